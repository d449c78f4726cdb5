"""What the build leaves behind (dice_amd/build.py): a library whose every object is of the
sources beside it, or none at all (no GPU, nothing is compiled)."""
import os
import shutil

import pytest

from dice_amd import build, lib


def test_library_is_built_from_the_sources_beside_it():
    with open(lib.LIB_PATH, "rb") as f:
        assert build.stale_units(f.read(), build.source_digest()) == []


def test_digest_covers_kernels_headers_generators_and_flags(tmp_path, monkeypatch):
    csrc, include = tmp_path / "csrc", tmp_path / "include"
    shutil.copytree(build.CSRC, csrc)
    shutil.copytree(build.INCLUDE, include)
    same = build.source_digest(str(csrc), str(include))
    assert same == build.source_digest()
    for path in (csrc / "gate.hip", csrc / "persist_dma.h", csrc / "gen_persist64_asm.py", include / "dice_moe.h"):
        old = path.read_bytes()
        path.write_bytes(old + b"\n")
        assert build.source_digest(str(csrc), str(include)) != same, path
        path.write_bytes(old)
    (csrc / "notes.txt").write_text("not a source")
    assert build.source_digest(str(csrc), str(include)) == same
    monkeypatch.setattr(build, "HIP_FLAGS", build.HIP_FLAGS + ["-DX"])
    assert build.source_digest(str(csrc), str(include)) != same
    shutil.rmtree(include)                               # nothing to build from: nothing to compare with
    assert build.source_digest(str(csrc), str(include)) is None


def test_one_object_of_other_sources_is_noticed(tmp_path, monkeypatch):
    digest, other = "a" * 64, "b" * 64
    image = {s: f"dice_moe unit {s} {digest}\0" for s in build.SOURCES}
    assert build.stale_units("..".join(image.values()).encode(), digest) == []
    name = build.SOURCES[-2]
    mixed = dict(image, **{name: f"dice_moe unit {name} {other}\0"})
    assert build.stale_units("..".join(mixed.values()).encode(), digest) == [name]
    both = "..".join([*image.values(), mixed[name]])
    assert build.stale_units(both.encode(), digest) == [name]
    del mixed[name]
    assert build.stale_units("..".join(mixed.values()).encode(), digest) == [name]
    assert build.stale_units(b"", digest) == build.SOURCES         # a library from before objects named their sources
    # ... and refused
    path = tmp_path / "libdice_moe.so"
    path.write_bytes("..".join(image.values()).encode())
    monkeypatch.setattr(lib, "LIB_PATH", str(path))
    monkeypatch.setattr(lib, "_lib", None)
    with pytest.raises(lib.DiceError, match="built from other sources"):
        lib.load()


@pytest.mark.parametrize("fails", ["compiler", "register check"])
def test_failed_build_leaves_no_library(tmp_path, monkeypatch, fails):
    monkeypatch.setattr(build, "BUILD_DIR", str(tmp_path / "_build"))
    os.makedirs(build.BUILD_DIR)
    objects = [os.path.join(build.BUILD_DIR, os.path.splitext(s)[0] + ".o") for s in build.SOURCES]
    target = tmp_path / "lib.so"
    for path in [target, *objects]:
        with open(path, "w") as f:
            f.write("of an older build")

    def run(cmd, **kw):
        if "-c" in cmd:
            obj = cmd[cmd.index("-o") + 1]
            bad = "grouped_gemm_persist_f8" in obj
            if not (bad and fails == "compiler"):
                open(obj, "w").close()
            return type("R", (), dict(returncode=1 if bad and fails == "compiler" else 0, stderr="no such operand"))()
        raise AssertionError("linked")

    def check(path):
        if fails == "register check" and "persist_f8" in path:
            raise RuntimeError("compiler placed values")

    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build.subprocess, "run", run)
    monkeypatch.setattr("dice_amd.check_acc_regs.check", check)
    with pytest.raises(RuntimeError):
        build.build_library(verbose=False, out=str(target))
    assert not target.exists()
    bad = os.path.join(build.BUILD_DIR, "grouped_gemm_persist_f8.o")
    assert not os.path.exists(bad)
