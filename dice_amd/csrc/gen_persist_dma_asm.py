"""Generates ``persist_dma_asm.inc``: the k-loop of the expert GEMM kernels whose
operands go from memory straight to LDS (gemm_persist_dma_body in csrc/persist_dma.h,
gemm_persist_f8_asm_body in csrc/grouped_gemm_persist_f8.hip), as inline assembly on
fixed registers.

Two things set it apart from the loop of gen_persist64_asm.py, which stages operands
in registers and multiplies with 32 x 32 x 16 instructions.

*   Products of 16 x 16 x 32 (16-bit operands).  The matrix pipe needs as many cycles as for two of
    32 x 32 x 16 and forms the same bits (bf16 and fp16, measured), but at the board's
    power limit it runs N(0,1) operands at 2020 TFLOP/s instead of 1780 (bf16, operands in
    registers, nothing else running; fp16 1890 / 1655; zeros, which the limit leaves
    alone, 2440 either way).
*   Copies from memory to LDS (``buffer_load_dwordx4 ... lds``).  An LDS write
    of 16 bytes per lane takes 13 cycles of the LDS and of the wave's issue, which an
    instruction of 16 cycles does not hide: 64 products of 16 x 16 x 32 (1024 cycles)
    with 16 fragment reads take 1073 cycles, with 8 LDS writes as well 1210 to 1340 by
    where these stand, with 8 copies instead 1072.

Register plan of a wave (fixed numbers):
  v[0:63], v[64:127]   fragments of k-block 0 / 1: weight block j at 8 j, row block i at 32 + 8 i (32 rows x
                       32 k; rows 0-15 of a block in the first four registers, 16-31 in the others)
  a[..]     the sums: block (i, j) at 16 (ACC0 + i TN + j), there half v of the rows
            and half u of the weights at + 8 v + 4 u
  everything else (addresses, descriptors) comes in as asm operands.

A step is 64 k (128-byte rows) in LDS slot s % 2, two k-blocks of 32.  What limits the loop is how
long a copy may take: the slot of step s + 2 is that of step s, so both k-blocks' fragments have
registers of their own, those of k-block 1 are read during the first half of k-block 0, and the
fragments of step s + 1 as late as its products allow.  Two statements per step s (of 2 n block
products, n = 16 for tiles of 256 weight rows):
  T1  products 0 .. n / 2: reads k-block 1's fragments.
  (compiled code moves the load side on, possibly into the next tile)
  T2  waits for this wave's reads of slot s, barrier: the slot is free.  The other products, the
      copies of step s + 2 spread over them.  At product 3 n / 2: waits for this wave's copies of
      step s + 1, barrier: every wave's have landed; reads the fragments of its k-block 0.
A copy has 25 to 48 block products (1600 to 3000 cycles) to land.  Activations go first and the weights
behind them: 16384 grouped rows of DiT-XL width, 8 experts, zero weights (so that the power limit plays no
part), fc1 / fc2 alone 234 / 128 us, alternating 250 / 148, weights first 249 / 144, one copy behind every product and
then none 260 / 151.  Fragments replaced in place, which leaves a copy 18 to 32 products: 249 / 149.
The first step of a tile waits for no copies: the kernel waits for all of them in front of the
epilogue's stores, which retire in another order (``_v1``; the first k-block's products then start the sums).

fp8 kinds: a step is 128 k (the same 128 bytes), a k-block 64; a block product is one instruction of
32 x 32 x 64 (its sums: element e in register e), the two parts of a fragment are the two 16-byte chunks of
a row that a lane holds.

The script simulates the instruction stream, finds for every instruction the memory
operations it depends on and emits ``s_waitcnt`` with the exact number of younger
operations that may still be outstanding (LDS reads complete in order, vector loads
too).

Usage: python gen_persist_dma_asm.py [out.inc] (dice_amd/build.py calls generate()).
"""
from __future__ import annotations

KINDS = {
    # weight blocks per wave, copies of weight rows per wave and step, row offsets of the weight blocks from the
    # wave's first, first block of sums, first copy that takes the second weight descriptor
    0: dict(name="fc1 SwiGLU, 256 weight rows", TN=4, CB=8, brow=[0, 32, 128, 160], acc0=0, up_from=4),
    1: dict(name="fc2, 192 weight rows", TN=3, CB=6, brow=[0, 32, 64], acc0=4, up_from=99),
    2: dict(name="fc2, 128 weight rows", TN=2, CB=4, brow=[0, 32], acc0=8, up_from=99),
    3: dict(name="256 weight rows", TN=4, CB=8, brow=[0, 32, 64, 96], acc0=0, up_from=99),
    4: dict(name="fc1 SwiGLU, 128 weight rows", TN=2, CB=4, brow=[0, 64], acc0=8, up_from=2),
    5: dict(name="fp8 fc1 SwiGLU, 256 weight rows", TN=4, CB=8, brow=[0, 32, 128, 160], acc0=0, up_from=4, f8=True),
    6: dict(name="fp8, 256 weight rows", TN=4, CB=8, brow=[0, 32, 64, 96], acc0=0, up_from=99, f8=True),
}
CA = 8                    # copies of activation rows per wave and step (load l: tile rows 32 l + 8 wave ..)
TM = 4
A_BYTES, SLOT = 256 * 128, 64 * 1024
LGKM_MAX = 15


class Stream:
    """An instruction stream with in-order LDS and vector-memory queues."""

    def __init__(self, kind, live):
        self.k = KINDS[kind]
        self.live = live
        self.lds_issued = self.lds_done = 0
        self.vm_issued = 0
        self.frag_op = {}         # first register of a fragment part -> index of the LDS read that fills it
        self.out = None           # lines of the statement being recorded
        self.waits, self.needed = {}, set()
        self.key, self.site = None, 0

    # ---- recording ----
    def begin(self, key):
        self.key, self.site, self.out = key, 0, []

    def end(self):
        lines, self.out = self.out, None
        return lines

    def emit(self, text):
        self.out.append(text)

    def wait_lds(self, need_done):
        """LDS reads up to index need_done (exclusive) must be complete.  The same statement runs in several places of
        the stream: the strictest count is kept, and the wait is written if any place needs it."""
        site = (self.key, self.site)
        self.site += 1
        n = max(0, min(self.lds_issued - need_done, LGKM_MAX))
        self.waits[site] = min(self.waits.get(site, n), n)
        if need_done > self.lds_done:
            self.needed.add(site)
            self.lds_done = max(self.lds_done, self.lds_issued - n)
        self.emit(("WAIT", site))

    # ---- instructions ----
    @staticmethod
    def frag_reg(kb, which, idx):
        return 64 * kb + 8 * idx + (0 if which == "w" else 32)

    def read(self, slot, kb, which, idx, t):
        """Part t of fragment (which, idx) of k-block kb of slot `slot`: rows 16 t .. (fp8: chunk t)."""
        reg = self.frag_reg(kb, which, idx) + 4 * t
        row = self.k["brow"][idx] if which == "w" else 64 * idx
        if self.k.get("f8"):
            addr = 2 * kb + t
        else:
            addr, row = kb, row + 16 * t
        self.emit(f"ds_read_b128 v[{reg}:{reg + 3}], %[r{'b' if which == 'w' else 'a'}{slot}{addr}] offset:{row * 128}")
        self.frag_op[reg] = self.lds_issued
        self.lds_issued += 1

    def copies(self):
        """A step's copies: l < CA activation rows, from CA on weight rows."""
        return list(range(CA + self.k["CB"]))

    def copy_address(self, slot, l):
        # (the LDS address of a copy sits in m0; whoever issues the copy puts an instruction between the two)
        off = slot * SLOT + (l * 4096 if l < CA else A_BYTES + (l - CA) * 4096)
        self.emit(f"s_add_u32 m0, %[lw], {off}")

    def copy(self, l):
        if l < CA:
            self.emit(f"buffer_load_dwordx4 %[va{l}], %[dA], %[koff] offen lds")
        else:
            i = l - CA
            self.emit(f"buffer_load_dwordx4 %[vb{i}], %[dB{1 if i >= self.k['up_from'] else 0}], %[koff] offen lds")
        self.vm_issued += 1

    def product(self, kb, i, j, first):
        """The instructions of a block product: (fragment parts it reads, text)."""
        w, a = self.frag_reg(kb, "w", j), self.frag_reg(kb, "a", i)
        acc = 16 * (self.k["acc0"] + i * self.k["TN"] + j)
        if self.k.get("f8"):
            d = f"a[{acc}:{acc + 15}]"
            return [((w, w + 4, a, a + 4), f"MFMA8 {d}, v[{w}:{w + 7}], v[{a}:{a + 7}], {'0' if first else d}")]
        four = []
        for u, v in ((0, 0), (0, 1), (1, 1), (1, 0)):   # (one operand changes at a time)
            d = f"a[{acc + 8 * v + 4 * u}:{acc + 8 * v + 4 * u + 3}]"
            four.append(((w + 4 * u, a + 4 * v), f"MFMA {d}, v[{w + 4 * u}:{w + 4 * u + 3}], "
                                                 f"v[{a + 4 * v}:{a + 4 * v + 3}], {'0' if first else d}"))
        return four

    # ---- the order of a k-block ----
    def quads(self):
        """The block products of a k-block, two rows x two columns at a time, down one column and up the next."""
        rows, tn = range(self.live), self.k["TN"]
        prods = []
        for r in range(0, self.live, 2):
            for c in range(0, tn, 2):
                pair = [i for i in (r, r + 1) if i in rows]
                prods += [(i, c) for i in pair] + [(i, c + 1) for i in reversed(pair) if c + 1 < tn]
        return prods

    def parts(self, slot, kb):
        """The reads of a k-block's fragments in the order in which its products need them."""
        seen = []
        for i, j in self.quads():
            seen += [f for f in (("w", j), ("a", i)) if f not in seen]
        return [(slot, kb, *f, t) for f in seen for t in (0, 1)]

    def run(self, prods, start, reads, copies, cslot):
        """The block products `prods` of (k-block, row block, weight block), of which those of k-block 0 start the sums
        if `start`; `reads` spread behind them, copies[g] behind product g, into slot cslot."""
        for g, prod in enumerate(prods):
            texts = self.product(*prod, start and prod[0] == 0)
            n_side = len(texts)
            side = [[] for _ in texts]
            mine = [r for n, r in enumerate(reads) if n * len(prods) // len(reads) == g]
            for n, what in enumerate(mine):
                side[n * n_side // len(mine)].append(("r", what))
            for n, l in enumerate(copies[g]):
                if len(copies[g]) * 2 <= n_side:
                    side[2 * n].append(("m", l))
                    side[2 * n + 1].append(("c", l))
                else:
                    side[n * n_side // len(copies[g])] += [("m", l), ("nop", 0), ("c", l)]
            for x, (parts, text) in enumerate(texts):
                self.wait_lds(max(self.frag_op[r] for r in parts) + 1)
                self.emit(text)
                for kind, what in side[x]:
                    if kind == "r":
                        self.read(*what)
                    elif kind == "m":
                        self.copy_address(cslot, what)
                    elif kind == "nop":
                        self.emit("s_nop 0")
                    else:
                        self.copy(what)

    def step(self):
        """(block products of a step, how many of them the first statement takes, the one behind the second barrier)."""
        kb = self.quads()
        return [(b, i, j) for b in (0, 1) for i, j in kb], max(1, len(kb) // 2), len(kb) * 3 // 2

    def t1(self, slot, var):
        prods, head, _ = self.step()
        self.run(prods[:head], var == 1, self.parts(slot, 1), [[]] * head, 0)

    def t2(self, slot, var):
        self.emit("s_waitcnt lgkmcnt(0)")
        self.lds_done = self.lds_issued
        self.emit("s_barrier")
        prods, head, land = self.step()
        copies = [[] for _ in prods]
        for n, l in enumerate(self.copies()):
            copies[head + n * (len(prods) - head) // len(self.copies())].append(l)
        self.run(prods[head:land], var == 1, [], copies[head:land], slot)
        if var != 1:
            self.emit(f"s_waitcnt vmcnt({sum(map(len, copies[:land]))})")    # (younger: these copies)
        self.emit("s_barrier")
        self.run(prods[land:], False, self.parts(slot ^ 1, 0), copies[land:], slot)

    def load(self, slot):
        for l in self.copies():
            self.copy_address(slot, l)
            self.emit("s_nop 0")
            self.copy(l)

    def read_first(self):
        for what in self.parts(0, 0):
            self.read(*what)


def render(lines, waits, needed):
    out = []
    for ln in lines:
        if isinstance(ln, tuple):
            if ln[1] in needed:
                out.append(f"s_waitcnt lgkmcnt({waits[ln[1]]})")
        else:
            out.append(ln)
    return out


def simulate(kind, live):
    """Runs the kernel's instruction stream: prologue, then tiles of eight steps.  Returns {name: lines}."""
    pieces = {}
    st = Stream(kind, live)

    def rec(name, fn, *args):
        st.begin(name)
        fn(*args)
        lines = st.end()
        if name in pieces:
            assert [x for x in pieces[name] if not isinstance(x, tuple)] == \
                   [x for x in lines if not isinstance(x, tuple)], name
        pieces[name] = lines

    rec("load_s0", st.load, 0)
    rec("load_s1", st.load, 1)
    for _ in range(3):
        rec("read_first", st.read_first)
        for s in range(8):
            slot, var = s & 1, 1 if s == 0 else 0
            rec(f"t1_s{slot}_v{var}", st.t1, slot, var)
            rec(f"t2_s{slot}_v{var}", st.t2, slot, var)
        st.lds_done = st.lds_issued       # the kernel waits for the LDS queue in front of the epilogue
    return {name: render(lines, st.waits, st.needed) for name, lines in pieces.items()}


def c_string(lines):
    return "\n".join(f'      "{ln}\\n"' for ln in lines)


def generate() -> str:
    out = ["// Generated by gen_persist_dma_asm.py - do not edit.  See that script for the register plan,",
           "// the order of the pieces and how the wait counts are derived.",
           "#pragma once"]
    for fam, macro, f8 in (("pdma", "PDMA", False), ("pdma8", "PDMA8", True)):
        table = {(kind, live): simulate(kind, live) for kind in KINDS for live in range(1, TM + 1)
                 if bool(KINDS[kind].get("f8")) == f8}
        for name in sorted(next(iter(table.values()))):
            out.append(f"template <int KIND, int LIVE>\n__device__ __forceinline__ void {fam}_{name}({macro}_PARAMS) {{")
            first = True
            for (kind, live), pcs in table.items():
                text = [ln.replace("MFMA8 ", '" DICE_MFMA8 " ').replace("MFMA ", '" DICE_MFMA_16X16 " ')
                        for ln in pcs[name]]
                out.append(f"  {'if' if first else 'else if'} constexpr (KIND == {kind} && LIVE == {live})")
                out.append("    asm volatile(")
                out.append(c_string(text))
                out.append(f"      {macro}_CONSTRAINTS);")
                first = False
            out.append("  else static_assert(KIND < 0, \"no such variant\");\n}")
    return "\n".join(out) + "\n"


if __name__ == "__main__":
    import sys
    if len(sys.argv) > 1:
        with open(sys.argv[1], "w") as f:
            f.write(generate())
    else:
        sys.stdout.write(generate())
