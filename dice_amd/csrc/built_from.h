// Included in front of every translation unit: leaves in its object which sources and flags it was compiled from
// (DICE_BUILT_FROM, set by the build), so that a library can be told from one of other sources, object by object.
#pragma once
#ifndef __HIP_DEVICE_COMPILE__
__attribute__((used)) static const char dice_built_from[] = DICE_BUILT_FROM;
#endif
