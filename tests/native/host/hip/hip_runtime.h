// What device_physics.h needs to compile for the host: its functions are plain
// C++ apart from the markers and a few hardware functions of the FP32 form.
#pragma once
#include <cmath>
#include <cstdint>
#include <math.h>
#define __host__
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_sinf(x) sinf(6.28318530717958647692f * (x))
#define __builtin_amdgcn_cosf(x) cosf(6.28318530717958647692f * (x))
#define __logf(x) logf(x)
