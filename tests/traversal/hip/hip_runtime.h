// What the traversal headers need of the HIP runtime to run on the CPU as a wave of one lane.
#pragma once
#include <cmath>
#include <cstdint>
#include <cstring>

#define __host__
#define __device__

struct float4 { float x, y, z, w; };
struct uint4 { uint32_t x, y, z, w; };
struct { uint32_t x = 1; } blockDim;
inline uint64_t __ballot(bool b) { return b ? 1u : 0u; }
inline int __popcll(uint64_t v) { return __builtin_popcountll(v); }
inline uint32_t __float_as_uint(float f) { uint32_t u; memcpy(&u, &f, 4); return u; }
inline float __uint_as_float(uint32_t u) { float f; memcpy(&f, &u, 4); return f; }
inline float4 make_float4(float x, float y, float z, float w) { return {x, y, z, w}; }
inline void atomicOr(uint32_t* p, uint32_t v) { *p |= v; }
