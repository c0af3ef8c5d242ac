// gk_probe.hpp - ambient-cube probe grid on the device: colour packing and the
// trilinear, occlusion-tested lookup interpolateAmbientCubesV2 (AmbientCube.slang:66-100,
// 135-232, 268-345). Used by the bake (probe.hip) and by REF_V2 path termination
// (wavefront.hip).
//
// Probe (x, y, z) sits at (x, y, z) * unit + offset and is element
// y * sxy * sxy + z * sxy + x of both arrays.
#pragma once
#include "gk_ctx.hpp"

namespace gk {

struct ProbeDev {
    const gk_ambient_cube* cubes;  // nullptr: no grid (every lookup is "outside")
    const gk_voxel* voxels;
    uint32_t sxy, sz;
    float unit;
    float off[3];
};

constexpr float kProbeMaxIlluminance = 512.f;  // MAX_ILLUMINANCE (AmbientCube.slang:4)

__host__ __device__ inline float clamp01(float x) { return fminf(fmaxf(x, 0.f), 1.f); }

// packRGB10A2 / unpackRGB10A2 (AmbientCube.slang:66-87)
__device__ inline uint32_t probe_pack(float4 c) {
    const float r = clamp01(c.x / kProbeMaxIlluminance), g = clamp01(c.y / kProbeMaxIlluminance);
    const float b = clamp01(c.z / kProbeMaxIlluminance), a = clamp01(c.w / kProbeMaxIlluminance);
    return uint32_t(r * 1023.0f) | (uint32_t(g * 1023.0f) << 10) | (uint32_t(b * 1023.0f) << 20) |
           (uint32_t(a * 3.0f) << 30);
}
// x / C, correctly rounded, for the whole numbers the packed fields hold (0 .. C): a product
// by the reciprocal and one residual step in place of an IEEE division, the same bits for
// every one of them
template <int C>
__device__ inline float div_field(uint32_t x) {
    constexpr float c = float(C), rc = 1.0f / float(C);
    const float f = float(x);
    const float q = f * rc;
    return fmaf(fmaf(-q, c, f), rc, q);
}
__device__ inline float4 probe_unpack(uint32_t p) {
    const float r = div_field<1023>(p & 0x3ffu);
    const float g = div_field<1023>((p >> 10) & 0x3ffu);
    const float b = div_field<1023>((p >> 20) & 0x3ffu);
    return make_float4(r * kProbeMaxIlluminance, g * kProbeMaxIlluminance, b * kProbeMaxIlluminance,
                       0.f * kProbeMaxIlluminance);
}

__device__ inline void acc_scaled(float4& acc, float w, float4 v) {
    acc.x = acc.x + w * v.x;
    acc.y = acc.y + w * v.y;
    acc.z = acc.z + w * v.z;
    acc.w = acc.w + w * v.w;
}

// A probe's faces as they lie in memory: the + and - face of an axis are neighbours
// ((+z, -z), (+y, -y), (+x, -x), bounced then direct, then the two sky words).
template <bool FULL>
struct ProbeFaces {
    uint2 d[3];
    uint2 b[FULL ? 3 : 1];
    uint2 sky;
};
template <bool FULL>
__device__ inline ProbeFaces<FULL> probe_faces(const gk_ambient_cube* cubes, size_t idx) {
    const uint2* w = reinterpret_cast<const uint2*>(cubes + idx);  // 56-byte records
    ProbeFaces<FULL> f;
#pragma unroll
    for (int k = 0; k < 3; ++k) f.d[k] = w[3 + k];
    if (FULL) {
#pragma unroll
        for (int k = 0; k < 3; ++k) f.b[FULL ? k : 0] = w[k];
        f.sky = w[6];
    }
    return f;
}

// sampleAmbientCubeHL2_DI (direct faces only) and sampleAmbientCubeHL2_Full (direct +
// bounced faces, sky visibility in w), AmbientCube.slang:117-232. Of an axis's two faces one
// has weight zero and adds an exact zero to sums that are not negative, so only the other one
// is unpacked (in the order +x or -x, +y or -y, +z or -z of the shader's sums).
__device__ inline uint32_t pick(bool first, uint2 v) {
    return first ? +v.x : +v.y;  // of values: a choice of the two members' addresses goes through scratch
}
template <bool FULL>
__device__ inline float4 probe_sample(const ProbeFaces<FULL>& c, f3 n) {
    const float wx = fmaxf(n.x, 0.f) + fmaxf(-n.x, 0.f);
    const float wy = fmaxf(n.y, 0.f) + fmaxf(-n.y, 0.f);
    const float wz = fmaxf(n.z, 0.f) + fmaxf(-n.z, 0.f);
    const bool px = n.x > 0.f, py = n.y > 0.f, pz = n.z > 0.f;
    const float sum = wx + wy + wz;
    float4 col = make_float4(0.f, 0.f, 0.f, 0.f);
    acc_scaled(col, wx, probe_unpack(pick(px, c.d[2])));
    acc_scaled(col, wy, probe_unpack(pick(py, c.d[1])));
    acc_scaled(col, wz, probe_unpack(pick(pz, c.d[0])));
    const float norm = sum > 0.f ? 1.0f / sum : 1.0f;
    if (FULL) {
        acc_scaled(col, wx, probe_unpack(pick(px, c.b[FULL ? 2 : 0])));
        acc_scaled(col, wy, probe_unpack(pick(py, c.b[FULL ? 1 : 0])));
        acc_scaled(col, wz, probe_unpack(pick(pz, c.b[0])));
        // sky bytes: +z -z +y -y, +x -x
        float skyvis = float((c.sky.x >> (pz ? 0 : 8)) & 0xffu) * wz;
        skyvis = skyvis + float((c.sky.x >> (py ? 16 : 24)) & 0xffu) * wy;
        skyvis = skyvis + float((c.sky.y >> (px ? 0 : 8)) & 0xffu) * wx;
        col.x = col.x * norm;
        col.y = col.y * norm;
        col.z = col.z * norm;
        skyvis = skyvis * norm;
        col.w = skyvis / 255.0f;
    } else {
        col.x = col.x * norm;
        col.y = col.y * norm;
        col.z = col.z * norm;
        col.w = col.w * norm;
    }
    return col;
}

// interpolateAmbientCubesV2 (AmbientCube.slang:268-345): the eight probes around pos,
// trilinear weights, a probe skipped when its voxel is inside geometry or when the
// direction-blended free distance of the voxel is shorter than the way to pos.
// Without branches: the eight voxels are loaded together and give the eight weights (zero for
// a skipped probe), then the cubes of several probes at a time; a skipped probe's cube is read
// where the last used one lies and adds an exact zero. Loads under a branch per probe were
// sixteen dependent memory round trips, which is what a launch with few threads waits for, and
// twelve unpacked faces with three divisions each were most of the arithmetic of a large one.
// k_bake_face over the city (64 x 32 x 64 probes, 13 M rays): 775 -> 380 us; the shading of a
// few hundred terminated paths 42 -> 24 us.
template <bool FULL>
__device__ inline float4 probe_lookup(const ProbeDev& P, f3 pos, f3 normal) {
    if (!P.cubes) return make_float4(0.f, 0.f, 0.f, 1.f);
    const f3 np = f3{(pos.x - P.off[0]) / P.unit, (pos.y - P.off[1]) / P.unit, (pos.z - P.off[2]) / P.unit};
    const float lim_xy = float(int(P.sxy) - 2), lim_z = float(int(P.sz) - 2);
    // written so that a NaN position also counts as outside
    if (!(np.x >= 0.f && np.y >= 0.f && np.z >= 0.f && np.x <= lim_xy && np.y <= lim_z && np.z <= lim_xy))
        return make_float4(0.f, 0.f, 0.f, 1.f);
    const f3 fl = f3{floorf(np.x), floorf(np.y), floorf(np.z)};
    const int bx = int(fl.x), by = int(fl.y), bz = int(fl.z);
    const f3 fr = np - fl;
    const uint32_t idx0 = (uint32_t(by) * P.sxy + uint32_t(bz)) * P.sxy + uint32_t(bx);  // at most 2^26 probes
    uint2 vox[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const uint32_t idx = idx0 + uint32_t(i & 1) + (uint32_t((i >> 1) & 1) * P.sxy + uint32_t((i >> 2) & 1)) * P.sxy;
        vox[i] = reinterpret_cast<const uint2*>(P.voxels + idx)[1];  // dist_gg_z01, dist_x01_y01
    }
    float wt[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int ox = i & 1, oy = (i >> 1) & 1, oz = (i >> 2) & 1;
        const uint32_t u0 = vox[i].x, u1 = vox[i].y;
        const float inside = div_field<255>((u0 >> 8) & 0xffu);
        const f3 to_local = fr - f3{float(ox), float(oy), float(oz)};
        const float dist = length(to_local);
        const f3 dir = normalize(to_local);
        // of an axis's two terms one is an exact zero; the sum's order is x, y, z
        const float dx = div_field<255>((u1 >> (dir.x > 0.f ? 0 : 8)) & 0xffu);
        const float dy = div_field<255>((u1 >> (dir.y > 0.f ? 16 : 24)) & 0xffu);
        const float dz = div_field<255>((u0 >> (dir.z > 0.f ? 16 : 24)) & 0xffu);
        const float hit_len = sqrtf(fabsf(dir.x)) * dx + sqrtf(fabsf(dir.y)) * dy + sqrtf(fabsf(dir.z)) * dz;
        const float wx = ox == 0 ? (1.0f - fr.x) : fr.x;
        const float wy = oy == 0 ? (1.0f - fr.y) : fr.y;
        const float wz = oz == 0 ? (1.0f - fr.z) : fr.z;
        wt[i] = (inside < 0.01f || dist > hit_len + 0.05f) ? 0.f : wx * wy * wz;
    }
    float total = 0.f;
    float4 res = make_float4(0.f, 0.f, 0.f, 0.f);
    uint32_t at = idx0;
    constexpr int G = FULL ? 2 : 4;  // cubes in flight (14 and 6 registers each)
#pragma unroll
    for (int q = 0; q < 8; q += G) {
        ProbeFaces<FULL> faces[G];
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const int i = q + k;
            const uint32_t idx = idx0 + uint32_t(i & 1) + (uint32_t((i >> 1) & 1) * P.sxy + uint32_t((i >> 2) & 1)) * P.sxy;
            at = wt[i] > 0.f ? idx : at;
            faces[k] = probe_faces<FULL>(P.cubes, at);
        }
#pragma unroll
        for (int k = 0; k < G; ++k) {
            const float w = wt[q + k];
            const float4 s = probe_sample<FULL>(faces[k], normal);
            res.x = res.x + s.x * w;
            res.y = res.y + s.y * w;
            res.z = res.z + s.z * w;
            res.w = res.w + s.w * w;
            total = total + w;
        }
    }
    if (!(total > 0.f)) return make_float4(0.f, 0.f, 0.f, 0.f);
    return make_float4(res.x / total, res.y / total, res.z / total, res.w / total);
}

}  // namespace gk
