// lvn_device.hpp — device-side arithmetic of the chunk mesher (gfx950).
//
// Every function follows the operation order of the reference formula it
// cites, with no contraction (the library is compiled with -ffp-contract=off),
// correctly rounded division and sqrt (HIP's default for FP32), and float
// constants in place of the reference's unsuffixed double literals.  The
// permutation table lives in LDS (64 KiB of bytes, row = texel y) together
// with the decoded gradient vectors.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

#include "lvn_shared.h"

namespace lvn {

// LDS-resident noise tables, built by the host.  The 256 x 256 permutation table is
// stored in rows of 258 bytes with a wrap row: texel (x, y) at y * 258 + 1 + x for x, y
// in 0..256 (256 repeating 0), so a corner's texel, whose coordinates are the cell's
// wrapped ones plus 0 or 1, is one add away from the cell's base index with no wrap
// masks per corner (REPEAT addressing, cl/simplex.cl:59).  Each byte holds the texel's
// value plus one, mod 256, and byte y * 258 holds texel (0, y): snoise3's second read,
// at x = value with 255 wrapping to 0, is then row + stored byte with no compare.  The
// 16-entry gradient table is indexed by the stored byte's low four bits (rotated by one
// entry, so no subtraction is needed).  The gradients are stored as (x, y) pairs, 8 bytes
// an entry, and z components at the same 8-byte stride, the two blocks on bank rows: the
// 16 pairs fill the 32 banks once and the 16 z values take the even banks once, so a
// wave's reads never meet two addresses in one bank (equal gradients share an address;
// whole 16-byte entries put entries 8 apart in the same banks).  The gradient blocks
// come first: their offsets then fit the LDS instructions' 16-bit immediate, and a
// corner's two reads share one address, its index times 8.  snoise2 reads a pair,
// snoise3 a pair and a z.  66,688 bytes per workgroup.
struct alignas(128) NoiseLds {
    float2 gxy[kGradEntries];  // entry j: gradient (j - 1) & 15, components x and y
    float2 gz[kGradEntries];   // entry j: (z component, unused)
    uint8_t perm[kPermPaddedBytes];
};
static_assert(offsetof(NoiseLds, gz) == 128 && offsetof(NoiseLds, perm) == 256,
              "gradient blocks on bank rows, ahead of the permutation table");

// Cooperative copy of the tables into LDS (all threads of the block call it).
__device__ __forceinline__ void load_noise_tables(NoiseLds& lds, const uint8_t* __restrict__ perm,
                                                  const float4* __restrict__ grads) {
    const uint4* src = reinterpret_cast<const uint4*>(perm);
    uint4* dst = reinterpret_cast<uint4*>(lds.perm);
    for (int i = threadIdx.x; i < kPermPaddedBytes / 16; i += blockDim.x) dst[i] = src[i];
    for (int i = threadIdx.x; i < kGradEntries; i += blockDim.x) {
        const float4 g = grads[i];
        lds.gxy[i] = make_float2(g.x, g.y);
        lds.gz[i] = make_float2(g.z, 0.f);
    }
    __syncthreads();
}

// Correctly rounded square root of x >= 1 (and of +inf): the hardware square root,
// within 1 ulp, replaced by its lower or upper neighbour when the FMA residual
// x - neighbour * root says that one is nearer.  These are the steps of the
// compiler's IEEE sqrtf without its range scaling (taken below 2^-96 only) and its
// zero / infinity select (+inf already comes out as +inf: both residuals are NaN).
__device__ __forceinline__ float sqrt_ge1(float x) {
    const float s = __builtin_amdgcn_sqrtf(x);
    const float lo = __int_as_float(__float_as_int(s) - 1);
    const float hi = __int_as_float(__float_as_int(s) + 1);
    const float r = fmaf(-lo, s, x) <= 0.f ? lo : s;
    return fmaf(-hi, s, x) > 0.f ? hi : r;
}

// Correctly rounded 1 / d for d in [1, 2): the hardware reciprocal refined by one
// Newton step, then the quotient corrected twice by its FMA residual.  These are the
// steps of the compiler's IEEE division 1.f / d with its operand scaling and its
// special-case fixup left out: for this range neither changes a value.
__device__ __forceinline__ float recip_1_2(float d) {
    const float r0 = __builtin_amdgcn_rcpf(d);
    const float r1 = fmaf(fmaf(-d, r0, 1.f), r0, r0);
    const float q1 = fmaf(fmaf(-d, r1, 1.f), r1, r1);
    return fmaf(fmaf(-d, q1, 1.f), r1, q1);
}

__device__ __forceinline__ float clamp01(float v) { return fminf(fmaxf(v, 0.f), 1.f); }

// One snoise2 corner (cl/simplex.cl:123-153).  The squared distance and the
// gradient dot product are fused multiply-adds, as the restatement defines them
// (the reference's -cl-fast-relaxed-math build, src/compute.cpp:213, allows it).
// A corner beyond the radius (r < 0) contributes zero: r is clamped at +0, which
// gives that zero up to its sign (+0 times the dot product).  No result can see the
// sign: the corner sum of a point with a non-zero corner is unchanged by it, and
// every noise value feeds either fBm's fma chain, which starts at +0 (a zero noise
// value then adds +0 to a sum that is never -0), or the ridged form's fabsf.
__device__ __forceinline__ float corner2(const NoiseLds& T, int texel, float fx, float fy) {
    const float r = clamp01(0.5f - fmaf(fy, fy, fx * fx));
    const float2 g = T.gxy[T.perm[texel] & 15];
    const float t = r * r;
    return (t * t) * fmaf(g.y, fy, g.x * fx);
}

// snoise2, cl/simplex.cl:99-157.
__device__ __forceinline__ float snoise2(const NoiseLds& T, float px, float py) {
    const float F2 = 0.366025403784f;
    const float G2 = 0.211324865405f;
    const float C2 = 1.f - 2.f * G2;
    const float s = (px + py) * F2;
    const float pix = floorf(px + s);
    const float piy = floorf(py + s);
    const float t = (pix + piy) * G2;
    const float f0x = px - (pix - t);
    const float f0y = py - (piy - t);
    const int base = ((int)piy & 255) * kPermPitch + ((int)pix & 255) + 1;  // texel of the cell corner
    const int o1x = f0x > f0y ? 1 : 0;
    const int o1y = 1 - o1x;
    const float n0 = corner2(T, base, f0x, f0y);
    const float n1 = corner2(T, base + o1y * kPermPitch + o1x, (f0x - (float)o1x) + G2, (f0y - (float)o1y) + G2);
    const float n2 = corner2(T, base + kPermPitch + 1, f0x - C2, f0y - C2);
    return 70.f * ((n0 + n1) + n2);
}

// One snoise3 corner (cl/simplex.cl:181-226).  The second table read uses the
// first read's value as x texel; value 255 wraps to texel 0 (normalised REPEAT).
// `texel` is the corner's (x, y) texel, `zrow` the start of its z texel's row; the
// stored byte (value + 1, or 0 for 255) is the second read's offset in that row.
// r is clamped at +0 as in corner2.
__device__ __forceinline__ float corner3(const NoiseLds& T, int texel, int zrow, float fx, float fy, float fz) {
    const int w = T.perm[texel];
    const float r = clamp01(0.6f - fmaf(fz, fz, fmaf(fy, fy, fx * fx)));
    const int j = T.perm[zrow + w] & 15;
    const float2 g = T.gxy[j];
    const float t = r * r;
    return (t * t) * fmaf(T.gz[j].x, fz, fmaf(g.y, fy, g.x * fx));
}

// snoise3, cl/simplex.cl:159-230 (simplex ranking of :74-97).
__device__ __forceinline__ float snoise3(const NoiseLds& T, float px, float py, float pz) {
    const float F3 = 0.333333333333f;
    const float G3 = 0.166666666667f;
    const float C2 = 2.f * G3;
    const float C3 = 1.f - 3.f * G3;
    const float s = ((px + py) + pz) * F3;
    const float pix = floorf(px + s);
    const float piy = floorf(py + s);
    const float piz = floorf(pz + s);
    const float t = ((pix + piy) + piz) * G3;
    const float f0x = px - (pix - t);
    const float f0y = py - (piy - t);
    const float f0z = pz - (piz - t);
    const int base = ((int)piy & 255) * kPermPitch + ((int)pix & 255) + 1;  // (x, y) texel of the cell corner
    const int zrow = ((int)piz & 255) * kPermPitch;
    const int xy = f0x >= f0y ? 1 : 0;
    const int xz = f0x >= f0z ? 1 : 0;
    const int yz = f0y >= f0z ? 1 : 0;
    const int rx = xy + xz;
    const int ry = (1 - xy) + yz;
    const int rz = (1 - xz) + (1 - yz);
    const int a1x = rx >> 1, a1y = ry >> 1, a1z = rz >> 1;            // rank 2 -> 1
    const int a2x = rx > 0 ? 1 : 0, a2y = ry > 0 ? 1 : 0, a2z = rz > 0 ? 1 : 0;  // rank >= 1 -> 1
    // f0 - offset for offsets 0 and 1: f0 - 0.f is f0 itself (also for -0)
    const float g0x = f0x - 1.f, g0y = f0y - 1.f, g0z = f0z - 1.f;
    const float n0 = corner3(T, base, zrow, f0x, f0y, f0z);
    const float n1 = corner3(T, base + a1y * kPermPitch + a1x, zrow + a1z * kPermPitch, (a1x ? g0x : f0x) + G3,
                             (a1y ? g0y : f0y) + G3, (a1z ? g0z : f0z) + G3);
    const float n2 = corner3(T, base + a2y * kPermPitch + a2x, zrow + a2z * kPermPitch, (a2x ? g0x : f0x) + C2,
                             (a2y ? g0y : f0y) + C2, (a2z ? g0z : f0z) + C2);
    const float n3 = corner3(T, base + kPermPitch + 1, zrow + kPermPitch, f0x - C3, f0y - C3, f0z - C3);
    return 32.f * (((n0 + n1) + n2) + n3);
}

// BasicFractal, cl/noise.cl:8-36.
__device__ __forceinline__ float fbm2(const NoiseLds& T, int octaves, float freq, float lac, float gain, float x,
                                      float y) {
    float px = x * freq, py = y * freq, amp = 1.f, n = 0.f;
    for (int i = 0; i < octaves; ++i) {
        n = fmaf(snoise2(T, px, py), amp, n);
        px = px * lac;
        py = py * lac;
        amp = amp * gain;
    }
    return n;
}

// The same fractal over snoise3.
__device__ __forceinline__ float fbm3(const NoiseLds& T, int octaves, float freq, float lac, float gain, float x,
                                      float y, float z) {
    float px = x * freq, py = y * freq, pz = z * freq, amp = 1.f, n = 0.f;
    for (int i = 0; i < octaves; ++i) {
        n = fmaf(snoise3(T, px, py, pz), amp, n);
        px = px * lac;
        py = py * lac;
        pz = pz * lac;
        amp = amp * gain;
    }
    return n;
}


// RidgedMultiFractal, cl/noise.cl:42-81 (pow(f, -1) as 1 / f).
__device__ __forceinline__ float ridged(const NoiseLds& T, int octaves, float lac, float gain, float offset, float x,
                                        float y) {
    float px = x, py = y;
    float signal = offset - fabsf(snoise2(T, px, py));
    signal = signal * signal;
    float n = signal, freq = 1.f;
    for (int i = 0; i < octaves; ++i) {
        px = px * lac;
        py = py * lac;
        const float weight = clamp01(signal * gain);
        signal = offset - fabsf(snoise2(T, px, py));
        signal = signal * weight;
        const float expo = 1.f / freq;
        freq = freq * lac;
        n = n + signal * expo;
    }
    return n * (1.f / (float)octaves);
}

// Terrain, cl/noise.cl:205-223.
__device__ __forceinline__ float leven_terrain(const NoiseLds& T, float x, float z) {
    const float qx = x * (1.f / 2000.f);
    const float qy = z * (1.f / 2000.f);
    const float r = clamp01(0.8f * ridged(T, 7, 2.114352f, 1.5241f, 1.f, qx, qy));
    float billow = 0.6f * fbm2(T, 4, 0.24f, 1.8754f, 0.433f, -4.33f * qx, 7.98f * qy);
    billow = (0.5f * billow) + 0.5f;
    const float n = billow * r;
    float b2 = 0.6f * fbm2(T, 2, 0.63f, 2.2f, 0.15f, qx, qy);
    b2 = (b2 * 0.5f) + 0.5f;
    return n + b2;
}

// A kernel's field kind: its template argument, or the descriptor's in the kernels that
// are not timed (kAnyField).  A kernel built for one kind holds no other kind's code, whose
// live values cost it scalar registers.
constexpr int kAnyField = -1;
template <int kKind>
__device__ __forceinline__ int field_kind(const FieldParams& F) {
    return kKind == kAnyField ? F.kind : kKind;
}

// Height term H(x, z) of every field kind: density = y - H (cl/noise.cl:265-266).
template <int kKind>
__device__ __forceinline__ float height_term(const FieldParams& F, const NoiseLds& T, float x, float z) {
    if (field_kind<kKind>(F) == LVN_FIELD_LEVEN_TERRAIN) return 900.f * leven_terrain(T, x, z);
    return F.hamp * fbm2(T, F.hoct, F.hfreq, F.hlac, F.hgain, x, z);
}

// Cave term of LVN_FIELD_TERRAIN_CAVES.
__device__ __forceinline__ float cave_term(const FieldParams& F, const NoiseLds& T, float x, float y, float z) {
    return fbm3(T, F.coct, F.cfreq, F.clac, F.cgain, x, y, z) - F.cthr;
}

// density = max(a, cave) with a = y - H.  The cave term is bounded by F.cave_cut
// (|snoise3| <= 1.19 times the sum of octave amplitudes, minus the threshold);
// when a exceeds it, max(a, cave) == a exactly and the cave term is skipped.
template <int kKind>
__device__ __forceinline__ float combine(const FieldParams& F, const NoiseLds& T, float a, float x, float y, float z) {
    if (field_kind<kKind>(F) != LVN_FIELD_TERRAIN_CAVES || a > F.cave_cut) return a;
    return fmaxf(a, cave_term(F, T, x, y, z));
}

// ---------------------------------------------------------------------------
// leven's height term at the four points of a central difference, (x + h, z), (x - h, z),
// (x, z + h), (x, z - h).  They lie 0.002 apart, so at almost every octave all four of a
// lane's points fall into one simplex cell, and the cell's gradients (all of snoise2's LDS
// reads and their addresses) are found once for them.  Each point's value is formed by
// snoise2's own expressions, so nothing changes in it; a wave with a lane whose points
// straddle a cell takes the plain form for that octave.  A coordinate's three values
// c[0..2] = (c, c + h, c - h) are scaled octave by octave as fbm2 and ridged scale a point's.
// Only for this field: the others' frequencies and lacunarities are powers of two and edges
// sample them at multiples of 1/16 voxel, so the points around which they are differenced
// lie on cell borders so often that no wave has 64 lanes without one (measured there: no
// LDS read saved, 10% more VALU).
// ---------------------------------------------------------------------------

__device__ constexpr int kNear2X[4] = {1, 2, 0, 0}, kNear2Z[4] = {0, 0, 1, 2};

__device__ __forceinline__ void snoise2_near(const NoiseLds& T, const float x[3], const float z[3], float out[4]) {
    const float F2 = 0.366025403784f;
    const float G2 = 0.211324865405f;
    const float C2 = 1.f - 2.f * G2;
    float fx[4], fy[4], cx = 0.f, cy = 0.f;
    bool upper = false, same = true;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float px = x[kNear2X[i]], py = z[kNear2Z[i]];
        const float s = (px + py) * F2;
        const float pix = floorf(px + s);
        const float piy = floorf(py + s);
        const float t = (pix + piy) * G2;
        fx[i] = px - (pix - t);
        fy[i] = py - (piy - t);
        const bool u = fx[i] > fy[i];
        if (i == 0) {
            cx = pix;
            cy = piy;
            upper = u;
        } else {
            same = same && pix == cx && piy == cy && u == upper;
        }
    }
    if (__ballot(!same) == 0) {
        const int base = ((int)cy & 255) * kPermPitch + ((int)cx & 255) + 1;
        const int o1x = upper ? 1 : 0, o1y = 1 - o1x;
        const float ox = (float)o1x, oy = (float)o1y;
        const float2 g0 = T.gxy[T.perm[base] & 15];
        const float2 g1 = T.gxy[T.perm[base + o1y * kPermPitch + o1x] & 15];
        const float2 g2 = T.gxy[T.perm[base + kPermPitch + 1] & 15];
        auto corner = [](float2 g, float ax, float ay) {  // corner2 with its gradient at hand
            const float r = fmaxf(0.5f - fmaf(ay, ay, ax * ax), 0.f);
            const float t = r * r;
            return (t * t) * fmaf(g.y, ay, g.x * ax);
        };
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float n0 = corner(g0, fx[i], fy[i]);
            const float n1 = corner(g1, (fx[i] - ox) + G2, (fy[i] - oy) + G2);
            const float n2 = corner(g2, fx[i] - C2, fy[i] - C2);
            out[i] = 70.f * ((n0 + n1) + n2);
        }
        return;
    }
    float px[4], py[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        px[i] = x[kNear2X[i]];
        py[i] = z[kNear2Z[i]];
    }
#pragma unroll 1
    for (int k = 0; k < 4; ++k) {  // one copy of snoise2's code: the points rotate through it
        const float n = snoise2(T, px[0], py[0]), ax = px[0], ay = py[0];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            px[i] = px[i + 1];
            py[i] = py[i + 1];
            out[i] = out[i + 1];
        }
        px[3] = ax;
        py[3] = ay;
        out[3] = n;
    }
}

// leven's 900 * Terrain as one loop over its 14 octaves (8 ridged, 4 of the billow, 2 of
// the base), for the point (x[0], z[0]) when N is 1 or the four near points when N is 4:
// leven_terrain's steps in its order, with one copy of the noise's code: written out, the four
// points' octaves made the crossing kernel 39 KB of code.  (leven_terrain stays written out:
// its three parts are independent chains, which overlap there.)
struct LevenExpo {  // 1 / lacunarity^o as RidgedMultiFractal's loop forms it
    float v[7];
    constexpr LevenExpo() : v() {
        float freq = 1.f;
        for (int o = 0; o < 7; ++o) {
            v[o] = 1.f / freq;
            freq = freq * 2.114352f;
        }
    }
};
__constant__ constexpr LevenExpo kLevenExpo{};

template <int N>
__device__ __forceinline__ void leven_heights(const NoiseLds& T, const float x[], const float z[], float out[]) {
    constexpr int M = N == 1 ? 1 : 3;
    float qx[M], qy[M], px[M], py[M], signal[N], sum[N], v[N], amp = 1.f, lac = 2.114352f, gain = 0.f;
#pragma unroll
    for (int j = 0; j < M; ++j) {
        px[j] = qx[j] = x[j] * (1.f / 2000.f);
        py[j] = qy[j] = z[j] * (1.f / 2000.f);
    }
#pragma unroll
    for (int i = 0; i < N; ++i) signal[i] = sum[i] = v[i] = 0.f;
#pragma unroll 1
    for (int step = 0; step < 14; ++step) {
        if (step == 8 || step == 12) {  // the next part starts
            const bool billow = step == 8;
            const float freq = billow ? 0.24f : 0.63f;
#pragma unroll
            for (int j = 0; j < M; ++j) {
                px[j] = (billow ? -4.33f * qx[j] : qx[j]) * freq;
                py[j] = (billow ? 7.98f * qy[j] : qy[j]) * freq;
            }
            lac = billow ? 1.8754f : 2.2f;
            gain = billow ? 0.433f : 0.15f;
            amp = 1.f;
#pragma unroll
            for (int i = 0; i < N; ++i) sum[i] = 0.f;
        }
        if constexpr (N == 1)
            v[0] = snoise2(T, px[0], py[0]);
        else
            snoise2_near(T, px, py, v);
        if (step < 8) {
            const float expo = step == 0 ? 1.f : kLevenExpo.v[step - 1];
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float weight = clamp01(signal[i] * 1.5241f);
                float s = 1.f - fabsf(v[i]);
                s = s * (step == 0 ? s : weight);
                signal[i] = s;
                sum[i] = step == 0 ? s : sum[i] + s * expo;
            }
        } else {
#pragma unroll
            for (int i = 0; i < N; ++i) sum[i] = fmaf(v[i], amp, sum[i]);
            amp = amp * gain;
        }
#pragma unroll
        for (int j = 0; j < M; ++j) {
            px[j] = px[j] * lac;
            py[j] = py[j] * lac;
        }
        if (step == 7) {
#pragma unroll
            for (int i = 0; i < N; ++i) out[i] = clamp01(0.8f * (sum[i] * (1.f / (float)7)));
        } else if (step == 11) {
#pragma unroll
            for (int i = 0; i < N; ++i) {
                const float billow = 0.6f * sum[i];
                out[i] = ((0.5f * billow) + 0.5f) * out[i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < N; ++i) {
        const float b2 = 0.6f * sum[i];
        out[i] = 900.f * (out[i] + ((b2 * 0.5f) + 0.5f));
    }
}

// height_term in the small form, for calls that are rare.
template <int kKind>
__device__ __forceinline__ float height_small(const FieldParams& F, const NoiseLds& T, float x, float z) {
    if (field_kind<kKind>(F) != LVN_FIELD_LEVEN_TERRAIN) return height_term<kKind>(F, T, x, z);
    float out;
    leven_heights<1>(T, &x, &z, &out);
    return out;
}

// height_term at (x + h, z), (x - h, z), (x, z + h), (x, z - h).
template <int kKind>
__device__ __forceinline__ void height_near(const FieldParams& F, const NoiseLds& T, const float x[3], const float z[3],
                                            float out[4]) {
    if (field_kind<kKind>(F) == LVN_FIELD_LEVEN_TERRAIN) {
        leven_heights<4>(T, x, z, out);
        return;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) out[i] = height_term<kKind>(F, T, x[kNear2X[i]], z[kNear2Z[i]]);
}

// ---------------------------------------------------------------------------
// CSG brushes (cl/apply_csg_operation.cl:42-81)
// ---------------------------------------------------------------------------

__device__ __forceinline__ float len3(float x, float y, float z) { return sqrtf((x * x + y * y) + z * z); }

// Density_Sphere / Density_Cuboid (pR rotation of xz, then the box SDF
// length(max(d,0)) + max(min(d,0)) with d = |p| - half extents).
__device__ __forceinline__ float brush_density(const DevOp& op, float x, float y, float z) {
    const float lx = x - op.ox;
    const float ly = y - op.oy;
    const float lz = z - op.oz;
    if (op.brush == 1) return len3(lx, ly, lz) - op.dx;
    const float rx = op.c * lx + op.s * lz;
    const float rz = op.c * lz + op.s * (-lx);
    const float ex = fabsf(rx) - op.dx;
    const float ey = fabsf(ly) - op.dy;
    const float ez = fabsf(rz) - op.dz;
    const float outside = len3(fmaxf(ex, 0.f), fmaxf(ey, 0.f), fmaxf(ez, 0.f));
    const float inside = fmaxf(fmaxf(fminf(ex, 0.f), fminf(ey, 0.f)), fminf(ez, 0.f));
    return outside + inside;
}

// normalize with zero vectors passed through.
__device__ __forceinline__ float3 normalize_or_zero(float x, float y, float z) {
    if (x == 0.f && y == 0.f && z == 0.f) return make_float3(x, y, z);
    const float l = len3(x, y, z);
    return make_float3(x / l, y / l, z / l);
}

// ---------------------------------------------------------------------------
// Octree codes (cl/octree.cl:34-72)
// ---------------------------------------------------------------------------

// The codes interleave x, y and z (bits 3 d + 2, 3 d + 1, 3 d) below a leading one at bit
// 3 depth; depth is at most 6, so a coordinate's six bits are spread and gathered by masks.
__device__ __forceinline__ uint32_t spread3(uint32_t v) {
    v = (v | (v << 8)) & 0x300fu;
    v = (v | (v << 4)) & 0x30c3u;
    return (v | (v << 2)) & 0x9249u;
}
__device__ __forceinline__ int gather3(uint32_t v) {
    v &= 0x9249u;
    v = (v | (v >> 2)) & 0x30c3u;
    v = (v | (v >> 4)) & 0x300fu;
    return (int)((v | (v >> 8)) & 0x3fu);
}

__device__ __forceinline__ uint32_t code_for_position(int x, int y, int z, int depth) {
    return (1u << (3 * depth)) | (spread3((uint32_t)x) << 2) | (spread3((uint32_t)y) << 1) | spread3((uint32_t)z);
}

// The position of a leaf's code (leading one at bit 3 depth).
__device__ __forceinline__ int3 position_for_code(uint32_t code, int depth) {
    return make_int3(gather3(code >> 2), gather3(code >> 1), gather3(code & ~(1u << (3 * depth))));
}

}  // namespace lvn
