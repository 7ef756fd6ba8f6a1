// Device core of the direct sum over unordered pairs, shared by the
// single-system kernel and the batch executor (a description and its
// measurements are in direct_sym.hip).
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/nbody.h"
#include "direct.hpp"
#include "direct_core.hpp"

namespace nbody {
namespace core {

constexpr int kPer = 4;                // resident particles per lane
constexpr int kSet = 64;               // streamed particles per set
constexpr int kRes = kSet * kPer;      // residents per wavefront
constexpr int kWaves = 4;              // wavefronts per workgroup
constexpr int kStream = kSet * kWaves;  // streamed particles per tile
static_assert(kStream == kTile && kRes == kTile, "blocks are whole tiles");

// The value of lane l + 1 (mod 64) of the wavefront.
__device__ __forceinline__ float from_next_lane(float x) {
    constexpr int kWaveRol1 = 0x134;
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kWaveRol1, 0xf, 0xf, false));
}

struct SymArgs {
    const float4* src;  // n_pad records (x, y, z, G m)
    float4* part;       // [rows][n_pad]
    int n_pad;
    SymPlan plan;
    DirectScale sc;
    float alpha, soft;  // SymUnits
};

// A particle in scaled units: (x', y', z', G m / c).  With EQ the masses do not
// enter the pairs, so a massless one (the padding) is placed at
// (2^100, 2^100, 2^100): its squared distances are +inf and their reciprocal
// square roots 0; so is, under law R, a massless particle that has no finite
// position (sums_of_a_lost_particle).
template <int LAW, bool EQ>
__device__ __forceinline__ float4 scaled(const float4 p, const DirectScale& sc) {
    float4 q = make_float4(p.x * sc.inv_len, p.y * sc.inv_len, p.z * sc.inv_len,
                           p.w * (LAW == NBODY_LAW_R ? 1.0f / sc.mass_k : sc.mass_k));
    if constexpr (EQ) {
        if (!(p.w > 0.f)) q.x = q.y = q.z = 0x1p100f;
    } else if constexpr (LAW == NBODY_LAW_R) {
        if (!(p.w > 0.f) && !finite3(q)) q.x = q.y = q.z = 0x1p100f;
    }
    return q;
}

// Row r of the partial sums, a record a particle.
__device__ __forceinline__ float4* part_row(float4* part, int r, int n_pad) {
    return part + static_cast<size_t>(r) * n_pad;
}

struct SymShared {
    float4 set[2][kWaves][2 * kSet];  // two tiles, every set twice in a row
    float sum[3][kWaves][kSet];       // the tile's sums
};

// 64 steps of a set past the wavefront's residents.  Adds to the residents'
// sums a[] and, with BOTH, returns the set's sums in (bx, by, bz), particle l
// in lane l.
template <int LAW, bool BOTH, bool EQ>
__device__ __forceinline__ void pass_set(const float4* set, const float (&x)[kPer], const float (&y)[kPer],
                                         const float (&z)[kPer], const float (&m)[kPer], float alpha, float soft,
                                         float tiny, float (&ax)[kPer], float (&ay)[kPer], float (&az)[kPer], float& bx, float& by,
                                         float& bz) {
    bx = by = bz = 0.f;
#pragma unroll 4
    for (int s = 0; s < kSet; ++s) {
        const float4 q = set[s];
        float dx[kPer], dy[kPer], dz[kPer], g[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            dx[k] = q.x - x[k];
            dy[k] = q.y - y[k];
            dz[k] = q.z - z[k];
            if constexpr (LAW == NBODY_LAW_R) {
                const float r2 = __builtin_fmaf(dz[k], dz[k], __builtin_fmaf(dy[k], dy[k], dx[k] * dx[k]));
                const float t = EQ ? r2 + soft : __builtin_fmaf(r2, alpha, soft);
                const float u = r2 * t;
                g[k] = __builtin_fmaf(u, t, tiny);
            } else {
                g[k] = __builtin_fmaf(dz[k], dz[k], __builtin_fmaf(dy[k], dy[k], __builtin_fmaf(dx[k], dx[k], soft)));
            }
        }
        rsq4(g[0], g[1], g[2], g[3]);
        float px = 0.f, py = 0.f, pz = 0.f;
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            if constexpr (LAW == NBODY_LAW_P) g[k] = g[k] * (g[k] * g[k]);
            const float f = EQ ? g[k] : g[k] * q.w;
            ax[k] = __builtin_fmaf(dx[k], f, ax[k]);
            ay[k] = __builtin_fmaf(dy[k], f, ay[k]);
            az[k] = __builtin_fmaf(dz[k], f, az[k]);
            if constexpr (BOTH) {
                const float h = EQ ? g[k] : g[k] * m[k];
                px = k == 0 ? dx[k] * h : __builtin_fmaf(dx[k], h, px);
                py = k == 0 ? dy[k] * h : __builtin_fmaf(dy[k], h, py);
                pz = k == 0 ? dz[k] * h : __builtin_fmaf(dz[k], h, pz);
            }
        }
        if constexpr (BOTH) {
            // before the first step the sums are zero in every lane
            bx = from_next_lane(bx) - px;
            by = from_next_lane(by) - py;
            bz = from_next_lane(bz) - pz;
        }
    }
    if constexpr (BOTH) {
        // step s's sums belong to particle l + s: one more lane brings each
        // particle's to its own lane
        bx = from_next_lane(bx);
        by = from_next_lane(by);
        bz = from_next_lane(bz);
    }
}

template <int LAW, bool BOTH, bool EQ>
__device__ __forceinline__ void sym_task(const SymArgs& A, SymShared& S, int blockA, int blockB, int h, int rowi,
                                         int rowj) {
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
    const float tiny = in_vgpr(__FLT_MIN__);
    constexpr bool kAlpha = LAW == NBODY_LAW_R && !EQ;
    float alpha = 1.0f;
    if constexpr (kAlpha) alpha = in_vgpr(A.alpha);
    const float soft = in_vgpr(A.soft);
    const int B = A.plan.block, S0 = B / A.plan.split;
    const int i0 = blockA * B, i1 = min(i0 + B, A.n_pad);
    const int j0 = blockB * B + h * S0, j1 = min(j0 + S0, A.n_pad);
    const float4 none = make_float4(0.f, 0.f, 0.f, 0.f);
    auto stage = [&](const float4 p, int buf) {
        const float4 q = scaled<LAW, EQ>(p, A.sc);
        S.set[buf][wave][lane] = q;
        S.set[buf][wave][lane + kSet] = q;
    };
    for (int ib = i0; ib < i1; ib += kRes * kWaves) {
        float x[kPer], y[kPer], z[kPer], m[kPer];
        float ax[kPer], ay[kPer], az[kPer], sx[kPer], sy[kPer], sz[kPer];
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = ib + wave * kRes + k * kSet + lane;
            const float4 q = scaled<LAW, EQ>(i < i1 ? A.src[i] : none, A.sc);
            x[k] = q.x, y[k] = q.y, z[k] = q.z, m[k] = q.w;
            ax[k] = ay[k] = az[k] = 0.f;
            sx[k] = sy[k] = sz[k] = 0.f;
        }
        // A wavefront without residents (the last block's end) only keeps the
        // barriers and starts its first set's sums.
        const bool any = ib + wave * kRes < i1;
        int buf = 0;
        if (j0 < j1) {
            const int j = j0 + static_cast<int>(threadIdx.x);
            __syncthreads();  // the previous residents' last tile has been read
            stage(j < j1 ? A.src[j] : none, 0);
            __syncthreads();
        }
        for (int jt = j0; jt < j1; jt += kStream) {
            const int j = jt + static_cast<int>(threadIdx.x);
            const bool more = jt + kStream < j1;
            float bx = 0.f, by = 0.f, bz = 0.f;
#pragma unroll 1
            for (int p = 0; p < kWaves; ++p) {
                const int set = (wave + p) & (kWaves - 1);
                if (any)
                    pass_set<LAW, BOTH, EQ>(&S.set[buf][set][lane], x, y, z, m, alpha, soft, tiny, ax, ay, az, bx, by,
                                            bz);
                if constexpr (BOTH) {
                    if (p == 0) S.sum[0][set][lane] = bx, S.sum[1][set][lane] = by, S.sum[2][set][lane] = bz;
                    else if (any) S.sum[0][set][lane] += bx, S.sum[1][set][lane] += by, S.sum[2][set][lane] += bz;
                }
                // The other buffer was last read before the previous tile's
                // end.  (Loaded here, not a tile ahead: the four registers
                // would cost a wave per SIMD, and the other waves cover it.)
                if (p == kWaves - 1 && more) stage(j + kStream < j1 ? A.src[j + kStream] : none, buf ^ 1);
                __syncthreads();  // the next wavefront to meet a set adds to the sums left here
            }
            // compensated: the next tile's sums start from what is left out here
            if (jt == j0) {
#pragma unroll
                for (int k = 0; k < kPer; ++k) {
                    sx[k] = ax[k], sy[k] = ay[k], sz[k] = az[k];
                    ax[k] = ay[k] = az[k] = 0.f;
                }
            } else {
#pragma unroll
                for (int k = 0; k < kPer; ++k)
                    add_keeping_rest(sx[k], ax[k]), add_keeping_rest(sy[k], ay[k]), add_keeping_rest(sz[k], az[k]);
            }
            if constexpr (BOTH) {
                // the tile's sums over these residents: thread t's particle is
                // set `wave`, lane `lane`, which only this thread touches again
                // before the next barrier
                if (j < j1) {
                    float4* out = part_row(A.part, rowj, A.n_pad) + j;
                    const float b[3] = {S.sum[0][wave][lane], S.sum[1][wave][lane], S.sum[2][wave][lane]};
                    if (ib == i0) {
                        *out = make_float4(b[0], b[1], b[2], 0.f);
                    } else {
                        float s[3], r[3];
                        unpack_sums(*out, s, r);
#pragma unroll
                        for (int a = 0; a < 3; ++a) {
                            r[a] += b[a];
                            add_keeping_rest(s[a], r[a]);
                        }
                        *out = pack_sums(s, r);
                    }
                }
            }
            buf ^= 1;
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = ib + wave * kRes + k * kSet + lane;
            if (i < i1) {
                const float s[3] = {sx[k], sy[k], sz[k]}, r[3] = {ax[k], ay[k], az[k]};
                part_row(A.part, rowi, A.n_pad)[i] =
                    j1 - j0 > kStream ? pack_sums(s, r) : make_float4(s[0], s[1], s[2], 0.f);
            }
        }
    }
}

// The sum of particle i's rows (i in block i / plan.block) in row order,
// compensated: the workgroup's wave w takes a quarter of the rows, then the
// waves' sums in order.  i is the same in every wave; every thread of the
// workgroup must call it, and only wave 0 returns the sums, times out and
// rounded once, in s.
__device__ __forceinline__ void sum_rows(const float4* __restrict__ part, const SymPlan& P, int n_pad, int i, SliceSums& sums,
                                         int wave, int lane, float out_hi, float out_lo, float (&s)[3]) {
    const int b = i / P.block;
    const int H = P.nsb / 2, rows = (H + 1) * P.split + H, per = (rows + 3) / 4;
    float c[3] = {0.f, 0.f, 0.f};
    s[0] = s[1] = s[2] = 0.f;
    const int r1 = min(rows, (wave + 1) * per);
#pragma unroll 4
    for (int r = wave * per; r < r1; ++r) {
        // the half distance of an even number of blocks is one task for each
        // two blocks: residents in the first half, streamed in the second
        const bool resident = r < (H + 1) * P.split;
        const int d = resident ? r / P.split : r - (H + 1) * P.split + 1;
        if (2 * d == P.nsb && (b >= d) == resident) continue;
        float x[3], rest[3];
        unpack_sums(part[static_cast<size_t>(r) * n_pad + i], x, rest);
        // a row is not small beside the sum of a few: no Kahan addition
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            add_keeping_rest(s[a], x[a]);
            c[a] -= x[a] + rest[a];
        }
    }
    add_slices(sums, wave, lane, s, c);
#pragma unroll
    for (int a = 0; a < 3; ++a) s[a] = __builtin_fmaf(s[a], out_hi, __builtin_fmaf(s[a], out_lo, -(c[a] * out_hi)));
}

}  // namespace core
}  // namespace nbody
