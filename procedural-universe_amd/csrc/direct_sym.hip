// Direct sum over unordered pairs (Newton's third law): each pair's separation
// and reciprocal square root are computed once and applied to both particles.
//
// The one-sided pair (direct_core.hpp) costs 12 FP32 instructions and one
// v_rsq_f32 per interaction and is bound by their issue.  Taken once for both
// sides a law-R pair costs 17 (15 when all masses are equal) and one
// v_rsq_f32, and 0.75 for moving the streamed sums from lane to lane: 8.9 (7.9)
// + 0.5 per interaction.  Measured, one step of N = 2^20: one-sided 288 ms
// (3.8e12 interactions/s), 193 ms (5.7e12) here, 177 ms (6.2e12) with equal
// masses; N = 65,536: 1.25, 0.79, 0.72 ms; N = 20,011 (law P): 0.151, 0.120,
// 0.108 ms.  Still bound by issue: 0.32 VALU instructions per SIMD per cycle
// were measured at N = 524,288, where the same step in a register-only loop
// reaches 0.34.
//
// Layout.  A wavefront holds 256 resident particles, four per lane, with their
// sums in registers, and streams sets of 64 particles past them: at step s
// lane l meets the set's particle (l + s) mod 64, read from LDS (the set is
// stored twice in a row, so the address is the lane's plus a constant), and
// the set's 64 sums travel the other way, one lane per step (a DPP wave
// rotation folded into the subtraction), so that after 64 steps every sum is
// back in its particle's lane.  (The sums kept in LDS instead, read and written
// each step, took 198 against 190 ms at N = 2^20: the DPP costs less than
// six LDS instructions.)  A workgroup is four such wavefronts, which share a
// tile of 256 streamed particles, each wavefront taking the tile's four sets in
// turn, starting with its own; single-wave workgroups with 64-particle tiles
// were slower at every size.  Six waves per SIMD (80 VGPRs): 190 ms against
// 197 ms with the 87 VGPRs the compiler takes freely, 225 ms held to seven.
//
// Tasks.  The particles are cut into nsb blocks; task (A, d) takes block A as
// residents and block A + d (mod nsb) as the stream, d = 1 .. nsb / 2 (with an
// even nsb the last distance only for the first half of the blocks), and d = 0
// is the block with itself, one-sided over all ordered pairs.  Every task
// writes the sums of its residents and of its stream to rows of `part` that no
// other task writes, and a second kernel adds each particle's rows in a fixed
// order: no atomics, the same bits every run.
//
// Summation: FP32 sums of 256 pairs, added over the task (at most about 30
// of them) and then, compensated, over the tasks.  RMS error against FP64 at
// N = 2^20: 2.9e-8, one-sided 2.6e-8; at 65,536 3.4e-8 either way.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/nbody.h"
#include "common.hpp"
#include "direct.hpp"
#include "direct_core.hpp"

namespace nbody {

namespace {

using core::kahan_add;

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
    float* part;        // [rows][3][n_pad]
    int n_pad;
    SymPlan plan;
    DirectScale sc;
};

// A particle in scaled units: (x', y', z', G m / c).  With EQ the masses do not
// enter the pairs, so a massless one (the padding) is placed at
// (2^100, 2^100, 2^100): its squared distances are +inf and their reciprocal
// square roots 0.
template <int LAW, bool EQ>
__device__ __forceinline__ float4 scaled(const float4 p, const DirectScale& sc) {
    float4 q = make_float4(p.x * sc.inv_len, p.y * sc.inv_len, p.z * sc.inv_len,
                           p.w * (LAW == NBODY_LAW_R ? 1.0f / sc.mass_k : sc.mass_k));
    if constexpr (EQ) {
        if (!(p.w > 0.f)) q.x = q.y = q.z = 0x1p100f;
    }
    return q;
}

// Row r of the partial sums: n_pad x, then y, then z.
__device__ __forceinline__ float* part_row(float* part, int r, int n_pad) {
    return part + static_cast<size_t>(3 * r) * n_pad;
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
                                         const float (&z)[kPer], const float (&m)[kPer], float soft, float tiny,
                                         float (&ax)[kPer], float (&ay)[kPer], float (&az)[kPer], float& bx, float& by,
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
                const float t = r2 + soft;
                const float u = r2 * t;
                g[k] = __builtin_fmaf(u, t, tiny);
            } else {
                g[k] = __builtin_fmaf(dz[k], dz[k], __builtin_fmaf(dy[k], dy[k], __builtin_fmaf(dx[k], dx[k], soft)));
            }
        }
        core::rsq4(g[0], g[1], g[2], g[3]);
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
    const float tiny = core::in_vgpr(__FLT_MIN__);
    const float soft = core::in_vgpr(A.sc.soft);
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
            float bx, by, bz;
#pragma unroll 1
            for (int p = 0; p < kWaves; ++p) {
                const int set = (wave + p) & (kWaves - 1);
                pass_set<LAW, BOTH, EQ>(&S.set[buf][set][lane], x, y, z, m, soft, tiny, ax, ay, az, bx, by, bz);
                if constexpr (BOTH) {
                    if (p == 0) S.sum[0][set][lane] = bx, S.sum[1][set][lane] = by, S.sum[2][set][lane] = bz;
                    else S.sum[0][set][lane] += bx, S.sum[1][set][lane] += by, S.sum[2][set][lane] += bz;
                }
                // The other buffer was last read before the previous tile's
                // end.  (Loaded here, not a tile ahead: the four registers
                // would cost a wave per SIMD, and the other waves cover it.)
                if (p == kWaves - 1 && more) stage(j + kStream < j1 ? A.src[j + kStream] : none, buf ^ 1);
                __syncthreads();  // the next wavefront to meet a set adds to the sums left here
            }
#pragma unroll
            for (int k = 0; k < kPer; ++k) {
                sx[k] += ax[k], sy[k] += ay[k], sz[k] += az[k];
                ax[k] = ay[k] = az[k] = 0.f;
            }
            if constexpr (BOTH) {
                // the tile's sums over these residents: thread t's particle is
                // set `wave`, lane `lane`, which only this thread touches again
                // before the next barrier
                if (j < j1) {
                    float* out = part_row(A.part, rowj, A.n_pad) + j;
                    const size_t n = A.n_pad;
                    bx = S.sum[0][wave][lane], by = S.sum[1][wave][lane], bz = S.sum[2][wave][lane];
                    if (ib > i0) bx += out[0], by += out[n], bz += out[2 * n];
                    out[0] = bx, out[n] = by, out[2 * n] = bz;
                }
            }
            buf ^= 1;
        }
#pragma unroll
        for (int k = 0; k < kPer; ++k) {
            const int i = ib + wave * kRes + k * kSet + lane;
            if (i < i1) {
                float* out = part_row(A.part, rowi, A.n_pad) + i;
                const size_t n = A.n_pad;
                out[0] = sx[k], out[n] = sy[k], out[2 * n] = sz[k];
            }
        }
    }
}

// Task (A, d, h): blockIdx.x = A; blockIdx.y runs over the distances 1 .. H,
// each with its `split` runs of the streamed block, then d = 0 (shorter, so
// last).
template <int LAW, bool EQ>
__global__ __launch_bounds__(kTile) __attribute__((amdgpu_waves_per_eu(6))) void sym_force_kernel(SymArgs A) {
    __shared__ SymShared S;
    const SymPlan& P = A.plan;
    const int a = blockIdx.x, H = P.nsb / 2;
    const int y = blockIdx.y / P.split, h = blockIdx.y - y * P.split;
    if (y == H) {
        sym_task<LAW, false, EQ>(A, S, a, a, h, h, 0);
        return;
    }
    const int d = y + 1;
    if (2 * d == P.nsb && a >= d) return;
    int b = a + d;
    if (b >= P.nsb) b -= P.nsb;
    sym_task<LAW, true, EQ>(A, S, a, b, h, d * P.split + h, (H + 1) * P.split + d - 1);
}

// Adds a particle's rows in row order (compensated): a workgroup takes 64
// particles, wave w a quarter of the rows, then the waves' sums in order;
// wave 0 scales them back and kicks and drifts (kick != 0) or stores the
// acceleration only.
__global__ __launch_bounds__(256) void sym_reduce_kernel(DirectLaunch L, SymPlan P, int kick) {
    __shared__ core::SliceSums sums;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    const int b = (blockIdx.x * 64) / P.block;  // blocks are multiples of 64 particles
    const int H = P.nsb / 2, rows = (H + 1) * P.split + H, per = (rows + 3) / 4;
    float s[3] = {0.f, 0.f, 0.f}, c[3] = {0.f, 0.f, 0.f};
    const int r1 = min(rows, (wave + 1) * per);
#pragma unroll 4
    for (int r = wave * per; r < r1; ++r) {
        // the half distance of an even number of blocks is one task for each
        // two blocks: residents in the first half, streamed in the second
        const bool resident = r < (H + 1) * P.split;
        const int d = resident ? r / P.split : r - (H + 1) * P.split + 1;
        if (2 * d == P.nsb && (b >= d) == resident) continue;
        const float* p = part_row(reinterpret_cast<float*>(L.part), r, L.n_pad) + i;
        kahan_add(s[0], c[0], p[0]);
        kahan_add(s[1], c[1], p[L.n_pad]);
        kahan_add(s[2], c[2], p[2 * static_cast<size_t>(L.n_pad)]);
    }
    core::add_slices(sums, wave, lane, s, c);
    if (wave != 0 || i >= L.n) return;
    // equal masses: the rows are sums without the mass, in scaled units
    const float out = L.gm_equal > 0.f ? L.gm_equal * L.sc.out : L.sc.out;
    const float ax = s[0] * out, ay = s[1] * out, az = s[2] * out;
    L.acc[i] = make_float4(ax, ay, az, 0.f);
    if (!kick) return;
    float4 v = L.vel[i], x = L.src[i];
    v.x = __builtin_fmaf(ax, L.dt, v.x);
    v.y = __builtin_fmaf(ay, L.dt, v.y);
    v.z = __builtin_fmaf(az, L.dt, v.z);
    x.x = __builtin_fmaf(v.x, L.dts, x.x);
    x.y = __builtin_fmaf(v.y, L.dts, x.y);
    x.z = __builtin_fmaf(v.z, L.dts, x.z);
    L.vel[i] = v;
    L.pos_out[i] = x;
}

}  // namespace

SymPlan sym_plan(int n_pad) {
    // Below 16,384 particles there are too few tasks for the chip (12,288:
    // 0.058 ms against 0.059 one-sided; 16,384: 0.081 against 0.093).
    SymPlan p{};
    if (n_pad < 16384) return p;
    // About 192 blocks: more give more rows of partial sums (12 bytes per
    // particle and block, 2.1 GB at 2^20 with 171 blocks, 3.2 GB and 1% less
    // time with 256), fewer leave a longer tail (128: 1% more time).
    constexpr int kStep = kRes * kWaves;
    p.block = ((n_pad + 191) / 192 + kStep - 1) / kStep * kStep;
    p.nsb = (n_pad + p.block - 1) / p.block;
    // Smaller systems' streams in up to four runs (each a whole tile), until
    // there are 4,096 tasks for the 1,536 workgroup places.
    const int tasks = p.nsb * (p.nsb + 1) / 2;
    p.split = tasks >= 4096 ? 1 : tasks >= 2048 ? 2 : 4;
    return p;
}

size_t sym_part_records(const SymPlan& p, int n_pad) {
    const size_t H = p.nsb / 2;
    return (((H + 1) * p.split + H) * 3 * static_cast<size_t>(n_pad) + 3) / 4;
}

hipError_t sym_step(const DirectLaunch& L, const SymPlan& P, bool kick, hipStream_t stream, hipEvent_t ev_b,
                    hipEvent_t ev_e) {
    const SymArgs A{L.src, reinterpret_cast<float*>(L.part), L.n_pad, P, L.sc};
    const dim3 grid(P.nsb, (P.nsb / 2 + 1) * P.split);
    hipError_t e = hipSuccess;
    if (ev_b && (e = hipEventRecord(ev_b, stream)) != hipSuccess) return e;
    using Fn = void (*)(SymArgs);
    const bool r = L.law == NBODY_LAW_R, eq = L.gm_equal > 0.f;
    const Fn fn = r ? (eq ? sym_force_kernel<NBODY_LAW_R, true> : sym_force_kernel<NBODY_LAW_R, false>)
                    : (eq ? sym_force_kernel<NBODY_LAW_P, true> : sym_force_kernel<NBODY_LAW_P, false>);
    hipLaunchKernelGGL(fn, grid, dim3(kTile), 0, stream, A);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (ev_e && (e = hipEventRecord(ev_e, stream)) != hipSuccess) return e;
    hipLaunchKernelGGL(sym_reduce_kernel, dim3(L.n_pad / 64), dim3(256), 0, stream, L, P, kick ? 1 : 0);
    return hipGetLastError();
}

}  // namespace nbody
