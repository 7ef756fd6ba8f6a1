// Direct sum over unordered pairs (Newton's third law): each pair's separation
// and reciprocal square root are computed once and applied to both particles.
//
// The one-sided pair (direct_core.hpp) costs 12 FP32 instructions and one
// v_rsq_f32 per interaction and is bound by their issue.  Taken once for both
// sides a law-R pair costs 17 (15 when all masses are equal) and one
// v_rsq_f32, and 0.75 for moving the streamed sums from lane to lane: 8.9 (7.9)
// + 0.5 per interaction.  Measured, one step of N = 2^20: one-sided 288 ms
// (3.8e12 interactions/s), 197 ms (5.6e12) here, 180 ms (6.1e12) with equal
// masses; N = 65,536: 1.25, 0.81, 0.74 ms; N = 20,011 (law P): 0.151, 0.123,
// 0.111 ms.  Still bound by issue: 0.389 VALU instructions per SIMD per cycle at
// N = 2^20 (2.13 GHz under this load), 0.326 one-sided.
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
// Summation: a resident's FP32 sums of 256 pairs (a streamed particle's of 1,024,
// four at a time and in four parts) are added with compensation over the task
// and then over the tasks: what the rounding of a resident's sum leaves out is where
// its next tile starts, so that it takes no registers, and a row keeps it too.
// RMS error against FP64, one-sided / here: N = 2^20 2.8e-8 / 2.7e-8 (a disc of unequal
// masses), 3.1e-8 / 3.1e-8 (a sphere of equal ones), 2^21 2.7e-8 / 2.7e-8, 20,011 5.2e-8 /
// 4.5e-8; with the tiles' and the rows' sums added plainly 3.2e-8 to 3.3e-8 and 6.3e-8,
// in 1.6% (equal masses) and 2.2% less time.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "../../include/nbody.h"
#include "common.hpp"
#include "direct.hpp"
#include "direct_core.hpp"
#include "direct_sym_core.hpp"

namespace nbody {

namespace {

// Task (A, d, h): blockIdx.x = A; blockIdx.y runs over the distances 1 .. H,
// each with its `split` runs of the streamed block, then d = 0 (shorter, so
// last).
template <int LAW, bool EQ>
__global__ __launch_bounds__(kTile) __attribute__((amdgpu_waves_per_eu(6))) void sym_force_kernel(core::SymArgs A) {
    __shared__ core::SymShared S;
    const SymPlan& P = A.plan;
    const int a = blockIdx.x, H = P.nsb / 2;
    const int y = blockIdx.y / P.split, h = blockIdx.y - y * P.split;
    if (y == H) {
        core::sym_task<LAW, false, EQ>(A, S, a, a, h, h, 0);
        return;
    }
    const int d = y + 1;
    if (2 * d == P.nsb && a >= d) return;
    int b = a + d;
    if (b >= P.nsb) b -= P.nsb;
    core::sym_task<LAW, true, EQ>(A, S, a, b, h, d * P.split + h, (H + 1) * P.split + d - 1);
}

// Adds each particle's rows, 64 particles a workgroup, scales the sums back and
// kicks and drifts (kick != 0) or stores the acceleration only.
template <int LAW>
__global__ __launch_bounds__(256) void sym_reduce_kernel(DirectLaunch L, SymPlan P, float out_hi, float out_lo,
                                                         int kick) {
    __shared__ core::SliceSums sums;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    float s[3];
    core::sum_rows(L.part, P, L.n_pad, i, sums, wave, lane, out_hi, out_lo, s);
    if (wave != 0 || i >= L.n) return;
    float4 x = L.src[i];
    core::sums_of_a_lost_particle<LAW>(x, L.sc, s);
    const float ax = s[0], ay = s[1], az = s[2];
    L.acc[i] = make_float4(ax, ay, az, 0.f);
    if (!kick) return;
    float4 v = L.vel[i];
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
    // About 192 blocks: more give more rows of partial sums (16 bytes per
    // particle and block, 2.9 GB at 2^20 with 171 blocks, 4.3 GB and 1% less
    // time with 256), fewer leave a longer tail (128: 1% more time).
    constexpr int kStep = core::kRes * core::kWaves;
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
    return ((H + 1) * p.split + H) * static_cast<size_t>(n_pad);
}

hipError_t sym_step(const DirectLaunch& L, const SymPlan& P, const SymUnits& U, bool kick, hipStream_t stream,
                    hipEvent_t ev_b, hipEvent_t ev_e) {
    const core::SymArgs A{L.src, L.part, L.n_pad, P, L.sc, U.alpha, U.soft};
    const dim3 grid(P.nsb, (P.nsb / 2 + 1) * P.split);
    hipError_t e = hipSuccess;
    if (ev_b && (e = hipEventRecord(ev_b, stream)) != hipSuccess) return e;
    using Fn = void (*)(core::SymArgs);
    const bool r = L.law == NBODY_LAW_R, eq = U.equal != 0;
    const Fn fn = r ? (eq ? sym_force_kernel<NBODY_LAW_R, true> : sym_force_kernel<NBODY_LAW_R, false>)
                    : (eq ? sym_force_kernel<NBODY_LAW_P, true> : sym_force_kernel<NBODY_LAW_P, false>);
    hipLaunchKernelGGL(fn, grid, dim3(kTile), 0, stream, A);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (ev_e && (e = hipEventRecord(ev_e, stream)) != hipSuccess) return e;
    hipLaunchKernelGGL((r ? sym_reduce_kernel<NBODY_LAW_R> : sym_reduce_kernel<NBODY_LAW_P>), dim3(L.n_pad / 64), dim3(256), 0, stream, L, P, U.out_hi, U.out_lo, kick ? 1 : 0);
    return hipGetLastError();
}

}  // namespace nbody
