// FP64 diagnostics of a device-resident state: kinetic energy, pair
// potential energy, linear and angular momentum.
//
// Positions are the FP32 state; masses come from an FP64 copy so that the
// diagnostics do not inherit the FP32 rounding of G*m.  Every sum is formed in
// a fixed order (per-block tree in LDS, then blocks in index order on the
// host), so the result is reproducible run to run.
//
// Pair potentials (the integral of each law's pair force from r to infinity):
//   law R: U(r) = -(G m_i m_j / sqrt(S)) * (pi/2 - atan(r / sqrt(S)));  S = 0: -G m_i m_j / r
//   law P: U(r) = -G m_i m_j / sqrt(r^2 + eps^2)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "../../include/nbody.h"
#include "diag.hpp"

namespace nbody {

namespace {

constexpr int kDiagBlock = 256;
constexpr int kDiagTile = 256;

__device__ double block_sum(double v, double* red) {
    const int t = threadIdx.x;
    red[t] = v;
    __syncthreads();
    for (int w = kDiagBlock / 2; w > 0; w >>= 1) {
        if (t < w) red[t] += red[t + w];
        __syncthreads();
    }
    const double r = red[0];
    __syncthreads();
    return r;
}

// out[block * 8 + {0: kinetic, 1-3: momentum, 4-6: angular momentum, 7: mass}]
__global__ __launch_bounds__(kDiagBlock) void diag_local_kernel(const float4* __restrict__ pos,
                                                                const float4* __restrict__ vel,
                                                                const double* __restrict__ mass, int n,
                                                                double* __restrict__ out) {
    __shared__ double red[kDiagBlock];
    double q[8] = {0, 0, 0, 0, 0, 0, 0, 0};
    for (int i = blockIdx.x * kDiagBlock + threadIdx.x; i < n; i += gridDim.x * kDiagBlock) {
        const double m = mass[i];
        const float4 x = pos[i];
        const float4 v = vel[i];
        const double vx = v.x, vy = v.y, vz = v.z;
        const double px = x.x, py = x.y, pz = x.z;
        q[0] += 0.5 * m * (vx * vx + vy * vy + vz * vz);
        q[1] += m * vx;
        q[2] += m * vy;
        q[3] += m * vz;
        q[4] += m * (py * vz - pz * vy);
        q[5] += m * (pz * vx - px * vz);
        q[6] += m * (px * vy - py * vx);
        q[7] += m;
    }
    for (int c = 0; c < 8; ++c) {
        const double s = block_sum(q[c], red);
        if (threadIdx.x == 0) out[blockIdx.x * 8 + c] = s;
    }
}

// atan(z) for 0 <= z <= 1 as z + z w P(w), w = z^2: the polynomial that meets
// atan(sqrt(w)) / sqrt(w) at the 21 Chebyshev points of [0, 1] (its value at 0
// rounds to 1), formed in 90-digit arithmetic; 5e-18 off, and with the rounding
// within 1.5 x 2^-53 of the value over 2e7 points.
constexpr double kAtan[20] = {
    -0x1.5555555555500p-2, 0x1.9999999993702p-3, -0x1.2492492327bf2p-3, 0x1.c71c716e724e1p-4,
    -0x1.745d1099f743ep-4, 0x1.3b135af6a0e88p-4, -0x1.110df7e57b3d8p-4, 0x1.e1b7b5bcacd55p-5,
    -0x1.ae4da39abd8c9p-5, 0x1.82a3c93dd0230p-5, -0x1.59180bd7d7b67p-5, 0x1.2b18b9c197546p-5,
    -0x1.e69dd6d612131p-6, 0x1.643110da5054fp-6, -0x1.c012fe85b6413p-7, 0x1.cd48e33ffd1aep-8,
    -0x1.6fa050a5cad37p-9, 0x1.a53135c884a6dp-11, -0x1.328ae5000addbp-13, 0x1.a7d4ff1d17f2cp-17,
};

__device__ __forceinline__ double atan_unit(double z) {
    const double w = z * z;
    double p = kAtan[19];
#pragma unroll
    for (int k = 18; k >= 0; --k) p = fma(p, w, kAtan[k]);
    return fma(z * w, p, z);
}

// 1 / sqrt(x) for finite x > 0: v_rsq_f64 (within 2^-22) and one third-order
// step (the error's cube, 2^-67, is below the rounding).
__device__ __forceinline__ double rsqrt_pos(double x) {
    const double y = __builtin_amdgcn_rsq(x);
    const double e = fma(-x * y, y, 1.0);
    return fma(y, e * fma(e, 0.375, 0.5), y);
}

// A pair's potential over -G m_i m_j (law R: times rs = sqrt(soft)).
//
// law R: (pi / 2 - atan(r / rs)) / rs = atan(rs / r) / rs, 1 / rs applied to the
// whole sum; r = 0 gives atan(inf).  PLAIN: every position is finite and soft >
// 0.  Then r2 is finite and, with 1e-300 (below the square of any difference of
// floats) added, positive; the arctangent's argument is rs / r or r / rs,
// whichever is at most 1, both products of the one reciprocal square root.
template <int LAW, bool PLAIN>
__device__ __forceinline__ double pair_potential(double dx, double dy, double dz, double soft, double rs,
                                                 double inv_rs) {
    if constexpr (PLAIN) {
        if constexpr (LAW == NBODY_LAW_R) {
            const double r2 = fma(dz, dz, fma(dy, dy, fma(dx, dx, 1e-300)));
            const double y = rsqrt_pos(r2);
            const double t = rs * y, u = r2 * y * inv_rs;
            const bool far = t < u;
            const double a = atan_unit(far ? t : u);
            return far ? a : 0x1.921fb54442d18p+0 - a;
        } else {
            return rsqrt_pos(fma(dz, dz, fma(dy, dy, fma(dx, dx, soft))));
        }
    }
    const double r2 = dx * dx + dy * dy + dz * dz;
    if constexpr (LAW == NBODY_LAW_R) {
        const double y = rsqrt(r2);
        if (rs > 0) return atan(rs * y);
        return r2 > 0 ? y : 0.0;
    }
    return rsqrt(r2 + soft);
}

// Every unordered pair of blocks of kDiagBlock particles once: block I with the
// blocks I, I + 1, ..., I + nb / 2 (mod nb), so each block has the same work;
// with an even number of blocks the opposite block only for the first half of
// them.  A block with itself takes every ordered pair at half weight.
// Workgroup (I, c) takes the c-th run of `per` of those distances:
// out[c * nb + I] = -sum m_i (G m_j) g(r_ij).
//
// Bound by FP64 arithmetic (law R: about 45 instructions a pair).  20,000
// particles, law R: 0.34 ms for the whole call, 0.64 ms with the library's
// reciprocal square root and arctangent, 7.61 ms with one workgroup per 256
// particles over every ordered pair (79 workgroups on 256 CUs) and a square
// root, a division and an arctangent a pair.
template <int LAW>
__global__ __launch_bounds__(kDiagBlock) void diag_potential_kernel(const float4* __restrict__ pos,
                                                                    const double* __restrict__ mass,
                                                                    const double* __restrict__ gm, int n, int nb,
                                                                    int per, double soft, double* __restrict__ out) {
    __shared__ double red[kDiagBlock];
    __shared__ double2 txy[kDiagTile], tzg[kDiagTile];
    const int i = blockIdx.x * kDiagBlock + threadIdx.x;
    const bool active = i < n;
    double xi = 0, yi = 0, zi = 0, mi = 0;
    if (active) {
        const float4 p = pos[i];
        xi = p.x;
        yi = p.y;
        zi = p.z;
        mi = mass[i];
    }
    const double rs = sqrt(soft), inv_rs = 1.0 / rs;
    const bool mine = __builtin_isfinite(xi + yi + zi);  // sums of doubles: no overflow from finite floats
    double phi = 0.0;
    const int last = min((static_cast<int>(blockIdx.y) + 1) * per, nb / 2 + 1);
    for (int d = blockIdx.y * per; d < last; ++d) {
        if (d > 0 && 2 * d == nb && static_cast<int>(blockIdx.x) >= d) break;  // counted from the other side
        int J = blockIdx.x + d;
        if (J >= nb) J -= nb;
        const int jt = J * kDiagTile, j = jt + threadIdx.x;
        double2 xy = make_double2(0.0, 0.0), zg = make_double2(0.0, 0.0);
        if (j < n) {
            const float4 p = pos[j];
            xy = make_double2(p.x, p.y);
            zg = make_double2(p.z, gm[j]);
        }
        const bool finite = mine && __builtin_isfinite(xy.x + xy.y + zg.x);
        // also the barrier after the previous tile's last read
        const bool plain = __syncthreads_and(finite && soft > 0.0);
        txy[threadIdx.x] = xy;
        tzg[threadIdx.x] = zg;
        __syncthreads();
        if (!active) continue;
        const int jn = min(kDiagTile, n - jt);
        double sum = 0.0;
        auto pairs = [&](auto is_plain, auto own) {
#pragma unroll 2
            for (int l = 0; l < jn; ++l) {
                const double g = pair_potential<LAW, is_plain.value>(txy[l].x - xi, txy[l].y - yi, tzg[l].x - zi, soft,
                                                                     rs, inv_rs);
                if constexpr (own.value) sum += jt + l == i ? 0.0 : tzg[l].y * g;
                else sum = fma(tzg[l].y, g, sum);
            }
        };
        using yes = std::true_type;
        using no = std::false_type;
        if (d == 0) plain ? pairs(yes{}, yes{}) : pairs(no{}, yes{});
        else plain ? pairs(yes{}, no{}) : pairs(no{}, no{});
        phi -= d == 0 ? 0.5 * sum : sum;
    }
    if (LAW == NBODY_LAW_R && rs > 0) phi /= rs;
    const double s = block_sum(active ? mi * phi : 0.0, red);
    if (threadIdx.x == 0) out[blockIdx.y * nb + blockIdx.x] = s;
}

// The distances' runs: enough workgroups for eight waves per SIMD (2,048 on
// 256 CUs), never an empty run.
struct DiagGrid {
    int nb, per, runs;
};

DiagGrid diag_grid(int n) {
    DiagGrid g{};
    g.nb = n < 1 ? 1 : (n + kDiagBlock - 1) / kDiagBlock;
    const int dists = g.nb / 2 + 1;
    const int want = std::min(dists, (2048 + g.nb - 1) / g.nb);
    g.per = (dists + want - 1) / want;
    g.runs = (dists + g.per - 1) / g.per;
    return g;
}

}  // namespace

int diag_local_blocks(int n) {
    int b = (n + kDiagBlock - 1) / kDiagBlock;
    return b < 1 ? 1 : (b > 1024 ? 1024 : b);
}

int diag_potential_blocks(int n) {
    const DiagGrid g = diag_grid(n);
    return g.nb * g.runs;
}

hipError_t diag_launch(const float4* pos, const float4* vel, const double* mass, const double* gm, int n,
                       int law, double soft, double* local_out, double* pot_out, hipStream_t stream) {
    hipLaunchKernelGGL(diag_local_kernel, dim3(diag_local_blocks(n)), dim3(kDiagBlock), 0, stream, pos, vel,
                       mass, n, local_out);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const DiagGrid g = diag_grid(n);
    const auto potential =
        law == NBODY_LAW_R ? diag_potential_kernel<NBODY_LAW_R> : diag_potential_kernel<NBODY_LAW_P>;
    hipLaunchKernelGGL(potential, dim3(g.nb, g.runs), dim3(kDiagBlock), 0, stream, pos, mass, gm, n, g.nb, g.per, soft,
                       pot_out);
    return hipGetLastError();
}

}  // namespace nbody
