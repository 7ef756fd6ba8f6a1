// Direct-sum gravity on gfx950: O(N^2) pair forces with LDS j-tiles.
//
// A step of fewer than 16,384 particles is one launch (small_step_kernel below),
// a larger one takes every unordered pair once (direct_sym.hip).  The one-sided
// sum described here, direct_force_kernel, runs where the launch is tuned by hand,
// where the rows of the pair sums find no room, and as the batch's baseline.
//
// Replaces the reference's BruteForceCPU::Exec/Update
// (src/Sim/BruteForceCPU.cpp:25-73) and the D3D11 pair of compute shaders
// (shaders/Compute/Gravity.csh:28-48, Update.csh:22-36), written from the
// force law, not translated.
//
// Layout: one float4 (x, y, z, G*m) per particle, padded to a multiple of
// kTile with massless dummies at the origin.  A workgroup owns
// block * i_per_lane targets; each lane keeps i_per_lane targets in registers.
// The workgroup streams its j-range through LDS one tile of kTile particles at
// a time (the next tile is prefetched into registers while the current one is
// consumed), and every lane reads the same LDS record per j, so the read is a
// broadcast.  Per tile the lane sums into plain FP32 registers; the tile sums
// are then added into a per-target compensated (Kahan) accumulator, so the
// rounding of the long sum grows with the number of tiles, not of particles.
//
// The pair arithmetic, the issue-rate choices behind it and the compensated
// summation are described with the shared core in direct_core.hpp.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <cmath>

#include "../../include/nbody.h"
#include "common.hpp"
#include "direct.hpp"
#include "direct_core.hpp"

namespace nbody {

namespace {

using core::kahan_add;

// Kick then drift of target i with the acceleration (ax, ay, az).
__device__ __forceinline__ void kick_drift(const DirectLaunch& L, int i, float ax, float ay, float az) {
    float4 v = L.vel[i];
    float4 x = L.src[i];
    v.x = __builtin_fmaf(ax, L.dt, v.x);
    v.y = __builtin_fmaf(ay, L.dt, v.y);
    v.z = __builtin_fmaf(az, L.dt, v.z);
    x.x = __builtin_fmaf(v.x, L.dts, x.x);
    x.y = __builtin_fmaf(v.y, L.dts, x.y);
    x.z = __builtin_fmaf(v.z, L.dts, x.z);
    L.vel[i] = v;
    L.pos_out[i] = x;
}

// One workgroup: targets [blockIdx.x * BLOCK * K, +BLOCK*K), sources
// [blockIdx.y * jchunk, +jchunk) clipped to n_pad.  KICK fuses the kick-drift
// update (only launched with a single j-chunk).
template <int LAW, int K, int BLOCK, bool KICK>
__global__ __launch_bounds__(BLOCK) void direct_force_kernel(DirectLaunch L, int jchunk) {
    __shared__ core::SrcTile tiles[2];

    const int tid = threadIdx.x;
    const int ibase = blockIdx.x * (BLOCK * K);

    float xi[K], yi[K], zi[K];
#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = min(ibase + tid + k * BLOCK, L.n_pad - 1);
        const float4 q = L.src[i];
        xi[k] = q.x * L.sc.inv_len;
        yi[k] = q.y * L.sc.inv_len;
        zi[k] = q.z * L.sc.inv_len;
    }

    const int j0 = blockIdx.y * jchunk;
    const int j1 = min(j0 + jchunk, L.n_pad);
    float sx[K], sy[K], sz[K];
    core::block_forces<LAW, K, BLOCK>(tiles, L.src, j0, j1, L.sc, xi, yi, zi, sx, sy, sz);

#pragma unroll
    for (int k = 0; k < K; ++k) {
        const int i = ibase + tid + k * BLOCK;
        if constexpr (KICK) {
            if (i < L.n) {
                const float ax = sx[k] * L.sc.out, ay = sy[k] * L.sc.out, az = sz[k] * L.sc.out;
                kick_drift(L, i, ax, ay, az);
                L.acc[i] = make_float4(ax, ay, az, 0.f);
            }
        } else {
            if (i < L.n_pad) L.part[(size_t)blockIdx.y * L.n_pad + i] = make_float4(sx[k], sy[k], sz[k], 0.f);
        }
    }
}

// Adds the j-chunk partial sums of each target in chunk order (compensated),
// scales them back, then either kicks and drifts (kick != 0) or only stores
// the acceleration.
__global__ __launch_bounds__(256) void reduce_kick_kernel(DirectLaunch L, int split, int kick) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= L.n) return;
    float sx = 0.f, sy = 0.f, sz = 0.f, cx = 0.f, cy = 0.f, cz = 0.f;
    for (int s = 0; s < split; ++s) {
        const float4 p = L.part[(size_t)s * L.n_pad + i];
        kahan_add(sx, cx, p.x);
        kahan_add(sy, cy, p.y);
        kahan_add(sz, cz, p.z);
    }
    const float ax = sx * L.sc.out, ay = sy * L.sc.out, az = sz * L.sc.out;
    L.acc[i] = make_float4(ax, ay, az, 0.f);
    if (kick) kick_drift(L, i, ax, ay, az);
}

// A whole step of a small system in one launch.  A workgroup of sixteen
// wavefronts owns T targets and all sources: a wavefront holds its T targets
// 64 / T times over, and each of the 1,024 / T copies takes every (1,024 / T)-th
// source of a tile of 1,024, so that a system of a few thousand particles fills
// the chip without chunks of sources whose sums a second kernel has to add.
// The copies' compensated sums are added lane by lane, then wave by wave, in a
// fixed order.  The pair is unfolded (13 FP32 instructions and one v_rsq_f32,
// the mass multiplied in last): folding it costs a division per staged source,
// and every workgroup stages them all.
//
// Bound by latency up to about 4,000 particles (a launch, the staging, one to
// four tiles), then by the pair arithmetic.  A step, ms, against the chunked
// one-sided sum and its second kernel, with T = 8 / 16 targets: 1,000 particles
// 0.0127 -> 0.0050 / 0.0053; 2,000 0.0130 -> 0.0062 / 0.0070; 3,000 0.0152 ->
// 0.0095 / 0.0087; 4,096 0.0147 -> 0.0112 / 0.0103; 8,192 0.0276 -> 0.0299 /
// 0.0252; 12,288 0.0549 -> 0.0600 / 0.0516.  (T = 4 and 32 lose everywhere.)
constexpr int kSmallThreads = 1024;
constexpr int kSmallWaves = kSmallThreads / 64;

//
// FAR (law R, some real particle has no mass): massless sources are staged far
// away, as core::stage_source does; they pull nothing then, even from a position
// that is not finite.  Always done, it costs 1% at 12,288 particles.
template <int LAW, int T, bool KICK, bool FAR>
__global__ __launch_bounds__(kSmallThreads) __attribute__((amdgpu_waves_per_eu(8))) void small_step_kernel(DirectLaunch L) {
    constexpr int COPIES = kSmallThreads / T;       // copies of each target
    constexpr int PER = kSmallThreads / COPIES;     // sources a copy takes of a tile
    static_assert(PER % 4 == 0, "whole groups of four reciprocal square roots");
    __shared__ float4 tile[2][kSmallThreads];
    __shared__ float sums[6][kSmallWaves][T];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int i = blockIdx.x * T + (lane & (T - 1));
    const int copy = wave * (64 / T) + lane / T;
    const float tiny = core::in_vgpr(__FLT_MIN__);
    const float soft = core::in_vgpr(L.sc.soft);
    const float inv_c = LAW == NBODY_LAW_R ? 1.0f / L.sc.mass_k : L.sc.mass_k;  // a power of two
    auto scaled = [&](int j) {
        const float4 p = j < L.n_pad ? L.src[j] : make_float4(0.f, 0.f, 0.f, 0.f);
        return make_float4(p.x * L.sc.inv_len, p.y * L.sc.inv_len, p.z * L.sc.inv_len, p.w * inv_c);
    };
    auto source = [&](int j) {
        float4 q = scaled(j);
        if constexpr (FAR) {
            if (!(q.w > 0.f)) q.x = q.y = q.z = 0x1p100f;
        }
        return q;
    };
    const float4 me = scaled(min(i, L.n_pad - 1));
    float s[3] = {0.f, 0.f, 0.f}, c[3] = {0.f, 0.f, 0.f};
    tile[0][tid] = source(tid);
    __syncthreads();
    int buf = 0;
    for (int jt = 0; jt < L.n_pad; jt += kSmallThreads) {
        const bool more = jt + kSmallThreads < L.n_pad;
        float4 next;
        if (more) next = source(jt + kSmallThreads + tid);
        float ax = 0.f, ay = 0.f, az = 0.f;
#pragma unroll 2
        for (int g = 0; g < PER; g += 4) {
            float4 p[4];
            float dx[4], dy[4], dz[4], q[4];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                p[k] = tile[buf][(g + k) * COPIES + copy];
                dx[k] = p[k].x - me.x;
                dy[k] = p[k].y - me.y;
                dz[k] = p[k].z - me.z;
                if constexpr (LAW == NBODY_LAW_R) {
                    const float r2 = __builtin_fmaf(dz[k], dz[k], __builtin_fmaf(dy[k], dy[k], dx[k] * dx[k]));
                    const float t = r2 + soft;
                    const float u = r2 * t;
                    q[k] = __builtin_fmaf(u, t, tiny);
                } else {
                    q[k] = __builtin_fmaf(dz[k], dz[k], __builtin_fmaf(dy[k], dy[k], __builtin_fmaf(dx[k], dx[k], soft)));
                }
            }
            core::rsq4(q[0], q[1], q[2], q[3]);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const float f = LAW == NBODY_LAW_R ? q[k] * p[k].w : (p[k].w * q[k]) * (q[k] * q[k]);
                ax = __builtin_fmaf(dx[k], f, ax);
                ay = __builtin_fmaf(dy[k], f, ay);
                az = __builtin_fmaf(dz[k], f, az);
            }
        }
        kahan_add(s[0], c[0], ax);
        kahan_add(s[1], c[1], ay);
        kahan_add(s[2], c[2], az);
        if (more) {
            // the other buffer was last read before the previous barrier
            tile[buf ^ 1][tid] = next;
            __syncthreads();
            buf ^= 1;
        }
    }
#pragma unroll
    for (int off = T; off < 64; off <<= 1) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            const float os = __shfl_xor(s[a], off), oc = __shfl_xor(c[a], off);
            kahan_add(s[a], c[a], os);
            kahan_add(s[a], c[a], -oc);
        }
    }
    if (lane < T) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            sums[a][wave][lane] = s[a];
            sums[3 + a][wave][lane] = c[a];
        }
    }
    __syncthreads();
    if (tid >= T || i >= L.n) return;
    for (int w = 1; w < kSmallWaves; ++w)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            kahan_add(s[a], c[a], sums[a][w][lane]);
            kahan_add(s[a], c[a], -sums[3 + a][w][lane]);
        }
    const float ax = s[0] * L.sc.out, ay = s[1] * L.sc.out, az = s[2] * L.sc.out;
    L.acc[i] = make_float4(ax, ay, az, 0.f);
    if constexpr (KICK) kick_drift(L, i, ax, ay, az);
}

// Acceleration at arbitrary points (3m packed floats) from all sources: one
// target per lane, every workgroup over the whole source range.
template <int LAW>
__global__ __launch_bounds__(256) void field_kernel(const float4* __restrict__ src, int n_src_pad,
                                                    const float* __restrict__ pts, int m, DirectScale sc,
                                                    float* __restrict__ out) {
    __shared__ core::SrcTile tiles[2];
    const int i = blockIdx.x * 256 + threadIdx.x;
    const size_t p = 3 * static_cast<size_t>(min(i, m - 1));
    float xi[1] = {pts[p] * sc.inv_len}, yi[1] = {pts[p + 1] * sc.inv_len}, zi[1] = {pts[p + 2] * sc.inv_len};
    float sx[1], sy[1], sz[1];
    core::block_forces<LAW, 1, 256>(tiles, src, 0, n_src_pad, sc, xi, yi, zi, sx, sy, sz);
    if (i < m) {
        out[p] = sx[0] * sc.out;
        out[p + 1] = sy[0] * sc.out;
        out[p + 2] = sz[0] * sc.out;
    }
}

// The same with the sources shared out three times, for few points: a workgroup
// holds 64 points and takes the tiles of one chunk, [blockIdx.y * jchunk,
// +jchunk); each half of it takes half of the chunk's tiles, and wave w of the half
// a quarter of each.  part[chunk * m + i] receives the chunk's sums in scaled
// units.
//
// Bound by the pair arithmetic once the chip is full: 65,536 points from 262,144
// sources 4.9 ms (3.5e12 pairs/s), 5.5 with 256 threads to a workgroup (the
// partial sums allow 1,024 workgroups, half the waves that the chip holds); with
// 1,024 threads 4.8, but 100 points take 57 us against 47.  4,096 points 0.36 ms
// with the copies and the sum, 0.39 with 256 threads, 8.60 ms on the 16
// workgroups that one per 256 points over all sources makes.
constexpr int kFieldParts = 2;
constexpr int kFieldThreads = 256 * kFieldParts;

template <int LAW>
__global__ __launch_bounds__(kFieldThreads) __attribute__((amdgpu_waves_per_eu(8))) void field_slice_kernel(const float4* __restrict__ src, int n_src_pad,
                                                          const float* __restrict__ pts, int m, DirectScale sc,
                                                          int jchunk, float4* __restrict__ part) {
    __shared__ core::SrcTile tiles[kFieldParts][2];
    __shared__ core::WaveSums<kFieldThreads / 64> sums;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int i = blockIdx.x * 64 + lane;
    const size_t p = 3 * static_cast<size_t>(min(i, m - 1));
    float xi[1] = {pts[p] * sc.inv_len}, yi[1] = {pts[p + 1] * sc.inv_len}, zi[1] = {pts[p + 2] * sc.inv_len};
    float sx[1], sy[1], sz[1], cx[1], cy[1], cz[1];
    const int j0 = blockIdx.y * jchunk, j1 = min(j0 + jchunk, n_src_pad);
    const int turns = ((j1 - j0) / kTile + kFieldParts - 1) / kFieldParts;
    const int part_id = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) / 256);
    const int p0 = j0 + part_id * turns * kTile, p1 = min(p0 + turns * kTile, j1);
    core::block_forces_comp<LAW, 1, 256, 4, kFieldParts>(tiles[part_id], src, p0, p1, sc, xi, yi, zi, sx, sy, sz, cx,
                                                         cy, cz, turns);
    float s[3] = {sx[0], sy[0], sz[0]}, c[3] = {cx[0], cy[0], cz[0]};
    core::add_slices(sums, wave, lane, s, c);
    if (wave != 0 || i >= m) return;
    float r[3] = {-c[0], -c[1], -c[2]};
#pragma unroll
    for (int a = 0; a < 3; ++a) core::add_keeping_rest(s[a], r[a]);
    part[static_cast<size_t>(blockIdx.y) * m + i] = core::pack_sums(s, r);
}

// Adds the chunks' sums of each point (compensated, in a fixed order) and scales
// them back.  A workgroup takes 16 points, the 16 threads of each every 16th
// chunk: with one thread to a point the 1,024 chunks of a single point among
// 262,144 sources took 0.1 ms of its 0.143.
__global__ __launch_bounds__(256) void field_sum_kernel(const float4* __restrict__ part, int split, int m,
                                                        DirectScale sc, float* __restrict__ out) {
    __shared__ float sums[6][16][16];
    const int pt = threadIdx.x & 15, row = threadIdx.x >> 4;
    const int i = blockIdx.x * 16 + pt;
    float s[3] = {0.f, 0.f, 0.f}, c[3] = {0.f, 0.f, 0.f};
    if (i < m) {
#pragma unroll 4
        for (int k = row; k < split; k += 16) {
            float x[3], r[3];
            core::unpack_sums(part[static_cast<size_t>(k) * m + i], x, r);
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                core::add_keeping_rest(s[a], x[a]);
                c[a] -= x[a] + r[a];
            }
        }
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) sums[a][row][pt] = s[a], sums[3 + a][row][pt] = c[a];
    __syncthreads();
    if (row != 0 || i >= m) return;
    float* o = out + 3 * static_cast<size_t>(i);
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        for (int r = 1; r < min(16, split); ++r) {
            float x = sums[a][r][pt];
            core::add_keeping_rest(s[a], x);
            c[a] += sums[3 + a][r][pt] - x;
        }
        o[a] = (s[a] - c[a]) * sc.out;
    }
}

// Chunks the field's sources are split into (0: field_kernel, no partial
// sums).  One workgroup per 256 points over all sources fills the chip's
// 2,048 workgroup places of eight waves per SIMD only from 524,288 points on;
// below 262,144 (the half of it, still faster than 64 points each, whose
// workgroups stage every tile four times as often per pair) a workgroup takes
// 64 points and the sources are split until there are 2,048 workgroups, as far
// as there are tiles and as the partial sums fit kFieldPartials records (from
// 65,537 points on a single chunk).  Depends on the two sizes only, so the
// entry with a staging array of its own gives the same bits.
constexpr int kFieldPartials = NBODY_FIELD_NOALLOC_MAX_POINTS;

int field_split(int m, int n_src_pad) {
    if (m >= 262144) return 0;
    const int tiles = n_src_pad / kTile, blocks = (m + 63) / 64;
    const int want = std::max(1, std::min({(2048 + blocks - 1) / blocks, kFieldPartials / m, tiles}));
    const int per = (tiles + want - 1) / want;
    return (tiles + per - 1) / per;  // no empty chunk
}

using ForceFn = void (*)(DirectLaunch, int);

template <int LAW, int K, int BLOCK>
ForceFn pick_kick(bool kick) {
    return kick ? direct_force_kernel<LAW, K, BLOCK, true> : direct_force_kernel<LAW, K, BLOCK, false>;
}

template <int LAW, int K>
ForceFn pick_block(int block, bool kick) {
    switch (block) {
        case 64: return pick_kick<LAW, K, 64>(kick);
        case 128: return pick_kick<LAW, K, 128>(kick);
        case 256: return pick_kick<LAW, K, 256>(kick);
        default: return nullptr;
    }
}

template <int LAW>
ForceFn pick_k(int k, int block, bool kick) {
    switch (k) {
        case 1: return pick_block<LAW, 1>(block, kick);
        case 2: return pick_block<LAW, 2>(block, kick);
        case 4: return pick_block<LAW, 4>(block, kick);
        case 8: return pick_block<LAW, 8>(block, kick);
        default: return nullptr;
    }
}

ForceFn pick(int law, int k, int block, bool kick) {
    return law == NBODY_LAW_R ? pick_k<NBODY_LAW_R>(k, block, kick) : pick_k<NBODY_LAW_P>(k, block, kick);
}

using SmallFn = void (*)(DirectLaunch);

template <int T>
SmallFn pick_small(const DirectLaunch& L, bool kick) {
    if (L.law == NBODY_LAW_P)
        return kick ? small_step_kernel<NBODY_LAW_P, T, true, false> : small_step_kernel<NBODY_LAW_P, T, false, false>;
    if (L.massless)
        return kick ? small_step_kernel<NBODY_LAW_R, T, true, true> : small_step_kernel<NBODY_LAW_R, T, false, true>;
    return kick ? small_step_kernel<NBODY_LAW_R, T, true, false> : small_step_kernel<NBODY_LAW_R, T, false, false>;
}

}  // namespace

bool direct_shape_valid(const DirectShape& s) {
    const bool k_ok = s.i_per_lane == 1 || s.i_per_lane == 2 || s.i_per_lane == 4 || s.i_per_lane == 8;
    const bool b_ok = s.block == 64 || s.block == 128 || s.block == 256;
    return k_ok && b_ok && s.split >= 1;
}

DirectScale direct_scale_for(int law, double softening, double extent, double max_gm) {
    DirectScale sc{};
    // lambda: the power of two nearest the geometric mean of the shortest and
    // longest distances that matter, so that their sixth powers (law R's rsq
    // argument grows as r^6) sit symmetrically inside FP32's range.  The
    // longest is the diagonal of the extent; the shortest is the softening
    // length, or the spacing of FP32 positions across the extent (2^-24 of it)
    // when that is larger.
    const double r_hi = std::sqrt(3.0) * std::max(extent, 0.0);
    const double r_lo = std::max(std::sqrt(std::max(softening, 0.0)), std::ldexp(std::max(extent, 0.0), -24));
    int e_len = 0;
    if (r_hi > 0 && r_lo > 0 && std::isfinite(r_hi) && std::isfinite(r_lo))
        e_len = static_cast<int>(std::lround(0.5 * (std::log2(r_hi) + std::log2(r_lo))));
    else if (r_lo > 0 && std::isfinite(r_lo))
        e_len = static_cast<int>(std::lround(std::log2(r_lo)));
    e_len = std::max(-120, std::min(120, e_len));
    // c: the power of two at or below the largest G m
    int e_mass = 0;
    if (max_gm > 0 && std::isfinite(max_gm)) {
        (void)std::frexp(max_gm, &e_mass);  // max_gm in [2^(e-1), 2^e)
        e_mass -= 1;
    }
    e_mass = std::max(-120, std::min(120, e_mass));
    // keep out = 2^(e_mass - 2 e_len) a normal float
    e_mass = std::max(2 * e_len - 120, std::min(2 * e_len + 120, e_mass));
    sc.inv_len = std::ldexp(1.0f, -e_len);
    sc.mass_k = law == NBODY_LAW_R ? std::ldexp(1.0f, e_mass) : std::ldexp(1.0f, -e_mass);
    sc.soft = static_cast<float>(std::ldexp(softening, -2 * e_len));
    sc.out = std::ldexp(1.0f, e_mass - 2 * e_len);
    return sc;
}

double equal_gm(double G, const double* mass, size_t n) {
    const float first = n ? static_cast<float>(G * mass[0]) : 0.f;
    if (!(first > 0.f) || !std::isfinite(first)) return 0.0;
    bool same = true;
    for (size_t i = 1; i < n; ++i) {
        if (static_cast<float>(G * mass[i]) != first) return 0.0;
        same = same && mass[i] == mass[0];
    }
    return same ? G * mass[0] : static_cast<double>(first);
}

SymUnits sym_units(int law, double softening, const DirectScale& sc, double gm_equal) {
    SymUnits u{gm_equal > 0, 1.0f, sc.soft, 0.f, 0.f};
    double out = sc.out;
    if (u.equal) {
        out *= gm_equal * (law == NBODY_LAW_R ? 1.0 / sc.mass_k : sc.mass_k);
    } else if (law == NBODY_LAW_R) {
        // With alpha = 1 the sum of r2, rounded already, and S' rounds the same way
        // for every r2 of a binade, an error that no number of pairs averages out: 3%
        // of the RMS error at N = 2^20, 7% at 2^21.  The product's bits below r2's
        // last make it a random one, as the one-sided sum's folded mass does.  Of
        // the 64 factors with seven such bits the one whose alpha S' is nearest a
        // float.
        const double s = softening * static_cast<double>(sc.inv_len) * static_cast<double>(sc.inv_len);
        double best = 1.0;
        for (int k = 1; k < 128; k += 2) {
            const double as = s * (128 + k) / 128.0, off = std::fabs(static_cast<double>(static_cast<float>(as)) - as);
            if (s == 0.0 || off < best * as) best = s == 0.0 ? 0.0 : off / as, u.alpha = (128 + k) / 128.0f;
        }
        u.soft = static_cast<float>(s * static_cast<double>(u.alpha));
        out *= u.alpha;
    }
    u.out_hi = static_cast<float>(out);
    if (std::isfinite(u.out_hi)) u.out_lo = static_cast<float>(out - static_cast<double>(u.out_hi));
    return u;
}

int direct_effective_split(const DirectShape& s, int n_pad) {
    const int tiles = n_pad / kTile;
    int split = s.split < 1 ? 1 : s.split;
    if (split > tiles) split = tiles;
    const int tiles_per_chunk = (tiles + split - 1) / split;
    return (tiles + tiles_per_chunk - 1) / tiles_per_chunk;
}

DirectShape direct_default_shape(int n_pad) {
    // One target per lane keeps the register count, and so the waves per SIMD,
    // highest; below ~1024 workgroups of targets the j-range is split so that
    // the 256 CUs still see about a thousand workgroups.
    DirectShape s{1, 256, 1};
    const int iblocks = (n_pad + s.block - 1) / s.block;
    if (iblocks < 1024) s.split = (1024 + iblocks - 1) / iblocks;
    return s;
}

size_t direct_field_scratch(int m, int n_src_pad) {
    return static_cast<size_t>(field_split(m, n_src_pad)) * static_cast<size_t>(m);
}

hipError_t direct_field(const float4* src, int n_src_pad, const float* pts, int m, int law, const DirectScale& sc,
                        float4* part, float* out, hipStream_t stream) {
    if (m <= 0) return hipSuccess;
    const bool r = law == NBODY_LAW_R;
    const int split = field_split(m, n_src_pad);
    if (split == 0) {
        hipLaunchKernelGGL((r ? field_kernel<NBODY_LAW_R> : field_kernel<NBODY_LAW_P>), dim3((m + 255) / 256),
                           dim3(256), 0, stream, src, n_src_pad, pts, m, sc, out);
        return hipGetLastError();
    }
    const int tiles = n_src_pad / kTile;
    const int jchunk = ((tiles + split - 1) / split) * kTile;
    hipLaunchKernelGGL((r ? field_slice_kernel<NBODY_LAW_R> : field_slice_kernel<NBODY_LAW_P>),
                       dim3((m + 63) / 64, split), dim3(kFieldThreads), 0, stream, src, n_src_pad, pts, m, sc, jchunk, part);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(field_sum_kernel, dim3((m + 15) / 16), dim3(256), 0, stream, part, split, m, sc, out);
    return hipGetLastError();
}

hipError_t small_step(const DirectLaunch& L, bool kick, hipStream_t stream, hipEvent_t ev_b, hipEvent_t ev_e) {
    // Fewer targets a workgroup while the workgroups do not fill the 256 CUs.
    const int t = L.n_pad <= 2048 ? 8 : 16;
    const SmallFn fn = t == 8 ? pick_small<8>(L, kick) : pick_small<16>(L, kick);
    hipError_t e = hipSuccess;
    if (ev_b && (e = hipEventRecord(ev_b, stream)) != hipSuccess) return e;
    hipLaunchKernelGGL(fn, dim3((L.n + t - 1) / t), dim3(kSmallThreads), 0, stream, L);
    if ((e = hipGetLastError()) != hipSuccess) return e;
    if (ev_e && (e = hipEventRecord(ev_e, stream)) != hipSuccess) return e;
    return hipSuccess;
}

hipError_t direct_step(const DirectLaunch& L, const DirectShape& s, bool kick, hipStream_t stream,
                       hipEvent_t ev_force_begin, hipEvent_t ev_force_end) {
    const int split = direct_effective_split(s, L.n_pad);
    const int tiles = L.n_pad / kTile;
    const int jchunk = ((tiles + split - 1) / split) * kTile;
    const bool fused = kick && split == 1;
    ForceFn fn = pick(L.law, s.i_per_lane, s.block, fused);
    if (!fn) return hipErrorInvalidValue;
    const int per_block = s.block * s.i_per_lane;
    dim3 grid((L.n_pad + per_block - 1) / per_block, split);
    if (ev_force_begin) {
        hipError_t e = hipEventRecord(ev_force_begin, stream);
        if (e != hipSuccess) return e;
    }
    hipLaunchKernelGGL(fn, grid, dim3(s.block), 0, stream, L, jchunk);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (ev_force_end) {
        e = hipEventRecord(ev_force_end, stream);
        if (e != hipSuccess) return e;
    }
    if (!fused) {
        DirectLaunch R = L;
        hipLaunchKernelGGL(reduce_kick_kernel, dim3((L.n + 255) / 256), dim3(256), 0, stream, R, split,
                           kick ? 1 : 0);
        e = hipGetLastError();
        if (e != hipSuccess) return e;
    }
    return hipSuccess;
}

}  // namespace nbody

extern "C" nbody_status nbody_direct_scale(int32_t law, double softening, double extent, double max_gm,
                                           float* out4) {
    nbody::clear_error();
    NB_CHECK(out4, NBODY_ERR_INVALID_ARG, "out is null");
    NB_CHECK(law == NBODY_LAW_R || law == NBODY_LAW_P, NBODY_ERR_INVALID_ARG, "unknown law %d", law);
    const nbody::DirectScale sc = nbody::direct_scale_for(law, softening, extent, max_gm);
    out4[0] = sc.inv_len;
    out4[1] = sc.mass_k;
    out4[2] = sc.soft;
    out4[3] = sc.out;
    return NBODY_OK;
}
