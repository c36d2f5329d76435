// lus_fluid.hip -- the reference's simulate_fluid (src/Simulate.cpp:27-115) on
// the GPU, with the reference's semantics kept exactly:
//
//   * dt clamped to [0.001, 0.01]; v += g * mass * dt; x* = x + v dt (:31, :48-51)
//   * neighbour lists of find_neighbors_uniform_grid (Neighbors.cpp:366-450):
//     per particle the 27 cells in (dy, dx, dz) order, each cell's moving
//     particles in ascending slot then its solids in ascending slot, self
//     included; built from a stable counting sort of the predicted positions
//   * lambda per particle with the cubic kernel (Kernels.cpp:5-41), self
//     counted twice in the density (:58-88) -- independent per particle
//   * the pressure sweep (:90-113) is sequential in the reference: particle i
//     reads x* of the particles before it as already corrected (in place) and
//     of those after it as predicted, and uses lambdas[t] for the t-th entry
//     of its list.  Here it runs as a data flow: the corrected positions go to
//     an array of their own, cleared to a "not yet" pattern before the sweep,
//     and particle i waits for the entries of its neighbours j < i there and
//     reads the predicted positions of those after it.  So a particle reads
//     every earlier neighbour corrected and every later one predicted: exactly
//     the reference's sequential sweep, in parallel (k_fl_sweep).
//
// Arithmetic follows the reference's operation order with no contraction and
// IEEE divide and square root (the library's build flags).  One call differs
// from the reference's binary: std::pow(float, float) in s_coor is glibc's
// powf; here the power is taken in double and rounded once (the correctly
// rounded value), which glibc's powf returns except for about 7 in 10,000
// arguments, where it is one ulp away.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cmath>
#include <cstring>
#include <vector>

#include "lus_device.hpp"
#include "lus_internal.hpp"
#include "lus_launch.hpp"
#include "lustrine_gpu.h"

namespace lus {

struct FluidK {
    float r, h, h2, f, ck, cl, mass, rho0, eps, scorr_k, scorr_n, W0, Wdq;
    float gm[3];          // gravity * mass, per component (float products)
    float hi[3];          // (int)domain - r, per axis: resolve_collision's max
    float cs;
    int gX, gY, gZ, gXZ;
    int s0, n;            // first moving slot, moving count
    int nl;               // entries of the lambdas array
    int ipow;             // s_corr_n as an exact small integer, or -1
};

struct FluidState {
    LusFluidParams p{};
    FluidK k{};
    int total = 0, s0 = 0, s1 = 0, t0 = 0, t1 = 0, C = 0, ns = 0;
    bool stepped = false;
    int last_levels = 0;
    long last_entries = 0;
    std::vector<void*> ptrs;
    float4 *x = nullptr, *xs = nullptr, *v = nullptr, *sorted = nullptr, *osorted = nullptr;
    float* lam = nullptr;
    int *key = nullptr, *slot = nullptr, *counts = nullptr, *cs = nullptr, *tmp = nullptr,
        *perm = nullptr, *ks = nullptr, *tiles = nullptr, *inv = nullptr;
    int *ocs = nullptr, *oref = nullptr;
    int *cnt = nullptr, *off = nullptr, *ltiles = nullptr, *idx = nullptr;
    long cap = 0;
    void* idx_mem = nullptr;
    float4* xs2 = nullptr;    // the sweep's output; swapped with xs after it
    int* ctl = nullptr;       // see kCtl*
    int* host_ctl = nullptr;  // pinned mirror of ctl
    float* stage = nullptr;   // a download's packed arrays
};

constexpr int kCtlTicket = 0;    // next block of the sweep
constexpr int kCtlLevels = 1;    // longest chain of waits of the sweep
constexpr int kCtlErr = 2;       // error bits
constexpr int kCtlInts = 4;
constexpr int kErrKey = 1;       // a predicted position lies outside the grid
constexpr int kErrLambda = 2;    // a list is longer than the lambdas array
constexpr int kErrStall = 4;     // the sweep gave up waiting

void fluid_free(FluidState* F) {
    if (!F) return;
    for (void* q : F->ptrs) (void)hipFree(q);
    if (F->idx_mem) (void)hipFree(F->idx_mem);
    if (F->host_ctl) (void)hipHostFree(F->host_ctl);
    delete F;
}

// ------------------------------------------------------------------ kernels
// cubic_kernel (Kernels.cpp:5-19); with kernelFactor 1/2 and neighbours within
// h, q <= 1/2 and only the first branch is taken
__device__ __forceinline__ float fl_cubic(const FluidK& k, float r) {
    const float q = (r * k.f) / k.h;
    float result = 0.0f;
    if ((double)q <= 1.0) {
        if ((double)q <= 0.5) {
            const float q2 = q * q;
            const float q3 = q2 * q;
            const float a = 6.0f * q3;
            const float b = 6.0f * q2;
            result = k.ck * ((a - b) + 1.0f);
        } else {
            const float t = 1.0f - q;
            const double t3 = ((double)t * (double)t) * (double)t;
            result = k.ck * (2.0f * (float)t3);
        }
    }
    return result;
}

// cubic_kernel_grad (Kernels.cpp:26-41)
__device__ __forceinline__ void fl_cubic_grad(const FluidK& k, float dx, float dy, float dz, float* gx,
                                              float* gy, float* gz) {
    const float rl = sqrtf(dot3(dx, dy, dz, dx, dy, dz)) * k.f;
    const float q = rl / k.h;
    float ox = 0.0f, oy = 0.0f, oz = 0.0f;
    if ((double)rl > 1.0e-5 && (double)q <= 1.0) {
        const float c = 1.0f / (rl * k.h);
        const float qx = c * dx, qy = c * dy, qz = c * dz;
        float sc;
        if ((double)q <= 0.5) {
            sc = (k.cl * q) * (3.0f * q - 2.0f);
        } else {
            const float t = 1.0f - q;
            sc = k.cl * ((-t) * t);
        }
        ox = sc * qx;
        oy = sc * qy;
        oz = sc * qz;
    }
    *gx = ox;
    *gy = oy;
    *gz = oz;
}

// std::pow(x, n) of s_coor (Simulate.cpp:7-9), rounded once from double
__device__ __forceinline__ float fl_pow(const FluidK& k, float x) {
    if (k.ipow >= 0) {
        double acc = 1.0, b = (double)x;
        int e = k.ipow;
        while (e) {
            if (e & 1) acc *= b;
            b *= b;
            e >>= 1;
        }
        return (float)acc;
    }
    return (float)pow((double)x, (double)k.scorr_n);
}

// resolve_collision (Simulate.cpp:11-24)
__device__ __forceinline__ float fl_resolve(float value, float lo, float hi) {
    if (value <= lo) return 0.01f;
    if (value > hi) return hi - 0.01f;
    return value;
}

// integration (:48-51) and the cell key of each moving particle
// and its "not yet" mark in the sweep's output
__global__ __launch_bounds__(kBlock) void k_fl_predict(float4* __restrict__ x, float4* __restrict__ v,
                                                        float4* __restrict__ xs, float4* __restrict__ xs2, FluidK k,
                                                        float dt, int* __restrict__ key, int C,
                                                        int* __restrict__ ctl) {
    const int t = xcd_index();
    if (t >= k.n) return;
    const int i = k.s0 + t;
    float4 vi = v[i];
    vi.x = vi.x + k.gm[0] * dt;
    vi.y = vi.y + k.gm[1] * dt;
    vi.z = vi.z + k.gm[2] * dt;
    const float4 p = x[i];
    float4 q;
    q.x = p.x + vi.x * dt;
    q.y = p.y + vi.y * dt;
    q.z = p.z + vi.z * dt;
    q.w = 0.0f;
    v[i] = vi;
    xs[i] = q;
    const float open = __uint_as_float(~0u);
    xs2[i] = make_float4(open, open, open, open);
    // get_cell_id (Utils.hpp:24-33) has no clamp: a cell index outside
    // [0, C) indexes outside the reference's cell vector; here it is reported
    // (an index inside [0, C) is used as the reference uses it, even when a
    // coordinate lies past its axis)
    const float px = q.x / k.cs, py = q.y / k.cs, pz = q.z / k.cs;
    bool bad = !(fabsf(px) < 1.0e9f && fabsf(py) < 1.0e9f && fabsf(pz) < 1.0e9f);
    int c = 0;
    if (!bad) {
        const long long cl = (long long)(int)py * k.gXZ + (long long)(int)px * k.gZ + (long long)(int)pz;
        bad = cl < 0 || cl >= C;
        c = (int)cl;
    }
    if (bad) {
        atomicOr(&ctl[kCtlErr], kErrKey);
        c = 0;
    }
    key[t] = c;
}

__global__ __launch_bounds__(kBlock) void k_fl_gather(const float4* __restrict__ xs, const int* __restrict__ perm,
                                                       int s0, int n, float4* __restrict__ sorted,
                                                       int* __restrict__ inv) {
    const int p = xcd_index();
    if (p >= n) return;
    const int t = perm[p];
    sorted[p] = xs[s0 + t];
    inv[t] = p;
}

// find_neighbors_uniform_grid: counts (fill == 0) or entries (fill == 1) of
// moving particle t's list; entries are reference slots
__global__ __launch_bounds__(kBlock) void k_fl_lists(const float4* __restrict__ sorted,
                                                      const int* __restrict__ skey,
                                                      const int* __restrict__ scs,
                                                      const int* __restrict__ sperm,
                                                      const int* __restrict__ inv,
                                                      const float4* __restrict__ osorted,
                                                      const int* __restrict__ ocs,
                                                      const int* __restrict__ oref, FluidK k,
                                                      const int* __restrict__ off, int* __restrict__ cnt,
                                                      int* __restrict__ idx, int fill) {
    const int t = xcd_index();
    if (t >= k.n) return;
    const int p = inv[t];
    const float4 me = sorted[p];
    const int c = skey[p];
    const int yy = c / k.gXZ;
    const int rm = c - yy * k.gXZ;
    const int xx = rm / k.gZ;
    const int zz = rm - xx * k.gZ;
    int o = fill ? off[t] : 0;
    int count = 0;
    for (int y = -1; y <= 1; ++y) {
        if (yy + y < 0 || yy + y >= k.gY) continue;
        for (int x = -1; x <= 1; ++x) {
            if (xx + x < 0 || xx + x >= k.gX) continue;
            for (int z = -1; z <= 1; ++z) {
                if (zz + z < 0 || zz + z >= k.gZ) continue;
                const int nc = (yy + y) * k.gXZ + (xx + x) * k.gZ + (zz + z);
                const int a = scs[nc], b = scs[nc + 1];
                for (int j = a; j < b; ++j) {
                    const float4 q = sorted[j];
                    const float dx = me.x - q.x, dy = me.y - q.y, dz = me.z - q.z;
                    if (dot3(dx, dy, dz, dx, dy, dz) <= k.h2) {
                        if (fill) idx[o + count] = k.s0 + sperm[j];
                        ++count;
                    }
                }
                if (osorted) {
                    const int oa = ocs[nc], ob = ocs[nc + 1];
                    for (int j = oa; j < ob; ++j) {
                        const float4 q = osorted[j];
                        const float dx = me.x - q.x, dy = me.y - q.y, dz = me.z - q.z;
                        if (dot3(dx, dy, dz, dx, dy, dz) <= k.h2) {
                            if (fill) idx[o + count] = oref[j];
                            ++count;
                        }
                    }
                }
            }
        }
    }
    if (!fill) cnt[t] = count;
}

// lambda of each moving particle (:58-88)
__global__ __launch_bounds__(kBlock) void k_fl_lambda(const float4* __restrict__ xs, const int* __restrict__ off,
                                                       const int* __restrict__ idx, FluidK k,
                                                       float* __restrict__ lam, int* __restrict__ ctl) {
    const int t = xcd_index();
    if (t >= k.n) return;
    const int i = k.s0 + t;
    const int a = off[t], b = off[t + 1];
    const float4 pi = xs[i];
    float density = 0.0f;
    for (int e = a; e < b; ++e) {
        const int j = idx[e];
        const float4 pj = xs[j];
        const float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
        const float len = sqrtf(dot3(dx, dy, dz, dx, dy, dz));
        density = density + k.mass * fl_cubic(k, len);
    }
    density = density + k.mass * k.W0;
    const float constraint = (float)((double)(density / k.rho0) - 1.0);
    float gsum = 0.0f, gcx = 0.0f, gcy = 0.0f, gcz = 0.0f;
    const float m = -(k.mass / k.rho0);
    for (int e = a; e < b; ++e) {
        const int j = idx[e];
        const float4 pj = xs[j];
        float gx, gy, gz;
        fl_cubic_grad(k, pi.x - pj.x, pi.y - pj.y, pi.z - pj.z, &gx, &gy, &gz);
        const float nx = m * gx, ny = m * gy, nz = m * gz;
        gsum = gsum + dot3(nx, ny, nz, nx, ny, nz);
        gcx = gcx - nx;
        gcy = gcy - ny;
        gcz = gcz - nz;
    }
    gsum = gsum + dot3(gcx, gcy, gcz, gcx, gcy, gcz);
    float l = 0.0f;
    if ((double)gsum > 0.0) l = -constraint / (gsum + k.eps);
    lam[i] = l;
    if (b - a > k.nl) atomicOr(&ctl[kCtlErr], kErrLambda);
}

// The pressure sweep (:90-113) as a data flow.  A term whose neighbour is a solid or comes later in the
// sweep (predicted position) is computed at once; an earlier neighbour's is
// computed when its corrected position shows up in xs2.  The terms meet in LDS
// and are added in list order, one lane per component, so the sums are the
// sequential sweep's bit for bit.
//
// A corrected position is its own signal: x, y, z and the chain length are
// agent-scope 4-byte stores over the all-ones words k_fl_predict left, and a
// reader takes the position when none of them is all ones (no flag, no fence,
// which would write back and invalidate an XCD's whole L2).
//
// Blocks take their particles in slot order by ticket, so every particle waited for
// belongs to the same wave (whose loop serves all its particles) or to a wave
// that already runs: every wait ends.  (kSweepSpins passes without progress
// end it with an error all the same.)
//
// At 32 K particles the longest chain of waits bounds it, 2.7 to 3.2 us a link
// (a bare store and load between two XCDs takes 0.6; the rest is the last term,
// its sum and the divides): 218 links 0.82 ms a step, 905 links 2.8 ms, where one
// launch per level (36 us a link and more) took 8.7 and 66.  At 1 M (762 links,
// 17.5 ms, 37 with launches) it is the window of particles in flight.  A
// particle that waits for at most kSweepFew neighbours asks for each; one that waits
// for more asks for the latest of each eight lanes (of each four with 16 lanes a
// particle), so that the waves far from the front leave the ones at it alone.
// The latest of the whole particle alone took 32 K (800 steps) 949 ms, 262 K
// 4.28 ms and 1 M 19.0 ms; every missing one 925, 3.85, 16.9; this 887, 4.00, 17.5.
// Between two askings it pauses (1, 4, 10, 30 x 64 cycles at the 905 links: 2.95,
// 2.86, 2.78, 2.86 ms).
//
// kLanes lanes hold one particle and take its list kLanes * kPer entries at a
// time, entry e in lane e % kLanes.  Few particles per wave shorten a link
// (they take turns), many widen the window of particles in flight, which bounds
// large scenes (launch_sweep).
// kPow4: s_corr_n = 4 (the Simulation default), else any exponent.
constexpr unsigned int kOpen = ~0u;                      // "not yet"
constexpr int kSweepSpins = 1 << 22;
constexpr int kSweepPause = 10;                          // x 64 cycles between two askings
constexpr int kSweepFew = 4;

// max over the kLanes lanes of a particle, in every one of them
template <int kCtrl>
__device__ __forceinline__ int dpp_max(int v) {
    const int o = __builtin_amdgcn_update_dpp(v, v, kCtrl, 0xF, 0xF, false);
    return o > v ? o : v;
}
__device__ __forceinline__ int quad_max(int v) {  // of the lane's four
    v = dpp_max<0xB1>(v);                        // lane ^ 1
    return dpp_max<0x4E>(v);                     // lane ^ 2
}
template <int kLanes>
__device__ __forceinline__ int sweep_max(int v) {
    v = quad_max(v);
    v = dpp_max<0x141>(v);                       // half row mirrored
    v = dpp_max<0x140>(v);                       // row mirrored
#pragma unroll
    for (int d = 16; d < kLanes; d <<= 1) {
        const int o = __shfl_xor(v, d, 64);
        v = o > v ? o : v;
    }
    return v;
}

struct SweepPos {
    unsigned long long xy, zc;  // (x, y), (z, chain length)
    __device__ __forceinline__ bool here() const {
        return (unsigned int)xy != kOpen && (unsigned int)(xy >> 32) != kOpen && (unsigned int)zc != kOpen &&
               (unsigned int)(zc >> 32) != kOpen;
    }
};
__device__ __forceinline__ SweepPos sweep_load(const unsigned long long* out, int j) {
    SweepPos q;
    q.xy = __hip_atomic_load(out + 2 * (size_t)j, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    q.zc = __hip_atomic_load(out + 2 * (size_t)j + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    return q;
}
__device__ __forceinline__ unsigned long long pack2(float a, float b) {
    return (unsigned long long)__float_as_uint(b) << 32 | __float_as_uint(a);
}

// one term of the sweep's sum: (lambda_i + lambdas[t] + s_corr) grad W
template <bool kPow4, int kRow>
__device__ __forceinline__ void fl_term(const FluidK& k, const float4 pi, float px, float py, float pz, float ll,
                                        float* __restrict__ out) {
    const float dx = pi.x - px, dy = pi.y - py, dz = pi.z - pz;
    const float len = sqrtf(dot3(dx, dy, dz, dx, dy, dz));
    const float ratio = fl_cubic(k, len) / k.Wdq;
    float pw;
    if constexpr (kPow4) {
        const double b = (double)ratio, b2 = b * b;
        pw = (float)(b2 * b2);
    } else {
        pw = fl_pow(k, ratio);
    }
    const float coef = ll + -k.scorr_k * pw;
    float gx, gy, gz;
    fl_cubic_grad(k, dx, dy, dz, &gx, &gy, &gz);
    out[0] = coef * gx;
    out[kRow] = coef * gy;
    out[2 * kRow] = coef * gz;
}

template <bool kPow4, int kLanes, int kPer>
__global__ __launch_bounds__(kBlock) void k_fl_sweep(float4* __restrict__ x, const float4* __restrict__ xs, float4* xs2,
                                                      float4* __restrict__ v, const float* __restrict__ lam,
                                                      const int* __restrict__ off, const int* __restrict__ idx,
                                                      FluidK k, float dt, int* __restrict__ ctl) {
    static_assert(kLanes == 16 || kLanes == 32 || kLanes == 64, "DPP rows");
    constexpr int kChunk = kLanes * kPer, kBlockP = kBlock / kLanes;
    constexpr int kRow = kChunk + 8;  // LDS floats per component (read eight at a time)
    __shared__ float terms[kBlockP][3 * kRow];
    __shared__ int ticket;
    if (threadIdx.x == 0) ticket = atomicAdd(&ctl[kCtlTicket], 1);
    __syncthreads();
    const int lane = (int)(threadIdx.x & 63);
    const int sub = lane & (kLanes - 1);
    const int first = lane - sub;  // the particle's first lane
    const unsigned long long group = (~0ull >> (64 - kLanes)) << first;
    const int t = ticket * kBlockP + (int)threadIdx.x / kLanes;
    float* const T = terms[threadIdx.x / kLanes];
    bool live = t < k.n;
    const int i = k.s0 + (live ? t : 0);
    const int a = live ? off[t] : 0, b = live ? off[t + 1] : 0;
    const float4 pi = xs[i];
    const float p0 = reinterpret_cast<const float*>(x + i)[sub & 3];
    const float li = lam[i];
    unsigned long long* const out = reinterpret_cast<unsigned long long*>(xs2);
    int j[kPer];
    float ll[kPer];
    SweepPos w[kPer];   // entry u's neighbour
    unsigned int pend = 0u;  // bit u: it is missing
    bool fresh = live;       // the chunk at c0 is to be taken
    bool ask = live;         // ask for everything missing
    int c0 = a, summed = 0;  // entries of the chunk in the sum
    float f = 0.0f;          // component sub (< 3) of the sum
    int chain = 0;
    unsigned int have = 0u;  // bit u: entry u's position is here, its term is not
    while (__any(live)) {
        if (fresh) {
            fresh = false;
            summed = 0;
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const int e = c0 + sub + u * kLanes;
                j[u] = e < b ? idx[e] : -1;
                // lambdas[t] with t the list position (:97); a list longer
                // than the lambdas array is reported after the step
                ll[u] = li + (e < b && e - a < k.nl ? lam[e - a] : 0.0f);
            }
#pragma unroll
            for (int u = 0; u < kPer; ++u) {
                const float4 p = xs[j[u] < 0 ? i : j[u]];
                w[u].xy = pack2(p.x, p.y);
                w[u].zc = pack2(p.z, 0.0f);
                if (j[u] >= k.s0 && j[u] < i)
                    pend |= 1u << u;
                else if (j[u] >= 0)
                    have |= 1u << u;
            }
        }
        if (ask) {
#pragma unroll
            for (int u = 0; u < kPer; ++u)
                if (pend >> u & 1u) w[u] = sweep_load(out, j[u]);
#pragma unroll
            for (int u = 0; u < kPer; ++u)
                if ((pend >> u & 1u) && w[u].here()) {
                    pend &= ~(1u << u);
                    have |= 1u << u;
                }
        }
        // a term per lane and turn, whichever entry it is
        while (__any((int)have)) {
            if (have) {
                // (a predicted position's chain length is 0)
                SweepPos q = w[0];
                float ql = ll[0];
                int e = sub;
#pragma unroll
                for (int u = 1; u < kPer; ++u)
                    if (!(have & ((1u << u) - 1u))) {
                        q = w[u];
                        ql = ll[u];
                        e = sub + u * kLanes;
                    }
                fl_term<kPow4, kRow>(k, pi, __uint_as_float((unsigned int)q.xy), __uint_as_float((unsigned int)(q.xy >> 32)),
                               __uint_as_float((unsigned int)q.zc), ql, T + e);
                const int c = (int)(q.zc >> 32);
                chain = c > chain ? c : chain;
                have &= have - 1u;
            }
        }
        wave_lds_sync();  // the terms are seen by the particle's other lanes
        // the sum goes on, in list order, up to the first missing term
        const int m = b - c0 < kChunk ? b - c0 : kChunk;
        int upto = m;
#pragma unroll
        for (int u = kPer - 1; u >= 0; --u) {
            const unsigned long long miss = __ballot(pend >> u & 1u) & group;
            if (miss) upto = __ffsll(miss) - 1 - first + u * kLanes;
        }
        if (live && sub < 3) {
            const float* const q = T + sub * kRow;
            for (int e = summed; e < upto; e += 8) {
                float w8[8];
#pragma unroll
                for (int d = 0; d < 8; ++d) w8[d] = q[e + d];
#pragma unroll
                for (int d = 0; d < 8; ++d)
                    if (e + d < upto) f = f + w8[d];
            }
        }
        summed = upto;
        if (live && upto == m) {
            c0 += kChunk;
            if (c0 < b) {
                fresh = true;
            } else {
                live = false;
                chain = sweep_max<kLanes>(chain) + 1;
                if (sub < 4) {
                    // lanes 0..2: the components; lane 3: the chain length
                    const float pc = sub == 0 ? pi.x : (sub == 1 ? pi.y : pi.z);
                    const float hc = sub == 0 ? k.hi[0] : (sub == 1 ? k.hi[1] : k.hi[2]);
                    const float o = fl_resolve(pc + f / k.rho0, k.r, hc);
                    // an all-ones NaN is published as another NaN
                    unsigned int word = __float_as_uint(o);
                    word = word == kOpen ? kOpen >> 1 : word;
                    __hip_atomic_store(reinterpret_cast<unsigned int*>(xs2 + i) + sub, sub < 3 ? word : (unsigned int)chain,
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    reinterpret_cast<float*>(x + i)[sub] = sub < 3 ? o : 0.0f;
                    reinterpret_cast<float*>(v + i)[sub] = sub < 3 ? (o - p0) / dt : 0.0f;
                }
            }
        }
        ask = fresh;
        if (__any(fresh) || !__any(live)) continue;
        // wait for a missing neighbour of any of the wave's particles
        int top = -1, u0 = 0;
#pragma unroll
        for (int u = 0; u < kPer; ++u)
            if ((pend >> u & 1u) && j[u] > top) {
                top = j[u];
                u0 = u;
            }
        const bool few = __popcll(__ballot(pend != 0u) & group) <= kSweepFew;
        const int latest = kLanes == 64 ? dpp_max<0x141>(quad_max(top)) : quad_max(top);
        const bool asks = top >= 0 && (few || latest == top);
        SweepPos q = {};
        bool here = false;
        int spins = 0;
        do {
            if (asks) {
                q = sweep_load(out, top);
                here = q.here();
            }
            if (__any(here)) break;
            __builtin_amdgcn_s_sleep(kSweepPause);
        } while (++spins < kSweepSpins);
        if (spins >= kSweepSpins) {
            if (lane == 0) atomicOr(&ctl[kCtlErr], kErrStall);
            break;
        }
        if (here) {
#pragma unroll
            for (int u = 0; u < kPer; ++u)
                if (u == u0) w[u] = q;
            pend &= ~(1u << u0);
            have |= 1u << u0;
        }
        ask = !few && (__ballot(here) & group) != 0ull;
    }
    // the longest chain, one atomic per wave
    for (int d = 32; d >= 1; d >>= 1) {
        const int o = __shfl_xor(chain, d, 64);
        chain = o > chain ? o : chain;
    }
    if (lane == 0) atomicMax(&ctl[kCtlLevels], chain);
}

template <int kLanes, int kPer>
static void launch_sweep_lanes(float4* x, const float4* xs, float4* xs2, float4* v, const float* lam, const int* off,
                               const int* idx, const FluidK& k, float dt, int* ctl, hipStream_t s) {
    const dim3 g((k.n + kBlock / kLanes - 1) / (kBlock / kLanes)), b(kBlock);
    if (k.ipow == 4)
        launch_kernel((k_fl_sweep<true, kLanes, kPer>), g, b, 0, s, x, xs, xs2, v, lam, off, idx, k, dt, ctl);
    else
        launch_kernel((k_fl_sweep<false, kLanes, kPer>), g, b, 0, s, x, xs, xs2, v, lam, off, idx, k, dt, ctl);
}

// A wave per particle while the particles in flight (8,192 at 8 waves per
// SIMD) cover most of the sweep's front, else four particles per wave
// (measured, one / two / four per wave: 32 K at 870 links 2.8 / 3.6 / 4.4 ms,
// 262 K 6.4 / 4.6 / 4.0 ms, 1 M 27 / 20 / 17.5 ms).
constexpr int kSweepWideN = 65536;

static hipError_t launch_sweep(float4* x, const float4* xs, float4* xs2, float4* v, const float* lam, const int* off,
                               const int* idx, const FluidK& k, float dt, int* ctl, hipStream_t s) {
    if (k.n <= kSweepWideN)
        launch_sweep_lanes<64, 1>(x, xs, xs2, v, lam, off, idx, k, dt, ctl, s);
    else
        launch_sweep_lanes<16, 4>(x, xs, xs2, v, lam, off, idx, k, dt, ctl, s);
    return hipGetLastError();
}

}  // namespace lus

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
namespace {

#define FL_HIP(call)                                                                                \
    do {                                                                                            \
        hipError_t e_ = (call);                                                                     \
        if (e_ != hipSuccess)                                                                       \
            return lus::report_error(LUS_EHIP, "%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), \
                                     __FILE__, __LINE__);                                           \
    } while (0)

template <class T>
hipError_t fl_alloc(lus::FluidState* F, T** out, size_t count) {
    void* q = nullptr;
    hipError_t e = hipMalloc(&q, std::max<size_t>(count, 1) * sizeof(T));
    if (e == hipSuccess) F->ptrs.push_back(q);
    *out = static_cast<T*>(q);
    return e;
}

std::vector<float4> aos_to_f4(const float* xyz, int first, int count) {
    std::vector<float4> out((size_t)std::max(count, 0));
    for (int i = 0; i < count; ++i) {
        const float* q = xyz + 3 * (size_t)(first + i);
        out[i] = make_float4(q[0], q[1], q[2], 0.0f);
    }
    return out;
}

int fl_grid_ok(const LusGrid& g) {
    return g.cell_size > 0.0f && g.gridX > 0 && g.gridY > 0 && g.gridZ > 0 &&
           (long long)g.gridX * g.gridY * g.gridZ < (1LL << 30);
}

}  // namespace

int lus_fluid_init(LusGpu* c, const LusFluidParams* p, int total, int sand_start, int sand_end, int solid_start,
                   int solid_end, const float* positions, const float* positions_star, const float* velocities,
                   int n_lambdas, const float* lambdas) {
    if (!c || !p || total <= 0 || !positions || !positions_star || !velocities || n_lambdas < 0 ||
        (n_lambdas && !lambdas))
        return lus::report_error(LUS_EINVAL, "lus_fluid_init: bad arguments");
    if (sand_start < 0 || sand_end < sand_start || sand_end > total || solid_start < 0 ||
        solid_end < solid_start || solid_end > total || (sand_end > sand_start && solid_end > solid_start &&
                                                         solid_start < sand_end && sand_start < solid_end))
        return lus::report_error(LUS_EINVAL, "lus_fluid_init: bad particle ranges");
    if (n_lambdas < sand_end)
        return lus::report_error(LUS_EINVAL,
                                 "lus_fluid_init: lambdas has %d entries, the moving slots reach %d (the "
                                 "reference writes lambdas[i] for every moving slot)",
                                 n_lambdas, sand_end);
    if (!fl_grid_ok(p->grid)) return lus::report_error(LUS_EINVAL, "lus_fluid_init: bad grid");
    if (!(p->kernelRadius > 0.0f) || !(p->rest_density != 0.0f) || !(p->mass > 0.0f))
        return lus::report_error(LUS_EINVAL, "lus_fluid_init: bad constants");
    const LusGrid& g = p->grid;
    const int C = g.gridX * g.gridY * g.gridZ;
    // solids never move: their cells are fixed, and must exist
    for (int i = solid_start; i < solid_end; ++i) {
        const float* q = positions_star + 3 * (size_t)i;
        const float px = q[0] / g.cell_size, py = q[1] / g.cell_size, pz = q[2] / g.cell_size;
        if (!(px >= 0.0f && py >= 0.0f && pz >= 0.0f) || (int)px >= g.gridX || (int)py >= g.gridY ||
            (int)pz >= g.gridZ)
            return lus::report_error(LUS_EINVAL, "lus_fluid_init: solid slot %d lies outside the grid", i);
    }
    const int dev = lus::ctx_device(c);
    hipStream_t s = lus::ctx_stream(c);
    FL_HIP(hipSetDevice(dev));
    FL_HIP(hipStreamSynchronize(s));
    lus::FluidState*& slot = lus::ctx_fluid(c);
    lus::fluid_free(slot);
    slot = nullptr;
    auto* F = new lus::FluidState();
    slot = F;
    F->p = *p;
    F->total = total;
    F->s0 = sand_start;
    F->s1 = sand_end;
    F->t0 = solid_start;
    F->t1 = solid_end;
    F->C = C;
    F->ns = solid_end - solid_start;
    const int n = sand_end - sand_start;
    lus::FluidK& k = F->k;
    k.r = p->particleRadius;
    k.h = p->kernelRadius;
    {
        volatile float hh = p->kernelRadius;
        k.h2 = hh * hh;
    }
    k.f = p->kernelFactor;
    k.ck = p->cubic_kernel_k;
    k.cl = p->cubic_kernel_l;
    k.mass = p->mass;
    k.rho0 = p->rest_density;
    k.eps = p->relaxation_epsilon;
    k.scorr_k = p->s_corr_k;
    k.scorr_n = p->s_corr_n;
    k.ipow = (p->s_corr_n >= 0.0f && p->s_corr_n <= 64.0f && p->s_corr_n == std::floor(p->s_corr_n))
                 ? (int)p->s_corr_n
                 : -1;
    for (int a = 0; a < 3; ++a) {
        volatile float gma = p->gravity[a] * p->mass;
        k.gm[a] = gma;
        volatile float hi = (float)(int)p->domain[a] - p->particleRadius;
        k.hi[a] = hi;
    }
    k.cs = g.cell_size;
    k.gX = g.gridX;
    k.gY = g.gridY;
    k.gZ = g.gridZ;
    k.gXZ = g.gridX * g.gridZ;
    k.s0 = sand_start;
    k.n = n;
    k.nl = n_lambdas;
    // W(0) and W(dq), the host evaluating the device's formula
    auto cubic = [&](float r) {
        volatile float q = (r * k.f) / k.h;
        if ((double)q > 1.0) return 0.0f;
        if ((double)q <= 0.5) {
            volatile float q2 = q * q;
            volatile float q3 = q2 * q;
            volatile float a = 6.0f * q3;
            volatile float b = 6.0f * q2;
            volatile float ab = a - b;
            volatile float ab1 = ab + 1.0f;
            return k.ck * ab1;
        }
        volatile float t = 1.0f - q;
        const double t3 = ((double)t * (double)t) * (double)t;
        volatile float two = 2.0f * (float)t3;
        return k.ck * two;
    };
    k.W0 = cubic(0.0f);
    k.Wdq = cubic(p->s_corr_dq);

    FL_HIP(fl_alloc(F, &F->x, total));
    FL_HIP(fl_alloc(F, &F->xs, total));
    FL_HIP(fl_alloc(F, &F->v, total));
    FL_HIP(fl_alloc(F, &F->lam, std::max(n_lambdas, 1)));
    FL_HIP(fl_alloc(F, &F->sorted, n));
    FL_HIP(fl_alloc(F, &F->key, n));
    FL_HIP(fl_alloc(F, &F->slot, n));
    FL_HIP(fl_alloc(F, &F->counts, C + 1));
    FL_HIP(fl_alloc(F, &F->cs, C + 1));
    FL_HIP(fl_alloc(F, &F->tmp, n));
    FL_HIP(fl_alloc(F, &F->perm, n));
    FL_HIP(fl_alloc(F, &F->ks, n));
    FL_HIP(fl_alloc(F, &F->tiles, lus::scan_tile_count(C + 1) + 1));
    FL_HIP(fl_alloc(F, &F->inv, n));
    FL_HIP(fl_alloc(F, &F->cnt, n + 1));
    FL_HIP(fl_alloc(F, &F->off, n + 1));
    FL_HIP(fl_alloc(F, &F->ltiles, lus::scan_tile_count(n + 1) + 1));
    FL_HIP(fl_alloc(F, &F->xs2, total));
    FL_HIP(fl_alloc(F, &F->ctl, lus::kCtlInts));
    FL_HIP(hipHostMalloc((void**)&F->host_ctl, sizeof(int) * lus::kCtlInts, hipHostMallocDefault));
    FL_HIP(hipMemsetAsync(F->counts, 0, sizeof(int) * (C + 1), s));

    std::vector<float4> h = aos_to_f4(positions, 0, total);
    FL_HIP(hipMemcpyAsync(F->x, h.data(), sizeof(float4) * total, hipMemcpyHostToDevice, s));
    FL_HIP(hipStreamSynchronize(s));
    h = aos_to_f4(positions_star, 0, total);
    FL_HIP(hipMemcpyAsync(F->xs, h.data(), sizeof(float4) * total, hipMemcpyHostToDevice, s));
    FL_HIP(hipMemcpyAsync(F->xs2, F->xs, sizeof(float4) * total, hipMemcpyDeviceToDevice, s));
    FL_HIP(hipStreamSynchronize(s));
    std::vector<float4> hv((size_t)total, make_float4(0.0f, 0.0f, 0.0f, 0.0f));
    for (int i = sand_start; i < sand_end; ++i) {
        const float* q = velocities + 3 * (size_t)i;
        hv[i] = make_float4(q[0], q[1], q[2], 0.0f);
    }
    FL_HIP(hipMemcpyAsync(F->v, hv.data(), sizeof(float4) * total, hipMemcpyHostToDevice, s));
    if (n_lambdas) FL_HIP(hipMemcpyAsync(F->lam, lambdas, sizeof(float) * n_lambdas, hipMemcpyHostToDevice, s));

    // solids: sorted once by cell (ascending slot inside a cell, as they
    // enter the reference's cell vectors)
    const int ns = F->ns;
    FL_HIP(fl_alloc(F, &F->osorted, ns));
    FL_HIP(fl_alloc(F, &F->ocs, C + 1));
    FL_HIP(fl_alloc(F, &F->oref, ns));
    {
        std::vector<int> okey((size_t)ns);
        for (int q = 0; q < ns; ++q) {
            const float* pp = positions_star + 3 * (size_t)(solid_start + q);
            okey[q] = ((int)(pp[1] / g.cell_size)) * g.gridX * g.gridZ + ((int)(pp[0] / g.cell_size)) * g.gridZ +
                      (int)(pp[2] / g.cell_size);
        }
        std::vector<int> ocnt((size_t)C + 1, 0), order((size_t)ns);
        for (int q = 0; q < ns; ++q) ocnt[okey[q] + 1]++;
        for (int cc = 0; cc < C; ++cc) ocnt[cc + 1] += ocnt[cc];
        std::vector<int> fillp(ocnt.begin(), ocnt.end() - 1);
        for (int q = 0; q < ns; ++q) order[fillp[okey[q]]++] = q;  // stable: ascending slot
        std::vector<float4> os((size_t)ns);
        std::vector<int> orf((size_t)ns);
        for (int q = 0; q < ns; ++q) {
            const float* pp = positions_star + 3 * (size_t)(solid_start + order[q]);
            os[q] = make_float4(pp[0], pp[1], pp[2], 0.0f);
            orf[q] = solid_start + order[q];
        }
        if (ns) {
            FL_HIP(hipMemcpyAsync(F->osorted, os.data(), sizeof(float4) * ns, hipMemcpyHostToDevice, s));
            FL_HIP(hipMemcpyAsync(F->oref, orf.data(), sizeof(int) * ns, hipMemcpyHostToDevice, s));
        }
        FL_HIP(hipMemcpyAsync(F->ocs, ocnt.data(), sizeof(int) * (C + 1), hipMemcpyHostToDevice, s));
        FL_HIP(hipStreamSynchronize(s));
    }
    F->stepped = false;
    return LUS_OK;
}

int lus_fluid_step(LusGpu* c, float dt) {
    if (!c) return lus::report_error(LUS_EINVAL, "lus_fluid_step: bad arguments");
    lus::FluidState* F = lus::ctx_fluid(c);
    if (!F) return lus::report_error(LUS_ESTATE, "lus_fluid_step: lus_fluid_init first");
    const int dev = lus::ctx_device(c);
    hipStream_t s = lus::ctx_stream(c);
    FL_HIP(hipSetDevice(dev));
    // dt = glm::clamp(dt, 0.001f, 0.01f) (Simulate.cpp:31)
    float t = dt < 0.001f ? 0.001f : dt;
    dt = 0.01f < t ? 0.01f : t;
    const lus::FluidK& k = F->k;
    const int n = k.n;
    FL_HIP(hipMemsetAsync(F->ctl, 0, sizeof(int) * lus::kCtlInts, s));
    F->last_levels = 0;
    F->last_entries = 0;
    if (n == 0) {
        F->stepped = true;
        return LUS_OK;
    }
    const int gb = lus::grid_for(n);
    lus::launch_kernel(lus::k_fl_predict, dim3(gb), dim3(lus::kBlock), 0, s, F->x, F->v, F->xs, F->xs2, k, dt,
                       F->key, F->C, F->ctl);
    FL_HIP(hipGetLastError());
    // stable counting sort of the moving particles by cell
    FL_HIP(lus::launch_count_keys(F->key, n, F->counts, F->slot, s));
    FL_HIP(lus::launch_exclusive_scan(F->counts, F->cs, F->C + 1, F->tiles, 1, s));
    FL_HIP(lus::launch_scatter(F->key, F->slot, F->cs, n, F->tmp, s));
    FL_HIP(lus::launch_stable_rank(F->tmp, F->key, F->cs, n, F->perm, F->ks, s));
    lus::launch_kernel(lus::k_fl_gather, dim3(gb), dim3(lus::kBlock), 0, s, F->xs, F->perm, k.s0, n, F->sorted,
                       F->inv);
    FL_HIP(hipGetLastError());
    // lists: counts, offsets, entries
    const float4* os = F->ns ? F->osorted : nullptr;
    lus::launch_kernel(lus::k_fl_lists, dim3(gb), dim3(lus::kBlock), 0, s, F->sorted, F->ks, F->cs, F->perm, F->inv,
                       os, F->ocs, F->oref, k, (const int*)nullptr, F->cnt, (int*)nullptr, 0);
    FL_HIP(hipGetLastError());
    FL_HIP(hipMemsetAsync(F->cnt + n, 0, sizeof(int), s));
    FL_HIP(lus::launch_exclusive_scan(F->cnt, F->off, n + 1, F->ltiles, 0, s));
    FL_HIP(hipMemcpyAsync(F->host_ctl, F->off + n, sizeof(int), hipMemcpyDeviceToHost, s));
    FL_HIP(hipMemcpyAsync(F->host_ctl + 1, F->ctl + lus::kCtlErr, sizeof(int), hipMemcpyDeviceToHost, s));
    FL_HIP(hipStreamSynchronize(s));
    if (F->host_ctl[1] & lus::kErrKey)
        return lus::report_error(LUS_EINVAL,
                                 "lus_fluid_step: a predicted position lies outside the grid (the reference "
                                 "indexes outside its cell vector there)");
    const long total = F->host_ctl[0];
    if (total < 0) return lus::report_error(LUS_EINVAL, "lus_fluid_step: more than 2^31 list entries");
    if (total > F->cap) {
        if (F->idx_mem) (void)hipFree(F->idx_mem);
        F->idx_mem = nullptr;
        F->cap = 0;
        const long want = total + total / 4 + 1024;
        FL_HIP(hipMalloc(&F->idx_mem, sizeof(int) * (size_t)want));
        F->cap = want;
    }
    F->idx = static_cast<int*>(F->idx_mem);
    F->last_entries = total;
    lus::launch_kernel(lus::k_fl_lists, dim3(gb), dim3(lus::kBlock), 0, s, F->sorted, F->ks, F->cs, F->perm, F->inv,
                       os, F->ocs, F->oref, k, (const int*)F->off, F->cnt, F->idx, 1);
    FL_HIP(hipGetLastError());
    lus::launch_kernel(lus::k_fl_lambda, dim3(gb), dim3(lus::kBlock), 0, s, (const float4*)F->xs,
                       (const int*)F->off, (const int*)F->idx, k, F->lam, F->ctl);
    FL_HIP(hipGetLastError());
    FL_HIP(lus::launch_sweep(F->x, F->xs, F->xs2, F->v, F->lam, F->off, F->idx, k, dt, F->ctl, s));
    std::swap(F->xs, F->xs2);
    FL_HIP(hipMemcpyAsync(F->host_ctl, F->ctl, sizeof(int) * lus::kCtlInts, hipMemcpyDeviceToHost, s));
    FL_HIP(hipStreamSynchronize(s));
    if (F->host_ctl[lus::kCtlErr] & lus::kErrStall)
        return lus::report_error(LUS_EHIP, "lus_fluid_step: the sweep stopped waiting for a particle");
    F->last_levels = F->host_ctl[lus::kCtlLevels];
    if (F->host_ctl[lus::kCtlErr] & lus::kErrLambda)
        return lus::report_error(LUS_EINVAL,
                                 "lus_fluid_step: a neighbour list is longer than the lambdas array (the "
                                 "reference reads past its vector there)");
    F->stepped = true;
    return LUS_OK;
}

int lus_fluid_download(LusGpu* c, float* positions, float* positions_star, float* velocities, float* lambdas) {
    if (!c) return lus::report_error(LUS_EINVAL, "lus_fluid_download: bad arguments");
    lus::FluidState* F = lus::ctx_fluid(c);
    if (!F) return lus::report_error(LUS_ESTATE, "lus_fluid_download: lus_fluid_init first");
    hipStream_t s = lus::ctx_stream(c);
    FL_HIP(hipSetDevice(lus::ctx_device(c)));
    // the arrays are packed on the device into one block: positions,
    // positions_star, the moving slots' velocities, lambdas (alone they come
    // from where they lie)
    const int total = F->total, moving = F->s1 - F->s0, nl = F->k.nl;
    const bool rows = positions || positions_star || velocities;
    if (rows && !F->stage) FL_HIP(fl_alloc(F, &F->stage, 6 * (size_t)total + 3 * (size_t)moving + (size_t)nl));
    lus::PackArgs pk{};
    lus::HostPiece pc[4];
    int np = 0;
    float* at = F->stage;
    if (positions) {
        pk.f[0] = {F->x, at, 0, total};
        pc[np++] = {positions, nullptr, sizeof(float) * 3 * (size_t)total};
        at += 3 * (size_t)total;
    }
    if (positions_star) {
        pk.f[1] = {F->xs, at, 0, total};
        pc[np++] = {positions_star, nullptr, sizeof(float) * 3 * (size_t)total};
        at += 3 * (size_t)total;
    }
    if (velocities) {
        pk.f[2] = {F->v, at, F->s0, F->s1};
        pc[np++] = {velocities + 3 * (size_t)F->s0, nullptr, sizeof(float) * 3 * (size_t)moving};
        at += 3 * (size_t)moving;
    }
    if (lambdas && nl) {
        if (rows) pk.i[0] = {reinterpret_cast<const int*>(F->lam), reinterpret_cast<int*>(at), nl};
        pc[np++] = {lambdas, nullptr, sizeof(float) * (size_t)nl};
    }
    if (np) {
        if (rows) FL_HIP(lus::launch_pack(pk, std::max(total, nl), s));
        FL_HIP(lus::pull_to_host(c, rows ? F->stage : F->lam, pc, np));
    } else {
        FL_HIP(hipStreamSynchronize(s));
    }
    return LUS_OK;
}

int lus_fluid_stats(LusGpu* c, int* levels, long* list_entries) {
    if (!c) return lus::report_error(LUS_EINVAL, "lus_fluid_stats: bad arguments");
    lus::FluidState* F = lus::ctx_fluid(c);
    if (!F) return lus::report_error(LUS_ESTATE, "lus_fluid_stats: lus_fluid_init first");
    if (levels) *levels = F->last_levels;
    if (list_entries) *list_entries = F->last_entries;
    return LUS_OK;
}
