// fs2d_pcg_loop.hpp -- the whole PCG loop of applyProjection
// (src/FluidSim2D.cpp:423-466) in one launch, for grids of few strips and for
// ensembles of them.
//
// Each strip of 64 rows belongs to one workgroup for the whole solve: it runs
// the strip's forward and backward solves (sweep_run), its SpMV and its p/r
// update, iteration after iteration.  Everything a strip reads is then its own,
// in its own XCD's L2, except
//   - the solves' boundary rows (HandRows, as in the separate launches);
//   - z of the two rows next to the strip, for the SpMV: the upper one is the
//     backward solve's boundary row, the lower one (the neighbour's last row)
//     is published as tagged words after that solve.  Each strip keeps s' of
//     both rows in LDS and updates it with the neighbour's own arithmetic;
//   - the partial sums of sigma, w.s and the maximum |r|, published as tagged
//     words {half, epoch + iteration} and added by every strip in one order.
// A word or row entry is itself the message, so nothing waits for caches or
// launches.  Separate launches of a small grid are mostly gaps and heads: of a
// 256^2 box's 44 us an iteration (48 in separate launches) the two solves'
// dependent steps take 30, and what is left, the SpMV and the update of a
// strip, is bound by one CU's loads from its L2.  More waves (10, 12) and p
// updated beside the next forward solve were 5-25% slower: the compiler then
// spills, and the solve's wave shares its SIMD.
//
// Strips of one simulation wait for each other, so all of them must be
// resident: every one first announces itself and waits for the others.
// Workgroups take (simulation, strip) from a ticket in order, so at most one
// simulation per launch is partly resident, and it holds fewer than
// kLoopMaxStrips workgroups while it waits for earlier simulations (which
// finish without it) or other streams' kernels to leave.  With one workgroup
// per CU, 256 CUs and HIP's 4 hardware queues, 16 strips leave room four times
// over; a device with fewer CUs takes the separate launches (loop_fits), and so
// do a process that asks for more queues and a stream with few CUs (loop_room).
#pragma once

#include "fs2d_kernels.hpp"

namespace fs2d {

constexpr int kLoopMaxStrips = 16;  // strips of one simulation: 1024 rows
// Columns.  A strip's SpMV and update run on its one CU, so their time grows
// with the width, where separate launches spread them.  us per iteration, loop
// and launches, boxes full of FLUID: 100^2 23/29, 256^2 44/48, 400x500 79/81,
// 512^2 84/86, 700^2 117/114, 1000x700 142/131.
constexpr int kLoopMaxNx = 576;
constexpr int kLoopWaves = 8;  // the sweep's 7, and the one that collects |r|
constexpr int kLoopThreads = 64 * kLoopWaves;
constexpr int kLoopSteps = kLoopMaxNx + 96;  // >= 4 T4
constexpr int kLoopPU = 3;  // groups of the p/r update in flight (4 arrays each)
constexpr int kLoopWords = 16;       // tagged words per strip
// word of a strip: sigma halves per loader, |r|_inf, w.s halves, its arrival
enum { kLwSigma = 0, kLwRmax = 2 * kLoaders, kLwWs = kLwRmax + 1, kLwArrive = kLwWs + 2 };
static_assert(kLwArrive < kLoopWords && kLoaders * kLoopMaxStrips <= 64, "one lane per sigma partial");
static_assert(kLoopWaves > 1 + kLoaders + kPollers, "a spare wave collects |r|");

inline bool loop_fits(const SkGeom& g, int ncu) {
    return g.S <= kLoopMaxStrips && g.nx <= kLoopMaxNx && ncu >= 8 * kLoopMaxStrips;
}
// Whether the strips that wait for each other, at most kLoopMaxStrips per launch
// and one launch per hardware queue, leave half of a stream's CUs to others: on
// 256 CUs with up to 8 queues.  The other side is separate launches with the
// same order of the sums, so no result depends on it.
inline bool loop_room(int cus, int queues) { return cus >= 2 * queues * kLoopMaxStrips; }
// Device words of one simulation: kLoopWords per strip, then a tagged row per strip.
__host__ __device__ inline size_t loop_words(const SkGeom& g) { return (size_t)g.S * (kLoopWords + 4 * g.T4); }

struct LoopArgs {
    SkGeom g;
    const float* Adiag;
    float *r, *p, *s0, *s1, *w, *z, *q;
    const float *P, *fx, *fy, *G;
    PcgScalars* sc;
    const int2* range;  // nullptr: every strip is active throughout
    HandRows rows;
    unsigned long long* words;  // loop_words
    int max_iters;
};

// One SK4 group of a strip's SpMV: w = A s' for the lane's 4 steps, and their
// share of w.s'.  The group's neighbours in the row come from the groups before
// and after it, those in the column from the next lanes; the edge lanes take
// dn / up, s' of the rows next to the strip.  s' is zero in every cell that is
// not FLUID, so the neighbours' sum needs no coupling bits; the terms and their
// order are spmv_core's.
__device__ __forceinline__ float4 spmv_group(const float4& prev, const float4& cur, const float4& nxt,
                                             const float4& ad, const float4& dn, const float4& up, double& acc) {
    const float left[4] = {prev.w, cur.x, cur.y, cur.z}, right[4] = {cur.y, cur.z, cur.w, nxt.x};
    float wv[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const float below = u2f(nbr<false, true>(f2u(f4get(dn, q)), f2u(left[q])));
        const float above = u2f(nbr<true, true>(f2u(f4get(up, q)), f2u(right[q])));
        const float nsum = ((left[q] + right[q]) + below) + above;
        const float a = f4get(ad, q), sc_ = f4get(cur, q);
        wv[q] = a != 0.0f ? fmaf(a, sc_, -nsum) : 0.0f;
        acc += (double)wv[q] * (double)sc_;
    }
    return make_float4(wv[0], wv[1], wv[2], wv[3]);
}
__device__ __forceinline__ float4 s_next(float beta, const float4& so, const float4& zc) {
    return make_float4(fmaf(beta, so.x, zc.x), fmaf(beta, so.y, zc.y), fmaf(beta, so.z, zc.z), fmaf(beta, so.w, zc.w));
}
__device__ __forceinline__ float4 ld4(const float* p) { return *(const float4*)p; }
// A strip's entries of one SK4 array, by group: scalar base and group offset,
// one register of lane offset for all of them (flat addresses of 12 groups of
// three arrays cost some 200 registers, and spilled).
struct StripArr {
    __amdgpu_buffer_rsrc_t rs;
    __device__ __forceinline__ StripArr(const float* a, const SkGeom& g, int s)
        : rs(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(a) + (long)s * g.T4 * 256, 0, g.T4 * 1024,
                                               kBufferCfg)) {}
    __device__ __forceinline__ float4 ld(int k) const {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        const u4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)(threadIdx.x & 63) * 16, k * 1024, 0);
        return make_float4(u2f(v.x), u2f(v.y), u2f(v.z), u2f(v.w));
    }
    __device__ __forceinline__ void st(int k, const float4& v) const {
        typedef uint32_t u4 __attribute__((ext_vector_type(4)));
        const u4 u = {f2u(v.x), f2u(v.y), f2u(v.z), f2u(v.w)};
        // no scalar offset: see sweep_compute's buffer stores
        __builtin_amdgcn_raw_buffer_store_b128(u, rs, (int)(threadIdx.x & 63) * 16 + k * 1024, 0, 0);
    }
};

// SpMV of a strip's groups ga .. gb-1 (of active groups lo .. hi-1) by one
// wave: s' = z + beta s, w = A s' and the lane's share of w.s'; kLoopU groups
// in flight at a time.
constexpr int kLoopU = 6;  // 10 with 8 groups in the update: 5% slower an iteration at 512^2
__device__ __forceinline__ double spmv_strip(int lo, int hi, int ga, int gb, const StripArr& Ad, const StripArr& Z,
                                             const StripArr& So, const StripArr& Sn, const StripArr& W, float beta,
                                             const float* dn, const float* up) {
    double acc = 0;
    if (ga >= gb) return acc;
    // the two groups before the first batch's are loaded with it, not before it
    const float4 so_p = So.ld(max(ga - 1, lo)), z_p = Z.ld(max(ga - 1, lo)), so_c = So.ld(ga), z_c = Z.ld(ga);
    float4 prev, cur;
    for (int g0 = ga; g0 < gb; g0 += kLoopU) {
        // the next groups' s and z (clamped into the range, tested below) and
        // this batch's matrix entries
        float4 so[kLoopU], zc[kLoopU], ad[kLoopU];
#pragma unroll
        for (int u = 0; u < kLoopU; u++) {
            so[u] = So.ld(min(g0 + u + 1, hi - 1));
            zc[u] = Z.ld(min(g0 + u + 1, hi - 1));
            ad[u] = Ad.ld(min(g0 + u, hi - 1));
        }
        if (g0 == ga) {
            prev = ga > lo ? s_next(beta, so_p, z_p) : make_float4(0, 0, 0, 0);
            cur = s_next(beta, so_c, z_c);
        }
#pragma unroll
        for (int u = 0; u < kLoopU; u++) {
            const int k = g0 + u;
            if (k >= gb) break;
            const float4 nxt = k + 1 < hi ? s_next(beta, so[u], zc[u]) : make_float4(0, 0, 0, 0);
            W.st(k, spmv_group(prev, cur, nxt, ad[u], ld4(dn + 4 * k), ld4(up + 4 * k), acc));
            Sn.st(k, cur);
            prev = cur;
            cur = nxt;
        }
    }
    return acc;
}
// r -= a w of one group; the largest |r|.
__device__ __forceinline__ float r_update(const StripArr& R, int k, float a, const float4& w, float4 v, float m) {
    v.x = fmaf(-a, w.x, v.x);
    v.y = fmaf(-a, w.y, v.y);
    v.z = fmaf(-a, w.z, v.z);
    v.w = fmaf(-a, w.w, v.w);
    R.st(k, v);
    return fmaxf(m, fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
}
// Sum of `acc` over a workgroup of kLoopThreads, in thread 0: lanes by
// butterfly, then waves in order.
__device__ __forceinline__ double loop_block_sum(double acc, double* part) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = acc;
    __syncthreads();
    double t = 0;
    for (int k = 0; k < kLoopWaves; k++) t += part[k];
    return t;
}

// The SpMV alone, a strip per workgroup, with the partial w.s of each strip:
// what the loop computes, for the separate launches that timing their phases,
// batches with larger members and streams without room for the loop need.  s' of the neighbouring rows is formed from
// their own s and z; outside the active range s' and w are set to zero, for the
// p/r update's launch, which covers the whole array.
__device__ __forceinline__ void spmv_strip_body(const SkGeom& g, const float* __restrict__ Adiag,
                                                const float* __restrict__ z, const float* __restrict__ s_old,
                                                float* __restrict__ s_new,
                                                float* __restrict__ w, float beta, double* partials,
                                                const int2* range, int s) {
    __shared__ __align__(16) float dn[kLoopSteps], up[kLoopSteps];
    __shared__ double part[kLoopWaves];
    const int wave = (int)uniform(threadIdx.x >> 6);
    const StripSpan sp = strip_span<false>(g, range, s), above = strip_span<false>(g, range, s + 1);
    for (int t = threadIdx.x; t < 4 * g.T4; t += kLoopThreads) {
        // lane 0 at step t is column t, lane 63 column t - 63
        const int td = t + 63, tu = t - 63;
        float d = 0, u = 0;
        if (td >= sp.up_lo && td < sp.up_hi) {
            const long e = (((long)(s - 1) * g.T4 + (td >> 2)) * 64 + 63) * 4 + (td & 3);
            d = fmaf(beta, s_old[e], z[e]);
        }
        if (tu >= 16 * above.lo && tu < 16 * above.hi) {
            const long e = ((long)(s + 1) * g.T4 + (tu >> 2)) * 256 + (tu & 3);
            u = fmaf(beta, s_old[e], z[e]);
        }
        dn[t] = d;
        up[t] = u;
    }
    __syncthreads();
    const int lo = 4 * sp.lo, hi = 4 * sp.hi, n = hi - lo;
    const StripArr Sn(s_new, g, s), W(w, g, s);
    const double acc = spmv_strip(lo, hi, lo + n * wave / kLoopWaves, lo + n * (wave + 1) / kLoopWaves,
                                  StripArr(Adiag, g, s), StripArr(z, g, s), StripArr(s_old, g, s), Sn, W, beta, dn, up);
    for (int k = wave; k < g.T4; k += kLoopWaves)
        if (k < lo || k >= hi) {
            Sn.st(k, make_float4(0, 0, 0, 0));
            W.st(k, make_float4(0, 0, 0, 0));
        }
    const double t = loop_block_sum(acc, part);
    if (threadIdx.x == 0) partials[s] = t;
}
__global__ __launch_bounds__(kLoopThreads) void pcg_spmv_strip_kernel(
    SkGeom g, const float* __restrict__ Adiag, const float* __restrict__ z, const float* __restrict__ s_old,
    float* __restrict__ s_new, float* __restrict__ w, PcgScalars* sc,
    const double* sig_cur, const double* sig_prev, int first, double* partials, const int2* range) {
    if (sc->done) return;
    const SpmvScalars S = spmv_scalars(g, sig_cur, sig_prev, first);
    if (blockIdx.x == 0 && threadIdx.x == 0) sc->sigma = S.sig;
    spmv_strip_body(g, Adiag, z, s_old, s_new, w, S.beta, partials, range, blockIdx.x);
}

// The backward solve inside the loop: its loaders' sigma partials are published.
struct LoopBwdOp : BwdOp {
    unsigned long long* words;
    unsigned tag;
    __device__ void loader_done(int, int me, double acc) const {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
        if ((threadIdx.x & 63) == 0) {
            const unsigned long long b = (unsigned long long)__double_as_longlong(acc);
            const unsigned long long t = (unsigned long long)tag << 32;
            atomic_st64(words + kLwSigma + 2 * me, (b & 0xffffffffull) | t);
            atomic_st64(words + kLwSigma + 2 * me + 1, (b >> 32) | t);
        }
    }
};

struct LoopLds {
    union {
        SweepLds<FwdOp, kRing> fwd;
        SweepLds<LoopBwdOp, kRing> bwd;
    };
    float dn[kLoopSteps], up[kLoopSteps];  // s' of the rows next to the strip, by step
    int2 range[kLoopMaxStrips];
    double part[kLoopWaves];
    double sig, ws, rn;
    unsigned rmax;
    int bad, active;
    __device__ LoopLds() {}
};

// Polls until `ready()` holds on every lane; false (and the error flag) on expiry.
template <class F>
__device__ __forceinline__ bool loop_wait(int* err, int site, int limit, F ready) {
    for (int spin = 0;; spin++) {
        if (__all(ready())) return true;
        if (spin >= limit || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
            raise_wait(err, site);
            return false;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}
// One wave: the sum over the simulation's strips of a double published as two
// tagged words each, `per` of them per strip (inactive strips count zero), in
// wave_sum_of's order over [strip][k].
__device__ __forceinline__ bool loop_gather(const unsigned long long* words, int S, unsigned act, int word, int per,
                                            unsigned tag, int* err, double& out) {
    const int i = threadIdx.x & 63, s = i / per;
    const bool mine = i < S * per && ((act >> s) & 1);
    const unsigned long long* p = words + (size_t)s * kLoopWords + word + 2 * (i % per);
    double v = 0;
    const bool ok = loop_wait(err, kWaitLoopWords, kSpinLimit, [&]() {
        if (!mine) return true;
        const unsigned long long a = atomic_ld64(p), b = atomic_ld64(p + 1);
        v = __longlong_as_double((long long)(((b & 0xffffffffull) << 32) | (a & 0xffffffffull)));
        return (unsigned)(a >> 32) == tag && (unsigned)(b >> 32) == tag;
    });
    v = mine ? v : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    out = v;
    return ok;
}

// The solve of one strip: s of a simulation whose matrix is factored, with r =
// rhs, p = s0 = 0 and sc initialised by the factor.
__device__ __forceinline__ void pcg_loop_strip(const LoopArgs& A, int s, LoopLds& L, int* err) {
    const SkGeom& g = A.g;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = (int)uniform((unsigned)tid >> 6);  // scalar: its group bounds then branch without masks
    const int NSG = g.T4 / kSub;
    if (tid == 0) {
        L.bad = __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        L.active = A.sc->done == 0;
        L.rmax = 0;
        L.fwd.abort_flag = 0;
    }
    if (tid < g.S) L.range[tid] = A.range ? A.range[tid] : make_int2(0, NSG);
    for (int t = tid; t < kLoopSteps; t += kLoopThreads) L.dn[t] = L.up[t] = 0.0f;
    __syncthreads();
    if (!L.active || L.bad) return;
    unsigned act = 0;  // strips with FLUID cells
    for (int k = 0; k < g.S; k++) act |= (L.range[k].x < L.range[k].y ? 1u : 0u) << k;
    act = uniform(act);
    if (!((act >> s) & 1)) return;
    const unsigned tag0 = uniform(A.sc->epoch);
    const double stop = A.sc->tol * A.sc->rhs_norm;
    unsigned long long* const mine = A.words + (size_t)s * kLoopWords;
    unsigned long long* const zrows = A.words + (size_t)g.S * kLoopWords;  // [S][4 T4]
    const unsigned long long tagw0 = (unsigned long long)tag0 << 32;
    // every strip of the simulation is resident before any waits for another
    if (wave == 0) {
        if (lane == 0) atomic_st64(mine + kLwArrive, tagw0);
        const bool m = lane < g.S && ((act >> lane) & 1);
        const bool ok = loop_wait(err, kWaitArrive, 1 << 23, [&]() {
            return !m || (unsigned)(atomic_ld64(A.words + (size_t)lane * kLoopWords + kLwArrive) >> 32) == tag0;
        });
        if (lane == 0) L.bad = !ok;
    }
    __syncthreads();
    if (L.bad) return;

    const SkCtl ctl{nullptr, nullptr, err, L.range};
    const bool below = s > 0 && ((act >> (s - 1)) & 1), above = s + 1 < g.S && ((act >> (s + 1)) & 1);
    const int lo = 4 * (int)uniform((unsigned)L.range[s].x), hi = 4 * (int)uniform((unsigned)L.range[s].y);
    const int ga = lo + (hi - lo) * wave / kLoopWaves, gb = lo + (hi - lo) * (wave + 1) / kLoopWaves;
    const int2 rd = below ? L.range[s - 1] : make_int2(0, 0), ru = above ? L.range[s + 1] : make_int2(0, 0);
    double sig_prev = 0, rn = A.sc->rhs_norm;
    int iter = 0, done = 0;
    // after an expired wait: the next solve's tags start past those in use here
    auto fail = [&](int it) {
        if (tid == 0) atomicMax(&A.sc->iter, it);
    };
    for (int it = 0;; it++) {
        const unsigned tag = tag0 + (unsigned)it;
        const unsigned long long tagw = (unsigned long long)tag << 32;
        {
            FwdOp op{{A.r, A.P, A.fx, A.fy}, nullptr, {A.q}, A.rows.set(g, false, it), A.rows.set(g, false, it + 1)};
            if (tid == 0) L.fwd.abort_flag = 0;
            // meanwhile the spare wave collects |r|_inf of the update before (:453)
            sweep_run<FwdOp, false, true, kRing, true>(op, g, ctl, s, 0, L.fwd, [&]() {
                if (it == 0) return;
                const bool m = lane < g.S && ((act >> lane) & 1);
                unsigned v = 0;
                const bool ok = loop_wait(err, kWaitLoopWords, kSpinLimit, [&]() {
                    if (!m) return true;
                    const unsigned long long a = atomic_ld64(A.words + (size_t)lane * kLoopWords + kLwRmax);
                    v = (unsigned)a;
                    return (unsigned)(a >> 32) == tag - 1u;
                });
                double x = m ? (double)u2f(v) : 0.0;
#pragma unroll
                for (int o = 32; o > 0; o >>= 1) {
                    const double y = __shfl_xor(x, o, 64);
                    x = y > x ? y : x;
                }
                if (lane == 0) {
                    L.rn = x;
                    if (!ok) L.bad = 1;
                }
            });
        }
        __syncthreads();
        if (L.bad || L.fwd.abort_flag) return fail(it);
        if (it > 0) {
            rn = L.rn;
            if (rn <= stop) {
                done = 1;
                break;
            }
        }
        __syncthreads();  // the flags are read: the backward solve may set its LDS up
        {
            LoopBwdOp op;
            op.in[0] = A.q;
            op.in[1] = A.P;
            op.in[2] = A.G;
            op.bytes = nullptr;
            op.out[0] = A.z;
            op.row = A.rows.set(g, true, it);
            op.row_next = A.rows.set(g, true, it + 1);
            op.words = mine;
            op.tag = tag;
            if (tid == 0) L.bwd.abort_flag = 0;
            sweep_run<LoopBwdOp, true, true, kRing, true>(op, g, ctl, s, 0, L.bwd);
        }
        __syncthreads();
        if (L.bwd.abort_flag) return fail(it);
        iter = it;
        if (it >= A.max_iters) break;

        const StripArr Ad(A.Adiag, g, s), Z(A.z, g, s), So((it & 1) ? A.s1 : A.s0, g, s),
            Sn((it & 1) ? A.s0 : A.s1, g, s), Wv(A.w, g, s), Rr(A.r, g, s), Pv(A.p, g, s);
        // wave 0: sigma of all strips; waves 1-4: z of the rows next to the
        // strip, by step: lane 0 at step t is column t (step t + 63 of the strip
        // below's last row), lane 63 column t - 63 (that step of the strip
        // above's first row, which the backward solve has waited for in every
        // column of the grid); waves 5-7: z of the last row for the strip above
        constexpr int kPer = (kLoopSteps + 255) / 256;
        float zd[kPer], zu[kPer];
        if (wave == 0) {
            double sig;
            if (!loop_gather(A.words, g.S, act, kLwSigma, kLoaders, tag, err, sig)) L.bad = 1;
            if (lane == 0) L.sig = sig;
        } else if (wave <= 4) {
            unsigned long long v[kPer];
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const int t = 4 * lo + tid - 64 + k * 256, tu = t - 63;
                zu[k] = 0.0f;
                if (t < 4 * hi && tu >= 16 * ru.x && tu < 16 * ru.y && tu < g.nx)
                    zu[k] = u2f(__hip_atomic_load(A.rows.set(g, true, it) + (size_t)(s + 1) * 4 * g.T4 + tu,
                                                  __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                v[k] = 0;
            }
            const bool ok = loop_wait(err, kWaitLoopRow, kSpinLimit, [&]() {
                bool all = true;
#pragma unroll
                for (int k = 0; k < kPer; k++) {
                    const int t = 4 * lo + tid - 64 + k * 256, td = t + 63;
                    if (t < 4 * hi && td >= 16 * rd.x && td < 16 * rd.y) {
                        v[k] = atomic_ld64(zrows + (size_t)(s - 1) * 4 * g.T4 + td);
                        all = all && (unsigned)(v[k] >> 32) == tag;
                    }
                }
                return all;
            });
            if (!ok) L.bad = 1;
#pragma unroll
            for (int k = 0; k < kPer; k++) zd[k] = u2f((unsigned)v[k]);
        } else if (above) {
            for (int t = 4 * lo + tid - 320; t < 4 * hi; t += kLoopThreads - 320) {
                const float v = A.z[(((long)s * g.T4 + (t >> 2)) * 64 + 63) * 4 + (t & 3)];
                atomic_st64(zrows + (size_t)s * 4 * g.T4 + t, (unsigned long long)f2u(v) | tagw);
            }
        }
        __syncthreads();
        if (L.bad) return fail(it);
        const double sig = L.sig;
        const float beta = it > 0 ? (float)(sig / sig_prev) : 0.0f;
        sig_prev = sig;
        if (wave >= 1 && wave <= 4)
#pragma unroll
            for (int k = 0; k < kPer; k++) {
                const int t = 4 * lo + tid - 64 + k * 256;
                if (t < 4 * hi) {
                    L.dn[t] = fmaf(beta, L.dn[t], zd[k]);
                    L.up[t] = fmaf(beta, L.up[t], zu[k]);
                }
            }
        __syncthreads();
        const double acc = spmv_strip(lo, hi, ga, gb, Ad, Z, So, Sn, Wv, beta, L.dn, L.up);
        const double ws_s = loop_block_sum(acc, L.part);
        if (wave == 0) {
            if (lane == 0) {
                const unsigned long long b = (unsigned long long)__double_as_longlong(ws_s);
                atomic_st64(mine + kLwWs, (b & 0xffffffffull) | tagw);
                atomic_st64(mine + kLwWs + 1, (b >> 32) | tagw);
                L.rmax = 0;
            }
            double ws;
            if (!loop_gather(A.words, g.S, act, kLwWs, 1, tag, err, ws)) L.bad = 1;
            if (lane == 0) L.ws = ws;
        }
        __syncthreads();
        if (L.bad) return fail(it);
        // alpha = sigma / w.s' (:450); p += alpha s', r -= alpha w (:451-452)
        const float alpha = (float)(sig / L.ws);
        float m = 0.0f;
        for (int g0 = ga; g0 < gb; g0 += kLoopPU) {
            float4 wv[kLoopPU], rr[kLoopPU], sv[kLoopPU], pv[kLoopPU];
#pragma unroll
            for (int u = 0; u < kLoopPU; u++) {
                const int k = min(g0 + u, gb - 1);
                wv[u] = Wv.ld(k);
                rr[u] = Rr.ld(k);
                sv[u] = Sn.ld(k);
                pv[u] = Pv.ld(k);
            }
#pragma unroll
            for (int u = 0; u < kLoopPU; u++)
                if (g0 + u < gb) {
                    m = r_update(Rr, g0 + u, alpha, wv[u], rr[u], m);
                    Pv.st(g0 + u, s_next(alpha, sv[u], pv[u]));
                }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
        if (lane == 0) atomicMax(&L.rmax, f2u(m));  // m >= 0: its bits order as it does
        // this wave's s', w and r stores are done before other waves read them
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
        asm volatile("" ::: "memory");
        __syncthreads();
        if (tid == 0) atomic_st64(mine + kLwRmax, (unsigned long long)L.rmax | tagw);
    }
    // done: the stopping test of iteration iter (the update before) passed;
    // otherwise max_iters iterations ran
    if (tid == 0 && (act & ((1u << s) - 1)) == 0) {
        A.sc->sigma = sig_prev;
        A.sc->r_norm = rn;
        A.sc->iter = iter;
        A.sc->done = done;
    }
}

__global__ __launch_bounds__(kLoopThreads) void pcg_loop_kernel(LoopArgs A, int* err) {
    __shared__ __align__(16) LoopLds L;
    pcg_loop_strip(A, blockIdx.x, L, err);
}

}  // namespace fs2d
