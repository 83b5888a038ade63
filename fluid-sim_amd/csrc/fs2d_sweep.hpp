// fs2d_sweep.hpp -- warp-specialised wavefront passes: the pressure solve's
// recurrences and the level set's Gauss-Seidel sweeps.
//
// The MIC(0) factor and both triangular solves of applyPreconditioner
// (src/FluidSim2D.cpp:364-421) are lexicographic recurrences: cell (i, j)
// needs (i-1, j) and (i, j-1) (forward) or (i+1, j) and (i, j+1) (backward).
// So are the closest-particle and eikonal sweeps of the level set
// (src/FluidSim2D.cpp:775-792, 845-902), each a forward sweep in coordinates
// mirrored by its direction.
//
// One workgroup owns a strip of 64 rows j = 64 s + l.  Its compute wave holds
// row l in lane l and at step t processes column i = t - l: the row neighbour
// is the lane's own previous result, the column neighbour is lane l-1's
// previous result moved by one DPP wave_shr:1 (wave_shl:1 backward), and the
// strip's edge lane receives the neighbouring strip's boundary row through the
// DPP `old` operand.
//
// A solve step is one DPP and two FMAs.  A lone wave issues about one
// instruction per 4 clocks whatever its type, so the compute wave does nothing
// else it can hand to another wave:
//   wave 0          compute: supergroups of 16 steps; the LDS reads of the
//                   next supergroup are issued while the current one computes
//                   (two register buffers, no copies); readiness flags are read
//                   one supergroup ahead; one dwordx4 store per output array
//                   and 4 steps; no global loads and no waits on them.
//   waves 1..L      loaders: stream the strip's inputs (SK4 layout, 1 KB per
//                   wave-wide dwordx4 load), apply the operator's per-cell
//                   transform (e.g. P*r) and fill an LDS ring of supergroups.
//   waves L+1, L+2  pollers: read the neighbouring strip's boundary row into an
//                   LDS ring indexed by step: the solves' from untagged words
//                   that hold kUnset until written (HandRows), the other
//                   passes' from tagged words ({payload, epoch}), both with
//                   agent-scope relaxed atomics (fs2d_gmem.hpp); steps whose
//                   edge column is outside the grid get the boundary value.
// The solves' producing lane stores its row with the buffer stores of the step
// (other lanes' offsets are out of range).  In the other passes its 16 boundary
// values per supergroup go through a 2-entry LDS outbox and are stored as
// tagged words by 16 lanes after the first sub-group of the next supergroup,
// into a padded row (no range tests).
//
// Waves signal each other through LDS counters without s_waitcnt: LDS executes
// one wave's operations in order, so a flag written after data (or after the
// reads that free a slot) is seen only after them; compiler barriers keep the
// accesses on their side of the flag.
//
// Strips are taken from a 64-bit ticket (strip = ticket mod S, launch =
// ticket / S, epoch = launch + 1): a strip only ever waits on a strip owned by
// a workgroup that started earlier, and no reset is needed between launches.
// Every wait is bounded; on expiry the workgroup raises the error flag and all
// its waves run to completion.
//
// SK4 layout: element (s, t, l) at ((s * T4 + t/4) * 64 + l) * 4 + t%4 (float
// arrays; byte arrays use the same element index), T4 a multiple of 8 (an even
// number of supergroups) with 4 T4 >= nx + 64.  Padding entries hold zero
// coefficients, so every lane computes every step.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fs2d_gmem.hpp"

namespace fs2d {

struct SkGeom {
    int nx, ny, S, T4;  // S strips of 64 rows, T4 groups of 4 steps per strip
    __host__ __device__ long size() const { return (long)S * T4 * 256; }
    __host__ __device__ long idx(int i, int j) const {
        const int s = j >> 6, l = j & 63, t = i + l;
        return (((long)s * T4 + (t >> 2)) * 64 + l) * 4 + (t & 3);
    }
};

__host__ inline SkGeom make_geom(int nx, int ny) {
    SkGeom g;
    g.nx = nx;
    g.ny = ny;
    g.S = (ny + 63) / 64;
    g.T4 = (nx + 64 + 31) / 32 * 8;
    return g;
}

// Boundary rows of the solves' strips.  Entry [4 T4 s + t] is strip s's edge
// lane at step t, one word without a tag: a row is kUnset (a signalling NaN,
// which no arithmetic result can be) until its pass writes it, four steps per
// store.  A solve's passes alternate between two sets of rows; each pass
// resets the set that the pass before it used, and the first one's is set by
// pcg_init_kernel.  Tagged words cost the compute wave four LDS writes (28
// clocks each), an LDS read and a store per 16 steps, and reach the next strip
// 16 to 20 steps after the first of them is known; rows cost four stores (13
// clocks) and leave with each group of four.
constexpr uint32_t kUnset = 0x7f9abcdeu;
struct HandRows {
    uint32_t* base;  // forward passes 0, 1, backward passes 0, 1: S * 4 T4 words each
    __host__ __device__ static size_t words(const SkGeom& g) { return 4 * (size_t)g.S * g.T4 * 4; }
    __host__ __device__ uint32_t* set(const SkGeom& g, bool backward, int pass) const {
        return base + (size_t)(2 * (backward ? 1 : 0) + (pass & 1)) * g.S * g.T4 * 4;
    }
};

struct SkCtl {
    unsigned long long* ticket;
    unsigned long long* handoff;  // per strip: [kHandPadLo + nx + kHandPadHi][NW] tagged words + 64 scratch words
    int* err;
    const int2* range = nullptr;  // per strip: its active supergroups (strip_span); nullptr: all of them
};
// A strip's hand-off row holds columns -kHandPadLo .. nx + kHandPadHi - 1:
// every column a producing lane can name (-79 .. nx + 110, since 4 T4 <=
// nx + 95), so the stores need no range test; only columns 0 .. nx-1 are read.
constexpr int kHandPadLo = 80, kHandPadHi = 112;
__host__ __device__ inline size_t sk_hand_cols(int nx) { return (size_t)nx + kHandPadLo + kHandPadHi; }
__host__ __device__ inline size_t sk_handoff_stride(int nx, int nw) { return sk_hand_cols(nx) * nw + 64; }

// Coupling bits of a FLUID cell: the off-diagonal entries of row (i, j) are
// -scaleA towards each coupled neighbour (FluidSim2D.cpp:266-301).
enum : uint32_t { CPL_L = 1, CPL_R = 2, CPL_D = 4, CPL_U = 8 };

constexpr int kSub = 4;         // SK4 groups per supergroup (16 steps)
constexpr int kLoaders = 4;       // with 3 the first strip waits for its loaders (13 of 132 supergroups at 2048^2), with 5 nothing changes
constexpr int kRing = 8;        // supergroups in the LDS ring of a single launch (a power of two)
constexpr int kHandRing = 256;  // steps in the hand-off ring
constexpr int kPollers = 2;     // poller waves: their polls interleave in time
constexpr int kSweepThreads = 64 * (1 + kLoaders + kPollers);  // at least 64 + kMaxStrips (sweep_ticket)
constexpr int kLdsSpin = 1 << 26;  // bounded LDS waits (~seconds)
// A ring of kLoaders + 2 supergroups lets every loader keep its loads in
// flight.  A smaller ring (batched launches, where more workgroups per CU
// matter more) only makes loaders wait for free slots: a loader waits for the
// consumption of supergroups below its own, which other loaders fill without
// waiting on it, so any power of two >= 2 is deadlock-free.
static_assert(kRing >= kLoaders + 2, "ring too small for the loaders");

__device__ __forceinline__ float f4get(const float4& v, int q) {
    return q == 0 ? v.x : (q == 1 ? v.y : (q == 2 ? v.z : v.w));
}
__device__ __forceinline__ uint32_t u4get(const uint4& v, int q) {
    return q == 0 ? v.x : (q == 1 ? v.y : (q == 2 ? v.z : v.w));
}

__device__ __forceinline__ unsigned lds_ld(unsigned* p) {
    unsigned v = __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    asm volatile("" ::: "memory");
    return v;
}
__device__ __forceinline__ void lds_st(unsigned* p, unsigned v) {
    asm volatile("" ::: "memory");
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void lds_max(unsigned* p, unsigned v) {
    asm volatile("" ::: "memory");
    __hip_atomic_fetch_max(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ unsigned uniform(unsigned v) { return (unsigned)__builtin_amdgcn_readfirstlane((int)v); }

// Neighbour-row value: lane l-1's (forward) or lane l+1's (backward) register.
// The edge lane gets `edge` (C: a strip upstream) or zero (no strip upstream;
// every operator's boundary state is zero).
template <bool B, bool C>
__device__ __forceinline__ uint32_t nbr(uint32_t edge, uint32_t v) {
    constexpr int ctl = B ? 0x130 /* wave_shl:1 */ : 0x138 /* wave_shr:1 */;
    if (C) return (uint32_t)__builtin_amdgcn_update_dpp((int)edge, (int)v, ctl, 0xf, 0xf, false);
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, ctl, 0xf, 0xf, true);
}

// Operators whose outputs other workgroups read within the same launch
// declare kOutThrough: their stores then carry device scope (SC1), so each is
// written through to memory, and a completion flag needs only those stores'
// own completion (vmcnt) before it, not a write-back of the whole L2.
template <class Op>
constexpr auto out_through_(int) -> decltype(Op::kOutThrough) {
    return Op::kOutThrough;
}
template <class Op>
constexpr bool out_through_(long) {
    return false;
}
template <class Op>
constexpr bool out_through() {
    return out_through_<Op>(0);
}
// Operators whose inputs other workgroups of the same launch produce declare
// kWaitInputs and wait_inputs(s, err): each loader wave calls it before its
// first load of strip s.
template <class Op>
constexpr auto wait_inputs_(int) -> decltype(Op::kWaitInputs) {
    return Op::kWaitInputs;
}
template <class Op>
constexpr bool wait_inputs_(long) {
    return false;
}
template <class Op>
constexpr bool waits_inputs() {
    return wait_inputs_<Op>(0);
}
// Operators of one state word whose boundary values travel through untagged
// rows declare kRow and hold row / row_next (HandRows).
template <class Op>
constexpr auto row_(int) -> decltype(Op::kRow) {
    return Op::kRow;
}
template <class Op>
constexpr bool row_(long) {
    return false;
}
constexpr int kBufferCfg = 0x00020000;  // raw buffer resource word 3 of gfx9-family targets
constexpr int kCpolSc1 = 16;            // cache policy operand: SC1 (device scope)
constexpr unsigned kWaitVm0 = 0x0F70u;  // s_waitcnt vmcnt(0), gfx9 encoding

// What one strip of a pass does, in processing order (supergroup sg of a
// backward pass is supergroup NSG - 1 - sg of the array).  A pressure solve
// runs only the strip's active supergroups, [range.x, range.y) of the array
// (even bounds, tile_act): outside them there is no FLUID cell, so every
// coefficient and every result is zero.  A neighbour's boundary row is read
// where the neighbour is active and zero elsewhere.  On the 512^2 dam break
// (a block of 0.4 x 0.6 of the box) a solve's chain of dependent steps halves.
struct StripSpan {
    int s, lo, hi;         // strip; supergroups lo .. hi-1, processing order (lo, hi even)
    int up_lo, up_hi;      // the upstream strip's active steps (array order)
    bool consume, produce; // an active strip upstream / downstream
};
template <bool BACKWARD>
__device__ __forceinline__ StripSpan strip_span(const SkGeom& g, const int2* range, int s) {
    const int NSG = g.T4 / 4;
    // in scalar registers: the compiler does not know that a range read from
    // LDS is uniform, and bounds in vector registers turn the compute wave's
    // loop into a divergent one (4% per iteration at 1000 x 700)
    auto rng = [&](int k) {
        if (k < 0 || k >= g.S) return make_int2(0, 0);
        if (!range) return make_int2(0, NSG);
        const int2 r = range[k];
        return make_int2((int)uniform((unsigned)r.x), (int)uniform((unsigned)r.y));
    };
    const int2 own = rng(s), up = rng(BACKWARD ? s + 1 : s - 1), down = rng(BACKWARD ? s - 1 : s + 1);
    return {s, BACKWARD ? NSG - own.y : own.x, BACKWARD ? NSG - own.x : own.y, 16 * up.x, 16 * up.y, up.x < up.y,
            down.x < down.y};
}

template <class Op, int RING = kRing>
struct SweepLds {
    static_assert(RING >= 2 && (RING & (RING - 1)) == 0, "ring slots are taken modulo RING");
    float4 ring_f[RING][kSub][Op::NF][64];
    uint32_t ring_b[Op::NB ? RING : 1][kSub][64];
    uint32_t hand[Op::NW][kHandRing];
    uint32_t outbox[2][Op::NW][16];
    uint32_t unread[64 * 4 + 2 * Op::NW * 16];  // where the lanes that produce nothing write (sweep_compute)
    unsigned slot_tag[RING];
    unsigned consumed_sg, hand_ready, abort_flag;
};

// Op interface:
//   NW    32-bit words of carried state; NIN float input arrays in[]; NF float
//         arrays in the ring; NB (0/1) byte input array `bytes`; NOUT float
//         output arrays out[]
//   bool skip(bool first)      wave 0 only; first: strip order 0
//   void xform(const float4 (&in)[NIN], float4 (&x)[NF], double& acc, int t, int s)
//         loader: ring values of one SK4 group from its inputs; t and s as
//         for group()
//   void loader_done(int s, int loader, double acc)
//   template <bool B, bool C, class H> void group(const float4 (&x)[NF], uint32_t b4,
//        uint32_t (&st)[NW], const uint4 (&hb)[NW], float (&o)[NOUT][4],
//        uint32_t (&prod)[NW][4], int t, int s, H hook)
//         4 steps; step q uses component q of x[a], byte q of b4 and, on the
//         edge lane of a consuming strip, component q of hb[w]; st is the
//         lane's state after the previous step, updated; o[n][q] output n;
//         prod[w][q] state word w after step q; t is the group's first step
//         and s the strip, so step q of lane l is cell (t + q - l, 64 s + l)
//   kRow (optional, true; NW = 1 and out[0] is the state): boundary values
//         through the rows row / row_next (HandRows), and group calls hook(i) in
//         its i-th step, between the step's row term and its lane shift: there
//         the next supergroup's LDS reads go out one or two at a time, in the
//         wait states the shift needs anyway
//   void strip_done(int s)     wave 0, after the last step (also of a strip with an empty span)
template <class Op, bool B, bool C, bool P, int RING>
__device__ __forceinline__ void sweep_compute(Op& op, const SkGeom& g, SweepLds<Op, RING>& L, const StripSpan& sp,
                                              unsigned epoch, unsigned long long* dst, int* err) {
    constexpr int NW = Op::NW, NF = Op::NF, NB = Op::NB, NOUT = Op::NOUT;
    const int lane = threadIdx.x & 63;
    const int s = sp.s, nx = g.nx;
    const int T = g.T4 * 4;
    const int prod_lane = B ? 0 : 63;
    const long strip_base = (long)s * g.T4 * 256;
    constexpr bool THROUGH = out_through<Op>(), ROW = row_<Op>(0);
    __amdgpu_buffer_rsrc_t out_rs[NOUT];
    if (THROUGH)
#pragma unroll
        for (int n = 0; n < NOUT; n++)
            out_rs[n] = __builtin_amdgcn_make_buffer_rsrc(op.out[n], 0, (int)(g.size() * 4), kBufferCfg);

    // the edge lane's row stores: every other lane's offset is out of range, so
    // the hardware drops its part (no exec mask, no branch)
    __amdgpu_buffer_rsrc_t row_rs;
    int row_off = 0;
    if constexpr (ROW) {
        row_rs = __builtin_amdgcn_make_buffer_rsrc(op.row + (size_t)s * T, 0, T * 4, kBufferCfg);
        row_off = (lane == prod_lane ? 0 : 0x40000000) + 4 * (B ? T - 16 * (sp.lo + 1) : 16 * sp.lo);
    }
    // Byte offsets of the buffer stores, advanced by a supergroup at a time: in
    // registers, not in the instruction's scalar offset.  A 16-byte buffer store
    // with a scalar offset still reads its data while the next instruction
    // executes, and where that one overwrites the data, lanes 28-31 stored the
    // new value (seen on gfx950; the compiler places the wait states only for
    // stores without one).
    int out_off = (int)((strip_base + (B ? T - 16 * (sp.lo + 1) : 16 * sp.lo) * 64L + lane * 4) * 4);
    constexpr int kOutInc = B ? -4096 : 4096, kRowInc = B ? -64 : 64;

    struct Buf {
        float4 x[kSub][NF];
        uint32_t b[kSub];
        uint4 h[kSub][NW];
    };
    // first step of supergroup sg (processing order)
    auto sg_t0 = [&](int sg) { return B ? T - 16 * (sg + 1) : 16 * sg; };
    // x data of a supergroup is in the ring (loaders); hand values of its
    // steps are in the hand ring (poller)
    auto x_ready = [&](int sg, unsigned tag) { return tag == (unsigned)sg + 1u; };
    auto h_ready = [&](int sg, unsigned hr) { return hr >= 16u * (unsigned)(sg + 1); };
    // LDS bases in a VGPR (mbcnt_lo(0, 0) is 0 in every lane but not known to
    // be uniform), so that the hand ring's and tags' constant offsets fold
    // into the ds_read offset fields instead of one address move per read
    const unsigned zero_v = __builtin_amdgcn_mbcnt_lo(0u, 0u);
    const uint32_t* const hand_v = &L.hand[0][0] + zero_v;
    unsigned* const tag_v = &L.slot_tag[0] + zero_v;
    // The LDS reads of a supergroup, numbered in the order the steps need
    // them: per sub-group its hand words (C; a supergroup's 16 steps sit at
    // (t0 & 255) .. +15 of the hand ring, no wrap), then its ring words.
    constexpr int kHandReads = C ? NW : 0;
    constexpr int kPerSub = kHandReads + NF + NB;
    constexpr int kReads = kSub * kPerSub;
    auto fetch = [&](int sg, Buf& f, int first, int last) {
        const int slot = sg & (RING - 1), h0 = sg_t0(sg) & (kHandRing - 1);
#pragma unroll
        for (int n = 0; n < kReads; n++) {
            if (n < first || n >= last) continue;
            const int j = B ? kSub - 1 - n / kPerSub : n / kPerSub, a = n % kPerSub;
            if (a < kHandReads) f.h[j][a] = *(const uint4*)(hand_v + a * kHandRing + h0 + 4 * j);
            else if (a < kHandReads + NF) f.x[j][a - kHandReads] = L.ring_f[slot][j][a - kHandReads][lane];
            else f.b[j] = L.ring_b[NB ? slot : 0][j][lane];
        }
    };
    auto fetch_all = [&](int sg, Buf& f) { fetch(sg, f, 0, kReads); };
    bool bad = false;
    auto give_up = [&](int spin) {
        if (spin >= kLdsSpin || lds_ld(&L.abort_flag)) {
            bad = true;
            raise_wait(err, kWaitCompute);
            atomicExch(&L.abort_flag, 1u);
        }
        __builtin_amdgcn_s_sleep(0);
    };
    auto wait_x = [&](int sg) {
        for (int spin = 0; !bad && !x_ready(sg, uniform(lds_ld(&L.slot_tag[sg & (RING - 1)]))); spin++) give_up(spin);
    };
    auto wait_h = [&](int sg) {
        for (int spin = 0; !bad && !h_ready(sg, uniform(lds_ld(&L.hand_ready))); spin++) give_up(spin);
    };

    uint32_t st[NW];
#pragma unroll
    for (int w = 0; w < NW; w++) st[w] = 0u;
    // Hand-off stores: at supergroup sg, lane 16 w + q stores word w of step q
    // of supergroup sg-1 (at the first one columns where this strip is not
    // active, never read).
    // Each such lane walks 16 columns per supergroup through the padded row;
    // lanes past 16 NW keep one scratch word each.  No per-supergroup address
    // arithmetic, no range test.
    const bool hreal = lane < 16 * NW;
    const int hcol0 = sg_t0(sp.lo - 1) + (lane & 15) - prod_lane;
    unsigned long long* hp = hreal ? dst + (size_t)(hcol0 + kHandPadLo) * NW + (lane >> 4)
                                   : dst + sk_hand_cols(nx) * NW + lane;
    const long hinc = hreal ? (B ? -16L : 16L) * NW : 0L;

    // One supergroup: compute `cur` while the LDS reads of the next one go
    // into `nxt` speculatively: the readiness flags are read just before the
    // data (LDS executes a wave's operations in order), and checked after
    // the compute; only a failed check branches (wait, then read again).  The
    // prefetch index is clamped, so the last supergroup re-reads its own slot
    // and every iteration has the same shape.
    // LDS order per supergroup: an explicit wait at the top for all but the
    // last sub-group's outbox and consumed_sg writes (the data of `cur` arrived
    // before, so it costs nothing); the outbox read and the first sub-group;
    // the readiness flags; then the reads of the next supergroup: in one burst,
    // or (kRow) over the second and third sub-groups, one or two per step in
    // the wait states that the lane shifts need (a read costs the wave 11
    // clocks, 6 of them hidden there).  Every lane writes (those that do not
    // produce to `unread`): behind an exec-mask branch the compiler cannot
    // count the writes, and waited at the top of each supergroup for those
    // just issued.
    // s_waitcnt immediates (gfx9 encoding: lgkmcnt in bits 8-11, vmcnt and
    // expcnt at their maxima): lgkmcnt(young writes) and lgkmcnt(0)
    constexpr unsigned kYoung = P && !ROW ? NW + 1 : 1;
    static_assert(kYoung <= 15, "outbox writes exceed lgkmcnt's range");
    constexpr unsigned kWaitOld = 0xC07Fu | (kYoung << 8);
    constexpr unsigned kWaitAll = 0xC07Fu;
    const bool is_prod = lane == prod_lane;
    uint32_t* const out_v = is_prod ? &L.outbox[0][0][0] : &L.unread[lane * 4];
    unsigned* const done_v = is_prod ? &L.consumed_sg : &L.unread[lane * 4];
    const uint32_t* const box_v = &L.outbox[0][min(lane >> 4, NW - 1)][lane & 15];
    // PAR: sg & 1 (lo is even)
    auto step = [&](auto par, int sg, Buf& cur, Buf& nxt) {
        constexpr int PAR = decltype(par)::value;
        const int t0 = sg_t0(sg);
        const int sn = min(sg + 1, sp.hi - 1);
        __builtin_amdgcn_s_waitcnt(kWaitOld);
        uint32_t ob = 0;
        if (P && !ROW) ob = box_v[(PAR ^ 1) * NW * 16];
        __builtin_amdgcn_sched_barrier(0);
        unsigned tagv = 0, hrv = 0;
#pragma unroll
        for (int k = 0; k < kSub; k++) {
            const int j = B ? kSub - 1 - k : k;
            float o[NOUT][4];
            uint32_t prod[NW][4];
            op.template group<B, C>(cur.x[j], cur.b[j], st, cur.h[j], o, prod, t0 + 4 * j, s, [&](int i) {
                if (ROW && (k == 1 || k == 2)) {
                    const int n = 4 * (k - 1) + i;
                    __builtin_amdgcn_sched_barrier(0);
                    fetch(sn, nxt, n * kReads / 8, (n + 1) * kReads / 8);
                    __builtin_amdgcn_sched_barrier(0);
                }
            });
#pragma unroll
            for (int n = 0; n < NOUT; n++) {
                if (THROUGH) {
                    typedef float f4 __attribute__((ext_vector_type(4)));
                    const f4 v = {o[n][0], o[n][1], o[n][2], o[n][3]};
                    __builtin_amdgcn_raw_buffer_store_b128(v, out_rs[n], out_off + j * 1024, 0, kCpolSc1);
                } else {
                    float* base = op.out[n] + strip_base + (long)t0 * 64;  // uniform
                    *(float4*)(base + j * 256 + lane * 4) = make_float4(o[n][0], o[n][1], o[n][2], o[n][3]);
                }
            }
            if constexpr (ROW) {
                if (P) {
                    typedef float f4 __attribute__((ext_vector_type(4)));
                    const f4 v = {o[0][0], o[0][1], o[0][2], o[0][3]};
                    __builtin_amdgcn_raw_buffer_store_b128(v, row_rs, row_off + 16 * j, 0, kCpolSc1);
                }
            } else if (P)
#pragma unroll
                for (int w = 0; w < NW; w++)
                    *(uint4*)(out_v + (PAR * NW + w) * 16 + 4 * j) =
                        make_uint4(prod[w][0], prod[w][1], prod[w][2], prod[w][3]);
            if (k == 0) {
                // the previous supergroup's boundary values leave once the
                // outbox read has had a sub-group's time to return
                if (P && !ROW) {
                    atomic_st64(hp, (unsigned long long)ob | ((unsigned long long)epoch << 32));
                    hp += hinc;
                }
                __builtin_amdgcn_sched_barrier(0);
                tagv = lds_ld(tag_v + (sn & (RING - 1)));
                if (C) hrv = lds_ld(&L.hand_ready);
                if (!ROW) fetch_all(sn, nxt);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        if (THROUGH) out_off += kOutInc;
        if (ROW && P) row_off += kRowInc;
        lds_st(done_v, (unsigned)sg + 1u);
        const unsigned sn1 = (unsigned)sn + 1u;
        const unsigned tv = uniform(tagv), hv = C ? uniform(hrv) : 0u;
        // nonzero unless the slot holds supergroup sn and its hand values are in
        // (hand_ready < 2^31, so the difference's sign bit is hv < 16 sn1)
        if ((tv ^ sn1) | (C ? (hv - 16u * sn1) >> 31 : 0u)) {
            if (tv != sn1) wait_x(sn);
            if (C && hv < 16u * sn1) wait_h(sn);
            fetch_all(sn, nxt);
            __builtin_amdgcn_s_waitcnt(kWaitAll);  // re-read data in registers, as on the fast path
        }
    };

    Buf b0, b1;
    wait_x(sp.lo);
    if (C) wait_h(sp.lo);
    fetch_all(sp.lo, b0);
    __builtin_amdgcn_s_waitcnt(kWaitAll);  // the first supergroup's data in registers
    for (int sg = sp.lo; sg < sp.hi; sg += 2) {  // an even number of supergroups
        step(std::integral_constant<int, 0>{}, sg, b0, b1);
        step(std::integral_constant<int, 1>{}, sg + 1, b1, b0);
    }
    if (P && !ROW && hreal) {
        const uint32_t ob = box_v[NW * 16];  // sp.hi - 1 is odd
        atomic_st64(hp, (unsigned long long)ob | ((unsigned long long)epoch << 32));
    }
    op.strip_done(s);
}

// Workgroup prologue: take a ticket and clear the LDS counters.  A single
// simulation's ranges are copied to LDS (`range` then points there) by other
// waves than the ticket's, beside its atomic: in one wave, or after it, they
// would put another memory round trip before every launch's first loads.
constexpr int kMaxStrips = 256;  // 16384 rows
template <class Op, int RING>
__device__ __forceinline__ unsigned long long sweep_ticket(SweepLds<Op, RING>& L, unsigned long long* ticket,
                                                           const int2*& range, int S) {
    __shared__ unsigned long long sh_ticket;
    __shared__ int2 sh_range[kMaxStrips];
    if (range) {
        const int k = (int)threadIdx.x - 64;
        if (k >= 0 && k < S) sh_range[k] = range[k];
        range = sh_range;
    }
    if (threadIdx.x == 0) {
        sh_ticket = atomicAdd(ticket, 1ull);
        L.consumed_sg = 0;
        L.hand_ready = 0;
        L.abort_flag = 0;
    }
    if (threadIdx.x < RING) L.slot_tag[threadIdx.x] = 0;
    __syncthreads();
    return sh_ticket;
}

// One strip of a pass: `order` is the strip's position in the pass (strip
// order for forward passes, reversed for backward ones), `epoch` tags its
// hand-off words.
// LOOP: one pass of many by a workgroup that keeps its strip (`order` is the
// strip, fs2d_pcg_loop.hpp): no stopping test, the LDS counters are set here,
// and the wave past the pollers calls spare() meanwhile.  The caller has a
// barrier before and after.
struct NoSpare {
    __device__ void operator()() const {}
};
template <class Op, bool BACKWARD, bool PREFETCH, int RING, bool LOOP = false, class Spare = NoSpare>
__device__ __forceinline__ void sweep_run(Op& op, const SkGeom& g, const SkCtl& c, int order, unsigned epoch,
                                          SweepLds<Op, RING>& L, Spare spare = Spare{}) {
    constexpr int NW = Op::NW, NIN = Op::NIN, NF = Op::NF, NB = Op::NB;
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
    __shared__ int sh_skip;
    const int s = BACKWARD && !LOOP ? g.S - 1 - order : order;
    const StripSpan sp = strip_span<BACKWARD>(g, c.range, s);
    const int T = g.T4 * 4, nx = g.nx;

    // A loader's supergroup: all loads in flight together; indices past the
    // span are clamped, so every register index stays a constant.
    const long strip_base = (long)s * g.T4 * 256 + lane * 4;
    float4 v[kSub][NIN];
    uint32_t vb[kSub];
    auto load_sg = [&](int sg) {
        const int sc = max(0, min(sg, sp.hi - 1));
        const int t0 = BACKWARD ? T - 16 * (sc + 1) : 16 * sc;
#pragma unroll
        for (int j = 0; j < kSub; j++) {
            const long e = strip_base + (long)(t0 + 4 * j) * 64;
#pragma unroll
            for (int a = 0; a < NIN; a++) v[j][a] = *(const float4*)(op.in[a] + e);
            vb[j] = NB ? *(const uint32_t*)(op.bytes + e) : 0u;
        }
    };
    // Loader m takes the span's supergroups sg with sg mod kLoaders = m (not
    // counted from the span's start, so a q.q partial's terms, and bits, do
    // not depend on how far the zeros outside the span are skipped).
    const int me = wave - 1;
    const int sg0 = sp.lo + (me + kLoaders - sp.lo % kLoaders) % kLoaders;
    // With PREFETCH a loader's first loads go out before the skip test,
    // whose reads they overlap (loads only: a skipped pass discards them).
    if (wave >= 1 && wave <= kLoaders && sp.lo < sp.hi) {
        if constexpr (waits_inputs<Op>()) op.wait_inputs(s, c.err);
        if (PREFETCH) load_sg(sg0);
    }
    if (LOOP) {
        if (threadIdx.x == 0) {
            L.consumed_sg = (unsigned)sp.lo;
            L.hand_ready = 0;
        }
        if (threadIdx.x < RING) L.slot_tag[threadIdx.x] = 0;
    } else if (wave == 0) {
        int sk = __hip_atomic_load(c.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0;
        if (!sk) sk = op.skip(order == 0);
        if (lane == 0) {
            sh_skip = sk;
            L.consumed_sg = (unsigned)sp.lo;
        }
    }
    __syncthreads();
    if (!LOOP && sh_skip) return;
    if (sp.lo >= sp.hi) {  // nothing in this strip
        if (wave == 0) op.strip_done(s);
        else if (wave <= kLoaders) op.loader_done(s, me, 0.0);
        return;
    }

    const int edge_lane = BACKWARD ? 63 : 0;
    auto raise = [&](int site) {
        raise_wait(c.err, site);
        atomicExch(&L.abort_flag, 1u);
    };

    // the rows of the pass before this one are free: reset them for the next
    if constexpr (row_<Op>(0)) {
        if (wave == kLoaders + 2 && sp.produce) {
            typedef uint32_t u4 __attribute__((ext_vector_type(4)));
            const __amdgpu_buffer_rsrc_t rs =
                __builtin_amdgcn_make_buffer_rsrc(op.row_next + (size_t)s * T, 0, T * 4, kBufferCfg);
            const int lo = BACKWARD ? T - 16 * sp.hi : 16 * sp.lo, hi = BACKWARD ? T - 16 * sp.lo : 16 * sp.hi;
            for (int t = lo + 4 * lane; t < hi; t += 256) {
                const u4 v = {kUnset, kUnset, kUnset, kUnset};
                __builtin_amdgcn_raw_buffer_store_b128(v, rs, 4 * t, 0, kCpolSc1);
            }
        }
    }

    if (wave == 0) {
        // the compute wave is the critical path: issue priority over the
        // loaders and pollers that share its SIMD
        __builtin_amdgcn_s_setprio(3);
        unsigned long long* dst = c.handoff + (size_t)s * sk_handoff_stride(nx, NW);
        if (sp.consume && sp.produce)
            sweep_compute<Op, BACKWARD, true, true>(op, g, L, sp, epoch, dst, c.err);
        else if (sp.consume)
            sweep_compute<Op, BACKWARD, true, false>(op, g, L, sp, epoch, dst, c.err);
        else if (sp.produce)
            sweep_compute<Op, BACKWARD, false, true>(op, g, L, sp, epoch, dst, c.err);
        else
            sweep_compute<Op, BACKWARD, false, false>(op, g, L, sp, epoch, dst, c.err);
    } else if (wave <= kLoaders) {
        // ------------------------------------------------------------- loaders
        bool bad = false;
        double acc = 0.0;
        for (int sg = sg0; sg < sp.hi; sg += kLoaders) {
            // slot of supergroup sg is free once sg - RING has been consumed
            for (int spin = 0; !bad && (int)lds_ld(&L.consumed_sg) < sg - RING + 1; spin++) {
                if (spin >= kLdsSpin || lds_ld(&L.abort_flag)) {
                    bad = true;
                    raise(kWaitLoader);
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (!PREFETCH || sg != sg0) load_sg(sg);  // with PREFETCH the first one is loaded
            const int slot = sg & (RING - 1);
            const int t0 = BACKWARD ? T - 16 * (sg + 1) : 16 * sg;
#pragma unroll
            for (int j = 0; j < kSub; j++) {
                float4 x[NF];
                op.xform(v[j], x, acc, t0 + 4 * j, s);
#pragma unroll
                for (int a = 0; a < NF; a++) L.ring_f[slot][j][a][lane] = x[a];
                if (NB) L.ring_b[NB ? slot : 0][j][lane] = vb[j];
            }
            if (lane == 0) lds_st(&L.slot_tag[slot], (unsigned)sg + 1u);
        }
        op.loader_done(s, me, acc);
    } else if (wave > kLoaders + kPollers) {
        spare();
    } else if (sp.consume) {
        // ------------------------------------------------------------- pollers
        // Steps in consumption order kk = 16 lo .. 16 hi - 1 (step t = kk
        // forward, T-1-kk backward); the edge lane reads column t - edge_lane,
        // which the upstream strip computes at its step col + up_lane.  The
        // pollers run the same loop, the second one half a poll behind, so a
        // hand-off word is seen about half a memory round trip sooner; both
        // write identical values and hand_ready only grows (LDS max).
        const int src_strip = BACKWARD ? s + 1 : s - 1;
        if (wave == kLoaders + 2) __builtin_amdgcn_s_sleep(4);
        constexpr bool ROW = row_<Op>(0);
        const uint32_t* row_src = nullptr;
        if constexpr (ROW) row_src = op.row + (size_t)src_strip * T;
        const unsigned long long* src = c.handoff + (size_t)src_strip * sk_handoff_stride(nx, NW);
        const int up_lane = 63 - edge_lane, K = 16 * sp.hi;
        bool bad = false;
        for (int k0 = 16 * sp.lo; k0 < K && !bad; k0 += 64) {
            const int kk = k0 + lane;
            const int t = BACKWARD ? T - 1 - kk : kk;
            const int col = t - edge_lane;
            const bool in_grid =
                kk < K && col >= 0 && col < nx && col + up_lane >= sp.up_lo && col + up_lane < sp.up_hi;
            // ring entries of k0 .. k0+63 were used by k - kHandRing
            for (int spin = 0; !bad && 16 * (int)lds_ld(&L.consumed_sg) < k0 + 64 - kHandRing; spin++) {
                if (spin >= kLdsSpin || lds_ld(&L.abort_flag)) {
                    bad = true;
                    raise(kWaitPollerRing);
                }
                __builtin_amdgcn_s_sleep(1);
            }
            if (!in_grid && kk < K)
#pragma unroll
                for (int w = 0; w < NW; w++) L.hand[w][t & (kHandRing - 1)] = 0u;  // boundary state
            unsigned long long hv[NW];
#pragma unroll
            for (int w = 0; w < NW; w++) hv[w] = 0;
            bool got = !in_grid;
            for (int spin = 0; !bad; spin++) {
                if (!got) {
                    bool ok = true;
                    if (ROW) {
                        hv[0] = __hip_atomic_load(const_cast<uint32_t*>(row_src) + col + up_lane, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT);
                        ok = (uint32_t)hv[0] != kUnset;
                    }
#pragma unroll
                    for (int w = 0; w < (ROW ? 0 : NW); w++) {
                        if ((unsigned)(hv[w] >> 32) != epoch)
                            hv[w] = atomic_ld64(src + (size_t)(col + kHandPadLo) * NW + w);
                        ok = ok && (unsigned)(hv[w] >> 32) == epoch;
                    }
                    if (ok) {
#pragma unroll
                        for (int w = 0; w < NW; w++) L.hand[w][t & (kHandRing - 1)] = (uint32_t)hv[w];
                        got = true;
                    }
                }
                // publish the ready prefix of this chunk
                const unsigned long long rdy = __ballot(got);
                const int prefix = rdy == ~0ull ? 64 : __ffsll((long long)~rdy) - 1;
                if (lane == 0) lds_max(&L.hand_ready, (unsigned)min(k0 + prefix, K));
                if (prefix == 64) break;
                if (spin >= kSpinLimit || lds_ld(&L.abort_flag)) {
                    bad = true;
                    if (lane == 0) raise(kWaitHandoff);
                    break;
                }
                __builtin_amdgcn_s_sleep(1);
            }
        }
    }
    if (LOOP) {  // rows reset, results stored
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWaitVm0);
        asm volatile("" ::: "memory");
    }
}

// Supergroups in a single launch's ring: kRing, or 4 for operators with more
// than 3 ring arrays (8 slots of 5 arrays would need 160 KB of LDS).
template <class Op>
constexpr int sweep_ring() {
    return Op::NF > 3 ? 4 : kRing;
}

template <class Op, bool BACKWARD>
__global__ __launch_bounds__(kSweepThreads) void sweep_kernel(Op op, SkGeom g, SkCtl c) {
    __shared__ __align__(16) SweepLds<Op, sweep_ring<Op>()> L;
    const unsigned long long ticket = sweep_ticket(L, c.ticket, c.range, g.S);
    const int order = (int)(ticket % (unsigned long long)g.S);
    const unsigned epoch = (unsigned)(ticket / (unsigned long long)g.S) + 1u;
    sweep_run<Op, BACKWARD, true>(op, g, c, order, epoch, L);
}

// ---------------------------------------------------------------------------
// Operators.  scaleA = dt / (rho dx^2) is the magnitude of every off-diagonal
// (FluidSim2D.cpp:261, 277, 294).
// ---------------------------------------------------------------------------

// Scalars of one projection, each written by exactly one workgroup of the
// kernel that produces it and read by later kernels.
struct PcgScalars {
    double rhs_norm, r_norm, sigma, tol;
    double ws;  // w.s of the current iteration when a separate reduction formed it
    int iter;
    int done;  // 0: iterating.  Non-zero: stopped; the launch whose stopping test runs beside
               // strips that read this (bwd_spmv_kernel) writes its next_iter + 1 (>= 2)
    float beta;  // beta of the current iteration when a separate reduction formed it
    unsigned epoch;  // tags of a solve in one launch: epoch + iteration (fs2d_pcg_loop.hpp)
};

__device__ __forceinline__ double wave_max_of(const double* a, int n) {
    // lane k takes a[k], a[k + 64], ... in that order, with 8 loads in flight
    double m = 0;
    for (int k0 = threadIdx.x & 63; k0 < n; k0 += 64 * 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = k0 + 64 * u < n ? a[k0 + 64 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k0 + 64 * u < n) m = v[u] > m ? v[u] : m;
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        double x = __shfl_xor(m, o, 64);
        m = x > m ? x : m;
    }
    return m;
}
// wave_max_of with every load of a lane in flight at once (n <= 64 W): one
// memory round trip instead of n / 512.  Indices are clamped, not tested: a
// branch around each load cost the head of a launch 0.4 us.
template <int W>
__device__ __forceinline__ double wave_max_of_wide(const double* a, int n) {
    const int lane = threadIdx.x & 63;
    double v[W];
#pragma unroll
    for (int u = 0; u < W; u++) v[u] = a[min(lane + 64 * u, n - 1)];
    double m = 0;
#pragma unroll
    for (int u = 0; u < W; u++) m = v[u] > m ? v[u] : m;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        double x = __shfl_xor(m, o, 64);
        m = x > m ? x : m;
    }
    return m;
}
// The narrowest of them that takes n partials (256 up to 512^2 grids, 2048 at 2048^2).
__device__ __forceinline__ double wave_max_of_any(const double* a, int n) {
    if (n <= 64 * 4) return wave_max_of_wide<4>(a, n);
    if (n <= 64 * 32) return wave_max_of_wide<32>(a, n);
    return wave_max_of(a, n);
}
// Two wave_sum_of sums with every load of both in flight together (n1 <=
// 64 W1, n2 <= 64 W2): one memory round trip instead of several; the same
// additions in the same order.
template <int W1, int W2>
__device__ __forceinline__ void wave_sum_of_wide2(const double* a, int n1, const double* b, int n2, double& sa,
                                                  double& sb) {
    const int lane = threadIdx.x & 63;
    double va[W1], vb[W2];
#pragma unroll
    for (int u = 0; u < W1; u++) va[u] = a[min(lane + 64 * u, n1 - 1)];
#pragma unroll
    for (int u = 0; u < W2; u++) vb[u] = b[min(lane + 64 * u, n2 - 1)];
    double ta = 0, tb = 0;
#pragma unroll
    for (int u = 0; u < W1; u++) ta += lane + 64 * u < n1 ? va[u] : 0.0;
#pragma unroll
    for (int u = 0; u < W2; u++) tb += lane + 64 * u < n2 ? vb[u] : 0.0;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
        ta += __shfl_xor(ta, o, 64);
        tb += __shfl_xor(tb, o, 64);
    }
    sa = ta;
    sb = tb;
}
__device__ __forceinline__ double wave_sum_of(const double* a, int n) {
    double t = 0;
    for (int k0 = threadIdx.x & 63; k0 < n; k0 += 64 * 8) {
        double v[8];
#pragma unroll
        for (int u = 0; u < 8; u++) v[u] = k0 + 64 * u < n ? a[k0 + 64 * u] : 0.0;
#pragma unroll
        for (int u = 0; u < 8; u++)
            if (k0 + 64 * u < n) t += v[u];
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) t += __shfl_xor(t, o, 64);
    return t;
}

// Two wave_sum_of sums, in one round trip where the counts allow it.
__device__ __forceinline__ void wave_sum_of_any2(const double* a, int n1, const double* b, int n2, double& sa,
                                                 double& sb) {
    if (n1 <= 64 && n2 <= 64 * 4) {
        wave_sum_of_wide2<1, 4>(a, n1, b, n2, sa, sb);
    } else if (n1 <= 64 * 4 && n2 <= 64 * 32) {
        wave_sum_of_wide2<4, 32>(a, n1, b, n2, sa, sb);
    } else {
        sa = wave_sum_of(a, n1);
        sb = wave_sum_of(b, n2);
    }
}

// MIC(0) factor (:364-388) and the solve coefficients, in solver units (the
// matrix divided by scaleA: the neighbours' Ax, Ay are -1 times their coupling
// bits).  State: precon (FP64) and the cell's coupling bits.  Outputs (Lt =
// diag(1/P) + lower(A) diag(P), M = Lt Lt^T):
//   P,  fx = c_L P P_L,  fy = c_D P P_D   (q = P r + fx q_L + fy q_D)
//   G = P^2                               (z = P q + G z_R + G z_U)
// The backward terms' couplings c_R and c_U need no factor: a neighbour that is
// not FLUID has P = G = 0, so its z is zero.  One coefficient array instead of
// two takes 4 of the 20 bytes per cell off the solve, and a quarter of the LDS
// reads off its compute wave.
// Products are rounded one by one, as the reference's expression reads
// (no contraction, the same in every launch path).  The first workgroup also
// finishes |rhs|_inf and initialises the solver (:424-430, 447-448).
struct FactorOp {
    static constexpr int NW = 3, NIN = 1, NF = 1, NB = 1, NOUT = 4;
    const float* in[NIN];  // Adiag
    const uint8_t* bytes;  // coupling bits
    float* out[NOUT];      // P, fx, fy, G
    double tau, sigma;
    const double* rhs_partials;
    int n_partials, max_iters;
    PcgScalars* sc;
    double rhs_zero;  // |rhs|_inf at or below which no iteration runs (1e-12, :448, in the rhs' units)
    __device__ bool skip(bool first) const {
        if (first) {
            const double rn = wave_max_of(rhs_partials, n_partials);
            if ((threadIdx.x & 63) == 0) {
                sc->rhs_norm = rn;
                sc->r_norm = rn;
                sc->iter = 0;
                sc->sigma = 0;
                sc->done = (rn <= rhs_zero) || (max_iters <= 0) ? -1 : 0;
            }
        }
        return false;
    }
    __device__ void xform(const float4 (&in)[NIN], float4 (&x)[NF], double&, int, int) const { x[0] = in[0]; }
    __device__ void loader_done(int, int, double) const {}
    template <bool B, bool C, class H>
    __device__ void group(const float4 (&x)[NF], uint32_t b4, uint32_t (&st)[NW], const uint4 (&hb)[NW],
                          float (&o)[NOUT][4], uint32_t (&prod)[NW][4], int, int, H hook) const {
#pragma clang fp contract(off)
#pragma unroll
        for (int q = 0; q < 4; q++) {
            uint32_t nb[NW];
#pragma unroll
            for (int w = 0; w < NW; w++) nb[w] = nbr<B, C>(u4get(hb[w], q), st[w]);
            const uint32_t f = (b4 >> (8 * q)) & 0xffu;
            const double A0 = f4get(x[0], q);
            const double PL = u2d(st), PB = u2d(nb);
            const uint32_t fL = st[2], fB = nb[2];
            // Ax(i-1,j), Ay(i-1,j), Ay(i,j-1), Ax(i,j-1)
            const double axl = (f & CPL_L) ? -1.0 : 0.0, ayl = (fL & CPL_U) ? -1.0 : 0.0;
            const double ayb = (f & CPL_D) ? -1.0 : 0.0, axb = (fB & CPL_R) ? -1.0 : 0.0;
            double Pc = 0;
            if (A0 != 0.0) {  // FLUID cells have a non-zero diagonal, all others zero
                const double t1 = axl * PL, t2 = ayb * PB;
                double e = A0 - t1 * t1 - t2 * t2 - tau * (axl * ayl * PL * PL + ayb * axb * PB * PB);
                if (e < sigma * A0) e = A0;
                Pc = 1.0 / sqrt(e);
            }
            o[0][q] = (float)Pc;
            o[1][q] = (float)(-axl * Pc * PL);
            o[2][q] = (float)(-ayb * Pc * PB);
            o[3][q] = (float)(Pc * Pc);
            d2u(Pc, st);
            st[2] = f;
#pragma unroll
            for (int w = 0; w < NW; w++) prod[w][q] = st[w];
        }
    }
    __device__ void strip_done(int) const {}
};

// Forward solve q = Lt^-1 r (:400-409), q = P r + fx q_L + fy q_D; the loaders
// form P r.
//   FUSED false: in iteration mode the first workgroup finishes |r|_inf and
//     applies the stopping test (:453) before any preconditioning, as the
//     reference does.
//   FUSED true: the solve's strips inside fwd_axpy_kernel, after the same
//     launch's p/r update.  Strip s's loaders first wait for the update's runs
//     over strip s (run_flags[vb] = the launch's epoch, published after the
//     runs' device-scope r stores); the stopping test moves to the backward
//     solve's launch, so the last solve of a projection runs once more than
//     needed, writing only q.
template <bool FUSED>
struct FwdOpT {
    static constexpr int NW = 1, NIN = 4, NF = 3, NB = 0, NOUT = 1;
    static constexpr bool kWaitInputs = FUSED, kRow = true;
    const float* in[NIN];  // r, P, fx, fy
    const uint8_t* bytes;
    float* out[NOUT];      // q
    uint32_t *row, *row_next;
    PcgScalars* sc;
    const double* rmax_partials;
    int n_partials, check;
    const unsigned* run_flags;  // FUSED: [n_partials] p/r update runs
    SkGeom geom;                // FUSED: the runs' strips
    unsigned epoch;
    __device__ bool skip(bool first) {
        if (sc->done) return true;
        if (FUSED || !check) return false;
        const double rn = wave_max_of(rmax_partials, n_partials);
        const bool conv = rn <= sc->tol * sc->rhs_norm;
        if (first && (threadIdx.x & 63) == 0) {
            sc->r_norm = rn;
            if (conv) sc->done = 1;
        }
        return conv;
    }
    // Runs of the p/r update are whole 256-entry groups, the n / 256 groups
    // split evenly over n_partials runs (pcg_run); strip s is groups
    // s T4 .. (s+1) T4 - 1.
    __device__ void wait_inputs(int s, int* err) const {
        if (!FUSED || sc->done) return;
        const long ng = geom.size() >> 8, nr = n_partials;
        const long g0 = (long)s * geom.T4, g1 = g0 + geom.T4;  // the strip's groups
        // runs vb with ng vb / nr < g1 and ng (vb + 1) / nr > g0
        const int lo = (int)(g0 * nr / ng), hi = (int)min(nr - 1, (g1 * nr + ng - 1) / ng);
        const int lane = threadIdx.x & 63;
        for (int v0 = lo; v0 <= hi; v0 += 64) {
            const int vb = v0 + lane;
            for (int spin = 0;; spin++) {
                const bool ok = vb > hi || __hip_atomic_load(run_flags + vb, __ATOMIC_RELAXED,
                                                              __HIP_MEMORY_SCOPE_AGENT) == epoch;
                if (__all(ok)) break;
                if (spin >= kSpinLimit || __hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) {
                    if (lane == 0) raise_wait(err, kWaitRuns);
                    return;
                }
                __builtin_amdgcn_s_sleep(4);
            }
        }
    }
    __device__ void xform(const float4 (&in)[NIN], float4 (&x)[NF], double&, int, int) const {
        x[0] = make_float4(in[1].x * in[0].x, in[1].y * in[0].y, in[1].z * in[0].z, in[1].w * in[0].w);
        x[1] = in[2];
        x[2] = in[3];
    }
    __device__ void loader_done(int, int, double) const {}
    template <bool B, bool C, class H>
    __device__ void group(const float4 (&x)[NF], uint32_t, uint32_t (&st)[NW], const uint4 (&hb)[NW],
                          float (&o)[NOUT][4], uint32_t (&prod)[NW][4], int, int, H hook) const {
        float qp = u2f(st[0]);
#pragma unroll
        for (int q = 0; q < 4; q++) {
            // the row term first: the DPP then reads qp one instruction later
            const float t1 = fmaf(f4get(x[1], q), qp, f4get(x[0], q));
            hook(q);
            const float qd = u2f(nbr<B, C>(u4get(hb[0], q), f2u(qp)));
            const float qn = fmaf(f4get(x[2], q), qd, t1);
            o[0][q] = qn;
            prod[0][q] = f2u(qn);
            qp = qn;
        }
        st[0] = f2u(qp);
    }
    __device__ void strip_done(int) const {}
};
using FwdOp = FwdOpT<false>;
using FwdFusedOp = FwdOpT<true>;

// Backward solve z = Lt^-T q (:410-419), z = P q + G z_R + G z_U; steps run
// q = 3, 2, 1, 0 within a group; the loaders form P q.  The first workgroup
// records the iteration count (:462).
//   FUSED false: the loaders also sum q.q per strip: z.r = r.M^-1 r =
//     |Lt^-1 r|^2 = q.q is sigma (:428, :457), into qq_partials[S][kLoaders].
//   FUSED true: the solve's strips inside bwd_spmv_kernel; sigma is summed by
//     that launch's own workgroups (in the loaders' order), and each strip's
//     compute wave publishes its completion for the SpMV workgroups of the
//     same launch: z is stored with device scope (kOutThrough), so once those
//     stores have completed (vmcnt 0) the flag may follow.
__device__ __forceinline__ double qq4(const float4& q) {
    return (double)fmaf(q.w, q.w, fmaf(q.z, q.z, fmaf(q.y, q.y, q.x * q.x)));
}
template <bool FUSED>
struct BwdOpT {
    static constexpr int NW = 1, NIN = 3, NF = 2, NB = 0, NOUT = 1;
    static constexpr bool kOutThrough = FUSED, kRow = true;
    const float* in[NIN];  // q, P, G
    const uint8_t* bytes;
    float* out[NOUT];      // z
    uint32_t *row, *row_next;
    PcgScalars* sc;
    double* qq_partials;   // [S][kLoaders] (FUSED false)
    int next_iter;         // iterations completed after this solve (0: initial solve)
    unsigned* strip_flags; // [S] (FUSED true): the launch's epoch once the strip's z is stored
    unsigned epoch;
    int check;                    // FUSED false: the iteration's stopping test (:453) first, as
                                  // FwdOp's, when the p/r update ran with the forward solves
                                  // (b_fwd_axpy_kernel)
    const double* rmax_partials;  // |r|_inf partials of the iteration's p/r update
    int n_partials;
    __device__ bool skip(bool first) const {
        // fused: the kernel has tested sc->done, the launch's SpMV workgroups
        // apply the stopping test and record the count; the strips run
        // regardless (the solve of the iteration that converges writes only z
        // and sigma, which no later launch reads)
        if (FUSED) return false;
        if (sc->done) return true;
        if (check) {
            const double rn = wave_max_of_any(rmax_partials, n_partials);
            const bool conv = rn <= sc->tol * sc->rhs_norm;
            if (first && (threadIdx.x & 63) == 0) {
                sc->r_norm = rn;
                if (conv) sc->done = 1;
            }
            if (conv) return true;
        }
        if (first && (threadIdx.x & 63) == 0 && next_iter > 0) sc->iter = next_iter;
        return false;
    }
    __device__ void xform(const float4 (&in)[NIN], float4 (&x)[NF], double& acc, int, int) const {
        const float4 q = in[0], P = in[1];
        x[0] = make_float4(P.x * q.x, P.y * q.y, P.z * q.z, P.w * q.w);
        x[1] = in[2];
        if (!FUSED) acc += qq4(q);
    }
    __device__ void loader_done(int s, int me, double acc) const {
        if (FUSED) return;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
        if ((threadIdx.x & 63) == 0) qq_partials[s * kLoaders + me] = acc;
    }
    template <bool B, bool C, class H>
    __device__ void group(const float4 (&x)[NF], uint32_t, uint32_t (&st)[NW], const uint4 (&hb)[NW],
                          float (&o)[NOUT][4], uint32_t (&prod)[NW][4], int, int, H hook) const {
        float zp = u2f(st[0]);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int q = 3 - i;
            const float t1 = fmaf(f4get(x[1], q), zp, f4get(x[0], q));
            hook(i);
            const float zu = u2f(nbr<B, C>(u4get(hb[0], q), f2u(zp)));
            const float zn = fmaf(f4get(x[1], q), zu, t1);
            o[0][q] = zn;
            prod[0][q] = f2u(zn);
            zp = zn;
        }
        st[0] = f2u(zp);
    }
    __device__ void strip_done(int s) const {
        if (!FUSED) return;
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_waitcnt(kWaitVm0);  // every z store of the strip is in memory
        asm volatile("" ::: "memory");
        if ((threadIdx.x & 63) == 0)
            __hip_atomic_store(strip_flags + s, epoch, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
};
using BwdOp = BwdOpT<false>;
using BwdFusedOp = BwdOpT<true>;

}  // namespace fs2d
