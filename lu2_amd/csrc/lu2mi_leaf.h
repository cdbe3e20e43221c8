// lu2mi_leaf.h -- the panel's leaf (a W-column strip factored by co-resident
// workgroups), the row-swap strip and the persistent sub-panel kernel.
#pragma once
#include "lu2mi_internal.h"
#include "lu2mi_dev.h"
#include "lu2mi_gemm_tile.h"
#include <limits.h>

// ---------------------------------------------------------------------------
// Leaf factorization: persistent kernel over rows [c, n), W columns; all
// workgroups are co-resident and exchange messages once per column.
namespace {
constexpr int NTL = 256;        // threads per workgroup in the leaf kernel
constexpr int LEAF_GMAX = 128;  // most workgroups a leaf launch may use

__device__ __forceinline__ void st_relaxed(unsigned long long *p, unsigned long long v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long ld_relaxed(unsigned long long *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ unsigned long long dbits(double v) { return __double_as_longlong(v); }
__device__ __forceinline__ double bitsd(unsigned long long v) { return __longlong_as_double(v); }
// device-scope (coherent across XCDs) scalar loads and stores of a vector element
__device__ __forceinline__ double ld_dev(const double *p)
{
    return bitsd(__hip_atomic_load((unsigned long long *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
__device__ __forceinline__ float ld_dev(const float *p)
{
    return __uint_as_float(__hip_atomic_load((unsigned *)p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
}
// device-scope loads through a buffer resource: same coherence as ld_dev but
// without a wait after every load, so independent loads overlap
__device__ __forceinline__ double ld_buf(__amdgpu_buffer_rsrc_t r, int byte_off, double)
{
    const unsigned int lo = __builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, 16);
    const unsigned int hi = __builtin_amdgcn_raw_buffer_load_b32(r, byte_off + 4, 0, 16);
    return bitsd(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ float ld_buf(__amdgpu_buffer_rsrc_t r, int byte_off, float)
{
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, byte_off, 0, 16));
}
__device__ __forceinline__ void st_dev(double *p, double v)
{
    __hip_atomic_store((unsigned long long *)p, dbits(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void st_dev(float *p, float v)
{
    __hip_atomic_store((unsigned *)p, __float_as_uint(v), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Publication of a sequence word (the back-substitution frontier) after the
// data it announces.  Every exchanged word is written and read with
// device-coherent (agent-scope, sc1) accesses, so no cache maintenance is
// needed, only completion order: the compiler barriers keep the data stores
// ahead of the sequence store in program order and s_waitcnt vmcnt(0) makes
// them complete before it is issued.  strict: an agent-scope release store
// instead (on gfx950 it adds buffer_wbl2, an L2 writeback, per publication;
// the matching acquire on the reader adds buffer_inv, an L2 invalidate).
__device__ __forceinline__ void publish_seq(unsigned long long *p, unsigned long long v, int strict)
{
    if (strict) {
        __hip_atomic_store(p, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_AGENT);
    } else {
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __builtin_amdgcn_s_waitcnt(0);
        __atomic_signal_fence(__ATOMIC_SEQ_CST);
        __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}
// reader side, after the spin on a sequence word has seen the new value
__device__ __forceinline__ void acquire_seq(int strict)
{
    if (strict) __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    else __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

// rank-1 update of one element: x - l * us, us = u * s rounded (the stored U
// value), one fused multiply-subtract, written out so that every copy of a
// row computes bit-identical values
__device__ __forceinline__ double fused_update(double x, double l, double us) { return fma(-l, us, x); }
__device__ __forceinline__ float fused_update(float x, float l, float us) { return fmaf(-l, us, x); }

// A pivot candidate's key: |x| as the bits of a non-negative number (they
// order as the numbers do) in two words, and its row; no candidate is
// (0, 0, INT_MAX), which loses to any row.
struct alignas(16) PivKey {
    unsigned hi, lo;
    int r;
};
__device__ __forceinline__ PivKey piv_key(double v, int r)
{
    const unsigned long long b = dbits(v);
    PivKey k;
    k.hi = r == INT_MAX ? 0u : (unsigned)(b >> 32);
    k.lo = r == INT_MAX ? 0u : (unsigned)b;
    k.r = r;
    return k;
}
__device__ __forceinline__ bool better(const PivKey &a, const PivKey &b)
{
    const unsigned long long x = ((unsigned long long)a.hi << 32) | a.lo, y = ((unsigned long long)b.hi << 32) | b.lo;
    return x > y || (x == y && a.r < b.r);
}

template <int CTRL>
__device__ __forceinline__ unsigned dpp_lane(unsigned v)
{
    return (unsigned)__builtin_amdgcn_update_dpp((int)v, (int)v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ double lane_bcast(double v, int l)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)b, l), hi = __builtin_amdgcn_readlane((int)(b >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ __forceinline__ float lane_bcast(float v, int l)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l));
}

// maximum over four lanes
__device__ __forceinline__ unsigned quad_max(unsigned v)
{
    v = max(v, dpp_lane<0xB1>(v));
    return max(v, dpp_lane<0x4E>(v));
}
// maximum over the wavefront: within 16 lanes by DPP (xor 1, xor 2, mirrored
// halves, mirrored rows), across the four 16-lane rows by readlane -- no LDS
// permutes, whose latency a step of the leaf would pay six times in a row
__device__ __forceinline__ unsigned wave_max(unsigned v)
{
    v = quad_max(v);
    v = max(v, dpp_lane<0x141>(v));
    v = max(v, dpp_lane<0x140>(v));
    const unsigned a = (unsigned)__builtin_amdgcn_readlane((int)v, 0), b = (unsigned)__builtin_amdgcn_readlane((int)v, 16);
    const unsigned c = (unsigned)__builtin_amdgcn_readlane((int)v, 32), d = (unsigned)__builtin_amdgcn_readlane((int)v, 48);
    return max(max(a, b), max(c, d));
}

// The lane of the best key (largest |x|, lowest row), the same in every lane.
// The upper words nearly always decide; only a tie looks further.
__device__ __forceinline__ int wave_argmax(const PivKey &k)
{
    unsigned long long m = __ballot(k.hi == wave_max(k.hi));
    if (m & (m - 1)) {
        const bool in = (m >> (threadIdx.x & 63)) & 1;
        const unsigned lo = wave_max(in ? k.lo : 0u);
        const bool in2 = in && k.lo == lo;
        const unsigned nr = wave_max(in2 ? ~(unsigned)k.r : 0u);   // rows are >= 0: ~r is never 0
        m = __ballot(in2 && ~(unsigned)k.r == nr);
    }
    return (int)__builtin_ctzll(m);
}
// the same over the keys of four wavefronts, lane l holding key l % 4
__device__ __forceinline__ int quad_argmax(const PivKey &k)
{
    unsigned long long m = __ballot(k.hi == quad_max(k.hi)) & 15;
    if (m & (m - 1)) {
        const bool in = (m >> (threadIdx.x & 3)) & 1;
        const unsigned lo = quad_max(in ? k.lo : 0u);
        const bool in2 = in && k.lo == lo;
        const unsigned nr = quad_max(in2 ? ~(unsigned)k.r : 0u);
        m = __ballot(in2 && ~(unsigned)k.r == nr) & 15;
    }
    return (int)__builtin_ctzll(m);
}
}  // namespace

template <typename T>
struct LeafArgs {
    T *A;
    long lda;
    int n, c, i, compat;
    int G;                        // number of workgroups (grid size)
    int *piv;                     // global pivots, piv[j] for j in [c, c+W)
    int *orig;                    // block-level origin row ids
    T *invd;                      // 1/d per pivot row
    int *pair_dst, *pair_src;     // 2W pairs for the panel row permutation
    T *linv;                      // nb x nb inverse of D^-1 L11 (this leaf's block)
    int ldl;
    unsigned long long *slots;    // 2 * G messages of LeafMsg<T, W>::NW words, G <= LEAF_GMAX
    unsigned long long seq_base;  // step tags seq_base+1 .. seq_base+W
    int *err;
};

// One workgroup's message of a column step: its candidate row's W values, the
// row number and the row's two origins, as 32-bit words (and one spare, so
// that messages lie at 16-byte multiples in LDS).  In memory every word
// travels with its step's tag in one 8-byte store, so a reader that sees the
// tag has the word: no sequence word behind the data, no wait between them,
// and one round trip instead of a poll followed by a copy.
constexpr int LEAF_NB = 10;   // message words per thread in one batch of loads: 64 FP64 messages of 16 columns
template <typename T, int W>
struct LeafMsg {
    static constexpr int VW = W * (int)sizeof(T) / 4;
    static constexpr int NW = VW + 4;
    // LDS words of a step's messages, whole batches
    static constexpr int XW = (LEAF_GMAX * NW + LEAF_NB * NTL - 1) / (LEAF_NB * NTL) * (LEAF_NB * NTL);
};

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
template <int V>
struct IntC {
    static constexpr int value = V;
};

// Per column step j (one grid-wide exchange):
//   gather   every workgroup polls all words of all messages (the candidate
//            row of every workgroup) and puts them into LDS: the threads'
//            loads are all in flight at once, and a thread repeats its own
//            until their tags are the step's;
//   reduce   each wavefront reduces the G candidates (largest |x|, lowest
//            row on ties) -- identical result everywhere, no extra barrier;
//   swap     the owners of rows j and p exchange rows, row j scaled by 1/d;
//   column j+1 updated first, its candidate reduced in the workgroup and
//            published (lookahead), then the other columns updated while
//            the exchange is in flight.
// With one workgroup (G == 1) the messages go straight to LDS.
//
// What bounds it: a step is one chain of latencies, whatever the number of
// rows -- candidate reduction, publication, the way through the
// device-coherent level, the reduction of the candidates, 1/d.  FP64, 16
// columns, alone on the device, before and after the tagged messages, the
// DPP reductions, the rotation and the copies of the current rows: 60 -> 30 us
// for 256 rows (one workgroup), 60 -> 43.5 us for 4096 (16 of them), 64.5 -> 48
// us for 9984 rows (39 workgroups), about 105 -> 61 us for 60000 rows; of the
// 48 us, 2.8 us per column: 1.4 the wait for the other workgroups' messages,
// 0.3 reduction and 1/d, 0.3 swap, 0.6 update, candidate and sending, the rest
// reading and writing the panel.
template <typename T, int W>
struct LeafSmem {
    union {
        T stage[NTL * (W + 1)];
        unsigned xch[2][LeafMsg<T, W>::XW];
    };
    alignas(16) unsigned pub[LeafMsg<T, W>::NW];   // the candidate before it is sent
    alignas(16) T cur[W];                          // row j in the order of the messages, where it is the pivot row
    T top[W * W];                                  // rows c .. c+W-1 as they stand, in column order
    int top_lorig[W], top_borig[W];
    PivKey red[NTL / 64];
    int pivs[W];
};

// the leaf as workgroup bid of a.G (a stand-alone launch, or a phase of the
// persistent sub-panel kernel)
template <typename T, int W, int RPT>
__device__ __forceinline__ void leaf_body(const LeafArgs<T> &a, const int bid, LeafSmem<T, W> &sm)
{
    typedef LeafMsg<T, W> Msg;
    constexpr int RS = 64 / W;   // rows one load or store of a wavefront covers
    constexpr int VW = Msg::VW, NW = Msg::NW, TW = (int)sizeof(T) / 4;
    T *const stage = sm.stage;
    auto &xch = sm.xch;
    PivKey *const red = sm.red;
    int *const pivs = sm.pivs;

    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int G = a.G;
    const long TT = (long)G * NTL;
    const int n = a.n, c = a.c;
    T *__restrict__ A = a.A;
    unsigned long long *const slots = a.slots;
    const int total = G * NW;   // words of one step
    const __amdgpu_buffer_rsrc_t srsrc =
        __builtin_amdgcn_make_buffer_rsrc(slots, 0, 2 * total * 8, 0x00020000);

    T row[RPT][W];
    int lorig[RPT], borig[RPT], rq[RPT];

    // coalesced load of the rows (all layers in flight); each wavefront
    // transposes its own 64 rows through its own part of the LDS
    T *const wst = stage + wave * 64 * (W + 1);
    auto wave_sync = [&]() __attribute__((always_inline)) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
#pragma clang loop unroll(full)
    for (int q = 0; q < RPT; q++) {
        const long base = (long)c + (long)bid * NTL + (long)q * TT;
        rq[q] = (int)min((long)INT_MAX, base + t);
        const long r0 = base + wave * 64 + lane / W;   // then every RS-th row
        const T *src = A + r0 * a.lda + c + lane % W;
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++, src += RS * a.lda) row[q][k] = (r0 + k * RS < n) ? *src : T(0);
        lorig[q] = rq[q];
        borig[q] = (rq[q] < n) ? ((c == a.i) ? rq[q] : a.orig[rq[q]]) : -1;
    }
#pragma clang loop unroll(full)
    for (int q = 0; q < RPT; q++) {
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++) {
            const int e = lane + k * 64;
            wst[(e / W) * (W + 1) + e % W] = row[q][k];
        }
        wave_sync();
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++) row[q][k] = wst[lane * (W + 1) + k];
        wave_sync();
    }

    // Registers rotate by one column per step: at step jl position k holds
    // column (jl + k) mod W, so the step's own column is position 0 and one
    // copy of the step's code serves all of them.  (Unrolled over the columns
    // the leaf was 123 to 194 KB of code that ran once: every step waited for
    // its instructions.)  Messages hold the row in the order of their step.
    //
    // local candidate of step jc, workgroup reduction, publication of the
    // message.  LATE: the
    // registers are still in the order of step jc - 1, whose update of the
    // columns beyond jc is pending (lookahead) with the scaled pivot row us:
    // the published values carry it, computed as the bulk update does.
    auto publish = [&](auto late, const int jc, const T (&us)[W]) __attribute__((always_inline)) {
        constexpr int P0 = decltype(late)::value;   // position of column jc
        const int j = c + jc;
        const int par = jc & 1;
        const bool odd_rule = a.compat && (jc & 1);
        double bv = -1.0;
        int br = INT_MAX;
#pragma clang loop unroll(full)
        for (int q = 0; q < RPT; q++) {
            const int r = rq[q];
            const double v = fabs((double)(odd_rule ? row[q][0] : row[q][P0]));   // odd_rule: LATE, column jc - 1
            if (r >= j && r < n && v > bv) { bv = v; br = r; }
        }
        const PivKey key = piv_key(bv, br);
        const int wl = wave_argmax(key);
        if (lane == wl) red[wave] = key;
        __syncthreads();
        const PivKey wkey = red[lane & 3];
        const int wr = __builtin_amdgcn_readlane(wkey.r, quad_argmax(wkey));
        // row q of the lane that has own set (at most one of the wavefront)
        auto send = [&](const bool own, const int q) __attribute__((always_inline)) {
            if (!__any(own)) return;
            unsigned *const m = (G == 1) ? xch[par] : sm.pub;
            if (own) {
#pragma clang loop unroll(full)
                for (int k = 0; k < W; k++) {
                    T v = row[q][k];
                    if (P0 == 1 && k >= 2) {
                        const T y = fused_update(v, row[q][0], us[k]);
                        v = (k <= W - jc) ? y : v;
                    }
                    ((T *)m)[(k + W - P0) % W] = v;
                }
                m[VW] = (unsigned)rq[q];
                m[VW + 1] = (unsigned)lorig[q];
                m[VW + 2] = (unsigned)borig[q];
            }
            if (G == 1) return;
            // the wavefront stores what its lane put into LDS
            wave_sync();
            const unsigned long long tag = (a.seq_base + (unsigned long long)jc + 1) << 32;
            unsigned long long *const sl = slots + (long)par * total + bid * NW;
#pragma clang loop unroll(full)
            for (int w0 = 0; w0 < NW; w0 += 64)
                if (w0 + lane < NW) st_relaxed(sl + w0 + lane, tag | m[w0 + lane]);
        };
        if (wr < n) {
#pragma clang loop unroll(full)
            for (int q = 0; q < RPT; q++) send(rq[q] == wr, q);
        } else if (G == 1) {   // no candidate: only the row number is looked at
            if (t == 0) xch[par][VW] = (unsigned)INT_MAX;
        } else if (t < NW) {
            const unsigned long long tag = (a.seq_base + (unsigned long long)jc + 1) << 32;
            st_relaxed(slots + (long)par * total + bid * NW + t, tag | (unsigned)INT_MAX);
        }
    };

    // all words of step par with tag tg from the slots into LDS, NB loads per
    // thread in flight; words beyond the last are out of the buffer's range
    auto gather = [&](auto nb_, const int base, const int par, const unsigned tg) __attribute__((always_inline)) {
        constexpr int NB = decltype(nb_)::value;
        u32x2 v[NB];
        unsigned long spins = 0;
        for (;;) {
            bool ok = true;
#pragma clang loop unroll(full)
            for (int k = 0; k < NB; k++) {
                const int w = base + k * NTL + t;
                v[k] = __builtin_amdgcn_raw_buffer_load_b64(srsrc, w < total ? (par * total + w) * 8 : -8, 0, 16);
            }
#pragma clang loop unroll(full)
            for (int k = 0; k < NB; k++) ok = ok && (base + k * NTL + t >= total || v[k].y == tg);
            if (ok) break;
            asm volatile("" ::: "memory");   // the loads are repeated, not kept
            if (((++spins) & 1023) == 0) {
                if (__hip_atomic_load(a.err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
                if (spins > (1UL << 25)) {
                    __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
            }
        }
#pragma clang loop unroll(full)
        for (int k = 0; k < NB; k++) xch[par][base + k * NTL + t] = v[k].x;
    };

    // Every workgroup keeps its own copy of the W rows that become the current
    // rows (same arithmetic, same bits as the owner's registers): the owner of
    // a pivot finds the row it receives there, and no second message has to
    // leave workgroup 0, whose sending it was the longest part of a step.
    for (int e = t; e < W * W; e += NTL) sm.top[e] = A[(long)(c + e / W) * a.lda + c + e % W];
    if (t < W) {
        sm.top_lorig[t] = c + t;
        sm.top_borig[t] = (c == a.i) ? c + t : a.orig[c + t];
    }
    T us[W];   // the step's pivot row (rotated like the rows) times 1/d; [0] unused
#pragma clang loop unroll(full)
    for (int k = 0; k < W; k++) us[k] = T(0);
    __syncthreads();   // every wavefront is done with its staged rows (LDS shared with xch)
    publish(IntC<0>(), 0, us);
#pragma clang loop unroll(disable)
    for (int jl = 0; jl < W; jl++) {
        const int j = c + jl;
        const int par = jl & 1;
        const unsigned *const xb = xch[par];
        if (G > 1) {
            const unsigned tg = (unsigned)(a.seq_base + (unsigned long long)jl + 1);
            if (total <= NTL) gather(IntC<1>(), 0, par, tg);
            else if (total <= 4 * NTL) gather(IntC<4>(), 0, par, tg);
            else
                for (int b0 = 0; b0 < total; b0 += LEAF_NB * NTL) gather(IntC<LEAF_NB>(), b0, par, tg);
        }
        __syncthreads();
        // ---- every wavefront reduces the G candidates (same result everywhere)
        int br, bg = 0;
        if (G == 1) {
            br = (int)xb[VW];
        } else {
            // the column that decides: this one, or under the odd rule the
            // one before it, which the rotation has left at the end
            const int kv = ((a.compat && (jl & 1)) ? W - 1 : 0) * TW;
            const int g1 = min(lane, G - 1);   // spare lanes repeat the last slot
            PivKey key = piv_key(fabs((double)*(const T *)&xb[g1 * NW + kv]), (int)xb[g1 * NW + VW]);
            bg = g1;
            if (G > 64) {
                const int g2 = min(lane + 64, G - 1);
                const PivKey o = piv_key(fabs((double)*(const T *)&xb[g2 * NW + kv]), (int)xb[g2 * NW + VW]);
                if (better(o, key)) { key = o; bg = g2; }
            }
            const int wl = wave_argmax(key);
            br = __builtin_amdgcn_readlane(key.r, wl);
            bg = __builtin_amdgcn_readlane(bg, wl);
        }
        // no comparable candidate (every |x| is NaN): pivot on the current
        // row, as BLAS idamax returns the first index for NaN input
        const bool none = (br < j || br >= n);
        const int p = none ? j : br;
        const unsigned *pslot = xb + bg * NW;
        if (none) {   // row j in the messages' order (every wavefront writes the same)
            if (lane < W) sm.cur[lane] = sm.top[jl * W + (jl + lane) % W];
            wave_sync();
            pslot = (const unsigned *)sm.cur;
        }
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++) us[k] = ((const T *)pslot)[k];
        const T d = us[0];
        const T s = T(1) / d;
#pragma clang loop unroll(full)
        for (int k = 1; k < W; k++) us[k] = us[k] * s;   // rounded: the stored U values
        // ---- swap rows j and p; row j becomes the pivot row scaled by 1/d
#pragma clang loop unroll(full)
        for (int q = 0; q < RPT; q++) {
            const int r = rq[q];
            if (r == j) {
                row[q][0] = d;
#pragma clang loop unroll(full)
                for (int k = 1; k < W; k++) row[q][k] = us[k];
                lorig[q] = none ? lorig[q] : (int)pslot[VW + 1];
                borig[q] = none ? borig[q] : (int)pslot[VW + 2];
            } else if (r == p) {
#pragma clang loop unroll(full)
                for (int k = 0; k < W; k++) row[q][k] = sm.top[jl * W + (jl + k) % W];
                lorig[q] = sm.top_lorig[jl];
                borig[q] = sm.top_borig[jl];
            }
        }
        // ---- column j+1 first, then publish its candidate (lookahead)
        if (jl + 1 < W) {
#pragma clang loop unroll(full)
            for (int q = 0; q < RPT; q++)
                if (rq[q] > j) row[q][1] = fused_update(row[q][1], row[q][0], us[1]);
            publish(IntC<1>(), jl + 1, us);
        }
        // ---- the remaining columns while the exchange is in flight, and the
        // rotation (rows past the matrix's end hold zeros that nothing reads)
        const int live = W - jl;
#pragma clang loop unroll(full)
        for (int q = 0; q < RPT; q++) {
            const T l = row[q][0];
            const bool upd = rq[q] > j;
            row[q][0] = row[q][1];
#pragma clang loop unroll(full)
            for (int k = 2; k < W; k++) {
                T x = row[q][k];
                if (k < live) {
                    const T y = fused_update(x, l, us[k]);
                    x = upd ? y : x;
                }
                row[q][k - 1] = x;
            }
            row[q][W - 1] = l;
        }
        // the copy of the rows below row j; row j itself, which the row
        // that leaves it may still be read from, stays
        for (int e = t; e < W * W; e += NTL) {
            const int r = e / W, col = e % W;
            if (r > jl) {
                const int from = (c + r == p) ? jl : r;
                const int k = (col + W - jl) % W;
                const T u = ((const T *)pslot)[k];
                const T x = sm.top[from * W + col];
                const T y = fused_update(x, sm.top[from * W + jl], u * s);
                const T z = (col > jl) ? y : x;
                if (from != r || col > jl) sm.top[e] = z;
            }
        }
        if (t < W && t > jl && c + t == p) {
            sm.top_lorig[t] = sm.top_lorig[jl];
            sm.top_borig[t] = sm.top_borig[jl];
        }
        if (t == 0) {
            pivs[jl] = p;
            if (bid == 0) {
                a.piv[j] = p;
                a.invd[j] = s;
            }
        }
    }
    __syncthreads();

    // ---- write back rows (coalesced, each wavefront through its part of the
    // LDS), origins and row pairs
#pragma clang loop unroll(full)
    for (int q = RPT - 1; q >= 0; q--) {   // layer 0 last: the inverse below reads it
        const long base = (long)c + (long)bid * NTL + (long)q * TT;
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++) wst[lane * (W + 1) + k] = row[q][k];
        wave_sync();
        const long r0 = base + wave * 64 + lane / W;
        T *dst = A + r0 * a.lda + c + lane % W;
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++, dst += RS * a.lda)
            if (r0 + k * RS < n) *dst = wst[(lane / W + k * RS) * (W + 1) + lane % W];
        wave_sync();
        const int r = rq[q];
        if (r < n) {
            a.orig[r] = borig[q];
#pragma clang loop unroll(full)
            for (int k = 0; k < W; k++)
                if (pivs[k] == r) {
                    a.pair_dst[W + k] = r;
                    a.pair_src[W + k] = lorig[q];
                }
        }
    }
    if (bid == 0 && t < W) {
        a.pair_dst[t] = c + t;
        a.pair_src[t] = lorig[0];
        // leaf block of the inverse of the unit-lower D^-1 L11, whose rows
        // this wavefront staged last: thread t forms column t, every finished
        // x[k] applied to all sums below it at once
        T x[W], acc[W], l[W], lnext[W];   // l: column k of the staged rows, one step ahead
#pragma clang loop unroll(full)
        for (int r = 0; r < W; r++) {
            acc[r] = T(0);
            lnext[r] = wst[r * (W + 1)];
        }
#pragma clang loop unroll(full)
        for (int k = 0; k < W; k++) {
            x[k] = (k < t) ? T(0) : (k == t) ? T(1) : -acc[k];
#pragma clang loop unroll(full)
            for (int r = k + 1; r < W; r++) {
                l[r] = lnext[r];
                if (r > k + 1) lnext[r] = wst[r * (W + 1) + k + 1];
            }
            if (k >= t) {
#pragma clang loop unroll(full)
                for (int r = k + 1; r < W; r++) acc[r] = fma(l[r], x[k], acc[r]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        const long off = (long)(c - a.i);
#pragma clang loop unroll(full)
        for (int r = 0; r < W; r++) a.linv[(off + r) * a.ldl + off + t] = x[r];
    }
}

// at most 256 VGPRs for the 16-wide leaf, so that it fits on a SIMD beside one
// wavefront of the trailing update.  Within them (FP64) one row per thread
// takes 146, two 209; four, for more than 32768 rows, spill 34 (140 bytes of
// scratch a lane): 61 us a leaf at 60000 rows all the same, where the kernel
// before the tagged messages took 105 with 220 VGPRs and no scratch
template <typename T, int W, int RPT>
__global__ __launch_bounds__(NTL, W == 16 ? 2 : 1) void leaf_kernel(LeafArgs<T> a)
{
    __shared__ LeafSmem<T, W> sm;
    __builtin_amdgcn_s_setprio(3);   // ahead of the trailing update's waves beside it, as all of the panel's kernels
    leaf_body<T, W, RPT>(a, blockIdx.x, sm);
}

// ---------------------------------------------------------------------------
// Row permutation of a column range: all sources of a column strip are read
// into LDS before any destination is written, so in-place permutations are
// safe.  Destinations in [d0, d1) are scaled by invd[dst] on columns < sce;
// destinations in [w0, w1) are written to the staging buffer instead.
template <typename T>
struct PermArgs {
    T *A;
    long lda;
    const int *dst, *src;
    int np;
    int c0, c1, k0, k1;   // columns [c0, c1) except [k0, k1)
    int sce;              // scale columns < sce
    int d0, d1;
    const T *invd;
    T *W;
    long ldw;
    int w0, w1;
    int sw;               // strip width
};

template <typename T>
__device__ __forceinline__ void rowperm_strip(const PermArgs<T> &a, const int strip, T *buf)
{
    const int cs = a.c0 + strip * a.sw;
    const int total = a.np * a.sw;
    for (int e = threadIdx.x; e < total; e += 256) {
        const int pr = e / a.sw, cc = e % a.sw;
        const int col = cs + cc;
        if (col < a.c1 && (col < a.k0 || col >= a.k1)) buf[e] = a.A[(long)a.src[pr] * a.lda + col];
    }
    __syncthreads();
    for (int e = threadIdx.x; e < total; e += 256) {
        const int pr = e / a.sw, cc = e % a.sw;
        const int col = cs + cc;
        if (col < a.c1 && (col < a.k0 || col >= a.k1)) {
            const int d = a.dst[pr];
            T v = buf[e];
            if (d >= a.d0 && d < a.d1 && col < a.sce) v *= a.invd[d];
            if (d >= a.w0 && d < a.w1) a.W[(long)(d - a.w0) * a.ldw + (col - a.c0)] = v;
            else a.A[(long)d * a.lda + col] = v;
        }
    }
}

// ---------------------------------------------------------------------------
// Persistent sub-panel: one launch factors w columns [c, c+w) of the block's
// panel (w a power of two <= SUB_WMAX, 16-column leaves): every leaf, its row
// swaps over the panel's other columns, and every recursion node inside the
// sub-panel (1/d scaling and staging, explicit-inverse TRSM, update of the
// rows below, off-diagonal block of the inverse), in the order of the
// recursion of lu2.c:1187-1235, separated by grid barriers instead of kernel
// boundaries.  The steps run the same device code as the separate launches
// (leaf body, row-swap strip, GEMM tile), so the factors are bit-identical;
// the difference is one dispatch instead of about seven per leaf, which is
// what a panel factored beside the trailing update waits on.
constexpr int SUB_W = 16;       // leaf width inside the sub-panel kernel
constexpr int SUB_WMAX = 256;   // widest sub-panel
constexpr int SUB_SWMAX = 128;  // widest row-swap strip (LDS: 2*SUB_W pairs x strip)
// the widest message is a 32-column FP64 leaf's
constexpr size_t SLOTS_BYTES = sizeof(unsigned long long) * 2 * (size_t)LEAF_GMAX * LeafMsg<double, 32>::NW;

template <typename T>
struct SubArgs {
    LeafArgs<T> leaf;            // first leaf: c = sub-panel start, seq_base of its first column
    int nb, w, sw;               // block size, sub-panel width, row-swap strip width
    T *wbuf, *tmp;               // h x h staging of the scaled rows; h x h product scratch
    unsigned long long *gbar;    // grid barrier arrivals (monotonic within a factorization)
    unsigned long long gbar_base;
};

// Barrier over the G co-resident workgroups: arrivals counted on one word,
// agent-scope fences on both sides so that every step's global writes (on
// any XCD) are visible to the next step.  Bounded: a timeout raises *err and
// lets every wave run to the end of the kernel.
__device__ __forceinline__ void grid_sync(unsigned long long *ctr, unsigned long long target, int *err)
{
    __syncthreads();
    if (threadIdx.x == 0) {
        __threadfence();
        __hip_atomic_fetch_add(ctr, 1ULL, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        unsigned long spins = 0;
        while (__hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) < target) {
            __builtin_amdgcn_s_sleep(1);
            if (((++spins) & 1023) == 0) {
                if (__hip_atomic_load(err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) break;
                if (spins > (1UL << 25)) {
                    __hip_atomic_store(err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    break;
                }
            }
        }
        __threadfence();
    }
    __syncthreads();
}

// C = alpha A B + beta C over the G workgroups in 64x64 tiles, each with the
// K range of the stand-alone GEMM's 128x128 tile that contains it
template <typename T, int EPI>
__device__ __forceinline__ void gemm_steps(int M, int N, int K, double alpha, const T *A, long lda, const T *B,
                                           long ldb, double beta, T *C, long ldc, int a_lower, int bid, int G,
                                           lu2mi_gemm::Tile64Smem<T> &ts)
{
    using namespace lu2mi_gemm;
    GemmDesc g;
    g.M = M; g.N = N; g.K = K; g.alpha = alpha; g.beta = beta;
    g.A = A; g.lda = lda; g.B = B; g.ldb = ldb; g.C = C; g.ldc = ldc; g.a_lower = a_lower;
    const int tiles_m = (M + BT64 - 1) / BT64, tiles_n = (N + BT64 - 1) / BT64;
    const int total = (M > 0 && N > 0) ? tiles_m * tiles_n : 0;
    for (int tile = bid; tile < total; tile += G) {
        const int m0 = (tile / tiles_n) * BT64, n0 = (tile % tiles_n) * BT64;
        const int Kt = a_lower ? min(K, (m0 & ~(BM - 1)) + BM) : K;
        const bool interior = (m0 + BT64 <= M) && (n0 + BT64 <= N) && (Kt % Mfma<T>::BK == 0);
        if (interior) gemm_tile64<T, false, EPI>(g, A, B, C, m0, n0, Kt, ts);
        else gemm_tile64<T, true, EPI>(g, A, B, C, m0, n0, Kt, ts);
        __syncthreads();   // the next tile restages the same LDS
    }
}

template <typename T, int RPT>
__global__ __launch_bounds__(NTL, 2) void subpanel_kernel(SubArgs<T> s)
{
    using namespace lu2mi_gemm;
    constexpr int W = SUB_W;
    __shared__ union {
        LeafSmem<T, W> leaf;
        Tile64Smem<T> tile;
        T perm[2 * W * SUB_SWMAX];
    } sm;
    const int bid = blockIdx.x, G = s.leaf.G;
    const int i = s.leaf.i, n = s.leaf.n, c0 = s.leaf.c, nb = s.nb, L = s.w / W;
    const long lda = s.leaf.lda;
    const int ldl = s.leaf.ldl;
    T *const A = s.leaf.A;
    T *const linv = s.leaf.linv;
    unsigned long long target = s.gbar_base;
    auto sync = [&]() __attribute__((always_inline)) {
        target += (unsigned long long)G;
        grid_sync(s.gbar, target, s.leaf.err);
    };
    // node (cn, 2h) after its left half: rows [cn, cn+h) of the right half
    // scaled by 1/d and staged, X = inv(D^-1 L11) * staged rows, then the
    // rows below (host path: Factor::panel)
    auto node_mid = [&](const int cn, const int h) __attribute__((always_inline)) {
        const long off = cn - i;
        for (long e = (long)bid * NTL + threadIdx.x; e < (long)h * h; e += (long)G * NTL) {
            const int r = (int)(e / h), col = (int)(e % h);
            s.wbuf[e] = A[(long)(cn + r) * lda + cn + h + col] * s.leaf.invd[cn + r];
        }
        sync();
        gemm_steps<T, EPI_SET>(h, h, h, 1.0, linv + off * ldl + off, ldl, s.wbuf, h, 0.0,
                               A + (long)cn * lda + cn + h, lda, 1, bid, G, sm.tile);
        sync();
        gemm_steps<T, EPI_SUB>(n - cn - h, h, h, -1.0, A + (long)(cn + h) * lda + cn, lda,
                               A + (long)cn * lda + cn + h, lda, 1.0, A + (long)(cn + h) * lda + cn + h, lda, 0,
                               bid, G, sm.tile);
        sync();
    };
    // node (cn, 2h) after its right half: X21 = -inv22 * L21 * inv11
    auto node_end = [&](const int cn, const int h) __attribute__((always_inline)) {
        const long off = cn - i;
        gemm_steps<T, EPI_SET>(h, h, h, 1.0, A + (long)(cn + h) * lda + cn, lda, linv + off * ldl + off, ldl, 0.0,
                               s.tmp, h, 0, bid, G, sm.tile);
        sync();
        gemm_steps<T, EPI_GENERAL>(h, h, h, -1.0, linv + (off + h) * ldl + off + h, ldl, s.tmp, h, 0.0,
                                   linv + (off + h) * ldl + off, ldl, 1, bid, G, sm.tile);
        sync();
    };
    // post-order walk: before leaf k the nodes whose right half ended at
    // leaf k-1 (deepest first) get their inverse block, then the node whose
    // left half ended there gets its right half updated
    for (int k = 0; k <= L; k++) {
        if (k > 0) {
            const int tz = __builtin_ctz(k);
            for (int lv = 1; lv <= tz; lv++) node_end(c0 + (k - (1 << lv)) * W, W << (lv - 1));
            if (k == L) break;
            node_mid(c0 + (k - (1 << tz)) * W, W << tz);
        }
        LeafArgs<T> la = s.leaf;
        la.c = c0 + k * W;
        la.seq_base = s.leaf.seq_base + (unsigned long long)k * W;
        leaf_body<T, W, RPT>(la, bid, sm.leaf);
        sync();
        // the leaf's swaps on the panel's other columns; its diagonal rows'
        // L part (columns left of the leaf) scaled by 1/d
        PermArgs<T> p;
        p.A = A; p.lda = lda; p.dst = la.pair_dst; p.src = la.pair_src; p.np = 2 * W;
        p.c0 = i; p.c1 = i + nb; p.k0 = la.c; p.k1 = la.c + W; p.sce = la.c; p.d0 = la.c; p.d1 = la.c + W;
        p.invd = la.invd; p.W = nullptr; p.ldw = 0; p.w0 = 0; p.w1 = 0; p.sw = s.sw;
        const int strips = (nb + s.sw - 1) / s.sw;
        for (int st = bid; st < strips; st += G) {
            rowperm_strip<T>(p, st, sm.perm);
            __syncthreads();
        }
        sync();
    }
}

// grid barriers one sub-panel launch of L leaves passes: two per leaf, three
// per node before its right half, two per node after it
__host__ __device__ constexpr int sub_barriers(int L) { return 2 * L + 5 * (L - 1); }
