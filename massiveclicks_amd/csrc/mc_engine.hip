// mc_engine.hip -- kernels and C ABI of the MI355X EM engine.
//
// Per EM iteration these kernels run on the model's stream (the held-out
// evaluation is in mc_eval.hip, the gradient path in mc_grad.hip):
//   em_item_kernel   E-step of one work item per workgroup, per-item
//                    reduction of the expected counts, in-place M-step of the
//                    entries the item owns (parallel_em/kernel.cu:42-89 and
//                    click_models/common.cu:114-192 fused); when every item
//                    has an LDS window, also the M-step of merged entries and
//                    of the shared (rank-indexed) tables;
//   em_merge_kernel  otherwise that M-step.
// theta_t is read from buffer `cur`, theta_{t+1} written to `cur ^ 1`, so the
// (1,2) reset of the reference (common.cu:71-82, a host fill plus H2D per
// iteration) disappears: the M-step writes prior + sum directly.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <numeric>
#include <string>
#include <thread>
#include <vector>

#include "mclicks.h"
#include "mc_internal.h"
#include "mc_kernels.h"
#include "mc_layout.h"
#include "mc_model.h"

namespace mc {

namespace {
thread_local std::string g_last_error;
}
void set_error(const std::string& msg) { g_last_error = msg; }

// ---------------------------------------------------------------------------
// Kernels
// ---------------------------------------------------------------------------

// Session code of lists of L ranks: LC > 0 a length known at compile time,
// 0 any (PBM and UBM).
template <int MODEL, int LC, class Src, class Emit>
__device__ __forceinline__ void run_session_len(const int (&pv)[kL], int len, uint32_t m, const Src& src, Emit& em,
                                                const float* sh, float (&acc)[55]) {
    constexpr bool VARLEN = LC < kL;
    const int L = LC > 0 ? LC : len;
    const uint32_t mm = m & ((1u << L) - 1u);
    if (MODEL == kPBM) {
        pbm_session(pv, L, mm, src, em, sh, acc);
    } else if (MODEL == kUBM) {
        ubm_session(pv, L, mm, src, em, sh, acc);
    } else if (MODEL == kDBN) {
        if (mm == 0) return;   // every count of a click-free session is a constant
        // The gamma and tau sums go straight into the lane's accumulators
        // (shared_sums gives them their factors at the end of the item).
        dbn_session<VARLEN>(pv, LC, mm, src, em, sh[0], acc[0], acc[1]);
    } else {
        if (mm == 0) return;
        ccm_session<VARLEN>(pv, LC, mm, src, em, sh[0], sh[1], sh[2], acc);
    }
}

// Uneven lists run the session code specialised for their length, so that
// every rank loop and tail index is static; sessions of a work item are
// ordered by length, so a wavefront mostly takes one case.  In items of few
// sessions a wavefront holds several lengths, whose cases run one after
// another.  The PBM and UBM, whose code for any length is as long as that for
// ten ranks, then run that once, and test the length per wavefront: 2M
// sessions, us per iteration with a case per lane / per wavefront: PBM 21.9 /
// 20.5, UBM 26.9 / 24.4.  The chains of the DBN and CCM need a static length
// for their tails (3M DBN sessions 26.7 us with a case per lane, 36.6 with
// general code for the mixed wavefronts).
template <int MODEL, bool VARLEN, class Src, class Emit>
__device__ __forceinline__ void run_session(const int (&pv)[kL], int L, uint32_t m, const Src& src, Emit& em,
                                            const float* sh, float (&acc)[55]) {
    if (!VARLEN) {
        run_session_len<MODEL, kL>(pv, kL, m, src, em, sh, acc);
        return;
    }
    constexpr bool general = MODEL == kPBM || MODEL == kUBM;
    int which = L;
    if (general) {
        const int first = __builtin_amdgcn_readfirstlane(L);
        which = __builtin_amdgcn_ballot_w64(L != first) ? 0 : first;
    }
    switch (which) {
        case 0:
            if (general) run_session_len<MODEL, 0>(pv, L, m, src, em, sh, acc);
            break;
        case 1: run_session_len<MODEL, 1>(pv, 1, m, src, em, sh, acc); break;
        case 2: run_session_len<MODEL, 2>(pv, 2, m, src, em, sh, acc); break;
        case 3: run_session_len<MODEL, 3>(pv, 3, m, src, em, sh, acc); break;
        case 4: run_session_len<MODEL, 4>(pv, 4, m, src, em, sh, acc); break;
        case 5: run_session_len<MODEL, 5>(pv, 5, m, src, em, sh, acc); break;
        case 6: run_session_len<MODEL, 6>(pv, 6, m, src, em, sh, acc); break;
        case 7: run_session_len<MODEL, 7>(pv, 7, m, src, em, sh, acc); break;
        case 8: run_session_len<MODEL, 8>(pv, 8, m, src, em, sh, acc); break;
        case 9: run_session_len<MODEL, 9>(pv, 9, m, src, em, sh, acc); break;
        default: run_session_len<MODEL, 10>(pv, 10, m, src, em, sh, acc); break;
    }
}

// One lane walks the sessions s0 + tid, s0 + tid + blockDim, ...; the
// indices of the next session are in flight while one is processed.  The
// first session is passed in already loaded.
template <int MODEL, bool VARLEN, bool WIN, class Src, class Emit>
__device__ __forceinline__ void run_item(const Stream& st, const Item& it, const Src& src, Emit& em, const float* sh,
                                         float (&acc)[55], uint32_t m, int L, int (&pv)[kL]) {
    const int nthr = blockDim.x;
    if (VARLEN) {
        // Two-stage prefetch: the length of session s + 2 nthr arrives one
        // session ahead of its indices, which are read only up to it.
        uint32_t mn;
        int Ln;
        load_head(st, it.s0 + (int)threadIdx.x + nthr, it.e1, mn, Ln);
        for (int s = it.s0 + (int)threadIdx.x; s < it.e1; s += nthr) {
            uint32_t m3;
            int L3;
            int pv2[kL];
            load_head(st, s + 2 * nthr, it.e1, m3, L3);
            load_pidx_upto<WIN>(st, s + nthr, it.e1, Ln, pv2);
            run_session<MODEL, VARLEN>(pv, L, m, src, em, sh, acc);
            m = mn;
            L = Ln;
            mn = m3;
            Ln = L3;
#pragma unroll
            for (int r = 0; r < kL; r++) pv[r] = pv2[r];
        }
        return;
    }
    for (int s = it.s0 + (int)threadIdx.x; s < it.e1; s += nthr) {
        uint32_t m2;
        int L2;
        int pv2[kL];
        load_session<VARLEN, WIN>(st, s + nthr, it.e1, m2, L2, pv2);
        run_session<MODEL, VARLEN>(pv, L, m, src, em, sh, acc);
        m = m2;
        L = L2;
#pragma unroll
        for (int r = 0; r < kL; r++) pv[r] = pv2[r];
    }
}

// run_item for packed items: one 16-byte record per session; the next
// session's record is in flight while one is processed (4 registers
// instead of the 12 of a rank-major session).
template <int MODEL, bool VARLEN, class Src, class Emit>
__device__ __forceinline__ void run_item_packed(const Stream& st, const Item& it, const Src& src, Emit& em,
                                                const float* sh, float (&acc)[55], PackedSession cur) {
    const int nthr = blockDim.x;
    for (int s = it.s0 + (int)threadIdx.x; s < it.e1; s += nthr) {
        const PackedSession nxt = load_packed(st, s + nthr, it.e1);
        uint32_t m;
        int L;
        int pv[kL];
        decode_packed<VARLEN>(cur, m, L, pv);
        run_session<MODEL, VARLEN>(pv, L, m, src, em, sh, acc);
        cur = nxt;
    }
}

// Direct items: every session is the only one of its query, so its entries
// receive no other counts; the lane writes theta_{t+1} of its entries itself.
template <int MODEL, bool VARLEN, class Src>
__device__ __forceinline__ void run_item_direct(const KArgs& A, const Stream& st, const Item& it, const Src& src,
                                                const float* sh, float (&acc)[55], uint32_t m, int L,
                                                int (&pv)[kL]) {
    constexpr int T = Shape<MODEL>::T;
    const int nthr = blockDim.x;
    for (int s = it.s0 + (int)threadIdx.x; s < it.e1; s += nthr) {
        uint32_t m2;
        int L2;
        int pv2[kL];
        load_session<VARLEN, false>(st, s + nthr, it.e1, m2, L2, pv2);
        EmitRegs em;
        em.clear();
        run_session<MODEL, VARLEN>(pv, L, m, src, em, sh, acc);
#pragma unroll
        for (int r = 0; r < kL; r++) {
            if (!VARLEN || r < L) {
                const int p = pv[r];
                const int2 oc = A.counts[p];
#pragma unroll
                for (int t = 0; t < T; t++) {
                    const float2 bd = base_den<MODEL>(t, oc);
                    const float num = bd.x + em.x[t][r];
                    A.tab[t].val_out[p] = clamp_value(num, bd.y);
                    if (A.write_num) A.tab[t].num_out[p] = num;
                }
            }
        }
        m = m2;
        L = L2;
#pragma unroll
        for (int r = 0; r < kL; r++) pv[r] = pv2[r];
    }
}

// Cross-workgroup hand-over inside one launch (fused M-step).  The data
// handed over (fixed-point sums, counters) is only ever written with
// device-scope atomics, which are performed at the device's coherence point;
// so the writer only has to wait until its atomics have completed before it
// bumps a counter (an agent-scope release fence would also write back the
// XCD's L2 for plain stores, which nothing here needs and which cost 4x the
// kernel's time), and the reader reads with device-coherent loads.
__device__ __forceinline__ void wait_memory() { __builtin_amdgcn_s_waitcnt(0); }

__device__ __forceinline__ unsigned long long load_acc(const unsigned long long* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// M-step of the shared (rank-indexed) tables from their fixed-point sums and
// FP64 bases, threads tid < K; then the accumulators are cleared for the next
// iteration.  COHERENT: the sums were added during this launch.
template <bool COHERENT>
__device__ __forceinline__ void finalize_shared(const KArgs& A, int tid, int nthr, unsigned long long* tot) {
    for (int j = tid; j < A.kacc; j += nthr) tot[j] = 0ull;
    __syncthreads();
    for (int j = tid & (kShStride - 1); j < A.kacc; j += kShStride) {   // one pass: kacc <= kShStride
        for (int c = tid / kShStride; c < A.sh_parts; c += 8 * (nthr / kShStride)) {
            unsigned long long v[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int cu = c + u * (nthr / kShStride);
                unsigned long long* p = &A.sh_acc[cu * kShStride + j];
                v[u] = cu < A.sh_parts ? (COHERENT ? load_acc(p) : *p) : 0ull;
            }
            unsigned long long w = 0ull;
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int cu = c + u * (nthr / kShStride);
                w += v[u];
                if (v[u] != 0ull) A.sh_acc[cu * kShStride + j] = 0ull;
            }
            if (w != 0ull) atomicAdd(&tot[j], w);
        }
    }
    __syncthreads();
    const int k = tid;
    if (k < A.K) {
        const int an = A.sh_acc_map[2 * k], ad = A.sh_acc_map[2 * k + 1];
        const long long tn = an >= 0 ? (long long)tot[an] : 0;
        const long long td = ad >= 0 ? (long long)tot[ad] : 0;
        const float num = (float)(A.sh_base[2 * k] + (double)tn * kFixInv);
        const float den = (float)(A.sh_base[2 * k + 1] + (double)td * kFixInv);
        A.sh_num_out[k] = num;
        A.sh_den_out[k] = den;
        A.sh_val_out[k] = clamp_value(num, den);
    }
}

// M-step of a per-qd entry whose sums several work items added to gacc; the
// accumulators are cleared for the next iteration.
template <int MODEL, bool COHERENT>
__device__ __forceinline__ void finalize_merged_entry(const KArgs& A, int p) {
    constexpr int T = Shape<MODEL>::T;
    const int2 oc = A.counts[p];
#pragma unroll
    for (int t = 0; t < T; t++) {
        const float2 bd = base_den<MODEL>(t, oc);
        const unsigned long long v = COHERENT ? load_acc(&A.tab[t].gacc[p]) : A.tab[t].gacc[p];
        const float num = fix_to_float(bd.x, v);
        A.tab[t].val_out[p] = clamp_value(num, bd.y);
        if (A.write_num) A.tab[t].num_out[p] = num;
        A.tab[t].gacc[p] = 0ull;
    }
}

// Counting finished work items in two levels: `c[0]` counts the `parts`
// counters, c[(1 + p) * kDoneStride] the items p, p + parts, ... of n.
// done_first counts an item in counter `part` and returns whether that
// counter is complete; done_last then counts the counter.  One address takes
// about 13 ns per atomic, so a single counter would serialise the end of a
// launch of thousands of workgroups.
__device__ __forceinline__ bool done_first(unsigned* c, unsigned parts, unsigned part, unsigned n) {
    if (parts == 1u) return true;
    return atomicAdd(&c[(1u + part) * kDoneStride], 1u) == (n - part + parts - 1u) / parts - 1u;
}
__device__ __forceinline__ bool done_last(unsigned* c, unsigned parts, unsigned part, unsigned n) {
    if (parts > 1u) c[(1u + part) * kDoneStride] = 0u;
    const bool last = atomicAdd(c, 1u) == (parts > 1u ? min(parts, n) : n) - 1u;
    if (last) c[0] = 0u;
    return last;
}

// Accumulators of the slice's split group in table t (fused M-step).
__device__ __forceinline__ unsigned long long* split_target(const KArgs& A, const SplitGroup& g, int slice, int t) {
    return A.split_acc + (int64_t)t * A.n_split_acc + g.acc + (int64_t)(slice & (g.parts - 1)) * (g.hi - g.lo);
}

// M-step of a split group's entries from the copies of their sums.
template <int MODEL>
__device__ __forceinline__ void finalize_split_group(const KArgs& A, const SplitGroup& g, int tid, int nthr) {
    constexpr int T = Shape<MODEL>::T;
    const int W = g.hi - g.lo;
    for (int i = tid; i < W; i += nthr) {
        const int p = g.lo + i;
        const int2 oc = A.counts[p];
#pragma unroll
        for (int t = 0; t < T; t++) {
            unsigned long long* a = A.split_acc + (int64_t)t * A.n_split_acc + g.acc + i;
            const float2 bd = base_den<MODEL>(t, oc);
            unsigned long long v = 0ull;
            for (int c = 0; c < g.parts; c++) v += load_acc(a + (int64_t)c * W);
            for (int c = 0; c < g.parts; c++) a[(int64_t)c * W] = 0ull;
            const float num = fix_to_float(bd.x, v);
            A.tab[t].val_out[p] = clamp_value(num, bd.y);
            if (A.write_num) A.tab[t].num_out[p] = num;
        }
    }
}

// Fused M-step at the end of work item `item`, all of whose sums are on their
// way: the workgroup that completes its item's split group finalises the
// group's entries, the last of the iteration's A.n_items items the shared
// tables.  Block-uniform call; `flag` is a shared int, `tot` shared scratch
// of kacc sums.
template <int MODEL>
__device__ __forceinline__ void fused_merge(const KArgs& A, int item, const Item& it, int tid, int nthr, int& flag,
                                            unsigned long long* tot) {
    const int split = it.split, slice = it.flags >> kItemSliceShift;
    SplitGroup g{};
    if (split >= 0) g = A.split_groups[split];
    wait_memory();
    __syncthreads();
    if (tid == 0) {
        const unsigned n = (unsigned)A.n_items, parts = (unsigned)A.sh_parts, part = (unsigned)item & (parts - 1u);
        const unsigned gparts = (unsigned)g.parts, gpart = (unsigned)slice & (gparts - 1u);
        bool a = done_first(A.grid_done, parts, part, n);
        bool b = split >= 0 && done_first(A.split_done + g.done, gparts, gpart, (unsigned)g.slices);
        if (a) a = done_last(A.grid_done, parts, part, n);
        if (b) b = done_last(A.split_done + g.done, gparts, gpart, (unsigned)g.slices);
        flag = (a ? 1 : 0) | (b ? 2 : 0);
    }
    __syncthreads();
    const int f = flag;
    if (f & 2) finalize_split_group<MODEL>(A, g, tid, nthr);
    if (f & 1) finalize_shared<true>(A, tid, nthr, tot);
}

// Sums of the lanes' shared-table accumulators over the workgroup, in fixed
// point (order-independent integer adds), one atomic per accumulator into the
// workgroup's copy.  `red` holds KACC x NWMAX.
template <int KACC, int NWMAX>
__device__ __forceinline__ void add_shared_sums(const KArgs& A, int item, const float (&acc)[55], long long (&red)[KACC][NWMAX],
                                                int tid, int nthr) {
    const int wave = tid >> 6, lane = tid & 63, nwave = nthr >> 6;
#pragma unroll
    for (int k = 0; k < KACC; k++) {
        const long long v = wave_sum_last(to_fix(acc[k]));
        if (lane == 63) red[k][wave] = v;
    }
    __syncthreads();
    for (int k = tid; k < KACC; k += nthr) {
        long long v = 0;
        for (int w = 0; w < nwave; w++) v += red[k][w];
        if (v != 0)
            atomicAdd(&A.sh_acc[(item & (A.sh_parts - 1)) * kShStride + k], (unsigned long long)v);
    }
}

// The same through LDS slots (fixed-point window paths): every lane adds its
// sums to its copy of the slots, then eight lanes add up each slot's copies.
// The UBM's lanes hold only the rows' "no earlier click" sums, its sessions
// add to the other slots themselves.  One LDS atomic per sum and wavefront:
// wavefront sums by DPP take about 24 VALU instructions per sum instead, a
// tenth of the launch (per iteration, with DPP / with slots: 2M CCM sessions
// 32.7 / 28.8 us, 8M PBM 62.4 / 56.1, 8M DBN 80.0 / 77.9).
template <int MODEL>
__device__ __forceinline__ void add_shared_slots(const KArgs& A, int item, const float (&acc)[55], unsigned long long* slots,
                                                 int tid, int nthr) {
    constexpr int KACC = Shape<MODEL>::KACC;
    unsigned long long* mine = slots + (tid & (kSlotCopies - 1));
#pragma unroll
    for (int r = 0; r < (MODEL == kUBM ? kL : KACC); r++) {
        const int k = MODEL == kUBM ? r * (r + 1) / 2 + kL - 1 : r;
        if (MODEL != kUBM || acc[k] != 0.f) atomicAdd(&mine[k * kSlotCopies], (unsigned long long)to_fix(acc[k]));
    }
    __syncthreads();
    for (int q = tid; q < (KACC + 7) / 8 * 64; q += nthr) {
        const int k = q >> 3, c = q & 7;
        long long v = 0;
        if (k < KACC)
#pragma unroll
            for (int j = 0; j < kSlotCopies / 8; j++) v += (long long)slots[k * kSlotCopies + c + 8 * j];
        v = sum_of_eight(v);
        if (c == 0 && v != 0)
            atomicAdd(&A.sh_acc[(item & (A.sh_parts - 1)) * kShStride + k], (unsigned long long)v);
    }
}

// Session paths, one kernel instantiation each (each gets its own register
// allocation): window items in LDS (rank-major or packed sessions), items
// without a window (global 64-bit fixed-point atomics), and the float-atomic
// mode.
enum { kPathLds = 0, kPathGlobal = 1, kPathAtomic = 2, kPathDirect = 3, kPathLdsFloat = 4, kPathPacked = 5 };

// E-step and in-item M-step of one work item (item index item_offset +
// blockIdx.x).  Bound by the VALU on large sets (8M sessions, instructions at
// four cycles of the launch: DBN 58 of 76 us, CCM 67 of 73), by the latency
// of the rare queries' items on medium ones and by the chain of load,
// session, flush and counter round trips on small ones (32,000 PBM sessions:
// 5 us of 7.4, the launch gap included).  At 37-64 VGPRs the packed paths
// keep 32 wavefronts on a CU, and the hardware hands each freed slot the next
// item: a persistent form with a fixed item list per workgroup held the next
// item's window in 77-103 VGPRs and took 87 us on 8M DBN sessions where this,
// with the same session code, took 82.  Dynamic LDS (window path): width x T
// fixed-point accumulators (AccWindow), then width x T staged values of
// theta_t, interleaved per entry, then the UBM's slots.  kPathLdsFloat (float-atomic mode) pre-reduces in
// float LDS accumulators and adds every window entry to global float
// accumulators, which the merge kernel finalises.
template <int MODEL, bool VARLEN, int PATH>
__global__ void __launch_bounds__(512) em_item_kernel(KArgs A, int item_offset) {
    constexpr int T = Shape<MODEL>::T;
    constexpr int K = Shape<MODEL>::K;
    constexpr int KACC = Shape<MODEL>::KACC;
    extern __shared__ unsigned long long lds[];
    __shared__ float sh[K < 64 ? 64 : K];
    __shared__ long long red[KACC][PATH == kPathLds || PATH == kPathPacked ? 1 : 8];
    __shared__ int last_one;

    const int item = item_offset + (int)blockIdx.x;
    const Item it = A.items[item];
    const int tid = threadIdx.x;
    const int nthr = blockDim.x;
    const int W = it.width;
    constexpr bool fwin = PATH == kPathLdsFloat;
    constexpr bool packed = PATH == kPathPacked;
    constexpr bool fixwin = PATH == kPathLds || packed;   // fixed-point LDS window
    constexpr bool win = fixwin || fwin;
    unsigned long long* lacc = lds;
    float* facc = (float*)lds;
    // Fixed-point windows take max_width slots per table (copies of the
    // entries of narrow windows), then the staged values.
    const int Wmax = A.max_width;
    const AccWindow<T> aw{lacc, Wmax, fixwin ? acc_copies_log2(W, Wmax) : 0};
    const int WS = W << aw.rsh;
    float* lval = fwin ? facc + T * W : (float*)(lds + T * Wmax);
    // Slots of the shared tables' sums: the UBM's after the window.
    constexpr bool lslots = fixwin;
    __shared__ unsigned long long few[lslots && MODEL != kUBM ? KACC * kSlotCopies : 1];
    unsigned long long* slots = MODEL == kUBM ? lds + ((size_t)T * Wmax * 12 + 7) / 8 : few;

    // First session's loads go out before the window is staged.
    const Stream st = make_stream(A);
    uint32_t m0 = 0;
    int L0 = 0;
    int pv0[kL];
    PackedSession r0;
    if (packed) r0 = load_packed(st, it.s0 + tid, it.e1);
    else load_session<VARLEN, win>(st, it.s0 + tid, it.e1, m0, L0, pv0);
    float shv = tid < K ? A.sh_val_in[tid] : 0.f;
    if (win) {
        // Three entries' values per lane and pass in flight together, the
        // first pass's while the accumulators are cleared (1-2 % faster than
        // one at a time).
        constexpr int U = 3;
        for (int i0 = 0; i0 < W; i0 += U * nthr) {
            float v[U][T];
#pragma unroll
            for (int u = 0; u < U; u++) {
                if (i0 + u * nthr >= W) break;
                const int i = min(i0 + u * nthr + tid, W - 1);
#pragma unroll
                for (int t = 0; t < T; t++) v[u][t] = A.tab[t].val_in[it.base + i];
            }
            if (i0 == 0) {
                if (fwin) {
                    for (int i = tid; i < W * T; i += nthr) facc[i] = 0.f;
                } else {
                    for (int i = tid; i < WS; i += nthr)
#pragma unroll
                        for (int t = 0; t < T; t++) lacc[aw.slot(t, i)] = 0ull;
                }
                if (lslots)
                    for (int i = tid; i < KACC * kSlotCopies; i += nthr) slots[i] = 0ull;
            }
#pragma unroll
            for (int u = 0; u < U; u++) {
                const int i = i0 + u * nthr + tid;
                if (i0 + u * nthr >= W) break;
#pragma unroll
                for (int t = 0; t < T; t++)
                    if (i < W) lval[i * T + t] = v[u][t];
            }
        }
    }
    if (tid < K) sh[tid] = shv;
    __syncthreads();

    float acc[55];
#pragma unroll
    for (int k = 0; k < 55; k++) acc[k] = 0.f;

    const SrcGlobal gsrc{A.tab[0].val_in, A.tab[1].val_in};
    if (PATH == kPathAtomic) {
        EmitGlobalFloat em{A.tab[0].gaccf, A.tab[1].gaccf};
        run_item<MODEL, VARLEN, false>(st, it, gsrc, em, sh, acc, m0, L0, pv0);
    } else if (fixwin) {
        EmitLds<T> em{aw, tid & ((1 << aw.rsh) - 1), slots + (tid & (kSlotCopies - 1))};
        const SrcLds<T> lsrc{lval};
        if (packed) run_item_packed<MODEL, VARLEN>(st, it, lsrc, em, sh, acc, r0);
        else run_item<MODEL, VARLEN, true>(st, it, lsrc, em, sh, acc, m0, L0, pv0);
    } else if (PATH == kPathLdsFloat) {
        EmitLdsFloat<T> em{facc};
        const SrcLds<T> lsrc{lval};
        run_item<MODEL, VARLEN, true>(st, it, lsrc, em, sh, acc, m0, L0, pv0);
    } else if (PATH == kPathDirect) {
        run_item_direct<MODEL, VARLEN>(A, st, it, gsrc, sh, acc, m0, L0, pv0);
    } else {
        EmitGlobalFix em{A.tab[0].gacc, A.tab[1].gacc};
        run_item<MODEL, VARLEN, false>(st, it, gsrc, em, sh, acc, m0, L0, pv0);
    }

    // Shared tables (also the barrier before the window is flushed).
    shared_sums<MODEL>(sh, acc);
    if constexpr (lslots) add_shared_slots<MODEL>(A, item, acc, slots, tid, nthr);
    else add_shared_sums<KACC>(A, item, acc, red, tid, nthr);

    if (fwin) {
        for (int i = tid; i < W; i += nthr) {
#pragma unroll
            for (int t = 0; t < T; t++) {
                const float v = facc[i * T + t];
                if (v != 0.f) unsafeAtomicAdd(&A.tab[t].gaccf[it.base + i], v);
            }
        }
    }
    // Flush the LDS window, four entries per thread per pass with the
    // constant loads issued together.
    if (fixwin) {
        const bool interior = (it.flags & kItemInterior) != 0;
        unsigned long long* sink[T];
#pragma unroll
        for (int t = 0; t < T; t++)
            sink[t] = (A.fuse_merge && it.split >= 0)
                          ? split_target(A, A.split_groups[it.split], it.flags >> kItemSliceShift, t)
                          : A.tab[t].gacc + it.base;
        for (int i0 = 0; i0 < W; i0 += 4 * nthr) {
            uint32_t pk[4];
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = i0 + u * nthr + tid;
                pk[u] = (interior && i < W) ? A.counts16[it.base + i] : 0u;
            }
#pragma unroll
            for (int u = 0; u < 4; u++) {
                const int i = i0 + u * nthr + tid;
                if (i >= W) continue;
                const int p = it.base + i;
                const int2 oc = interior ? unpack_counts(pk[u], A.counts, p) : make_int2(0, 0);
#pragma unroll
                for (int t = 0; t < T; t++) {
                    const unsigned long long v = aw.sum(t, i);
                    if (interior) {
                        const float2 bd = base_den<MODEL>(t, oc);
                        const float num = fix_to_float(bd.x, v);
                        A.tab[t].val_out[p] = clamp_value(num, bd.y);
                        if (A.write_num) A.tab[t].num_out[p] = num;
                    } else if (v != 0ull) {
                        atomicAdd(&sink[t][i], v);
                    }
                }
            }
        }
    }
    if (A.fuse_merge) fused_merge<MODEL>(A, item, it, tid, nthr, last_one, (unsigned long long*)red);
}

// Merge kernel: block 0 finalises the shared tables, the other blocks
// finalise per-qd entries accumulated in global memory (entries merged across
// items in segmented mode, every entry in atomic mode).
template <int MODEL>
__global__ void __launch_bounds__(256) em_merge_kernel(KArgs A) {
    constexpr int T = Shape<MODEL>::T;
    const int tid = threadIdx.x;
    if (blockIdx.x == 0) {
        __shared__ unsigned long long tot[kShStride];
        finalize_shared<false>(A, tid, (int)blockDim.x, tot);
        return;
    }
    const int64_t i = (int64_t)(blockIdx.x - 1) * blockDim.x + tid;
    if (A.mode == 1) {
        if (i >= A.n_qd) return;
        const int2 oc = A.counts[i];
#pragma unroll
        for (int t = 0; t < T; t++) {
            const float2 bd = base_den<MODEL>(t, oc);
            const float v = A.tab[t].gaccf[i];
            const float num = (float)((double)bd.x + (double)v);
            A.tab[t].val_out[i] = clamp_value(num, bd.y);
            if (A.write_num) A.tab[t].num_out[i] = num;
            A.tab[t].gaccf[i] = 0.f;
        }
    } else {
        if (i >= A.n_shared) return;
        finalize_merged_entry<MODEL, false>(A, A.shared_idx[i]);
    }
}

// Copies n 4-byte words to pinned host memory, 16 bytes a lane.
__global__ void __launch_bounds__(256) copy_out_kernel(const uint32_t* src, uint32_t* out, int64_t n) {
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (4 * i + 4 <= n) reinterpret_cast<uint4*>(out)[i] = reinterpret_cast<const uint4*>(src)[i];
    else
        for (int64_t j = 4 * i; j < n; j++) out[j] = src[j];
}

// Fills a float array with a constant (used instead of memsets so that the
// same code is safe inside captured graphs).
__global__ void fill_kernel(float* p, float v, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

// reset_parameters in one launch: every per-qd entry and the shared table
// (the last workgroup) to (1, 2), value 1/2.
struct ResetArgs {
    float *val[2], *num[2];
    float *sh_val, *sh_num, *sh_den;
    int64_t n_qd;
    int32_t T, K;
};
__global__ void __launch_bounds__(256) reset_kernel(ResetArgs R) {
    if (blockIdx.x == gridDim.x - 1) {
        if ((int)threadIdx.x < R.K) {
            R.sh_val[threadIdx.x] = 0.5f;
            R.sh_num[threadIdx.x] = 1.f;
            R.sh_den[threadIdx.x] = 2.f;
        }
        return;
    }
    const int64_t i = 4 * ((int64_t)blockIdx.x * blockDim.x + threadIdx.x);
    for (int t = 0; t < R.T; t++) {
        if (i + 4 <= R.n_qd) {
            *reinterpret_cast<float4*>(R.val[t] + i) = make_float4(0.5f, 0.5f, 0.5f, 0.5f);
            *reinterpret_cast<float4*>(R.num[t] + i) = make_float4(1.f, 1.f, 1.f, 1.f);
        } else {
            for (int64_t j = i; j < R.n_qd; j++) {
                R.val[t][j] = 0.5f;
                R.num[t][j] = 1.f;
            }
        }
    }
}

}  // namespace mc

// ===========================================================================
// Host side
// ===========================================================================
using namespace mc;

namespace mc {

const char* table_name(int type, int t) {
    switch (type) {
        case MC_PBM: return t == 0 ? "attractiveness" : "examination";
        case MC_UBM: return t == 0 ? "attractiveness" : "examination";
        case MC_CCM: return t == 0 ? "attractiveness" : "continuation";
        case MC_DBN: return t == 0 ? "attractiveness" : (t == 1 ? "satisfaction" : "continuation");
    }
    return "?";
}

void release(mc_model* m) {
    if (m->adam_graph) { (void)hipGraphExecDestroy(m->adam_graph); m->adam_graph = nullptr; }
    m->grad_ready = false;
    for (int b = 0; b < 2; b++)
        if (m->graph[b]) { (void)hipGraphExecDestroy(m->graph[b]); m->graph[b] = nullptr; }
    for (void* p : m->allocations) (void)hipFree(p);
    m->allocations.clear();
    m->mem_bytes = 0;
    // What later calls allocate when they first need it.
    for (float*& d : m->d_den_user) d = nullptr;
    m->d_test_packed = nullptr;
    m->d_test_pidx = nullptr;
    m->d_test_mask = nullptr;
    m->d_test_len = nullptr;
    m->d_test_perm = nullptr;
    m->d_test_part = nullptr;
    m->d_eval_part = nullptr;
    m->n_test = 0;
    m->test_bytes = 0;
    m->initialized = false;
}

mc_status stage_reserve(mc_model* m, size_t bytes) {
    for (hipEvent_t& e : m->stage_ev)
        if (!e) MC_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    if (bytes <= m->stage_cap) return MC_OK;
    m->stage_cap = 0;
    if (m->stage[0]) MC_HIP(hipHostFree(m->stage[0]));
    m->stage[0] = nullptr;
    const size_t step = (bytes + 255) / 256 * 256;
    const hipError_t e = hipHostMalloc((void**)&m->stage[0], step * kStages, hipHostMallocCoherent);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        m->stage[0] = nullptr;
        set_error("hipHostMalloc of " + std::to_string(step * kStages) + " bytes failed: " + hipGetErrorString(e));
        return e == hipErrorOutOfMemory ? MC_ERR_OOM : MC_ERR_HIP;
    }
    for (int k = 1; k < kStages; k++) m->stage[k] = m->stage[0] + (size_t)k * step;
    m->stage_cap = bytes;
    return MC_OK;
}

namespace {
// Host array of n bytes from chunks that produce(dst, offset, bytes) enqueues
// into pinned memory; beside(offset, bytes) is the host's own work for the
// same range, done while the chunk is on its way.  The copies out of the
// pinned chunks are spread over a few threads: the destination is usually
// fresh memory, whose page faults cost one thread more than the link does.
// Numerators and denominators of a table into new numpy arrays, us by the
// runtime's pageable copy and a loop over the counts / so: 2,000 entries 21 /
// 18, 90,000 38 / 35, 250,000 83 / 68, 4M 1,900 / 490.  (Denominators by a
// kernel and a second pass: 31, 56, 101 and 840.)
constexpr size_t kStageChunk = (size_t)1 << 20;
constexpr size_t kStageSmallChunk = (size_t)256 << 10;
constexpr size_t kStageThreadsFrom = (size_t)8 << 20;   // below, starting threads costs more than they save
// One chunk up to 1 MB: an event costs as much as the overlap saves (130,000
// entries 42 us in one chunk, 46 in two; 250,000 68, 79 in four).  About four
// chunks of a somewhat larger array, so that copies overlap.
size_t stage_chunk(size_t n) {
    if (n <= kStageChunk) return n;
    return std::min(kStageChunk, std::max(kStageSmallChunk, (n / 4 + 255) / 256 * 256));
}
// Bytes of each of the kStages slots, which lie side by side: a single chunk
// takes as many of them as it needs.
size_t stage_slot(size_t n) { return n <= kStageChunk ? (n + kStages - 1) / kStages : stage_chunk(n); }
template <class Produce, class Beside>
mc_status staged_out(mc_model* m, char* dst, size_t n, Produce produce, Beside beside) {
    if (n == 0) return MC_OK;
    const size_t chunk = stage_chunk(n);
    MC_TRY(stage_reserve(m, stage_slot(n)));
    const size_t chunks = (n + chunk - 1) / chunk;
    auto size_of = [&](size_t k) { return std::min(chunk, n - k * chunk); };
    auto copy_here = [&]() -> mc_status {   // by this thread alone
        for (size_t k = 0; k < chunks + kStages - 1; k++) {
            if (k < chunks) {
                MC_TRY(produce(m->stage[k % kStages], k * chunk, size_of(k)));
                if (k + 1 < chunks) MC_HIP(hipEventRecord(m->stage_ev[k % kStages], m->stream));
                beside(k * chunk, size_of(k));
            }
            if (k + 1 < kStages) continue;
            const size_t j = k + 1 - kStages;
            // The stream's end instead of the last event: the next call's
            // first launch otherwise takes 20 us longer.
            if (j + 1 < chunks) MC_HIP(hipEventSynchronize(m->stage_ev[j % kStages]));
            else MC_HIP(hipStreamSynchronize(m->stream));
            std::memcpy(dst + j * chunk, m->stage[j % kStages], size_of(j));
        }
        return MC_OK;
    };
    if (n < kStageThreadsFrom) return copy_here();
    std::atomic<size_t> issued{0}, freed[kStages];
    std::atomic<int> error{(int)hipSuccess};
    for (auto& x : freed) x = 0;
    // Worker w of W copies chunks w, w + W, ...; chunk k is in slot
    // k % kStages, whose use number is k / kStages.
    auto work = [&](size_t w, size_t W) {
        for (size_t k = w; k < chunks; k += W) {
            beside(k * chunk, size_of(k));
            while (issued.load(std::memory_order_acquire) <= k) {
                if (error.load() != (int)hipSuccess) return;
                std::this_thread::yield();
            }
            const hipError_t e = hipEventSynchronize(m->stage_ev[k % kStages]);
            if (e != hipSuccess) {
                error = (int)e;
                return;
            }
            std::memcpy(dst + k * chunk, m->stage[k % kStages], size_of(k));
            freed[k % kStages].store(k / kStages + 1, std::memory_order_release);
        }
    };
    auto issue = [&](size_t k) -> mc_status {
        while (freed[k % kStages].load(std::memory_order_acquire) < k / kStages) {
            if (error.load() != (int)hipSuccess) MC_HIP((hipError_t)error.load());
            std::this_thread::yield();
        }
        MC_TRY(produce(m->stage[k % kStages], k * chunk, size_of(k)));
        MC_HIP(hipEventRecord(m->stage_ev[k % kStages], m->stream));
        issued.store(k + 1, std::memory_order_release);
        return MC_OK;
    };
    const size_t want = std::min<size_t>(kStageThreads, chunks);
    std::vector<std::thread> team;
    try {
        team.reserve(want);
        for (size_t w = 0; w < want; w++) team.emplace_back(work, w, want);
    } catch (...) {   // no thread to be had: end those there are, copy here
        error = (int)hipErrorUnknown;
        for (auto& t : team) t.join();
        return copy_here();
    }
    mc_status st = MC_OK;
    for (size_t k = 0; k < chunks && st == MC_OK; k++) st = issue(k);
    if (st != MC_OK && error.load() == (int)hipSuccess) error = (int)hipErrorUnknown;
    for (auto& t : team) t.join();
    if (st == MC_OK) MC_HIP((hipError_t)error.load());
    return st;
}

// Enqueues a copy of a chunk.
mc_status copy_out(mc_model* m, const void* src, char* to, size_t at, size_t bytes) {
    const int64_t words = (int64_t)(bytes / 4);
    hipLaunchKernelGGL(copy_out_kernel, dim3((unsigned)((words + 1023) / 1024)), dim3(256), 0, m->stream,
                       (const uint32_t*)((const char*)src + at), (uint32_t*)to, words);
    MC_HIP(hipGetLastError());
    return MC_OK;
}

// Denominators of per-qd table t after an M-step, as base_den in the kernels:
// entries [first, first + n).
void constant_den(const mc_model* m, int t, float* out, size_t first, size_t n) {
    // All from the packed counts, then those that do not fit there.
    const int kind = m->type == MC_CCM ? 2 : m->type == MC_DBN && t == 1 ? 1 : 0;
    auto den = [kind](int o, int c) {
        return kind == 2 ? 2.f + (float)o + (float)c : kind == 1 ? 2.f + 2.f * (float)o - (float)c : 2.f + (float)o;
    };
    const uint16_t* c = m->h_counts16.data();
    if (kind == 2)
        for (size_t i = first; i < first + n; i++) out[i] = 2.f + (float)(c[i] & 0xff) + (float)(c[i] >> 8);
    else if (kind == 1)
        for (size_t i = first; i < first + n; i++) out[i] = 2.f + 2.f * (float)(c[i] & 0xff) - (float)(c[i] >> 8);
    else
        for (size_t i = first; i < first + n; i++) out[i] = 2.f + (float)(c[i] & 0xff);
    auto big = std::lower_bound(m->h_big_counts.begin(), m->h_big_counts.end(), first,
                                [](const mc_model::BigCount& b, size_t p) { return (size_t)b.entry < p; });
    for (; big != m->h_big_counts.end() && (size_t)big->entry < first + n; ++big)
        out[big->entry] = den(big->counts.x, big->counts.y);
}
}  // namespace

mc_status download(mc_model* m, void* dst, const void* src, size_t n) {
    return staged_out(
        m, (char*)dst, n, [&](char* to, size_t at, size_t bytes) { return copy_out(m, src, to, at, bytes); },
        [](size_t, size_t) {});
}

mc_status fill(mc_model* m, float* p, float v, int64_t n) {
    if (n <= 0) return MC_OK;
    hipLaunchKernelGGL(fill_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, m->stream, p, v, n);
    MC_HIP(hipGetLastError());
    return MC_OK;
}

}  // namespace mc

namespace {

void shape_of(int type, int* T, int* K, int* KACC) {
    switch (type) {
        case MC_PBM: *T = 1; *K = 10; *KACC = 10; break;
        case MC_UBM: *T = 1; *K = 55; *KACC = 55; break;
        case MC_DBN: *T = 2; *K = 1; *KACC = 2; break;
        default: *T = 1; *K = 3; *KACC = 6; break;
    }
}

KArgs make_args(mc_model* m, int cur, int write_num) {
    KArgs A;
    std::memset(&A, 0, sizeof(A));
    A.packed = m->d_packed;
    A.pidx16 = m->d_pidx16;
    A.pidx = m->d_pidx;
    A.mask = m->d_mask;
    A.len = m->varlen ? m->d_len : nullptr;
    A.N = m->N;
    A.n_w = m->n_w;
    A.n_pk = m->n_pk;
    A.items = m->d_items;
    A.n_items = m->n_items;
    A.mode = m->reduce_mode;
    for (int t = 0; t < 2; t++) {
        int tt = t < m->T ? t : 0;
        A.tab[t].val_in = m->d_val[cur][tt];
        A.tab[t].val_out = m->d_val[cur ^ 1][tt];
        A.tab[t].num_out = m->d_num[cur ^ 1][tt];
        A.tab[t].gacc = m->d_gacc[tt];
        A.tab[t].gaccf = (float*)m->d_gacc[tt];
    }
    A.sh_val_in = m->d_sh_val[cur];
    A.sh_acc = m->d_sh_acc;
    A.shared_idx = m->d_shared_idx;
    A.n_shared = m->n_shared;
    A.n_qd = m->n_qd;
    A.n_tables = m->T;
    A.write_num = write_num;
    A.counts = m->d_counts;
    A.counts16 = m->d_counts16;
    A.max_width = m->max_width;
    A.K = m->K;
    A.kacc = m->KACC;
    A.sh_base = m->d_sh_base;
    A.sh_acc_map = m->d_sh_acc_map;
    A.sh_val_out = m->d_sh_val[cur ^ 1];
    A.sh_num_out = m->d_sh_num[cur ^ 1];
    A.sh_den_out = m->d_sh_den[cur ^ 1];
    A.fuse_merge = m->fuse ? 1 : 0;
    A.split_groups = m->d_split_groups;
    A.split_acc = m->d_split_acc;
    A.n_split_acc = m->n_split_acc;
    A.split_done = m->d_split_done;
    A.grid_done = m->d_grid_done;
    A.sh_parts = m->sh_parts;
    return A;
}

// `width`: the launch's window entries (LDS), 0 for items without a window.
template <int MODEL, int PATH>
void launch_path(mc_model* m, KArgs A, int first, int count, int width) {
    if (count <= 0) return;
    A.max_width = width;
    const size_t lds = width ? window_lds_bytes(m->type, m->reduce_mode, width) : 0;
    if (m->varlen)
        hipLaunchKernelGGL((em_item_kernel<MODEL, true, PATH>), dim3(count), dim3(m->block), lds, m->stream, A, first);
    else
        hipLaunchKernelGGL((em_item_kernel<MODEL, false, PATH>), dim3(count), dim3(m->block), lds, m->stream, A, first);
}

template <int MODEL>
void launch_item(mc_model* m, const KArgs& A) {
    if (m->reduce_mode == MC_REDUCE_ATOMIC) {
        // LDS pre-reduction of window items, then float atomics; items
        // without a window add straight to the global accumulators.
        launch_path<MODEL, kPathLdsFloat>(m, A, 0, m->n_win_items, m->max_width);
        launch_path<MODEL, kPathAtomic>(m, A, m->n_win_items, m->n_glob_items, 0);
    } else {
        const int wide = m->n_win_items - m->n_wide_items;
        launch_path<MODEL, kPathPacked>(m, A, 0, m->n_pk_items, m->max_width);
        launch_path<MODEL, kPathLds>(m, A, m->n_pk_items, wide - m->n_pk_items, m->max_width);
        launch_path<MODEL, kPathLds>(m, A, wide, m->n_wide_items, m->wide_width);
        launch_path<MODEL, kPathGlobal>(m, A, m->n_win_items, m->n_glob_items, 0);
        launch_path<MODEL, kPathDirect>(m, A, m->n_win_items + m->n_glob_items, m->n_dir_items, 0);
    }
}

mc_status launch_estep(mc_model* m, int cur, int write_num) {
    KArgs A = make_args(m, cur, write_num);
    switch (m->type) {
        case MC_PBM: launch_item<kPBM>(m, A); break;
        case MC_UBM: launch_item<kUBM>(m, A); break;
        case MC_DBN: launch_item<kDBN>(m, A); break;
        default: launch_item<kCCM>(m, A); break;
    }
    MC_HIP(hipGetLastError());
    return MC_OK;
}

mc_status launch_mstep(mc_model* m, int cur, int write_num) {
    if (m->fuse) return MC_OK;   // done by the E-step launches
    KArgs A = make_args(m, cur, write_num);
    int64_t n_entries = m->reduce_mode == MC_REDUCE_ATOMIC ? m->n_qd : m->n_shared;
    unsigned grid = (unsigned)(1 + (n_entries + 255) / 256);
    switch (m->type) {
        case MC_PBM: hipLaunchKernelGGL(em_merge_kernel<kPBM>, dim3(grid), dim3(256), 0, m->stream, A); break;
        case MC_UBM: hipLaunchKernelGGL(em_merge_kernel<kUBM>, dim3(grid), dim3(256), 0, m->stream, A); break;
        case MC_DBN: hipLaunchKernelGGL(em_merge_kernel<kDBN>, dim3(grid), dim3(256), 0, m->stream, A); break;
        default: hipLaunchKernelGGL(em_merge_kernel<kCCM>, dim3(grid), dim3(256), 0, m->stream, A); break;
    }
    MC_HIP(hipGetLastError());
    return MC_OK;
}

// Captures n_iter iterations starting from buffer parity `cur` into a graph
// (cached per parity).
mc_status get_graph(mc_model* m, int n_iter, int cur, hipGraphExec_t* out) {
    if (m->graph[cur] && m->graph_iters[cur] == n_iter) { *out = m->graph[cur]; return MC_OK; }
    if (m->graph[cur]) { MC_HIP(hipGraphExecDestroy(m->graph[cur])); m->graph[cur] = nullptr; }
    hipGraph_t g;
    MC_HIP(hipStreamBeginCapture(m->stream, hipStreamCaptureModeThreadLocal));
    int c = cur;
    mc_status st = MC_OK;
    for (int i = 0; i < n_iter && st == MC_OK; i++) {
        const int wn = i == n_iter - 1;   // numerators only for the final state
        st = launch_estep(m, c, wn);
        if (st == MC_OK) st = launch_mstep(m, c, wn);
        c ^= 1;
    }
    hipError_t e = hipStreamEndCapture(m->stream, &g);
    if (st != MC_OK) return st;
    MC_HIP(e);
    e = hipGraphInstantiate(&m->graph[cur], g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    MC_HIP(e);
    m->graph_iters[cur] = n_iter;
    *out = m->graph[cur];
    return MC_OK;
}


}  // namespace

// ---------------------------------------------------------------------------
// C ABI
// ---------------------------------------------------------------------------
extern "C" {

const char* mc_last_error(void) { return g_last_error.c_str(); }

mc_status mc_model_create(int model_type, int device, mc_model** out) {
    MC_REQUIRE(out, "null output pointer");
    MC_REQUIRE(model_type >= 0 && model_type <= 3, "model_type must be 0 (PBM), 1 (CCM), 2 (DBN) or 3 (UBM)");
    int n_dev = 0;
    MC_HIP(hipGetDeviceCount(&n_dev));
    MC_REQUIRE(device >= 0 && device < n_dev, "no such HIP device");
    MC_HIP(hipSetDevice(device));
    mc_model* m = new mc_model;
    m->type = model_type;
    m->device = device;
    shape_of(model_type, &m->T, &m->K, &m->KACC);
    const mc_status ss = eval_scratch_setup(device);
    if (ss != MC_OK) {
        delete m;
        return ss;
    }
    hipError_t e = hipStreamCreateWithFlags(&m->stream, hipStreamNonBlocking);
    if (e != hipSuccess) {
        delete m;
        set_error(std::string("hipStreamCreate: ") + hipGetErrorString(e));
        return MC_ERR_HIP;
    }
    e = hipHostMalloc((void**)&m->h_totals, 21 * sizeof(double), hipHostMallocDefault);
    if (e != hipSuccess) {
        (void)hipGetLastError();
        (void)hipStreamDestroy(m->stream);
        delete m;
        set_error(std::string("hipHostMalloc: ") + hipGetErrorString(e));
        return MC_ERR_HIP;
    }
    *out = m;
    return MC_OK;
}

mc_status mc_get_model_type(const mc_model* m, int* model_type) {
    MC_REQUIRE(m && model_type, "null argument");
    *model_type = m->type;
    return MC_OK;
}

mc_status mc_model_set_option(mc_model* m, int option, int64_t value) {
    MC_REQUIRE(m, "null model");
    MC_REQUIRE(!m->initialized, "options must be set before mc_init_parameters");
    switch (option) {
        case MC_OPT_REDUCE_MODE:
            MC_REQUIRE(value == MC_REDUCE_SEGMENTED || value == MC_REDUCE_ATOMIC, "bad reduce mode");
            m->reduce_mode = (int)value;
            break;
        case MC_OPT_ITEM_SESSIONS:
            MC_REQUIRE(value == MC_AUTO || (value >= 64 && value <= (1 << 20)),
                       "item sessions out of range [64, 2^20]");
            m->item_sessions = (int)value;
            m->item_sessions_set = value != MC_AUTO;
            break;
        case MC_OPT_ITEM_WINDOW:
            MC_REQUIRE(value == MC_AUTO || (value >= 0 && value <= 16384), "item window out of range [0, 16384]");
            m->item_window = (int)value;
            m->item_window_set = value != MC_AUTO;
            break;
        case MC_OPT_SORT_BY_LCR:
            m->sort_by_lcr = value != 0;
            break;
        case MC_OPT_DIRECT:
            m->direct = value != 0;
            break;
        case MC_OPT_PERSISTENT:
            break;   // no effect
        case MC_OPT_PACKED:
            m->packed = value != 0;
            break;
        case MC_OPT_SKIP_CONSTANT:
            m->skip_constant = value != 0;
            break;
        case MC_OPT_FUSED_MERGE:
            m->fused_merge = value != 0;
            break;
        case MC_OPT_BATCHES:
            MC_REQUIRE(value >= 1 && value <= 4096, "batches out of range [1, 4096]");
            m->n_batches = (int)value;
            break;
        case MC_OPT_BLOCK:
            MC_REQUIRE(value == MC_AUTO || value == 64 || value == 128 || value == 256 || value == 512,
                       "block must be 64/128/256/512");
            m->block = (int)value;
            m->block_set = value != MC_AUTO;
            break;
        default:
            set_error("unknown option");
            return MC_ERR_INVALID_ARG;
    }
    return MC_OK;
}

mc_status mc_init_parameters(mc_model* m, int64_t n, const int32_t* query, const int32_t* pidx,
                             const uint8_t* clicks, const uint8_t* len, int64_t n_qd) {
    MC_REQUIRE(m && query && pidx && clicks, "null argument");
    // The session stream is addressed with 32-bit buffer offsets: 20 B per
    // session of a window item (checked here), 40 B per other session
    // (checked by the planner, which decides which sessions those are).
    MC_REQUIRE(n >= 1 && n * 20 < (int64_t)UINT32_MAX, "session count out of range (at most 214,748,364)");
    MC_REQUIRE(n_qd >= 1 && n_qd <= INT32_MAX - 1, "n_qd out of range");
    MC_HIP(hipSetDevice(m->device));
    if (m->initialized) release(m);
    const int T = m->T, K = m->K, KACC = m->KACC;
    m->N = n;
    m->n_qd = n_qd;
    m->varlen = len != nullptr;

    HostLayout h;
    try {
        MC_TRY(plan_layout(m, n, query, pidx, clicks, len, n_qd, &h));
    } catch (std::bad_alloc&) {
        set_error("out of host memory while planning the device layout");
        return MC_ERR_OOM;
    }
    const std::vector<Item>& items = h.items;
    const std::vector<int32_t>& shared_idx = h.shared_idx;
    const std::vector<int32_t>& lists = h.lists;
    const std::vector<int2>& counts = h.counts;
    const std::vector<double>& sh_base = h.sh_base;
    const std::vector<int32_t>& sh_map = h.sh_map;
    const std::vector<uint16_t>& h_pidx16 = h.pidx16;
    const std::vector<int32_t>& h_pidx = h.pidx32;
    const std::vector<uint16_t>& h_mask = h.mask;
    const std::vector<uint8_t>& h_len = h.len;
    {
        // The window (plus the kernels' few KB of static LDS) must fit one
        // workgroup's LDS.
        int max_lds = 0;
        MC_HIP(hipDeviceGetAttribute(&max_lds, hipDeviceAttributeMaxSharedMemoryPerBlock, m->device));
        const size_t lds = window_lds_bytes(m->type, m->reduce_mode, std::max(m->max_width, m->wide_width));
        MC_REQUIRE(lds + 4096 <= (size_t)max_lds,
                   "item window too large for this device's LDS (" + std::to_string(m->max_width) + " entries need " +
                       std::to_string(lds) + " bytes, at most " + std::to_string(max_lds) +
                       " per workgroup): use a smaller MC_OPT_ITEM_WINDOW");
    }

    // The M-step runs inside the E-step launches when every work item is a
    // window item of the segmented mode.
    m->fuse = m->fused_merge && m->reduce_mode == MC_REDUCE_SEGMENTED && m->n_win_items == m->n_items;
    m->sh_parts = 1;
    while (m->sh_parts < kMaxShParts && m->sh_parts * 32 < m->n_items) m->sh_parts *= 2;
    MC_TRY(dalloc(m, &m->d_packed, std::max<size_t>(h.packed.size() * 4, 16)));
    MC_TRY(dalloc(m, &m->d_pidx16, std::max<size_t>(h_pidx16.size() * 2, 4)));
    MC_TRY(dalloc(m, &m->d_pidx, std::max<size_t>(h_pidx.size() * 4, 4)));
    MC_TRY(dalloc(m, &m->d_mask, h_mask.size() * 2));
    if (m->varlen) MC_TRY(dalloc(m, &m->d_len, h_len.size()));
    MC_TRY(dalloc(m, &m->d_items, items.size() * sizeof(Item)));
    MC_TRY(dalloc(m, &m->d_shared_idx, shared_idx.size() * 4));
    // Copies of the split groups' sums and counters: one copy per eight
    // slices, at most 16 and 4096 accumulators a group.
    int64_t n_split_done = 0;
    m->n_split_acc = 0;
    if (m->fuse)
        for (SplitGroup& g : h.split_groups) {
            g.parts = 1;
            while (g.parts < 16 && g.parts * 16 <= g.slices && (int64_t)g.parts * 2 * (g.hi - g.lo) <= 4096) g.parts *= 2;
            MC_REQUIRE(m->n_split_acc < (1 << 30) && n_split_done < (1 << 30), "internal: split group sums");
            g.acc = (int32_t)m->n_split_acc;
            g.done = (int32_t)n_split_done;
            m->n_split_acc += (int64_t)g.parts * (g.hi - g.lo);
            n_split_done += (int64_t)(1 + g.parts) * kDoneStride;
        }
    const size_t split_acc_bytes = (size_t)std::max<int64_t>(m->n_split_acc, 1) * T * 8;
    const size_t split_done_bytes = (size_t)std::max<int64_t>(n_split_done, 1) * 4;
    MC_TRY(dalloc(m, &m->d_split_groups, std::max<size_t>(h.split_groups.size(), 1) * sizeof(SplitGroup)));
    MC_TRY(dalloc(m, &m->d_split_acc, split_acc_bytes));
    MC_TRY(dalloc(m, &m->d_split_done, split_done_bytes));
    MC_TRY(dalloc(m, &m->d_grid_done, (size_t)(1 + m->sh_parts) * kDoneStride * 4));
    MC_TRY(dalloc(m, &m->d_lists, lists.size() * 4));
    for (int t = 0; t < T; t++) {
        for (int b = 0; b < 2; b++) {
            MC_TRY(dalloc(m, &m->d_val[b][t], (size_t)n_qd * 4));
            MC_TRY(dalloc(m, &m->d_num[b][t], (size_t)n_qd * 4));
        }
        MC_TRY(dalloc(m, &m->d_gacc[t], (size_t)n_qd * 8));
    }
    for (int b = 0; b < 2; b++) {
        MC_TRY(dalloc(m, &m->d_sh_val[b], (size_t)K * 4));
        MC_TRY(dalloc(m, &m->d_sh_num[b], (size_t)K * 4));
        MC_TRY(dalloc(m, &m->d_sh_den[b], (size_t)K * 4));
    }
    MC_TRY(dalloc(m, &m->d_counts, (size_t)n_qd * 8));
    MC_TRY(dalloc(m, &m->d_counts16, (size_t)n_qd * 2));
    MC_TRY(dalloc(m, &m->d_sh_base, sh_base.size() * 8));
    MC_TRY(dalloc(m, &m->d_sh_acc_map, sh_map.size() * 4));
    MC_TRY(dalloc(m, &m->d_sh_acc, (size_t)m->sh_parts * kShStride * 8));

    if (!h.packed.empty())
        MC_HIP(hipMemcpyAsync(m->d_packed, h.packed.data(), h.packed.size() * 4, hipMemcpyHostToDevice, m->stream));
    if (!h_pidx16.empty())
        MC_HIP(hipMemcpyAsync(m->d_pidx16, h_pidx16.data(), h_pidx16.size() * 2, hipMemcpyHostToDevice, m->stream));
    if (!h_pidx.empty())
        MC_HIP(hipMemcpyAsync(m->d_pidx, h_pidx.data(), h_pidx.size() * 4, hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemcpyAsync(m->d_mask, h_mask.data(), h_mask.size() * 2, hipMemcpyHostToDevice, m->stream));
    if (m->varlen)
        MC_HIP(hipMemcpyAsync(m->d_len, h_len.data(), h_len.size(), hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemcpyAsync(m->d_items, items.data(), items.size() * sizeof(Item), hipMemcpyHostToDevice, m->stream));
    if (!shared_idx.empty())
        MC_HIP(hipMemcpyAsync(m->d_shared_idx, shared_idx.data(), shared_idx.size() * 4, hipMemcpyHostToDevice,
                              m->stream));
    if (!h.split_groups.empty())
        MC_HIP(hipMemcpyAsync(m->d_split_groups, h.split_groups.data(), h.split_groups.size() * sizeof(SplitGroup),
                              hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemsetAsync(m->d_split_acc, 0, split_acc_bytes, m->stream));
    MC_HIP(hipMemsetAsync(m->d_split_done, 0, split_done_bytes, m->stream));
    MC_HIP(hipMemsetAsync(m->d_grid_done, 0, (size_t)(1 + m->sh_parts) * kDoneStride * 4, m->stream));
    if (!lists.empty())
        MC_HIP(hipMemcpyAsync(m->d_lists, lists.data(), lists.size() * 4, hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemcpyAsync(m->d_counts, counts.data(), counts.size() * 8, hipMemcpyHostToDevice, m->stream));
    std::vector<uint16_t> counts16((size_t)n_qd);
    m->h_big_counts.clear();
    for (int64_t p = 0; p < n_qd; p++) {
        const int2 c = counts[(size_t)p];
        counts16[(size_t)p] = c.x < 255 ? (uint16_t)(c.x | (c.y << 8)) : (uint16_t)kCountsEscape;
        if (c.x >= 255) m->h_big_counts.push_back({(int32_t)p, c});
    }
    MC_HIP(hipMemcpyAsync(m->d_counts16, counts16.data(), counts16.size() * 2, hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemcpyAsync(m->d_sh_base, sh_base.data(), sh_base.size() * 8, hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemcpyAsync(m->d_sh_acc_map, sh_map.data(), sh_map.size() * 4, hipMemcpyHostToDevice, m->stream));
    MC_HIP(hipMemsetAsync(m->d_sh_acc, 0, (size_t)m->sh_parts * kShStride * 8, m->stream));
    for (int t = 0; t < T; t++) {
        MC_HIP(hipMemsetAsync(m->d_gacc[t], 0, (size_t)n_qd * 8, m->stream));
        for (int b = 0; b < 2; b++) {
            MC_TRY(fill(m, m->d_val[b][t], 0.5f, n_qd));
            MC_TRY(fill(m, m->d_num[b][t], 1.f, n_qd));
        }
        m->den_state[t] = 0;
    }
    for (int b = 0; b < 2; b++) {
        MC_TRY(fill(m, m->d_sh_val[b], 0.5f, K));
        MC_TRY(fill(m, m->d_sh_num[b], 1.f, K));
        MC_TRY(fill(m, m->d_sh_den[b], 2.f, K));
    }
    m->den_state[T] = 0;
    // For the tables' readback and evaluations of a few thousand host rows.
    MC_TRY(stage_reserve(m, std::max(stage_slot((size_t)n_qd * 4), (size_t)64 << 10)));
    MC_HIP(hipStreamSynchronize(m->stream));
    m->h_counts16 = std::move(counts16);
    m->cur = 0;
    m->estep_pending = false;
    m->initialized = true;
    return MC_OK;
}

mc_status mc_init_from_dataset(mc_model* m, const mc_dataset* ds) {
    MC_REQUIRE(m && ds, "null argument");
    const HostDataset& d = ds->d;
    return mc_init_parameters(m, (int64_t)d.train_query.size(), d.train_query.data(), d.train_pidx.data(),
                              d.train_clicks.data(), d.train_len.empty() ? nullptr : d.train_len.data(), d.n_qd);
}

mc_status mc_process_session(mc_model* m) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    MC_REQUIRE(!m->estep_pending, "E-step already pending; call mc_update_parameters");
    MC_HIP(hipSetDevice(m->device));
    MC_TRY(launch_estep(m, m->cur, 1));
    MC_HIP(hipStreamSynchronize(m->stream));
    m->estep_pending = true;
    return MC_OK;
}

mc_status mc_update_parameters(mc_model* m) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    MC_REQUIRE(m->estep_pending, "no pending E-step; call mc_process_session first");
    MC_HIP(hipSetDevice(m->device));
    MC_TRY(launch_mstep(m, m->cur, 1));
    MC_HIP(hipStreamSynchronize(m->stream));
    m->cur ^= 1;
    m->estep_pending = false;
    for (int t = 0; t <= m->T; t++) m->den_state[t] = 2;
    return MC_OK;
}

mc_status mc_em_iterations(mc_model* m, int n_iter, int use_graph) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    MC_REQUIRE(!m->estep_pending, "an E-step is pending");
    MC_REQUIRE(n_iter >= 0, "n_iter must be >= 0");
    if (n_iter == 0) return MC_OK;
    MC_HIP(hipSetDevice(m->device));
    if (use_graph && n_iter > 1) {   // a graph of one launch costs more than the launch
        hipGraphExec_t g = nullptr;
        MC_TRY(get_graph(m, n_iter, m->cur, &g));
        MC_HIP(hipGraphLaunch(g, m->stream));
    } else {
        int c = m->cur;
        for (int i = 0; i < n_iter; i++) {
            const int wn = i == n_iter - 1;
            MC_TRY(launch_estep(m, c, wn));
            MC_TRY(launch_mstep(m, c, wn));
            c ^= 1;
        }
    }
    MC_HIP(hipStreamSynchronize(m->stream));
    m->cur ^= (n_iter & 1);
    for (int t = 0; t <= m->T; t++) m->den_state[t] = 2;
    return MC_OK;
}

mc_status mc_em_iterations_timed(mc_model* m, int n_iter, double* ms_total, double* ms_estep_avg,
                                 double* ms_mstep_avg) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    MC_REQUIRE(!m->estep_pending, "an E-step is pending");
    MC_REQUIRE(n_iter >= 1, "n_iter must be >= 1");
    MC_HIP(hipSetDevice(m->device));
    std::vector<hipEvent_t> ev((size_t)(3 * n_iter + 1));
    for (auto& e : ev) MC_HIP(hipEventCreate(&e));
    int c = m->cur;
    MC_HIP(hipEventRecord(ev[0], m->stream));
    for (int i = 0; i < n_iter; i++) {
        const int wn = i == n_iter - 1;
        MC_HIP(hipEventRecord(ev[3 * i + 1], m->stream));
        MC_TRY(launch_estep(m, c, wn));
        MC_HIP(hipEventRecord(ev[3 * i + 2], m->stream));
        MC_TRY(launch_mstep(m, c, wn));
        MC_HIP(hipEventRecord(ev[3 * i + 3], m->stream));
        c ^= 1;
    }
    MC_HIP(hipStreamSynchronize(m->stream));
    double te = 0, tm = 0;
    for (int i = 0; i < n_iter; i++) {
        float a = 0, b = 0;
        MC_HIP(hipEventElapsedTime(&a, ev[3 * i + 1], ev[3 * i + 2]));
        MC_HIP(hipEventElapsedTime(&b, ev[3 * i + 2], ev[3 * i + 3]));
        te += a;
        tm += b;
    }
    float tot = 0;
    MC_HIP(hipEventElapsedTime(&tot, ev[0], ev[3 * n_iter]));
    for (auto& e : ev) (void)hipEventDestroy(e);
    if (ms_total) *ms_total = tot;
    if (ms_estep_avg) *ms_estep_avg = te / n_iter;
    if (ms_mstep_avg) *ms_mstep_avg = tm / n_iter;
    m->cur ^= (n_iter & 1);
    for (int t = 0; t <= m->T; t++) m->den_state[t] = 2;
    return MC_OK;
}

mc_status mc_em_graph_timed(mc_model* m, int n_iter, double* ms_total) {
    MC_REQUIRE(m && m->initialized && n_iter >= 1, "invalid argument");
    MC_REQUIRE(!m->estep_pending, "an E-step is pending");
    MC_HIP(hipSetDevice(m->device));
    // One warm replay, then the timed replay (graphs built outside the timing).
    MC_TRY(mc_em_iterations(m, n_iter, 1));
    hipGraphExec_t g = nullptr;
    MC_TRY(get_graph(m, n_iter, m->cur, &g));
    hipEvent_t a, b;
    MC_HIP(hipEventCreate(&a));
    MC_HIP(hipEventCreate(&b));
    MC_HIP(hipEventRecord(a, m->stream));
    MC_HIP(hipGraphLaunch(g, m->stream));
    MC_HIP(hipEventRecord(b, m->stream));
    MC_HIP(hipStreamSynchronize(m->stream));
    float ms = 0;
    MC_HIP(hipEventElapsedTime(&ms, a, b));
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    m->cur ^= (n_iter & 1);
    for (int t = 0; t <= m->T; t++) m->den_state[t] = 2;
    if (ms_total) *ms_total = ms;
    return MC_OK;
}

mc_status mc_synchronize(mc_model* m) {
    MC_REQUIRE(m, "null model");
    MC_HIP(hipStreamSynchronize(m->stream));
    return MC_OK;
}

mc_status mc_get_n_tables(const mc_model* m, int* n_tables) {
    MC_REQUIRE(m && n_tables, "null argument");
    *n_tables = m->T + 1;
    return MC_OK;
}

mc_status mc_get_table_info(const mc_model* m, int t, const char** name, int* is_public, int64_t* size) {
    MC_REQUIRE(m && t >= 0 && t <= m->T, "bad table index");
    if (name) *name = table_name(m->type, t);
    if (is_public) *is_public = t == m->T;
    if (size) *size = t == m->T ? m->K : m->n_qd;
    return MC_OK;
}

mc_status mc_get_parameters(mc_model* m, int t, float* num, float* den) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    MC_REQUIRE(t >= 0 && t <= m->T, "bad table index");
    MC_HIP(hipSetDevice(m->device));
    const bool shared = t == m->T;
    const int64_t n = shared ? m->K : m->n_qd;
    if (!shared && m->den_state[t] == 3) {
        // Values set by the gradient path: (value, 1).
        if (num) MC_TRY(download(m, num, m->d_val[m->cur][t], n * 4));
        if (den) std::fill(den, den + n, 1.f);
        return MC_OK;
    }
    // The host fills in denominators that it knows (the prior's, or the
    // M-step's constants) while the numerators are on their way.
    const float* src = shared ? m->d_sh_num[m->cur] : m->d_num[m->cur][t];
    auto host_den = [&](size_t at, size_t bytes) {
        const size_t first = at / 4, k = bytes / 4;
        if (!den || shared || m->den_state[t] == 1) return;
        if (m->den_state[t] == 0) std::fill(den + first, den + first + k, 2.f);
        else constant_den(m, t, den, first, k);
    };
    if (num)
        MC_TRY(staged_out(
            m, (char*)num, (size_t)n * 4,
            [&](char* to, size_t at, size_t bytes) { return copy_out(m, src, to, at, bytes); }, host_den));
    else
        host_den(0, (size_t)n * 4);
    if (den && shared) return download(m, den, m->d_sh_den[m->cur], n * 4);
    if (den && m->den_state[t] == 1) return download(m, den, m->d_den_user[t], n * 4);
    return MC_OK;
}

mc_status mc_set_parameters(mc_model* m, int t, const float* num, const float* den) {
    MC_REQUIRE(m && m->initialized && num && den, "invalid argument");
    MC_REQUIRE(t >= 0 && t <= m->T, "bad table index");
    MC_REQUIRE(!m->estep_pending, "an E-step is pending");
    MC_HIP(hipSetDevice(m->device));
    const bool shared = t == m->T;
    const int64_t n = shared ? m->K : m->n_qd;
    std::vector<float> val((size_t)n);
    for (int64_t i = 0; i < n; i++) {   // Param::value, param.cu:75-87
        const float v = num[i] / den[i];
        val[i] = v < kClampMax ? v : kClampMax;
    }
    float* dv = shared ? m->d_sh_val[m->cur] : m->d_val[m->cur][t];
    float* dn = shared ? m->d_sh_num[m->cur] : m->d_num[m->cur][t];
    MC_HIP(hipMemcpy(dv, val.data(), n * 4, hipMemcpyHostToDevice));
    MC_HIP(hipMemcpy(dn, num, n * 4, hipMemcpyHostToDevice));
    if (shared) {
        MC_HIP(hipMemcpy(m->d_sh_den[m->cur], den, n * 4, hipMemcpyHostToDevice));
    } else {
        if (!m->d_den_user[t]) MC_TRY(dalloc(m, &m->d_den_user[t], (size_t)n * 4));
        MC_HIP(hipMemcpy(m->d_den_user[t], den, n * 4, hipMemcpyHostToDevice));
        m->den_state[t] = 1;
    }
    return MC_OK;
}

mc_status mc_reset_parameters(mc_model* m) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    MC_HIP(hipSetDevice(m->device));
    ResetArgs R;
    for (int t = 0; t < 2; t++) {
        R.val[t] = m->d_val[m->cur][t < m->T ? t : 0];
        R.num[t] = m->d_num[m->cur][t < m->T ? t : 0];
    }
    R.sh_val = m->d_sh_val[m->cur];
    R.sh_num = m->d_sh_num[m->cur];
    R.sh_den = m->d_sh_den[m->cur];
    R.n_qd = m->n_qd;
    R.T = m->T;
    R.K = m->K;
    hipLaunchKernelGGL(reset_kernel, dim3((unsigned)((m->n_qd + 1023) / 1024 + 1)), dim3(256), 0, m->stream, R);
    MC_HIP(hipGetLastError());
    MC_HIP(hipStreamSynchronize(m->stream));
    for (int t = 0; t < m->T; t++) m->den_state[t] = 0;
    m->estep_pending = false;
    return MC_OK;
}

mc_status mc_get_memory_usage(const mc_model* m, size_t* bytes) {
    MC_REQUIRE(m && bytes, "null argument");
    *bytes = m->mem_bytes;
    return MC_OK;
}

mc_status mc_compute_memory_footprint(int model_type, int64_t n, int64_t n_qd, size_t* bytes) {
    MC_REQUIRE(bytes && model_type >= 0 && model_type <= 3 && n >= 0 && n_qd >= 0, "invalid argument");
    int T, K, KACC;
    shape_of(model_type, &T, &K, &KACC);
    // EM buffers, for the default layout.  Sessions: at most 40 B of indices
    // (20 B for sessions of window items), 2 B mask, 1 B length.  Per entry
    // and table: two values, two numerators, an 8-byte accumulator; per
    // entry: 8 B counts, 2 B packed counts, 4 B if merged across items.
    // Work items of at least 64 sessions (24 B each, 8 B of batch lists).
    const size_t items = (size_t)(n / 64 + 1);
    // Shared tables: values, numerators, denominators (two each), FP64 bases,
    // accumulator map; plus the 16-byte minimum of small allocations.
    size_t b = (size_t)n * 43 + (size_t)n_qd * ((size_t)T * 24 + 14) + (size_t)K * 64;
    b += (size_t)KACC * 8 + items * (sizeof(Item) + 8) + 256;
    *bytes = b;
    return MC_OK;
}

mc_status mc_get_layout_info(const mc_model* m, int64_t* n_items, int64_t* n_shared_entries,
                             int64_t* max_item_sessions, int64_t* n_em_sessions) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    if (n_items) *n_items = m->n_items;
    if (n_shared_entries) *n_shared_entries = m->n_shared;
    if (max_item_sessions) *max_item_sessions = m->max_item_sessions;
    if (n_em_sessions) *n_em_sessions = m->n_em_sessions;
    return MC_OK;
}

mc_status mc_get_stream_info(const mc_model* m, int64_t* n_window_sessions, int64_t* index_bytes) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    if (n_window_sessions) *n_window_sessions = m->n_w;
    if (index_bytes) *index_bytes = m->n_pk * 16 + (m->n_w - m->n_pk) * kMaxSerp * 2 + (m->N - m->n_w) * kMaxSerp * 4;
    return MC_OK;
}

mc_status mc_get_session_formats(const mc_model* m, int64_t* n_packed, int64_t* n_window16, int64_t* n_absolute) {
    MC_REQUIRE(m && m->initialized, "model not initialised");
    if (n_packed) *n_packed = m->n_pk;
    if (n_window16) *n_window16 = m->n_w - m->n_pk;
    if (n_absolute) *n_absolute = m->N - m->n_w;
    return MC_OK;
}

void mc_model_destroy(mc_model* m) {
    if (!m) return;
    (void)hipSetDevice(m->device);
    (void)hipStreamSynchronize(m->stream);
    release(m);
    (void)hipHostFree(m->h_totals);
    if (m->stage[0]) (void)hipHostFree(m->stage[0]);
    for (hipEvent_t e : m->stage_ev)
        if (e) (void)hipEventDestroy(e);
    (void)hipStreamDestroy(m->stream);
    delete m;
}

}  // extern "C"
