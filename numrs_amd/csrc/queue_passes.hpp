// queue_passes.hpp -- uneven batches in two launches, one a pass, for the batches that
// run slower as one list (queue_api.hip says which) or whose ring finds no room: here
// only 1-D items of two passes need memory, 2-D ones use the output.
//
// The host turns every item into tiles of one pass each:
//   1-D, one pass             one row tile (the whole transform)
//   1-D, longer               four-step: N1 column tiles with the W_N twiddle
//                             (in -> workspace), then N2 row tiles stored
//                             transposed (workspace -> out)
//   2-D, n0 x n1              row tiles along n1 (in -> out), then column
//                             tiles along n0 (in place in out)
// First passes and single-pass items are ordered largest first, second passes
// follow in the same item order.  Groups of a launch take tiles from a counter; the
// end of a launch makes the first passes' results visible to the second ones on
// another XCD.
//
// What bounds it: the latency of a tile.  A tile is 16 values a thread (1024
// threads FP32, 512 FP64, whole values in LDS, one group a CU), against 32 of 512
// threads and two groups a CU in the one-launch form, so a tile of three or four
// stages is done sooner, and a list that does not fill the chip with it.
#pragma once
#include "pass_c2c.hpp"

namespace nrfft {

// Tile points (TI x L) of the queue kernel: EPT = 16 values per thread, so a
// group has qp_pts / 16 threads.
template <typename T>
constexpr int qp_pts() {
    return sizeof(T) == 4 ? 16384 : 8192;
}
constexpr int QP_MIN_LOGL = 6;
// Longest pass of a tile: at most the tile itself and 8192 points (a single
// 16384-point FP32 tile -- four stages, one transform -- measured slower on
// the 10,000-item batch than the two-pass four-step it replaces).
constexpr int QP_MAX_LOGL = 13;
template <typename T>
constexpr int qp_max_logl() {
    return ilog2c(qp_pts<T>()) < QP_MAX_LOGL ? ilog2c(qp_pts<T>()) : QP_MAX_LOGL;
}
constexpr int QP_MODES = 3;  // 0: row (JJ), 1: column (TT), 2: row load / column store (JT)

template <typename T>
constexpr int qp_nclasses() {
    return (qp_max_logl<T>() - QP_MIN_LOGL + 1) * QP_MODES;
}

template <typename T>
constexpr int qp_lds_elems() {
    return qp_pts<T>() + qp_pts<T>() / NRFFT_LDS_PAD + 1;
}

struct QPass {
    int32_t cls;        // (log2 L - QP_MIN_LOGL) * QP_MODES + mode
    int32_t nvalid;     // transforms of the tile that exist
    int32_t src, dst;   // 0 = in, 1 = out, 2 = workspace
    int64_t ioff, ooff; // element offsets of the tile base
    int32_t si0, esi, so0, eso;
    int32_t tw_logn;    // four-step twiddle W_N^{k (tw_n2base + t)}, N = 2^tw_logn (0 = none)
    int32_t tw_n2base;
};

struct QPState {
    uint32_t next[2];  // task counters of the two phases
};

// Stages 1 .. NST-2 of a tile class read their twiddles from an LDS copy
// (at most the 8192-point tables: 612 entries); a group refreshes it when
// its next task has another transform length.
template <int L>
constexpr int qp_ltm() {
    return RadixPlan<L>::NST >= 3 ? RadixPlan<L>::NST - 2 : 0;
}
constexpr int QP_LTW_ELEMS = 612;

template <typename T, int S, int C>
__device__ __forceinline__ void qp_run_class(const QPass& q, cpx<T>* const* bufs, cpx<T>* lds, cpx<T>* ltw,
                                            bool fresh_tw, const Twiddles<T>& tw, int tid) {
    constexpr int LOGL = C / QP_MODES + QP_MIN_LOGL;
    constexpr int MODE = C % QP_MODES;
    constexpr int L = 1 << LOGL;
    if constexpr (L > qp_pts<T>()) {
        return;
    } else {
        constexpr int TI = qp_pts<T>() / L;
        constexpr int NT = qp_pts<T>() / 16;
        constexpr int ML = MODE == 1 ? MAP_T : MAP_J;
        constexpr int MS = MODE == 0 ? MAP_J : MAP_T;
        using E = Engine<T, S, L, TI, NT, ML, MS>;
        static_assert(E::LDS_ELEMS <= qp_lds_elems<T>(), "queue LDS too small for a tile class");
        static_assert(TI * L == qp_pts<T>() && E::EPT == 16, "queue tile shape");
        constexpr int LTM = qp_ltm<L>();
        static_assert(LTM == 0 || E::tw_elems(LTM) <= QP_LTW_ELEMS, "queue twiddle copy too small");
        // Published by the first exchange barrier; the loop-top barrier of
        // k_queue_pass ordered the previous task's reads before this overwrite.
        if constexpr (LTM > 0)
            if (fresh_tw) E::template stage_tw_to_lds<LTM>(ltw, tw.stage, tid);
        const cpx<T>* ib = bufs[q.src] + q.ioff;
        cpx<T>* ob = bufs[q.dst] + q.ooff;
        const int nvalid = q.nvalid, si0 = q.si0, esi = q.esi, so0 = q.so0, eso = q.eso;
        cpx<T> v[E::EPT];
        E::load0(v, tid, [&](int t, int i) -> cpx<T> {
            if (t < nvalid) return ib[t * si0 + i * esi];
            return cpx<T>{(T)0, (T)0};
        });
        E::template compute<0>(v, tid, tw.stage);
        E::template middle<1, LTM>(v, tid, lds, tw.stage, false, ltw);
        if (q.tw_logn) {
            const int logn = q.tw_logn;
            const uint32_t mask = (1u << logn) - 1u;
            E::store_last(v, tid, [&](int t, int j, const cpx<T>* w) {
                if (t < nvalid) {
                    const uint32_t n2 = uint32_t(q.tw_n2base + t);
                    cpx<T> f[E::RLAST];
                    twiddle_run<E::RLAST, S>(tw, (uint32_t(j) * n2) & mask, (uint32_t(E::NBLAST) * n2) & mask, logn, f);
#pragma unroll
                    for (int r = 0; r < E::RLAST; ++r) ob[t * so0 + (j + r * E::NBLAST) * eso] = cmul(w[r], f[r]);
                }
            });
        } else {
            E::store_last(v, tid, [&](int t, int j, const cpx<T>* w) {
                if (t < nvalid) {
#pragma unroll
                    for (int r = 0; r < E::RLAST; ++r) ob[t * so0 + (j + r * E::NBLAST) * eso] = w[r];
                }
            });
        }
    }
}

template <typename T, int S, int... Cs>
__device__ __forceinline__ void qp_dispatch(int cls, const QPass& q, cpx<T>* const* bufs, cpx<T>* lds, cpx<T>* ltw,
                                           bool fresh_tw, const Twiddles<T>& tw, int tid,
                                           std::integer_sequence<int, Cs...>) {
    ((cls == Cs ? qp_run_class<T, S, Cs>(q, bufs, lds, ltw, fresh_tw, tw, tid) : void()), ...);
}

// Reset of the queue counters (a fill kernel, so the sequence can live in a
// captured graph).
__global__ void k_queue_reset(QPState* st) {
    if (threadIdx.x < 2) st->next[threadIdx.x] = 0;
}

// One phase: tasks [base, base + count) of the task list.
template <typename T, int S>
__global__ __launch_bounds__(qp_pts<T>() / 16) void k_queue_pass(cpx<T>* in, cpx<T>* out, cpx<T>* ws, const QPass* tasks,
                                                            int base, int count, int phase, QPState* st,
                                                            Twiddles<T> tw) {
    __shared__ cpx<T> lds[qp_lds_elems<T>()];
    __shared__ __align__(16) cpx<T> ltw[QP_LTW_ELEMS];
    __shared__ int sh_task;
    cpx<T>* bufs[3] = {in, out, ws};
    const int tid = threadIdx.x;
    int tw_logl = -1;  // transform length whose twiddles ltw holds
    for (;;) {
        lds_barrier();  // previous task's LDS readers are done; sh_task free
        if (tid == 0) sh_task = (int)atomicAdd(&st->next[phase], 1u);
        lds_barrier();
        const int k = sh_task;
        if (k >= count) break;
        const QPass q = tasks[base + k];
        const int logl = q.cls / QP_MODES + QP_MIN_LOGL;
        qp_dispatch<T, S>(q.cls, q, bufs, lds, ltw, logl != tw_logl, tw, fresh_tid(tid),
                         std::make_integer_sequence<int, qp_nclasses<T>()>{});
        tw_logl = logl;
    }
}

}  // namespace nrfft
