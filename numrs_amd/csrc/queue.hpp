// queue.hpp -- uneven batches in one launch: every pass of every item is a
// list of tiles, run in list order by the groups of a persistent kernel.
//
// Tile classes (transform length L, mode), tiles of FS_TILE bytes in the
// stage engine of the fused four-step (fused_c2c.hpp):
//   Q_ROW   1-D items of one length of up to 8192 points, in -> out (wherever
//           they lie: a list of offsets)
//   Q_COL   columns of a longer 1-D item, times W_N^{k n2}, in -> ring
//   Q_ROWS  rows of a 2-D item, in -> ring
//   Q_RING  second passes (rows of the four-step, columns of a 2-D item), ring -> out
//
// The intermediate of an item's two passes lies in a ring that fits the last-level
// cache.  Items are taken largest first and collected into slabs; a slab gets the
// next part of the ring, and its second passes stand in the list half a ring
// behind its first ones.  Each slab has two counters that run down to 0: tiles
// its first pass still has to store (its second-pass tiles wait for that) and
// tiles its second pass still has to load (the first-pass tiles of the slabs that
// get its part of the ring next wait for that).  A tile waits only for tiles that
// stand before it in the list, so the first unfinished tile never waits.
// Coherence across XCDs as in fused_c2c.hpp: SC1 stores and loads.
//
// What bounds it: as the fused four-step, the fabric between the XCDs and the
// memory side (2.1 times the algorithmic bytes pass it).  500 items of mixed shapes,
// FP32 (914 MB): 583 us; as two launches,
// one a pass with the whole intermediate in memory, 840 (HBM traffic twice).
// 16 of 2048 x 2048 382 us against 575 (second-pass tiles of eight columns write
// 64-byte runs), 64 of 1024 x 1024 335 against 525.  Batches that are faster as two
// launches (few tiles of long passes): queue_passes.hpp.
//
// In the ring an item lies in blocks [second-pass tile][first-pass tile][kk][t]
// (kk: transform of the second-pass tile, t: of the first), so that a tile of
// either pass moves whole runs of kk x t values.
#pragma once
#include "fused_c2c.hpp"

namespace nrfft {

constexpr int Q_MIN_LOGL = 6, Q_MAX_LOGL = 13;
enum { Q_ROW = 0, Q_COL, Q_ROWS, Q_RING, Q_MODES };
constexpr int Q_NCLASSES = (Q_MAX_LOGL - Q_MIN_LOGL + 1) * Q_MODES;

struct QTask {
    int32_t cls;             // (log2 L - Q_MIN_LOGL) * Q_MODES + mode
    int32_t nvalid;          // transforms of the tile that exist
    int64_t ioff, ooff;      // element offsets of the tile's base in its buffers
    uint32_t ibytes, obytes; // bytes from there to the end of the item
    int32_t ist;             // Q_ROWS, Q_RING: distance of the tile's transforms in the input
    int32_t ish, ihi;        // input element i at (i >> ish) ihi + (i mod 2^ish)
    int32_t osh, ohi, olo;   // output element k at (k >> osh) ohi + (k mod 2^osh) olo
    int32_t tw_logn;         // Q_COL: N = 2^tw_logn
    int32_t first;           // Q_COL: n2 of the tile's first column; Q_ROW: its first entry of the offset list
    int32_t wait, nwait;     // counters [wait, wait + nwait), nwait <= 64, that have to be 0
    int32_t count;           // counter of this tile (Q_COL, Q_ROWS: stored, Q_RING: loaded; 0: none)
    int32_t last;            // no second tile in this ticket
};

// Counters, each on a cache line of its own: tickets taken, groups that have
// left, tickets taken in the last launch, whether a wait has given up (set until a
// check reads it), then the slabs'.
constexpr int Q_LINE = 32, Q_TICKET = 0, Q_DONE = 1, Q_LAST = 2, Q_EXPIRED = 3, Q_SLABS = 4;
constexpr size_t Q_SLAB_TILES = 64, Q_PAIR_TILES = 640, Q_FEW_TILES = 768;

// Stage-1 twiddles of all lengths: W_{n^2}^{r k} for k, r < n, n = 32 (FP32) and
// 16, rows of n + 2 entries.  A class of NS rows and radix R reads every n / NS-th
// row and n / R-th column.
template <typename T>
constexpr int q_tw_elems() {
    return (sizeof(T) == 4 ? 32 * 34 : 0) + 16 * 18;
}
template <typename T, int R, int NS>
__device__ __forceinline__ auto q_ltw(const cpx<T>* ltw) {
    constexpr int n = R == 32 ? 32 : 16;
    return FsLtw<T, n / NS * (n + 2), n / R>{n == 32 ? ltw + 16 * 18 : ltw};
}
template <typename T>
__device__ __forceinline__ void q_fill_tw(cpx<T>* ltw, const cpx<T>* coarse, int tid) {
    for (int e = tid; e < 256; e += FS_NT) ltw[(e / 16) * 18 + e % 16] = coarse[(e / 16) * (e % 16) * (TW_COARSE / 256)];
    if constexpr (sizeof(T) == 4)
        for (int e = tid; e < 1024; e += FS_NT)
            ltw[16 * 18 + (e / 32) * 34 + e % 32] = coarse[(e / 32) * (e % 32) * (TW_COARSE / 1024)];
}

// Which classes exist: a column tile holds at least 4 transforms, the columns
// of a 2-D item at least 2; rows of 8192 are stored along the row.
template <typename T>
constexpr bool q_has(int logl, int mode) {
    constexpr int ql = ilog2c(fs_tile<T>());
    return logl <= ql && (mode != Q_COL || logl <= ql - 2) && (mode != Q_RING || logl <= ql - 1);
}
template <typename T, int S, int LOGL, int MODE>
using QEng = FsEng<T, S, (1 << LOGL), MODE == Q_COL ? MAP_T : MAP_J,
                   (MODE == Q_ROW || LOGL == Q_MAX_LOGL) ? MAP_J : MAP_T>;
template <typename T, int C = 0>
constexpr int q_ex_elems() {
    if constexpr (C == Q_NCLASSES) {
        return 0;
    } else {
        constexpr int rest = q_ex_elems<T, C + 1>();
        if constexpr (q_has<T>(C / Q_MODES + Q_MIN_LOGL, C % Q_MODES)) {
            using E = QEng<T, 1, C / Q_MODES + Q_MIN_LOGL, C % Q_MODES>;
            return E::EX_ELEMS > rest ? E::EX_ELEMS : rest;
        } else {
            return rest;
        }
    }
}

// One tile.  publish: after its loads are issued; loaded: every wave's have
// arrived (FsEng's hook `read`); mid / late: FsEng's hooks.
template <typename T, int S, int C, class PUB, class LOADED, class MID, class LATE>
__device__ __forceinline__ void q_tile(const QTask& q, const cpx<T>* in, cpx<T>* out, cpx<T>* ring,
                                       const uint32_t* __restrict__ offs, T* ex,
                                       const cpx<T>* ltw, const Twiddles<T>& tw, int tid, PUB&& publish,
                                       LOADED&& loaded, MID&& mid, LATE&& late) {
    constexpr int LOGL = C / Q_MODES + Q_MIN_LOGL, MODE = C % Q_MODES, L = 1 << LOGL, CS = (int)sizeof(cpx<T>);
    if constexpr (q_has<T>(LOGL, MODE)) {
        using E = QEng<T, S, LOGL, MODE>;
        constexpr int EPT = E::EPT;
        constexpr int AUX_IN = MODE == Q_RING ? FS_AUX_SC1 : FS_AUX_NT;
        // Results are not read again (NT), but runs of less than 64 bytes (sides of 4096
        // and 8192) have to meet their line's other runs in the L2 first: 4096 x 4096 FP32
        // 228 us against 388, 8 of 2048 x 2048 (64-byte runs) 242 against 221 with NT.
        constexpr int AUX_OUT = MODE == Q_COL || MODE == Q_ROWS ? FS_AUX_SC1
                                : MODE == Q_RING && E::TI * CS < 64 ? 0 : FS_AUX_NT;
        // A transform that does not exist is out of its buffer's range: loads
        // give 0, stores are dropped.  (Four-step tiles are always full.)
        auto valid = [&](uint32_t off, int t) {
            return MODE == Q_COL || t < q.nvalid ? off * uint32_t(CS) : 0x80000000u;
        };
        auto ioff = [&](uint32_t i) {
            if constexpr (MODE == Q_COL) return i * uint32_t(q.ihi);
            else if constexpr (MODE == Q_RING) return (i >> q.ish) * uint32_t(q.ihi) + (i & ((1u << q.ish) - 1u));
            else return i;
        };
        auto ooff = [&](uint32_t k) {
            if constexpr (MODE == Q_ROW) return k;
            else if constexpr (MODE == Q_RING) return k * uint32_t(q.ohi);
            else return (k >> q.osh) * uint32_t(q.ohi) + (k & ((1u << q.osh) - 1u)) * uint32_t(q.olo);
        };
        // Where transform t begins: a list entry, or t times a distance.
        auto start = [&](int t, uint32_t dist) {
            if constexpr (MODE == Q_ROW) return offs[q.first + (t < q.nvalid ? t : 0)];
            else return uint32_t(t) * dist;
        };
        cpx<T> v[EPT];
        const __amdgpu_buffer_rsrc_t ri = fs_rsrc((MODE == Q_RING ? ring : in) + q.ioff, q.ibytes);
        uint32_t at0[EPT / E::R0];
        E::template each_butterfly<0>(tid, [&](int b, int t, int) { at0[b] = start(t, MODE == Q_COL ? 1u : uint32_t(q.ist)); });
        E::template each_butterfly<0>(tid, [&](int b, int t, int j) {
            constexpr int R = E::R0, NB = L / R;
            const uint32_t voff = valid(ioff(uint32_t(j)) + at0[b], t);
            // j and r NB have no bits in common, so their offsets add up
#pragma unroll
            for (int r = 0; r < R; ++r) v[b * R + r] = fs_load<T, AUX_IN>(ri, voff, ioff(uint32_t(r * NB)) * uint32_t(CS));
        });
        publish();
        __builtin_amdgcn_s_setprio(1);
        E::template butterflies<0>(v);
        FsTw<T, S, E::RL, EPT / E::RL, E::NBL> f;
        uint32_t at1[EPT / E::RL];  // where the outputs go
        auto load_tw = [&]() {
            if constexpr (MODE == Q_ROW) {
                E::template each_butterfly<E::NST - 1>(tid, [&](int b, int t, int) { at1[b] = start(t, 0); });
            } else if constexpr (MODE == Q_COL) {
                uint32_t n2 = 0, jl[EPT / E::RL];
                E::template each_butterfly<E::NST - 1>(tid, [&](int b, int t, int j) {
                    n2 = uint32_t(q.first + t);  // the same for every b
                    jl[b] = uint32_t(j);
                });
                f.load(tw, n2, jl, q.tw_logn);
            }
        };
        E::rest(
            v, tid, ex, q_ltw<T, E::P::R[1], E::ns(1)>(ltw), tw.stage,
            [&]() {
                if constexpr (MODE == Q_RING) loaded();
            },
            load_tw,
            [&]() {
                __builtin_amdgcn_s_setprio(2);
                if constexpr (MODE == Q_COL) f.join();
                mid();
            },
            [&]() {
                late();
                __builtin_amdgcn_s_setprio(3);
            });
        if constexpr (MODE == Q_COL) f.apply(v);
        const __amdgpu_buffer_rsrc_t ro = fs_rsrc((MODE == Q_COL || MODE == Q_ROWS ? ring : out) + q.ooff, q.obytes);
        E::template each_butterfly<E::NST - 1>(tid, [&](int b, int t, int j) {
            constexpr int R = E::RL, NB = E::NBL;
            const uint32_t voff = valid(ooff(uint32_t(j)) + (MODE == Q_ROW ? at1[b] : uint32_t(t)), t);
#pragma unroll
            for (int r = 0; r < R; ++r) fs_store<T, AUX_OUT>(v[b * R + r], ro, voff, ooff(uint32_t(r * NB)) * uint32_t(CS));
        });
        __builtin_amdgcn_s_setprio(0);
    }
}

template <typename T, int S, int... Cs, class... A>
__device__ __forceinline__ void q_dispatch(std::integer_sequence<int, Cs...>, int cls, A&&... a) {
    ((cls == Cs ? q_tile<T, S, Cs>(a...) : void()), ...);
}

__device__ __forceinline__ void q_count(uint32_t* p) {
    __hip_atomic_fetch_sub(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// A ticket u is one or two tiles, 2 u and 2 u + 1 (an atomic on one line takes
// about 40 ns here whoever asks: a tile each would bound a long list).
template <typename T, int S>
__global__ __attribute__((amdgpu_flat_work_group_size(FS_NT, FS_NT), amdgpu_waves_per_eu(4, 4))) void
k_queue(const cpx<T>* in, cpx<T>* out, cpx<T>* ring, const QTask* __restrict__ tasks, int ntasks,
        const uint32_t* __restrict__ offs, uint32_t* ctr, const uint32_t* __restrict__ init, int lines, Twiddles<T> tw) {
    __shared__ __align__(16) T ex[q_ex_elems<T>()];
    __shared__ __align__(16) cpx<T> ltw[q_tw_elems<T>()];
    __shared__ uint32_t sh[2], arrive;
    static_assert(sizeof(ex) + sizeof(ltw) + 64 <= 81920, "two groups share a CU");
    const int tid = threadIdx.x;
    const bool wave0 = __builtin_amdgcn_readfirstlane(tid >> 6) == 0;
    uint32_t taken = 0;                // lane 0: the ticket as it arrives
    uint32_t next = 0, seen = 1;       // wave 0: the coming tile, and its counters as last read (one a lane)
    int next_wait = 0, next_n = 0;     // wave 0: what it waits for
    int patience = FS_SPIN;            // polls (as k_fused4: once in vain)
    uint32_t* pending = nullptr;       // counter of the group's last tile, its stores perhaps in flight
    auto line = [&](int c) { return ctr + c * Q_LINE; };
    auto peek = [&](int wait, int n) { return tid < n ? fs_peek(line(wait + tid)) : 0u; };  // wave 0
    // (fresh_tid: see k_fused4.)
    auto take_ticket = [&]() {
        if (tid == 0)
            taken = __hip_atomic_fetch_add(ctr + fresh_tid(0), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto aim = [&](uint32_t k) {
        next = k;
        next_n = 0;
        if (int(next) < ntasks) {
            next_wait = tasks[next].wait;
            next_n = tasks[next].nwait;
        }
    };
    if (tid == 0) arrive = 0;
    take_ticket();
    q_fill_tw(ltw, tw.coarse, tid);
    if (wave0) aim(2u * __builtin_amdgcn_readfirstlane(taken));
    for (;;) {
        if (wave0) {
            const bool ok = next_n == 0 || __ballot(seen != 0) == 0;
            if (tid == 0) {
                sh[0] = next;
                sh[1] = ok;
            }
        }
        lds_barrier();  // also: the previous tile's exchange has been read
        const int k = __builtin_amdgcn_readfirstlane(int(sh[0]));
        const bool ready = __builtin_amdgcn_readfirstlane(int(sh[1])) != 0;
        if (k >= ntasks) break;
        const QTask q = tasks[k];
        if (!ready) {
            // Publish the last tile before waiting for anything.
            if (pending) {
                fs_drain<0>();
                lds_barrier();
                if (tid == 0) q_count(pending);
                pending = nullptr;
            }
            if (wave0) {
                int i = 0;
                for (; i < patience; ++i) {
                    if (__ballot(peek(q.wait, q.nwait) != 0) == 0) break;
                    __builtin_amdgcn_s_sleep(8);
                }
                if (i == patience) {
                    patience = 0;
                    if (tid == 0) fs_flag(line(Q_EXPIRED));
                }
            }
            lds_barrier();
        }
        const int ltid = fresh_tid(tid);
        const bool last = q.last != 0;
        auto publish = [&]() {
            if (pending) {
                fs_drain<fs_ept<T>()>();
                if ((tid & 63) == 0 && atomicAdd(&arrive, 1u) == FS_NT / 64 - 1) {
                    arrive = 0;
                    q_count(pending);
                }
            }
            if (last) take_ticket();
        };
        auto loaded = [&]() {
            fs_release_mark();
            if (tid == 0) q_count(line(q.count));
        };
        auto mid = [&]() {
            if (wave0) aim(last ? 2u * __builtin_amdgcn_readfirstlane(taken) : uint32_t(k) + 1);
        };
        auto late = [&]() {
            if (wave0 && next_n) seen = peek(next_wait, next_n);
        };
        q_dispatch<T, S>(std::make_integer_sequence<int, Q_NCLASSES>{}, q.cls, q, in, out, ring, offs, ex, ltw, tw, ltid,
                         publish, loaded, mid, late);
        const int mode = q.cls % Q_MODES;
        pending = mode == Q_COL || mode == Q_ROWS ? line(q.count) : nullptr;
    }
    // Leave; the last group sets the counters for the next launch.
    fs_drain<0>();
    lds_barrier();
    uint32_t left = 0;  // (as k_fused4)
    if (tid == 0) {
        if (pending) q_count(pending);
        fs_drain<0>();
        left = __hip_atomic_fetch_add(line(Q_DONE), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
        sh[0] = left % gridDim.x == 0;
    }
    lds_barrier();
    if (sh[0]) {
        if (tid == 0) {
            __hip_atomic_store(line(Q_LAST), fs_peek(line(Q_TICKET)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(line(Q_TICKET), 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            fs_all_left(line(Q_DONE), left);
        }
        for (int i = Q_SLABS + tid; i < lines; i += FS_NT)
            __hip_atomic_store(line(i), init[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
}

}  // namespace nrfft
