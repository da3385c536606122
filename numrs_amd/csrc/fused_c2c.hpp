// fused_c2c.hpp -- both passes of a batched four-step C2C in one persistent
// kernel, the intermediate in a small ring that stays in the last-level cache.
//
// N = LA * LB, x viewed as [n1][n2] (n1 < LA, n2 < LB).  Pass A transforms
// columns of TA adjacent n2 (LA points each), times W_N^{k1 n2}; pass B
// transforms TB adjacent rows k1 (LB points each) into X[k2 LA + k1].  A tile
// of either pass is FS_TILE bytes (16384 FP32 / 8192 FP64 points), held in the
// registers of 512 threads.
//
// What bounds it: the fabric between the XCDs and the memory side.  HBM sees
// each point once in and once out, the last-level cache (MALL) the
// intermediate once in and once out; a copy kernel with these four streams,
// this tile shape and this ticket order takes 297 us for 64 x 2^20 FP32 on
// MI355X (random data; 2 GiB past the L2s, 7.2 TB/s), this kernel 324.  Two
// launches per batch chunk (k_c2c_dma / k_c2c) took 445: each pays a ramp and a
// drain, and their chunks have to be 64-128 MiB to fill the chip, so input,
// intermediate and output share the MALL.  FP64 45 x 2^18 150 -> 124 us.
//
// Groups take work from one ticket counter.  A ticket is a unit: A tile u,
// then B tile u - lead, with lead = `lag` slabs; a slab is 64 tiles
// of consecutive transforms (at least one transform), and slab s lies in ring
// slot s mod `slots`.  (One ticket a tile made the counter the limit: an atomic
// on one line takes about 40 ns here whoever asks, 8704 tickets 340 us.)
//
// Order and coherence.  The intermediate crosses XCDs, whose L2s are not
// coherent with each other: A stores it and B loads it at device scope (SC1:
// the store goes through to memory, the load does not hit a stale line), so
// no L2 write-back or invalidate is needed (and it costs nothing: 292 us
// against 293 with plain stores).  A group that has waited for its stores
// counts its tile in the slab's counter; a B tile starts once the counter has
// reached the slab's tiles.  An A tile that reuses a slot starts once the B
// tiles of the slab that was there have all loaded: one thread counts a B tile
// behind the first barrier of its exchange, which no wave passes without its values.  A tile depends only on
// units with smaller tickets, and a group that holds a ticket runs, so the
// smallest unfinished unit never waits: no deadlock, however few groups are
// resident.  Every wait is bounded all the same (a group polls FS_SPIN times in
// vain at most once, about a second), so misuse (one plan on two streams at once)
// gives wrong results, not a hang.  A group that gives up sets `expired`, which
// stays set until a check reads it (nrfft_plan_check).
//
// The last group to leave clears the counters, so a launch leaves the state
// as it found it and needs no reset launch or memset before it.  (Launches of one
// plan have equal grids.  If some overlapped against the rules, the very last group
// still brings the count of those that have left to a multiple of the grid, finds
// it unchanged and clears everything; a state that a plan gives back is cleared.)
#pragma once
#include "pass_c2c.hpp"
#include "real_fft.hpp"

namespace nrfft {

constexpr int FS_NT = 512;
constexpr int FS_MAX_SLOTS = 32;
constexpr int FS_SPIN = 1 << 20;

// Counters of a fused plan, each on a cache line of its own (operations on
// one line queue up behind each other).  All but `expired` are zero between
// launches.
struct FsState {
    uint32_t expired, pad0[31];  // a wait has given up
    uint32_t ticket, pad1[31];
    uint32_t done, pad2[31];
    uint32_t stored[FS_MAX_SLOTS][32];  // [slot][0]: A tiles of the slot's slabs that are stored
    uint32_t loaded[FS_MAX_SLOTS][32];  // [slot][0]: B tiles of the slot's slabs that are loaded
};

struct FsDesc {
    int32_t batch;       // transforms
    int32_t split;       // transforms of `in` and `out`; the others are those of `in2` and `out2`
    int32_t slab_log;    // log2 transforms per slab
    int32_t slots;       // ring slots (slabs)
    int32_t lag;         // slabs pass B trails pass A by, 1 .. slots - 1
};

template <typename T>
constexpr int fs_tile() {
    return sizeof(T) == 4 ? 16384 : 8192;
}
template <typename T>
constexpr int fs_ept() {
    return fs_tile<T>() / FS_NT;
}

// ---------------------------------------------------------------------------
// 32-point DFT: 4 x 8 (DFT4 down the columns j1 of x[8 j1 + j2], twiddle
// w32^(j2 k1), DFT8 along j2, output X[k1 + 4 k2]).
// ---------------------------------------------------------------------------
template <int S, int M, typename T>
__device__ __forceinline__ cpx<T> rot32(cpx<T> a) {
    if constexpr (M % 2 == 0) {
        return rot16<S, M / 2, true>(a);
    } else {
        // In 32 bits cos(pi/16) is the neighbour above (errors 2.99e-8 and 2.97e-8): see rot16.
        constexpr double c16 = sizeof(T) == 4 ? 0.98078531026840210 : 0.98078528040323044912618223613424;
        constexpr double c[4] = {c16, 0.83146961230254523707878837761791, 0.55557023301960222474283081394853,
                                 0.19509032201612826784828486847702};
        constexpr double s[4] = {0.19509032201612826784828486847702, 0.55557023301960222474283081394853,
                                 0.83146961230254523707878837761791, c16};
        // exp(i pi M / 16): M = 8 q + (1, 3, 5, 7), a quarter turn per 8
        constexpr int q = M / 8, h = (M % 8) / 2;
        constexpr double cr = q == 0 ? c[h] : q == 1 ? -s[h] : -c[h];
        constexpr double ci = q == 0 ? s[h] : q == 1 ? c[h] : -s[h];
        const T cc = (T)cr, ss = (T)((double)S * ci);
        return {a.x * cc - a.y * ss, a.x * ss + a.y * cc};
    }
}

template <int S, int K1, int J2, typename T>
__device__ __forceinline__ void rot32_row(cpx<T>* v) {
    if constexpr (J2 < 8) {
        v[8 * K1 + J2] = rot32<S, K1 * J2>(v[8 * K1 + J2]);
        rot32_row<S, K1, J2 + 1>(v);
    }
}

template <int S, typename T>
__device__ __forceinline__ void dft32(cpx<T>* v) {
#pragma unroll
    for (int j2 = 0; j2 < 8; ++j2) dft4<S>(v[j2], v[8 + j2], v[16 + j2], v[24 + j2]);
    rot32_row<S, 1, 1>(v);
    rot32_row<S, 2, 1>(v);
    rot32_row<S, 3, 1>(v);
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1) dft8<S>(v + 8 * k1);
    cpx<T> t[32];
#pragma unroll
    for (int k1 = 0; k1 < 4; ++k1)
#pragma unroll
        for (int k2 = 0; k2 < 8; ++k2) t[k1 + 4 * k2] = v[8 * k1 + k2];
#pragma unroll
    for (int i = 0; i < 32; ++i) v[i] = t[i];
}

template <int R, int S, typename T>
__device__ __forceinline__ void fs_dft(cpx<T>* v) {
    if constexpr (R == 32) dft32<S>(v);
    else if constexpr (R == 16) dft16<S, true>(v);
    else dft<R, S>(v);
}

// Radix plan of a tile's transforms: two stages (one exchange) where the
// values per thread allow it, else the plan of RadixPlan (stages from the third
// on read the global per-stage table).
template <int... RS>
struct FsRadices {
    static constexpr int NST = sizeof...(RS);
    static constexpr int R[NST] = {RS...};
};
template <int L>
using FsTablePlan = std::conditional_t<
    RadixPlan<L>::NST == 2, FsRadices<RadixPlan<L>::radix(0), RadixPlan<L>::radix(1)>,
    std::conditional_t<RadixPlan<L>::NST == 3,
                       FsRadices<RadixPlan<L>::radix(0), RadixPlan<L>::radix(1), RadixPlan<L>::radix(2)>,
                       FsRadices<RadixPlan<L>::radix(0), RadixPlan<L>::radix(1), RadixPlan<L>::radix(2),
                                 RadixPlan<L>::radix(3)>>>;
template <typename T, int L>
struct FsPlan : FsTablePlan<L> {};
template <typename T> struct FsPlan<T, 64> : FsRadices<8, 8> {};
template <> struct FsPlan<float, 512> : FsRadices<16, 32> {};
template <> struct FsPlan<float, 1024> : FsRadices<32, 32> {};

// Stage-1 twiddle rows in LDS: entry (k, r) at p[k ROW_ + r COL_].
template <typename T, int ROW_, int COL_>
struct FsLtw {
    static constexpr int ROW = ROW_, COL = COL_;
    const cpx<T>* p;
};

// ---------------------------------------------------------------------------
// Stage engine of one tile: EPT values per thread.  Stage 0 is mapped along
// (MAP_J) or across (MAP_T) the transforms, later stages by MAPS.  The exchanges
// move one real component at a time, so a tile needs half the LDS and two
// groups share a CU: one's loads and stores run under the other's arithmetic.
// LDS layout with gaps that keep the first exchange's writes in distinct
// banks (LANES lanes meet in the banks); elements of a transform are
//   MAPS = MAP_T  TI apart ([i][TI]).  Lanes across the transforms (MAPL =
//          MAP_T): LANES holds G = LANES / TI (at most 16) butterflies j; they
//          are taken L / (R0 G) apart (j = (jj mod G) L / (R0 G) + jj / G, jj =
//          thread / TI), and each of the G parts of the tile is moved on by TI
//          values.  Lanes along j (MAPL = MAP_J) write R0 TI apart: a gap after
//          every R0 TI values.
//   MAPS = MAP_J  contiguous ([t][L]), a gap of one after every LANES values.
// Reads and the later exchanges' writes take (nearly) consecutive addresses.
// ---------------------------------------------------------------------------
//
// PAIR = FS_PAIR_FIRST / FS_PAIR_LAST: the values of the first (last) stage are
// held in mirror pairs.  Lane l + 32 of a wave then has butterfly NB - 1 - j of
// transform t + TI / 2 where lane l has butterfly j of transform t < TI / 2, so
// element i of one and L - 1 - i of the other stand in registers r and R - 1 - r.
enum { FS_PAIR_FIRST = 1, FS_PAIR_LAST = 2 };
template <typename T, int S, int L, int MAPL, int MAPS = MAP_T, int PAIR = 0>
struct FsEng {
    static_assert(!(PAIR & FS_PAIR_FIRST) || MAPL == MAP_T, "pairs lie across the transforms");
    static_assert(!(PAIR & FS_PAIR_LAST) || MAPS == MAP_T, "pairs lie across the transforms");
    static_assert(MAPS == MAP_T || MAPL == MAP_J, "row stores come with row loads");
    using P = FsPlan<T, L>;
    static constexpr int EPT = fs_ept<T>(), NT = FS_NT, TI = fs_tile<T>() / L, NST = P::NST;
    static constexpr int R0 = P::R[0];
    static constexpr int ns(int s) {
        int n = 1;
        for (int q = 0; q < s; ++q) n *= P::R[q];
        return n;
    }
    static constexpr int RL = P::R[NST - 1];   // last radix
    static constexpr int NBL = L / RL;         // output k = j + r NBL
    static constexpr int LANES = 256 / (int)sizeof(T);
    static constexpr bool COLS = MAPL == MAP_T;  // stage 0 across the transforms
    static constexpr int G = (COLS && TI < LANES) ? (LANES / TI < 16 ? LANES / TI : 16) : 1;
    static constexpr int TS = MAPS == MAP_T ? TI : 1;  // distance of neighbouring elements
    static constexpr int BLK = MAPS == MAP_J ? LANES : COLS ? TI * L / G : R0 * TI;
    static constexpr int PADQ = MAPS == MAP_J ? 1 : COLS ? (G > 1 ? TI : 0) : (L / R0 >= LANES ? 1 : LANES / (L / R0));
    static constexpr int EX_ELEMS = TI * L + (TI * L / BLK) * PADQ;
    static constexpr bool parts_whole() {
        if (G == 1) return true;
        for (int s = 1; s < NST; ++s)
            if (P::R[s] % G) return false;
        return (L / R0) % G == 0;
    }
    static_assert(parts_whole(), "gaps fall on whole radix steps");
    static constexpr int phys(int raw) { return raw + raw / BLK * PADQ; }
    static __device__ __forceinline__ int raw_of(int t, int i) { return MAPS == MAP_T ? i * TI + t : t * L + i; }

    template <int s, class F>
    static __device__ __forceinline__ void each_butterfly(int tid, F&& f) {
        constexpr int R = P::R[s], NB = L / R, BPT = EPT / R;
        static_assert(BPT >= 1 && EPT % R == 0, "a thread holds whole butterflies");
#pragma unroll
        for (int b = 0; b < BPT; ++b) {
            const unsigned q = unsigned(tid) + unsigned(b * NT);
            int t, j;
            if constexpr ((s == 0 && (PAIR & FS_PAIR_FIRST)) || (s == NST - 1 && (PAIR & FS_PAIR_LAST))) {
                const unsigned ql = unsigned(tid / 64 * 32 + tid % 32) + unsigned(b * (NT / 2)), jj = ql / unsigned(TI / 2);
                const bool up = (tid & 32) != 0;
                j = (s == 0 && G > 1) ? int((jj % unsigned(G)) * unsigned(NB / G) + jj / unsigned(G)) : int(jj);
                t = int(ql % unsigned(TI / 2)) + (up ? TI / 2 : 0);
                j = up ? NB - 1 - j : j;
            } else if constexpr ((s == 0 ? MAPL : MAPS) == MAP_J) {
                t = int(q / unsigned(NB));
                j = int(q % unsigned(NB));
            } else {
                t = int(q % unsigned(TI));
                const unsigned jj = q / unsigned(TI);
                j = (s == 0 && G > 1) ? int((jj % unsigned(G)) * unsigned(NB / G) + jj / unsigned(G)) : int(jj);
            }
            f(b, t, j);
        }
    }
    // Component C (0 re, 1 im) of the stage-s outputs to LDS / of the
    // stage-s inputs from it.
    template <int s, int C>
    static __device__ __forceinline__ void put(const cpx<T>* v, int tid, T* ex) {
        constexpr int R = P::R[s], NS = ns(s);
        each_butterfly<s>(tid, [&](int b, int t, int j) {
            T* base = ex + phys(raw_of(t, (j / NS) * NS * R + (j % NS)));
            // Columns: a butterfly's outputs lie in one gap-free part.  Rows in,
            // columns out: R0 of them do (s = 0), or they lie whole parts apart.
            // Rows: at compile-time distances (NS divides LANES or is a multiple).
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int o = r * NS * TS + (MAPS == MAP_J ? r * NS / LANES : COLS || s == 0 ? 0 : r * (NS / R0) * PADQ);
                base[o] = C == 0 ? v[b * R + r].x : v[b * R + r].y;
            }
        });
    }
    template <int s, int C>
    static __device__ __forceinline__ void get(cpx<T>* v, int tid, const T* ex) {
        constexpr int R = P::R[s], NB = L / R;
        each_butterfly<s>(tid, [&](int b, int t, int j) {
            // element j + r NB: r alone says in which part it lies (columns), or
            // r NB TS / BLK is its share of the gaps
            const T* base = ex + (COLS ? j * TI + t : phys(raw_of(t, j)));
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int o = r * NB * TS + (r * NB * TS) / BLK * PADQ;
                if constexpr (C == 0) v[b * R + r].x = base[o];
                else v[b * R + r].y = base[o];
            }
        });
    }
    // Stage 1's twiddles W_{NS R}^{r k} come from LDS (FsLtw: rows k; by default NS
    // rows of R + 2 entries, exact entries of the coarse table), later ones from
    // the per-stage table.
    static constexpr int TW_ELEMS = ns(1) * (P::R[1] + 2);
    static __device__ __forceinline__ void fill_tw(cpx<T>* ltw, const cpx<T>* coarse, int tid) {
        constexpr int R = P::R[1], NS = ns(1);
        for (int e = tid; e < NS * R; e += NT) {
            const int k = e / R, r = e % R;
            ltw[k * (R + 2) + r] = coarse[(r * k) * (TW_COARSE / (NS * R))];
        }
    }
    using Ltw = FsLtw<T, P::R[1] + 2, 1>;
    template <int s, class LTW>
    static __device__ __forceinline__ void twiddle(cpx<T>* v, int tid, LTW ltw, const cpx<T>* stage_tw) {
        constexpr int R = P::R[s], NS = ns(s), RS = s == 1 ? LTW::COL : 1;
        each_butterfly<s>(tid, [&](int b, int, int j) {
            const cpx<T>* row = s == 1 ? ltw.p + (j % NS) * LTW::ROW
                                       : stage_tw + 2 * L + StageTable<L>::off(s) + (j % NS) * R;
#pragma unroll
            for (int r = 1; r < R; ++r) v[b * R + r] = cmul(v[b * R + r], dirw<S>(row[r * RS]));
        });
    }
    template <int s>
    static __device__ __forceinline__ void butterflies(cpx<T>* v) {
        constexpr int R = P::R[s];
#pragma unroll
        for (int b = 0; b < EPT / R; ++b) fs_dft<R, S>(v + b * R);
    }
    // Stages 1 .. NST-1; stage 0's outputs are in v.  Hook behind the first
    // exchange's first barrier: `read`; there every wave has written outputs of all
    // its stage-0 butterflies, so each value the group loaded has arrived.  Hooks in
    // the last exchange: `pre` before it, `mid` behind its first barrier, `late`
    // before its last read.
    template <int s = 1, class LTW, class READ, class PRE, class MID, class LATE>
    static __device__ __forceinline__ void rest(cpx<T>* v, int tid, T* ex, LTW ltw, const cpx<T>* stage_tw, READ&& read,
                                                PRE&& pre, MID&& mid, LATE&& late) {
        static_assert(NST == 2 || std::is_base_of_v<FsTablePlan<L>, P>, "stage 2 reads the per-stage table");
        if constexpr (s < NST) {
            if constexpr (s > 1) lds_barrier();  // the previous exchange has been read
            if constexpr (s == NST - 1) pre();
            put<s - 1, 0>(v, tid, ex);
            lds_barrier();
            if constexpr (s == 1) read();
            if constexpr (s == NST - 1) mid();
            get<s, 0>(v, tid, ex);
            lds_barrier();
            put<s - 1, 1>(v, tid, ex);
            lds_barrier();
            if constexpr (s == NST - 1) late();
            get<s, 1>(v, tid, ex);
            twiddle<s>(v, tid, ltw, stage_tw);
            butterflies<s>(v);
            rest<s + 1>(v, tid, ex, ltw, stage_tw, read, pre, mid, late);
        }
    }
};

// Four-step twiddles W_N^{S n2 (j + r NB)}, r < R (N = 2^logn), of a thread's
// BPT last-stage butterflies (one n2): factors a[h] b[l] for r = 4 h + l, a[h]
// = W^{n2 (j + 4 h NB)}, b[l] = W^{n2 l NB}.  Every second a[h] and the b[l]
// (FP64: b[1], b[2]) are table products, so a factor is at most three products
// away from them.
// The table values are loaded before the last exchange and joined behind its
// first barrier: loaded with the tile they took 32 registers through the first
// stages (64 x 2^20 FP32 337 us against 324; FP64 C2C 2^19 and 2^20 spilled).  All
// a[h] from the tables: 2% less error in FP32, 2 to 4% more time.
template <typename T, int S, int R, int BPT, int NB>
struct FsTw {
    static_assert(R >= 8 && R % 8 == 0, "last radix 8, 16 or 32");
    static constexpr bool B3 = sizeof(T) == 4;  // b3 from the tables too
    static constexpr int H = R / 4, A0 = B3 ? 4 : 3, NP = A0 + BPT * (H / 2);
    cpx<T> x[NP], y[NP];  // table values, then x: b1, b2, W^{4 n2 NB}, (b3,) a[0], a[2], ..
    __device__ __forceinline__ void load(const Twiddles<T>& tw, uint32_t n2, const uint32_t* j, int logn) {
        const uint32_t mask = (1u << logn) - 1u, st = n2 * uint32_t(NB);
#pragma unroll
        for (int i = 0; i < A0; ++i) twiddle_parts(tw, (i == 3 ? 3 * st : st << i) & mask, logn, x[i], y[i]);
#pragma unroll
        for (int b = 0; b < BPT; ++b)
#pragma unroll
            for (int h = 0; h < H / 2; ++h)
                twiddle_parts(tw, (n2 * j[b] + uint32_t(8 * h) * st) & mask, logn, x[A0 + b * (H / 2) + h],
                              y[A0 + b * (H / 2) + h]);
    }
    __device__ __forceinline__ void join() {
#pragma unroll
        for (int i = 0; i < NP; ++i) x[i] = twiddle_join<S>(x[i], y[i]);
    }
    __device__ __forceinline__ void apply(cpx<T>* v) const {
        const cpx<T> b1 = x[0], b2 = x[1], p4 = x[2], b3 = B3 ? x[3] : cmul(b1, b2);
#pragma unroll
        for (int b = 0; b < BPT; ++b)
#pragma unroll
            for (int h = 0; h < H / 2; ++h) {
                const cpx<T> a0 = x[A0 + b * (H / 2) + h], a1 = cmul(a0, p4);
                cpx<T>* w = v + b * R + 8 * h;
                w[0] = cmul(w[0], a0);
                w[1] = cmul(w[1], cmul(a0, b1));
                w[2] = cmul(w[2], cmul(a0, b2));
                w[3] = cmul(w[3], cmul(a0, b3));
                w[4] = cmul(w[4], a1);
                w[5] = cmul(w[5], cmul(a1, b1));
                w[6] = cmul(w[6], cmul(a1, b2));
                w[7] = cmul(w[7], cmul(a1, b3));
            }
    }
};

// ---------------------------------------------------------------------------
// Buffer accesses: a 128-bit resource per tile base, one 32-bit offset
// register per thread and constant steps in scalar registers.
// ---------------------------------------------------------------------------
typedef unsigned fs_u2 __attribute__((ext_vector_type(2)));
typedef unsigned fs_u4 __attribute__((ext_vector_type(4)));
constexpr int FS_AUX_NT = 2, FS_AUX_SC1 = 16;

__device__ __forceinline__ __amdgpu_buffer_rsrc_t fs_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, (int)bytes, 0x00020000);
}
template <typename T, int AUX>
__device__ __forceinline__ cpx<T> fs_load(__amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(T) == 4) {
        return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b64(r, (int)voff, (int)soff, AUX));
    } else {
        return __builtin_bit_cast(cpx<T>, __builtin_amdgcn_raw_buffer_load_b128(r, (int)voff, (int)soff, AUX));
    }
}
template <typename T, int AUX>
__device__ __forceinline__ void fs_store(cpx<T> v, __amdgpu_buffer_rsrc_t r, uint32_t voff, uint32_t soff) {
    if constexpr (sizeof(T) == 4) {
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(fs_u2, v), r, (int)voff, (int)soff, AUX);
    } else {
        // No scalar offset register: with one, 16-byte stores were seen to
        // write data of a later VALU result (lanes 12-15 of 16; the compiler
        // keeps the wait states that a store of more than 8 bytes needs
        // before its data registers change only for stores without one).
        __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(fs_u4, v), r, (int)(voff + soff), 0, AUX);
    }
}

// At most N vector memory operations of this wave are outstanding.
template <int N = 0>
__device__ __forceinline__ void fs_drain() {
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ uint32_t fs_peek(const uint32_t* p) {
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void fs_count(uint32_t* p) {
    __hip_atomic_fetch_add(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ void fs_flag(uint32_t* p) {
    __hip_atomic_store(p, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// The count of groups that have left back to 0 unless more have left since.
__device__ __forceinline__ void fs_all_left(uint32_t* done, uint32_t left) {
    __hip_atomic_compare_exchange_strong(done, &left, 0u, __ATOMIC_RELAXED, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Where a ring slot's tile is counted as loaded: the next tile's stores to the slot
// may follow.  (The comment marks the place in the assembly, where
// tests/test_ring_release.py finds every load from the ring waited for.)
__device__ __forceinline__ void fs_release_mark() { asm volatile("; ring slot released" ::: "memory"); }

// ---------------------------------------------------------------------------
// The untangle of a real transform (untangle_pair, real_fft.hpp) on mirror pairs
// in registers: bins p and N - p of the packed signal stand in registers r and
// R - 1 - r of a thread and of the one 32 lanes away (FS_PAIR_*).
// ---------------------------------------------------------------------------
// exp(i pi r / R), r < R <= 32.
template <int R, int r, typename T>
__device__ __forceinline__ cpx<T> fs_half_root() {
    constexpr double c[17] = {1.0, 0.99518472667219688624483695310948, 0.98078528040323044912618223613424,
                              0.95694033573220886493579788698027, 0.92387953251128675612818318939679,
                              0.88192126434835502971275686366039, 0.83146961230254523707878837761791,
                              0.77301045336273696081090660975847, 0.70710678118654752440084436210485,
                              0.63439328416364549821517161322549, 0.55557023301960222474283081394853,
                              0.47139673682599764855638762590525, 0.38268343236508977172845998403040,
                              0.29028467725446236763619237581740, 0.19509032201612826784828486847702,
                              0.09801714032956060199419556388864, 0.0};
    constexpr int k = r * (32 / R);
    constexpr double re = k <= 16 ? c[k <= 16 ? k : 0] : -c[k <= 16 ? 0 : 32 - k];
    constexpr double im = c[k <= 16 ? 16 - k : k - 16];
    return {(T)re, (T)im};
}
// The value of the lane 32 away.
__device__ __forceinline__ float fs_cross(float x, bool up) {
    const unsigned u = __builtin_bit_cast(unsigned, x);
    const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);  // {low half twice, high half twice}
    return __builtin_bit_cast(float, up ? r[0] : r[1]);
}
__device__ __forceinline__ double fs_cross(double x, bool up) {
    const auto u = __builtin_bit_cast(fs_u2, x);
    const auto a = __builtin_amdgcn_permlane32_swap(u[0], u[0], false, false);
    const auto b = __builtin_amdgcn_permlane32_swap(u[1], u[1], false, false);
    return __builtin_bit_cast(double, fs_u2{up ? a[0] : a[1], up ? b[0] : b[1]});
}
template <typename T>
__device__ __forceinline__ cpx<T> fs_cross(cpx<T> v, bool up) {
    return {fs_cross(v.x, up), fs_cross(v.y, up)};
}
// Butterfly of R values at v, w0 = exp(i pi p / N) of its bin r = 0 (DIR = -1:
// the conjugate).  v[R - 1 - r] becomes the mirror of v[r]'s bin, r < R / 2.
template <int DIR, int R, int r = 0, typename T>
__device__ __forceinline__ void fs_untangle(cpx<T>* v, cpx<T> w0, bool up) {
    if constexpr (r < R / 2) {
        const cpx<T> w = cmul(w0, dirw<DIR>(fs_half_root<R, r, T>()));
        cpx<T> x, y;
        untangle_pair(v[r], fs_cross(v[R - 1 - r], up), w, (T)(-0.5 * DIR), x, y);
        v[r] = x;
        v[R - 1 - r] = y;
        fs_untangle<DIR, R, r + 1>(v, w0, up);
    }
}
// Likewise of a transform that is its own mirror, partner(r) = the value at the
// mirror of bin r: v[r] stays bin r.  dc: v[0] is bin 0.
template <int DIR, int R, int r = 0, typename T, class P>
__device__ __forceinline__ void fs_untangle_self(cpx<T>* v, cpx<T> w0, bool dc, P&& partner) {
    if constexpr (r < R) {
        const cpx<T> w = cmul(w0, dirw<DIR>(fs_half_root<R, r, T>()));
        cpx<T> x, y;
        untangle_pair(v[r], partner(r), w, (T)(-0.5 * DIR), x, y);
        v[r] = r == 0 && dc ? (DIR > 0 ? dc_forward(v[r]) : dc_inverse(v[r])) : x;
        fs_untangle_self<DIR, R, r + 1>(v, w0, dc, partner);
    }
}

template <typename T, int LA, int LB>
struct FsShape {
    static constexpr int TILE = fs_tile<T>();
    static constexpr int TA = TILE / LA, TB = TILE / LB;
    static constexpr int64_t N = int64_t(LA) * LB;
    static constexpr int NTA = LB / TA, NTB = LA / TB;  // tiles per transform (equal: N / TILE)
    static_assert(TA <= LB && TB <= LA, "a tile lies in one transform");
    static_assert(NTA == NTB, "both passes have N / TILE tiles");
    static constexpr int LOGN = ilog2c(N);
    static constexpr bool SAME_TW = LA == LB;
    using EA = FsEng<T, 1, LA, MAP_T>;
    using EB = FsEng<T, 1, LB, MAP_J>;
    static constexpr int EX = EA::EX_ELEMS > EB::EX_ELEMS ? EA::EX_ELEMS : EB::EX_ELEMS;
    static constexpr int TWA = EA::TW_ELEMS, TWB = SAME_TW ? 1 : EB::TW_ELEMS;
    static_assert(EX * (int)sizeof(T) + (TWA + TWB) * (int)sizeof(cpx<T>) + 64 <= 81920, "two groups share a CU");
};

// Vector memory operations complete in order, so what a group waits for is
// issued ahead of the stores that would otherwise hold it up: wave 0 takes
// the next ticket behind a tile's loads and looks at the next tile's counter
// before the tile's stores.  The wave priority rises through a tile, so of a
// CU's two groups the one further along finishes first (oldest-first issue let
// the younger group's A tiles take 30 us beside 14, and every slab waits for
// its slowest tile: 311 -> 302 us with a lag of 8 slabs, zero data).
//
// RE = 1: the forward transform of 2 N reals (S = 1), RE = -1: its inverse (S =
// -1); N and the tables are those of the packed signal.  Bin p = k2 LA + k1 pairs
// with N - p in row LA - k1 (row 0 with itself, row LA / 2 too), so a pass-B tile of
// RE = 1 holds TB / 2 rows k1 = c .. and their mirror rows, taken from the ring
// where they lie; the rows 0 and LA / 2 share a pair's place and are untangled
// through the LDS.  RE = -1 takes column tiles likewise (columns n2 and LB - n2),
// untangles before pass A, and pass B picks the columns up in their order.  So the
// untangle costs no pass over memory.  64 x 2^19 reals FP32 forward 99 us, inverse
// 98, in passes 158 and 129; 36 x 2^20 130 and 101 against 198 and 131.  What it pays
// instead: half as long runs in memory, one of two at an odd element (11% of the
// forward's write requests are below 64 bytes).
//
// RE = -2: the inverse of the correlation of the spectra `in` and `in2`: as RE = -1
// on a conj(b) / N, taken where a tile is loaded (b in pieces of 8 values a thread;
// more would not fit beside a).
//
// 128 registers a thread (two groups a CU).  The C2C forms keep to them; of the others
// the FP32 inverses of 2^20 and 2^21 points spill 112 and 116 bytes a lane, the FP32
// forwards from 2^18 and most FP64 ones 8 to 40.
template <typename T, int S, int LA, int LB, int RE = 0>
__global__ __attribute__((amdgpu_flat_work_group_size(FS_NT, FS_NT), amdgpu_waves_per_eu(4, 4))) void
k_fused4(const cpx<T>* in, cpx<T>* out, cpx<T>* ring, FsState* st, FsDesc d, Twiddles<T> tw, const cpx<T>* in2,
         cpx<T>* out2) {
    static_assert(RE == 0 || (RE > 0) == (S > 0), "forward untangles behind, the inverse ahead");
    using SH = FsShape<T, LA, LB>;
    using EA = FsEng<T, S, LA, MAP_T, MAP_T, (RE < 0 ? FS_PAIR_FIRST : 0)>;
    using EB = FsEng<T, S, LB, MAP_J, MAP_T, (RE > 0 ? FS_PAIR_LAST : 0)>;
    constexpr int TILE = SH::TILE, TA = SH::TA, TB = SH::TB, EPT = fs_ept<T>(), CS = (int)sizeof(cpx<T>);
    constexpr int TPT_LOG = ilog2c(SH::NTA);  // tiles per transform
    constexpr int64_t N = SH::N;
    constexpr int LOGN = SH::LOGN;
    __shared__ __align__(16) T ex[SH::EX];
    __shared__ __align__(16) cpx<T> ltwa[SH::TWA];
    __shared__ __align__(16) cpx<T> ltwb_[SH::TWB];
    __shared__ uint32_t sh[2], arrive;
    const cpx<T>* ltwb = SH::SAME_TW ? ltwa : ltwb_;
    const int tid = threadIdx.x;

    const uint32_t slab_tiles_log = uint32_t(TPT_LOG + d.slab_log), slab_mask = (1u << slab_tiles_log) - 1u;
    const uint32_t nt = uint32_t(d.batch) << TPT_LOG;  // tiles of one pass
    const uint32_t lead = uint32_t(d.lag) << slab_tiles_log;
    const uint32_t nlead = lead < nt ? lead : nt;
    // A ticket u is a unit of work: A tile u (u < nt), then B tile u - nlead
    // (u >= nlead).  Task 2 u is the unit's A tile, 2 u + 1 its B tile.
    const uint32_t units = nt + nlead;
    struct Task {
        bool b;
        uint32_t tile, slot, gen, in_slab;  // in_slab: tiles of the slab (the last may be short)
    };
    auto task_of = [&](uint32_t k) {
        Task t;
        t.b = (k & 1) != 0;
        t.tile = t.b ? (k >> 1) - nlead : k >> 1;
        const uint32_t slab = t.tile >> slab_tiles_log;
        t.gen = slab / uint32_t(d.slots);
        t.slot = slab - t.gen * uint32_t(d.slots);
        const uint32_t left = nt - (slab << slab_tiles_log);
        t.in_slab = left < slab_mask + 1 ? left : slab_mask + 1;
        return t;
    };
    auto first_of = [&](uint32_t u) { return u < nt ? 2 * u : 2 * u + 1; };
    auto last_of_unit = [&](uint32_t k) { return (k & 1) != 0 || (k >> 1) < nlead; };
    // The counter a task waits for and the value it needs.
    auto waits_on = [&](const Task& t) -> const uint32_t* { return t.b ? st->stored[t.slot] : st->loaded[t.slot]; };
    auto need_of = [&](const Task& t) {
        return t.b ? (t.gen << slab_tiles_log) + t.in_slab : t.gen << slab_tiles_log;
    };
    // Wave 0 takes the tickets and watches the counters; its decisions are
    // scalar (a ticket is read from lane 0 once it has arrived).
    const bool wave0 = __builtin_amdgcn_readfirstlane(tid >> 6) == 0;
    uint32_t taken = 0;            // lane 0: the ticket as it arrives
    uint32_t next = 0, seen = 0;   // wave 0: the coming task, and its counter as last read
    int patience = FS_SPIN;        // polls
    uint32_t* pending = nullptr;   // counter of the group's last A tile, its stores perhaps in flight
    // (Through a pointer the compiler must take for lane-dependent: for a
    // uniform one it broadcasts the result at once, i.e. waits for the atomic
    // and every operation before it.)
    auto take_ticket = [&]() {
        if (tid == 0)
            taken = __hip_atomic_fetch_add(&st->ticket + fresh_tid(0), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };
    auto look = [&](uint32_t k) {
        if (wave0) {
            next = last_of_unit(k) ? first_of(__builtin_amdgcn_readfirstlane(taken)) : k + 1;
            if (next < 2 * units) seen = fs_peek(waits_on(task_of(next)));
        }
    };
    if (tid == 0) arrive = 0;  // (before the first barrier)
    take_ticket();
    EA::fill_tw(ltwa, tw.coarse, tid);
    if constexpr (!SH::SAME_TW) EB::fill_tw(ltwb_, tw.coarse, tid);
    if (wave0) next = first_of(__builtin_amdgcn_readfirstlane(taken));
    for (;;) {
        if (wave0) {
            const bool ok = next < 2 * units && uint32_t(__builtin_amdgcn_readfirstlane(int(seen))) >= need_of(task_of(next));
            if (tid == 0) {
                sh[0] = next;
                sh[1] = ok;
            }
        }
        lds_barrier();  // also: the previous tile's exchange has been read
        const uint32_t k = __builtin_amdgcn_readfirstlane(sh[0]);
        const bool ready = __builtin_amdgcn_readfirstlane(sh[1]) != 0;
        if (k >= 2 * units) break;
        const Task t = task_of(k);
        if (!ready) {
            // Publish the last A tile before waiting for anything.
            if (pending) {
                fs_drain<0>();
                lds_barrier();
                if (tid == 0) fs_count(pending);
                pending = nullptr;
            }
            if (wave0) {
                const uint32_t* p = waits_on(t);
                const uint32_t need = need_of(t);
                int i = 0;
                for (; i < patience; ++i) {
                    if (__builtin_amdgcn_readfirstlane(fs_peek(p)) >= need) break;
                    __builtin_amdgcn_s_sleep(8);
                }
                if (i == patience) {
                    patience = 0;
                    if (tid == 0) fs_flag(&st->expired);
                }
            }
            lds_barrier();
        }
        const uint32_t tr = t.tile >> TPT_LOG, idx = t.tile & ((1u << TPT_LOG) - 1u);  // transform, its tile
        const uint32_t in_slot = tr & ((1u << d.slab_log) - 1u);
        cpx<T>* rt = ring + ((int64_t(t.slot) << d.slab_log) + in_slot) * N;  // this transform's intermediate
        cpx<T> v[EPT];
        const int ltid = fresh_tid(tid);
        // Once a tile's loads are issued, a wave with no more operations
        // outstanding than those has finished the stores before them; the
        // group's last such wave counts the previous A tile as stored.
        auto publish = [&]() {
            if (!pending) return;
            fs_drain<EPT>();
            if ((tid & 63) == 0 && atomicAdd(&arrive, 1u) == FS_NT / 64 - 1) {
                arrive = 0;
                fs_count(pending);
            }
        };
        // Column (RE < 0) or row (RE > 0) tt of the tile.
        auto paired = [&](int tt, int half, int len) {
            const uint32_t u = idx * uint32_t(half) + uint32_t(tt & (half - 1));
            return tt < half ? u : u ? uint32_t(len) - u : uint32_t(len / 2);
        };
        auto column = [&](int tt) -> uint32_t {
            if constexpr (RE < 0) return paired(tt, TA / 2, LB);
            else return idx * uint32_t(TA) + uint32_t(tt);
        };
        // Untangle of the tile's mirror pairs, transforms of
        // length L in butterflies of radix R: each(f) goes through the butterflies, bin(t, j) is the bin of
        // a butterfly's first value; back: the mirrors return to their threads.
        auto untangle = [&](auto radix, auto len, cpx<T>* x, int id, auto&& each, auto&& bin, bool back) {
            constexpr int R = decltype(radix)::value, L = decltype(len)::value, NB = L / R;
            const bool up = (id & 32) != 0;
            constexpr int HALF = TILE / L / 2;
            auto own = [&](int tt) { return idx == 0 && (tt & (HALF - 1)) == 0; };
            if (idx == 0) {  // transforms that are their own mirrors
                cpx<T>* z = reinterpret_cast<cpx<T>*>(ex) + (up ? L : 0);
                lds_barrier();
                each([&](int b, int tt, int j) {
                    if (own(tt))
#pragma unroll
                        for (int r = 0; r < R; ++r) z[j + r * NB] = x[b * R + r];
                });
                lds_barrier();
                each([&](int b, int tt, int j) {
                    if (own(tt))
                        fs_untangle_self<(RE > 0 ? 1 : -1), R>(x + b * R, twiddle_big<S>(tw, bin(tt, j), LOGN + 1), j == 0 && !up,
                                                [&](int r) {
                                                    const int k = j + r * NB;
                                                    return z[up ? L - 1 - k : (L - k) & (L - 1)];
                                                });
                });
                lds_barrier();
            }
            each([&](int b, int tt, int j) {
                if (!own(tt)) {
                    fs_untangle<(RE > 0 ? 1 : -1), R>(x + b * R, twiddle_big<S>(tw, bin(tt, j), LOGN + 1), up);
                    if (back)
#pragma unroll
                        for (int r = R / 2; r < R; ++r) x[b * R + r] = fs_cross(x[b * R + r], up);
                }
            });
        };
        const bool second = RE != -2 && tr >= uint32_t(d.split);
        const int64_t at = int64_t(second ? tr - uint32_t(d.split) : tr) * N;
        if (!t.b) {
            const __amdgpu_buffer_rsrc_t rin = fs_rsrc((second ? in2 : in) + at, uint32_t(N * CS));
            // x[(j + r NB0) LB + idx TA + t]
            EA::template each_butterfly<0>(ltid, [&](int b, int tt, int j) {
                constexpr int R = EA::R0, NB = LA / R;
                const uint32_t voff = uint32_t(j * LB) * CS + (RE < 0 ? column(tt) * uint32_t(CS) : uint32_t(tt * CS));
#pragma unroll
                for (int r = 0; r < R; ++r)
                    v[b * R + r] = fs_load<T, FS_AUX_NT>(
                        rin, voff, uint32_t(r * NB * LB) * CS + (RE < 0 ? 0u : idx * uint32_t(TA * CS)));
            });
            publish();
            if (last_of_unit(k)) take_ticket();
            FsTw<T, S, EA::RL, EPT / EA::RL, EA::NBL> f;
            auto load_tw = [&]() {
                uint32_t n2 = 0, jl[EPT / EA::RL];
                EA::template each_butterfly<EA::NST - 1>(ltid, [&](int b, int tt, int j) {
                    n2 = column(tt);  // the same for every b
                    jl[b] = uint32_t(j);
                });
                f.load(tw, n2, jl, LOGN);
            };
            __builtin_amdgcn_s_setprio(1);
            if constexpr (RE == -2) {
                const __amdgpu_buffer_rsrc_t ry = fs_rsrc(in2 + at, uint32_t(N * CS));
                constexpr T scale = (T)1 / (T)N;
                EA::template each_butterfly<0>(ltid, [&](int b, int tt, int j) {
                    constexpr int R = EA::R0, NB = LA / R, U = R < 8 ? R : 8;
                    const uint32_t voff = (uint32_t(j * LB) + column(tt)) * uint32_t(CS);
                    const bool dc = voff == 0;  // [F_0, F_N] in one slot
#pragma unroll
                    for (int r0 = 0; r0 < R; r0 += U) {
                        cpx<T> y[U];
#pragma unroll
                        for (int u = 0; u < U; ++u) y[u] = fs_load<T, FS_AUX_NT>(ry, voff, uint32_t((r0 + u) * NB * LB) * CS);
#pragma unroll
                        for (int u = 0; u < U; ++u) {
                            cpx<T>& x = v[b * R + r0 + u];
                            const cpx<T> q = spec_apply(OP_CORREL, x, y[u], scale);
                            if (r0 + u == 0)
                                x = cpx<T>{dc ? spec_apply_real(OP_CORREL, x.x, y[u].x, scale) : q.x,
                                           dc ? spec_apply_real(OP_CORREL, x.y, y[u].y, scale) : q.y};
                            else x = q;
                        }
                    }
                });
            }
            if constexpr (RE < 0) {
                untangle(
                    std::integral_constant<int, EA::R0>{}, std::integral_constant<int, LA>{}, v, ltid,
                    [&](auto&& f) { EA::template each_butterfly<0>(ltid, f); },
                    [&](int tt, int j) { return uint32_t(j * LB) + column(tt); }, true);
            }
            EA::template butterflies<0>(v);
            EA::rest(
                v, ltid, ex, typename EA::Ltw{ltwa}, tw.stage, []() {}, load_tw,
                [&]() {
                    __builtin_amdgcn_s_setprio(2);
                    f.join();
                },
                [&]() {
                    look(k);
                    __builtin_amdgcn_s_setprio(3);
                });
            f.apply(v);
            // ring: [block b = k1 / TB][block a = idx][k1 mod TB][n2 mod TA]
            const __amdgpu_buffer_rsrc_t rr = fs_rsrc(rt, uint32_t(N * CS));
            EA::template each_butterfly<EA::NST - 1>(ltid, [&](int b, int tt, int j) {
                constexpr int R = EA::RL, NB = EA::NBL;
                static_assert(NB % TB == 0 || TB % NB == 0, "output steps are constant");
                const uint32_t voff = uint32_t((j / TB) * TILE + (j % TB) * TA + tt) * CS;
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const uint32_t so = uint32_t(((r * NB) / TB) * TILE + ((r * NB) % TB) * TA) * CS;
                    fs_store<T, FS_AUX_SC1>(v[b * R + r], rr, voff, so + idx * uint32_t(TB * TA * CS));
                }
            });
            __builtin_amdgcn_s_setprio(0);
            pending = st->stored[t.slot];
        } else {
            // row t, element i: (i / TA) TB TA + t TA + i mod TA from its tile
            const __amdgpu_buffer_rsrc_t rr =
                RE > 0 ? fs_rsrc(rt, uint32_t(N * CS)) : fs_rsrc(rt + int64_t(idx) * TILE, uint32_t(TILE * CS));
            EB::template each_butterfly<0>(ltid, [&](int b, int tt, int j) {
                constexpr int R = EB::R0, NB = LB / R, H = TA / 2;
                static_assert(NB % TA == 0 || TA % NB == 0, "input steps are constant");
                uint32_t row = uint32_t(tt * TA);
                if constexpr (RE > 0) {
                    const uint32_t k1 = paired(tt, TB / 2, LA);
                    row = (k1 / TB) * uint32_t(TILE) + (k1 % TB) * uint32_t(TA);
                }
                if constexpr (RE < 0) {
                    // column n2 < LB / 2 is column n2 mod H of tile n2 / H, its mirror LB - n2 (column
                    // 0: LB / 2) the one H further on
                    auto at = [&](uint32_t n) { return (n / H) * uint32_t(TB * TA) + n % H; };
#pragma unroll
                    for (int r = 0; r < R; ++r) {
                        uint32_t voff, soff;
                        if constexpr (NB % H == 0) {  // steps are constant
                            if (r < R / 2) {
                                voff = at(uint32_t(j));
                                soff = uint32_t((r * NB) / H * (TB * TA));
                            } else {
                                voff = at(uint32_t(NB - j)) + H;
                                soff = uint32_t(((R - 1 - r) * NB) / H * (TB * TA));
                                if (r == R / 2 && j == 0) voff = H - soff;
                            }
                        } else {
                            const uint32_t n2 = uint32_t(j + r * NB);
                            voff = n2 < uint32_t(LB / 2) ? at(n2) : at(n2 == LB / 2 ? 0u : uint32_t(LB) - n2) + H;
                            soff = 0;
                        }
                        v[b * R + r] = fs_load<T, FS_AUX_SC1>(rr, (voff + soff + row) * uint32_t(CS), 0);
                    }
                } else {
                    const uint32_t voff = ((j / TA) * uint32_t(TB * TA) + row + uint32_t(j % TA)) * uint32_t(CS);
#pragma unroll
                    for (int r = 0; r < R; ++r)
                        v[b * R + r] = fs_load<T, FS_AUX_SC1>(
                            rr, voff, uint32_t(((r * NB) / TA) * (TB * TA) + (r * NB) % TA) * CS);
                }
            });
            publish();
            if (last_of_unit(k)) take_ticket();
            __builtin_amdgcn_s_setprio(1);
            EB::template butterflies<0>(v);
            EB::rest(
                v, ltid, ex, typename EB::Ltw{ltwb}, tw.stage,
                [&]() {
                    fs_release_mark();
                    if (tid == 0) fs_count(st->loaded[t.slot]);
                },
                []() {}, []() { __builtin_amdgcn_s_setprio(2); },
                [&]() {
                    look(k);
                    __builtin_amdgcn_s_setprio(3);
                });
            const __amdgpu_buffer_rsrc_t ro = fs_rsrc((second ? out2 : out) + at, uint32_t(N * CS));
            if constexpr (RE > 0)
                untangle(
                    std::integral_constant<int, EB::RL>{}, std::integral_constant<int, LB>{}, v, ltid,
                    [&](auto&& f) { EB::template each_butterfly<EB::NST - 1>(ltid, f); },
                    [&](int tt, int j) { return uint32_t(j * LA) + paired(tt, TB / 2, LA); }, false);
            EB::template each_butterfly<EB::NST - 1>(ltid, [&](int b, int tt, int j) {
                constexpr int R = EB::RL, NB = EB::NBL;
                uint32_t voff = uint32_t(j * LA + tt) * CS, mirror = voff;
                if constexpr (RE > 0) {
                    const uint32_t k1 = paired(tt, TB / 2, LA);
                    voff = (uint32_t(j * LA) + k1) * uint32_t(CS);
                    mirror = idx == 0 && (tt & (TB / 2 - 1)) == 0
                                 ? voff
                                 : (uint32_t((NB - 1 - j) * LA) + uint32_t(LA) - k1) * uint32_t(CS);
                }
#pragma unroll
                for (int r = 0; r < R; ++r)
                    fs_store<T, FS_AUX_NT>(v[b * R + r], ro, r < R / 2 ? voff : mirror,
                                           uint32_t(r * NB * LA) * CS + (RE > 0 ? 0u : idx * uint32_t(TB * CS)));
            });
            __builtin_amdgcn_s_setprio(0);
            pending = nullptr;
        }
    }
    // Leave: the last A tile counted, then the group; the last group clears
    // the state (nobody reads it any more).
    fs_drain<0>();
    lds_barrier();
    uint32_t left = 0;  // thread 0: groups that have left, this one included
    if (tid == 0) {
        if (pending) fs_count(pending);
        fs_drain<0>();
        left = __hip_atomic_fetch_add(&st->done, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1;
        sh[0] = left % gridDim.x == 0;
    }
    lds_barrier();
    if (sh[0]) {
        if (tid < FS_MAX_SLOTS) {
            __hip_atomic_store(st->stored[tid], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(st->loaded[tid], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        if (tid == 0) {
            __hip_atomic_store(&st->ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            fs_all_left(&st->done, left);
        }
    }
}

}  // namespace nrfft
