// queue_api.hip -- uneven-batch plans: task lists, the persistent queue
// kernel, hipGraph capture and the extern "C" entry points.
#include <algorithm>
#include <cstring>
#include <memory>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/nrfft.h"
#include "internal.hpp"
#include "queue.hpp"
#include "uneven.hpp"

namespace nrfft {

#define HIPCHK(x)                                                                                      \
    do {                                                                                               \
        hipError_t e_ = (x);                                                                           \
        if (e_ != hipSuccess) return fail(NRFFT_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

struct UnevenState {
    int dtype = 0;
    std::vector<UnevenItem> items;
    std::unique_ptr<UnevenPasses> passes;  // one launch a pass; the list below is then not used
    std::vector<QTask> tasks;  // in the order in which they are taken, two to a ticket
    int n1 = 0, n2 = 0;        // single- and first-pass tiles, second-pass tiles
    std::vector<uint32_t> offs;  // of the items of single-pass tiles, from their tile's base
    bool few = false;          // one group per CU
    bool slow_list = false;    // faster with one launch a pass
    bool reused = false;       // parts of the ring are handed out more than once
    std::vector<uint32_t> init;  // the counters' initial values
    size_t ring_elems = 0;
    size_t total_elems = 0;
    QTask* d_tasks = nullptr;
    uint32_t* d_offs = nullptr;
    uint32_t* d_init = nullptr;
    uint32_t* d_ctr = nullptr;
    void* d_ring = nullptr;
    unsigned grid[2] = {0, 0};  // per direction (different kernels)
    // graph cache
    hipGraphExec_t gexec = nullptr;
    hipGraph_t graph = nullptr;
    hipStream_t cap = nullptr;
    const void* g_in = nullptr;
    void* g_out = nullptr;
    int g_isign = 0;
    std::mutex mu;
    ~UnevenState() {
        if (gexec) (void)hipGraphExecDestroy(gexec);
        if (graph) (void)hipGraphDestroy(graph);
        if (cap) (void)hipStreamDestroy(cap);
        drop_list();
    }
    void drop_list() {
        for (void* p : {(void*)d_tasks, (void*)d_offs, (void*)d_init, (void*)d_ctr, d_ring})
            if (p) (void)hipFree(p);
        d_tasks = nullptr;
        d_offs = d_init = d_ctr = nullptr;
        d_ring = nullptr;
        tasks = {};
        offs = init = {};
    }
};

template <typename T>
static const void* queue_kernel(int isign) {
    return isign > 0 ? reinterpret_cast<const void*>(&k_queue<T, 1>) : reinterpret_cast<const void*>(&k_queue<T, -1>);
}

static int q_cls(int logl, int mode) { return (logl - Q_MIN_LOGL) * Q_MODES + mode; }

// The two passes of an item: n1a transforms of length 2^la, then n1b = 2^la of
// length 2^lb = n1a.  First-pass tiles hold ta transforms, second-pass tiles tb.
struct PassPair {
    int la, lb;
    bool cols;  // first pass along columns (four-step), else rows (2-D)
};

static void add_first(std::vector<QTask>& out, int dtype, const PassPair& p, int64_t off, int64_t ring) {
    const int64_t pts = dtype == NRFFT_F32 ? fs_tile<float>() : fs_tile<double>();
    const int64_t LA = int64_t(1) << p.la, LB = int64_t(1) << p.lb, n = LA * LB, cs = (int64_t)csize(dtype);
    const int64_t ta = std::min(pts / LA, LB), tb = std::min(pts / LB, LA);
    for (int64_t b0 = 0; b0 < LB; b0 += ta) {
        QTask q{};
        q.cls = q_cls(p.la, p.cols ? Q_COL : Q_ROWS);
        q.nvalid = (int32_t)ta;
        q.ioff = off + (p.cols ? b0 : b0 * LA);
        q.ibytes = uint32_t((n - (q.ioff - off)) * cs);
        q.ooff = ring + b0 * tb;
        q.obytes = uint32_t((n - b0 * tb) * cs);
        q.ist = (int32_t)(p.cols ? 1 : LA);
        q.ihi = (int32_t)LB;  // columns
        q.osh = ilog2((size_t)tb);
        q.ohi = (int32_t)(LB * tb);
        q.olo = (int32_t)ta;
        q.tw_logn = p.la + p.lb;
        q.first = (int32_t)b0;
        out.push_back(q);
    }
}

static void add_second(std::vector<QTask>& out, int dtype, const PassPair& p, int64_t off, int64_t ring) {
    const int64_t pts = dtype == NRFFT_F32 ? fs_tile<float>() : fs_tile<double>();
    const int64_t LA = int64_t(1) << p.la, LB = int64_t(1) << p.lb, n = LA * LB, cs = (int64_t)csize(dtype);
    const int64_t ta = std::min(pts / LA, LB), tb = std::min(pts / LB, LA);
    for (int64_t b0 = 0; b0 < LA; b0 += tb) {
        QTask q{};
        q.cls = q_cls(p.lb, Q_RING);
        q.nvalid = (int32_t)tb;
        q.ioff = ring + b0 * LB;
        q.ibytes = uint32_t((n - b0 * LB) * cs);
        q.ist = (int32_t)ta;
        q.ish = ilog2((size_t)ta);
        q.ihi = (int32_t)(tb * ta);
        q.ooff = off + b0;
        q.obytes = uint32_t((n - b0) * cs);
        q.ohi = (int32_t)LA;
        out.push_back(q);
    }
}

// Single-pass items (length, offset; sorted) as tiles of one length: as many
// items as a tile holds and as its 32-bit offsets reach.
static std::vector<QTask> single_tiles(int dtype, const std::vector<std::pair<int, int64_t>>& one,
                                       std::vector<uint32_t>& offs) {
    std::vector<QTask> out;
    const int64_t pts = dtype == NRFFT_F32 ? fs_tile<float>() : fs_tile<double>(), cs = (int64_t)csize(dtype);
    offs.clear();
    for (size_t i = 0; i < one.size();) {
        const int logn = one[i].first;
        const int64_t n = int64_t(1) << logn, base = one[i].second, room = pts >> logn;
        QTask q{};
        q.cls = q_cls(logn, Q_ROW);
        q.ioff = q.ooff = base;
        q.first = (int32_t)offs.size();
        for (; i < one.size() && one[i].first == logn && q.nvalid < room; ++i, ++q.nvalid) {
            const int64_t end = (one[i].second - base + n) * cs;
            if (end >= int64_t(1) << 31) break;
            q.ibytes = q.obytes = uint32_t(end);
            offs.push_back(uint32_t(one[i].second - base));
        }
        out.push_back(q);
    }
    return out;
}

// Four-step split of a 1-D item of 2^logn points: the autotuned choice for
// its size class when the tune cache holds one, else N1 = 2^floor(logn / 2).
int uneven_split(int dtype, int logn, int lo, int hi, const std::vector<int>* force) {
    if (force && (size_t)logn < force->size() && (*force)[logn] > 0) return (*force)[logn];
    Tune t;
    if (tune_find(PK_UNEVEN, dtype, {size_t(1) << logn}, 0, &t) && t.split_log1 >= lo && t.split_log1 <= hi)
        return t.split_log1;
    return std::min(hi, std::max(lo, logn / 2));
}

// Whether an item of two passes of 2^la and 2^lb points runs faster with one launch
// a pass, in a batch of `tiles` first-pass tiles.  A tile of three or four stages
// (2048 points and more) takes longer in the list's engine, which shows while the
// tiles are few; 8192-point passes and the 32-byte runs of a 4096 x 4096 item's
// columns lose at any number.  Batches of one shape, MI355X, one launch a pass / list
// (us):
//   FP32 1 of 2^21 41 / 48, 2: 47 / 56, 4: 75 / 73; 1 of 2^22 49 / 71, 2: 81 / 85,
//   4: 167 / 142; 1 of 2048 x 2048 50 / 64, 2: 83 / 73; 2 of 1024 x 2048 48 / 54, 4: 76 / 70;
//   1 of 4096 x 4096 172 / 230, 2: 386 / 433; 1 of 256 x 8192 42 / 49, 8: 129 / 145, 16:
//   267 / 265; 1 of 8192 x 256 58 / 61, of 8192 x 2048 244 / 387; 1 of 2^20 36 / 33, of
//   1024 x 1024 38 / 32.
//   FP64 1 of 2^20 41 / 41, 2: 46 / 55, 4: 73 / 66; 1 of 2^22 82 / 106, 2: 175 / 157;
//   8 of 2^18 45 / 49, 16: 72 / 62; 1 of 4096 x 4096 381 / 509, of 4096 x 2048 170 / 211.
static bool item_faster_in_passes(bool f32, int la, int lb, bool cols, size_t tiles) {
    const int s = la + lb, longest = std::max(la, lb);
    if (s >= 24) return true;
    if (f32) {
        if (longest == 13) return tiles <= 2048;
        if (s == 23) return tiles <= (cols ? 640 : 512);
        if (s == 22) return tiles <= (cols ? 640 : 256);
        return s == 21 && tiles <= 256 && (cols || tiles > 128);
    }
    if (!cols && lb == 12 && la >= 10) return true;
    if (s == 23) return tiles <= 1024;
    if (s == 22) return tiles <= (longest == 13 ? 1024 : 896);
    if (tiles > 256) return false;
    return s == 21 || longest == 13 || (s >= 18 && tiles > 128 && lb <= 10);
}
// Likewise for single-pass items: only 8192-point ones (FP64 256 of them 31 / 43 us,
// 100: 26 / 24, 800: 70 / 69; FP32 16 23 / 24, as plain launches 15 / 19, 256 28 / 26).
static bool row_faster_in_passes(bool f32, int logn, size_t tiles) {
    return logn == 13 && (f32 ? tiles <= 64 : tiles > 128 && tiles < 700);
}

// The list of tiles (queue.hpp): items largest first, collected into slabs of
// at most Q_SLAB_TILES first-pass tiles (or one item) and those into ring slots;
// second passes stand half a ring behind the first ones; single-pass items are
// spread evenly over the list, where their arithmetic runs under the others'
// memory traffic.
static int build_uneven(UnevenState& u, const std::vector<int>* force_split = nullptr) {
    const bool f32 = u.dtype == NRFFT_F32;
    const int qlog = ilog2(f32 ? fs_tile<float>() : fs_tile<double>());
    const int maxl = std::min(Q_MAX_LOGL, qlog);
    // a column tile of a four-step holds at least 4 transforms
    const int maxl_col = std::min(maxl, qlog - 2);
    struct Two {
        size_t work;
        int64_t off;
        PassPair p;
    };
    std::vector<Two> two;
    std::vector<std::pair<int, int64_t>> one;  // (logn, offset)
    for (const UnevenItem& it : u.items) {
        if (it.ndim == 1) {
            const int logn = ilog2(it.n0);
            if (logn <= maxl) {
                if (logn < Q_MIN_LOGL) return fail(NRFFT_E_UNSUPPORTED, "uneven items need N >= 64");
                one.emplace_back(logn, (int64_t)it.off);
            } else {
                const int lo = std::max(Q_MIN_LOGL, logn - maxl_col), hi = std::min(maxl_col, logn - Q_MIN_LOGL);
                if (lo > hi) return fail(NRFFT_E_UNSUPPORTED, "uneven 1-D item longer than the queue supports");
                const int l1 = uneven_split(u.dtype, logn, lo, hi, force_split);
                two.push_back(Two{it.n0, (int64_t)it.off, PassPair{l1, logn - l1, true}});
            }
        } else {
            const int l0 = ilog2(it.n0), l1 = ilog2(it.n1);
            if (l0 < Q_MIN_LOGL || l1 < Q_MIN_LOGL || l1 > maxl || l0 > std::min(maxl, qlog - 1))
                return fail(NRFFT_E_UNSUPPORTED, "uneven 2-D sides out of the supported range");
            two.push_back(Two{it.n0 * it.n1, (int64_t)it.off, PassPair{l1, l0, false}});
        }
    }
    std::stable_sort(two.begin(), two.end(), [](const Two& x, const Two& y) { return x.work > y.work; });
    std::sort(one.begin(), one.end(), [](const auto& x, const auto& y) {
        return x.first != y.first ? x.first > y.first : x.second < y.second;
    });
    const std::vector<QTask> singles = single_tiles(u.dtype, one, u.offs);

    // The ring is handed out front to back, over and over.  Its size is a multiple
    // of the largest item (and holds at least four), and the items' sizes are powers
    // of two that do not grow along the list, so no item crosses its end.
    const size_t largest = two.empty() ? 1 : two[0].work;
    size_t total = 0;
    for (const Two& t : two) total += t.work;
    const size_t ring = std::min(total, std::max<size_t>(4, FUSED_RING_BYTES / csize(u.dtype) / largest) * largest);
    u.ring_elems = ring;
    u.reused = ring < total;
    // Slabs: consecutive items.
    const size_t tile = size_t(1) << qlog, slab_elems = Q_SLAB_TILES * tile;
    struct Slab {
        size_t i0, i1, elems, tiles;
        size_t from;  // ring elements handed out before it; its place is from mod ring
        int w0, w1;   // slabs [w0, w1) had its place before
        std::vector<QTask> a, b;
    };
    std::vector<Slab> slabs;
    size_t handed = 0;
    for (size_t i = 0; i < two.size(); ++i) {
        const size_t tiles = std::max<size_t>(1, two[i].work / tile);
        if (slabs.empty() || handed % ring == 0 || slabs.back().elems + two[i].work > slab_elems ||
            slabs.back().tiles + tiles > Q_SLAB_TILES)
            slabs.push_back(Slab{i, i, 0, 0, handed, 0, 0, {}, {}});
        Slab& s = slabs.back();
        s.i1 = i + 1;
        s.elems += two[i].work;
        s.tiles += tiles;
        handed += two[i].work;
    }
    // (A slab's place may begin inside the last one that its predecessor waits for.)
    for (size_t k = 0, o = 0; k < slabs.size(); ++k) {
        Slab& s = slabs[k];
        if (s.from < ring) continue;
        while (slabs[o].from + slabs[o].elems + ring <= s.from) ++o;
        s.w0 = (int)o;
        size_t e = o;
        while (e < k && slabs[e].from + ring < s.from + s.elems) ++e;
        s.w1 = (int)e;
    }
    u.init.assign(Q_SLABS + 2 * slabs.size(), 0);
    u.n1 = (int)singles.size();
    u.n2 = 0;
    for (size_t k = 0; k < slabs.size(); ++k) {
        Slab& s = slabs[k];
        int64_t at = int64_t(s.from % ring);
        for (size_t i = s.i0; i < s.i1; ++i) {
            add_first(s.a, u.dtype, two[i].p, two[i].off, at);
            add_second(s.b, u.dtype, two[i].p, two[i].off, at);
            at += (int64_t)two[i].work;
        }
        const int stored = Q_SLABS + (int)k, loaded = stored + (int)slabs.size();
        for (QTask& q : s.a) {
            q.count = stored;
            q.wait = Q_SLABS + (int)slabs.size() + s.w0;
            q.nwait = s.w1 - s.w0;
        }
        for (QTask& q : s.b) {
            q.wait = stored;
            q.nwait = 1;
            q.count = loaded;
        }
        u.init[stored] = (uint32_t)s.a.size();
        u.init[loaded] = (uint32_t)s.b.size();
        u.n1 += (int)s.a.size();
        u.n2 += (int)s.b.size();
        // (A slab holds at most 64 items, none larger than those before, or one: its place
        // held two or three slabs.)
        if (s.w1 - s.w0 > 64) return fail(NRFFT_E_UNSUPPORTED, "uneven ring order");
    }
    // One launch a pass if that is faster for most of the work.
    size_t points = 0, slow = 0;
    for (const Two& t : two) {
        points += t.work;
        if (item_faster_in_passes(f32, t.p.la, t.p.lb, t.p.cols, (size_t)u.n1)) slow += t.work;
    }
    for (const auto& o : one) {
        points += size_t(1) << o.first;
        if (row_faster_in_passes(f32, o.first, (size_t)u.n1)) slow += size_t(1) << o.first;
    }
    u.slow_list = 2 * slow > points;
    if ((size_t)u.n1 + (size_t)u.n2 > size_t(1) << 30) return fail(NRFFT_E_UNSUPPORTED, "uneven batch of too many tiles");

    // Few tiles: one group per CU, so that they spread over the chip (720 first-pass
    // tiles, FP32: 98 us, two per CU 112; 1024: 119 against 108).  If nothing in the
    // ring is replaced, second passes follow all first ones (925 tiles: 113 us, half
    // a ring behind 134; 1280: 125 and 136).
    u.few = (size_t)u.n1 <= Q_FEW_TILES;
    const size_t lag = ring == total ? ring : ring / 2;
    // Tickets: a first-pass tile and, once the second passes have begun, one of
    // theirs, if the distance from a slab's end to its second passes exceeds the
    // 512 tickets in flight (else second passes wait: 500 items whose largest is
    // 2048 x 2048, FP32, 680 us against 630); single tiles otherwise.
    u.tasks.clear();
    u.tasks.reserve(2 * size_t(u.n1 + u.n2));
    auto ticket = [&](const QTask& x, const QTask* y) {
        u.tasks.push_back(x);
        u.tasks.back().last = y == nullptr;
        u.tasks.push_back(y ? *y : QTask{});
        u.tasks.back().last = 1;
    };
    size_t kb = 0, ib = 0;  // next second-pass tile: slab, index
    auto second = [&]() -> const QTask* {
        const QTask* q = &slabs[kb].b[ib];
        if (++ib == slabs[kb].b.size()) {
            ib = 0;
            ++kb;
        }
        return q;
    };
    size_t done = 0, taken = 0;
    auto spread = [&](size_t n) {  // n of the two-pass tiles are in the list
        done += n;
        const size_t all = size_t(u.n1 + u.n2) - singles.size(), upto = all ? singles.size() * done / all : singles.size();
        for (; taken < upto; ++taken) ticket(singles[taken], nullptr);
    };
    for (const Slab& s : slabs) {
        for (; (int)kb < s.w1; spread(1)) ticket(*second(), nullptr);
        for (const QTask& q : s.a) {
            const bool due = slabs[kb].from + lag <= s.from;
            const bool pair = due && ring / 2 >= slabs[kb].elems + Q_PAIR_TILES * tile;
            ticket(q, pair ? second() : nullptr);
            if (due && !pair) ticket(*second(), nullptr);
            spread(due ? 2 : 1);
        }
    }
    for (; kb < slabs.size(); spread(1)) ticket(*second(), nullptr);
    spread(0);
    return NRFFT_OK;
}

static int uneven_setup_device(UnevenState& u) {
    DeviceCtx* ctx = nullptr;
    int rc = get_ctx(&ctx);
    if (rc) return rc;
    HIPCHK(hipMalloc(&u.d_tasks, std::max<size_t>(1, u.tasks.size()) * sizeof(QTask)));
    if (!u.tasks.empty())
        HIPCHK(hipMemcpy(u.d_tasks, u.tasks.data(), u.tasks.size() * sizeof(QTask), hipMemcpyHostToDevice));
    HIPCHK(hipMalloc(&u.d_offs, std::max<size_t>(1, u.offs.size()) * sizeof(uint32_t)));
    if (!u.offs.empty())
        HIPCHK(hipMemcpy(u.d_offs, u.offs.data(), u.offs.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    HIPCHK(hipMalloc(&u.d_init, u.init.size() * sizeof(uint32_t)));
    HIPCHK(hipMemcpy(u.d_init, u.init.data(), u.init.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    std::vector<uint32_t> ctr(u.init.size() * Q_LINE, 0);
    for (size_t i = 0; i < u.init.size(); ++i) ctr[i * Q_LINE] = u.init[i];
    HIPCHK(hipMalloc(&u.d_ctr, ctr.size() * sizeof(uint32_t)));
    HIPCHK(hipMemcpy(u.d_ctr, ctr.data(), ctr.size() * sizeof(uint32_t), hipMemcpyHostToDevice));
    if (u.ring_elems) {
        const size_t bytes = u.ring_elems * csize(u.dtype);
        if (dev_malloc(&u.d_ring, bytes) != hipSuccess) return fail(NRFFT_E_NOMEM, "uneven workspace");
    }
    for (int d = 0; d < 2; ++d) {
        const void* fn = u.dtype == NRFFT_F32 ? queue_kernel<float>(d == 0 ? 1 : -1)
                                              : queue_kernel<double>(d == 0 ? 1 : -1);
        int per_cu = 0;
        HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, FS_NT, 0));
        if (per_cu < 1) return fail(NRFFT_E_UNSUPPORTED, "queue kernel does not fit a CU");
        u.grid[d] = (unsigned)((u.few ? 1 : per_cu) * ctx->ncu);
    }
    return NRFFT_OK;
}

// The plan's launches: one list, or one launch a pass where that is faster or the
// ring finds no room.
static int uneven_make(UnevenState& u, const std::vector<int>* force_split = nullptr) {
    int rc = build_uneven(u, force_split);
    if (rc) return rc;
    bool passes = u.slow_list;
    if (!passes) {
        rc = uneven_setup_device(u);
        passes = rc == NRFFT_E_NOMEM;
        if (rc && !passes) return rc;
    }
    if (passes) {
        u.drop_list();
        u.passes = std::make_unique<UnevenPasses>();
        if ((rc = u.passes->build(u.dtype, u.items, force_split)) || (rc = u.passes->setup_device())) return rc;
    }
    HIPCHK(hipStreamCreateWithFlags(&u.cap, hipStreamNonBlocking));
    return NRFFT_OK;
}

template <typename T>
static int uneven_enqueue(UnevenState& u, const void* in, void* out, int isign, hipStream_t s) {
    if (u.passes) return u.passes->enqueue(in, out, isign, s);
    DeviceCtx* ctx = nullptr;
    int rc = get_ctx(&ctx);
    if (rc) return rc;
    Twiddles<T> tw = ctx_twiddles<T>(ctx);
    const cpx<T>* pin = static_cast<const cpx<T>*>(in);
    cpx<T>* pout = static_cast<cpx<T>*>(out);
    cpx<T>* ring = static_cast<cpx<T>*>(u.d_ring);
    const QTask* tk = u.d_tasks;
    uint32_t* ctr = u.d_ctr;
    const uint32_t* init = u.d_init;
    int lines = (int)u.init.size();
    const uint32_t* offs = u.d_offs;
    int count = (int)u.tasks.size();
    const unsigned grid = std::min<unsigned>(u.grid[isign > 0 ? 0 : 1], unsigned(count / 2));
    void* args[] = {&pin, &pout, &ring, &tk, &count, &offs, &ctr, &init, &lines, &tw};
    HIPCHK(hipLaunchKernel(queue_kernel<T>(isign), dim3(grid), dim3(FS_NT), args, 0, s));
    return NRFFT_OK;
}

static int uneven_execute(UnevenState& u, const void* in, void* out, int isign, hipStream_t stream, bool use_graph) {
    std::lock_guard<std::mutex> lk(u.mu);
    if (!use_graph) {
        return u.dtype == NRFFT_F32 ? uneven_enqueue<float>(u, in, out, isign, stream)
                                    : uneven_enqueue<double>(u, in, out, isign, stream);
    }
    if (!u.gexec || u.g_in != in || u.g_out != out || u.g_isign != isign) {
        if (u.gexec) {
            (void)hipGraphExecDestroy(u.gexec);
            u.gexec = nullptr;
        }
        if (u.graph) {
            (void)hipGraphDestroy(u.graph);
            u.graph = nullptr;
        }
        HIPCHK(hipStreamBeginCapture(u.cap, hipStreamCaptureModeThreadLocal));
        int rc = u.dtype == NRFFT_F32 ? uneven_enqueue<float>(u, in, out, isign, u.cap)
                                      : uneven_enqueue<double>(u, in, out, isign, u.cap);
        hipGraph_t g = nullptr;
        hipError_t e = hipStreamEndCapture(u.cap, &g);
        if (rc) {
            if (g) (void)hipGraphDestroy(g);
            return rc;
        }
        if (e != hipSuccess) return fail(NRFFT_E_HIP, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
        u.graph = g;
        HIPCHK(hipGraphInstantiate(&u.gexec, u.graph, nullptr, nullptr, 0));
        u.g_in = in;
        u.g_out = out;
        u.g_isign = isign;
    }
    HIPCHK(hipGraphLaunch(u.gexec, stream));
    return NRFFT_OK;
}

// Average ms of `iters` executions of an uneven plan (plain launches).
template <typename T>
static int time_uneven(UnevenState& u, void* in, void* out, int iters, hipStream_t s, hipEvent_t e0, hipEvent_t e1,
                       float* ms) {
    int rc = uneven_enqueue<T>(u, in, out, 1, s);
    if (rc) return rc;
    HIPCHK(hipEventRecord(e0, s));
    for (int i = 0; i < iters; ++i)
        if ((rc = uneven_enqueue<T>(u, in, out, 1, s))) return rc;
    HIPCHK(hipEventRecord(e1, s));
    HIPCHK(hipEventSynchronize(e1));
    HIPCHK(hipEventElapsedTime(ms, e0, e1));
    *ms /= (float)iters;
    return NRFFT_OK;
}

// Every four-step split of the 1-D size classes 2^lmin .. 2^lmax, timed on a
// batch of that class (2^25 FP32 / 2^24 FP64 points); the fastest goes to the
// tune cache under (PK_UNEVEN, dtype, {N}).
static int autotune_uneven(int dtype, int lmin, int lmax, int iters, int* best_l1, float* best_ms) {
    const bool f32 = dtype == NRFFT_F32;
    const int qlog = ilog2(f32 ? fs_tile<float>() : fs_tile<double>());
    const int maxl = std::min(Q_MAX_LOGL, qlog);
    const int maxl_col = std::min(maxl, qlog - 2);
    const size_t pts = size_t(1) << (f32 ? 25 : 24);
    struct Res {
        hipStream_t s = nullptr;
        hipEvent_t e0 = nullptr, e1 = nullptr;
        void* in = nullptr;
        void* out = nullptr;
        ~Res() {
            if (e0) (void)hipEventDestroy(e0);
            if (e1) (void)hipEventDestroy(e1);
            if (in) (void)hipFree(in);
            if (out) (void)hipFree(out);
            if (s) (void)hipStreamDestroy(s);
        }
    } r;
    HIPCHK(hipStreamCreateWithFlags(&r.s, hipStreamNonBlocking));
    HIPCHK(hipEventCreate(&r.e0));
    HIPCHK(hipEventCreate(&r.e1));
    if (hipMalloc(&r.in, pts * csize(dtype)) != hipSuccess || hipMalloc(&r.out, pts * csize(dtype)) != hipSuccess)
        return fail(NRFFT_E_NOMEM, "autotune buffers");
    HIPCHK(hipMemsetAsync(r.in, 0, pts * csize(dtype), r.s));
    for (int logn = lmin; logn <= lmax; ++logn) {
        const int slot = logn - lmin;
        if (best_l1) best_l1[slot] = 0;
        if (best_ms) best_ms[slot] = 0.f;
        const int lo = std::max(Q_MIN_LOGL, logn - maxl_col), hi = std::min(maxl_col, logn - Q_MIN_LOGL);
        if (logn <= maxl || lo > hi) continue;  // single pass: nothing to choose
        const size_t n = size_t(1) << logn;
        const size_t count = std::max<size_t>(1, pts / n);
        float best = 0.f;
        int arg = 0;
        for (int l1 = lo; l1 <= hi; ++l1) {
            UnevenState u;
            u.dtype = dtype;
            for (size_t k = 0; k < count; ++k) u.items.push_back(UnevenItem{1, n, 1, k * n});
            u.total_elems = count * n;
            std::vector<int> force(size_t(logn) + 1, 0);
            force[logn] = l1;
            int rc = uneven_make(u, &force);
            float ms = 0.f;
            if (!rc) rc = f32 ? time_uneven<float>(u, r.in, r.out, iters, r.s, r.e0, r.e1, &ms)
                              : time_uneven<double>(u, r.in, r.out, iters, r.s, r.e0, r.e1, &ms);
            if (rc) return rc;
            if (arg == 0 || ms < best) {
                best = ms;
                arg = l1;
            }
        }
        Tune t;
        t.split_log1 = arg;
        tune_store(PK_UNEVEN, dtype, {n}, 0, t);
        if (best_l1) best_l1[slot] = arg;
        if (best_ms) best_ms[slot] = best;
    }
    HIPCHK(hipStreamSynchronize(r.s));
    return NRFFT_OK;
}

}  // namespace nrfft

using namespace nrfft;

struct nrfft_uneven_s {
    UnevenState u;
};

// FFTProcessor::fft_batch (FFT_1.rs:185-189) over host buffers of mixed
// lengths: packed into one HBM buffer, run as one uneven queue launch.
template <typename T>
static int host_fft_batch(T* const* data, const size_t* nn, size_t count, int isign, int dtype) {
    if (isign != 1 && isign != -1) return fail(NRFFT_E_ISIGN, "isign must be 1 or -1");
    if (count == 0) return NRFFT_OK;
    if (!data || !nn) return fail(NRFFT_E_INVALID, "null array");
    std::vector<int> nd(count, 1);
    std::vector<size_t> dims(2 * count, 1), offs(count);
    size_t total = 0;
    for (size_t i = 0; i < count; ++i) {
        if (!data[i]) return fail(NRFFT_E_INVALID, "null buffer");
        if (nn[i] == 0) return fail(NRFFT_E_EMPTY, "nn == 0");
        if (!is_pow2(nn[i])) return fail(NRFFT_E_NOT_POW2, "nn must be a power of two");
        dims[2 * i] = nn[i];
        offs[i] = total;
        total += nn[i];
    }
    // Items shorter than the queue's minimum go through the batched C2C call.
    std::vector<size_t> big, small;
    for (size_t i = 0; i < count; ++i) (nn[i] >= 64 ? big : small).push_back(i);
    for (size_t i : small) {
        int rc = dtype == NRFFT_F32 ? nrfft_four1_f32(reinterpret_cast<float*>(data[i]), nn[i], isign)
                                    : nrfft_four1_f64(reinterpret_cast<double*>(data[i]), nn[i], isign);
        if (rc) return rc;
    }
    if (big.empty()) return NRFFT_OK;
    std::vector<int> bnd(big.size(), 1);
    std::vector<size_t> bdims(2 * big.size(), 1), boffs(big.size());
    size_t btotal = 0;
    for (size_t k = 0; k < big.size(); ++k) {
        bdims[2 * k] = nn[big[k]];
        boffs[k] = btotal;
        btotal += nn[big[k]];
    }
    nrfft_uneven plan = nullptr;
    int rc = nrfft_plan_uneven(&plan, dtype, big.size(), bnd.data(), bdims.data(), boffs.data());
    if (rc) return rc;
    std::unique_ptr<nrfft_uneven_s> guard(plan);
    hipStream_t s = hipStreamPerThread;
    DevBuf buf;
    const size_t bytes = btotal * 2 * sizeof(T);
    if ((rc = dev_alloc(buf, bytes, s))) return rc;
    for (size_t k = 0; k < big.size(); ++k)
        HIPCHK(hipMemcpyAsync(static_cast<T*>(buf.p) + 2 * boffs[k], data[big[k]], nn[big[k]] * 2 * sizeof(T),
                              hipMemcpyHostToDevice, s));
    if ((rc = uneven_execute(plan->u, buf.p, buf.p, isign, s, false))) return rc;
    for (size_t k = 0; k < big.size(); ++k)
        HIPCHK(hipMemcpyAsync(data[big[k]], static_cast<T*>(buf.p) + 2 * boffs[k], nn[big[k]] * 2 * sizeof(T),
                              hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    if ((rc = nrfft_uneven_check(plan, s))) return rc;
    return NRFFT_OK;
}

extern "C" {

int nrfft_plan_uneven(nrfft_uneven* plan, int dtype, size_t nitems, const int* ndim, const size_t* dims,
                      const size_t* offs) {
    g_err.clear();
    if (!plan) return fail(NRFFT_E_INVALID, "null plan pointer");
    *plan = nullptr;
    if (dtype != NRFFT_F32 && dtype != NRFFT_F64) return fail(NRFFT_E_INVALID, "dtype");
    if (nitems == 0) return fail(NRFFT_E_EMPTY, "no items");
    if (!ndim || !dims || !offs) return fail(NRFFT_E_INVALID, "null array");
    auto p = std::make_unique<nrfft_uneven_s>();
    p->u.dtype = dtype;
    size_t end = 0;
    for (size_t i = 0; i < nitems; ++i) {
        UnevenItem it;
        it.ndim = ndim[i];
        if (it.ndim != 1 && it.ndim != 2) return fail(NRFFT_E_DIMS, "uneven items are 1-D or 2-D");
        it.n0 = dims[2 * i];
        it.n1 = it.ndim == 2 ? dims[2 * i + 1] : 1;
        if (it.n0 <= 1 || (it.ndim == 2 && it.n1 <= 1)) return fail(NRFFT_E_DIMS, "Invalid dimension size");
        if (!is_pow2(it.n0) || !is_pow2(it.n1)) return fail(NRFFT_E_NOT_POW2, "dimension must be a power of two");
        it.off = offs[i];
        end = std::max(end, it.off + it.n0 * it.n1);
        p->u.items.push_back(it);
    }
    p->u.total_elems = end;
    int rc = uneven_make(p->u);
    if (rc) return rc;
    *plan = p.release();
    return NRFFT_OK;
}

int nrfft_execute_uneven(nrfft_uneven plan, const void* d_in, void* d_out, int isign, void* stream) {
    g_err.clear();
    if (!plan) return fail(NRFFT_E_INVALID, "null plan");
    if (isign != 1 && isign != -1) return fail(NRFFT_E_ISIGN, "isign must be 1 or -1");
    if (!d_in || !d_out) return fail(NRFFT_E_INVALID, "null buffer");
    return uneven_execute(plan->u, d_in, d_out, isign, (hipStream_t)stream, true);
}

int nrfft_execute_uneven_nograph(nrfft_uneven plan, const void* d_in, void* d_out, int isign, void* stream) {
    g_err.clear();
    if (!plan) return fail(NRFFT_E_INVALID, "null plan");
    if (isign != 1 && isign != -1) return fail(NRFFT_E_ISIGN, "isign must be 1 or -1");
    if (!d_in || !d_out) return fail(NRFFT_E_INVALID, "null buffer");
    return uneven_execute(plan->u, d_in, d_out, isign, (hipStream_t)stream, false);
}

int nrfft_uneven_check(nrfft_uneven plan, void* stream) {
    g_err.clear();
    if (!plan) return fail(NRFFT_E_INVALID, "null plan");
    if (plan->u.passes) return plan->u.passes->check((hipStream_t)stream);
    uint32_t tickets = 0;
    HIPCHK(hipMemcpyAsync(&tickets, plan->u.d_ctr + Q_LAST * Q_LINE, sizeof tickets, hipMemcpyDeviceToHost, (hipStream_t)stream));
    HIPCHK(hipStreamSynchronize((hipStream_t)stream));
    // every group leaves after drawing one ticket past the end
    if (2 * (uint64_t)tickets < (uint64_t)plan->u.tasks.size())
        return fail(NRFFT_E_HIP, "uneven queue: the task list was not drained");
    return expired_check(plan->u.d_ctr + Q_EXPIRED * Q_LINE, (hipStream_t)stream);
}

int nrfft_uneven_launch_info(nrfft_uneven plan, int* launches, int* ring_reused, void** expired) {
    g_err.clear();
    if (!plan) return fail(NRFFT_E_INVALID, "null plan");
    const UnevenState& u = plan->u;
    if (launches) *launches = u.passes ? u.passes->launches() : 1;
    if (ring_reused) *ring_reused = !u.passes && u.reused ? 1 : 0;
    if (expired) *expired = u.passes ? nullptr : u.d_ctr + Q_EXPIRED * Q_LINE;
    return NRFFT_OK;
}

int nrfft_uneven_info(nrfft_uneven plan, size_t* tasks_phase1, size_t* tasks_phase2, size_t* workspace_bytes,
                      unsigned* groups) {
    g_err.clear();
    if (!plan) return fail(NRFFT_E_INVALID, "null plan");
    const UnevenState& u = plan->u;
    if (tasks_phase1) *tasks_phase1 = (size_t)(u.passes ? u.passes->n1 : u.n1);
    if (tasks_phase2) *tasks_phase2 = (size_t)(u.passes ? u.passes->n2 : u.n2);
    if (workspace_bytes) *workspace_bytes = (u.passes ? u.passes->ws_elems : u.ring_elems) * csize(u.dtype);
    if (groups) *groups = u.passes ? u.passes->grid[0] : u.grid[0];
    return NRFFT_OK;
}

int nrfft_uneven_destroy(nrfft_uneven plan) {
    delete plan;
    return NRFFT_OK;
}

int nrfft_autotune_uneven(int dtype, int log2n_min, int log2n_max, int iters, int* best_l1, float* best_ms) {
    g_err.clear();
    if (dtype != NRFFT_F32 && dtype != NRFFT_F64) return fail(NRFFT_E_INVALID, "dtype");
    if (log2n_min < Q_MIN_LOGL || log2n_max < log2n_min || log2n_max > 26)
        return fail(NRFFT_E_INVALID, "size-class range");
    if (iters < 1) iters = 1;
    return autotune_uneven(dtype, log2n_min, log2n_max, iters, best_l1, best_ms);
}

int nrfft_fft_batch_f64(double* const* data, const size_t* nn, size_t count, int isign) {
    g_err.clear();
    return host_fft_batch<double>(data, nn, count, isign, NRFFT_F64);
}
int nrfft_fft_batch_f32(float* const* data, const size_t* nn, size_t count, int isign) {
    g_err.clear();
    return host_fft_batch<float>(data, nn, count, isign, NRFFT_F32);
}

}  // extern "C"
