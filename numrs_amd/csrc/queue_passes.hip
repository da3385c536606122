// queue_passes.hip -- uneven plans that run one launch a pass: task lists and launches.
#include <algorithm>
#include <string>
#include <utility>

#include "../../include/nrfft.h"
#include "queue_passes.hpp"
#include "uneven.hpp"

namespace nrfft {

#define HIPCHK(x)                                                                                      \
    do {                                                                                               \
        hipError_t e_ = (x);                                                                           \
        if (e_ != hipSuccess) return fail(NRFFT_E_HIP, std::string(#x) + ": " + hipGetErrorString(e_)); \
    } while (0)

template <typename T>
static const void* pass_kernel(int isign) {
    return isign > 0 ? reinterpret_cast<const void*>(&k_queue_pass<T, 1>)
                     : reinterpret_cast<const void*>(&k_queue_pass<T, -1>);
}

UnevenPasses::UnevenPasses() = default;
UnevenPasses::~UnevenPasses() {
    if (d_tasks) (void)hipFree(d_tasks);
    if (d_state) (void)hipFree(d_state);
    if (d_ws) (void)hipFree(d_ws);
}

// Tiles of one pass over `count` transforms of length L = 2^logl: TI transforms
// along b (b-th transform at base + b * bstride), element stride es.
static void add_pass(std::vector<QPass>& out, int dtype, int logl, int mode, int64_t count, int src, int dst,
                     int64_t ibase, int64_t ibstride, int32_t iesi, int64_t obase, int64_t obstride, int32_t oeso,
                     int tw_logn) {
    const int qp = dtype == NRFFT_F32 ? qp_pts<float>() : qp_pts<double>();
    const int64_t TI = qp >> logl;
    for (int64_t b0 = 0; b0 < count; b0 += TI) {
        QPass q{};
        q.cls = (logl - QP_MIN_LOGL) * QP_MODES + mode;
        q.nvalid = (int32_t)std::min<int64_t>(TI, count - b0);
        q.src = src;
        q.dst = dst;
        q.ioff = ibase + b0 * ibstride;
        q.ooff = obase + b0 * obstride;
        q.si0 = (int32_t)ibstride;
        q.esi = iesi;
        q.so0 = (int32_t)obstride;
        q.eso = oeso;
        q.tw_logn = tw_logn;
        q.tw_n2base = (int32_t)b0;
        out.push_back(q);
    }
}

int UnevenPasses::build(int dt, const std::vector<UnevenItem>& items, const std::vector<int>* force_split) {
    dtype = dt;
    const bool f32 = dtype == NRFFT_F32;
    const int qlog = ilog2(f32 ? qp_pts<float>() : qp_pts<double>());
    const int maxl = f32 ? qp_max_logl<float>() : qp_max_logl<double>();
    const int maxl_col = std::min(maxl, qlog - 2);  // a column tile holds at least 4 transforms
    std::vector<std::pair<int64_t, std::vector<QPass>>> p1, p2;  // (work, tiles) per item
    size_t ws = 0;
    for (const UnevenItem& it : items) {
        std::vector<QPass> a, b;
        if (it.ndim == 1) {
            const int logn = ilog2(it.n0);
            if (logn <= maxl) {
                if (logn < QP_MIN_LOGL) return fail(NRFFT_E_UNSUPPORTED, "uneven items need N >= 64");
                add_pass(a, dtype, logn, 0, 1, B_IN, B_OUT, it.off, it.n0, 1, it.off, it.n0, 1, 0);
            } else {
                const int lo = std::max(QP_MIN_LOGL, logn - maxl_col), hi = std::min(maxl_col, logn - QP_MIN_LOGL);
                if (lo > hi) return fail(NRFFT_E_UNSUPPORTED, "uneven 1-D item longer than the queue supports");
                const int l1 = uneven_split(dtype, logn, lo, hi, force_split);
                const int l2 = logn - l1;
                const int64_t N1 = int64_t(1) << l1, N2 = int64_t(1) << l2;
                // pass A: columns n2 (stride N2), length N1, twiddle -> workspace [k1][n2]
                add_pass(a, dtype, l1, 1, N2, B_IN, B_TMP, (int64_t)it.off, 1, (int32_t)N2, (int64_t)ws, 1,
                         (int32_t)N2, logn);
                // pass B: rows k1 of the workspace, length N2, stored at X[k2 N1 + k1]
                add_pass(b, dtype, l2, 2, N1, B_TMP, B_OUT, (int64_t)ws, N2, 1, (int64_t)it.off, 1, (int32_t)N1, 0);
                ws += size_t(N1 * N2);
            }
        } else {
            const int l0 = ilog2(it.n0), l1 = ilog2(it.n1);
            if (l0 < QP_MIN_LOGL || l1 < QP_MIN_LOGL || l1 > maxl || l0 > std::min(maxl, qlog - 1))
                return fail(NRFFT_E_UNSUPPORTED, "uneven 2-D sides out of the supported range");
            // rows along n1 (contiguous), then columns along n0 (stride n1) in place in out
            add_pass(a, dtype, l1, 0, (int64_t)it.n0, B_IN, B_OUT, it.off, it.n1, 1, it.off, it.n1, 1, 0);
            add_pass(b, dtype, l0, 1, (int64_t)it.n1, B_OUT, B_OUT, it.off, 1, (int32_t)it.n1, it.off, 1,
                     (int32_t)it.n1, 0);
        }
        const int64_t work = int64_t(it.n0 * it.n1);
        p1.emplace_back(work, std::move(a));
        if (!b.empty()) p2.emplace_back(work, std::move(b));
    }
    // Largest items first in each launch (longest-processing-time order).
    auto by_work = [](const auto& x, const auto& y) { return x.first > y.first; };
    std::stable_sort(p1.begin(), p1.end(), by_work);
    std::stable_sort(p2.begin(), p2.end(), by_work);
    tasks.clear();
    for (auto& e : p1) tasks.insert(tasks.end(), e.second.begin(), e.second.end());
    n1 = (int)tasks.size();
    for (auto& e : p2) tasks.insert(tasks.end(), e.second.begin(), e.second.end());
    n2 = (int)tasks.size() - n1;
    ws_elems = ws;
    return NRFFT_OK;
}

int UnevenPasses::setup_device() {
    DeviceCtx* ctx = nullptr;
    int rc = get_ctx(&ctx);
    if (rc) return rc;
    HIPCHK(hipMalloc(&d_tasks, std::max<size_t>(1, tasks.size()) * sizeof(QPass)));
    if (!tasks.empty()) HIPCHK(hipMemcpy(d_tasks, tasks.data(), tasks.size() * sizeof(QPass), hipMemcpyHostToDevice));
    HIPCHK(hipMalloc(&d_state, sizeof(QPState)));
    if (ws_elems && dev_malloc(&d_ws, ws_elems * csize(dtype)) != hipSuccess)
        return fail(NRFFT_E_NOMEM, "uneven workspace");
    for (int d = 0; d < 2; ++d) {
        const void* fn = dtype == NRFFT_F32 ? pass_kernel<float>(d == 0 ? 1 : -1) : pass_kernel<double>(d == 0 ? 1 : -1);
        const int nt = dtype == NRFFT_F32 ? qp_pts<float>() / 16 : qp_pts<double>() / 16;
        int per_cu = 0;
        HIPCHK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, fn, nt, 0));
        if (per_cu < 1) return fail(NRFFT_E_UNSUPPORTED, "queue kernel does not fit a CU");
        grid[d] = (unsigned)(per_cu * ctx->ncu);
    }
    return NRFFT_OK;
}

template <typename T>
static int enqueue_as(UnevenPasses& u, const void* in, void* out, int isign, hipStream_t s) {
    DeviceCtx* ctx = nullptr;
    int rc = get_ctx(&ctx);
    if (rc) return rc;
    Twiddles<T> tw = ctx_twiddles<T>(ctx);
    cpx<T>* pin = const_cast<cpx<T>*>(static_cast<const cpx<T>*>(in));
    cpx<T>* pout = static_cast<cpx<T>*>(out);
    cpx<T>* pws = static_cast<cpx<T>*>(u.d_ws);
    const QPass* tk = u.d_tasks;
    QPState* st = u.d_state;
    const int d = isign > 0 ? 0 : 1;
    hipLaunchKernelGGL(k_queue_reset, dim3(1), dim3(64), 0, s, st);
    HIPCHK(hipGetLastError());
    const int nt = (int)(qp_pts<T>() / 16);
    for (int phase = 0; phase < 2; ++phase) {
        int base = phase ? u.n1 : 0, count = phase ? u.n2 : u.n1, ph = phase;
        if (count == 0) continue;
        const unsigned grid = std::min<unsigned>(u.grid[d], (unsigned)count);
        void* args[] = {&pin, &pout, &pws, &tk, &base, &count, &ph, &st, &tw};
        HIPCHK(hipLaunchKernel(pass_kernel<T>(isign), dim3(grid), dim3(nt), args, 0, s));
    }
    return NRFFT_OK;
}

int UnevenPasses::enqueue(const void* in, void* out, int isign, hipStream_t s) {
    return dtype == NRFFT_F32 ? enqueue_as<float>(*this, in, out, isign, s)
                              : enqueue_as<double>(*this, in, out, isign, s);
}

int UnevenPasses::check(hipStream_t s) {
    QPState st{};
    HIPCHK(hipMemcpyAsync(&st, d_state, sizeof st, hipMemcpyDeviceToHost, s));
    HIPCHK(hipStreamSynchronize(s));
    // every group leaves after drawing one index past the end of its launch
    if (st.next[0] < (uint32_t)n1 || st.next[1] < (uint32_t)n2)
        return fail(NRFFT_E_HIP, "uneven queue: a pass did not drain its task list");
    return NRFFT_OK;
}

}  // namespace nrfft
