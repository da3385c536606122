// uneven.hpp -- what the two forms of an uneven plan share: its items, and the form
// that runs one launch a pass (queue_passes.hip).
#pragma once
#include <vector>

#include "internal.hpp"

namespace nrfft {

struct UnevenItem {
    int ndim;
    size_t n0, n1;  // ndim == 1: n0 = N, n1 = 1
    size_t off;     // complex elements
};

// Four-step split of a 1-D item of 2^logn points, lo <= log2 N1 <= hi.
int uneven_split(int dtype, int logn, int lo, int hi, const std::vector<int>* force);

struct QPass;
struct QPState;
struct UnevenPasses {
    int dtype = 0;
    std::vector<QPass> tasks;  // first passes, then second ones
    int n1 = 0, n2 = 0;
    size_t ws_elems = 0;  // the 1-D items of two passes; 2-D ones run in the output
    QPass* d_tasks = nullptr;
    QPState* d_state = nullptr;
    void* d_ws = nullptr;
    unsigned grid[2] = {0, 0};  // per direction (different kernels)
    UnevenPasses();
    ~UnevenPasses();
    int build(int dt, const std::vector<UnevenItem>& items, const std::vector<int>* force_split);
    int setup_device();
    int launches() const { return 1 + (n1 > 0) + (n2 > 0); }
    int enqueue(const void* in, void* out, int isign, hipStream_t s);
    int check(hipStream_t s);
};

}  // namespace nrfft
