// fused_f64.hip -- instances of the fused four-step (FP64).
#include "internal.hpp"

namespace nrfft {

// LA x LB of pass A and B; FA x FB of the forward real transform (as FP32: 4096
// tiles, 2^17 256 x 512 442 us, 512 x 256 311; 2^18 512 x 512 372, 1024 x 256 309).
template <int LA, int LB, int FA = LB, int FB = LA>
static FusedRef ref(int sign, bool real) {
    using SH = FsShape<double, LA, LB>;
    const void* fn = real ? (sign > 0 ? reinterpret_cast<const void*>(&k_fused4<double, 1, FA, FB, 1>)
                                      : reinterpret_cast<const void*>(&k_fused4<double, -1, LA, LB, -1>))
                          : (sign > 0 ? reinterpret_cast<const void*>(&k_fused4<double, 1, LA, LB>)
                                      : reinterpret_cast<const void*>(&k_fused4<double, -1, LA, LB>));
    return FusedRef{fn, ilog2c(SH::NTA)};
}

FusedRef fused_lookup_f64(int sign, int logn, bool real) {
    switch (logn) {
        case 14: return ref<128, 128, 256, 64>(sign, real);
        case 15: return ref<128, 256>(sign, real);
        case 16: return ref<256, 256, 512, 128>(sign, real);
        case 17: return ref<256, 512>(sign, real);
        case 18: return ref<512, 512, 1024, 256>(sign, real);
        case 19: return ref<512, 1024>(sign, real);
        case 20: return ref<1024, 1024, 2048, 512>(sign, real);
        default: return FusedRef{nullptr, 0};
    }
}

}  // namespace nrfft
