// fused_f32.hip -- instances of the fused four-step (FP32).
#include "internal.hpp"

namespace nrfft {

template <int LA, int LB>
static FusedRef ref(int sign) {
    using SH = FsShape<float, LA, LB>;
    return FusedRef{sign > 0 ? reinterpret_cast<const void*>(&k_fused4<float, 1, LA, LB>)
                             : reinterpret_cast<const void*>(&k_fused4<float, -1, LA, LB>),
                    ilog2c(SH::NTA)};
}

FusedRef fused_lookup_f32(int sign, int logn) {
    switch (logn) {
        case 15: return ref<128, 256>(sign);
        case 16: return ref<256, 256>(sign);
        case 17: return ref<256, 512>(sign);
        case 18: return ref<512, 512>(sign);
        case 19: return ref<512, 1024>(sign);
        case 20: return ref<1024, 1024>(sign);
        case 21: return ref<1024, 2048>(sign);
        default: return FusedRef{nullptr, 0};
    }
}

}  // namespace nrfft
