// fused_f32.hip -- instances of the fused four-step (FP32).
#include "internal.hpp"

namespace nrfft {

// LA x LB of pass A and B; FA x FB of the forward real transform, whose pass-B
// tiles store runs of half as many rows at an odd element: more rows a tile pay
// (4096 tiles, FP32: 2^18 512 x 512 446 us, 1024 x 256 321; 2^19 512 x 1024 541,
// 1024 x 512 381; 2^21 1024 x 2048 890, 2048 x 1024 555).
template <int LA, int LB, int FA = LB, int FB = LA>
static FusedRef ref(int sign, bool real) {
    using SH = FsShape<float, LA, LB>;
    const void* fn = real ? (sign > 0 ? reinterpret_cast<const void*>(&k_fused4<float, 1, FA, FB, 1>)
                                      : reinterpret_cast<const void*>(&k_fused4<float, -1, LA, LB, -1>))
                          : (sign > 0 ? reinterpret_cast<const void*>(&k_fused4<float, 1, LA, LB>)
                                      : reinterpret_cast<const void*>(&k_fused4<float, -1, LA, LB>));
    return FusedRef{fn, ilog2c(SH::NTA)};
}

FusedRef fused_lookup_f32(int sign, int logn, bool real) {
    switch (logn) {
        case 15: return ref<128, 256>(sign, real);
        case 16: return ref<256, 256>(sign, real);
        case 17: return ref<256, 512>(sign, real);
        case 18: return ref<512, 512, 1024, 256>(sign, real);
        case 19: return ref<512, 1024>(sign, real);
        case 20: return ref<1024, 1024, 2048, 512>(sign, real);
        case 21: return ref<1024, 2048>(sign, real);
        default: return FusedRef{nullptr, 0};
    }
}

}  // namespace nrfft
