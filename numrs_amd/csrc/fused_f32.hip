// fused_f32.hip -- instances of the fused four-step (FP32).
#include "internal.hpp"

namespace nrfft {

// LA x LB of pass A and B; FA x FB of the forward real transform, whose pass-B
// tiles store runs of half as many rows at an odd element: more rows a tile pay
// (4096 tiles, FP32: 2^18 512 x 512 446 us, 1024 x 256 321; 2^19 512 x 1024 541,
// 1024 x 512 381; 2^21 1024 x 2048 890, 2048 x 1024 555).
template <int LA, int LB, int FA = LB, int FB = LA>
static FusedRef ref(int sign, int form) {
    using SH = FsShape<float, LA, LB>;
    const void* fn;
    if (sign > 0)
        fn = form == FUSED_C2C ? reinterpret_cast<const void*>(&k_fused4<float, 1, LA, LB>)
                               : reinterpret_cast<const void*>(&k_fused4<float, 1, FA, FB, 1>);
    else if (form == FUSED_CORREL)
        fn = reinterpret_cast<const void*>(&k_fused4<float, -1, LA, LB, (SH::LOGN <= 19 ? -2 : -1)>);
    else
        fn = form == FUSED_C2C ? reinterpret_cast<const void*>(&k_fused4<float, -1, LA, LB>)
                               : reinterpret_cast<const void*>(&k_fused4<float, -1, LA, LB, -1>);
    return FusedRef{fn, ilog2c(SH::NTA)};
}

FusedRef fused_lookup_f32(int sign, int logn, int form) {
    // Correlations of longer spectra are faster with a pass for the product (1184
    // tiles a spectrum: FP32 2^20 503 us against 491, 2^19 408 against 493).
    if (form == FUSED_CORREL && logn > 19) return FusedRef{nullptr, 0};
    switch (logn) {
        case 15: return ref<128, 256>(sign, form);
        case 16: return ref<256, 256>(sign, form);
        case 17: return ref<256, 512>(sign, form);
        case 18: return ref<512, 512, 1024, 256>(sign, form);
        case 19: return ref<512, 1024>(sign, form);
        case 20: return ref<1024, 1024, 2048, 512>(sign, form);
        case 21: return ref<1024, 2048>(sign, form);
        default: return FusedRef{nullptr, 0};
    }
}

}  // namespace nrfft
