// fused_f64.hip -- instances of the fused four-step (FP64).
#include "internal.hpp"

namespace nrfft {

// LA x LB of pass A and B; FA x FB of the forward real transform (as FP32: 4096
// tiles, 2^17 256 x 512 442 us, 512 x 256 311; 2^18 512 x 512 372, 1024 x 256 309).
template <int LA, int LB, int FA = LB, int FB = LA>
static FusedRef ref(int sign, int form) {
    using SH = FsShape<double, LA, LB>;
    const void* fn;
    if (sign > 0)
        fn = form == FUSED_C2C ? reinterpret_cast<const void*>(&k_fused4<double, 1, LA, LB>)
                               : reinterpret_cast<const void*>(&k_fused4<double, 1, FA, FB, 1>);
    else if (form == FUSED_CORREL)
        fn = reinterpret_cast<const void*>(&k_fused4<double, -1, LA, LB, (SH::LOGN <= 19 ? -2 : -1)>);
    else
        fn = form == FUSED_C2C ? reinterpret_cast<const void*>(&k_fused4<double, -1, LA, LB>)
                               : reinterpret_cast<const void*>(&k_fused4<double, -1, LA, LB, -1>);
    return FusedRef{fn, ilog2c(SH::NTA)};
}

FusedRef fused_lookup_f64(int sign, int logn, int form) {
    // Correlations of longer spectra are faster with a pass for the product (1184
    // tiles a spectrum: FP64 2^20 499 us against 467, 2^19 400 against 439).
    if (form == FUSED_CORREL && logn > 19) return FusedRef{nullptr, 0};
    switch (logn) {
        case 14: return ref<128, 128, 256, 64>(sign, form);
        case 15: return ref<128, 256>(sign, form);
        case 16: return ref<256, 256, 512, 128>(sign, form);
        case 17: return ref<256, 512>(sign, form);
        case 18: return ref<512, 512, 1024, 256>(sign, form);
        case 19: return ref<512, 1024>(sign, form);
        case 20: return ref<1024, 1024, 2048, 512>(sign, form);
        default: return FusedRef{nullptr, 0};
    }
}

}  // namespace nrfft
