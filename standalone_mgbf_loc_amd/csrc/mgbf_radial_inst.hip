// One translation unit per radial half-width and part, compiled for each
// MGBF_RADIAL_H in 1..10 and MGBF_RADIAL_PART: 0 the box of taps and the
// matrix-core engine, 1 the disc, 2 the product of line factors, 3 and 4 the
// disc and the product with 2 columns a lane.
#include "mgbf_radial.hpp"

#if !defined(MGBF_RADIAL_H) || !defined(MGBF_RADIAL_PART)
#error "MGBF_RADIAL_H and MGBF_RADIAL_PART must be defined"
#endif
#if MGBF_RADIAL_PART == 0
#include "mgbf_radial_mx.hpp"
#endif

#define MGBF_CAT2(a, b) a##b
#define MGBF_CAT(a, b) MGBF_CAT2(a, b)

namespace mgbf {
#if MGBF_RADIAL_PART == 0
hipError_t MGBF_CAT(launch_radial_mx_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_mx_h<MGBF_RADIAL_H>(a, st);
}
hipError_t MGBF_CAT(launch_radial_box_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_taps<MGBF_RADIAL_H, kTapsBox>(a, st);
}
hipError_t MGBF_CAT(launch_radial_box2_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_taps2<MGBF_RADIAL_H, kTapsBox>(a, st);
}
#elif MGBF_RADIAL_PART == 1
hipError_t MGBF_CAT(launch_radial_disc_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_taps<MGBF_RADIAL_H, kTapsDisc>(a, st);
}
#elif MGBF_RADIAL_PART == 2
hipError_t MGBF_CAT(launch_radial_sep_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_taps<MGBF_RADIAL_H, kTapsSep>(a, st);
}
#elif MGBF_RADIAL_PART == 3
hipError_t MGBF_CAT(launch_radial_disc2_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_taps2<MGBF_RADIAL_H, kTapsDisc>(a, st);
}
#else
hipError_t MGBF_CAT(launch_radial_sep2_H, MGBF_RADIAL_H)(const RadialArgs& a, hipStream_t st) {
    return launch_radial_taps2<MGBF_RADIAL_H, kTapsSep>(a, st);
}
#endif
}  // namespace mgbf
