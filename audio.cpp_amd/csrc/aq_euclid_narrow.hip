// Euclidean RVQ at K = 256: the narrow one-launch cascade.
#include "aq_euclid_kernels.hpp"

namespace {
// Keys per lane after the merge.  The Q8_0 variant for top-4 keeps six in
// place of four: its fp16 images of q * d leave about 2.7 % of the frames of
// each stage uncertified with four (their verification then costs more than
// the cascade saves), a few with six.
template <bool Q8, int TOPL>
constexpr int merged_keys() { return Q8 && TOPL == 4 ? 6 : TOPL; }
template <int RECIPE, bool Q8, int FG, int TOPL>
constexpr int narrow_lds() { return NwLayout<8, FG, merged_keys<Q8, TOPL>(), Q8>::BYTES; }
template <int RECIPE, bool Q8, int FG, int TOPL>
constexpr CascadeFn narrow_fn() { return euclid_narrow_kernel<RECIPE, Q8, 8, FG, merged_keys<Q8, TOPL>()>; }

template <int FG>
const NarrowKernels *table() {
    static const NarrowKernels t = {
        {{narrow_fn<OMNI, false, FG, 3>(), narrow_fn<OMNI, false, FG, 4>()},
         {narrow_fn<HIGGS, false, FG, 3>(), narrow_fn<HIGGS, false, FG, 4>()},
         {narrow_fn<DIRECT, false, FG, 3>(), narrow_fn<DIRECT, false, FG, 4>()},
         {narrow_fn<HIGGS, true, FG, 3>(), narrow_fn<HIGGS, true, FG, 4>()}},
        {{narrow_lds<OMNI, false, FG, 3>(), narrow_lds<OMNI, false, FG, 4>()},
         {narrow_lds<HIGGS, false, FG, 3>(), narrow_lds<HIGGS, false, FG, 4>()},
         {narrow_lds<DIRECT, false, FG, 3>(), narrow_lds<DIRECT, false, FG, 4>()},
         {narrow_lds<HIGGS, true, FG, 3>(), narrow_lds<HIGGS, true, FG, 4>()}},
        FG * 16};
    return &t;
}
}  // namespace

namespace aq_euclid {
const NarrowKernels *kernels_narrow(int fg) {
    switch (fg) {
        case 1: return table<1>();
        case 2: return table<2>();
        case 4: return table<4>();
        default: return nullptr;
    }
}
}  // namespace aq_euclid
