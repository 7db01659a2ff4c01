// Three-phase keyswitch at N = 4096 (a translation unit of its own: the
// kernels of one size take a minute to compile).
#include "keyswitch_rows.hpp"

namespace praghip {

template <int LOG>
hipError_t run_keyswitch_rows_small(const KsArgs& a, const KsConst* kc_dev, const KsConst& kc, const NttDevice& d,
                                    hipStream_t s) {
  return run_keyswitch_rows<LOG>(a, kc_dev, kc, d, s);
}
template hipError_t run_keyswitch_rows_small<12>(const KsArgs&, const KsConst*, const KsConst&, const NttDevice&,
                                                 hipStream_t);

}  // namespace praghip
