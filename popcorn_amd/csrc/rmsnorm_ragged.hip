// RMSNorm on rows that are not whole, aligned 16-byte packs: the row kernels of
// rmsnorm_rows.h instantiated for them. Reading such rows element by element
// left most of every memory access unused: fp32 [5003, 1537] with a bias took
// 45 us backward (whose dw columns went through memory row by row) and takes
// 24; bf16 [9264, 174] 8.7 us forward and 9.4 backward, 5.9 and 9.4 now.
#include "rmsnorm_rows.h"

namespace pk {

template <typename T, typename W, int MODE> void Ragged<T, W, MODE>::fwd(const FwdArgs& a, const Plan& p) {
  fwd_vec<T, W, MODE, false>(a, p);
}
template <typename T, typename W, int MODE> void Ragged<T, W, MODE>::bwd(const BwdArgs& a, const Plan& p, int64_t blocks) {
  bwd_vec<T, W, MODE, false>(a, p, blocks);
}
template <typename T, typename W, int MODE> int Ragged<T, W, MODE>::resident(const Plan& p) {
  return bwd_vec_resident<T, W, MODE, false>(p);
}

#define PK_MODES(T, W)               \
  template struct Ragged<T, W, kPlain>; \
  template struct Ragged<T, W, kBias>;  \
  template struct Ragged<T, W, kAdd>;
PK_MODES(float, float)
PK_MODES(bf16, bf16)
PK_MODES(f16, f16)
PK_MODES(bf16, float)
PK_MODES(f16, float)
#undef PK_MODES

}  // namespace pk
