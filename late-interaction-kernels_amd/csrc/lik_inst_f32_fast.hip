// Instantiations of the dense MaxSim kernel for fp32 tokens at 65 .. 128 dims
// with the token normalise alone compiled in, what retrieval calls use: the
// all-features kernel's token-scale, packed-doc and mask branches sit in a tile
// loop whose splitting of fp32 rows already takes the VALU's time (32 queries x
// 2048 docs, normalised: 314 -> 295 us).
#include "lik_kernel.h"

namespace lik {
int launch_dense_f32_generic(const Plan& pl, const Params& p, int64_t nb, hipStream_t s);

int launch_dense_f32(const Plan& pl, const Params& p, int64_t nb, hipStream_t s) {
  // (Feature sets without a per-column query scale are not for fp32: the split
  // of a zero has a tiny low part, so padding columns need their scale of 0.)
  if (pl.dpad == 128 && needed_feat(p) == F_NORM) return launch_cfg<EK_F32, 128, SRC_DENSE, 0, F_NORM>(pl, p, nb, s);
  return launch_dense_f32_generic(pl, p, nb, s);
}
}  // namespace lik
