// Instantiates the skinny kernel (qgemm_skinny_kernel.h) for Q5_K weights; one translation unit
// per quant type keeps the build parallel.
#include "qgemm_skinny_kernel.h"

namespace mlxr {
namespace skinny {

const SkinnyKern& kern_q5k(bool f16, int xr, int rt, int kg, bool sw, bool split) {
  return f16 ? kern_of<QT_Q5_K, X_F16>(xr, rt, kg, sw, split) : kern_of<QT_Q5_K, X_BF16>(xr, rt, kg, sw, split);
}

}  // namespace skinny
}  // namespace mlxr
