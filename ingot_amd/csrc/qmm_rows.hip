// The few-row int4 product on the caller's bf16 rows (ih_qmm_int4): the kernel of qmm_kernel.h with its row-major
// activation reads, in the three output forms of the C ABI.
#include "qmm_kernel.h"

namespace ih {

template <int T, bool X16>
static bool by_mode(const TimedLaunch& tl, QmmShape sh, dim3 grid, hipStream_t st, const QmmParams& p, int mode) {
  switch (mode) {
    case QM_F32: return qmm_dispatch_mode<T, X16, QM_F32, true>(tl, sh, grid, st, p);
    case QM_F32_ADD: return qmm_dispatch_mode<T, X16, QM_F32_ADD, true>(tl, sh, grid, st, p);
    case QM_BF16: return qmm_dispatch_mode<T, X16, QM_BF16, true>(tl, sh, grid, st, p);
    default: return false;
  }
}

bool qmm_rows_dispatch(const TimedLaunch& tl, QmmShape sh, dim3 grid, hipStream_t st, const QmmParams& p, int M,
                       int mode) {
  if (M > 17 && grid.z == 1) return by_mode<2, false>(tl, sh, grid, st, p, mode);
  if (M == 17) return by_mode<1, true>(tl, sh, grid, st, p, mode);
  return by_mode<1, false>(tl, sh, grid, st, p, mode);
}

}  // namespace ih
