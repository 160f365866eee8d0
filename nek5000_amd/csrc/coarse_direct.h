// Direct coarse solver: the assembled trilinear problem by explicit inverses
// (see coarse_direct.hip).
#pragma once
#include <vector>

#include "nekamd_internal.h"

namespace nekamd {

struct DirectCoarse {
  int n = 0;              // unknowns; 0: not set up
  int np = 0;             // parts
  int kld = 0;            // rows and row length a part is padded to (multiple of 64)
  int ns = 0, sld = 0;    // separator unknowns, padded
  double *inv = nullptr;  // np inverses of the parts' blocks, kld x kld each
  double *sinv = nullptr; // inverse of the separator's Schur complement, sld x sld
  int32_t *prow = nullptr;  // np*kld: unknown of a part's row, -1 where padded
  int32_t *srow = nullptr;  // ns: unknown of a separator row
  // couplings in CSR: part rows -> separator rows, separator rows -> part rows
  int32_t *is_rp = nullptr, *is_ci = nullptr;
  double *is_v = nullptr;
  int32_t *si_rp = nullptr, *si_ci = nullptr;
  double *si_v = nullptr;
  double *y = nullptr, *g = nullptr, *xs = nullptr;
  // steps of refinement in a solve; where there are any, the problem's rows, a
  // residual and a correction
  int refine = 0;
  int32_t *a_rp = nullptr, *a_ci = nullptr;
  double *a_v = nullptr, *rr = nullptr, *dd = nullptr;

  bool ready() const { return n > 0; }
  // rows of the assembled SPD problem, and three coordinates per unknown (the
  // dissection splits along them).  *ok = false, nothing kept: the problem is
  // too large for this solver, a pivot is rounding or the residual of a solve
  // is too large (kPivotMin, kMaxResidual), or memory is short.
  int setup(const std::vector<int32_t> &rp, const std::vector<int32_t> &ci,
            const std::vector<double> &v, const std::vector<double> &xyz, hipStream_t s,
            bool *ok);
  // x = A^-1 b, enqueued on s (x and b distinct)
  int solve(double *x, const double *b, hipStream_t s) const;
  void release();

 private:
  // one pass of the inverses, without refinement
  int apply(double *x, const double *b, hipStream_t s) const;
  bool refine_to(const std::vector<int32_t> &rp, const std::vector<int32_t> &ci,
                 const std::vector<double> &v, const std::vector<double> &xyz, hipStream_t s);
};

}  // namespace nekamd
