// The dense operator of the untransposed cycle from one level down: the
// cycle applied to all unit vectors of that level at once, in FP64.  A
// multi-vector is row-major (row i of all ld columns consecutive), so every
// sparse product streams whole rows, and the triangular solves of all columns
// go through the level sets together.
//
// On MI355X the cycle applied to one unit vector after the other (about ten
// launches each) took 28 ms for 473 rows below an l1-Jacobi hierarchy; this
// form takes 2.1 ms for 3308 rows, and makes tails of that size possible.
#pragma once
#include "mld_devcommon.hpp"

namespace mld {
namespace tail {

// acc of row i, column c; EPI: 0 y = acc, 1 y += acc, 2 y = b - acc,
// 3 y = d (b - acc), 4 y += d (b - acc)
template <int EPI>
__global__ __launch_bounds__(256) void mspmm_kernel(int ncol, int ld, const int* __restrict__ irp,
                                                    const int* __restrict__ ja, const double* __restrict__ val,
                                                    const double* __restrict__ x, const double* __restrict__ d,
                                                    const double* __restrict__ b, double* __restrict__ y) {
  const int i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= ncol) return;
  double acc = 0.0;
  const int k1 = irp[i + 1];
#pragma unroll 4
  for (int k = irp[i]; k < k1; ++k) acc = acc + val[k] * x[(size_t)ja[k] * ld + c];
  const size_t q = (size_t)i * ld + c;
  if (EPI == 0) y[q] = acc;
  else if (EPI == 1) y[q] = y[q] + acc;
  else if (EPI == 2) y[q] = b[q] - acc;
  else if (EPI == 3) y[q] = d[i] * (b[q] - acc);
  else y[q] = y[q] + d[i] * (b[q] - acc);
}
// y (+)= B x with the dense row-major n x n B
__global__ __launch_bounds__(256) void mdense_kernel(int n, int ncol, int ld, const double* __restrict__ B,
                                                     const double* __restrict__ x, double* __restrict__ y, int add) {
  const int i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= ncol) return;
  double acc = 0.0;
#pragma unroll 4
  for (int k = 0; k < n; ++k) acc = acc + B[(size_t)i * n + k] * x[(size_t)k * ld + c];
  const size_t q = (size_t)i * ld + c;
  y[q] = add ? y[q] + acc : acc;
}
// y (+)= d x (d null: 1)
__global__ __launch_bounds__(256) void mvmul_kernel(int ncol, int ld, const double* __restrict__ d,
                                                    const double* __restrict__ x, double* __restrict__ y, int add) {
  const int i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c >= ncol) return;
  const size_t q = (size_t)i * ld + c;
  const double t = d ? d[i] * x[q] : x[q];
  y[q] = add ? y[q] + t : t;
}
__global__ __launch_bounds__(256) void munit_kernel(int ncol, int ld, double* __restrict__ x, int identity) {
  const int i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c < ncol) x[(size_t)i * ld + c] = (identity && i == c) ? 1.0 : 0.0;
}
// t = solution of a triangular system: 64 columns per workgroup, its
// wavefronts share the rows of a level set, with a barrier between level sets
// (one thread per column going through all rows took 2.9 us per row, four
// dependent loads).  SC as in tri_row: 0 unit diagonal, 1 d b - acc, 2 (b -
// acc) / d.  b and t may be the same array.
constexpr int TRI_W = 8;
template <int SC>
__global__ __launch_bounds__(64 * TRI_W) void mtri_kernel(int nlv, const int* __restrict__ ptr,
                                                          const int* __restrict__ rows, int ncol, int ld,
                                                          const int* __restrict__ irp, const int* __restrict__ ja,
                                                          const double* __restrict__ val,
                                                          const double* __restrict__ d, const double* b, double* t) {
  const int c = min(blockIdx.x * 64 + (threadIdx.x & 63), ncol - 1);  // (a clamped column is computed twice, alike)
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  for (int lv = 0; lv < nlv; ++lv) {
    for (int q = ptr[lv] + w; q < ptr[lv + 1]; q += TRI_W) {
      const int i = rows[q];
      const double bi = b[(size_t)i * ld + c];
      double acc = 0.0;
      const int k1 = irp[i + 1];
#pragma unroll 4
      for (int k = irp[i]; k < k1; ++k) acc = acc + val[k] * t[(size_t)ja[k] * ld + c];
      if (blockIdx.x * 64 + (threadIdx.x & 63) < ncol)
        t[(size_t)i * ld + c] = SC == 1 ? d[i] * bi - acc : (SC == 2 ? (bi - acc) / d[i] : bi - acc);
    }
    __syncthreads();
  }
}
// the operator in the level's value type, rows of ldb entries (padding zero)
template <typename V>
__global__ __launch_bounds__(256) void mstore_kernel(int n, int ld, const double* __restrict__ y, int ldb,
                                                     V* __restrict__ B) {
  const int i = blockIdx.x, c = blockIdx.y * 256 + threadIdx.x;
  if (c < ldb) B[(size_t)i * ldb + c] = c < n ? (V)y[(size_t)i * ld + c] : (V)0;
}

struct Sm {
  int smoother = JAC, solver = DIAG_SCALE;
  int64_t nnz_nd = 0;
  DevSrc nd, l, u;
  const int *lptr = nullptr, *lrows = nullptr, *uptr = nullptr, *urows = nullptr;  // level sets of l and u
  int nl = 0, nu = 0;
  double* dv = nullptr;
  const double* dinv = nullptr;
};
struct Lev {
  int n = 0, pre = 0, post = 0, cycle = VCYCLE;
  DevSrc a, p, r;
  Sm sm, sm2;
  bool has2 = false;
  double *x = nullptr, *y = nullptr, *ty = nullptr, *tx = nullptr, *t1 = nullptr;
};

// The cycle of mld_dmlprec_aply (untransposed; no K-cycle) on multi-vectors
// of ncol columns.  run() leaves M X of the first level in its y; false where
// a smoother has no multi-vector form.
class Cycle {
 public:
  Cycle(std::vector<Lev>& L, int ncol, int ld, hipStream_t s) : L_(L), ncol_(ncol), ld_(ld), s_(s) {}
  bool run() {
    Lev& D = L_[0];
    munit_kernel<<<grid(D.n), 256, 0, s_>>>(ncol_, ld_, D.x, 1);
    return cycle(0);
  }

 private:
  std::vector<Lev>& L_;
  int ncol_, ld_;
  hipStream_t s_;
  dim3 grid(int n) const { return dim3(n, (ncol_ + 255) / 256); }
  template <int EPI>
  void mul(const DevSrc& m, const double* x, double* y, const double* b = nullptr, const double* d = nullptr) {
    if (m.nr > 0) mspmm_kernel<EPI><<<grid(m.nr), 256, 0, s_>>>(ncol_, ld_, m.irp, m.ja, m.val, x, d, b, y);
  }
  template <int SC>
  void tri(const Sm& S, bool lower, const double* d, const double* b, double* t) {
    const DevSrc& m = lower ? S.l : S.u;
    mtri_kernel<SC><<<(ncol_ + 63) / 64, 64 * TRI_W, 0, s_>>>(lower ? S.nl : S.nu, lower ? S.lptr : S.uptr,
                                                              lower ? S.lrows : S.urows, ncol_, ld_, m.irp, m.ja,
                                                              m.val, d, b, t);
  }
  void vmul(int n, const double* d, const double* x, double* y, int add) {
    mvmul_kernel<<<grid(n), 256, 0, s_>>>(ncol_, ld_, d, x, y, add);
  }
  bool solver(Lev& D, Sm& S, const double* x, int beta, double* y) {
    switch (S.solver) {
      case F_NONE: vmul(D.n, nullptr, x, y, beta); return true;
      case DIAG_SCALE:
      case L1_DIAG: vmul(D.n, S.dv, x, y, beta); return true;
      case ILU_N:
        tri<0>(S, true, nullptr, x, D.tx);
        tri<1>(S, false, S.dv, D.tx, D.tx);  // (row i of the right-hand side is read before it is overwritten)
        vmul(D.n, nullptr, D.tx, y, beta);
        return true;
      case DENSE_LU:
        mdense_kernel<<<grid(D.n), 256, 0, s_>>>(D.n, ncol_, ld_, S.dinv, x, y, beta);
        return true;
    }
    return false;
  }
  bool smooth(Lev& D, Sm& S, const double* x, int beta, double* y, int sweeps) {
    if (S.smoother == NOPREC) {
      vmul(D.n, nullptr, x, y, beta);
      return true;
    }
    if (sweeps < 0) return false;
    if (S.solver == GS || S.solver == BWGS) {
      const bool fw = S.solver == GS;
      for (int sw = 1; sw <= std::max(1, sweeps); ++sw) {
        const double* b = x;
        if (sw > 1) {
          mul<2>(fw ? S.u : S.l, D.tx, D.t1, x);
          b = D.t1;
        }
        tri<2>(S, fw, S.dv, b, D.tx);
      }
      vmul(D.n, nullptr, D.tx, y, beta);
      return true;
    }
    if (sweeps <= 1 || S.nnz_nd == 0) return solver(D, S, x, beta, y);
    if (S.solver != DIAG_SCALE && S.solver != L1_DIAG) return false;
    double *ta = D.tx, *tb = D.t1;
    vmul(D.n, S.dv, x, ta, 0);
    for (int sw = 2; sw < sweeps; ++sw) {
      mul<3>(S.nd, ta, tb, x, S.dv);
      std::swap(ta, tb);
    }
    if (beta) mul<4>(S.nd, ta, y, x, S.dv);
    else mul<3>(S.nd, ta, y, x, S.dv);
    return true;
  }
  bool down(Lev& D, size_t l, const double* r) {
    Lev& C = L_[l + 1];
    mul<0>(C.r, r, C.x);
    if (!cycle(l + 1)) return false;
    mul<1>(C.p, C.y, D.y);
    return true;
  }
  bool cycle(size_t l) {
    Lev& D = L_[l];
    if (D.cycle == ADD_ML) {
      if (D.has2) {
        vmul(D.n, nullptr, D.x, D.y, 0);
        for (int k = 0; k < std::max(D.pre, D.post); ++k)
          if (!smooth(D, D.sm, D.y, 0, D.ty, 1) || !smooth(D, D.sm2, D.ty, 0, D.y, 1)) return false;
      } else if (!smooth(D, D.sm, D.x, 0, D.y, D.pre)) {
        return false;
      }
      return l + 1 == L_.size() || down(D, l, D.x);
    }
    if (D.cycle != MULT_ML && D.cycle != VCYCLE && D.cycle != WCYCLE) return false;
    if (l + 1 == L_.size()) return smooth(D, D.sm, D.x, 0, D.y, D.pre);
    if (D.pre > 0) {
      if (!smooth(D, D.sm, D.x, 0, D.y, D.pre)) return false;
      mul<2>(D.a, D.y, D.ty, D.x);
      if (!down(D, l, D.ty)) return false;
    } else {
      munit_kernel<<<grid(D.n), 256, 0, s_>>>(ncol_, ld_, D.y, 0);
      if (!down(D, l, D.x)) return false;
    }
    if (D.cycle == WCYCLE) {
      mul<2>(D.a, D.y, D.ty, D.x);
      if (!down(D, l, D.ty)) return false;
    }
    if (D.post > 0) {
      mul<2>(D.a, D.y, D.ty, D.x);
      return smooth(D, D.has2 ? D.sm2 : D.sm, D.ty, 1, D.y, D.post);
    }
    return true;
  }
};

}  // namespace tail
}  // namespace mld
