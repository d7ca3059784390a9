// One-workgroup kernels of FGMRES for small systems (fgmres_small.hip).
#pragma once

#include "fgmres_dev.h"
#include "kernels.h"

namespace impes {

// Systems up to this size take them. One workgroup reads the basis at one CU's rate,
// so a step's time grows with rows times basis vectors, while the separate kernels
// cost about 25 us of launches per step.
constexpr int kSmallRows = 4096;
constexpr long long kSmallRowNnz = 16;

struct SmallOperator {
  bool stencil = false;
  Stencil7<double> st{};
  CsrF64 csr{};
  const double* dinv = nullptr;
  int n = 0;
};

// S, sout: the preconditioner's input and output scalings; bout, x: its input and
// output vectors in precision T; host: device address of the pinned scalars.
void small_start(const SmallOperator& A, FgmresLayout L, double* sm, const double* b, double* x, bool use_x0, double* V,
                 double* host, hipStream_t s);
template <class T>
void small_begin(int n, FgmresLayout L, double* sm, double* V, const double* S, T* bout, hipStream_t s);
template <class T>
void small_step(const SmallOperator& A, FgmresLayout L, int j, double* sm, const T* x, const double* sout, double* Z,
                double* V, const double* S, T* bout, double* est, hipStream_t s);
template <class T>
void small_end(const SmallOperator& A, FgmresLayout L, int k, bool close, double* sm, const double* Z, double* V,
               const double* b, double* x, const double* S, T* bout, double* host, hipStream_t s);
template <class T>
void small_input(int n, const double* V, const double* S, T* bout, hipStream_t s);
template <class T>
void small_check(const SmallOperator& A, FgmresLayout L, double* sm, const T* xc, const double* sout, double* V,
                 const double* b, double* x, double* host, hipStream_t s);

}  // namespace impes
