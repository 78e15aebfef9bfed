// One matrix on the host through the route that a batch of `batch` matrices of
// its order takes (the per-matrix entries of veig_compat.hpp: the kernels differ
// in the order of their operations, and the values are to be the batch entry's).
// Contiguous planes; each returns a veig_status.
#pragma once

#include <cstdint>

namespace veig {
int slot_zgehrd(int dim, int64_t batch, double *rA, double *iA, double *rtau, double *itau);
int slot_zunghr(int dim, int64_t batch, double *rA, double *iA, double *rtau, double *itau);
int slot_zlahqr(int dim, int64_t batch, double *rE, double *iE, double *rH, double *iH, double *rZ, double *iZ);
int slot_ztrevc(int dim, int64_t batch, double *rT, double *iT, double *rR, double *iR);
}  // namespace veig
