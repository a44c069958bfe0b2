// Host-callable launchers of the SpMV kernels (spmv.hip).
#pragma once

#include "mirror.hpp"

namespace tbsla {
namespace hip {

// One product with the reference's Ax semantics on device vectors:
//   CSR, ELL   y[i]  = sum_j A(i,j) x(j)   for the rows the matrix defines
//   COO, SCOO  y[r + vect_incr (- f_row)] += A(r,c) x(c (- f_col)), entry order per row
//   DENSE      y[i] += sum_j A(i,j) x(j)
// Supported element types: values F64 with x, y F64; values F32/BF16 with
// x, y F32 (float accumulation).  Throws on an unsupported combination.
void launch_spmv(const DeviceMatrix &d, const void *x, Dtype xdt, void *y, Dtype ydt, int vect_incr,
                 hipStream_t s);

// d.col24 (pairs: d.col24_pairs) from d.colidx, if every local column (x_need
// of them) fits 24 bits and the memory is there: the tile products then read
// 11 instead of 12 bytes an entry in FP64, 7 instead of 8 in FP32.  Packed
// against not: 62 million entries CSR FP64 141.5 -> 132.7 us, SCOO 148.0 ->
// 140.0, CSR FP32 105.7 -> 100.3; 1,000,003 rows of 16 FP64 56.1 -> 53.8 and
// FP32 34.9 -> 32.5, 500,009 FP64 28.0 -> 26.7.
void pack_columns(DeviceMatrix &d, bool pairs);

// The same for an ELL mirror, whose slots' columns are replaced (groups of
// four; plain if the memory for both during the change is not there): 4194304
// rows of 16 FP64 150.0 -> 142.0 us, 1,000,003 rows FP64 43.3 -> 41.2 and FP32
// 30.7 -> 28.5, 300,007 rows of 12 FP64 15.3 -> 11.9.  A group is three words
// whatever it holds, so up to three slots, and at five, six and nine, rows stay
// plain: packed, 4,000,001 rows of one FP32 slot took 22.0 us against 18.3, of
// two 27.6 against 24.5, of five 45.5 against 43.0.
void pack_ell_columns(DeviceMatrix &d);

// y[0:n) = value
void launch_fill(void *y, Dtype ydt, long n, double value, hipStream_t s);

// Kernel symbol names (for profiles): one per format.
const char *spmv_kernel_name(cpp::Format f);

}  // namespace hip
}  // namespace tbsla
