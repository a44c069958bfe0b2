// SpMV kernels for gfx950 (MI355X, CDNA4, 64-wide wavefronts).
//
// csr_tile_kernel   one workgroup per tile of 1024, 2048 or 3072 entries.
//                   Entries are read with 16-byte loads (4, 8 or 12 entries
//                   per thread), multiplied by the gathered x, and staged in
//                   LDS; each row that starts in the tile is then summed by
//                   one thread in entry order.  With FP64 this reproduces the
//                   reference loop MatrixCSR.cpp:133-139 bit for bit (product
//                   rounded, then a left-to-right sum starting from 0).
//                   Columns are read packed in three bytes where they fit
//                   (pack_columns).
// csr_long_kernel   rows longer than 1536 entries, one workgroup each.
// ell_kernel        one row per thread over the sliced column-major slots (one
//                   contiguous block per workgroup), eight slots per step;
//                   same order as MatrixELL.cpp:105-113 (contraction off, so
//                   bit-identical in FP64).
// coo_tile_kernel   COO/SCOO: the CSR entry-tile kernel on the row segments of
//                   the row-sorted view, each segment's sum starting from
//                   y[row], so each row is accumulated in entry order
//                   (MatrixCOO.cpp:113-115 / MatrixSCOO.cpp:120-122 with one
//                   thread).
// dense_kernel      one row per wavefront, or four sharing each x load, butterfly
//                   reduction
//                   (MatrixDENSE.cpp:67-72, different summation order).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "tile_csr.hpp"

namespace tbsla {
namespace hip {
namespace {

using dev::bf16;
using dev::block_tree_sum;
using dev::nt_load;
using dev::Val;

template <typename YT>
struct StoreRow {
  YT *y;
  template <typename AT>
  __device__ void operator()(int row, AT s) const {
    y[row] = static_cast<YT>(s);
  }
};

template <typename VT, typename XT, typename YT, int TN, int LOADS>
__global__ __launch_bounds__(kTileThreads) void csr_tile_kernel(dev::CsrView<VT> m, const XT *__restrict__ x,
                                                                YT *__restrict__ y) {
  __shared__ dev::CsrTileLds<typename Val<VT>::A, TN> lds;
  StoreRow<YT> epi{y};
  dev::csr_tile_rows<VT, XT, TN, static_cast<dev::TileLoads>(LOADS)>(m, x, lds, epi);
}

template <typename VT, typename XT, typename YT>
__global__ __launch_bounds__(kTileThreads) void csr_long_kernel(dev::CsrView<VT> m, const XT *__restrict__ x,
                                                                YT *__restrict__ y) {
  __shared__ dev::CsrTileLds<typename Val<VT>::A, kTileThreads> lds;
  StoreRow<YT> epi{y};
  dev::csr_long_row<VT, XT, kTileThreads>(m, x, lds, epi);
}

// ELL: one row per thread, one workgroup per slice of kEllSlice rows, whose
// K slots lie in one contiguous block (slot j of the slice's row t at
// j * kEllSlice + t), so a workgroup streams one block of HBM and every slot
// is one coalesced load per wavefront.  Slots go in groups of kEllGroup; the
// next group's loads are issued before this group's gathers (two register
// sets, alternating), so each group waits on one round trip.  Each row still
// sums its slots in order 0..K-1.  Bound by the HBM reads of the slots: columns
// are read packed in three bytes where they fit (pack_ell_columns).
constexpr int kEllGroup = 8;

__device__ inline double ell_value(const double *p, long i) { return __builtin_nontemporal_load(p + i); }
__device__ inline float ell_value(const float *p, long i) { return __builtin_nontemporal_load(p + i); }
__device__ inline float ell_value(const bf16 *p, long i) {
  return Val<bf16>::cvt(__builtin_nontemporal_load(reinterpret_cast<const unsigned short *>(p) + i));
}

// Columns of N slots from slot j of the slice: `cols` points at the thread's
// first slot (plain) or its first group's words (packed; j a multiple of 4).
template <bool PACK, int N>
__device__ inline void ell_columns(const int *__restrict__ cols, int j, int (&c)[kEllGroup]) {
  if constexpr (PACK) {
#pragma unroll
    for (int g = 0; g < (N + 3) / 4; g++) {
      const int *w = cols + static_cast<long>(j / 4 + g) * kEllSlice * 3;
      const unsigned a = static_cast<unsigned>(__builtin_nontemporal_load(w)),
                     b = static_cast<unsigned>(__builtin_nontemporal_load(w + 1)),
                     d = static_cast<unsigned>(__builtin_nontemporal_load(w + 2));
      c[4 * g] = static_cast<int>(a & 0xFFFFFFu);
      c[4 * g + 1] = static_cast<int>(a >> 24 | (b & 0xFFFFu) << 8);
      c[4 * g + 2] = static_cast<int>(b >> 16 | (d & 0xFFu) << 16);
      c[4 * g + 3] = static_cast<int>(d >> 8);
    }
  } else {
#pragma unroll
    for (int u = 0; u < N; u++) c[u] = nt_load(cols, static_cast<long>(j + u) * kEllSlice);
  }
}

template <typename VT, bool PACK>
struct EllGroup {
  using AT = typename Val<VT>::A;
  int c[kEllGroup];
  AT v[kEllGroup];

  // slots j, j + 1, ... (N of them)
  template <int N>
  __device__ void load(const int *__restrict__ cols, const VT *__restrict__ vals, int j) {
    ell_columns<PACK, N>(cols, j, c);
#pragma unroll
    for (int u = 0; u < N; u++) v[u] = ell_value(vals, static_cast<long>(j + u) * kEllSlice);
  }
  template <int N, typename XT>
  __device__ void accumulate(const XT *__restrict__ x, AT &acc) const {
#pragma clang fp contract(off)
    AT xv[N];
#pragma unroll
    for (int u = 0; u < N; u++) xv[u] = static_cast<AT>(x[c[u]]);
#pragma unroll
    for (int u = 0; u < N; u++) acc += v[u] * xv[u];
  }
};

// GROUPS: K is at least kEllGroup.  Rows of fewer slots are bound by the loads
// in flight, so by the wavefronts, and carry no registers for a second group
// (4,000,001 rows FP32: one slot 18.3 -> 16.3 us, five 43.0 -> 39.8).
template <typename VT, typename XT, typename YT, bool PACK, bool GROUPS>
__global__ __launch_bounds__(kEllSlice) void ell_kernel(const int *__restrict__ cols, const VT *__restrict__ vals,
                                                        const XT *__restrict__ x, YT *__restrict__ y, int rows,
                                                        int K) {
  using AT = typename Val<VT>::A;
  const long i = static_cast<long>(blockIdx.x) * kEllSlice + threadIdx.x;
  if (i >= rows) return;
  vals += static_cast<long>(blockIdx.x) * K * kEllSlice + threadIdx.x;
  cols += PACK ? (static_cast<long>(blockIdx.x) * ((K + 3) / 4) * kEllSlice + threadIdx.x) * 3
               : static_cast<long>(blockIdx.x) * K * kEllSlice + threadIdx.x;
  const int KG = K - K % kEllGroup;  // slots in whole groups
  AT acc = 0;
  EllGroup<VT, PACK> A;
  int j = 0;
  if constexpr (GROUPS) {
    EllGroup<VT, PACK> B;
    A.template load<kEllGroup>(cols, vals, 0);
    while (j < KG) {
      if (j + kEllGroup < KG) B.template load<kEllGroup>(cols, vals, j + kEllGroup);
      A.template accumulate<kEllGroup>(x, acc);
      j += kEllGroup;
      if (j >= KG) break;
      if (j + kEllGroup < KG) A.template load<kEllGroup>(cols, vals, j + kEllGroup);
      B.template accumulate<kEllGroup>(x, acc);
      j += kEllGroup;
    }
  }
  // the last K % kEllGroup slots: four together, then one to three
  if (K - j >= 4) {
    A.template load<4>(cols, vals, j);
    A.template accumulate<4>(x, acc);
    j += 4;
  }
  if (K - j == 3) {
    A.template load<3>(cols, vals, j);
    A.template accumulate<3>(x, acc);
  } else if (K - j == 2) {
    A.template load<2>(cols, vals, j);
    A.template accumulate<2>(x, acc);
  } else if (K - j == 1) {
    A.template load<1>(cols, vals, j);
    A.template accumulate<1>(x, acc);
  }
  y[i] = static_cast<YT>(acc);
}

// COO/SCOO segment epilogue: the segment's sum started from y[row], so the
// row is accumulated y[row] += v * x in entry order (MatrixCOO.cpp:113-115).
template <typename YT>
struct AccRow {
  YT *y;
  const int *segrow;
  long y_off;
  template <typename AT>
  __device__ AT init(int s) const {
    return static_cast<AT>(y[segrow[s] + y_off]);
  }
  template <typename AT>
  __device__ void operator()(int s, AT v) const {
    y[segrow[s] + y_off] = static_cast<YT>(v);
  }
};

template <typename VT, typename XT, typename YT, int TN, int LOADS, bool LONG>
__global__ __launch_bounds__(kTileThreads) void coo_tile_kernel(dev::CsrView<VT> m, const XT *__restrict__ x,
                                                                YT *__restrict__ y, const int *__restrict__ segrow,
                                                                long y_off) {
  __shared__ dev::CsrTileLds<typename Val<VT>::A, TN> lds;
  AccRow<YT> epi{y, segrow, y_off};
  if constexpr (LONG)
    dev::csr_long_row<VT, XT, TN>(m, x, lds, epi);
  else
    dev::csr_tile_rows<VT, XT, TN, static_cast<dev::TileLoads>(LOADS)>(m, x, lds, epi);
}

// R consecutive rows per wavefront, so each x load serves all of them; per row
// and lane the columns are summed in one order whatever R is (j = 2*lane +
// 128*k; short rows lane + 64*k), then a butterfly.  Bound by the HBM reads of
// A: two steps of R 16-byte loads in flight, non-temporal, and with an odd row
// length every other row starts 8 bytes off a 16-byte boundary, which the loads
// allow (8191 x 8191: 247 us with 8-byte loads, 83 now; 8192 x 8192 83 in both,
// 6.5 TB/s).
// Rows of at most kDenseShortRow columns take a column a lane: two columns a
// lane leave half the lanes of a short row idle (1,000,000 x 15 224.5 us, 173.7
// so; x 16 216 and 172; x 63 260 and 198; 300,000 x 161 142 and 116; x 192 114.5
// and 115.7; x 208 117 and 141).
constexpr int kDenseShortRow = 192;
template <typename XT, typename YT, int R>
__global__ __launch_bounds__(256) void dense_kernel(const double *__restrict__ A, const XT *__restrict__ x,
                                                    YT *__restrict__ y, int rows, int cols, long ld) {
  const int w = (blockIdx.x * 256 + threadIdx.x) >> 6;
  const int lane = threadIdx.x & 63;
  const long r0 = static_cast<long>(w) * R;
  if (r0 >= rows) return;
  const int nr = static_cast<int>(min(static_cast<long>(R), rows - r0));  // rows of this wavefront
  double acc[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = 0;
  typedef double v2d_8 __attribute__((ext_vector_type(2), aligned(8)));
  if (cols <= kDenseShortRow) {
#pragma unroll
    for (int r = 0; r < R; r++)
      if (r < nr)
        for (int k = lane; k < cols; k += 64)
          acc[r] += __builtin_nontemporal_load(A + (r0 + r) * ld + k) * static_cast<double>(x[k]);
  }
  int j = cols <= kDenseShortRow ? cols : 2 * lane;
  for (; j + 128 + 1 < cols; j += 2 * 128) {
    v2d_8 av[2][R];
    double xv[2][2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      xv[u][0] = static_cast<double>(x[j + u * 128]);
      xv[u][1] = static_cast<double>(x[j + u * 128 + 1]);
#pragma unroll
      for (int r = 0; r < R; r++)
        av[u][r] = r < nr ? __builtin_nontemporal_load(
                                reinterpret_cast<const v2d_8 *>(A + (r0 + r) * ld + j + u * 128))
                          : v2d_8{0, 0};
    }
#pragma unroll
    for (int u = 0; u < 2; u++)
#pragma unroll
      for (int r = 0; r < R; r++) acc[r] += av[u][r].x * xv[u][0] + av[u][r].y * xv[u][1];
  }
  for (; j < cols; j += 128)
#pragma unroll
    for (int r = 0; r < R; r++)
      if (r < nr) {
        const double *a = A + (r0 + r) * ld;
        acc[r] += __builtin_nontemporal_load(a + j) * static_cast<double>(x[j]);
        if (j + 1 < cols) acc[r] += __builtin_nontemporal_load(a + j + 1) * static_cast<double>(x[j + 1]);
      }
#pragma unroll
  for (int r = 0; r < R; r++) {
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc[r] += __shfl_xor(acc[r], off, 64);
  }
  if (lane == 0)
#pragma unroll
    for (int r = 0; r < R; r++)
      if (r < nr) y[r0 + r] = static_cast<YT>(static_cast<double>(y[r0 + r]) + acc[r]);
}

template <typename T>
__global__ void fill_kernel(T *y, long n, T v) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256) y[i] = v;
}

// three words of packed columns for the four entries of group g (0 past the end)
__global__ __launch_bounds__(256) void pack24_kernel(const int *__restrict__ colidx, long nnz, int f_col, bool pairs,
                                                     unsigned *__restrict__ out) {
  const long groups = (nnz + 255) / 256 * 64;
  for (long g = blockIdx.x * 256L + threadIdx.x; g < groups; g += static_cast<long>(gridDim.x) * 256) {
    unsigned c[4];
    for (int q = 0; q < 4; q++) {
      const long e = pairs ? (g & ~63L) * 4 + 2 * (g & 63) + (q >> 1) * 128 + (q & 1) : 4 * g + q;
      c[q] = e < nnz ? static_cast<unsigned>(colidx[e] - f_col) : 0u;
    }
    out[3 * g] = c[0] | c[1] << 24;
    out[3 * g + 1] = c[1] >> 8 | c[2] << 16;
    out[3 * g + 2] = c[2] >> 16 | c[3] << 8;
  }
}

// the columns of slot group j / 4 of every row of every slice (plain layout
// `in`, K slots; slots past K: column 0), as DeviceMatrix::ecols packed
__global__ __launch_bounds__(kEllSlice) void pack_ell_kernel(const int *__restrict__ in, int K,
                                                             unsigned *__restrict__ out) {
  const int KQ = (K + 3) / 4;
  for (int g = 0; g < KQ; g++) {
    unsigned c[4];
    for (int q = 0; q < 4; q++)
      c[q] = 4 * g + q < K ? static_cast<unsigned>(in[(static_cast<long>(blockIdx.x) * K + 4 * g + q) * kEllSlice +
                                                      threadIdx.x])
                           : 0u;
    unsigned *o = out + ((static_cast<long>(blockIdx.x) * KQ + g) * kEllSlice + threadIdx.x) * 3;
    o[0] = c[0] | c[1] << 24;
    o[1] = c[1] >> 8 | c[2] << 16;
    o[2] = c[2] >> 16 | c[3] << 8;
  }
}

inline unsigned blocks_for(long n, int per_block) { return static_cast<unsigned>((n + per_block - 1) / per_block); }

// Four rows per wavefront from 7168 rows on, where that still fills the chip
// (seven wavefronts a CU); one below: 2000 x 2000 10.9 us with four, 8.3 with
// one, 4096 28.3 and 21.6, 7001 66.2 and 64.4, 8192 83.0 and 85.9.
constexpr int kDenseRows = 4, kDenseManyRows = 7168;

template <typename XT, typename YT>
void launch_dense(const DeviceMatrix &d, const XT *x, YT *y, hipStream_t s) {
  const bool many = d.rows >= kDenseManyRows;
  const long waves = many ? (static_cast<long>(d.rows) + kDenseRows - 1) / kDenseRows : d.rows;
  const auto kernel = many ? dense_kernel<XT, YT, kDenseRows> : dense_kernel<XT, YT, 1>;
  hipLaunchKernelGGL(kernel, dim3(blocks_for(waves * 64, 256)), dim3(256), 0, s, d.dvals.as<double>(), x, y, d.rows,
                     d.dcols, static_cast<long>(d.dcols));
}

template <typename VT, typename F>
void with_loads(const dev::CsrView<VT> &m, F f) {
  if (m.col24 && m.stream)
    f(std::integral_constant<int, dev::kPackedStream>());
  else if (m.col24)
    f(std::integral_constant<int, dev::kPacked>());
  else if (m.stream)
    f(std::integral_constant<int, dev::kStream>());
  else
    f(std::integral_constant<int, dev::kPlain>());
}

template <typename VT, typename XT, typename YT>
void run_typed(const DeviceMatrix &d, const XT *x, YT *y, int vect_incr, hipStream_t s) {
  switch (d.format) {
    case cpp::FORMAT_CSR: {
      const dev::CsrView<VT> m = dev::csr_view<VT>(d);
      if (d.ntiles > 0)
        with_tile_size(d, [&](auto tn) {
          constexpr int TN = decltype(tn)::value;
          with_loads(m, [&](auto loads) {
            hipLaunchKernelGGL((csr_tile_kernel<VT, XT, YT, TN, decltype(loads)::value>), dim3(d.ntiles),
                               dim3(kTileThreads), 0, s, m, x, y);
          });
        });
      if (d.nlong > 0)
        hipLaunchKernelGGL((csr_long_kernel<VT, XT, YT>), dim3(d.nlong), dim3(kTileThreads), 0, s, m, x, y);
      break;
    }
    case cpp::FORMAT_ELL:
      if (d.rows > 0)
        hipLaunchKernelGGL((d.K < kEllGroup ? (d.epacked ? ell_kernel<VT, XT, YT, true, false>
                                                         : ell_kernel<VT, XT, YT, false, false>)
                                            : (d.epacked ? ell_kernel<VT, XT, YT, true, true>
                                                         : ell_kernel<VT, XT, YT, false, true>)),
                           dim3(blocks_for(d.rows, kEllSlice)), dim3(kEllSlice), 0, s, d.ecols.as<int>(),
                           d.evals.as<VT>(), x, y, d.rows, d.K);
      break;
    case cpp::FORMAT_COO:
    case cpp::FORMAT_SCOO: {
      // columns: global (COO) or minus f_col (SCOO, the view's f_col);
      // rows: + vect_incr (- f_row for SCOO)
      const dev::CsrView<VT> m = dev::csr_view<VT>(d);
      const long y_off = vect_incr - (d.format == cpp::FORMAT_SCOO ? d.f_row : 0);
      if (d.ntiles > 0)
        with_tile_size(d, [&](auto tn) {
          constexpr int TN = decltype(tn)::value;
          with_loads(m, [&](auto loads) {
            hipLaunchKernelGGL((coo_tile_kernel<VT, XT, YT, TN, decltype(loads)::value, false>), dim3(d.ntiles),
                               dim3(kTileThreads), 0, s, m, x, y, d.segrow.as<int>(), y_off);
          });
        });
      if (d.nlong > 0)
        hipLaunchKernelGGL((coo_tile_kernel<VT, XT, YT, kTileThreads, dev::kPlain, true>), dim3(d.nlong), dim3(kTileThreads), 0, s, m, x, y,
                           d.segrow.as<int>(), y_off);
      break;
    }
    case cpp::FORMAT_DENSE:
      if (d.rows > 0) launch_dense<XT, YT>(d, x, y, s);
      break;
  }
  TBSLA_HIP_CHECK(hipGetLastError());
}

}  // namespace

void launch_spmv(const DeviceMatrix &d, const void *x, Dtype xdt, void *y, Dtype ydt, int vect_incr,
                 hipStream_t s) {
  if (d.noop) return;
  if (d.vdt == Dtype::F64 && xdt == Dtype::F64 && ydt == Dtype::F64) {
    run_typed<double, double, double>(d, static_cast<const double *>(x), static_cast<double *>(y), vect_incr, s);
  } else if (d.vdt == Dtype::F32 && xdt == Dtype::F32 && ydt == Dtype::F32 && d.format != cpp::FORMAT_DENSE) {
    run_typed<float, float, float>(d, static_cast<const float *>(x), static_cast<float *>(y), vect_incr, s);
  } else if (d.vdt == Dtype::BF16 && xdt == Dtype::F32 && ydt == Dtype::F32 && d.format != cpp::FORMAT_DENSE) {
    run_typed<bf16, float, float>(d, static_cast<const float *>(x), static_cast<float *>(y), vect_incr, s);
  } else {
    throw std::invalid_argument("tbsla: unsupported value/vector type combination for this format");
  }
}

void pack_columns(DeviceMatrix &d, bool pairs) {
  if (d.entries <= 0 || d.x_need > (1L << 24)) return;
  DevBuf &out = pairs ? d.col24_pairs : d.col24;
  const long groups = (d.entries + 255) / 256 * 64;
  if (!out.try_reserve(static_cast<std::size_t>(groups) * 12)) return;
  hipLaunchKernelGGL(pack24_kernel, dim3(static_cast<unsigned>(std::min<long>((groups + 255) / 256, 65536))), dim3(256),
                     0, nullptr, d.colidx.as<int>(), d.entries, d.f_col, pairs, out.as<unsigned>());
  TBSLA_HIP_CHECK(hipGetLastError());
}

void pack_ell_columns(DeviceMatrix &d) {
  if (d.rows <= 0 || d.x_need > (1L << 24) || 3 * ((d.K + 3) / 4) >= d.K) return;
  const unsigned slices = blocks_for(d.rows, kEllSlice);
  DevBuf out;
  if (!out.try_reserve(static_cast<std::size_t>(slices) * static_cast<std::size_t>((d.K + 3) / 4) * kEllSlice * 12))
    return;
  hipLaunchKernelGGL(pack_ell_kernel, dim3(slices), dim3(kEllSlice), 0, nullptr, d.ecols.as<int>(), d.K,
                     out.as<unsigned>());
  TBSLA_HIP_CHECK(hipGetLastError());
  TBSLA_HIP_CHECK(hipDeviceSynchronize());
  d.ecols = std::move(out);
  d.epacked = true;
}

void launch_fill(void *y, Dtype ydt, long n, double value, hipStream_t s) {
  if (n <= 0) return;
  const unsigned g = static_cast<unsigned>(std::min<long>((n + 255) / 256, 65536));
  if (ydt == Dtype::F64)
    hipLaunchKernelGGL(fill_kernel<double>, dim3(g), dim3(256), 0, s, static_cast<double *>(y), n, value);
  else if (ydt == Dtype::F32)
    hipLaunchKernelGGL(fill_kernel<float>, dim3(g), dim3(256), 0, s, static_cast<float *>(y), n,
                       static_cast<float>(value));
  else
    throw std::invalid_argument("tbsla: fill supports F64/F32 vectors");
  TBSLA_HIP_CHECK(hipGetLastError());
}

const char *spmv_kernel_name(cpp::Format f) {
  switch (f) {
    case cpp::FORMAT_CSR: return "csr_tile_kernel";
    case cpp::FORMAT_ELL: return "ell_kernel";
    case cpp::FORMAT_COO:
    case cpp::FORMAT_SCOO: return "coo_tile_kernel";
    case cpp::FORMAT_DENSE: return "dense_kernel";
  }
  return "";
}

}  // namespace hip
}  // namespace tbsla
