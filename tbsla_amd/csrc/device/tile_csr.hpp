// Device building blocks shared by spmv.hip and pagerank.hip (device code;
// include only from .hip translation units).
//
// CSR products use fixed entry tiles: tile t holds entries [t*T, (t+1)*T)
// (T = the caller's TN, 1024 to kCsrTileNnz) and owns the rows whose first
// entry lies in it (tile_row[t] .. tile_row[t+1]).  A tile's entries are read
// with 16-byte loads (packed columns: 12 bytes) at an aligned offset that needs
// no descriptor load, the products v * x[c] are rounded and staged in LDS, and
// each owned row is summed by one thread from 0, left to right; of a row that
// runs past the tile the rest is staged too (kTileTail).  That reproduces the
// sequential FP64 row sum of MatrixCSR.cpp:133-139 exactly.  Rows longer than
// kCsrLongRow entries (the batch: kBatchLongRow) are left to csr_long_row (one
// workgroup per row, fixed-order tree).
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "mirror.hpp"

namespace tbsla {
namespace hip {
namespace dev {

struct bf16 {
  unsigned short bits;
};

// round to nearest even via FP32, as the CSR mirror's values
__device__ inline unsigned short bf16_of(double d) {
  const float f = static_cast<float>(d);
  unsigned u = __float_as_uint(f);
  if ((u & 0x7f800000u) == 0x7f800000u) return static_cast<unsigned short>(u >> 16);
  u += 0x7fffu + ((u >> 16) & 1u);
  return static_cast<unsigned short>(u >> 16);
}

typedef double v2d __attribute__((ext_vector_type(2)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef unsigned short v4us __attribute__((ext_vector_type(4)));

// A load, non-temporal or plain.
template <bool NT, typename V>
__device__ inline V vec_load(const V *p) {
  if constexpr (NT) return __builtin_nontemporal_load(p);
  return *p;
}

template <typename T>
struct Val;
template <>
struct Val<double> {
  using A = double;
  static constexpr int kXBytes = 8;
  __device__ static double get(const double *p, long i) { return p[i]; }
  // four consecutive values starting at a multiple of 4
  __device__ static void get4(const double *p, long i, double (&v)[4]) { get22<false>(p, i, i + 2, v); }
  // two from i, two from j
  template <bool NT>
  __device__ static void get22(const double *p, long i, long j, double (&v)[4]) {
    const v2d a = vec_load<NT>(reinterpret_cast<const v2d *>(p + i));
    const v2d b = vec_load<NT>(reinterpret_cast<const v2d *>(p + j));
    v[0] = a.x;
    v[1] = a.y;
    v[2] = b.x;
    v[3] = b.y;
  }
};
template <>
struct Val<float> {
  using A = float;
  static constexpr int kXBytes = 4;
  __device__ static float get(const float *p, long i) { return p[i]; }
  template <bool NT = false>
  __device__ static void get4(const float *p, long i, float (&v)[4]) {
    const v4f a = vec_load<NT>(reinterpret_cast<const v4f *>(p + i));
    v[0] = a.x;
    v[1] = a.y;
    v[2] = a.z;
    v[3] = a.w;
  }
};
template <>
struct Val<bf16> {
  using A = float;
  static constexpr int kXBytes = 4;
  __device__ static float cvt(unsigned short b) { return __uint_as_float(static_cast<unsigned>(b) << 16); }
  __device__ static float get(const bf16 *p, long i) { return cvt(reinterpret_cast<const unsigned short *>(p)[i]); }
  template <bool NT = false>
  __device__ static void get4(const bf16 *p, long i, float (&v)[4]) {
    const v4us a = vec_load<NT>(reinterpret_cast<const v4us *>(reinterpret_cast<const unsigned short *>(p) + i));
    v[0] = cvt(a.x);
    v[1] = cvt(a.y);
    v[2] = cvt(a.z);
    v[3] = cvt(a.w);
  }
};

__device__ inline int nt_load(const int *p, long i) { return __builtin_nontemporal_load(p + i); }

// Sum of one value per thread over a block of kTileThreads, fixed order.
template <typename AT>
__device__ inline AT block_tree_sum(AT v, AT *part) {
  part[threadIdx.x] = v;
  __syncthreads();
  for (int s = kTileThreads / 2; s > 0; s >>= 1) {
    if (static_cast<int>(threadIdx.x) < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  AT r = part[0];
  __syncthreads();
  return r;
}

template <typename AT>
__device__ inline AT block_tree_max(AT v, AT *part) {
  part[threadIdx.x] = v;
  __syncthreads();
  for (int s = kTileThreads / 2; s > 0; s >>= 1) {
    if (static_cast<int>(threadIdx.x) < s) part[threadIdx.x] = fmax(part[threadIdx.x], part[threadIdx.x + s]);
    __syncthreads();
  }
  AT r = part[0];
  __syncthreads();
  return r;
}

// The four entries of a tile's group in a thread: eight-byte values go two and
// two (lane l of the wavefront's 256 entries has 2l, 2l + 1, 128 + 2l, 129 +
// 2l), so that each 16-byte load of a wavefront is one run of 1 KB (with 32
// bytes a lane, read in halves, non-temporal loads fetched lines twice: 62
// million entries 161.8 us, 142.5 so); smaller values four in a row.
template <typename VT>
__host__ __device__ constexpr bool tile_pairs() {
  return sizeof(typename Val<VT>::A) == 8;
}
// Place of entry e in the order of the groups' threads.
template <typename VT>
__device__ inline long tile_place(long e) {
  return tile_pairs<VT>() ? (e & ~255L) + 4 * ((e & 127) >> 1) + ((e & 128) >> 6) + (e & 1) : e;
}

// Device view of a CSR mirror (entry j of the matrix is colidx[j], vals[j],
// with j = rowptr[i] - rp0 + k for the k-th entry of row i).  colidx is the
// mirror's padded buffer; vals may be a caller's array of exactly nnz
// values, so no value is read at index nnz or beyond.
template <typename VT>
struct CsrView {
  const int *rowptr;
  const int *colidx;
  const VT *vals;  // nullptr for the value-free view
  const int *tile_row;
  const int *long_rows;
  long nnz;
  int rp0, f_col;
  // the columns minus f_col packed in three bytes each (little endian, four
  // in three words; column of entry e at 3 * tile_place<VT>(e)), or nullptr
  const unsigned *col24 = nullptr;
  bool stream = false;  // the entries are read non-temporally (stream_entries)

  // the local column of entry e, in a load and what is done with its word
  __device__ unsigned col_word(long e) const {
    typedef unsigned u32_u __attribute__((aligned(1)));
    if (col24)
      return *reinterpret_cast<const u32_u *>(reinterpret_cast<const char *>(col24) + 3 * tile_place<VT>(e));
    return static_cast<unsigned>(colidx[e]);
  }
  __device__ int col_of(unsigned w) const { return col24 ? static_cast<int>(w & 0xFFFFFFu) : static_cast<int>(w) - f_col; }
  __device__ int col(long e) const { return col_of(col_word(e)); }
};

// Entries are read non-temporally where x does not stay in an L2 (4 MB) beside
// them otherwise: 1,000,003 rows of 16 FP64 46.3 -> 42.6 us, 3,000,003 FP32 110
// -> 98, 600,007 of 8 FP64 (4.8 MB of x) 16.5 -> 15.4; a smaller x stays, and
// then the caches' share of the entries counts: 800,003 of 16 FP32 (3.2 MB)
// 23.9 plain and 27.6 so, 300,007 of 31 FP64 (2.4 MB) 22.1 and 23.7.
inline bool stream_entries(long x_bytes) { return x_bytes > (7L << 19); }

template <typename VT>
inline CsrView<VT> csr_view(const DeviceMatrix &d) {
  const unsigned *col24 = (tile_pairs<VT>() ? d.col24_pairs : d.col24).template as<unsigned>();
  return CsrView<VT>{d.rowptr.as<int>(), d.colidx.as<int>(), d.vals.as<VT>(), d.tiles.as<int>(),
                     d.long_rows.as<int>(), d.entries, d.rp0, d.f_col, col24,
                     stream_entries(d.x_need * Val<VT>::kXBytes)};
}

// A row's sum reads its products from LDS kSumRun at a time, all reads issued
// before the adds; the slack slots after the tile keep those reads in bounds
// (their contents are never added).
constexpr int kSumRun = 16;
// A row of more products than this goes on, from a multiple of kSumRun, in whole
// runs: their slots are consecutive and every product is added, where a run from
// anywhere takes an address and a select each (a row of 1500 among 20,000 of 8:
// 35.7 -> 14.4 us in FP64, 23.9 -> 11.4 in FP32; 30,000 of 200 FP64 21.0 -> 15.8).
// From 16 on, the steps to the multiple cost what they save: 20,000 of 24 4.2 us
// and 4.65 so, 50,000 of 100 13.6 and 13.1.
constexpr int kLongSum = 64;

// Entries past the tile's end that are staged after the tile's, one a thread,
// for the tile's last row where it goes on: loaded beside the tile's own, where
// one thread fetching them after the barrier was a chain of memory round trips
// in every tile (50,000 rows of 100 FP64 35.9 -> 13.4 us, 200,001 of 37 27.1 ->
// 18.0, 300,007 of 12 13.0 -> 11.8, 62 million entries 146.2 -> 144.8).
constexpr int kTileTail = kTileThreads;

// TN: entries per tile of the caller's table.
// Product i of the tile is at slot(i): a free slot after every 16, so that the
// threads of a wavefront, each reading its own row, meet in few LDS banks (rows
// of 16 doubles start in two of the 64 without it): 500,009 rows of 16 FP64
// 27.0 -> 25.1 us, 1,000,003 52.2 -> 49.8 and FP32 32.4 -> 31.2.  FP32 in the
// largest tiles, which stream from HBM, stays packed (62 million entries 100.8
// us, 101.6 spread; FP64 146.2 and 146.0).
// TAIL: kTileTail, or 0 where the staging does not pay: a persistent kernel's
// registers (batch_step: 20.3 -> 21.9 ms for the mixed-size batch with it); one
// thread then finishes the last row.
template <typename AT, int TN, int TAIL = kTileTail>
struct CsrTileLds {
  static constexpr bool kSpread = sizeof(AT) == 8 || TN < kCsrTileNnz;
  __device__ static constexpr int slot(int i) { return kSpread ? i + (i >> 4) : i; }
  static constexpr int kEnd = TN + TAIL + kSumRun;
  AT prod[kEnd + (kSpread ? kEnd / 16 : 0)];
};

// Value source: stored values (VT) or value-free (every product is z[c]).
// load4 reads the four values of a group (issued before the gathers that need
// the column indices), apply4 gathers x and forms the rounded products.
template <typename VT, typename XT>
struct Prod {
  using AT = typename Val<VT>::A;
  template <bool NT>
  __device__ static void load4(const CsrView<VT> &m, long e, AT (&v)[4]) {
    if constexpr (tile_pairs<VT>())
      Val<VT>::template get22<NT>(m.vals, e, e + 128, v);
    else
      Val<VT>::template get4<NT>(m.vals, e, v);
  }
  __device__ static void apply4(const AT (&v)[4], const XT *__restrict__ x, const int (&c)[4], AT (&p)[4]) {
#pragma unroll
    for (int q = 0; q < 4; q++) p[q] = v[q] * static_cast<AT>(x[c[q]]);
  }
  __device__ static AT load1(const CsrView<VT> &m, long e) { return Val<VT>::get(m.vals, e); }
  __device__ static AT apply1(AT v, const XT *__restrict__ x, int c) { return v * static_cast<AT>(x[c]); }
  __device__ static AT one(const CsrView<VT> &m, const XT *__restrict__ x, long e) {
    const AT v = load1(m, e);
    return apply1(v, x, m.col(e));
  }
};
struct Pattern {};
template <>
struct Val<Pattern> {
  using A = double;
  static constexpr int kXBytes = 8;
};
template <typename XT>
struct Prod<Pattern, XT> {
  using AT = double;
  template <bool NT>
  __device__ static void load4(const CsrView<Pattern> &, long, double (&)[4]) {}
  __device__ static void apply4(const double (&)[4], const XT *__restrict__ z, const int (&c)[4], double (&p)[4]) {
#pragma unroll
    for (int q = 0; q < 4; q++) p[q] = static_cast<double>(z[c[q]]);
  }
  __device__ static double load1(const CsrView<Pattern> &, long) { return 1.0; }
  __device__ static double apply1(double, const XT *__restrict__ z, int c) { return static_cast<double>(z[c]); }
  __device__ static double one(const CsrView<Pattern> &m, const XT *__restrict__ z, long e) {
    return static_cast<double>(z[m.col(e)]);
  }
};

// A row sum starts from epi.init<AT>(row) when the epilogue has one (an
// accumulating product, y[row] += ...), else from 0.
template <typename AT, typename E>
__device__ inline auto epi_init(const E &e, int r, int) -> decltype(e.template init<AT>(r)) {
  return e.template init<AT>(r);
}
template <typename AT, typename E>
__device__ inline AT epi_init(const E &, int, long) {
  return AT(0);
}

// The entries [e0, e0 + ne) of one tile held by the calling thread, in groups
// of four (at(k, q): place of group k's entry q in the tile).  load() issues
// the index and value loads; products() gathers x and forms the rounded
// products, store() writes them to the slots of prod.  FULL (ne == TN, every
// tile but the matrix's last) reads with no per-entry guard; otherwise entries
// at or past ne are not read (a caller's value array holds exactly nnz values).
template <bool FULL, bool PACK, bool NT, typename VT, typename XT, int TN>
struct TileEntries {
  using AT = typename Val<VT>::A;
  static constexpr int G = TN / 4 / kTileThreads;  // 4-entry groups per thread
  static constexpr bool PAIRS = tile_pairs<VT>();
  v4i raw[G];  // the groups' columns as loaded: four ints, or three words of packed ones
  AT v[G][4];

  __device__ static int at(int k, int q) {
    const int t = static_cast<int>(threadIdx.x);
    return PAIRS ? 4 * (k * kTileThreads + (t & ~63)) + 2 * (t & 63) + (q >> 1) * 128 + (q & 1)
                 : 4 * (k * kTileThreads + t) + q;
  }

  __device__ void load(const CsrView<VT> &m, long e0, int ne) {
    typedef unsigned v3u __attribute__((ext_vector_type(3), aligned(4)));
    typedef int v2i __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int k = 0; k < G; k++) {
      if (FULL || at(k, 0) < ne) {
        if constexpr (PACK) {
          const int g = k * kTileThreads + threadIdx.x;
          const v3u w = vec_load<NT>(reinterpret_cast<const v3u *>(m.col24 + (e0 / 4 + g) * 3));
          raw[k].x = static_cast<int>(w.x);
          raw[k].y = static_cast<int>(w.y);
          raw[k].z = static_cast<int>(w.z);
        } else if constexpr (PAIRS) {
          const v2i c01 = vec_load<NT>(reinterpret_cast<const v2i *>(m.colidx + e0 + at(k, 0)));
          raw[k].x = c01.x;
          raw[k].y = c01.y;
          if (FULL || at(k, 2) < ne) {
            const v2i c23 = vec_load<NT>(reinterpret_cast<const v2i *>(m.colidx + e0 + at(k, 2)));
            raw[k].z = c23.x;
            raw[k].w = c23.y;
          }
        } else {
          raw[k] = vec_load<NT>(reinterpret_cast<const v4i *>(m.colidx + e0 + at(k, 0)));
        }
      }
    }
    // (after every group's columns: the gathers wait for those alone)
#pragma unroll
    for (int k = 0; k < G; k++)
      if (FULL || at(k, 3) < ne) Prod<VT, XT>::template load4<NT>(m, e0 + at(k, 0), v[k]);
  }

  __device__ void columns(const CsrView<VT> &m, int ne, int (&c)[G][4]) const {
#pragma unroll
    for (int k = 0; k < G; k++) {
      if constexpr (PACK) {
        const unsigned a = static_cast<unsigned>(raw[k].x), b = static_cast<unsigned>(raw[k].y),
                       d = static_cast<unsigned>(raw[k].z);
        c[k][0] = static_cast<int>(a & 0xFFFFFFu);
        c[k][1] = static_cast<int>(a >> 24 | (b & 0xFFFFu) << 8);
        c[k][2] = static_cast<int>(b >> 16 | (d & 0xFFu) << 16);
        c[k][3] = static_cast<int>(d >> 8);
      } else {
        c[k][0] = raw[k].x - m.f_col;
        c[k][1] = raw[k].y - m.f_col;
        c[k][2] = raw[k].z - m.f_col;
        c[k][3] = raw[k].w - m.f_col;
      }
      if (!FULL)  // entries past the matrix end: column 0
        for (int q = 0; q < 4; q++)
          if (at(k, q) >= ne) c[k][q] = 0;
    }
  }

  // gathers and rounded products into p
  __device__ void products(const CsrView<VT> &m, const XT *__restrict__ x, long e0, int ne, AT (&p)[G][4]) const {
#pragma clang fp contract(off)
    int c[G][4];
    columns(m, ne, c);
#pragma unroll
    for (int k = 0; k < G; k++) {
      if (FULL || at(k, 3) < ne)
        Prod<VT, XT>::apply4(v[k], x, c[k], p[k]);
      else  // the matrix's last entries: no value read past nnz
#pragma unroll
        for (int q = 0; q < 4; q++) p[k][q] = at(k, q) < ne ? Prod<VT, XT>::one(m, x, e0 + at(k, q)) : AT(0);
    }
  }

  static __device__ void store(const AT (&p)[G][4], AT *prod, int ne) {
#pragma unroll
    for (int k = 0; k < G; k++) {
#pragma unroll
      for (int q = 0; q < 4; q += 2) {  // (entries q and q + 1 are neighbours, in one run of 16)
        AT *o = prod + CsrTileLds<AT, TN>::slot(at(k, q));
        if (FULL || at(k, q) < ne) o[0] = p[k][q];
        if (FULL || at(k, q + 1) < ne) o[1] = p[k][q + 1];
      }
    }
  }
};

// Work of the caller's own that a tile does beside its loads: issue() (loads)
// after the tile's index and value loads, finish() after its products, before
// the barrier that precedes the row sums.
struct NoPre {
  __device__ void issue() {}
  __device__ void finish() {}
};

// The bounds of the thread's first owned row, then the index/value loads,
// gathers and products into prod.  (Issuing the row table first measured
// faster than deferring it behind the tile loads.)
template <bool FULL, bool PACK, bool NT, int TAIL, typename VT, typename XT, int TN, typename Pre>
__device__ inline void csr_tile_stage(const CsrView<VT> &m, const XT *__restrict__ x, typename Val<VT>::A *prod,
                                      long e0, int ne, int rlo, int rhi, int &a, int &b, int &last, Pre &pre) {
  // loaded with no branch so they stay in flight under the tile loads
  // (indices clamped to rhi <= rows: in bounds, and exact for every thread
  // that owns a row)
  a = m.rowptr[min(rlo + static_cast<int>(threadIdx.x), rhi)] - m.rp0;
  b = m.rowptr[min(rlo + static_cast<int>(threadIdx.x) + 1, rhi)] - m.rp0;
  using AT = typename Val<VT>::A;
  TileEntries<FULL, PACK, NT, VT, XT, TN> t;
  t.load(m, e0, ne);
  last = TAIL > 0 && FULL && rlo < rhi ? m.rowptr[rhi] - m.rp0 : 0;
  const int tail = min(max(last - static_cast<int>(e0) - ne, 0), TAIL);
  unsigned tc = 0;
  AT tv = 0;
  if (static_cast<int>(threadIdx.x) < tail) {
    tc = m.col_word(e0 + ne + threadIdx.x);
    tv = Prod<VT, XT>::load1(m, e0 + ne + threadIdx.x);
  }
  pre.issue();
  AT p[TileEntries<FULL, PACK, NT, VT, XT, TN>::G][4];
  t.products(m, x, e0, ne, p);
  AT tp = 0;
  if (static_cast<int>(threadIdx.x) < tail) tp = Prod<VT, XT>::apply1(tv, x, m.col_of(tc));
  pre.finish();
  TileEntries<FULL, PACK, NT, VT, XT, TN>::store(p, prod, ne);
  if (static_cast<int>(threadIdx.x) < tail) prod[CsrTileLds<AT, TN>::slot(ne + static_cast<int>(threadIdx.x))] = tp;
}

// s + the products [e, end) of the tile, in order.
template <typename AT, int TN, int TAIL>
__device__ inline AT sum_staged(const CsrTileLds<AT, TN, TAIL> &lds, int e, int end, AT s) {
#pragma clang fp contract(off)
  if (end - e > kLongSum) {
    for (; e & (kSumRun - 1); e++) s = s + lds.prod[lds.slot(e)];
    for (; e + kSumRun <= end; e += kSumRun) {
      const AT *p = lds.prod + lds.slot(e);
      AT v[kSumRun];
#pragma unroll
      for (int u = 0; u < kSumRun; u++) v[u] = p[u];
#pragma unroll
      for (int u = 0; u < kSumRun; u++) s = s + v[u];
    }
  }
  for (; e < end; e += kSumRun) {
    AT v[kSumRun];
#pragma unroll
    for (int u = 0; u < kSumRun; u++) v[u] = lds.prod[lds.slot(e + u)];
#pragma unroll
    for (int u = 0; u < kSumRun; u++) s = e + u < end ? s + v[u] : s;
  }
  return s;
}

// Rows of entry tile `tile`; epi(row, sum) once per owned row by the thread
// that sums it, rows longer than LT left to csr_long_row.  The caller
// synchronises the block before reusing `lds`.
// LOADS: what is known of m where the kernel is compiled: nothing (kEither), or
// whether the columns are packed and the entries stream.
enum TileLoads { kEither = -1, kPlain = 0, kPacked = 1, kStream = 2, kPackedStream = 3 };
template <typename VT, typename XT, typename Epi, int TN, int LT, TileLoads LOADS = kEither, int TAIL = kTileTail,
          typename Pre = NoPre>
__device__ inline void csr_tile_rows_at(const CsrView<VT> &mat, const XT *__restrict__ x,
                                        CsrTileLds<typename Val<VT>::A, TN, TAIL> &lds, Epi &epi, int tile,
                                        Pre &&pre = Pre()) {
#pragma clang fp contract(off)
  CsrView<VT> m = mat;
  if (LOADS == kPlain || LOADS == kStream) m.col24 = nullptr;
  using AT = typename Val<VT>::A;
  const int tid = threadIdx.x;
  const long e0 = static_cast<long>(tile) * TN;
  const int ne = static_cast<int>(min(static_cast<long>(TN), m.nnz - e0));
  const int rlo = m.tile_row[tile], rhi = m.tile_row[tile + 1];
  int a, b, last;  // last: end of the last owned row (0 in the matrix's last tile)
  const bool packed = LOADS == kEither ? m.col24 != nullptr : LOADS & 1;
  const bool stream = LOADS == kEither ? m.stream : LOADS & 2;
  const auto stage = [&](auto full, auto pack, auto nt) {
    csr_tile_stage<decltype(full)::value, decltype(pack)::value, decltype(nt)::value, TAIL, VT, XT, TN>(
        m, x, lds.prod, e0, ne, rlo, rhi, a, b, last, pre);
  };
  constexpr std::true_type yes{};
  constexpr std::false_type no{};
  if (ne == TN) {
    if (packed && stream)
      stage(yes, yes, yes);
    else if (packed)
      stage(yes, yes, no);
    else if (stream)
      stage(yes, no, yes);
    else
      stage(yes, no, no);
  } else {  // the matrix's last tile
    if (packed)
      stage(no, yes, no);
    else
      stage(no, no, no);
  }
  __syncthreads();
  const int t0 = static_cast<int>(e0);
  const int e1 = t0 + ne + min(max(last - t0 - ne, 0), TAIL);  // end of what is staged
  AT s = 0;
  int r = rlo + tid;
  for (; r < rhi; r += kTileThreads) {
    if (r != rlo + tid) {
      a = m.rowptr[r] - m.rp0;
      b = m.rowptr[r + 1] - m.rp0;
    }
    if (b - a > LT) continue;  // summed by csr_long_row
    s = epi_init<AT>(epi, r, 0);
    // a row owned by the tile starts in it and what is staged of it ends by
    // TN + kTileTail, so the reads below stay under slot(kEnd)
    s = sum_staged(lds, a - t0, min(b, e1) - t0, s);
    if (TAIL > 0 && b > e1) break;  // the last row, below
    // (no staging) the rest of the last row, same order, 8 loads in flight
    for (int e = e1; TAIL == 0 && e < b; e += 8) {
      AT q8[8];
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (e + u < b) q8[u] = Prod<VT, XT>::one(m, x, e + u);
#pragma unroll
      for (int u = 0; u < 8; u++)
        if (e + u < b) s += q8[u];
    }
    epi(r, s);
  }
  if (TAIL == 0 || last <= e1) return;
  // the last row runs past what is staged: the whole block stages the rest,
  // kTileThreads entries at a time, for the thread that sums it
  if (last - (m.rowptr[rhi - 1] - m.rp0) > LT) return;
  const bool mine = r == rhi - 1;
  for (int e = e1; e < last; e += kTileThreads) {
    const int n = min(last - e, kTileThreads);
    __syncthreads();
    if (tid < n) lds.prod[lds.slot(tid)] = Prod<VT, XT>::one(m, x, e + tid);
    __syncthreads();
    if (mine) s = sum_staged(lds, 0, n, s);
  }
  if (mine) epi(rhi - 1, s);
}

// Rows of entry tile blockIdx.x.
template <typename VT, typename XT, int TN, TileLoads LOADS = kEither, typename Epi, typename Pre = NoPre>
__device__ inline void csr_tile_rows(const CsrView<VT> &m, const XT *__restrict__ x,
                                     CsrTileLds<typename Val<VT>::A, TN> &lds, Epi &epi, Pre &&pre = Pre()) {
  csr_tile_rows_at<VT, XT, Epi, TN, kCsrLongRow, LOADS>(m, x, lds, epi, blockIdx.x, pre);
}

// One long row (m.long_rows[idx]) per workgroup: chunk products (LC
// entries per chunk), a fixed-order tree per chunk, chunk totals added in
// order.  epi by thread 0.  Bound by the latency of one workgroup's loads, so
// the columns are read from colidx: packed ones take more instructions to find
// and to part, and one row's bytes are few (a row of 20,000 among 20,000 of 8:
// 32.9 us packed, 28.9 so; among 1,000,003 157 and 146).
template <typename VT, typename XT, typename Epi, int TN, int LC, int TAIL>
__device__ inline void csr_long_row_at(const CsrView<VT> &mat, const XT *__restrict__ x,
                                       CsrTileLds<typename Val<VT>::A, TN, TAIL> &lds, Epi &epi, int idx) {
  using AT = typename Val<VT>::A;
  CsrView<VT> m = mat;
  m.col24 = nullptr;
  const int r = m.long_rows[idx];
  const long a = m.rowptr[r] - m.rp0, b = m.rowptr[r + 1] - m.rp0;
  AT total = 0;
  for (long base = a; base < b; base += LC) {
    const long cnt = min(static_cast<long>(LC), b - base);
    AT acc = 0;
    for (long e = threadIdx.x; e < cnt; e += kTileThreads) acc += Prod<VT, XT>::one(m, x, base + e);
    total += block_tree_sum<AT>(acc, lds.prod);
  }
  if (threadIdx.x == 0) epi(r, epi_init<AT>(epi, r, 0) + total);
}

template <typename VT, typename XT, int TN, typename Epi>
__device__ inline void csr_long_row(const CsrView<VT> &m, const XT *__restrict__ x,
                                    CsrTileLds<typename Val<VT>::A, TN> &lds, Epi &epi) {
  csr_long_row_at<VT, XT, Epi, TN, kCsrTileNnz, kTileTail>(m, x, lds, epi, blockIdx.x);
}

}  // namespace dev
}  // namespace hip
}  // namespace tbsla
