// PageRank iteration kernels and their host driver (see pagerank.hpp).
//
// One iteration of the CSR engine on the entry tiles is two launches on
// matrices of up to 2^20 entries (three with long rows):
//   pr_update_csr     first the step decision of the iteration before (every
//                     block merges that normalise pass's partials, at most
//                     256, and takes the same decision; block 0 stores it),
//                     then the entry-tile SpMV of the current iterate fused
//                     with b = beta*(A b_t) + tele and the block max of b,
//                     merged into 64 atomic-max slots.
//   pr_normalize      the max over the slots (every block), then b /= max, the
//                     L1 residual against b_t and the compensated sum of b,
//                     as per-block partials.
// The step decision updates the state: iteration count, convergence, the next
// teleport term, and (mixed precision) whether to move the anchor.  A launch
// of its own (pr_finalize_norm) takes it at the end of a launch batch, before
// the host reads the state, and in every iteration on larger matrices.
// Partial results cross workgroups only at kernel boundaries, so no kernel
// needs a device-wide fence.
// Every kernel returns at once when the state says the run has converged, so
// the host launches `check_every` iterations between two reads of the state.
#include <hip/hip_runtime.h>

#include <tbsla/cpp/MatrixCSR.hpp>

#include <chrono>
#include <cmath>
#include <mutex>
#include <stdexcept>
#include <string>
#include <vector>

#include "kernels.hpp"
#include "mirror.hpp"
#include <type_traits>

#include "pagerank.hpp"
#include "tile_csr.hpp"

namespace tbsla {
namespace hip {
namespace {

struct PrState {
  double beta, eps, bound_target, tele_scale;
  double tele;          // teleport term used by the next update
  double maxv;          // max of the last update
  double err;           // reference residual sum|b_k - b_{k-1}| of the last iteration
  double err_prev;      // ... and of the one before
  double sum, sum_prev; // sum of the last / previous normalised iterate (compensated)
  double bound, bound_prev, bound_anchor;
  double anchor_tau, floor_eps;
  // sum-normalised propagation-blocked runs: 1 / sum of the last iterate
  // (the next iterate's scale), and for mixed runs the sum of the anchor,
  // the teleport term and the scale of the iteration that moved it
  double inv_sum, sum_hat, t_anchor, c_anchor;
  // reference-rule runs with propagation-blocked products keep the update's
  // unnormalised b (raw = 1): the iterate is b * xscale, xscale = 1 / max of
  // the update that wrote it (1 for the start and in every other run)
  // xnext: that scale as the normalise pass leaves it for the next products,
  // before the step decision moves it to xscale
  double xscale, xnext;
  int it, max_it, done, rule;
  int need_anchor, anchors, anchor_it, mixed, raw;
};

constexpr int kNormBlocks = 1024;
// blocks of a normalise pass (1024 threads each): as many partials as the
// first wavefront of the next kernel merges in one step of four loads a lane
// (mixed runs, six streams instead of three: twice as many)
constexpr int kPassBlocks = 256;
constexpr int kMergeTileNnz = 1024;

// Neumaier-compensated running sum and its exact-error merge (TwoSum).
struct CSum {
  double s, c;
};
__device__ inline void csum_add(CSum &a, double v) {
  const double t = a.s + v;
  if (fabs(a.s) >= fabs(v))
    a.c += (a.s - t) + v;
  else
    a.c += (v - t) + a.s;
  a.s = t;
}
__device__ inline CSum csum_merge(CSum a, CSum b) {
  const double t = a.s + b.s;
  const double bp = t - a.s;
  const double e = (a.s - (t - bp)) + (b.s - bp);
  return CSum{t, a.c + b.c + e};
}

// Fixed-order butterfly reductions over one wavefront (every lane gets the
// result) and over the 16 wavefronts of a 1024-thread workgroup (thread 0
// gets the result; red holds 48 doubles).
// The partner of each step holds the other group's value: lanes 1 and 2 away
// (quad permutes), then the mirrored lane of 8 and of 16 (every lane of a
// group holds the group's value), which are VALU moves; the 16-lane rows are
// exchanged through LDS shuffles.  (Six LDS shuffles in a chain take three
// times as long.)
template <int CTRL>
__device__ inline double dpp_f64(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp(static_cast<int>(b), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp(static_cast<int>(b >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned>(lo));
}
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppHalfMirror = 0x141, kDppMirror = 0x140;
// f(partner) over the steps of a 16-lane row
template <typename T, typename Get, typename Op>
__device__ inline T row_reduce(T v, Get get, Op op) {
  v = op(v, get(std::integral_constant<int, kDppXor1>(), v));
  v = op(v, get(std::integral_constant<int, kDppXor2>(), v));
  v = op(v, get(std::integral_constant<int, kDppHalfMirror>(), v));
  v = op(v, get(std::integral_constant<int, kDppMirror>(), v));
  return v;
}
struct GetF64 {
  template <typename C>
  __device__ double operator()(C, double v) const {
    return dpp_f64<C::value>(v);
  }
};
struct GetCSum {
  template <typename C>
  __device__ CSum operator()(C, CSum v) const {
    return CSum{dpp_f64<C::value>(v.s), dpp_f64<C::value>(v.c)};
  }
};
struct AddF64 {
  __device__ double operator()(double a, double b) const { return a + b; }
};
struct MaxF64 {
  __device__ double operator()(double a, double b) const { return fmax(a, b); }
};
struct MergeCSum {
  __device__ CSum operator()(CSum a, CSum b) const { return csum_merge(a, b); }
};
__device__ inline CSum wave_csum(CSum v) {
  v = row_reduce(v, GetCSum(), MergeCSum());
#pragma unroll
  for (int off = 16; off <= 32; off <<= 1) v = csum_merge(v, CSum{__shfl_xor(v.s, off, 64), __shfl_xor(v.c, off, 64)});
  return v;
}
__device__ inline double wave_sum(double v) {
  v = row_reduce(v, GetF64(), AddF64());
  v += __shfl_xor(v, 16, 64);
  return v + __shfl_xor(v, 32, 64);
}
__device__ inline double wave_max(double v) {
  v = row_reduce(v, GetF64(), MaxF64());
  v = fmax(v, __shfl_xor(v, 16, 64));
  return fmax(v, __shfl_xor(v, 32, 64));
}
__device__ inline void block1024_err_csum(double err, CSum cs, double *red, double &err_out, CSum &cs_out) {
  err = wave_sum(err);
  cs = wave_csum(cs);
  const int w = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (lane == 0) {
    red[w] = err;
    red[16 + w] = cs.s;
    red[32 + w] = cs.c;
  }
  __syncthreads();
  if (w == 0) {  // the 16 wavefronts' sums on 16 lanes (each 16-lane group the same)
    err_out = red[lane & 15];
    cs_out = CSum{red[16 + (lane & 15)], red[32 + (lane & 15)]};
    err_out = row_reduce(err_out, GetF64(), AddF64());
    cs_out = row_reduce(cs_out, GetCSum(), MergeCSum());
  }
}

__device__ inline CSum block_csum(CSum v, double *ps, double *pc) {
  ps[threadIdx.x] = v.s;
  pc[threadIdx.x] = v.c;
  __syncthreads();
  for (int s = kTileThreads / 2; s > 0; s >>= 1) {
    if (static_cast<int>(threadIdx.x) < s) {
      CSum m = csum_merge(CSum{ps[threadIdx.x], pc[threadIdx.x]}, CSum{ps[threadIdx.x + s], pc[threadIdx.x + s]});
      ps[threadIdx.x] = m.s;
      pc[threadIdx.x] = m.c;
    }
    __syncthreads();
  }
  CSum r{ps[0], pc[0]};
  __syncthreads();
  return r;
}

// Teleport term of row i, by mode:
//   TM = 0  uniform: + tele on every row (tele = (1-beta)/n * sum b_t)
//   TM = 1  node set: + tele on listed rows (tele = (1-beta)/|nodes| * sum b_t)
//   TM = 2  distribution v: + tele * v[i] (tele = (1-beta) * sum b_t)
struct Teleport {
  const unsigned char *member;
  const double *v;
};
template <int TM>
__device__ inline double add_teleport(double bi, double tele, const Teleport &tp, long i) {
#pragma clang fp contract(off)
  if (TM == 0) return bi + tele;
  if (TM == 1) return tp.member[i] ? bi + tele : bi;
  return bi + tele * tp.v[i];
}

// What an update needs of the state, in LDS (written by the first wavefront
// before the products, read after the barrier that ends them).
struct StepIn {
  double beta, tele;
  int go;  // 0: the run had converged, nothing is written
};

// Per-row update epilogue: b = beta*(yhat + s) + teleport (MIXED) or beta*s + teleport.
template <typename AT, bool MIXED, int TM>
struct UpdateRow {
  double *b;
  const double *yhat;
  Teleport tp;
  const StepIn *in;
  double lmax;
  __device__ void operator()(int row, AT s) {
#pragma clang fp contract(off)
    if (!in->go) return;
    const double v = MIXED ? yhat[row] + static_cast<double>(s) : static_cast<double>(s);
    const double bi = add_teleport<TM>(in->beta * v, in->tele, tp, row);
    b[row] = bi;
    lmax = fmax(lmax, bi);
  }
};

// Block maxima are merged with integer atomicMax on 64 slots (a block uses
// slot blockIdx % 64), each slot holding an order-preserving encoding of a
// double (0 = empty), so the finalize reads 64 numbers however many blocks ran.
constexpr int kMaxSlots = 64;

__device__ inline unsigned long long ord_encode(double v) {
  const unsigned long long u = static_cast<unsigned long long>(__double_as_longlong(v));
  return (u >> 63) ? ~u : (u | 0x8000000000000000ull);
}
__device__ inline double ord_decode(unsigned long long u) {
  if (u == 0) return -INFINITY;
  return __longlong_as_double(static_cast<long long>((u >> 63) ? (u & 0x7fffffffffffffffull) : ~u));
}
__device__ inline void slot_max(unsigned long long *slots, double v, double *red) {
  const double bm = dev::block_tree_max<double>(v, red);
  if (threadIdx.x == 0) atomicMax(slots + (blockIdx.x % kMaxSlots), ord_encode(bm));
}

__device__ inline double step_bound(double err, double S, double sum_prev) {
  return err / S + fabs(sum_prev / S - 1.0);
}
__device__ inline bool step_converged(const PrState &st, double err, double bound) {
  return st.rule == 0 ? (err < st.eps) : (bound <= st.bound_target);
}

// The step decision from an iteration's residual and sum (one thread).
// MIXED = false leaves out what only mixed runs do.
template <bool MIXED = true>
__device__ inline void finalize_step(PrState *st, double err, double S) {
  // (mixed runs) this iteration moved the anchor: its step is the FP64
  // anchor product's, so its bound is free of the low-precision error
  const bool moved = MIXED && st->mixed && st->need_anchor;
  st->it += 1;
  st->err_prev = st->err;
  st->err = err;
  st->sum_prev = st->sum;
  st->sum = S;
  const double bound = step_bound(err, S, st->sum_prev);
  st->bound_prev = st->bound;
  st->bound = bound;
  bool converged = step_converged(*st, err, bound);
  int anchor = 0;
  if (MIXED && st->mixed) {
    // A low-precision phase converges to a point off the FP64 fixed point by
    // up to about floor_eps * (bound at its anchor) / (1 - rho)^2, rho the
    // phase's mean contraction per iteration.  When that may exceed the
    // target, convergence is only declared after an iteration that moved the
    // anchor (an FP64 step) meets the bound.
    if (converged && !moved) {
      const int k = st->it - st->anchor_it > 0 ? st->it - st->anchor_it : 1;
      double rho = 0.999;
      if (st->bound_anchor > 0.0 && bound > 0.0) rho = fmin(0.999, pow(bound / st->bound_anchor, 1.0 / k));
      const double floor = st->floor_eps * st->bound_anchor * 10.0 / ((1.0 - rho) * (1.0 - rho));
      if (floor > st->bound_target) {
        converged = false;
        anchor = 1;
      }
    }
    if (!converged) {
      if (bound <= st->anchor_tau * st->bound_anchor) anchor = 1;
      // progress has stopped (the phase reached its low-precision floor)
      if (st->it - st->anchor_it >= 3 && bound > 0.99 * st->bound_prev) anchor = 1;
    }
    if (anchor) {
      st->bound_anchor = bound;
      st->anchor_it = st->it;
      st->anchors += 1;
    }
  }
  st->need_anchor = anchor;
  st->done = (converged || st->it >= st->max_it) ? 1 : 0;
  st->tele = S * st->tele_scale;
  st->xscale = st->xnext;
}

// The partials of a normalise pass; n = 0: the state is up to date.
struct Partials {
  const double *perr, *ps, *pc;
  int n;
};

// The first wavefront of every block of an update: merges the partials of
// the iteration before (at most kPassBlocks, four a lane) and takes its step
// decision, the same in every block; block 0 stores the new state to `out`
// (a buffer of its own: other blocks still read `in`).  issue() loads,
// finish() decides; both are the Pre work of a tile, so the loads wait beside
// the tile's.
struct StepMerge {
  static constexpr int U = kPassBlocks / 64;
  const PrState *in;
  PrState *out;
  Partials pp;
  StepIn *sh;
  double pe[U], pv[U], pw[U];

  __device__ void issue() {
    if (threadIdx.x >= 64) return;
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = max(0, min(static_cast<int>(threadIdx.x) + 64 * u, pp.n - 1));
      pe[u] = pp.perr[i];
      pv[u] = pp.ps[i];
      pw[u] = pp.pc[i];
    }
  }
  __device__ void finish() {
    if (threadIdx.x >= 64) return;
    double e = 0, S = 0;
    if (pp.n > 0) {
      CSum t{0, 0};
#pragma unroll
      for (int u = 0; u < U; u++)
        if (static_cast<int>(threadIdx.x) + 64 * u < pp.n) {
          e += pe[u];
          t = csum_merge(t, CSum{pv[u], pw[u]});
        }
      e = wave_sum(e);
      t = wave_csum(t);
      S = t.s + t.c;
    }
    if (threadIdx.x != 0) return;
    if (blockIdx.x == 0) {
      *out = *in;
      if (pp.n > 0) finalize_step<false>(out, e, S);
    }
    // what finalize_step leaves in tele and done
    StepIn v{in->beta, in->tele, !in->done};
    if (pp.n > 0) {
      v.tele = S * in->tele_scale;
      v.go = !(step_converged(*in, e, step_bound(e, S, in->sum)) || in->it + 1 >= in->max_it);
    }
    *sh = v;
  }
};
// The state is up to date and only read.
struct StepRead {
  const PrState *in;
  StepIn *sh;
  __device__ void issue() {}
  __device__ void finish() {
    if (threadIdx.x == 0) *sh = StepIn{in->beta, in->tele, !in->done};
  }
};

// Fused update over the CSR tiles (LONG = false) or the long rows (LONG =
// true): b = beta * (A x) + tele, block max into the slots.  VT = dev::Pattern
// is the value-free product over z = colscale .* b_t.
// MERGE: the step decision of the iteration before is taken here (StepMerge).
template <typename VT, typename XT, bool MIXED, int TM, int TN, bool MERGE, bool LONG>
__global__ __launch_bounds__(kTileThreads) void pr_update_csr(dev::CsrView<VT> m, const XT *__restrict__ x,
                                                              const double *__restrict__ yhat, Teleport tp,
                                                              double *__restrict__ b, const PrState *st,
                                                              PrState *st_out, Partials pp,
                                                              unsigned long long *slots) {
  if (st->done) {
    if (MERGE && blockIdx.x == 0 && threadIdx.x == 0) *st_out = *st;
    return;
  }
  using AT = typename dev::Val<VT>::A;
  __shared__ dev::CsrTileLds<AT, TN> lds;
  __shared__ double red[kTileThreads];
  __shared__ StepIn in;
  UpdateRow<AT, MIXED, TM> epi{b, yhat, tp, &in, -INFINITY};
  if constexpr (LONG) {
    StepRead{st, &in}.finish();
    __syncthreads();
    dev::csr_long_row<VT, XT, TN>(m, x, lds, epi);
  } else if constexpr (MERGE) {
    StepMerge pre{st, st_out, pp, &in};
    dev::csr_tile_rows<VT, XT, TN>(m, x, lds, epi, pre);
  } else {
    dev::csr_tile_rows<VT, XT, TN>(m, x, lds, epi, StepRead{st, &in});
  }
  if (in.go) slot_max(slots, epi.lmax, red);
}

// Update for any format after a plain product y = A b_t (generic engine).
template <int TM>
__global__ __launch_bounds__(kTileThreads) void pr_update_vec(double *__restrict__ b, long n, Teleport tp,
                                                              const PrState *st, PrState *st_out, Partials pp,
                                                              unsigned long long *slots) {
#pragma clang fp contract(off)
  if (st->done) {
    if (blockIdx.x == 0 && threadIdx.x == 0) *st_out = *st;
    return;
  }
  __shared__ double red[kTileThreads];
  __shared__ StepIn in;
  StepMerge pre{st, st_out, pp, &in};
  pre.issue();
  pre.finish();
  __syncthreads();
  if (!in.go) return;
  const double beta = in.beta, tele = in.tele;
  double lmax = -INFINITY;
  for (long i = blockIdx.x * static_cast<long>(kTileThreads) + threadIdx.x; i < n;
       i += static_cast<long>(gridDim.x) * kTileThreads) {
    const double bi = add_teleport<TM>(beta * b[i], tele, tp, i);
    b[i] = bi;
    lmax = fmax(lmax, bi);
  }
  slot_max(slots, lmax, red);
}

// MODE 0: FP64, b normalised in place, previous iterate `prev`.
// MODE 4: MODE 0 with b and prev left unnormalised (raw runs): b * (1/max)
//         and prev * xscale are the iterates, nothing is written.
// MODE 1: mixed, previous iterate xhat + dold, writes dnew = b - xhat (FP32).
// MODE 2: FP64 + z = colscale .* b for the next value-free product.
// MODE 3: MODE 1 + zd = colscale .* (b - xhat) in FP32 (colscale32) for the
//         next value-free FP32 product.
//
// Every block takes the maximum of the update's slots (64 loads by its first
// wavefront); block 0 leaves it in the state and clears slots_next, the slots
// of the next update (the two sets alternate).
template <int MODE>
__global__ __launch_bounds__(1024) void pr_normalize(double *__restrict__ b, const double *__restrict__ prev,
                                                     const double *__restrict__ xhat, const float *__restrict__ dold,
                                                     float *__restrict__ dnew, double *__restrict__ z,
                                                     const double *__restrict__ colscale, float *__restrict__ zd,
                                                     const float *__restrict__ colscale32, long n, PrState *st,
                                                     const unsigned long long *slots, unsigned long long *slots_next,
                                                     double *__restrict__ perr, double *__restrict__ ps,
                                                     double *__restrict__ pc) {
#pragma clang fp contract(off)
  if (st->done) return;
  __shared__ double red[48];
  __shared__ double smax;
  const long stride = static_cast<long>(gridDim.x) * 1024;
  const long i_first = blockIdx.x * 1024L + threadIdx.x;
  // four elements of the thread's sequence per step, loads first; the first
  // step's are in flight beside the slots
  double bv[4], pv[4];
  const auto load4 = [&](long i0) {
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const long i = min(i0 + u * stride, n - 1);
      bv[u] = b[i];
      pv[u] = prev[i];
    }
  };
  if (MODE == 4 || MODE == 0) load4(i_first);
  if (threadIdx.x < 64) {
    unsigned long long u = __hip_atomic_load(slots + threadIdx.x, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
      const unsigned long long o = __shfl_xor(u, off, 64);
      u = o > u ? o : u;
    }
    if (threadIdx.x == 0) smax = ord_decode(u);
  }
  if (blockIdx.x == 0 && threadIdx.x >= 64 && threadIdx.x < 64 + kMaxSlots)
    __hip_atomic_store(slots_next + (threadIdx.x - 64), 0ull, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  const double pscale = st->xscale;  // (MODE 4)
  const bool moved = st->need_anchor != 0, raw = st->raw != 0;
  __syncthreads();
  const double m = smax, inv_m = 1.0 / m;
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    st->maxv = m;
    st->xnext = raw ? inv_m : 1.0;  // the scale of the b just written
  }
  double err = 0;
  CSum cs{0, 0};
  if (MODE == 4 || MODE == 0) {
    for (long i0 = i_first; i0 < n; i0 += 4 * stride) {
      if (i0 != i_first) load4(i0);
#pragma unroll
      for (int u = 0; u < 4; u++)
        if (i0 + u * stride < n) {
          const double bi = MODE == 4 ? bv[u] * inv_m : bv[u] / m;
          err += fabs(bi - (MODE == 4 ? pv[u] * pscale : pv[u]));
          csum_add(cs, bi);
          if (MODE == 0) b[i0 + u * stride] = bi;
        }
    }
  } else {
    for (long i = blockIdx.x * 1024L + threadIdx.x; i < n; i += stride) {
      const double bi = b[i] / m;
      const bool mixed = MODE == 1 || MODE == 3;
      // an iteration that moved the anchor starts from xhat itself (its delta
      // was folded into xhat and is not read)
      const double pi = mixed ? (moved ? xhat[i] : xhat[i] + static_cast<double>(dold[i])) : prev[i];
      err += fabs(bi - pi);
      csum_add(cs, bi);
      if (mixed) {
        const double dd = bi - xhat[i];
        dnew[i] = static_cast<float>(dd);
        if (MODE == 3) zd[i] = static_cast<float>(static_cast<double>(colscale32[i]) * dd);
      } else {
        b[i] = bi;
        z[i] = colscale[i] * bi;
      }
    }
  }
  double e;
  CSum t;
  block1024_err_csum(err, cs, red, e, t);
  if (threadIdx.x == 0) {
    perr[blockIdx.x] = e;
    ps[blockIdx.x] = t.s;
    pc[blockIdx.x] = t.c;
  }
}

// Sum of the per-block partials (err, compensated sum) over nb blocks by one
// block of T threads, in the fixed order thread t: t, t + T, ...
// The loads of 8 partials per thread are issued together (a loop that loads
// one partial per step waits for each load in turn).
template <int T = kTileThreads>
__device__ inline void sum_partials(const double *__restrict__ perr, const double *__restrict__ ps,
                                    const double *__restrict__ pc, int nb, double &e, CSum &t) {
  constexpr int U = 8;
  for (int i0 = threadIdx.x; i0 < nb; i0 += U * T) {
    double pe[U], pv[U], pw[U];
#pragma unroll
    for (int u = 0; u < U; u++) {
      const int i = min(i0 + u * T, nb - 1);
      pe[u] = perr ? perr[i] : 0.0;
      pv[u] = ps[i];
      pw[u] = pc[i];
    }
#pragma unroll
    for (int u = 0; u < U; u++)
      if (i0 + u * T < nb) {
        e += pe[u];
        t = csum_merge(t, CSum{pv[u], pw[u]});
      }
  }
}

// One block: residual and compensated sum of the normalise pass, then the
// step decision.
__global__ __launch_bounds__(kTileThreads) void pr_finalize_norm(const double *__restrict__ perr,
                                                                 const double *__restrict__ ps,
                                                                 const double *__restrict__ pc, int nb, PrState *st) {
  if (st->done) return;
  __shared__ double red_s[kTileThreads], red_c[kTileThreads];
  double e = 0;
  CSum t{0, 0};
  sum_partials(perr, ps, pc, nb, e, t);
  e = dev::block_tree_sum<double>(e, red_s);
  t = block_csum(t, red_s, red_c);
  if (threadIdx.x == 0) finalize_step(st, e, t.s + t.c);
}

// Mixed precision with tile products: move the anchor to the current iterate
// when requested, xhat += delta (and z = colscale .* xhat for the value-free
// anchor product).  The tile products still add the delta product in that
// iteration, so its input `clear` (the delta, or the scaled delta of
// PATTERN_F32) is zeroed; the normalise pass of that iteration starts from
// xhat.  (With propagation-blocked products the move is part of the scatter,
// and that iteration has no delta product.)
__global__ __launch_bounds__(256) void pr_anchor_move(double *__restrict__ xhat, const float *delta, float *clear,
                                                      double *__restrict__ z, const double *__restrict__ colscale,
                                                      long n, const PrState *st) {
  if (st->done || !st->need_anchor) return;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256) {
    const double v = xhat[i] + static_cast<double>(delta[i]);
    xhat[i] = v;
    if (clear) clear[i] = 0.0f;
    if (z) z[i] = colscale[i] * v;
  }
}

// A small graph's whole run in one workgroup and one launch (at most
// `iterations` of them, so that every launch ends): the iterate, the update
// and the row bounds stay in LDS, and the entries are read from L2, row by
// row, C per thread at a time.  The arithmetic is that of pr_update_csr and
// pr_normalize (row sums left to right, b = beta*s + tele, b / max).  VF: the
// entries of a column agree, so only the indices are read and the products
// are those of the column values (cs), formed once per column in LDS.
//
// Bound by the latency of a row's loads and by the cache lines one CU reads
// (a lane reads its own row); the two launches of an iteration took 11.5 us
// whatever the size.  Value-free, 8 entries a row, us an iteration: 100 nodes
// 11.6 -> 2.5, 1,000 12.2 -> 3.2, 2,500 12.1 -> 4.1, 5,003 12.5 -> 6.1; 4,000
// of 16 12.4 -> 8.1.  With stored values (three times the bytes, and most of
// each line another lane's) 2,500 of 8 took 6.2 and 5,003 9.5, 3,000 of 16
// 16.3: the lines kOneBlockEntries* draw.
// A long row is one thread's, a load of a chunk after the other, 0.2 us each:
// past kOneBlockChain of them (DeviceMatrix::one_block_chain) in a wavefront the
// tiles are sooner.  4,000 nodes of 4 (us an iteration, value-free, here and
// tiles): one row of 400 (53 loads) 13.7 and 14.8, 12 of 200 (52) 13.9 and 14.0,
// 40 of 100 (52) 16.4 and 13.3, one of 800 (103) 23.5 and 17.6, one of 1500 39.4
// and 24.0, 40 of 200 (100) 28.5 and 14.4; with stored values one of 400 15.6
// and 14.9, 12 of 400 (102) 37.2 and 17.1.
static_assert(kOneBlockRows * 28 <= 158 << 10, "28 bytes of LDS a row");
constexpr int kOneBlockChain = 64;
constexpr long kOneBlockEntries = 65536;       // value-free
constexpr long kOneBlockEntriesVal = 24576;    // with stored values
constexpr int kOneBlockLenBits = 11;
static_assert(kCsrLongRow < (1 << kOneBlockLenBits) && kOneBlockEntries < (1L << (31 - kOneBlockLenBits)),
              "a row's first entry and length fit one int");

typedef int v4i_u __attribute__((ext_vector_type(4), aligned(4)));
typedef double v2d_u __attribute__((ext_vector_type(2), aligned(8)));

// C entries from entry e (past the row's end they are the next row's, or the
// mirror's zeroed padding: loaded, never added).
template <bool VF, int C>
struct RowChunk {
  v4i_u c[C / 4];
  v2d_u v[VF ? 1 : C / 2];
  __device__ void load(const dev::CsrView<double> &m, int e) {
#pragma unroll
    for (int k = 0; k < C / 4; k++) c[k] = reinterpret_cast<const v4i_u *>(m.colidx + e)[k];
    if (!VF)
#pragma unroll
      for (int k = 0; k < C / 2; k++) v[k] = reinterpret_cast<const v2d_u *>(m.vals + e)[k];
  }
  // s plus the first `len` products, in entry order
  __device__ double add(double s, int len, const double *xs) const {
#pragma clang fp contract(off)
    double p[C];
#pragma unroll
    for (int k = 0; k < C / 4; k++) {
      p[4 * k] = xs[c[k].x];
      p[4 * k + 1] = xs[c[k].y];
      p[4 * k + 2] = xs[c[k].z];
      p[4 * k + 3] = xs[c[k].w];
      if (!VF) {
        p[4 * k] = v[2 * k].x * p[4 * k];
        p[4 * k + 1] = v[2 * k].y * p[4 * k + 1];
        p[4 * k + 2] = v[2 * k + 1].x * p[4 * k + 2];
        p[4 * k + 3] = v[2 * k + 1].y * p[4 * k + 3];
      }
    }
#pragma unroll
    for (int k = 0; k < C; k++) s = k < len ? s + p[k] : s;
    return s;
  }
};

template <int TM, bool VF, int C>
__global__ __launch_bounds__(1024) void pr_one_block(dev::CsrView<double> m, const double *__restrict__ colval, int n,
                                                     Teleport tp, double *__restrict__ x, double *__restrict__ out,
                                                     PrState *st, int iterations) {
#pragma clang fp contract(off)
  __shared__ double xs[kOneBlockRows], ys[kOneBlockRows], zbuf[VF ? kOneBlockRows : 1];
  __shared__ int bounds[kOneBlockRows];  // first entry << kOneBlockLenBits | length
  __shared__ double red[48];
  __shared__ PrState sh;
  double *const zs = VF ? zbuf : xs;  // the products' input
  constexpr int T = 1024, kLen = (1 << kOneBlockLenBits) - 1;
  const int tid = threadIdx.x;
  if (tid == 0) sh = *st;
  for (int r = tid; r < n; r += T) {
    const int a = m.rowptr[r] - m.rp0, b = m.rowptr[r + 1] - m.rp0;
    bounds[r] = a << kOneBlockLenBits | (b - a);
    const double v = x[r];
    xs[r] = v;
    if (VF) zs[r] = colval[r] * v;
  }
  __syncthreads();
  for (int it = 0; it < iterations && !sh.done; it++) {
    const double beta = sh.beta, tele = sh.tele;
    double lmax = -INFINITY;
    // the first chunk of the thread's next row is loaded while this one is summed
    RowChunk<VF, C> ck;
    int bd = tid < n ? bounds[tid] : 0;
    ck.load(m, bd >> kOneBlockLenBits);
#pragma unroll 1
    for (int r = tid; r < n; r += T) {
      const int bn = r + T < n ? bounds[r + T] : 0;
      RowChunk<VF, C> nx;
      nx.load(m, bn >> kOneBlockLenBits);
      const int a = bd >> kOneBlockLenBits, len = bd & kLen;
      double s = ck.add(0.0, len, zs);
      for (int k = C; k < len; k += C) {
        RowChunk<VF, C> c;
        c.load(m, a + k);
        s = c.add(s, len - k, zs);
      }
      const double b = add_teleport<TM>(beta * s, tele, tp, r);
      ys[r] = b;
      lmax = fmax(lmax, b);
      ck = nx;
      bd = bn;
    }
    lmax = wave_max(lmax);
    if ((tid & 63) == 0) red[tid >> 6] = lmax;
    __syncthreads();  // (every read of the old iterate by a row sum is done too)
    const double mx = row_reduce(red[tid & 15], GetF64(), MaxF64());
    double err = 0, e;
    CSum cs{0, 0}, t;
    for (int r = tid; r < n; r += T) {
      const double b = ys[r] / mx;
      err += fabs(b - xs[r]);
      csum_add(cs, b);
      xs[r] = b;
      if (VF) zs[r] = colval[r] * b;
    }
    __syncthreads();  // (red is written again)
    block1024_err_csum(err, cs, red, e, t);
    if (tid == 0) {
      sh.maxv = mx;
      finalize_step<false>(&sh, e, t.s + t.c);
    }
    __syncthreads();
  }
  const double S = sh.sum;
  for (int r = tid; r < n; r += T) {
    x[r] = xs[r];
    if (sh.done) out[r] = xs[r] / S;
  }
  if (tid == 0) *st = sh;
}

template <int TM>
void launch_one_block(const DeviceMatrix &d, const double *colval, int n, const Teleport &tp, double *x, double *out,
                      PrState *st, int iterations, hipStream_t s) {
  const dev::CsrView<double> m = dev::csr_view<double>(d);
  const auto kernel = !colval ? pr_one_block<TM, false, 8>
                      : d.entries > 10L * n ? pr_one_block<TM, true, 16>
                                            : pr_one_block<TM, true, 8>;
  hipLaunchKernelGGL(kernel, dim3(1), dim3(1024), 0, s, m, colval, n, tp, x, out, st, iterations);
}

template <typename YT>
struct StoreRowD {
  YT *y;
  template <typename AT>
  __device__ void operator()(int row, AT s) {
    y[row] = static_cast<YT>(s);
  }
};

// Mixed precision: the FP64 anchor product yhat = A64 xhat (VT = double) or
// its value-free form over z = colscale .* xhat (VT = dev::Pattern).
template <typename VT, int TN, bool LONG>
__global__ __launch_bounds__(kTileThreads) void pr_anchor_spmv(dev::CsrView<VT> m, const double *__restrict__ x,
                                                               double *__restrict__ yhat, const PrState *st) {
  if (st->done || !st->need_anchor) return;
  __shared__ dev::CsrTileLds<double, TN> lds;
  StoreRowD<double> epi{yhat};
  if constexpr (LONG)
    dev::csr_long_row<VT, double, TN>(m, x, lds, epi);
  else
    dev::csr_tile_rows<VT, double, TN>(m, x, lds, epi);
}

// Mixed runs on the tile products, once per run: the state's sum becomes the
// compensated sum of the anchor plus the FP32 delta, from one partial per block
// (2^24 nodes: 3.8 ms in one workgroup, 39 us so).
__global__ __launch_bounds__(1024) void pr_sum_rounded(const double *__restrict__ a, const float *__restrict__ d,
                                                       long n, double *__restrict__ ps, double *__restrict__ pc) {
#pragma clang fp contract(off)
  __shared__ double red[48];
  const long stride = static_cast<long>(gridDim.x) * 1024;
  CSum cs{0, 0}, t;
  for (long i0 = blockIdx.x * 1024L + threadIdx.x; i0 < n; i0 += 8 * stride) {
    double v[8];
#pragma unroll
    for (int u = 0; u < 8; u++) {
      const long i = min(i0 + u * stride, n - 1);
      v[u] = a[i] + static_cast<double>(d[i]);
    }
#pragma unroll
    for (int u = 0; u < 8; u++)
      if (i0 + u * stride < n) csum_add(cs, v[u]);
  }
  double unused;
  block1024_err_csum(0.0, cs, red, unused, t);
  if (threadIdx.x == 0) {
    ps[blockIdx.x] = t.s;
    pc[blockIdx.x] = t.c;
  }
}
__global__ __launch_bounds__(kTileThreads) void pr_sum_merge(const double *__restrict__ ps,
                                                             const double *__restrict__ pc, int nb, PrState *st) {
  __shared__ double red_s[kTileThreads], red_c[kTileThreads];
  double unused = 0;
  CSum t{0, 0};
  sum_partials(nullptr, ps, pc, nb, unused, t);
  t = block_csum(t, red_s, red_c);
  if (threadIdx.x == 0) st->sum = t.s + t.c;
}

// out = v / sum(v), v = (a (+ d)) * xscale (xscale is 1 except in raw runs):
// the state holds the compensated sum of the last iterate.
__global__ __launch_bounds__(256) void pr_scale_kernel(const double *__restrict__ a, const float *__restrict__ d,
                                                       long n, const PrState *st, double *__restrict__ out) {
#pragma clang fp contract(off)
  const double S = st->sum, sc = st->xscale;
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256)
    out[i] = ((d ? a[i] + static_cast<double>(d[i]) : a[i]) * sc) / S;
}

// cs[colidx[k] - f_col] = vals[k] over the stored entries: for a
// count-stochastic matrix every entry of a column holds the same value, so
// the order of the writes does not matter.
__global__ __launch_bounds__(256) void colscale_kernel(const int *__restrict__ colidx, const double *__restrict__ vals,
                                                       long nnz, int f_col, long n, double *__restrict__ cs) {
  for (long k = blockIdx.x * 256L + threadIdx.x; k < nnz; k += static_cast<long>(gridDim.x) * 256) {
    const long c = static_cast<long>(colidx[k]) - f_col;
    if (c >= 0 && c < n) cs[c] = vals[k];
  }
}
__global__ __launch_bounds__(256) void to_f32(const double *__restrict__ a, float *__restrict__ b, long n) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256)
    b[i] = static_cast<float>(a[i]);
}

__global__ __launch_bounds__(256) void fill_f64(double *y, long n, double v) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256) y[i] = v;
}
// Everything a run starts from: the state, the max slots (both sets) and the
// start vectors that are not nullptr.
struct PrInit {
  PrState h;
  PrState *st;
  unsigned long long *slots;
  long n;
  double *x;          // = x0
  double x0;
  double *xhat, *yhat, *z;  // = 0, 0, z_scale .* x0
  const double *z_scale;
  float *d, *w, *xhat32;    // = fl32(x0), 0, 0
  float *zd;                // = fl32(zd_scale32 .* fl32(x0)), or fl32(zd_scale64 * x0)
  const float *zd_scale32;
  const double *zd_scale64;
};
__global__ __launch_bounds__(256) void pr_init(PrInit a) {
  if (blockIdx.x == 0) {
    if (threadIdx.x == 0) *a.st = a.h;
    if (threadIdx.x < 2 * kMaxSlots) a.slots[threadIdx.x] = 0;
  }
  const float f0 = static_cast<float>(a.x0);
  for (long i = blockIdx.x * 256L + threadIdx.x; i < a.n; i += static_cast<long>(gridDim.x) * 256) {
    if (a.x) a.x[i] = a.x0;
    if (a.xhat) a.xhat[i] = 0.0;
    if (a.yhat) a.yhat[i] = 0.0;
    if (a.z) a.z[i] = a.z_scale[i] * a.x0;
    if (a.d) a.d[i] = f0;
    if (a.w) a.w[i] = 0.0f;
    if (a.xhat32) a.xhat32[i] = 0.0f;
    if (a.zd)
      a.zd[i] = a.zd_scale32 ? static_cast<float>(static_cast<double>(a.zd_scale32[i]) * static_cast<double>(f0))
                             : static_cast<float>(a.zd_scale64[i] * a.x0);
  }
}

unsigned grid_for(long n, long cap = kNormBlocks) {
  return static_cast<unsigned>(std::max<long>(1, std::min<long>(cap, (n + 255) / 256)));
}

// bad[0] = 1 unless every stored value of column j has the bits of cs[j]
// (colscale_kernel's: one of the column's stored values).
__global__ __launch_bounds__(256) void colscale_check(const int *__restrict__ colidx, const double *__restrict__ vals,
                                                      long nnz, int f_col, const double *__restrict__ cs,
                                                      int *__restrict__ bad) {
  if (*bad) return;  // (another block found one: nothing left to decide)
  for (long k = blockIdx.x * 256L + threadIdx.x; k < nnz; k += static_cast<long>(gridDim.x) * 256)
    if (__double_as_longlong(vals[k]) != __double_as_longlong(cs[static_cast<long>(colidx[k]) - f_col])) *bad = 1;
}
__global__ __launch_bounds__(256) void to_bf16_f32(const double *__restrict__ a, float *__restrict__ b, long n) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256)
    b[i] = dev::Val<dev::bf16>::cvt(dev::bf16_of(a[i]));
}

// The column values of an n-column CSR matrix into cs (0 for a column with no
// entries).  Returns whether the stored entries of every column hold one
// value: true of fill_cqmat_stochastic's by construction, found from the
// values otherwise (with `flag`, 8 bytes).  x_need <= n has been checked.
bool find_column_values(const cpp::Matrix &m, const DeviceMatrix &d64, long n, double *cs, double *flag,
                        hipStream_t s) {
  const unsigned ge = grid_for(d64.entries, 16L * kNormBlocks);
  hipLaunchKernelGGL(fill_f64, dim3(grid_for(n)), dim3(256), 0, s, cs, n, 0.0);
  if (d64.entries == 0) return true;
  hipLaunchKernelGGL(colscale_kernel, dim3(ge), dim3(256), 0, s, d64.colidx.as<int>(), d64.vals.as<double>(),
                     d64.entries, d64.f_col, n, cs);
  if (m.count_stochastic()) return true;
  int differs = 0;
  hipLaunchKernelGGL(fill_f64, dim3(1), dim3(256), 0, s, flag, 1L, 0.0);
  hipLaunchKernelGGL(colscale_check, dim3(ge), dim3(256), 0, s, d64.colidx.as<int>(), d64.vals.as<double>(),
                     d64.entries, d64.f_col, cs, reinterpret_cast<int *>(flag));
  TBSLA_HIP_CHECK(hipMemcpyAsync(&differs, flag, sizeof(int), hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  return !differs;
}

// find_column_values, decided once per matrix: if true, the column values are
// in the matrix's device cache in FP64, FP32 and as BF16 rounds them.
bool column_values(const cpp::Matrix &m, const DeviceMatrix &d64, long n, hipStream_t s) {
  DeviceCache &cache = m.device_cache();
  std::lock_guard<std::mutex> g(cache.mu);
  if (cache.col_values != DeviceCache::kUnknown) return cache.col_values == DeviceCache::kPerColumn;
  DevBuf c64, c32, cbf, flag;
  c64.reserve(sizeof(double) * static_cast<std::size_t>(n));
  flag.reserve(sizeof(double));
  const bool same = find_column_values(m, d64, n, c64.as<double>(), flag.as<double>(), s);
  if (same) {
    c32.reserve(sizeof(float) * static_cast<std::size_t>(n));
    cbf.reserve(sizeof(float) * static_cast<std::size_t>(n));
    hipLaunchKernelGGL(to_f32, dim3(grid_for(n)), dim3(256), 0, s, c64.as<double>(), c32.as<float>(), n);
    hipLaunchKernelGGL(to_bf16_f32, dim3(grid_for(n)), dim3(256), 0, s, c64.as<double>(), cbf.as<float>(), n);
  }
  TBSLA_HIP_CHECK(hipGetLastError());
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  if (same) {
    cache.colscale64 = std::move(c64);
    cache.colscale32 = std::move(c32);
    cache.colscale_bf16 = std::move(cbf);
  }
  cache.col_values = same ? DeviceCache::kPerColumn : DeviceCache::kDiffer;
  return same;
}

// ---------------------------------------------------------------------------
// Propagation-blocked product (layout in mirror.hpp, PbMatrix).
//   pb_scatter  one workgroup per column superblock (at most 8192 columns, in
//               the wide order 16384; fewer on small graphs, pb_width): the
//               superblock's slice of x is staged in LDS, then every far
//               product v * x[c] is written to its slot in the bin-grouped
//               product array; entries come in (bin, column) order, so
//               consecutive threads write runs of consecutive slots.
//   pb_gather   one 1024-thread workgroup per bin (at most 8192 rows): the bin's
//               far products and local products (x from the bin's own slice)
//               are added into LDS, then the row epilogue runs on the sums.
// The LDS additions are atomic, so the summation order within a row is not
// fixed (the result can differ in the last bits from run to run).
template <typename VT>
struct PbVal {
  template <typename AT>
  __device__ static AT prod(const VT *v, long k, AT x) {
    return static_cast<AT>(dev::Val<VT>::get(v, k)) * x;
  }
  // four values from a multiple of four
  template <typename AT>
  __device__ static void get4(const VT *v, long k, AT (&out)[4]) {
    typename dev::Val<VT>::A t[4];
    dev::Val<VT>::get4(v, k, t);
#pragma unroll
    for (int q = 0; q < 4; q++) out[q] = static_cast<AT>(t[q]);
  }
  template <typename AT>
  __device__ static AT mul(AT v, AT x) {
    return v * x;
  }
};
template <>
struct PbVal<dev::Pattern> {
  template <typename AT>
  __device__ static AT prod(const dev::Pattern *, long, AT x) {
    return x;
  }
  template <typename AT>
  __device__ static void get4(const dev::Pattern *, long, AT (&out)[4]) {
#pragma unroll
    for (int q = 0; q < 4; q++) out[q] = AT(1);
  }
  template <typename AT>
  __device__ static AT mul(AT, AT x) {
    return x;
  }
};

constexpr int kPbScatterThreads = 1024;

struct PbScatterArgs {
  const int *sp;              // far entries of superblock s: [sp[s], sp[s+1])
  const unsigned short *fkey; // column within the superblock | kPbRunStart
  const int *rp;              // runs of superblock s: [rp[s], rp[s+1])
  const int *rdelta;          // slot - entry of each run
  const int *cbase;           // run of the first entry of each 64-entry chunk
  const int *cp;              // chunks of superblock s: [cp[s], cp[s+1])
  int nsb, n;
  int cols;                   // columns per superblock
  long nfar;                  // product slots; kPbChunk spare slots follow them
};

// The anchor move of a mixed run, folded into the scatter of the iteration
// that makes it: over the superblock's columns c, xhat[c] += delta[c], and
// the product's input is colscale[c] * xhat[c] (value-free anchor product;
// the gather forms the same product for its local entries) or xhat[c] itself
// (colscale == nullptr), and xhat32[c] = fl32(xhat[c]).  Each superblock
// leaves the compensated sum of its new xhat in (psum, pcomp)[superblock].
struct AnchorMove {
  double *xhat;
  float *xhat32;  // fl32(xhat), for the scale term of the mixed iterations (or nullptr)
  const float *delta;
  // value-free anchor products: 1/count of each column (the product's input
  // is colscale .* xhat, formed where it is read), else nullptr
  const double *colscale;
  double *psum, *pcomp;
  int first;  // set on the device: the run's first move, whose anchor is still 0
};

// The far products of one superblock (picked from blockIdx): its slice of x
// staged in xs (LDS), then every far product v * x[c] written to its slot.
// With MOVE the slice is the anchor move's result instead of x.  COLS: the
// widest superblock of the layout `a` (kPbCols or kPbColsWide).  xcs (value-
// free FP64 products): the column values; the slice is xcs .* x.
template <typename VT, typename XT, typename AT, bool MOVE, int COLS, bool XCS = false>
__device__ inline void pb_scatter_sb(const PbScatterArgs &a, const VT *__restrict__ val, const XT *__restrict__ x,
                                     AT *__restrict__ prod, XT *xs, const AnchorMove &am, double *red,
                                     XT xsc = XT(1), const XT *__restrict__ xcs = nullptr) {
#pragma clang fp contract(off)
  // superblocks of one XCD (blockIdx % 8) are contiguous, so the runs that
  // share a cache line at a run boundary are written through the same L2
  // (the grid may be larger than the layout needs: the mixed kernel serves
  // two layouts)
  const int per = (a.nsb + 7) / 8;
  if (static_cast<int>(blockIdx.x) >= 8 * per) return;
  const int sb = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (sb >= a.nsb) return;
  const int k0 = a.sp[sb], k1 = a.sp[sb + 1];
  const int *__restrict__ delta = a.rdelta + a.rp[sb];  // slot - entry of each run of this superblock
  const int *__restrict__ cbase = a.cbase + a.cp[sb];   // run of the first entry of each chunk
  const long c0 = static_cast<long>(sb) * a.cols;
  const int nc = static_cast<int>(min(static_cast<long>(a.cols), static_cast<long>(a.n) - c0));
  {
    constexpr int S = COLS / kPbScatterThreads;  // x values per thread, all loads issued first
    XT t[S];
    CSum cs{0, 0};
#pragma unroll
    for (int u = 0; u < S; u++) {
      const int i = threadIdx.x + u * kPbScatterThreads;
      if (MOVE) {
        if (i < nc) {
          const long c = c0 + i;
          // (0 + d is d: the first move need not read the zero anchor)
          const double v = am.first ? static_cast<double>(am.delta[c]) : am.xhat[c] + static_cast<double>(am.delta[c]);
          am.xhat[c] = v;
          if (am.xhat32) am.xhat32[c] = static_cast<float>(v);
          csum_add(cs, v);
          t[u] = static_cast<XT>(am.colscale ? am.colscale[c] * v : v);
        } else {
          t[u] = XT(0);
        }
      } else {
        t[u] = i < nc ? static_cast<XT>(x[c0 + i] * xsc) : XT(0);
        if (XCS && i < nc) t[u] *= xcs[c0 + i];
      }
    }
#pragma unroll
    for (int u = 0; u < S; u++) xs[threadIdx.x + u * kPbScatterThreads] = t[u];
    if (MOVE) {
      double e_unused;
      CSum tot;
      block1024_err_csum(0.0, cs, red, e_unused, tot);
      if (threadIdx.x == 0) {
        am.psum[sb] = tot.s;
        am.pcomp[sb] = tot.c;
      }
    }
  }
  __syncthreads();
  // Each wavefront walks chunks wv + 16u + 16*UC*it (u < UC) of the
  // superblock, one entry per lane, as a software pipeline: the run of each
  // chunk's first entry (cbase) is loaded two iterations ahead; the keys,
  // the values and the slot offsets of the chunk's runs (rdelta[cb .. cb +
  // 63], one coalesced load, each lane's offset picked with a lane shuffle)
  // one iteration ahead, so no load of an iteration waits on another.  An
  // entry's run is the chunk's first run plus the run starts on lanes
  // 1..lane (a ballot).
  static_assert(kPbScatterThreads == 16 * kPbChunk && kPbChunk == 64, "16 wavefronts of 64-entry chunks");
  // chunks per wavefront per stage (two stages in flight fit 64 VGPRs)
  constexpr int UC = sizeof(AT) == 8 ? 2 : 4;
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int nent = k1 - k0, nck = (nent + kPbChunk - 1) / kPbChunk;
  const int nr = a.rp[sb + 1] - a.rp[sb];  // runs of this superblock
  const int nit = (nck + 16 * UC - 1) / (16 * UC);
  struct Stage {
    unsigned key[UC];
    AT v[UC];
    int dl[UC];
  };
  if (nent == 0) return;
  // Every load is unconditional (indices clamped into the superblock) and
  // every store too (lanes past the end write spare slots), so the loop is
  // straight-line code and each wait covers only the loads it needs; the
  // loop is unrolled twice with the two stages in fixed registers (no
  // register copies, which would wait for the loads in flight).  On the
  // 2^24-node graph this took the FP32 delta scatter from 193 to 177 us.
  auto load_cb = [&](int it, int (&cb)[UC]) {
#pragma unroll
    for (int u = 0; u < UC; u++) cb[u] = cbase[min(wv + 16 * u + 16 * UC * it, nck - 1)];
  };
  // (lanes past the end keep what they load: their run starts only count
  // for lanes past the end, and their products go to the spare slots)
  auto load_stage = [&](int it, const int (&cb)[UC], Stage &g) {
#pragma unroll
    for (int u = 0; u < UC; u++) {
      const int ec = k0 + min((wv + 16 * u + 16 * UC * it) * kPbChunk + lane, nent - 1);
      g.key[u] = a.fkey[ec];
      g.v[u] = PbVal<VT>::template prod<AT>(val, ec, AT(1));
      g.dl[u] = delta[min(cb[u] + lane, nr - 1)];
    }
  };
  auto store = [&](int it, const Stage &g) {
#pragma unroll
    for (int u = 0; u < UC; u++) {
      const int e = (wv + 16 * u + 16 * UC * it) * kPbChunk + lane;
      const unsigned long long starts = __ballot((g.key[u] & kPbRunStart) != 0u);
      // run starts on lanes 1..lane: those below this lane (mbcnt) plus its own
      const unsigned long long s1 = starts & ~1ull;
      const int below = static_cast<int>(__builtin_amdgcn_mbcnt_hi(
          static_cast<unsigned>(s1 >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(s1), 0u)));
      const int d = __shfl(g.dl[u], below + static_cast<int>((s1 >> lane) & 1ull), 64);
      // lanes past the end write a spare slot, so the store is unconditional
      const long o = e < nent ? static_cast<long>(k0 + e + d) : a.nfar + lane;
      prod[o] = g.v[u] * static_cast<AT>(xs[g.key[u] & (kPbRunStart - 1)]);
    }
  };
  // iteration it: the loads of stage it + 1 (its chunk runs were loaded in
  // iteration it - 1) and of the chunk runs of it + 2, then the stores of
  // stage it (loaded in iteration it - 1); chunks past the end load the
  // superblock's last entry and store to the spare slots
  int cb0[UC], cb1[UC];
  Stage s0, s1;
  load_cb(0, cb0);
  load_cb(1, cb1);
  __builtin_amdgcn_sched_barrier(0);  // (the loop's order: chunk runs, then a stage)
  load_stage(0, cb0, s0);
  // (both halves of an iteration use what they load: the compiler would
  // sink a load past a branch into the block that uses it)
  int it = 0;
  for (; it + 1 < nit; it += 2) {
    load_cb(it + 2, cb0);  // (first: the next half waits for it, not for the stage loads)
    load_stage(it + 1, cb1, s1);
    __builtin_amdgcn_sched_barrier(0);  // keep the loads ahead of the stores
    store(it, s0);
    load_cb(it + 3, cb1);
    load_stage(it + 2, cb0, s0);
    __builtin_amdgcn_sched_barrier(0);
    store(it + 1, s1);
  }
  if (it < nit) store(it, s0);
}

template <typename VT>
constexpr bool pb_value_free() {
  return std::is_same<VT, dev::Pattern>::value;
}

// FP64 runs: the far products of x (value-free: of cs .* x).  The last block
// takes the step decision of the iteration before from its partials instead
// (pp.n > 0): the products need only the iterate and, in raw runs, its scale
// xnext, so the decision costs no launch of its own.  The other blocks may
// read `done` before or after it is set; a scatter past convergence writes
// products that nothing reads.
template <typename VT, int COLS>
__global__ __launch_bounds__(kPbScatterThreads) void pb_scatter(PbScatterArgs a, const VT *__restrict__ val,
                                                                const double *__restrict__ cs,
                                                                const double *__restrict__ x,
                                                                double *__restrict__ prod, PrState *st, Partials pp) {
  if (st->done) return;
  __shared__ double xs[COLS];
  if (blockIdx.x == gridDim.x - 1) {
    if (pp.n > 0) {
      double e = 0, eb = 0;
      CSum t{0, 0}, tb{0, 0};
      sum_partials<kPbScatterThreads>(pp.perr, pp.ps, pp.pc, pp.n, e, t);
      block1024_err_csum(e, t, xs, eb, tb);
      if (threadIdx.x == 0) {
        finalize_step<false>(st, eb, tb.s + tb.c);
        st->inv_sum = 1.0 / (tb.s + tb.c);
      }
    }
    return;
  }
  // (raw reference-rule runs: x is the unnormalised b, the iterate x * xnext)
  pb_scatter_sb<VT, double, double, false, COLS, pb_value_free<VT>()>(a, val, x, prod, xs, AnchorMove{}, nullptr,
                                                                      st->xnext, cs);
}

// The value-free FP64 anchor product takes the wide scatter order (a 128 KB
// x slice, runs of about 32 products), as the value-free FP64 runs do; with
// FP64 values the narrow order was faster.
template <typename VA>
constexpr bool pb_anchor_wide() {
  return pb_value_free<VA>();
}

// Mixed runs, one launch per iteration: in an iteration that moves the
// anchor, the anchor move and the FP64 anchor product's far products (values
// VA, FP64, layout a: the wide order for value-free anchors, else the
// narrow one); otherwise the delta product's (values VD, delta XD, sums AD)
// over layout ad of superblocks up to DCOLS wide (kPbColsWide: the 4-byte x
// slice fills the LDS of a narrow FP64 slice).
template <typename VA, typename VD, typename XD, typename AD, int DCOLS>
__global__ __launch_bounds__(kPbScatterThreads) void pb_scatter_mx(PbScatterArgs a, PbScatterArgs ad,
                                                                   const VA *__restrict__ vala,
                                                                   const VD *__restrict__ vald,
                                                                   const XD *__restrict__ xd, void *prod,
                                                                   AnchorMove am, const PrState *st) {
  constexpr int ACOLS = pb_anchor_wide<VA>() ? kPbColsWide : kPbCols;
  static_assert(sizeof(XD) * DCOLS <= sizeof(double) * ACOLS, "the delta slice fits the LDS");
  if (st->done) return;
  __shared__ double xs[ACOLS];
  __shared__ double red[48];
  if (st->need_anchor) {
    AnchorMove m = am;
    m.first = st->anchors == 1;  // (the count includes the move this iteration makes)
    pb_scatter_sb<VA, double, double, true, ACOLS>(a, vala, nullptr, static_cast<double *>(prod), xs, m, red);
  } else {
    pb_scatter_sb<VD, XD, AD, false, DCOLS>(ad, vald, xd, static_cast<AD *>(prod), reinterpret_cast<XD *>(xs), am,
                                            nullptr);
  }
}

struct PbView {
  const int *bp, *lp;
  const unsigned short *frow, *lkey, *lbase;
  int n, rows;  // rows per bin
  long n_far;
};

// Far products are read non-temporally where they are past the L2s but partly
// in the 256 MB memory-side cache, whose lines the next scatter writes again
// (per iteration, graphs of 8 entries a row, half of them random: 3,000,003
// nodes FP64 82 -> 75 us, 5,000,011 150 -> 142.6 and FP32 112.3 -> 108.5,
// 8,000,009 241 -> 226).  Fewer are read sooner plain (2,000,003 nodes 51.3
// against 52.5; 3,000,003 in FP32, half the bytes, 58.1 and 59.3), more come
// from HBM either way (2^24 nodes 528 and 529).
template <typename AT>
__device__ inline bool pb_stream(long n_far) {
  return n_far > (sizeof(AT) == 8 ? 10L << 20 : 16L << 20) && n_far <= 48L << 20;
}

// Two products of type T in one vector load.
template <typename T>
struct PbPair;
template <>
struct PbPair<float> {
  typedef float type __attribute__((ext_vector_type(2)));
};
template <>
struct PbPair<double> {
  typedef double type __attribute__((ext_vector_type(2)));
};

// The row sums of one bin (blockIdx) into the FP64 LDS accumulator ybin
// (v.rows <= kPbRows entries): the bin's far products and its local products, x read
// from the bin's own slice, scaled by xsc (XCS: and by xcs[j], the column
// values of a value-free FP64 product, where they are read or once per column
// into zbin, in LDS).  Ends with a barrier.
//
// Local entries whose columns lie apart are bound by the lines that their loads
// touch, and two arrays are twice the lines, and more than an L1: 2^22 nodes of
// 12, columns within 4000 of the row's, 499 us an iteration with x and xcs read
// per entry, 316 with stored values, 114 staged; within 16000 (a quarter of the
// entries local) 351, 334 and 212.  zbin leaves a CU one workgroup instead of
// two, which far entries feel (2^24 nodes of 8, half of them far and the others
// beside each other: 530 us read, 541 staged; 40% far 489 and 483), and costs a
// pass over the slice (300,007 nodes of 12, 15% local: 24.5 and 25.4).  Hence
// PbMatrix::stage_local: scattered local entries are staged from a quarter of
// the far ones on, the others where they are 4/3 of them.
enum PbColumnValues { kNoColumnValues, kReadColumnValues, kStagedColumnValues };
template <typename VT, typename XT, typename AT, PbColumnValues XCS = kNoColumnValues>
__device__ inline void pb_accumulate(const PbView &v, const VT *__restrict__ lval, const XT *__restrict__ x,
                                     const AT *__restrict__ prod, double *ybin, XT xsc = XT(1),
                                     const double *__restrict__ xcs = nullptr, double *zbin = nullptr) {
#pragma clang fp contract(off)
  const int bin = blockIdx.x, tid = threadIdx.x;
  const int base = bin * v.rows;
  for (int i = tid; i < v.rows; i += 1024) ybin[i] = 0.0;
  if constexpr (XCS == kStagedColumnValues)
    for (int i = tid; i < min(v.rows, v.n - base); i += 1024) zbin[i] = xcs[base + i] * (x[base + i] * xsc);
  __syncthreads();
  const int f1 = v.bp[bin + 1], l1 = v.lp[bin + 1];
  // far products in pairs: one 4-byte load of two rows and one 8- or
  // 16-byte load of two products, four pairs per thread per round, 1024
  // pairs apart (an odd first or last entry of the bin's run goes alone).
  // Rounds with all four pairs in range run unmasked as a software
  // pipeline: the next round's loads are issued before this round's LDS
  // additions (the compiler does not move global loads across LDS atomics);
  // one masked round ends the run
  int f0 = v.bp[bin], fe = f1;
  if ((f0 & 1) && f0 < fe) {
    if (tid == 0) atomicAdd(&ybin[v.frow[f0]], static_cast<double>(prod[f0]));
    f0++;
  }
  if (((fe - f0) & 1) && fe > f0) {
    if (tid == 1023) atomicAdd(&ybin[v.frow[fe - 1]], static_cast<double>(prod[fe - 1]));
    fe--;
  }
  const auto far = [&](auto nt) {
    constexpr bool NT = decltype(nt)::value;
    using AT2 = typename PbPair<AT>::type;
    const unsigned *__restrict__ frow2 = reinterpret_cast<const unsigned *>(v.frow);
    const AT2 *__restrict__ prod2 = reinterpret_cast<const AT2 *>(prod);
    const int p1 = fe >> 1;
    constexpr int U = 4;
    int kp = (f0 >> 1) + tid;
    auto add = [&](unsigned rr, AT2 pp) {
      atomicAdd(&ybin[rr & 0xFFFFu], static_cast<double>(pp.x));
      atomicAdd(&ybin[rr >> 16], static_cast<double>(pp.y));
    };
    if (kp + (U - 1) * 1024 < p1) {
      unsigned rA[U];
      AT2 pA[U];
#pragma unroll
      for (int u = 0; u < U; u++) rA[u] = dev::vec_load<NT>(frow2 + kp + u * 1024), pA[u] = dev::vec_load<NT>(prod2 + kp + u * 1024);
      for (;;) {
        const int kn = kp + U * 1024;
        const bool more = kn + (U - 1) * 1024 < p1;
        unsigned rB[U];
        AT2 pB[U];
        if (more)
#pragma unroll
          for (int u = 0; u < U; u++)
            rB[u] = dev::vec_load<NT>(frow2 + kn + u * 1024), pB[u] = dev::vec_load<NT>(prod2 + kn + u * 1024);
#pragma unroll
        for (int u = 0; u < U; u++) add(rA[u], pA[u]);
        kp = kn;
        if (!more) break;
#pragma unroll
        for (int u = 0; u < U; u++) rA[u] = rB[u], pA[u] = pB[u];
      }
    }
    if (kp < p1) {
      unsigned r[U];
      AT2 pv[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const int kk = kp + u * 1024;
        r[u] = kk < p1 ? frow2[kk] : 0u;
        pv[u] = kk < p1 ? prod2[kk] : AT2{AT(0), AT(0)};
      }
#pragma unroll
      for (int u = 0; u < U; u++)
        if (kp + u * 1024 < p1) add(r[u], pv[u]);
    }
  };
  if (pb_stream<AT>(v.n_far))
    far(std::true_type{});
  else
    far(std::false_type{});
  // local entries: one group of four per thread (a 2-byte base row, one
  // 8-byte key load, aligned value loads), rows decoded from the keys; runs
  // of one row summed and added once
  constexpr int LU = 2;  // groups per thread in flight (4 measured slower)
  constexpr int kPad = -1;
  for (int k = v.lp[bin] + kPbLocalGroup * tid; k < l1; k += LU * kPbLocalGroup * 1024) {
    int r[LU][4], c[LU][4];
    AT lv[LU][4], xv[LU][4];
#pragma unroll
    for (int g = 0; g < LU; g++) {
      const int kg = k + g * kPbLocalGroup * 1024;
      if (g == 0 || kg < l1) {
        const int rb = v.lbase[kg / kPbLocalGroup];
        const dev::v4us kk = *reinterpret_cast<const dev::v4us *>(v.lkey + kg);
        PbVal<VT>::template get4<AT>(lval, kg, lv[g]);
        const unsigned key[4] = {kk.x, kk.y, kk.z, kk.w};
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const int dr = static_cast<int>(key[u] >> kPbShift);
          r[g][u] = dr == kPbLocalPad ? kPad : rb + dr;
          c[g][u] = static_cast<int>(key[u] & static_cast<unsigned>(kPbRows - 1));
        }
      } else {  // past the bin's run: a group of padding
#pragma unroll
        for (int u = 0; u < 4; u++) r[g][u] = kPad, c[g][u] = 0, lv[g][u] = AT(0);
      }
    }
#pragma unroll
    for (int g = 0; g < LU; g++)
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int j = base + c[g][u];
        if constexpr (XCS == kStagedColumnValues)
          xv[g][u] = zbin[c[g][u]];
        else if constexpr (XCS == kReadColumnValues)
          xv[g][u] = xcs[j] * (x[j] * xsc);
        else
          xv[g][u] = static_cast<AT>(x[j] * xsc);
      }
#pragma unroll
    for (int g = 0; g < LU; g++) {
      double acc = 0.0;
      int row = r[g][0];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        if (r[g][u] == kPad) break;  // padding closes a group
        if (r[g][u] != row) {
          atomicAdd(&ybin[row], acc);
          acc = 0.0;
          row = r[g][u];
        }
        acc += static_cast<double>(PbVal<VT>::template mul<AT>(lv[g][u], xv[g][u]));
      }
      if (row != kPad) atomicAdd(&ybin[row], acc);
    }
  }
  __syncthreads();
}

template <typename VT, bool STAGE>
constexpr PbColumnValues pb_columns() {
  return !pb_value_free<VT>() ? kNoColumnValues : STAGE ? kStagedColumnValues : kReadColumnValues;
}

// FP64 runs under the reference rule: b = beta*(A x) + t into out, block
// max into the slots (normalised by a separate pass).
template <typename VT, int TM, bool STAGE>
__global__ __launch_bounds__(1024) void pb_gather(PbView v, const VT *__restrict__ lval, const double *__restrict__ cs,
                                                  const double *__restrict__ x, const double *__restrict__ prod,
                                                  Teleport tp, double *__restrict__ out, PrState *st,
                                                  unsigned long long *slots) {
#pragma clang fp contract(off)
  if (st->done) return;
  __shared__ double ybin[kPbRows];
  __shared__ double red[16];
  __shared__ double zbin[STAGE ? kPbRows : 1];
  pb_accumulate<VT, double, double, pb_columns<VT, STAGE>()>(v, lval, x, prod, ybin, st->xnext, cs, zbin);
  const int bin = blockIdx.x, tid = threadIdx.x;
  const int base = bin * v.rows;
  const int rows = min(v.rows, v.n - base);
  double lmax = -INFINITY;
  const double beta = st->beta, tele = st->tele;
  for (int i = tid; i < rows; i += 1024) {
    const int r = base + i;
    const double bi = add_teleport<TM>(beta * ybin[i], tele, tp, r);
    out[r] = bi;
    lmax = fmax(lmax, bi);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) lmax = fmax(lmax, __shfl_xor(lmax, off, 64));
  if ((tid & 63) == 0) red[tid >> 6] = lmax;
  __syncthreads();
  if (tid == 0) {
    double m = red[0];
    for (int w = 1; w < 16; w++) m = fmax(m, red[w]);
    atomicMax(slots + (bin % kMaxSlots), ord_encode(m));
  }
}

// FP64 runs under the sum-normalised rule, update and normalisation in one
// pass: x' = (beta*(A x) + t) * inv_sum, where inv_sum = 1 / sum(x) (the
// sum-normalised iterate does not depend on the scale, so the scale of the
// last iterate serves), with sum|x' - x| and the compensated sum of x' as
// per-bin partials.
template <typename VT, int TM, bool STAGE>
__global__ __launch_bounds__(1024) void pb_gather_sn(PbView v, const VT *__restrict__ lval,
                                                     const double *__restrict__ colscale,
                                                     const double *__restrict__ x, const double *__restrict__ prod,
                                                     Teleport tp, double *__restrict__ xout, const PrState *st,
                                                     double *__restrict__ perr, double *__restrict__ ps,
                                                     double *__restrict__ pc) {
#pragma clang fp contract(off)
  if (st->done) return;
  __shared__ double ybin[kPbRows];
  __shared__ double red[48];
  __shared__ double zbin[STAGE ? kPbRows : 1];
  pb_accumulate<VT, double, double, pb_columns<VT, STAGE>()>(v, lval, x, prod, ybin, 1.0, colscale, zbin);
  const int bin = blockIdx.x, tid = threadIdx.x;
  const int base = bin * v.rows;
  const int rows = min(v.rows, v.n - base);
  const double beta = st->beta, tele = st->tele, inv = st->inv_sum;
  double err = 0.0;
  CSum cs{0, 0};
  for (int i = tid; i < rows; i += 1024) {
    const int r = base + i;
    const double xn = add_teleport<TM>(beta * ybin[i], tele, tp, r) * inv;
    xout[r] = xn;
    err += fabs(xn - x[r]);
    csum_add(cs, xn);
  }
  double e;
  CSum t;
  block1024_err_csum(err, cs, red, e, t);
  if (tid == 0) {
    perr[bin] = e;
    ps[bin] = t.s;
    pc[bin] = t.c;
  }
}

// Mixed runs (the partner of pb_scatter_mx).  The iterate is xhat + delta
// (FP64 anchor, FP32 delta) and is scaled by c = 1 / sum each iteration, as
// the FP64 runs are: x' = c*(beta*A x + t*e), e the teleport pattern.  The
// iteration that moves the anchor (xhat += delta, then delta = 0) sums the
// FP64 anchor product (values VA, input xhat; value-free anchors: acs .*
// xhat, acs = 1/count of each column, as the scatter forms it) and stores the
// anchor's scaled one-step change w = c_a*(beta*A xhat + t_a*e) - xhat in
// FP32 (c_a, t_a: that iteration's scale and teleport term); the next delta
// is d' = w.  The other iterations sum the delta product (values VD, input
// xd): with r = c / c_a,
//   d' = r*w + (r - 1)*xhat + c*(beta*(A_lo d) + (t - t_a)*e),
// which is x' - xhat.  w and r - 1 stay of the order of the iterate's
// change (the scale moves with the iterate's sum, which leaks at dangling
// columns), so the FP32 delta carries no part of the iterate itself.
// Writes d' (PAT32: also zd' = fl32(colscale32 * d')), with sum|d' - d| and
// the compensated sum of d' as per-bin partials.
template <typename VA, typename VD, typename XD, typename AD, int TM, bool PAT32>
__global__ __launch_bounds__(1024) void pb_gather_mx(PbView v, const VA *__restrict__ lvala,
                                                     const double *__restrict__ acs, const VD *__restrict__ lvald,
                                                     const XD *__restrict__ xd, const void *prod, Teleport tp,
                                                     const double *__restrict__ xhat,
                                                     const float *__restrict__ xhat32, float *__restrict__ w,
                                                     const float *__restrict__ dold, float *__restrict__ dnew,
                                                     float *__restrict__ zdnew, const float *__restrict__ colscale32,
                                                     const PrState *st, double *__restrict__ perr,
                                                     double *__restrict__ ps, double *__restrict__ pc) {
#pragma clang fp contract(off)
  if (st->done) return;
  __shared__ double ybin[kPbRows];
  __shared__ double red[48];
  const bool anchor = st->need_anchor != 0;
  if (anchor)
    pb_accumulate<VA, double, double, pb_columns<VA, false>()>(v, lvala, xhat, static_cast<const double *>(prod), ybin,
                                                              1.0, acs);
  else
    pb_accumulate<VD, XD, AD>(v, lvald, xd, static_cast<const AD *>(prod), ybin);
  const int bin = blockIdx.x, tid = threadIdx.x;
  const int base = bin * v.rows;
  const int rows = min(v.rows, v.n - base);
  const double beta = st->beta, c = st->inv_sum;
  // the anchor iteration's teleport term and scale (kept by the finalize
  // pass of that iteration for the phase)
  const double ta = anchor ? st->tele : st->t_anchor;
  const double r = anchor ? 1.0 : c / st->c_anchor, r1 = r - 1.0;
  const double dt = st->tele - ta;
  double err = 0.0;
  CSum cs{0, 0};
  for (int i = tid; i < rows; i += 1024) {
    const int row = base + i;
    float d32;
    if (anchor) {
      d32 = static_cast<float>(c * add_teleport<TM>(beta * ybin[i], ta, tp, row) - xhat[row]);
      w[row] = d32;
      err += fabs(static_cast<double>(d32));
    } else {
      // (r - 1) is of the order of the change of the leak since the anchor,
      // so the FP32 anchor copy carries this term to well below FP32 delta
      // precision
      d32 = static_cast<float>(r * static_cast<double>(w[row]) + r1 * static_cast<double>(xhat32[row]) +
                               c * add_teleport<TM>(beta * ybin[i], dt, tp, row));
      err += fabs(static_cast<double>(d32) - static_cast<double>(dold[row]));
    }
    dnew[row] = d32;
    if (PAT32) zdnew[row] = static_cast<float>(static_cast<double>(colscale32[row]) * static_cast<double>(d32));
    csum_add(cs, static_cast<double>(d32));
  }
  double e;
  CSum t;
  block1024_err_csum(err, cs, red, e, t);
  if (tid == 0) {
    perr[bin] = e;
    ps[bin] = t.s;
    pc[bin] = t.c;
  }
}

PbView pb_view(const PbMatrix &pb) {
  return PbView{pb.bp.as<int>(), pb.lp.as<int>(), pb.frow.as<unsigned short>(), pb.lkey.as<unsigned short>(),
                pb.lbase.as<unsigned short>(), pb.n, pb.rows, pb.n_far};
}

PbScatterArgs pb_args(const PbMatrix &pb) {
  return PbScatterArgs{pb.sp.as<int>(),    pb.fkey.as<unsigned short>(), pb.rp.as<int>(), pb.rdelta.as<int>(),
                       pb.cbase.as<int>(), pb.cp.as<int>(),              pb.nsb,          pb.n,
                       pb.cols,            pb.n_far};
}

// The scatter order of the delta products with values VD (the far values of
// dtype F32 are stored narrow, BF16 wide; the pb_mirror build follows this).
template <typename VD>
constexpr bool pb_delta_wide() {
  return !std::is_same<VD, float>::value;
}

PbScatterArgs pb_args_wide(const PbMatrix &pb) {
  if (pb.cols_w == pb.cols) return pb_args(pb);
  return PbScatterArgs{pb.sp_w.as<int>(),    pb.fkey_w.as<unsigned short>(), pb.rp_w.as<int>(), pb.rdelta_w.as<int>(),
                       pb.cbase_w.as<int>(), pb.cp_w.as<int>(),              pb.nsb_w,          pb.n,
                       pb.cols_w,            pb.n_far};
}

// The scatter order of value-free products.
PbScatterArgs pb_args_free(const PbMatrix &pb) { return pb.wide_free() ? pb_args_wide(pb) : pb_args(pb); }

dim3 pb_scatter_grid(int nsb) { return dim3((nsb + 7) / 8 * 8); }

// Dynamic LDS added to the scatter launches whose static LDS (a 64 KB x
// slice) would let two blocks share a CU: one scatter block per CU writes
// its products faster (2^24-node graph: FP64 scatter 345 -> 315 us, and the
// gather after it 374 -> 362 us; two blocks per CU for the mixed scatters:
// 199 -> 207 us).  The value-free FP64 scatter takes the wide order, whose
// 128 KB slice already holds a CU alone (234 -> 210 us; with values, FP64
// and FP32, the wide order measured slower).
constexpr unsigned kPbScatterLdsPad = 24 * 1024;

// The far products of one FP64 iteration (values VT): value-free ones (cs:
// the column values) over the wide order, the others over the narrow one.
template <typename VT>
void launch_pb_scatter(const PbMatrix &pb, const VT *fval, const double *cs, const double *x, double *prod,
                       PrState *st, const Partials &pp, hipStream_t s) {
  if constexpr (pb_value_free<VT>()) {
    const PbScatterArgs a = pb_args_free(pb);
    hipLaunchKernelGGL((pb_scatter<VT, kPbColsWide>), dim3(pb_scatter_grid(a.nsb).x + 1), dim3(kPbScatterThreads),
                       0, s, a, fval, cs, x, prod, st, pp);
  } else {
    hipLaunchKernelGGL((pb_scatter<VT, kPbCols>), dim3(pb_scatter_grid(pb.nsb).x + 1), dim3(kPbScatterThreads),
                       kPbScatterLdsPad, s, pb_args(pb), fval, cs, x, prod, st, pp);
  }
}

// The per-bin partials of a sum-normalised iteration.
struct SnPartials {
  double *perr, *ps, *pc;
};

// One FP64 iteration on the blocked products (values VT; dev::Pattern: value-
// free, cs the column values): scatter and gather, through the run's product
// slots prod.  sp == nullptr: the reference-rule update, block maxima into the
// slots; else the sum-normalised one with its partials.  pp: the partials of the iteration before, whose step
// decision the scatter takes (pp.n = 0: taken already).
template <typename VT, int TM>
void launch_pb_tm(const PbMatrix &pb, const double *cs, const double *x, double *prod, const Teleport &tp, double *out,
                  PrState *st, unsigned long long *slots, const SnPartials *sp, const Partials &pp, hipStream_t s) {
  constexpr int slot = static_cast<int>(Dtype::F64);
  const VT *fval = pb_value_free<VT>() ? nullptr : pb.fval[slot].as<VT>();
  const VT *lval = pb_value_free<VT>() ? nullptr : pb.lval[slot].as<VT>();
  launch_pb_scatter<VT>(pb, fval, cs, x, prod, st, pp, s);
  const auto gather = [&](auto stage) {
    constexpr bool STAGE = decltype(stage)::value;
    if (sp)
      hipLaunchKernelGGL((pb_gather_sn<VT, TM, STAGE>), dim3(pb.nbins), dim3(1024), 0, s, pb_view(pb), lval, cs, x,
                         prod, tp, out, st, sp->perr, sp->ps, sp->pc);
    else
      hipLaunchKernelGGL((pb_gather<VT, TM, STAGE>), dim3(pb.nbins), dim3(1024), 0, s, pb_view(pb), lval, cs, x, prod,
                         tp, out, st, slots);
  };
  if constexpr (pb_value_free<VT>()) {
    if (pb.stage_local()) return gather(std::true_type());
  }
  gather(std::false_type());
}

void launch_pb(int tmode, const PbMatrix &pb, const double *cs, const double *x, double *prod, const Teleport &tp,
               double *out, PrState *st, unsigned long long *slots, const SnPartials *sp, const Partials &pp,
               hipStream_t s) {
  const auto go = [&](auto tag) {
    using VT = decltype(tag);
    if (tmode == 1)
      launch_pb_tm<VT, 1>(pb, cs, x, prod, tp, out, st, slots, sp, pp, s);
    else if (tmode == 2)
      launch_pb_tm<VT, 2>(pb, cs, x, prod, tp, out, st, slots, sp, pp, s);
    else
      launch_pb_tm<VT, 0>(pb, cs, x, prod, tp, out, st, slots, sp, pp, s);
  };
  if (cs)
    go(dev::Pattern());
  else
    go(double());
}

// Buffers of a mixed sum-normalised iteration.
struct MxBufs {
  AnchorMove am;           // anchor xhat (and 1/count, value-free) with the scatter's sum partials
  const void *xd;          // the delta product's input: delta (F32/BF16) or zd (PATTERN_F32)
  void *prod;              // the run's product slots
  float *w;                // FP32 one-step change of the anchor
  const float *dold;       // delta of the current iterate
  float *dnew, *zdnew;     // delta (and zd) of the next
  const float *colscale32; // PATTERN_F32
};

// One mixed iteration: the anchor move and the FP64 anchor product (values
// VA at slot va, input z or xhat) when the state asks for it, else the delta
// product (values VD at slot vd); the finalize pass follows.
template <typename VA, typename VD, typename XD, int TM, bool PAT32>
void launch_pb_mx_tm(const PbMatrix &pb, int va, int vd, const MxBufs &b, const Teleport &tp, PrState *st,
                     const SnPartials &sp, hipStream_t s) {
  const VA *fa = va >= 0 ? pb.fval[va].as<VA>() : nullptr;
  const VA *la = va >= 0 ? pb.lval[va].as<VA>() : nullptr;
  const VD *fd = vd >= 0 ? pb.fval[vd].as<VD>() : nullptr;
  const VD *ld = vd >= 0 ? pb.lval[vd].as<VD>() : nullptr;
  const XD *xd = static_cast<const XD *>(b.xd);
  // the delta products of BF16-valued and value-free runs take the wide
  // scatter order, FP32-valued ones the narrow one (measured: value-free FP32
  // delta scatter 154 -> 140 us wide, BF16 196 -> 192, FP32 191 -> 196)
  constexpr bool wide = pb_delta_wide<VD>();
  // (a wide anchor's 128 KB slice leaves room for one block per CU without
  // the LDS pad)
  constexpr bool awide = pb_anchor_wide<VA>();
  const PbScatterArgs aa = awide ? pb_args_free(pb) : pb_args(pb);
  const PbScatterArgs ad = pb_value_free<VD>() ? pb_args_free(pb) : wide ? pb_args_wide(pb) : pb_args(pb);
  hipLaunchKernelGGL((pb_scatter_mx<VA, VD, XD, float, wide ? kPbColsWide : kPbCols>),
                     pb_scatter_grid(std::max(aa.nsb, ad.nsb)), dim3(kPbScatterThreads),
                     awide ? 0 : kPbScatterLdsPad, s, aa, ad, fa, fd, xd, b.prod, b.am, st);
  hipLaunchKernelGGL((pb_gather_mx<VA, VD, XD, float, TM, PAT32>), dim3(pb.nbins), dim3(1024), 0, s, pb_view(pb), la,
                     b.am.colscale, ld, xd, b.prod, tp, b.am.xhat, b.am.xhat32, b.w, b.dold, b.dnew, b.zdnew,
                     b.colscale32, st, sp.perr, sp.ps, sp.pc);
}

template <typename VA, typename VD, typename XD, bool PAT32>
void launch_pb_mx(int tmode, const PbMatrix &pb, int va, int vd, const MxBufs &b, const Teleport &tp, PrState *st,
                  const SnPartials &sp, hipStream_t s) {
  if (tmode == 1)
    launch_pb_mx_tm<VA, VD, XD, 1, PAT32>(pb, va, vd, b, tp, st, sp, s);
  else if (tmode == 2)
    launch_pb_mx_tm<VA, VD, XD, 2, PAT32>(pb, va, vd, b, tp, st, sp, s);
  else
    launch_pb_mx_tm<VA, VD, XD, 0, PAT32>(pb, va, vd, b, tp, st, sp, s);
}

// The state an update reads, where its block 0 leaves the state after the
// step decision it takes (nullptr: none to take), and the partials for it.
struct StepArgs {
  const PrState *in;
  PrState *out;
  Partials pp;
};

template <typename VT, typename XT, bool MIXED, int TM>
void launch_update(const DeviceMatrix &d, const VT *vals, const XT *x, const double *yhat, const Teleport &tp,
                   double *b, const StepArgs &a, unsigned long long *slots, hipStream_t s) {
  dev::CsrView<VT> m = dev::csr_view<VT>(d);
  if (vals) m.vals = vals;
  // (nnz / tile size + 1 tiles, so at least one block stores the state)
  if constexpr (!MIXED) {
    if (a.out)
      hipLaunchKernelGGL((pr_update_csr<VT, XT, MIXED, TM, kMergeTileNnz, true, false>), dim3(d.ntiles),
                         dim3(kTileThreads), 0, s, m, x, yhat, tp, b, a.in, a.out, a.pp, slots);
  }
  if (!a.out)
    with_tile_size(d, [&](auto tn) {
      hipLaunchKernelGGL((pr_update_csr<VT, XT, MIXED, TM, decltype(tn)::value, false, false>), dim3(d.ntiles),
                         dim3(kTileThreads), 0, s, m, x, yhat, tp, b, a.in, a.out, a.pp, slots);
    });
  if (d.nlong > 0)
    hipLaunchKernelGGL((pr_update_csr<VT, XT, MIXED, TM, kTileThreads, false, true>), dim3(d.nlong),
                       dim3(kTileThreads), 0, s, m, x, yhat, tp, b, a.out ? a.out : a.in,
                       static_cast<PrState *>(nullptr), Partials{}, slots);
}

// Values override `vals` (nullptr: the mirror's own values).
template <typename VT, typename XT, bool MIXED>
void launch_update(int tmode, const DeviceMatrix &d, const VT *vals, const XT *x, const double *yhat,
                   const Teleport &tp, double *b, const StepArgs &a, unsigned long long *slots, hipStream_t s) {
  if (tmode == 1)
    launch_update<VT, XT, MIXED, 1>(d, vals, x, yhat, tp, b, a, slots, s);
  else if (tmode == 2)
    launch_update<VT, XT, MIXED, 2>(d, vals, x, yhat, tp, b, a, slots, s);
  else
    launch_update<VT, XT, MIXED, 0>(d, vals, x, yhat, tp, b, a, slots, s);
}

template <typename VT>
void launch_anchor(const DeviceMatrix &d, const double *x, double *yhat, const PrState *st, hipStream_t s) {
  const dev::CsrView<VT> m = dev::csr_view<VT>(d);
  if (d.ntiles > 0)
    with_tile_size(d, [&](auto tn) {
      hipLaunchKernelGGL((pr_anchor_spmv<VT, decltype(tn)::value, false>), dim3(d.ntiles), dim3(kTileThreads), 0, s, m,
                         x, yhat, st);
    });
  if (d.nlong > 0)
    hipLaunchKernelGGL((pr_anchor_spmv<VT, kTileThreads, true>), dim3(d.nlong), dim3(kTileThreads), 0, s, m, x, yhat, st);
}

struct Scratch {
  WsBuf st, slots, perr, ps, pc, member, nodes, hsum, hcomp;
  WsBuf X0, X1, Z, yhat, xhat, xhat32, D0, D1, ZD0, ZD1, W, out, cs, flag, prod;
};

// One block: the step decision of a sum-normalised propagation-blocked
// iteration from the gather's per-bin partials (nb) and, after a mixed run's
// anchor move, the scatter's per-superblock sums of the new anchor (nsb).
// S is the sum of the new iterate: sum(x') (FP64 runs), sum(xhat) + sum(d')
// (mixed runs).  The iteration that moved the anchor starts from the
// rescaled anchor, whose sum replaces the previous one in the bound.
__global__ __launch_bounds__(kTileThreads) void pr_finalize_sn(const double *__restrict__ perr,
                                                               const double *__restrict__ ps,
                                                               const double *__restrict__ pc, int nb,
                                                               const double *__restrict__ hs,
                                                               const double *__restrict__ hc, int nsb, PrState *st) {
  if (st->done) return;
  __shared__ double red_s[kTileThreads], red_c[kTileThreads];
  double e = 0;
  CSum t{0, 0};
  sum_partials(perr, ps, pc, nb, e, t);
  e = dev::block_tree_sum<double>(e, red_s);
  t = block_csum(t, red_s, red_c);
  const bool moved = st->mixed && st->need_anchor;
  CSum h{0, 0};
  if (moved) {
    double unused = 0;
    sum_partials(nullptr, hs, hc, nsb, unused, h);
    h = block_csum(h, red_s, red_c);
  }
  if (threadIdx.x == 0) {
    double S = t.s + t.c;
    if (st->mixed) {
      if (moved) {
        st->sum_hat = h.s + h.c;
        st->sum = st->sum_hat;  // the iterate the step started from: the moved anchor
        st->t_anchor = st->tele;
        st->c_anchor = st->inv_sum;
      }
      S += st->sum_hat;
    }
    finalize_step(st, e, S);
    st->inv_sum = 1.0 / S;
  }
}

// member[i] = 1 for the listed nodes in [0, n) (member cleared first).
__global__ __launch_bounds__(256) void set_members(unsigned char *member, long n, const int *nodes, int n_nodes) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n_nodes; i += static_cast<long>(gridDim.x) * 256) {
    const int v = nodes[i];
    if (v >= 0 && v < n) member[v] = 1;
  }
}
__global__ __launch_bounds__(256) void fill_u8(unsigned char *y, long n, unsigned char v) {
  for (long i = blockIdx.x * 256L + threadIdx.x; i < n; i += static_cast<long>(gridDim.x) * 256) y[i] = v;
}

}  // namespace

// Iterations to launch before the next state read: the iterations the last
// two residuals predict are left (geometric decay of the quantity the rule
// tests), at least 1 and at most `check`.  Kernels launched past convergence
// return at once, so this only trims those launches.
int next_batch(const PrState &h, int check) {
  const bool sumnorm = h.rule != 0;
  const double cur = sumnorm ? h.bound : h.err, prev = sumnorm ? h.bound_prev : h.err_prev;
  const double target = sumnorm ? h.bound_target : h.eps;
  if (!(cur > 0.0) || !(prev > cur) || !(target > 0.0) || cur <= target) return check;
  const double left = std::log(target / cur) / std::log(cur / prev);
  if (!(left > 0.0)) return check;
  return static_cast<int>(std::min<double>(check, std::max(1.0, std::ceil(left))));
}

namespace {

// Iterations the state h predicts are left (as next_batch, unclamped): 1
// once the bound is met (a certification step of a mixed run may follow),
// `check` when the last two residuals give no decay to extrapolate.
int iterations_left(const PrState &h, int check) {
  const bool sumnorm = h.rule != 0;
  const double cur = sumnorm ? h.bound : h.err, prev = sumnorm ? h.bound_prev : h.err_prev;
  const double target = sumnorm ? h.bound_target : h.eps;
  if (cur <= target) return 1;
  if (!(cur > 0.0) || !(prev > cur) || !(target > 0.0)) return check;
  const double left = std::log(target / cur) / std::log(cur / prev);
  if (!(left > 0.0) || !(left < 1e6)) return check;
  return static_cast<int>(std::ceil(left));
}

}  // namespace

namespace {

// The engine.  The result goes to out_dev, or (out_dev == nullptr) to a buffer
// of the run, and from there to out_host if given.  arena != nullptr: every buffer of the run is a slice of the
// arena (cap bytes) and nothing is allocated (the caller has checked that
// the mirror exists and that no lazily built layout is needed).
PageRankReport run_page_rank(const cpp::Matrix &m, const PageRankParams &p, double *out_dev, double *out_host,
                             hipStream_t s, unsigned char *arena, std::size_t cap) {
  const long n = m.get_n_col();
  // (COO keeps NR/NC in ln_row/ln_col, MatrixCOO.cpp:344-345, so the block
  // layout is read from NR/NC)
  if (m.get_n_row() != m.get_n_col() || m.get_NR() != 1 || m.get_NC() != 1)
    throw std::invalid_argument("tbsla: page_rank needs a square matrix held in one block");
  PageRankReport rep;
  if (n == 0) return rep;
  const bool pat32 = p.precision == PrPrecision::PATTERN_F32;
  const bool pattern = p.precision == PrPrecision::PATTERN;
  const bool mixed = p.precision == PrPrecision::F32 || p.precision == PrPrecision::BF16 || pat32;
  const bool csr = m.format() == cpp::FORMAT_CSR;
  if ((mixed || p.precision == PrPrecision::PATTERN) && !csr)
    throw std::invalid_argument("tbsla: mixed-precision and value-free PageRank need a CSR matrix");
  if ((p.precision == PrPrecision::PATTERN || pat32) && !m.count_stochastic())
    throw std::invalid_argument("tbsla: value-free PageRank needs values from fill_cqmat_stochastic");
  if (mixed && p.rule != PrRule::SUMNORM)
    throw std::invalid_argument("tbsla: mixed-precision PageRank uses the SUMNORM stopping rule");
  if (p.values && (!csr || p.precision != PrPrecision::F64))
    throw std::invalid_argument("tbsla: explicit edge values need a CSR matrix and FP64 precision");

  const DeviceMatrix &d64 = mirror(m, Dtype::F64);
  if (csr && !d64.noop && d64.rows != n)
    throw std::invalid_argument("tbsla: CSR rowptr does not cover every row");
  if (d64.x_need > n) throw std::invalid_argument("tbsla: column index beyond n_col");
  const bool fused = csr && !d64.noop && d64.rows == n;
  // propagation-blocked products: explicit choice, or by default on graphs
  // of 2^16 nodes and more, whatever the stopping rule (their row sums are
  // rounded in a run-dependent order; gather = 1 keeps the fixed-order tile
  // products, whose sums are the reference's)
  const bool use_pb = fused && !p.values && (p.gather == 2 || (p.gather == 0 && n >= (1L << 16)));
  const PbMatrix *pbm = nullptr;
  // small graphs with few long rows: the whole run in one workgroup.  (The
  // stored values' padding is read, so explicit ones take the tiles; f_col is
  // 0 in a matrix of one block.)
  const bool small = fused && !use_pb && !mixed && !p.values && n <= kOneBlockRows && d64.nlong == 0 &&
                     d64.one_block_chain <= kOneBlockChain && d64.f_col == 0 && p.max_iteration > 0;
  // Blocked products of a matrix whose stored entries agree within every
  // column (a link graph: 1/out-degree) read no values: the input is scaled
  // by the column's value once, which gives the same rounded products.  (On
  // fill_cqmat_stochastic(2^24,2^24,8,0.5,7): FP64 iteration 696 -> 536 us,
  // FP32 437 -> 385, BF16 436 -> 428.)
  bool vfree = false;
  const bool try_vfree = small && d64.entries <= kOneBlockEntries;
  if (try_vfree && !arena) vfree = column_values(m, d64, n, s);
  if (use_pb) {
    vfree = column_values(m, d64, n, s);
    pbm = &pb_mirror(m, vfree ? Dtype::PATTERN : Dtype::F64);
    if (!vfree && p.precision == PrPrecision::F32) pbm = &pb_mirror(m, Dtype::F32);
    if (!vfree && p.precision == PrPrecision::BF16) pbm = &pb_mirror(m, Dtype::BF16);
  }
  // the tile products of a mixed run read the values in the low precision
  // (the blocked ones read them from the blocked layout)
  const DeviceMatrix *dlo = nullptr;
  if (!use_pb && p.precision == PrPrecision::F32) dlo = &mirror(m, Dtype::F32);
  if (!use_pb && p.precision == PrPrecision::BF16) dlo = &mirror(m, Dtype::BF16);
  Scratch w;
  RunLayout ws;
  const unsigned gN = grid_for(n);
  // blocks of the normalise pass.  The mixed one (six streams) measured
  // faster with twice the blocks (four and eight times: slower); the FP64 one
  // (three streams) slower
  const unsigned gM = static_cast<unsigned>(std::min<long>(mixed ? 2 * kPassBlocks : kPassBlocks, (n + 1023) / 1024));
  // sum-normalised rule with propagation-blocked products: the update, the
  // normalisation and the residual in the gather pass
  const bool sn = pbm && p.rule == PrRule::SUMNORM;
  const unsigned nparts = std::max(gM, sn ? static_cast<unsigned>(pbm->nbins) : 0u);
  ws.alloc(w.st, 2 * sizeof(PrState));
  ws.alloc(w.slots, 2 * sizeof(unsigned long long) * kMaxSlots);
  ws.alloc(w.perr, sizeof(double) * nparts);
  ws.alloc(w.ps, sizeof(double) * nparts);
  ws.alloc(w.pc, sizeof(double) * nparts);
  // (mixed runs on propagation-blocked products keep the iterate as the
  // anchor plus the delta and never use X)
  const bool pb_mixed = mixed && sn;
  if (!pb_mixed) {
    ws.alloc(w.X0, sizeof(double) * n);
    ws.alloc(w.X1, sizeof(double) * n);
  }
  // blocked products: 8 bytes per far entry, and kPbChunk spare slots that the
  // scatter's idle lanes write (the run's own: the layout is shared between
  // the runs of a matrix)
  if (pbm) ws.alloc(w.prod, sizeof(double) * (static_cast<std::size_t>(pbm->n_far) + kPbChunk));
  // teleport mode: 0 uniform, 1 node set (Matrix.cpp:63-114), 2 distribution vector
  const int tmode = p.teleport ? 2 : (p.personalized ? 1 : 0);
  Teleport tp{nullptr, p.teleport};
  const double b0 = p.personalized && !p.teleport ? 0.25 : 1.0;
  if (tmode == 1) {
    ws.alloc(w.member, static_cast<std::size_t>(n));
    ws.alloc(w.nodes, sizeof(int) * static_cast<std::size_t>(std::max(0, p.n_nodes)));
  }
  if (mixed) {
    ws.alloc(w.xhat, sizeof(double) * n);
    ws.alloc(w.D0, sizeof(float) * n);
    ws.alloc(w.D1, sizeof(float) * n);
    if (sn) {
      // the anchor's FP32 one-step change and FP32 copy, and the scatter's
      // per-superblock sums of a moved anchor
      ws.alloc(w.W, sizeof(float) * n);
      ws.alloc(w.xhat32, sizeof(float) * n);
      ws.alloc(w.hsum, sizeof(double) * std::max(1, pbm->nsb));
      ws.alloc(w.hcomp, sizeof(double) * std::max(1, pbm->nsb));
    } else {
      ws.alloc(w.yhat, sizeof(double) * n);
    }
  }
  // value-free deltas: the product's input zd = colscale32 .* delta
  const bool zdelta = pat32 || (pb_mixed && vfree);
  if (zdelta) {
    ws.alloc(w.ZD0, sizeof(float) * n);
    ws.alloc(w.ZD1, sizeof(float) * n);
  }
  // (propagation-blocked runs form z = colscale .* x where they read it)
  const bool stored_z = !pbm && (pattern || (mixed && m.count_stochastic()));
  if (stored_z) ws.alloc(w.Z, sizeof(double) * n);
  if (!out_dev) ws.alloc(w.out, sizeof(double) * n);
  // (allocation-free runs find the column values again in each run)
  if (try_vfree && arena) {
    ws.alloc(w.cs, sizeof(double) * n);
    ws.alloc(w.flag, sizeof(double));
  }
  std::unique_ptr<RunSpace> space;
  if (arena) {
    if (ws.bytes() > cap)
      throw std::invalid_argument("tbsla: the allocation-free PageRank needs more than its " +
                                  std::to_string(cap >> 20) + " MiB scratch buffer");
    ws.place(arena);
  } else {
    space = m.device_cache().spaces.take(ws.bytes());
    ws.place(space->mem.get());
  }
  if (!out_dev) out_dev = w.out.as<double>();
  if (tmode == 1) {
    hipLaunchKernelGGL(fill_u8, dim3(grid_for(n)), dim3(256), 0, s, w.member.as<unsigned char>(), n,
                       static_cast<unsigned char>(0));
    if (p.n_nodes > 0) {
      // (p.nodes stays valid until the run has ended)
      TBSLA_HIP_CHECK(hipMemcpyAsync(w.nodes.p, p.nodes, sizeof(int) * static_cast<std::size_t>(p.n_nodes),
                                     hipMemcpyHostToDevice, s));
      hipLaunchKernelGGL(set_members, dim3(grid_for(p.n_nodes)), dim3(256), 0, s, w.member.as<unsigned char>(), n,
                         w.nodes.as<int>(), p.n_nodes);
    }
    tp.member = w.member.as<unsigned char>();
  }
  // the column values of a value-free run (1/count per column after
  // fill_cqmat_stochastic), and those of its deltas in FP32 (as rounded for
  // the run's precision)
  const double *colscale64 = nullptr;
  const float *colscale32 = nullptr;
  if (arena) {
    if (try_vfree) vfree = find_column_values(m, d64, n, w.cs.as<double>(), w.flag.as<double>(), s);
    if (vfree) colscale64 = w.cs.as<double>();
  } else if (vfree || pattern || pat32 || (mixed && m.count_stochastic())) {
    (void)column_values(m, d64, n, s);
    const DeviceCache &cache = m.device_cache();
    colscale64 = cache.colscale64.as<double>();
    colscale32 = p.precision == PrPrecision::BF16 ? cache.colscale_bf16.as<float>() : cache.colscale32.as<float>();
  }
  const bool one_block = small && d64.entries <= (vfree ? kOneBlockEntries : kOneBlockEntriesVal);
  PrState h{};
  h.beta = p.beta;
  h.eps = p.epsilon;
  h.bound_target = p.epsilon * (1.0 - p.beta) / p.beta;
  h.tele_scale = tmode == 2   ? (1.0 - p.beta)
                 : tmode == 1 ? (1.0 - p.beta) / static_cast<double>(static_cast<std::size_t>(p.n_nodes))
                              : (1.0 - p.beta) / static_cast<double>(n);
  // sum-normalised propagation-blocked runs start from 1/n (any uniform
  // start gives the same sum-normalised iterates; this one keeps the
  // iterates near sum 1 from the start)
  const double x0 = sn ? 1.0 / static_cast<double>(n) : b0;
  const double x0s = mixed ? static_cast<double>(static_cast<float>(x0)) : x0;  // as stored
  h.sum = x0s * static_cast<double>(n);
  h.tele = h.sum * h.tele_scale;
  h.inv_sum = 1.0 / h.sum;
  h.sum_hat = 0.0;
  h.t_anchor = 0.0;
  h.c_anchor = 1.0;
  h.bound = 2.0;
  h.bound_prev = 2.0;
  h.bound_anchor = 2.0;
  h.max_it = p.max_iteration;
  h.rule = static_cast<int>(p.rule);
  h.mixed = mixed ? 1 : 0;
  // FP64 reference-rule runs on propagation-blocked products keep each
  // update's b unnormalised and carry its scale (1/max) to the readers of
  // the iterate, so the normalise pass writes nothing (a pass over the
  // iterate less per iteration)
  h.raw = (fused && pbm && !sn && !mixed) ? 1 : 0;
  h.xscale = 1.0;
  h.xnext = 1.0;
  // mixed runs start from the anchor xhat = 0 (so yhat = A xhat = 0 with no
  // product) and delta = b0: the first phase carries the whole iterate in the
  // low precision, and the first anchor move comes when it has converged to
  // that precision's floor
  h.need_anchor = 0;
  h.anchors = 0;
  h.floor_eps = p.precision == PrPrecision::BF16 ? 4e-3 : 6e-8;  // FP32 and PATTERN_F32: 6e-8
  // (a sweep on fill_cqmat_stochastic(2^24,2^24,8,0.5,7): BF16 5e-2 -> 7
  // anchor moves, 2e-2 -> 6, 1e-2 -> 5 and the fastest, 5e-3 -> 5 with one
  // more iteration; FP32 3e-6 and 1e-6 -> 1 move, 1e-5 and above -> 2)
  h.anchor_tau = p.anchor_tau > 0 ? p.anchor_tau : (p.precision == PrPrecision::BF16 ? 1e-2 : 3e-6);
  h.done = p.max_iteration <= 0 ? 1 : 0;
  // one launch writes the state, the slots and every start vector (the other
  // buffers are written before they are read)
  PrInit in{};
  in.h = h;
  in.st = w.st.as<PrState>();
  in.slots = w.slots.as<unsigned long long>();
  in.n = n;
  in.x = w.X0.as<double>();
  in.x0 = x0;
  PrState *const st = w.st.as<PrState>();
  double *X[2] = {w.X0.as<double>(), w.X1.as<double>()};
  unsigned long long *const slots = w.slots.as<unsigned long long>();
  float *D[2] = {nullptr, nullptr};
  if (mixed) {
    D[0] = in.d = w.D0.as<float>();
    D[1] = w.D1.as<float>();
    in.xhat = w.xhat.as<double>();
    if (sn) {
      // (w is 0 before the first anchor, whose anchor is 0)
      in.w = w.W.as<float>();
      in.xhat32 = w.xhat32.as<float>();
    } else {
      in.yhat = w.yhat.as<double>();
    }
  }
  float *ZD[2] = {w.ZD0.as<float>(), w.ZD1.as<float>()};
  if (zdelta) {
    in.zd = ZD[0];
    if (sn)
      in.zd_scale32 = colscale32;
    else
      in.zd_scale64 = colscale64;
  }
  if (stored_z) {
    in.z = w.Z.as<double>();
    in.z_scale = colscale64;
  }
  hipLaunchKernelGGL(pr_init, dim3(gN), dim3(256), 0, s, in);
  TBSLA_HIP_CHECK(hipGetLastError());

  // device time of the loop: HIP events, or (allocation-free runs, which
  // create no events) the host clock between two stream synchronisations
  if (arena) TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  const auto h0 = std::chrono::steady_clock::now();
  if (space) TBSLA_HIP_CHECK(hipEventRecord(space->timing[0], s));
  const int check = one_block ? 256 : (fused ? std::max(1, p.check_every) : 1);
  int next = check;  // iterations in the next launch batch
  PrState hs{};
  int launched = 0;
  const bool mixed_pattern = mixed && m.count_stochastic();
  // runs whose updates take the step decision of the iteration before: the
  // tile products and the generic engine in one precision (their state
  // alternates between two buffers).  On larger matrices than those with
  // kMergeTileNnz-entry tiles the decision repeated in every block costs more
  // than a launch of its own.
  const bool merged = !pbm && !mixed && !one_block && (!fused || d64.tile_nnz == kMergeTileNnz);
  const auto state = [&](int it) { return merged ? st + (it & 1) : st; };
  const SnPartials sp{w.perr.as<double>(), w.ps.as<double>(), w.pc.as<double>()};
  const Partials parts{sp.perr, sp.ps, sp.pc, static_cast<int>(sn ? static_cast<unsigned>(pbm->nbins) : gM)};
  const Partials none{sp.perr, sp.ps, sp.pc, 0};
  double *Z = w.Z.as<double>();
  const double *colscale = colscale64;
  const auto normalize = [&](auto mode, double *xout, const double *xin, const float *dcur, float *dnext, float *zdnext,
                             double *z, int it) {
    hipLaunchKernelGGL(pr_normalize<decltype(mode)::value>, dim3(gM), dim3(1024), 0, s, xout, xin,
                       w.xhat.as<double>(), dcur, dnext, z, colscale, zdnext, colscale32, n, state(it + 1),
                       slots + (it & 1) * kMaxSlots, slots + ((it + 1) & 1) * kMaxSlots, sp.perr, sp.ps, sp.pc);
  };
  const auto decide = [&](PrState *to) {
    hipLaunchKernelGGL(pr_finalize_norm, dim3(1), dim3(kTileThreads), 0, s, sp.perr, sp.ps, sp.pc,
                       static_cast<int>(gM), to);
  };
  using std::integral_constant;
  auto launch_batch = [&](int batch) {
    if (one_block) {
      if (tmode == 1)
        launch_one_block<1>(d64, colscale64, static_cast<int>(n), tp, X[0], out_dev, st, batch, s);
      else if (tmode == 2)
        launch_one_block<2>(d64, colscale64, static_cast<int>(n), tp, X[0], out_dev, st, batch, s);
      else
        launch_one_block<0>(d64, colscale64, static_cast<int>(n), tp, X[0], out_dev, st, batch, s);
    }
    for (int k = 0; k < batch && !one_block; k++) {
      const int it = launched + k;
      double *xin = X[it & 1], *xout = X[(it + 1) & 1];
      // the step decision of the iteration before is taken by this one, the
      // last of the batch's by a launch of its own
      const Partials &pp = k > 0 ? parts : none;
      unsigned long long *const slot = slots + (it & 1) * kMaxSlots;
      const StepArgs step = merged ? StepArgs{state(it), state(it + 1), pp} : StepArgs{st, nullptr, none};
      if (sn) {
        if (mixed) {
          MxBufs b;
          b.am = AnchorMove{w.xhat.as<double>(), w.xhat32.as<float>(), D[it & 1], colscale, w.hsum.as<double>(),
                            w.hcomp.as<double>(), 0};
          b.xd = vfree ? static_cast<const void *>(ZD[it & 1]) : static_cast<const void *>(D[it & 1]);
          b.prod = w.prod.p;
          b.w = w.W.as<float>();
          b.dold = D[it & 1];
          b.dnew = D[(it + 1) & 1];
          b.zdnew = vfree ? ZD[(it + 1) & 1] : nullptr;
          b.colscale32 = colscale32;
          if (vfree)
            launch_pb_mx<dev::Pattern, dev::Pattern, float, true>(tmode, *pbm, -1, -1, b, tp, st, sp, s);
          else if (p.precision == PrPrecision::F32)
            launch_pb_mx<double, float, float, false>(tmode, *pbm, 0, 1, b, tp, st, sp, s);
          else
            launch_pb_mx<double, dev::bf16, float, false>(tmode, *pbm, 0, 2, b, tp, st, sp, s);
        } else {
          launch_pb(tmode, *pbm, colscale, xin, w.prod.as<double>(), tp, xout, st, nullptr, &sp, pp, s);
        }
        // (the anchor move's sum partials: one per superblock of the anchor
        // product's scatter order)
        const int nsb_anchor = vfree ? pb_args_free(*pbm).nsb : pbm->nsb;
        if (mixed || k == batch - 1)
          hipLaunchKernelGGL(pr_finalize_sn, dim3(1), dim3(kTileThreads), 0, s, sp.perr, sp.ps, sp.pc, pbm->nbins,
                             mixed ? w.hsum.as<double>() : nullptr, mixed ? w.hcomp.as<double>() : nullptr,
                             nsb_anchor, st);
      } else if (fused) {
        if (mixed) {
          float *dcur = D[it & 1], *dnext = D[(it + 1) & 1];
          float *zdcur = ZD[it & 1], *zdnext = ZD[(it + 1) & 1];
          double *xhat = w.xhat.as<double>(), *yhat = w.yhat.as<double>();
          {
            // (mixed runs take the tile products here: with propagation-
            // blocked products they run the sum-normalised branch above)
            hipLaunchKernelGGL(pr_anchor_move, dim3(gN), dim3(256), 0, s, xhat, dcur, pat32 ? zdcur : dcur,
                               mixed_pattern ? Z : nullptr, colscale, n, st);
            if (mixed_pattern)
              launch_anchor<dev::Pattern>(d64, Z, yhat, st, s);
            else
              launch_anchor<double>(d64, xhat, yhat, st, s);
            if (pat32)
              launch_update<dev::Pattern, float, true>(tmode, d64, nullptr, zdcur, yhat, tp, xout, step, slot, s);
            else if (p.precision == PrPrecision::F32)
              launch_update<float, float, true>(tmode, *dlo, nullptr, dcur, yhat, tp, xout, step, slot, s);
            else
              launch_update<dev::bf16, float, true>(tmode, *dlo, nullptr, dcur, yhat, tp, xout, step, slot, s);
          }
          if (pat32)
            normalize(integral_constant<int, 3>(), xout, nullptr, dcur, dnext, zdnext, nullptr, it);
          else
            normalize(integral_constant<int, 1>(), xout, nullptr, dcur, dnext, nullptr, nullptr, it);
          decide(st);
        } else if (pbm) {
          launch_pb(tmode, *pbm, colscale, xin, w.prod.as<double>(), tp, xout, st, slot, nullptr, pp, s);
          normalize(integral_constant<int, 4>(), xout, xin, nullptr, nullptr, nullptr, nullptr, it);
          if (k == batch - 1) decide(st);
        } else {
          if (pattern) {
            launch_update<dev::Pattern, double, false>(tmode, d64, nullptr, Z, nullptr, tp, xout, step, slot, s);
            normalize(integral_constant<int, 2>(), xout, xin, nullptr, nullptr, nullptr, Z, it);
          } else {
            launch_update<double, double, false>(tmode, d64, p.values, xin, nullptr, tp, xout, step, slot, s);
            normalize(integral_constant<int, 0>(), xout, xin, nullptr, nullptr, nullptr, nullptr, it);
          }
          if (!merged || k == batch - 1) decide(state(it + 1));
        }
      } else {
        // any format: y = 0 (accumulating formats), y += A b_t, update, normalise
        hipLaunchKernelGGL(fill_f64, dim3(gN), dim3(256), 0, s, xout, n, 0.0);
        if (!d64.noop) launch_spmv(d64, xin, Dtype::F64, xout, Dtype::F64, 0, s);
        if (tmode == 1)
          hipLaunchKernelGGL(pr_update_vec<1>, dim3(gN), dim3(kTileThreads), 0, s, xout, n, tp, step.in, step.out, pp,
                             slot);
        else if (tmode == 2)
          hipLaunchKernelGGL(pr_update_vec<2>, dim3(gN), dim3(kTileThreads), 0, s, xout, n, tp, step.in, step.out, pp,
                             slot);
        else
          hipLaunchKernelGGL(pr_update_vec<0>, dim3(gN), dim3(kTileThreads), 0, s, xout, n, tp, step.in, step.out, pp,
                             slot);
        normalize(integral_constant<int, 0>(), xout, xin, nullptr, nullptr, nullptr, nullptr, it);
        if (k == batch - 1) decide(state(it + 1));
      }
    }
    TBSLA_HIP_CHECK(hipGetLastError());
    launched += batch;
  };
  if (arena) {
    // allocation-free runs: the state is read after every batch
    while (launched < p.max_iteration) {
      launch_batch(std::min(next, p.max_iteration - launched));
      TBSLA_HIP_CHECK(hipMemcpyAsync(&hs, state(launched), sizeof(hs), hipMemcpyDeviceToHost, s));
      TBSLA_HIP_CHECK(hipStreamSynchronize(s));
      if (hs.done) break;
      next = next_batch(hs, check);
    }
  } else {
    // Up to two batches in flight, each followed by a copy of the state to
    // pinned memory and an event: while the host waits for one batch's
    // state, the next batch is already queued when the state read before
    // predicts more iterations than are in flight, so the GPU does not idle
    // at the reads (kernels launched past convergence return at once).
    static_assert(2 * sizeof(PrState) <= kReadBackBytes, "two states fit the read-back buffer");
    PrState *const hbuf = static_cast<PrState *>(space->pinned);
    hipEvent_t *const cev = space->ready;
    int head = 0, npend = 0;  // slot of the oldest batch in flight, batches in flight
    auto enqueue = [&](int batch) {
      launch_batch(batch);
      const int sl = (head + npend) & 1;
      TBSLA_HIP_CHECK(hipMemcpyAsync(hbuf + sl, state(launched), sizeof(PrState), hipMemcpyDeviceToHost, s));
      TBSLA_HIP_CHECK(hipEventRecord(cev[sl], s));
      npend++;
    };
    bool have = false;  // hs holds a state read back
    if (launched < p.max_iteration) enqueue(std::min(check, p.max_iteration - launched));
    while (npend > 0) {
      if (npend == 1 && launched < p.max_iteration && !one_block) {
        int nb = check;
        if (have) nb = std::min(check, iterations_left(hs, check) - (launched - hs.it));
        nb = std::min(nb, p.max_iteration - launched);
        if (nb > 0) enqueue(nb);
      }
      TBSLA_HIP_CHECK(hipEventSynchronize(cev[head]));
      hs = hbuf[head];
      head ^= 1;
      npend--;
      have = true;
      if (hs.done) break;
      if (npend == 0 && launched < p.max_iteration) enqueue(std::min(next_batch(hs, check), p.max_iteration - launched));
    }
  }
  if (space) TBSLA_HIP_CHECK(hipEventRecord(space->timing[1], s));
  const double host_seconds = std::chrono::duration<double>(std::chrono::steady_clock::now() - h0).count();
  const int it = hs.it;
  // final sum normalisation (Matrix.cpp:52-59), compensated
  const double *a = mixed ? w.xhat.as<double>() : X[it & 1];
  const float *dd = mixed ? D[it & 1] : nullptr;
  if (mixed && !sn) {  // the state's sum is that of the FP64 update; the result's elements are rounded
    hipLaunchKernelGGL(pr_sum_rounded, dim3(gM), dim3(1024), 0, s, a, dd, n, sp.ps, sp.pc);
    hipLaunchKernelGGL(pr_sum_merge, dim3(1), dim3(kTileThreads), 0, s, sp.ps, sp.pc, static_cast<int>(gM), st);
  }
  if (!one_block)  // (which wrote the result)
    hipLaunchKernelGGL(pr_scale_kernel, dim3(gN), dim3(256), 0, s, a, dd, n, state(launched), out_dev);
  TBSLA_HIP_CHECK(hipGetLastError());
  if (out_host)
    TBSLA_HIP_CHECK(hipMemcpyAsync(out_host, out_dev, sizeof(double) * static_cast<std::size_t>(n),
                                   hipMemcpyDeviceToHost, s));
  TBSLA_HIP_CHECK(hipStreamSynchronize(s));
  float ms = 0;
  if (space) {
    TBSLA_HIP_CHECK(hipEventElapsedTime(&ms, space->timing[0], space->timing[1]));
    m.device_cache().spaces.give(std::move(space));
  }
  rep.iterations = it;
  rep.anchors = hs.anchors;
  rep.last_error = hs.err;
  rep.bound = hs.bound;
  rep.seconds = arena ? host_seconds : ms * 1e-3;
  return rep;
}

}  // namespace

PageRankReport page_rank_device(const cpp::Matrix &m, const PageRankParams &p, double *out_dev, hipStream_t s) {
  return run_page_rank(m, p, out_dev, nullptr, s, nullptr, 0);
}

// ---- allocation-free PageRank ----------------------------------------------
// The scratch memory of page_rank_device_noalloc: one fixed buffer in each
// GPU's copy of this code object, held until the process ends.  Host code
// never passes `scratch` itself (in host code it names a host-side stand-in):
// it uses the device address hipGetSymbolAddress returns for the current
// device, looked up once per device.
static __device__ __align__(256) unsigned char scratch[kNoAllocScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mu;
unsigned char *g_scratch[kMaxDevices] = {};

unsigned char *scratch_of_current_device() {
  int dev = 0;
  TBSLA_HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw std::runtime_error("tbsla: device index beyond the scratch table");
  std::lock_guard<std::mutex> g(g_scratch_mu);
  if (!g_scratch[dev]) {
    void *ptr = nullptr;
    TBSLA_HIP_CHECK(hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
    if (!ptr) throw std::runtime_error("tbsla: no device address for the scratch buffer");
    g_scratch[dev] = static_cast<unsigned char *>(ptr);
  }
  return g_scratch[dev];
}

std::size_t slice(std::size_t bytes) { return (std::max<std::size_t>(bytes, 1) + 255) & ~std::size_t(255); }

}  // namespace

std::size_t page_rank_noalloc_bytes(long n, int n_nodes) {
  const std::size_t gM = static_cast<std::size_t>(std::min<long>(kPassBlocks, (n + 1023) / 1024));
  std::size_t b = slice(2 * sizeof(PrState)) + slice(2 * sizeof(unsigned long long) * kMaxSlots) +
                  3 * slice(sizeof(double) * gM) + 2 * slice(sizeof(double) * static_cast<std::size_t>(n));
  if (n <= kOneBlockRows) b += slice(sizeof(double) * static_cast<std::size_t>(n)) + slice(sizeof(double));
  if (n_nodes > 0) b += slice(static_cast<std::size_t>(n)) + slice(sizeof(int) * static_cast<std::size_t>(n_nodes));
  return b;
}

PageRankReport page_rank_device_noalloc(const cpp::Matrix &m, const PageRankParams &p, double *out_dev,
                                        hipStream_t s) {
  if (p.precision != PrPrecision::F64)
    throw std::invalid_argument("tbsla: the allocation-free PageRank computes in FP64 (precision TBSLA_F64)");
  if (p.gather == 2)
    throw std::invalid_argument("tbsla: the allocation-free PageRank uses the fixed-order tile products "
                                "(gather 0 or 1): the propagation-blocked layout is built, and allocated, on first use");
  const long n = m.get_n_col();
  const int nodes = p.personalized && !p.teleport ? std::max(p.n_nodes, 0) : 0;
  const std::size_t need = page_rank_noalloc_bytes(n, nodes);
  if (need > kNoAllocScratchBytes)
    throw std::invalid_argument("tbsla: allocation-free PageRank on " + std::to_string(n) + " nodes needs " +
                                std::to_string(need) + " bytes of scratch; the buffer holds " +
                                std::to_string(kNoAllocScratchBytes));
  if (!mirror_if_built(m, Dtype::F64))
    throw std::invalid_argument("tbsla: the allocation-free PageRank needs the FP64 mirror: call "
                                "tbsla_hip_prepare(m, TBSLA_F64) first");
  PageRankParams q = p;
  q.gather = 1;
  return run_page_rank(m, q, out_dev, nullptr, s, scratch_of_current_device(), kNoAllocScratchBytes);
}

PageRankReport page_rank(const cpp::Matrix &m, const PageRankParams &p, double *out) {
  return run_page_rank(m, p, nullptr, out, nullptr, nullptr, 0);
}

}  // namespace hip
}  // namespace tbsla
