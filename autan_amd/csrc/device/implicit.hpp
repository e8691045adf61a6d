// The steady implicit step on the device: pseudo-transient continuation
// (V / dt + dR/dU) du = -R with the approximate Jacobian, as EulerPhysics::steady_step takes it
// with linear_solver = "gauss-seidel" (physics/src/euler_physics.cpp:1056-1250):
//   k_impl_diag, k_impl_off   Euler::assemble (physics/src/euler.cpp:993-1053): per cell
//                             lambda_c / CFL I + the sum over its faces, in cell_faces order, of
//                             +-J D_c; per interior face A(owner, neighbour) = J_R D_neighbour and
//                             A(neighbour, owner) = -J_L D_owner; each J D entry summed over k from 0
//                             and added as sign * t;
//   k_impl_invert             BlockMatrix::factor: each diagonal block's inverse by Gauss-Jordan
//                             elimination with partial pivoting (physics/src/block_matrix.cpp:14-45);
//   k_impl_relax(_run)        BlockMatrix::relax over the cells of one colour (a colour's cells share
//                             no face, so they update together), or of a run of small colours;
//   k_impl_multiply           BlockMatrix::multiply;
//   k_impl_start, k_impl_scale_dot   the GCR's residual, its largest entry (owned_max_abs), scaled by it;
//                             inner products as exact sums (EulerPhysics::owned_dot), fused into the
//                             GCR's updates (k_impl_orth_dots, k_impl_advance_dot);
//   k_impl_admissible         EulerPhysics::admissible_step: each cell's largest fraction of du that
//                             keeps its density and pressure above half their values, the least over
//                             the cells (an exact minimum of the FP64 values);
// and the GCR's vector updates (solvers/src/gcr.cpp). Everything in FP64, no contraction, so every
// value equals the host restatement's. Layouts (chosen for the relaxation, which streams a colour's
// rows): the rows are numbered by position, colour by colour, in each colour those with a neighbour of
// a higher colour first; each of these groups is cut into slices of kSlice = 12 rows (the last padded
// with empty rows), one wave's five lanes per row: lane 5 g + r holds row r of the slice's g-th block.
// The slice's blocks are stored as the wave reads them, 60 consecutive values per block column: the
// diagonal and inverse blocks of slice s at 300 s + 60 j + lane, its off-diagonal blocks slot by slot
// (its rows' k-th entries together, rows with fewer padded with zero blocks) at 300 slot + 60 j +
// lane. The solve's vectors (the right-hand side, du, the GCR's directions) hold value q of position p
// at 5 p + q, 60 values per slice; the padding rows' are 0.
#pragma once

#include "exact.hpp"
#include "jacobian.hpp"

namespace mxe {

static_assert(kWords == kExactWords, "the device's exact-sum words are exact_value's");

// Row r of out += sign * (j d) for 5 x 5 row-major blocks: out_r[c] += sign * sum_k j_r[k] dm[5 k + c],
// each entry's product summed over k from zero.
__device__ __forceinline__ void impl_add_product_row(double* out_r, const double* j_r, const double* dm, double sign) {
#pragma unroll
  for (int c = 0; c < 5; ++c) {
    double t = 0.0;
#pragma unroll
    for (int k = 0; k < 5; ++k) t += j_r[k] * dm[5 * k + c];
    out_r[c] += sign * t;
  }
}

// Row r of a block stored as impl_block reads it.
__device__ __forceinline__ void impl_block_row(const double* __restrict__ v, long long n, long long e, int k, int r,
                                               double* b_r) {
#pragma unroll
  for (int c = 0; c < 5; ++c) b_r[c] = v[(25LL * k + 5 * r + c) * n + e];
}

__device__ __forceinline__ void impl_block(const double* __restrict__ v, long long n, long long e, int k, double* b) {
#pragma unroll
  for (int q = 0; q < 25; ++q) b[q] = v[(25LL * k + q) * n + e];
}

// Cell c's 5 x 5 dW/dq block from the cell-major copy (25 contiguous values per cell).
__device__ __forceinline__ void impl_cell_block(const double* __restrict__ dwdu, long long c, double* b) {
  const double* p = dwdu + 25 * c;
#pragma unroll
  for (int q = 0; q < 25; ++q) b[q] = p[q];
}

constexpr int kSlice = kWave / 5;          // rows per slice
constexpr int kSliceVec = 5 * kSlice;      // values of a vector per slice, the lanes at work
constexpr int kSliceBlock = 25 * kSlice;   // values of a slice's blocks

// The address of value (0, 0) of entry e (its slot times kSlice plus its row's place in the slice);
// value (r, j) is 60 j + r further.
__device__ __forceinline__ long long impl_entry(int e) {
  return static_cast<long long>(e / kSlice) * kSliceBlock + 5 * (e % kSlice);
}

// The diagonal blocks: lam_c / cfl on the diagonal, then the cell's faces in cell_faces order.
// An interior face's term is the negated off-diagonal block of the transposed position, which
// k_impl_off has stored: the owner's +J_L D_owner is -A(neighbour, owner) (entry at[f].y), the
// neighbour's -J_R D_neighbour is -A(owner, neighbour) (entry at[f].x). Each such block is the
// same sum from zero, negated exactly, and a running sum from +0 is never -0, so adding the
// negated entry gives the bits of adding the product; it reads each entry's 25 contiguous values
// instead of recomputing the product from the face blocks. A boundary face's term J_b D_c from
// bj (25 x nb) and the cell's dW/dq block (cell-major). One wave per slice, lane 5 g + r row r of the
// g-th row's block; an empty row's block is 0.
template <class C>
__global__ __launch_bounds__(kBlock) void k_impl_diag(Dev<C> d, const double* __restrict__ dwdu,
                                                      const double* __restrict__ bj, const double* __restrict__ offd,
                                                      const int2* __restrict__ at, double cfl,
                                                      const int* __restrict__ cell, int slices,
                                                      double* __restrict__ diag) {
  const int lane = threadIdx.x % kWave;
  const int s = blockIdx.x * (kBlock / kWave) + static_cast<int>(threadIdx.x / kWave);
  if (s >= slices || lane >= kSliceVec) return;
  const int r = lane % 5;
  const int c = cell[kSlice * s + lane / 5];
  double dg[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  if (c >= 0) {
    const double shift = static_cast<double>(d.lam[c]) / cfl;
    dg[r] += shift;
    for (int k = d.cfo[c]; k < d.cfo[c + 1]; ++k) {
      const int e = d.inc[k];
      const int f = e & 0x7fffffff;
      if (f >= d.ni) {
        double dc[25], j[5];
        impl_cell_block(dwdu, c, dc);
        impl_block_row(bj, d.nb, f - d.ni, 0, r, j);
        impl_add_product_row(dg, j, dc, 1.0);
      } else {
        const int2 a = at[f];
        const double* o = offd + impl_entry(e >= 0 ? a.y : a.x) + r;
#pragma unroll
        for (int q = 0; q < 5; ++q) dg[q] += -o[kSliceVec * q];
      }
    }
  }
  double* out = diag + static_cast<long long>(kSliceBlock) * s + lane;
#pragma unroll
  for (int q = 0; q < 5; ++q) out[kSliceVec * q] = dg[q];
}

// The off-diagonal blocks of every interior face, at their entries (at[f].x in the owner's row,
// at[f].y in the neighbour's): J_R D_neighbour (row owner), -J_L D_owner (row neighbour). One
// thread per face: five lanes per face would each load the cells' whole dW/dq blocks, and a block
// computed a row at a time stores in pieces too small (measured twice the time).
template <class C>
__global__ __launch_bounds__(kBlock) void k_impl_off(Dev<C> d, const double* __restrict__ dwdu,
                                                     const double* __restrict__ fj, const int2* __restrict__ at,
                                                     double* __restrict__ offd) {
  const int f = blockIdx.x * kBlock + threadIdx.x;
  if (f >= d.ni) return;
  const int2 lr = d.lr[f];
  const int2 k = at[f];
  double j[25], dm[25], out[25];
  impl_block(fj, d.ni, f, 1, j);
  impl_cell_block(dwdu, lr.y, dm);
#pragma unroll
  for (int q = 0; q < 25; ++q) out[q] = 0.0;
#pragma unroll
  for (int r = 0; r < 5; ++r) impl_add_product_row(out + 5 * r, j + 5 * r, dm, 1.0);
  double* up = offd + impl_entry(k.x);
#pragma unroll
  for (int q = 0; q < 25; ++q) up[kSliceVec * (q % 5) + q / 5] = out[q];
  impl_block(fj, d.ni, f, 0, j);
  impl_cell_block(dwdu, lr.x, dm);
#pragma unroll
  for (int q = 0; q < 25; ++q) out[q] = 0.0;
#pragma unroll
  for (int r = 0; r < 5; ++r) impl_add_product_row(out + 5 * r, j + 5 * r, dm, -1.0);
  double* lo = offd + impl_entry(k.y);
#pragma unroll
  for (int q = 0; q < 25; ++q) lo[kSliceVec * (q % 5) + q / 5] = out[q];
}

// Each diagonal block's inverse: Gauss-Jordan on [A | I] with partial pivoting (the first row
// holding the largest |pivot| below the diagonal, rows swapped whole, the pivot row scaled by the
// pivot's reciprocal, every other row reduced). A zero or non-finite pivot marks the cell in
// *singular (the least such cell). One thread per position p, cell[p] its cell.
__global__ __launch_bounds__(kBlock) void k_impl_invert(const double* __restrict__ diag, const int* __restrict__ cell,
                                                        int n, double* __restrict__ inverse,
                                                        int* __restrict__ singular) {
  const int p = blockIdx.x * kBlock + threadIdx.x;
  if (p >= n) return;
  if (cell[p] < 0) return;  // an empty row: its inverse stays 0
  const double* dp = diag + static_cast<long long>(kSliceBlock) * (p / kSlice) + 5 * (p % kSlice);
  double m[5][10];
#pragma unroll
  for (int i = 0; i < 5; ++i) {
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      m[i][j] = dp[kSliceVec * j + i];
      m[i][5 + j] = i == j ? 1.0 : 0.0;
    }
  }
  bool ok = true;
#pragma unroll
  for (int k = 0; k < 5; ++k) {
    // The pivot row by its value's magnitude carried along, so that no register is indexed at
    // run time (the first strictly larger one wins, as when comparing with m[piv][k]).
    int piv = k;
    double best = fabs(m[k][k]);
#pragma unroll
    for (int i = k + 1; i < 5; ++i) {
      const double a = fabs(m[i][k]);
      if (a > best) {
        best = a;
        piv = i;
      }
    }
    // Swapped by selects, row by row.
#pragma unroll
    for (int i = k + 1; i < 5; ++i) {
      if (i == piv) {
#pragma unroll
        for (int j = 0; j < 10; ++j) {
          const double t = m[k][j];
          m[k][j] = m[i][j];
          m[i][j] = t;
        }
      }
    }
    if (m[k][k] == 0.0 || !__builtin_isfinite(m[k][k])) ok = false;
    const double dv = 1.0 / m[k][k];
#pragma unroll
    for (int j = 0; j < 10; ++j) m[k][j] *= dv;
#pragma unroll
    for (int i = 0; i < 5; ++i) {
      if (i == k) continue;
      const double f = m[i][k];
#pragma unroll
      for (int j = 0; j < 10; ++j) m[i][j] -= f * m[k][j];
    }
  }
  if (!ok) atomicMin(singular, cell[p]);
  double* ip = inverse + static_cast<long long>(kSliceBlock) * (p / kSlice) + 5 * (p % kSlice);
#pragma unroll
  for (int j = 0; j < 5; ++j) {
#pragma unroll
    for (int i = 0; i < 5; ++i) ip[kSliceVec * j + i] = m[i][5 + j];
  }
}

// The rows by position: the cell of each (-1: an empty row), slice s's slots slot[s] .. slot[s + 1],
// and the position of the other cell of every entry (kSlice per slot; -1: padding). A row's entries
// are the cell's interior faces in ascending face order, one per slot from the slice's first.
struct ImplRows {
  const int* slot;
  const int* other;
  const int* cell;
};

// Sum over a slice's slots of A_cf x_other, row by row, added to (ADD) or taken from r: slot by slot,
// then column by column, the one-thread order. kSlots slots' loads are issued together (the entry's
// place, five block columns, one value of the other cell per lane; the group's five values reach its
// lanes by shuffles), since the sums that use them are one chain. A padding entry is a zero block
// times zeros, which leaves r's bits (a sum from +0, or r - 0) as they are.
constexpr int kSlots = 3;

template <bool ADD>
__device__ __forceinline__ double impl_slots(const ImplRows& rows, int s, int lane, const double* __restrict__ offd,
                                             const double* x, double r) {
  // No load stands behind a condition (the compiler moves one that does to its use): the idle lanes
  // read the last row's, a slot past the slice the last slot's, and zeros take their place.
  const int at = lane < kSliceVec ? lane : kSliceVec - 1;
  const int g = at / 5, q = at % 5, base = lane - lane % 5;
  const int k1 = rows.slot[s + 1];
  int next[kSlots];
  // The places are read kSlots ahead, so that a long row's chain is one load per kSlots, not two.
  auto places = [&](int k) {
#pragma unroll
    for (int u = 0; u < kSlots; ++u) next[u] = rows.other[kSlice * (k + u < k1 ? k + u : k1 - 1) + g];
  };
  const int first = rows.slot[s];
  if (first < k1) places(first);
  for (int k0 = first; k0 < k1; k0 += kSlots) {
    int o[kSlots];
    double a[kSlots][5], xq[kSlots];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      o[u] = k0 + u < k1 ? next[u] : -1;
      const double* block = offd + static_cast<long long>(kSliceBlock) * (k0 + u < k1 ? k0 + u : k1 - 1) + at;
#pragma unroll
      for (int j = 0; j < 5; ++j) a[u][j] = block[kSliceVec * j];
    }
    places(k0 + kSlots < k1 ? k0 + kSlots : first);
#pragma unroll
    for (int u = 0; u < kSlots; ++u) xq[u] = x[5LL * (o[u] >= 0 ? o[u] : 0) + q];
#pragma unroll
    for (int u = 0; u < kSlots; ++u) {
      const double xu = o[u] >= 0 ? xq[u] : 0.0;
#pragma unroll
      for (int j = 0; j < 5; ++j) {
        const double xj = __shfl(xu, (base + j) % kWave);
        const double aj = k0 + u < k1 ? a[u][j] : 0.0;
        if constexpr (ADD) {
          r += aj * xj;
        } else {
          r -= aj * xj;
        }
      }
    }
  }
  return r;
}

// BlockMatrix::relax of a slice's rows by one wave, lane 5 g + q row q of the g-th: x_c = D_c^-1 (b_c -
// sum_f A_cf x_other). The group's five rows reach its lanes by shuffles for the inverse's product.
// Bound by the blocks' bytes on a large colour and by the chain of loads (slot, place, value) on a
// small one: the inverse, the right-hand side and three slots' blocks are in flight at once. With the
// blocks row by row (each lane five consecutive values, a wave's loads 40 bytes apart) and one entry
// in flight, two iterations of a 1.03M-cell channel took 54.1 ms where they now take 48.7 (the
// relaxations 5.5 TB/s of blocks and values; each lane reading the other cell's five values itself 54.2),
// a 39.5k-cell fp64 channel's 6.56 and 6.0 ms.
__device__ __forceinline__ void impl_relax_slice(const ImplRows& rows, int s, const double* __restrict__ offd,
                                                 const double* __restrict__ inverse, const double* __restrict__ b,
                                                 double* x) {
  const int lane = threadIdx.x % kWave;
  const bool on = lane < kSliceVec;
  const int base = lane - lane % 5;
  const int at = on ? lane : kSliceVec - 1;  // the idle lanes repeat the last row's loads
  const long long v = static_cast<long long>(kSliceVec) * s + at;
  double ip[5];
#pragma unroll
  for (int j = 0; j < 5; ++j) ip[j] = inverse[static_cast<long long>(kSliceBlock) * s + kSliceVec * j + at];
  const double r = impl_slots<false>(rows, s, lane, offd, x, b[v]);
  double sum = 0.0;
#pragma unroll
  for (int j = 0; j < 5; ++j) sum += ip[j] * __shfl(r, (base + j) % kWave);
  if (on) x[v] = sum;
}

// The slice of this wave in a launch over `count` slices, -1 past them: each XCD takes a contiguous
// run, whose neighbours' values share its L2.
__device__ __forceinline__ int impl_slice(int count) {
  const int waves = blockDim.x / kWave;
  const int t = __builtin_amdgcn_readfirstlane(xcd_block() * waves + static_cast<int>(threadIdx.x / kWave));
  return t < count ? t : -1;
}

// Threads of a block and blocks of a launch over `count` slices: four waves per block, or one where
// that leaves fewer than two blocks per CU.
constexpr int kImplFewSlices = 4 * 512;
inline int impl_threads(int count) { return count < kImplFewSlices ? kWave : kBlock; }
inline int impl_grid(int count) {
  const int waves = impl_threads(count) / kWave;
  return xcd_grid((count + waves - 1) / waves);
}

// BlockMatrix::relax of the slices first .. first + count (rows of one colour).
__global__ __launch_bounds__(kBlock) void k_impl_relax(ImplRows rows, int first, int count,
                                                       const double* __restrict__ offd,
                                                       const double* __restrict__ inverse,
                                                       const double* __restrict__ b, double* x) {
  const int t = impl_slice(count);
  if (t >= 0) impl_relax_slice(rows, first + t, offd, inverse, b, x);
}

// The first relaxation of the sweeps from x = 0, colour 0's `count` slices: x_c = D_c^-1 b_c, every
// neighbour's value being zero, without reading an off-diagonal block; and x = 0 on the other slices
// up to n. The blocks are finite here (each is a term of a diagonal block, and an inverse met a
// non-finite pivot otherwise and the solve was refused), so the products left out are zeros; a zero's
// sign in b_c - 0 is lost in the inverse's product, whose sum starts at +0.
__global__ __launch_bounds__(kBlock) void k_impl_relax_start(int count, int n, const double* __restrict__ inverse,
                                                             const double* __restrict__ b, double* __restrict__ x) {
  const int s = impl_slice(n);
  if (s < 0) return;
  const int lane = threadIdx.x % kWave;
  const bool on = lane < kSliceVec;
  const int base = lane - lane % 5;
  const long long v = static_cast<long long>(kSliceVec) * s + lane;
  double sum = 0.0;
  if (s < count) {
    const double r = on ? b[v] : 0.0;
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      const double a = on ? inverse[static_cast<long long>(kSliceBlock) * s + kSliceVec * j + lane] : 0.0;
      sum += a * __shfl(r, (base + j) % kWave);
    }
  }
  if (on) x[v] = sum;
}

// A run of small colours relaxed in order by one workgroup: phase p relaxes the slices first[p] ..
// first[p] + count[p], the barrier between phases making each phase's x visible to the next (the
// workgroup shares one CU's cache), as separate launches would. Saves a launch per colour where a
// colour is too small to fill the device.
constexpr int kRelaxRunThreads = 1024;
constexpr int kRelaxRunMax = 32;
// Colours of at most this many slots join a run: their blocks (2.4 KB a slot) come into one CU, 64 bytes
// a cycle, in 3 us or less, what a launch costs. A colour of 600 slots (1.03M-cell channel) took 13 us of
// a run.
constexpr int kRelaxRunSlots = 192;
struct ImplRun {
  int first[kRelaxRunMax];
  int count[kRelaxRunMax];
  int phases;
};

__global__ __launch_bounds__(kRelaxRunThreads) void k_impl_relax_run(ImplRows rows, ImplRun run,
                                                                     const double* __restrict__ offd,
                                                                     const double* __restrict__ inverse,
                                                                     const double* __restrict__ b, double* x) {
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x / kWave));
  for (int p = 0; p < run.phases; ++p) {
    for (int t = wave; t < run.count[p]; t += kRelaxRunThreads / kWave) {
      impl_relax_slice(rows, run.first[p] + t, offd, inverse, b, x);
    }
    __syncthreads();
  }
}

// BlockMatrix::multiply: y_c = D_c x_c + sum_f A_cf x_other, the diagonal block first, in slices as the
// relaxation.
__global__ __launch_bounds__(kBlock) void k_impl_multiply(ImplRows rows, int slices, const double* __restrict__ diag,
                                                          const double* __restrict__ offd,
                                                          const double* __restrict__ x, double* __restrict__ y) {
  const int s = impl_slice(slices);
  if (s < 0) return;
  const int lane = threadIdx.x % kWave;
  const bool on = lane < kSliceVec;
  const int base = lane - lane % 5;
  const int at = on ? lane : kSliceVec - 1;
  const long long v = static_cast<long long>(kSliceVec) * s + at;
  const double xq = x[v];
  double r = 0.0;
#pragma unroll
  for (int j = 0; j < 5; ++j) {
    const double a = diag[static_cast<long long>(kSliceBlock) * s + kSliceVec * j + at];
    r += a * __shfl(xq, (base + j) % kWave);
  }
  r = impl_slots<true>(rows, s, lane, offd, x, r);
  if (on) y[v] = r;
}

// A block's exact sum in LDS: kReplicas copies of the words, lane l adding to copy l mod 32, so that a
// wave's terms (whose limbs are mostly the same few) meet two at a time on an address, and no lane
// waits on another. The copies of a word lie one after the other with one place left empty, so that
// the words' final sums read different banks. Summing each limb across the wave in registers instead
// took about 230 instructions a term and made these kernels bound by them: a Gram-Schmidt launch on
// 198k values 26 us on average and 12.5 now, on 5.2M values 72 and 59 (5 TB/s).
constexpr int kReplicas = 32;
constexpr int kReplicaRow = kReplicas + 1;
struct ImplSum {
  long long copies[kWords * kReplicaRow];
  long long words[kWords];
};

__device__ __forceinline__ void impl_sum_clear(ImplSum& s) {
  for (int t = threadIdx.x; t < kWords * kReplicaRow; t += kBlock) s.copies[t] = 0;
}

// The term split into three 32-bit limbs from limb i, as exact_add_wave splits it.
__device__ __forceinline__ void impl_sum_add(ImplSum& s, double t) {
  const unsigned long long bits = static_cast<unsigned long long>(__double_as_longlong(t));
  if ((bits << 1) == 0) return;
  const int biased = static_cast<int>((bits >> 52) & 0x7ff);
  const unsigned long long fraction = bits & ((1ULL << 52) - 1);
  const bool negative = (bits >> 63) != 0;
  unsigned long long* col = reinterpret_cast<unsigned long long*>(s.copies) + threadIdx.x % kReplicas;
  if (biased == 0x7ff) {
    atomicAdd(col + (fraction != 0 ? kLimbs + 2 : (negative ? kLimbs + 1 : kLimbs)) * kReplicaRow, 1ULL);
    return;
  }
  const unsigned long long m = biased == 0 ? fraction : (fraction | (1ULL << 52));
  const int p = (biased == 0 ? -1074 : biased - 1075) + 1088;
  const int sh = p & 31;
  const unsigned long long lo = (m & 0xffffffffULL) << sh, hi = (m >> 32) << sh;
  unsigned long long part[3] = {lo & 0xffffffffULL, (lo >> 32) + (hi & 0xffffffffULL), hi >> 32};
  col += (p >> 5) * kReplicaRow;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    if (part[k] != 0) atomicAdd(col + k * kReplicaRow, negative ? 0ULL - part[k] : part[k]);
  }
}

// The block's N sums added into their global words.
template <int N>
__device__ __forceinline__ void impl_sum_flush(ImplSum* s, long long* const* words) {
  static_assert(N * 128 <= kBlock && kWords <= 128);
  __syncthreads();
  const int n = threadIdx.x / 128, t = threadIdx.x % 128;
  if (n < N && t < kWords) {
    long long v = 0;
#pragma unroll 8
    for (int r = 0; r < kReplicas; ++r) v += s[n].copies[t * kReplicaRow + r];
    s[n].words[t] = v;
  }
  __syncthreads();
  if (n < N && t < kWords) {
    const long long v = carried_word(s[n].words, t);
    if (v != 0) atomicAdd(reinterpret_cast<unsigned long long*>(words[n] + t), static_cast<unsigned long long>(v));
  }
}

// r /= s, s the number of these bits, and sum_i r_i r_i over the m values as exact words (added into
// `words`, cleared beforehand): each product rounded to FP64, then added exactly. Grid-stride.
__global__ __launch_bounds__(kBlock) void k_impl_scale_dot(double* __restrict__ r, long long m,
                                                           const unsigned long long* __restrict__ scale_bits,
                                                           long long* __restrict__ words) {
  __shared__ ImplSum acc[1];
  impl_sum_clear(acc[0]);
  const double s = __longlong_as_double(static_cast<long long>(*scale_bits));
  __syncthreads();
  const long long stride = static_cast<long long>(gridDim.x) * kBlock;
  for (long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i < m; i += stride) {
    const double v = r[i] / s;
    r[i] = v;
    impl_sum_add(acc[0], v * v);
  }
  long long* out[1] = {words};
  impl_sum_flush<1>(acc, out);
}

// The GCR's modified Gram-Schmidt step fused with the inner products that follow it: when zj is
// given, beta = (w, w_j) / (w_j, w_j) from the words of the last inner product and the device's
// (w_j, w_j) (each block rounds them with exact_value), z -= beta zj and w -= beta wj; then sum
// w_i p_i into wp and, with two SUMS, sum w_i q_i into wq, each over the updated w. The sums are
// exact, so fusing them changes no bit.
template <int SUMS>
__global__ __launch_bounds__(kBlock) void k_impl_orth_dots(double* __restrict__ z, double* w,
                                                           const double* __restrict__ zj,
                                                           const double* __restrict__ wj, long long m,
                                                           const long long* __restrict__ beta_words,
                                                           const double* __restrict__ beta_den,
                                                           const double* p, long long* __restrict__ wp,
                                                           const double* __restrict__ q, long long* __restrict__ wq) {
  __shared__ ImplSum acc[SUMS];
  __shared__ double beta_sh;
#pragma unroll
  for (int n = 0; n < SUMS; ++n) impl_sum_clear(acc[n]);
  if (zj != nullptr && threadIdx.x < kWave) {
    const double v = exact_value_wave(beta_words) / *beta_den;
    if (threadIdx.x == 0) beta_sh = v;
  }
  __syncthreads();
  const double beta = zj != nullptr ? beta_sh : 0.0;
  const long long stride = static_cast<long long>(gridDim.x) * kBlock;
  for (long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i < m; i += stride) {
    double wi = w[i];
    if (zj != nullptr) {
      z[i] -= beta * zj[i];
      wi -= beta * wj[i];
      w[i] = wi;
    }
    // p may be w itself ((w, w) after the step): its value here is the updated one.
    impl_sum_add(acc[0], wi * (p == w ? wi : p[i]));
    if constexpr (SUMS == 2) impl_sum_add(acc[1], wi * q[i]);
  }
  long long* out[2] = {wp, wq};
  impl_sum_flush<SUMS>(acc, out);
}

// The GCR's update fused with the scalars before it and the inner product after it: each block
// rounds (w, w) and alpha = (r, w) / (w, w) from their words (block 0 stores (w, w) for the host and
// the next directions), then, when (w, w) > 0 (else the GCR stops before its update), x += sa z
// (sa = scale * alpha, scale the residual's largest magnitude from its bits) and r -= alpha w;
// then sum r_i r_i into words.
__global__ __launch_bounds__(kBlock) void k_impl_advance_dot(double* __restrict__ x, double* __restrict__ r,
                                                             const double* __restrict__ z,
                                                             const double* __restrict__ w, long long m,
                                                             const unsigned long long* __restrict__ scale_bits,
                                                             const long long* __restrict__ ww_words,
                                                             const long long* __restrict__ rw_words,
                                                             double* __restrict__ ww_out,
                                                             long long* __restrict__ words) {
  __shared__ ImplSum acc[1];
  __shared__ double product[2];
  impl_sum_clear(acc[0]);
  if (threadIdx.x < 2 * kWave) {  // one wave per product
    const double v = exact_value_wave(threadIdx.x < kWave ? ww_words : rw_words);
    if (threadIdx.x % kWave == 0) product[threadIdx.x / kWave] = v;
    if (threadIdx.x == 0 && blockIdx.x == 0) *ww_out = v;
  }
  __syncthreads();
  const bool update = product[0] > 0.0;
  const double alpha = product[1] / product[0];
  const double sa = __longlong_as_double(static_cast<long long>(*scale_bits)) * alpha;
  const long long stride = static_cast<long long>(gridDim.x) * kBlock;
  for (long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i < m; i += stride) {
    double ri = r[i];
    if (update) {
      x[i] += sa * z[i];
      ri -= alpha * w[i];
      r[i] = ri;
    }
    impl_sum_add(acc[0], ri * ri);
  }
  long long* out[1] = {words};
  impl_sum_flush<1>(acc, out);
}

// What a solve leaves besides its sums: bits[0] the admissible fraction's minimum, bits[1] the residual's
// largest entry, bits[2] the least cell with a singular diagonal block.
constexpr int kImplBits = 3;
__device__ __host__ inline int* impl_singular(unsigned long long* bits) { return reinterpret_cast<int*>(bits + 2); }

// Clears n exact-sum words and sets the fraction to 1.0's bits, the largest entry's to 0 and the
// singular cell to INT32_MAX.
__global__ void k_impl_clear(long long* __restrict__ words, int n, unsigned long long* __restrict__ bits) {
  for (int t = threadIdx.x; t < n; t += blockDim.x) words[t] = 0;
  if (threadIdx.x == 0) {
    bits[0] = static_cast<unsigned long long>(__double_as_longlong(1.0));
    bits[1] = 0;
    *impl_singular(bits) = INT32_MAX;
  }
}

// EulerPhysics::pressure(c, a): the pressure of u + a du in FP64.
__device__ __forceinline__ double impl_pressure(const double* v0, const double* dv, double a, double gamma) {
  double v[5];
#pragma unroll
  for (int k = 0; k < 5; ++k) v[k] = v0[k] + a * dv[k];
  return (gamma - 1.0) * (v[4] - 0.5 * (v[1] * v[1] + v[2] * v[2] + v[3] * v[3]) / v[0]);
}

constexpr double kImplMaxDecrease = 0.5;
constexpr double kImplMinStep = 1e-6;

// Each cell's admissible fraction (its density bound, then halved until its pressure bound holds),
// and their least as the bits of a non-negative double (atomicMin of the bits).
__global__ __launch_bounds__(kBlock) void k_impl_admissible(const double* __restrict__ u,
                                                            const double* __restrict__ du,
                                                            const int* __restrict__ rank, int n, double gamma,
                                                            unsigned long long* __restrict__ bits) {
  const int c = blockIdx.x * kBlock + threadIdx.x;
  unsigned long long key = ~0ULL;
  if (c < n) {
    const long long at = 5LL * rank[c];
    double v0[5], dv[5];
#pragma unroll
    for (int k = 0; k < 5; ++k) {
      v0[k] = u[static_cast<long long>(k) * n + c];
      dv[k] = du[at + k];
    }
    double a = 1.0;
    if (dv[0] < 0.0) {
      const double b = kImplMaxDecrease * v0[0] / -dv[0];
      a = b < a ? b : a;  // std::min(a, b): b when b < a
    }
    const double p = impl_pressure(v0, dv, 0.0, gamma);
    while (a >= kImplMinStep && !(impl_pressure(v0, dv, a, gamma) >= (1.0 - kImplMaxDecrease) * p)) a *= 0.5;
    key = static_cast<unsigned long long>(__double_as_longlong(a));
  }
  // *bits starts at 1.0's, so a wave whose cells all take the full step has nothing to lower (one atomic
  // per wave on that address took 188 us on 1.03M cells).
  key = wave_min(key);
  if ((threadIdx.x % kWave) == 0 && key < static_cast<unsigned long long>(__double_as_longlong(1.0))) atomicMin(bits, key);
}

// The Krylov operator's boundary term (EulerPhysics::add_boundary_gradient_term with
// Euler::gradient_tangent, physics/src/euler_physics.cpp:1300-1320, physics/src/euler.cpp:1081-1119):
// y += B v, the boundary faces' fluxes' derivative through the reconstruction's gradients, which
// the assembled blocks drop. Per cell owning a boundary face (`cells`, ascending): the
// primitive tangents dW = dW/dq v of the cell and its stencil cells (the direction rounded to the
// compute type, the products summed in it; k_impl_tangents, for the cells `near` lists), the gradient's
// tangent sum_k (dW_k - dW_c) w_k (FP64 sums, boundary values held), then over its boundary faces in
// cell_faces order, where the reconstruction did not fall back to the cell value, bnd_jac applied to
// phi (grad_tan . r), and on warped slip and wall faces the wall-warp term's tangent phi_p M^T grad_tan p.
// dwdu cell-major (25 c + 5 i + j), v by position (5 p + j).
template <class C>
__device__ __forceinline__ void impl_tangent(const double* __restrict__ dwdu, const double* __restrict__ v, long long c,
                                             long long p, C* dw) {
  C vc[5];
#pragma unroll
  for (int j = 0; j < 5; ++j) vc[j] = static_cast<C>(v[5 * p + j]);
#pragma unroll
  for (int i = 0; i < 5; ++i) {
    C t = C(0);
#pragma unroll
    for (int j = 0; j < 5; ++j) t = t + static_cast<C>(dwdu[25 * c + 5 * i + j]) * vc[j];
    dw[i] = t;
  }
}

// Marks the listed cells and the cells of their gradient stencils: those whose tangents the boundary term
// reads. Threads that mark one cell write the same byte.
template <class C>
__global__ __launch_bounds__(kBlock) void k_impl_near(Dev<C> d, const int* __restrict__ cells, int count,
                                                      unsigned char* __restrict__ mark) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= count) return;
  const int c = cells[t];
  mark[c] = 1;
  const long long at = d.soff[c / kWave] + c % kWave;
  const int len = d.slen[c];
  for (int j = 0; j < len; ++j) {
    const int e = d.sidx[at + static_cast<long long>(j) * kWave];
    if (e >= 0) mark[e] = 1;
  }
}

// The primitive tangent dW/dq v (impl_tangent) of the listed cells, 5 consecutive values per cell in the
// compute type, for the boundary term's stencils.
template <class C>
__global__ __launch_bounds__(kBlock) void k_impl_tangents(const double* __restrict__ dwdu, const double* __restrict__ v,
                                                          const int* __restrict__ rank, const int* __restrict__ near,
                                                          int count, C* __restrict__ out) {
  const int t = blockIdx.x * kBlock + threadIdx.x;
  if (t >= count) return;
  const int c = near[t];
  C dw[5];
  impl_tangent<C>(dwdu, v, c, rank[c], dw);
#pragma unroll
  for (int i = 0; i < 5; ++i) out[5LL * c + i] = dw[i];
}

// Five lanes per cell (12 cells per wave), lane i the tangents of variable i and then row i of the
// faces' blocks, eight stencil entries in flight. The few thousand boundary cells leave most of the GPU
// idle, so what counts is the chain of one cell's loads: with one thread per cell and one entry at a
// time this took 57 us on 7.7k cells, 26 now.
template <class C>
__global__ __launch_bounds__(kBlock) void k_impl_bgrad(Dev<C> d, const int* __restrict__ cells, int count,
                                                       const C* __restrict__ tangents, const double* __restrict__ bj,
                                                       const int* __restrict__ rank, double* __restrict__ y) {
  const int lane = threadIdx.x % kWave, wave = threadIdx.x / kWave;
  const int g = lane / 5, i = lane % 5, base = lane - i;
  const int t = (blockIdx.x * (kBlock / kWave) + wave) * kSlice + g;
  // Lanes without a cell (60 .. 63, and past the list) repeat the last one: every lane shuffles.
  const bool on = lane < kSliceVec && t < count;
  const int c = cells[t < count ? t : count - 1];
  const Params<C>& pa = d.ptab[cell_case(d, c)];
  const C dwc = tangents[5LL * c + i];
  double acc[3] = {0.0, 0.0, 0.0};
  const long long at = d.soff[c / kWave] + (c % kWave);
  const int len = d.slen[c];
  constexpr int kEntries = 8;
  for (int j = 0; j < len; j += kEntries) {
    int e[kEntries];
    C w[kEntries][3], dwn[kEntries];
#pragma unroll
    for (int u = 0; u < kEntries; ++u) {
      const long long k = at + static_cast<long long>(j + u < len ? j + u : len - 1) * kWave;
      e[u] = d.sidx[k];
      w[u][0] = d.sw0[k];
      w[u][1] = d.sw1[k];
      w[u][2] = d.sw2[k];
    }
#pragma unroll
    for (int u = 0; u < kEntries; ++u) {
      const C v = tangents[5LL * (e[u] >= 0 ? e[u] : c) + i];
      dwn[u] = e[u] >= 0 ? v : C(0);
    }
    // Past the cell's entries the last is read again and a zero added: a branch would have the
    // compiler move the loads behind it.
#pragma unroll
    for (int u = 0; u < kEntries; ++u) {
      const C dd = dwn[u] - dwc;
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        const double v = static_cast<double>(dd * w[u][q]);
        acc[q] += j + u < len ? v : 0.0;
      }
    }
  }
  C gt[3], gp[3];
#pragma unroll
  for (int q = 0; q < 3; ++q) gt[q] = static_cast<C>(acc[q]);
#pragma unroll
  for (int q = 0; q < 3; ++q) gp[q] = __shfl(gt[q], base + 4 < kWave ? base + 4 : lane);  // the pressure's
  const W5<C> w = load_w(d.prim, c);
  C rec[20];
  load_rec(d.rec, c, rec);
  const C* gc = rec;
  const C* pc = rec + 15;
  const C phi = i == 0 ? pc[0] : i == 1 ? pc[1] : i == 2 ? pc[2] : i == 3 ? pc[3] : pc[4];
  double dres = 0.0;
  // Every lane of a group takes the same faces; groups of unlike counts meet no shuffle of another's.
  for (int k = d.cfo[c]; k < d.cfo[c + 1]; ++k) {
    const int f = d.inc[k] & 0x7fffffff;
    if (f < d.ni) continue;
    const int b = f - d.ni;
    C g8[8];
    load_n<C, 8>(d.fgeo + 8LL * f, g8);
    const C r[3] = {g8[4], g8[5], g8[6]};
    const C d00 = gc[0] * r[0] + gc[1] * r[1] + gc[2] * r[2];
    const C d04 = gc[12] * r[0] + gc[13] * r[1] + gc[14] * r[2];
    const bool fell_back = !((w.r + pc[0] * d00) > C(0.0) && (w.p + pc[4] * d04) + pa.pref > C(0.0));
    if (fell_back) continue;
    const C dwf = phi * (gt[0] * r[0] + gt[1] * r[1] + gt[2] * r[2]);
    double s = 0.0;
#pragma unroll
    for (int j = 0; j < 5; ++j) {
      const double v = static_cast<double>(__shfl(dwf, (base + j) % kWave));
      s += bj[static_cast<long long>(5 * i + j) * d.nb + b] * v;
    }
    dres += s;
    const int kind = d.bkind[b];
    if (d.moment != nullptr && (kind == 2 || kind >= 5) && i >= 1 && i <= 3) {
      const long long n = d.nf;
      const C* m = d.moment + static_cast<long long>(i - 1) * n + f;
      dres += static_cast<double>(pc[4] * (m[0] * gp[0] + m[3 * n] * gp[1] + m[6 * n] * gp[2]));
    }
  }
  if (on) y[5LL * rank[c] + i] += dres;
}

// ---- the solve's start and end, on the state's layout

// r = -x and du = 0: x as the residual holds it (value q of cell c at q n + c), r and du by position (m
// values; an empty row's are 0); and the largest |r_i| into *largest as the bits of a non-negative
// double (their integer order is their order; a NaN's are above every number's), one atomic per block.
__global__ __launch_bounds__(kBlock) void k_impl_start(const double* __restrict__ x, const int* __restrict__ cell,
                                                       double* __restrict__ r, double* __restrict__ du, long long n,
                                                       long long m, unsigned long long* __restrict__ largest) {
  __shared__ unsigned long long wave_best[kBlock / kWave];
  unsigned long long best = 0;
  const long long stride = static_cast<long long>(gridDim.x) * kBlock;
  for (long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x; i < m; i += stride) {
    const int c = cell[i / 5];
    const double v = c >= 0 ? -x[(i % 5) * n + c] : 0.0;
    r[i] = v;
    du[i] = 0.0;
    const unsigned long long b = static_cast<unsigned long long>(__double_as_longlong(fabs(v)));
    best = b > best ? b : best;
  }
  best = wave_max(best);
  if (threadIdx.x % kWave == 0) wave_best[threadIdx.x / kWave] = best;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kBlock / kWave; ++w) best = wave_best[w] > best ? wave_best[w] : best;
    if (best != 0) atomicMax(largest, best);
  }
}

// u += alpha du, alpha the number of these bits, unless it is below the least step; u as the state holds
// it (value q of cell c at q n + c), du by position.
__global__ __launch_bounds__(kBlock) void k_impl_update(double* __restrict__ u, const double* __restrict__ du,
                                                        const int* __restrict__ rank, long long n,
                                                        const unsigned long long* __restrict__ alpha_bits) {
  const double alpha = __longlong_as_double(static_cast<long long>(*alpha_bits));
  if (alpha < kImplMinStep) return;
  const long long i = static_cast<long long>(blockIdx.x) * kBlock + threadIdx.x;
  if (i < 5 * n) u[i] += alpha * du[5LL * rank[i % n] + i / n];
}

}  // namespace mxe
