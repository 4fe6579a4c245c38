// UDT decomposition (column-pivoted Householder QR) and rdivp on gfx950.
//
// Reference: udt_AVX_pivot! (linalg/UDT.jl:216-334) and rdivp! (linalg/real.jl:198-226).
//
// The reference picks, at every column step, the trailing column of largest 2-norm
// (recomputed exactly, strict ">" so the first maximum wins), applies one Householder
// reflector at a time (BLAS-2), then accumulates Q backwards, sets D = |diag R| (0 -> 1)
// and T = D^-1 R, column-permuted (apply_pivot) or left "dirty upper" for rdivp.
//
// GPU form (a short sequence of launches per batch of matrices):
//  * Blocked Householder with panels of w <= 16 columns factorised by one workgroup (one
//    wave per column), and the trailing matrix updated with the compact-WY block reflector
//    I - V T V^T by one wave per 16-column strip on the matrix cores, so the trailing
//    matrix is streamed once per panel instead of once per column.  The same launch
//    accumulates Q = H_1 ... H_P forward on 16-row strips of U (U <- U (I - V T V^T),
//    the first panel's launch starting from the identity without reading U), so Q needs
//    no launches of its own.
//  * Pivoting: at every panel start the trailing columns' residual norms are recomputed
//    exactly and the w largest (first index wins ties) are moved to the front with the
//    reference's sequential swap semantics.  Inside a panel the order is kept.  This is
//    a column-pivoted QR whose pivot choices can differ from the reference's only where
//    the residual-norm order changes inside one panel; U D T reconstructs the input and
//    the Green's functions built from it agree with the reference's to ~1e-11 relative.
//  * Reflector convention as the reference: nu = copysign(||x||, x1), R_jj = -nu,
//    tau = (x1 + nu) / nu, v = x / (x1 + nu) with v_j = 1.
#include "common.h"

#include <vector>

namespace dqmc {

constexpr int kQrMaxW = 16;

// Wave64 sum of a double, result in every lane: butterflies inside each 16-lane row
// with DPP (quad_perm xor 1, xor 2, row_ror 4, row_ror 8), then the four row sums are
// combined through v_readlane.
template <int CTRL>
__device__ __forceinline__ double dpp_mov(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double readlane_d(double v, int l) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), l);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), l);
  return __hiloint2double(hi, lo);
}
__device__ __forceinline__ double wsum(double v) {
  v += dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_mov<0x124>(v);  // row_ror 4
  v += dpp_mov<0x128>(v);  // row_ror 8
  return (readlane_d(v, 0) + readlane_d(v, 16)) + (readlane_d(v, 32) + readlane_d(v, 48));
}

typedef double dx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dx4 mfma16(double a, double b, dx4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// The UDT runs as a sequence of launches per batch (one stream, so each sees the previous
// one's results): column norms; per panel a single-workgroup panel kernel (pivot choice,
// column moves, Householder factorisation of the panel) and a many-workgroup launch that
// forms the panel's compact-WY factor T, applies the block reflector to the trailing matrix
// and accumulates Q forward on U's rows (U <- U H); finally D and T.  Per-item state
// between launches: it.tau holds the residual norms, it.pivot the working permutation,
// it.tfac the taus of each panel.

// Panel width for `rows` remaining rows: one wave per column, the panel's reflectors held in
// LDS (width x rows doubles, at most 128 KB), so 16 columns up to 1024 rows and 8 beyond.
constexpr int kPanelWideRows = 1024;
__host__ __device__ static int udt_panel_width(int rows) {
  int w = rows <= kPanelWideRows ? kQrMaxW : kQrMaxW / 2;
  if (w > rows) w = rows;
  if (w < 1) w = 1;
  return w;
}

// TAB (all UDT and rdivp kernels): items from the device table batch.items with their own n
// and panel (many-chain launches), else from the kernel arguments (a separate instantiation
// for the one-chain path)
template <bool TAB>
__global__ __launch_bounds__(256) void udt_norms_kernel(UdtBatch batch) {
  constexpr bool tab = TAB;
  const UdtItem it = tab ? batch.items[blockIdx.y] : batch.it[blockIdx.y];
  const int n = tab ? it.n : batch.n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = blockIdx.x * 4 + wave;
  if (col >= n) return;  // per-wave work only: no workgroup barrier in this kernel
  const double* a = it.A + (size_t)col * n;
  double s = 0.0;
  for (int i0 = 0; i0 < n; i0 += 64 * 8) {
    double x[8];
#pragma unroll
    for (int q = 0; q < 8; q++) {
      const int i = i0 + 64 * q + lane;
      x[q] = i < n ? a[i] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < 8; q++) s += x[q] * x[q];
  }
  s = wsum(s);
  if (lane == 0) {
    it.tau[col] = s;
    it.pivot[col] = col;
  }
}

// (a, ia) comes before (b, ib): larger norm first, the lower column on ties.
__device__ __forceinline__ bool pivot_before(double a, int ia, double b, int ib) {
  return a > b || (a == b && ia < ib);
}

// Value of lane (lane ^ S).  Inside a 16-lane row with DPP: xor 1 and xor 2 are quad
// permutations, xor 4 a half-row mirror (i <-> 7 - i) followed by a quad reversal, xor 8
// a row rotation by 8.  Across rows with the gfx950 swaps of two registers (here two
// copies of x): permlane16_swap exchanges the odd rows of the first with the even rows of
// the second, so lanes of odd rows find lane - 16 in the first result and lanes of even
// rows lane + 16 in the second; permlane32_swap does the same with the two 32-lane halves.
template <int S>
__device__ __forceinline__ int lane_xor(int x) {
  if constexpr (S == 1) {
    return __builtin_amdgcn_update_dpp(0, x, 0xB1, 0xF, 0xF, false);    // quad_perm [1,0,3,2]
  } else if constexpr (S == 2) {
    return __builtin_amdgcn_update_dpp(0, x, 0x4E, 0xF, 0xF, false);    // quad_perm [2,3,0,1]
  } else if constexpr (S == 4) {
    const int m = __builtin_amdgcn_update_dpp(0, x, 0x141, 0xF, 0xF, false);  // row_half_mirror
    return __builtin_amdgcn_update_dpp(0, m, 0x1B, 0xF, 0xF, false);    // quad_perm [3,2,1,0]
  } else if constexpr (S == 8) {
    return __builtin_amdgcn_update_dpp(0, x, 0x128, 0xF, 0xF, false);   // row_ror 8
  } else if constexpr (S == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
    return (__lane_id() & 16) ? (int)r[0] : (int)r[1];
  } else {
    static_assert(S == 32, "lane_xor: strides 1 .. 32");
    const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
    return (__lane_id() & 32) ? (int)r[0] : (int)r[1];
  }
}

template <int S>
__device__ __forceinline__ double lane_xor_d(double x) {
  const int lo = lane_xor<S>(__double2loint(x));
  const int hi = lane_xor<S>(__double2hiint(x));
  return __hiloint2double(hi, lo);
}

template <int SIZE, int STRIDE>
__device__ __forceinline__ void bitonic_stage(double& kv, int& ki, int lane) {
  const int lo = lane_xor<STRIDE>(__double2loint(kv));
  const int hi = lane_xor<STRIDE>(__double2hiint(kv));
  const double pv = __hiloint2double(hi, lo);
  const int pi = lane_xor<STRIDE>(ki);
  const bool up = (lane & SIZE) == 0 || SIZE == 64;
  const bool lower = (lane & STRIDE) == 0;
  const bool pb = pivot_before(pv, pi, kv, ki);
  const bool take = lower == up ? pb : !pb;
  kv = take ? pv : kv;
  ki = take ? pi : ki;
  if constexpr (STRIDE > 1) bitonic_stage<SIZE, STRIDE / 2>(kv, ki, lane);
}

// Bitonic sort of one (norm, column) pair per lane of a wave into pivot order.
__device__ __forceinline__ void bitonic64(double& kv, int& ki, int lane) {
  bitonic_stage<2, 1>(kv, ki, lane);
  bitonic_stage<4, 2>(kv, ki, lane);
  bitonic_stage<8, 4>(kv, ki, lane);
  bitonic_stage<16, 8>(kv, ki, lane);
  bitonic_stage<32, 16>(kv, ki, lane);
  bitonic_stage<64, 32>(kv, ki, lane);
}

// Sum of a double over the wave, wave-uniform: butterflies inside each 16-lane row, then the
// row totals through row_bcast 15 (rows 1 and 3 take the row below) and row_bcast 31 (rows 2
// and 3 take lane 31), so lane 63 holds the total.
__device__ __forceinline__ double wave_total(double v) {
  v += dpp_mov<0xB1>(v);   // quad_perm [1,0,3,2]
  v += dpp_mov<0x4E>(v);   // quad_perm [2,3,0,1]
  v += dpp_mov<0x124>(v);  // row_ror 4
  v += dpp_mov<0x128>(v);  // row_ror 8
  {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x142, 0xA, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x142, 0xA, 0xF, false);
    v += __hiloint2double(hi, lo);
  }
  {
    const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), 0x143, 0xC, 0xF, false);
    const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), 0x143, 0xC, 0xF, false);
    v += __hiloint2double(hi, lo);
  }
  return readlane_d(v, 63);
}

// nu = copysign(||x||, x1), xi = x1 + nu and g = 1 / (nu xi) from normu = ||x||^2 > 0, so that
// H a = a - u (u^T a) g with u = (xi, x_2, x_3, ...).  Inside a range where nothing can overflow
// or turn subnormal the root comes from the hardware estimate by Goldschmidt's iteration and the
// reciprocal by Newton's (each to the last bits of a double); outside, where nu xi need not have a
// finite reciprocal, g = -xi / nu = -tau, and H a = a - v tau (v^T a) with v = u / xi.
__device__ __forceinline__ void reflector_scalars(double normu, double x1, double& nu, double& xi, double& g) {
  if (__builtin_expect(normu >= 0x1p-900 && normu <= 0x1p900, 1)) {
    const double y = __builtin_amdgcn_rsq(normu);
    double s = normu * y, h = 0.5 * y;
    const double r = fma(-s, h, 0.5);
    s = fma(s, r, s);
    h = fma(h, r, h);
    s = fma(fma(-s, s, normu), h, s);
    s = fma(fma(-s, s, normu), h, s);
    nu = copysign(s, x1);
    xi = x1 + nu;
    const double den = fma(fabs(x1), s, normu);    // nu xi
    double q = __builtin_amdgcn_rcp(den);
    q = fma(fma(-den, q, 1.0), q, q);
    q = fma(fma(-den, q, 1.0), q, q);
    g = q;
  } else {
    nu = copysign(sqrt(normu), x1);
    xi = x1 + nu;
    g = -(xi / nu);
  }
}

// LDS of a panel workgroup of NWV waves and RT rows per lane: the published columns (the pivot
// choice's candidate lists alias them), the steps' scalars, the progress counters, the choice.
template <int RT, int NWV>
constexpr size_t panel_lds() { return (size_t)NWV * 64 * RT * 8 + 32 * 8 + 4 * 4 + 16 * 4; }

// The w largest residual norms of columns [p0, n) in order, ties to the lower column
// (reference: strict ">"), into selr.  Every 64 columns are sorted by one wave, which keeps
// their best 16; groups of four such lists are merged until one is left.  With the odd lists of
// a group stored reversed, the 64 candidates are in the state the bitonic network reaches after
// its size-16 stage, so a merge is its size-32 and size-64 stages.  A NaN norm orders as the
// largest and is counted as a device error.
template <int RT, int NWV>
__device__ __forceinline__ void panel_choice(const UdtItem& it, int n, int p0, int w, int lane, int wave, double* cv,
                                             int* selr) {
  constexpr int kLists = RT < 4 ? 4 : RT;            // RT lists, padded to whole groups of four
  constexpr int kMerged = kLists <= 4 ? 0 : kLists <= 16 ? 4 : 8 + 4;   // lists of the later levels
  static_assert((kLists + kMerged) * 16 * 12 <= NWV * 64 * RT * 8, "lists fit the columns they alias");
  int* ci = reinterpret_cast<int*>(cv + (kLists + kMerged) * 16);
  for (int l = wave; l < kLists; l += NWV) {
    const int k = p0 + 64 * l + lane;
    double kv = k < n ? it.tau[k] : -HUGE_VAL;
    int ki = k;
    const bool bad = kv != kv;
    if (bad) kv = HUGE_VAL;
    if (__ballot(bad) && lane == 0 && it.err) atomicAdd(it.err, 1ull);
    if (p0 + 64 * l < n) bitonic64(kv, ki, lane);    // (an empty list is in order)
    if (RT == 1) {
      if (l == 0 && lane < 16) selr[lane] = lane < w ? ki : p0;
    } else if (lane < 16) {
      const int slot = l * 16 + ((l & 1) ? 15 - lane : lane);
      cv[slot] = kv;
      ci[slot] = ki;
    }
  }
  __syncthreads();
  if constexpr (RT > 1) {
    int base = 0;
#pragma unroll
    for (int lists = kLists; lists > 1;) {
      const int groups = lists / 4, pad = groups > 1 ? (groups + 3) / 4 * 4 : 1;
      for (int m = wave; m < pad; m += NWV) {
        double kv = -HUGE_VAL;
        int ki = n + 4096 + m * 64 + lane;
        if (m < groups) {
          kv = cv[base + m * 64 + lane];
          ki = ci[base + m * 64 + lane];
          bitonic_stage<32, 16>(kv, ki, lane);
          bitonic_stage<64, 32>(kv, ki, lane);
        }
        if (pad == 1) {
          if (lane < 16) selr[lane] = lane < w ? ki : p0;
        } else if (lane < 16) {
          const int slot = base + lists * 16 + m * 16 + ((m & 1) ? 15 - lane : lane);
          cv[slot] = kv;
          ci[slot] = ki;
        }
      }
      __syncthreads();
      base += lists * 16;
      lists = pad;
    }
  }
}

// Householder panel of one item: pivot choice, column moves, factorisation, the taus.
//
// One wave per panel column (lane l holds rows l + 64 k, k < RT), so a column step is a few
// instructions per wave and the waves' work runs beside each other.  Column j, once final, is
// published in LDS (x below its diagonal, zero elsewhere); every later column's wave forms its
// x^T a while column j's wave forms ||x||^2 and the scalars, and then applies
//   a <- a - u (u^T a) g,  u = (xi, x), g = 1 / (nu xi)   (reflector_scalars, with its form for
// squared norms next to the ends of the range; marked unlikely, which keeps that form off the straight
// path: 16x16 sites 51.2 -> 50.8 ms per sweep).
// A column's wave depends only on lower columns' waves of the same workgroup, in order, so the
// waits end; the chain is 16 steps of one reduction, one root and one reciprocal.
// What bounds it is that chain's latency, and beside it the issue slots of the 16 waves on four
// SIMDs.  Against one wave for all columns (up to 256 rows) and four waves with a barrier per step
// and an n^2 count for the choice (above), per launch, one or two matrices:
//   1024 rows 183 -> 21 us, 512 rows 77 -> 16 us, 256 rows 19.8 -> 14.0 us, 64 rows 19 -> 12.5 us;
// a sweep of 32x32 sites 382 -> 230 ms, 24x24 323 -> 215 ms, 16x16 72.6 -> 66.8 ms.
//
// The swaps of the reference ("slot p0 + t <-> slot that holds choice t", t = 0, 1, ...) leave
// choice t in slot p0 + t.  A panel column that was not chosen ends in the slot of a choice from
// outside the panel: the path choice t -> the choice that was column p0 + t -> ... ends at it,
// since every swap stays among the slots and columns of one such path.  Waves 0 to 3, done with
// their columns first, move the columns; a row is moved by one lane, which reads all its sources
// before it writes.
template <int RT, int NWV>
__device__ __forceinline__ void panel_body(const UdtItem& it, int n, int p0, int w, int last, unsigned char* smem) {
  constexpr int LR = 64 * RT;
  const int rows = n - p0;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double* V = reinterpret_cast<double*>(smem);   // [NWV][LR] published columns
  double* scal = V + NWV * LR;                   // [16][2] xi, g of each step
  int* pub = reinterpret_cast<int*>(scal + 32);  // [0] columns published, [1] steps' scalars published
  int* selr = pub + 4;                           // [16] the choice
  double* __restrict__ A = it.A;

  if (tid < 2) pub[tid] = 0;
  panel_choice<RT, NWV>(it, n, p0, w, lane, wave, V, selr);

  const int c = wave;
  double a[RT];
  if (c < w) {
    const double* src = A + (size_t)p0 + (size_t)selr[c] * n;
#pragma unroll
    for (int k = 0; k < RT; k++) {
      const int i = lane + 64 * k;
      a[k] = src[i < rows ? i : rows - 1];
    }
#pragma unroll
    for (int k = 0; k < RT; k++) a[k] = lane + 64 * k < rows ? a[k] : 0.0;
  }
  // movers: lane e < w: choice e and, if it comes from outside the panel, the column that
  // takes its slot
  constexpr int kMovers = 4;
  int sel = p0, out = -1;
  if (wave < kMovers) {
    const int le = lane & 15;
    sel = le < w ? selr[le] : p0 + le;
    int nxt = le;                                // the choice that was column p0 + le (else le)
#pragma unroll
    for (int t = 0; t < kQrMaxW; t++) nxt = __builtin_amdgcn_readlane(sel, t) == p0 + le ? t : nxt;
#pragma unroll
    for (int q = 0; q < 4; q++) nxt = __shfl(nxt, nxt, 64);
    if (le < w && sel >= p0 + w) out = p0 + nxt;
    if (wave == 0) {
      // the permutation: every entry is read before one is written
      const int pv0 = it.pivot[sel < n ? sel : n - 1];
      const int pv1 = out >= 0 ? it.pivot[out] : 0;
      if (lane < w) {
        it.pivot[p0 + lane] = pv0;
        if (out >= 0) it.pivot[sel] = pv1;
      }
    }
  }
  __syncthreads();   // the panel's sources are read (and the candidate lists free)

  double nu = 0.0, tau = 0.0, xi = 0.0, normu = 0.0;
  if (c < w) {
    for (int j = 0; j < c; j++) {
      if (j == c - 1) __builtin_amdgcn_s_setprio(3);   // the next column to be published
      while (__hip_atomic_load(pub, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= j) {}
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      double x[RT];
#pragma unroll
      for (int k = 0; k < RT; k++) x[k] = V[j * LR + lane + 64 * k];
      double s0 = x[0] * a[0], s1 = 0.0;
#pragma unroll
      for (int k = 1; k < RT; k++) {
        if (k & 1) s1 = fma(x[k], a[k], s1);
        else s0 = fma(x[k], a[k], s0);
      }
      const double tot = wave_total(s0 + s1);
      const double aj = readlane_d(a[0], j);
      while (__hip_atomic_load(pub + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) <= j) {}
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
      const double xj = scal[2 * j], g = scal[2 * j + 1];
      if (__builtin_expect(g > 0.0, 1)) {
        const double f = fma(aj, xj, tot) * g;
        a[0] = fma(-(lane == j ? xj : x[0]), f, a[0]);
#pragma unroll
        for (int k = 1; k < RT; k++) a[k] = fma(-x[k], f, a[k]);
      } else if (__builtin_expect(g != 0.0, 0)) {   // -tau (or NaN); 0: a zero column, H = I
        const double r = 1.0 / xj, f = -g * fma(tot, r, aj);
        a[0] = fma(-(lane == j ? 1.0 : x[0] * r), f, a[0]);
#pragma unroll
        for (int k = 1; k < RT; k++) a[k] = fma(-(x[k] * r), f, a[k]);
      }
    }
    // column c is final: x below the diagonal, then the scalars
    const double xc = lane > c ? a[0] : 0.0;
    if (c + 1 < w) {
      V[c * LR + lane] = xc;
#pragma unroll
      for (int k = 1; k < RT; k++) V[c * LR + lane + 64 * k] = a[k];
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if (lane == 0) __hip_atomic_store(pub, c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    double s0 = lane >= c ? a[0] * a[0] : 0.0, s1 = 0.0;
#pragma unroll
    for (int k = 1; k < RT; k++) {
      if (k & 1) s1 = fma(a[k], a[k], s1);
      else s0 = fma(a[k], a[k], s0);
    }
    normu = wave_total(s0 + s1);
    double g = 0.0;
    if (normu != 0.0) reflector_scalars(normu, readlane_d(a[0], c), nu, xi, g);
    if (c + 1 < w) {
      if (lane == 0) {
        scal[2 * c] = xi;
        scal[2 * c + 1] = g;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
      if (lane == 0) __hip_atomic_store(pub + 1, c + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    }
    __builtin_amdgcn_s_setprio(0);
    if (normu != 0.0) {
      tau = xi / nu;
      const double rxi = 1.0 / xi;
      a[0] = lane > c ? a[0] * rxi : (lane == c ? -nu : a[0]);
#pragma unroll
      for (int k = 1; k < RT; k++) a[k] *= rxi;
    }
  }
  if (wave < kMovers) {
    for (int r0 = 64 * wave; r0 < n; r0 += 64 * kMovers) {
      const int rr = r0 + lane, rc = rr < n ? rr : n - 1;
      double v[kQrMaxW], v2[kQrMaxW];
      const bool above = r0 < p0;              // (uniform) rows < p0: R's part of the panel columns
#pragma unroll
      for (int e = 0; e < kQrMaxW; e++) {
        const int d = __builtin_amdgcn_readlane(out, e), s = __builtin_amdgcn_readlane(sel, e);
        v[e] = A[(size_t)rc + (size_t)(d >= 0 ? d : p0) * n];
        if (above) v2[e] = A[(size_t)rc + (size_t)(e < w ? s : p0) * n];
      }
#pragma unroll
      for (int e = 0; e < kQrMaxW; e++) {
        const int d = __builtin_amdgcn_readlane(out, e), s = __builtin_amdgcn_readlane(sel, e);
        if (d >= 0 && rr < n) A[(size_t)rr + (size_t)s * n] = v[e];
        if (above && e < w && rr < p0) A[(size_t)rr + (size_t)(p0 + e) * n] = v2[e];
      }
    }
  }
  __syncthreads();   // the moves have read the panel's slots
  if (c < w) {
    double* dst = A + (size_t)p0 + (size_t)(p0 + c) * n;
#pragma unroll
    for (int k = 0; k < RT; k++) {
      const int i = lane + 64 * k;
      if (i < rows) dst[i] = a[k];
    }
    if (last && lane == c) {   // D = |diag R| (0 -> 1) of this panel
      const double x = fabs(a[0]);
      it.D[p0 + c] = x == 0.0 ? 1.0 : x;
    }
    if (lane == 0) it.tfac[(size_t)p0 * 16 + c] = tau;
  } else if (c < kQrMaxW) {
    if (lane == 0) it.tfac[(size_t)p0 * 16 + c] = 0.0;
  }
  if (NWV < kQrMaxW && tid < kQrMaxW - NWV) it.tfac[(size_t)p0 * 16 + NWV + tid] = 0.0;
  if (last) {
    // D = |diag R| (0 -> 1) of the earlier panels (final since their launches)
    for (int i = tid; i < p0; i += 64 * NWV) {
      const double x = fabs(A[(size_t)i + (size_t)i * n]);
      it.D[i] = x == 0.0 ? 1.0 : x;
    }
  }
}

// 16-column panels of at most 64 RT rows (one chain).
template <int RT>
__global__ __launch_bounds__(1024) void udt_panel_kernel(UdtBatch batch, int p0, int w, int last) {
  extern __shared__ __align__(16) unsigned char smem[];
  panel_body<RT, 16>(batch.it[blockIdx.x], batch.n, p0, w, last, smem);
}

// Item table: each item's own panel, rows per lane by its own size.
__global__ __launch_bounds__(1024) void udt_panel_tab_kernel(UdtBatch batch) {
  extern __shared__ __align__(16) unsigned char smem[];
  const UdtItem& it = batch.items[blockIdx.x];
  const int n = it.n, p0 = it.p0, w = it.w, last = it.last, rows = n - p0;
  if (rows <= 64) panel_body<1, 16>(it, n, p0, w, last, smem);
  else if (rows <= 128) panel_body<2, 16>(it, n, p0, w, last, smem);
  else if (rows <= 256) panel_body<4, 16>(it, n, p0, w, last, smem);
  else if (rows <= 512) panel_body<8, 16>(it, n, p0, w, last, smem);
  else panel_body<16, 16>(it, n, p0, w, last, smem);
}

// 8-column panels of 1025 to 2048 rows.
template <bool TAB>
__global__ __launch_bounds__(512) void udt_panel_tall_kernel(UdtBatch batch, int p0a, int wa, int lasta) {
  extern __shared__ __align__(16) unsigned char smem[];
  const UdtItem& it = TAB ? batch.items[blockIdx.x] : batch.it[blockIdx.x];
  panel_body<32, 8>(it, TAB ? it.n : batch.n, TAB ? it.p0 : p0a, TAB ? it.w : wa, TAB ? it.last : lasta, smem);
}

// One workgroup per 16-column strip: X[p0:n, strip] -= V op(T) V^T X[p0:n, strip].
// mode 0 = trailing update of A with T^T, plus the residual norms of the updated columns
// over rows >= p0 + w; mode 1 = Q accumulation into U with T.  The four waves split the
// 16-row blocks of the strip.  X is held in the f64 MFMA B/D layout (lane l: rows
// l/16 + 4r of a block, column l%16), which is at once the B operand of W = V^T X and
// the accumulator of X - V Y, so each block is loaded once; V is read in both
// orientations.  All loads of a group of blocks are issued before the first product.
constexpr int kReflRB = 4;   // 16-row blocks per wave and group

__device__ __forceinline__ double vpanel(const double* Vp, int n, int rows, int w, int i, int a) {
  if (a >= w || i >= rows || i < a) return 0.0;
  if (i == a) return 1.0;
  return Vp[(size_t)i + (size_t)a * n];
}

__device__ __forceinline__ void reflect_strip(const UdtItem& it, int n, int p0, int w, int cb, int mode,
                                              double (&red)[4][4][64], double (&sred)[4][4][64],
                                              double (&stm)[4][2][256], double (&nred)[4][16]) {
  const int rows = n - p0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const bool trans = mode != 1;
  const double* Vp = it.A + (size_t)p0 * n + p0;
  const int col = cb + li;
  const bool colok = col < n;
  const int colc = colok ? col : n - 1;
  // X[i][c] (i >= p0): column cb + c of A (mode 0) or of U (mode 1), or row cb + c of U
  // (mode 2: X = U^T, so X -= V T^T V^T X is U <- U - U V T V^T on those rows)
  const size_t xs = mode == 2 ? (size_t)n : 1;
  double* Xc = mode == 2 ? it.U + colc + (size_t)p0 * n : (mode == 0 ? it.A : it.U) + (size_t)colc * n + p0;
  // the first panel's Q strips start from the identity (U is not read; every column of the
  // strip is written)
  const bool ident = mode == 2 && p0 == 0;
  // the panel's taus (zero beyond w)
  double tz[16];
#pragma unroll
  for (int j = 0; j < 16; j++) tz[j] = it.tfac[(size_t)p0 * 16 + j];
  const int nblk = (rows + 15) / 16;
  const int ngroups = (nblk + 4 * kReflRB - 1) / (4 * kReflRB);
  double xb[kReflRB][4], vb[kReflRB][4], va[kReflRB][4];
  dx4 Wacc = dx4{0, 0, 0, 0};
  dx4 Sacc = dx4{0, 0, 0, 0};   // S = V^T V: vb is both operands
  for (int g = 0; g < ngroups; g++) {
#pragma unroll
    for (int q = 0; q < kReflRB; q++) {
      const int blk = g * 4 * kReflRB + wave + 4 * q;
#pragma unroll
      for (int kc = 0; kc < 4; kc++) {
        const int i = 16 * blk + 4 * kc + lk;
        const int ic = i < rows ? i : rows - 1;
        const double x = ident ? (ic == colc ? 1.0 : 0.0) : Xc[ic * xs];
        xb[q][kc] = (i < rows && colok) ? x : 0.0;
        vb[q][kc] = vpanel(Vp, n, rows, w, i, li);
      }
    }
    if (ngroups == 1) {      // the second product's operand, loaded with the first's
#pragma unroll
      for (int q = 0; q < kReflRB; q++) {
        const int blk = wave + 4 * q;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) va[q][kc] = vpanel(Vp, n, rows, w, 16 * blk + li, 4 * kc + lk);
      }
    }
#pragma unroll
    for (int q = 0; q < kReflRB; q++)
#pragma unroll
      for (int kc = 0; kc < 4; kc++) {
        Wacc = mfma16(vb[q][kc], xb[q][kc], Wacc);
        Sacc = mfma16(vb[q][kc], vb[q][kc], Sacc);
      }
  }
#pragma unroll
  for (int r = 0; r < 4; r++) {
    red[wave][r][lane] = Wacc[r];
    sred[wave][r][lane] = Sacc[r];
  }
  __syncthreads();
  dx4 Wt;
#pragma unroll
  for (int r = 0; r < 4; r++) Wt[r] = (red[0][r][lane] + red[1][r][lane]) + (red[2][r][lane] + red[3][r][lane]);
  // compact-WY factor T (upper triangular, 16 x 16, zero beyond w): H_1..H_w = I - V T V^T.
  // Every wave forms it on its own (no workgroup barrier): S row-major into the wave's
  // space, then lane i builds row i of T from its own earlier entries,
  // T[i][j] = -tau_j sum_{k=i}^{j-1} T[i][k] S[k][j] (T[i][k] = 0 for k < i, so the sum may
  // start at 0), with S[k][j] read from LDS, the same address in every lane.
  double ta[4];
  {
    double* Sm = stm[wave][0];
    double* Tm = stm[wave][1];
#pragma unroll
    for (int r = 0; r < 4; r++)
      Sm[(4 * r + lk) * 16 + li] = (sred[0][r][lane] + sred[1][r][lane]) + (sred[2][r][lane] + sred[3][r][lane]);
    __builtin_amdgcn_wave_barrier();
    double row[16];
#pragma unroll
    for (int j = 0; j < 16; j++) {
      double acc = 0.0;
#pragma unroll
      for (int k = 0; k < j; k++) acc += row[k] * Sm[k * 16 + j];
      double t = 0.0;
      if (lane < w && j < w) {
        if (j == lane) t = tz[j];
        else if (j > lane) t = -tz[j] * acc;
      }
      row[j] = t;
    }
    if (lane < 16) {
#pragma unroll
      for (int j = 0; j < 16; j++) Tm[lane * 16 + j] = row[j];
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int kc = 0; kc < 4; kc++) {
      const int kk = 4 * kc + lk;
      ta[kc] = trans ? Tm[kk * 16 + li] : Tm[li * 16 + kk];
    }
  }
  dx4 Y = dx4{0, 0, 0, 0};
#pragma unroll
  for (int kc = 0; kc < 4; kc++) Y = mfma16(ta[kc], Wt[kc], Y);

  double ss = 0.0;
  for (int g = 0; g < ngroups; g++) {
    if (ngroups > 1) {
#pragma unroll
      for (int q = 0; q < kReflRB; q++) {
        const int blk = g * 4 * kReflRB + wave + 4 * q;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) {
          const int i = 16 * blk + 4 * kc + lk;
          const int ic = i < rows ? i : rows - 1;
          const double x = ident ? (ic == colc ? 1.0 : 0.0) : Xc[ic * xs];
          xb[q][kc] = (i < rows && colok) ? x : 0.0;
        }
      }
#pragma unroll
      for (int q = 0; q < kReflRB; q++) {
        const int blk = g * 4 * kReflRB + wave + 4 * q;
#pragma unroll
        for (int kc = 0; kc < 4; kc++) va[q][kc] = vpanel(Vp, n, rows, w, 16 * blk + li, 4 * kc + lk);
      }
    }
#pragma unroll
    for (int q = 0; q < kReflRB; q++) {
      const int blk = g * 4 * kReflRB + wave + 4 * q;
      if (16 * blk < rows) {
        dx4 acc;
#pragma unroll
        for (int r = 0; r < 4; r++) acc[r] = xb[q][r];
#pragma unroll
        for (int kc = 0; kc < 4; kc++) acc = mfma16(-va[q][kc], Y[kc], acc);
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int i = 16 * blk + lk + 4 * r;
          if (i < rows && colok) {
            Xc[i * xs] = acc[r];
            if (i >= w) ss += acc[r] * acc[r];
          }
        }
      }
    }
  }
  if (mode == 0) {
    ss += lane_xor_d<16>(ss);
    ss += lane_xor_d<32>(ss);
    if (lk == 0) nred[wave][li] = ss;
    __syncthreads();
    if (tid < 16 && cb + tid < n)
      it.tau[cb + tid] = (nred[0][tid] + nred[1][tid]) + (nred[2][tid] + nred[3][tid]);
  }
}

// Panel p0's block reflector applied in one launch: workgroups [0, nA) update the trailing
// 16-column strips of A from column c0 (with residual norms), the rest accumulate Q on
// 16-row strips of U (U <- U H, forward: U holds H_1 ... H_k after panel k).
template <bool TAB>
__global__ __launch_bounds__(256) void udt_reflect_kernel(UdtBatch batch, int p0, int w, int c0, int nA) {
  __shared__ double red[4][4][64];
  __shared__ double sred[4][4][64];
  __shared__ double stm[4][2][256];
  __shared__ double nred[4][16];
  const int bx = blockIdx.x;
  if constexpr (TAB) {
    // item table: this item's own panel; workgroups beyond its strips leave at once
    const UdtItem& it = batch.items[blockIdx.y];
    const int n = it.n, c0i = it.p0 + it.w;
    const int nAi = c0i < n ? (n - c0i + 15) / 16 : 0, nQi = (n + 15) / 16;
    if (bx >= nAi + nQi) return;
    if (bx < nAi) reflect_strip(it, n, it.p0, it.w, c0i + 16 * bx, 0, red, sred, stm, nred);
    else reflect_strip(it, n, it.p0, it.w, 16 * (bx - nAi), 2, red, sred, stm, nred);
    return;
  }
  if (bx < nA) reflect_strip(batch.it[blockIdx.y], batch.n, p0, w, c0 + 16 * bx, 0, red, sred, stm, nred);
  else reflect_strip(batch.it[blockIdx.y], batch.n, p0, w, 16 * (bx - nA), 2, red, sred, stm, nred);
}

// T = D^-1 R (pivoted: column j of R goes to column pivot[j]; dirty: the strict lower part
// is copied), one wave per column.
template <bool TAB>
__global__ __launch_bounds__(256) void udt_finish_kernel(UdtBatch batch) {
  constexpr bool tab = TAB;
  const UdtItem it = tab ? batch.items[blockIdx.y] : batch.it[blockIdx.y];
  const int n = tab ? it.n : batch.n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = blockIdx.x * 4 + wave;
  if (j >= n) return;
  const double* __restrict__ A = it.A;
  double* To = it.T;
  const size_t cj = (size_t)j * n;
  if (batch.apply_pivot) {
    const size_t co = (size_t)it.pivot[j] * n;
    for (int i = lane; i < n; i += 64) {
      const double d = 1.0 / it.D[i];
      To[co + i] = j >= i ? d * A[cj + i] : 0.0;
    }
  } else {
    for (int i = lane; i < n; i += 64) {
      if (j >= i) {
        const double d = 1.0 / it.D[i];
        To[cj + i] = d * A[cj + i];
      } else if (To != A) {
        To[cj + i] = A[cj + i];
      }
    }
  }
}


int udt_plan_fixed(int n, int* starts, int* widths, int cap) {
  int np = 0;
  for (int p0 = 0; p0 < n;) {
    const int w = udt_panel_width(n - p0);
    if (np == cap) return -1;
    starts[np] = p0;
    widths[np] = w;
    np++;
    p0 += w;
  }
  return np;
}

void udt_plan(int n, std::vector<int>& starts, std::vector<int>& widths) {
  starts.clear();
  widths.clear();
  for (int p0 = 0; p0 < n;) {
    const int w = udt_panel_width(n - p0);
    starts.push_back(p0);
    widths.push_back(w);
    p0 += w;
  }
}

hipError_t udt_check(const UdtBatch& b) {
  if (b.count < 0 || b.count > kMaxUdtItems || b.n < 1 || b.n > 2048) return hipErrorInvalidValue;
  for (int k = 0; k < b.count; k++) {
    // U is written while A's reflectors are read: it must be its own buffer
    if (b.it[k].U == b.it[k].A || b.it[k].U == b.it[k].T) return hipErrorInvalidValue;
    if (b.apply_pivot && b.it[k].T == b.it[k].A) return hipErrorInvalidValue;  // pivoted T is written out of place
  }
  return hipSuccess;
}

hipError_t launch_udt_norms(const UdtBatch& b, hipStream_t s) {
  if (b.items) hipLaunchKernelGGL(udt_norms_kernel<true>, dim3((b.max_n + 3) / 4, b.count), dim3(256), 0, s, b);
  else hipLaunchKernelGGL(udt_norms_kernel<false>, dim3((b.n + 3) / 4, b.count), dim3(256), 0, s, b);
  return hipGetLastError();
}

template <int RT>
static void launch_panel_t(const UdtBatch& b, int p0, int w, int last, hipStream_t s) {
  hipLaunchKernelGGL(udt_panel_kernel<RT>, dim3(b.count), dim3(1024), (panel_lds<RT, 16>()), s, b, p0, w, last);
}

hipError_t launch_udt_panel(const UdtBatch& b, int p0, int w, int last, hipStream_t s) {
  const int rows = b.n - p0;
  if (rows < 1 || rows > 2048 || w < 1 || w > udt_panel_width(rows)) return hipErrorInvalidValue;
  if (rows <= 64) launch_panel_t<1>(b, p0, w, last, s);
  else if (rows <= 128) launch_panel_t<2>(b, p0, w, last, s);
  else if (rows <= 256) launch_panel_t<4>(b, p0, w, last, s);
  else if (rows <= 512) launch_panel_t<8>(b, p0, w, last, s);
  else if (rows <= kPanelWideRows) launch_panel_t<16>(b, p0, w, last, s);
  else
    hipLaunchKernelGGL(udt_panel_tall_kernel<false>, dim3(b.count), dim3(512), (panel_lds<32, 8>()), s, b, p0, w,
                       last);
  return hipGetLastError();
}

hipError_t launch_udt_reflect(const UdtBatch& b, int p0, int w, hipStream_t s) {
  const int c0 = p0 + w;
  const int nA = c0 < b.n ? (b.n - c0 + 15) / 16 : 0;
  const int nQ = (b.n + 15) / 16;
  hipLaunchKernelGGL(udt_reflect_kernel<false>, dim3(nA + nQ, b.count), dim3(256), 0, s, b, p0, w, c0, nA);
  return hipGetLastError();
}

hipError_t launch_udt_finish(const UdtBatch& b, hipStream_t s) {
  if (b.items) hipLaunchKernelGGL(udt_finish_kernel<true>, dim3((b.max_n + 3) / 4, b.count), dim3(256), 0, s, b);
  else hipLaunchKernelGGL(udt_finish_kernel<false>, dim3((b.n + 3) / 4, b.count), dim3(256), 0, s, b);
  return hipGetLastError();
}

// Panels of one launch share the kernel: 16 waves and columns, or the tall form.
int udt_rows_class(int rows) { return rows <= kPanelWideRows ? 1 : 8; }
int udt_width_for(int rows) { return udt_panel_width(rows); }

hipError_t launch_udt_panel_tab(const UdtBatch& b, int R, hipStream_t s) {
  if (!b.items || b.count < 1 || b.max_n < 1 || b.max_n > 2048) return hipErrorInvalidValue;
  if (R == 1) {
    // LDS for the tallest panel of the launch (an item of n sites in this class has at most
    // min(n, 1024) rows)
    const size_t lds = b.max_n <= 64 ? panel_lds<1, 16>()
                     : b.max_n <= 128 ? panel_lds<2, 16>()
                     : b.max_n <= 256 ? panel_lds<4, 16>()
                     : b.max_n <= 512 ? panel_lds<8, 16>() : panel_lds<16, 16>();
    hipLaunchKernelGGL(udt_panel_tab_kernel, dim3(b.count), dim3(1024), lds, s, b);
  } else if (R == 8) {
    hipLaunchKernelGGL(udt_panel_tall_kernel<true>, dim3(b.count), dim3(512), (panel_lds<32, 8>()), s, b, 0, 0, 0);
  } else {
    return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_udt_reflect_tab(const UdtBatch& b, int max_grid, hipStream_t s) {
  if (!b.items || b.count < 1 || max_grid < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(udt_reflect_kernel<true>, dim3(max_grid, b.count), dim3(256), 0, s, b, 0, 0, 0, 0);
  return hipGetLastError();
}

// The whole sequence on one stream (the chain's own path times the steps separately).
hipError_t launch_udt(const UdtBatch& b, hipStream_t s) {
  if (b.count == 0) return hipSuccess;
  hipError_t e = udt_check(b);
  if (e != hipSuccess) return e;
  std::vector<int> st, wd;
  udt_plan(b.n, st, wd);
  const int np = (int)st.size();
  if ((e = launch_udt_norms(b, s)) != hipSuccess) return e;
  for (int pi = 0; pi < np; pi++) {
    if ((e = launch_udt_panel(b, st[pi], wd[pi], pi == np - 1, s)) != hipSuccess) return e;
    if ((e = launch_udt_reflect(b, st[pi], wd[pi], s)) != hipSuccess) return e;
  }
  return launch_udt_finish(b, s);
}

// rdivp: A <- A[:, pivot] * triu(T)^-1 (only the upper triangle of T is read).
// Rows are independent.  Each wave owns 16 rows; for every 16-column panel J the
// coupling to the already solved columns, X_{<J} T_{<J,J}, is a 16 x 16 x j0 product on
// the matrix cores, then the 16 x 16 triangular block is solved by 16 lanes (one row each)
// in the reference's order: x_j = (o_j - sum_{k<j} x_k T_kj) / T_jj.
template <bool TAB>
__global__ __launch_bounds__(256) void rdivp_kernel(RdivpBatch batch) {
  constexpr bool tab = TAB;
  const RdivpItem it = tab ? batch.items[blockIdx.y] : batch.it[blockIdx.y];
  const int n = tab ? it.n : batch.n;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int li = lane & 15, lk = lane >> 4;
  const int r0 = blockIdx.x * 64 + wave * 16;
  __shared__ double Ysh[4][16][17];
  __shared__ double Tsh[4][16][17];
  if (r0 >= n) return;  // per-wave work only: no workgroup barrier below
  double* __restrict__ A = it.A;
  double* __restrict__ O = it.O;
  const double* __restrict__ T = it.T;
  const int* __restrict__ piv = it.pivot;
  {
    const int r = r0 + li;
    if (r < n)
      for (int j = lk; j < n; j += 4) O[(size_t)r + (size_t)j * n] = A[(size_t)r + (size_t)piv[j] * n];
  }
  __threadfence_block();
  for (int j0 = 0; j0 < n; j0 += 16) {
    const int w = n - j0 < 16 ? n - j0 : 16;
    dx4 acc = dx4{0, 0, 0, 0};
    const int ra = r0 + li;
    const int cb = j0 + li;
#pragma unroll 4
    for (int k0 = 0; k0 < j0; k0 += 4) {
      const int k = k0 + lk;
      const double av = ra < n ? A[(size_t)ra + (size_t)k * n] : 0.0;
      const double bv = cb < n ? T[(size_t)k + (size_t)cb * n] : 0.0;
      acc = mfma16(av, bv, acc);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const int row = mfma_row<double>(lane, r);
      const int gr = r0 + row, gc = j0 + li;
      Ysh[wave][row][li] = (gr < n && gc < n) ? O[(size_t)gr + (size_t)gc * n] - acc[r] : 0.0;
      const int tr = j0 + row;
      Tsh[wave][row][li] = (tr < n && gc < n) ? T[(size_t)tr + (size_t)gc * n] : 1.0;
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_s_waitcnt(0);
    if (lane < 16 && r0 + lane < n) {
      double x[16];
#pragma unroll
      for (int c = 0; c < 16; c++) {
        double v = Ysh[wave][lane][c];
#pragma unroll
        for (int cp = 0; cp < 16; cp++)
          if (cp < c) v -= x[cp] * Tsh[wave][cp][c];
        x[c] = v / Tsh[wave][c][c];
      }
#pragma unroll
      for (int c = 0; c < 16; c++)
        if (c < w) A[(size_t)(r0 + lane) + (size_t)(j0 + c) * n] = x[c];
    }
    __threadfence_block();
    __builtin_amdgcn_wave_barrier();
  }
}

// rdivp for kRdivpBlockMaxN < n <= kRdivpStripMaxN: four waves per 16-row strip, the strip in LDS.
// Per 16-column panel p:
//   the waves share Y = X_p - X_{<p} T_{<p,p} on the matrix cores (wave w takes k-steps w, w + 4,
//   ...) and then issue the loads of T's coupling column of panel p + 1;
//   wave 0 solves X_p T_pp = Y by substitution, row l % 16 in lane l (the quarters of the wave alike),
//   T_pp's entries read from LDS at one address for all lanes;
//   wave 1 brings T's diagonal block of panel p + 1 and its reciprocals to LDS beside it.
// What bounds a panel is the substitution's chain and the latency of T's column (16 lines per load,
// issued a solve ahead).  One matrix, n = 576 and 1024: one wave per strip 279 and 751 us; five waves,
// one of which inverts the next diagonal block for a product in place of the substitution, 204 and
// 568 us; this, four waves with all their registers (no spills), 170 and 439 us.  The product's residual
// also grows with the inverse's entries (one unit-diagonal block with normal entries of size 3: up to
// 2e-13 of |X| |T|, the substitution's 2e-16), and its 0 times infinity spoils columns that do not depend
// on an infinite entry.
// KS = 40 (n <= 640) or 64: k-steps of one wave per panel, at most.
static size_t rdivp_wide_lds_bytes(int n) {
  return ((size_t)n * 17 + 2 * 16 * 17 + 2 * 16 + 4 * 4 * 64 + 16 * 17) * 8 + (size_t)n * 4;
}

template <bool TAB, int KS>
__global__ __launch_bounds__(256) void rdivp_wide_kernel(RdivpBatch batch) {
  const RdivpItem it = TAB ? batch.items[blockIdx.y] : batch.it[blockIdx.y];
  const int n = TAB ? it.n : batch.n;
  const int r0 = blockIdx.x * 16;
  if (TAB && r0 >= n) return;   // item-table launches size the grid for the largest item
  const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, lk = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nb = (n + 15) / 16;
  extern __shared__ __align__(16) unsigned char smem[];
  double* X = reinterpret_cast<double*>(smem);          // [n][17]: X[j * 17 + row]
  double* Tsh = X + (size_t)n * 17;                     // [2][16][17]: diagonal blocks of even and odd panels
  double* rec = Tsh + 2 * 16 * 17;                      // [2][16]: their diagonals' reciprocals
  double* red = rec + 2 * 16;                           // [4 waves][4][64]
  double* Ysh = red + 4 * 4 * 64;                       // [16][17]: Y[row][col]
  int* pv = reinterpret_cast<int*>(Ysh + 16 * 17);
  double* __restrict__ A = it.A;
  const double* __restrict__ T = it.T;

  for (int j = tid; j < n; j += 256) pv[j] = it.pivot[j];
  __syncthreads();
  // the strip's pivoted input (thread: row tid % 16, columns tid / 16 + 16 q)
  const int grow = tid & 15, gcol = tid >> 4;
  const int grr = r0 + grow, grc = grr < n ? grr : n - 1;
  for (int jb = 0; jb < n; jb += 256) {
    double v[16];
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int j = jb + gcol + 16 * q;
      v[q] = A[(size_t)grc + (size_t)pv[j < n ? j : n - 1] * n];
    }
#pragma unroll
    for (int q = 0; q < 16; q++) {
      const int j = jb + gcol + 16 * q;
      if (j < n) X[(size_t)j * 17 + grow] = v[q];
    }
  }
  // wave 1: the diagonal block of panel p (lane: rows lk + 4 q of column li), the identity beyond n
  double ub[4];
  auto load_block = [&](int p) {
#pragma unroll
    for (int q = 0; q < 4; q++) {
      const int ra = 16 * p + lk + 4 * q, cc = 16 * p + li;
      const double v = T[(size_t)(ra < n ? ra : n - 1) + (size_t)(cc < n ? cc : n - 1) * n];
      ub[q] = ra < n && cc < n ? v : (lk + 4 * q == li ? 1.0 : 0.0);
    }
  };
  auto store_block = [&](int p) {
    double* Tp = Tsh + (size_t)(p & 1) * 16 * 17;
    double d = 1.0;
#pragma unroll
    for (int q = 0; q < 4; q++) {
      Tp[(lk + 4 * q) * 17 + li] = ub[q];
      d = lk + 4 * q == li ? ub[q] : d;
    }
    if (lk == (li & 3)) rec[(p & 1) * 16 + li] = 1.0 / d;
  };
  // T's coupling column of panel j0 for this wave's k-steps q = wave + 4 s (4 q < j0)
  double tb[KS];
  auto load_tb = [&](int j0) {
    const int cb = j0 + li, cbc = cb < n ? cb : n - 1;
#pragma unroll
    for (int g = 0; g < KS / 8; g++)
      if (128 * g < j0) {
#pragma unroll
        for (int s = 8 * g; s < 8 * g + 8; s++) {
          const int k = 4 * (wave + 4 * s) + lk;
          tb[s] = T[(size_t)(k < j0 ? k : 0) + (size_t)cbc * n];
        }
      }
  };
  if (wave == 1) {
    load_block(0);
    store_block(0);
    if (nb > 1) load_block(1);
  }
  if (nb > 1) load_tb(16);
  __syncthreads();
  for (int p = 0; p < nb; p++) {
    const int j0 = 16 * p;
    dx4 acc = dx4{0, 0, 0, 0};
#pragma unroll
    for (int g = 0; g < KS / 8; g++)
      if (128 * g < j0) {
#pragma unroll
        for (int s = 8 * g; s < 8 * g + 8; s++) {
          const int q = wave + 4 * s;
          if (4 * q < j0) acc = mfma16(X[(size_t)(4 * q + lk) * 17 + li], tb[s], acc);
        }
      }
#pragma unroll
    for (int r = 0; r < 4; r++) red[(wave * 4 + r) * 64 + lane] = acc[r];
    if (p >= 1 && p + 1 < nb) load_tb(j0 + 16);
    __syncthreads();
    if (wave == 0) {
      const int cb = j0 + li;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = mfma_row<double>(lane, r);
        const double u = (red[r * 64 + lane] + red[(4 + r) * 64 + lane]) +
                         (red[(8 + r) * 64 + lane] + red[(12 + r) * 64 + lane]);
        Ysh[row * 17 + li] = cb < n ? X[(size_t)cb * 17 + row] - u : 0.0;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      const double* Tp = Tsh + (size_t)(p & 1) * 16 * 17;
      const double dl = Tp[li * 17 + li], yl = rec[(p & 1) * 16 + li];
      double v[16];
#pragma unroll
      for (int c = 0; c < 16; c++) v[c] = Ysh[li * 17 + c];
      // x_c = v_c / T_cc, then v_c' -= x_c T_cc' for every later c'.  The quotient comes from the
      // reciprocal y = 1 / T_cc with one correction, x = q + (v - T_cc q) y, q = v y, which is the
      // correctly rounded v / T_cc (Markstein) for the unit-modulus diagonal of a UDT's T (an infinite
      // q stays); any other diagonal value divides.
#pragma unroll
      for (int c = 0; c < 16; c++) {
        const double d = readlane_d(dl, c), y = readlane_d(yl, c);
        double xc;
        if (fabs(d) >= 0.5 && fabs(d) <= 2.0) {
          const double q0 = v[c] * y;
          xc = fma(fma(-d, q0, v[c]), y, q0);
          xc = fabs(q0) < HUGE_VAL ? xc : q0;
        } else {
          xc = v[c] / d;
        }
        v[c] = xc;
#pragma unroll
        for (int c2 = c + 1; c2 < 16; c2++) v[c2] = fma(-xc, Tp[c * 17 + c2], v[c2]);
      }
      if (lane < 16) {
#pragma unroll
        for (int c = 0; c < 16; c++)
          if (j0 + c < n) X[(size_t)(j0 + c) * 17 + lane] = v[c];
      }
    } else if (wave == 1 && p + 1 < nb) {
      store_block(p + 1);
      if (p + 2 < nb) load_block(p + 2);
    }
    __syncthreads();
  }
  if (grr < n) {
    for (int j = gcol; j < n; j += 16) A[(size_t)grr + (size_t)j * n] = X[(size_t)j * 17 + grow];
  }
}

// rdivp for n <= kRdivpBlockMaxN: four waves per 16-row strip.  Every 16 x 16 diagonal block
// of T is inverted first (thread (b, c) solves U_b x = e_c upwards), beside the loads of
// the strip's pivoted input; then per 16-column panel p the four waves share the update
// Y = X_p - X_{<p} T_{<p,p} on the matrix cores (wave w takes k-steps w, w + 4, ...; T's
// coupling column of the next panel is loaded while the current one is formed), and wave 0
// forms X_p = Y inv(T_pp), one 16 x 16 x 16 product.  In exact arithmetic this is the
// column-by-column substitution of the reference; the products round differently (the
// bound of the kernel tests: 1e-12 of the largest entry).
static size_t rdivp_block_lds_bytes(int n) {
  const size_t nb = (size_t)(n + 15) / 16;
  return ((size_t)n * 17 + nb * 16 * 17 + 4 * 4 * 64 + 16 * 17) * 8 + (size_t)n * 4;
}

// KS = 16 (n <= 256) or 32 (n <= 512): loads per thread of the gather and k-steps of one wave
// per panel, at most.  Every batch of loads has this fixed count (clamped addresses), so the
// wait for one batch never waits for the prefetch behind it.
template <bool TAB, int KS>
__global__ __launch_bounds__(256) void rdivp_block_kernel(RdivpBatch batch) {
  constexpr int kRdivpBlockSteps = KS;
  const RdivpItem it = TAB ? batch.items[blockIdx.y] : batch.it[blockIdx.y];
  const int n = TAB ? it.n : batch.n;
  const int r0 = blockIdx.x * 16;
  if (TAB && r0 >= n) return;   // item-table launches size the grid for the largest item
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, li = lane & 15, lk = lane >> 4;
  const int nb = (n + 15) / 16;
  extern __shared__ __align__(16) unsigned char smem[];
  double* X = reinterpret_cast<double*>(smem);          // [n][17]: X[j * 17 + row]
  double* Ti = X + (size_t)n * 17;                      // [nb][16][17]: block b, row a, column c
  double* red = Ti + (size_t)nb * 16 * 17;              // [4 waves][4][64]
  double* Ysh = red + 4 * 4 * 64;                       // [16][17]: Y[row][col]
  int* pv = reinterpret_cast<int*>(Ysh + 16 * 17);
  double* __restrict__ A = it.A;
  const double* __restrict__ T = it.T;

  for (int j = tid; j < n; j += 256) pv[j] = it.pivot[j];
  __syncthreads();
  // the strip's pivoted input (thread: row tid % 16, columns tid / 16 + 16 q), held in
  // registers while the diagonal blocks are inverted
  const int grow = tid & 15, gcol = tid >> 4;
  const int grr = r0 + grow, grc = grr < n ? grr : n - 1;
  double gv[kRdivpBlockSteps];
#pragma unroll
  for (int q = 0; q < kRdivpBlockSteps; q++) {
    const int j = gcol + 16 * q;
    gv[q] = A[(size_t)grc + (size_t)pv[j < n ? j : n - 1] * n];
  }
  // diagonal blocks of T: the upper part, the identity beyond n (consecutive threads read
  // consecutive rows of a column)
  for (int e = tid; e < nb * 256; e += 256) {
    const int b = e >> 8, c = (e >> 4) & 15, a = e & 15;
    const int ra = 16 * b + a, cc = 16 * b + c;
    double v;
    if (ra < n && cc < n) v = a <= c ? T[(size_t)ra + (size_t)cc * n] : 0.0;
    else v = a == c ? 1.0 : 0.0;
    Ti[(size_t)(b * 16 + a) * 17 + c] = v;
  }
  __syncthreads();
  for (int b0 = 0; b0 < nb; b0 += 16) {
    const int b = b0 + (tid >> 4), c = tid & 15;
    double x[16];
    if (b < nb) {
      const double* U = Ti + (size_t)b * 16 * 17;
      // x[k] = 0 for k > c, so every row runs the same straight-line sum
#pragma unroll
      for (int i = 15; i >= 0; i--) {
        double sum = i == c ? 1.0 : 0.0;
#pragma unroll
        for (int k = i + 1; k < 16; k++) sum -= U[i * 17 + k] * x[k];
        x[i] = i <= c ? sum / U[i * 17 + i] : 0.0;
      }
    }
    __syncthreads();
    if (b < nb) {
#pragma unroll
      for (int a = 0; a < 16; a++) Ti[(size_t)(b * 16 + a) * 17 + c] = x[a];
    }
  }
#pragma unroll
  for (int q = 0; q < kRdivpBlockSteps; q++) {
    const int j = gcol + 16 * q;
    if (j < n) X[(size_t)j * 17 + grow] = gv[q];
  }
  __syncthreads();

  // T's coupling column of panel j0 for this wave's k-steps q = wave + 4 s (4 q < j0)
  auto load_tb = [&](double (&tb)[KS], int j0) {
    const int cb = j0 + li, cbc = cb < n ? cb : n - 1;
#pragma unroll
    for (int s = 0; s < kRdivpBlockSteps; s++) {
      const int k = 4 * (wave + 4 * s) + lk;
      tb[s] = T[(size_t)(k < n ? k : n - 1) + (size_t)cbc * n];
    }
  };
  auto panel = [&](int p, const double (&tb)[KS]) {
    const int j0 = 16 * p;
    dx4 acc = dx4{0, 0, 0, 0};
#pragma unroll
    for (int s = 0; s < kRdivpBlockSteps; s++) {
      const int q = wave + 4 * s;
      if (4 * q < j0) acc = mfma16(X[(size_t)(4 * q + lk) * 17 + li], tb[s], acc);
    }
#pragma unroll
    for (int r = 0; r < 4; r++) red[(wave * 4 + r) * 64 + lane] = acc[r];
    __syncthreads();
    if (wave == 0) {
      const int cb = j0 + li;
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int row = mfma_row<double>(lane, r);
        const double u = (red[r * 64 + lane] + red[(4 + r) * 64 + lane]) +
                         (red[(8 + r) * 64 + lane] + red[(12 + r) * 64 + lane]);
        Ysh[row * 17 + li] = cb < n ? X[(size_t)cb * 17 + row] - u : 0.0;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
      dx4 o = dx4{0, 0, 0, 0};
#pragma unroll
      for (int ks = 0; ks < 4; ks++) {
        const int k = 4 * ks + lk;
        o = mfma16(Ysh[li * 17 + k], Ti[(size_t)(p * 16 + k) * 17 + li], o);
      }
      if (cb < n) {
#pragma unroll
        for (int r = 0; r < 4; r++) X[(size_t)cb * 17 + mfma_row<double>(lane, r)] = o[r];
      }
    }
    __syncthreads();
  };
  double tbA[kRdivpBlockSteps], tbB[kRdivpBlockSteps];
  load_tb(tbA, 0);
  for (int p = 0; p < nb; p += 2) {
    if (p + 1 < nb) load_tb(tbB, 16 * (p + 1));
    panel(p, tbA);
    if (p + 1 < nb) {
      if (p + 2 < nb) load_tb(tbA, 16 * (p + 2));
      panel(p + 1, tbB);
    }
  }
  if (grr < n) {
    for (int j = gcol; j < n; j += 16) A[(size_t)grr + (size_t)j * n] = X[(size_t)j * 17 + grow];
  }
}

hipError_t launch_rdivp(const RdivpBatch& b, hipStream_t s) {
  if (b.count <= 0) return hipSuccess;
  if (b.items) {
    // item table: one kernel class per launch (the host packs items of n <= kRdivpBlockMaxN, of
    // n <= kRdivpStripMaxN and larger ones apart); the grid and LDS are sized for the largest item
    if (b.max_n < 1 || b.max_n > 2048) return hipErrorInvalidValue;
    if (b.max_n <= 256)
      hipLaunchKernelGGL((rdivp_block_kernel<true, 16>), dim3((b.max_n + 15) / 16, b.count), dim3(256),
                         rdivp_block_lds_bytes(b.max_n), s, b);
    else if (b.max_n <= kRdivpBlockMaxN)
      hipLaunchKernelGGL((rdivp_block_kernel<true, 32>), dim3((b.max_n + 15) / 16, b.count), dim3(256),
                         rdivp_block_lds_bytes(b.max_n), s, b);
    else if (b.max_n <= 640)
      hipLaunchKernelGGL((rdivp_wide_kernel<true, 40>), dim3((b.max_n + 15) / 16, b.count), dim3(256),
                         rdivp_wide_lds_bytes(b.max_n), s, b);
    else if (b.max_n <= kRdivpStripMaxN)
      hipLaunchKernelGGL((rdivp_wide_kernel<true, 64>), dim3((b.max_n + 15) / 16, b.count), dim3(256),
                         rdivp_wide_lds_bytes(b.max_n), s, b);
    else
      hipLaunchKernelGGL(rdivp_kernel<true>, dim3((b.max_n + 63) / 64, b.count), dim3(256), 0, s, b);
    return hipGetLastError();
  }
  if (b.count > kMaxUdtItems) return hipErrorInvalidValue;
  if (b.n <= 256)
    hipLaunchKernelGGL((rdivp_block_kernel<false, 16>), dim3((b.n + 15) / 16, b.count), dim3(256),
                       rdivp_block_lds_bytes(b.n), s, b);
  else if (b.n <= kRdivpBlockMaxN)
    hipLaunchKernelGGL((rdivp_block_kernel<false, 32>), dim3((b.n + 15) / 16, b.count), dim3(256),
                       rdivp_block_lds_bytes(b.n), s, b);
  else if (b.n <= 640)
    hipLaunchKernelGGL((rdivp_wide_kernel<false, 40>), dim3((b.n + 15) / 16, b.count), dim3(256),
                       rdivp_wide_lds_bytes(b.n), s, b);
  else if (b.n <= kRdivpStripMaxN)
    hipLaunchKernelGGL((rdivp_wide_kernel<false, 64>), dim3((b.n + 15) / 16, b.count), dim3(256),
                       rdivp_wide_lds_bytes(b.n), s, b);
  else
    hipLaunchKernelGGL(rdivp_kernel<false>, dim3((b.n + 63) / 64, b.count), dim3(256), 0, s, b);
  return hipGetLastError();
}

hipError_t qr_kernels_init() {
  const void* fns[] = {reinterpret_cast<const void*>(udt_panel_kernel<1>),
                       reinterpret_cast<const void*>(udt_panel_kernel<2>),
                       reinterpret_cast<const void*>(udt_panel_kernel<4>),
                       reinterpret_cast<const void*>(udt_panel_kernel<8>),
                       reinterpret_cast<const void*>(udt_panel_kernel<16>),
                       reinterpret_cast<const void*>(udt_panel_tall_kernel<false>),
                       reinterpret_cast<const void*>(udt_panel_tall_kernel<true>),
                       reinterpret_cast<const void*>(udt_panel_tab_kernel),
                       reinterpret_cast<const void*>(rdivp_wide_kernel<false, 40>),
                       reinterpret_cast<const void*>(rdivp_wide_kernel<true, 40>),
                       reinterpret_cast<const void*>(rdivp_wide_kernel<false, 64>),
                       reinterpret_cast<const void*>(rdivp_wide_kernel<true, 64>),
                       reinterpret_cast<const void*>(rdivp_block_kernel<false, 16>),
                       reinterpret_cast<const void*>(rdivp_block_kernel<true, 16>),
                       reinterpret_cast<const void*>(rdivp_block_kernel<false, 32>),
                       reinterpret_cast<const void*>(rdivp_block_kernel<true, 32>)};
  for (const void* f : fns) {
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

}  // namespace dqmc
