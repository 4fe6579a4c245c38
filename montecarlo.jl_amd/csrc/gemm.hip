// Batched dense products on the gfx950 matrix cores.
//
// C = alpha * diag(dl) * op(A) * diag(dmid) * op(B) * diag(dr) + beta * C + diag(dadd)
//
// Every slice-matrix multiply of the DQMC stack (reference stack.jl:319-367: eT^2 eV M,
// M eT^2 eV, M eV^-1 eT^-2, eV^-1 eT^-2 M, eV' eT^2' M), the Green's-function wraps
// (stack.jl:594-603), the products of calculate_greens_AVX! (stack.jl:442-496) and the
// physical-greens transform (greens.jl:114-125) are one or two launches of this kernel:
// the diagonal interaction matrices enter as row / inner / column scalings generated
// straight from the Hirsch field column, so they never exist as separate arrays.
//
// Tile: 32 x 32 per workgroup of 16 waves or 64 x 64 per workgroup of 8: each quadrant of the
// tile has four (or two) waves, each with v_mfma_f64_16x16x4f64 (FP64) or
// v_mfma_f32_16x16x4f32 (FP32) accumulators over their part of K, added through LDS at the end.
// The waves of a SIMD share the loads and hide each other's latencies, where one wave per SIMD was
// bound by its own instruction stream.  (The 64-wide FP64 form has 128 registers per wave, two
// workgroups per CU, and spills 8 to 21 of them.)  Operand layout of the 16x16x4 instructions (wave64, lane l):
//   A (16 x 4): lane l supplies A[l % 16][l / 16]
//   B (4 x 16): lane l supplies B[l / 16][l % 16]
//   D (16 x 16): lane l holds D[row][l % 16], r = 0..3, with row = l / 16 + 4 r (FP64)
//                or 4 (l / 16) + r (FP32); see mfma_row in common.h
// K is staged through LDS in chunks with two buffers: a chunk's global loads are all issued at
// once and the next chunk's loads are in flight during the current chunk's products, so a
// 32 x 32 tile with K <= 256 costs about one memory round trip.
#include "common.h"

namespace dqmc {

typedef double dx4 __attribute__((ext_vector_type(4)));
typedef float fx4 __attribute__((ext_vector_type(4)));

template <typename T> struct AccT;
template <> struct AccT<double> { typedef dx4 type; };
template <> struct AccT<float> { typedef fx4 type; };

__device__ __forceinline__ dx4 mfma16(double a, double b, dx4 c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ fx4 mfma16(float a, float b, fx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// Tile geometry: TILE x TILE outputs per workgroup, K staged in chunks of KC.  TILE = 32
// (a wave: one 16x16 fragment) where a launch has few tiles, TILE = 64 (a wave: a 32x32 quadrant
// as 2 x 2 fragments; two workgroups per CU) where it has many: half the operand traffic per
// flop.  With either, an element is the sum (p0 + p2) + (p1 + p3) of four accumulators, p_q over
// the pieces k = 16 (4 i + q) .. + 15, i = 0, 1, ..., in order, so the two give identical
// results: a wave of the 32-wide tile holds one of the four, a wave of the 64-wide tile p_g and
// p_(g+2), whose sum it forms itself.
template <int TILE> struct TileCfg {
  static constexpr int Threads = TILE == 32 ? 1024 : 512;
  static constexpr int Groups = Threads / 256;            // waves per quadrant
  static constexpr int Parts = 4 / Groups;                // accumulators per wave and fragment
  static constexpr int KC = TILE == 32 ? 128 : 32;
  static constexpr int LD = TILE + 1;
  static constexpr int F = TILE / 32;                     // 16x16 fragments per wave and side
  static constexpr int LPT = 2 * TILE * KC / Threads;     // loads per thread per chunk (8)
  static constexpr int Blocks = TILE == 32 ? 1 : 2;       // workgroups per CU
};

template <typename T, int TILE>
constexpr size_t gemm_lds_bytes() {
  const size_t stage = sizeof(T) * 2 * 2 * TileCfg<TILE>::KC * TileCfg<TILE>::LD;
  const size_t sums = sizeof(T) * TileCfg<TILE>::Groups * 4 * TileCfg<TILE>::F * TileCfg<TILE>::F * 16 * 17;
  return stage > sums ? stage : sums;
}

// XCD-aware tile order.  Workgroups go to the 8 XCDs round-robin by linear id, and each XCD
// has its own L2: with the plain order, XCD k gets the tiles of row block k, so every XCD
// fetches every column panel of B.  When the grid splits evenly, the tiles are renumbered
// so that XCD k holds a contiguous run of 4 x 4 super-tiles (of one item), whose 4 row and
// 4 column panels then come from its own L2.  A permutation of the tiles: results are equal.
constexpr int kXcds = 8, kSuper = 4;
__device__ __forceinline__ void xcd_tile(int& bx, int& by, int& bz) {
  const int gx = gridDim.x, gy = gridDim.y, gz = gridDim.z;
  bx = blockIdx.x; by = blockIdx.y; bz = blockIdx.z;
  const int per_item = gx * gy;
  const int total = per_item * gz;
  if (gx % kSuper || gy % kSuper || total % kXcds) return;
  const int hw = blockIdx.x + gx * (blockIdx.y + gy * blockIdx.z);
  const int logical = (hw % kXcds) * (total / kXcds) + hw / kXcds;
  bz = logical / per_item;
  const int t = logical % per_item;
  const int sb = t / (kSuper * kSuper), w = t % (kSuper * kSuper);
  const int sbx = sb % (gx / kSuper), sby = sb / (gx / kSuper);
  bx = sbx * kSuper + w % kSuper;
  by = sby * kSuper + w / kSuper;
}

// TAB: the items come from the device table batch.items (many-chain launches), else from
// the kernel arguments (a separate instantiation, so the one-chain path reads its items
// straight from the argument segment)
template <typename T, int TA, int TB, bool TAB, int TILE>
__global__ __launch_bounds__(TileCfg<TILE>::Threads, TileCfg<TILE>::Threads * TileCfg<TILE>::Blocks / 256) void gemm_kernel(GemmBatch<T> batch) {
  typedef typename AccT<T>::type acc_t;
  constexpr int kTM = TILE, kTN = TILE, kKC = TileCfg<TILE>::KC, kLD = TileCfg<TILE>::LD;
  constexpr int kF = TileCfg<TILE>::F, kLoadsPerThread = TileCfg<TILE>::LPT;
  constexpr int kHalf = kLoadsPerThread / 2;
  constexpr int kThreads = TileCfg<TILE>::Threads, kGroups = TileCfg<TILE>::Groups, kParts = TileCfg<TILE>::Parts;
  int bx, by, bz;
  xcd_tile(bx, by, bz);
  const GemmItem<T>& it = TAB ? batch.items[bz] : batch.it[bz];
  const int M = it.M, N = it.N, K = it.K;
  const int m0 = bx * kTM, n0 = by * kTN;
  if (m0 >= M || n0 >= N) return;  // uniform per workgroup, before any barrier

  extern __shared__ __align__(16) unsigned char smem[];
  T* As = reinterpret_cast<T*>(smem);              // [2][kKC][kLD]  As[k][m]
  T* Bs = As + 2 * kKC * kLD;                      // [2][kKC][kLD]  Bs[k][n]

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int quad = wave & 3, kq = wave >> 2;       // quadrant of the tile, first piece of K
  const int wm = (quad & 1) * (16 * kF), wn = (quad >> 1) * (16 * kF);
  const T* __restrict__ A = it.A;
  const T* __restrict__ B = it.B;
  const int lda = it.lda, ldb = it.ldb;
  const bool has_mid = diag_active(it.dmid);
  const int nch = (K + kKC - 1) / kKC;

  // element q of this thread in a chunk: q < kHalf -> A, else B; index e = tid + kThreads (q % kHalf)
  auto coord = [&](int q, int& mn, int& kk) {
    const int e = tid + kThreads * (q % kHalf);
    const bool isA = q < kHalf;
    const bool kfast = isA ? TA == 1 : TB == 0;    // consecutive threads along k in memory
    if (kfast) { kk = e % kKC; mn = e / kKC; }
    else { mn = e % kTM; kk = e / kTM; }
  };
  // A chunk's loads are all issued before any is used: in-range (clamped) addresses, then
  // the out-of-range elements zeroed; the middle diagonal (a uniform choice per launch) is
  // gathered for the chunk's k values in a second batch of loads.
  auto load = [&](int c, T* reg) {
    const int k0 = c * kKC;
    const int kl = K - 1 - k0, ml = M - 1 - m0, nl = N - 1 - n0;   // last in-range offsets
    const T* Ac = TA == 0 ? A + m0 + (size_t)k0 * lda : A + k0 + (size_t)m0 * lda;
    const T* Bc = TB == 0 ? B + k0 + (size_t)n0 * ldb : B + n0 + (size_t)k0 * ldb;
#pragma unroll
    for (int q = 0; q < kLoadsPerThread; q++) {
      int mn, kk;
      coord(q, mn, kk);
      const bool isA = q < kHalf;
      const int last = isA ? ml : nl;
      mn = mn < last ? mn : last;
      kk = kk < kl ? kk : kl;
      // a uniform base and a 32-bit lane offset inside the chunk
      const bool kfast = isA ? TA == 1 : TB == 0;
      const unsigned int ld = isA ? lda : ldb;
      const unsigned int off = (unsigned int)sizeof(T) * (kfast ? kk + mn * ld : mn + kk * ld);
      reg[q] = *reinterpret_cast<const T*>(reinterpret_cast<const char*>(isA ? Ac : Bc) + off);
    }
    if (has_mid) {
      double f[kHalf];
      if (it.dmid.vec) {
#pragma unroll
        for (int q = 0; q < kHalf; q++) {
          int mn, kk;
          coord(q, mn, kk);
          const int gk = k0 + kk;
          f[q] = it.dmid.vec[gk < K ? gk : K - 1];
        }
        if (it.dmid.mode == kDiagInv) {
#pragma unroll
          for (int q = 0; q < kHalf; q++) f[q] = 1.0 / f[q];
        } else if (it.dmid.mode != kDiagPlain) {
#pragma unroll
          for (int q = 0; q < kHalf; q++) f[q] = diag_map(f[q], it.dmid.mode);
        }
      } else {
        int8_t cf[kHalf];
#pragma unroll
        for (int q = 0; q < kHalf; q++) {
          int mn, kk;
          coord(q, mn, kk);
          const int gk = k0 + kk;
          cf[q] = it.dmid.conf[gk < K ? gk : K - 1];
        }
#pragma unroll
        for (int q = 0; q < kHalf; q++) f[q] = cf[q] > 0 ? it.dmid.pos : it.dmid.neg;
      }
#pragma unroll
      for (int q = 0; q < kHalf; q++) reg[q] = T(reg[q] * f[q]);
    }
    if (m0 + kTM > M || n0 + kTN > N || k0 + kKC > K) {
#pragma unroll
      for (int q = 0; q < kLoadsPerThread; q++) {
        int mn, kk;
        coord(q, mn, kk);
        const int gk = k0 + kk;
        const bool ok = q < kHalf ? (m0 + mn < M && gk < K) : (n0 + mn < N && gk < K);
        reg[q] = ok ? reg[q] : T(0);
      }
    }
  };
  auto store = [&](int buf, const T* reg) {
    T* Ab = As + buf * kKC * kLD;
    T* Bb = Bs + buf * kKC * kLD;
#pragma unroll
    for (int q = 0; q < kLoadsPerThread; q++) {
      int mn, kk;
      coord(q, mn, kk);
      if (q < kHalf) Ab[kk * kLD + mn] = reg[q];
      else Bb[kk * kLD + mn] = reg[q];
    }
  };
  acc_t acc[kParts][kF][kF];
#pragma unroll
  for (int h = 0; h < kParts; h++)
#pragma unroll
    for (int i = 0; i < kF; i++)
#pragma unroll
      for (int j = 0; j < kF; j++) acc[h][i][j] = acc_t{0, 0, 0, 0};
  const int li = lane & 15, lk = lane >> 4;
  auto step = [&](const T* Ab, const T* Bb, int kk, int h) {
    T av[kF], bv[kF];
#pragma unroll
    for (int i = 0; i < kF; i++) av[i] = Ab[(kk + lk) * kLD + wm + 16 * i + li];
#pragma unroll
    for (int j = 0; j < kF; j++) bv[j] = Bb[(kk + lk) * kLD + wn + 16 * j + li];
#pragma unroll
    for (int i = 0; i < kF; i++)
#pragma unroll
      for (int j = 0; j < kF; j++) acc[h][i][j] = mfma16(av[i], bv[j], acc[h][i][j]);
  };
  // 16 k-steps of a piece (offset k0 in a chunk with kend of K left): a whole one straight-line,
  // so that the LDS reads run ahead of the products
  auto piece = [&](const T* Ab, const T* Bb, int k0, int kend, int h) {
    if (k0 + 16 <= kend) {
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4) step(Ab, Bb, k0 + kk, h);
    } else {
#pragma unroll
      for (int kk = 0; kk < 16; kk += 4)
        if (k0 + kk < kend) step(Ab, Bb, k0 + kk, h);
    }
  };

  if constexpr (TILE == 32) {
    auto compute = [&](int c, int buf) {
      // (not unrolled over the pieces: the registers of 16 waves)
#pragma unroll 1
      for (int p = 0; p < kKC; p += 64)
        piece(As + buf * kKC * kLD, Bs + buf * kKC * kLD, p + 16 * kq, K - c * kKC, 0);
    };
    // chunk c lives in buffer c % 2 and arrives in register set ra (even c) or rb (odd c), so
    // that two chunks are in flight
    T ra[kLoadsPerThread], rb[kLoadsPerThread];
    load(0, ra);
    if (nch > 1) load(1, rb);
    store(0, ra);
    __syncthreads();
    for (int c = 0; c < nch; c += 2) {
      if (c + 2 < nch) load(c + 2, ra);
      compute(c, 0);
      if (c + 1 < nch) store(1, rb);
      __syncthreads();
      if (c + 1 < nch) {
        if (c + 3 < nch) load(c + 3, rb);
        compute(c + 1, 1);
        if (c + 2 < nch) store(0, ra);
        __syncthreads();
      }
    }
  } else {
    // a chunk holds two of the four pieces, in turn; one chunk ahead (the CU's other workgroup
    // computes while this one waits)
    T ra[kLoadsPerThread];
    load(0, ra);
    store(0, ra);
    __syncthreads();
    for (int c = 0; c < nch; c += 2) {
      if (c + 1 < nch) load(c + 1, ra);
      piece(As, Bs, 16 * kq, K - c * kKC, 0);
      if (c + 1 < nch) store(1, ra);
      __syncthreads();
      if (c + 1 < nch) {
        if (c + 2 < nch) load(c + 2, ra);
        piece(As + kKC * kLD, Bs + kKC * kLD, 16 * kq, K - (c + 1) * kKC, 1);
        if (c + 2 < nch) store(0, ra);
        __syncthreads();
      }
    }
  }

  // the partial sums of every element through LDS (free after the last barrier): fragment
  // (group, quadrant, i, j) at 272 elements each, column by column with leading dimension 17
  T* red = reinterpret_cast<T*>(smem);
  constexpr int kFrag = 16 * 17, kGroup = 4 * kF * kF * kFrag;
#pragma unroll
  for (int i = 0; i < kF; i++)
#pragma unroll
    for (int j = 0; j < kF; j++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        T x = acc[0][i][j][r];
        if constexpr (kParts == 2) x += acc[1][i][j][r];
        red[kq * kGroup + ((quad * kF + i) * kF + j) * kFrag + li * 17 + mfma_row<T>(lane, r)] = x;
      }
  __syncthreads();

  const T alpha = T(batch.alpha), beta = T(batch.beta);
  const bool has_l = diag_active(it.dl), has_r = diag_active(it.dr), has_add = diag_active(it.dadd);
  T* __restrict__ Cm = it.C;
  const int ldc = it.ldc;
#pragma unroll
  for (int q = 0; q < TILE * TILE / kThreads; q++) {
    // consecutive threads write consecutive rows of a column
    const int e = tid + kThreads * q;
    const int rt = e % TILE, ct = e / TILE;
    const int row = m0 + rt, col = n0 + ct;
    if (row >= M || col >= N) continue;
    const int qd = rt / (16 * kF) + 2 * (ct / (16 * kF)), i = rt / 16 % kF, j = ct / 16 % kF;
    const T* x = red + ((qd * kF + i) * kF + j) * kFrag + (ct & 15) * 17 + (rt & 15);
    T sum;
    if constexpr (kParts == 2) sum = x[0] + x[kGroup];
    else sum = (x[0] + x[2 * kGroup]) + (x[kGroup] + x[3 * kGroup]);
    T v = alpha * sum;
    if (has_l) v *= T(diag_at(it.dl, row));
    if (has_r) v *= T(diag_at(it.dr, col));
    T* dst = Cm + (size_t)row + (size_t)col * ldc;
    if (beta != T(0)) v += beta * (*dst);
    if (has_add && row == col) v += T(diag_at(it.dadd, row));
    *dst = v;
  }
}

// Which tile, by an estimate in clocks.  32-wide: workgroups of a CU follow each other, each with its
// products (K / 4 steps of 64 clocks on every SIMD) and about 6000 clocks of fill, sums and stores.
// 64-wide: a CU's workgroups run in pairs that share the matrix cores, so four times the products for
// each of them, and 8000 clocks once, for the fill and stores that no neighbour hides.  That
// counts a partly filled turn of 256 as a whole one, which is too much beside a neighbour: for one
// matrix of n = 1025 to 1248, 1409 to 1536 and 1729 to 1824, 32-wide tiles are taken although 64-wide
// ones are faster, by a quarter at most.
// Measured, 32- and 64-wide, one matrix: n = 576 27 and 40 us, 784 54 and 56, 864 55 and 62, 865 70
// and 62, 1024 80 and 70, 1100 115 and 105, 1300 162 and 121, 1800 435 and 330, 2048 565 and 362; sweeps
// of 32 chains of n = 256, two flavours, 23.4 and 19.5 ms, of 256 chains of n = 64 22.0 and 18.4 ms,
// of 256 chains of n = 16 15.8 and 18.3 ms (16.4 ms by the rule).
constexpr int64_t kGemmCUs = 256;
static bool wide_tiles(int64_t t32, int64_t t64, int K) {
  const int64_t step = (int64_t)((K + 3) / 4) * 64;
  const int64_t c32 = (t32 + kGemmCUs - 1) / kGemmCUs * (step + 6000);
  const int64_t c64 = (t64 + kGemmCUs - 1) / kGemmCUs * 4 * step + 8000;
  return c64 < c32;
}

template <typename T, int TILE>
static void launch_gemm_tile(const GemmBatch<T>& b, int Mx, int Nx, hipStream_t s) {
  dim3 grid((Mx + TILE - 1) / TILE, (Nx + TILE - 1) / TILE, b.count);
  dim3 block(TileCfg<TILE>::Threads);
  const size_t lds = gemm_lds_bytes<T, TILE>();
  const int sel = b.transA * 2 + b.transB;
  if (b.items) {
    switch (sel) {
      case 0: hipLaunchKernelGGL((gemm_kernel<T, 0, 0, true, TILE>), grid, block, lds, s, b); break;
      case 1: hipLaunchKernelGGL((gemm_kernel<T, 0, 1, true, TILE>), grid, block, lds, s, b); break;
      case 2: hipLaunchKernelGGL((gemm_kernel<T, 1, 0, true, TILE>), grid, block, lds, s, b); break;
      default: hipLaunchKernelGGL((gemm_kernel<T, 1, 1, true, TILE>), grid, block, lds, s, b); break;
    }
  } else {
    switch (sel) {
      case 0: hipLaunchKernelGGL((gemm_kernel<T, 0, 0, false, TILE>), grid, block, lds, s, b); break;
      case 1: hipLaunchKernelGGL((gemm_kernel<T, 0, 1, false, TILE>), grid, block, lds, s, b); break;
      case 2: hipLaunchKernelGGL((gemm_kernel<T, 1, 0, false, TILE>), grid, block, lds, s, b); break;
      default: hipLaunchKernelGGL((gemm_kernel<T, 1, 1, false, TILE>), grid, block, lds, s, b); break;
    }
  }
}

template <typename T>
static hipError_t launch_gemm_t(const GemmBatch<T>& b, hipStream_t s) {
  if (b.count <= 0) return hipSuccess;
  int Mx = 0, Nx = 0, Kx = 0;
  if (b.items) {
    // item table in device memory (checked by the host code that packed it)
    if (b.max_m < 1 || b.max_n < 1 || b.count > 65535) return hipErrorInvalidValue;
    Mx = b.max_m;
    Nx = b.max_n;
    Kx = Mx;                       // (square products)
  } else {
    if (b.count > kMaxGemmItems) return hipErrorInvalidValue;
    for (int i = 0; i < b.count; i++) {
      if (b.it[i].K < 1) return hipErrorInvalidValue;
      if (b.it[i].M > Mx) Mx = b.it[i].M;
      if (b.it[i].N > Nx) Nx = b.it[i].N;
      if (b.it[i].K > Kx) Kx = b.it[i].K;
    }
  }
  const int64_t t32 = (int64_t)((Mx + 31) / 32) * ((Nx + 31) / 32) * b.count;
  const int64_t t64 = (int64_t)((Mx + 63) / 64) * ((Nx + 63) / 64) * b.count;
  if (wide_tiles(t32, t64, Kx)) launch_gemm_tile<T, 64>(b, Mx, Nx, s);
  else launch_gemm_tile<T, 32>(b, Mx, Nx, s);
  return hipGetLastError();
}

template <typename T, bool TAB, int TILE>
static hipError_t set_gemm_lds() {
  const void* fns[] = {reinterpret_cast<const void*>(gemm_kernel<T, 0, 0, TAB, TILE>),
                       reinterpret_cast<const void*>(gemm_kernel<T, 0, 1, TAB, TILE>),
                       reinterpret_cast<const void*>(gemm_kernel<T, 1, 0, TAB, TILE>),
                       reinterpret_cast<const void*>(gemm_kernel<T, 1, 1, TAB, TILE>)};
  for (const void* f : fns) {
    hipError_t e = hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) return e;
  }
  return hipSuccess;
}

hipError_t gemm_kernels_init() {
  hipError_t e = set_gemm_lds<double, false, 32>();
  if (e == hipSuccess) e = set_gemm_lds<double, true, 32>();
  if (e == hipSuccess) e = set_gemm_lds<double, false, 64>();
  if (e == hipSuccess) e = set_gemm_lds<double, true, 64>();
  if (e == hipSuccess) e = set_gemm_lds<float, false, 32>();
  if (e == hipSuccess) e = set_gemm_lds<float, true, 32>();
  if (e == hipSuccess) e = set_gemm_lds<float, false, 64>();
  if (e == hipSuccess) e = set_gemm_lds<float, true, 64>();
  return e;
}

hipError_t launch_gemm_f64(const GemmBatch<double>& b, hipStream_t s) { return launch_gemm_t(b, s); }
hipError_t launch_gemm_f32(const GemmBatch<float>& b, hipStream_t s) { return launch_gemm_t(b, s); }

}  // namespace dqmc
