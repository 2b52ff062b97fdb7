// Grouped, energy-batched complex GEMM on CDNA4 FP64 matrix cores.
//
// Each launch carries up to kMaxProblems independent problems
//   D = sum_t alpha_t op(A_t) op(B_t) + sum_a (c1_a F_a + c2_a F_a^H)
// over nE energies.  Two kernels:
//  * zgemm_grouped_kernel (second half of the file), the FP64 products of the
//    sweeps: three real MFMAs per complex product;
//  * zgemm4m_kernel: four real MFMAs (v_mfma_f64_16x16x4f64),
//    re += ar*br - ai*bi, im += ar*bi + ai*br, in FP64 or with FP32 operands.
// In zgemm4m_kernel, tiles of op(A) (TM x TK) and op(B) (TK x TN) are staged through LDS,
// k-major so that every MFMA fragment read is 16 contiguous complex values;
// conjugation and alpha are applied while staging, so the inner loop is the
// same for every op combination.  Global loads are issued for the next k-tile
// before the MFMAs of the current one (register double buffering, two LDS
// stages, one barrier per k-tile).
#include <type_traits>

#include "qx_common.h"

namespace qx {

namespace {

constexpr int PAD = 1;

// kTK: k-depth of one LDS stage.  kSlab: epilogue rows per LDS pass (the rows
// of one wave row).  The one-wave 32x32 tile (blocks below 64, where the
// products are bound by HBM) halves both for FP64, so that its LDS (8.4 KB
// instead of 16.9 KB) does not cap the number of workgroups per CU below what
// its registers allow (measured: equal at b = 32, +13-34% at b = 48); FP32
// products, whose MFMAs take half as long, lose more to the extra barriers
// than they gain and keep the deeper stage (k = 16 made the 4M 128x64 tile
// slower: 99 KB of LDS cost it a workgroup per CU).
template <int TM, int TN, bool kF32 = false>
struct TileShape {
  static constexpr bool kSmall = TM == 32 && TN == 32 && !kF32;
  static constexpr int kTK = kSmall ? 4 : 8;
  static constexpr int kSlab = kSmall ? 16 : 32;
  static constexpr int kWavesM = TM / 32;
  static constexpr int kWavesN = TN / 32;
  static constexpr int kThreads = 64 * kWavesM * kWavesN;
  static constexpr int kAPer = TM * kTK / kThreads;
  static constexpr int kBPer = kTK * TN / kThreads;
};

template <int TM, int TN, bool F32>
__device__ inline void load_a(const ZTerm& t, int e, int m, int m0, int k0, int tid,
                              double2 (&ra)[TileShape<TM, TN, F32>::kAPer]) {
  using S = TileShape<TM, TN, F32>;
  const double2* A = t.A + (int64_t)e * t.sA;
  const double2 zero = cmk(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < S::kAPer; ++i) {
    const int idx = tid + i * S::kThreads;
    int mm, kk;
    if (t.opA == kOpN) { mm = idx / S::kTK; kk = idx % S::kTK; }
    else { mm = idx % TM; kk = idx / TM; }
    const int gm = m0 + mm, gk = k0 + kk;
    double2 v = zero;
    if (gm < m && gk < t.k) {
      v = (t.opA == kOpN) ? A[(int64_t)gm * t.lda + gk] : A[(int64_t)gk * t.lda + gm];
    }
    ra[i] = v;
  }
}

__device__ inline void put(double2* p, double2 v) { *p = v; }
__device__ inline void put(float2* p, double2 v) { *p = make_float2((float)v.x, (float)v.y); }

template <int TM, int TN, bool F32, typename LT>
__device__ inline void store_a(const ZTerm& t, int tid,
                               const double2 (&ra)[TileShape<TM, TN, F32>::kAPer],
                               LT (*As)[TM + PAD]) {
  using S = TileShape<TM, TN, F32>;
  const bool cj = (t.opA == kOpC);
#pragma unroll
  for (int i = 0; i < S::kAPer; ++i) {
    const int idx = tid + i * S::kThreads;
    int mm, kk;
    if (!cj) { mm = idx / S::kTK; kk = idx % S::kTK; }
    else { mm = idx % TM; kk = idx / TM; }
    double2 v = ra[i];
    if (cj) v.y = -v.y;
    put(&As[kk][mm], cmul(t.alpha, v));
  }
}

template <int TM, int TN, bool F32>
__device__ inline void load_b(const ZTerm& t, int e, int n, int n0, int k0, int tid,
                              double2 (&rb)[TileShape<TM, TN, F32>::kBPer]) {
  using S = TileShape<TM, TN, F32>;
  const double2* B = t.B + (int64_t)e * t.sB;
  const double2 zero = cmk(0.0, 0.0);
#pragma unroll
  for (int i = 0; i < S::kBPer; ++i) {
    const int idx = tid + i * S::kThreads;
    int kk, nn;
    if (t.opB == kOpN) { kk = idx / TN; nn = idx % TN; }
    else { kk = idx % S::kTK; nn = idx / S::kTK; }
    const int gk = k0 + kk, gn = n0 + nn;
    double2 v = zero;
    if (gn < n && gk < t.k) {
      v = (t.opB == kOpN) ? B[(int64_t)gk * t.ldb + gn] : B[(int64_t)gn * t.ldb + gk];
    }
    rb[i] = v;
  }
}

template <int TM, int TN, bool F32, typename LT>
__device__ inline void store_b(const ZTerm& t, int tid,
                               const double2 (&rb)[TileShape<TM, TN, F32>::kBPer],
                               LT (*Bs)[TN + PAD]) {
  using S = TileShape<TM, TN, F32>;
  const bool cj = (t.opB == kOpC);
#pragma unroll
  for (int i = 0; i < S::kBPer; ++i) {
    const int idx = tid + i * S::kThreads;
    int kk, nn;
    if (!cj) { kk = idx / TN; nn = idx % TN; }
    else { kk = idx % S::kTK; nn = idx / S::kTK; }
    double2 v = rb[i];
    if (cj) v.y = -v.y;
    put(&Bs[kk][nn], v);
  }
}

template <int TM, int TN, typename LT>
struct Smem {
  using S = TileShape<TM, TN, std::is_same<LT, float2>::value>;
  static constexpr int kA = S::kTK * (TM + PAD);  // one LDS stage of op(A), k-major (LT elements)
  static constexpr int kB = S::kTK * (TN + PAD);  // one LDS stage of op(B), k-major
  static constexpr int kMainBytes = (2 * kA + 2 * kB) * (int)sizeof(LT);
  // the epilogue stages one kSlab-row slab of the output tile at a time
  static constexpr int kTileBytes = S::kSlab * (TN + 1) * (int)sizeof(double2);
  static constexpr int kBytes = kMainBytes > kTileBytes ? kMainBytes : kTileBytes;
};

// f64 MFMA with the BLGP field used as the negate-A modifier.
__device__ inline double4_t mfma(double a, double b, double4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}
__device__ inline double4_t mfma_nega(double a, double b, double4_t c) {
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 1);
}

// kRole only separates kernel names in traces: 0 = sweep products,
// 1 = trailing updates inside the blocked inversion.
// kF32: operands are rounded to complex64 while staged into LDS and the
// products run on v_mfma_f32_16x16x4f32 with FP32 accumulation; loads,
// addends and stores stay complex128 (the mixed-precision sweeps).
// Occupancy target: four 64x64 workgroups per CU (33 KB LDS each, <= 128
// VGPRs), measured faster than three.
template <int TM, int TN, int kRole, bool kF32>
__global__ void __launch_bounds__((TileShape<TM, TN, kF32>::kThreads),
                                  (TM * TN > 4096 ? 1 : (TM * TN == 4096 ? 4 : 2)))
zgemm4m_kernel(const ZGroup g) {
  using S = TileShape<TM, TN, kF32>;
  using LT = typename std::conditional<kF32, float2, double2>::type;
  using AccT = typename std::conditional<kF32, float4_t, double4_t>::type;
  using L = Smem<TM, TN, LT>;
  constexpr int TK = S::kTK;
  constexpr int kSlab = S::kSlab;
  __shared__ __align__(16) char smem_raw[L::kBytes];
  LT* smem = reinterpret_cast<LT*>(smem_raw);
  auto As = [&](int buf) { return reinterpret_cast<LT(*)[TM + PAD]>(smem + buf * L::kA); };
  auto Bs = [&](int buf) {
    return reinterpret_cast<LT(*)[TN + PAD]>(smem + 2 * L::kA + buf * L::kB);
  };

  // Energy-major order: logical id = e * per + (tile offset of the problem
  // within the energy) + tile.  The XCD remap gives every XCD a contiguous
  // range of energies with all their problems, so XCDs receive equal work even
  // when the problems of a launch differ in cost (number of terms, addends).
  const int per = g.wg_base[g.nprob];
  const int wid = xcd_remap(blockIdx.x, per * g.nE);
  const int e = wid / per;
  const int r = wid - e * per;
  int p = 0;
  while (p + 1 < g.nprob && r >= g.wg_base[p + 1]) ++p;
  const ZProblem& P = g.p[p];
  const int t = r - g.wg_base[p];
  const int m0 = (t / g.tiles_n[p]) * TM;
  const int n0 = (t % g.tiles_n[p]) * TN;
  const int m = P.m, n = P.n;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int wm = wave / S::kWavesN;
  const int wn = wave % S::kWavesN;

  AccT accr[2][2], acci[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      accr[i][j] = AccT{0, 0, 0, 0};
      acci[i][j] = AccT{0, 0, 0, 0};
    }

  for (int ti = 0; ti < P.nterms; ++ti) {
    // by value: the term's fields are loaded once into scalar registers
    // instead of being re-read from the kernel-argument segment in the loop
    const ZTerm T = P.t[ti];
    const int nk = (T.k + TK - 1) / TK;
    double2 ra[S::kAPer], rb[S::kBPer];
    load_a<TM, TN, kF32>(T, e, m, m0, 0, tid, ra);
    load_b<TM, TN, kF32>(T, e, n, n0, 0, tid, rb);
    store_a<TM, TN, kF32, LT>(T, tid, ra, As(0));
    store_b<TM, TN, kF32, LT>(T, tid, rb, Bs(0));
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
      const int cur = kt & 1;
      const bool more = (kt + 1 < nk);
      if (more) {
        load_a<TM, TN, kF32>(T, e, m, m0, (kt + 1) * TK, tid, ra);
        load_b<TM, TN, kF32>(T, e, n, n0, (kt + 1) * TK, tid, rb);
      }
      auto as = As(cur);
      auto bs = Bs(cur);
      // fragments double-buffered across the k-steps of this LDS stage
      LT fa[2][2], fb[2][2];
#pragma unroll
      for (int i = 0; i < 2; ++i) fa[0][i] = as[lane >> 4][wm * 32 + i * 16 + (lane & 15)];
#pragma unroll
      for (int j = 0; j < 2; ++j) fb[0][j] = bs[lane >> 4][wn * 32 + j * 16 + (lane & 15)];
#pragma unroll
      for (int ks = 0; ks < TK / 4; ++ks) {
        const int c = ks & 1;
        if (ks + 1 < TK / 4) {
          const int kk = (ks + 1) * 4 + (lane >> 4);
#pragma unroll
          for (int i = 0; i < 2; ++i) fa[c ^ 1][i] = as[kk][wm * 32 + i * 16 + (lane & 15)];
#pragma unroll
          for (int j = 0; j < 2; ++j) fb[c ^ 1][j] = bs[kk][wn * 32 + j * 16 + (lane & 15)];
        }
        if constexpr (kF32) {
          float nai[2];
#pragma unroll
          for (int i = 0; i < 2; ++i) nai[i] = -fa[c][i].y;
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              accr[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[c][i].x, fb[c][j].x, accr[i][j], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acci[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[c][i].x, fb[c][j].y, acci[i][j], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              accr[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(nai[i], fb[c][j].y, accr[i][j], 0, 0, 0);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j)
              acci[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(fa[c][i].y, fb[c][j].x, acci[i][j], 0, 0, 0);
        } else {
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) accr[i][j] = mfma(fa[c][i].x, fb[c][j].x, accr[i][j]);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acci[i][j] = mfma(fa[c][i].x, fb[c][j].y, acci[i][j]);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) accr[i][j] = mfma_nega(fa[c][i].y, fb[c][j].y, accr[i][j]);
#pragma unroll
          for (int i = 0; i < 2; ++i)
#pragma unroll
            for (int j = 0; j < 2; ++j) acci[i][j] = mfma(fa[c][i].y, fb[c][j].x, acci[i][j]);
        }
      }
      if (more) {
        store_a<TM, TN, kF32, LT>(T, tid, ra, As(cur ^ 1));
        store_b<TM, TN, kF32, LT>(T, tid, rb, Bs(cur ^ 1));
      }
      __syncthreads();
    }
  }

  // ---- epilogue: one 32-row slab (the rows of one wave row) at a time,
  // staged through LDS so that global accesses are row-coalesced ----
  // For v_mfma_f64_16x16x4f64 register r of a lane holds D[4*r + lane/16][lane%16]
  // of each 16x16 sub-tile (probed on gfx950).
  // (v_mfma_f32_16x16x4f32: register r of lane l holds D[4*(l/16) + r][l%16].)
  constexpr int kPer = kSlab * TN / S::kThreads;
  static_assert(kPer % 2 == 0, "addends are applied in pairs");
  auto Cs = reinterpret_cast<double2(*)[TN + 1]>(smem_raw);
  const int64_t eo = (int64_t)e;
  double2* D = P.D + eo * P.sD;
  double2* D2 = P.D2 ? P.D2 + eo * P.sD2 : nullptr;
  constexpr int kSlabsPerWaveRow = 32 / kSlab;  // 1, or 2 for the 32x32 tile
#pragma unroll 1
  for (int h = 0; h < TM / kSlab; ++h) {
    const int r0 = m0 + h * kSlab;  // first global row of the slab
    if (wm == h / kSlabsPerWaveRow) {
      const int isub = h % kSlabsPerWaveRow;  // sub-tile row held by a half-row slab
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if (kSlabsPerWaveRow == 2 && i != isub) continue;
        const int ri = kSlabsPerWaveRow == 1 ? i * 16 : 0;
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int rr = kF32 ? ((lane >> 4) * 4 + r) : (r * 4 + (lane >> 4));
            Cs[ri + rr][wn * 32 + j * 16 + (lane & 15)] =
                cmk((double)accr[i][j][r], (double)acci[i][j][r]);
          }
      }
    }
    __syncthreads();
    // Each thread owns elements idx = tid + q*kThreads of the slab (row-major,
    // so global accesses are coalesced along rows); values live in Cs and are
    // updated in pairs: loads of a pair are issued before its stores (pairs,
    // not larger groups, keep the 64x64 kernel within 128 VGPRs unspilled).
    for (int a = 0; a <= P.naddends; ++a) {
      if (a == P.npre && P.d2mode == kD2Partial) {
#pragma unroll 4
        for (int q = 0; q < kPer; ++q) {
          const int idx = tid + q * S::kThreads;
          const int row = r0 + idx / TN, col = n0 + idx % TN;
          if (row < m && col < n) D2[(int64_t)row * P.ldd2 + col] = Cs[idx / TN][idx % TN];
        }
      }
      if (a == P.naddends) break;
      const ZAddend& A = P.ad[a];
      const double2* F = A.F + eo * A.sF;
      const bool use1 = cnz(A.c1), use2 = cnz(A.c2);
#pragma unroll 1
      for (int q0 = 0; q0 < kPer; q0 += 2) {
        double2 f1[2], f2[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int idx = tid + (q0 + u) * S::kThreads;
          const int row = r0 + idx / TN, col = n0 + idx % TN;
          const bool in = row < m && col < n;
          f1[u] = (use1 && in) ? F[(int64_t)row * A.ldf + col] : cmk(0.0, 0.0);
          f2[u] = (use2 && in) ? F[(int64_t)col * A.ldf + row] : cmk(0.0, 0.0);
        }
#pragma unroll
        for (int u = 0; u < 2; ++u) {
          const int idx = tid + (q0 + u) * S::kThreads;
          double2 v = Cs[idx / TN][idx % TN];
          v = cadd(v, cadd(cmul(A.c1, f1[u]), cmul(A.c2, cconj(f2[u]))));
          Cs[idx / TN][idx % TN] = v;
        }
      }
    }
#pragma unroll 4
    for (int q = 0; q < kPer; ++q) {
      const int idx = tid + q * S::kThreads;
      const int row = r0 + idx / TN, col = n0 + idx % TN;
      if (row < m && col < n) {
        const double2 v = Cs[idx / TN][idx % TN];
        D[(int64_t)row * P.ldd + col] = v;
        if (P.d2mode == kD2Copy) D2[(int64_t)row * P.ldd2 + col] = cmul(P.s2, v);
      }
    }
    if (P.d2mode == kD2ConjT) {
      // D2[c][r] = s2 conj(D[r][c]): read the slab transposed from LDS, store
      // runs of kSlab consecutive elements of rows of D2.  The transposed read
      // takes elements that other waves finished in the addend pass: wait for
      // them (the condition is uniform over the workgroup).
      __syncthreads();
#pragma unroll 4
      for (int q = 0; q < kPer; ++q) {
        const int idx = tid + q * S::kThreads;
        const int tr = idx / kSlab, tc = idx % kSlab;
        const int row2 = n0 + tr, col2 = r0 + tc;
        if (row2 < n && col2 < m) D2[(int64_t)row2 * P.ldd2 + col2] = cmul(P.s2, cconj(Cs[tc][tr]));
      }
    }
    __syncthreads();  // the next slab overwrites Cs
  }
}

template <int TM, int TN, int kRole, bool kF32 = false>
hipError_t launch_cfg(const ZGroup& g0, hipStream_t stream) {
  ZGroup g = g0;
  int per = 0;  // workgroups per energy (all problems)
  for (int p = 0; p < g.nprob; ++p) {
    const int tm = (g.p[p].m + TM - 1) / TM, tn = (g.p[p].n + TN - 1) / TN;
    g.tiles_n[p] = tn;
    g.tiles_mn[p] = tm * tn;
    g.wg_base[p] = per;
    per += tm * tn;
  }
  g.wg_base[g.nprob] = per;
  const int64_t total = (int64_t)per * g.nE;
  if (total == 0) return hipSuccess;
  if (total > 0x7fffffff) return hipErrorInvalidValue;
  hipLaunchKernelGGL((zgemm4m_kernel<TM, TN, kRole, kF32>), dim3((unsigned)total),
                     dim3(TileShape<TM, TN, kF32>::kThreads), 0, stream, g);
  return hipGetLastError();
}

// ---------------------------------------------------------------------------
// FP64 products of the sweeps: three real MFMAs per complex product
// ---------------------------------------------------------------------------
//
// P1 = ar br, P2 = ai bi and P3 = (ar + ai)(br + bi) accumulate in three
// accumulator sets; re = P1 - P2, im = P3 - P1 - P2 in the epilogue.  Bound by
// the matrix cores: v_mfma_f64_16x16x4f64 takes 64 cycles of its SIMD, and every
// vector instruction takes its issue cycles from the same pipe (measured with
// twelve independent MFMAs in a loop: 64.4 cycles per MFMA alone; each FP64 add
// in the loop costs 7.8 cycles of MFMA time, each 32-bit VALU instruction or
// LDS access about 3).  So the loop holds almost nothing but MFMAs:
//  * alpha = +-1 and the conjugations never touch an operand.  A conjugated
//    operand changes the sign with which its imaginary part enters the two
//    fragment sums (an fma with a scalar +-1 in the place of the add) and the
//    sign of P2, and a negative term that of all three; the accumulators keep
//    the sum up to those signs, are negated where a term's signs differ from
//    the one before it, and the last signs are applied in the epilogue.  (No
//    product has another alpha: the launch refuses it.)
//  * operands come by buffer loads with one lane offset per element and a scalar
//    offset per k-tile; rows and columns beyond the edge have an offset beyond
//    the buffer, which reads as zero, and so have the inner indices beyond K
//    (kTail: K not a multiple of 8 costs a compare and a select per element).
//  * two k-tiles per loop pass, so that every LDS address is a constant offset.
//  * the reads of the next k-step's fragments, the stores of the next k-tile and
//    the loads of the one after it sit between the MFMAs (scheduled by
//    sched_group_barrier), with one barrier per k-tile, placed between its two
//    k-steps: what is read after it was stored a whole k-step before.
// The epilogue works on the accumulators: register r of a lane holds D[4 r +
// lane / 16][lane % 16] of its 16 x 16 tile, so a store covers four rows of
// 256 contiguous bytes; no LDS pass, no barrier.  Waves whose part of the tile lies beyond the
// matrix only help to stage.
// Measured (MI355X, TFLOP/s by 8 m n k, against the kernel it replaced, which
// staged its epilogue through LDS, waited for its own LDS traffic and relied on
// a third workgroup per CU): 256^3 x 512 energies 93 (76), 512^3 x 16 96 (76),
// 256^3 x 8 81 (48), 208^3 x 64 74 (49), 96^3 x 64 69 (36), 91 x 77 x 65 x 48
// 33 (17); results are bit for bit the same.  92% of the time the matrix cores
// are busy at 512^3; the rest is the FP64 adds of the fragment sums (5%) and
// the epilogue.  Three waves per SIMD at 64 x 64 (162 registers) hide prologues
// and epilogues that two did not (256^3 x 512: 89).
#define QX_SGB(mask, n) __builtin_amdgcn_sched_group_barrier(mask, n, 0)
constexpr int kSgMfma = 0x8, kSgVmemRead = 0x20, kSgDsRead = 0x100, kSgDsWrite = 0x200;

// kFast: every K a multiple of 8; kFastTail: any K; kPlain4M: any K, four MFMAs per
// product (no conjugation, alpha = 1).
enum Form : int { kFast = 0, kFastTail = 1, kPlain4M = 2 };

template <int TM, int TN, int WM, int WN>
struct Tile3M {
  static constexpr int kTK = 8;
  static constexpr int kThreads = 64 * WM * WN;
  static constexpr int SI = TM / WM / 16, SJ = TN / WN / 16;  // 16 x 16 tiles of a wave
  static constexpr int kAPer = TM * kTK / kThreads, kBPer = kTK * TN / kThreads;
  static constexpr int LA = TM + 1, LB = TN + 1;
};

// TM x TN output tile, WM x WN waves, at least MINW waves per SIMD.  kRole only
// separates kernel names in traces: 0 = sweep products, 1 = trailing updates
// inside the blocked inversion.
template <int TM, int TN, int kRole, int WM, int WN, int MINW, int kForm>
__global__ void __launch_bounds__(64 * WM * WN, MINW) zgemm_grouped_kernel(const ZGroup g) {
  if (kRole == 1) __builtin_amdgcn_s_setprio(2);  // the inversion is the longer chain
  using S = Tile3M<TM, TN, WM, WN>;
  constexpr int SI = S::SI, SJ = S::SJ, TK = S::kTK;
  constexpr bool kTail = kForm != kFast, k4M = kForm == kPlain4M;
  __shared__ double2 lds_a[2 * TK * S::LA];
  __shared__ double2 lds_b[2 * TK * S::LB];

  const int per = g.wg_base[g.nprob];
  const int wid = xcd_remap(blockIdx.x, per * g.nE);
  const int e = wid / per;
  const int rem = wid - e * per;
  int p = 0;
  while (p + 1 < g.nprob && rem >= g.wg_base[p + 1]) ++p;
  const ZProblem& P = g.p[p];
  const int tt = rem - g.wg_base[p];
  const int m0 = (tt / g.tiles_n[p]) * TM;
  const int n0 = (tt % g.tiles_n[p]) * TN;
  const int m = P.m, n = P.n;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WN, wn = wave % WN;
  const int l16 = lane & 15, kq = lane >> 4;
  const int mw = m0 + wm * (16 * SI), nw = n0 + wn * (16 * SJ);
  const bool some = mw < m && nw < n;  // this wave has valid outputs

  // `live` waves multiply, the others only stage (two copies of the code, so
  // that the copy without MFMAs does not weigh on the other's registers)
  auto body = [&](auto live) {
  constexpr bool kLive = decltype(live)::value;
  double4_t acc1[SI][SJ], acc2[SI][SJ], acc3[SI][SJ];
#pragma unroll
  for (int i = 0; i < SI; ++i)
#pragma unroll
    for (int j = 0; j < SJ; ++j) acc1[i][j] = acc2[i][j] = acc3[i][j] = double4_t{0, 0, 0, 0};

  double2 ra[S::kAPer], rb[S::kBPer];
  double2 fa[2][SI], fb[2][SJ];
  auto sync = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  };
  const double2* fra = lds_a + kq * S::LA + wm * (16 * SI) + l16;
  const double2* frb = lds_b + kq * S::LB + wn * (16 * SJ) + l16;
  auto read = [&](int fbuf, int buf, int ks) {
#pragma unroll
    for (int i = 0; i < SI; ++i) fa[fbuf][i] = fra[buf * (TK * S::LA) + ks * 4 * S::LA + 16 * i];
#pragma unroll
    for (int j = 0; j < SJ; ++j) fb[fbuf][j] = frb[buf * (TK * S::LB) + ks * 4 * S::LB + 16 * j];
  };
  double sgn_a = 1.0, sgn_b = 1.0;  // -1: the operand is conjugated
  auto mma = [&](int f) {
    if constexpr (k4M) {
#pragma unroll
      for (int i = 0; i < SI; ++i)
#pragma unroll
        for (int j = 0; j < SJ; ++j) {
          acc1[i][j] = mfma(fa[f][i].x, fb[f][j].x, acc1[i][j]);
          acc2[i][j] = mfma(fa[f][i].x, fb[f][j].y, acc2[i][j]);
          acc1[i][j] = mfma_nega(fa[f][i].y, fb[f][j].y, acc1[i][j]);
          acc2[i][j] = mfma(fa[f][i].y, fb[f][j].x, acc2[i][j]);
        }
      return;
    }
    double sa[SI], sb[SJ];
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
      for (int j = 0; j < SJ; ++j) acc1[i][j] = mfma(fa[f][i].x, fb[f][j].x, acc1[i][j]);
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
      for (int j = 0; j < SJ; ++j) acc2[i][j] = mfma(fa[f][i].y, fb[f][j].y, acc2[i][j]);
#pragma unroll
    for (int i = 0; i < SI; ++i) sa[i] = fma(sgn_a, fa[f][i].y, fa[f][i].x);
#pragma unroll
    for (int j = 0; j < SJ; ++j) sb[j] = fma(sgn_b, fb[f][j].y, fb[f][j].x);
#pragma unroll
    for (int i = 0; i < SI; ++i)
#pragma unroll
      for (int j = 0; j < SJ; ++j) acc3[i][j] = mfma(sa[i], sb[j], acc3[i][j]);
  };

  // acc1 and acc3 hold (neg1 ? -1 : 1) times the sum over the terms so far, acc2 (neg2 ? -1 : 1) times it
  bool neg1 = false, neg2 = false;
  auto term = [&](int ti) {
    const ZTerm& T = P.t[ti];
    const bool aN = T.opA == kOpN, bN = T.opB == kOpN;
    const int K = T.k, lda = T.lda, ldb = T.ldb;
    const int nt = (K + TK - 1) / TK;
    if (nt == 0) return;
    const auto rsa = buf_of(T.A + (int64_t)e * T.sA), rsb = buf_of(T.B + (int64_t)e * T.sB);
    const unsigned step_a = 16u * TK * (aN ? 1 : lda), step_b = 16u * TK * (bN ? ldb : 1);
    unsigned offa[S::kAPer], offb[S::kBPer];
    int ka[S::kAPer], kb[S::kBPer];
#pragma unroll
    for (int i = 0; i < S::kAPer; ++i) {
      const int idx = tid + i * S::kThreads;
      const int gm = m0 + (aN ? idx / TK : idx % TM);
      ka[i] = aN ? idx % TK : idx / TM;
      offa[i] = gm < m ? 16u * (aN ? gm * lda + ka[i] : ka[i] * lda + gm) : kOob;
    }
#pragma unroll
    for (int i = 0; i < S::kBPer; ++i) {
      const int idx = tid + i * S::kThreads;
      const int gn = n0 + (bN ? idx % TN : idx / TK);
      kb[i] = bN ? idx / TN : idx % TK;
      offb[i] = gn < n ? 16u * (bN ? kb[i] * ldb + gn : gn * ldb + kb[i]) : kOob;
    }
    {
      const bool t1 = T.alpha.x < 0.0, t2 = t1 != (aN != bN);
      if (ti > 0 && t1 != neg1) {
#pragma unroll
        for (int i = 0; i < SI; ++i)
#pragma unroll
          for (int j = 0; j < SJ; ++j) {
            acc1[i][j] = -acc1[i][j];
            acc3[i][j] = -acc3[i][j];
          }
      }
      if (ti > 0 && t2 != neg2) {
#pragma unroll
        for (int i = 0; i < SI; ++i)
#pragma unroll
          for (int j = 0; j < SJ; ++j) acc2[i][j] = -acc2[i][j];
      }
      neg1 = t1;
      neg2 = t2;
      sgn_a = aN ? 1.0 : -1.0;
      sgn_b = bN ? 1.0 : -1.0;
    }
    double2* wa[S::kAPer];
#pragma unroll
    for (int i = 0; i < S::kAPer; ++i) {
      const int idx = tid + i * S::kThreads;
      wa[i] = lds_a + (aN ? (idx % TK) * S::LA + idx / TK : (idx / TM) * S::LA + idx % TM);
    }
    double2* wb[S::kBPer];
#pragma unroll
    for (int i = 0; i < S::kBPer; ++i) {
      const int idx = tid + i * S::kThreads;
      wb[i] = lds_b + (bN ? (idx / TN) * S::LB + idx % TN : (idx % TK) * S::LB + idx / TK);
    }
    auto load = [&](int t) {
      t = min(t, nt - 1);
      const int kr = K - t * TK;
      const unsigned sa = t * step_a, sb = t * step_b;
#pragma unroll
      for (int i = 0; i < S::kAPer; ++i) ra[i] = buf_load(rsa, !kTail || ka[i] < kr ? offa[i] : kOob, sa);
#pragma unroll
      for (int i = 0; i < S::kBPer; ++i) rb[i] = buf_load(rsb, !kTail || kb[i] < kr ? offb[i] : kOob, sb);
    };
    auto store = [&](int buf) {
#pragma unroll
      for (int i = 0; i < S::kAPer; ++i) wa[i][buf * (TK * S::LA)] = ra[i];
#pragma unroll
      for (int i = 0; i < S::kBPer; ++i) wb[i][buf * (TK * S::LB)] = rb[i];
    };
    load(0);
    store(0);
    load(1);
    sync();
    // One k-tile in LDS stage `cur`; the tile after the last one is loaded and
    // stored again in its place, so that the loop has no condition.
    auto tile = [&](int t, int cur) {
      constexpr int kM = (k4M ? 4 : 3) * SI * SJ, kMem = S::kAPer + S::kBPer;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kLive) read(1, cur, 1);
      store(cur ^ 1);
      load(t + 2);
      if constexpr (kLive) {
        mma(0);
#pragma unroll
        for (int i = 0; i < SI + SJ; ++i) { QX_SGB(kSgMfma, 1); QX_SGB(kSgDsRead, 1); }
#pragma unroll
        for (int i = 0; i < kMem; ++i) { QX_SGB(kSgMfma, 1); QX_SGB(kSgDsWrite, 1); QX_SGB(kSgVmemRead, 1); }
        QX_SGB(kSgMfma, kM);
      }
      __builtin_amdgcn_sched_barrier(0);
      sync();
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (kLive) {
        read(0, cur ^ 1, 0);
        mma(1);
#pragma unroll
        for (int i = 0; i < SI + SJ; ++i) { QX_SGB(kSgMfma, 1); QX_SGB(kSgDsRead, 1); }
        QX_SGB(kSgMfma, kM);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (kLive) read(0, 0, 0);
#pragma unroll 1
    for (int t = 0; t < nt; t += 2) {
      tile(t, 0);
      if (t + 1 == nt) break;
      tile(t + 1, 1);
    }
    // every wave has read this term's last tile before the barrier in its
    // middle; what the last store and read touched is not used
    if (ti + 1 < P.nterms) sync();
  };
  // Written out, not a loop: round a loop the compiler keeps a second copy of
  // every accumulator (64 x 64: 256 registers instead of 166).
  static_assert(sizeof(P.t) / sizeof(P.t[0]) == 2, "a problem has up to two terms");
  if (P.nterms > 0) term(0);
  if (P.nterms > 1) term(1);

  // ---- epilogue, straight from the accumulators ----
  if constexpr (!kLive) return;
  const int64_t eo = e;
  const auto rd = buf_of(P.D + eo * P.sD);
  const auto rd2 = buf_of(P.D2 ? P.D2 + eo * P.sD2 : P.D);
#pragma unroll
  for (int i = 0; i < SI; ++i) {
#pragma unroll
    for (int j = 0; j < SJ; ++j) {
      __builtin_amdgcn_sched_barrier(0);
      const int col = nw + 16 * j + l16, row0 = mw + 16 * i + kq;
      const int rows = col < n ? m : 0;  // rows of this column that are valid
      auto at = [&](int ld, int r) { return row0 + 4 * r < rows ? 16u * ((row0 + 4 * r) * ld + col) : kOob; };
      auto at_t = [&](int ld, int r) { return row0 + 4 * r < rows ? 16u * (col * ld + row0 + 4 * r) : kOob; };
      double2 v[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double p1 = neg1 ? -acc1[i][j][r] : acc1[i][j][r], p2 = neg2 ? -acc2[i][j][r] : acc2[i][j][r];
        const double p3 = neg1 ? -acc3[i][j][r] : acc3[i][j][r];
        v[r] = k4M ? cmk(p1, p2) : cmk(p1 - p2, p3 - p1 - p2);
      }
      for (int a = 0; a <= P.naddends; ++a) {
        if (a == P.npre && P.d2mode == kD2Partial) {
#pragma unroll
          for (int r = 0; r < 4; ++r) buf_store(rd2, at(P.ldd2, r), v[r]);
        }
        if (a == P.naddends) break;
        const ZAddend& A = P.ad[a];
        const auto rf = buf_of(A.F + eo * A.sF);
        if (cnz(A.c1)) {
          double2 f[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) f[r] = buf_load(rf, at(A.ldf, r), 0);
          if (cnz(A.c2)) {
            double2 f2[4];
#pragma unroll
            for (int r = 0; r < 4; ++r) f2[r] = buf_load(rf, at_t(A.ldf, r), 0);
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = cadd(v[r], cadd(cmul(A.c1, f[r]), cmul(A.c2, cconj(f2[r]))));
          } else {
#pragma unroll
            for (int r = 0; r < 4; ++r) v[r] = cadd(v[r], cmul(A.c1, f[r]));
          }
        } else if (cnz(A.c2)) {
          double2 f2[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) f2[r] = buf_load(rf, at_t(A.ldf, r), 0);
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = cadd(v[r], cmul(A.c2, cconj(f2[r])));
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) buf_store(rd, at(P.ldd, r), v[r]);
      if (P.d2mode == kD2Copy) {
#pragma unroll
        for (int r = 0; r < 4; ++r) buf_store(rd2, at(P.ldd2, r), cmul(P.s2, v[r]));
      }
      if (P.d2mode == kD2ConjT) {
#pragma unroll
        for (int r = 0; r < 4; ++r) buf_store(rd2, at_t(P.ldd2, r), cmul(P.s2, cconj(v[r])));
      }
    }
  }
  };
  if (some) body(std::true_type{});
  else body(std::false_type{});
}

template <int TM, int TN, int WM, int WN, int MINW, int kRole>
hipError_t launch_3m(const ZGroup& g0, hipStream_t stream, bool plain4m = false) {
  ZGroup g = g0;
  int per = 0;
  bool unit = true, tail = false;
  for (int p = 0; p < g.nprob; ++p) {
    const int tm = (g.p[p].m + TM - 1) / TM, tn = (g.p[p].n + TN - 1) / TN;
    g.tiles_n[p] = tn;
    g.tiles_mn[p] = tm * tn;
    g.wg_base[p] = per;
    per += tm * tn;
    for (int t = 0; t < g.p[p].nterms; ++t) {
      const ZTerm& T = g.p[p].t[t];
      unit &= T.alpha.y == 0.0 && (T.alpha.x == 1.0 || T.alpha.x == -1.0);
      tail |= T.k % Tile3M<TM, TN, WM, WN>::kTK != 0;
    }
  }
  g.wg_base[g.nprob] = per;
  const int64_t total = (int64_t)per * g.nE;
  if (total == 0) return hipSuccess;
  if (total > 0x7fffffff || !unit) return hipErrorInvalidValue;
  const dim3 grid((unsigned)total), block(64 * WM * WN);
  if constexpr (kRole == 1 && TM == 32 && TN == 32) {
    if (plain4m) {
      hipLaunchKernelGGL((zgemm_grouped_kernel<TM, TN, kRole, WM, WN, MINW, kPlain4M>), grid, block, 0, stream, g);
      return hipGetLastError();
    }
  }
  if (tail) hipLaunchKernelGGL((zgemm_grouped_kernel<TM, TN, kRole, WM, WN, MINW, kFastTail>), grid, block, 0, stream, g);
  else hipLaunchKernelGGL((zgemm_grouped_kernel<TM, TN, kRole, WM, WN, MINW, kFast>), grid, block, 0, stream, g);
  return hipGetLastError();
}

// The 3M tile of a launch: 64 x 64, 64 x 32 or 32 x 32, each by four waves.  A
// larger tile reads less and spends fewer instructions per MFMA (relative
// rates 1, 0.944 and 0.884 at 256^3 x 512), a smaller one wastes less at the edges and
// in the last round over the 256 CUs: time ~ area (rounds + 1/2) / rate, with the
// half round for a first load and an epilogue that nothing hides.  It
// agrees with the fastest of the three at b = 48 ... 512, 8 ... 1024 energies, to
// 4% (us for 64 x 64 / 64 x 32 / 32 x 32: 3 products of 256^3 x 8 49.6 / 39.8 / 40.6,
// 2 of 192^3 x 32 55.6 / 48.5 / 47.0, 4 of 208^3 x 64 303 / 270 / 251, 3 of
// 512^3 x 16 538 / 558 / 592).  Products with K up to 64 (small blocks and the inversion's
// trailing updates) are bound by the latency of that first load and by the
// epilogue, which more and smaller workgroups hide better: no 64 x 64 tile, and 32 x 32 as
// fast per element as 64 x 32 (256 x 192, K = 64, 64 energies: 32.0 / 30.4 /
// 30.0; 3 of 64^3 x 256 34.2 / 34.3 / 32.0; 3 of 48^3 x 1024 87 / 84 / 79).
int pick_3m(const ZGroup& g) {
  const int tm[3] = {64, 64, 32}, tn[3] = {64, 32, 32};
  int kmax = 0;
  for (int p = 0; p < g.nprob; ++p) {
    int k = 0;
    for (int t = 0; t < g.p[p].nterms; ++t) k += g.p[p].t[t].k;
    kmax = k > kmax ? k : kmax;
  }
  const double rate[3] = {1.0, 0.944, kmax <= 64 ? 0.935 : 0.884};
  int best = 0;
  double tbest = 0;
  for (int c = kmax <= 64 ? 1 : 0; c < 3; ++c) {
    int64_t wgs = 0;
    for (int p = 0; p < g.nprob; ++p)
      wgs += (int64_t)((g.p[p].m + tm[c] - 1) / tm[c]) * ((g.p[p].n + tn[c] - 1) / tn[c]);
    wgs *= g.nE;
    const double t = tm[c] * tn[c] * ((double)((wgs + 255) / 256) + 0.5) / rate[c];
    if (tbest == 0 || t < tbest) {
      best = c;
      tbest = t;
    }
  }
  return best;
}

template <int kRole>
hipError_t launch_3m_auto(const ZGroup& g, hipStream_t stream) {
  switch (pick_3m(g)) {
    case 0: return launch_3m<64, 64, 2, 2, 3, kRole>(g, stream);
    case 1: return launch_3m<64, 32, 2, 2, 4, kRole>(g, stream);
    default: return launch_3m<32, 32, 2, 2, 4, kRole>(g, stream);
  }
}

}  // namespace

static_assert(sizeof(ZGroup) <= 4000, "kernel argument block too large");

int tile_m(int cfg) {
  switch (cfg) {
    case kTile32x32: case kTile32x32_3M: return 32;
    case kTile64x32: return 64;
    case kTile128x64: case kTile128x64_3M: return 128;
    default: return 64;
  }
}
int tile_n(int cfg) {
  switch (cfg) {
    case kTile32x32: case kTile32x32_3M: return 32;
    case kTile64x32: return 32;
    case kTile128x64: case kTile128x64_3M: return 64;
    default: return 64;
  }
}

hipError_t launch_zgemm(const ZGroup& g, int cfg, hipStream_t stream) {
  switch (cfg) {
    case kTile32x32: return launch_cfg<32, 32, 0>(g, stream);
    case kTile64x32: return launch_cfg<64, 32, 0>(g, stream);
    case kTile128x64: return launch_cfg<128, 64, 0>(g, stream);
    case kTile64x64_3M: return launch_3m_auto<0>(g, stream);
    case kTile32x32_3M: return launch_3m<32, 32, 2, 2, 4, 0>(g, stream);
    case kTile128x64_3M: return launch_3m<128, 64, 4, 2, 2, 0>(g, stream);
    default: return launch_cfg<64, 64, 0>(g, stream);
  }
}

hipError_t launch_zgemm_f32(const ZGroup& g, int cfg, hipStream_t stream) {
  switch (cfg) {
    case kTile32x32: return launch_cfg<32, 32, 0, true>(g, stream);
    case kTile128x64: return launch_cfg<128, 64, 0, true>(g, stream);
    default: return launch_cfg<64, 64, 0, true>(g, stream);
  }
}

hipError_t launch_zgemm_update(const ZGroup& g, int cfg, hipStream_t stream) {
  switch (cfg) {
    case kTile32x32: return launch_cfg<32, 32, 1>(g, stream);
    case kTile32x32_3M: case kTile64x64_3M: case kTile128x64_3M: return launch_3m_auto<1>(g, stream);
    default: return launch_cfg<64, 64, 1>(g, stream);
  }
}

hipError_t launch_zgemm_narrow(const ZGroup& g, hipStream_t stream) {
  return launch_3m<32, 32, 2, 2, 4, 1>(g, stream, true);
}

}  // namespace qx
