// Batched complex FP64 matrix inverse: blocked in-place Gauss-Jordan
// elimination with partial pivoting, rows never moved (implicit pivoting).
//
// Step c eliminates column c with pivot row pi(c), the row of largest
// |re|+|im| among the rows not yet used as pivots (LAPACK izamax's measure,
// first physical row on ties; from 33 to 512 rows compared by its ten highest
// mantissa bits).  Nothing is swapped: after all steps the matrix
// holds M with A^{-1}[i][j] = M[pi(i)][pi^{-1}(j)].  A panel of NB columns
// [k, k+nb) is eliminated by a panel kernel, one workgroup per energy and
// unblocked GJE on the panel: zinv_panel2_kernel up to 32 rows (two threads per
// row), zinv_panel8_kernel up to 512 (sub-panels of 8 columns), zinv_panel_kernel above
// (16-column panels, one physical row per thread with its panel part in
// registers).  In zinv_panel_kernel a step takes one barrier: before it every
// wave publishes its best candidate row (DPP maximum of the key) and the
// key; after it every thread takes the winner and applies
//   row <- keep row + g prow   (keep = 1, g = -a_r / a_p; for the pivot row
//   keep = 0, g = 1 / a_p)
// with the unscaled pivot row prow, a_r the row's pivot-column value and a_p
// the pivot, so no thread scales the pivot row alone while the others wait.
// The panel kernels write the transformed panel T in place, move the pivot
// rows' non-panel columns to Wp (nb x n) and zero them in S.  The blocked
// GJE update is
//   S[:, nonpanel] += T * Wp[:, nonpanel],
// i.e. S += (T - J) Wp with J[pi(k+q)][q] = 1: J Wp restores the pivot rows,
// which the move to Wp left at zero.
//
// Each update reads and writes all of S (with short K it waits on memory more
// than on the matrix cores), so panels are taken in pairs (P1, P2) and the
// columns R outside both are updated once, with K = nb1 + nb2:
//   1. panel P1 -> T1, WA
//   2. S[:, P2] += T1 WA[:, P2]                   (P2 columns only)
//   3. panel P2 -> T2, WB; the move zeroes rows pi(P2) of T1 as well, and
//      WB[:, P1] holds those rows of T1
//   4. S[:, P1] += T2 WB[:, P1]  (T1 -> T1')
//   5. S[:, R] += T1' WA[:, R] + T2 WB[:, R]     (one pass over R)
// (2 and 4 are K = nb updates of nb columns, run on 32 x 32 tiles.)
// Row by row this is the sequence of the two single-panel updates: rows
// pi(P1) and pi(P2) are zero in S[:, R] before step 5, and rows pi(P2) of T1
// are zero there, so their P1 contribution enters only through WB.  WB's R
// columns were moved before P1's update reached them; the missing
// WB[:, P1] WA[:, R] enters step 5 through T2 WB[:, P1] WA[:, R], which
// T1' carries (step 4 before step 5).
// zinv_finish_kernel then writes Out[i][j] = S[pi(i)][pi^{-1}(j)].
#include <algorithm>

#include "qx_common.h"

namespace qx {

namespace {

template <int NB>
struct PanelAux {
  // byte offsets inside one energy's aux area: two pivot-row buffers (the
  // panels of a pair), then the pivot bookkeeping
  __host__ __device__ static size_t wp(int n, int slot) {
    return (size_t)slot * n * NB * sizeof(double2);
  }
  // pivot row of each step (pi)
  __host__ __device__ static size_t piv(int n) { return wp(n, 2); }
  // step at which each row was the pivot (pi^{-1}; -1 while unused)
  __host__ __device__ static size_t step(int n) { return piv(n) + (size_t)n * sizeof(int); }
  __host__ __device__ static size_t bytes(int n) {
    size_t b = step(n) + (size_t)n * sizeof(int);
    return (b + 255) & ~(size_t)255;
  }
};

inline int panel_nb(int n) { return n <= 512 ? 32 : 16; }

// Maximum over each row of 16 lanes, left in the row's last lane (row_shr
// 1, 2, 4, 8 on both halves of the double; a lane whose source lies before its
// row keeps its own value).
template <int CTRL>
__device__ inline double dpp_d(double v) {
  const long long b = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_update_dpp((int)(b & 0xffffffffll), (int)(b & 0xffffffffll), CTRL,
                                             0xf, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), CTRL, 0xf, 0xf, false);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}
__device__ inline double row_max16_d(double v) {
  v = fmax(v, dpp_d<0x111>(v));
  v = fmax(v, dpp_d<0x112>(v));
  v = fmax(v, dpp_d<0x114>(v));
  v = fmax(v, dpp_d<0x118>(v));
  return v;
}

__device__ inline unsigned row_max16_u(unsigned v) {
  // (a lane whose source lies before its row takes 0)
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, true));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, true));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, true));
  v = max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, true));
  return v;
}
// 1 / d = conj(d) / |d|^2 without a branch: d scaled by a power of two to
// max(|re|, |im|) in [1/2, 1), the reciprocal of |d|^2 by v_rcp_f64 and two
// Newton steps, and the same power of two on the result.
__device__ inline double2 scaled_recip(double2 d) {
  const int ex = __builtin_amdgcn_frexp_exp(fmax(fabs(d.x), fabs(d.y)));
  const double x = __builtin_amdgcn_ldexp(d.x, -ex), y = __builtin_amdgcn_ldexp(d.y, -ex);
  const double m = x * x + y * y;
  double r = __builtin_amdgcn_rcp(m);
  r = fma(r, fma(-m, r, 1.0), r);
  r = fma(r, fma(-m, r, 1.0), r);
  return cmk(__builtin_amdgcn_ldexp(x * r, -ex), __builtin_amdgcn_ldexp(-y * r, -ex));
}
// Maximum of two wave-uniform values, on the scalar unit.
__device__ inline unsigned max_uniform(unsigned a, unsigned b) {
  unsigned r;
  asm("s_max_u32 %0, %1, %2" : "=s"(r) : "s"(a), "s"(b) : "scc");
  return r;
}

// Shared state of one panel workgroup.
// Panel rows are moved between HBM and registers through LDS in chunks of
// kChunk columns, so that global accesses are row-contiguous.  That staging
// area is dynamic LDS of blockDim.x x (kChunk + 1) elements, sized by the
// launch (one row per thread): a static one sized for the largest block
// would cap small matrices at two workgroups per CU.
constexpr int kChunk = 8;

template <int NB>
struct PanelShared {
  double red_key[16];
  int red_idx[16];
  double2 piv_row[NB];
  int s_piv[NB];
};
// The one-thread-per-row panel kernel: per wave its candidate pivot row and
// (key, row), both double-buffered by step.
template <int NB, int MAXW>
struct PanelShared1 {
  double2 cand[2][MAXW][NB];
  double2 red[2][16];
  int s_piv[NB];
};

inline size_t panel_stage_bytes(int threads) {
  return (size_t)threads * (kChunk + 1) * sizeof(double2);
}

template <int NB, int MAXT>
__global__ void __launch_bounds__(MAXT)
zinv_panel_kernel(double2* S, int64_t sS, int n, int k, int nbe, char* aux, int64_t sAux,
                  int wp_slot, int* info, int info_tag, int64_t e0) {
  const int e = blockIdx.x;
  double2* A = S + (int64_t)e * sS;
  char* ax = aux + (int64_t)e * sAux;
  double2* Wp = reinterpret_cast<double2*>(ax + PanelAux<NB>::wp(n, wp_slot));
  int* piv = reinterpret_cast<int*>(ax + PanelAux<NB>::piv(n));
  int* step_of = reinterpret_cast<int*>(ax + PanelAux<NB>::step(n));

  __shared__ PanelShared1<NB, MAXT / 64> sh;
  extern __shared__ __align__(16) double2 stage_raw[];
  auto stage = reinterpret_cast<double2(*)[kChunk + 1]>(stage_raw);

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int r = tid;
  const bool valid = r < n;

  int step = -1;
  if (valid && k > 0) step = step_of[r];
  // The row's panel part lives in registers and is rotated by one position
  // after every step, so the current pivot column is always position 0 and
  // the (rolled) loop body indexes registers with constants only.
  double re[NB], im[NB];
  const int rows = blockDim.x;
  // rows x kChunk tiles, kChunk consecutive lanes per row segment
  // (coalesced); thread tid moves column cc of rows rr0, rr0 + rstep, ...
  // (rows is a multiple of kChunk).  The next chunk's global loads are in
  // flight while the current one passes through LDS.
  const int cc = tid % kChunk, rr0 = tid / kChunk, rstep = rows / kChunk;
  double2 ld[2][kChunk];
  auto fetch = [&](int q0, double2* dst) {
    const bool col_ok = q0 + cc < nbe;
    const double2* src = A + (int64_t)rr0 * n + k + q0 + cc;
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      const int rr = rr0 + i * rstep;
      dst[i] = (rr < n && col_ok) ? src[(int64_t)i * rstep * n] : cmk(0.0, 0.0);
    }
  };
  fetch(0, ld[0]);
#pragma unroll
  for (int c = 0; c < NB / kChunk; ++c) {
    if (c + 1 < NB / kChunk) fetch((c + 1) * kChunk, ld[(c + 1) & 1]);
#pragma unroll
    for (int i = 0; i < kChunk; ++i) stage[rr0 + i * rstep][cc] = ld[c & 1][i];
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kChunk; ++q) {
      const double2 v = stage[r][q];
      re[c * kChunk + q] = v.x;
      im[c * kChunk + q] = v.y;
    }
    __syncthreads();
  }

  // Wave maximum of the pivot key of the current pivot column (position 0)
  // and the lane of its row (lowest on ties; -1 when the wave has no
  // candidate row left): DPP maxima of the four 16-lane rows.
  auto wave_pick = [&](double& wmax, int& cl) {
    double key = (valid && step < 0) ? fabs(re[0]) + fabs(im[0]) : -1.0;
    key = (key != key) ? HUGE_VAL : key;  // NaN: keep the order total
    const double v = row_max16_d(key);
    wmax = fmax(fmax(readlane_d(v, 15), readlane_d(v, 31)),
                fmax(readlane_d(v, 47), readlane_d(v, 63)));
    cl = (int)__builtin_ctzll(__ballot(key == wmax));
  };
  // Every wave publishes its candidate row (unscaled) and (key, row) before
  // the step's one barrier, double-buffered by step; after it every thread
  // takes the winner (first wave on ties: rows ascend with the wave).
  auto publish = [&](int b, double wmax, int cl) {
    if (lane == cl) {
      // as 8-byte halves (ds_write2_b64 takes them from any registers)
      double* ps = reinterpret_cast<double*>(sh.cand[b][wave]);
#pragma unroll
      for (int q = 0; q < NB; ++q) {
        ps[2 * q] = re[q];
        ps[2 * q + 1] = im[q];
      }
    }
    if (lane == 0) sh.red[b][wave] = cmk(wmax, (double)(wave * 64 + cl));
  };
  {
    double wmax;
    int cl;
    wave_pick(wmax, cl);
    publish(0, wmax, cl);
  }

#pragma unroll 1
  for (int jj = 0; jj < nbe; ++jj) {
    const int c = k + jj;
    const int b = jj & 1;
    __syncthreads();
    int p, wb;
    {
      // lane w < nw holds wave w's entry
      const double2 ent = sh.red[b][lane & 15];
      const double key = (lane < nw) ? ent.x : -2.0;
      const double v = row_max16_d(key);
      const double mx = readlane_d(v, 15);
      wb = (int)__builtin_ctzll(__ballot(key == mx) & 0xffffull);
      p = (int)readlane_d(ent.y, wb);
      p = (p < n) ? p : n - 1;  // memory safety only; a candidate row always wins
    }
    const double2* prow = sh.cand[b][wb];
    const double2 pa = prow[0];
    if (tid == 0) {
      sh.s_piv[jj] = p;
      if (pa.x == 0.0 && pa.y == 0.0 && atomicCAS(info, 0, info_tag) == 0) {
        info[1] = (int)(e0 + e);
        info[2] = c;
      }
    }
    const bool me = r == p;
    if (me) step = c;
    // new[q - 1] = keep row[q] + g prow[q] (q >= 1), new[NB - 1] = g, with
    // keep = 1, g = -a_r / a_p for the other rows and keep = 0, g = 1 / a_p
    // for the pivot row (a_r: the row's pivot-column value, a_p: the pivot);
    // pivot-row values in groups of four, the next group's reads issued
    // before the current group's update
    constexpr int G = 4, NG = (NB - 1 + G - 1) / G;
    double2 pv[2][G];
    auto load = [&](int grp, double2* dst) {
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int q = 1 + G * grp + i;
        if (q < NB) dst[i] = prow[q];
      }
    };
    load(0, pv[0]);
    const double2 inv = pivot_recip_inline(pa);
    const double gr = me ? inv.x : -(re[0] * inv.x - im[0] * inv.y);
    const double gi = me ? inv.y : -(re[0] * inv.y + im[0] * inv.x);
    const double keep = me ? 0.0 : 1.0;
    double wmax = -1.0;
    int cl = 0;
#pragma unroll
    for (int grp = 0; grp < NG; ++grp) {
      if (grp + 1 < NG) load(grp + 1, pv[(grp + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < G; ++i) {
        const int q = 1 + G * grp + i;
        if (q < NB) {
          const double2 v = pv[grp & 1][i];
          re[q - 1] = fma(gr, v.x, fma(-gi, v.y, keep * re[q]));
          im[q - 1] = fma(gr, v.y, fma(gi, v.x, keep * im[q]));
        }
      }
      // the next step's pivot search (position 0 is final after the first
      // group) beside the second group's update
      if (grp == 1) wave_pick(wmax, cl);
      __builtin_amdgcn_sched_barrier(0);
    }
    re[NB - 1] = gr;  // the eliminated column rotates into the last position
    im[NB - 1] = gi;
    publish(b ^ 1, wmax, cl);
  }
  __syncthreads();

  // after nbe rotations position q holds panel column (q + nbe) mod NB
  if (valid) step_of[r] = step;
  if (tid < nbe) piv[k + tid] = sh.s_piv[tid];
#pragma unroll
  for (int q0 = 0; q0 < NB; q0 += kChunk) {
#pragma unroll
    for (int q = 0; q < NB; ++q) {
      int col = q + nbe;
      col = (col >= NB) ? col - NB : col;
      if (col >= q0 && col < q0 + kChunk) stage[r][col - q0] = cmk(re[q], im[q]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kChunk; ++i) {
      const int idx = tid + i * rows;
      const int rr = idx / kChunk, q = q0 + idx % kChunk;
      if (rr < n && q < nbe) A[(int64_t)rr * n + k + q] = stage[rr][idx % kChunk];
    }
    __syncthreads();
  }
  // move the pivot rows' non-panel columns to Wp, leaving zeros in S.  Every
  // thread owns one column (rows >= n); the values of 16 pivot rows are loaded
  // before any of them is stored, so the loads are not serialised behind the
  // stores (the pointers may alias as far as the compiler knows).
  if (nbe < n) {
    const int c = tid;
    const bool outside = c < n && (c < k || c >= k + nbe);
#pragma unroll 1
    for (int q0 = 0; q0 < nbe; q0 += 16) {
      double2 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int q = q0 + u;
        v[u] = (outside && q < nbe) ? A[(int64_t)sh.s_piv[q] * n + c] : cmk(0.0, 0.0);
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int q = q0 + u;
        if (outside && q < nbe) {
          Wp[(int64_t)q * n + c] = v[u];
          A[(int64_t)sh.s_piv[q] * n + c] = cmk(0.0, 0.0);
        }
      }
    }
  }
}

// The panel kernel of 33 to 512 rows: 32 columns in four sub-panels of 8.
//
// A step of the elimination is a chain (update the next pivot column, find its
// largest unused entry, publish that row, read it back, scale), and the kernel is bound
// by the length of that chain times n steps: at 4.1 cycles per FP64
// instruction of a wave, 8.5 between dependent ones, 60 per LDS read and 25-55 per
// 16-byte LDS write of a single lane.  So the unblocked elimination runs on 8
// columns, one physical row per thread with its 8 values in registers (7 complex updates
// and 8 published values per step instead of 31 and 32), and the panel's other 24 columns
// follow once per sub-panel on the matrix cores: X += T W, with T the n x 8
// result and W the 8 pivot rows of X (moved out of X, which keeps zeros there; the same
// block step as between panels).  The panel itself stays in registers in the MFMA
// accumulator layout, a wave's 64 rows as 4 x 2 tiles of 16 x 16, and a sub-panel passes
// through the wave's own LDS area into the row layout and back, without a barrier.
//  * pivot key: high word of |re| + |im| with the row in its low bits (10 of its 20
//    mantissa bits decide, the first row on ties), so that a wave's maximum is four
//    32-bit DPP steps and one word says key, row and wave.  A pivot up to 0.1% below the
//    largest entry costs no accuracy (rms error of the selected solve against 64 bits, whole keys / these: 48 rows
//    1.77e-14 / 1.67e-14, 77 1.68e-14 / 1.72e-14, 128 2.06e-14 / 2.06e-14, 512 1.18e-14 / 1.17e-14);
//  * two barriers per step: the waves' keys before the first, and only the winning row
//    is written, before the second (one lane's 8 writes: 264 cycles, by four waves at
//    once 468);
//  * every lane forms the reciprocal of its own value beside the search, so the pivot's
//    is there when its row wins; the pivot row starts from zero (its registers are
//    cleared while the published row is on its way), so an update is four FMAs;
//  * the panel is read and written in 256-byte row segments, all loads in flight,
//    and the pivot rows' columns outside the panel move to Wp under the MFMAs.
// Measured (MI355X, per launch, against one row of 32 columns per thread before): 128 and
// 256 rows, 8 matrices 39.7 us (68), 512 rows, 16 matrices 58 (138), 512 matrices of 256
// rows 82 (131).  Of the 39.7 us the 32 steps take about 19 (some 1400 cycles each), the 256 MFMAs
// of a wave 7, their operands' way through LDS and the pivot rows 8, panel I/O 3.
// Sub-panels of 16 (half the MFMAs, twice the published values) took 47 us, of 16 with
// four lanes per row 57.
constexpr int kSub = 8;
constexpr int kWaveElems = 64 * 9;  // one wave's LDS area (row-major or k-major)

// MW: at most this many waves.
template <int MW>
__global__ void __launch_bounds__(64 * MW, 2)
zinv_panel8_kernel(double2* S, int64_t sS, int n, int k, int nbe, char* aux, int64_t sAux,
                   int wp_slot, int* info, int info_tag, int64_t e0) {
  __builtin_amdgcn_s_setprio(3);  // before the products that share its CU (+1% of a solve)
  constexpr int NB = 32;
  constexpr unsigned kRow = 511u;  // row bits of a pivot key
  const int e = blockIdx.x;
  double2* A = S + (int64_t)e * sS;
  char* ax = aux + (int64_t)e * sAux;
  double2* Wp = reinterpret_cast<double2*>(ax + PanelAux<NB>::wp(n, wp_slot));
  int* piv = reinterpret_cast<int*>(ax + PanelAux<NB>::piv(n));
  int* step_of = reinterpret_cast<int*>(ax + PanelAux<NB>::step(n));

  // the step's pivot row (with the reciprocal of the pivot in its place), and by
  // step parity the key of each wave's best row (0: no unused row left)
  __shared__ double2 cand[kSub];
  __shared__ __align__(16) unsigned ckey[2][(MW + 3) & ~3];
  __shared__ double2 W[kSub][NB];
  __shared__ int s_piv[NB];
  extern __shared__ __align__(16) double2 wave_area[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nw = blockDim.x >> 6;
  const int l16 = lane & 15, kq = lane >> 4;
  const int row = tid, row0 = wave * 64;
  const bool valid = row < n;
  double2* T = wave_area + wave * kWaveElems;
  if (tid < ((MW + 3) & ~3) && tid >= nw) ckey[0][tid] = ckey[1][tid] = 0u;
  // step at which the row was the pivot (-1: unused; rows beyond the matrix count as used)
  int step = valid ? (k > 0 ? step_of[row] : -1) : 0x7fffffff;

  // the panel, zero beyond its rows and columns; register r of tile (rt, ct)
  // is row 16 rt + 4 r + lane / 16 of the wave, column 16 ct + lane % 16
  const auto rs = buf_of(A);
  auto off = [&](int rt, int ct, int r, int kq_, int l16_) {
    const int rr = row0 + rt * 16 + 4 * r + kq_, cc = ct * 16 + l16_;
    return rr < n && cc < nbe ? 16u * (rr * n + k + cc) : kOob;
  };
  double4_t ar[4][2], ai[4][2];
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const double2 v = buf_load(rs, off(rt, ct, r, kq, l16), 0);
        ar[rt][ct][r] = v.x;
        ai[rt][ct][r] = v.y;
      }
  // LDS accesses of one wave are in order; this keeps the compiler from moving them
  auto wave_fence = [&]() {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };

#pragma unroll
  for (int ct = 0; ct < 2; ++ct) {
#pragma unroll 1
    for (int h = 0; h < 2; ++h) {
      const int c0 = ct * 16 + h * 8;  // first column of the sub-panel
      if (c0 >= nbe) break;
      const int steps = min(kSub, nbe - c0);
      const bool own = (l16 >> 3) == h;  // this lane's column of tile ct belongs to it
      if (own) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            T[(rt * 16 + 4 * r + kq) * 9 + (l16 & 7)] = cmk(ar[rt][ct][r], ai[rt][ct][r]);
      }
      wave_fence();
      // the row's 8 values, rotated by one position after every step: the
      // current pivot column is always position 0 and the step loop stays rolled
      double re[kSub], im[kSub];
#pragma unroll
      for (int q = 0; q < kSub; ++q) {
        const double2 v = T[lane * 9 + q];
        re[q] = v.x;
        im[q] = v.y;
      }
      int sub = -1;  // this row's step within the sub-panel
      unsigned kw = 0;
      int cl = 0;
      double2 inv = cmk(0.0, 0.0);
      // the wave's candidate for the column of values (x, y): its key kw, lane cl and
      // reciprocal
      auto search = [&](double x, double y) {
        const unsigned hi = (unsigned)(__double_as_longlong(fabs(x) + fabs(y)) >> 32);
        unsigned key = (hi & ~(2 * kRow + 1)) | (kRow + 1) | (kRow - row);
        key = row_max16_u(step < 0 ? key : 0u);
        kw = max_uniform(max_uniform((unsigned)__builtin_amdgcn_readlane((int)key, 15),
                                     (unsigned)__builtin_amdgcn_readlane((int)key, 31)),
                         max_uniform((unsigned)__builtin_amdgcn_readlane((int)key, 47),
                                     (unsigned)__builtin_amdgcn_readlane((int)key, 63)));
        cl = (int)(kRow - (kw & kRow)) & 63;
        // (every lane that of its own value, beside the search and the row update; the
        // empty asm keeps it from being sunk into the publishing lane's branch)
        inv = scaled_recip(cmk(x, y));
        asm volatile("" : "+v"(inv.x), "+v"(inv.y));
      };
      search(re[0], im[0]);
      if (lane == 0) ckey[0][wave] = kw;
#pragma unroll 1
      for (int j = 0; j < kSub; ++j) {
        const int b = j & 1;
        __syncthreads();
        if (j >= steps) {  // beyond the panel: rotate only
          const double r0 = re[0], i0 = im[0];
#pragma unroll
          for (int q = 1; q < kSub; ++q) {
            re[q - 1] = re[q];
            im[q - 1] = im[q];
          }
          re[kSub - 1] = r0;
          im[kSub - 1] = i0;
          continue;
        }
        unsigned km = 0;
        if constexpr (MW <= 2) {
          km = max(ckey[b][0], MW > 1 ? ckey[b][1] : 0u);
        } else {
#pragma unroll
          for (int w = 0; w < MW; w += 4) {
            const uint4 kk = *reinterpret_cast<const uint4*>(&ckey[b][w]);
            km = max(max(km, max(kk.x, kk.y)), max(kk.z, kk.w));
          }
        }
        km = (unsigned)__builtin_amdgcn_readfirstlane((int)km);
        const int p = min((int)(kRow - (km & kRow)), n - 1);  // (the bound is for memory safety only)
        if (row == p) {
          cand[0] = inv;
#pragma unroll
          for (int q = 1; q < kSub; ++q) cand[q] = cmk(re[q], im[q]);
        }
        // The update is new[q - 1] = row[q] + g prow[q], new[last] = g with
        // g = -a_r / a_p; the pivot row has g = 1 / a_p and starts from zero (while
        // the published row is on its way)
        const bool me = row == p;
        const double a_re = re[0], a_im = im[0];
        if (me) {
          step = k + c0 + j;
          sub = j;
          s_piv[c0 + j] = p;
          if (a_re == 0.0 && a_im == 0.0 && atomicCAS(info, 0, info_tag) == 0) {
            info[1] = (int)(e0 + e);
            info[2] = step;
          }
#pragma unroll
          for (int q = 1; q < kSub; ++q) re[q] = im[q] = 0.0;
        }
        __syncthreads();
        double2 pv[kSub];
#pragma unroll
        for (int q = 0; q < kSub; ++q) pv[q] = cand[q];
        const double2 iv = pv[0];
        const double gr = me ? iv.x : -(a_re * iv.x - a_im * iv.y);
        const double gi = me ? iv.y : -(a_re * iv.y + a_im * iv.x);
        auto upd = [&](int q) {
          re[q - 1] = fma(gr, pv[q].x, fma(-gi, pv[q].y, re[q]));
          im[q - 1] = fma(gr, pv[q].y, fma(gi, pv[q].x, im[q]));
        };
        upd(1);
        search(re[0], im[0]);  // (after the last step: of a finished column, not used)
        if (lane == 0) ckey[b ^ 1][wave] = kw;
#pragma unroll
        for (int q = 2; q < kSub; ++q) upd(q);
        re[kSub - 1] = gr;
        im[kSub - 1] = gi;
      }
      // T, k-major, for the MFMAs and the way back into the tile
      wave_fence();
#pragma unroll
      for (int q = 0; q < kSub; ++q) T[q * 65 + lane] = cmk(re[q], im[q]);
      // the pivot rows leave the panel and leave zeros
      const unsigned long long chosen = __ballot(sub >= 0);
#pragma unroll
      for (int rt = 0; rt < 4; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int base = rt * 16 + 4 * r;
          if (((chosen >> base) & 15) == 0) continue;
          const int s0 = __builtin_amdgcn_readlane(sub, base), s1 = __builtin_amdgcn_readlane(sub, base + 1);
          const int s2 = __builtin_amdgcn_readlane(sub, base + 2), s3 = __builtin_amdgcn_readlane(sub, base + 3);
          const int ps = kq == 0 ? s0 : kq == 1 ? s1 : kq == 2 ? s2 : s3;
          if (ps >= 0) {
#pragma unroll
            for (int t2 = 0; t2 < 2; ++t2) {
              W[ps][t2 * 16 + l16] = cmk(ar[rt][t2][r], ai[rt][t2][r]);
              ar[rt][t2][r] = 0.0;
              ai[rt][t2][r] = 0.0;
            }
          }
        }
      __syncthreads();
      double2 bw[2][2], a[4][2];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int t2 = 0; t2 < 2; ++t2) {
          bw[ks][t2] = W[ks * 4 + kq][t2 * 16 + l16];
          if (ks * 4 + kq >= steps || (t2 == ct && own)) bw[ks][t2] = cmk(0.0, 0.0);
        }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int rt = 0; rt < 4; ++rt) a[rt][ks] = T[(ks * 4 + kq) * 65 + rt * 16 + l16];
      auto mul = [&](int ks) {
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int t2 = 0; t2 < 2; ++t2) {
            ar[rt][t2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt][ks].x, bw[ks][t2].x, ar[rt][t2], 0, 0, 0);
            ai[rt][t2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt][ks].x, bw[ks][t2].y, ai[rt][t2], 0, 0, 0);
            ar[rt][t2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt][ks].y, bw[ks][t2].y, ar[rt][t2], 0, 0, 1);
            ai[rt][t2] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[rt][ks].y, bw[ks][t2].x, ai[rt][t2], 0, 0, 0);
          }
      };
      mul(0);
      __builtin_amdgcn_sched_barrier(0);
      // the pivot rows' columns outside the panel, one column per thread: loaded
      // and, after the other half of the MFMAs, stored
      const bool outside = tid < n && (tid < k || tid >= k + nbe);
      int pr[kSub];
      double2 mv[kSub];
#pragma unroll
      for (int q = 0; q < kSub; ++q) pr[q] = s_piv[c0 + q];
#pragma unroll
      for (int q = 0; q < kSub; ++q)
        mv[q] = buf_load(rs, outside && q < steps ? 16u * (pr[q] * n + tid) : kOob, 0);
      __builtin_amdgcn_sched_barrier(0);
      mul(1);
      __builtin_amdgcn_sched_barrier(0);
      // the sub-panel's columns come back into the tile
      {
        double2 v[16];
#pragma unroll
        for (int q = 0; q < 16; ++q) v[q] = T[(l16 & 7) * 65 + 4 * q + kq];
#pragma unroll
        for (int rt = 0; rt < 4; ++rt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            ar[rt][ct][r] = own ? v[4 * rt + r].x : ar[rt][ct][r];
            ai[rt][ct][r] = own ? v[4 * rt + r].y : ai[rt][ct][r];
          }
      }
      if (outside) {
#pragma unroll
        for (int q = 0; q < kSub; ++q)
          if (q < steps) {
            Wp[(int64_t)(c0 + q) * n + tid] = mv[q];
            A[(int64_t)pr[q] * n + tid] = cmk(0.0, 0.0);
          }
      }
      wave_fence();
    }
  }
  if (valid) step_of[row] = step;
  if (tid < nbe) piv[k + tid] = s_piv[tid];
  // (the offsets are formed again instead of living through the kernel)
  int kq2 = kq, l2 = l16;
  asm volatile("" : "+v"(kq2), "+v"(l2));
#pragma unroll
  for (int ct = 0; ct < 2; ++ct)
#pragma unroll
    for (int rt = 0; rt < 4; ++rt)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        buf_store(rs, off(rt, ct, r, kq2, l2), cmk(ar[rt][ct][r], ai[rt][ct][r]));
}

// The same elimination with two threads per row for 32-column panels: lanes l and l + 32 of a wave hold the two 16-column halves of
// row 32 * wave + (l & 31), so each thread updates 16 values per step instead
// of 32, twice as many waves hide the pivot search, and a 32 x 32 matrix fills
// its wave instead of half of it.  The halves exchange their position 0 once
// per step (the lower half needs the row's pivot-column value, the upper one
// the value that rotates into its last position).  Combined position
// P = 16 h + q rotates exactly as the single-thread row does.
template <int MAXT>
__global__ void __launch_bounds__(MAXT)
zinv_panel2_kernel(double2* S, int64_t sS, int n, int k, int nbe, char* aux, int64_t sAux,
                   int wp_slot, int* info, int info_tag, int64_t e0) {
  constexpr int NB = 32, H = 16;
  const int e = blockIdx.x;
  double2* A = S + (int64_t)e * sS;
  char* ax = aux + (int64_t)e * sAux;
  double2* Wp = reinterpret_cast<double2*>(ax + PanelAux<NB>::wp(n, wp_slot));
  int* piv = reinterpret_cast<int*>(ax + PanelAux<NB>::piv(n));
  int* step_of = reinterpret_cast<int*>(ax + PanelAux<NB>::step(n));

  __shared__ PanelShared<NB> sh;
  extern __shared__ __align__(16) double2 stage_raw[];
  auto stage = reinterpret_cast<double2(*)[kChunk + 1]>(stage_raw);  // [blockDim.x / 2] rows

  const int tid = threadIdx.x;
  const int lane = tid & 63, wave = tid >> 6, nw = blockDim.x >> 6;
  const int h = lane >> 5;
  const int r = wave * 32 + (lane & 31);
  const bool valid = r < n;
  const int nthr = blockDim.x;

  int step = -1;
  if (valid && k > 0) step = step_of[r];
  double re[H], im[H];
#pragma unroll
  for (int q0 = 0; q0 < NB; q0 += kChunk) {
#pragma unroll
    for (int i = 0; i < kChunk / 2; ++i) {
      const int idx = tid + i * nthr;
      const int rr = idx / kChunk, q = q0 + idx % kChunk;
      stage[rr][idx % kChunk] = (rr < n && q < nbe) ? A[(int64_t)rr * n + k + q] : cmk(0.0, 0.0);
    }
    __syncthreads();
    if (h == q0 / H) {
#pragma unroll
      for (int q = 0; q < kChunk; ++q) {
        const double2 v = stage[r][q];
        re[q0 % H + q] = v.x;
        im[q0 % H + q] = v.y;
      }
    }
    __syncthreads();
  }

#pragma unroll 1
  for (int jj = 0; jj < nbe; ++jj) {
    const int c = k + jj;
    const double ore = __shfl_xor(re[0], 32), oim = __shfl_xor(im[0], 32);
    const double pre = h ? ore : re[0], pim = h ? oim : im[0];  // the row's pivot-column value
    double key = (valid && step < 0 && h == 0) ? fabs(pre) + fabs(pim) : -1.0;
    key = (key != key) ? HUGE_VAL : key;  // NaN: keep the order total
    double wmax = key;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) wmax = fmax(wmax, __shfl_xor(wmax, off));
    const unsigned long long hit = __ballot(key == wmax);
    if (lane == 0) {
      sh.red_key[wave] = wmax;
      sh.red_idx[wave] = wave * 32 + ((int)__builtin_ctzll(hit) & 31);
    }
    __syncthreads();
    double bk = sh.red_key[0];
    int p = sh.red_idx[0];
    for (int w = 1; w < nw; ++w) {
      const double ok = sh.red_key[w];
      if (ok > bk) { bk = ok; p = sh.red_idx[w]; }  // waves in row order: first wins ties
    }
    p = (p < n) ? p : n - 1;  // memory safety only; a candidate row always wins
    const bool me = (r == p);
    if (me) {
      if (h == 0 && pre == 0.0 && pim == 0.0) {
        if (atomicCAS(info, 0, info_tag) == 0) {
          info[1] = (int)(e0 + e);
          info[2] = c;
        }
      }
      const double2 inv = crecip(cmk(pre, pim));
      if (h == 0) sh.piv_row[0] = inv;
#pragma unroll
      for (int q = 0; q < H; ++q) {
        if (h == 0 && q == 0) continue;
        sh.piv_row[h * H + q] = cmk(re[q] * inv.x - im[q] * inv.y, re[q] * inv.y + im[q] * inv.x);
      }
      step = c;
    }
    if (tid == 0) sh.s_piv[jj] = p;
    __syncthreads();
    const double keep = me ? 0.0 : 1.0;
    const double fr = me ? -1.0 : pre, fi = me ? 0.0 : pim;
    // the value rotating into the last position: for the lower half the
    // partner's position 0 (panel column 16 + ...), for the upper half the
    // eliminated column itself
    double lr, li;
    if (h == 0) {
      const double2 pv = sh.piv_row[H];
      lr = keep * ore - (fr * pv.x - fi * pv.y);
      li = keep * oim - (fr * pv.y + fi * pv.x);
    } else {
      const double2 p0 = sh.piv_row[0];
      lr = -(fr * p0.x - fi * p0.y);
      li = -(fr * p0.y + fi * p0.x);
    }
    const int base = h * H;
#pragma unroll
    for (int q0 = 1; q0 < H; q0 += 8) {
      asm volatile("" ::: "memory");
#pragma unroll
      for (int q = q0; q < q0 + 8 && q < H; ++q) {
        const double2 pv = sh.piv_row[base + q];
        const double nr = keep * re[q] - (fr * pv.x - fi * pv.y);
        const double ni = keep * im[q] - (fr * pv.y + fi * pv.x);
        re[q - 1] = nr;
        im[q - 1] = ni;
      }
    }
    re[H - 1] = lr;
    im[H - 1] = li;
  }

  // after nbe rotations combined position P = 16 h + q holds panel column (P + nbe) mod NB
  if (valid && h == 0) step_of[r] = step;
  if (tid < nbe) piv[k + tid] = sh.s_piv[tid];
#pragma unroll
  for (int q0 = 0; q0 < NB; q0 += kChunk) {
#pragma unroll
    for (int q = 0; q < H; ++q) {
      int col = h * H + q + nbe;
      col = (col >= NB) ? col - NB : col;
      if (col >= q0 && col < q0 + kChunk) stage[r][col - q0] = cmk(re[q], im[q]);
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < kChunk / 2; ++i) {
      const int idx = tid + i * nthr;
      const int rr = idx / kChunk, q = q0 + idx % kChunk;
      if (rr < n && q < nbe) A[(int64_t)rr * n + k + q] = stage[rr][idx % kChunk];
    }
    __syncthreads();
  }
  // move the pivot rows' non-panel columns to Wp (one column per thread), as
  // in the single-thread-per-row kernel
  if (nbe < n) {
    const int c = tid;
    const bool outside = c < n && (c < k || c >= k + nbe);
#pragma unroll 1
    for (int q0 = 0; q0 < nbe; q0 += 16) {
      double2 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int q = q0 + u;
        v[u] = (outside && q < nbe) ? A[(int64_t)sh.s_piv[q] * n + c] : cmk(0.0, 0.0);
      }
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        const int q = q0 + u;
        if (outside && q < nbe) {
          Wp[(int64_t)q * n + c] = v[u];
          A[(int64_t)sh.s_piv[q] * n + c] = cmk(0.0, 0.0);
        }
      }
    }
  }
}

// Rows staged per workgroup of the finish kernel: rows * n <= kFinishElems,
// rows <= kFinishRows; kFinishThreads threads per workgroup.
constexpr int kFinishElems = 2048;
constexpr int kFinishRows = 256;
constexpr int kFinishThreads = 256;

template <int NB>
__global__ void __launch_bounds__(256)
zinv_finish_kernel(const double2* S, int64_t sS, int n, const char* aux, int64_t sAux,
                   double2* Out, int64_t sOut, int ldo, int rows_per_wg) {
  __shared__ int colsrc[1024];
  __shared__ int rowsrc[kFinishRows];
  __shared__ double2 rows_lds[kFinishElems];
  const int e = blockIdx.y;
  const char* ax = aux + (int64_t)e * sAux;
  const int* piv = reinterpret_cast<const int*>(ax + PanelAux<NB>::piv(n));
  const int* step_of = reinterpret_cast<const int*>(ax + PanelAux<NB>::step(n));
  const int r0 = blockIdx.x * rows_per_wg;
  // (the clamps only matter for NaN input, where the pivot order is meaningless)
  for (int t = threadIdx.x; t < n; t += blockDim.x) {
    const int s = step_of[t];
    colsrc[t] = (s >= 0 && s < n) ? s : 0;
  }
  for (int t = threadIdx.x; t < rows_per_wg; t += blockDim.x) {
    const int pr = (r0 + t < n) ? piv[r0 + t] : 0;
    rowsrc[t] = (pr >= 0 && pr < n) ? pr : 0;
  }
  __syncthreads();
  const double2* A = S + (int64_t)e * sS;
  double2* O = Out + (int64_t)e * sOut;
  const int total = rows_per_wg * n;
  // source rows pi(r) read whole and coalesced, all of a thread's loads in
  // flight before their LDS stores ...
  constexpr int kU = kFinishElems / kFinishThreads;
  double2 v[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int idx = threadIdx.x + u * kFinishThreads;
    const int rr = idx / n, t = idx - rr * n;
    // (indexes clamped so that even a speculated LDS read stays in its array)
    v[u] = (idx < total && r0 + rr < n) ? A[(int64_t)rowsrc[min(rr, kFinishRows - 1)] * n + t]
                                        : cmk(0.0, 0.0);
  }
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int idx = threadIdx.x + u * kFinishThreads;
    if (idx < total) rows_lds[idx] = v[u];
  }
  __syncthreads();
  // ... and permuted by column inside LDS: Out[r][j] = S[pi(r)][pi^{-1}(j)]
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    const int idx = threadIdx.x + u * kFinishThreads;
    const int rr = idx / n, j = idx - rr * n, r = r0 + rr;
    if (idx < total && r < n) O[(int64_t)r * ldo + j] = rows_lds[min(rr * n + colsrc[j], kFinishElems - 1)];
  }
}

template <int NB, int MAXT>
hipError_t zinv_run(double2* S, int64_t sS, int n, int nE, double2* Out, int64_t sOut, int ldo,
                    void* aux, int* info, int info_tag, int64_t e0, int tile_cfg,
                    hipStream_t stream) {
  char* ax = static_cast<char*>(aux);
  const int64_t sAux = (int64_t)PanelAux<NB>::bytes(n);
  const int64_t sAuxC = sAux / (int64_t)sizeof(double2);
  double2* wa = reinterpret_cast<double2*>(ax + PanelAux<NB>::wp(n, 0));
  double2* wb = reinterpret_cast<double2*>(ax + PanelAux<NB>::wp(n, 1));
  // blocks up to 32: two threads per row, which fills the wave that one thread
  // per row would leave half idle (measured at 4096 matrices of 32 x 32: 0.196
  // against 0.275 ms)
  const bool two = NB == 32 && n <= 32;
  const int threads = two ? 2 * ((n + 31) / 32) * 32 : ((n + 63) / 64) * 64;
  auto panel = [&](int k, int nbe, int slot) {
    auto go = [&](auto kern, size_t lds) {
      hipLaunchKernelGGL(kern, dim3(nE), dim3(threads), lds, stream, S, sS, n, k, nbe, ax, sAux, slot, info,
                         info_tag, e0);
    };
    if constexpr (NB == 32) {
      const size_t lds = (size_t)(threads / 64) * kWaveElems * sizeof(double2);
      if (two) go(zinv_panel2_kernel<512>, panel_stage_bytes(threads / 2));
      else if (threads <= 128) go(zinv_panel8_kernel<2>, lds);
      else if (threads <= 256) go(zinv_panel8_kernel<4>, lds);
      else go(zinv_panel8_kernel<8>, lds);
    } else {
      go(zinv_panel_kernel<NB, MAXT>, panel_stage_bytes(threads));
    }
  };
  // operands: columns c0.. of S (stride sS) or of a pivot-row buffer (stride sAuxC), ld n
  auto tS = [&](int c0, const double2* B, int k) {
    return ZTerm{S + c0, B, sS, sAuxC, n, n, kOpN, kOpN, k, 0, cmk(1.0, 0.0)};
  };
  // D (m x nc at D, per-energy stride sD, ld n) += sum of the terms
  auto add = [&](ZGroup& g, int m, int nc, double2* D, int64_t sD, ZTerm t0, const ZTerm* t1) {
    if (m <= 0 || nc <= 0) return;
    ZProblem& P = g.p[g.nprob++];
    P.m = m; P.n = nc; P.nterms = t1 ? 2 : 1; P.naddends = 1; P.npre = 1; P.d2mode = kD2None;
    P.t[0] = t0;
    if (t1) P.t[1] = *t1;
    P.ad[0] = ZAddend{D, sD, n, 0, cmk(1.0, 0.0), cmk(0.0, 0.0)};
    P.D = D; P.sD = sD; P.ldd = n;
  };
  auto run = [&](ZGroup& g) { return g.nprob ? launch_zgemm_update(g, tile_cfg, stream) : hipSuccess; };
  // the narrow K = NB updates of a pair's panel columns on full 32 x 32 tiles
  // (a 64 x 64 tile would be half empty), four waves of 16 x 16 each (256 x 32,
  // K = 32, 64 energies: 7.0 us, one wave of 32 x 32 15.0; 512 energies 37 / 40)
  auto run_narrow = [&](ZGroup& g) {
    return g.nprob ? launch_zgemm_narrow(g, stream) : hipSuccess;
  };
  hipError_t err = hipSuccess;
  for (int k = 0; k < n;) {
    const int nb1 = (n - k < NB) ? (n - k) : NB;
    const int k2 = k + nb1;
    const int nb2 = (n - k2 < NB) ? (n - k2) : NB;
    panel(k, nb1, 0);
    if (nb1 == n) break;  // single panel: nothing else to update
    if (nb2 == 0) {       // last panel, unpaired: columns before it
      ZGroup g{};
      g.nE = nE;
      add(g, n, k, S, sS, tS(k, wa, nb1), nullptr);
      err = run(g);
      break;
    }
    const int k3 = k2 + nb2;  // R = [0, k) and [k3, n)
    {
      ZGroup g{};
      g.nE = nE;
      add(g, n, nb2, S + k2, sS, tS(k, wa + k2, nb1), nullptr);
      if ((err = run_narrow(g)) != hipSuccess) return err;
    }
    panel(k2, nb2, 1);
    {
      // S[:, P1] += T2 WB[:, P1]: T1 becomes T1' = T1 + T2 WB[:, P1], which
      // carries WB's missing P1 contribution into the pass over R below
      ZGroup g{};
      g.nE = nE;
      add(g, n, nb1, S + k, sS, tS(k2, wb + k, nb2), nullptr);
      if ((err = run_narrow(g)) != hipSuccess) return err;
    }
    {
      // S[:, R] += T1' WA[:, R] + T2 WB[:, R]
      ZGroup g{};
      g.nE = nE;
      const ZTerm l2 = tS(k2, wb, nb2), r2 = tS(k2, wb + k3, nb2);
      add(g, n, k, S, sS, tS(k, wa, nb1), &l2);
      add(g, n, n - k3, S + k3, sS, tS(k, wa + k3, nb1), &r2);
      if ((err = run(g)) != hipSuccess) return err;
    }
    k = k3;
  }
  if (err != hipSuccess) return err;
  const int rows = std::min(kFinishElems / n, kFinishRows);  // n <= 1024: at least 2
  hipLaunchKernelGGL((zinv_finish_kernel<NB>), dim3((n + rows - 1) / rows, nE), dim3(256), 0,
                     stream, S, sS, n, ax, sAux, Out, sOut, ldo, rows);
  return hipGetLastError();
}

}  // namespace

// Non-decreasing in n: a workspace sized for the largest block of a geometry
// also holds the need of every smaller block.  Blocks up to 512 use 32-column
// panels (about 1032 n bytes), larger ones 16-column panels (about 520 n), so
// for n > 512 the need of a 512-row block can exceed that of n itself.
size_t zinv_aux_bytes(int n) {
  if (panel_nb(n) == 32) return PanelAux<32>::bytes(n);
  return std::max(PanelAux<32>::bytes(512), PanelAux<16>::bytes(n));
}

hipError_t launch_zinv(double2* S, int64_t sS, int n, int nE, double2* Out, int64_t sOut, int ldo,
                       void* aux, int* info, int info_tag, int64_t e0, int tile_cfg,
                       hipStream_t stream) {
  if (n < 1 || n > 1024) return hipErrorInvalidValue;
  if (nE == 0) return hipSuccess;
  if (panel_nb(n) == 32)
    return zinv_run<32, 512>(S, sS, n, nE, Out, sOut, ldo, aux, info, info_tag, e0, tile_cfg,
                             stream);
  return zinv_run<16, 1024>(S, sS, n, nE, Out, sOut, ldo, aux, info, info_tag, e0, tile_cfg,
                            stream);
}

}  // namespace qx
