// Persistent, on-chip selected solve for geometries whose blocks are all at
// most 32 x 32 (the regime where the launch-per-product sweep is bound by
// HBM round trips of its intermediates and by launch count).
//
// One workgroup (4 waves) runs the whole forward and backward sweep of one
// energy point with every intermediate block in LDS: nine 32 x 32 complex128
// block slots (152 KB, one workgroup per CU).  Inputs are read from HBM when a
// step needs them and results are written once; the only blocks that travel
// back through memory are the left-connected g_i, g^<>_i written by the
// forward sweep and read by the backward one (they are outputs too) and,
// when the current is requested, the Sigma~ blocks.  Workgroups are persistent
// (about one per CU) and pull energy points from a device work queue that
// spans several problems (geometries), ordered by cost on the host; the
// triple products g W g^H run back to back with V = g W never leaving LDS.
//
// The recurrences are those of RGF.selected_solve (rgf.py:216-412); the
// backward lesser/greater blocks use B = g_i Sigma_ij G_jj^H, which serves
// both G^<_ij = -g^<_i R^H + B - U G^<_jj and, as B U^H = Z M^H, the
// T1 = K g^<_i - B U^H term (the same products as the reference, grouped
// to fit the nine slots).
//
// The forward sweep is bound by the inversions, one wave's serial pivot steps (39000
// cycles for 32 x 32, of 100000 per block), so only P = A_ji g_i and S = A_jj - P A_ij stand
// between two of them: while wave 3 inverts S, waves 0 and 1 run the lesser and greater
// chains (V = g_i W_i, g^<>_i = V g_i^H, Y = A_ji g^<>_i, W_j; whole products by one
// wave, in place, no barrier) and wave 2 forms their Q, stores g_i and brings
// the next step's blocks.  Bytes are no limit (2.4 TB/s with 256 energies in flight).
//
// Elsewhere products run in rounds: a round is a set of products that do not depend
// on one another, each wave computes one 16 x 16 output tile of each of them, and
// the round ends with one barrier.  A round whose outputs overwrite one of its own operands
// waits for every wave once more before writing.  With every block above 16 a
// wave has the same tile in all products of a round and their common fragments are read once;
// otherwise tile (w - p) mod 4 of product p, so that products smaller than 16 x 16
// spread over the waves.  Outputs that are only stored (G^R_ij, G^R_ji,
// G^<>_ij and their conjugate transposes) go from registers to HBM without
// an LDS slot.  A round's product takes 2250 cycles, 1536 of them MFMAs; the rest is what a single
// wave per SIMD cannot put beside them (the FP64 adds of 3M, 7.8 cycles each,
// LDS and issue).  The blocks of the next backward step are loaded a
// step ahead, a few in each round.
//
// Measured (MI355X): 32 blocks of 32 x 32, 1024 energies 8.47 -> 5.1 ms, 8 blocks, one energy
// 488 -> 315 us, against the inversion beside the W products only, loads at the
// start of each step and accumulators in AGPRs (copied to be read; this file is
// built with MFMA results in VGPRs).  Errors against 64 bits, rms over four seeds, the elimination column
// by column / in sub-panels: 12 blocks of 16 6.3e-14 / 6.7e-14, 16 of 24 1.09e-13 / 0.86e-13, 8 of 32 8.3e-15 /
// 8.5e-15, 32 of 32 4.58e-14 / 4.45e-14.
//
// Tile products: v_mfma_f64_16x16x4f64, complex as three real products (3M:
// ar br, ai bi, (ar + ai)(br + bi)) into three accumulators; the sign of a
// term and the conjugations of op(A) / op(B) are the MFMA's negate-A
// modifier and the sign of the fragment sums, so no fragment is scaled.  The
// inner index always runs over the 32 padded rows: blocks smaller than 32 are
// zero-padded and inverted blocks carry an identity pad, and no valid output
// element sees a pad product (a pad column of one operand meets a zero pad row
// of the other, or an identity pad meets zeros), so only the pad region of an
// output can differ from zero (it is never stored).  With every block at most
// 16 the inner loop runs over 16 (the KS = 4 kernel).
#include <utility>

#include "qx_common.h"

namespace qx {

namespace {

constexpr int kB = 32;
constexpr int kLd = 33;
constexpr int kNS = 9;
constexpr int kThreads = 256;
typedef double2 Slot[kB][kLd];

struct SmallShared {
  Slot s[kNS];
  double2 w[8][kB + 1];  // inversion: pivot rows of a sub-panel
  int piv[kB];           // inversion: pivot row of each elimination step
  int q_done;            // blocks whose Q^< (odd: and Q^>) is in LDS, times two
  double red[2][4];
  int job;
};

struct Acc {
  double4_t p1, p2, p3;  // ar br, ai bi, (ar + ai)(br + bi)
};

template <bool NEG>
__device__ inline double4_t mf(double a, double b, double4_t c) {
  // f64 MFMA with the BLGP field used as the negate-A modifier
  return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, NEG ? 1 : 0);
}

__device__ inline Acc acc_zero() {
  Acc a;
  a.p1 = double4_t{0, 0, 0, 0};
  a.p2 = a.p1;
  a.p3 = a.p1;
  return a;
}

// acc += (NEG ? -1 : 1) op(A) op(B) over one k-step of 4; op = plain or conjugate
// transpose (AH / BH).  With op(A) = (ar, sa ai) and op(B) = (br, sb bi): P1 +=
// ar br, P2 += sa sb ai bi, P3 += (ar + sa ai)(br + sb bi), each negated for NEG.
template <bool AH, bool BH, bool NEG>
__device__ inline void mma_step(Acc& c, double2 a, double2 b) {
  const double sa = AH ? a.x - a.y : a.x + a.y;
  const double sb = BH ? b.x - b.y : b.x + b.y;
  c.p1 = mf<NEG>(a.x, b.x, c.p1);
  c.p2 = mf<NEG != (AH != BH)>(a.y, b.y, c.p2);
  c.p3 = mf<NEG>(sa, sb, c.p3);
}

// The same over KS k-steps for this wave's tile (tr, tc).  All fragments are read
// before the first MFMA, so the MFMA chain does not wait on LDS.
template <int KS, bool AH, bool BH, bool NEG>
__device__ inline void mma(Acc& c, const Slot& A, const Slot& B, int tr, int tc, int lane) {
  const int l16 = lane & 15, kq = lane >> 4;
  const int row = tr * 16 + l16, col = tc * 16 + l16;
  double2 a[KS], b[KS];
#pragma unroll
  for (int s = 0; s < KS; ++s) {
    const int kk = s * 4 + kq;
    a[s] = AH ? A[kk][row] : A[row][kk];
    b[s] = BH ? B[col][kk] : B[kk][col];
  }
#pragma unroll
  for (int s = 0; s < KS; ++s) mma_step<AH, BH, NEG>(c, a[s], b[s]);
}

// Register r of a lane holds tile element (4 r + lane / 16, lane % 16).
__device__ inline void tile_vals(const Acc& c, double2 (&v)[4]) {
#pragma unroll
  for (int r = 0; r < 4; ++r) v[r] = cmk(c.p1[r] - c.p2[r], c.p3[r] - c.p1[r] - c.p2[r]);
}

__device__ inline int tile_row(int tr, int r, int lane) { return tr * 16 + 4 * r + (lane >> 4); }
__device__ inline int tile_col(int tc, int lane) { return tc * 16 + (lane & 15); }
// Tile of product p of a round computed by `wave`: with every block above 16 (kFull)
// the same one for all products, which then share operand fragments; else
// rotated, so that products with a single live tile spread over the waves.
template <bool kFull>
__device__ inline void tile_of(int p, int wave, int& tr, int& tc) {
  const int t = kFull ? wave : (wave - p) & 3;
  tr = t >> 1;
  tc = t & 1;
}

// Global memory is accessed by buffer loads and stores: an element outside its
// block has an offset beyond the buffer, which reads as zero and is not
// written, so that no access needs a branch.  (They count on the vector-memory counter
// only: an LDS wait does not also wait for prefetches still in flight.)
__device__ inline unsigned goff(int ld, int rows, int cols, int r, int c) {
  return r < rows && c < cols ? 16u * (unsigned)(r * ld + c) : kOob;
}
// Element i of what begins at p: within 2 GiB, so p is an energy's own part of an array.
__device__ inline void gput(double2* p, int i, double2 v) { buf_store(buf_of(p), 16u * (unsigned)i, v); }
__device__ void gput(double2* p, int64_t i, double2 v) = delete;

// Element of a global block (row-major, ld), zero outside rows x cols and without a block.
__device__ inline double2 gld(const double2* F, int ld, int rows, int cols, int r, int c) {
  return buf_load(buf_of(F), goff(ld, F ? rows : 0, cols, r, c), 0);
}

// One product's epilogue ingredients: up to three addends
//   c1 * F[r][c] + c2 * conj(F[c][r])
// from an LDS slot (s), or this thread's four tile elements prefetched into
// registers (r).
struct Add {
  const Slot* s;
  double c1, c2;  // real coefficients suffice for every use here
  const double2* r;
};
__device__ inline Add add_slot(const Slot& s, double c1, double c2 = 0.0) { return Add{&s, c1, c2, nullptr}; }
__device__ inline Add add_regs(const double2* r) { return Add{nullptr, 1.0, 0.0, r}; }
__device__ inline Add add_none() { return Add{nullptr, 0.0, 0.0, nullptr}; }

__device__ inline double2 add_val(const Add& a, int q, int r, int c) {
  if (a.r) return a.r[q];
  double2 out = cmk(0.0, 0.0);
  if (a.s) {
    const Slot& s = *a.s;
    if (a.c1 != 0.0) out = cmk(a.c1 * s[r][c].x, a.c1 * s[r][c].y);
    if (a.c2 != 0.0) {
      const double2 t = s[c][r];
      out = cadd(out, cmk(a.c2 * t.x, -a.c2 * t.y));
    }
  }
  return out;
}

// Where a product's tile goes: an LDS slot (whole padded tile), a global
// block (valid rows x cols, row-major, scaled) and / or the conjugate
// transpose of the valid part into a second global block (gt[c][r]).
struct Dst {
  int slot = -1;
  double2* g = nullptr;
  int ld = 0, rows = 0, cols = 0;
  double gs = 1.0;
  double2* gt = nullptr;
  int ldt = 0;
  double ts = 1.0;
  double2* keep = nullptr;  // this thread's four elements (registers)
  __device__ Dst glob(double2* p, int ld_, int rows_, int cols_, double s = 1.0) const {
    Dst d = *this;
    d.g = p;
    d.ld = ld_;
    d.rows = rows_;
    d.cols = cols_;
    d.gs = s;
    return d;
  }
  __device__ Dst globT(double2* p, int ldt_, double s) const {
    Dst d = *this;
    d.gt = p;
    d.ldt = ldt_;
    d.ts = s;
    return d;
  }
};
__device__ inline Dst kept(Dst d, double2* keep) {
  d.keep = keep;
  return d;
}
__device__ inline Dst to_slot(int s) {
  Dst d;
  d.slot = s;
  return d;
}
__device__ inline Dst to_glob(double2* p, int ld, int rows, int cols, double s = 1.0) {
  return Dst{}.glob(p, ld, rows, cols, s);
}

// A product of a round: D (m x n valid) = terms + addends.  `on` = false skips
// the product (uniform).
template <typename T>
struct Prod {
  bool on;
  int m, n;
  T terms;  // void(Acc&, int tr, int tc, int lane)
  Dst d;
  Add a0, a1, a2;
};
template <typename T>
__device__ inline Prod<T> prod(int m, int n, T terms, Dst d, Add a0 = add_none(), Add a1 = add_none(),
                               Add a2 = add_none(), bool on = true) {
  return Prod<T>{on, m, n, terms, d, a0, a1, a2};
}

template <bool kFull, int I, typename T>
__device__ inline void compute(const Prod<T>& p, double2 (&v)[4], int wave, int lane) {
  int tr, tc;
  tile_of<kFull>(I, wave, tr, tc);
  if (!p.on) return;
  if (kFull || (tr * 16 < p.m && tc * 16 < p.n)) {
    Acc acc = acc_zero();
    p.terms(acc, tr, tc, lane);
    tile_vals(acc, v);
  } else {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = cmk(0.0, 0.0);
  }
  const Add adds[3] = {p.a0, p.a1, p.a2};
  const int col = tile_col(tc, lane);
#pragma unroll
  for (int a = 0; a < 3; ++a) {
#pragma unroll
    for (int r = 0; r < 4; ++r) v[r] = cadd(v[r], add_val(adds[a], r, tile_row(tr, r, lane), col));
  }
}

template <bool kFull, int I, typename T>
__device__ inline void emit(SmallShared& sh, const Prod<T>& p, const double2 (&v)[4], int wave,
                            int lane) {
  if (!p.on) return;
  int tr, tc;
  tile_of<kFull>(I, wave, tr, tc);
  const int col = tile_col(tc, lane);
  const Dst& d = p.d;
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    const int row = tile_row(tr, r, lane);
    if (d.keep) d.keep[r] = v[r];
    if (d.slot >= 0) sh.s[d.slot][row][col] = v[r];
    if (d.g) buf_store(buf_of(d.g), goff(d.ld, d.rows, d.cols, row, col), cmk(d.gs * v[r].x, d.gs * v[r].y));
    if (d.gt) buf_store(buf_of(d.gt), goff(d.ldt, d.cols, d.rows, col, row), cmk(d.ts * v[r].x, -d.ts * v[r].y));
  }
}

template <bool kFull, typename... P, size_t... I>
__device__ inline void round_impl(SmallShared& sh, bool sync_first, std::index_sequence<I...>,
                                  const P&... ps) {
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  double2 v[sizeof...(P)][4];
  (compute<kFull, I>(ps, v[I], wave, lane), ...);
  if (sync_first) __syncthreads();
  (emit<kFull, I>(sh, ps, v[I], wave, lane), ...);
  __syncthreads();
}

// Runs the products of one round and publishes their outputs (trailing
// barrier).  `sync_first`: wait for every wave between computing and writing,
// needed when an output slot is an operand or slot addend of any product of
// the round (other than its own elements as an addend).
template <bool kFull, typename... P>
__device__ inline void run_round(SmallShared& sh, bool sync_first, const P&... ps) {
  round_impl<kFull>(sh, sync_first, std::index_sequence_for<P...>{}, ps...);
}

// A global block (rows x cols, ld) on its way into a slot, zero-filled, with c2 *
// src2 (same shape; optional) added and `pad` on the diagonal beyond the valid
// square (the identity pad of a block about to be inverted).  Thread t moves
// elements t + 256 q (q < 4) of the padded 32 x 32 block.
struct Blk {
  int s;
  const double2* src;
  int ld, rows, cols;
  const double2* src2;
  double c2, pad;
};
__device__ inline Blk blk(int s, const double2* src, int ld, int rows, int cols,
                          const double2* src2 = nullptr, double c2 = 0.0, double pad = 0.0) {
  return Blk{s, src, ld, rows, cols, src2, c2, pad};
}
// Only loads (unless there is a src2): nothing here waits for them.
__device__ inline void fetch_blk(const Blk& b, double2 (&v)[4]) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int idx = tid + q * kThreads;
    v[q] = gld(b.src, b.ld, b.rows, b.cols, idx >> 5, idx & 31);
  }
  if (b.src2) {
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const int idx = tid + q * kThreads;
      const double2 w = gld(b.src2, b.ld, b.rows, b.cols, idx >> 5, idx & 31);
      v[q] = cmk(v[q].x + b.c2 * w.x, v[q].y + b.c2 * w.y);
    }
  }
}
__device__ inline void commit_blk(SmallShared& sh, int s, const double2 (&v)[4], int rows = kB, double pad = 0.0) {
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const int idx = tid + q * kThreads;
    const int r = idx >> 5, c = idx & 31;
    double2 x = v[q];
    if (pad != 0.0 && r == c && r >= rows) x.x = pad;
    sh.s[s][r][c] = x;
  }
}
// The global loads of all NB blocks are issued before the barrier that
// protects the slots' previous readers, so the blocks share one memory
// latency; the caller synchronises before reading the slots.
template <int NB>
__device__ inline void load_blks(SmallShared& sh, const Blk (&b)[NB]) {
  double2 v[NB][4];
#pragma unroll
  for (int i = 0; i < NB; ++i) fetch_blk(b[i], v[i]);
  __syncthreads();  // the slots' previous content may still be read
#pragma unroll
  for (int i = 0; i < NB; ++i) commit_blk(sh, b[i].s, v[i], b[i].rows, b[i].pad);
}

// The same by one wave alone: global loads now, the slot written by wave_commit.
__device__ inline void wave_fetch(double2 (&v)[16], const double2* src, int ld, int rows, int cols, int lane) {
#pragma unroll
  for (int q = 0; q < 16; ++q) v[q] = gld(src, ld, rows, cols, 2 * q + (lane >> 5), lane & 31);
}
__device__ inline void wave_commit(SmallShared& sh, int s, const double2 (&v)[16], int lane, int rows = kB,
                                   double pad = 0.0) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int r = 2 * q + (lane >> 5), c = lane & 31;
    double2 x = v[q];
    if (pad != 0.0 && r == c && r >= rows) x.x = pad;
    sh.s[s][r][c] = x;
  }
}

// Global write of the valid part of a square slot by one wave.
__device__ inline void wave_store_blk(double2* dst, int ld, int b, const Slot& s, int lane) {
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int r = 2 * q + (lane >> 5), c = lane & 31;
    buf_store(buf_of(dst), goff(ld, b, b, r, c), s[r][c]);
  }
}

// Global write of a slot's valid part after a barrier.  mode 0: dst = s;
// 2: dst = (s - s^H) / 2 (square).
__device__ inline void store_blk(double2* dst, int ld, int rows, int cols, const Slot& s, int mode) {
  if (!dst) return;
  const int tid = threadIdx.x;
#pragma unroll
  for (int q = 0; q < kB * kB / kThreads; ++q) {
    const int idx = tid + q * kThreads;
    const int r = idx >> 5, c = idx & 31;
    double2 v = s[r][c];
    if (mode == 2) {
      const double2 l = s[c][r];
      v = cmk(0.5 * (v.x - l.x), 0.5 * (v.y + l.y));
    }
    buf_store(buf_of(dst), goff(ld, rows, cols, r, c), v);
  }
}

// Maximum with the value kCtl (row_shr 1, 2, 4, 8) lanes before, zero where that lies
// before the row of 16: the four in turn leave the row's maximum in its last lane.
template <int kCtl>
__device__ inline unsigned dpp_max(unsigned v) {
  return max(v, (unsigned)__builtin_amdgcn_update_dpp(0, (int)v, kCtl, 0xf, 0xf, true));
}

// v_permlane16_swap: lanes 16-31 and 48-63 of x and lanes 0-15 and 32-47 of y
// change places; v_permlane32_swap: lanes 32-63 of x and 0-31 of y.
__device__ inline void swap16(double& x, double& y) {
  const long long a = __double_as_longlong(x), b = __double_as_longlong(y);
  const auto lo = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
  x = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
  y = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}
__device__ inline void swap32(double& x, double& y) {
  const long long a = __double_as_longlong(x), b = __double_as_longlong(y);
  const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(a >> 32), (unsigned)(b >> 32), false, false);
  x = __longlong_as_double(((long long)hi[0] << 32) | lo[0]);
  y = __longlong_as_double(((long long)hi[1] << 32) | lo[1]);
}

__device__ inline void wave_fence() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// Gauss-Jordan inverse of the n x n valid part of slot ms (identity pad beyond n) in place,
// with partial pivoting and no row moves, by ONE wave (the others work
// meanwhile; no barrier).  Column c is eliminated with the unused row of largest |re| + |im|
// (compared on its high word without six bits, first row on ties): pad rows have
// zeros in valid columns, so they are picked for pad columns only.
//
// Blocked like the larger inversion's panels: 8 columns at a time, the other
// columns once per sub-panel by MFMA, X += T W with T the sub-panel's result and W the pivot
// rows of X (which leave X as zeros).  A step is bound by the instructions of one wave (660
// cycles; 1800 with 16 columns per lane updated in every step), so:
//  * a lane holds row l % 32 of the sub-panel (both halves the same rows) and the pivot row
//    comes as scalars: 32 v_readlane at 8 cycles, cheaper than ds_bpermute (11 each)
//    or a way through LDS;
//  * every lane forms the reciprocal of its own entry beside the search (DPP maximum)
//    and the other columns' updates;
//  * the matrix is held transposed in the MFMA accumulator layout (lane: row 16 rt + l % 16,
//    register u: column 4 u + l / 16), where one v_permlane16_swap and two v_permlane32_swap
//    turn four columns into rows, and one v_permlane16_swap turns T into the right operand,
//    which is also the sub-panel's new content.  Only W goes through LDS.
// Of 9400 cycles per sub-panel the steps take 5300, the 32 MFMAs 2000, W 1100, the
// change of layout 600.  NT: 16 x 16 tiles per side (1: n <= 16).
template <int NT>
__device__ __forceinline__ void invert_wave(SmallShared& sh, int ms, int n, int* info, int tag,
                                            int64_t energy) {
  constexpr int NU = 4 * NT;  // units of four columns
  const int lane = threadIdx.x & 63, l16 = lane & 15, kq = lane >> 4, row = lane & 31;
  const bool low = lane < 32;
  double xr[NT][NU], xi[NT][NU];
#pragma unroll
  for (int rt = 0; rt < NT; ++rt)
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const double2 v = sh.s[ms][16 * rt + l16][4 * u + kq];
      xr[rt][u] = v.x;
      xi[rt][u] = v.y;
    }
  unsigned unused = row < 16 * NT ? ~0u : 0u;
  int step = row, zero_at = -1;
  const int panels = (n + 7) >> 3;
#pragma unroll 1
  for (int s = 0; s < panels; ++s) {
    // units 0 and 1 into rows
    double re[8], im[8];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      auto rows = [&](double a, double b, double* t) {
        swap16(a, b);
        double a2 = a, b2 = b;
        swap32(a, a2);
        swap32(b, b2);
        t[4 * ks] = a;
        t[4 * ks + 1] = b;
        t[4 * ks + 2] = a2;
        t[4 * ks + 3] = b2;
      };
      rows(xr[0][ks], NT > 1 ? xr[NT - 1][ks] : 0.0, re);
      rows(xi[0][ks], NT > 1 ? xi[NT - 1][ks] : 0.0, im);
    }
    int sub = -1, p = 0;
    unsigned mx = 0;
    double2 iv = cmk(0.0, 0.0);
    // The search of the next pivot column (its values x, y in re[0], im[0]) and the
    // reciprocals of its entries, in stages with beside(k) between them
    auto search = [&](auto beside) {
      const double x = re[0], y = im[0];
      auto stage = [&](auto k) {
        beside(k);
        __builtin_amdgcn_sched_barrier(0);
      };
      const double sum = fabs(x) + fabs(y);
      double big;
      asm("v_max_f64 %0, |%1|, |%2|" : "=v"(big) : "v"(x), "v"(y));
      stage(std::integral_constant<int, 0>{});
      unsigned key = (((unsigned)(__double_as_longlong(sum) >> 32) & ~63u) | (unsigned)(63 - row)) & unused;
      const int ex = -__builtin_amdgcn_frexp_exp(big);
      stage(std::integral_constant<int, 1>{});
      key = dpp_max<0x111>(key);
      const double sx = __builtin_amdgcn_ldexp(x, ex), sy = __builtin_amdgcn_ldexp(y, ex);
      stage(std::integral_constant<int, 2>{});
      key = dpp_max<0x112>(key);
      double m = sx * sx;
      stage(std::integral_constant<int, 3>{});
      m = fma(sy, sy, m);
      stage(std::integral_constant<int, 4>{});
      key = dpp_max<0x114>(key);
      double r = __builtin_amdgcn_rcp(m);
      stage(std::integral_constant<int, 5>{});
      double d = fma(-m, r, 1.0);
      stage(std::integral_constant<int, 6>{});
      key = dpp_max<0x118>(key);
      r = fma(r, d, r);
      stage(std::integral_constant<int, 7>{});
      d = fma(-m, r, 1.0);
      unsigned m0 = (unsigned)__builtin_amdgcn_readlane((int)key, 15);
      unsigned m1 = NT > 1 ? (unsigned)__builtin_amdgcn_readlane((int)key, 31) : 0u;
      stage(std::integral_constant<int, 8>{});
      r = fma(r, d, r);
      mx = m0 > m1 ? m0 : m1;
      p = 31 - (int)(mx & 31u);
      stage(std::integral_constant<int, 9>{});
      double ix = sx * r, iy = -sy * r;
      stage(std::integral_constant<int, 10>{});
      ix = __builtin_amdgcn_ldexp(ix, ex);
      iy = __builtin_amdgcn_ldexp(iy, ex);
      stage(std::integral_constant<int, 11>{});
      iv = cmk(readlane_d(ix, p), readlane_d(iy, p));
    };
    search([](auto) {});
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      double2 pv[8];
#pragma unroll
      for (int q = 1; q < 8; ++q) pv[q] = cmk(readlane_d(re[q], p), readlane_d(im[q], p));
      double ax = re[0], ay = im[0];
      if (mx < 64u) {  // (a pivot of zero or next to it)
        if (row == p && ax == 0.0 && ay == 0.0 && 8 * s + j < n) zero_at = 8 * s + j;
      }
      // new[q - 1] = row[q] - g prow[q], new[last] = -g with g = a_r / a_p; the
      // pivot row has a_r = -1 and starts from zero
      if (row == p) {
        unused = 0u;
        step = 8 * s + j;
        sub = j;
        ax = -1.0;
        ay = 0.0;
#pragma unroll
        for (int q = 1; q < 8; ++q) re[q] = im[q] = 0.0;
      }
      const double gx = ax * iv.x - ay * iv.y, gy = ax * iv.y + ay * iv.x;
      double ur = 0.0, ui = 0.0;
      auto inner = [&](int q) {
        ur = fma(gy, pv[q].y, re[q]);
        ui = fma(-gy, pv[q].x, im[q]);
      };
      auto outer = [&](int q) {
        re[q - 1] = fma(-gx, pv[q].x, ur);
        im[q - 1] = fma(-gx, pv[q].y, ui);
      };
      inner(1);
      outer(1);
      if (j < 7) {
        search([&](auto k) {
          constexpr int q = 2 + decltype(k)::value / 2;
          if constexpr (decltype(k)::value % 2 == 0) inner(q);
          else outer(q);
        });
      } else {
#pragma unroll
        for (int q = 2; q < 8; ++q) {
          inner(q);
          outer(q);
        }
      }
      re[7] = -gx;
      im[7] = -gy;
    }
    // the pivot rows leave the other columns and leave zeros
    {
      const auto sw = __builtin_amdgcn_permlane16_swap((unsigned)sub, (unsigned)sub, false, false);
#pragma unroll
      for (int rt = 0; rt < NT; ++rt) {
        const int ps = (int)sw[rt];
        if (ps >= 0) {
#pragma unroll
          for (int u = 2; u < NU; ++u) {
            sh.w[ps][4 * u + kq] = cmk(xr[rt][u], xi[rt][u]);
            xr[rt][u] = xi[rt][u] = 0.0;
          }
        }
      }
    }
    // T as the right operand, which is also the new content of its units
    double tr[2][2], ti[2][2];  // [ks][rt]
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      tr[ks][0] = low ? re[4 * ks] : re[4 * ks + 2];
      tr[ks][1] = low ? re[4 * ks + 1] : re[4 * ks + 3];
      ti[ks][0] = low ? im[4 * ks] : im[4 * ks + 2];
      ti[ks][1] = low ? im[4 * ks + 1] : im[4 * ks + 3];
      swap16(tr[ks][0], tr[ks][1]);
      swap16(ti[ks][0], ti[ks][1]);
    }
    wave_fence();
    double2 w[2][NT];  // [ks][ct]
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int ct = 0; ct < NT; ++ct) {
        w[ks][ct] = sh.w[4 * ks + kq][16 * ct + l16];
        if (ct == 0 && l16 < 8) w[ks][ct] = cmk(0.0, 0.0);
      }
    wave_fence();
    double4_t dr[NT][NT], di[NT][NT];
#pragma unroll
    for (int ct = 0; ct < NT; ++ct)
#pragma unroll
      for (int rt = 0; rt < NT; ++rt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          dr[rt][ct][r] = xr[rt][4 * ct + r];
          di[rt][ct][r] = xi[rt][4 * ct + r];
        }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int ct = 0; ct < NT; ++ct)
#pragma unroll
          for (int rt = 0; rt < NT; ++rt) {
            if (f == 0) dr[rt][ct] = mf<false>(w[ks][ct].x, tr[ks][rt], dr[rt][ct]);
            if (f == 1) di[rt][ct] = mf<false>(w[ks][ct].x, ti[ks][rt], di[rt][ct]);
            if (f == 2) dr[rt][ct] = mf<true>(w[ks][ct].y, ti[ks][rt], dr[rt][ct]);
            if (f == 3) di[rt][ct] = mf<false>(w[ks][ct].y, tr[ks][rt], di[rt][ct]);
          }
    // the next sub-panel's units come first
#pragma unroll
    for (int rt = 0; rt < NT; ++rt) {
#pragma unroll
      for (int u = 0; u < NU - 2; ++u) {
        xr[rt][u] = dr[rt][(u + 2) >> 2][(u + 2) & 3];
        xi[rt][u] = di[rt][(u + 2) >> 2][(u + 2) & 3];
      }
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        xr[rt][NU - 2 + ks] = tr[ks][rt];
        xi[rt][NU - 2 + ks] = ti[ks][rt];
      }
    }
  }
  if (__any(zero_at >= 0)) {
    int first = zero_at >= 0 ? zero_at : kB;
#pragma unroll
    for (int o = 16; o > 0; o >>= 1) first = min(first, __shfl_xor(first, o));
    if (lane == 0 && atomicCAS(info, 0, tag) == 0) {
      info[1] = (int)energy;
      info[2] = first;
    }
  }
  // units 0 .. NU - 1 now hold columns 8 panels .. in turn; Out[i][j] = M[pi(i)][pi^-1(j)]: row R goes to row step(R), column C to column pi(C)
  if (low) sh.piv[step & 31] = row;
  const auto so = __builtin_amdgcn_permlane16_swap((unsigned)step, (unsigned)step, false, false);
  wave_fence();
  int pc[NU];
#pragma unroll
  for (int u = 0; u < NU; ++u) pc[u] = sh.piv[(4 * u + 8 * panels + kq) & (16 * NT - 1)] & 31;
#pragma unroll
  for (int rt = 0; rt < NT; ++rt)
#pragma unroll
    for (int u = 0; u < NU; ++u) sh.s[ms][(int)so[rt] & 31][pc[u]] = cmk(xr[rt][u], xi[rt][u]);
}

// tr(X1 Y1) - tr(X2 Y2) over the valid b x b parts; every thread gets it.
__device__ double2 trace2(SmallShared& sh, const Slot& X1, const Slot& Y1, const Slot& X2,
                          const Slot& Y2, int b) {
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  double sr = 0.0, si = 0.0;
#pragma unroll
  for (int q = 0; q < kB * kB / kThreads; ++q) {
    const int idx = tid + q * kThreads;
    const int r = idx >> 5, c = idx & 31;
    if (r < b && c < b) {
      const double2 p = cmul(X1[r][c], Y1[c][r]);
      const double2 m = cmul(X2[r][c], Y2[c][r]);
      sr += p.x - m.x;
      si += p.y - m.y;
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) {
    sr += __shfl_xor(sr, off);
    si += __shfl_xor(si, off);
  }
  if (lane == 0) {
    sh.red[0][wave] = sr;
    sh.red[1][wave] = si;
  }
  __syncthreads();
  double2 out = cmk(sh.red[0][0] + sh.red[0][1] + sh.red[0][2] + sh.red[0][3],
                    sh.red[1][0] + sh.red[1][1] + sh.red[1][2] + sh.red[1][3]);
  __syncthreads();
  return out;
}

// Fragments of an operand read from a global block (rows x cols, ld) as the
// right operand of a product: element (4 s + kq, 16 tc + l16), zero outside.
template <int KS>
__device__ inline void fetch_right(double2 (&b)[KS / 4][KS], const double2* F, int ld, int rows, int cols, int lane) {
  const int l16 = lane & 15, kq = lane >> 4;
#pragma unroll
  for (int tc = 0; tc < KS / 4; ++tc)
#pragma unroll
    for (int s = 0; s < KS; ++s) b[tc][s] = gld(F, ld, rows, cols, 4 * s + kq, 16 * tc + l16);
}

// All tiles of op(A) op(B) (m x n valid) by one wave, A (and B, unless its fragments
// are given) in LDS.  Unless kFull, dead tiles are left out (zero).
template <int KS, bool kFull, bool AH, bool BH>
__device__ inline void wave_product(double2 (&v)[KS / 4][KS / 4][4], const Slot& A, const Slot* B,
                                    const double2 (*given)[KS], int m, int n, int lane) {
  constexpr int NT = KS / 4, H = 4;  // inner steps whose fragments are held at a time
  const int l16 = lane & 15, kq = lane >> 4;
  if constexpr (!kFull && NT > 1) {
#pragma unroll
    for (int tr = 0; tr < NT; ++tr)
#pragma unroll
      for (int tc = 0; tc < NT; ++tc) {
        if (16 * tr < m && 16 * tc < n) {
          Acc c = acc_zero();
#pragma unroll
          for (int s = 0; s < KS; ++s) {
            const int kk = 4 * s + kq, x = 16 * tr + l16, y = 16 * tc + l16;
            mma_step<AH, BH, false>(c, AH ? A[kk][x] : A[x][kk], B ? (BH ? (*B)[y][kk] : (*B)[kk][y]) : given[tc][s]);
          }
          tile_vals(c, v[tr][tc]);
        } else {
#pragma unroll
          for (int r = 0; r < 4; ++r) v[tr][tc][r] = cmk(0.0, 0.0);
        }
      }
    return;
  }
  Acc acc[NT][NT];
#pragma unroll
  for (int tr = 0; tr < NT; ++tr)
#pragma unroll
    for (int tc = 0; tc < NT; ++tc) acc[tr][tc] = acc_zero();
#pragma unroll
  for (int s0 = 0; s0 < KS; s0 += H) {
    double2 a[NT][H], b[NT][H];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int u = 0; u < H; ++u) {
        const int kk = (s0 + u) * 4 + kq, x = 16 * t + l16;
        a[t][u] = AH ? A[kk][x] : A[x][kk];
        b[t][u] = B ? (BH ? (*B)[x][kk] : (*B)[kk][x]) : given[t][s0 + u];
      }
#pragma unroll
    for (int u = 0; u < H; ++u)
#pragma unroll
      for (int tr = 0; tr < NT; ++tr)
#pragma unroll
        for (int tc = 0; tc < NT; ++tc) mma_step<AH, BH, false>(acc[tr][tc], a[tr][u], b[tc][u]);
  }
#pragma unroll
  for (int tr = 0; tr < NT; ++tr)
#pragma unroll
    for (int tc = 0; tc < NT; ++tc) tile_vals(acc[tr][tc], v[tr][tc]);
}
template <int NT>
__device__ inline void wave_store(SmallShared& sh, int slot, const double2 (&v)[NT][NT][4], int lane) {
#pragma unroll
  for (int tr = 0; tr < NT; ++tr)
#pragma unroll
    for (int tc = 0; tc < NT; ++tc)
#pragma unroll
      for (int r = 0; r < 4; ++r) sh.s[slot][tile_row(tr, r, lane)][tile_col(tc, lane)] = v[tr][tc][r];
}

// The lesser (or greater) part of forward step j by one wave, in place in slot w
// (W_i on entry, W_j on exit): V = g_i W_i, g^<_i = V g_i^H (to global memory), Y = A_ji
// g^<_i, W_j = Y A_ji^H + Q^H - Q [= Sigma~, to `partial`] + Sigma_jj + B_j.  Waits for Q
// before its last product's epilogue.
template <int KS, bool kFull>
__device__ inline void lesser_chain(SmallShared& sh, int g, int w, int a, int q, int q_ready, double2* gi, int bi,
                                    const double2* sd, const double2* ob, int bj, double2* partial, int lane) {
  constexpr int NT = KS / 4;
  double2 v[NT][NT][4];
  wave_product<KS, kFull, false, false>(v, sh.s[g], &sh.s[w], nullptr, bi, bi, lane);
  wave_fence();
  wave_store<NT>(sh, w, v, lane);
  wave_fence();
  wave_product<KS, kFull, false, true>(v, sh.s[w], &sh.s[g], nullptr, bi, bi, lane);
  wave_fence();
  wave_store<NT>(sh, w, v, lane);
#pragma unroll
  for (int tr = 0; tr < NT; ++tr)
#pragma unroll
    for (int tc = 0; tc < NT; ++tc)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = tile_row(tr, r, lane), col = tile_col(tc, lane);
        buf_store(buf_of(gi), goff(bi, bi, bi, row, col), v[tr][tc][r]);
      }
  // (used by the last product's epilogue)
  double2 add[NT][NT][4];
#pragma unroll
  for (int tr = 0; tr < NT; ++tr)
#pragma unroll
    for (int tc = 0; tc < NT; ++tc)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        add[tr][tc][r] = gld(sd, bj, bj, bj, tile_row(tr, r, lane), tile_col(tc, lane));
  wave_fence();
  wave_product<KS, kFull, false, false>(v, sh.s[a], &sh.s[w], nullptr, bj, bi, lane);
  wave_fence();
  wave_store<NT>(sh, w, v, lane);
  if (ob) {
#pragma unroll
    for (int tr = 0; tr < NT; ++tr)
#pragma unroll
      for (int tc = 0; tc < NT; ++tc)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          add[tr][tc][r] = cadd(add[tr][tc][r], gld(ob, bj, bj, bj, tile_row(tr, r, lane), tile_col(tc, lane)));
  }
  wave_fence();
  wave_product<KS, kFull, false, true>(v, sh.s[w], &sh.s[a], nullptr, bj, bj, lane);
  while (__hip_atomic_load(&sh.q_done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < q_ready)
    __builtin_amdgcn_s_sleep(1);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  const Add qa = add_slot(sh.s[q], -1.0, 1.0);
#pragma unroll
  for (int tr = 0; tr < NT; ++tr)
#pragma unroll
    for (int tc = 0; tc < NT; ++tc)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int row = tile_row(tr, r, lane), col = tile_col(tc, lane);
        const double2 x = cadd(v[tr][tc][r], add_val(qa, r, row, col));
        if (partial) gput(partial, row * kB + col, x);
        v[tr][tc][r] = cadd(x, add[tr][tc][r]);
      }
  wave_store<NT>(sh, w, v, lane);
}

// Q = P Sigma_ij (from global memory) into slot q by one wave; then announces it.
template <int KS, bool kFull>
__device__ inline void q_product(SmallShared& sh, int p, const double2 (&b)[KS / 4][KS], int q, int done, int n,
                                 int lane) {
  double2 v[KS / 4][KS / 4][4];
  wave_product<KS, kFull, false, false>(v, sh.s[p], nullptr, b, n, n, lane);
  wave_store<KS / 4>(sh, q, v, lane);
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  if (lane == 0) __hip_atomic_store(&sh.q_done, done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Uniform slot allocator (every thread holds the same mask).
struct Slots {
  unsigned used = 0;
  __device__ int take() {
    const int s = __builtin_ctz(~used);
    used |= 1u << s;
    return s;
  }
  __device__ void give(int s) { used &= ~(1u << s); }
};

// Product terms: T<AH, BH, NEG>(A, B) is acc += (-1)^NEG op(A) op(B).
#define QX_T(AH, BH, NEG, A_, B_)                                                   \
  [&](Acc& ac, int tr, int tc, int lane) {                                          \
    mma<KS, AH, BH, NEG>(ac, sh.s[A_], sh.s[B_], tr, tc, lane);                     \
  }
#define QX_T2(AH1, BH1, NEG1, A1, B1, AH2, BH2, NEG2, A2, B2)                       \
  [&](Acc& ac, int tr, int tc, int lane) {                                          \
    mma<KS, AH1, BH1, NEG1>(ac, sh.s[A1], sh.s[B1], tr, tc, lane);                  \
    mma<KS, AH2, BH2, NEG2>(ac, sh.s[A2], sh.s[B2], tr, tc, lane);                  \
  }

// the problem table and its index tables are read through the scalar
// (constant) path
typedef __attribute__((address_space(4))) const SmallProblem cprob;

// One energy point.
template <int KS, bool kFull>
__device__ __forceinline__ void sweep_one(SmallShared& sh, const SmallLaunch& L, const cprob& P, int e,
                                          double2* wg_scratch) {
  constexpr int NT = KS / 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t eg = P.e_base + e;
  const int N = P.N;
  const __attribute__((address_space(4))) int* bs = (const __attribute__((address_space(4))) int*)P.bs;
  const __attribute__((address_space(4))) int64_t* od = (const __attribute__((address_space(4))) int64_t*)P.od;
  const __attribute__((address_space(4))) int64_t* ou = (const __attribute__((address_space(4))) int64_t*)P.ou;
  auto D_ = [&](const double2* base, int i) { return base ? base + (int64_t)e * P.Dsz + od[i] : nullptr; };
  auto U_ = [&](const double2* base, int i) { return base ? base + (int64_t)e * P.Usz + ou[i] : nullptr; };
  auto Dw = [&](double2* base, int i) { return base ? base + (int64_t)e * P.Dsz + od[i] : nullptr; };
  auto Uw = [&](double2* base, int i) { return base ? base + (int64_t)e * P.Usz + ou[i] : nullptr; };
  auto OB = [&](const double2* const* arr, int i) -> const double2* {
    if (!arr) return nullptr;
    typedef const double2* cptr;
    typedef __attribute__((address_space(4))) const cptr ccptr;
    const double2* b = ((const ccptr*)arr)[i];
    return b ? b + (int64_t)e * bs[i] * bs[i] : nullptr;
  };
  // left-connected g_i: the G^R diagonal output, or this workgroup's scratch
  double2* gstore = P.GRd ? nullptr : wg_scratch;
  double2* sigt = wg_scratch ? wg_scratch + (int64_t)(P.GRd ? 0 : N) * kB * kB : nullptr;
  auto Gd = [&](int i) -> double2* { return P.GRd ? Dw(P.GRd, i) : gstore + (int64_t)i * kB * kB; };
  auto Gld = [&](int i) { return P.GRd ? bs[i] : kB; };
  auto SigT = [&](int k, int i) { return sigt + ((int64_t)k * N + i) * kB * kB; };
  const bool cur = P.cur != nullptr;
  double2* current = cur ? P.cur + (int64_t)e * (N + 1) : nullptr;
  Slots S;

  // ---- block 0 (rgf.py:216-239): W_0 = Sigma_00 + B_0 ----
  int cg = S.take(), wl = S.take(), wg = S.take();
  {
    const int b = bs[0];
    const Blk blks[3] = {blk(cg, D_(P.Ad, 0), b, b, b, OB(P.obr, 0), -1.0, 1.0),
                         blk(wl, D_(P.SLd, 0), b, b, b, OB(P.obl, 0), 1.0),
                         blk(wg, D_(P.SGd, 0), b, b, b, OB(P.obg, 0), 1.0)};
    load_blks<3>(sh, blks);
  }
  // A_ji, A_ij and A_jj - B^R_j of step j come by wave 2 while block j - 1 is
  // inverted: the last two into their slots, A_ji into registers
  int s = S.take(), pp = S.take();
  const int a = S.take(), t = S.take(), ql = S.take(), qg = S.take();
  double2 fa[16];
  auto fetch_step = [&](int j, int slot_s) {
    const int bi = bs[j - 1], bj = bs[j];
    double2 fs[16], ft[16];
    wave_fetch(fs, D_(P.Ad, j), bj, bj, bj, lane);
    wave_fetch(ft, U_(P.Au, j - 1), bj, bi, bj, lane);  // (bi x bj)
    wave_fetch(fa, U_(P.Al, j - 1), bi, bj, bi, lane);  // (bj x bi)
    if (const double2* ob = OB(P.obr, j)) {
      double2 fo[16];
      wave_fetch(fo, ob, bj, bj, bj, lane);
#pragma unroll
      for (int q = 0; q < 16; ++q) fs[q] = csub(fs[q], fo[q]);
    }
    wave_commit(sh, slot_s, fs, lane, bj, 1.0);
    wave_commit(sh, t, ft, lane);
  };
  __syncthreads();
  if (wave == 3) invert_wave<NT>(sh, cg, bs[0], L.info, 1, eg);
  if (wave == 2 && N > 1) fetch_step(1, s);
  __syncthreads();

  // ---- forward sweep (rgf.py:241-302) ----
  // Only P = A_ji g_i and S = A_jj - B^R_j - P A_ij stand between two inversions:
  // wave 3 inverts S, and meanwhile waves 0 and 1 take g^<_i and g^>_i from W_i and go on
  // to W_j (in place), with Q = P Sigma_ij from wave 2, which then stores g_i and brings
  // the next step's blocks.
  for (int j = 1; j < N; ++j) {
    const int i = j - 1;
    const int bi = bs[i], bj = bs[j];
    if (wave == 2) wave_commit(sh, a, fa, lane);
    __syncthreads();
    run_round<kFull>(sh, false, prod(bj, bi, QX_T(false, false, false, a, cg), to_slot(pp)));
    run_round<kFull>(sh, false,
                     prod(bj, bj, QX_T(false, false, true, pp, t), to_slot(s), add_slot(sh.s[s], 1.0)));
    if (wave == 3) {
      invert_wave<NT>(sh, s, bj, L.info, j + 1, eg);
    } else if (wave == 2) {
      double2 bl[NT][KS], bg[NT][KS];
      fetch_right<KS>(bl, U_(P.SLu, i), bj, bi, bj, lane);  // Sigma^<_ij
      fetch_right<KS>(bg, U_(P.SGu, i), bj, bi, bj, lane);  // Sigma^>_ij
      q_product<KS, kFull>(sh, pp, bl, ql, 2 * j, bj, lane);
      q_product<KS, kFull>(sh, pp, bg, qg, 2 * j + 1, bj, lane);
      wave_store_blk(Gd(i), Gld(i), bi, sh.s[cg], lane);
      if (j + 1 < N) fetch_step(j + 1, pp);
    } else {
      const bool gr = wave == 1;
      lesser_chain<KS, kFull>(sh, cg, gr ? wg : wl, a, gr ? qg : ql, 2 * j + (gr ? 1 : 0),
                              Dw(gr ? P.GGd : P.GLd, i), bi, D_(gr ? P.SGd : P.SLd, j),
                              OB(gr ? P.obg : P.obl, j), bj, cur ? SigT(gr ? 1 : 0, j) : nullptr, lane);
    }
    __syncthreads();
    const int g = cg;
    cg = s;
    s = pp;
    pp = g;
  }
  store_blk(Gd(N - 1), Gld(N - 1), bs[N - 1], bs[N - 1], sh.s[cg], 0);
  for (const int x : {a, t, s, pp, ql, qg}) S.give(x);
  // the backward sweep's input blocks of step i, fetched one step ahead: g_i,
  // Sigma^<_ij, Sigma^>_ij, A_ij, A_ji
  double2 pre[5][4];
  auto fetch_back = [&](int i, int k) {
    const int bi = bs[i], bj = bs[i + 1];
    if (k == 0) fetch_blk(blk(0, Gd(i), Gld(i), bi, bi), pre[0]);
    if (k == 1) fetch_blk(blk(0, U_(P.SLu, i), bj, bi, bj), pre[1]);
    if (k == 2) fetch_blk(blk(0, U_(P.SGu, i), bj, bi, bj), pre[2]);
    if (k == 3) fetch_blk(blk(0, U_(P.Au, i), bj, bi, bj), pre[3]);
    if (k == 4) fetch_blk(blk(0, U_(P.Al, i), bi, bj, bi), pre[4]);
  };
  if (N > 1)
#pragma unroll
    for (int k = 0; k < 5; ++k) fetch_back(N - 2, k);
  // V = g W, g^<> = V g^H of the last block
  {
    const int b = bs[N - 1], vl = S.take(), vg = S.take();
    run_round<kFull>(sh, false, prod(b, b, QX_T(false, false, false, cg, wl), to_slot(vl)),
                     prod(b, b, QX_T(false, false, false, cg, wg), to_slot(vg)));
    run_round<kFull>(sh, false, prod(b, b, QX_T(false, true, false, vl, cg), to_slot(wl)),
                     prod(b, b, QX_T(false, true, false, vg, cg), to_slot(wg)));
    S.give(vl);
    S.give(vg);
  }
  const int cl = wl, cgg = wg;

  // ---- last block: G_{N-1} = g_{N-1}; stored diagonal G^<> projected ----
  {
    const int n1 = N - 1, b = bs[n1];
    store_blk(Dw(P.GLd, n1), b, b, b, sh.s[cl], 2);
    store_blk(Dw(P.GGd, n1), b, b, b, sh.s[cgg], 2);
    if (cur) {
      const int x = S.take(), y = S.take();
      if (N > 1) {
        const Blk xy[2] = {blk(x, SigT(1, n1), kB, b, b), blk(y, SigT(0, n1), kB, b, b)};
        load_blks<2>(sh, xy);
        __syncthreads();
        const double2 jv = trace2(sh, sh.s[x], sh.s[cl], sh.s[cgg], sh.s[y], b);
        if (tid == 0) gput(current, n1, jv);
      }
      const Blk xy[2] = {blk(x, OB(P.obg, n1), b, b, b), blk(y, OB(P.obl, n1), b, b, b)};
      load_blks<2>(sh, xy);
      __syncthreads();
      const double2 jn = trace2(sh, sh.s[x], sh.s[cl], sh.s[cgg], sh.s[y], b);
      if (tid == 0) gput(current, N, cmk(-jn.x, -jn.y));
      if (N == 1) {
        // J_0 with the same (first = last) block
        if (tid == 0) gput(current, 0, jn);
      }
      S.give(x);
      S.give(y);
    }
  }

  // ---- backward sweep (rgf.py:315-412) ----
  int X = cg, Xl = cl, Xg = cgg;  // G_jj, G^<>_jj (unprojected)
  for (int i = N - 2; i >= 0; --i) {
    const int j = i + 1;
    const int bi = bs[i], bj = bs[j];
    // the left-connected g^<>_i (unprojected) are fetched into registers one round
    // before slots free up for them
    const int g = S.take(), sgl = S.take(), sgg = S.take(), aij = S.take(), aji = S.take();
    const Blk gb[2] = {blk(0, Dw(P.GLd, i), bi, bi, bi), blk(0, Dw(P.GGd, i), bi, bi, bi)};
    double2 gpre[4], gnew[4];
    commit_blk(sh, g, pre[0]);
    commit_blk(sh, sgl, pre[1]);
    commit_blk(sh, sgg, pre[2]);
    commit_blk(sh, aij, pre[3]);
    commit_blk(sh, aji, pre[4]);
    __syncthreads();
    // Z^<> = g_i Sigma^<>_ij ; U = g_i A_ij ; R = G_jj A_ji (over their B operands)
    run_round<kFull>(sh, true, prod(bi, bj, QX_T(false, false, false, g, sgl), to_slot(sgl)),
              prod(bi, bj, QX_T(false, false, false, g, sgg), to_slot(sgg)),
              prod(bi, bj, QX_T(false, false, false, g, aij), to_slot(aij)),
              prod(bj, bi, QX_T(false, false, false, X, aji), to_slot(aji)));
    const int zl = sgl, zg = sgg, u = aij, rr = aji;
    fetch_blk(gb[0], gpre);
    // B^<> = Z^<> G_jj^H ; G^R_ij = -U G_jj ; G^R_ji = -R g_i ; K = U R ;
    // T2^<> = U G^<>_jj (over Z, G_jj and the carried G^<>_jj)
    run_round<kFull>(sh, true, prod(bi, bj, QX_T(false, true, false, zl, X), to_slot(zl)),
              prod(bi, bj, QX_T(false, true, false, zg, X), to_slot(zg)),
              prod(bi, bi, QX_T(false, false, false, u, rr), to_slot(X)),
              prod(bi, bj, QX_T(false, false, false, u, Xl), to_slot(Xl)),
              prod(bi, bj, QX_T(false, false, false, u, Xg), to_slot(Xg)),
              prod(bi, bj, QX_T(false, false, true, u, X), to_glob(Uw(P.GRu, i), bj, bi, bj), add_none(),
                   add_none(), add_none(), P.GRu != nullptr),
              prod(bj, bi, QX_T(false, false, true, rr, g), to_glob(Uw(P.GRl, i), bi, bj, bi), add_none(),
                   add_none(), add_none(), P.GRl != nullptr));
    const int bl = zl, bg = zg, kk = X, t2l = Xl, t2g = Xg;
    // g^<_i into the free slot
    const int gl = S.take();
    commit_blk(sh, gl, gpre);
    fetch_blk(gb[1], gpre);
    __syncthreads();
    if (i > 0) {
      fetch_back(i - 1, 0);
      fetch_back(i - 1, 1);
    }
    // G_ii = g_i + K g_i ; G^<_ij = -g^<_i R^H + B^< - T2^< (and G^<_ji =
    // -(G^<_ij)^H) ; T1^< = K g^<_i - B^< U^H over g_i
    run_round<kFull>(sh, true,
              prod(bi, bi, QX_T(false, false, false, kk, g), kept(to_glob(Gd(i), Gld(i), bi, bi), gnew),
                   add_slot(sh.s[g], 1.0)),
              prod(bi, bj, QX_T(false, true, true, gl, rr),
                   to_glob(Uw(P.GLu, i), bj, bi, bj).globT(Uw(P.GLl, i), bi, -1.0), add_slot(sh.s[bl], 1.0),
                   add_slot(sh.s[t2l], -1.0)),
              prod(bi, bi, QX_T2(false, false, false, kk, gl, false, true, true, bl, u), to_slot(g)));
    const int t1l = g;
    S.give(bl);
    // g^>_i into the slot of B^<
    const int gg = S.take();
    commit_blk(sh, gg, gpre);
    __syncthreads();
    if (i > 0) {
      fetch_back(i - 1, 2);
      fetch_back(i - 1, 3);
    }
    // G^>_ij, G^>_ji ; T1^> = K g^>_i - B^> U^H over K ;
    // G^<_ii = g^<_i + T2^< U^H + T1^< - T1^<^H (in place)
    run_round<kFull>(sh, true,
              prod(bi, bj, QX_T(false, true, true, gg, rr),
                   to_glob(Uw(P.GGu, i), bj, bi, bj).globT(Uw(P.GGl, i), bi, -1.0), add_slot(sh.s[bg], 1.0),
                   add_slot(sh.s[t2g], -1.0)),
              prod(bi, bi, QX_T2(false, false, false, kk, gg, false, true, true, bg, u), to_slot(kk)),
              prod(bi, bi, QX_T(false, true, false, t2l, u), to_slot(gl), add_slot(sh.s[gl], 1.0),
                   add_slot(sh.s[t1l], 1.0, -1.0)));
    const int t1g = kk;
    if (i > 0) fetch_back(i - 1, 4);
    // G^>_ii = g^>_i + T2^> U^H + T1^> - T1^>^H (in place)
    run_round<kFull>(sh, false,
              prod(bi, bi, QX_T(false, true, false, t2g, u), to_slot(gg), add_slot(sh.s[gg], 1.0),
                   add_slot(sh.s[t1g], 1.0, -1.0)));
    store_blk(Dw(P.GLd, i), bi, bi, bi, sh.s[gl], 2);
    store_blk(Dw(P.GGd, i), bi, bi, bi, sh.s[gg], 2);
    S.give(t1g);
    S.give(t1l);
    S.give(bg);
    S.give(u);
    S.give(rr);
    S.give(t2l);
    S.give(t2g);
    Xl = gl;
    Xg = gg;
    X = S.take();
    {
      int tr, tc;
      tile_of<kFull>(0, wave, tr, tc);
#pragma unroll
      for (int r = 0; r < 4; ++r) sh.s[X][tile_row(tr, r, lane)][tile_col(tc, lane)] = gnew[r];
    }
    if (cur) {
      const int x = S.take(), y = S.take();
      if (i >= 1) {
        const Blk xy[2] = {blk(x, SigT(1, i), kB, bi, bi), blk(y, SigT(0, i), kB, bi, bi)};
        load_blks<2>(sh, xy);
      } else {
        const Blk xy[2] = {blk(x, OB(P.obg, 0), bi, bi, bi), blk(y, OB(P.obl, 0), bi, bi, bi)};
        load_blks<2>(sh, xy);
      }
      __syncthreads();
      const double2 jv = trace2(sh, sh.s[x], sh.s[Xl], sh.s[Xg], sh.s[y], bi);
      if (tid == 0) gput(current, i, jv);
      S.give(x);
      S.give(y);
    }
  }
}

template <int KS>
__global__ void __launch_bounds__(kThreads, 1) sweep_small_kernel(SmallLaunch L) {
  __shared__ SmallShared sh;
  double2* wg_scratch = L.scratch ? (double2*)(L.scratch + (int64_t)blockIdx.x * L.scratch_per_wg) : nullptr;
  for (;;) {
    if (threadIdx.x == 0) {
      sh.job = atomicAdd(L.counter, 1);
      sh.q_done = 0;
    }
    __syncthreads();
    const int job = __builtin_amdgcn_readfirstlane(sh.job);
    __syncthreads();
    if (job >= L.total_jobs) break;
    int p = 0;
    const cprob* probs = (const cprob*)L.probs;
    while (p + 1 < L.nprob && job >= probs[p + 1].job0) ++p;
    const cprob& P = probs[p];
    const int e = job - P.job0;
    if (KS == 8 && P.full)
      sweep_one<KS, KS == 8>(sh, L, P, e, wg_scratch);
    else
      sweep_one<KS, false>(sh, L, P, e, wg_scratch);
    __syncthreads();
  }
}


#undef QX_T
#undef QX_T2

}  // namespace

size_t sweep_small_scratch_per_wg(int n_blocks, bool need_g, bool current) {
  const size_t blk = (size_t)kB * kB * sizeof(double2);
  return blk * ((need_g ? n_blocks : 0) + (current ? 2 * n_blocks : 0));
}

hipError_t launch_sweep_small(const SmallLaunch& L, int grid, hipStream_t stream) {
  if (L.total_jobs == 0) return hipSuccess;
  if (L.bmax <= 16)
    hipLaunchKernelGGL(sweep_small_kernel<4>, dim3(grid), dim3(kThreads), 0, stream, L);
  else
    hipLaunchKernelGGL(sweep_small_kernel<8>, dim3(grid), dim3(kThreads), 0, stream, L);
  return hipGetLastError();
}

}  // namespace qx
