// hn_inv.hip -- batched complex block inverse with partial pivoting.
//
// Replaces zinv (ZGETRF + ZGETRS against I, inversions.F90:807-839) and
// cu_Zinverse (gpuroutines.cu:449-523) for whole batches of blocks.
//
// Blocks up to 96 (FP32: 128): one workgroup per block, LU with partial pivoting
// and the substitutions in registers, on the matrix cores (k_lu_inv_mx; FP64 up
// to 16 on a thread grid, k_lu_inv_2d).  FP32 blocks of 129 to 140, the largest
// that fit: Gauss-Jordan with partial pivoting in LDS, followed by the column
// interchanges that undo the row pivoting (k_inv_lds).
//
// Large blocks (up to n = 1024): in-place Gauss-Jordan with lazy pivoting on
// the row-major view M = A^T, so that rows of M are contiguous columns of A
// (inverting M and reading the result back column-major gives A^-1; the row
// pivoting of M is column pivoting of A).  Rows are never moved; the pivot
// row of each logical column is recorded.  Per super-panel S of up to 64
// columns, one launch (one workgroup of 512 threads per item, the n x |S|
// panel in registers) runs the |S| elimination steps on S and writes the
// accumulated transform; the other columns of M then take ONE deferred
// rank-|S| update on the matrix cores.  After the last super-panel,
// M^-1(i, c) = B(pi(i), pi^-1(c)) with pi(c) the pivot row of column c.
#include <cfloat>
#include <utility>

#include "hn_gemm.h"
#include "hn_inv.h"
#include "hn_prof.h"

namespace hn {

namespace {

constexpr int NT = 256;
constexpr int kLdsBudget = 160 * 1024 - 2048;

template <typename R> struct CT_;
template <> struct CT_<double> { typedef double2 t; };
template <> struct CT_<float> { typedef float2 t; };

template <typename C> __device__ inline C cmul(C a, C b) {
  return C{a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x};
}
template <typename C> __device__ inline C csub(C a, C b) { return C{a.x - b.x, a.y - b.y}; }
template <typename C> __device__ inline C cneg(C a) { return C{-a.x, -a.y}; }
template <typename C> __device__ inline C crecip(C b) {
  // 1/b, Smith's algorithm; 0 for b == 0 (singular: flagged by the caller)
  typedef decltype(b.x) R;
  if (b.x == R(0) && b.y == R(0)) return C{0, 0};
  if (fabs(b.x) >= fabs(b.y)) {
    R r = b.y / b.x, d = b.x + r * b.y;
    return C{R(1) / d, -r / d};
  } else {
    R r = b.x / b.y, d = b.y + r * b.x;
    return C{r / d, R(-1) / d};
  }
}
template <typename C> __device__ inline auto cabs1(C a) -> decltype(a.x) {
  return fabs(a.x) + fabs(a.y);
}

// wave-level argmax of (v, i): larger v wins, ties -> smaller index
template <typename R> __device__ inline void wave_argmax(R &v, int &i) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    R ov = __shfl_xor(v, off);
    int oi = __shfl_xor(i, off);
    if (ov > v || (ov == v && oi >= 0 && (i < 0 || oi < i))) {
      v = ov;
      i = oi;
    }
  }
}

// ---------------------------------------------------------------------------
// single-workgroup LDS Gauss-Jordan (FP32 blocks of order 129 to 140)
// ---------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(NT) void k_inv_lds(int n, typename CT_<R>::t *A, long long sA,
                                                typename CT_<R>::t *Ainv, long long sAinv,
                                                const int *active, int *status) {
  typedef typename CT_<R>::t C;
  extern __shared__ __align__(16) unsigned char smem[];
  const int b = blockIdx.x;
  if (active && active[b] == 0) return;
  C *M = (C *)smem;
  C *rowbuf = M + (size_t)n * n;
  C *colbuf = rowbuf + n;
  int *perm = (int *)(colbuf + n);
  __shared__ int s_p, s_sing;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const C *Ab = A + (long long)b * sA;
  for (int e = tid; e < n * n; e += NT) M[e] = Ab[e];
  if (tid == 0) s_sing = 0;
  // 2-D thread mapping for the rank-1 update: thread -> (row i, column phase)
  const int cpar = NT / n;  // n <= NT here
  const int ui = tid % n, uj0 = tid / n;
  const bool upd = uj0 < cpar;
  __syncthreads();
  for (int k = 0; k < n; ++k) {
    if (wave == 0) {
      R best = R(-1);
      int bi = -1;
      for (int i = k + lane; i < n; i += 64) {
        R v = cabs1(M[i + (size_t)k * n]);
        if (v > best) { best = v; bi = i; }
      }
      wave_argmax(best, bi);
      if (lane == 0) {
        s_p = bi < 0 ? k : bi;
        if (!(best > R(0))) s_sing = 1;
      }
    }
    __syncthreads();
    const int p = s_p;
    if (p != k)
      for (int j = tid; j < n; j += NT) {
        C t = M[k + (size_t)j * n];
        M[k + (size_t)j * n] = M[p + (size_t)j * n];
        M[p + (size_t)j * n] = t;
      }
    if (tid == 0) perm[k] = p;
    __syncthreads();
    const C pinv = crecip(M[k + (size_t)k * n]);
    for (int j = tid; j < n; j += NT) rowbuf[j] = (j == k) ? pinv : cmul(M[k + (size_t)j * n], pinv);
    for (int i = tid; i < n; i += NT) colbuf[i] = (i == k) ? C{0, 0} : M[i + (size_t)k * n];
    __syncthreads();
    if (upd) {
      const C ci = colbuf[ui];
      for (int j = uj0; j < n; j += cpar) {
        size_t e = ui + (size_t)j * n;
        if (ui == k) M[e] = rowbuf[j];
        else if (j == k) M[e] = cneg(cmul(ci, pinv));
        else M[e] = csub(M[e], cmul(ci, rowbuf[j]));
      }
    }
    __syncthreads();
  }
  for (int k = n - 1; k >= 0; --k) {
    const int p = perm[k];
    if (p != k)
      for (int i = tid; i < n; i += NT) {
        C t = M[i + (size_t)k * n];
        M[i + (size_t)k * n] = M[i + (size_t)p * n];
        M[i + (size_t)p * n] = t;
      }
    __syncthreads();
  }
  C *Ob = Ainv + (long long)b * sAinv;
  for (int e = tid; e < n * n; e += NT) Ob[e] = M[e];
  if (tid == 0 && s_sing && status) atomicOr(&status[b], (int)ST_SINGULAR);
}

// ---------------------------------------------------------------------------
// blocked path
// ---------------------------------------------------------------------------
constexpr int NTG = 512;  // threads of the Gauss-Jordan kernel: two halves of 256 rows

// Encoding of a chosen pivot row r (r < 1024) with its FP64 |.|_1 (the row
// itself comes from the exact 64-bit search): the high word of the magnitude
// (exponent and 9 mantissa bits), a flag bit and 1023 - r; the row is read
// back from the low bits and a magnitude below 2^-1011 (the high word below
// 0x800) flags a zero pivot.
__device__ inline unsigned pivot_key(double v, int r) {
  const unsigned hi = min((unsigned)((unsigned long long)__double_as_longlong(v) >> 32), 0x7FF00000u);
  return (hi & ~0x7FFu) | 0x400u | (unsigned)(1023 - r);
}
__device__ inline unsigned pivot_key(float v, int r) {
  return pivot_key((double)v, r);
}
// 1/b for a pivot: b scaled by a power of two (exact) so that |b'|^2 lies in
// [1/4, 2), the hardware reciprocal of |b'|^2 refined by two Newton-Raphson
// steps (r <- r + r (1 - d r)), and conj(b') r scaled back; 0 for b == 0.
__device__ inline double2 crecip_fast(double2 b) {
  const double mx = fmax(fabs(b.x), fabs(b.y));
  if (mx == 0.0) return double2{0, 0};
  const int e = __builtin_amdgcn_frexp_exp(mx);
  const double x = __builtin_amdgcn_ldexp(b.x, -e), y = __builtin_amdgcn_ldexp(b.y, -e);
  const double d = fma(x, x, y * y);
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  r = fma(r, fma(-d, r, 1.0), r);
  return double2{__builtin_amdgcn_ldexp(x * r, -e), __builtin_amdgcn_ldexp(-y * r, -e)};
}
__device__ inline float2 crecip_fast(float2 b) { return crecip(b); }

// value held by lane `lane` (uniform) of the wave
__device__ inline double lane_read(double v, int lane) {
  const int lo = __builtin_amdgcn_readlane(__double2loint(v), lane);
  const int hi = __builtin_amdgcn_readlane(__double2hiint(v), lane);
  return __hiloint2double(hi, lo);
}
__device__ inline float lane_read(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// 64-bit key helpers for the exact pivot search: DPP butterflies inside each
// row of 16 lanes on both halves, then the four row results read as scalars.
template <int CTRL> __device__ inline unsigned long long dpp64(unsigned long long k) {
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(k >> 32), CTRL, 0xF, 0xF, false);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)k, CTRL, 0xF, 0xF, false);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ inline unsigned long long rl64(unsigned long long k, int lane) {
  const unsigned hi = __builtin_amdgcn_readlane((int)(k >> 32), lane);
  const unsigned lo = __builtin_amdgcn_readlane((int)(unsigned)k, lane);
  return ((unsigned long long)hi << 32) | lo;
}
__device__ inline unsigned long long wave_max64(unsigned long long k) {
  k = max(k, dpp64<0xB1>(k));   // quad_perm [1,0,3,2]
  k = max(k, dpp64<0x4E>(k));   // quad_perm [2,3,0,1]
  k = max(k, dpp64<0x124>(k));  // row_ror:4
  k = max(k, dpp64<0x128>(k));  // row_ror:8
  return max(max(rl64(k, 0), rl64(k, 16)), max(rl64(k, 32), rl64(k, 48)));
}
template <int CTRL> __device__ inline unsigned dpp_min(unsigned k) {
  return min(k, (unsigned)__builtin_amdgcn_update_dpp(-1, (int)k, CTRL, 0xF, 0xF, false));
}
__device__ inline unsigned wave_min32(unsigned k) {
  k = dpp_min<0xB1>(k);
  k = dpp_min<0x4E>(k);
  k = dpp_min<0x124>(k);
  k = dpp_min<0x128>(k);
  const unsigned a = __builtin_amdgcn_readlane((int)k, 0), b = __builtin_amdgcn_readlane((int)k, 16);
  const unsigned c = __builtin_amdgcn_readlane((int)k, 32), d = __builtin_amdgcn_readlane((int)k, 48);
  return min(min(a, b), min(c, d));
}

// ---------------------------------------------------------------------------
// LU inverse of blocks up to 16 (complex double), one workgroup per block
// ---------------------------------------------------------------------------
// The reference's algorithm: ZGETRF (partial pivoting; the pivot is the first
// largest |Re| + |Im| of the column in the current row order, as IZAMAX
// picks it) followed by ZGETRS against the identity (inversions.F90:807-839).
//
// G x G threads, thread (cb, rb) = threadIdx cb*G + rb holding the TB x TB
// sub-block rows rb*TB.., columns cb*TB.. in registers.  The G threads of one
// thread column are G consecutive lanes of one wave.  Rows are never moved:
// pos is a row's current position in LAPACK's row order, and a pivot step
// exchanges two positions.  One register block holds both factors in place:
// columns right of the current step hold A, columns at or left of it hold
// Y = L^-1 P (the forward substitution of ZGETRS against P I; column j of Y
// belongs to the row pivoted at step j, so the pivoted rows' entries of Y
// right of their own step are zero).
//
// Step k: the pivot p (row, position, reciprocal) and column k after step
// k-1 are in LDS.  The thread column owning column k turns that register
// column into Y's column k (1 on row p, 0 elsewhere).  Every thread takes row
// p for its columns from the lane of its own thread column that holds it
// (ds_bpermute inside the wave) and applies X(r, c) -= m_r X(p, c),
// m_r = A(r, k)/A(p, k), to its unpivoted rows -- ZGETRF's elimination on
// A's columns and ZGETRS's forward substitution on Y's, in one pass with no
// branches.  Then the thread column owning column k+1 publishes it: the
// entries of pivoted rows (U above the diagonal) into a triangular LDS array
// by position, the others for the next multipliers, and the pivot -- the
// largest |Re| + |Im| over the unpivoted rows as an exact 64-bit key, ties to
// the smallest position, reduced by DPP inside the G lanes.  One barrier per
// step.
//
// Every register index is a compile-time constant (static_for, the k loop
// unrolled by TB, and run-time rows read through select chains), so the
// block stays in registers.
//
// Back substitution U X = Y, positions i = n-1 .. 0, without barriers: row i
// of X (the row pivoted at step i, divided by U(i, i)) from the lanes of the
// same thread column, U's column i from the triangular array; the division
// of a row's own registers is applied at the end (a row is not updated after
// its own position).  Row pos(r) of X ends in the threads of row r; column j of X is
// column perm(j) of the inverse (the row pivoted at step j).

template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
// f(std::integral_constant<int, i>) for i = 0 .. N-1, unrolled at compile time
template <int N, typename F> __device__ __forceinline__ void static_for(F &&f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

// (key, pos) pair reduction over 8 consecutive lanes: the larger key wins, equal
// keys go to the smaller pos
template <int CTRL> __device__ inline void best_dpp(unsigned long long &k, int &p) {
  const unsigned hi = __builtin_amdgcn_update_dpp(0, (int)(k >> 32), CTRL, 0xF, 0xF, false);
  const unsigned lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)k, CTRL, 0xF, 0xF, false);
  const int op = __builtin_amdgcn_update_dpp(0, p, CTRL, 0xF, 0xF, false);
  const unsigned long long ok = ((unsigned long long)hi << 32) | lo;
  if (ok > k || (ok == k && op < p)) {
    k = ok;
    p = op;
  }
}
__device__ inline void group_best8(unsigned long long &k, int &p) {
  best_dpp<0xB1>(k, p);   // quad_perm [1,0,3,2]
  best_dpp<0x4E>(k, p);   // quad_perm [2,3,0,1]
  best_dpp<0x141>(k, p);  // row_half_mirror
}
// x - m y with the FMA order of the elimination updates
__device__ inline double2 fms_c(double2 x, double2 m, double2 y) {
  x.x = fma(-m.x, y.x, x.x);
  x.x = fma(m.y, y.y, x.x);
  x.y = fma(-m.x, y.y, x.y);
  x.y = fma(-m.y, y.x, x.y);
  return x;
}

// value `v` of the lane at byte index `src` (4 x lane) within the wave, for every lane
__device__ inline double bperm(double v, int src) {
  const int lo = __builtin_amdgcn_ds_bpermute(src, __double2loint(v));
  const int hi = __builtin_amdgcn_ds_bpermute(src, __double2hiint(v));
  return __hiloint2double(hi, lo);
}
__device__ inline double2 bperm(double2 v, int src) {
  return double2{bperm(v.x, src), bperm(v.y, src)};
}
// offset of U(i, c), i < c, in the triangular LDS array (by position)
__device__ inline int utri(int i, int c) { return (c * (c - 1)) / 2 + i; }

template <int TB> struct LuBlk {
  double2 v[TB][TB];
  int pos[TB];
  bool done[TB];
};

// element (r, J) of the register block for the uniform run-time row r < TB,
// as a select chain that starts from zero (so it is not folded into a
// register-indexed load, which would move the block out of registers)
template <int TB, int J>
__device__ __forceinline__ double2 pick0(const double2 (&v)[TB][TB], int r) {
  double xr = 0.0, xi = 0.0;
  static_for<TB>([&](auto I) {
    const bool hit = r == (int)I;
    xr = hit ? v[I][J].x : xr;
    xi = hit ? v[I][J].y : xi;
  });
  return double2{xr, xi};
}

// The thread column owning column col (register column JJ) publishes it:
// pivoted rows' entries into the triangular U array, unpivoted rows' into
// colbuf (the next multipliers), and the pivot's row, position and
// reciprocal.
template <int G, int TB, int JJ>
__device__ __forceinline__ void lu_publish(int col, int tid, const LuBlk<TB> &B, double2 *Ut,
                                           double2 *colbuf, int *s_perm, int *s_pospiv,
                                           double2 *s_uinv, int *s_sing) {
  const int cb = tid / G, rb = tid % G;
  const int oc = col / TB;
  unsigned long long key = 0, kk[TB];
  int bp = 0x7fffffff;
  static_for<TB>([&](auto I) {
    constexpr int i = I;
    const double2 v = B.v[i][JJ];
    kk[i] = B.done[i] ? 0ull
                      : (unsigned long long)__double_as_longlong(fabs(v.x) + fabs(v.y)) + 1ull;
    if (cb == oc) {
      if (B.done[i]) Ut[utri(B.pos[i], col)] = v;
      else colbuf[rb * TB + i] = v;
    }
    if (kk[i] > key || (kk[i] == key && B.pos[i] < bp)) {
      key = kk[i];
      bp = B.pos[i];
    }
  });
  group_best8(key, bp);
  if (cb == oc) {
    static_for<TB>([&](auto I) {
      constexpr int i = I;
      if (!B.done[i] && kk[i] == key && B.pos[i] == bp) {
        s_perm[col] = rb * TB + i;
        s_pospiv[col & 1] = bp;
        s_uinv[col] = crecip_fast(B.v[i][JJ]);
        if (key <= 1ull) *s_sing = 1;  // the largest candidate is zero
      }
    });
  }
}

template <int G, int TB>
__global__ __launch_bounds__(G * G) void k_lu_inv_2d(int n, const double2 *__restrict__ A,
                                                     long long sA, double2 *__restrict__ Ainv,
                                                     long long sAinv,
                                                     const int *__restrict__ active,
                                                     int *__restrict__ status) {
  typedef double2 C;
  constexpr int LD = G * TB;  // rows (and columns) of the padded block
  static_assert(G == 8, "one wave, thread columns of 8 lanes");
  const int b = blockIdx.x;
  if (active && active[b] == 0) return;
  extern __shared__ __align__(16) unsigned char lsm[];
  C *Ut = (C *)lsm;  // U(i, c), i < c (positions), at utri(i, c)
  __shared__ int s_perm[LD];
  __shared__ C s_uinv[LD];
  __shared__ int s_pospiv[2];
  __shared__ int s_sing;
  __shared__ C colbuf[2][LD];
  const int tid = threadIdx.x, cb = tid / G, rb = tid % G;
  const int gbase = (tid & 63) - rb;  // lane of this thread column's rb = 0
  const C *Ab = A + (long long)b * sA;
  LuBlk<TB> B;
  static_for<TB>([&](auto I) {
    constexpr int i = I;
    const int r = rb * TB + i;
    B.pos[i] = r;
    B.done[i] = r >= n;
    static_for<TB>([&](auto J) {
      const int c = cb * TB + J;
      B.v[i][J] = (r < n && c < n) ? Ab[r + (size_t)c * n] : C{0, 0};
    });
  });
  if (tid == 0) s_sing = 0;
  lu_publish<G, TB, 0>(0, tid, B, Ut, colbuf[0], s_perm, s_pospiv, s_uinv, &s_sing);
  __syncthreads();

  for (int k0 = 0; k0 < n; k0 += TB) {
    static_for<TB>([&](auto KK) {
      constexpr int kk = KK;
      const int k = k0 + kk;
      if (k >= n) return;  // uniform
      const int p = s_perm[k], pos_p = s_pospiv[k & 1];
      const C pinv = s_uinv[k];
      const int prb = p / TB, pi = p - prb * TB;
      const bool own_k = cb == k0 / TB;
      C m[TB];
      static_for<TB>([&](auto I) {
        constexpr int i = I;
        const int r = rb * TB + i;
        if (r == p) {
          B.pos[i] = k;
          B.done[i] = true;
        } else if (B.pos[i] == k) {
          B.pos[i] = pos_p;
        }
        m[i] = B.done[i] ? C{0, 0} : cmul(colbuf[k & 1][r], pinv);
        // register column k becomes Y's column k: 1 on the pivot row
        if (own_k) B.v[i][kk] = C{r == p ? 1.0 : 0.0, 0.0};
      });
      // row p for this thread's columns, from the lane of this thread column
      // that holds it (same wave)
      const int ps = __builtin_amdgcn_readfirstlane(pi);
      static_for<TB>([&](auto J) {
        const C u = bperm(pick0<TB, J>(B.v, ps), (gbase + prb) << 2);
        static_for<TB>([&](auto I) { B.v[I][J] = fms_c(B.v[I][J], m[I], u); });
      });
      if (k + 1 < n)
        lu_publish<G, TB, (kk + 1) % TB>(k + 1, tid, B, Ut, colbuf[(k + 1) & 1], s_perm,
                                         s_pospiv, s_uinv, &s_sing);
      __syncthreads();
    });
  }

  // back substitution U X = Y, position i = n-1 .. 0, each wave on its own
  // columns: row i of X (row q of Y / U(i, i), left unscaled in the registers
  // of row q) from the lane of this thread column that holds row q
  for (int i = n - 1; i >= 0; --i) {
    const int q = s_perm[i];
    const C uinv = s_uinv[i];
    const int qrb = q / TB, qs = __builtin_amdgcn_readfirstlane(q - qrb * TB);
    C coef[TB];
    static_for<TB>([&](auto T) {
      coef[T] = (B.pos[T] < i) ? Ut[utri(B.pos[T], i)] : C{0, 0};
    });
    static_for<TB>([&](auto J) {
      const C xq = bperm(cmul(pick0<TB, J>(B.v, qs), uinv), (gbase + qrb) << 2);
      // coef = 0 on row q and below position i
      static_for<TB>([&](auto T) { B.v[T][J] = fms_c(B.v[T][J], coef[T], xq); });
    });
  }
  // rows of X: the scaling by 1 / U(pos, pos) left out above
  static_for<TB>([&](auto I) {
    if (rb * TB + I < n) {
      const C ui = s_uinv[B.pos[I]];
      static_for<TB>([&](auto J) { B.v[I][J] = cmul(B.v[I][J], ui); });
    }
  });
  // column j of X = U^-1 L^-1 is column perm(j) of the inverse
  C *Ob = Ainv + (long long)b * sAinv;
  static_for<TB>([&](auto J) {
    const int c = cb * TB + J;
    if (c < n) {
      const int pc = s_perm[c];
      static_for<TB>([&](auto I) {
        if (rb * TB + I < n) Ob[B.pos[I] + (size_t)pc * n] = B.v[I][J];
      });
    }
  });
  if (tid == 0 && s_sing && status) atomicOr(&status[b], (int)ST_SINGULAR);
}

// ---------------------------------------------------------------------------
// LU inverse of blocks up to 128 on the matrix cores, one workgroup per block
// ---------------------------------------------------------------------------
// The reference's algorithm: ZGETRF (partial pivoting; the pivot is the first
// largest |Re| + |Im| of the column in the current row order, as IZAMAX picks
// it) followed by ZGETRS against the identity (inversions.F90:807-839).
//
// NP = ceil(n / 16) waves; wave w holds columns 16w .. 16w+15 of all
// R = 16 NP rows in the accumulator layout of v_mfma_f64_4x4x4: lane
// 16a + 4b + c, strip s, quad q <-> row 16s + 4b + a, column 16w + 4q + c.
// Rows are never moved during the elimination: pos is a row's position in
// LAPACK's row order and a pivot step exchanges two positions.  One register
// block holds both factors in place: a row pivoted at step k keeps U at
// columns >= k and Y = L^-1 P left of it (unit diagonal implied), rows not
// pivoted yet hold A right of the current step and Y left of it.
//
// Per panel of 4 columns: the wave that owns them turns them into one row per
// lane (two above n = 64) through its LDS scratch and runs the 4 steps alone --
// pivot search by DPP, the pivot row by readlane, no barrier -- and publishes
// the panel (two buffers, one barrier per panel).  Every wave then adds
// Z * (pivot rows of its own columns), Z the panel's Y (L11^-1 - I on the pivot
// rows, -L21 L11^-1 below, 0 on rows pivoted before): one K = 4 product, 16 NP
// matrix instructions per wave.  Four columns, since the explicit L11^-1 costs
// accuracy as it grows: on blocks with random +-0.97 multipliers 16 columns gave
// 2.4 - 2.9 times LAPACK's error, four give 0.95 - 0.99, and the transmission of
// ribbons of 24 to 90 orbitals had 4 - 22 % more error in the mean over 800
// energies than elimination one column at a time, now 4 % more to 6 % less.  And
// since four columns take 16 registers per row of a lane instead of 64, so that
// more waves share a SIMD.
//
// Then every wave sorts its rows by position and the back substitution
// U X = Y runs by blocks of 16: U_ii X_i = Y_i row by row (explicit U_ii^-1 lost
// a digit on nearly singular ribbon blocks), then Y_s -= U_si X_i (s < i) on the
// matrix cores.  Operand B of these
// products is the register block itself: block b of the instruction takes its
// k index from quad (b + r) % 4, r = 0 .. 3, which is a DPP row rotation, and
// A is read from LDS in the matching order.  Column j of X is column perm(j)
// of the inverse (the row pivoted at step j).
//
// FP32 blocks are converted on load and store and run in FP64.

// 1/b for a pivot without a branch, so that it overlaps the search (0 for
// b == 0): b scaled as in crecip_fast, one Newton-Raphson step on 1/|b'|^2 and
// one on the complex reciprocal itself, p <- p + p (1 - b p), which leaves
// little but the rounding of p (inverses of a ribbon's first decimation step:
// error 3.2e-16, with crecip_fast's two real steps 3.5e-16)
__device__ inline double2 crecip_sel(double2 b) {
  const double mx = fmax(fabs(b.x), fabs(b.y));
  const int e = __builtin_amdgcn_frexp_exp(mx);
  const double x = __builtin_amdgcn_ldexp(b.x, -e), y = __builtin_amdgcn_ldexp(b.y, -e);
  const double d = fma(x, x, y * y);
  double r = __builtin_amdgcn_rcp(d);
  r = fma(r, fma(-d, r, 1.0), r);
  r = mx == 0.0 ? 0.0 : r;
  const double px = x * r, py = -y * r;
  const double er = fma(y, py, fma(-x, px, 1.0)), ei = fma(-y, px, -x * py);
  return double2{__builtin_amdgcn_ldexp(fma(-py, ei, fma(px, er, px)), -e),
                 __builtin_amdgcn_ldexp(fma(px, ei, fma(py, er, py)), -e)};
}
// f64 maximum over the wave, in every lane's SGPR copy
template <int CTRL, int ROWS> __device__ inline double dpp_max(double v) {
  const int lo = __double2loint(v), hi = __double2hiint(v);
  // every lane of a row pattern has a source; the broadcasts leave masked rows
  const int l2 = ROWS == 0xF ? __builtin_amdgcn_update_dpp(0, lo, CTRL, ROWS, 0xF, true)
                             : __builtin_amdgcn_update_dpp(lo, lo, CTRL, ROWS, 0xF, false);
  const int h2 = ROWS == 0xF ? __builtin_amdgcn_update_dpp(0, hi, CTRL, ROWS, 0xF, true)
                             : __builtin_amdgcn_update_dpp(hi, hi, CTRL, ROWS, 0xF, false);
  return fmax(v, __hiloint2double(h2, l2));
}
__device__ inline double wave_fmax(double v) {
  v = dpp_max<0xB1, 0xF>(v);   // quad_perm [1,0,3,2]
  v = dpp_max<0x4E, 0xF>(v);   // quad_perm [2,3,0,1]
  v = dpp_max<0x141, 0xF>(v);  // row_half_mirror
  v = dpp_max<0x140, 0xF>(v);  // row_mirror
  v = dpp_max<0x142, 0xA>(v);  // row_bcast:15
  v = dpp_max<0x143, 0xC>(v);  // row_bcast:31
  return lane_read(v, 63);
}
template <int CTRL> __device__ inline double dpp_mov(double v) {
  return __hiloint2double(
      __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, true),
      __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, true));
}
// quad (b + r) % 4 of every row of 16 lanes, into quad b
template <int r> __device__ inline double quad_rot(double v) {
  if constexpr (r == 0) return v;
  else if constexpr (r == 1) return dpp_mov<0x12C>(v);  // row_ror:12
  else if constexpr (r == 2) return dpp_mov<0x128>(v);  // row_ror:8
  else return dpp_mov<0x124>(v);                        // row_ror:4
}

// LDS of k_lu_inv_mx<NP>, in double2: two published panels (4 columns of R + 1
// rows each) and per wave a scratch of 4 columns x R rows or of 4 x 17 pivot-row
// entries; then the packed triangles U_ii and every U_si, s < i
template <int NP> struct LuLds {
  static constexpr int R = 16 * NP, LD = R + 1;
  static constexpr int UI = 136;                 // packed 16 x 16 triangle
  static constexpr int SHARED = 2 * 4 * LD;
  static constexpr int SCR = 4 * R > 4 * 17 ? 4 * R : 4 * 17;
  static constexpr int ELIM = SHARED + NP * SCR;
  static constexpr int BACK = NP * UI + (NP * (NP - 1)) / 2 * 272;
  static constexpr size_t bytes = (size_t)(ELIM > BACK ? ELIM : BACK) * sizeof(double2);
};

// c[q] += a b[q] for four column quads on the matrix cores, the K = 4 products
// summed apart and added once: into c itself every one of their eight terms is
// rounded at the size of c (inverses of a ribbon's converged surface blocks and
// of its sweep blocks, order 64: error 8.0e-16 and 16e-16, apart 3.9e-16 and
// 7.8e-16; 3 % longer)
__device__ __forceinline__ void mfma_c4(double ar, double ai, const double (&br)[4],
                                        const double (&bi)[4], double (&cr)[4], double (&ci)[4]) {
  const double nai = -ai;
  double tr[4], ti[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    tr[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, br[q], 0.0, 0, 0, 0);
    ti[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(ar, bi[q], 0.0, 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    tr[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(nai, bi[q], tr[q], 0, 0, 0);
    ti[q] = __builtin_amdgcn_mfma_f64_4x4x4f64(ai, br[q], ti[q], 0, 0, 0);
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    cr[q] += tr[q];
    ci[q] += ti[q];
  }
}

// Keeps a value's computation here: the compiler otherwise sinks the updates
// of an unrolled section to their last use and holds all of its operands.
__device__ __forceinline__ void pin(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void pin(double2 &v) {
  pin(v.x);
  pin(v.y);
}
// orders the LDS accesses of one wave among its own lanes
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Waves per SIMD the registers are kept for.  Workgroups of 5 waves need 4: with
// 3 (no spills) the second workgroup of a CU found no room on the SIMD that
// holds two waves of the first; order 65, 1 / 500 / 2000 blocks 122 / 241 / 874
// us with 3, 128 / 181 / 708 with 4.  Of 6 waves 3: LDS and 263 spilled registers
// eat up what the second workgroup gives (order 96, 189 / 376 / 1394 us with 3,
// 222 / 337 / 1387 with 4).
constexpr int lu_waves(int np) { return np <= 5 ? 4 : np <= 6 ? 3 : 2; }

template <int NP, typename IO>
__global__ __launch_bounds__(64 * NP, lu_waves(NP)) void k_lu_inv_mx(int n, const IO *__restrict__ A,
                                                       long long sA, IO *__restrict__ Ainv,
                                                       long long sAinv,
                                                       const int *__restrict__ active,
                                                       int *__restrict__ status) {
  typedef double2 C;
  typedef LuLds<NP> L;
  constexpr int R = L::R, LD = L::LD, RT = (R + 63) / 64;
  const int b = blockIdx.x;
  if (active && active[b] == 0) return;
  extern __shared__ __align__(16) unsigned char lsm[];
  C *pan = (C *)lsm;
  __shared__ int s_pos[R];     // position of each row
  __shared__ int s_rowt[2][R];  // a panel's rows: -1 pivoted before, 0..3 pivot step, 4 not pivoted
  __shared__ int s_perm[R];    // row pivoted at each step
  __shared__ C s_uinv[R];      // reciprocal pivots by step
  __shared__ int s_sing;
  const int tid = threadIdx.x;
  // Wave -> columns, rotated by the dispatch round: the waves of a workgroup go
  // to the SIMDs in order, so without it the panel waves of all workgroups that
  // share a CU (started together) would run on one SIMD at a time.
  const int w = __builtin_amdgcn_readfirstlane((int)((tid >> 6) + (blockIdx.x >> 8)) % NP);
  C *scr = pan + L::SHARED + w * L::SCR;
  int l = tid & 63;
  int la = l >> 4, lb = (l >> 2) & 3, lc = l & 3;
  int drow = 4 * lb + la;  // row of the lane inside a strip
  // the lane's indices anew: addresses are then formed where they are used
  // instead of being kept in registers across the whole kernel
  auto fresh_lane = [&] {
    asm volatile("" : "+v"(l));
    la = l >> 4;
    lb = (l >> 2) & 3;
    lc = l & 3;
    drow = 4 * lb + la;
  };

  // ---- load ----
  double mr[NP][4], mi[NP][4];
  {
    const IO *Ab = A + (long long)b * sA;
    static_for<NP>([&](auto S) {
      static_for<4>([&](auto Q) {
        const int r = 16 * S + drow, c = 16 * w + 4 * Q + lc;
        const bool in = r < n && c < n;
        const IO v = Ab[in ? r + c * n : 0];
        mr[S][Q] = in ? v.x : 0.0;
        mi[S][Q] = in ? v.y : 0.0;
      });
    });
  }
  for (int r = tid; r < R; r += 64 * NP) {
    s_pos[r] = r;
    s_uinv[r] = C{0, 0};
  }
  if (tid == 0) s_sing = 0;
  __syncthreads();

  // ---- elimination ----
#pragma unroll 1
  for (int P = 0; P < NP; ++P) {
    static_for<4>([&](auto G) {
      constexpr int buf = G & 1;
      const int k0 = 16 * P + 4 * G, kmax = min(4, n - k0);
      if (kmax <= 0) return;  // uniform
      C *pn = pan + buf * 4 * LD;
      fresh_lane();
      if (w == P) {
        C v[RT][4];
        int pos[RT], rowt[RT];
        // own columns: one row per lane (and l + 64)
        static_for<NP>([&](auto S) { scr[lc * R + 16 * S + drow] = C{mr[S][G], mi[S][G]}; });
        wave_lds_fence();
        static_for<RT>([&](auto T) {
          const int r = l + 64 * T, rr = min(r, R - 1);
          static_for<4>([&](auto J) { v[T][J] = scr[J * R + rr]; });
          pos[T] = r < n ? s_pos[r] : -1;  // padding rows count as pivoted
          rowt[T] = pos[T] < k0 ? -1 : 4;
        });
        bool sing = false;
        static_for<4>([&](auto J) {
          constexpr int j = J;
          const int k = k0 + j;
          if (k >= n) return;  // uniform
          // the lane's largest candidate, its position and reciprocal, and the
          // wave's maximum; NaN and Inf count as the largest finite number: a
          // NaN is a pivot like any other and spreads over the inverse
          double best = -1.0;
          int bp = 0x7fffffff;
          C cand = C{0, 0};
          static_for<RT>([&](auto T) {
            const double m = pos[T] >= k ? fmin(fabs(v[T][j].x) + fabs(v[T][j].y), DBL_MAX) : -1.0;
            const bool hit = m > best || (T > 0 && m == best && m >= 0.0 && pos[T] < bp);
            best = hit ? m : best;
            bp = hit ? pos[T] : bp;
            cand.x = hit ? v[T][j].x : cand.x;
            cand.y = hit ? v[T][j].y : cand.y;
          });
          const C rc = crecip_sel(cand);
          const double vmax = wave_fmax(best);
          unsigned long long hits = __ballot(best == vmax && bp != 0x7fffffff);
          if (hits & (hits - 1)) {  // ties go to the smallest position
            const unsigned key = ((hits >> l) & 1) ? (unsigned)bp : 0xFFFFFFFFu;
            const unsigned mn = wave_min32(key);
            hits = __ballot(key == mn);
          }
          const int pl = __ffsll((long long)hits) - 1;  // n - k rows are left
          // which of the lane's rows, and its position
          int psel = 0;
          if constexpr (RT > 1) psel = __builtin_amdgcn_readlane(bp == pos[1] ? 1 : 0, pl);
          const int pp = __builtin_amdgcn_readlane(bp, pl);
          C pinv = C{lane_read(rc.x, pl), lane_read(rc.y, pl)};
          if constexpr (sizeof(IO) == sizeof(float2))
            if (vmax == DBL_MAX) {  // FP32: a NaN is flagged, the reciprocal of Inf is 0
              const double px = lane_read(cand.x, pl), py = lane_read(cand.y, pl);
              pinv = crecip(C{px, py});
              sing |= px != px || py != py;
            }
          sing |= vmax == 0.0;
          if (l == j) {
            s_perm[k] = pl + 64 * psel;
            s_uinv[k] = pinv;
          }
          C m[RT];
          static_for<RT>([&](auto T) {
            const bool piv = l == pl && psel == T;
            if (piv) {
              pos[T] = k;
              rowt[T] = j;
            } else if (pos[T] == k) {
              pos[T] = pp;
            }
            const bool live = pos[T] > k;
            const C t = cmul(v[T][j], pinv);
            m[T] = live ? t : C{0, 0};
          });
          // the other columns, from the pivot row in lane pl
          C y[4];
          if (RT > 1 && psel)
            static_for<4>([&](auto I) {
              if (I != j) y[I] = C{lane_read(v[RT - 1][I].x, pl), lane_read(v[RT - 1][I].y, pl)};
            });
          else
            static_for<4>([&](auto I) {
              if (I != j) y[I] = C{lane_read(v[0][I].x, pl), lane_read(v[0][I].y, pl)};
            });
          static_for<RT>([&](auto T) {
            static_for<3>([&](auto I) {  // the next column first
              constexpr int c = (j + 1 + I) & 3;
              v[T][c] = fms_c(v[T][c], m[T], y[c]);
            });
            // the column becomes Y's: -m below, U above and on the pivot row
            const bool live = pos[T] > k;
            v[T][j].x = live ? -m[T].x : v[T][j].x;
            v[T][j].y = live ? -m[T].y : v[T][j].y;
          });
        });
        if (sing && l == 0) s_sing = 1;
        static_for<RT>([&](auto T) {
          const int r = l + 64 * T;
          if (r < n) s_pos[r] = pos[T];
          if (r < R) {
            s_rowt[buf][r] = rowt[T];
            static_for<4>([&](auto J) { pn[J * LD + r] = v[T][J]; });
          }
        });
      }
      // the panel is published; everyone has read the one before the last
      __syncthreads();
      // pivot rows of the wave's own columns -> scratch, row t = pivot step
      if (kmax < 4) {
        for (int e = l; e < 4 * 17; e += 64) scr[e] = C{0, 0};
        wave_lds_fence();
      }
      static_for<NP>([&](auto S) {
        const int t = s_rowt[buf][16 * S + drow];
        if (t >= 0 && t < 4)
          static_for<4>([&](auto Q) { scr[t * 17 + 4 * Q + lc] = C{mr[S][Q], mi[S][Q]}; });
      });
      wave_lds_fence();
      double br[4], bi[4];
      static_for<4>([&](auto Q) {
        const C x = scr[la * 17 + 4 * Q + lc];
        br[Q] = x.x;
        bi[Q] = x.y;
      });
      static_for<NP>([&](auto S) {
        C z = pn[la * LD + 16 * S + (l & 15)];
        if (la >= s_rowt[buf][16 * S + (l & 15)]) z = C{0, 0};
        mfma_c4(z.x, z.y, br, bi, mr[S], mi[S]);
        static_for<4>([&](auto Q) { pin(mr[S][Q]); pin(mi[S][Q]); });
      });
      if (w == P)  // the panel's own columns
        static_for<NP>([&](auto S) {
          const C x = pn[lc * LD + 16 * S + drow];
          mr[S][G] = x.x;
          mi[S][G] = x.y;
        });
      wave_lds_fence();
    });
  }

  // ---- rows into position order ----
  fresh_lane();
  {
    int ps[NP];
    static_for<NP>([&](auto S) { ps[S] = s_pos[16 * S + drow]; });
    static_for<4>([&](auto Q) {
      static_for<NP>([&](auto S) { scr[lc * R + ps[S]] = C{mr[S][Q], mi[S][Q]}; });
      wave_lds_fence();
      static_for<NP>([&](auto S) {
        const C x = scr[lc * R + 16 * S + drow];
        mr[S][Q] = x.x;
        mi[S][Q] = x.y;
      });
      wave_lds_fence();
    });
  }
  __syncthreads();  // the last panel has been read: pan is reused
  fresh_lane();
  // ---- U to LDS: the triangles U_ww (packed by columns) and U_sw (s < w); the
  // registers keep Y, unit lower triangular ----
  C *ut = pan, *ub = pan + NP * L::UI;
  static_for<NP>([&](auto S) {
    if (S < w) {
      C *u = ub + ((w * (w - 1)) / 2 + S) * 272;
      static_for<4>([&](auto Q) {
        u[(4 * Q + lc) * 17 + drow] = C{mr[S][Q], mi[S][Q]};
        mr[S][Q] = 0.0;
        mi[S][Q] = 0.0;
      });
    } else if (S == w) {
      static_for<4>([&](auto Q) {
        const int c = 4 * Q + lc;
        if (drow <= c) ut[w * L::UI + (c * (c + 1)) / 2 + drow] = C{mr[S][Q], mi[S][Q]};
        mr[S][Q] = c < drow ? mr[S][Q] : (c == drow ? 1.0 : 0.0);
        mi[S][Q] = c < drow ? mi[S][Q] : 0.0;
      });
    }
  });
  __syncthreads();
  // ---- back substitution by blocks of 16 positions, every wave on its own ----
  static_for<NP>([&](auto K) {
    constexpr int i = NP - 1 - K;
    fresh_lane();
    // U_ii X_i = Y_i row by row: row k of every column from the lanes holding it
#pragma unroll 1
    for (int k = min(15, n - 1 - 16 * i); k >= 0; --k) {
      const int src = (16 * (k & 3) + 4 * (k >> 2) + lc) << 2;
      const C ui = s_uinv[16 * i + k];
      C t = C{0, 0};
      if (drow < k) t = ut[i * L::UI + (k * (k + 1)) / 2 + drow];
      static_for<4>([&](auto Q) {
        const C x = cmul(C{bperm(mr[i][Q], src), bperm(mi[i][Q], src)}, ui);
        const C y = fms_c(C{mr[i][Q], mi[i][Q]}, t, x);
        mr[i][Q] = drow == k ? x.x : y.x;
        mi[i][Q] = drow == k ? x.y : y.y;
      });
    }
    if constexpr (i > 0) {
      static_for<4>([&](auto Rr) {
        double br[4], bi[4];
        static_for<4>([&](auto Q) {
          br[Q] = quad_rot<Rr>(mr[i][Q]);
          bi[Q] = quad_rot<Rr>(mi[i][Q]);
        });
        const int row = 4 * lb + lc, col = 4 * ((lb + Rr) & 3) + la;
        static_for<i>([&](auto S) {
          const C u = ub[((i * (i - 1)) / 2 + S) * 272 + col * 17 + row];
          mfma_c4(-u.x, -u.y, br, bi, mr[S], mi[S]);
          static_for<4>([&](auto Q) { pin(mr[S][Q]); pin(mi[S][Q]); });
        });
      });
    }
  });
  // ---- column j of X = U^-1 L^-1 is column perm(j) of the inverse ----
  fresh_lane();
  IO *Ob = Ainv + (long long)b * sAinv;
  static_for<4>([&](auto Q) {
    const int c = 16 * w + 4 * Q + lc;
    if (c < n) {
      const size_t pc = (size_t)s_perm[c] * n;
      static_for<NP>([&](auto S) {
        const int r = 16 * S + drow;
        if (r < n) {
          IO o;
          o.x = mr[S][Q];
          o.y = mi[S][Q];
          Ob[r + pc] = o;
        }
      });
    }
  });
  if (tid == 0 && s_sing && status) atomicOr(&status[b], (int)ST_SINGULAR);
}


// "row already pivoted" flags of a lane's RT register rows: an array, or at
// 16 rows per lane the bits of one register (the panel then holds 128)
template <int RT, bool BITS = (RT >= 16)> struct RowFlags {
  int f[RT];
  __device__ __forceinline__ int get(int i) const { return f[i]; }
  __device__ __forceinline__ void set(int i, int v) { f[i] = v; }
};
template <int RT> struct RowFlags<RT, true> {
  static_assert(RT <= 32, "one 32-bit mask");
  unsigned m = 0;
  __device__ __forceinline__ int get(int i) const { return (int)((m >> i) & 1u); }
  __device__ __forceinline__ void set(int i, int v) { m = v ? (m | (1u << i)) : (m & ~(1u << i)); }
};

// rows of the LDS staging buffer of k_inv_gj (a chunk of the n x 8CT panel,
// rows padded by one element); at 16 rows per lane the multiplier buffers
// (2 x 64 RT elements) take their share of the budget
template <typename R, int RT, int CT>
constexpr int gj_stage_rows() {
  constexpr int rowb = (8 * CT + 1) * 2 * (int)sizeof(R);
  constexpr int budget = 140 * 1024 - (RT >= 16 ? 2 * 64 * RT * 2 * (int)sizeof(R) : 0);
  constexpr int cr = (budget / rowb) & ~63;
  return cr < 64 * RT ? cr : 64 * RT;
}
template <typename R, int RT, int CT>
constexpr size_t gj_stage_bytes() {
  return (size_t)gj_stage_rows<R, RT, CT>() * (8 * CT + 1) * 2 * sizeof(R);
}

// Gauss-Jordan elimination over one super-panel S = columns [s0, s0+sw),
// sw <= 8 CT, of the row-major view M = A^T of an item (row r of M is column r
// of A, so rows of M are contiguous in memory).
//
// Wave w (of 8) holds columns s0 + w*CT .. +CT, lane l the rows l + 64 i
// (i < RT), in registers (loaded and stored through an LDS staging buffer so
// that global accesses run along rows).  Every step writes each updated value
// one register lower (register 0 moves to the last), so the wave owning the
// current pivot column always finds it in register 0 and no register is
// indexed at run time; CT steps restore the order.
//
// Step j, pivot column owned by wave wj = j / CT, one barrier:
//   every thread reads the pivot key (row p, the largest |.|_1 over the
//   unpivoted rows) and 1/B(p, j); each wave reads its CT entries of row p
//   from the lane holding them (1 in place of column j); every row applies
//   B(r, :) -= (B(r, j)/B(p, j)) B(p, :), the multipliers of the other waves'
//   rows coming from LDS, and the pivot row becomes B(p, :)/B(p, j) (1/B(p, j)
//   in column j).  The wave owning the next pivot column updates that column
//   first and, before its other columns, publishes the column (the next
//   multipliers) and its pivot candidate with the reciprocal, so the search
//   overlaps the update.  LDS buffers alternate between steps.
//
// With Ẑ = B(:, S) - E (E: ones at (pivot row, column)) the columns J outside
// S then take B(:, J) += Ẑ B_old(piv, J).  In A's column-major layout that is
// A(J', :) += Rb Ẑ^T with Rb(c, k) = A(c, piv_k) -- contiguous columns of A --
// and J' the rows of A outside S.  Ẑ^T is the rows S of A less E^T, and
// -Rb E^T only cancels A(J', piv_k): the kernel moves those entries into Rb
// (ld n; rows of S are not written) and leaves zeros, so that the deferred
// update on the matrix cores is the plain product A(J', :) += Rb A(S, :).
template <typename R, int RT, int CT>
__global__ __launch_bounds__(NTG) void k_inv_gj(int n, int s0, int sw,
                                                typename CT_<R>::t *__restrict__ A, long long sA,
                                                typename CT_<R>::t *__restrict__ Rb,
                                                int *__restrict__ used_g, int *__restrict__ piv_g,
                                                const int *__restrict__ active,
                                                int *__restrict__ status) {
  typedef typename CT_<R>::t C;
  static_assert(CT >= 2, "the look-ahead needs two columns per wave");
  constexpr int SWC = 8 * CT, LDST = SWC + 1;
  constexpr int CR = gj_stage_rows<R, RT, CT>();
  constexpr int PER = CR * SWC / NTG;  // staged elements per thread and chunk
  const int b = blockIdx.x;
  if (active && active[b] == 0) return;
  extern __shared__ __align__(16) unsigned char gsm[];
  C *stage = (C *)gsm;
  __shared__ C mcol[2][64 * RT];
  __shared__ unsigned redk[2];
  __shared__ C redinv[2];
  __shared__ int spiv[SWC];
  __shared__ int s_sing;
  const int tid = threadIdx.x, w = tid >> 6, l = tid & 63;
  C *Xb = A + (long long)b * sA;
  int *ug = used_g + (long long)b * n;

  C P[RT][CT];
  RowFlags<RT> used;
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = l + 64 * i;
    used.set(i, r >= n ? 1 : (s0 == 0 ? 0 : ug[r]));
#pragma unroll
    for (int c = 0; c < CT; ++c) P[i][c] = C{0, 0};
  }
  if (tid == 0) s_sing = 0;
  // ---- load the panel in chunks of CR rows, NPF chunks' global loads
  // issued together (one at 16 rows per lane, where the panel itself holds
  // 128 registers), coalesced along rows of M ----
  static_assert(CR % 64 == 0, "a lane's rows fall in one chunk each");
  constexpr int NCH = (64 * RT + CR - 1) / CR;
  constexpr int NPF = RT >= 16 ? 1 : 2;
#pragma unroll
  for (int h0 = 0; h0 < NCH; h0 += NPF) {
  C ld[NPF][PER];
#pragma unroll
  for (int h = 0; h < NPF; ++h)
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + NTG * k;
      const int row = (h0 + h) * CR + e / SWC, col = e % SWC;
      ld[h][k] = (h0 + h < NCH && row < n && col < sw) ? Xb[(size_t)row * n + s0 + col] : C{0, 0};
    }
#pragma unroll
  for (int h = 0; h < NPF; ++h) {
    const int cr0 = (h0 + h) * CR;
    if (h0 + h < NCH && cr0 < n) {  // uniform
#pragma unroll
      for (int k = 0; k < PER; ++k) {
        const int e = tid + NTG * k;
        stage[(e / SWC) * LDST + e % SWC] = ld[h][k];
      }
      __syncthreads();
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int r = l + 64 * i;
        if (r >= cr0 && r < cr0 + CR) {
          const C *src = stage + (r - cr0) * LDST + w * CT;
#pragma unroll
          for (int c = 0; c < CT; ++c) P[i][c] = src[c];
        }
      }
      __syncthreads();
    }
  }
  }

  // the owning wave's column (register 0) -> multipliers in mcol[bb] and the
  // pivot candidate (largest key over the wave's unpivoted rows) with its
  // reciprocal in redk[bb] / redinv[bb]
  // exact search: the largest |Re| + |Im| (its FP64 bit pattern as a 64-bit
  // key), ties to the smallest row; the winner publishes its row as a
  // pivot_key (decoded by every wave) and its reciprocal
  auto candidate = [&](int bb) {
    unsigned long long kb = 0;
    int rb = 0x7fffffff;
    double vb = 0.0;
    C cv = C{0, 0};
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int r = l + 64 * i;
      if (r < n) mcol[bb][r] = P[i][0];
      const double v = (double)cabs1(P[i][0]);
      const unsigned long long key =
          used.get(i) ? 0ull : (unsigned long long)__double_as_longlong(v) + 1ull;
      if (key > kb) { kb = key; rb = r; vb = v; cv = P[i][0]; }  // rows grow with i
    }
    const unsigned long long km = wave_max64(kb);
    const unsigned rmin = wave_min32(kb == km ? (unsigned)rb : 0xFFFFFFFFu);
    if (km != 0 && kb == km && (unsigned)rb == rmin) {
      redk[bb] = pivot_key(vb, rb);
      redinv[bb] = crecip_fast(cv);
    }
    if (km == 0 && l == 0) redk[bb] = 0;
  };
  if (w == 0) candidate(0);
  __syncthreads();

  for (int j = 0; j < sw; ++j) {
    const int bf = j & 1, wj = j / CT;
    // ---- pivot row p and 1/B(p, j); each wave reads its columns of row p
    // from the lane holding it ----
    const unsigned kx = redk[bf];
    const int p = kx ? 1023 - (int)(kx & 1023) : -1;
    if (tid == 0 && (kx >> 11) == 0) s_sing = 1;  // zero (or NaN) pivot
    const C pinv = kx ? redinv[bf] : C{0, 0};
    const int lp = p & 63, ip = p >> 6;  // p < 0 cannot happen: j < n unpivoted rows remain
    C y[CT];
#pragma unroll
    for (int c = 0; c < CT; ++c) y[c] = C{0, 0};
#pragma unroll
    for (int i = 0; i < RT; ++i)
      if (p >= 0 && ip == i) {
#pragma unroll
        for (int c = 0; c < CT; ++c) y[c] = C{lane_read(P[i][c].x, lp), lane_read(P[i][c].y, lp)};
        if (l == lp) used.set(i, 1);
      }
    if (w == wj) y[0] = C{R(1), R(0)};  // column j itself
    if (w == wj && l == 0) spiv[j] = p < 0 ? 0 : p;
    // ---- B(r, :) -= l_r B(p, :), l_r = B(r, j) / B(p, j); old register k + 1
    // -> register k (the owning wave's column j, taken as 0, enters the last
    // register against the 1 in y[0]) ----
    if constexpr (RT >= 16) {
      // 16 rows per lane: row by row (multiplier, then the row's CT registers),
      // so no per-row arrays are held; the next column is published after the
      // whole update.  The same operations on every element as below.
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        const int r = l + 64 * i;
        const C m = (w == wj) ? P[i][0] : (r < n ? mcol[bf][r] : C{0, 0});
        C lmi = cmul(m, pinv);
        C x0i = (w == wj) ? C{0, 0} : P[i][0];
        if (r == p) {
          lmi = C{-pinv.x, -pinv.y};
          x0i = C{0, 0};
#pragma unroll
          for (int c = 1; c < CT; ++c) P[i][c] = C{0, 0};
        }
        const R nr = -lmi.x, ni = -lmi.y;
#pragma unroll
        for (int k = 0; k < CT; ++k) {
          const C yk = y[(k + 1) % CT];
          C x = k + 1 < CT ? P[i][k + 1] : x0i;
          x.x = fma(nr, yk.x, x.x);
          x.x = fma(-ni, yk.y, x.x);
          x.y = fma(nr, yk.y, x.y);
          x.y = fma(ni, yk.x, x.y);
          P[i][k] = x;
        }
      }
      if (j + 1 < sw && w == (j + 1) / CT) candidate(bf ^ 1);
      __syncthreads();
      continue;
    }
    C lm[RT], x0[RT];
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int r = l + 64 * i;
      const C m = (w == wj) ? P[i][0] : (r < n ? mcol[bf][r] : C{0, 0});
      lm[i] = cmul(m, pinv);
      x0[i] = (w == wj) ? C{0, 0} : P[i][0];
      if (r == p) {  // the pivot row becomes B(p, :) / B(p, j)
        lm[i] = C{-pinv.x, -pinv.y};
        x0[i] = C{0, 0};
#pragma unroll
        for (int c = 1; c < CT; ++c) P[i][c] = C{0, 0};
      }
    }
    auto upd = [&](int k) {
      const C yk = y[(k + 1) % CT];
#pragma unroll
      for (int i = 0; i < RT; ++i) {
        C x = k + 1 < CT ? P[i][k + 1] : x0[i];
        const R nr = -lm[i].x, ni = -lm[i].y;
        x.x = fma(nr, yk.x, x.x);
        x.x = fma(-ni, yk.y, x.x);
        x.y = fma(nr, yk.y, x.y);
        x.y = fma(ni, yk.x, x.y);
        P[i][k] = x;
      }
    };
    upd(0);  // the next pivot column of its wave lands in register 0
    if (j + 1 < sw && w == (j + 1) / CT) candidate(bf ^ 1);
#pragma unroll
    for (int k = 1; k < CT; ++k) upd(k);
    __syncthreads();
  }
  // restore the register order after a narrow super-panel
  for (int j = sw; j % CT != 0; ++j) {
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const C first = P[i][0];
#pragma unroll
      for (int c = 1; c < CT; ++c) P[i][c - 1] = P[i][c];
      P[i][CT - 1] = first;
    }
  }

  // ---- write the super-panel back, CR rows at a time ----
  for (int cr0 = 0; cr0 < n; cr0 += CR) {
    const int nr = min(CR, n - cr0);
    if (cr0 > 0) __syncthreads();  // the previous chunk has been read
#pragma unroll
    for (int i = 0; i < RT; ++i) {
      const int r = l + 64 * i;
      if (r >= cr0 && r < cr0 + nr) {
        C *dst = stage + (r - cr0) * LDST + w * CT;
#pragma unroll
        for (int c = 0; c < CT; ++c) dst[c] = P[i][c];
      }
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < PER; ++k) {
      const int e = tid + NTG * k;
      const int row = e / SWC, col = e % SWC;
      if (row < nr && col < sw) Xb[(size_t)(cr0 + row) * n + s0 + col] = stage[row * LDST + col];
    }
  }
#pragma unroll
  for (int i = 0; i < RT; ++i) {
    const int r = l + 64 * i;
    if (w == 0 && r < n) ug[r] = used.get(i);
  }
  if (tid < sw) piv_g[(long long)b * n + s0 + tid] = spiv[tid];
  if (Rb) {  // pivot columns of A outside the rows of S, moved to Rb; element e = (c, k)
    C *Rbb = Rb + (long long)b * kInvSuper * n;
    constexpr int GU = 8;  // loads in flight per thread
    const float inv_n = 1.0f / (float)n;  // e / n below is exact: e < 2^15, n <= 1024
    const int tot = sw * n;
    for (int base = 0; base < tot; base += NTG * GU) {
      C v[GU];
      long long o[GU];
#pragma unroll
      for (int u = 0; u < GU; ++u) {
        const int e = base + tid + NTG * u;
        const int k = (int)(((float)e + 0.5f) * inv_n), c = e - k * n;
        o[u] = (e < tot && (c < s0 || c >= s0 + sw)) ? c + (long long)spiv[k] * n : -1;
        v[u] = o[u] >= 0 ? Xb[o[u]] : C{0, 0};
      }
#pragma unroll
      for (int u = 0; u < GU; ++u)
        if (o[u] >= 0) {
          Rbb[base + tid + NTG * u] = v[u];
          Xb[o[u]] = C{0, 0};
        }
    }
  }
  if (tid == 0 && s_sing && status) atomicOr(&status[b], (int)ST_SINGULAR);
}

// Ainv(c, i) = B(ip[c], pv[i]): column i of the inverse is column pv[i] of
// the working matrix with its rows taken in the order ip (pv: pivot row of
// each logical column of M = A^T, ip its inverse permutation).
template <typename R>
__global__ __launch_bounds__(NT) void k_inv_unperm(int n, const typename CT_<R>::t *B,
                                                   long long sB, typename CT_<R>::t *Out,
                                                   long long sOut, const int *piv_g,
                                                   const int *active) {
  typedef typename CT_<R>::t C;
  extern __shared__ __align__(16) unsigned char smem[];
  const int b = blockIdx.y;
  if (active && active[b] == 0) return;
  int *pv = (int *)smem;
  int *ip = pv + n;
  const int *pg = piv_g + (long long)b * n;
  for (int c = threadIdx.x; c < n; c += NT) {
    int p = pg[c];
    pv[c] = (p >= 0 && p < n) ? p : 0;  // pivots are a permutation of [0, n)
    ip[c] = 0;
  }
  __syncthreads();
  for (int c = threadIdx.x; c < n; c += NT) ip[pv[c]] = c;
  __syncthreads();
  const C *Bb = B + (long long)b * sB;
  C *Ob = Out + (long long)b * sOut;
  // output columns handled by this workgroup: blockIdx.x * 8 .. +8
  for (int ii = 0; ii < 8; ++ii) {
    const int i = blockIdx.x * 8 + ii;
    if (i >= n) break;
    const C *src = Bb + (size_t)pv[i] * n;
    for (int c = threadIdx.x; c < n; c += NT) Ob[c + (size_t)i * n] = src[ip[c]];
  }
}

// Largest order of the one-workgroup LU kernel, above it the blocked
// Gauss-Jordan path.  1 / 500 / 2000 FP64 blocks, here against the thread-grid
// LU kernel used before (us, launch and wait included), at every batch no slower:
//   order 17   34 /  38 /   65    51 /  55 /   69
//   order 32   45 /  58 /   95    79 /  89 /  119
//   order 48   67 /  89 /  206   118 / 160 /  461
//   order 64   92 / 131 /  332   152 / 213 /  612
//   order 65  128 / 181 /  708   199 / 276 /  958
//   order 80  151 / 218 /  847   241 / 332 / 1165
//   order 96  189 / 380 / 1394   330 / 491 / 1697
// FP64 orders 97 to 128 stay on the blocked path, whose residuals are up to 15 %
// smaller (2.4e-16 ||A|| ||X||, here 2.4e-16 to 2.8e-16), though it takes longer:
// order 97 229 / 646 / 2635 us against 213 / 434 / 1660 here, order 128 292 / 831 /
// 3376 against 294 / 615 / 2346.  FP32
// (the block computed in FP64), 1 / 2000 blocks against Gauss-Jordan in LDS: order
// 64 93 / 321 against 260 / 676 us, order 65 134 / 721 against 314 / 790, order 128
// 0.28 / 2.2 against 1.4 / 11.3 ms; with one row or column beyond a multiple of 16
// and 2000 blocks it is 9 % slower at orders 17 and 33 (63 against 58 us, 147
// against 135), where one block takes 34 against 46 us and 53 against 88.
template <typename R> constexpr int kLuMaxN = sizeof(R) == 8 ? 96 : 128;

// FP32 blocks above it that still fit in LDS (up to order 140) take Gauss-Jordan
// there: residuals 1.0e-7, in the blocked FP32 path 1.5e-7 to 2.1e-7, though
// that is 5 to 9 times faster (order 129, 1 block: 2.6 against 0.31 ms).
template <typename R>
size_t gj_lds_bytes(int n) {
  typedef typename CT_<R>::t C;
  return (size_t)n * n * sizeof(C) + 2 * (size_t)n * sizeof(C) + (size_t)n * sizeof(int);
}
template <typename R>
bool gj_in_lds(int n) {
  return sizeof(R) == 4 && n <= NT && gj_lds_bytes<R>(n) <= (size_t)kLdsBudget;
}

template <typename Kern>
void allow_lds(Kern k, size_t bytes) {
  if (bytes > 64 * 1024)
    HN_CHECK(hipFuncSetAttribute((const void *)k, hipFuncAttributeMaxDynamicSharedMemorySize,
                                 (int)bytes));
}

template <int NP, typename IO>
void launch_lu(int n, IO *A, long long sA, IO *Ainv, long long sAinv, int batch, const int *active,
               int *status, hipStream_t s) {
  allow_lds(k_lu_inv_mx<NP, IO>, LuLds<NP>::bytes);
  hipLaunchKernelGGL((k_lu_inv_mx<NP, IO>), dim3(batch), dim3(64 * NP), LuLds<NP>::bytes, s, n, A, sA,
                     Ainv, sAinv, active, status);
  HN_CHECK(hipGetLastError());
}
template <typename IO>
void lu_mx(int n, IO *A, long long sA, IO *Ainv, long long sAinv, int batch, const int *active,
           int *status, hipStream_t s) {
  if constexpr (sizeof(IO) == sizeof(float2))  // FP64 up to 16: k_lu_inv_2d
    if (n <= 16) return launch_lu<1>(n, A, sA, Ainv, sAinv, batch, active, status, s);
  switch ((n + 15) / 16) {
    case 2: return launch_lu<2>(n, A, sA, Ainv, sAinv, batch, active, status, s);
    case 3: return launch_lu<3>(n, A, sA, Ainv, sAinv, batch, active, status, s);
    case 4: return launch_lu<4>(n, A, sA, Ainv, sAinv, batch, active, status, s);
    case 5: return launch_lu<5>(n, A, sA, Ainv, sAinv, batch, active, status, s);
    case 6: return launch_lu<6>(n, A, sA, Ainv, sAinv, batch, active, status, s);
    default: break;
  }
  if constexpr (sizeof(IO) == sizeof(float2)) {
    if (n <= 112) return launch_lu<7>(n, A, sA, Ainv, sAinv, batch, active, status, s);
    return launch_lu<8>(n, A, sA, Ainv, sAinv, batch, active, status, s);
  }
}

template <typename R>
void inv_impl(int n, typename CT_<R>::t *A, long long sA, typename CT_<R>::t *Ainv,
              long long sAinv, int batch, const int *active, int *status, const InvWork<R> &w,
              hipStream_t s) {
  if (n <= 0 || batch <= 0) return;
  // algorithmic work of the one-launch inverses: 8 n^3 flops and the block read
  // and written per item (items unknown for a mask without a count: -1)
  const double items = w.prof_items >= 0 ? (double)w.prof_items : (active ? -1.0 : (double)batch);
  const double sm_fl = items < 0 ? -1.0 : 8.0 * (double)n * n * n * items;
  const double sm_by = items < 0 ? 0.0 : 2.0 * sizeof(typename CT_<R>::t) * (double)n * n * items;
  if (n <= kLuMaxN<R>) {
    ProfScope ps(PT_INV_SMALL, sm_fl, sm_by, s);
    if constexpr (sizeof(R) == 8) {
      if (n <= 16) {  // one wave either way: 2000 blocks of order 10 take 32 us here, 36 below
        const size_t lds = std::max<size_t>(1, (size_t)n * (n - 1) / 2) * sizeof(double2);
        hipLaunchKernelGGL((k_lu_inv_2d<8, 2>), dim3(batch), dim3(64), lds, s, n, A, sA, Ainv, sAinv,
                           active, status);
        HN_CHECK(hipGetLastError());
        return;
      }
    }
    lu_mx(n, A, sA, Ainv, sAinv, batch, active, status, s);
    return;
  }
  if constexpr (sizeof(R) == 4) {
    if (gj_in_lds<R>(n)) {
      const size_t lds = gj_lds_bytes<R>(n);
      allow_lds(k_inv_lds<R>, lds);
      ProfScope ps(PT_INV_SMALL, sm_fl, sm_by, s);
      hipLaunchKernelGGL(k_inv_lds<R>, dim3(batch), dim3(NT), lds, s, n, A, sA, Ainv, sAinv,
                         active, status);
      HN_CHECK(hipGetLastError());
      return;
    }
  }
  if (n > 1024) throw std::runtime_error("inverse: block order > 1024 is not supported");
  if (sA < (long long)n * n || sAinv < (long long)n * n)
    throw std::runtime_error("inverse: item stride smaller than n*n");
  if (!w.Rb || w.n < n || w.batch < batch) throw std::runtime_error("inverse: workspace too small");
  // register tile per thread: 4 rows x 8 columns (super-panel 64) up to
  // n = 256, 8 rows x 4 columns (super-panel 32) up to n = 512, 16 rows x 2
  // columns (super-panel 16) up to n = 1024
  const int rpt = n <= 256 ? 1 : n <= 512 ? 2 : 4;
  const int spw = rpt == 1 ? 64 : rpt == 2 ? 32 : 16;
  for (int s0 = 0; s0 < n; s0 += spw) {
    const int sw = std::min(spw, n - s0);
    typename CT_<R>::t *rb = n > sw ? w.Rb : nullptr;
    {
      ProfScope ps(PT_INV_PANEL, -1.0, 0.0, s);
      if (rpt == 1) {
        allow_lds(k_inv_gj<R, 4, 8>, gj_stage_bytes<R, 4, 8>());
        hipLaunchKernelGGL((k_inv_gj<R, 4, 8>), dim3(batch), dim3(NTG),
                           (gj_stage_bytes<R, 4, 8>()), s, n, s0, sw, A, sA, rb, w.used,
                           w.piv, active, status);
      } else if (rpt == 2) {
        allow_lds(k_inv_gj<R, 8, 4>, gj_stage_bytes<R, 8, 4>());
        hipLaunchKernelGGL((k_inv_gj<R, 8, 4>), dim3(batch), dim3(NTG),
                           (gj_stage_bytes<R, 8, 4>()), s, n, s0, sw, A, sA, rb, w.used,
                           w.piv, active, status);
      } else {
        allow_lds(k_inv_gj<R, 16, 2>, gj_stage_bytes<R, 16, 2>());
        hipLaunchKernelGGL((k_inv_gj<R, 16, 2>), dim3(batch), dim3(NTG),
                           (gj_stage_bytes<R, 16, 2>()), s, n, s0, sw, A, sA, rb, w.used,
                           w.piv, active, status);
      }
    }
    HN_CHECK(hipGetLastError());
    if (rb) {  // deferred rank-sw update of every row of A outside the super-panel
      GemmArgs<R> g;
      g.m = n; g.n = n; g.k = sw;
      g.A = rb; g.sA = (long long)kInvSuper * n; g.lda = n; g.opA = OP_N;
      g.B = A + s0; g.sB = sA; g.ldb = n; g.opB = OP_N;
      g.C = A; g.sC = sA; g.ldc = n;
      g.alpha = {1.0, 0.0}; g.beta = {1.0, 0.0};
      g.active = active; g.skip_r0 = s0; g.skip_r1 = s0 + sw;
      g.batch = batch; g.tag = PT_GEMM_INV; g.prof_items = w.prof_items;
      if constexpr (sizeof(R) == 8) gemm_z(g, s);
      else gemm_c(g, s);
    }
  }
  hipLaunchKernelGGL(k_inv_unperm<R>, dim3((n + 7) / 8, batch), dim3(NT), 2 * n * sizeof(int), s,
                     n, A, sA, Ainv, sAinv, w.piv, active);
  HN_CHECK(hipGetLastError());
}

}  // namespace

int inv_wg_max_n(int real_bytes) {
  if (real_bytes == 8) return kLuMaxN<double>;
  int n = kLuMaxN<float>;
  while (gj_in_lds<float>(n + 1)) ++n;
  return n;
}

size_t inv_work_bytes(int n, int batch, int real_bytes) {
  size_t c = 2 * (size_t)real_bytes;
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  return al((size_t)n * kInvSuper * c * batch) + al((size_t)n * batch * sizeof(int)) * 2;
}

template <typename R>
InvWork<R> inv_work_carve(void *buf, int n, int batch) {
  typedef typename InvWork<R>::CT C;
  auto al = [](size_t x) { return (x + 255) & ~(size_t)255; };
  InvWork<R> w;
  char *p = (char *)buf;
  w.Rb = (C *)p; p += al((size_t)n * kInvSuper * sizeof(C) * batch);
  w.used = (int *)p; p += al((size_t)n * batch * sizeof(int));
  w.piv = (int *)p;
  w.n = n;
  w.batch = batch;
  return w;
}
template InvWork<double> inv_work_carve<double>(void *, int, int);
template InvWork<float> inv_work_carve<float>(void *, int, int);

void inv_z(int n, double2 *A, long long sA, double2 *Ainv, long long sAinv, int batch,
           const int *active, int *status, const InvWork<double> &w, hipStream_t s) {
  inv_impl<double>(n, A, sA, Ainv, sAinv, batch, active, status, w, s);
}
void inv_c(int n, float2 *A, long long sA, float2 *Ainv, long long sAinv, int batch,
           const int *active, int *status, const InvWork<float> &w, hipStream_t s) {
  inv_impl<float>(n, A, sA, Ainv, sAinv, batch, active, status, w, s);
}

}  // namespace hn
