// f2d_coarse.h -- the coarse multigrid levels of one instance on one
// workgroup, operator rows held in registers (device code and the host rule
// that says which hierarchies it takes).
//
// What bounds it: a chain of about 25 phases (a sweep, a residual, a transfer
// each), every one waiting for the one before it; bytes and flops are nothing.
// So each phase is made short.  Four wavefronts, one per SIMD, instead of
// sixteen: a barrier is cheap and a thread may hold 250 registers, in which
// the operator rows of every level stay for the whole launch (with 1024
// threads they came from LDS, 18 operands a cell and sweep).  A strip of four
// rows per thread takes 18 LDS values for four cells, its four serial sums
// advance together (the FP64 latency of one hides in the others), and a
// coarse cell's owner computes its restriction into a register.  The operands
// are packed per strip at set-up, so that the load is 33 coalesced 16-byte
// loads per thread which wait for no descriptor.  V-cycle tail from 32 x 32
// (32, 16, 8, 4): 21.5 -> 11.6 us; F-cycle tail 47.5 -> 26.2 us; of the first,
// operands 2.7, the 4 x 4 solve 2.4.  Whole steps: 128^2 859 -> 617 us,
// 1024^2 2080 -> 1680 us.  Strips of 8 rows on 64 x 32 cells need the
// accumulation registers too (2048 x 1024 Boussinesq 1247 -> 1261 us), so a
// top level over 1024 cells is taken only where the generic kernel's LDS
// budget would take it (FP32 operators: 48 x 24).
//
// Every level here lies below the finest, so its operator, mask, right-hand
// side and iterate are stored with periodic images in their halo: a value at
// a halo position equals the value at its image, and each level is a torus of
// its M x N interior cells.
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <stdint.h>
#include <string.h>

#include "f2d_dev.h"

namespace f2d {
namespace coarse {

// Level slots.  A level has a quarter of the cells of the level above it, so
// a hierarchy that ends at the coarsest level fills consecutive slots:
//   0  1025..4096 cells  strips of 8 rows per thread
//   1   257..1024        strips of 4 rows
//   2    65..256         one cell per thread
//   3    17..64, or the coarsest level of at most 64   wavefront 0, one cell per lane
//   4   the coarsest level under a slot-3 level        wavefront 0
constexpr int NSLOT = 5;
constexpr int PB = 64;  // LDS row pitch (values) of slots 0-2
constexpr int PW = 16;  // of slots 3-4
constexpr int MAXM = 64;

struct Slot {
  int M, N;  // interior rows, columns
  int lds;   // first LDS value of the level's x; t follows M rows later
  int pad;
};
struct Desc {
  Slot s[NSLOT];
  const void* b;  // top level's right-hand side
  double omega;
  int top, deep;  // first and last slot in use
};

// Strip rows and threads of a slot, and the packed operand record of a
// strip: its R cells' c1 / |A_5|, prolongation weights and masks (one word,
// bit r), then the operator rows -- what own_load reads, laid out so that each
// load takes two values per thread from consecutive addresses.
constexpr int slot_rows(int s) { return s == 0 ? 8 : (s == 1 ? 4 : 1); }
constexpr int slot_threads(int s) { return s <= 2 ? 256 : 64; }
constexpr int rec_values(int R) { return (10 * R + 2 + 1) / 2 * 2; }
// first value of slot s's records in an instance's block, and its length
constexpr size_t pack_first(int s) {
  size_t v = 0;
  for (int q = 0; q < s; q++) v += (size_t)rec_values(slot_rows(q)) * slot_threads(q);
  return v;
}
constexpr size_t PACK_VALUES = pack_first(NSLOT);

#define F2D_GLB __attribute__((address_space(1)))
#define F2D_LDS __attribute__((address_space(3)))

// element i of a global array, 32-bit byte offset from a uniform base
template <typename T>
__device__ __forceinline__ T gl32(const void* p, uint32_t i) {
  return *(F2D_GLB const T*)((F2D_GLB const char*)p + (size_t)(uint32_t)(i * (uint32_t)sizeof(T)));
}

// v where bit r of `bits` is set, else +0
__device__ __forceinline__ double keep(double v, int bits, int r) {
  const int m = __builtin_amdgcn_sbfe(bits, (unsigned)r, 1u);
  const long long u = __double_as_longlong(v);
  const int lo = (int)u & m, hi = (int)(u >> 32) & m;
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// One level as its owning threads see it: R consecutive rows of one column,
// the operator row of each cell (a1[R] is the south coupling of the row
// below the strip), c1 / |A_5|, right-hand side, iterate and
// prolongation weight; and the
// LDS offsets of the strip's neighbours on the torus.
template <int R>
struct Own {
  double a0[R], a1[R + 1], a2[R], a3[R], a4[R], a3e[R], a2s[R], a0s[R];
  double c3[R], b[R], x[R], w[R];
  int m;               // the cells' masks, bit r
  bool act;
  int j, i;            // first interior row, column
  int du, dd, dw, de;  // LDS offsets: row above, row below the strip; west, east
  F2D_LDS double *x0, *t0;  // the strip's first cell in the level's x and t
};

template <int R, int P>
__device__ __forceinline__ void own_place(Own<R>& o, const Slot& s, int tid, F2D_LDS double* lds) {
  const int M = s.M, N = s.N;
  // tid / N for tid < 512, N <= 64 (exact: the quotient is at least 0.5 / 64
  // from an integer, the float product within 1e-4 of it)
  const int g = (int)(((float)tid + 0.5f) * __builtin_amdgcn_rcpf((float)N));
  o.i = tid - g * N;
  o.j = g * R;
  o.act = o.j < M;
  if (!o.act) {
    o.j = 0;
    o.i = 0;
  }
  o.dw = o.i == 0 ? N - 1 : -1;
  o.de = o.i == N - 1 ? 1 - N : 1;
  o.du = o.j == 0 ? (M - 1) * P : -P;
  o.dd = o.j + R == M ? -o.j * P : R * P;
  o.x0 = lds + s.lds + o.j * P + o.i;
  o.t0 = o.x0 + M * P;
}

// the strip's record from the packed block
template <int R, int S>
__device__ __forceinline__ void own_load(Own<R>& o, const double* pk, int tid) {
  constexpr int NV = rec_values(R), NT = slot_threads(S);
  static_assert(R == slot_rows(S), "strip rows");
  typedef double v2 __attribute__((ext_vector_type(2)));
  double v[NV];
#pragma unroll
  for (int q = 0; q < NV / 2; q++) {
    const v2 w = gl32<v2>(pk + pack_first(S) + 2 * q * NT, (uint32_t)tid);
    v[2 * q] = w.x;
    v[2 * q + 1] = w.y;
  }
  int k = 0;
#pragma unroll
  for (int r = 0; r < R; r++) o.c3[r] = v[k++];
  o.m = (int)__double_as_longlong(v[k++]);
  double* const rows[8] = {o.a0, o.a1, o.a2, o.a3, o.a3e, o.a2s, o.a0s, o.a4};
#pragma unroll
  for (int q = 0; q < 8; q++)
#pragma unroll
    for (int r = 0; r < R; r++) rows[q][r] = v[k++];
  o.a1[R] = v[k++];
#pragma unroll
  for (int r = 0; r < R; r++) o.w[r] = v[k++];
}

// An instance's packed block, slot S's part (host): the level's operator
// planes A and mask (with halo), c1 the damped-Jacobi weight, mc the next
// coarser level's mask (null for the coarsest level).  Strips past the level
// stay zero.
template <int S>
inline void pack_slot(double* block, const double* A, const int8_t* mf, int M, int N,
                      const int8_t* mc, double c1) {
  constexpr int R = slot_rows(S), NT = slot_threads(S), NV = rec_values(R);
  const int n = N + 2 * NH, nc = N / 2 + 2 * NH;
  const size_t P = (size_t)(M + 2 * NH) * n;
  for (int t = 0; t < NT; t++) {
    const int j0 = t / N * R, i = t % N;
    if (j0 >= M) break;
    double v[NV] = {};
    int k = 0;
    const size_t c = (size_t)(j0 + NH) * n + i + NH;
    for (int r = 0; r < R; r++) v[k++] = c1 / fabs(A[4 * P + c + (size_t)r * n]);
    long long bits = 0;
    for (int r = 0; r < R; r++) bits |= (long long)(mf[c + (size_t)r * n] != 0) << r;
    memcpy(&v[k++], &bits, sizeof bits);
    const ptrdiff_t off[8] = {0,
                              (ptrdiff_t)P,
                              (ptrdiff_t)(2 * P),
                              (ptrdiff_t)(3 * P),
                              (ptrdiff_t)(3 * P + 1),
                              (ptrdiff_t)(2 * P + n - 1),
                              (ptrdiff_t)(n + 1),
                              (ptrdiff_t)(4 * P)};
    for (int q = 0; q < 8; q++)
      for (int r = 0; r < R; r++) v[k++] = A[c + (size_t)r * n + off[q]];
    v[k++] = A[P + c + (size_t)R * n];
    for (int r = 0; r < R; r++) {
      // prolongation weight (core/gmg/fortran_multigrid.f90:439, 454-492)
      const int j = j0 + r + NH, q = i + NH;
      double w = 0.;
      if (mc && mf[(size_t)j * n + q] > 0) {
        const int8_t* m = mc + (size_t)((j + 2) >> 1) * nc + ((q + 2) >> 1);
        const double c3[5] = {0., 1., 0.5, (double)0.3333333333333333333333333333f, 0.25};
        if (!(j & 1) && !(q & 1))
          w = 1.;
        else if (!(j & 1))
          w = c3[m[0] + m[1]];
        else if (!(q & 1))
          w = c3[m[0] + m[nc]];
        else
          w = c3[m[0] + m[1] + m[nc] + m[nc + 1]];
      }
      v[k++] = w;
    }
    for (int e = 0; e < NV; e++)
      block[pack_first(S) + ((size_t)(e / 2) * NT + t) * 2 + e % 2] = v[e];
  }
}

// the strip's 3 x (R + 2) torus neighbourhood of array p
template <int R, int P>
__device__ __forceinline__ void gather(const Own<R>& o, F2D_LDS const double* p,
                                       double (&v)[R + 2][3]) {
  auto row = [&](int k, int d) {
    v[k][0] = p[d + o.dw];
    v[k][1] = p[d];
    v[k][2] = p[d + o.de];
  };
  row(0, o.du);
#pragma unroll
  for (int r = 0; r < R; r++) row(r + 1, r * P);
  row(R + 1, o.dd);
}

// The rows' serial sums advance together, each stage's products issued one
// stage ahead of the sum that takes them: with one wavefront per SIMD nothing
// else hides the latency of a dependent FP64 operation, and the scheduler on
// its own runs one row's chain after the other.
#define F2D_STAGE() __builtin_amdgcn_sched_barrier(0)

// s[r] = ((t(r, 0) + t(r, 1)) + t(r, 2)) + ... + t(r, 7)
template <int R, typename F>
__device__ __forceinline__ void chain(F t, double (&s)[R]) {
  double p[R];
#pragma unroll
  for (int r = 0; r < R; r++) s[r] = t(r, 0);
#pragma unroll
  for (int r = 0; r < R; r++) p[r] = t(r, 1);
#pragma unroll
  for (int k = 2; k <= 8; k++) {
    F2D_STAGE();
#pragma unroll
    for (int r = 0; r < R; r++) {
      const double n = k < 8 ? t(r, k) : 0.;
      s[r] = s[r] + p[r];
      p[r] = n;
    }
  }
  F2D_STAGE();
}

// First damped-Jacobi sweep from x = 0: every product with x is a zero, so
// the value of jacobi_2d is 0 + c3 (0 - b), bit for bit (a zero sum's sign
// is lost in the final sum with +0).
template <int R, int P>
__device__ __forceinline__ void sweep_zero(Own<R>& o) {
  if (!o.act) return;
#pragma unroll
  for (int r = 0; r < R; r++) {
    const double v = 0. + o.c3[r] * (0. - o.b[r]);
    o.t0[r * P] = keep(v, o.m, r);
  }
}

// one damped-Jacobi sweep (jacobi_2d, operand for operand) from array p into
// q; the value stays in o.x
template <int R, int P>
__device__ __forceinline__ void sweep(Own<R>& o, F2D_LDS const double* p, F2D_LDS double* q,
                                      double c2) {
  if (!o.act) return;
  double v[R + 2][3];
  gather<R, P>(o, p, v);
  double q0[R];
  chain<R>(
      [&](int r, int k) {
        switch (k) {
          case 0: return o.a0[r] * v[r][0];
          case 1: return o.a1[r] * v[r][1];
          case 2: return o.a2[r] * v[r][2];
          case 3: return o.a3[r] * v[r + 1][0];
          case 4: return o.a3e[r] * v[r + 1][2];
          case 5: return o.a2s[r] * v[r + 2][0];
          case 6: return o.a1[r + 1] * v[r + 2][1];
          default: return o.a0s[r] * v[r + 2][2];
        }
      },
      q0);
  double w[R], u[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    q0[r] = q0[r] - o.b[r];
    u[r] = v[r + 1][1] * c2;
  }
  F2D_STAGE();
#pragma unroll
  for (int r = 0; r < R; r++) w[r] = o.c3[r] * q0[r];
  F2D_STAGE();
#pragma unroll
  for (int r = 0; r < R; r++) {
    o.x[r] = keep(u[r] + w[r], o.m, r);
    q[r * P] = o.x[r];
  }
}

// residual b - A x (residual_2d, operand for operand) into t
template <int R, int P>
__device__ __forceinline__ void residual(Own<R>& o) {
  if (!o.act) return;
  double v[R + 2][3];
  gather<R, P>(o, o.x0, v);
  double s[R], p[R];
#pragma unroll
  for (int r = 0; r < R; r++) {
    s[r] = o.b[r];
    p[r] = o.a0[r] * v[r][0];
  }
#pragma unroll
  for (int k = 1; k <= 9; k++) {
    F2D_STAGE();
#pragma unroll
    for (int r = 0; r < R; r++) {
      double n = 0.;
      if (k == 1) n = o.a1[r] * v[r][1];
      if (k == 2) n = o.a2[r] * v[r][2];
      if (k == 3) n = o.a3[r] * v[r + 1][0];
      if (k == 4) n = o.a4[r] * v[r + 1][1];
      if (k == 5) n = o.a3e[r] * v[r + 1][2];
      if (k == 6) n = o.a2s[r] * v[r + 2][0];
      if (k == 7) n = o.a1[r + 1] * v[r + 2][1];
      if (k == 8) n = o.a0s[r] * v[r + 2][2];
      s[r] = s[r] - p[r];
      p[r] = n;
    }
  }
#pragma unroll
  for (int r = 0; r < R; r++) {
    o.t0[r * P] = keep(s[r], o.m, r);
  }
}

// full weighting of the finer level's t (restrict_r): coarse cell (J, I)
// lies on fine (2 J + 1, 2 I + 1)
template <int R, int PF>
__device__ __forceinline__ void restrict_t(Own<R>& o, const Slot& f, F2D_LDS double* lds) {
  if (!o.act) return;
  const int M = f.M, N = f.N;
  F2D_LDS const double* t = lds + f.lds + M * PF;
  const int i0 = 2 * o.i, i1 = i0 + 1, i2 = i0 + 2 == N ? 0 : i0 + 2;
  const int last = 2 * (o.j + R) == M ? 0 : 2 * (o.j + R);  // fine row under the strip's end
  F2D_LDS const double* q = t + 2 * o.j * PF;
  double v[2 * R + 1][3];
#pragma unroll
  for (int k = 0; k < 2 * R; k++) {
    v[k][0] = q[k * PF + i0];
    v[k][1] = q[k * PF + i1];
    v[k][2] = q[k * PF + i2];
  }
  q = t + last * PF;
  v[2 * R][0] = q[i0];
  v[2 * R][1] = q[i1];
  v[2 * R][2] = q[i2];
#pragma unroll
  for (int r = 0; r < R; r++) {
    const double w = restrict_r<double>([&](int dj, int di) { return v[2 * r + 1 + dj][1 + di]; });
    o.b[r] = keep(w, o.m, r);
  }
}

// x + I(coarse x) (ACC) or I(coarse x) (interp_at) of the strip, stored to x
template <int R, int P, int PC>
__device__ __forceinline__ void prolong(Own<R>& o, const Slot& c, F2D_LDS double* lds, bool acc) {
  if (!o.act) return;
  const int M = c.M, N = c.N;
  F2D_LDS const double* xc = lds + c.lds;
  // coarse column (i - 1) >> 1 and the next, even i: between the two
  const bool pi = !(o.i & 1);
  const int I = ((o.i - 1) >> 1) < 0 ? N - 1 : (o.i - 1) >> 1;
  const int Ie = I + 1 == N ? 0 : I + 1;
  if constexpr (R == 1) {
    const bool pj = !(o.j & 1);
    const int J = ((o.j - 1) >> 1) < 0 ? M - 1 : (o.j - 1) >> 1;
    const int Jn = J + 1 == M ? 0 : J + 1;
    const double a = xc[J * PC + I], b = xc[J * PC + Ie], d = xc[Jn * PC + I],
                 e = xc[Jn * PC + Ie];
    double s = pi ? a + b : a;
    s = pj ? s + d : s;
    s = (pi && pj) ? s + e : s;
    const double r = keep(s * o.w[0], o.m, 0);
    o.x[0] = acc ? o.x[0] + r : r;
    o.x0[0] = o.x[0];
  } else {
    // strips start on even rows: coarse rows j / 2 - 1 .. j / 2 + R / 2 - 1
    double v[R / 2 + 1][2];
    const int J = o.j / 2, Jm = J == 0 ? M - 1 : J - 1;
    v[0][0] = xc[Jm * PC + I];
    v[0][1] = xc[Jm * PC + Ie];
#pragma unroll
    for (int k = 0; k < R / 2; k++) {
      v[k + 1][0] = xc[(J + k) * PC + I];
      v[k + 1][1] = xc[(J + k) * PC + Ie];
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      const int k = (r + 1) / 2;
      double s;
      if (r & 1) {  // odd row: on coarse row (j + r - 1) / 2
        s = pi ? v[k][0] + v[k][1] : v[k][0];
      } else {
        const double a = pi ? v[k][0] + v[k][1] : v[k][0];
        s = a + v[k + 1][0];
        s = pi ? s + v[k + 1][1] : s;
      }
      const double q = keep(s * o.w[r], o.m, r);
      o.x[r] = acc ? o.x[r] + q : q;
      o.x0[r * P] = o.x[r];
    }
  }
}

// a double from lane (lane moved by the DPP control CTRL) of the same row of
// 16 lanes: two 32-bit DPP moves
template <int CTRL>
__device__ __forceinline__ double dpp_move(double v) {
  const long long u = __double_as_longlong(v);
  const int lo = __builtin_amdgcn_mov_dpp((int)u, CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_mov_dpp((int)(u >> 32), CTRL, 0xF, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (long long)(unsigned)lo);
}

// wavefront-level ordering of LDS accesses (a wavefront's LDS operations
// execute in order)
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// The coarsest level: 16 smoothings from zero (hierarchy.py:117-118), result
// in o.x and in LDS.  A 4 x 4 level runs on the torus held by the first row
// of 16 lanes, lane 4 r + c: neighbours by DPP (row rotations by 4 and 12
// lanes for the rows, quad permutes for the columns); other shapes exchange
// through LDS.
__device__ __forceinline__ void coarsest(Own<1>& o, const Slot& s, double c2) {
  if (s.M == 4 && s.N == 4) {
    constexpr int DN = 0x124, DS = 0x12C, DW = 0x93, DE = 0x39;
    auto step = [&](double v) {
      const double n = dpp_move<DN>(v), d = dpp_move<DS>(v);
      // the moves and products run one stage ahead of the serial sum
      const double vw = dpp_move<DW>(v), nw = dpp_move<DW>(n);
      double q = o.a0[0] * nw, p = o.a1[0] * n;
      const double ne = dpp_move<DE>(n);
      F2D_STAGE();
      double r = o.a2[0] * ne;
      q = q + p;
      const double ve = dpp_move<DE>(v);
      F2D_STAGE();
      p = o.a3[0] * vw;
      q = q + r;
      const double dw = dpp_move<DW>(d);
      F2D_STAGE();
      r = o.a3e[0] * ve;
      q = q + p;
      const double de = dpp_move<DE>(d);
      F2D_STAGE();
      p = o.a2s[0] * dw;
      q = q + r;
      F2D_STAGE();
      r = o.a1[1] * d;
      q = q + p;
      F2D_STAGE();
      p = o.a0s[0] * de;
      q = q + r;
      F2D_STAGE();
      r = v * c2;
      q = q + p;
      const double w = r + o.c3[0] * (q - o.b[0]);
      return keep(w, o.m, 0);
    };
    double v = keep(0. + o.c3[0] * (0. - o.b[0]), o.m, 0);
    // 31 steps, five to a turn of the loop (a taken branch costs a refetch)
    v = step(v);
#pragma unroll 1
    for (int k = 0; k < 6; k++) v = step(step(step(step(step(v)))));
    o.x[0] = v;
    if (o.act) o.x0[0] = v;
  } else {
    sweep_zero<1, PW>(o);
    wave_sync();
    F2D_LDS double *p = o.t0, *q = o.x0;
#pragma unroll 1
    for (int k = 0; k < 31; k++) {
      sweep<1, PW>(o, p, q, c2);
      wave_sync();
      F2D_LDS double* h = p;
      p = q;
      q = h;
    }
  }
  wave_sync();
}

// MODE 0: the tail of a V-cycle from the top level entered with x = 0
// (hierarchy.py:98-126); 1: an F-cycle from the top level
// (hierarchy.py:131-151).  The top level's x goes to xg with its images.
// pk: the instance's packed block, of which slots first .. 4 are read before
// anything else is known.  `skip` is evaluated after the loads are issued; a
// skipped instance writes nothing.
template <typename T, bool S0, int MODE, typename SKIP, typename STAMP>
__device__ __forceinline__ void coarse_body(const Desc& D, const double* pk, int first, T* xg,
                                            F2D_LDS double* lds, SKIP skip, STAMP stamp) {
  const int tid = threadIdx.x;
  const bool w0 = tid < 64;
  constexpr int mode = MODE;
  Own<8> o0;
  Own<4> o1;
  Own<1> o2, o3, o4;
  // The order of the loads: the top level's operands, then its right-hand
  // side (its address waits for the descriptor), then the levels below,
  // which arrive while the top level is swept.
  const int top = D.top, deep = D.deep;
  const double c2 = 1. - D.omega;
  auto top_b = [&](auto& o, const Slot& s) {
    constexpr int R = sizeof(o.b) / sizeof(double);
    const uint32_t n = (uint32_t)s.N + 2 * NH;
    const uint32_t c = (uint32_t)(o.j + NH) * n + (uint32_t)(o.i + NH);
#pragma unroll
    for (int r = 0; r < R; r++) o.b[r] = (double)gl32<T>(D.b, c + (uint32_t)r * n);
  };
  if constexpr (S0) {
    own_load<8, 0>(o0, pk, tid);
    if (top <= 0) {
      own_place<8, PB>(o0, D.s[0], tid, lds);
      top_b(o0, D.s[0]);
    }
  }
  if (first <= 1) own_load<4, 1>(o1, pk, tid);
  if (top <= 1) {
    own_place<4, PB>(o1, D.s[1], tid, lds);
    if (top == 1) top_b(o1, D.s[1]);
  }
  if (first <= 2) own_load<1, 2>(o2, pk, tid);
  if (top <= 2) {
    own_place<1, PB>(o2, D.s[2], tid, lds);
    if (top == 2) top_b(o2, D.s[2]);
  }
  if (w0) {
    own_load<1, 3>(o3, pk, tid);
    own_load<1, 4>(o4, pk, tid);
    if (top <= 3) {
      own_place<1, PW>(o3, D.s[3], tid, lds);
      if (top == 3) top_b(o3, D.s[3]);
    }
    if (deep == 4) {
      own_place<1, PW>(o4, D.s[4], tid, lds);
      if (top == 4) top_b(o4, D.s[4]);
    }
  }
  if (skip()) return;
  stamp(1);
  // Two sweeps of a block level: from zero, or from x in LDS.
  auto pair = [&](auto& o, bool zero) {
    constexpr int R = sizeof(o.b) / sizeof(double);
    if (zero)
      sweep_zero<R, PB>(o);
    else
      sweep<R, PB>(o, o.x0, o.t0, c2);
    __syncthreads();
    sweep<R, PB>(o, o.t0, o.x0, c2);
    __syncthreads();
  };
  auto put_b = [&](auto& o, auto pitch) {  // b into t, to be restricted
    constexpr int R = sizeof(o.b) / sizeof(double), P = decltype(pitch)::value;
    if (o.act) {
#pragma unroll
      for (int r = 0; r < R; r++) o.t0[r * P] = o.b[r];
    }
  };
  using IB = std::integral_constant<int, PB>;
  using IW = std::integral_constant<int, PW>;
  int s = top;
  if (mode == 1) {  // b restricted down, then the coarsest solve
    if (S0 && top <= 0) {
      put_b(o0, IB());
      __syncthreads();
      restrict_t<4, PB>(o1, D.s[0], lds);
    }
    if (top <= 1) {
      put_b(o1, IB());
      __syncthreads();
      restrict_t<1, PB>(o2, D.s[1], lds);
    }
    if (top <= 2) {
      put_b(o2, IB());
      __syncthreads();
      if (w0) restrict_t<1, PB>(o3, D.s[2], lds);
    }
    if (w0 && deep == 4 && top <= 3) {
      put_b(o3, IW());
      wave_sync();
      restrict_t<1, PW>(o4, D.s[3], lds);
    }
    stamp(40);
    if (w0) {
      if (deep == 4)
        coarsest(o4, D.s[4], c2);
      else
        coarsest(o3, D.s[3], c2);
    }
    __syncthreads();
    stamp(20);
    s = deep - 1;
  }
  // V-cycles: one from the top level (mode 0), or one from each level
  // upward, entered from the prolongation (mode 1)
  constexpr bool zero = mode == 0;
#pragma unroll 1
  for (;; s--) {
    if (mode == 1) {
      if (s < top) break;
      if (S0 && s == 0) prolong<8, PB, PB>(o0, D.s[1], lds, false);
      if (s == 1) prolong<4, PB, PB>(o1, D.s[2], lds, false);
      if (s == 2) prolong<1, PB, PW>(o2, D.s[3], lds, false);
      if (s == 3 && w0) {
        prolong<1, PW, PW>(o3, D.s[4], lds, false);
        wave_sync();
      }
      if (s < 3) __syncthreads();
      stamp(50 + s);
    }
    if (S0 && s <= 0) {
      pair(o0, zero || s < 0);
      residual<8, PB>(o0);
      __syncthreads();
      restrict_t<4, PB>(o1, D.s[0], lds);
      stamp(10);
    }
    if (s <= 1) {
      pair(o1, zero || s < 1);
      residual<4, PB>(o1);
      __syncthreads();
      restrict_t<1, PB>(o2, D.s[1], lds);
      stamp(11);
    }
    if (s <= 2) {
      pair(o2, zero || s < 2);
      residual<1, PB>(o2);
      __syncthreads();
      stamp(12);
    }
    if (w0) {
      if (s <= 2) restrict_t<1, PB>(o3, D.s[2], lds);
      if (deep == 4) {
        if (s <= 3) {
          if (zero || s < 3)
            sweep_zero<1, PW>(o3);
          else
            sweep<1, PW>(o3, o3.x0, o3.t0, c2);
          wave_sync();
          sweep<1, PW>(o3, o3.t0, o3.x0, c2);
          wave_sync();
          residual<1, PW>(o3);
          wave_sync();
          restrict_t<1, PW>(o4, D.s[3], lds);
        }
        stamp(13);
        coarsest(o4, D.s[4], c2);
        stamp(20);
        if (s <= 3) {
          prolong<1, PW, PW>(o3, D.s[4], lds, true);
          wave_sync();
          sweep<1, PW>(o3, o3.x0, o3.t0, c2);
          wave_sync();
          sweep<1, PW>(o3, o3.t0, o3.x0, c2);
          wave_sync();
        }
        stamp(33);
      } else {
        coarsest(o3, D.s[3], c2);
        stamp(20);
      }
    }
    if (s <= 2) {
      __syncthreads();
      prolong<1, PB, PW>(o2, D.s[3], lds, true);
      __syncthreads();
      pair(o2, false);
      stamp(32);
    }
    if (s <= 1) {
      prolong<4, PB, PB>(o1, D.s[2], lds, true);
      __syncthreads();
      pair(o1, false);
      stamp(31);
    }
    if (S0 && s <= 0) {
      prolong<8, PB, PB>(o0, D.s[1], lds, true);
      __syncthreads();
      pair(o0, false);
      stamp(30);
    }
    if (mode == 0) break;
    if (s == 3) __syncthreads();  // the next level up reads what wavefront 0 wrote
  }
  // the top level's x with its periodic images
  auto put_x = [&](auto& o, const Slot& q) {
    constexpr int R = sizeof(o.b) / sizeof(double);
    const int M = q.M, N = q.N;
    const uint32_t n = (uint32_t)N + 2 * NH;
    if (!o.act) return;
    F2D_GLB T* xq = (F2D_GLB T*)xg;
    auto put = [&](int j, int i, T v) {
      *(F2D_GLB T*)((F2D_GLB char*)xq + (size_t)(uint32_t)(((uint32_t)j * n + (uint32_t)i) *
                                                           (uint32_t)sizeof(T))) = v;
    };
    // rows and columns within 3 of an edge have one image beyond the other
    // edge, or (interiors narrower than 6) one beyond each
    const bool thin = M < 2 * NH || N < 2 * NH;
    const int I = NH + o.i, Ii = o.i < NH ? I + N : I - N;
    const bool ci = o.i < NH || o.i >= N - NH;
    if (thin) {
#pragma unroll 1
      for (int dj = -M; dj <= M; dj += M)
#pragma unroll 1
        for (int di = -N; di <= N; di += N)
#pragma unroll
          for (int r = 0; r < R; r++) {
            const int j = NH + o.j + r + dj, i = I + di;
            if (j >= 0 && j < M + 2 * NH && i >= 0 && i < N + 2 * NH) put(j, i, T(o.x[r]));
          }
      return;
    }
#pragma unroll
    for (int r = 0; r < R; r++) {
      const T v = T(o.x[r]);
      const int J = NH + o.j + r;
      const int Ji = o.j + r < NH ? J + M : J - M;
      const bool cj = o.j + r < NH || o.j + r >= M - NH;
      put(J, I, v);
      if (ci) put(J, Ii, v);
      if (cj) put(Ji, I, v);
      if (ci && cj) put(Ji, Ii, v);
    }
  };
  if (S0 && top == 0) put_x(o0, D.s[0]);
  if (top == 1) put_x(o1, D.s[1]);
  if (top == 2) put_x(o2, D.s[2]);
  if (w0) {
    if (top == 3) put_x(o3, D.s[3]);
    if (top == 4) put_x(o4, D.s[4]);
  }
  stamp(2);
}

// The slots of the levels k0 .. nlev - 1 with interiors M[l] x N[l]: false
// when they do not fit them (the generic coarse kernel takes those).
// most_top: the most cells of the top level.
inline bool slots(int k0, int nlev, const int* M, const int* N, int most_top, int* slot_of_top,
                  int* deep) {
  const int nl = nlev - k0;
  if (nl < 1 || nl > NSLOT) return false;
  // the coarsest level's slot: 4 when the level above it (in this kernel or
  // not) also fits a wavefront, else 3
  const int d = nlev - 1;
  if (M[d] * N[d] > 64 || N[d] > PW) return false;
  const bool two = d >= 1 && M[d - 1] * N[d - 1] <= 64 && N[d - 1] <= PW;
  *deep = two ? 4 : 3;
  *slot_of_top = *deep - (nl - 1);
  if (*slot_of_top < 0) return false;
  const int lim[NSLOT] = {most_top, 1024, 256, 64, 64}, rows[NSLOT] = {8, 4, 1, 1, 1};
  for (int l = k0; l < nlev; l++) {
    const int s = *deep - (nlev - 1 - l);
    if (M[l] * N[l] > lim[s] || M[l] > MAXM || M[l] % rows[s]) return false;
    if (N[l] > (s >= 3 ? PW : PB)) return false;
    // the prolongation and restriction assume exact halving
    if (l + 1 < nlev && (M[l] != 2 * M[l + 1] || N[l] != 2 * N[l + 1])) return false;
  }
  return true;
}
// LDS values of the levels in slots top .. deep
inline int lds_values(const Desc& D) {
  int v = 0;
  for (int s = D.top; s <= D.deep; s++) v += 2 * D.s[s].M * (s >= 3 ? PW : PB);
  return v;
}

}  // namespace coarse
}  // namespace f2d
