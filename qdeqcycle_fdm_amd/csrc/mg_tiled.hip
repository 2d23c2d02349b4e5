// mg_tiled.hip -- the fast V-cycle: temporally blocked LDS tile kernels.
//
// One V-cycle of the fast cycle costs two launches per level above the coarse
// tail plus one launch for the whole tail:
//   k_down  (level l): n_pre red/black sweeps, residual, full-weighting
//           restriction to level l+1, all on one LDS tile with a halo of
//           2 n_pre + 2 points, so the ring of redundant updates makes every
//           interior value exactly what global sweeps would produce;
//   k_tail  (levels with N <= TAIL_MAX_N): one workgroup runs the rest of the
//           V-cycle in LDS with workgroup barriers only (k_tail_direct: the
//           production tail of one level and the direct coarsest solve;
//           k_coarse_rows: a tail of that solve alone, over workgroups);
//   k_up    (level l): bilinear prolongation + correction (folded into the
//           tile load), n_post sweeps, and on level 0 either the
//           residual-norm partials (FP64 solve) or the FP64 update u += e
//           (FP32 correction of iterative refinement).
// The tiles live in registers as 2x2 quads of points, their values shared
// through the LDS.
// Every update, residual, restriction and prolongation is evaluated with the
// same expressions as the one-launch-per-half-sweep kernels of mg.hip, so the
// tiled cycle reproduces them bit for bit.  The input and output u of a tile
// kernel are different buffers (tiles read their neighbours' interiors as
// halo).
#include <cmath>

#include <algorithm>
#include <type_traits>
#include <utility>
#include <vector>

#include "qdeq_internal.h"

namespace qdeq {

constexpr int TX_THREADS = 64;   // one wavefront across a tile row
constexpr int TY_THREADS = 16;   // 16 rows of lanes: 1024 threads per tile
constexpr int TILE_THREADS = TX_THREADS * TY_THREADS;
constexpr int TAIL_THREADS = 1024;
constexpr int TAIL_MAX_N = 33;  // levels with N, K <= this run in the tail
// threads of the tail of one level and the direct solve, whose coarsest level
// has at most 17 x 15 unknowns
constexpr int DIRECT_THREADS = 512;
// one quad of a tail level per thread
static_assert(((TAIL_MAX_N + 1) / 2) * ((TAIL_MAX_N + 1) / 2) <= DIRECT_THREADS, "tail quads");
static_assert(DIRECT_THREADS <= TAIL_THREADS, "tail quads");

// Update of one point with its quantity a = relax / (m1 + m2 + m3 + m4)
// (EXACT, the reference's form) or m1 + m2 + m3 + m4 (plain) formed once: the
// operations of k_rbgs in the same order, so the same bits.
template <typename T, bool EXACT>
__device__ inline T rbgs_update_pre(T a, T m1, T m2, T m3, T m4, T uW, T uE, T uS,
                                    T uN, T uC, T fDH2, bool has_f, T relax) {
  T num = m1 * uW + m2 * uE + m3 * uS + m4 * uN;
  if (has_f) num = num - fDH2;
  if (EXACT) return a * num + (T(1) - relax) * uC;
  const T unew = num / a;
  return (relax == T(1)) ? unew : uC + relax * (unew - uC);
}

template <typename T, bool EXACT>
__device__ inline T rbgs_factor(T m1, T m2, T m3, T m4, T relax) {
  return EXACT ? relax / (m1 + m2 + m3 + m4) : m1 + m2 + m3 + m4;
}

// Tile handled by this workgroup.  Workgroups are dispatched to the 8 XCDs
// in turn (linear id mod 8), and each XCD has its own L2; the tiles are
// dealt out in 8 contiguous bands of row-major tile order, one per XCD, so
// neighbouring tiles (their halos overlap) and the tiles of consecutive
// levels over the same part of the grid run on the same XCD.  XCD x holds
// q + (x < r) workgroups for n = 8 q + r tiles.
__device__ inline int tile_id() {
  const int n = gridDim.x * gridDim.y;
  const int id = blockIdx.y * gridDim.x + blockIdx.x;
  const int x = id & 7, slot = id >> 3;
  const int q = n >> 3, r = n & 7;
  return x * q + min(x, r) + slot;
}

// Tiles as 2x2 quads held in registers.
//
// A tile is R x C points (both even) starting at the even global row j0 and
// even column k0, so that quad (a, b) = local rows 2a, 2a+1 and columns 2b,
// 2b+1 has colour 0 on its diagonal and colour 1 on the anti-diagonal, its
// point (0, 0) is the coarse point under it, and its two points of a row are
// one aligned 16-byte load (8-byte in FP32).  Quad id = a (C/2) + b belongs
// to thread id mod nthr; a thread keeps S quads: values, coefficients,
// relaxation factor and right-hand side stay in registers from the tile load
// to the store, and only the values are shared through the LDS, in four
// planes (one per position in the quad), so that every neighbour of quad id
// sits at id, id +- 1 or id +- C/2 of a plane: consecutive lanes read
// consecutive words (no bank conflicts) and a point update costs two LDS
// reads and one write.
//
// Against tiles of points in three or four LDS arrays (8-byte loads with
// per-point address arithmetic, the relaxation factor's division in every
// half-sweep), launched back to back with tuned shapes, FP64 down / up in us:
// level 0 of 1025^2 16.1 / 22.5 -> 10.2 / 13.4, level 1 7.4 / 9.4 -> 4.5 /
// 5.5, level 2 5.5 / 6.4 -> 3.6 / 3.9; level 0 of 2049^2 53 / 96 -> 32 / 44
// (FP32 42 / 55 -> 22 / 33).  What bounds them now: the tile's loads (41 MB
// with the halos at level 0 of 1025^2, all workgroups at once), and below
// level 1 the launch and one round trip of loads (3.3 us whatever the size).
//
// The sweeps update every point of the tile that the grid's sweeps update,
// without shrinking the window: the neighbours of the outermost ring are
// wrong (they read a guard cell or another row), so each half-sweep spoils
// one more ring from the edge, and a halo of as many rings as half-sweeps
// keeps the interior exact.
template <typename T>
struct Vec2 {
  typedef T type __attribute__((ext_vector_type(2)));
};

// PS: words from one plane to the next, or 0 where it follows the tile's size.
// With a constant distance a quad's LDS addresses are three registers (own,
// south and north quad) and immediate offsets; otherwise each plane has its
// own, which two FP64 quads per thread cannot afford.
template <typename T, int PS>
struct QTile {
  T *p;        // plane 0
  int stride;  // words between planes (PS == 0)
  int C2, nq;  // quads per row, quads
  int j0, k0;  // global row and column of the tile's first point
  // the planes of the points (0,0), (0,1), (1,0) and (1,1), indexed by quad
  __device__ T *plane(int n) const { return p + n * (PS ? PS : stride); }
  __device__ T *p00() const { return plane(0); }
  __device__ T *p01() const { return plane(1); }
  __device__ T *p10() const { return plane(2); }
  __device__ T *p11() const { return plane(3); }
};

template <typename T>
struct Quad {
  T u00, u01, u10, u11;
  T x0, x1, x2, y0, y1, y2;      // west faces: row j columns k..k+2, row j+1
  T z0, z1, w0, w1, v0, v1;      // south faces of rows j, j+1, j+2
  T a00, a01, a10, a11;          // relax / (m1+m2+m3+m4), or the sum (plain)
  T f00, f01, f10, f11;          // f, or DH^2 f (up kernels)
  int id;                        // index in the planes
  bool valid;                    // a quad of the tile
  bool first, top, topn;         // row j is the grid's first, last; row j+1 the last
  bool k00, k01, k10, k11;       // points that the sweeps update
};

// Quads a thread may hold: what the 128 registers of a thread in a 1024-thread
// workgroup take (about 45 per FP64 quad, 24 per FP32 one).
template <typename T>
constexpr int kMaxQuads = sizeof(T) == 8 ? 2 : 3;

// Keeps the scheduler from running the quads of a thread side by side where
// their registers fill the file (two FP64 quads, three FP32 ones).
template <typename T, int S>
__device__ inline void one_quad_at_a_time() {
  if (S == kMaxQuads<T>) __builtin_amdgcn_sched_barrier(0);
}

// Guard words before, between and after the planes: reads at id +- C/2 and
// id +- 1 of the outermost quads stay inside the LDS (their values go into
// spoiled rings only).
__host__ __device__ inline int quad_guard(int C2) { return C2 + 1; }
__host__ __device__ inline size_t quad_lds_words(int R, int C, int ps) {
  const int C2 = C / 2, nq = (R / 2) * C2, G = quad_guard(C2);
  return 3 * (size_t)(ps ? ps : nq + G) + nq + 2 * (size_t)G;
}
// Plane distance of a kernel with S quads per thread: constant for the most
// quads, at least those of 1024 threads and a guard (C/2 is at most 161; an
// LDS instruction's offset reaches 64 KB, three planes).
template <typename T, int S>
constexpr int kPlaneWords = S < kMaxQuads<T> ? 0 : kMaxQuads<T> * 1024 + 168;

template <typename T, int PS>
__device__ inline QTile<T, PS> make_qtile(unsigned char *smem, int TX, int TY, int H) {
  QTile<T, PS> t;
  const int R = TY + 2 * H, C = TX + 2 * H;
  t.C2 = C >> 1;
  t.nq = (R >> 1) * t.C2;
  const int tile = tile_id();
  t.j0 = (tile / (int)gridDim.x) * TY - H;
  t.k0 = (tile % (int)gridDim.x) * TX - H;
  const int G = quad_guard(t.C2);
  t.p = reinterpret_cast<T *>(smem) + G;
  t.stride = t.nq + G;
  return t;
}

// The quad's place in the tile and the grid.
template <typename T, int PS>
__device__ inline void quad_place(const QTile<T, PS> &t, Quad<T> &q, int id, int N, int K) {
  q.valid = id < t.nq;
  q.id = q.valid ? id : t.nq - 1;
  const int a = q.id / t.C2;
  const int j = t.j0 + 2 * a, k = t.k0 + 2 * (q.id - a * t.C2);
  // rows 0 and N-1 reflect: the row across the boundary is the one on the
  // other side.  Row 0 is a quad's first row (j0 is even); the last row is
  // either.
  q.first = j == 0;
  q.top = j == N - 1;
  q.topn = j + 1 == N - 1;
  const bool j0in = q.valid && j >= 0 && j < N, j1in = q.valid && j >= -1 && j + 1 < N;
  const bool k0in = k >= 1 && k <= K - 2, k1in = k >= 0 && k + 1 <= K - 2;
  q.k00 = j0in && k0in;
  q.k01 = j0in && k1in;
  q.k10 = j1in && k0in;
  q.k11 = j1in && k1in;
}

// Quad whose planes hold the row south of row j, and north of row j+1 (the
// quad itself at a reflecting boundary).
template <typename T, int PS>
__device__ inline int quad_south(const QTile<T, PS> &t, const Quad<T> &q) {
  return q.first ? q.id : q.id - t.C2;
}
template <typename T, int PS>
__device__ inline int quad_north(const QTile<T, PS> &t, const Quad<T> &q) {
  return q.topn ? q.id : q.id + t.C2;
}

// Local row and column of the quad's point (0, 0) (formed again where they
// are needed rather than kept in registers through the sweeps).
template <typename T, int PS>
__device__ inline void quad_rc(const QTile<T, PS> &t, int id, int &r, int &c) {
  const int a = id / t.C2;
  r = 2 * a;
  c = 2 * (id - a * t.C2);
}

// Element at a 32-bit byte offset from a uniform base (one address register
// per load, shared by the arrays of a level).
template <typename V, typename T>
__device__ inline V load_at(const T *base, unsigned bytes) {
  return *reinterpret_cast<const V *>(reinterpret_cast<const char *>(base) + bytes);
}

// Global loads of a quad, at clamped in-range addresses (what lies outside
// the grid is never used by a point that is updated, normed or stored).
// zero_u: the values are zero (first visit of a coarse level).
template <typename T, bool HAS_F, int PS>
__device__ inline void quad_load(const QTile<T, PS> &t, Quad<T> &q, const T *__restrict__ u,
                                 const T *__restrict__ f, const T *__restrict__ cx,
                                 const T *__restrict__ cz, int N, int K, int P,
                                 bool zero_u) {
  typedef typename Vec2<T>::type V2;
  constexpr unsigned E = sizeof(T);
  int j, k;
  quad_rc(t, q.id, j, k);
  j += t.j0;
  k += t.k0;
  // offsets from the tile's first row inside the grid
  const int jt = max(t.j0, 0);
  const size_t base = (size_t)jt * P;
  const int ja = min(max(j, 0), N - 1) - jt, jb = min(max(j + 1, 0), N - 1) - jt;
  // an even column whose pair lies in the row (the pitch is a multiple of 64)
  const int kc = min(max(k, 0), (K - 1) & ~1), kx = min(kc + 2, K - 1);
  const unsigned oa = (unsigned)(ja * P + kc) * E, ob = (unsigned)(jb * P + kc) * E;
  V2 ua = {T(0), T(0)}, ub = {T(0), T(0)};
  if (!zero_u) {
    ua = load_at<V2>(u + base, oa);
    ub = load_at<V2>(u + base, ob);
  }
  const V2 xa = load_at<V2>(cx + base, oa), xb = load_at<V2>(cx + base, ob);
  q.x2 = load_at<T>(cx + base, (unsigned)(ja * P + kx) * E);
  q.y2 = load_at<T>(cx + base, (unsigned)(jb * P + kx) * E);
  const int jz = min(max(j, 0), N) - jt, jw = min(max(j + 1, 0), N) - jt,
            jv = min(max(j + 2, 0), N) - jt;
  const V2 za = load_at<V2>(cz + base, (unsigned)(jz * P + kc) * E);
  const V2 zb = load_at<V2>(cz + base, (unsigned)(jw * P + kc) * E);
  const V2 zc = load_at<V2>(cz + base, (unsigned)(jv * P + kc) * E);
  V2 fa = {T(0), T(0)}, fb = {T(0), T(0)};
  if (HAS_F) {
    fa = load_at<V2>(f + base, oa);
    fb = load_at<V2>(f + base, ob);
  }
  q.u00 = ua.x; q.u01 = ua.y; q.u10 = ub.x; q.u11 = ub.y;
  q.x0 = xa.x; q.x1 = xa.y; q.y0 = xb.x; q.y1 = xb.y;
  q.z0 = za.x; q.z1 = za.y; q.w0 = zb.x; q.w1 = zb.y; q.v0 = zc.x; q.v1 = zc.y;
  q.f00 = fa.x; q.f01 = fa.y; q.f10 = fb.x; q.f11 = fb.y;
}

// u + P e on a quad (prolongate_kernel, odeSolver.cpp:1017-1043): point
// (0, 0) sits on coarse point (cj, ck).  The same single addition per point
// as a separate pass over u makes; the reference leaves the last row alone
// (FULL_TOP = false), the fast cycle corrects it.
template <typename T, bool FULL_TOP, int PS>
__device__ inline void quad_prolong(const QTile<T, PS> &t, Quad<T> &q, const T *__restrict__ e,
                                    int Nc, int Kc, int Pc, int N, int K) {
  int j, k;
  quad_rc(t, q.id, j, k);
  j += t.j0;
  k += t.k0;
  const int cj = j >> 1, ck = k >> 1;
  const int ct = min(max(t.j0, 0) >> 1, Nc - 1);
  const T *eb = e + (size_t)ct * Pc;
  const int ca = min(max(cj, 0), Nc - 1) - ct, cb = min(max(cj + 1, 0), Nc - 1) - ct;
  const int ka = min(max(ck, 0), Kc - 1), kb = min(max(ck + 1, 0), Kc - 1);
  constexpr unsigned E = sizeof(T);
  const T e00 = load_at<T>(eb, (unsigned)(ca * Pc + ka) * E);
  const T e01 = load_at<T>(eb, (unsigned)(ca * Pc + kb) * E);
  const T e10 = load_at<T>(eb, (unsigned)(cb * Pc + ka) * E);
  const T e11 = load_at<T>(eb, (unsigned)(cb * Pc + kb) * E);
  const bool in = q.valid && j >= 0 && k >= 0 && k < K && ck < Kc - 1;
  const bool p0 = in && j < N && (FULL_TOP ? cj <= Nc - 1 : cj < Nc - 1);
  const bool p1 = in && j + 1 < N && cj < Nc - 1;
  const bool kin = k + 1 < K;
  if (p0) {
    q.u00 += e00;
    if (kin) q.u01 += T(0.5) * (e00 + e01);
  }
  if (p1) {
    q.u10 += T(0.5) * (e00 + e10);
    if (kin) q.u11 += T(0.25) * (e00 + e01 + e10 + e11);
  }
}

template <typename T, bool EXACT>
__device__ inline void quad_factors(Quad<T> &q, T relax) {
  q.a00 = rbgs_factor<T, EXACT>(q.x0, q.x1, q.z0, q.w0, relax);
  q.a01 = rbgs_factor<T, EXACT>(q.x1, q.x2, q.z1, q.w1, relax);
  q.a10 = rbgs_factor<T, EXACT>(q.y0, q.y1, q.w0, q.v0, relax);
  q.a11 = rbgs_factor<T, EXACT>(q.y1, q.y2, q.w1, q.v1, relax);
}

template <typename T, int PS>
__device__ inline void quad_put(const QTile<T, PS> &t, const Quad<T> &q) {
  if (q.valid) {
    t.p00()[q.id] = q.u00;
    t.p01()[q.id] = q.u01;
    t.p10()[q.id] = q.u10;
    t.p11()[q.id] = q.u11;
  }
}

// One half-sweep on the quads of a thread; SCALED: the quads hold DH^2 f.
template <typename T, bool HAS_F, bool EXACT, bool SCALED, int COL, int S, int PS>
__device__ inline void quads_half_sweep(const QTile<T, PS> &t, Quad<T> (&q)[S], T DH2,
                                        T relax) {
#pragma unroll
  for (int i = 0; i < S; i++) {
    Quad<T> &p = q[i];
    one_quad_at_a_time<T, S>();
    const int so = quad_south(t, p), no = quad_north(t, p);
    if (COL == 0) {
      const T W = t.p01()[p.id - 1], So = t.p10()[so];
      const T E = t.p10()[p.id + 1], No = t.p01()[no];
      const T n0 = rbgs_update_pre<T, EXACT>(
          p.a00, p.x0, p.x1, p.z0, p.w0, W, p.u01, So, p.top ? So : p.u10, p.u00,
          HAS_F ? (SCALED ? p.f00 : DH2 * p.f00) : T(0), HAS_F, relax);
      const T n1 = rbgs_update_pre<T, EXACT>(
          p.a11, p.y1, p.y2, p.w1, p.v1, p.u10, E, p.u01, No, p.u11,
          HAS_F ? (SCALED ? p.f11 : DH2 * p.f11) : T(0), HAS_F, relax);
      if (p.k00) t.p00()[p.id] = p.u00 = n0;
      if (p.k11) t.p11()[p.id] = p.u11 = n1;
    } else {
      const T E = t.p00()[p.id + 1], So = t.p11()[so];
      const T W = t.p11()[p.id - 1], No = t.p00()[no];
      const T n0 = rbgs_update_pre<T, EXACT>(
          p.a01, p.x1, p.x2, p.z1, p.w1, p.u00, E, So, p.top ? So : p.u11, p.u01,
          HAS_F ? (SCALED ? p.f01 : DH2 * p.f01) : T(0), HAS_F, relax);
      const T n1 = rbgs_update_pre<T, EXACT>(
          p.a10, p.y0, p.y1, p.w0, p.v0, W, p.u11, p.u00, No, p.u10,
          HAS_F ? (SCALED ? p.f10 : DH2 * p.f10) : T(0), HAS_F, relax);
      if (p.k01) t.p01()[p.id] = p.u01 = n0;
      if (p.k10) t.p10()[p.id] = p.u10 = n1;
    }
  }
}

// nu red/black sweeps; the planes are current (and every thread past a
// barrier) before and after.
template <typename T, bool HAS_F, bool EXACT, bool SCALED, int S, int PS>
__device__ inline void quads_sweep(const QTile<T, PS> &t, Quad<T> (&q)[S], int nu, T DH2,
                                   T relax) {
  for (int s = 0; s < nu; s++) {
    quads_half_sweep<T, HAS_F, EXACT, SCALED, 0, S>(t, q, DH2, relax);
    __syncthreads();
    quads_half_sweep<T, HAS_F, EXACT, SCALED, 1, S>(t, q, DH2, relax);
    __syncthreads();
  }
}

// Residual of one point, the expression of k_residual.
template <typename T>
__device__ inline T point_residual(T fv, T m1, T m2, T m3, T m4, T uW, T uE, T uS, T uN,
                                   T uC, T DH2) {
  return fv - (m1 * uW + m2 * uE + m3 * uS + m4 * uN - (m1 + m2 + m3 + m4) * uC) / DH2;
}

// Residuals of a quad (zero where the grid has none), and the fault and
// remote neighbours' values for the boundary-data residual.
template <typename T, bool HAS_F, int PS>
__device__ inline void quad_residual(const QTile<T, PS> &t, const Quad<T> &p, T DH2, T &r00,
                                     T &r01, T &r10, T &r11) {
  const T W0 = t.p01()[p.id - 1], S0 = t.p10()[quad_south(t, p)];
  const T E0 = t.p00()[p.id + 1], S1 = t.p11()[quad_south(t, p)];
  const T W1 = t.p11()[p.id - 1], N0 = t.p00()[quad_north(t, p)];
  const T E1 = t.p10()[p.id + 1], N1 = t.p01()[quad_north(t, p)];
  const T a = point_residual<T>(HAS_F ? p.f00 : T(0), p.x0, p.x1, p.z0, p.w0, W0, p.u01,
                                S0, p.top ? S0 : p.u10, p.u00, DH2);
  const T b = point_residual<T>(HAS_F ? p.f01 : T(0), p.x1, p.x2, p.z1, p.w1, p.u00, E0,
                                S1, p.top ? S1 : p.u11, p.u01, DH2);
  const T c = point_residual<T>(HAS_F ? p.f10 : T(0), p.y0, p.y1, p.w0, p.v0, W1, p.u11,
                                p.u00, N0, p.u10, DH2);
  const T d = point_residual<T>(HAS_F ? p.f11 : T(0), p.y1, p.y2, p.w1, p.v1, p.u10, E1,
                                p.u01, N1, p.u11, DH2);
  r00 = p.k00 ? a : T(0);
  r01 = p.k01 ? b : T(0);
  r10 = p.k10 ? c : T(0);
  r11 = p.k11 ? d : T(0);
}

// Full weighting onto the coarse point under a quad's (0, 0) (the expression
// of k_restrict): the quad's own residuals and those of its west, south and
// south-west quads in the planes of r.  The first and last coarse rows use
// their one fine neighbour row twice.
template <typename T, int PS>
__device__ inline T quad_restrict(const QTile<T, PS> &r, int id, T r00, T r01, T r10, T r11,
                                  bool first, bool last) {
  const int s = id - r.C2;
  const T nm = r.p11()[id - 1];
  const T s0 = r.p10()[s], sm = r.p11()[s - 1], sp = r.p11()[s];
  const T rs0 = first ? r10 : s0, rsm = first ? nm : sm, rsp = first ? r11 : sp;
  const T rn0 = last ? s0 : r10, rnm = last ? sm : nm, rnp = last ? sp : r11;
  return T(0.0625) * (T(4.0) * r00 + T(2.0) * r.p01()[id - 1] + T(2.0) * r01 +
                      T(2.0) * rs0 + T(2.0) * rn0 + rsm + rsp + rnm + rnp);
}

// Whether the quad lies in the tile's interior (H and the tile are even),
// and the global row and column of its point (0, 0).
template <typename T, int PS>
__device__ inline bool quad_interior(const QTile<T, PS> &t, const Quad<T> &q, int H, int TX,
                                     int TY, int &j, int &k) {
  int r, c;
  quad_rc(t, q.id, r, c);
  j = t.j0 + r;
  k = t.k0 + c;
  return q.valid && r >= H && r < H + TY && c >= H && c < H + TX;
}

// The interior quad's values into the grid array, 16 bytes a row.
template <typename T>
__device__ inline void quad_store(const Quad<T> &q, int j, int k, T *__restrict__ u, int N,
                                  int K, int P) {
  typedef typename Vec2<T>::type V2;
  if (j >= N || k >= K) return;
  T *g = u + (size_t)j * P + k;
  const bool pair = k + 1 < K;
  if (pair)
    *reinterpret_cast<V2 *>(g) = V2{q.u00, q.u01};
  else
    g[0] = q.u00;
  if (j + 1 < N) {
    if (pair)
      *reinterpret_cast<V2 *>(g + P) = V2{q.u10, q.u11};
    else
      g[P] = q.u10;
  }
}

// Start of a plain FP64 solve folded into its first V-cycle (no separate
// start kernels): the level-0 down kernel (START_PARTIALS) forms, per tile
// and before smoothing, the residual-norm partials of the start and of the
// boundary data (the residual with the interior at zero), the expressions of
// k_start_partials; the level-1 down kernel (START_TEST) sums them in a
// fixed order (every workgroup the same bits), applies the start test of
// k_start_gate, returns at once if the start already meets the threshold,
// and its workgroup (0, 0) publishes the start as k_start_gate does.  Both
// ignore the gate flag, which the previous solve left set.
enum { DOWN_PLAIN = 0, START_PARTIALS = 1, START_TEST = 2 };
// partials in c->partial: start norm at kStartOff + tile, boundary data at
// kStartOff + kStartCap + tile (the level-0 up kernel's norm partials stay
// below kStartOff)
constexpr int kStartOff = 8192, kStartCap = 4096;
static_assert(kStartOff + 2 * kStartCap <= kPartialCap, "start partials");

struct StartArgs {
  double *part;    // c->partial + kStartOff
  int nb;          // tiles of the level-0 down kernel (partials per kind)
  double *scal, *mb;
  int *gate;
  int rel, cap;
  double tol;
  // launched ahead (spec: the gate word it waits on, else 0): START_PARTIALS
  // goes on only if gate[spec] == 1 (2: the solve before it converged; 7:
  // k_combine accepted the attempt) and records that decision in gate[6];
  // START_TEST abandons the start when gate[6] is 0 (gate[0] = 1 stops the
  // batch behind it, the mailbox step carries outcome 4)
  int spec;
  // DOWN_PLAIN at level 0: the stop test of the previous V-cycle (that of
  // k_norm_gate, on its nb norm partials at part, at most 256 in FP64) runs
  // here
  int fold;
};

// Halo of an up kernel: one ring per half-sweep and one for the residual
// norm, rounded up to even so that quads start on even rows and columns.
__host__ __device__ inline int up_halo(int nu, bool norm) {
  return 2 * nu + (norm ? 2 : 0);
}

// Pre-smoothing + residual + restriction (levels above the tail), S quads
// per thread.  The gate is read with the tile's loads in flight and obeyed
// after the first barrier.
template <typename T, bool HAS_F, bool EXACT, int SMODE, int S>
__global__ __launch_bounds__(TILE_THREADS) void k_down(
    const T *__restrict__ uin, T *__restrict__ uout, const T *__restrict__ f,
    const T *__restrict__ cx, const T *__restrict__ cz, int N, int K, int P,
    T DH2, T relax, int nu, int zero_u, T *__restrict__ r2, int Nc, int Kc,
    int Pc, int TX, int TY, int H, const int *__restrict__ gate, StartArgs sa) {
  extern __shared__ __align__(16) unsigned char smem[];
  __shared__ double sdec[16 * 2];
  const int nthr = blockDim.x * blockDim.y;
  const int ltid = threadIdx.y * blockDim.x + threadIdx.x;
  const bool wg0 = blockIdx.x == 0 && blockIdx.y == 0 && ltid == 0;
  // (FP64 has no right-hand side on level 0, FP32 refinement has one)
  const bool folding = SMODE == DOWN_PLAIN && (!HAS_F || !EXACT) && sa.fold;
  // whether this launch does nothing: the solve has stopped, or (launched
  // ahead) what it waits on did not go through
  bool leave = false;
  if (SMODE == DOWN_PLAIN) leave = gate && gate[0];
  if (SMODE == START_PARTIALS) leave = sa.spec && sa.gate[sa.spec] != 1;
  if (SMODE == START_TEST) leave = sa.spec && sa.gate[6] == 0;

  constexpr int PS = kPlaneWords<T, S>;
  const QTile<T, PS> t = make_qtile<T, PS>(smem, TX, TY, H);
  Quad<T> q[S];
#pragma unroll
  for (int i = 0; i < S; i++) {
    quad_place(t, q[i], ltid + i * nthr, N, K);
    quad_load<T, HAS_F>(t, q[i], uin, f, cx, cz, N, K, P, zero_u != 0);
  }
  // folded stop test: each of k_norm_gate's 256 threads (the first four
  // wavefronts here) loads its partials with the tile and sums in
  // k_norm_gate's order, so every workgroup takes the same decision
  double fold_p = 0.0;
  if (folding && EXACT && ltid < sa.nb) fold_p = 0.0 + sa.part[ltid];
  if (folding && !EXACT && ltid < 256) fold_p = strided_sum(sa.part, sa.nb, ltid);
  // the start norms from the level-0 tiles' partials, summed by the whole
  // workgroup (every workgroup alike), four loads of a thread in flight
  double v2[2] = {0.0, 0.0};
  if (SMODE == START_TEST) {
    for (int i0 = ltid; i0 < sa.nb; i0 += 4 * nthr) {
      double p[4], b[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int at = min(i0 + i * nthr, sa.nb - 1);
        p[i] = sa.part[at];
        b[i] = sa.part[kStartCap + at];
      }
#pragma unroll
      for (int i = 0; i < 4; i++)
        if (i0 + i * nthr < sa.nb) {
          v2[0] += p[i];
          v2[1] += b[i];
        }
    }
  }
#pragma unroll
  for (int i = 0; i < S; i++) {
    quad_put(t, q[i]);
    quad_factors<T, EXACT>(q[i], relax);
    one_quad_at_a_time<T, S>();
  }
  if (folding && ltid < 256) {
    const double w = wave_sum(fold_p);
    if ((ltid & 63) == 0) sdec[ltid >> 6] = w;
  }
  if (SMODE == START_TEST)
    block_sums<2>(v2, sdec);  // with the tile's barrier
  else
    __syncthreads();
  if (SMODE == START_PARTIALS && sa.spec && wg0) sa.gate[6] = leave ? 0 : 1;
  if (leave) {
    // a folded stop test still takes its step of the mailbox sequence
    if (folding && wg0) sa.gate[3] = sa.gate[3] + 1;
    if (SMODE == START_TEST && wg0) {
      sa.gate[0] = 1;
      const int seq = sa.gate[3] + 1;
      sa.gate[3] = seq;
      sa.mb[MB_CODE] = 4.0;
      __threadfence_system();
      sa.mb[MB_SEQ] = (double)seq;
    }
    return;
  }
  if (SMODE == START_TEST) {
    const double du = sqrt(v2[0]);
    const double r0 = sa.rel ? sqrt(v2[1]) : du;
    const double thr = sa.rel ? sa.tol * r0 : sa.tol;
    int code = 0;
    if (!(du > thr))
      code = 1;
    else if (sa.cap < 1)
      code = 3;
    if (wg0) {
      sa.scal[SC_NORM] = du;
      sa.scal[SC_NORM0] = r0;
      sa.gate[0] = code ? 1 : 0;
      sa.gate[1] = 0;
      sa.gate[2] = code;
      sa.gate[4] = 0;
      sa.gate[5] = 0;
      sa.mb[SC_NORM] = du;
      sa.mb[SC_NORM0] = r0;
      sa.mb[MB_START] = du;
      sa.mb[MB_USED] = 0.0;
      sa.mb[MB_COUNT] = 0.0;
      sa.mb[MB_CODE] = (double)code;
      const int seq = sa.gate[3] + 1;
      sa.gate[3] = seq;
      __threadfence_system();
      sa.mb[MB_SEQ] = (double)seq;
    }
    if (code) return;  // no V-cycle needed
  }
  if (folding) {
    const double v = sqrt(((sdec[0] + sdec[1]) + sdec[2]) + sdec[3]);
    const int code = stop_code(v, sa.rel, sa.tol, sa.scal);
    if (wg0) {
      // what k_norm_gate records (the V-cycle cap is left to it: the host
      // folds no test that could reach the cap)
      const int cnt = sa.gate[1] + 1;
      sa.gate[1] = cnt;
      sa.gate[2] = code;
      sa.gate[3] = sa.gate[3] + 1;
      sa.scal[SC_NORM] = v;
      if (code) {
        sa.gate[0] = 1;
        sa.mb[SC_NORM] = v;
        sa.mb[MB_COUNT] = (double)cnt;
        sa.mb[MB_CODE] = (double)code;
        __threadfence_system();
      }
    }
    if (code) return;
  }
  if (SMODE == START_PARTIALS) {
    // the start as loaded: residual norm and boundary-data norm partials of
    // the interior points
#pragma unroll
    for (int i = 0; i < S; i++) {
      const Quad<T> &p = q[i];
      int j, k;
      if (!quad_interior(t, p, H, TX, TY, j, k)) continue;
      T r00, r01, r10, r11;
      quad_residual<T, false>(t, p, DH2, r00, r01, r10, r11);
      v2[0] += (double)(r00 * r00);
      v2[0] += (double)(r01 * r01);
      v2[0] += (double)(r10 * r10);
      v2[0] += (double)(r11 * r11);
      // the residual with a zero interior: only next to the Dirichlet columns
      auto bd = [&](bool in, int kp, T m1, T m2, T uW, T uE) {
        if (!in || (kp != 1 && kp != K - 2)) return;
        const T w = (kp - 1 == 0) ? uW : T(0), e = (kp + 1 == K - 1) ? uE : T(0);
        const T rb = T(0) - (m1 * w + m2 * e) / DH2;
        v2[1] += (double)(rb * rb);
      };
      bd(p.k00, k, p.x0, p.x1, t.p01()[p.id - 1], p.u01);
      bd(p.k01, k + 1, p.x1, p.x2, p.u00, t.p00()[p.id + 1]);
      bd(p.k10, k, p.y0, p.y1, t.p11()[p.id - 1], p.u11);
      bd(p.k11, k + 1, p.y1, p.y2, p.u10, t.p10()[p.id + 1]);
    }
    block_sums<2>(v2, sdec);
    if (ltid == 0) {
      const int bid = tile_id();
      sa.part[bid] = v2[0];
      sa.part[kStartCap + bid] = v2[1];
    }
  }
  quads_sweep<T, HAS_F, EXACT, false, S>(t, q, nu, DH2, relax);
  // residuals of the interior and the ring below and left of it, in the
  // planes of their points (the values stay in the registers); point (0, 0)
  // is only needed by its own quad
  T r00[S], r01[S], r10[S], r11[S];
#pragma unroll
  for (int i = 0; i < S; i++) {
    quad_residual<T, HAS_F>(t, q[i], DH2, r00[i], r01[i], r10[i], r11[i]);
    one_quad_at_a_time<T, S>();
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < S; i++)
    if (q[i].valid) {
      t.p01()[q[i].id] = r01[i];
      t.p10()[q[i].id] = r10[i];
      t.p11()[q[i].id] = r11[i];
    }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < S; i++) {
    const Quad<T> &p = q[i];
    int j, k;
    if (!quad_interior(t, p, H, TX, TY, j, k)) continue;
    quad_store(p, j, k, uout, N, K, P);
    // restriction onto the coarse point under (0, 0); the first and last
    // coarse rows use their one fine neighbour row twice
    const int jc = j >> 1, kc = k >> 1;
    if (jc >= Nc || kc < 1 || kc > Kc - 2) continue;
    const T v = quad_restrict(t, p.id, r00[i], r01[i], r10[i], r11[i], jc == 0,
                              jc == Nc - 1);
    r2[(size_t)jc * Pc + kc] = v;
  }
}

// Level-0 finishing modes of k_up.
enum { UP_STORE = 0, UP_NORM = 1, UP_ADD64 = 2 };

// Prolongation at the load: none (further sweeps, or the first sweeps of a
// level when zero_u), the reference's, or with the last row too.
enum { PROL_NONE = 0, PROL_REF = 1, PROL_FULL = 2 };

// Prolongation + correction + post-smoothing, S quads per thread.
template <typename T, bool HAS_F, bool EXACT, int PROL, int MODE, int S>
__global__ __launch_bounds__(TILE_THREADS) void k_up(
    const T *__restrict__ uin, T *__restrict__ uout, const T *__restrict__ f,
    const T *__restrict__ cx, const T *__restrict__ cz, int N, int K, int P,
    T DH2, T relax, int nu, int zero_u, const T *__restrict__ e, int Nc, int Kc, int Pc,
    int TX, int TY, int H, double *__restrict__ partial, double *__restrict__ u64,
    const int *__restrict__ gate) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int nthr = blockDim.x * blockDim.y;
  const int ltid = threadIdx.y * blockDim.x + threadIdx.x;
  const bool leave = gate && gate[0];  // the solve has converged
  constexpr int PS = kPlaneWords<T, S>;
  const QTile<T, PS> t = make_qtile<T, PS>(smem, TX, TY, H);
  Quad<T> q[S];
#pragma unroll
  for (int i = 0; i < S; i++) {
    quad_place(t, q[i], ltid + i * nthr, N, K);
    quad_load<T, HAS_F>(t, q[i], uin, f, cx, cz, N, K, P, PROL == PROL_NONE && zero_u);
    if (PROL != PROL_NONE)
      quad_prolong<T, PROL == PROL_FULL>(t, q[i], e, Nc, Kc, Pc, N, K);
  }
#pragma unroll
  for (int i = 0; i < S; i++) {
    quad_put(t, q[i]);
    quad_factors<T, EXACT>(q[i], relax);
    one_quad_at_a_time<T, S>();
    if (HAS_F) {
      q[i].f00 = DH2 * q[i].f00;
      q[i].f01 = DH2 * q[i].f01;
      q[i].f10 = DH2 * q[i].f10;
      q[i].f11 = DH2 * q[i].f11;
    }
  }
  __syncthreads();
  if (leave) return;
  quads_sweep<T, HAS_F, EXACT, true, S>(t, q, nu, DH2, relax);
  if (MODE == UP_NORM) {
    // the residual-norm partial of the tile's interior first: the block
    // sum's barrier then has no global stores of this kernel to wait for
    double acc = 0.0;
#pragma unroll
    for (int i = 0; i < S; i++) {
      int j, k;
      if (!quad_interior(t, q[i], H, TX, TY, j, k)) continue;
      T r00, r01, r10, r11;
      quad_residual<T, false>(t, q[i], DH2, r00, r01, r10, r11);
      acc += (double)(r00 * r00);
      acc += (double)(r01 * r01);
      acc += (double)(r10 * r10);
      acc += (double)(r11 * r11);
      one_quad_at_a_time<T, S>();
    }
    __shared__ double red[16];
    const double s = block_sum1(acc, red);
    if (ltid == 0) partial[tile_id()] = s;
  }
#pragma unroll
  for (int i = 0; i < S; i++) {
    const Quad<T> &p = q[i];
    int j, k;
    if (!quad_interior(t, p, H, TX, TY, j, k)) continue;
    if (MODE == UP_ADD64) {
      const size_t g = (size_t)j * P + k;
      if (p.k00) u64[g] += (double)p.u00;
      if (p.k01) u64[g + 1] += (double)p.u01;
      if (p.k10) u64[g + P] += (double)p.u10;
      if (p.k11) u64[g + P + 1] += (double)p.u11;
    } else {
      quad_store(p, j, k, uout, N, K, P);
    }
  }
}

// ---------------------------------------------------------------------------
// Coarse tail: one workgroup runs every level with N, K <= 33.
// ---------------------------------------------------------------------------
//
// One quad per thread and level (289 of them at 33^2, so five wavefronts
// sweep and the others only wait); values in planes, residuals, right-hand
// sides and corrections in the LDS.  A V-cycle's tail is a serial chain of
// small steps in one CU, bound by LDS and barrier latency and by its loads.
// Against one point of each colour per thread over all 16 wavefronts, FP64
// with entry level 33^2: the production cycle's tail 13.9 -> 10.4 us, the
// reference's (192 half-sweeps) 84 -> 44 us.

struct TailLevel {
  const void *cx, *cz;  // global coefficients of the level
  int N, K, P;          // dims and global pitch
  double DH2;
};

struct TailArgs {
  TailLevel lv[6];
  int nlev;             // levels in the tail (first = entry level)
  const void *f_in;     // restricted residual of the entry level (global)
  void *e_out;          // correction of the entry level (global)
  int nu_pre, nu_post, nu_coarse;
  double relax;
  const void *minv;     // direct coarsest solve (FP32 inverse: column-major cinv32 in
                        // k_tail, else cinv4) or null
  int cn;               // coarsest unknowns for minv
  const int *gate;      // skip flag of a batched solve, or null
};

constexpr int kTailAhead = 32;

// LDS words of a tail level: its value planes, and its right-hand side
// (rows 0..N, so that a quad's second row of the last one stays inside).
__host__ __device__ inline int tail_quads(int N, int K) {
  return ((N + 1) / 2) * ((K + 1) / 2);
}
constexpr int kTailPlane = ((TAIL_MAX_N + 1) / 2) * ((TAIL_MAX_N + 1) / 2) +
                           (TAIL_MAX_N + 1) / 2 + 1;
__host__ __device__ inline size_t tail_plane_words(int K) {
  return 4 * (size_t)kTailPlane + (size_t)quad_guard((K + 1) / 2);
}
__host__ __device__ inline size_t tail_level_words(int N, int K) {
  return tail_plane_words(K) + (size_t)(N + 1) * K + 2;
}

// Level l's planes as a tile that covers the level, and its right-hand side;
// recomputed from the level dimensions (uniform values) at each use: a
// per-level table indexed by a loop variable would live in per-lane scratch
// memory.
template <typename T>
__device__ inline QTile<T, kTailPlane> tail_tile(T *base, const TailArgs &a, int l) {
  for (int i = 0; i < l; i++) base += tail_level_words(a.lv[i].N, a.lv[i].K);
  QTile<T, kTailPlane> t;
  t.C2 = (a.lv[l].K + 1) / 2;
  t.nq = tail_quads(a.lv[l].N, a.lv[l].K);
  t.j0 = t.k0 = 0;
  t.p = base + quad_guard(t.C2);
  t.stride = 0;
  return t;
}
template <typename T>
__device__ inline T *tail_rhs(T *base, const TailArgs &a, int l) {
  for (int i = 0; i < l; i++) base += tail_level_words(a.lv[i].N, a.lv[i].K);
  return base + tail_plane_words(a.lv[l].K);
}

// The thread's quad of level l: place, coefficients and factors (values zero).
template <typename T, bool EXACT>
__device__ inline void tail_quad(const QTile<T, kTailPlane> &t, Quad<T> &q, const TailLevel &L,
                                 T relax) {
  quad_place(t, q, (int)threadIdx.x, L.N, L.K);
  if (!q.valid) return;
  quad_load<T, false>(t, q, (const T *)nullptr, (const T *)nullptr, (const T *)L.cx,
                      (const T *)L.cz, L.N, L.K, L.P, true);
  quad_factors<T, EXACT>(q, relax);
}

// Its right-hand side from the LDS.
template <typename T>
__device__ inline void tail_quad_rhs(const QTile<T, kTailPlane> &t, Quad<T> &q, const T *F, int K) {
  if (!q.valid) return;
  int j, k;
  quad_rc(t, q.id, j, k);
  const T *f = F + j * K + k;
  q.f00 = f[0];
  q.f01 = f[1];
  q.f10 = f[K];
  q.f11 = f[K + 1];
}

// Sweeps of the level by the threads that hold a quad.
template <typename T, bool EXACT>
__device__ inline void tail_sweep(const QTile<T, kTailPlane> &t, Quad<T> &q, int nu, T DH2, T relax) {
  Quad<T>(&qs)[1] = reinterpret_cast<Quad<T>(&)[1]>(q);
  for (int s = 0; s < nu; s++) {
    if (q.valid) quads_half_sweep<T, true, EXACT, false, 0, 1>(t, qs, DH2, relax);
    __syncthreads();
    if (q.valid) quads_half_sweep<T, true, EXACT, false, 1, 1>(t, qs, DH2, relax);
    __syncthreads();
  }
}

// Values of the level into the row-major correction E (boundary columns too).
template <typename T>
__device__ inline void tail_put_e(const QTile<T, kTailPlane> &t, const Quad<T> &q, T *E, int N,
                                  int K) {
  if (!q.valid) return;
  int j, k;
  quad_rc(t, q.id, j, k);
  T *e = E + j * K + k;
  e[0] = q.u00;
  if (k + 1 < K) e[1] = q.u01;
  if (j + 1 < N) {
    e[K] = q.u10;
    if (k + 1 < K) e[K + 1] = q.u11;
  }
}

// Residual of level l and its restriction into F (the next level's right-hand
// side) and, for a direct coarsest solve, DH^2 times it into G.
template <typename T>
__device__ inline void tail_restrict(const QTile<T, kTailPlane> &t, const Quad<T> &q, T *R, T DH2,
                                     T *F, T *G, T DH2c, int Nc, int Kc) {
  QTile<T, kTailPlane> r = t;
  r.p = R + quad_guard(t.C2);
  T r00, r01, r10, r11;
  if (q.valid) {
    quad_residual<T, true>(t, q, DH2, r00, r01, r10, r11);
    r.p01()[q.id] = r01;
    r.p10()[q.id] = r10;
    r.p11()[q.id] = r11;
  }
  __syncthreads();
  if (q.valid) {
    const int jc = q.id / t.C2, kc = q.id - jc * t.C2;
    if (jc < Nc && kc >= 1 && kc <= Kc - 2) {
      const T v = quad_restrict(r, q.id, r00, r01, r10, r11, jc == 0, jc == Nc - 1);
      F[jc * Kc + kc] = v;
      if (G) G[jc * (Kc - 2) + kc - 1] = DH2c * v;
    }
  }
  __syncthreads();
}

// LDS behind the levels' arrays: residual planes, corrections, the direct
// solve's right-hand side and partial sums.
template <typename T>
struct TailScratch {
  T *R, *E, *G, *part;
  __device__ TailScratch(T *base, const TailArgs &a) {
    R = base;
    for (int i = 0; i < a.nlev; i++) R += tail_level_words(a.lv[i].N, a.lv[i].K);
    E = R + tail_plane_words(a.lv[0].K);
    G = E + a.lv[0].N * a.lv[0].K;
    part = G + a.cn + 4;
  }
};

// The chunks' sums of the direct coarsest solve added in order, into s.E with
// its boundary columns; ends with a barrier.
template <typename T, int THREADS>
__device__ inline void tail_sum_chunks(const TailScratch<T> &s, int n, int Q, int K, int W) {
  for (int i = threadIdx.x; i < n; i += THREADS) {
    T v = s.part[i];
    for (int ch = 1; ch < Q; ch++) v = v + s.part[ch * n + i];
    const int j = i / W, k = i - j * W + 1;
    s.E[j * K + k] = v;
    if (k == 1) s.E[j * K] = T(0);
    if (k == W) s.E[j * K + W + 1] = T(0);
  }
  __syncthreads();
}

// Direct coarsest solve from s.G into s.E (level L); starts after and ends
// with a barrier.
template <typename T>
__device__ inline void tail_solve(const TailArgs &a, const TailScratch<T> &s, const TailLevel &L) {
  const float *minv = reinterpret_cast<const float *>(a.minv);
  const int n = a.cn, W = L.K - 2, Q = coarse_chunks(n), C = coarse_chunk_len(n);
  const int ch = threadIdx.x / n, row = threadIdx.x - ch * n;
  const int c0 = min(ch * C, n), c1 = ch < Q ? min((ch + 1) * C, n) : c0;
  T acc = T(0);
#pragma unroll 8
  for (int col = c0; col < c1; col++)
    acc = acc + (T)load_at<float>(minv, (unsigned)(col * n + row) * 4u) * s.G[col];
  s.part[threadIdx.x] = acc;
  __syncthreads();
  tail_sum_chunks<T, TAIL_THREADS>(s, n, Q, L.K, W);
}

// 16-byte groups of the inverse that a thread of TailDirect sums, and the most
// over the sizes of the level below an entry level.
__host__ __device__ constexpr int tail_direct_groups(int n) {
  const int Q = coarse_chunks(n), fit = DIRECT_THREADS / n, parts = Q < fit ? Q : fit;
  return (Q + parts - 1) / parts * coarse_chunk_quads(n);
}
constexpr int tail_direct_most() {
  constexpr int N = (TAIL_MAX_N + 1) / 2;
  int most = 0;
  for (int n = 1; n <= N * (N - 2); n++) most = std::max(most, tail_direct_groups(n));
  return most;
}
static_assert(tail_direct_most() <= kTailAhead, "the inverse's entries of a thread");

// The same by DIRECT_THREADS threads with the inverse's entries, in 16-byte
// groups, all fetched ahead: a thread has one row and whole chunks from ch0 on,
// each with its own sum.
template <typename T, int AHEAD>
struct TailDirect {
  float4 ahead[AHEAD];
  int row, ch0;
  unsigned off, end;  // next group and the last one, in bytes
  __device__ void place(const TailArgs &a) {
    const int n = a.cn, Q = coarse_chunks(n), GC = coarse_chunk_quads(n);
    const int parts = min(Q, DIRECT_THREADS / n), per = (Q + parts - 1) / parts;
    const int part = (int)threadIdx.x / n;
    row = threadIdx.x - part * n;
    ch0 = min(part * per, Q);
    end = (unsigned)((Q * GC - 1) * n + row) * 16u;
    off = min((unsigned)(ch0 * GC * n + row) * 16u, end);
  }
  template <int FROM, int TO>
  __device__ void fetch(const TailArgs &a) {
#pragma unroll
    for (int i = FROM; i < TO; i++) {
      ahead[i] = load_at<float4>(reinterpret_cast<const float4 *>(a.minv), off);
      off = min(off + (unsigned)a.cn * 16u, end);
    }
  }
  // The group's four values of s.G are read two groups ahead.  Padding entries
  // are zero and s.G has four zeros behind it, so no group needs a test.
  __device__ void solve(const TailArgs &a, const TailScratch<T> &s, const TailLevel &L) {
    const int n = a.cn, Q = coarse_chunks(n), C = coarse_chunk_len(n);
    const int GC = coarse_chunk_quads(n), skip = C - 4 * (GC - 1);
    int ch = ch0, left = GC, col = min(ch0 * C, n), left_col = GC;
    struct Four {
      T v[4];
    } g[3];
    auto read = [&](Four &f) {
#pragma unroll
      for (int e = 0; e < 4; e++) f.v[e] = s.G[col + e];
      const bool end = --left_col == 0;
      col = min(col + (end ? skip : 4), n);
      if (end) left_col = GC;
    };
    T acc = T(0);
    auto add = [&](const float4 &m, const Four &f) {
      acc = acc + (T)m.x * f.v[0];
      acc = acc + (T)m.y * f.v[1];
      acc = acc + (T)m.z * f.v[2];
      acc = acc + (T)m.w * f.v[3];
      if (--left == 0) {
        if (ch < Q) s.part[ch * n + row] = acc;
        acc = T(0);
        ch++;
        left = GC;
      }
    };
    const int most = tail_direct_groups(n);
    read(g[0]);
    read(g[1]);
#pragma unroll
    for (int i = 0; i < AHEAD; i++)
      if (i < most) {
        read(g[(i + 2) % 3]);
        add(ahead[i], g[i % 3]);
      }
    __syncthreads();
    tail_sum_chunks<T, DIRECT_THREADS>(s, n, Q, L.K, L.K - 2);
  }
};

// Any tail: each visit of a level loads its quads' coefficients again.
template <typename T, bool EXACT, bool FULL_TOP>
__global__ __launch_bounds__(TAIL_THREADS) void k_tail(TailArgs a) {
  if (a.gate && a.gate[0]) return;  // the solve has converged
  extern __shared__ __align__(16) unsigned char smem[];
  T *base = reinterpret_cast<T *>(smem);
  const TailScratch<T> s(base, a);
  const int tid = threadIdx.x, last = a.nlev - 1;
  const T relax = (T)a.relax;
  const bool direct = a.minv != nullptr;
  const TailLevel &L0 = a.lv[0], &LC = a.lv[last];
  {
    T *F = tail_rhs(base, a, 0);
    for (int i = tid; i < L0.N * L0.K; i += TAIL_THREADS) {
      const int j = i / L0.K, k = i - j * L0.K;
      F[i] = ((const T *)a.f_in)[(size_t)j * L0.P + k];
    }
  }
  Quad<T> p;
  for (int l = 0; l < last; l++) {
    const TailLevel &L = a.lv[l], &C = a.lv[l + 1];
    const QTile<T, kTailPlane> t = tail_tile(base, a, l);
    tail_quad<T, EXACT>(t, p, L, relax);
    if (p.valid) quad_put(t, p);
    __syncthreads();
    tail_quad_rhs(t, p, tail_rhs(base, a, l), L.K);
    tail_sweep<T, EXACT>(t, p, a.nu_pre, (T)L.DH2, relax);
    tail_restrict(t, p, s.R, (T)L.DH2, tail_rhs(base, a, l + 1),
                  direct && l + 1 == last ? s.G : nullptr, (T)C.DH2, C.N, C.K);
  }
  if (direct) {  // below two levels or more (k_coarse_rows, k_tail_direct else)
    tail_solve(a, s, LC);
  } else {
    const QTile<T, kTailPlane> t = tail_tile(base, a, last);
    tail_quad<T, EXACT>(t, p, LC, relax);
    if (p.valid) quad_put(t, p);
    __syncthreads();
    tail_quad_rhs(t, p, tail_rhs(base, a, last), LC.K);
    tail_sweep<T, EXACT>(t, p, a.nu_coarse, (T)LC.DH2, relax);
    tail_put_e(t, p, s.E, LC.N, LC.K);
    __syncthreads();
  }
  for (int l = last - 1; l >= 0; l--) {
    const TailLevel &L = a.lv[l], &C = a.lv[l + 1];
    const QTile<T, kTailPlane> t = tail_tile(base, a, l);
    tail_quad<T, EXACT>(t, p, L, relax);
    tail_quad_rhs(t, p, tail_rhs(base, a, l), L.K);
    if (p.valid) {
      p.u00 = t.p00()[p.id];
      p.u01 = t.p01()[p.id];
      p.u10 = t.p10()[p.id];
      p.u11 = t.p11()[p.id];
      quad_prolong<T, FULL_TOP>(t, p, s.E, C.N, C.K, C.K, L.N, L.K);
    }
    __syncthreads();
    if (p.valid) quad_put(t, p);
    __syncthreads();
    tail_sweep<T, EXACT>(t, p, a.nu_post, (T)L.DH2, relax);
    tail_put_e(t, p, s.E, L.N, L.K);
    __syncthreads();
  }
  T *eo = reinterpret_cast<T *>(a.e_out);
  for (int i = tid; i < L0.N * L0.K; i += TAIL_THREADS) {
    const int j = i / L0.K, k = i - j * L0.K;
    eo[(size_t)j * L0.P + k] = s.E[i];
  }
}

// The tail of the production cycle: one level and the direct coarsest solve.
// The level's quads stay in registers from the load to the store, and each
// thread fetches its entries of the coarsest inverse (255^2 floats at 1025^2)
// before they are needed, two chunks of a row in 128 registers: half of them
// with the level's data, half behind the sweeps (all at once they hold up the
// first sweep, at the 64 bytes a clock of one CU).  With 1024 threads
// the registers held half of a thread's chunk and the rest was loaded during
// the solve, which took 5.5 us between the other kernels of a V-cycle; 3.5
// now, the FP32 to FP64 conversions and the products' issue (V-cycle at 1025^2
// 80.7 -> 79.3 us; launched back to back, with the inverse in the L2, the
// kernel takes 10.4 us either way).
template <typename T, bool EXACT>
__global__ __launch_bounds__(DIRECT_THREADS) void k_tail_direct(TailArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  T *base = reinterpret_cast<T *>(smem);
  const TailScratch<T> s(base, a);
  const T relax = (T)a.relax;
  const bool leave = a.gate && a.gate[0];  // the solve has converged
  const TailLevel &L = a.lv[0], &C = a.lv[1];
  const QTile<T, kTailPlane> t = tail_tile(base, a, 0);
  const T DH2 = (T)L.DH2;
  Quad<T> q;
  quad_place(t, q, (int)threadIdx.x, L.N, L.K);
  if (q.valid)
    quad_load<T, true>(t, q, (const T *)nullptr, (const T *)a.f_in, (const T *)L.cx,
                       (const T *)L.cz, L.N, L.K, L.P, true);
  TailDirect<T, kTailAhead> d;
  d.place(a);
  d.template fetch<0, kTailAhead / 2>(a);
  if (threadIdx.x < 4) s.G[a.cn + threadIdx.x] = T(0);
  if (q.valid) {
    quad_factors<T, EXACT>(q, relax);
    quad_put(t, q);
  }
  __syncthreads();
  if (leave) return;
  tail_sweep<T, EXACT>(t, q, a.nu_pre, DH2, relax);
  d.template fetch<kTailAhead / 2, kTailAhead>(a);
  tail_restrict(t, q, s.R, DH2, tail_rhs(base, a, 1), s.G, (T)C.DH2, C.N, C.K);
  d.solve(a, s, C);
  if (q.valid) {
    quad_prolong<T, true>(t, q, s.E, C.N, C.K, C.K, L.N, L.K);
    quad_put(t, q);
  }
  __syncthreads();
  tail_sweep<T, EXACT>(t, q, a.nu_post, DH2, relax);
  if (q.valid) {
    int j, k;
    quad_rc(t, q.id, j, k);
    quad_store(q, j, k, reinterpret_cast<T *>(a.e_out), L.N, L.K, L.P);
  }
}

// A tail of the direct coarsest solve alone (the next finer level is too large
// for the tail): e = inverse (DH^2 f), COARSE_ROWS rows per workgroup, whose
// entries of the inverse are staged in the LDS by all threads before one
// wavefront sums a chunk of a row per lane.  In one workgroup (k_tail) 384
// unknowns took 9.6 us, bound by one CU's loads; 5.5 us in 24
// workgroups (V-cycle at 801 x 481 64 -> 60 us).
constexpr int COARSE_ROWS = 16, COARSE_THREADS = 512;
__host__ __device__ inline size_t coarse_rows_lds(int n, size_t esz) {
  return (size_t)coarse_chunks(n) * coarse_chunk_quads(n) * COARSE_ROWS * 16 +
         (n + 4 + 4 * COARSE_ROWS) * esz;
}
template <typename T>
__global__ __launch_bounds__(COARSE_THREADS) void k_coarse_rows(TailArgs a) {
  extern __shared__ __align__(16) unsigned char smem[];
  const TailLevel &L = a.lv[0];
  const bool leave = a.gate && a.gate[0];  // the solve has converged
  const int n = a.cn, W = L.K - 2, Q = coarse_chunks(n), C = coarse_chunk_len(n);
  const int GC = coarse_chunk_quads(n), groups = Q * GC * COARSE_ROWS, tid = threadIdx.x;
  float4 *M = reinterpret_cast<float4 *>(smem);
  T *G = reinterpret_cast<T *>(M + groups), *part = G + n + 4;
  const int row0 = blockIdx.x * COARSE_ROWS;
  const float4 *inv = reinterpret_cast<const float4 *>(a.minv);
#pragma unroll 4
  for (int i = tid; i < groups; i += COARSE_THREADS)
    M[i] = inv[(size_t)(i / COARSE_ROWS) * n + min(row0 + i % COARSE_ROWS, n - 1)];
  for (int i = tid; i < n + 4; i += COARSE_THREADS) {
    const int j = i / W, k = i - j * W + 1;
    G[i] = i < n ? (T)L.DH2 * ((const T *)a.f_in)[(size_t)j * L.P + k] : T(0);
  }
  __syncthreads();
  if (leave) return;
  const int ch = tid / COARSE_ROWS, r = tid % COARSE_ROWS, row = row0 + r;
  if (ch < Q) {
    T acc = T(0);
#pragma unroll 8
    for (int g = 0; g < GC; g++) {
      // padding entries are zero; so is G behind its end
      const float4 m = M[(ch * GC + g) * COARSE_ROWS + r];
      const T *p = G + min(ch * C + 4 * g, n);
      acc = acc + (T)m.x * p[0];
      acc = acc + (T)m.y * p[1];
      acc = acc + (T)m.z * p[2];
      acc = acc + (T)m.w * p[3];
    }
    part[tid] = acc;
  }
  __syncthreads();
  if (ch != 0 || row >= n) return;
  T v = part[r];
  for (int q = 1; q < Q; q++) v = v + part[q * COARSE_ROWS + r];
  const int j = row / W, k = row - j * W + 1;
  T *e = (T *)a.e_out + (size_t)j * L.P;
  e[k] = v;
  if (k == 1) e[0] = T(0);
  if (k == W) e[W + 1] = T(0);
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------

// The sizes of tiles that the shape checks accept: three words per point of
// the tile and its halo (an up kernel's of 2 n_post + 1), one more with a
// right-hand side (or, for a level-0 down tile, beyond eight residuals per
// thread) within the LDS.  The quads need one word per point, and a workgroup
// holds kMaxQuads per thread of 1024 threads: enough at every such size but the
// FP64 level-0 up kernel's with one more ring of halo, whose tiles of two or
// four columns and 1000 rows or more (n_post = 0) are cut (up_shape).
static size_t tile_budget_bytes(int TX, int TY, int H, bool has_f, size_t esz,
                                bool down, int threads) {
  const size_t R = TY + 2 * H, C = TX + 2 * H;
  size_t words = 3 * R * C + C;
  if (has_f || (down && (TX + 2) * (TY + 2) > 8 * threads)) words += R * C;
  return words * esz;
}

// Launch of a tile kernel: quads per thread, thread rows and LDS.
template <typename T>
struct QuadLaunch {
  int quads, rows;
  size_t lds;
  QuadLaunch(const TileShape &s, int H) {
    constexpr int most = kMaxQuads<T>;
    const int R = s.ty + 2 * H, C = s.tx + 2 * H, nq = (R / 2) * (C / 2);
    // as few quads per thread as the shape's rows allow, then no more rows
    // than hold them (but four: a folded stop test sums with 256 threads)
    quads = std::min(most, (nq + TX_THREADS * s.tyt - 1) / (TX_THREADS * s.tyt));
    rows = std::max((nq + TX_THREADS * quads - 1) / (TX_THREADS * quads),
                    std::min(s.tyt, 4));
    lds = quad_lds_words(R, C, quads < most ? 0 : kPlaneWords<T, most>) * sizeof(T);
  }
};

// First level handled by the tail (or L if the coarsest level is too big).
int tail_entry_level(const qdeq_ctx *c) {
  for (int l = 0; l < c->L; l++)
    if (c->lv[l].N <= TAIL_MAX_N && c->lv[l].K <= TAIL_MAX_N && l > 0) {
      if (c->L - l > 6) return c->L;
      return l;
    }
  return c->L;
}

template <typename T>
static size_t tail_lds_bytes(const qdeq_ctx *c, int lt) {
  size_t n = 0;
  for (int l = lt; l < c->L; l++) n += tail_level_words(c->lv[l].N, c->lv[l].K);
  n += tail_plane_words(c->lv[lt].K);  // residuals
  n += (size_t)c->lv[lt].N * c->lv[lt].K;           // corrections
  n += c->coarse_n + 4;  // right-hand side of the direct coarsest solve
  n += 1024;         // its partial sums
  return n * sizeof(T);
}

bool tail_fits(const qdeq_ctx *c, bool fp64) {
  const int lt = tail_entry_level(c);
  if (lt >= c->L) return false;
  const size_t b = fp64 ? tail_lds_bytes<double>(c, lt) : tail_lds_bytes<float>(c, lt);
  return b + 4096 <= c->lds_max;
}

// Shape of the down (smoothing + restriction) or up (prolongation +
// smoothing) kernel of a level: tuned or pinned, else the caller's
// (qdeq_set_tiles), else the model's.
TileShape tile_shape(const qdeq_ctx *c, int level, bool down) {
  if (c->tuned) return down ? c->tdown[level] : c->tup[level];
  if (c->user_tiles) return TileShape{c->tile_tx, c->tile_ty, TY_THREADS};
  return down ? c->mdown[level] : c->mup[level];
}

// Rows of an up kernel's halo: the norm's ring on level 0 in FP64.
static int up_halo_of(const qdeq_ctx *c, int level) {
  return up_halo(c->cfg.n_post, level == 0 && c->cfg.precision != QDEQ_PREC_FP32_IR);
}

// The up kernel's tile of a level as it is launched: the chosen shape, with no
// more rows than the quads that a workgroup holds.  The results do not depend
// on it.
static TileShape up_shape(const qdeq_ctx *c, int level) {
  TileShape s = tile_shape(c, level, false);
  const int H = up_halo_of(c, level);
  const int most = TILE_THREADS * (c->cfg.precision != QDEQ_PREC_FP32_IR ? kMaxQuads<double>
                                                                         : kMaxQuads<float>);
  s.ty = std::min(s.ty, 2 * (most / (s.tx / 2 + H)) - 2 * H);
  return s;
}

// Model of a launch's time in us, from launches measured back to back: start,
// first loads and store; the tile data; the half-sweeps at their latency plus
// the issue of the quads that share a CU.
static double pass_us(int tiles, int nq, int sweeps, double mbytes) {
  const int per_cu = (tiles + 255) / 256;
  return 3.3 + mbytes / 6.0 + 2 * sweeps * (0.17 + 0.017 * per_cu * nq / 64.0);
}

// Whether a shape fits the kernels: even sizes, tile rows (with halo) of at
// most 320 points, and the LDS with 8 KiB to spare.
static bool shape_fits(const qdeq_ctx *c, const TileShape &s, bool down,
                       bool has_f, size_t esz) {
  const int nu = down ? c->cfg.n_pre : c->cfg.n_post;
  const int H = down ? 2 * nu + 2 : 2 * nu + 1;
  if (s.tx < 2 || s.ty < 2 || (s.tx & 1) || (s.ty & 1)) return false;
  if (s.tyt < 1 || s.tyt > TY_THREADS || (s.tyt & (s.tyt - 1))) return false;
  if (s.tx + 2 * H > 5 * TX_THREADS) return false;
  return tile_budget_bytes(s.tx, s.ty, H, has_f, esz, down, TX_THREADS * s.tyt) + 8192 <=
         c->lds_max;
}

// Candidate tile sizes of a level.
static const int kTuneTX[] = {32, 64, 96, 128, 192, 256};
static const int kTuneTY[] = {2, 4, 8, 16, 32, 64};
static const int kTuneTYT[] = {4, 8, 16};
// Tile sizes that split a level into a whole number of tiles: the grids are
// 2^k + 1 points wide, so the power-of-two sizes leave a last tile of one
// or two points.  With one tile per CU per round, a grid of 16 x 16 tiles
// of 66 points at 1025^2 runs in one round where 96 x 32 needs two.
static const int kFitTX[] = {4, 8, 12, 16};
static const int kFitTY[] = {8, 12, 16, 24, 32};

static void add_fitted(std::vector<int> &v, int n, const int *parts, int np) {
  for (int i = 0; i < np; i++) {
    int t = (n + parts[i] - 1) / parts[i];
    t += t & 1;
    if (t >= 2 && std::find(v.begin(), v.end(), t) == v.end()) v.push_back(t);
  }
}

static void tile_candidates(const LevelDims &d, std::vector<int> &txs, std::vector<int> &tys) {
  txs.assign(std::begin(kTuneTX), std::end(kTuneTX));
  tys.assign(std::begin(kTuneTY), std::end(kTuneTY));
  add_fitted(txs, d.K, kFitTX, (int)(sizeof(kFitTX) / sizeof(int)));
  add_fitted(tys, d.N, kFitTY, (int)(sizeof(kFitTY) / sizeof(int)));
}

// The model's time of a tile kernel: the tile's arrays (three, one more with
// a right-hand side), the half-sweeps, residual and restriction counted as
// one sweep.  In FP32, with two or more workgroups on a CU at a time and three
// or more rounds of them, one's loads run during another's sweeps (2049^2:
// 110 us a V-cycle against 124 without this; FP64 tiles that small re-read
// too much halo, 181 against 168).  A level-0 up kernel of more than 256
// tiles costs a stop-test kernel per V-cycle (see defer_fits).  With these
// shapes a V-cycle's kernels take 68.6 us at 1025^2 FP64 (93 with tiles of
// 64 x 16 on every level, 66.0 tuned), 52 at 801 x 481 (51 tuned).
template <typename T>
static double shape_us(const qdeq_ctx *c, int l, bool down, bool has_f, const TileShape &s) {
  const LevelDims &d = c->lv[l];
  const bool norm = !down && l == 0 && !has_f;
  const int nu = down ? c->cfg.n_pre : c->cfg.n_post;
  const int H = down ? 2 * nu + 2 : up_halo(nu, norm);
  const int nq = ((s.tx + 2 * H) / 2) * ((s.ty + 2 * H) / 2);
  const int tiles = ((d.K + s.tx - 1) / s.tx) * ((d.N + s.ty - 1) / s.ty);
  const double mem = 1e-6 * tiles * nq * 4.0 * (has_f ? 4 : 3) * sizeof(T) / 6.0;
  const int quads = (nq + TILE_THREADS - 1) / TILE_THREADS;
  const int waves = (nq + 64 * quads - 1) / (64 * quads);
  const int resident = std::max(1, (quads == 1 ? 20 : 16) / waves);
  const int per_cu = (tiles + 255) / 256, rounds = (per_cu + resident - 1) / resident;
  const double sweeps = 2 * (down || norm ? nu + 1 : nu) *
                        (0.17 * rounds + 0.017 * per_cu * nq / 64.0);
  const double body = sizeof(T) == 4 && resident >= 2 && rounds >= 3
                          ? std::max(mem, sweeps) + 0.25 * std::min(mem, sweeps)
                          : mem + sweeps;
  return 3.3 + body + (norm && tiles > 256 ? 4.0 : 0.0);
}

// The model's choice per level, for contexts that neither tune nor pin their
// shapes.  One quad per thread where a kernel with two spills (FP64 down).
template <typename T>
static void model_shapes(qdeq_ctx *c) {
  const int lt = tail_entry_level(c);
  for (int l = 0; l < lt && l < QDEQ_MAX_LEVELS; l++)
    for (int dir = 0; dir < 2; dir++) {
      const bool down = dir == 0, hf = l > 0 || sizeof(T) == 4;
      TileShape best{c->tile_tx, c->tile_ty, TY_THREADS};
      double best_us = 1e300;
      std::vector<int> txs, tys;
      tile_candidates(c->lv[l], txs, tys);
      for (int tx : txs)
        for (int ty : tys) {
          const TileShape s{tx, ty, TY_THREADS};
          if (!shape_fits(c, s, down, hf, sizeof(T))) continue;
          const int H = 2 * c->cfg.n_pre + 2;
          if (down && sizeof(T) == 8 && (tx / 2 + H) * (ty / 2 + H) > TILE_THREADS) continue;
          const LevelDims &d = c->lv[l];
          if (!down && l == 0 && !hf &&
              (long)((d.K + tx - 1) / tx) * ((d.N + ty - 1) / ty) > kPartialCap)
            continue;
          const double us = shape_us<T>(c, l, down, hf, s);
          if (us < best_us) {
            best_us = us;
            best = s;
          }
        }
      (down ? c->mdown[l] : c->mup[l]) = best;
    }
}

// Largest dynamic LDS the tile kernels of this context would request.
bool tiles_fit(const qdeq_ctx *c, int tx, int ty) {
  const bool fp64 = c->cfg.precision != QDEQ_PREC_FP32_IR;
  const size_t esz = fp64 ? 8 : 4;
  const size_t down = tile_budget_bytes(tx, ty, 2 * c->cfg.n_pre + 2, true, esz, true,
                                        TILE_THREADS);
  const size_t up = tile_budget_bytes(tx, ty, 2 * c->cfg.n_post + 1, true, esz, false,
                                      TILE_THREADS);
  // tile rows (with halo) of at most 320 points
  if (tx + 2 * (2 * c->cfg.n_pre + 2) > 5 * TX_THREADS) return false;
  if (tx + 2 * (2 * c->cfg.n_post + 1) > 5 * TX_THREADS) return false;
  return down + 8192 <= c->lds_max && up + 8192 <= c->lds_max;
}

// Calls fn with the quads per thread as a compile-time constant.
template <typename T, typename Fn>
static void with_quads(int quads, Fn fn) {
  if (quads <= 1)
    fn(std::integral_constant<int, 1>{});
  else if (quads == 2 || kMaxQuads<T> == 2)
    fn(std::integral_constant<int, 2>{});
  else
    fn(std::integral_constant<int, kMaxQuads<T>>{});
}

template <typename T, typename Fn>
static void with_quads_all(Fn fn) {
  for (int s = 1; s <= kMaxQuads<T>; s++) with_quads<T>(s, fn);
}

// One launch of k_down on level l: nu sweeps of src (zero with zero_u), the
// residual restricted onto level l + 1, the swept values into dst; tiles of
// shape sh with a halo of H points.
template <typename T, bool EXACT>
static void run_down(qdeq_ctx *c, LevelBufs<T> *B, int l, bool has_f, bool zero_u,
                     int smode, const TileShape &sh, int H, int nu, const T *src, T *dst,
                     const StartArgs &sa) {
  const LevelDims &d = c->lv[l];
  const LevelDims &dc = c->lv[l + 1];
  const QuadLaunch<T> ql(sh, H);
  const dim3 grd((d.K + sh.tx - 1) / sh.tx, (d.N + sh.ty - 1) / sh.ty);
  const dim3 blk(TX_THREADS, ql.rows);
  const T DH2 = (T)(d.DH * d.DH), relax = (T)c->cfg.relax;
#define DOWN_ARGS                                                                        \
  grd, blk, ql.lds, c->stream, src, dst, B[l].f, B[l].cx, B[l].cz, d.N, d.K, d.P, DH2,   \
      relax, nu, zero_u ? 1 : 0, B[l + 1].f, dc.N, dc.K, dc.P, sh.tx, sh.ty, H,          \
      (const int *)c->gate_ptr, sa
  auto launch = [&](auto quads) {
    constexpr int S = decltype(quads)::value;
    if (smode == START_PARTIALS)
      hipLaunchKernelGGL((k_down<T, false, EXACT, START_PARTIALS, S>), DOWN_ARGS);
    else if (smode == START_TEST)
      hipLaunchKernelGGL((k_down<T, true, EXACT, START_TEST, S>), DOWN_ARGS);
    else if (has_f)
      hipLaunchKernelGGL((k_down<T, true, EXACT, DOWN_PLAIN, S>), DOWN_ARGS);
    else
      hipLaunchKernelGGL((k_down<T, false, EXACT, DOWN_PLAIN, S>), DOWN_ARGS);
  };
  with_quads<T>(ql.quads, launch);
#undef DOWN_ARGS
}

// One launch of k_up on level l: src (zero with zero_u) with the prolonged
// correction of level l + 1 (PROL), nu sweeps, finished as MODE says.
// Returns the number of workgroups (norm partials).
template <typename T, bool EXACT, bool HAS_F, int PROL, int MODE>
static int run_up(qdeq_ctx *c, LevelBufs<T> *B, int l, const TileShape &sh, int H, int nu,
                  bool zero_u, const T *src, T *dst, double *partial, double *u64) {
  const LevelDims &d = c->lv[l];
  const LevelDims &dc = c->lv[PROL == PROL_NONE ? l : l + 1];
  const T *e = PROL == PROL_NONE ? nullptr : B[l + 1].u;
  const dim3 grd((d.K + sh.tx - 1) / sh.tx, (d.N + sh.ty - 1) / sh.ty);
  const QuadLaunch<T> ql(sh, H);
  const T DH2 = (T)(d.DH * d.DH), relax = (T)c->cfg.relax;
  auto launch = [&](auto quads) {
    constexpr int S = decltype(quads)::value;
    hipLaunchKernelGGL((k_up<T, HAS_F, EXACT, PROL, MODE, S>), grd,
                       dim3(TX_THREADS, ql.rows), ql.lds, c->stream, src, dst, B[l].f,
                       B[l].cx, B[l].cz, d.N, d.K, d.P, DH2, relax, nu, zero_u ? 1 : 0, e,
                       dc.N, dc.K, dc.P, sh.tx, sh.ty, H, partial, u64,
                       (const int *)c->gate_ptr);
  };
  with_quads<T>(ql.quads, launch);
  return (int)(grd.x * grd.y);
}

template <typename T, bool EXACT>
static void launch_down(qdeq_ctx *c, LevelBufs<T> *B, int l, bool has_f,
                        bool zero_u, int smode = DOWN_PLAIN) {
  const LevelDims &d = c->lv[l];
  StartArgs sa{};
  if (smode != DOWN_PLAIN) {
    const TileShape s0 = tile_shape(c, 0, true);
    const LevelDims &d0 = c->lv[0];
    sa.part = c->partial + kStartOff;
    sa.nb = ((d0.K + s0.tx - 1) / s0.tx) * ((d0.N + s0.ty - 1) / s0.ty);
    sa.scal = c->scal;
    sa.mb = mb_dev(c);
    sa.gate = c->gate;
    sa.spec = c->spec_launch ? c->spec_go : 0;
    sa.rel = c->cfg.tol_mode == QDEQ_TOL_REL ? 1 : 0;
    sa.cap = c->cfg.max_vcycles;
    sa.tol = c->cfg.tol;
  }
  if (smode == DOWN_PLAIN && l == 0 && c->fold_next && c->gate_ptr) {
    sa.fold = 1;
    sa.part = c->partial;
    sa.nb = norm_parts(c);
    sa.scal = c->scal;
    sa.mb = mb_dev(c);
    sa.gate = c->gate;
    sa.rel = c->cfg.tol_mode == QDEQ_TOL_REL ? 1 : 0;
    sa.cap = c->cfg.max_vcycles;
    sa.tol = c->cfg.tol;
  }
  const int nu = c->cfg.n_pre;
  run_down<T, EXACT>(c, B, l, has_f, zero_u, smode, tile_shape(c, l, true), 2 * nu + 2, nu,
                     B[l].u, B[l].r, sa);
}

// Norm partials of a V-cycle on the tile kernels: the level-0 tiles of its last
// launch in FP64, the rows of the FP64 residual in FP32 refinement.
int norm_parts(const qdeq_ctx *c) {
  if (c->cfg.precision == QDEQ_PREC_FP32_IR) return norm_blocks(c);
  const LevelDims &d = c->lv[0];
  const TileShape up = use_tiled(c) ? up_shape(c, 0) : c->ref_plan[0].sh;
  return ((d.K + up.tx - 1) / up.tx) * ((d.N + up.ty - 1) / up.ty);
}

// Whether a V-cycle's stop test may run in a kernel behind it: that of the tile
// kernels, in FP64 with at most 256 norm partials (one for each of
// k_norm_gate's threads; a register-bound kernel sums no more).
static bool test_moves(const qdeq_ctx *c) {
  return !c->fold_off && (use_tiled(c) || use_ref_tiles(c)) &&
         (c->cfg.precision == QDEQ_PREC_FP32_IR || norm_parts(c) <= 256);
}

// Whether the fault update that follows a batch launched kernel by kernel may
// run its last stop test.
bool defer_fits(const qdeq_ctx *c) { return launch_direct(c) && test_moves(c); }

// Whether a batch (launched kernel by kernel, or captured as a stage's graph)
// may fold its stop tests into the next V-cycle's level-0 down kernel: that
// of the fast cycle, with a workgroup of four wavefronts or more.  FP32
// refinement sums a partial per row in every workgroup: worth the stop test's
// launch up to 8 workgroups a CU (1089 at 1025^2: 220.5 -> 215.7 us a solve,
// 257^2: 135.5 -> 128.8; 4257 at 2049^2: 411.5 -> 413.5).
bool fold_fits(const qdeq_ctx *c) {
  if (!test_moves(c) || !use_tiled(c) || tail_entry_level(c) < 1) return false;
  const LevelDims &d = c->lv[0];
  const TileShape dn = tile_shape(c, 0, true);
  const long tiles = (long)((d.K + dn.tx - 1) / dn.tx) * ((d.N + dn.ty - 1) / dn.ty);
  return TX_THREADS * dn.tyt >= 256 &&
         (c->cfg.precision == QDEQ_PREC_FP64 || tiles <= 8 * 256);
}

// Whether the start of the next FP64 solve may be folded into its first
// V-cycle's down kernels: two tile levels at least, and the start
// partials of every level-0 tile and the up kernel's norm partials fit
// their regions of c->partial.
bool fused_start_fits(const qdeq_ctx *c) {
  if (c->cfg.precision != QDEQ_PREC_FP64 || !use_tiled(c) || tail_entry_level(c) < 2)
    return false;
  const LevelDims &d = c->lv[0];
  const TileShape dn = tile_shape(c, 0, true), up = up_shape(c, 0);
  const long nd = (long)((d.K + dn.tx - 1) / dn.tx) * ((d.N + dn.ty - 1) / dn.ty);
  const long nu = (long)((d.K + up.tx - 1) / up.tx) * ((d.N + up.ty - 1) / up.ty);
  return nd <= kStartCap && nu <= kStartOff;
}

template <typename T, bool EXACT, bool HAS_F, int MODE>
static void launch_up_t(qdeq_ctx *c, LevelBufs<T> *B, int l, double *partial,
                        double *u64, int *nblocks) {
  const int nu = c->cfg.n_post;
  const int n = run_up<T, EXACT, HAS_F, PROL_FULL, MODE>(
      c, B, l, up_shape(c, l), up_halo(nu, MODE == UP_NORM), nu, false, B[l].r,
      B[l].u, partial, u64);
  if (nblocks) *nblocks = n;
}

template <typename T, bool EXACT, bool FULL_TOP = true>
static void launch_tail(qdeq_ctx *c, LevelBufs<T> *B, int lt) {
  TailArgs a{};
  a.nlev = c->L - lt;
  for (int i = 0; i < a.nlev; i++) {
    const LevelDims &d = c->lv[lt + i];
    a.lv[i] = TailLevel{B[lt + i].cx, B[lt + i].cz, d.N, d.K, d.P, d.DH * d.DH};
  }
  a.f_in = B[lt].f;
  a.e_out = B[lt].u;
  a.nu_pre = c->cfg.n_pre;
  a.nu_post = c->cfg.n_post;
  a.nu_coarse = c->cfg.n_coarse;
  a.relax = c->cfg.relax;
  a.cn = c->coarse_n;
  a.minv = c->coarse_n > 0 ? (const void *)c->cinv32 : nullptr;
  a.gate = c->gate_ptr;
  const size_t lds = tail_lds_bytes<T>(c, lt);
  if (FULL_TOP && a.nlev == 1 && a.minv) {
    a.minv = c->cinv4;
    hipLaunchKernelGGL((k_coarse_rows<T>), dim3((a.cn + COARSE_ROWS - 1) / COARSE_ROWS),
                       dim3(COARSE_THREADS), coarse_rows_lds(a.cn, sizeof(T)), c->stream, a);
  } else if (FULL_TOP && a.nlev == 2 && a.minv) {
    a.minv = c->cinv4;
    hipLaunchKernelGGL((k_tail_direct<T, EXACT>), dim3(1), dim3(DIRECT_THREADS), lds,
                       c->stream, a);
  } else {
    hipLaunchKernelGGL((k_tail<T, EXACT, FULL_TOP>), dim3(1), dim3(TAIL_THREADS), lds,
                       c->stream, a);
  }
}

// Fast V-cycle for the FP64 solve (level 0 = the displacement, f = 0) or
// the FP32 correction of iterative refinement (level 0 = correction e,
// f = r32; the last up kernel adds e into the FP64 displacement).  The
// level-0 norm partials land in `partial` (FP64) and the count of partials
// in *nparts.
template <typename T, bool EXACT>
static void vcycle_tiled(qdeq_ctx *c, LevelBufs<T> *B, bool level0_has_f,
                         double *partial, double *u64, int *nparts) {
  const int lt = tail_entry_level(c);
  // the start of the solve folded into this cycle (FP64 only)
  const bool fuse = c->fuse_start_next && !level0_has_f && lt >= 2;
  c->fuse_start_next = false;
  for (int l = 0; l < lt; l++) {
    if (l == 1) timing_mark(c, QDEQ_TIME_DOWN1, 0);
    const int smode = !fuse ? DOWN_PLAIN : (l == 0 ? START_PARTIALS
                                                    : (l == 1 ? START_TEST : DOWN_PLAIN));
    launch_down<T, EXACT>(c, B, l, l > 0 || level0_has_f, l > 0 || level0_has_f, smode);
    if (l == 1) timing_mark(c, QDEQ_TIME_DOWN1, 1);
  }
  timing_mark(c, QDEQ_TIME_TAIL, 0);
  launch_tail<T, EXACT>(c, B, lt);
  timing_mark(c, QDEQ_TIME_TAIL, 1);
  for (int l = lt - 1; l >= 1; l--)
    launch_up_t<T, EXACT, true, UP_STORE>(c, B, l, nullptr, nullptr, nullptr);
  timing_mark(c, QDEQ_TIME_UP0, 0);
  if (u64)
    launch_up_t<T, EXACT, true, UP_ADD64>(c, B, 0, nullptr, u64, nullptr);
  else if (level0_has_f)
    launch_up_t<T, EXACT, true, UP_STORE>(c, B, 0, nullptr, nullptr, nullptr);
  else
    launch_up_t<T, EXACT, false, UP_NORM>(c, B, 0, partial, nullptr, nparts);
  timing_mark(c, QDEQ_TIME_UP0, 1);
}

void vcycle_tiled_fp64(qdeq_ctx *c, double *partial, int *nparts) {
  vcycle_tiled<double, true>(c, c->d, false, partial, nullptr, nparts);
}

void vcycle_tiled_fp32_ir(qdeq_ctx *c) {
  vcycle_tiled<float, false>(c, c->s, true, nullptr, c->d[0].u, nullptr);
}

// ---- the reference's V-cycle on the tile kernels ----
//
// Its 32 sweeps per smoothing (odeSolver.cpp:4) run as a few launches of
// several sweeps each: k_up without prolongation for the first ones of a
// descent, k_down for the last (with residual and restriction), k_up with the
// reference's prolongation (the last row left alone) for the first of the
// ascent; the levels that fit go to the tail.  Same expressions as the
// launches per half-sweep, so the same bits.  One launch per half-sweep cost
// 2.6 us each whatever the size up to 257^2 (448 of them a V-cycle at 129^2);
// here a half-sweep costs 0.2 to 0.7 us inside a launch.

// `sweeps` split into as even passes of at most `most` sweeps as there are.
static std::vector<int> split_sweeps(int sweeps, int most) {
  const int n = std::max(1, (sweeps + most - 1) / most);
  std::vector<int> v;
  for (int i = 0; i < n; i++) v.push_back(sweeps / n + (i < sweeps % n ? 1 : 0));
  return v;
}

// Tiles and passes of one level: the tile side and the sweeps per launch that
// the model finds fastest, among square tiles with a halo and, where the
// grid's quads fit one workgroup, one tile of the whole level without a halo
// and all sweeps in a launch.
template <typename T>
static bool plan_level(const qdeq_ctx *c, int l, int n_pre, int n_post, RefLevel *out) {
  const LevelDims &d = c->lv[l];
  const int most_quads = kMaxQuads<T> * TILE_THREADS;
  double best = 1e300;
  auto consider = [&](int tx, int ty, int sweeps, bool whole) {
    const std::vector<int> pre = split_sweeps(n_pre, sweeps);
    std::vector<int> post;
    if (n_post >= 0) post = split_sweeps(n_post, sweeps);
    const int tiles = ((d.K + tx - 1) / tx) * ((d.N + ty - 1) / ty);
    if (l == 0 && tiles > kPartialCap) return;
    double us = 0.0;
    for (const auto *v : {&pre, static_cast<const std::vector<int> *>(&post)})
      for (int s : *v) {
        const int H = whole ? 0 : 2 * s + 2;
        const int R = ty + 2 * H, C = tx + 2 * H, nq = (R / 2) * (C / 2);
        if (nq > most_quads || C > 5 * TX_THREADS) return;
        us += pass_us(tiles, nq, s, 1e-6 * tiles * nq * 4.0 * sizeof(T) * 4.0);
      }
    if (us < best) {
      best = us;
      *out = RefLevel{TileShape{tx, ty, TY_THREADS}, whole, pre, post};
    }
  };
  consider(d.K + (d.K & 1), d.N + (d.N & 1), std::max(1, std::max(n_pre, n_post)), true);
  for (int sweeps : {1, 2, 4, 6, 8, 11, 16})
    for (int t : {4, 6, 8, 10, 12, 14, 18, 22, 26, 30, 34, 38, 42, 46, 50, 54, 58, 62, 66})
      consider(t, t, sweeps, false);
  return best < 1e300;
}

// The plan of every level above the tail (or of all of them when the
// coarsest does not fit it), empty if some level has none.
template <typename T>
static void plan_reference(qdeq_ctx *c) {
  c->ref_plan.clear();
  if (c->cfg.cycle != QDEQ_CYCLE_REFERENCE) return;
  const int lt = tail_fits(c, sizeof(T) == 8) ? tail_entry_level(c) : c->L;
  c->ref_tail = lt;
  for (int l = 0; l < lt; l++) {
    const bool coarsest = l == c->L - 1;
    RefLevel p;
    if (!plan_level<T>(c, l, coarsest ? c->cfg.n_coarse : c->cfg.n_pre,
                       coarsest ? -1 : c->cfg.n_post, &p)) {
      c->ref_plan.clear();
      return;
    }
    // level 0 starts and ends in u: an even number of passes
    if (l == 0 && ((p.pre.size() + p.post.size()) & 1)) {
      std::vector<int> &v = p.pre;
      if (v[0] >= 2) {
        v.insert(v.begin(), v[0] / 2);
        v[1] -= v[0];
      } else {
        v.insert(v.begin(), 0);
      }
    }
    c->ref_plan.push_back(p);
  }
}

bool use_ref_tiles(const qdeq_ctx *c) { return c->ref_tiles && !c->ref_plan.empty(); }

template <typename T, bool EXACT>
static void vcycle_ref(qdeq_ctx *c, LevelBufs<T> *B, bool level0_has_f, double *partial,
                       double *u64, int *nparts) {
  const int lt = c->ref_tail;
  // pass i of a level's n writes u when an even number follows, else r, and
  // reads the other
  auto pass = [&](int l, int i, bool down) {
    const RefLevel &p = c->ref_plan[l];
    const int np = (int)p.pre.size(), n = np + (int)p.post.size();
    const int nu = i < np ? p.pre[i] : p.post[i - np];
    const bool last = i == n - 1, zero = i == 0 && (l > 0 || level0_has_f);
    const bool has_f = l > 0 || level0_has_f;
    const bool prol = i == np, add = l == 0 && last && u64;
    const bool norm = l == 0 && last && !level0_has_f;
    T *dst = ((n - 1 - i) & 1) ? B[l].r : B[l].u;
    const T *src = dst == B[l].u ? B[l].r : B[l].u;
    const int H = p.whole ? 0 : (down ? 2 * nu + 2 : up_halo(nu, norm));
    if (down) {
      run_down<T, EXACT>(c, B, l, has_f, zero, DOWN_PLAIN, p.sh, H, nu, src, dst,
                         StartArgs{});
      return;
    }
    auto up = [&](auto pr) {
      constexpr int PR = decltype(pr)::value;
      if (norm)
        *nparts = run_up<T, EXACT, false, PR, UP_NORM>(c, B, l, p.sh, H, nu, zero, src,
                                                       dst, partial, nullptr);
      else if (add)
        run_up<T, EXACT, true, PR, UP_ADD64>(c, B, l, p.sh, H, nu, zero, src, dst, nullptr,
                                             u64);
      else if (has_f)
        run_up<T, EXACT, true, PR, UP_STORE>(c, B, l, p.sh, H, nu, zero, src, dst, nullptr,
                                             nullptr);
      else
        run_up<T, EXACT, false, PR, UP_STORE>(c, B, l, p.sh, H, nu, zero, src, dst,
                                              nullptr, nullptr);
    };
    if (prol)
      up(std::integral_constant<int, PROL_REF>{});
    else
      up(std::integral_constant<int, PROL_NONE>{});
  };
  for (int l = 0; l < lt; l++) {
    const int np = (int)c->ref_plan[l].pre.size();
    for (int i = 0; i < np; i++) pass(l, i, i == np - 1 && l < c->L - 1);
  }
  if (lt < c->L) launch_tail<T, EXACT, false>(c, B, lt);
  for (int l = lt - 1; l >= 0; l--) {
    const RefLevel &p = c->ref_plan[l];
    for (int i = 0; i < (int)p.post.size(); i++) pass(l, (int)p.pre.size() + i, false);
  }
}

void vcycle_ref_fp64(qdeq_ctx *c, double *partial, int *nparts) {
  vcycle_ref<double, true>(c, c->d, false, partial, nullptr, nparts);
}

void vcycle_ref_fp32_ir(qdeq_ctx *c) {
  vcycle_ref<float, false>(c, c->s, true, nullptr, c->d[0].u, nullptr);
}

// ---- tile-shape autotuner ----

// Launches one tile kernel of level l (down or up, in the solve's mode).
template <typename T, bool EXACT>
static void launch_one(qdeq_ctx *c, LevelBufs<T> *B, int l, bool down,
                       bool level0_has_f, double *u64) {
  const bool hf = l > 0 || level0_has_f;
  if (down) {
    launch_down<T, EXACT>(c, B, l, hf, hf);
  } else if (l > 0) {
    launch_up_t<T, EXACT, true, UP_STORE>(c, B, l, nullptr, nullptr, nullptr);
  } else if (u64) {
    launch_up_t<T, EXACT, true, UP_ADD64>(c, B, 0, nullptr, u64, nullptr);
  } else {
    int nb = 0;
    launch_up_t<T, EXACT, false, UP_NORM>(c, B, 0, c->partial, nullptr, &nb);
  }
}

template <typename T, bool EXACT>
static int autotune_t(qdeq_ctx *c, LevelBufs<T> *B, bool level0_has_f,
                      double *u64, int reps) {
  const int lt = tail_entry_level(c);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  QDEQ_HIP(c, hipEventCreate(&e0));
  QDEQ_HIP(c, hipEventCreate(&e1));
  int st = QDEQ_OK;
  // an idle card takes about a millisecond of work to reach its clocks
  for (int r = 0; r < 100; r++) launch_one<T, EXACT>(c, B, 0, true, level0_has_f, u64);
  for (int l = 0; l < lt && st == QDEQ_OK; l++) {
    for (int dir = 0; dir < 2 && st == QDEQ_OK; dir++) {
      const bool down = dir == 0;
      const bool hf = l > 0 || level0_has_f;
      // every candidate's time, in a fixed order.  Among those within 3% of
      // the fastest (small levels' kernels all take as long as a launch by
      // the host) the model's best wins, the first of equals.
      std::vector<std::pair<TileShape, float>> times;
      std::vector<int> txs, tys;
      tile_candidates(c->lv[l], txs, tys);
      for (int tx : txs)
        for (int ty : tys) {
          int last_quads = 0, last_rows = 0;
          for (int tyt : kTuneTYT) {
            const TileShape cand{tx, ty, tyt};
            if (!shape_fits(c, cand, down, hf, sizeof(T))) continue;
            if (tyt > ty + 8) continue;  // more thread rows than tile rows
            // the same launch as with fewer thread rows
            const int H = down ? 2 * c->cfg.n_pre + 2
                               : up_halo(c->cfg.n_post, l == 0 && !u64 && !level0_has_f);
            const QuadLaunch<T> ql(cand, H);
            if (ql.quads == last_quads && ql.rows == last_rows) continue;
            last_quads = ql.quads;
            last_rows = ql.rows;
            const LevelDims &d = c->lv[l];
            const long blocks = (long)((d.K + tx - 1) / tx) * ((d.N + ty - 1) / ty);
            if (!down && l == 0 && !u64 && blocks > kPartialCap) continue;
            (down ? c->tdown[l] : c->tup[l]) = cand;
            launch_one<T, EXACT>(c, B, l, down, level0_has_f, u64);  // warm-up
            if (hipEventRecord(e0, c->stream) != hipSuccess) { st = QDEQ_ERR_HIP; break; }
            for (int r = 0; r < reps; r++)
              launch_one<T, EXACT>(c, B, l, down, level0_has_f, u64);
            if (hipEventRecord(e1, c->stream) != hipSuccess ||
                hipEventSynchronize(e1) != hipSuccess) { st = QDEQ_ERR_HIP; break; }
            float ms = 0.f;
            if (hipEventElapsedTime(&ms, e0, e1) != hipSuccess) { st = QDEQ_ERR_HIP; break; }
            times.emplace_back(cand, ms);
          }
        }
      if (times.empty()) continue;
      float best_ms = times[0].second;
      for (const auto &t : times) best_ms = std::min(best_ms, t.second);
      double best_us = 1e300;
      for (const auto &t : times) {
        if (t.second > 1.03f * best_ms) continue;
        const double us = shape_us<T>(c, l, down, hf, t.first);
        if (us < best_us) {
          best_us = us;
          (down ? c->tdown[l] : c->tup[l]) = t.first;
        }
      }
    }
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (st != QDEQ_OK)
    return set_error(c, st, std::string("autotune: ") + hipGetErrorString(hipGetLastError()));
  QDEQ_HIP(c, hipGetLastError());
  return QDEQ_OK;
}

// Sets the per-level shapes explicitly (validated like tuned ones).
int set_tile_shapes(qdeq_ctx *c, int nlevels, const int *shapes) {
  if (!use_tiled(c))
    return set_error(c, QDEQ_ERR_STATE, "tile shapes: the tiled fast cycle is not in use");
  const int lt = tail_entry_level(c);
  if (nlevels != lt)
    return set_error(c, QDEQ_ERR_ARG, "tile shapes: need one entry per tile level (" +
                                          std::to_string(lt) + ")");
  const bool ir = c->cfg.precision == QDEQ_PREC_FP32_IR;
  const size_t esz = ir ? 4 : 8;
  TileShape dn[QDEQ_MAX_LEVELS], up[QDEQ_MAX_LEVELS];
  for (int l = 0; l < lt; l++) {
    dn[l] = TileShape{shapes[6 * l], shapes[6 * l + 1], shapes[6 * l + 2]};
    up[l] = TileShape{shapes[6 * l + 3], shapes[6 * l + 4], shapes[6 * l + 5]};
    const bool hf = l > 0 || ir;
    if (!shape_fits(c, dn[l], true, hf, esz) || !shape_fits(c, up[l], false, hf, esz))
      return set_error(c, QDEQ_ERR_ARG, "tile shapes: level " + std::to_string(l) +
                                            " does not fit the kernels");
    const LevelDims &d = c->lv[l];
    const long blocks = (long)((d.K + up[l].tx - 1) / up[l].tx) *
                        ((d.N + up[l].ty - 1) / up[l].ty);
    if (l == 0 && !ir && blocks > kPartialCap)
      return set_error(c, QDEQ_ERR_ARG, "tile shapes: too many level-0 blocks");
  }
  for (int l = 0; l < lt; l++) {
    c->tdown[l] = dn[l];
    c->tup[l] = up[l];
  }
  c->tuned = true;
  mg_destroy_graphs(c);
  return QDEQ_OK;
}

// Times every candidate shape of each tile level's down and up kernel on the
// context's own buffers and keeps the fastest.  Any shape gives the same
// results; the level-0 displacement is saved and restored around the runs.
int autotune_tiles(qdeq_ctx *c, int reps) {
  if (!use_tiled(c))
    return set_error(c, QDEQ_ERR_STATE, "autotune: the tiled fast cycle is not in use");
  const LevelDims &d0 = c->lv[0];
  const size_t n0 = (size_t)d0.N * d0.P;
  if ((size_t)2 * c->nx * c->nz < n0)
    return set_error(c, QDEQ_ERR_STATE, "autotune: staging buffer too small");
  QDEQ_HIP(c, hipMemcpyAsync(c->stage_U, c->d[0].u, n0 * sizeof(double),
                             hipMemcpyDeviceToDevice, c->stream));
  // start from the current default shapes
  for (int l = 0; l < QDEQ_MAX_LEVELS; l++) {
    c->tdown[l] = c->tup[l] = TileShape{c->tile_tx, c->tile_ty, TY_THREADS};
  }
  c->tuned = true;
  int st;
  if (c->cfg.precision == QDEQ_PREC_FP32_IR)
    st = autotune_t<float, false>(c, c->s, true, c->d[0].u, reps);
  else
    st = autotune_t<double, true>(c, c->d, false, nullptr, reps);
  QDEQ_HIP(c, hipMemcpyAsync(c->d[0].u, c->stage_U, n0 * sizeof(double),
                             hipMemcpyDeviceToDevice, c->stream));
  QDEQ_HIP(c, hipStreamSynchronize(c->stream));
  mg_destroy_graphs(c);
  if (st != QDEQ_OK) c->tuned = false;
  return st;
}

// Average duration of each kernel of the tiled cycle launched `reps` times
// back to back in its current shape: us[0 .. lt-1] = down kernels of levels
// 0 .. lt-1, us[lt] = tail, us[lt+1 ..] = up kernels of levels lt-1 .. 0.
template <typename T, bool EXACT>
static int breakdown_t(qdeq_ctx *c, LevelBufs<T> *B, bool level0_has_f,
                       double *u64, int reps, double *us) {
  const int lt = tail_entry_level(c);
  hipEvent_t e0 = nullptr, e1 = nullptr;
  QDEQ_HIP(c, hipEventCreate(&e0));
  QDEQ_HIP(c, hipEventCreate(&e1));
  int st = QDEQ_OK;
  for (int r = 0; r < 100; r++)  // to the card's clocks, as in the tuner
    launch_one<T, EXACT>(c, B, 0, true, level0_has_f, u64);
  for (int i = 0; i < 2 * lt + 1 && st == QDEQ_OK; i++) {
    auto launch = [&]() {
      if (i < lt)
        launch_one<T, EXACT>(c, B, i, true, level0_has_f, u64);
      else if (i == lt)
        launch_tail<T, EXACT>(c, B, lt);
      else
        launch_one<T, EXACT>(c, B, 2 * lt - i, false, level0_has_f, u64);
    };
    launch();
    float ms = 0.f;
    if (hipEventRecord(e0, c->stream) != hipSuccess) st = QDEQ_ERR_HIP;
    for (int r = 0; r < reps && st == QDEQ_OK; r++) launch();
    if (st == QDEQ_OK &&
        (hipEventRecord(e1, c->stream) != hipSuccess ||
         hipEventSynchronize(e1) != hipSuccess ||
         hipEventElapsedTime(&ms, e0, e1) != hipSuccess))
      st = QDEQ_ERR_HIP;
    us[i] = 1e3 * (double)ms / reps;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (st != QDEQ_OK) return set_error(c, st, "kernel breakdown: HIP error");
  QDEQ_HIP(c, hipGetLastError());
  return QDEQ_OK;
}

int kernel_breakdown(qdeq_ctx *c, int reps, int *n, double *us) {
  if (!use_tiled(c))
    return set_error(c, QDEQ_ERR_STATE, "breakdown: the tiled fast cycle is not in use");
  const LevelDims &d0 = c->lv[0];
  const size_t n0 = (size_t)d0.N * d0.P;
  if ((size_t)2 * c->nx * c->nz < n0)
    return set_error(c, QDEQ_ERR_STATE, "breakdown: staging buffer too small");
  QDEQ_HIP(c, hipMemcpyAsync(c->stage_U, c->d[0].u, n0 * sizeof(double),
                             hipMemcpyDeviceToDevice, c->stream));
  *n = 2 * tail_entry_level(c) + 1;
  int st;
  if (c->cfg.precision == QDEQ_PREC_FP32_IR)
    st = breakdown_t<float, false>(c, c->s, true, c->d[0].u, reps, us);
  else
    st = breakdown_t<double, true>(c, c->d, false, nullptr, reps, us);
  QDEQ_HIP(c, hipMemcpyAsync(c->d[0].u, c->stage_U, n0 * sizeof(double),
                             hipMemcpyDeviceToDevice, c->stream));
  QDEQ_HIP(c, hipStreamSynchronize(c->stream));
  return st;
}

int tiled_setup(qdeq_ctx *c) {
  // Per-workgroup LDS available to dynamic allocations on this device; the
  // attribute raises the default cap where the runtime needs it.
  int dev = 0, optin = 0;
  hipDeviceProp_t prop;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipGetDeviceProperties(&prop, dev) == hipSuccess)
    c->lds_max = prop.sharedMemPerBlock;
  if (hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin,
                            dev) == hipSuccess &&
      (size_t)optin > c->lds_max)
    c->lds_max = (size_t)optin;
  const int big = (int)c->lds_max;
#define SETA(kern)                                                       \
  (void)hipFuncSetAttribute((const void *)(kern),                        \
                            hipFuncAttributeMaxDynamicSharedMemorySize, big)
  with_quads_all<double>([&](auto quads) {
    constexpr int S = decltype(quads)::value;
    SETA((k_down<double, true, true, DOWN_PLAIN, S>));
    SETA((k_down<double, false, true, DOWN_PLAIN, S>));
    SETA((k_down<double, false, true, START_PARTIALS, S>));
    SETA((k_down<double, true, true, START_TEST, S>));
    SETA((k_up<double, true, true, PROL_FULL, UP_STORE, S>));
    SETA((k_up<double, false, true, PROL_FULL, UP_NORM, S>));
    SETA((k_up<double, true, true, PROL_REF, UP_STORE, S>));
    SETA((k_up<double, true, true, PROL_NONE, UP_STORE, S>));
    SETA((k_up<double, false, true, PROL_REF, UP_STORE, S>));
    SETA((k_up<double, false, true, PROL_NONE, UP_STORE, S>));
    SETA((k_up<double, false, true, PROL_REF, UP_NORM, S>));
    SETA((k_up<double, false, true, PROL_NONE, UP_NORM, S>));
  });
  with_quads_all<float>([&](auto quads) {
    constexpr int S = decltype(quads)::value;
    SETA((k_down<float, true, false, DOWN_PLAIN, S>));
    SETA((k_up<float, true, false, PROL_FULL, UP_STORE, S>));
    SETA((k_up<float, true, false, PROL_FULL, UP_ADD64, S>));
    SETA((k_up<float, true, false, PROL_REF, UP_STORE, S>));
    SETA((k_up<float, true, false, PROL_NONE, UP_STORE, S>));
    SETA((k_up<float, true, false, PROL_REF, UP_ADD64, S>));
    SETA((k_up<float, true, false, PROL_NONE, UP_ADD64, S>));
  });
  SETA((k_coarse_rows<double>));
  SETA((k_coarse_rows<float>));
  SETA((k_tail_direct<double, true>));
  SETA((k_tail_direct<float, false>));
  SETA((k_tail<double, true, true>));
  SETA((k_tail<float, false, true>));
  SETA((k_tail<double, true, false>));
  SETA((k_tail<float, false, false>));
#undef SETA
  (void)hipGetLastError();
  if (!tiles_fit(c, c->tile_tx, c->tile_ty)) c->tiled = false;
  if (c->cfg.precision == QDEQ_PREC_FP32_IR) {
    model_shapes<float>(c);
    plan_reference<float>(c);
  } else {
    model_shapes<double>(c);
    plan_reference<double>(c);
  }
  return QDEQ_OK;
}

}  // namespace qdeq
