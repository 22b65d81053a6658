// Differentiable periodic box: one PIC step and its adjoint (reverse mode).
//
// Forward.  The discrete step of one lap of projects/pic-turbulence/pic.py:187-221
// on a single periodic box, with the expression order of the reference
// kernels (and of the tile path), compiled with -ffp-contract=off:
//   B1 = B + (cfl/2) curlE(E)                       emf/yee_lattice_fdtd2.c++:19-58
//   per particle: E, B at x (node means + lerp3D)   emf/yee_lattice_interpolate_linear_1st.h:29-138
//                 Boris: u', x' = x + cfl u'/gamma'  pic/particle_boris.h:15-62
//                 x'' = periodic wrap of x'          pic/tile_communication.c++:98-117
//                 zigzag deposit of (x'', u') -> J   pic/particle_current_zigzag_1st.c++:225-339
//   Jf = binomial2^P(J) (periodic)                  emf/yee_lattice_current_filter_binomial2.c++:23-76
//   B2 = B1 + (cfl/2) curlE(E)
//   E' = E + cfl curlB(B2) - Jf                     emf/yee_lattice_fdtd2.c++:68-111, yee_lattice.c++:170-179
// On a periodic box the tile halos, J_exchange and the copies between filter
// passes reduce to periodic indexing, so a step gives the tile path's particles
// bit for bit and its J up to rounding: of the order of the deposit's sums, and
// of the filter, whose passes are summed axis by axis (k_dfilter) instead of as
// the reference's 27 taps.
//
// Adjoint.  Vector-Jacobian products of each stage, in reverse order.  The
// discrete curls are negative transposes of each other (curlE^T = -curlB),
// the periodic binomial stencil is symmetric (F^T = F), so the field part
// reuses the forward stencils with negated time steps.  The particle part is
// one kernel per particle that recomputes its forward step and then applies,
// by hand-derived chain rule:
//   the deposit adjoint  (gather of lambda_J at the 24 zigzag nodes),
//   the position update and Boris Jacobian-transposes,
//   the interpolation adjoint (scatter of lambda_E, lambda_B to node-mean
//   adjoints, then one grid pass maps node means back to the staggered
//   components) and the gradient of the weights in x.
// The particle part of both directions runs brick by brick out of LDS (see
// "particles by brick" below).
// Floors, the zigzag relay point's branch and the wrap are piecewise
// constant / identity, so their derivatives are taken on the branch the
// forward step took.
#include "rk_internal.h"

#include <algorithm>
#include <cmath>

namespace rk {

namespace {

constexpr int DWG = 256;

template<class T>
struct DBox {
  int n[3];
  int nsp;
  int64_t off[RK_MAX_SPECIES + 1];  // species s holds particles [off[s], off[s+1])
  T q[RK_MAX_SPECIES];
  T qm[RK_MAX_SPECIES];
  T cfl;
};

template<class T>
struct G3 {
  T* c[3];
};

// A magic is ceil(2^40 / d): x * magic / 2^40 floors to x / d for x < 2^28.
struct Axis {
  int n, nb;
  uint64_t per_n, per_nb;  // magics of n and nb
};

// one box of an ensemble: its geometry and where its cells and particles
// start in the concatenated arrays (a single box is an ensemble of one)
template<class T>
struct DEnt {
  DBox<T> b;
  int64_t c0, p0;
  int64_t pb0;  // first particle block
  Axis ax[3];   // cells and bricks of each axis
  int64_t k0;   // first global brick number
  // runs of the sorted particle blocks: one row of rowlen words (two 16-bit
  // run starts each) per particle block, one run per group of 2^gsh bricks per axis
  int gsh;
  int ng[3];
  int ngroup, rowlen;
  int64_t nrow, row0;
};

template<class T>
__device__ inline G3<T> sh(G3<T> g, int64_t o)
{
#pragma unroll
  for(int c = 0; c < 3; ++c)
    if(g.c[c]) g.c[c] += o;
  return g;
}

__host__ __device__ inline int64_t cidx(const int n[3], int i, int j, int k)
{
  return (int64_t(i) * n[1] + j) * n[2] + k;
}

__device__ inline int wrap1(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

template<class T>
__device__ inline T dot3d(const T a[3], const T b[3])
{
  T r = a[0] * b[0];
  r = r + a[1] * b[1];
  r = r + a[2] * b[2];
  return r;
}

template<class T>
__device__ inline void cross3d(const T a[3], const T b[3], T r[3])
{
  r[0] = a[1] * b[2] - a[2] * b[1];
  r[1] = -a[0] * b[2] + a[2] * b[0];
  r[2] = a[0] * b[1] - a[1] * b[0];
}

template<class T>
__device__ inline T lerp_d(T x, T A, T B)
{
  return (T(1) - x) * A + x * B;
}

template<class T>
__device__ inline T lerp3_d(const T d[3], const T m[2][2][2])
{
  const T c00 = lerp_d(d[0], m[0][0][0], m[1][0][0]);
  const T c01 = lerp_d(d[0], m[0][0][1], m[1][0][1]);
  const T c10 = lerp_d(d[0], m[0][1][0], m[1][1][0]);
  const T c11 = lerp_d(d[0], m[0][1][1], m[1][1][1]);
  const T c0 = lerp_d(d[1], c00, c10);
  const T c1 = lerp_d(d[1], c01, c11);
  return lerp_d(d[2], c0, c1);
}

template<class T>
__device__ inline void atomic_add(T* p, T v)
{
  unsafeAtomicAdd(p, v);
}

// ---------------------------------------------------------------- field stencils
// out = in + dt * curlE(E)   (push_b_fdtd2 order; out may alias in); clears
// the planar field Z when it is given
template<class T>
struct CurlB {
  G3<T> out, in, E;
  T dt;
  G3<T> Z;
};

// The grid of a per-box launch (grid_of, block_of) as part of a launch of 1D
// workgroups of DWG threads (at most MERGED_BLOCKS of them, see merged()).
struct BoxGrid {
  int gx, gy, gz, bx, by;
  int seg;  // workgroups that share a row (few, long rows)
  __host__ __device__ int blocks() const { return gx * gy * gz; }
};
struct BoxPlace {
  int z, i, j, tx, step;
  bool ok;
};
__device__ inline BoxPlace place(const BoxGrid& g, int blk)
{
  const int tid = int(threadIdx.x), ty = tid / g.bx, x = blk % g.gx, q = blk / g.gx;
  return BoxPlace {q / g.gy, q % g.gy, x / g.seg * g.by + ty, x % g.seg * g.bx + tid - ty * g.bx, g.seg * g.bx, ty < g.by};
}

// the nodes (i, j, k), k = tx, tx + bx, ..., of a box
template<class T>
__device__ inline void curl_b_row(const DEnt<T>& en, const CurlB<T>& u, int i, int j, int tx, int bx)
{
  const DBox<T>& b = en.b;
  if(j >= b.n[1] || i >= b.n[0]) return;
  const G3<T> out = sh(u.out, en.c0);
  const G3<T> in = sh(u.in, en.c0);
  const G3<T> E = sh(u.E, en.c0);
  const int n0 = b.n[0], n1 = b.n[1], n2 = b.n[2];
  const int ip = wrap1(i + 1, n0), jp = wrap1(j + 1, n1);
  for(int k = tx; k < n2; k += bx) {
    const int kp = wrap1(k + 1, n2);
    const int64_t c = cidx(b.n, i, j, k);
    const T DkEy = E.c[1][cidx(b.n, i, j, kp)] - E.c[1][c];
    const T DjEz = E.c[2][cidx(b.n, i, jp, k)] - E.c[2][c];
    const T DiEz = E.c[2][cidx(b.n, ip, j, k)] - E.c[2][c];
    const T DkEx = E.c[0][cidx(b.n, i, j, kp)] - E.c[0][c];
    const T DjEx = E.c[0][cidx(b.n, i, jp, k)] - E.c[0][c];
    const T DiEy = E.c[1][cidx(b.n, ip, j, k)] - E.c[1][c];
    out.c[0][c] = in.c[0][c] + u.dt * (DkEy - DjEz);
    out.c[1][c] = in.c[1][c] + u.dt * (DiEz - DkEx);
    out.c[2][c] = in.c[2][c] + u.dt * (DjEx - DiEy);
    if(u.Z.c[0])
#pragma unroll
      for(int q = 0; q < 3; ++q) u.Z.c[q][en.c0 + c] = T(0);
  }
}

template<class T>
__global__ void __launch_bounds__(DWG) k_dcurl_b(const DEnt<T>* __restrict__ tab, CurlB<T> u)
{
  curl_b_row(tab[blockIdx.z], u, int(blockIdx.y), int(blockIdx.x * blockDim.y + threadIdx.y), int(threadIdx.x),
             int(blockDim.x));
}

// out = in + dt * curlB(B), then out -= J when J is given (push_e_fdtd2 +
// add_current order; out may alias in, not B)
template<class T>
__global__ void __launch_bounds__(DWG)
  k_dcurl_e(const DEnt<T>* __restrict__ tab, G3<T> out, G3<T> in, G3<T> B, T dt, G3<T> J)
{
  const DEnt<T>& en = tab[blockIdx.z];
  const DBox<T>& b = en.b;
  const int j = int(blockIdx.x * blockDim.y + threadIdx.y), i = int(blockIdx.y);
  if(j >= b.n[1] || i >= b.n[0]) return;
  out = sh(out, en.c0);
  in = sh(in, en.c0);
  B = sh(B, en.c0);
  J = sh(J, en.c0);
  const int n0 = b.n[0], n1 = b.n[1], n2 = b.n[2];
  const int im = wrap1(i - 1, n0), jm = wrap1(j - 1, n1);
  for(int k = int(threadIdx.x); k < n2; k += int(blockDim.x)) {
    const int km = wrap1(k - 1, n2);
    const int64_t c = cidx(b.n, i, j, k);
    const T DkBy = B.c[1][cidx(b.n, i, j, km)] - B.c[1][c];
    const T DjBz = B.c[2][cidx(b.n, i, jm, k)] - B.c[2][c];
    const T DiBz = B.c[2][cidx(b.n, im, j, k)] - B.c[2][c];
    const T DkBx = B.c[0][cidx(b.n, i, j, km)] - B.c[0][c];
    const T DjBx = B.c[0][cidx(b.n, i, jm, k)] - B.c[0][c];
    const T DiBy = B.c[1][cidx(b.n, im, j, k)] - B.c[1][c];
    T e0 = in.c[0][c] + dt * (DkBy - DjBz);
    T e1 = in.c[1][c] + dt * (DiBz - DkBx);
    T e2 = in.c[2][c] + dt * (DjBx - DiBy);
    if(J.c[0]) {
      e0 = e0 - J.c[0][c];
      e1 = e1 - J.c[1][c];
      e2 = e2 - J.c[2][c];
    }
    out.c[0][c] = e0;
    out.c[1][c] = e1;
    out.c[2][c] = e2;
  }
}

// R binomial2 passes (yee_lattice_current_filter_binomial2.c++:23-76) of a
// periodic box in one pass over memory: the passes are separable and commute,
// so together they are (2R+1)-tap binomials along z, y and x.  That is another
// rounding than the reference's 27 taps a pass, whose weights are powers of two
// (products with 6, 15 and 20 sixty-fourths round, so they are fused with their
// sums), and no worse: three FP32 passes against 64 bits 7.6e-8 on a current (27
// taps 9.3e-8; unfused 8.3e-8), 8.9e-8 on noise, as an adjoint may be (9.4e-8;
// 9.8e-8).  A workgroup
// owns FY x FZ columns of nodes of one component and marches over xseg planes:
// each arriving plane is staged in LDS with R nodes around the tile, summed
// along z (four nodes a thread, which share their reads) and then along y (four
// nodes a thread, one wave), and kept in registers for the 2R+1 sums along x
// that take it; the next plane's loads are in flight meanwhile.  LDS reads bound
// it on large boxes: 22.3 us on 96^3 cells (66 us as three 27-tap launches); on
// small ones the chain of a plane's two barriers does, shorter with a component
// a workgroup than with all three in one of 256 threads: 16^3 12.7 -> 9.4 us.
constexpr int FY = 8, FZ = 32, FT = 128;

template<class T, int R>
struct Taps {
  T w[R + 1];  // outermost first
};

template<class T, int R>
__device__ constexpr Taps<T, R> taps()
{
  if constexpr(R == 3) return {{T(1. / 64.), T(6. / 64.), T(15. / 64.), T(20. / 64.)}};
  else if constexpr(R == 2) return {{T(1. / 16.), T(4. / 16.), T(6. / 16.)}};
  else return {{T(1. / 4.), T(2. / 4.)}};
}

__device__ inline float fused(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ inline double fused(double a, double b, double c) { return __builtin_fma(a, b, c); }

template<class T, int R, int N>
__device__ inline T tap_sum(const T (&v)[N], int o)
{
  constexpr Taps<T, R> t = taps<T, R>();
  T s = t.w[R] * v[o + R];
#pragma unroll
  for(int k = R - 1; k >= 0; --k) s = fused(t.w[k], v[o + k] + v[o + 2 * R - k], s);
  return s;
}

template<class T, int R>
__global__ void __launch_bounds__(FT)
  k_dfilter(const DEnt<T>* __restrict__ tab, G3<T> out, G3<T> in, int tiles_z, int xseg)
{
  constexpr int IY = FY + 2 * R, IZ = FZ + 2 * R, NI = IY * IZ, NM = (NI + FT - 1) / FT;
  constexpr int PZ = (IZ + 3) / 4 * 4, ZG = FZ / 4, TASKS = IY * ZG;
  static_assert(TASKS <= FT && 2 * FZ <= FT && FY == 8, "a task a thread");
  __shared__ alignas(32) T pl[2][IY * PZ];
  __shared__ alignas(32) T zs[2][IY * FZ];
  const DEnt<T>& en = tab[blockIdx.z];
  const DBox<T>& b = en.b;
  const int comp = int(blockIdx.x) % 3, tile = int(blockIdx.x) / 3;
  const int j0 = tile / tiles_z * FY, k0 = tile % tiles_z * FZ, i0 = int(blockIdx.y) * xseg;
  if(i0 >= b.n[0] || j0 >= b.n[1] || k0 >= b.n[2]) return;  // uniform over the workgroup
  const int i1 = min(i0 + xseg, b.n[0]);
  const T* __restrict__ const src = (comp == 0 ? in.c[0] : (comp == 1 ? in.c[1] : in.c[2])) + en.c0;
  T* __restrict__ const dst = (comp == 0 ? out.c[0] : (comp == 1 ? out.c[1] : out.c[2])) + en.c0;
  const int tid = int(threadIdx.x);
  auto wrapm = [](int i, int n) {
    while(i < 0) i += n;
    while(i >= n) i -= n;
    return i;
  };
  int off[NM], at[NM];
#pragma unroll
  for(int m = 0; m < NM; ++m) {
    const int e = min(tid + m * FT, NI - 1);  // (the last threads repeat the last node)
    off[m] = wrapm(j0 - R + e / IZ, b.n[1]) * b.n[2] + wrapm(k0 - R + e % IZ, b.n[2]);
    at[m] = e / IZ * PZ + e % IZ;
  }
  T pre[NM];
  auto load = [&](int i) {
    const T* const plane = src + int64_t(wrapm(i, b.n[0])) * b.n[1] * b.n[2];
#pragma unroll
    for(int m = 0; m < NM; ++m) pre[m] = plane[off[m]];
  };
  T ring[4][2 * R + 1] = {};
  const int ty = tid / FZ * 4, tz = tid % FZ;  // the y and x sums: threads 0..63
  load(i0 - R);
  for(int i = i0 - R; i < i1 + R; ++i) {
    const int cur = i & 1;
#pragma unroll
    for(int m = 0; m < NM; ++m) pl[cur][at[m]] = pre[m];
    if(i + 1 < i1 + R) load(i + 1);
    __syncthreads();
    if(tid < TASKS) {
      const int row = tid / ZG, zg = tid % ZG;
      const T* p = &pl[cur][row * PZ + zg * 4];
      T v[4 + 2 * R];
#pragma unroll
      for(int k = 0; k < 4 + 2 * R; ++k) v[k] = p[k];
#pragma unroll
      for(int k = 0; k < 4; ++k) zs[cur][row * FZ + zg * 4 + k] = tap_sum<T, R>(v, k);
    }
    __syncthreads();
    if(tid < 2 * FZ) {
      T v[4 + 2 * R];
#pragma unroll
      for(int k = 0; k < 4 + 2 * R; ++k) v[k] = zs[cur][(ty + k) * FZ + tz];
#pragma unroll
      for(int y = 0; y < 4; ++y) {
#pragma unroll
        for(int k = 0; k < 2 * R; ++k) ring[y][k] = ring[y][k + 1];
        ring[y][2 * R] = tap_sum<T, R>(v, y);
        if(i >= i0 + R && j0 + ty + y < b.n[1] && k0 + tz < b.n[2])
          dst[cidx(b.n, i - R, j0 + ty + y, k0 + tz)] = tap_sum<T, R>(ring[y], 0);
      }
    }
  }
}

// ---------------------------------------------------------------- bricks
// Brick k of an axis with n cells and nb bricks holds the cells
// [k n / nb, (k+1) n / nb): sizes differ by at most one, and a brick has at
// most BR cells per axis.
__device__ inline int brick_start(const Axis& a, int k) { return int((uint64_t(uint32_t(k * a.n)) * a.per_nb) >> 40); }

// brick of cell i: the largest k with k n / nb <= i, ((i+1) nb - 1) / n
__device__ inline int brick_at(const Axis& a, int i)
{
  return int((uint64_t(uint32_t((i + 1) * a.nb - 1)) * a.per_n) >> 40);
}

// The windows (of LO nodes before a brick's cells to HI after them) that hold
// node i of one axis: its own brick's and a neighbour's (ok), or, on bricks of
// fewer than LO + HI cells, those of both neighbours (both).
struct Cov {
  bool ok, both;
  int brick[3], off[3];
};

template<int LO, int HI>
__device__ inline Cov covers(const Axis& a, int i)
{
  Cov c;
  const int k = brick_at(a, i), s = brick_start(a, k), e = brick_start(a, k + 1);
  const int kl = k == 0 ? a.nb - 1 : k - 1, kr = k == a.nb - 1 ? 0 : k + 1;
  const bool left = i - s < HI, right = e - i <= LO;
  const int ol = brick_start(a, kl + 1) - brick_start(a, kl) + LO + i - s, or_ = LO - (e - i);
  c.ok = left || right;
  c.both = left && right;
  c.brick[0] = k;
  c.off[0] = i - s + LO;
  // without a neighbour's window the own one stands in (read, not added)
  c.brick[1] = left ? kl : (right ? kr : k);
  c.off[1] = left ? ol : (right ? or_ : i - s + LO);
  c.brick[2] = kr;
  c.off[2] = or_;
  return c;
}

// sum of the NC components of node (i, j, k) over the windows (W nodes per
// axis) that hold it.  A node lies in at most eight windows as a rule: their
// loads are issued together, the absent ones on the own window and not added
// (k_djgather on 96^3 30.8 -> 26.3 us, on 16^3 7.8 -> 4.0 us; a chain of loads before).
// THIRD: bricks of two cells along an axis may put a node in a third window
// there; then up to three at a time (2 x 2 x 4096 cells, k_dfinish: 196 us in a
// chain by a workgroup a row, 120 us so, 10 us with sixteen workgroups a row).
template<class T, int NC, int W, bool THIRD>
__device__ inline void sum_windows(const DEnt<T>& en, const Cov& ci, const Cov& cj, const Cov& ck,
                                   const T* __restrict__ st, T (&sum)[NC])
{
  constexpr int V = W * W * W;
  auto window = [&](int x, int y, int z) {
    const int64_t br = (int64_t(ci.brick[x]) * en.ax[1].nb + cj.brick[y]) * en.ax[2].nb + ck.brick[z];
    return st + br * (NC * V) + (ci.off[x] * W + cj.off[y]) * W + ck.off[z];
  };
#pragma unroll
  for(int q = 0; q < NC; ++q) sum[q] = T(0);
  if(!THIRD || !(ci.both || cj.both || ck.both)) {
    T v[8][NC];
#pragma unroll
    for(int m = 0; m < 8; ++m) {
      const T* w = window(m >> 2, m >> 1 & 1, m & 1);
#pragma unroll
      for(int q = 0; q < NC; ++q) v[m][q] = w[q * V];
    }
#pragma unroll
    for(int m = 0; m < 8; ++m) {
      const bool in = (!(m & 4) || ci.ok) && (!(m & 2) || cj.ok) && (!(m & 1) || ck.ok);
#pragma unroll
      for(int q = 0; q < NC; ++q) {
        const T t = sum[q] + v[m][q];
        sum[q] = in ? t : sum[q];
      }
    }
    return;
  }
  if constexpr(THIRD) {
    auto held = [](const Cov& c, int o) { return o == 0 || (o == 1 ? c.ok : c.both); };
    auto pick = [](const int (&v)[3], int o) { return o == 0 ? v[0] : (o == 1 ? v[1] : v[2]); };
#pragma unroll 1
    for(int m = 0; m < 9; ++m) {
      const int x = m / 3, y = m % 3;
      if(!held(ci, x) || !held(cj, y)) continue;
      const int64_t row = (int64_t(pick(ci.brick, x)) * en.ax[1].nb + pick(cj.brick, y)) * en.ax[2].nb;
      const int at = (pick(ci.off, x) * W + pick(cj.off, y)) * W;
      T v[3][NC];
#pragma unroll
      for(int z = 0; z < 3; ++z) {
        const int k = held(ck, z) ? z : 0;
        const T* w = st + (row + pick(ck.brick, k)) * (NC * V) + at + pick(ck.off, k);
#pragma unroll
        for(int q = 0; q < NC; ++q) v[z][q] = w[q * V];
      }
#pragma unroll
      for(int z = 0; z < 3; ++z)
#pragma unroll
        for(int q = 0; q < NC; ++q) {
          const T t = sum[q] + v[z][q];
          sum[q] = held(ck, z) ? t : sum[q];
        }
    }
  }
}

// lambda_E += the bricks' windows of E adjoints (components 0..2 of mst),
// lambda_B1 = lambda_B2 + their windows of B adjoints (3..5)
template<class T, int BR>
__device__ inline void mgather_row(const DEnt<T>& en, G3<T> LE, G3<T> LB, G3<T> LBout, const T* __restrict__ mst, int i,
                                   int j, int tx, int bx)
{
  constexpr int W = BR + 2, V = W * W * W;
  const DBox<T>& b = en.b;
  if(j >= b.n[1] || i >= b.n[0]) return;
  mst += en.k0 * (6 * V);
  const Cov ci = covers<1, 1>(en.ax[0], i);
  const Cov cj = covers<1, 1>(en.ax[1], j);
  for(int k = tx; k < b.n[2]; k += bx) {
    const Cov ck = covers<1, 1>(en.ax[2], k);
    T s[6];
    sum_windows<T, 6, W, false>(en, ci, cj, ck, mst, s);
    const int64_t c = en.c0 + cidx(b.n, i, j, k);
#pragma unroll
    for(int q = 0; q < 3; ++q) {
      LE.c[q][c] += s[q];
      LBout.c[q][c] = LB.c[q][c] + s[3 + q];
    }
  }
}

template<class T, int BR>
__global__ void __launch_bounds__(DWG)
  k_dmgather(const DEnt<T>* __restrict__ tab, G3<T> LE, G3<T> LB, G3<T> LBout, const T* __restrict__ mst)
{
  mgather_row<T, BR>(tab[blockIdx.z], LE, LB, LBout, mst, int(blockIdx.y), int(blockIdx.x * blockDim.y + threadIdx.y),
                     int(threadIdx.x), int(blockDim.x));
}

// J += the bricks' current windows (jst, three components per brick).  J was
// cleared before the particle step; it holds only contributions that missed
// their brick's window.
template<class T, int BR>
__device__ inline void jgather_row(const DEnt<T>& en, G3<T> J, const T* __restrict__ jst, int i, int j, int tx, int bx)
{
  constexpr int D = BR + 3, V = D * D * D;
  const DBox<T>& b = en.b;
  if(j >= b.n[1] || i >= b.n[0]) return;
  J = sh(J, en.c0);
  jst += en.k0 * (3 * V);
  const Cov ci = covers<1, 2>(en.ax[0], i);
  const Cov cj = covers<1, 2>(en.ax[1], j);
  for(int k = tx; k < b.n[2]; k += bx) {
    const Cov ck = covers<1, 2>(en.ax[2], k);
    T s[3];
    sum_windows<T, 3, D, true>(en, ci, cj, ck, jst, s);
    const int64_t c = cidx(b.n, i, j, k);
#pragma unroll
    for(int q = 0; q < 3; ++q) J.c[q][c] += s[q];
  }
}

template<class T, int BR>
__global__ void __launch_bounds__(DWG)
  k_djgather(const DEnt<T>* __restrict__ tab, G3<T> J, const T* __restrict__ jst)
{
  jgather_row<T, BR>(tab[blockIdx.z], J, jst, int(blockIdx.y), int(blockIdx.x * blockDim.y + threadIdx.y),
                     int(threadIdx.x), int(blockDim.x));
}

// ---------------------------------------------------------------- particles
// forward quantities of one particle's step that its adjoint reuses
template<class T>
struct Fwd {
  T d[3];             // intra-cell offsets of the interpolation
  T EBE[3], EBB[3];   // interpolated fields
  T xn[3], un[3];     // position after the push (before the wrap), momentum
  T xw[3];            // wrapped position
};

template<class T>
__device__ inline bool in_box(const DBox<T>& b, const T x[3])
{
  // the stencils below address cells -1 .. n+1 around the box
  return x[0] >= T(-1) && x[0] <= T(b.n[0] + 1) && x[1] >= T(-1) && x[1] <= T(b.n[1] + 1) && x[2] >= T(-1) &&
         x[2] <= T(b.n[2] + 1);
}

template<class T>
struct BorisT {
  T v0[3], E0[3], u0[3], g, bfac, B0[3], f, w[3], u1[3], u2[3];
};

template<class T>
__device__ inline void boris_fwd(const T cfl, const T qm, const T EBE[3], const T EBB[3], const T x[3],
                                 const T vel[3], BorisT<T>& s, T xn[3], T un[3])
{
  const T hq = T(0.5) * qm;
#pragma unroll
  for(int c = 0; c < 3; ++c) s.v0[c] = vel[c] * cfl;
#pragma unroll
  for(int c = 0; c < 3; ++c) s.E0[c] = EBE[c] * hq;
#pragma unroll
  for(int c = 0; c < 3; ++c) s.u0[c] = s.v0[c] + s.E0[c];
  s.g = cfl / sqrt(cfl * cfl + dot3d(s.u0, s.u0));
  s.bfac = hq * s.g;
#pragma unroll
  for(int c = 0; c < 3; ++c) s.B0[c] = (EBB[c] * s.bfac) / cfl;
  s.f = T(2) / (T(1) + dot3d(s.B0, s.B0));
  T cr[3];
  cross3d(s.u0, s.B0, cr);
#pragma unroll
  for(int c = 0; c < 3; ++c) s.w[c] = s.u0[c] + cr[c];
#pragma unroll
  for(int c = 0; c < 3; ++c) s.u1[c] = s.w[c] * s.f;
  cross3d(s.u1, s.B0, cr);
#pragma unroll
  for(int c = 0; c < 3; ++c) s.u2[c] = (s.u0[c] + cr[c]) + s.E0[c];
#pragma unroll
  for(int c = 0; c < 3; ++c) un[c] = s.u2[c] / cfl;
  const T ginv2 = cfl / sqrt(cfl * cfl + dot3d(s.u2, s.u2));
#pragma unroll
  for(int c = 0; c < 3; ++c) xn[c] = x[c] + (un[c] * ginv2) * cfl;
}

template<class T>
__device__ inline void wrap_pos(const DBox<T>& b, const T xn[3], T xw[3])
{
  // leavers get (x < 0 ? L : 0) + fmod(x, L); |x| < 2L here, so fmod is x or x - L
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    const T L = T(b.n[a]);
    const T v = xn[a];
    xw[a] = v < T(0) ? L + v : (v >= L ? v - L : v);
  }
}

// zigzag geometry of one particle (particle_current_zigzag_1st.c++:225-339)
template<class T>
struct Zig {
  T x1[3], x2[3], fi1[3], fi2[3], xr[3], F1[3], F2[3], W1[3], W2[3];
  bool mid[3];   // relay point on its (x1+x2)/2 branch
  int i1[3], i2[3];  // cells of the segments, on the axes of xw (not wrapped)
  T s, invgam;
};

template<class T>
__device__ inline void zig_setup(const DBox<T>& b, const T xw[3], const T u[3], T charge, Zig<T>& z)
{
  const T one = T(1);
  z.invgam = one / sqrt(one + dot3d(u, u));
  z.s = b.cfl * z.invgam;
#pragma unroll
  for(int d = 0; d < 3; ++d) {
    z.x2[d] = xw[d] + T(3);
    z.x1[d] = z.x2[d] - u[d] * z.s;
    z.fi1[d] = floor(z.x1[d]);
    z.fi2[d] = floor(z.x2[d]);
    const T a = (z.fi1[d] < z.fi2[d] ? z.fi1[d] : z.fi2[d]) + one;
    const T b1 = (z.fi1[d] > z.fi2[d] ? z.fi1[d] : z.fi2[d]);
    const T b2 = T(0.5) * (z.x1[d] + z.x2[d]);
    const T bb = (b1 > b2 ? b1 : b2);
    z.xr[d] = (a < bb ? a : bb);
    z.mid[d] = !(b1 > b2) && !(a < bb);
    z.F1[d] = (z.xr[d] - z.x1[d]) * charge;
    z.F2[d] = (z.x2[d] - z.xr[d]) * charge;
    z.W1[d] = (z.x1[d] + z.xr[d]) * T(0.5) - z.fi1[d];
    z.W2[d] = (z.x2[d] + z.xr[d]) * T(0.5) - z.fi2[d];
    z.i1[d] = int(static_cast<uint32_t>(z.fi1[d])) - 3;
    z.i2[d] = int(static_cast<uint32_t>(z.fi2[d])) - 3;
  }
}

// the 7 (node, component) contributions of one segment, in store order:
// v[m][c] goes to node (c[0][o0], c[1][o1], c[2][o2]) with offsets ZOFF[m]
static __device__ constexpr int ZOFF[7][3] = {{0, 0, 0}, {1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {0, 1, 1}, {1, 0, 1}, {1, 1, 0}};

template<class T>
__device__ inline void zig_values(const T F[3], const T W[3], T v[7][3])
{
  const T one = T(1);
  v[0][0] = F[0] * (one - W[1]) * (one - W[2]);
  v[0][1] = F[1] * (one - W[0]) * (one - W[2]);
  v[0][2] = F[2] * (one - W[0]) * (one - W[1]);
  v[1][0] = T(0);
  v[1][1] = F[1] * W[0] * (one - W[2]);
  v[1][2] = F[2] * W[0] * (one - W[1]);
  v[2][0] = F[0] * W[1] * (one - W[2]);
  v[2][1] = T(0);
  v[2][2] = F[2] * (one - W[0]) * W[1];
  v[3][0] = F[0] * (one - W[1]) * W[2];
  v[3][1] = F[1] * (one - W[0]) * W[2];
  v[3][2] = T(0);
  v[4][0] = F[0] * W[1] * W[2];
  v[4][1] = T(0);
  v[4][2] = T(0);
  v[5][0] = T(0);
  v[5][1] = F[1] * W[0] * W[2];
  v[5][2] = T(0);
  v[6][0] = T(0);
  v[6][1] = T(0);
  v[6][2] = F[2] * W[0] * W[1];
}

// whether v[m][c] is structurally non-zero
__host__ __device__ constexpr bool zig_has(int m, int c)
{
  return m == 0 || (m < 4 ? c != m - 1 : c == m - 4);
}

template<class T>
__device__ inline int species_of(const DBox<T>& b, int64_t p)
{
  int s = 0;
  while(s + 1 < b.nsp && p >= b.off[s + 1]) ++s;
  return s;
}

// ---------------------------------------------------------------- particles by brick
// The state's particles keep their places in the arrays and mix over the box,
// so reading the 8 corner nodes and adding the current per particle touches
// memory at random: about 40 cache lines and an atomic or two per particle
// and step.  Instead every particle visits LDS once, in three passes:
//   k_dbin     a block takes P consecutive particles, counts them by brick in
//              LDS and writes them as 8-word records, sorted by brick, into
//              its own P slots; a row of run starts (one per brick) beside them;
//   k_dstep / k_dadj   a workgroup per brick walks its run of every row with
//              the brick's node means (and, for the adjoint, the current's
//              adjoint) in LDS, and sums its current (node-mean adjoints)
//              there in double precision; each record's result replaces it;
//   k_dunsort  a block puts its P records back in the arrays' order.
// The sort never leaves a block, so records move only inside P slots that
// stay in cache, with no global atomic and no scan over bricks (boxes of more
// than GROUPS_MAX bricks need both, see k_dcount).  About 220
// bytes per particle and step cross memory; the pass over 96^3 cells with 2.8e7
// mixed particles takes 2.3 ms (7.3 ms with random corner reads, records
// bucketed by cell through global counters and a scan), its adjoint 3.8 ms
// (12.1 ms).  Measured there: k_dbin 0.66 (adjoint 1.46), k_dstep 1.15 (vector
// issue and LDS adds, about half of the cycles each), k_dadj 1.89 (LDS adds),
// k_dunsort 0.49 ms.
template<class T>
struct alignas(8 * sizeof(T)) Rec {
  T v[8];  // x, u, species, unused; or the adjoint's lambda_x, lambda_u
};

// position -> cell of one axis (the interpolation's base cell, not wrapped) and offset in it
template<class T>
__device__ inline int base_cell(T x, T& d)
{
  const T p = x + T(3);  // x - origo, origo = mins - halo = -3
  const uint32_t ii = static_cast<uint32_t>(p);
  d = p - static_cast<T>(ii);
  return int(ii) - 3;
}

__device__ inline int wrap2(int i, int n) { return wrap1(wrap1(i, n), n); }

template<class T, int K, bool ADJ>
__device__ __forceinline__ void
bin_block(int block, const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, G3<T> x, G3<T> u, G3<T> lx, G3<T> lu,
         uint32_t* __restrict__ rows, uint16_t* __restrict__ slot, Rec<T>* __restrict__ A, Rec<T>* __restrict__ B,
         unsigned long long* err)
{
  extern __shared__ uint32_t hist[];  // two 16-bit counters per word: groups, then out-of-box particles
  __shared__ uint32_t wsum[16];
  const DEnt<T>& en = tab[pmap[block]];
  const DBox<T>& b = en.b;
  const int nt = int(blockDim.x), tid = int(threadIdx.x);
  const int64_t blk = int64_t(block) - en.pb0, P = int64_t(nt) * K;
  const int64_t np = b.off[b.nsp], p0 = blk * P;
  const int nw = en.rowlen;
  for(int w = tid; w < nw; w += nt) hist[w] = 0;
  __syncthreads();
  // (loads run ahead of their use: lanes past the end load the last particle)
  T px[K][3];
#pragma unroll
  for(int k = 0; k < K; ++k) {
    const int64_t q = en.p0 + min(p0 + k * nt + tid, np - 1);
#pragma unroll
    for(int a = 0; a < 3; ++a) px[k][a] = x.c[a][q];
  }
  uint32_t kr[K];
#pragma unroll
  for(int k = 0; k < K; ++k) {
    kr[k] = 0;
    if(p0 + k * nt + tid < np) {
      int key = en.ngroup;
      if(in_box(b, px[k])) {
        int g[3];
#pragma unroll
        for(int a = 0; a < 3; ++a) {
          T d;
          g[a] = brick_at(en.ax[a], wrap2(base_cell(px[k][a], d), b.n[a])) >> en.gsh;
        }
        key = (g[0] * en.ng[1] + g[1]) * en.ng[2] + g[2];
      } else if(!ADJ) {
        atomicAdd(err, 1ull);
      }
      const int s = (key & 1) * 16;
      const uint32_t old = atomicAdd(&hist[key >> 1], 1u << s);
      kr[k] = (uint32_t(key) << 16) | ((old >> s) & 0xffffu);
    }
  }
  __syncthreads();
  // counts -> exclusive run starts: a contiguous share of words per thread
  const int per = (nw + nt - 1) / nt, w0 = min(tid * per, nw), w1 = min(w0 + per, nw);
  uint32_t sum = 0;
  for(int w = w0; w < w1; ++w) sum += (hist[w] & 0xffffu) + (hist[w] >> 16);
  uint32_t inc = sum;
#pragma unroll
  for(int o = 1; o < 64; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o);
    if((tid & 63) >= o) inc += t;
  }
  if((tid & 63) == 63) wsum[tid >> 6] = inc;
  __syncthreads();
  uint32_t run = inc - sum;
  for(int w = 0; w < (tid >> 6); ++w) run += wsum[w];
  for(int w = w0; w < w1; ++w) {
    const uint32_t lo = hist[w] & 0xffffu, hi = hist[w] >> 16;
    hist[w] = run | ((run + lo) << 16);
    run += lo + hi;
  }
  __syncthreads();
  uint32_t* row = rows + en.row0 + blk * nw;
  for(int w = tid; w < nw; w += nt) row[w] = hist[w];
  constexpr int KC = K < 4 ? K : 4;  // particles whose loads are in flight together
#pragma unroll
  for(int k0 = 0; k0 < K; k0 += KC) {
    T pu[KC][3], lr[ADJ ? KC : 1][6];
#pragma unroll
    for(int k = 0; k < KC; ++k) {
      const int64_t q = en.p0 + min(p0 + (k0 + k) * nt + tid, np - 1);
#pragma unroll
      for(int a = 0; a < 3; ++a) {
        pu[k][a] = u.c[a][q];
        if constexpr(ADJ) {
          lr[k][a] = lx.c[a][q];
          lr[k][3 + a] = lu.c[a][q];
        }
      }
    }
#pragma unroll
    for(int k = 0; k < KC; ++k) {
      const int64_t p = p0 + (k0 + k) * nt + tid;
      if(p >= np) continue;
      const int key = int(kr[k0 + k] >> 16);
      const uint32_t dst = ((hist[key >> 1] >> ((key & 1) * 16)) & 0xffffu) + (kr[k0 + k] & 0xffffu);
      slot[en.p0 + p] = uint16_t(dst);
      const int64_t at = en.p0 + p0 + dst;
      Rec<T> r;
#pragma unroll
      for(int a = 0; a < 3; ++a) {
        r.v[a] = px[k0 + k][a];
        r.v[3 + a] = pu[k][a];
      }
      r.v[6] = T(species_of(b, p));
      r.v[7] = T(0);
      A[at] = r;
      if constexpr(ADJ) {
#pragma unroll
        for(int a = 0; a < 6; ++a) r.v[a] = lr[k][a];
        r.v[6] = T(0);
        B[at] = r;
      }
    }
  }
}

template<class T, int K, bool ADJ>
__global__ void __launch_bounds__(1024)
  k_dbin(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, G3<T> x, G3<T> u, G3<T> lx, G3<T> lu,
         uint32_t* __restrict__ rows, uint16_t* __restrict__ slot, Rec<T>* __restrict__ A, Rec<T>* __restrict__ B,
         unsigned long long* err)
{
  bin_block<T, K, ADJ>(int(blockIdx.x), tab, pmap, x, u, lx, lu, rows, slot, A, B, err);
}

template<class T, int K>
__device__ __forceinline__ void
unsort_block(int block, const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, const uint16_t* __restrict__ slot,
            const Rec<T>* __restrict__ A, G3<T> x, G3<T> u)
{
  const DEnt<T>& en = tab[pmap[block]];
  const int nt = int(blockDim.x);
  const int64_t np = en.b.off[en.b.nsp], p0 = (int64_t(block) - en.pb0) * nt * K;
  constexpr int KC = K < 4 ? K : 4;
#pragma unroll
  for(int k0 = 0; k0 < K; k0 += KC) {
    int64_t q[KC];
    Rec<T> r[KC];
#pragma unroll
    for(int k = 0; k < KC; ++k) q[k] = en.p0 + min(p0 + (k0 + k) * nt + int(threadIdx.x), np - 1);
#pragma unroll
    for(int k = 0; k < KC; ++k) r[k] = A[en.p0 + p0 + slot[q[k]]];
#pragma unroll
    for(int k = 0; k < KC; ++k)
      if(p0 + (k0 + k) * nt + int(threadIdx.x) < np)
#pragma unroll
        for(int a = 0; a < 3; ++a) {
          x.c[a][q[k]] = r[k].v[a];
          u.c[a][q[k]] = r[k].v[3 + a];
        }
  }
}

template<class T, int K>
__global__ void __launch_bounds__(1024)
  k_dunsort(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, const uint16_t* __restrict__ slot,
            const Rec<T>* __restrict__ A, G3<T> x, G3<T> u)
{
  unsort_block<T, K>(int(blockIdx.x), tab, pmap, slot, A, x, u);
}

// Boxes of more than GROUPS_MAX bricks, whose rows hold runs of groups of bricks:
// a brick's records through a list of their places, sorted by brick.  A record
// takes its number in its brick from a global counter (k_dcount), the counters
// become the bricks' starts (k_dsums, k_dstarts), and the places are stored
// (k_dorder).  A brick that walked its group's runs passed over the other
// bricks' records with most lanes idle: 512^3 cells, groups of 4^3, 1.34e8 mixed
// particles took 145 ms a step and 279 ms its adjoint, 31 and 46 ms so; 256^3
// cells, groups of 2^3, 27 and 50 ms, 18 and 25.5 so (k_dcount 2.4, k_dorder 2.3
// ms of each, bound by their scattered 4-byte accesses).
template<class T>
__device__ inline int64_t brick_number(const DEnt<T>& en, const T x[3])
{
  int k[3];
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    T d;
    k[a] = brick_at(en.ax[a], wrap2(base_cell(x[a], d), en.b.n[a]));
  }
  return en.k0 + (int64_t(k[0]) * en.ax[1].nb + k[1]) * en.ax[2].nb + k[2];
}

// a lane's number among those that take one of counter `key`: an atomic for all
// lanes of one key while they are many (particles in cell order), else one each
__device__ inline uint32_t take_number(uint32_t* __restrict__ count, int64_t key, bool live)
{
  const int lane = int(threadIdx.x) & 63;
  const uint64_t below = (uint64_t(1) << lane) - 1;
  uint64_t left = __ballot(live);
  while(left) {
    const int lead = __ffsll(static_cast<unsigned long long>(left)) - 1;
    const int64_t k = __shfl(key, lead);
    const uint64_t same = __ballot(live && key == k) & left;
    if(__popcll(same) < 8) break;
    uint32_t base = 0;
    if(lane == lead) base = atomicAdd(&count[k], uint32_t(__popcll(same)));
    base = __shfl(base, lead);
    if(same >> lane & 1) return base + uint32_t(__popcll(same & below));
    left &= ~same;
  }
  return (left >> lane & 1) ? atomicAdd(&count[key], 1u) : 0u;
}

constexpr uint32_t NO_RANK = UINT32_MAX;

template<class T>
__global__ void __launch_bounds__(DWG)
  k_dcount(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, int64_t P, const Rec<T>* __restrict__ A,
           uint32_t* __restrict__ count, uint32_t* __restrict__ rank)
{
  const DEnt<T>& en = tab[pmap[blockIdx.x]];
  const int64_t p0 = (int64_t(blockIdx.x) - en.pb0) * P, p1 = min(p0 + P, en.b.off[en.b.nsp]);
  for(int64_t q0 = p0; q0 < p1; q0 += DWG) {
    const int64_t q = q0 + threadIdx.x, at = en.p0 + min(q, p1 - 1);
    const T x[3] = {A[at].v[0], A[at].v[1], A[at].v[2]};
    const bool live = q < p1 && in_box(en.b, x);
    const uint32_t r = take_number(count, live ? brick_number(en, x) : 0, live);
    if(q < p1) rank[at] = live ? r : NO_RANK;
  }
}

constexpr int SCAN = 4096;  // counters of a workgroup

__device__ inline uint32_t block_sum(uint32_t v, uint32_t* wsum)
{
#pragma unroll
  for(int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o);
  __syncthreads();
  if((threadIdx.x & 63) == 0) wsum[threadIdx.x >> 6] = v;
  __syncthreads();
  uint32_t sum = 0;
#pragma unroll
  for(int w = 0; w < DWG / 64; ++w) sum += wsum[w];
  return sum;
}

static __global__ void __launch_bounds__(DWG) k_dzero(uint32_t* __restrict__ p, int64_t n)
{
  const int64_t i = int64_t(blockIdx.x) * DWG + threadIdx.x;
  if(i < n) p[i] = 0;
}

static __global__ void __launch_bounds__(DWG) k_dsums(const uint32_t* __restrict__ count, int64_t n, uint32_t* __restrict__ sums)
{
  __shared__ uint32_t wsum[DWG / 64];
  const int64_t c0 = int64_t(blockIdx.x) * SCAN, c1 = min(c0 + SCAN, n);
  uint32_t v = 0;
  for(int64_t c = c0 + threadIdx.x; c < c1; c += DWG) v += count[c];
  v = block_sum(v, wsum);
  if(threadIdx.x == 0) sums[blockIdx.x] = v;
}

// counts -> exclusive starts, in place; entry n takes the total
static __global__ void __launch_bounds__(DWG)
  k_dstarts(uint32_t* __restrict__ count, int64_t n, const uint32_t* __restrict__ sums)
{
  __shared__ uint32_t wsum[DWG / 64];
  uint32_t v = 0;
  for(int b = int(threadIdx.x); b < int(blockIdx.x); b += DWG) v += sums[b];
  uint32_t run = block_sum(v, wsum);
  const int64_t c0 = int64_t(blockIdx.x) * SCAN, c1 = min(c0 + SCAN, n);
  const int wave = int(threadIdx.x) >> 6;
  for(int64_t q = c0; q < c1; q += DWG) {
    const int64_t c = q + threadIdx.x;
    const uint32_t own = c < c1 ? count[c] : 0;
    uint32_t inc = own;
#pragma unroll
    for(int o = 1; o < 64; o <<= 1) {
      const uint32_t t = __shfl_up(inc, o);
      if((int(threadIdx.x) & 63) >= o) inc += t;
    }
    __syncthreads();
    if((threadIdx.x & 63) == 63) wsum[wave] = inc;
    __syncthreads();
    uint32_t before = run;
#pragma unroll
    for(int w = 0; w < DWG / 64; ++w) {
      before += w < wave ? wsum[w] : 0;
      run += wsum[w];
    }
    if(c < c1) count[c] = before + inc - own;
  }
  if(c1 == n && threadIdx.x == 0) count[n] = run;
}

template<class T>
__global__ void __launch_bounds__(DWG)
  k_dorder(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, int64_t P, const Rec<T>* __restrict__ A,
           const uint32_t* __restrict__ start, const uint32_t* __restrict__ rank, uint32_t* __restrict__ order)
{
  const DEnt<T>& en = tab[pmap[blockIdx.x]];
  const int64_t p0 = (int64_t(blockIdx.x) - en.pb0) * P, p1 = min(p0 + P, en.b.off[en.b.nsp]);
  for(int64_t q = p0 + threadIdx.x; q < p1; q += DWG) {
    const int64_t at = en.p0 + q;
    const uint32_t r = rank[at];
    if(r == NO_RANK) continue;
    const T x[3] = {A[at].v[0], A[at].v[1], A[at].v[2]};
    order[start[brick_number(en, x)] + r] = uint32_t(at);
  }
}

// Small boxes (a particle a thread in the particle blocks): a launch costs
// about 4 us whatever it does, so what needs nothing of each other shares one.
// Before the bricks' step, the particles' bins and the curls of the fields; a
// second curl (the adjoint's) when c2.out is given.  16^3 box, 16384 particles: six
// launches a step instead of eight (adjoint: of nine), eight steps and their
// gradient 1.02 -> 0.87 ms.
template<class T, bool ADJ>
__global__ void __launch_bounds__(DWG)
  k_dprep(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, G3<T> x, G3<T> u, G3<T> lx, G3<T> lu,
          uint32_t* __restrict__ rows, uint16_t* __restrict__ slot, Rec<T>* __restrict__ A, Rec<T>* __restrict__ B,
          unsigned long long* err, int pblocks, BoxGrid bg, CurlB<T> c1, CurlB<T> c2)
{
  int blk = int(blockIdx.x);
  if(blk < pblocks) {
    bin_block<T, 1, ADJ>(blk, tab, pmap, x, u, lx, lu, rows, slot, A, B, err);
    return;
  }
  blk -= pblocks;
  const bool second = blk >= bg.blocks();
  const BoxPlace pl = place(bg, second ? blk - bg.blocks() : blk);
  if(pl.ok) curl_b_row(tab[pl.z], second ? c2 : c1, pl.i, pl.j, pl.tx, pl.step);
}

// After it, the particles back into their order and the gather of the bricks'
// windows (the current's, or the adjoint's node means).
template<class T, int BR, bool ADJ>
__global__ void __launch_bounds__(DWG)
  k_dfinish(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ pmap, const uint16_t* __restrict__ slot,
            const Rec<T>* __restrict__ A, G3<T> x, G3<T> u, int pblocks, BoxGrid bg, G3<T> F, G3<T> LB, G3<T> LBout,
            const T* __restrict__ st)
{
  const int blk = int(blockIdx.x);
  if(blk < pblocks) {
    unsort_block<T, 1>(blk, tab, pmap, slot, A, x, u);
    return;
  }
  const BoxPlace pl = place(bg, blk - pblocks);
  if(!pl.ok) return;
  if constexpr(ADJ) mgather_row<T, BR>(tab[pl.z], F, LB, LBout, st, pl.i, pl.j, pl.tx, pl.step);
  else jgather_row<T, BR>(tab[pl.z], F, st, pl.i, pl.j, pl.tx, pl.step);
}

// one brick of a box
struct BrickOf {
  int s[3], n[3];  // first cell, cells
};

template<class T>
__device__ inline BrickOf brick_of_box(const DEnt<T>& en, int64_t k)
{
  BrickOf B;
  const uint32_t kk = uint32_t(k), n1 = uint32_t(en.ax[1].nb), n2 = uint32_t(en.ax[2].nb);
  const int kc[3] = {int(kk / n2 / n1), int(kk / n2 % n1), int(kk % n2)};
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    B.s[a] = brick_start(en.ax[a], kc[a]);
    B.n[a] = brick_start(en.ax[a], kc[a] + 1) - B.s[a];
  }
  return B;
}

// node means of E and B (interpolation_EB_linear_1st's corner values) of a
// brick's nodes 0..n, M = BR + 1 per axis:
// E_x(N) = (Ex[N-x] + Ex[N]) / 2, B_x(N) = (Bx[N] + (Bx[N-y] + (Bx[N-z] + Bx[N-y-z]))) / 4
template<class T, int BR, int NT>
__device__ inline void stage_nodes(const DBox<T>& b, const BrickOf& bk, const G3<T>& E, const G3<T>& B, T* nm)
{
  constexpr int M = BR + 1, V = M * M * M;
  for(int q = int(threadIdx.x); q < V; q += NT) {
    const int l[3] = {q / (M * M), q / M % M, q % M};
    if(l[0] > bk.n[0] || l[1] > bk.n[1] || l[2] > bk.n[2]) continue;
    const int i = wrap1(bk.s[0] + l[0], b.n[0]), j = wrap1(bk.s[1] + l[1], b.n[1]), k = wrap1(bk.s[2] + l[2], b.n[2]);
    const int im = wrap1(i - 1, b.n[0]), jm = wrap1(j - 1, b.n[1]), km = wrap1(k - 1, b.n[2]);
    const int64_t c = cidx(b.n, i, j, k);
    nm[q] = (E.c[0][cidx(b.n, im, j, k)] + E.c[0][c]) / T(2);
    nm[V + q] = (E.c[1][cidx(b.n, i, jm, k)] + E.c[1][c]) / T(2);
    nm[2 * V + q] = (E.c[2][cidx(b.n, i, j, km)] + E.c[2][c]) / T(2);
    nm[3 * V + q] =
      (B.c[0][c] + (B.c[0][cidx(b.n, i, jm, k)] + (B.c[0][cidx(b.n, i, j, km)] + B.c[0][cidx(b.n, i, jm, km)]))) / T(4);
    nm[4 * V + q] =
      (B.c[1][c] + (B.c[1][cidx(b.n, im, j, k)] + (B.c[1][cidx(b.n, i, j, km)] + B.c[1][cidx(b.n, im, j, km)]))) / T(4);
    nm[5 * V + q] =
      (B.c[2][c] + (B.c[2][cidx(b.n, im, j, k)] + (B.c[2][cidx(b.n, i, jm, k)] + B.c[2][cidx(b.n, im, jm, k)]))) / T(4);
  }
}

// E and B at a particle from the staged nodes: o is its base cell's node,
// f.d its offsets
template<class T, int BR>
__device__ inline void gather_nodes(const T* nm, int o, Fwd<T>& f)
{
  constexpr int M = BR + 1, V = M * M * M;
  T m[2][2][2];
#pragma unroll
  for(int comp = 0; comp < 6; ++comp) {
#pragma unroll
    for(int ic = 0; ic < 2; ++ic)
#pragma unroll
      for(int jc = 0; jc < 2; ++jc)
#pragma unroll
        for(int kc = 0; kc < 2; ++kc) m[ic][jc][kc] = nm[comp * V + o + (ic * M + jc) * M + kc];
    (comp < 3 ? f.EBE[comp] : f.EBB[comp - 3]) = lerp3_d(f.d, m);
  }
}

// What a particle's cells are counted from: window node (of a window of one
// node before the brick to two after) = cell + rel.  l: the base cell's place
// in the brick, cell: the base cell, both of the position before the push; the
// wrap after it shifts the axis by -n, 0 or n.
template<class T>
__device__ inline void window_rel(const DBox<T>& b, const int l[3], const int cell[3], const T xn[3], int rel[3])
{
#pragma unroll
  for(int a = 0; a < 3; ++a) {
    const int n = b.n[a];
    rel[a] = l[a] + 1 - cell[a] - (xn[a] < T(0) ? n : (xn[a] >= T(n) ? -n : 0));
  }
}

// window node of a segment's cell; -1 when it misses the window
template<int BR>
__device__ inline int window_node(const BrickOf& bk, const int rel[3], const int i[3])
{
  constexpr int D = BR + 3;
  const int w[3] = {i[0] + rel[0], i[1] + rel[1], i[2] + rel[2]};
  const bool in = uint32_t(w[0]) <= uint32_t(bk.n[0] + 1) && uint32_t(w[1]) <= uint32_t(bk.n[1] + 1) &&
                  uint32_t(w[2]) <= uint32_t(bk.n[2] + 1);
  return in ? (w[0] * D + w[1]) * D + w[2] : -1;
}

// a segment's cell in the box, however far (a large cfl) it lies outside
struct BoxCell {
  int c[3];
};

template<class T>
__device__ inline BoxCell box_cell(const DBox<T>& b, int i0, int i1, int i2)
{
  auto rem = [](int i, int n) {
    const int r = i % n;
    return r < 0 ? r + n : r;
  };
  return BoxCell {{rem(i0, b.n[0]), rem(i1, b.n[1]), rem(i2, b.n[2])}};
}

// box node at offsets o (0 or 1) of a cell
template<class T>
__device__ inline int64_t box_node(const DBox<T>& b, const BoxCell& k, const int o[3])
{
  return cidx(b.n, wrap1(k.c[0] + o[0], b.n[0]), wrap1(k.c[1] + o[1], b.n[1]), wrap1(k.c[2] + o[2], b.n[2]));
}

__device__ inline void lds_add(double* p, double v)
{
  __hip_atomic_fetch_add(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Where a brick's records are: its run in the row of every particle block, or,
// in a box of more than GROUPS_MAX bricks, its part of a list (k_dorder).
struct Runs {
  const uint32_t* rows;
  int64_t P;
  const uint32_t *bstart, *order;
};

// The records of brick k of a box, taken by its workgroup's NT threads: rows are
// scanned NT at a time; a thread takes a contiguous share of the records they
// hold, so neighbouring lanes are far apart in a run (the particles of a cell
// that lie one after the other go to one lane, and the lanes' LDS adds to
// different nodes).  body(record, its place).  SPLIT: the gridDim.y workgroups of
// a brick take a share of the rows each.
template<class T, int NT, bool LIST, bool SPLIT, class Body>
__device__ inline void for_records(const DEnt<T>& en, const Runs& runs, int64_t k, const Rec<T>* A, Body&& body)
{
  const int tid = int(threadIdx.x);
  if constexpr(LIST) {
    const uint32_t lo = runs.bstart[en.k0 + k], total = runs.bstart[en.k0 + k + 1] - lo;
    const uint32_t* __restrict__ const list = runs.order + lo;
    const uint32_t per = (total + NT - 1) / NT, end = min((uint32_t(tid) + 1) * per, total);
    uint32_t r = min(uint32_t(tid) * per, total);
    if(r >= end) return;
    int64_t at = list[r];
    Rec<T> rec = A[at];
    for(; r < end; ++r) {
      const int64_t here = at;
      const Rec<T> cur = rec;
      if(r + 1 < end) {
        at = list[r + 1];
        rec = A[at];
      }
      body(cur, here);
    }
    return;
  }
  __shared__ uint32_t pre[NT + 1];  // records of the rows before
  __shared__ uint16_t first[NT];
  __shared__ uint32_t wsum[NT / 64];
  const int64_t P = runs.P;
  const uint16_t* tabl = reinterpret_cast<const uint16_t*>(runs.rows + en.row0) + k;
  const int64_t stride = 2 * int64_t(en.rowlen);
  const int64_t ra = SPLIT ? en.nrow * blockIdx.y / gridDim.y : 0;
  const int64_t rb = SPLIT ? en.nrow * (blockIdx.y + 1) / gridDim.y : en.nrow;
  for(int64_t r0 = ra; r0 < rb; r0 += NT) {
    uint32_t a = 0, len = 0;
    if(r0 + tid < rb) {
      const uint16_t* e = tabl + (r0 + tid) * stride;
      a = e[0];
      len = e[1] - a;
    }
    uint32_t inc = len;
#pragma unroll
    for(int o = 1; o < 64; o <<= 1) {
      const uint32_t t = __shfl_up(inc, o);
      if((tid & 63) >= o) inc += t;
    }
    if((tid & 63) == 63) wsum[tid >> 6] = inc;
    __syncthreads();
    uint32_t base = 0, total = 0;
#pragma unroll
    for(int w = 0; w < NT / 64; ++w) {
      base += w < (tid >> 6) ? wsum[w] : 0;
      total += wsum[w];
    }
    pre[tid] = base + inc - len;
    first[tid] = uint16_t(a);
    if(tid == 0) pre[NT] = total;
    __syncthreads();
    const uint32_t per = (total + NT - 1) / NT;
    uint32_t r = min(uint32_t(tid) * per, total);
    const uint32_t end = min(r + per, total);
    if(r < end) {
      // the last row that starts at or before r
      int lo = 0, hi = NT - 1;
      while(lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if(pre[mid] <= r) lo = mid;
        else hi = mid - 1;
      }
      auto place = [&](uint32_t i) {
        while(i >= pre[lo + 1]) ++lo;
        return en.p0 + (r0 + lo) * P + first[lo] + (i - pre[lo]);
      };
      int64_t at = place(r);
      Rec<T> rec = A[at];
      for(; r < end; ++r) {
        const int64_t here = at;
        const Rec<T> cur = rec;
        if(r + 1 < end) {
          at = place(r + 1);
          rec = A[at];
        }
        body(cur, here);
      }
    }
    __syncthreads();
  }
}

// a segment further than a cell from its particle's base cell (cfl > 1):
// straight to the box, out of line with scalar arguments
template<class T>
__device__ __attribute__((noinline)) void deposit_far(const DBox<T>& b, T* J0, T* J1, T* J2, int i0, int i1, int i2,
                                                     T F0, T F1, T F2, T W0, T W1, T W2)
{
  T* const J[3] = {J0, J1, J2};
  const BoxCell k = box_cell(b, i0, i1, i2);
  const T F[3] = {F0, F1, F2}, W[3] = {W0, W1, W2};
  T v[7][3];
  zig_values(F, W, v);
#pragma unroll
  for(int m = 0; m < 7; ++m)
#pragma unroll
    for(int c = 0; c < 3; ++c)
      if(zig_has(m, c)) atomic_add(&J[c][box_node(b, k, ZOFF[m])], v[m][c]);
}

// a split brick's window as one of its workgroups summed it
template<int N, int NT>
__device__ inline void store_part(double* __restrict__ part, const double (&win)[N])
{
  double* p = part + (int64_t(blockIdx.x) * gridDim.y + blockIdx.y) * N;
  for(int q = int(threadIdx.x); q < N; q += NT) p[q] = win[q];
}

// their sum, brick blockIdx.x
template<int N, int NT>
__device__ inline void sum_parts(const double* __restrict__ part, int split, double (&win)[N])
{
  const double* p = part + int64_t(blockIdx.x) * split * N;
  for(int q = int(threadIdx.x); q < N; q += NT) {
    double v = 0.0;
#pragma unroll 8
    for(int k = 0; k < split; ++k) v += p[int64_t(k) * N + q];
    win[q] = v;
  }
}

// the forward step of one brick's particles; results replace the records (a
// second set of records made the step 12 to 35 % slower: twice the lines to
// hold in cache)
template<class T, int BR, int NT, bool LIST>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 5 : 4)))
  k_dstep(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ kmap, G3<T> E, G3<T> B,
          Runs runs, Rec<T>* A, T* __restrict__ jst, G3<T> J, double* __restrict__ part)
{
  constexpr int M = BR + 1, D = BR + 3, V = D * D * D;
  __shared__ double win[3 * V];
  __shared__ T nm[6 * M * M * M];
  const DEnt<T>& en = tab[kmap[blockIdx.x]];
  const DBox<T>& b = en.b;
  const int64_t kb = int64_t(blockIdx.x) - en.k0;
  const BrickOf bk = brick_of_box(en, kb);
  E = sh(E, en.c0);
  B = sh(B, en.c0);
  J = sh(J, en.c0);
  for(int q = int(threadIdx.x); q < 3 * V; q += NT) win[q] = 0.0;
  stage_nodes<T, BR, NT>(b, bk, E, B, nm);
  __syncthreads();
  for_records<T, NT, LIST, BR == 4>(en, runs, kb, A, [&](Rec<T> r, int64_t at) {
    Fwd<T> f;
    int cell[3], l[3];
#pragma unroll
    for(int a = 0; a < 3; ++a) {
      cell[a] = base_cell(r.v[a], f.d[a]);
      l[a] = wrap2(cell[a], b.n[a]) - bk.s[a];
    }
    const int s = int(r.v[6]);
    gather_nodes<T, BR>(nm, (l[0] * M + l[1]) * M + l[2], f);
    BorisT<T> bs;
    boris_fwd(b.cfl, b.qm[s], f.EBE, f.EBB, r.v, r.v + 3, bs, f.xn, f.un);
    wrap_pos(b, f.xn, f.xw);
    Zig<T> z;
    zig_setup(b, f.xw, f.un, b.q[s], z);
#pragma unroll
    for(int a = 0; a < 3; ++a) {
      r.v[a] = f.xw[a];
      r.v[3 + a] = f.un[a];
    }
    A[at] = r;
    int rel[3];
    window_rel(b, l, cell, f.xn, rel);
    const int o1 = window_node<BR>(bk, rel, z.i1), o2 = window_node<BR>(bk, rel, z.i2);
    T v1[7][3], v2[7][3];
    zig_values(z.F1, z.W1, v1);
    zig_values(z.F2, z.W2, v2);
    if(o1 < 0 || o2 < 0) {
      deposit_far(b, J.c[0], J.c[1], J.c[2], z.i1[0], z.i1[1], z.i1[2], z.F1[0], z.F1[1], z.F1[2], z.W1[0], z.W1[1],
                  z.W1[2]);
      deposit_far(b, J.c[0], J.c[1], J.c[2], z.i2[0], z.i2[1], z.i2[2], z.F2[0], z.F2[1], z.F2[2], z.W2[0], z.W2[1],
                  z.W2[2]);
      return;
    }
    const bool same = o1 == o2;
#pragma unroll
    for(int m = 0; m < 7; ++m)
#pragma unroll
      for(int c = 0; c < 3; ++c)
        if(zig_has(m, c)) {
          const int n = c * V + (ZOFF[m][0] * D + ZOFF[m][1]) * D + ZOFF[m][2];
          lds_add(&win[o1 + n], same ? double(v1[m][c]) + double(v2[m][c]) : double(v1[m][c]));
        }
    if(!same) {
#pragma unroll
      for(int m = 0; m < 7; ++m)
#pragma unroll
        for(int c = 0; c < 3; ++c)
          if(zig_has(m, c)) {
            const int n = c * V + (ZOFF[m][0] * D + ZOFF[m][1]) * D + ZOFF[m][2];
            lds_add(&win[o2 + n], double(v2[m][c]));
          }
    }
  });
  __syncthreads();
  if constexpr(BR == 4)
    if(gridDim.y > 1) {
      store_part<3 * V, NT>(part, win);
      return;
    }
  T* w = jst + int64_t(blockIdx.x) * (3 * V);
  for(int q = int(threadIdx.x); q < 3 * V; q += NT) w[q] = T(win[q]);
}

// split bricks: their current windows
template<class T, int BR, int NT>
__global__ void __launch_bounds__(NT) k_dstep_sum(const double* __restrict__ part, int split, T* __restrict__ jst)
{
  constexpr int N = 3 * (BR + 3) * (BR + 3) * (BR + 3);
  __shared__ double win[N];
  sum_parts<N, NT>(part, split, win);
  T* w = jst + int64_t(blockIdx.x) * N;
  for(int q = int(threadIdx.x); q < N; q += NT) w[q] = T(win[q]);  // (each thread its own)
}

// gathered adjoint of one zigzag segment: dL/dF and dL/dW (per axis); L(d, o)
// is the current's adjoint of component d at the node at offsets o of the cell
template<class T, class Read>
__device__ inline void zig_seg_adj(Read&& L, const T F[3], const T W[3], T gF[3], T gW[3])
{
  const T one = T(1);
  gW[0] = gW[1] = gW[2] = T(0);
#pragma unroll
  for(int d = 0; d < 3; ++d) {
    const int e = d == 0 ? 1 : 0, g = d == 2 ? 1 : 2;  // the other two axes, e < g
    T v[2][2];
#pragma unroll
    for(int de = 0; de < 2; ++de)
#pragma unroll
      for(int dg = 0; dg < 2; ++dg) {
        int o[3] = {0, 0, 0};
        o[e] = de;
        o[g] = dg;
        v[de][dg] = L(d, o);
      }
    const T we = W[e], wg = W[g];
    const T G = (v[0][0] * (one - we) + v[1][0] * we) * (one - wg) + (v[0][1] * (one - we) + v[1][1] * we) * wg;
    const T dGe = (v[1][0] - v[0][0]) * (one - wg) + (v[1][1] - v[0][1]) * wg;
    const T dGg = (v[0][1] - v[0][0]) * (one - we) + (v[1][1] - v[1][0]) * we;
    gF[d] = G;
    gW[e] += F[d] * dGe;
    gW[g] += F[d] * dGg;
  }
}

template<class T>
__device__ inline void cross_adj(const T a[3], const T b[3], const T gc[3], T ga[3], T gb[3])
{
  // c = a x b: dL/da = b x gc, dL/db = gc x a (accumulated)
  T t[3];
  cross3d(b, gc, t);
#pragma unroll
  for(int k = 0; k < 3; ++k) ga[k] += t[k];
  cross3d(gc, a, t);
#pragma unroll
  for(int k = 0; k < 3; ++k) gb[k] += t[k];
}

// a brick's window of field adjoints from its node-mean adjoints mw
template<class T, int BR, int NT>
__device__ inline void store_means(const BrickOf& bk, const double* mw, T* __restrict__ mst)
{
  constexpr int M = BR + 1, MV = M * M * M;
  // node means back to the staggered components.  E_x(node N) = (Ex[N-x] +
  // Ex[N]) / 2, so Ex[n] receives (ME_x[n] + ME_x[n+x]) / 2; B_x(node N) =
  // (Bx[N] + Bx[N-y] + Bx[N-z] + Bx[N-y-z]) / 4, so Bx[n] receives the mean of
  // MB_x over n, n+y, n+z, n+y+z: a window of one node before the brick to one after
  constexpr int W = BR + 2, WV = W * W * W;
  T* out = mst + int64_t(blockIdx.x) * (6 * WV);
  for(int q = int(threadIdx.x); q < WV; q += NT) {
    const int o[3] = {q / (W * W) - 1, q / W % W - 1, q % W - 1};
    auto at = [&](int c, int x, int y, int z) {
      const int p[3] = {o[0] + x, o[1] + y, o[2] + z};
#pragma unroll
      for(int a = 0; a < 3; ++a)
        if(p[a] < 0 || p[a] > bk.n[a]) return 0.0;
      return mw[c * MV + (p[0] * M + p[1]) * M + p[2]];
    };
    out[q] = T((at(0, 0, 0, 0) + at(0, 1, 0, 0)) * 0.5);
    out[WV + q] = T((at(1, 0, 0, 0) + at(1, 0, 1, 0)) * 0.5);
    out[2 * WV + q] = T((at(2, 0, 0, 0) + at(2, 0, 0, 1)) * 0.5);
    out[3 * WV + q] = T(((at(3, 0, 0, 0) + at(3, 0, 1, 0)) + (at(3, 0, 0, 1) + at(3, 0, 1, 1))) * 0.25);
    out[4 * WV + q] = T(((at(4, 0, 0, 0) + at(4, 1, 0, 0)) + (at(4, 0, 0, 1) + at(4, 1, 0, 1))) * 0.25);
    out[5 * WV + q] = T(((at(5, 0, 0, 0) + at(5, 1, 0, 0)) + (at(5, 0, 1, 0) + at(5, 1, 1, 0))) * 0.25);
  }
}

// the adjoint of one brick's particles.  L: the filtered adjoint of E', whose
// negative is the adjoint of J.  Each particle recomputes its forward step,
// applies the chain rule by hand and adds its node-mean adjoints (dL/dE, dL/dB
// at the particle times the trilinear weights of its 8 corners) to the
// brick's window; records of A (x, u) stay, records of B (lambda_x, lambda_u)
// are replaced.
template<class T, int BR, int NT, bool LIST>
__global__ void __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 4 : 2)))
  k_dadj(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ kmap, G3<T> E, G3<T> B, G3<T> L,
         Runs runs, const Rec<T>* __restrict__ A, Rec<T>* __restrict__ lam, T* __restrict__ mst,
         double* __restrict__ part)
{
  constexpr int M = BR + 1, MV = M * M * M, D = BR + 3, V = D * D * D;
  __shared__ double mw[6 * MV];
  __shared__ T nm[6 * MV];
  __shared__ T lw[3 * V];
  const DEnt<T>& en = tab[kmap[blockIdx.x]];
  const DBox<T>& b = en.b;
  const int64_t kb = int64_t(blockIdx.x) - en.k0;
  const BrickOf bk = brick_of_box(en, kb);
  E = sh(E, en.c0);
  B = sh(B, en.c0);
  L = sh(L, en.c0);
  for(int q = int(threadIdx.x); q < 6 * MV; q += NT) mw[q] = 0.0;
  stage_nodes<T, BR, NT>(b, bk, E, B, nm);
  for(int q = int(threadIdx.x); q < V; q += NT) {
    const int o[3] = {q / (D * D), q / D % D, q % D};
    if(o[0] > bk.n[0] + 2 || o[1] > bk.n[1] + 2 || o[2] > bk.n[2] + 2) continue;
    int c[3];
#pragma unroll
    for(int a = 0; a < 3; ++a) c[a] = wrap1(wrap1(bk.s[a] + o[a] - 1, b.n[a]), b.n[a]);
    const int64_t node = cidx(b.n, c[0], c[1], c[2]);
#pragma unroll
    for(int d = 0; d < 3; ++d) lw[d * V + q] = -L.c[d][node];
  }
  __syncthreads();
  const T cfl = b.cfl;
  for_records<T, NT, LIST, BR == 4>(en, runs, kb, A, [&](const Rec<T>& r, int64_t at) {
    Rec<T> g = lam[at];
    Fwd<T> f;
    int cell[3], l[3];
#pragma unroll
    for(int a = 0; a < 3; ++a) {
      cell[a] = base_cell(r.v[a], f.d[a]);
      l[a] = wrap2(cell[a], b.n[a]) - bk.s[a];
    }
    const int s = int(r.v[6]);
    const int node = (l[0] * M + l[1]) * M + l[2];
    const T gxo[3] = {g.v[0], g.v[1], g.v[2]}, guo[3] = {g.v[3], g.v[4], g.v[5]};
    // ---- recompute the forward step
    gather_nodes<T, BR>(nm, node, f);
    BorisT<T> bs;
    boris_fwd(cfl, b.qm[s], f.EBE, f.EBB, r.v, r.v + 3, bs, f.xn, f.un);
    wrap_pos(b, f.xn, f.xw);
    Zig<T> z;
    const T q = b.q[s];
    zig_setup(b, f.xw, f.un, q, z);

    // ---- deposit adjoint: J(F, W) -> x1, x2, xr -> x'' and u'
    T gF1[3], gW1[3], gF2[3], gW2[3];
    int rel[3];
    window_rel(b, l, cell, f.xn, rel);
    const int o1 = window_node<BR>(bk, rel, z.i1), o2 = window_node<BR>(bk, rel, z.i2);
    if(o1 >= 0 && o2 >= 0) {
      auto at_node = [&](int o0) {
        return [o0](int d, const int o[3]) { return lw[d * V + o0 + (o[0] * D + o[1]) * D + o[2]]; };
      };
      zig_seg_adj(at_node(o1), z.F1, z.W1, gF1, gW1);
      zig_seg_adj(at_node(o2), z.F2, z.W2, gF2, gW2);
    } else {
      // a segment further than a cell from the base cell (cfl > 1)
      auto in_box_at = [&](const int* i) {
        return [&b, &L, k = box_cell(b, i[0], i[1], i[2])](int d, const int o[3]) { return -L.c[d][box_node(b, k, o)]; };
      };
      zig_seg_adj(in_box_at(z.i1), z.F1, z.W1, gF1, gW1);
      zig_seg_adj(in_box_at(z.i2), z.F2, z.W2, gF2, gW2);
    }
    T gx1[3], gx2[3];
#pragma unroll
    for(int d = 0; d < 3; ++d) {
      const T gxr = q * gF1[d] - q * gF2[d] + T(0.5) * (gW1[d] + gW2[d]);
      gx1[d] = -q * gF1[d] + T(0.5) * gW1[d];
      gx2[d] = q * gF2[d] + T(0.5) * gW2[d];
      if(z.mid[d]) {
        gx1[d] += T(0.5) * gxr;
        gx2[d] += T(0.5) * gxr;
      }
    }
    // x1 = x2 - u' s(u'), s = cfl / sqrt(1 + u'.u')
    T gun[3], gxw[3];
    const T ig3 = z.invgam * z.invgam * z.invgam;
    const T g1u = dot3d(gx1, f.un);
#pragma unroll
    for(int d = 0; d < 3; ++d) {
      gxw[d] = gx2[d] + gx1[d] + gxo[d];
      gun[d] = guo[d] - z.s * gx1[d] + cfl * ig3 * g1u * f.un[d];
    }
    // ---- position update: x' = x + cfl u' / sqrt(1 + u'.u'); the wrap is the identity
    T gx[3];
    const T gxu = dot3d(gxw, f.un);
#pragma unroll
    for(int d = 0; d < 3; ++d) {
      gx[d] = gxw[d];
      gun[d] += cfl * (z.invgam * gxw[d] - ig3 * gxu * f.un[d]);
    }
    // ---- Boris Jacobian-transpose
    T gu2[3], gu0[3], gE0[3], gB0[3] = {T(0), T(0), T(0)}, gu1[3] = {T(0), T(0), T(0)};
#pragma unroll
    for(int d = 0; d < 3; ++d) {
      gu2[d] = gun[d] / cfl;
      gu0[d] = gu2[d];
      gE0[d] = gu2[d];
    }
    cross_adj(bs.u1, bs.B0, gu2, gu1, gB0);  // u2 = u0 + u1 x B0 + E0
    T gw[3];
#pragma unroll
    for(int d = 0; d < 3; ++d) gw[d] = gu1[d] * bs.f;  // u1 = w f
    const T gf = dot3d(gu1, bs.w);
#pragma unroll
    for(int d = 0; d < 3; ++d) gu0[d] += gw[d];  // w = u0 + u0 x B0
    cross_adj(bs.u0, bs.B0, gw, gu0, gB0);
#pragma unroll
    for(int d = 0; d < 3; ++d) gB0[d] += -(bs.f * bs.f) * gf * bs.B0[d];  // f = 2 / (1 + B0.B0)
    const T hq = T(0.5) * b.qm[s];
    T gEB[3], gEE[3];
#pragma unroll
    for(int d = 0; d < 3; ++d) gEB[d] = gB0[d] * (bs.bfac / cfl);  // B0 = EBB bfac / cfl
    const T gbfac = dot3d(gB0, f.EBB) / cfl;
    const T gg = hq * gbfac;  // bfac = hq g
    const T g3 = bs.g * bs.g * bs.g / (cfl * cfl);
#pragma unroll
    for(int d = 0; d < 3; ++d) gu0[d] += -gg * g3 * bs.u0[d];  // g = cfl / sqrt(cfl^2 + u0.u0)
    T gvel[3];
#pragma unroll
    for(int d = 0; d < 3; ++d) {
      gE0[d] += gu0[d];          // u0 = v0 + E0
      gvel[d] = gu0[d] * cfl;    // v0 = vel cfl
      gEE[d] = gE0[d] * hq;      // E0 = EBE hq
    }
    // ---- interpolation adjoint: node-mean adjoints, and the gradient of the
    // weights in x
    const T wx[2] = {T(1) - f.d[0], f.d[0]}, wy[2] = {T(1) - f.d[1], f.d[1]}, wz[2] = {T(1) - f.d[2], f.d[2]};
    // (the corners are read again: kept, their derivatives spill)
    T gd[3] = {T(0), T(0), T(0)};
#pragma unroll
    for(int ic = 0; ic < 2; ++ic)
#pragma unroll
      for(int jc = 0; jc < 2; ++jc)
#pragma unroll
        for(int kc = 0; kc < 2; ++kc) {
          const int n = node + (ic * M + jc) * M + kc;
          T sum = T(0);
#pragma unroll
          for(int c = 0; c < 3; ++c) sum += gEE[c] * nm[c * MV + n] + gEB[c] * nm[(3 + c) * MV + n];
          // d(trilinear weight)/dd: the weight with its own axis factor replaced by -1 / +1
          gd[0] += (ic ? sum : -sum) * (wy[jc] * wz[kc]);
          gd[1] += (jc ? sum : -sum) * (wx[ic] * wz[kc]);
          gd[2] += (kc ? sum : -sum) * (wx[ic] * wy[jc]);
          const T w = wx[ic] * wy[jc] * wz[kc];
#pragma unroll
          for(int c = 0; c < 3; ++c) {
            lds_add(&mw[c * MV + n], double(gEE[c] * w));
            lds_add(&mw[(3 + c) * MV + n], double(gEB[c] * w));
          }
        }
#pragma unroll
    for(int a = 0; a < 3; ++a) {
      g.v[a] = gx[a] + gd[a];
      g.v[3 + a] = gvel[a];
    }
    lam[at] = g;
  });
  __syncthreads();
  if constexpr(BR == 4)
    if(gridDim.y > 1) {
      store_part<6 * MV, NT>(part, mw);
      return;
    }
  store_means<T, BR, NT>(bk, mw, mst);
}

// split bricks: their windows of field adjoints
template<class T, int BR, int NT>
__global__ void __launch_bounds__(NT)
  k_dadj_sum(const DEnt<T>* __restrict__ tab, const uint16_t* __restrict__ kmap, const double* __restrict__ part, int split,
             T* __restrict__ mst)
{
  constexpr int MV = (BR + 1) * (BR + 1) * (BR + 1);
  __shared__ double mw[6 * MV];
  const DEnt<T>& en = tab[kmap[blockIdx.x]];
  sum_parts<6 * MV, NT>(part, split, mw);
  __syncthreads();
  store_means<T, BR, NT>(brick_of_box(en, int64_t(blockIdx.x) - en.k0), mw, mst);
}

}  // namespace

// ---------------------------------------------------------------- host side
struct DiffImpl {
  rk_diff_desc d;                    // the first box (precision, cfl, filter passes are common)
  std::vector<rk_diff_desc> boxes;   // every box of the ensemble
  std::vector<int64_t> c0, p0;       // first cell / particle of each box in the concatenated arrays
  int nmax[3] = {0, 0, 0};           // largest side per axis (the field kernels' grid)
  void* tab = nullptr;               // device DEnt<T>[boxes]
  int64_t ncell = 0, np = 0;         // totals
  size_t vb = 4;
  int br = 8;                        // most cells of a brick per axis (8 or 4)
  int bin_threads = 256, bin_k = 1;  // a particle block: threads and particles per thread
  int64_t pblocks = 0, nbricks = 0, row_words = 0;
  int rowlen_max = 0;
  bool listed = false;               // some box has too many bricks for a row: records through a list
  uint16_t* pmap = nullptr;          // particle block -> box
  uint16_t* kmap = nullptr;          // brick -> box
  void* scratch[5][3] = {};          // B1, J, Jt, LB2, LE (planar)
  void* recs[2] = {};                // the sorted blocks' records: x, u; lambda_x, lambda_u
  uint16_t* slot = nullptr;          // particle -> its record's slot in its block
  uint32_t* rows = nullptr;          // run starts of every block
  uint32_t* rank = nullptr;          // listed: a record's number in its brick
  uint32_t* order = nullptr;         // listed: the records' places, sorted by brick
  uint32_t* bstart = nullptr;        // listed: the bricks' starts in it
  uint32_t* bsums = nullptr;         // listed: sums of SCAN counters each
  void* stage = nullptr;             // per brick: its current or node-mean adjoint window
  int split = 1;                     // workgroups of a brick
  double* part = nullptr;            // split bricks: the window of each of their workgroups
  unsigned long long* err = nullptr;
};

namespace {

enum { S_B1 = 0, S_J, S_JT, S_LB2, S_LE };

// Threads per brick workgroup: an 8^3 brick at 16 particles per cell and
// species holds 16384 records, a 4^3 brick an eighth of that.
constexpr int brick_threads(int br) { return br == 8 ? 512 : 256; }

template<class T>
DBox<T> make_box(const rk_diff_desc& d)
{
  DBox<T> b {};
  for(int a = 0; a < 3; ++a) b.n[a] = d.n[a];
  b.nsp = d.n_species;
  b.off[0] = 0;
  for(int s = 0; s < b.nsp; ++s) {
    b.off[s + 1] = b.off[s] + d.count[s];
    b.q[s] = static_cast<T>(d.charge[s]);
    const double sg = (0.0 < d.charge[s]) - (d.charge[s] < 0.0);
    b.qm[s] = static_cast<T>(sg / d.mass[s]);
  }
  b.cfl = static_cast<T>(d.cfl);
  return b;
}

int64_t bricks_of_box(const rk_diff_desc& d, int br, int nb[3])
{
  for(int a = 0; a < 3; ++a) nb[a] = (d.n[a] + br - 1) / br;
  return int64_t(nb[0]) * nb[1] * nb[2];
}

// a row's run starts stay in one block's LDS as 16-bit counters (64 KiB)
constexpr int GROUPS_MAX = 32000;

// Layout of the particle phase.
//  * Bricks of 8 cells per axis, of 4 while those are fewer than one per CU.
//  * Bricks of 4 cells that are few and full are split over workgroups, a share
//    of the rows each, until there are two per CU or 1024 records for each.  One
//    workgroup a brick left the chip idle, below the particle kernels before
//    bricks: 4^3 cells with 2e5 particles, adjoint 3.48 ms (2.05 ms before), 0.14
//    ms so; 8^3 with 2e5 0.51 (0.39), 0.08; with 2e4 0.084, 0.062 (4096 records each:
//    0.14 and 0.084 ms).
//  * A particle block is as long as keeps two and more blocks per CU busy: its
//    runs (P / bricks records of a mixed box) are what a brick reads in one
//    piece.  2.8e7 mixed particles, P = 4096 and 8192: k_dbin<adjoint> + k_dadj
//    3.43 and 3.33 ms; 4.2e6 particles in cell order: k_dbin 60 and 66 us.
//  * Boxes of more than GROUPS_MAX bricks sort by groups of 2^gsh bricks per
//    axis, and their bricks take the records through a list (k_dorder).  Just
//    below and above the line, 1.34e8 mixed particles: 248 x 256 x 256 cells 16.6
//    ms a step and 30 ms its adjoint, 256^3 17.9 and 25.5 ms.
template<class T>
hipError_t upload_table(DiffImpl& h)
{
  int nb[3];
  int64_t total = 0;
  for(const auto& d : h.boxes) total += bricks_of_box(d, 8, nb);
  h.br = total >= 256 ? 8 : 4;
  const int64_t np = h.np;
  h.bin_threads = np >= (int64_t(1) << 23) ? 1024 : (np >= (int64_t(1) << 20) ? 512 : 256);
  h.bin_k = np >= (int64_t(1) << 20) ? 8 : (np >= (int64_t(1) << 17) ? 4 : 1);
  const int64_t P = int64_t(h.bin_threads) * h.bin_k;
  std::vector<DEnt<T>> t(h.boxes.size());
  std::vector<uint16_t> pm, km;
  for(size_t i = 0; i < t.size(); ++i) {
    DEnt<T>& e = t[i];
    e.b = make_box<T>(h.boxes[i]);
    e.c0 = h.c0[i];
    e.p0 = h.p0[i];
    e.pb0 = h.pblocks;
    e.k0 = h.nbricks;
    e.row0 = h.row_words;
    h.nbricks += bricks_of_box(h.boxes[i], h.br, nb);
    auto per = [](int d) { return ((uint64_t(1) << 40) + uint64_t(d) - 1) / uint64_t(d); };
    for(int a = 0; a < 3; ++a) e.ax[a] = Axis {e.b.n[a], nb[a], per(e.b.n[a]), per(nb[a])};
    e.gsh = 0;
    for(;; ++e.gsh) {
      for(int a = 0; a < 3; ++a) e.ng[a] = ((nb[a] - 1) >> e.gsh) + 1;
      if(int64_t(e.ng[0]) * e.ng[1] * e.ng[2] <= GROUPS_MAX) break;
    }
    e.ngroup = e.ng[0] * e.ng[1] * e.ng[2];
    e.rowlen = (e.ngroup + 2) / 2;  // run starts and the end of the last run
    e.nrow = (e.b.off[e.b.nsp] + P - 1) / P;
    h.pblocks += e.nrow;
    h.row_words += e.nrow * e.rowlen;
    h.rowlen_max = std::max(h.rowlen_max, e.rowlen);
    if(e.gsh > 0) h.listed = true;
    pm.resize(size_t(h.pblocks), uint16_t(i));
    km.resize(size_t(h.nbricks), uint16_t(i));
  }
  auto put = [](auto** dst, const auto& v) {
    const size_t bytes = sizeof(v[0]) * std::max<size_t>(v.size(), 1);
    hipError_t e = hipMalloc(reinterpret_cast<void**>(dst), bytes);
    if(e == hipSuccess && !v.empty()) e = hipMemcpy(*dst, v.data(), sizeof(v[0]) * v.size(), hipMemcpyHostToDevice);
    return e;
  };
  hipError_t e = put(&h.tab, t);
  if(e == hipSuccess) e = put(&h.pmap, pm);
  if(e == hipSuccess) e = put(&h.kmap, km);
  const size_t win = size_t(6) * (h.br + 2) * (h.br + 2) * (h.br + 2);  // the larger of the two windows
  if(e == hipSuccess) e = hipMalloc(&h.stage, h.vb * win * size_t(h.nbricks));
  if(h.br == 4) {
    h.split = int(std::clamp<int64_t>(std::min(np / (h.nbricks * 1024), 512 / h.nbricks), 1, 64));
    // doubles of the larger of the two windows as they are summed
    if(h.split > 1 && e == hipSuccess)
      e = hipMalloc(reinterpret_cast<void**>(&h.part), sizeof(double) * 3 * 7 * 7 * 7 * size_t(h.nbricks) * size_t(h.split));
  }
  const size_t n1 = size_t(std::max<int64_t>(np, 1));
  for(int i = 0; i < 2 && e == hipSuccess; ++i) e = hipMalloc(&h.recs[i], sizeof(Rec<T>) * n1);
  if(e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&h.slot), sizeof(uint16_t) * n1);
  if(e == hipSuccess)
    e = hipMalloc(reinterpret_cast<void**>(&h.rows), sizeof(uint32_t) * size_t(std::max<int64_t>(h.row_words, 1)));
  auto words = [&](uint32_t** p, size_t n) {
    if(h.listed && e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(p), sizeof(uint32_t) * n);
  };
  words(&h.rank, n1);
  words(&h.order, n1);
  words(&h.bstart, size_t(h.nbricks) + 1);
  words(&h.bsums, size_t(h.nbricks + SCAN - 1) / SCAN);
  return e;
}

template<class T>
const DEnt<T>* table(const DiffImpl& h)
{
  return static_cast<const DEnt<T>*>(h.tab);
}

template<class T>
G3<T> g3(void* const p[3])
{
  return G3<T> {{static_cast<T*>(p[0]), static_cast<T*>(p[1]), static_cast<T*>(p[2])}};
}

template<class T>
G3<T> g3s(const DiffImpl& h, int which)
{
  return G3<T> {{static_cast<T*>(h.scratch[which][0]), static_cast<T*>(h.scratch[which][1]),
                 static_cast<T*>(h.scratch[which][2])}};
}

int dfail(int code, const char* msg)
{
  set_error(msg);
  return code;
}

// per-box launches: blockIdx.z is the box; x (and y) are sized for the largest
// box.  Lanes run along z; rows shorter than a wave share a workgroup.
inline dim3 block_of(const DiffImpl& h)
{
  const int bx = std::min(h.nmax[2], DWG);
  return dim3(unsigned(bx), unsigned(bx >= 64 ? 1 : DWG / bx));
}
inline dim3 grid_of(const DiffImpl& h)
{
  const unsigned by = block_of(h).y;
  return dim3((unsigned(h.nmax[1]) + by - 1) / by, unsigned(h.nmax[0]), unsigned(h.boxes.size()));
}

// f = F^P(f) through the J / Jt pair (f may be either of them, or neither), up
// to three passes a launch
template<class T>
int filter_passes(const DiffImpl& h, const DEnt<T>* b, G3<T>& f, hipStream_t st)
{
  int o = f.c[0] == g3s<T>(h, S_J).c[0] ? S_JT : S_J;
  // x segments as long as leaves 512 workgroups a component, six per CU in all (a
  // segment reads 2R planes more than it writes).  With 256, 512 and 1024: 64^3
  // 12.6, 13.9 and 14.0 us, 96^3 22.0, 20.8 and 27.9, 128^3 43.6, 32.6 and 43.2;
  // below 64^3 all within 0.4 us
  const int tz = (h.nmax[2] + FZ - 1) / FZ, cols = tz * ((h.nmax[1] + FY - 1) / FY);
  int xseg = h.nmax[0];
  while(xseg > 2 && int64_t(cols) * ((h.nmax[0] + xseg - 1) / xseg) * int64_t(h.boxes.size()) < 512) xseg = (xseg + 1) / 2;
  const dim3 grid(3 * unsigned(cols), unsigned((h.nmax[0] + xseg - 1) / xseg), unsigned(h.boxes.size()));
  for(int left = h.d.filter_passes; left > 0;) {
    const int r = std::min(left, 3);
    const G3<T> out = g3s<T>(h, o);
    auto go = [&](auto kern) { hipLaunchKernelGGL(kern, grid, dim3(FT), 0, st, b, out, f, tz, xseg); };
    r == 3 ? go(k_dfilter<T, 3>) : (r == 2 ? go(k_dfilter<T, 2>) : go(k_dfilter<T, 1>));
    RK_HIP(hipGetLastError());
    f = out;
    o = o == S_J ? S_JT : S_J;
    left -= r;
  }
  return RK_OK;
}

// the particles of x, u (and lx, lu) into sorted records
template<class T, bool ADJ>
int bin_particles(const DiffImpl& h, G3<T> x, G3<T> u, G3<T> lx, G3<T> lu, hipStream_t st)
{
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(unsigned(h.pblocks)), dim3(unsigned(h.bin_threads)), sizeof(uint32_t) * size_t(h.rowlen_max),
                       st, table<T>(h), h.pmap, x, u, lx, lu, h.rows, h.slot, static_cast<Rec<T>*>(h.recs[0]),
                       static_cast<Rec<T>*>(h.recs[1]), h.err);
  };
  h.bin_k == 8 ? go(k_dbin<T, 8, ADJ>) : (h.bin_k == 4 ? go(k_dbin<T, 4, ADJ>) : go(k_dbin<T, 1, ADJ>));
  RK_HIP(hipGetLastError());
  return RK_OK;
}

// the bricks' lists of their records, where they need them
template<class T>
int list_records(const DiffImpl& h, hipStream_t st)
{
  if(!h.listed) return RK_OK;
  const int64_t P = int64_t(h.bin_threads) * h.bin_k;
  const Rec<T>* A = static_cast<const Rec<T>*>(h.recs[0]);
  const unsigned scan = unsigned((h.nbricks + SCAN - 1) / SCAN);
  hipLaunchKernelGGL(k_dzero, dim3(unsigned((h.nbricks + DWG - 1) / DWG)), dim3(DWG), 0, st, h.bstart, h.nbricks);
  RK_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_dcount<T>, dim3(unsigned(h.pblocks)), dim3(DWG), 0, st, table<T>(h), h.pmap, P, A, h.bstart, h.rank);
  RK_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_dsums, dim3(scan), dim3(DWG), 0, st, h.bstart, h.nbricks, h.bsums);
  RK_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_dstarts, dim3(scan), dim3(DWG), 0, st, h.bstart, h.nbricks, h.bsums);
  RK_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_dorder<T>, dim3(unsigned(h.pblocks)), dim3(DWG), 0, st, table<T>(h), h.pmap, P, A, h.bstart, h.rank,
                     h.order);
  RK_HIP(hipGetLastError());
  return RK_OK;
}

Runs runs_of(const DiffImpl& h) { return Runs {h.rows, int64_t(h.bin_threads) * h.bin_k, h.bstart, h.order}; }

// the records of set `which` back into x, u in the arrays' order
template<class T>
int unsort_particles(const DiffImpl& h, int which, G3<T> x, G3<T> u, hipStream_t st)
{
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(unsigned(h.pblocks)), dim3(unsigned(h.bin_threads)), 0, st, table<T>(h), h.pmap, h.slot,
                       static_cast<const Rec<T>*>(h.recs[which]), x, u);
  };
  h.bin_k == 8 ? go(k_dunsort<T, 8>) : (h.bin_k == 4 ? go(k_dunsort<T, 4>) : go(k_dunsort<T, 1>));
  RK_HIP(hipGetLastError());
  return RK_OK;
}

inline BoxGrid box_grid(const DiffImpl& h)
{
  const dim3 g = grid_of(h), b = block_of(h);
  // a row longer than a workgroup is shared while there are fewer rows than CUs
  const int64_t blocks = int64_t(g.x) * g.y * g.z;
  const int seg = blocks < 256 ? (h.nmax[2] + int(b.x) - 1) / int(b.x) : 1;
  return BoxGrid {int(g.x) * seg, int(g.y), int(g.z), int(b.x), int(b.y), seg};
}

// Launches are merged where they bound the step: particle blocks of DWG threads
// with a particle each (up to 2^17 particles) and up to 2^18 cells, beyond which
// the curls' rows (a workgroup of DWG threads however short) outweigh a launch.
// The merged launch lays the padded grid of the boxes (the largest side of every
// axis, times the boxes) out along x.  Boxes of one shape need at most 2^16
// blocks of it (every block holds two rows of two cells and more); boxes that
// are long along different axes need up to 2^31 and more, almost all empty, and
// a grid of 2^24 blocks of DWG threads is past what a launch takes: those keep
// the launches of their own, whose grid has three dimensions.
constexpr int64_t MERGED_BLOCKS = int64_t(1) << 16;

inline bool merged(const DiffImpl& h)
{
  const dim3 g = grid_of(h);
  return h.np > 0 && h.bin_k == 1 && h.bin_threads == DWG && h.ncell <= (int64_t(1) << 18) &&
         int64_t(g.x) * g.y * g.z <= MERGED_BLOCKS;
}

// the bins of the particles, and before them the curls (c2: if c2.out is given)
template<class T, bool ADJ>
int prepare(const DiffImpl& h, G3<T> x, G3<T> u, G3<T> lx, G3<T> lu, const CurlB<T>& c1, const CurlB<T>& c2, hipStream_t st)
{
  const bool two = c2.out.c[0] != nullptr;
  if(merged(h)) {
    const BoxGrid bg = box_grid(h);
    hipLaunchKernelGGL((k_dprep<T, ADJ>), dim3(unsigned(h.pblocks + (two ? 2 : 1) * bg.blocks())), dim3(DWG),
                       sizeof(uint32_t) * size_t(h.rowlen_max), st, table<T>(h), h.pmap, x, u, lx, lu, h.rows, h.slot,
                       static_cast<Rec<T>*>(h.recs[0]), static_cast<Rec<T>*>(h.recs[1]), h.err, int(h.pblocks), bg, c1, c2);
    RK_HIP(hipGetLastError());
    return RK_OK;
  }
  hipLaunchKernelGGL(k_dcurl_b<T>, grid_of(h), block_of(h), 0, st, table<T>(h), c1);
  RK_HIP(hipGetLastError());
  if(two) {
    hipLaunchKernelGGL(k_dcurl_b<T>, grid_of(h), block_of(h), 0, st, table<T>(h), c2);
    RK_HIP(hipGetLastError());
  }
  if(h.np == 0) return RK_OK;
  if(int rc = bin_particles<T, ADJ>(h, x, u, lx, lu, st)) return rc;
  return list_records<T>(h, st);
}

template<class T, int BR>
int step_t(DiffImpl& h, const rk_diff_state* in, rk_diff_state* out, hipStream_t st)
{
  const DEnt<T>* b = table<T>(h);
  const T half = static_cast<T>(h.d.cfl / 2), full = static_cast<T>(h.d.cfl);
  const G3<T> none {{nullptr, nullptr, nullptr}};
  const G3<T> E = g3<T>(in->E), B = g3<T>(in->B), B1 = g3s<T>(h, S_B1), J = g3s<T>(h, S_J);
  // B1 = B + cfl/2 curlE(E); J = 0
  if(int rc = prepare<T, false>(h, g3<T>(in->x), g3<T>(in->u), none, none, {B1, B, E, half, J}, {none, none, none, half, none}, st))
    return rc;
  if(h.np > 0) {
    constexpr int NT = brick_threads(BR);
    T* jst = static_cast<T*>(h.stage);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(unsigned(h.nbricks), unsigned(h.split)), dim3(NT), 0, st, b, h.kmap, E, B1, runs_of(h),
                         static_cast<Rec<T>*>(h.recs[0]), jst, J, h.part);
    };
    h.listed ? go(k_dstep<T, BR, NT, BR == 8>) : go(k_dstep<T, BR, NT, false>);  // (listed boxes have bricks of 8 cells)
    RK_HIP(hipGetLastError());
    if constexpr(BR == 4)
      if(h.split > 1) {
        hipLaunchKernelGGL((k_dstep_sum<T, BR, NT>), dim3(unsigned(h.nbricks)), dim3(NT), 0, st, h.part, h.split, jst);
        RK_HIP(hipGetLastError());
      }
    if(merged(h)) {
      const BoxGrid bg = box_grid(h);
      hipLaunchKernelGGL((k_dfinish<T, BR, false>), dim3(unsigned(h.pblocks + bg.blocks())), dim3(DWG), 0, st, b, h.pmap,
                         h.slot, static_cast<const Rec<T>*>(h.recs[0]), g3<T>(out->x), g3<T>(out->u),
                         int(h.pblocks), bg, J, none, none, jst);
      RK_HIP(hipGetLastError());
    } else {
      hipLaunchKernelGGL((k_djgather<T, BR>), grid_of(h), block_of(h), 0, st, b, J, jst);
      RK_HIP(hipGetLastError());
      if(int rc = unsort_particles<T>(h, 0, g3<T>(out->x), g3<T>(out->u), st)) return rc;
    }
  }
  G3<T> jf = J;
  if(int rc = filter_passes<T>(h, b, jf, st)) return rc;
  // B2 = B1 + cfl/2 curlE(E), written to out.B (E is still the input E)
  hipLaunchKernelGGL(k_dcurl_b<T>, grid_of(h), block_of(h), 0, st, b, CurlB<T> {g3<T>(out->B), B1, E, half, none});
  RK_HIP(hipGetLastError());
  // E' = E + cfl curlB(B2) - Jf
  hipLaunchKernelGGL(k_dcurl_e<T>, grid_of(h), block_of(h), 0, st, b, g3<T>(out->E), E, g3<T>(out->B), full, jf);
  RK_HIP(hipGetLastError());
  return RK_OK;
}

template<class T, int BR>
int adjoint_t(DiffImpl& h, const rk_diff_state* in, const rk_diff_state* ao, rk_diff_state* ai, hipStream_t st)
{
  const DEnt<T>* b = table<T>(h);
  const T half = static_cast<T>(h.d.cfl / 2), full = static_cast<T>(h.d.cfl);
  const G3<T> none {{nullptr, nullptr, nullptr}};
  const G3<T> E = g3<T>(in->E), B = g3<T>(in->B), B1 = g3s<T>(h, S_B1);
  const G3<T> LEo = g3<T>(ao->E), LBo = g3<T>(ao->B), LB2 = g3s<T>(h, S_LB2), LE = g3s<T>(h, S_LE);
  // forward B1, and
  // E' = E + cfl curlB(B2) - Jf:  lambda_B2 = LB' + cfl curlB^T(LE') = LB' - cfl curlE(LE')
  if(int rc = prepare<T, true>(h, g3<T>(in->x), g3<T>(in->u), g3<T>(ao->x), g3<T>(ao->u), {B1, B, E, half, none},
                               {LB2, LBo, LEo, T(-full), none}, st))
    return rc;
  // B2 = B1 + cfl/2 curlE(E):  lambda_E = LE' + cfl/2 curlE^T(LB2) = LE' - cfl/2 curlB(LB2)
  hipLaunchKernelGGL(k_dcurl_e<T>, grid_of(h), block_of(h), 0, st, b, LE, LEo, LB2, T(-half), none);
  RK_HIP(hipGetLastError());
  G3<T> LB1 = LB2;
  if(h.np > 0) {
    // lambda_J = -F^P(LE')
    G3<T> lj = LEo;
    if(int rc = filter_passes<T>(h, b, lj, st)) return rc;
    constexpr int NT = brick_threads(BR);
    T* mst = static_cast<T*>(h.stage);
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(unsigned(h.nbricks), unsigned(h.split)), dim3(NT), 0, st, b, h.kmap, E, B1, lj,
                         runs_of(h), static_cast<const Rec<T>*>(h.recs[0]), static_cast<Rec<T>*>(h.recs[1]), mst, h.part);
    };
    h.listed ? go(k_dadj<T, BR, NT, BR == 8>) : go(k_dadj<T, BR, NT, false>);
    RK_HIP(hipGetLastError());
    if constexpr(BR == 4)
      if(h.split > 1) {
        hipLaunchKernelGGL((k_dadj_sum<T, BR, NT>), dim3(unsigned(h.nbricks)), dim3(NT), 0, st, b, h.kmap, h.part, h.split, mst);
        RK_HIP(hipGetLastError());
      }
    // node-mean adjoints: lambda_E += NM_E^T(ME), lambda_B = lambda_B1 = LB2 + NM_B^T(MB)
    LB1 = g3<T>(ai->B);
    if(merged(h)) {
      const BoxGrid bg = box_grid(h);
      hipLaunchKernelGGL((k_dfinish<T, BR, true>), dim3(unsigned(h.pblocks + bg.blocks())), dim3(DWG), 0, st, b, h.pmap,
                         h.slot, static_cast<const Rec<T>*>(h.recs[1]), g3<T>(ai->x), g3<T>(ai->u), int(h.pblocks), bg, LE,
                         LB2, LB1, mst);
      RK_HIP(hipGetLastError());
    } else {
      if(int rc = unsort_particles<T>(h, 1, g3<T>(ai->x), g3<T>(ai->u), st)) return rc;
      hipLaunchKernelGGL((k_dmgather<T, BR>), grid_of(h), block_of(h), 0, st, b, LE, LB2, LB1, mst);
      RK_HIP(hipGetLastError());
    }
  } else {
    for(int c = 0; c < 3; ++c)
      RK_HIP(hipMemcpyAsync(ai->B[c], LB2.c[c], h.vb * size_t(h.ncell), hipMemcpyDeviceToDevice, st));
  }
  // B1 = B + cfl/2 curlE(E): lambda_E -= cfl/2 curlB(lambda_B1)
  hipLaunchKernelGGL(k_dcurl_e<T>, grid_of(h), block_of(h), 0, st, b, g3<T>(ai->E), LE, LB1, T(-half), none);
  RK_HIP(hipGetLastError());
  return RK_OK;
}

bool state_ok(const rk_diff_state* s, bool particles)
{
  if(!s) return false;
  for(int c = 0; c < 3; ++c) {
    if(!s->E[c] || !s->B[c]) return false;
    if(particles && (!s->x[c] || !s->u[c])) return false;
  }
  return true;
}

}  // namespace

}  // namespace rk

using namespace rk;

struct rk_diff : rk::DiffImpl {};

extern "C" {

int rk_diff_create_ensemble(rk_diff** out, const rk_diff_desc* descs, int32_t n_boxes)
{
  if(!out || !descs) return dfail(RK_EINVAL, "null argument");
  *out = nullptr;
  if(n_boxes < 1 || n_boxes > 65535) return dfail(RK_EINVAL, "diff ensemble: 1..65535 boxes");
  const rk_diff_desc& d0 = descs[0];
  if(d0.precision != 4 && d0.precision != 8) return dfail(RK_EINVAL, "diff box: precision must be 4 or 8");
  if(!(d0.cfl > 0.0) || d0.filter_passes < 0) return dfail(RK_EINVAL, "diff box: invalid cfl or filter passes");
  auto* h = new rk_diff();
  h->d = d0;
  h->vb = size_t(d0.precision);
  for(int i = 0; i < n_boxes; ++i) {
    const rk_diff_desc& d = descs[i];
    const char* bad = nullptr;
    for(int a = 0; a < 3; ++a)
      if(d.n[a] < 2 || d.n[a] > 4096) bad = "diff box: every side must be 2..4096 cells";
    if(d.n_species < 0 || d.n_species > RK_MAX_SPECIES) bad = "diff box: invalid species count";
    if(d.precision != d0.precision || d.cfl != d0.cfl || d.filter_passes != d0.filter_passes)
      bad = "diff ensemble: every box needs the same precision, cfl and filter passes";
    int64_t np = 0;
    for(int sp = 0; sp < d.n_species && !bad; ++sp) {
      if(d.count[sp] < 0 || !(d.mass[sp] > 0.0)) bad = "diff box: invalid particle count or mass";
      np += d.count[sp];
    }
    if(bad) {
      delete h;
      return dfail(RK_EINVAL, bad);
    }
    const int64_t nc = int64_t(d.n[0]) * d.n[1] * d.n[2];
    h->boxes.push_back(d);
    h->c0.push_back(h->ncell);
    h->p0.push_back(h->np);
    h->ncell += nc;
    h->np += np;
    for(int a = 0; a < 3; ++a) h->nmax[a] = std::max(h->nmax[a], d.n[a]);
  }
  if(h->ncell >= (int64_t(1) << 31) || h->np >= (int64_t(1) << 31)) {
    delete h;
    return dfail(RK_EINVAL, "diff ensemble: cells and particles must each total below 2^31");
  }
  hipError_t e = h->vb == 4 ? upload_table<float>(*h) : upload_table<double>(*h);
  for(int i = 0; i < 5 && e == hipSuccess; ++i)
    for(int c = 0; c < 3 && e == hipSuccess; ++c) e = hipMalloc(&h->scratch[i][c], h->vb * size_t(h->ncell));
  if(e == hipSuccess) e = hipMalloc(reinterpret_cast<void**>(&h->err), sizeof(unsigned long long));
  if(e == hipSuccess) e = hipMemset(h->err, 0, sizeof(unsigned long long));
  if(e != hipSuccess) {
    rk_diff_destroy(h);
    return hip_fail(e, "rk_diff_create");
  }
  *out = h;
  return RK_OK;
}

int rk_diff_create(rk_diff** out, const rk_diff_desc* desc)
{
  if(!desc) return dfail(RK_EINVAL, "null argument");
  return rk_diff_create_ensemble(out, desc, 1);
}

int rk_diff_destroy(rk_diff* h)
{
  if(!h) return RK_OK;
  for(auto& s : h->scratch)
    for(auto& p : s)
      if(p) (void)hipFree(p);
  for(void* q : {h->recs[0], h->recs[1], static_cast<void*>(h->slot), static_cast<void*>(h->rows),
                 static_cast<void*>(h->rank), static_cast<void*>(h->order), static_cast<void*>(h->bstart),
                 static_cast<void*>(h->bsums), h->stage, static_cast<void*>(h->part), static_cast<void*>(h->err), h->tab, static_cast<void*>(h->pmap),
                 static_cast<void*>(h->kmap)})
    if(q) (void)hipFree(q);
  delete h;
  return RK_OK;
}

int rk_diff_step(rk_diff* h, const rk_diff_state* in, rk_diff_state* out, void* stream)
{
  if(!h || !state_ok(in, h->np > 0) || !state_ok(out, h->np > 0)) return dfail(RK_EINVAL, "null state buffer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if(h->br == 8) return h->vb == 4 ? step_t<float, 8>(*h, in, out, st) : step_t<double, 8>(*h, in, out, st);
  return h->vb == 4 ? step_t<float, 4>(*h, in, out, st) : step_t<double, 4>(*h, in, out, st);
}

int rk_diff_step_adjoint(rk_diff* h, const rk_diff_state* in, const rk_diff_state* adj_out, rk_diff_state* adj_in,
                         void* stream)
{
  if(!h || !state_ok(in, h->np > 0) || !state_ok(adj_out, h->np > 0) || !state_ok(adj_in, h->np > 0))
    return dfail(RK_EINVAL, "null state buffer");
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  if(h->br == 8)
    return h->vb == 4 ? adjoint_t<float, 8>(*h, in, adj_out, adj_in, st) : adjoint_t<double, 8>(*h, in, adj_out, adj_in, st);
  return h->vb == 4 ? adjoint_t<float, 4>(*h, in, adj_out, adj_in, st) : adjoint_t<double, 4>(*h, in, adj_out, adj_in, st);
}

int rk_diff_error_count(rk_diff* h, int64_t* out, void* stream)
{
  if(!h || !out) return dfail(RK_EINVAL, "null argument");
  unsigned long long v = 0;
  hipStream_t st = reinterpret_cast<hipStream_t>(stream);
  RK_HIP(hipMemcpyAsync(&v, h->err, sizeof(v), hipMemcpyDeviceToHost, st));
  RK_HIP(hipStreamSynchronize(st));
  *out = int64_t(v);
  return RK_OK;
}

}  // extern "C"
