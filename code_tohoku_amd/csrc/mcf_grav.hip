// mcf_grav.hip -- self-gravity GRAVTY (3DMHD-CfCA/selfG_MPIfull8.f90, "SG8")
// for gfx950, FP64.
//
// Split levels (one block of nodes 0..n per reference rank): every operator
// is one launch over all ranks' blocks.  A halo exchange (BCsgr_MPI) is a
// single launch that pulls each ghost node's final value from where the
// reference's six sequential sendrecv phases (x low, x high, y low, y high,
// z low, z high; x ends closed, y and z periodic) would take it: walking the
// phases backwards from z, a ghost coordinate with its phase active moves to
// the neighbouring rank's opposite interior node.  The node it lands on is
// never written by any phase, so the pull reads pre-exchange values and
// one launch reproduces the reference's result exactly.
//
// Gauss-Seidel (relaxMPI, relax) runs over each block in lexicographic order
// in the reference.  Updating all nodes of one hyperplane i+j+k = t at once,
// planes in increasing t, gives the same values: a node's lower neighbours
// (and the wrapped-around upper neighbour of the whole-domain levels) lie on
// earlier planes, its upper neighbours on later ones, exactly as in the
// sequential order.  One workgroup sweeps one block, a barrier per plane.
//
// The split levels of at most 16^3 cells and all levels below them run whole
// V-cycles in one workgroup's LDS (k_grav_bottom).
//
// The whole-domain levels 1..NGcr (at most 17^3 nodes) of the set-up run as
// one workgroup (k_grav_coarse) with the potential, right-hand side and
// residual of all levels in LDS (3 x 45 KB), the reference's level-stacked
// layout kept so that the residual's reads past a level's ends hit the same
// neighbouring values.
//
// PB's boundary potential: the x planes' y-z Fourier modes by a radix-2 LDS
// FFT of the plane packed as nn1/2 complex values per row, then the
// reference's real-FFT unpacking (rlft3, SG8:1466-1512) including its
// single-precision twiddles and the in-place double pass over the middle
// column; the Green's-function weights and the sum over planes per mode;
// the same unpacking and FFT backwards.
#include "mcf_grav.h"

#include <type_traits>

namespace mcf {

__device__ __forceinline__ void g_rank(const GravGeo &G, int r, int c[3]) {
  c[0] = r % G.S[0];
  c[2] = r / (G.S[0] * G.S[1]);
  c[1] = r / G.S[0] - G.S[1] * c[2];
}
__device__ __forceinline__ int g_rid(const GravGeo &G, int a, int b, int c) { return a + G.S[0] * (b + G.S[1] * c); }
// Skewed block layout, hyperplane-major: node (i,j,k) at
// j + J (k + K (i+j+k)), J = n1+1, K = n2+1, so that one hyperplane
// i+j+k = t is one contiguous J*K slab, rows of j; the upper neighbours
// sit at +JK (x), +1+JK (y), +J+JK (z), the lower ones at the negatives.
// Slots with i outside 0..n0 are never used.
__device__ __forceinline__ long g_idx(const int *n, int i, int j, int k) {
  return j + (long)(n[1] + 1) * (k + (long)(n[2] + 1) * (i + j + k));
}
__device__ __forceinline__ long g_tid() { return blockIdx.x * (long)blockDim.x + threadIdx.x; }

// Node q (0 <= q < A B) of an A x B rectangle of nodes (a, b) in
// anti-diagonal order: a+b ascending, then b.  With a = i-1, b = j-1 of one
// k plane, neighbouring q are neighbouring slots of the skewed layout (j up,
// i down, i+j+k fixed).  The diagonals' lengths rise 1..m, stay at m, fall
// m-1..1 (m = min(A, B)); the rising and falling parts invert a triangular
// number, the float square root corrected to the exact integer.
__device__ __forceinline__ int g_tri(int q) { // largest s with s(s+1)/2 <= q
  int s = (int)((__builtin_amdgcn_sqrtf(8.0f * (float)q + 1.0f) - 1.0f) * 0.5f);
  while (s * (s + 1) / 2 > q) --s;
  while ((s + 1) * (s + 2) / 2 <= q) ++s;
  return s;
}
__device__ __forceinline__ void g_diag(int A, int B, int q, int &a, int &b) {
  const int m = min(A, B), M = max(A, B), T1 = m * (m + 1) / 2, F = (M - m) * m;
  int s, o;
  if (q < T1) {
    s = g_tri(q);
    o = q - s * (s + 1) / 2;
  } else if (q < T1 + F) {
    s = m + (q - T1) / m;
    o = (q - T1) % m;
  } else {
    const int r = A * B - 1 - q, u = g_tri(r);
    s = A + B - 2 - u;
    o = u - (r - u * (u + 1) / 2);
  }
  b = max(0, s - (A - 1)) + o;
  a = s - b;
}
// node q of a block's nodes 1..n0 x 1..n1 x 1..n2: k planes, each in
// anti-diagonal order
__device__ __forceinline__ void g_node(const int *n, long q, int &i, int &j, int &k) {
  const long AB = (long)n[0] * n[1];
  k = 1 + (int)(q / AB);
  int a, b;
  g_diag(n[0], n[1], (int)(q - (k - 1) * AB), a, b);
  i = 1 + a;
  j = 1 + b;
}

__global__ void k_grav_zero(double *a, long n) {
  for (long t = g_tid(); t < n; t += (long)gridDim.x * blockDim.x) a[t] = 0.0;
}

// mglin's right-hand side at the finest level (SG8:163-167): 4 pi G rho on
// every node 0..C+1 of every rank, the density ghosts included
__global__ void k_grav_rhs(GravGeo G, const double *rho, Geo g, double *rhs2) {
  const int L = G.NGL;
  const int *n = G.n[L];
  const long B = (long)(n[0] + 1) * (n[1] + 1) * (n[2] + 1), t = g_tid();
  if (t >= B * G.npe) return;
  const int r = (int)(t / B);
  long q = t - r * B;
  const int i = (int)(q % (n[0] + 1));
  q /= n[0] + 1;
  const int j = (int)(q % (n[1] + 1)), k = (int)(q / (n[1] + 1));
  int c[3];
  g_rank(G, r, c);
  rhs2[G.off[L] + r * G.bsz[L] + g_idx(n, i, j, k)] =
      rho[ix3(g, c[0] * G.C[0] + i, c[1] * G.C[1] + j, c[2] * G.C[2] + k)] * GRAV_G4PI;
}

// rstrctMPI (SG8:385-456) into split level lc from lc+1, coarse nodes
// 1..nc of every rank: the first node of the first rank and the last node
// of the last rank along an axis are copied, the other inner nodes take
// 1/2 + 6 x 1/12.  The exchange follows as its own launch.
__global__ void k_grav_rstrct(GravGeo G, double *uc2, const double *uf2, int lc) {
  const int *nc = G.n[lc], *nf = G.n[lc + 1];
  const long cnt = (long)nc[0] * nc[1] * nc[2], t = g_tid();
  if (t >= cnt * G.npe) return;
  const int r = (int)(t / cnt);
  int ic[3];
  g_node(nc, t - r * cnt, ic[0], ic[1], ic[2]);
  int c[3];
  g_rank(G, r, c);
  const double *uf = uf2 + G.off[lc + 1] + r * G.bsz[lc + 1];
  double *uc = uc2 + G.off[lc] + r * G.bsz[lc];
  bool copy = false, inner = true;
  for (int d = 0; d < 3; ++d) {
    const bool first = c[d] == 0, last = c[d] == G.S[d] - 1;
    if ((first && ic[d] == 1) || (last && ic[d] == nc[d])) copy = true;
    if (ic[d] < (first ? 2 : 1) || ic[d] > nc[d] - 1) inner = false;
  }
  const int fi = 2 * ic[0] - 1, fj = 2 * ic[1] - 1, fk = 2 * ic[2] - 1;
  const long p = g_idx(nf, fi, fj, fk), J = nf[1] + 1, JK = J * (nf[2] + 1);
  const long sx = JK, sy = 1 + JK, sz = J + JK;
  double v = 0.0;
  bool write = true;
  if (copy) {
    v = uf[p];
  } else if (inner) {
    const double w = 1.0 / 12.0;
    v = 0.5 * uf[p] + w * (uf[p + sx] + uf[p - sx] + uf[p + sy] + uf[p - sy] + uf[p + sz] + uf[p - sz]);
  } else {
    write = false;
  }
  if (write) uc[g_idx(nc, ic[0], ic[1], ic[2])] = v;
}

// Where BCsgr_MPI's six phases take ghost node (i,j,k) of rank c from: walks
// the phases backwards (z, y, x); returns false when no phase moves it.
__device__ __forceinline__ bool g_resolve(const GravGeo &G, const int *n, int c[3], int &i, int &j, int &k, int flags) {
  const int i0 = i, j0 = j, k0 = k;
  if (k == 0 && (flags & 16)) { c[2] = (c[2] + G.S[2] - 1) % G.S[2]; k = n[2] - 1; }
  else if (k == n[2] && (flags & 32)) { c[2] = (c[2] + 1) % G.S[2]; k = 1; }
  if (j == 0 && (flags & 4)) { c[1] = (c[1] + G.S[1] - 1) % G.S[1]; j = n[1] - 1; }
  else if (j == n[1] && (flags & 8)) { c[1] = (c[1] + 1) % G.S[1]; j = 1; }
  if (i == 0 && (flags & 1) && c[0] > 0) { c[0] -= 1; i = n[0] - 1; }
  else if (i == n[0] && (flags & 2) && c[0] < G.S[0] - 1) { c[0] += 1; i = 1; }
  return i != i0 || j != j0 || k != k0;
}

// Ghost node q (0 <= q < grav_nghost(n)) of a block: faces counted once,
// z planes whole, y planes without their z rows, x planes without both.  A
// z plane is walked as (i+j, j) with j fastest, so that neighbouring threads
// touch neighbouring slots of the skewed layout (there and at the source);
// the slots of that walk with i outside 0..n0 are not nodes (false).
__device__ __forceinline__ bool g_ghost(const int *n, int q, int &i, int &j, int &k) {
  const int gz = 2 * (n[0] + n[1] + 1) * (n[1] + 1), gy = 2 * (n[0] + 1) * (n[2] - 1);
  if (q < gz) {
    const int h = (n[0] + n[1] + 1) * (n[1] + 1);
    const int s = q / h, m = q - s * h;
    j = m % (n[1] + 1);
    i = m / (n[1] + 1) - j;
    k = s ? n[2] : 0;
    return i >= 0 && i <= n[0];
  }
  if (q < gz + gy) {
    q -= gz;
    const int h = (n[0] + 1) * (n[2] - 1);
    const int s = q / h, m = q - s * h;
    i = m % (n[0] + 1);
    k = 1 + m / (n[0] + 1);
    j = s ? n[1] : 0;
    return true;
  }
  q -= gz + gy;
  const int h = (n[1] - 1) * (n[2] - 1);
  const int s = q / h, m = q - s * h;
  j = 1 + m % (n[1] - 1);
  k = 1 + m / (n[1] - 1);
  i = s ? n[0] : 0;
  return true;
}

// BCsgr_MPI (SG8:298-336) at split level l.  flags: bit 0 x low, 1 x high,
// 2 y low, 3 y high, 4 z low, 5 z high (the reference's lx1..lz2).  One
// thread per ghost node (a node with a coordinate 0 or n); faces counted
// once: z planes whole, y planes without their z rows, x planes without both.
__global__ void k_grav_exchange(GravGeo G, double *u2, int l, int flags) {
  const int *n = G.n[l];
  const long per = grav_nghost(n), t = g_tid();
  if (t >= per * G.npe) return;
  const int r = (int)(t / per);
  int i, j, k;
  if (!g_ghost(n, (int)(t - r * per), i, j, k)) return;
  int c[3];
  g_rank(G, r, c);
  int si = i, sj = j, sk = k;
  if (!g_resolve(G, n, c, si, sj, sk, flags)) return;
  const int rs = g_rid(G, c[0], c[1], c[2]);
  u2[G.off[l] + r * G.bsz[l] + g_idx(n, i, j, k)] = u2[G.off[l] + rs * G.bsz[l] + g_idx(n, si, sj, sk)];
}

// relaxMPI (SG8:740-870): one Gauss-Seidel sweep of nodes 1..n-1 of one
// rank's block per workgroup, as hyperplanes i+j+k = t; node 1 of the first
// x rank is the boundary, kept by the reference's arithmetic mask.
__global__ __launch_bounds__(GRAV_RELAX_THREADS) void k_grav_relax(GravGeo G, double *phi2, const double *rhs2, int l) {
  const int r = blockIdx.x;
  const int *n = G.n[l];
  int c[3];
  g_rank(G, r, c);
  double *u = phi2 + G.off[l] + r * G.bsz[l];
  const double *rhs = rhs2 + G.off[l] + r * G.bsz[l];
  const double w = 1.0 / 6.0;
  const double h = G.Lbox / (double)((n[0] - 1) * G.S[0]);
  const double h2 = h * h;
  const int li = c[0] == 0 ? 1 : 0;
  const int m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1;
  const long J = n[1] + 1, JK = J * (n[2] + 1), sx = JK, sy = 1 + JK, sz = J + JK;
  for (int t = 3; t <= m0 + m1 + m2; ++t) {
    const int klo = max(1, t - m0 - m1), khi = min(m2, t - 2);
    const int cnt = m1 * (khi - klo + 1);
    for (int q = threadIdx.x; q < cnt; q += blockDim.x) {
      const int j = 1 + q % m1, k = klo + q / m1, i = t - j - k;
      if (i < 1 || i > m0) continue;
      const long p = g_idx(n, i, j, k);
      const int ifl = li * (1 / i);
      const double s = u[p + sx] + u[p - sx] + u[p + sy] + u[p - sy] + u[p + sz] + u[p - sz] - h2 * rhs[p];
      u[p] = w * s * (double)(1 - ifl) + (0.5 + copysign(0.5, (double)ifl - 0.5)) * u[p];
    }
    __syncthreads();
  }
}

// Barrier that orders LDS accesses only: the workgroup's threads exchange
// values through LDS, and global loads still in flight (the next plane's
// prefetch) need not complete first, as they would under __syncthreads.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Orders a wave's own LDS accesses (one lane's write before another's read):
// the LDS serves them in the order issued, so only the compiler is held.
__device__ __forceinline__ void wave_order() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// ---------------------------------------------------------------------------
// Sweeps from one copy of the level into another: a block reads its nodes and
// ghosts from src and writes the swept nodes to dst, then puts those next to
// its faces into the ghosts of the blocks that hold copies of them (in dst,
// which no block reads in this launch), so the level is exchanged when the
// launch ends, and no separate exchange is needed between sweeps or after
// them.  BCsgr_MPI's six phases give a ghost the value of the node that is
// its image along every axis on which it is a ghost (x: only inside the
// domain); seen from that node, it goes out along every combination of the
// axes on which it lies next to a face.  The boundary node n of the last x
// rank is carried along with its y and z images.  Node 0 of the first x rank
// is never written, in either copy.
// ---------------------------------------------------------------------------
struct GPush {
  const GravGeo &G;
  double *level; // dst of the level
  const int *n;
  int c[3];
  long bsz;
  __device__ __forceinline__ int axis(int d, int q) const { return q == 1 ? -1 : (q == n[d] - 1 ? 1 : 0); }
  __device__ __forceinline__ void put(int dx, int dy, int dz, int i, int j, int k, double v) const {
    int a = c[0] + dx, b = c[1] + dy, e = c[2] + dz;
    b = b < 0 ? G.S[1] - 1 : (b == G.S[1] ? 0 : b);
    e = e < 0 ? G.S[2] - 1 : (e == G.S[2] ? 0 : e);
    if (dx) i = dx < 0 ? n[0] : 0;
    if (dy) j = dy < 0 ? n[1] : 0;
    if (dz) k = dz < 0 ? n[2] : 0;
    level[g_rid(G, a, b, e) * bsz + g_idx(n, i, j, k)] = v;
  }
  // The images of all nodes next to a face; val(i, j, k) is the node's new
  // value.  Combinations with x over the x faces, with y but not x over the
  // y faces, z alone over the z faces.
  // xface: node 1 (s = 0) or n-1 (s = 1) along x of column (j, k).
  __device__ __forceinline__ void xface(int s, int j, int k, double v) const {
    const int i = s ? n[0] - 1 : 1, dx = s ? 1 : -1;
    if (c[0] + dx < 0 || c[0] + dx >= G.S[0]) return;
    const int dy = axis(1, j), dz = axis(2, k);
    put(dx, 0, 0, i, j, k, v);
    if (dy) put(dx, dy, 0, i, j, k, v);
    if (dz) put(dx, 0, dz, i, j, k, v);
    if (dy && dz) put(dx, dy, dz, i, j, k, v);
  }
  template <class F> __device__ __forceinline__ void all(F val) const {
    const int m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1;
    for (int q = threadIdx.x; q < 2 * m1 * m2; q += blockDim.x) {
      const int s = q >= m1 * m2, r = q - s * m1 * m2, j = 1 + r % m1, k = 1 + r / m1;
      xface(s, j, k, val(s ? m0 : 1, j, k));
    }
    yzfaces(val);
  }
  template <class F> __device__ __forceinline__ void yzfaces(F val) const {
    const int m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1;
    const int me = c[0] == G.S[0] - 1 ? n[0] : m0; // last node along x carried
    for (int q = threadIdx.x; q < 2 * me * m2; q += blockDim.x) {
      const int s = q >= me * m2, r = q - s * me * m2, i = 1 + r % me, k = 1 + r / me, j = s ? m1 : 1, dy = s ? 1 : -1;
      const int dz = axis(2, k);
      const double v = val(i, j, k);
      put(0, dy, 0, i, j, k, v);
      if (dz) put(0, dy, dz, i, j, k, v);
    }
    // (i+j, j) with j fastest: neighbouring slots, here and at the image
    const int zn = (me + m1 - 1) * m1;
    for (int q = threadIdx.x; q < 2 * zn; q += blockDim.x) {
      const int s = q >= zn, r = q - s * zn, j = 1 + r % m1, i = 2 + r / m1 - j, k = s ? m2 : 1;
      if (i >= 1 && i <= me) put(0, 0, s ? 1 : -1, i, j, k, val(i, j, k));
    }
  }
};

// A sweep of blocks that fit in LDS (at most GRAV_LDS_NODES nodes, ghosts
// included, at most 256 (j,k) columns): the block is loaded whole, swept
// plane by plane with one thread per column (a node's lower x neighbour is
// the thread's last result, the others come from LDS), and written out.  The
// right-hand side is loaded RD planes ahead by every lane, so the loads sit in
// no branch and the compiler can count them.  Bound by the chain of planes
// (an LDS round trip and seven dependent FP64 operations each, and a barrier of
// the waves that hold columns): 8 blocks of 16^3 cells 23 -> 19 us with the
// upper neighbours read a plane ahead, 512 of them 38 -> 34.
typedef unsigned g_u2 __attribute__((ext_vector_type(2)));
constexpr int RD = 4;
__global__ __launch_bounds__(GRAV_LDS_THREADS) void k_grav_relax_lds(GravGeo G, const double *src, double *dst,
                                                                     const double *rhs2, int l) {
  __shared__ double U[GRAV_LDS_NODES];
  const int r = blockIdx.x;
  const int *n = G.n[l];
  int c[3];
  g_rank(G, r, c);
  const long base = G.off[l] + r * G.bsz[l];
  const double *u = src + base, *rhs = rhs2 + base;
  const double w = 1.0 / 6.0;
  const double h = G.Lbox / (double)((n[0] - 1) * G.S[0]);
  const double h2 = h * h;
  const int li = c[0] == 0 ? 1 : 0;
  const int n0 = n[0], m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1, T = m0 + m1 + m2;
  const int I = n[0] + 1, J = n[1] + 1, JK = J * (n[2] + 1), IJ = I * J;
  // load: hyperplanes, contiguous over their (j,k) columns, dealt out to the
  // waves 64 columns at a time; a column without a node on a plane loads
  // nothing (the buffer resource drops its offset).  Sixteen loads in flight
  // per wave.
  const int TM = n[0] + n[1] + n[2], wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
  const __amdgpu_buffer_rsrc_t ub = __builtin_amdgcn_make_buffer_rsrc((void *)u, 0, (int)(8 * G.bsz[l]), 0x00020000);
  for (int q0 = 0; q0 < JK; q0 += 128) {
    int p0[2], jk[2], q[2];
#pragma unroll
    for (int h_ = 0; h_ < 2; ++h_) {
      q[h_] = q0 + 64 * h_ + (int)(threadIdx.x & 63);
      jk[h_] = q[h_] < JK ? q[h_] % J + q[h_] / J : 1 << 20;
      p0[h_] = I * q[h_];
    }
    for (int t0 = wave; t0 <= TM; t0 += 8 * nw) {
      double a[2][8];
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int h_ = 0; h_ < 2; ++h_) {
          const int t = t0 + s * nw;
          const bool ok = (unsigned)(t - jk[h_]) <= (unsigned)n0;
          a[h_][s] = __builtin_bit_cast(
              double, __builtin_amdgcn_raw_buffer_load_b64(ub, ok ? 8u * (unsigned)(q[h_] + JK * t) : 0xffffff00u, 0, 0));
        }
#pragma unroll
      for (int s = 0; s < 8; ++s)
#pragma unroll
        for (int h_ = 0; h_ < 2; ++h_) {
          const int i = t0 + s * nw - jk[h_];
          if ((unsigned)i <= (unsigned)n0) U[p0[h_] + i] = a[h_][s];
        }
    }
  }
  __syncthreads();
  const int q = min((int)threadIdx.x, m1 * m2 - 1), j = 1 + q % m1, k = 1 + q / m1, p0 = I * (j + J * k);
  const bool on = (int)threadIdx.x < m1 * m2; // further waves only load and store
  const double *rc = rhs + j + J * k;
  auto rat = [&](int t) { return rc[(long)JK * min(t, T)]; };
  const double u1 = U[p0 + 1];
  double prev = U[p0], rr[RD];
#pragma unroll
  for (int s = 0; s < RD; ++s) rr[s] = rat(3 + s);
  // the upper neighbours, values from before the sweep, are read a plane
  // ahead, so that a plane's chain is the round trip of the two lower ones.
  // Columns without a node on a plane read what lies there (i runs from 3-j-k
  // to T+RD+1-j-k: inside the block's array, as a row is shorter than the rows
  // before and behind it) and keep nothing.
  double *col = U + p0 - j - k;
  double xu = col[4], yu = col[3 + I], zu = col[3 + IJ];
  const int lo = j + k + 1, cnt = on ? m0 : 0;
  const bool idle = __builtin_amdgcn_readfirstlane((int)threadIdx.x) >= m1 * m2; // no column in this wave
  for (int tb = 3; tb <= T; tb += RD) {
    if (idle) {
#pragma unroll
      for (int s = 0; s < RD; ++s) lds_barrier();
      continue;
    }
#pragma unroll
    for (int s = 0; s < RD; ++s) {
      const int t = tb + s;
      const double ym = col[t - I], zm = col[t - IJ];
      const double sum = xu + prev + yu + ym + zu + zm - h2 * rr[s];
      xu = col[t + 2];
      yu = col[t + 1 + I];
      zu = col[t + 1 + IJ];
      const double v = (li && t == lo) ? u1 : w * sum;
      rr[s] = rat(t + RD);
      const bool act = (unsigned)(t - lo) < (unsigned)cnt;
      if (act) col[t] = v;
      prev = act ? v : prev; // a use outside the branch keeps the loads and the sum out of it
      lds_barrier();
    }
  }
  // write back nodes 1..m0 (to n0 on the last x rank), then the images
  const int me = c[0] == G.S[0] - 1 ? n0 : m0;
  double *d = dst + base + j + J * k;
  if (on)
    for (int t = 3; t <= T + 1; ++t) {
      const int i = t - j - k;
      if (i >= 1 && i <= me) d[(long)JK * t] = U[p0 + i];
    }
  const GPush P{G, dst + G.off[l], n, {c[0], c[1], c[2]}, G.bsz[l]};
  P.all([&](int a, int b, int e) { return U[a + I * (b + J * e)]; });
}

// A sweep of larger blocks, streamed: each thread owns one (j,k) column and
// walks i = t-j-k along it.  The node's lower x neighbour is the thread's own
// last result (a register), its lower y and z neighbours are the neighbouring
// columns' results of the previous plane (LDS, two buffers by plane parity).
// Its upper neighbours are values from before the sweep: along x the one
// loaded for this plane, along y and z the ones the neighbouring columns
// loaded for it (u(i,j+1,k) is the upper x neighbour of their node on the same
// plane), passed on through LDS one plane ahead.  Ghosts on the four j and k
// faces are staged in LDS at the start.  So a plane takes two loads per
// column (upper x neighbour, right-hand side), issued D planes ahead into a
// ring of registers: memory answers in about 2.4 us, four times a plane.
// Loads and stores go through buffer resources, which drop the offsets of idle
// lanes: with loads or stores inside a branch the compiler cannot count how
// many are in flight and waits for all of them.  A wave runs only the planes on
// which one of its columns, or a column next to them, has a node, and waits at
// the barriers of the others.
//
// The x faces go out from registers (a column's first and last result); read
// back from memory they take a cache line per node.  256^3 on 8x8x8: 295 -> 280
// us a sweep, 1.44 TB/s of its compulsory 24 B per node; it moves 1.2 GB, three
// times that, most of it lines of the ghost faces along x and y.  Not kept: the
// y and z faces put into LDS as they are formed (270 us there, but 50 -> 62 us
// for 8 blocks at 64^3, where the chain of planes counts), two workgroups per
// CU (no change), several face values fetched before the first goes out (no
// change).
template <int LMAX, int D>
__global__ __launch_bounds__(GRAV_RELAX_THREADS) void k_grav_relax_col(GravGeo G, const double *src, double *dst,
                                                                       const double *rhs2, int l) {
  // two planes of results (0, 1), two of old values (2, 3), the ghost faces
  // j = 0, k = 0, j = n1, k = n2 (4 .. 7); idle lanes read up to 128 entries
  // past either end of a face
  constexpr int PAD = 128;
  __shared__ double lds[8 * LMAX + PAD];
  const int r = blockIdx.x;
  const int *n = G.n[l];
  int c[3];
  g_rank(G, r, c);
  const long base = G.off[l] + r * G.bsz[l];
  const double *u = src + base, *rhs = rhs2 + base;
  double *d = dst + base;
  const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(d, 0, (int)(8 * G.bsz[l]), 0x00020000);
  const double w = 1.0 / 6.0;
  const double h = G.Lbox / (double)((n[0] - 1) * G.S[0]);
  const double h2 = h * h;
  const int li = c[0] == 0 ? 1 : 0;
  const int m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1, LJ = n[1] + 1, T = m0 + m1 + m2, I1 = n[0] + 1;
  const int JK = LJ * (n[2] + 1);
  {
    const int cy = I1 * (n[2] + 1), cz = I1 * (n[1] + 1); // nodes of a y and of a z face; eight loads in flight
    for (int q0 = threadIdx.x; q0 < max(cy, cz); q0 += 2 * blockDim.x) {
      double f[2][4];
#pragma unroll
      for (int h_ = 0; h_ < 2; ++h_) {
        const int q = q0 + h_ * blockDim.x, y = q < cy ? q : 0, z = q < cz ? q : 0;
        const int yi = y % I1, yk = y / I1, zi = z % I1, zj = z / I1;
        f[h_][0] = u[g_idx(n, yi, 0, yk)];
        f[h_][1] = u[g_idx(n, zi, zj, 0)];
        f[h_][2] = u[g_idx(n, yi, n[1], yk)];
        f[h_][3] = u[g_idx(n, zi, zj, n[2])];
      }
#pragma unroll
      for (int h_ = 0; h_ < 2; ++h_) {
        const int q = q0 + h_ * blockDim.x;
        if (q < cy) {
          lds[4 * LMAX + q] = f[h_][0];
          lds[6 * LMAX + q] = f[h_][2];
        }
        if (q < cz) {
          lds[5 * LMAX + q] = f[h_][1];
          lds[7 * LMAX + q] = f[h_][3];
        }
      }
    }
  }
  const int q = min((int)threadIdx.x, m1 * m2 - 1), j = 1 + q % m1, k = 1 + q / m1, jk = j + k, cell = j + LJ * k;
  // threads past the last column run it once more (the same values) and store nothing
  const bool on = (int)threadIdx.x < m1 * m2;
  double prev = u[cell + JK * jk], v1 = 0.0; // v1: the new value of node 1; prev ends as that of the last node
  const double u1 = u[cell + JK * (jk + 1)]; // nodes 0 and 1 before the sweep
  // planes of this wave: from two before its first column's first node (the
  // old value a neighbour needs, passed on one plane ahead) to its last one
  const int q0 = __builtin_amdgcn_readfirstlane((int)(threadIdx.x & ~63u)), q1 = min(q0 + 63, m1 * m2 - 1);
  const bool row = q0 / m1 == q1 / m1;
  const int t0 = (row ? 1 + q0 % m1 : 1) + 1 + q0 / m1 - 1;
  const int len = (m0 + (row ? 1 + q1 % m1 : m1) + 1 + q1 / m1 - t0 + 1 + D - 1) / D * D;
  const int NB = T + 2 * D; // barriers every wave reaches, planes 1 .. NB
  // Positions in lds of the neighbours read on plane t0 + s, s even (e) and
  // odd (o): fixed in the plane buffers, moving with i on a ghost face.
  // A face has row length I1; positions of idle lanes stay within PAD of it.
  const int pe = t0 & 1, i0 = t0 - jk; // parity of plane t0; i there (>= -m1 - 1, below m0 + m1 + D)
  auto pos = [&](bool face, int f, int fq, int plane, int off) { return face ? f * LMAX + fq + i0 : plane * LMAX + cell + off; };
  int ym[2], zm[2], yp[2], zp[2];
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    ym[s] = pos(j == 1, 4, I1 * k + s, pe ^ s ^ 1, -1);
    zm[s] = pos(k == 1, 5, I1 * j + s, pe ^ s ^ 1, -LJ);
    yp[s] = pos(j == m1, 6, I1 * k + s, 2 + (pe ^ s), 1);
    zp[s] = pos(k == m2, 7, I1 * j + s, 2 + (pe ^ s), LJ);
  }
  const int ay = j == 1 ? 2 : 0, az = k == 1 ? 2 : 0, by = j == m1 ? 2 : 0, bz = k == m2 ? 2 : 0;
  const int wc[2] = {pe * LMAX + cell, (pe ^ 1) * LMAX + cell};                   // own result on an even / odd plane
  const int wx[2] = {(2 + (pe ^ 1)) * LMAX + cell, (2 + pe) * LMAX + cell};       // old value for the next plane
  unsigned so = 8u * (unsigned)(cell + JK * t0);
  double rx[D], rr[D];
  const __amdgpu_buffer_rsrc_t ub = __builtin_amdgcn_make_buffer_rsrc((void *)u, 0, (int)(8 * G.bsz[l]), 0x00020000);
  const __amdgpu_buffer_rsrc_t rb = __builtin_amdgcn_make_buffer_rsrc((void *)rhs, 0, (int)(8 * G.bsz[l]), 0x00020000);
  auto fetch = [&](int s, int i, unsigned off) { // node i of the column, at byte offset off
    const unsigned o = (unsigned)i <= (unsigned)m0 ? off : 0xffffff00u;
    rx[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(ub, o, 8 * JK, 0));
    rr[s] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(rb, o, 0, 0));
  };
  const unsigned sk = 8u * (unsigned)JK;
#pragma unroll
  for (int s = 0; s < D; ++s) fetch(s, i0 + s, so + (unsigned)s * sk);
  __syncthreads();
  for (int b = 1; b < t0; ++b) lds_barrier();
  int i = i0;
  for (int tb = t0; tb < t0 + len; tb += D) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      const int e = s & 1;
      const double vyp = lds[yp[e]], vym = lds[ym[e]], vzp = lds[zp[e]], vzm = lds[zm[e]];
      const double sum = rx[s] + prev + vyp + vym + vzp + vzm - h2 * rr[s];
      const double v = (li && i == 1) ? u1 : w * sum;
      const bool act = (unsigned)(i - 1) < (unsigned)m0;
      lds[wc[e]] = v; // read only by the columns that have this i on the next plane
      lds[wx[e]] = rx[(s + 1) % D];
      prev = act ? v : prev;
      v1 = i == 1 ? v : v1;
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(g_u2, v), db, act && on ? so : 0xffffffffu, 0, 0);
      fetch(s, i + D, so + D * sk);
      ym[e] += ay;
      zm[e] += az;
      yp[e] += by;
      zp[e] += bz;
      so += sk;
      ++i;
      lds_barrier();
    }
  }
  for (int b = t0 + len; b <= NB; ++b) lds_barrier();
  if (c[0] == G.S[0] - 1) // the boundary nodes of the last x rank
    for (int e = threadIdx.x; e < m1 * m2; e += blockDim.x) {
      const long p = g_idx(n, n[0], 1 + e % m1, 1 + e / m1);
      d[p] = u[p];
    }
  __syncthreads(); // the block's stores, before they are read again
  const GPush P{G, dst + G.off[l], n, {c[0], c[1], c[2]}, G.bsz[l]};
  if (on) {
    P.xface(0, j, k, v1);
    P.xface(1, j, k, prev);
  }
  P.yzfaces([&](int a, int b, int e) { return d[g_idx(n, a, b, e)]; });
}
template __global__ void k_grav_relax_col<1156, GRAV_RELAX_D>(GravGeo, const double *, double *, const double *, int);

// The same for blocks of up to four columns per thread, whose faces and old
// values do not fit LDS: the upper y and z neighbours are loaded, the faces
// j = 0 and k = 0 staged.
template <int PP, int LMAX, int D>
__global__ __launch_bounds__(GRAV_RELAX_THREADS) void k_grav_relax_col4(GravGeo G, const double *src, double *dst,
                                                                       const double *rhs2, int l) {
  // two plane buffers, then the ghost faces j = 0 and k = 0
  __shared__ double lds[4 * LMAX];
  const int r = blockIdx.x;
  const int *n = G.n[l];
  int c[3];
  g_rank(G, r, c);
  const long base = G.off[l] + r * G.bsz[l];
  const double *u = src + base, *rhs = rhs2 + base;
  double *d = dst + base;
  const __amdgpu_buffer_rsrc_t db = __builtin_amdgcn_make_buffer_rsrc(d, 0, (int)(8 * G.bsz[l]), 0x00020000);
  const double w = 1.0 / 6.0;
  const double h = G.Lbox / (double)((n[0] - 1) * G.S[0]);
  const double h2 = h * h;
  const int li = c[0] == 0 ? 1 : 0;
  const int m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1, LJ = n[1] + 1, T = m0 + m1 + m2, I1 = n[0] + 1;
  const int JK = LJ * (n[2] + 1);
  double *gyf = lds + 2 * LMAX, *gzf = lds + 3 * LMAX;
  for (int q = threadIdx.x; q < I1 * (n[2] + 1); q += blockDim.x) gyf[q] = u[g_idx(n, q % I1, 0, q / I1)];
  for (int q = threadIdx.x; q < I1 * (n[1] + 1); q += blockDim.x) gzf[q] = u[g_idx(n, q % I1, q / I1, 0)];
  int pj[PP], pk[PP];
  bool on[PP];
  double prev[PP], u1[PP]; // the lower x neighbour; node 1 before the sweep
  // ring slot s: the loads of the node on plane t = t0 + s (mod D)
  double rx[D][PP], ry[D][PP], rz[D][PP], rr[D][PP];
#pragma unroll
  for (int p = 0; p < PP; ++p) {
    // columns past the last one run it once more (the same values) and store nothing
    const int q = min((int)(threadIdx.x + p * blockDim.x), m1 * m2 - 1);
    on[p] = (int)(threadIdx.x + p * blockDim.x) < m1 * m2;
    pj[p] = 1 + q % m1;
    pk[p] = 1 + q / m1;
    const long q1 = g_idx(n, 1, pj[p], pk[p]);
    prev[p] = u[q1 - JK];
    u1[p] = u[q1];
  }
  // 32-bit byte offsets from the block's (uniform) base: one register per address
  auto at = [](const double *b, unsigned off) { return *(const double *)((const char *)b + off); };
  const unsigned bx = 8u * (unsigned)JK, by = bx + 8u, bz = bx + 8u * (unsigned)LJ;
  auto fetch = [&](int s, int p, int t) {
    const unsigned q = 8u * (unsigned)(pj[p] + LJ * pk[p] + JK * min(t, T));
    rx[s][p] = at(u, q + bx);
    ry[s][p] = at(u, q + by);
    rz[s][p] = at(u, q + bz);
    rr[s][p] = at(rhs, q);
  };
  const int t0 = 3, len = (T - 2 + D - 1) / D * D;
#pragma unroll
  for (int s = 0; s < D; ++s)
#pragma unroll
    for (int p = 0; p < PP; ++p) fetch(s, p, t0 + s);
  __syncthreads();
  for (int tb = t0; tb < t0 + len; tb += D) {
#pragma unroll
    for (int s = 0; s < D; ++s) {
      const int t = tb + s;
      double *Lc = lds + (t & 1) * LMAX;
      const double *Lp = lds + ((t + 1) & 1) * LMAX;
#pragma unroll
      for (int p = 0; p < PP; ++p) {
        const int i = t - pj[p] - pk[p], ic = min(max(i, 1), m0), cell = pj[p] + LJ * pk[p];
        const double ym = *(pj[p] == 1 ? gyf + ic + I1 * pk[p] : Lp + cell - 1);
        const double zm = *(pk[p] == 1 ? gzf + ic + I1 * pj[p] : Lp + cell - LJ);
        const double sum = rx[s][p] + prev[p] + ry[s][p] + ym + rz[s][p] + zm - h2 * rr[s][p];
        const double v = (li && i == 1) ? u1[p] : w * sum;
        const bool act = i >= 1 && i <= m0;
        Lc[cell] = v; // read only by the columns that have this i on the next plane
        prev[p] = act ? v : prev[p];
        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(g_u2, v), db, act && on[p] ? 8u * (unsigned)(cell + JK * t) : 0xffffffffu, 0, 0);
        fetch(s, p, t + D);
      }
      lds_barrier();
    }
  }
  if (c[0] == G.S[0] - 1) // the boundary nodes of the last x rank
    for (int q = threadIdx.x; q < m1 * m2; q += blockDim.x) {
      const long p = g_idx(n, n[0], 1 + q % m1, 1 + q / m1);
      d[p] = u[p];
    }
  __syncthreads(); // the block's stores, before they are read again
  const GPush P{G, dst + G.off[l], n, {c[0], c[1], c[2]}, G.bsz[l]};
  P.all([&](int a, int b, int e) { return d[g_idx(n, a, b, e)]; });
}
template __global__ void k_grav_relax_col4<4, 4356, GRAV_RELAX_D4>(GravGeo, const double *, double *, const double *, int);

// residMPI's expression
__device__ __forceinline__ double g_res7(double xp, double xm, double yp, double ym, double zp, double zm, double u,
                                         double h2i, double rhs) {
  return -h2i * (xp + xm + yp + ym + zp + zm - 6.0 * u) + rhs;
}

// residMPI (SG8:918-952) and its exchange at one node of split level l: node
// (i,j,k) of rank c, a ghost taken to the node it is a copy of (whose
// neighbours, ghosts included, are in its own block); zero at the x-end nodes.
__device__ __forceinline__ double g_resid(const GravGeo &G, const double *phi2, const double *rhs2, int l, const int c_[3],
                                          int i, int j, int k) {
  const int *n = G.n[l];
  int c[3] = {c_[0], c_[1], c_[2]};
  g_resolve(G, n, c, i, j, k, 63);
  if ((c[0] == 0 && i <= 1) || (c[0] == G.S[0] - 1 && i == n[0])) return 0.0;
  const long p = G.off[l] + g_rid(G, c[0], c[1], c[2]) * G.bsz[l] + g_idx(n, i, j, k);
  const double *u = phi2 + p;
  const double h = G.Lbox / (double)((n[0] - 1) * G.S[0]);
  const double h2i = 1.0 / (h * h);
  const long J = n[1] + 1, JK = J * (n[2] + 1), sx = JK, sy = 1 + JK, sz = J + JK;
  return g_res7(u[sx], u[-sx], u[sy], u[-sy], u[sz], u[-sz], u[0], h2i, rhs2[p]);
}

// The way down from split level lc+1 to lc: residual, its restriction
// (rstrctMPI, mode 1) into the right-hand side of lc at the nodes 1..n-1
// (the only ones read there), and the potential of lc set to zero.  The
// residual is formed where the restriction reads it (7 points per coarse
// node, 7/8 of a pass over the fine nodes), so it is neither stored nor
// exchanged: one launch instead of residual, exchange, restriction, exchange
// and zeroing (20 ways down a solve; 256^3 on 8x8x8: 0.69 against 1.9 ms).
__global__ void k_grav_down(GravGeo G, const double *phif, double *phic, double *rhs2, int lc) {
  const int *nc = G.n[lc];
  const int m[3] = {nc[0] - 1, nc[1] - 1, nc[2] - 1};
  const long cnt = (long)m[0] * m[1] * m[2], t = g_tid();
  const long nz = G.bsz[lc] * G.npe, all = (long)gridDim.x * blockDim.x;
  for (long q = t; q < nz; q += all) phic[G.off[lc] + q] = 0.0;
  if (t >= cnt * G.npe) return;
  const int r = (int)(t / cnt);
  int ic[3];
  g_node(m, t - r * cnt, ic[0], ic[1], ic[2]);
  int c[3];
  g_rank(G, r, c);
  bool copy = false;
  for (int d = 0; d < 3; ++d)
    if (c[d] == 0 && ic[d] == 1) copy = true;
  const int fi = 2 * ic[0] - 1, fj = 2 * ic[1] - 1, fk = 2 * ic[2] - 1, lf = lc + 1;
  double v = 0.0;
  if (!(c[0] == 0 && ic[0] == 1)) {
    auto R = [&](int i, int j, int k) { return g_resid(G, phif, rhs2, lf, c, i, j, k); };
    v = R(fi, fj, fk);
    if (!copy) {
      const double w = 1.0 / 12.0;
      v = 0.5 * v + w * (R(fi + 1, fj, fk) + R(fi - 1, fj, fk) + R(fi, fj + 1, fk) + R(fi, fj - 1, fk) +
                         R(fi, fj, fk + 1) + R(fi, fj, fk - 1));
    }
  }
  rhs2[G.off[lc] + r * G.bsz[lc] + g_idx(nc, ic[0], ic[1], ic[2])] = v;
}

// Prolongation of interpMPI / interp (SG8:500-599): injection at odd
// nodes, then the mean of the two neighbours along x (odd y, z), along y
// (odd z) and along z, in that order; each node's value is formed directly
// from the coarse nodes with the same operations.
template <class F>
__device__ __forceinline__ double pro_w(const F &C, int i, int j, int k) { // j, k odd
  return (i & 1) ? C(i, j, k) : .5 * (C(i + 1, j, k) + C(i - 1, j, k));
}
template <class F>
__device__ __forceinline__ double pro_v(const F &C, int i, int j, int k) { // k odd
  return (j & 1) ? pro_w(C, i, j, k) : .5 * (pro_w(C, i, j + 1, k) + pro_w(C, i, j - 1, k));
}
template <class F>
__device__ __forceinline__ double pro_node(const F &C, int i, int j, int k) {
  return (k & 1) ? pro_v(C, i, j, k) : .5 * (pro_v(C, i, j, k + 1) + pro_v(C, i, j, k - 1));
}

// interpMPI into split level lf with its exchange of the low ghosts: nodes
// 0..nf of every rank, a low ghost taken to the node it is a copy of and
// formed from that rank's coarse block (node 0 of the first x rank stays).
// Mode 1 writes the potential, with the end-plane potential on the x-end
// nodes; mode 0 adds to it (addintMPI, SG8:602-624; the interpolant is
// neither stored nor exchanged).  An odd coordinate's two coarse nodes are
// one and the same, and 0.5 (c + c) = c, so every node takes eight loads and
// no branch.  flat: the coarse level lies as k_grav_bottom leaves it, whole,
// without ghosts.
__global__ void k_grav_prolong(GravGeo G, double *phif, const double *phic, int lf, int mode, const double *bphi2, int flat) {
  const int *nf = G.n[lf], *nc = G.n[lf - 1];
  const int m[3] = {nf[0] + 1, nf[1] + 1, nf[2] + 1};
  const long cnt = (long)m[0] * m[1] * m[2], t = g_tid();
  if (t >= cnt * G.npe) return;
  const int r = (int)(t / cnt);
  int i, j, k;
  g_node(m, t - r * cnt, i, j, k);
  --i; --j; --k;
  int c[3];
  g_rank(G, r, c);
  if (c[0] == 0 && i == 0) return;
  const long out = G.off[lf] + r * G.bsz[lf] + g_idx(nf, i, j, k);
  int rs = r;
  if (i == 0 || j == 0 || k == 0) {
    g_resolve(G, nf, c, i, j, k, 1 | 4 | 16);
    rs = g_rid(G, c[0], c[1], c[2]);
  }
  double v;
  const int side = (c[0] == 0 && i == 1) ? 0 : ((c[0] == G.S[0] - 1 && i == nf[0]) ? 1 : -1);
  if (mode == 1 && side >= 0) {
    v = bphi2[G.boff[lf] + (2L * rs + side) * (long)(nf[1] + 1) * (nf[2] + 1) + j + (long)(nf[1] + 1) * k];
  } else {
    // the upper coarse node of each axis is (f+2)/2; the lower one f/2 at an
    // even coordinate, the same node at an odd one
    const int iu = (i + 2) / 2, ju = (j + 2) / 2, ku = (k + 2) / 2;
    auto mean = [](const double *u, long sx, long sy, long sz) {
      auto w = [&](long o) { return .5 * (u[-o] + u[-o - sx]); };
      auto vv = [&](long o) { return .5 * (w(o) + w(o + sy)); };
      return .5 * (vv(0) + vv(sz));
    };
    if (flat) {
      const int Nc = 1 << (lf - 1), X = c[0] * (nc[0] - 1) + iu, Y = c[1] * (nc[1] - 1) + ju, Z = c[2] * (nc[2] - 1) + ku;
      const int Yw = Y > Nc ? 1 : Y, Zw = Z > Nc ? 1 : Z, sy = Nc + 1, sz = sy * Nc;
      v = mean(phic + (X - 1) + sy * (Yw - 1) + sz * (Zw - 1), !(i & 1), (j & 1) ? 0 : sy * (Yw == Y ? 1 : 1 - Nc),
               (k & 1) ? 0 : sz * (Zw == Z ? 1 : 1 - Nc));
    } else {
      const long J = nc[1] + 1, JK = J * (nc[2] + 1);
      v = mean(phic + G.off[lf - 1] + rs * G.bsz[lf - 1] + g_idx(nc, iu, ju, ku), (i & 1) ? 0 : JK, (j & 1) ? 0 : 1 + JK,
               (k & 1) ? 0 : J + JK);
    }
  }
  if (mode == 1) phif[out] = v;
  else phif[out] = phif[out] + v;
}

// collect (SG8:339-366): the level-NGcr rank blocks into the whole-domain
// level NGcr (2^NGcr+1 nodes per axis, node 1 first, 1-based offset p1)
__global__ void k_grav_collect(GravGeo G, double *u1, const double *u2) {
  const int L = G.NGcr, N1 = (1 << L) + 1;
  const int *m = G.n[L];
  const long t = g_tid();
  if (t >= (long)N1 * N1 * N1) return;
  const int gi = 1 + (int)(t % N1), gj = 1 + (int)((t / N1) % N1), gk = 1 + (int)(t / ((long)N1 * N1));
  const int g3[3] = {gi, gj, gk};
  int c[3], lo[3];
  for (int d = 0; d < 3; ++d) {
    c[d] = min((g3[d] - 1) / (m[d] - 1), G.S[d] - 1);
    lo[d] = g3[d] - c[d] * (m[d] - 1);
  }
  const int r = g_rid(G, c[0], c[1], c[2]);
  u1[G.p1[L] + t] = u2[G.off[L] + r * G.bsz[L] + g_idx(m, lo[0], lo[1], lo[2])];
}

// divide (SG8:369-382): whole-domain level NGcr into the rank blocks, the
// node-0 planes of the first rank along each axis left as they are
__global__ void k_grav_divide(GravGeo G, double *u2, const double *u1) {
  const int L = G.NGcr, N1 = (1 << L) + 1;
  const int *m = G.n[L];
  const long B = (long)(m[0] + 1) * (m[1] + 1) * (m[2] + 1), t = g_tid();
  if (t >= B * G.npe) return;
  const int r = (int)(t / B);
  long q = t - r * B;
  int id[3];
  id[0] = (int)(q % (m[0] + 1));
  q /= m[0] + 1;
  id[1] = (int)(q % (m[1] + 1));
  id[2] = (int)(q / (m[1] + 1));
  int c[3];
  g_rank(G, r, c);
  int g3[3];
  for (int d = 0; d < 3; ++d) {
    if (c[d] == 0 && id[d] == 0) return;
    g3[d] = c[d] * (m[d] - 1) + id[d];
  }
  u2[G.off[L] + r * G.bsz[L] + g_idx(m, id[0], id[1], id[2])] =
      u1[G.p1[L] + (g3[0] - 1) + (long)N1 * ((g3[1] - 1) + (long)N1 * (g3[2] - 1))];
}

// ---------------------------------------------------------------------------
// whole-domain levels, one workgroup
// ---------------------------------------------------------------------------
struct Coarse {
  const GravGeo &G;
  const GravBuf &B;
  double *phi, *rhs, *res; // LDS, 1-based
};

__device__ __forceinline__ int c_at(int off, int n, int i, int j, int k) {
  return off + (i - 1) + n * ((j - 1) + n * (k - 1));
}

// rstrct (SG8:459-497): inner nodes weighted, the six faces copied, mode 1
// zeroes the x faces
__device__ void c_rstrct(double *uc, int offc, const double *uf, int offf, int nc, int mode) {
  const int nf = 2 * nc - 1;
  const int cnt = nc * nc * nc;
  for (int q = threadIdx.x; q < cnt; q += blockDim.x) {
    const int ic = 1 + q % nc, jc = 1 + (q / nc) % nc, kc = 1 + q / (nc * nc);
    const bool face = ic == 1 || ic == nc || jc == 1 || jc == nc || kc == 1 || kc == nc;
    const int p = c_at(offf, nf, 2 * ic - 1, 2 * jc - 1, 2 * kc - 1);
    double v;
    if (face) {
      v = uf[p];
    } else {
      const double w = 1.0 / 12.0;
      v = 0.5 * uf[p] + w * (uf[p + 1] + uf[p - 1] + uf[p + nf] + uf[p - nf] + uf[p + nf * nf] + uf[p - nf * nf]);
    }
    if (mode == 1 && (ic == 1 || ic == nc)) v = 0.0;
    uc[c_at(offc, nc, ic, jc, kc)] = v;
  }
  __syncthreads();
}

// interp (SG8:557-599); mode 1 sets the x faces from the end-plane potential
__device__ void c_interp(const Coarse &S, double *uf, int offf, const double *uc, int offc, int nf, int np, int mode) {
  const int nc = nf / 2 + 1;
  const int cnt = nf * nf * nf;
  for (int q = threadIdx.x; q < cnt; q += blockDim.x) {
    const int i = 1 + q % nf, j = 1 + (q / nf) % nf, k = 1 + q / (nf * nf);
    double v;
    if (mode == 1 && (i == 1 || i == nf)) {
      v = S.B.bphi1[(i == 1 ? 0 : S.G.needb1 + 1) + np + (j - 1) + nf * (k - 1)];
    } else {
      auto C = [&](int a, int b, int e) { return uc[c_at(offc, nc, (a + 1) / 2, (b + 1) / 2, (e + 1) / 2)]; };
      v = pro_node(C, i, j, k);
    }
    uf[c_at(offf, nf, i, j, k)] = v;
  }
  __syncthreads();
}

// relax (SG8:873-915): x nodes 2..n-1, y and z wrapped with period n.
// Hyperplanes i+j+k = t; only levels below NGcr are relaxed here (n <= 9), so
// the workgroup's first wave sweeps alone, each lane on one or two (j,k)
// columns with their wrapped neighbours' offsets formed once.  The LDS serves
// a wave's accesses in order, so a plane needs no barrier: it takes an LDS
// round trip and its nine dependent operations (0.12 us; 0.55 us with a barrier
// of sixteen waves).
static_assert(((1 << (GRAV_MAX_NGCR - 1)) + 1) * ((1 << (GRAV_MAX_NGCR - 1)) + 1) <= 128, "two columns per lane");
__device__ __forceinline__ void c_relax(const Coarse &S, double *u, int off, const double *rhs, int n, int times) {
  const double w = 1.0 / 6.0;
  const double h = S.G.Lbox / (double)(n - 1);
  const double h2 = h * h;
  if (threadIdx.x < 64) {
    int base[2], oyp[2], oym[2], ozp[2], ozm[2], lo[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int q = threadIdx.x + 64 * e, j = q < n * n ? 1 + q % n : 1, k = q < n * n ? 1 + q / n : 1;
      lo[e] = q < n * n ? j + k + 2 : 1 << 20; // no node on any plane
      base[e] = c_at(off, n, 0, j, k) - j - k;
      oym[e] = n * ((j == 1 ? n : j - 1) - j);
      oyp[e] = n * ((j == n ? 1 : j + 1) - j);
      ozm[e] = n * n * ((k == 1 ? n : k - 1) - k);
      ozp[e] = n * n * ((k == n ? 1 : k + 1) - k);
    }
    // one or two columns per lane; the x, y and z upper neighbours and the
    // right-hand side are read a plane ahead (a wrapped one was written n-1
    // planes before); columns without a node on a plane read what lies there,
    // at most n+4 entries past the level, and keep nothing
    auto sweep = [&](auto two) {
      constexpr int E = decltype(two)::value;
      for (int s = 0; s < times; ++s) {
        double xu[E], yu[E], zu[E], rr[E], prev[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
          const double *P = u + base[e];
          prev[e] = P[lo[e] < 64 ? lo[e] - 1 : 3];
          xu[e] = P[5];
          yu[e] = P[4 + oyp[e]];
          zu[e] = P[4 + ozp[e]];
          rr[e] = rhs[base[e] + 4];
        }
        for (int tb = 4; tb <= (n - 1) + 2 * n; tb += 4) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int t = tb + g;
            double v[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
              const double *P = u + base[e];
              const double ym = P[t + oym[e]], zm = P[t + ozm[e]];
              v[e] = w * (xu[e] + prev[e] + yu[e] + ym + zu[e] + zm - h2 * rr[e]);
              xu[e] = P[t + 2];
              yu[e] = P[t + 1 + oyp[e]];
              zu[e] = P[t + 1 + ozp[e]];
              rr[e] = rhs[base[e] + t + 1];
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
              const bool act = (unsigned)(t - lo[e]) < (unsigned)(n - 2);
              if (act) u[base[e] + t] = v[e];
              prev[e] = act ? v[e] : prev[e];
            }
            wave_order();
          }
        }
      }
    };
    if (n * n <= 64) sweep(std::integral_constant<int, 1>{});
    else sweep(std::integral_constant<int, 2>{});
  }
  __syncthreads();
}

// resid (SG8:955-971): the y and z neighbours at flat offsets +-n, +-n^2,
// past the level's ends for its first and last rows and planes
__device__ void c_resid(const Coarse &S, double *res, const double *u, const double *rhs, int off, int n) {
  const double h = S.G.Lbox / (double)(n - 1);
  const double h2i = 1.0 / (h * h);
  const int cnt = n * n * n, nn = n * n;
  for (int q = threadIdx.x; q < cnt; q += blockDim.x) {
    const int i = 1 + q % n;
    const int p = off + q;
    if (i == 1 || i == n) {
      res[p] = 0.0;
    } else {
      res[p] = -h2i * (u[p + 1] + u[p - 1] + u[p + n] + u[p - n] + u[p + nn] + u[p - nn] - 6.0 * u[p]) + rhs[p];
    }
  }
  __syncthreads();
}

__device__ void c_fill0(double *u, int off, int n) {
  const int cnt = n * n * n;
  for (int q = threadIdx.x; q < cnt; q += blockDim.x) u[off + q] = 0.0;
  __syncthreads();
}

__device__ void c_copy(double *dst, int off, const double *src, int n) {
  const int cnt = n * n * n;
  for (int q = threadIdx.x; q < cnt; q += blockDim.x) dst[off + q] = src[off + q];
  __syncthreads();
}

__device__ __forceinline__ double w3(int j, int k, int jp, int kp) {
  return (j == jp && k == kp) ? 8.0 : ((j == jp || k == kp) ? 2.0 : 1.0);
}

// slvsml (SG8:651-679): exact 3^3 solve, zero x faces; b = 1 is slvsmlb
// (SG8:682-737) with the end-plane potential on the x faces
__device__ void c_slvsml(const Coarse &S, const double *rhs, int b) {
  const double h = 0.5 * S.G.Lbox;
  const int off = S.G.p1[1];
  double *u = S.phi;
  const int q = threadIdx.x;
  if (q < 9) {
    const int j = 1 + q % 3, k = 1 + q / 3;
    u[c_at(off, 3, 1, j, k)] = b ? S.B.bphi1[S.G.pb1[1] + (j - 1) + 3 * (k - 1)] : 0.0;
    u[c_at(off, 3, 3, j, k)] = b ? S.B.bphi1[S.G.needb1 + 1 + S.G.pb1[1] + (j - 1) + 3 * (k - 1)] : 0.0;
  }
  __syncthreads();
  if (q < 9) {
    const int j = 1 + q % 3, k = 1 + q / 3;
    double s = 0.0;
    if (b) {
      bool first = true;
      for (int side = 1; side <= 3; side += 2)
        for (int jp = 1; jp <= 3; ++jp)
          for (int kp = 1; kp <= 3; ++kp) {
            const double t = w3(j, k, jp, kp) * u[c_at(off, 3, side, jp, kp)];
            s = first ? t : s + t;
            first = false;
          }
      for (int jp = 1; jp <= 3; ++jp)
        for (int kp = 1; kp <= 3; ++kp) s = s - w3(j, k, jp, kp) * h * h * rhs[c_at(off, 3, 2, jp, kp)];
      s = 0.025 * s;
    } else {
      bool first = true;
      for (int jp = 1; jp <= 3; ++jp)
        for (int kp = 1; kp <= 3; ++kp) {
          const double t = w3(j, k, jp, kp) * rhs[c_at(off, 3, 2, jp, kp)];
          s = first ? -t : s - t;
          first = false;
        }
      s = 0.025 * h * h * s;
    }
    u[c_at(off, 3, 2, j, k)] = s;
  }
  __syncthreads();
}

// addint (SG8:627-648): res = prolongation of level l-1, phi(l) += res
__device__ void c_addint(const Coarse &S, int l) {
  const int nf = (1 << l) + 1;
  c_interp(S, S.res, S.G.p1[l], S.phi, S.G.p1[l - 1], nf, 0, 0);
  const int cnt = nf * nf * nf, off = S.G.p1[l];
  for (int q = threadIdx.x; q < cnt; q += blockDim.x) S.phi[off + q] = S.phi[off + q] + S.res[off + q];
  __syncthreads();
}

// the downward leg from level top-1 (whose right-hand side is set) to 2,
// the exact 3^3 solve and the upward leg to top-1 (mglin SG8:200-270)
__device__ void c_vcycle_lower(const Coarse &S, int top) {
  const GravGeo &G = S.G;
  for (int jj = top - 1; jj >= 2; --jj) {
    const int n = (1 << jj) + 1;
    c_relax(S, S.phi, G.p1[jj], S.rhs, n, 5);
    c_resid(S, S.res, S.phi, S.rhs, G.p1[jj], n);
    c_rstrct(S.rhs, G.p1[jj - 1], S.res, G.p1[jj], (1 << (jj - 1)) + 1, 1);
    c_fill0(S.phi, G.p1[jj - 1], (1 << (jj - 1)) + 1);
  }
  c_slvsml(S, S.rhs, 0);
  for (int jj = 2; jj <= top - 1; ++jj) {
    c_addint(S, jj);
    c_relax(S, S.phi, G.p1[jj], S.rhs, (1 << jj) + 1, 5);
  }
}

// 2D restriction of an end plane (PB, SG8:1394-1460): 1/2 centre + 1/8
// per in-plane neighbour, a missing neighbour's weight moved to the centre
__device__ __forceinline__ double plane_restrict(const double *bf, long kf, long stride, int ic, int jc, int mcx, int mcy) {
  const double w = 0.125;
  const bool hl = ic > 1, hr = ic < mcx, hd = jc > 1, hu = jc < mcy;
  const double cw = (double)(4 + !hl + !hr + !hd + !hu) * w;
  const long nb[4] = {kf - 1, kf + 1, kf - stride, kf + stride};
  const bool has[4] = {hl, hr, hd, hu};
  double sum = 0.0;
  bool first = true;
  for (int qq = 0; qq < 4; ++qq)
    if (has[qq]) {
      sum = first ? bf[nb[qq]] : sum + bf[nb[qq]];
      first = false;
    }
  return cw * bf[kf] + w * sum;
}

__global__ __launch_bounds__(GRAV_COARSE_THREADS) void k_grav_coarse(GravGeo G, GravBuf B, int prog, int jst) {
  __shared__ double sphi[GRAV_NEED1_MAX + 1], srhs[GRAV_NEED1_MAX + 1], sres[GRAV_NEED1_MAX + 1];
  // all loads of the three arrays in flight at once (GRAV_COARSE_THREADS
  // threads, GRAV_NEED1_MAX + 1 entries each)
  constexpr int CU = (GRAV_NEED1_MAX + GRAV_COARSE_THREADS) / GRAV_COARSE_THREADS;
  const long need = G.need1;
  {
    double a[CU], b[CU], c[CU];
#pragma unroll
    for (int q = 0; q < CU; ++q) {
      const long p = threadIdx.x + (long)q * GRAV_COARSE_THREADS;
      if (p <= need) {
        a[q] = B.phi1[p];
        b[q] = B.rhs1[p];
        c[q] = B.res1[p];
      }
    }
#pragma unroll
    for (int q = 0; q < CU; ++q) {
      const long p = threadIdx.x + (long)q * GRAV_COARSE_THREADS;
      if (p <= need) {
        sphi[p] = a[q];
        srhs[p] = b[q];
        sres[p] = c[q];
      }
    }
  }
  __syncthreads();
  const Coarse S{G, B, sphi, srhs, sres};
  const int L = G.NGcr, N1 = (1 << L) + 1;
  if (prog == 0) {
    // crho1 down to level 1, the end-plane potential likewise, slvsmlb
    for (int l = L - 1; l >= 1; --l) c_rstrct(B.rho1, G.p1[l], B.rho1, G.p1[l + 1], (1 << l) + 1, 0);
    for (int lc = L - 1; lc >= 1; --lc) {
      const int ncu = (1 << lc) + 1, nf = 2 * ncu - 1;
      for (long q = threadIdx.x; q < 2L * ncu * ncu; q += blockDim.x) {
        const int side = (int)(q / ((long)ncu * ncu)), m = (int)(q % ((long)ncu * ncu));
        const int ic = 1 + m % ncu, jc = 1 + m / ncu;
        double *bl = B.bphi1 + side * (G.needb1 + 1);
        const long kf = (2 * ic - 2) + (long)nf * (2 * jc - 2), kc = (ic - 1) + (long)ncu * (jc - 1);
        bl[G.pb1[lc] + kc] = plane_restrict(bl + G.pb1[lc + 1], kf, nf, ic, jc, ncu, ncu);
      }
      __syncthreads();
    }
    c_slvsml(S, B.rho1, 1);
  } else if (prog == 1) {
    // FMG stage jst < NGcr: candidate solution, then two V-cycles
    const int nf = (1 << jst) + 1;
    c_interp(S, sphi, G.p1[jst], sphi, G.p1[jst - 1], nf, G.pb1[jst], 1);
    c_copy(srhs, G.p1[jst], B.rho1, nf);
    for (int cyc = 0; cyc < 2; ++cyc) {
      c_relax(S, sphi, G.p1[jst], srhs, nf, 5);
      c_resid(S, sres, sphi, srhs, G.p1[jst], nf);
      c_rstrct(srhs, G.p1[jst - 1], sres, G.p1[jst], (1 << (jst - 1)) + 1, 1);
      c_fill0(sphi, G.p1[jst - 1], (1 << (jst - 1)) + 1);
      c_vcycle_lower(S, jst);
      c_addint(S, jst);
      c_relax(S, sphi, G.p1[jst], srhs, nf, 5);
    }
  } else {
    // FMG stage NGcr, whole-domain part
    c_interp(S, sphi, G.p1[L], sphi, G.p1[L - 1], N1, G.pb1[L], 1);
    c_copy(srhs, G.p1[L], B.rho1, N1);
  }
  for (long p = threadIdx.x; p <= need; p += blockDim.x) {
    B.phi1[p] = sphi[p];
    B.rhs1[p] = srhs[p];
    B.res1[p] = sres[p];
  }
}

// ---------------------------------------------------------------------------
// V-cycles of the small split levels, one workgroup
// ---------------------------------------------------------------------------
// Levels NGcr..top (top <= GRAV_BOT_TOP, NGcr >= 2) as whole domains in LDS:
// nodes 1..N+1 x 1..N x 1..N of each level (N = 2^l), y and z wrapped, in two
// copies, and the right-hand side.  Rows of x are N+2 apart and z planes
// N(N+2)+9: the columns of a hyperplane (x falls as y or z rises) then spread
// evenly over the banks (with N+1 eight of them met in one bank).  The blocks
// of the split show in the sweeps alone: a node's lower neighbours inside its
// block are the sweep's own results (the copy written), all others the values
// from before it (the copy read), which is what the exchanged ghosts of a
// split level hold.  The whole-domain levels below NGcr are k_grav_coarse's;
// the whole-domain form of NGcr itself is level NGcr here, its nodes N+1 along
// y and z apart from the wrapped node 1 only in the correction: divide hands
// them to the last ranks' high ghosts and leaves the first ranks' low ghosts
// as they were, so the first sweep after it takes these from ghost planes.
//
// Bound by the chain of planes (an LDS round trip of 68 cycles and seven
// dependent FP64 operations of 13 each: 0.1 us a plane in a wave alone; a
// barrier of eight waves a plane doubles it).  On separate launches these
// levels cost a launch per sweep, 5 to 9 us each for 0.3 to 3 us of work: a
// V-cycle from level 4 takes 80 us instead of about 300 on 2x2x2 blocks, 110
// instead of 190 on 8x8x8; a step with self-gravity 3.48 -> 2.0 ms at 64^3 on
// 2x2x2, 15.8 -> 15.0 ms at 256^3 on 8x8x8.

// The thread's index, read anew: what is formed from it is not carried in
// registers from one part of the kernel to the next (128 are all there are).
__device__ __forceinline__ int b_tid() {
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}

struct Bot {
  const GravGeo &G;
  double *s; // level NGcr's two copies and right-hand side, then the next level's
  int flip; // bit l: the level's current copy
  __device__ __forceinline__ static int rs(int l) { return (1 << l) + 2; }
  __device__ __forceinline__ static int zs(int l) { return (rs(l) << l) + 9; }
  __device__ __forceinline__ static int size(int l) { return zs(l) << l; }
  __device__ __forceinline__ double *level(int l) const { // two copies, then the right-hand side
    int o = 0;
    for (int q = G.NGcr; q < l; ++q) o += 3 * size(q);
    return s + o;
  }
  __device__ __forceinline__ double *cur(int l) const { return level(l) + ((flip >> l) & 1) * size(l); }
  __device__ __forceinline__ double *other(int l) const { return level(l) + (~(flip >> l) & 1) * size(l); }
  __device__ __forceinline__ double *rhs(int l) const { return level(l) + 2 * size(l); }
  // node (X, Y, Z), 1-based
  __device__ __forceinline__ static int at(int l, int X, int Y, int Z) {
    return (X - 1) + rs(l) * (Y - 1) + zs(l) * (Z - 1);
  }
  // f(X, Y, Z) at every node, dealt out to the threads
  template <class F> __device__ __forceinline__ static void each(int l, F f) {
    const int N = 1 << l, NX = N + 1;
    for (int q = b_tid(); q < NX << (2 * l); q += blockDim.x) {
      const int yz = q / NX;
      f(1 + q - yz * NX, 1 + (yz & (N - 1)), 1 + (yz >> l));
    }
  }
  __device__ __forceinline__ double h(int l) const { return G.Lbox / (double)((G.n[l][0] - 1) * G.S[0]); }
};

// ghost planes of level NGcr, size = (N+1) N each: low and high y, low and high z
struct BotGhost {
  double *base;
  int size;
  __device__ __forceinline__ double *p(int d) const { return base + d * size; }
};

// times Gauss-Seidel sweeps of level l, a thread per column of a block, two
// where there are more than 1024 (S0 N^2), the block's columns side by side: in one wave when
// there are at most 64, so that its planes need no barrier.  ghosts: the first
// sweep takes its y and z ghosts from the planes gh.
template <int E>
__device__ __forceinline__ void b_sweeps(Bot &b, int l, int times, const BotGhost &gh, bool ghosts) {
  const GravGeo &G = b.G;
  const int *n = G.n[l];
  const int m0 = n[0] - 1, m1 = n[1] - 1, m2 = n[2] - 1, T = m0 + m1 + m2, N = 1 << l, cols = N * N * G.S[0];
  const int s1 = __ffs(m1) - 1, s12 = s1 + __ffs(m2) - 1, s0 = __ffs(G.S[0]) - 1, s01 = s0 + __ffs(G.S[1]) - 1;
  const double w = 1.0 / 6.0, h = b.h(l), h2 = h * h;
  const int tid = b_tid();
  const bool bar = m1 * m2 > 64;
  const bool idle = __builtin_amdgcn_readfirstlane((int)threadIdx.x) >= cols; // no column in this wave
  // rows of the column and its neighbours, shifted so that entry t is the node
  // on plane t.  Columns without a node on a plane read what lies there (at
  // most m1+m2 entries before a row, as many and 6 past it: inside the LDS
  // array, whose ends are the ghost planes and the whole-domain levels).
  int row[E], ryp[E], rzp[E], rym[E], rzm[E], lo[E], cnt[E], d[E], Y[E], Z[E];
  bool iny[E], inz[E], last[E];
#pragma unroll
  for (int e = 0; e < E; ++e) {
    const int q_ = tid + GRAV_COARSE_THREADS * e, q = q_ < cols ? q_ : 0;
    const int r = q >> s12, jk = q & ((1 << s12) - 1), j = 1 + (jk & (m1 - 1)), k = 1 + (jk >> s1);
    const int c0 = r & (G.S[0] - 1), c1 = (r >> s0) & (G.S[1] - 1), c2 = r >> s01;
    const int X0 = c0 * m0;
    Y[e] = c1 * m1 + j;
    Z[e] = c2 * m2 + k;
    d[e] = j + k;
    row[e] = Bot::at(l, X0, Y[e], Z[e]) - d[e];
    ryp[e] = Bot::at(l, X0, Y[e] == N ? 1 : Y[e] + 1, Z[e]) - d[e];
    rzp[e] = Bot::at(l, X0, Y[e], Z[e] == N ? 1 : Z[e] + 1) - d[e];
    rym[e] = Bot::at(l, X0, Y[e] == 1 ? N : Y[e] - 1, Z[e]) - d[e];
    rzm[e] = Bot::at(l, X0, Y[e], Z[e] == 1 ? N : Z[e] - 1) - d[e];
    iny[e] = j > 1;
    inz[e] = k > 1;
    last[e] = q_ < cols && c0 == G.S[0] - 1;
    // node 1 of the first x block is the boundary, kept
    lo[e] = d[e] + (c0 == 0 ? 2 : 1);
    cnt[e] = q_ < cols ? d[e] + m0 + 1 - lo[e] : 0;
  }
#pragma unroll 1
  for (int s = 0; s < times; ++s) {
    if (idle) {
      if (bar)
        for (int t = 3; t <= T; t += 4) {
#pragma unroll
          for (int g = 0; g < 4; ++g) lds_barrier();
        }
    } else {
      double *U = gh.base; // everything as an offset from the LDS array's start
      const int A = (int)(b.cur(l) - U), B = (int)(b.other(l) - U), R = (int)(b.rhs(l) - U);
      int yp[E], zp[E], ym[E], zm[E];
      double xu[E], yu[E], zu[E], rr[E], prev[E];
#pragma unroll
      for (int e = 0; e < E; ++e) {
        yp[e] = A + ryp[e];
        zp[e] = A + rzp[e];
        ym[e] = (iny[e] ? B : A) + rym[e];
        zm[e] = (inz[e] ? B : A) + rzm[e];
        if (ghosts && s == 0) {
          const int X0 = row[e] + d[e] - Bot::at(l, 0, Y[e], Z[e]);
          const int gy = X0 - 1 + (N + 1) * (Z[e] - 1) - d[e], gz = X0 - 1 + (N + 1) * (Y[e] - 1) - d[e];
          if (Y[e] == 1) ym[e] = gy;
          if (Y[e] == N) yp[e] = gh.size + gy;
          if (Z[e] == 1) zm[e] = 2 * gh.size + gz;
          if (Z[e] == N) zp[e] = 3 * gh.size + gz;
        }
        const double *a = U + A + row[e];
        prev[e] = a[lo[e] - 1];
        xu[e] = a[4]; // the upper neighbours and the right-hand side a plane ahead, as in k_grav_relax_lds
        yu[e] = U[yp[e] + 3];
        zu[e] = U[zp[e] + 3];
        rr[e] = U[R + row[e] + 3];
        if (lo[e] - d[e] == 2 && cnt[e] > 0) U[B + row[e] + d[e] + 1] = a[d[e] + 1];
        if (last[e]) U[B + row[e] + d[e] + m0 + 1] = a[d[e] + m0 + 1];
      }
      wave_order();
      for (int tb = 3; tb <= T; tb += 4) {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int t = tb + g;
          double v[E];
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const double ymv = U[ym[e] + t], zmv = U[zm[e] + t];
            v[e] = w * (xu[e] + prev[e] + yu[e] + ymv + zu[e] + zmv - h2 * rr[e]);
            xu[e] = U[A + row[e] + t + 2];
            yu[e] = U[yp[e] + t + 1];
            zu[e] = U[zp[e] + t + 1];
            rr[e] = U[R + row[e] + t + 1];
          }
#pragma unroll
          for (int e = 0; e < E; ++e) {
            const bool act = (unsigned)(t - lo[e]) < (unsigned)cnt[e];
            if (act) U[B + row[e] + t] = v[e];
            prev[e] = act ? v[e] : prev[e];
          }
          if (bar) lds_barrier();
          else wave_order();
        }
      }
    }
    b.flip ^= 1 << l;
    __syncthreads();
  }
}
__device__ __forceinline__ void b_relax(Bot &b, int l, int times, const BotGhost &gh, bool ghosts) {
  if ((b.G.S[0] << (2 * l)) > GRAV_COARSE_THREADS) b_sweeps<2>(b, l, times, gh, ghosts);
  else b_sweeps<1>(b, l, times, gh, ghosts);
}

// residMPI at every node of level l into its other copy
__device__ void b_resid(Bot &b, int l) {
  const int N = 1 << l, sy = Bot::rs(l), sz = Bot::zs(l);
  const double h = b.h(l), h2i = 1.0 / (h * h);
  const double *u = b.cur(l), *rhs = b.rhs(l);
  double *res = b.other(l);
  Bot::each(l, [&](int X, int Y, int Z) {
    const int q = Bot::at(l, X, Y, Z);
    double v = 0.0;
    if (X > 1 && X <= N)
      v = g_res7(u[q + 1], u[q - 1], u[q + (Y == N ? 1 - N : 1) * sy], u[q + (Y == 1 ? N - 1 : -1) * sy],
                 u[q + (Z == N ? 1 - N : 1) * sz], u[q + (Z == 1 ? N - 1 : -1) * sz], u[q], h2i, rhs[q]);
    res[q] = v;
  });
  __syncthreads();
}

// the way down from level l (k_grav_down)
__device__ void b_down(Bot &b, int l) {
  b_resid(b, l);
  const int lc = l - 1, Nc = 1 << lc, sy = Bot::rs(l), sz = Bot::zs(l);
  const double *res = b.other(l);
  double *rhs = b.rhs(lc), *u = b.cur(lc);
  Bot::each(lc, [&](int X, int Y, int Z) {
    const int q = Bot::at(lc, X, Y, Z);
    u[q] = 0.0;
    double v = 0.0;
    if (X > 1 && X <= Nc) {
      const int p = Bot::at(l, 2 * X - 1, 2 * Y - 1, 2 * Z - 1);
      v = res[p];
      if (Y > 1 && Z > 1) {
        const double w = 1.0 / 12.0;
        v = 0.5 * v + w * (res[p + 1] + res[p - 1] + res[p + sy] + res[p - sy] + res[p + sz] + res[p - sz]);
      }
    }
    rhs[q] = v;
  });
  __syncthreads();
}

// the interpolant of a coarser level (row and plane strides sy, sz) at node
// (X, Y, Z); wrap: its nodes 1..Nc along y and z are periodic
__device__ __forceinline__ double b_interp(const double *uc, int Nc, int sy, int sz, bool wrap, int X, int Y, int Z) {
  const int xu = (X + 2) / 2 - 1, yu = (Y + 2) / 2 - 1, zu = (Z + 2) / 2 - 1; // 0-based
  const int xl = xu - !(X & 1), yl = yu - !(Y & 1), zl = zu - !(Z & 1);
  const int y0 = (wrap && yu == Nc ? 0 : yu) * sy, y1 = yl * sy, z0 = (wrap && zu == Nc ? 0 : zu) * sz, z1 = zl * sz;
  auto w = [&](int o) { return .5 * (uc[o + xu] + uc[o + xl]); };
  auto vv = [&](int o) { return .5 * (w(o + y0) + w(o + y1)); };
  return .5 * (vv(z0) + vv(z1));
}

// addintMPI from level l-1 (k_grav_prolong, mode 0)
__device__ void b_add(Bot &b, int l) {
  const int lc = l - 1;
  const double *uc = b.cur(lc);
  double *u = b.cur(l);
  Bot::each(l, [&](int X, int Y, int Z) {
    const int q = Bot::at(l, X, Y, Z);
    u[q] = u[q] + b_interp(uc, 1 << lc, Bot::rs(lc), Bot::zs(lc), true, X, Y, Z);
  });
  __syncthreads();
}

// the whole-domain levels below L = NGcr: the residual of L restricted
// (rstrct, mode 1; its nodes N+1 along y and z are the wrapped first ones),
// the lower levels, the correction of L (addint) with the ghost planes of the
// sweep after it
__device__ void b_below(Bot &b, const Coarse &S, const BotGhost &gh) {
  const GravGeo &G = b.G;
  const int L = G.NGcr, N = 1 << L, NX = N + 1, nc = N / 2 + 1, sy = Bot::rs(L), sz = Bot::zs(L);
  b_resid(b, L);
  const double *res = b.other(L);
  double *u = b.cur(L);
  for (int q = b_tid(); q < nc * nc * nc; q += blockDim.x) {
    const int ic = 1 + q % nc, jc = 1 + (q / nc) % nc, kc = 1 + q / (nc * nc);
    double v = 0.0;
    if (ic > 1 && ic < nc) {
      const int p = Bot::at(L, 2 * ic - 1, jc == nc ? 1 : 2 * jc - 1, kc == nc ? 1 : 2 * kc - 1);
      v = res[p];
      if (jc > 1 && jc < nc && kc > 1 && kc < nc) {
        const double w = 1.0 / 12.0;
        v = 0.5 * v + w * (res[p + 1] + res[p - 1] + res[p + sy] + res[p - sy] + res[p + sz] + res[p - sz]);
      }
    }
    S.rhs[G.p1[L - 1] + q] = v;
    S.phi[G.p1[L - 1] + q] = 0.0;
  }
  // the residual of level L-1 reads on into the first rows of level L
  for (int q = b_tid(); q < nc * nc; q += blockDim.x) S.phi[G.p1[L] + q] = u[Bot::at(L, 1 + q % NX, 1 + q / NX, 1)];
  __syncthreads();
  c_vcycle_lower(S, L);
  const double *uc = S.phi + G.p1[L - 1];
  Bot::each(L, [&](int X, int Y, int Z) {
    const int q = Bot::at(L, X, Y, Z), gy = (X - 1) + NX * (Z - 1), gz = (X - 1) + NX * (Y - 1);
    const double o = u[q];
    auto pro = [&](int y, int z) { return b_interp(uc, N / 2, nc, nc * nc, false, X, y, z); };
    if (Y == N) gh.p(0)[gy] = o;
    if (Y == 1) gh.p(1)[gy] = o + pro(NX, Z);
    if (Z == N) gh.p(2)[gz] = o;
    if (Z == 1) gh.p(3)[gz] = o + pro(Y, NX);
    u[q] = o + pro(Y, Z);
  });
  __syncthreads();
}

// cycles V-cycles from split level top: right-hand side from its blocks, the
// potential from its blocks (phi) or zero (no phi), the result to out, nodes
// 1..N+1 x 1..N x 1..N (k_grav_prolong reads it there).  sweeps before and
// after on the levels above NGcr, five after the correction of NGcr.
__global__ __launch_bounds__(GRAV_COARSE_THREADS) void k_grav_bottom(GravGeo G, GravBuf B, const double *phi, double *out,
                                                                     int top, int sweeps, int cycles) {
  __shared__ double lds[GRAV_BOT_LDS];
  const int L = G.NGcr, N1 = (1 << L) + 1, Ng = 1 << L, need = (int)G.p1[L], tail = (Ng / 2 + 1) * (Ng / 2 + 1);
  const BotGhost gh{lds, N1 * Ng};
  Bot b{G, lds + 4 * gh.size, 0};
  double *sphi = b.level(top + 1), *srhs = sphi + need + tail, *sres = srhs + need;
  const Coarse S{G, B, sphi, srhs, sres};
  const int *n = G.n[top], N = 1 << top, NX = N + 1;
  const int h0 = __ffs(n[0] - 1) - 1, h1 = __ffs(n[1] - 1) - 1, h2 = __ffs(n[2] - 1) - 1;
  const int bs = (int)G.bsz[top];
  const double *u2 = phi ? phi + G.off[top] : nullptr, *r2 = B.rhs2 + G.off[top];
  // node (X, Y, Z) of the level, its high ghosts included, in its block
  auto slot = [&](int X, int Y, int Z) {
    const int c0 = min((X - 1) >> h0, G.S[0] - 1), c1 = min((Y - 1) >> h1, G.S[1] - 1), c2 = min((Z - 1) >> h2, G.S[2] - 1);
    return g_rid(G, c0, c1, c2) * bs + (int)g_idx(n, X - (c0 << h0), Y - (c1 << h1), Z - (c2 << h2));
  };
  {
    double *u = b.cur(top), *rhs = b.rhs(top);
    Bot::each(top, [&](int X, int Y, int Z) {
      const int a = slot(X, Y, Z), q = Bot::at(top, X, Y, Z);
      u[q] = u2 ? u2[a] : 0.0;
      rhs[q] = r2[a];
    });
    for (int q = b_tid(); q < need; q += blockDim.x) {
      sphi[q] = B.phi1[q];
      srhs[q] = B.rhs1[q];
      sres[q] = B.res1[q];
    }
    if (top == L) // the ghosts as they are
      for (int q = b_tid(); q < gh.size; q += blockDim.x) {
        const int X = 1 + q % N1, e = 1 + q / N1;
        gh.p(0)[q] = u2 ? u2[slot(X, 1, e) - 1 - (n[1] + 1) * (n[2] + 1)] : 0.0;
        gh.p(1)[q] = u2 ? u2[slot(X, Ng + 1, e)] : 0.0;
        gh.p(2)[q] = u2 ? u2[slot(X, e, 1) - (n[1] + 1) * (n[2] + 2)] : 0.0;
        gh.p(3)[q] = u2 ? u2[slot(X, e, Ng + 1)] : 0.0;
      }
  }
  __syncthreads();
  for (int cyc = 0; cyc < cycles; ++cyc) {
    for (int l = top; l > L; --l) {
      b_relax(b, l, sweeps, gh, false);
      b_down(b, l);
    }
    b_relax(b, L, sweeps, gh, top == L && cyc == 0);
    b_below(b, S, gh);
    b_relax(b, L, 5, gh, true);
    for (int l = L + 1; l <= top; ++l) {
      b_add(b, l);
      b_relax(b, l, sweeps, gh, false);
    }
  }
  const double *u = b.cur(top);
  Bot::each(top, [&](int X, int Y, int Z) { out[(X - 1) + NX * ((Y - 1) + ((Z - 1) << top))] = u[Bot::at(top, X, Y, Z)]; });
  for (int q = b_tid(); q < need; q += blockDim.x) {
    B.phi1[q] = sphi[q];
    B.rhs1[q] = srhs[q];
    B.res1[q] = sres[q];
  }
}

// ---------------------------------------------------------------------------
// PB: boundary potential on the x ends
// ---------------------------------------------------------------------------
// the real plane of global x index gx packed as nn1/2 complex values per
// row (y = 2k-1 real part, 2k imaginary part), rows along z
// Through an LDS tile of 64 planes x 64 rows at one z: the reads run along
// x (the planes, consecutive x within a block), the writes along the row
// pairs.  Grid (plane tiles, pair tiles of 32, nn2), 256 threads.
__global__ __launch_bounds__(256) void k_pb_pack(PbArgs P, const double *rho, Geo g, double2 *Z) {
  __shared__ double T[64][65];
  const int H = P.nn1 / 2, q = blockIdx.z;
  const int pl0 = 64 * blockIdx.x, pp0 = 32 * blockIdx.y;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int pl = pl0 + lane;
  const int gx = pl < P.np ? P.gx[pl] : 0;
  for (int r = w; r < 64; r += 4) { // row j = 2 pp0 + 1 + r
    const int pp = pp0 + (r >> 1);
    T[r][lane] = (pl < P.np && pp < H) ? rho[ix3(g, gx, 2 * pp0 + 1 + r, q + 1)] : 0.0;
  }
  __syncthreads();
  const int e = threadIdx.x & 31, h = threadIdx.x >> 5; // pair pp0 + e, planes h, h + 8, ...
  for (int c = h; c < 64; c += 8) {
    const int p2 = pl0 + c, pp = pp0 + e;
    if (p2 < P.np && pp < H) Z[((long)p2 * P.nn2 + q) * H + pp] = make_double2(T[2 * e][c], T[2 * e + 1][c]);
  }
}

// radix-2 FFT of lines of L complex values in LDS: X_k = sum_j z_j
// exp(sign 2 pi i j k / L).  Line id -> (outer, inner); element e of the
// line at outer*outer_stride + inner*inner_stride + e*es.  A workgroup
// transforms 2^lcw lines of consecutive inner index (ninner a multiple of
// it, 2^lcw L <= 2 GRAV_FFT_MAXL): with inner_stride 1 and es > 1 (the
// columns of a plane) its loads and stores run over 2^lcw neighbouring
// columns at once.
__global__ __launch_bounds__(512) void k_pb_fft(double2 *Z, int L, long es, long inner_stride, long outer_stride,
                                                 int ninner, int sign, int lcw) {
  __shared__ double2 buf[2 * GRAV_FFT_MAXL];
  // the twiddles exp(sign 2 pi i k / L), k < L/2, once per workgroup: stage
  // len takes k = pos L/len, whose sincospi argument 2k/L is the same double
  // as 2 pos/len
  __shared__ double2 tw[GRAV_FFT_MAXL / 2];
  const int CW = 1 << lcw, H2 = L / 2;
  const long line0 = (long)blockIdx.x << lcw;
  double2 *z = Z + (line0 / ninner) * outer_stride + (line0 % ninner) * inner_stride;
  int lg = 0;
  while ((1 << lg) < L) ++lg;
  for (int idx = threadIdx.x; idx < CW * L; idx += blockDim.x) {
    const int e = idx >> lcw, c = idx & (CW - 1);
    const int rev = (int)(__brev((unsigned)e) >> (32 - lg));
    buf[c * L + rev] = z[c * inner_stride + e * es];
  }
  for (int k = threadIdx.x; k < H2; k += blockDim.x) {
    double sn, cs;
    sincospi(2.0 * (double)k / (double)L, &sn, &cs);
    tw[k] = make_double2(cs, sign > 0 ? sn : -sn);
  }
  __syncthreads();
  for (int len = 2; len <= L; len <<= 1) {
    const int half = len >> 1;
    for (int b = threadIdx.x; b < CW * H2; b += blockDim.x) {
      const int c = b / H2, bb = b - c * H2;
      const int grp = bb / half, pos = bb - grp * half;
      const int i0 = c * L + grp * len + pos, i1 = i0 + half;
      const double2 W = tw[pos * (L / len)];
      const double cs = W.x, sn = W.y;
      const double2 a = buf[i0], d = buf[i1];
      const double tr = cs * d.x - sn * d.y, ti = cs * d.y + sn * d.x;
      buf[i1] = make_double2(a.x - tr, a.y - ti);
      buf[i0] = make_double2(a.x + tr, a.y + ti);
    }
    __syncthreads();
  }
  for (int idx = threadIdx.x; idx < CW * L; idx += blockDim.x) {
    const int e = idx >> lcw, c = idx & (CW - 1);
    z[c * inner_stride + e * es] = buf[c * L + e];
  }
}

// one rlft3 unpacking step: h1 = c1 (a + b), h2 = c2 (a - b) with
// c1 = (0.5, 0), c2 = (0, c2i), b already conjugated
struct H12 { double h1r, h1i, h2r, h2i; };
__device__ __forceinline__ H12 rl_h(double ar, double ai, double br, double bi, double c2i) {
  const double sr = ar + br, si = ai + bi, dr = ar - br, di = ai - bi;
  return {0.5 * sr - 0.0 * si, 0.5 * si + 0.0 * sr, 0.0 * dr - c2i * di, 0.0 * di + c2i * dr};
}

// rlft3's unpacking loop (SG8:1484-1508) after the forward FFT (isign 1:
// S receives the Nyquist column) or before the inverse one (isign -1: S
// holds it).  One thread per independent piece: a pair (i2, mirror) of
// the first column, an (i1, i2) of columns 2..nn1/4 with its partner
// (nn1/2-i1+2, mirror), or a pair of the middle column, which the
// reference's in-place loop passes twice.
__global__ void k_pb_unpack(PbArgs P, double2 *Z, double2 *S, int nplanes, int isign) {
  const int H = P.nn1 / 2, nn2 = P.nn2, q4 = P.nn1 / 4;
  const int npair = nn2 / 2 + 1;
  const long per = 2L * npair + (long)(q4 - 1) * nn2, t = g_tid();
  if (t >= per * nplanes) return;
  const int pl = (int)(t / per);
  long m = t - pl * per;
  double2 *D = Z + (long)pl * nn2 * H;
  double2 *Sp = S + (long)pl * nn2;
  const double c2i = -0.5 * (double)isign;
  const double2 *wt = isign > 0 ? P.wf : P.wi;
  auto at = [&](int i1, int i2) -> double2 & { return D[(long)(i2 - 1) * H + (i1 - 1)]; };
  auto mir = [&](int i2) { return i2 == 1 ? 1 : nn2 - i2 + 2; };
  if (m < npair) {
    const int a = (int)m + 1, b = mir(a);
    if (isign > 0) {
      const double2 za = at(1, a), zb = at(1, b);
      H12 h = rl_h(za.x, za.y, zb.x, -zb.y, c2i);
      at(1, a) = make_double2(h.h1r + h.h2r, h.h1i + h.h2i);
      Sp[b - 1] = make_double2(h.h1r - h.h2r, -(h.h1i - h.h2i));
      if (b != a) {
        h = rl_h(zb.x, zb.y, za.x, -za.y, c2i);
        at(1, b) = make_double2(h.h1r + h.h2r, h.h1i + h.h2i);
        Sp[a - 1] = make_double2(h.h1r - h.h2r, -(h.h1i - h.h2i));
      }
    } else {
      const double2 da = at(1, a), db = at(1, b), sa = Sp[a - 1], sb = Sp[b - 1];
      H12 h = rl_h(da.x, da.y, sb.x, -sb.y, c2i);
      at(1, a) = make_double2(h.h1r + h.h2r, h.h1i + h.h2i);
      if (b != a) {
        h = rl_h(db.x, db.y, sa.x, -sa.y, c2i);
        at(1, b) = make_double2(h.h1r + h.h2r, h.h1i + h.h2i);
      }
    }
    return;
  }
  m -= npair;
  if (m < npair) {
    // middle column i1 = nn1/4 + 1: step a, then step b on the new values
    const int i1 = q4 + 1, a = (int)m + 1, b = mir(a);
    const double wr = wt[i1].x, wi = wt[i1].y;
    double2 da = at(i1, a), db = at(i1, b);
    H12 h = rl_h(da.x, da.y, db.x, -db.y, c2i);
    double whr = wr * h.h2r - wi * h.h2i, whi = wr * h.h2i + wi * h.h2r;
    const double2 na = make_double2(h.h1r + whr, h.h1i + whi);
    const double2 nb = make_double2(h.h1r - whr, -(h.h1i - whi));
    if (b == a) {
      at(i1, a) = nb;
      return;
    }
    h = rl_h(nb.x, nb.y, na.x, -na.y, c2i);
    whr = wr * h.h2r - wi * h.h2i;
    whi = wr * h.h2i + wi * h.h2r;
    at(i1, b) = make_double2(h.h1r + whr, h.h1i + whi);
    at(i1, a) = make_double2(h.h1r - whr, -(h.h1i - whi));
    return;
  }
  m -= npair;
  const int i1 = 2 + (int)(m / nn2), i2 = 1 + (int)(m % nn2);
  const int j1 = H - i1 + 2, j2 = mir(i2);
  const double wr = wt[i1].x, wi = wt[i1].y;
  const double2 da = at(i1, i2), db = at(j1, j2);
  const H12 h = rl_h(da.x, da.y, db.x, -db.y, c2i);
  const double whr = wr * h.h2r - wi * h.h2i, whi = wr * h.h2i + wi * h.h2r;
  at(i1, i2) = make_double2(h.h1r + whr, h.h1i + whi);
  at(j1, j2) = make_double2(h.h1r - whr, -(h.h1i - whi));
}

// PB's mode weights (SG8:1146-1229) summed over the planes: for mode
// (l, m) of the y (nn1) and z (nn2) transforms, 0.5 exp(-z kappa)/kappa
// facG with kappa^2 = 4 (sin^2(pi (l-1)/nn1)/dy^2 + sin^2(pi (m-1)/nn2)/dz^2)
// for the left (z = zp) and right (z = Lbox - zp) end; the mean mode takes
// -0.5 z facG; the Nyquist column of y (the speq values) takes
// kappa = sqrt(sqrt(kappa^2) + 1e-20) for m <= nn2/2+1, as the reference.
// One thread per mode (pp = 0..nn1/2, q = 0..nn2-1).
// One wave per mode: the lanes take the planes in turn and the four sums
// are reduced across the wave (the reference's sum runs over each rank's
// planes and then over the ranks in the MPI library's order, so no order
// is the reference's bit for bit).
__global__ void k_pb_weight(PbArgs P, const double2 *Z, const double2 *S, double2 *D, double2 *SD) {
  const int H = P.nn1 / 2, nn1 = P.nn1, nn2 = P.nn2;
  const long t = g_tid() >> 6;
  const int lane = threadIdx.x & 63;
  if (t >= (long)(H + 1) * nn2) return;
  const int pp = (int)(t % (H + 1)), q = (int)(t / (H + 1));
  const double pi = 3.14159265359;
  const int l = pp + 1, m2 = q + 1;
  auto k2 = [&](int li, int mi) {
    const double s1 = sin(pi * (double)(li - 1) / (double)nn1), s2 = sin(pi * (double)(mi - 1) / (double)nn2);
    return 4.0 * (s1 * s1 / (P.dxx * P.dxx) + s2 * s2 / (P.dyy * P.dyy));
  };
  const bool dc = pp == 0 && m2 == 1;
  double kap = 0.0;
  if (pp < H) {
    if (!dc) kap = sqrt(k2(l, m2 <= nn2 / 2 + 1 ? m2 : nn2 + 2 - m2));
  } else {
    kap = m2 <= nn2 / 2 + 1 ? sqrt(sqrt(k2(l, m2)) + 1.0e-20) : sqrt(k2(l, nn2 + 2 - m2));
  }
  double ar[2] = {0.0, 0.0}, ai[2] = {0.0, 0.0};
  for (int pl = lane; pl < P.np; pl += 64) {
    const double2 X = pp < H ? Z[((long)pl * nn2 + q) * H + pp] : S[(long)pl * nn2 + q];
    const double fg = P.facG[pl];
    const double z[2] = {P.zp[pl], P.zq[pl]};
    for (int s = 0; s < 2; ++s) {
      if (dc) {
        ar[s] = ar[s] + (0.0 - X.x * 0.5 * z[s] * fg);
        ai[s] = ai[s] + (0.0 - X.y * 0.5 * z[s] * fg);
      } else {
        const double e = exp(-z[s] * kap);
        ar[s] = ar[s] + X.x * 0.5 * e / kap * fg;
        ai[s] = ai[s] + X.y * 0.5 * e / kap * fg;
      }
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1)
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      ar[s] += __shfl_xor(ar[s], o);
      ai[s] += __shfl_xor(ai[s], o);
    }
  if (lane != 0) return;
  for (int s = 0; s < 2; ++s) {
    if (pp < H) D[((long)s * nn2 + q) * H + pp] = make_double2(ar[s], ai[s]);
    else SD[(long)s * nn2 + q] = make_double2(ar[s], ai[s]);
  }
}

// the end-plane potential after the inverse transform, divided by
// 2 (nn1/2)^2, onto the finest split level of every rank (SG8:1259-1272):
// node (j, k) of the rank's plane, 0..C+1, the outer nodes wrapped
__global__ void k_pb_bphi(GravGeo G, PbArgs P, const double2 *D, double *bphi2) {
  const int L = G.NGL, ny = G.C[1] + 1, nz = G.C[2] + 1;
  const long per = (long)(ny + 1) * (nz + 1), t = g_tid();
  if (t >= per * 2 * G.npe) return;
  const int rs = (int)(t / per), r = rs / 2, s = rs % 2;
  const long nidx = t - rs * per;
  const int j = (int)(nidx % (ny + 1)), k = (int)(nidx / (ny + 1));
  int c[3];
  g_rank(G, r, c);
  int jb = c[1] * G.C[1] + j, kb = c[2] * G.C[2] + k;
  if (j == ny && c[1] == G.S[1] - 1) jb = 1;
  if (k == nz && c[2] == G.S[2] - 1) kb = 1;
  if (j == 0 && c[1] == 0) jb = P.nn1;
  if (k == 0 && c[2] == 0) kb = P.nn2;
  const int H = P.nn1 / 2;
  const double2 z = D[((long)s * P.nn2 + (kb - 1)) * H + (jb - 1) / 2];
  const double fac = (double)(2 * (P.nn1 / 2) * (P.nn1 / 2));
  bphi2[G.boff[L] + t] = ((jb & 1) ? z.x : z.y) / fac;
}

// the end planes restricted to split level lc (SG8:1288-1363)
__global__ void k_pb_restrict(GravGeo G, double *bphi2, int lc) {
  const int mcx = G.n[lc][1], mcy = G.n[lc][2];
  const long cper = (long)(mcx + 1) * (mcy + 1), fper = (long)(G.n[lc + 1][1] + 1) * (G.n[lc + 1][2] + 1);
  const long cnt = (long)mcx * mcy, t = g_tid();
  if (t >= cnt * 2 * G.npe) return;
  const int rs = (int)(t / cnt);
  const long m = t - rs * cnt;
  const int ic = 1 + (int)(m % mcx), jc = 1 + (int)(m / mcx);
  const double *bf = bphi2 + G.boff[lc + 1] + rs * fper;
  const long kf = (2 * ic - 1) + (long)(mcx * 2) * (2 * jc - 1), kc = ic + (long)(mcx + 1) * jc;
  bphi2[G.boff[lc] + rs * cper + kc] = plane_restrict(bf, kf, 2L * mcx, ic, jc, mcx, mcy);
}

// the level-NGcr end planes of the first / last x ranks gathered into the
// whole-domain level NGcr (SG8:1366-1390)
__global__ void k_pb_collect(GravGeo G, double *bphi1, const double *bphi2) {
  const int L = G.NGcr, N1 = (1 << L) + 1;
  const int *m = G.n[L];
  const long t = g_tid();
  if (t >= 2L * N1 * N1) return;
  const int s = (int)(t / ((long)N1 * N1));
  const long q = t - s * (long)N1 * N1;
  const int j = 1 + (int)(q % N1), k = 1 + (int)(q / N1);
  const int cy = min((j - 1) / (m[1] - 1), G.S[1] - 1), cz = min((k - 1) / (m[2] - 1), G.S[2] - 1);
  const int jj = j - cy * (m[1] - 1), kk = k - cz * (m[2] - 1);
  const int r = g_rid(G, s == 0 ? 0 : G.S[0] - 1, cy, cz);
  bphi1[s * (G.needb1 + 1) + G.pb1[L] + (j - 1) + (long)N1 * (k - 1)] =
      bphi2[G.boff[L] + (2L * r + s) * (long)(m[1] + 1) * (m[2] + 1) + jj + (long)(m[1] + 1) * kk];
}

// Phi at the cells: each rank's nodes 1..C of the finest level (SG8:282-291)
// (a rank block's cells in g_node's order: the reads of the skewed layout
// contiguous, the writes scattered)
__global__ void k_grav_phi(GravGeo G, const double *phi2, double *Phi, Geo g) {
  const long cnt = (long)G.C[0] * G.C[1] * G.C[2], t = g_tid();
  if (t >= cnt * G.npe) return;
  const int r = (int)(t / cnt), L = G.NGL;
  int i, j, k, c[3];
  g_node(G.C, t - r * cnt, i, j, k);
  g_rank(G, r, c);
  Phi[ix3(g, c[0] * G.C[0] + i, c[1] * G.C[1] + j, c[2] * G.C[2] + k)] = phi2[G.off[L] + r * G.bsz[L] + g_idx(G.n[L], i, j, k)];
}

// Phi's face ghosts (SG8:22-67): y and z periodic, the x ends copied from
// the first / last cell (zero gradient)
__global__ void k_grav_phi_ghosts(double *Phi, Geo g) {
  const int N0 = g.n[0], N1 = g.n[1], N2 = g.n[2];
  const long a0 = (long)N1 * N2, a1 = (long)N0 * N2, a2 = (long)N0 * N1, t = g_tid();
  if (t < a0) {
    const int j = 1 + (int)(t % N1), k = 1 + (int)(t / N1);
    const double l = Phi[ix3(g, 1, j, k)], r = Phi[ix3(g, N0, j, k)];
    Phi[ix3(g, 0, j, k)] = l;
    Phi[ix3(g, -1, j, k)] = l;
    Phi[ix3(g, N0 + 1, j, k)] = r;
    Phi[ix3(g, N0 + 2, j, k)] = r;
  } else if (t < a0 + a1) {
    const long u = t - a0;
    const int i = 1 + (int)(u % N0), k = 1 + (int)(u / N0);
    Phi[ix3(g, i, -1, k)] = Phi[ix3(g, i, N1 - 1, k)];
    Phi[ix3(g, i, 0, k)] = Phi[ix3(g, i, N1, k)];
    Phi[ix3(g, i, N1 + 1, k)] = Phi[ix3(g, i, 1, k)];
    Phi[ix3(g, i, N1 + 2, k)] = Phi[ix3(g, i, 2, k)];
  } else if (t < a0 + a1 + a2) {
    const long u = t - a0 - a1;
    const int i = 1 + (int)(u % N0), j = 1 + (int)(u / N0);
    Phi[ix3(g, i, j, -1)] = Phi[ix3(g, i, j, N2 - 1)];
    Phi[ix3(g, i, j, 0)] = Phi[ix3(g, i, j, N2)];
    Phi[ix3(g, i, j, N2 + 1)] = Phi[ix3(g, i, j, 1)];
    Phi[ix3(g, i, j, N2 + 2)] = Phi[ix3(g, i, j, 2)];
  }
}

// GRAVTY(dt,3) (SG8:82-89): v -= dt/2 * the fourth-order gradient of Phi,
// 1/(12 dx(0)) with dx(0) of the cell's x rank
__global__ void k_grav_kick(double *U2, double *U3, double *U4, const double *Phi, Geo g, const double *gdx0, int cx,
                            double dt) {
  const long N0 = g.n[0], N1 = g.n[1];
  const long t = g_tid();
  if (t >= N0 * N1 * g.n[2]) return;
  const int i = 1 + (int)(t % N0), j = 1 + (int)((t / N0) % N1), k = 1 + (int)(t / (N0 * N1));
  const int c = ix3(g, i, j, k), sx = 1, sy = g.st[1], sz = g.st[2];
  const double dxi = 1.0 / (12.0 * gdx0[((i - 1) / cx) * cx + 1]);
  const double *P = Phi;
  U2[c] = U2[c] - dt * (-P[c + 2 * sx] + 8.0 * P[c + sx] - 8.0 * P[c - sx] + P[c - 2 * sx]) * dxi * 0.5;
  U3[c] = U3[c] - dt * (-P[c + 2 * sy] + 8.0 * P[c + sy] - 8.0 * P[c - sy] + P[c - 2 * sy]) * dxi * 0.5;
  U4[c] = U4[c] - dt * (-P[c + 2 * sz] + 8.0 * P[c + sz] - 8.0 * P[c - sz] + P[c - 2 * sz]) * dxi * 0.5;
}

} // namespace mcf
