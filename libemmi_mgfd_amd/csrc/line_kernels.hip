// line_kernels.hip -- exact line block Gauss-Seidel, factored once per level.
//
// Line (a; pb, pc) holds the vertex patches of the nodes (p, pb, pc),
// p = 1..N-1, N = n_a (src/gmg.c:340-1298): the along-line edges E_a(e),
// e = 0..N-1, and per node four perpendicular edges, slots
//   0: E_b(p, pb-1, pc)  1: E_b(p, pb, pc)  2: E_c(p, pb, pc-1)  3: E_c(p, pb, pc)
// with (a, b, c) cyclic.  Each line system is solved exactly for the
// correction of the current residual.  An along-line edge couples only to
// the perpendicular edges of its two end nodes, through the constant vector
// v = (Hc, -Hc, Hb, -Hb):
//     d_e dE_a(e) + v.da_e - v.da_{e+1} = rho_e,
// so it is eliminated first; the node unknowns then form a complex
// symmetric 4x4 block-tridiagonal system
//     D_p = K_p - v v^T (1/d_{p-1} + 1/d_p),   B_p = diag(l_{p-1}) + v v^T / d_{p-1}
//     W_1 = D_1,  W_p = D_p - B_p W_{p-1}^{-1} B_p
// whose factors depend on the grid, the medium and the frequency only.
// k_line_factor stores, per node, W_p^{-1} (symmetric, 10 entries) and 1/d
// once; a sweep then computes the residuals sigma_p, rho_p of the lines and
// runs
//     y_p = g_p - B_p z_{p-1},  z_p = W_p^{-1} y_p          (forward)
//     da_p = z_p - W_p^{-1} B_{p+1} da_{p+1},
//     dE_a(p) = rho_p/d_p + v.(da_{p+1} - da_p) / d_p        (backward)
// with g_p = sigma_p + v (rho_{p-1}/d_{p-1} - rho_p/d_p) from the residual:
// k_line_solve_m does all of it in one launch on the matrix cores,
// k_line_long_* in two for lines whose records are in memory; k_line_rhs* and
// k_line_solve (one lane per line half) take colours of many long lines and
// packs whose lines differ in length, and serve as the others' check.
// Lines of one colour (pb%2, pc%2) are not coupled, so a launch sweeps one
// colour; every kernel computes in FP64 whatever the storage precision.  The
// substitutions keep a ring of the next D nodes' factor records in registers,
// so D nodes of loads are in flight while a node is computed.
#include "line_kernels.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <map>
#include <mutex>
#include <stdexcept>
#include "dynamic_lds.h"
#include "stencil.h"
#include "timing.h"

namespace emmi {

constexpr int FREC = 22;  // values per node in the factor records: W^-1 (10 complex), 1/d
constexpr int SREC = 10;  // values per node in the line records: sigma or z (4 complex), rho

// 16-byte chunk of record values
template <typename R>
struct alignas(16) Ch {
  static constexpr int V = 16 / (int)sizeof(R);
  R v[V];
};
template <typename R> constexpr int fchunks() { return (FREC + Ch<R>::V - 1) / Ch<R>::V; }
template <typename R> constexpr int schunks() { return (SREC + Ch<R>::V - 1) / Ch<R>::V; }
// minimum waves per SIMD the right-hand-side kernels are compiled for
// (bounds their registers; more waves keep more stencil loads in flight)
#ifndef EMMI_LINE_RHS_MIN_WAVES
#define EMMI_LINE_RHS_MIN_WAVES 1
#endif

template <typename T> using FacRec = typename LineFac<T>::type;
template <typename T> using ScrRec = typename LineScr<T>::type;

// nodes of records in flight in the substitution (build-time tunable)
// for FP32-storage and FP64 cycles
#ifndef EMMI_LINE_RING_F32
#define EMMI_LINE_RING_F32 2
#endif
#ifndef EMMI_LINE_RING_F64
#define EMMI_LINE_RING_F64 1
#endif
template <typename T> constexpr int ring_depth() { return sizeof(T) == 4 ? EMMI_LINE_RING_F32 : EMMI_LINE_RING_F64; }
// value k of a node's chunks, as double
template <typename R, int NC>
__device__ __forceinline__ double val(const Ch<R> (&c)[NC], int k) {
  return (double)c[k / Ch<R>::V].v[k % Ch<R>::V];
}
template <typename R, int NC>
__device__ __forceinline__ void put(Ch<R> (&c)[NC], int k, double x) {
  c[k / Ch<R>::V].v[k % Ch<R>::V] = (R)x;
}
// loads the NC chunks of one node; src points at chunk 0 of that node's line
template <typename R, int NC>
__device__ __forceinline__ void load_node(Ch<R> (&c)[NC], const Ch<R>* __restrict__ src, long stride) {
#pragma unroll
  for (int k = 0; k < NC; k++) c[k] = src[k * stride];
}

__device__ __forceinline__ int symidx(int i, int j) {
  const int a = i < j ? i : j, b = i < j ? j : i;
  return a * 4 - (a * (a - 1)) / 2 + (b - a);
}

__device__ __forceinline__ void inv4(cxd (&M)[4][4]) {
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const cxd piv = cinv(M[k][k]);
    M[k][k] = cxd(1.0, 0.0);
#pragma unroll
    for (int j = 0; j < 4; j++) M[k][j] = M[k][j] * piv;
#pragma unroll
    for (int i = 0; i < 4; i++) {
      if (i == k) continue;
      const cxd fct = M[i][k];
      M[i][k] = cxd(0.0, 0.0);
#pragma unroll
      for (int j = 0; j < 4; j++) M[i][j] -= fct * M[k][j];
    }
  }
}

// constants of one line
template <typename T, int A>
struct LineGeo {
  static constexpr int B = (A + 1) % 3, C = (A + 2) % 3;
  int N, pb, pc;
  long sa, base, oa, ob0, ob1, oc0, oc1;
  double Hb, Hc, Wb0, Wb1, Wc0, Wc1, sIb, sIc, dre_a;
  double v[4];

  __device__ __forceinline__ LineGeo() {}
  __device__ __forceinline__ LineGeo(const Level<T>& L, int pb_, int pc_) { init(L, pb_, pc_); }
  __device__ __forceinline__ void init(const Level<T>& L, int pb_, int pc_) {
    pb = pb_;
    pc = pc_;
    N = L.n[A];
    sa = L.es[A];
    base = (long)pb * L.es[B] + (long)pc * L.es[C];
    oa = A * L.nc + base;
    ob0 = B * L.nc + base - L.es[B];
    ob1 = B * L.nc + base;
    oc0 = C * L.nc + base - L.es[C];
    oc1 = C * L.nc + base;
    Hb = L.H[B][pb];
    Hc = L.H[C][pc];
    Wb0 = L.W[B][pb - 1];
    Wb1 = L.W[B][pb];
    Wc0 = L.W[C][pc - 1];
    Wc1 = L.W[C][pc];
    sIb = (double)L.IW[B][pb - 1] + (double)L.IW[B][pb];
    sIc = (double)L.IW[C][pc - 1] + (double)L.IW[C][pc];
    dre_a = Hc * sIb + Hb * sIc;
    v[0] = Hc; v[1] = -Hc; v[2] = Hb; v[3] = -Hb;
  }
  // diagonal of the along-line edge e
  __device__ __forceinline__ cxd d_edge(const Level<T>& L, int e) const {
    return cxd((double)L.W[A][e] * dre_a, -L.omu * (double)L.sbar[oa + e * sa]);
  }
  // along-line coupling of node p to node p+1, per slot
  __device__ __forceinline__ void lcoef(const Level<T>& L, int p, double (&l)[4]) const {
    const double iWa = L.IW[A][p];
    l[0] = -Wb0 * Hc * iWa; l[1] = -Wb1 * Hc * iWa; l[2] = -Wc0 * Hb * iWa; l[3] = -Wc1 * Hb * iWa;
  }
};

template <typename T, int A>
__device__ __forceinline__ bool line_of(const LineJob<T>& J, int tid, int& pb, int& pc) {
  constexpr int B = (A + 1) % 3, C = (A + 2) % 3;
  if (tid >= J.nlo * J.nhi) return false;
  const int sb = J.cb ? 1 : 2, sc = J.cc ? 1 : 2;
  // the perpendicular axis with the smaller stride varies fastest
  if (B < C) { pb = sb + 2 * (tid % J.nlo); pc = sc + 2 * (tid / J.nlo); }
  else { pc = sc + 2 * (tid % J.nlo); pb = sb + 2 * (tid / J.nlo); }
  return true;
}

// D_p: the diagonal block of node p after the along-line edges p-1 and p
// (with 1/d = rdm, rdp) are eliminated
template <typename T, int A>
__device__ __forceinline__ void diag_block(const Level<T>& L, const LineGeo<T, A>& G, int p, cxd rdm, cxd rdp,
                                           cxd (&D)[4][4]) {
  const double Ha = L.H[A][p];
  const double iWa0 = L.IW[A][p - 1], iWa1 = L.IW[A][p];
  const double Gb = Ha * G.sIc + G.Hc * (iWa1 + iWa0);
  const double Gc = G.Hb * (iWa1 + iWa0) + Ha * G.sIb;
  const long off = p * G.sa;
  D[0][0] = cxd(G.Wb0 * Gb, -L.omu * (double)L.sbar[G.ob0 + off]);
  D[1][1] = cxd(G.Wb1 * Gb, -L.omu * (double)L.sbar[G.ob1 + off]);
  D[2][2] = cxd(G.Wc0 * Gc, -L.omu * (double)L.sbar[G.oc0 + off]);
  D[3][3] = cxd(G.Wc1 * Gc, -L.omu * (double)L.sbar[G.oc1 + off]);
  D[0][1] = D[1][0] = cxd(0, 0);
  D[2][3] = D[3][2] = cxd(0, 0);
  D[0][2] = D[2][0] = cxd(-Ha, 0);
  D[0][3] = D[3][0] = cxd(Ha, 0);
  D[1][2] = D[2][1] = cxd(Ha, 0);
  D[1][3] = D[3][1] = cxd(-Ha, 0);
  const cxd s = rdm + rdp;
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) D[i][j] -= s * (G.v[i] * G.v[j]);
}

// D -= B Wi B for the coupling B = diag(l) + v v^T rd of two neighbouring
// nodes (Wi: the inverse factor of the neighbour)
__device__ __forceinline__ void sub_bwb(cxd (&D)[4][4], const cxd (&Wi)[4][4], const double (&l)[4], cxd rd,
                                        const double (&v)[4]) {
  cxd wv[4];
#pragma unroll
  for (int i = 0; i < 4; i++) wv[i] = Wi[i][0] * v[0] + Wi[i][1] * v[1] + Wi[i][2] * v[2] + Wi[i][3] * v[3];
  cxd Pm[4][4];   // Wi B
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) Pm[i][j] = Wi[i][j] * l[j] + (wv[i] * rd) * v[j];
  cxd vP[4];
#pragma unroll
  for (int j = 0; j < 4; j++) vP[j] = Pm[0][j] * v[0] + Pm[1][j] * v[1] + Pm[2][j] * v[2] + Pm[3][j] * v[3];
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = 0; j < 4; j++) D[i][j] -= Pm[i][j] * l[i] + (vP[j] * rd) * v[i];
}

// The factor records of a line stand in the order of the substitution: the
// two halves one after the other, each from its boundary node towards the
// meeting node m = N/2, then the meeting node,
//     record t            (t < T)   node t - (T - m)       (top half)
//     record T + t                  node N + (T - H) - t   (bottom half)
//     record 2 T                    node m
// with H = N - m.  A record holds the node's inverse block and 1/d of its
// inner edge (towards m): edge p of a top node p, edge p - 1 of a bottom
// node.  T is H rounded up to whole groups of line_ring nodes (the
// substitution loads and unrolls by groups); the boundary nodes and the
// records before them hold zero inverses, so that their corrections are zero.
// The group is 8 nodes where that pads a half by no more than an eighth, else
// 4, and 2 for halves of at most two nodes (a single group: the back pass
// reloads a slot one step late, which a ring of two could not wait for).
__host__ __device__ __forceinline__ int line_ring(int N) {
  const int H = N - N / 2;
  return (8 - H % 8) % 8 <= H / 8 ? 8 : H > 2 ? 4 : 2;
}
struct HalfOrder {
  int N, m, T, o, ob;   // o, ob: t of the boundary node on top and below
  __host__ __device__ explicit HalfOrder(int n) : N(n), m(n / 2) {
    const int H = N - m, D = line_ring(N);
    T = (H + D - 1) / D * D;
    o = T - m;
    ob = T - H;
  }
  __host__ __device__ int records() const { return 2 * T + 1; }
  // record of node p (0..N) and the record that holds 1/d of edge e (0..N-1)
  __host__ __device__ int node(int p) const { return p < m ? p + o : p > m ? T + N + ob - p : 2 * T; }
  __host__ __device__ int edge(int e) const { return e < m ? e + o : T + N + ob - e - 1; }
};

// Colours of many long lines keep their records across the lines (chunk k of
// record r of line l at (r FC + k) nl + l) for the one-lane kernel, which then
// reads them contiguously; the others line by line for the matrix cores.
// Where lines no longer fit the LDS by the half-dozen, more than 4096 of them
// are bound by memory traffic, of which one lane per line half has the least.
// One launch of a colour, matrix cores (the better of k_line_solve_m and
// k_line_long_*) against one lane: 160 x 160 lines of 1024 nodes along z, FP64
// 2165 and 1961 us, FP32 1376 and 1313; along x 2275 and 2058, 1801 and 1514;
// 224 x 224 lines of 288 nodes along z, FP64 1088 and 908, FP32 668 and 566; of
// 256 nodes FP32 590 and 525 (160 x 160: 336 and 332).  Along x the records in
// LDS win for longer lines, as its loads and stores of u run along the lines:
// 160 x 160 of 512 nodes FP64 893 and 1000, FP32 841 and 759; of 288 nodes FP32
// 360 and 407.
__host__ __device__ __forceinline__ bool line_across(int esize, int axis, int N, long nl) {
  if (nl <= 4096) return false;
  if (axis == 0) return N > (esize == 4 ? 384 : 512);
  return N > 256 || (esize == 4 && N > 128 && nl > 8192);
}
// the records of one line (BY_LINE: known to stand line by line)
template <typename T, int A, bool BY_LINE = false>
struct FacLine {
  using C = Ch<FacRec<T>>;
  static constexpr int FC = fchunks<FacRec<T>>();
  C* base;
  long rs, cs;   // strides of the records and of their chunks
  __device__ __forceinline__ FacLine(const LineJob<T>& J, const HalfOrder& O, int line) {
    const long nl = (long)J.nlo * J.nhi;
    const bool across = !BY_LINE && line_across(sizeof(T), A, O.N, nl);
    cs = across ? nl : 1;
    rs = FC * cs;
    base = reinterpret_cast<C*>(J.fac) + (across ? line : (long)line * O.records() * FC);
  }
  __device__ __forceinline__ C* at(int r) const { return base + r * rs; }
};

// inverts D in place and stores the symmetric part with 1/d of the inner edge
template <typename R>
__device__ __forceinline__ void store_factor(Ch<R>* r, long cs, cxd (&D)[4][4], cxd rd) {
  constexpr int FC = fchunks<R>();
  inv4(D);
  Ch<R> c[FC] = {};
#pragma unroll
  for (int i = 0; i < 4; i++)
#pragma unroll
    for (int j = i; j < 4; j++) {
      const int sidx = symidx(i, j);
      const cxd w = (i == j) ? D[i][j] : (D[i][j] + D[j][i]) * 0.5;
      put(c, 2 * sidx, w.re);
      put(c, 2 * sidx + 1, w.im);
    }
  put(c, 20, rd.re);
  put(c, 21, rd.im);
#pragma unroll
  for (int k = 0; k < FC; k++) r[k * cs] = c[k];
}

// Twisted factorization of each line, meeting at node m = N/2 of the nodes
// 1..M (M = N-1):
//   top     W_1 = D_1,  W_p = D_p - B_p W_{p-1}^-1 B_p        p = 2..m-1
//   bottom  U_M = D_M,  U_p = D_p - B_{p+1} U_{p+1}^-1 B_{p+1}  p = M-1..m+1
//   middle  S_m = D_m - B_m W_{m-1}^-1 B_m - B_{m+1} U_{m+1}^-1 B_{m+1}
// The records (HalfOrder) take the inverse of each node's factor (W, S or U).
// (BY_LINE: with constant offsets 128-node lines take 353 us, else 367.)
template <typename T, int A, bool BY_LINE>
__global__ void __launch_bounds__(64) k_line_factor(LinePack<T> P) {
  using R = FacRec<T>;
  constexpr int FC = fchunks<R>();
  const LineJob<T>& J = P.job[blockIdx.y];
  const Level<T>& L = J.L;
  const int tid = blockIdx.x * blockDim.x + threadIdx.x;
  int pb, pc;
  if (!line_of<T, A>(J, tid, pb, pc)) return;
  const LineGeo<T, A> G(L, pb, pc);
  const int N = G.N;
  if (N < 2) return;
  const int M = N - 1, m = N / 2;
  const HalfOrder O(N);
  const FacLine<T, A, BY_LINE> F(J, O, tid);
  const cxd rd0 = cinv(G.d_edge(L, 0)), rdM = cinv(G.d_edge(L, M));
  // boundary nodes and the padding before them
  auto zero_rec = [&](int r, cxd rd) {
    Ch<R> c[FC] = {};
    put(c, 20, rd.re);
    put(c, 21, rd.im);
#pragma unroll
    for (int k = 0; k < FC; k++) F.at(r)[k * F.cs] = c[k];
  };
  for (int t = 0; t < O.o; t++) zero_rec(t, cxd(0, 0));
  for (int t = 0; t < O.ob; t++) zero_rec(O.T + t, cxd(0, 0));
  zero_rec(O.o, rd0);
  zero_rec(O.T + O.ob, rdM);
  cxd Wt[4][4], Wb[4][4], Dm[4][4];
  double l[4];
  cxd rd_prev = rd0;
  for (int p = 1; p <= m - 1; p++) {
    const cxd rd = cinv(G.d_edge(L, p));
    diag_block(L, G, p, rd_prev, rd, Dm);
    if (p >= 2) {
      G.lcoef(L, p - 1, l);
      sub_bwb(Dm, Wt, l, rd_prev, G.v);
    }
    store_factor(F.at(O.node(p)), F.cs, Dm, rd);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) Wt[i][j] = Dm[i][j];
    rd_prev = rd;
  }
  for (int p = M; p >= m + 1; p--) {
    const cxd rdm = cinv(G.d_edge(L, p - 1)), rdp = cinv(G.d_edge(L, p));
    diag_block(L, G, p, rdm, rdp, Dm);
    if (p <= M - 1) {
      G.lcoef(L, p, l);
      sub_bwb(Dm, Wb, l, rdp, G.v);
    }
    store_factor(F.at(O.node(p)), F.cs, Dm, rdm);
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
      for (int j = 0; j < 4; j++) Wb[i][j] = Dm[i][j];
  }
  {
    const cxd rdm = cinv(G.d_edge(L, m - 1)), rdp = cinv(G.d_edge(L, m));
    diag_block(L, G, m, rdm, rdp, Dm);
    if (m >= 2) {
      G.lcoef(L, m - 1, l);
      sub_bwb(Dm, Wt, l, rdm, G.v);
    }
    if (m <= M - 1) {
      G.lcoef(L, m, l);
      sub_bwb(Dm, Wb, l, rdp, G.v);
    }
    store_factor(F.at(O.node(m)), F.cs, Dm, cxd(0, 0));
  }
}

// z = W^{-1} y with the packed symmetric inverse held in values 0..19
template <typename R, int NC>
__device__ __forceinline__ void symv(const Ch<R> (&w)[NC], const cxd (&y)[4], cxd (&z)[4]) {
#pragma unroll
  for (int i = 0; i < 4; i++) {
    cxd acc(0, 0);
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const int s = symidx(i, j);
      acc += cxd(val(w, 2 * s), val(w, 2 * s + 1)) * y[j];
    }
    z[i] = acc;
  }
}

// Right-hand sides of the lines of one colour: one thread per (node, line),
// lines fastest, so the chunked records are written contiguously.
//   record p, slots 0..7: sigma_p, the residual of the four perpendicular
//                          edges of node p (p >= 1)
//   record p, slots 8..9: rho_p, the residual of the along-line edge p
// Lines of one colour are not coupled, so these are the residuals each line
// solve of the colour starts from.
// the records of node p of line `line` (at (pb, pc)) of job J
// the ten values of that record (node 0: rho only, the rest zero)
template <typename T, int A, typename RS>
__device__ __forceinline__ void node_rhs_rec(const LineJob<T>& J, int pb, int pc, int p, Ch<RS> (&c)[schunks<RS>()]) {
  constexpr int B = (A + 1) % 3, C = (A + 2) % 3;
  const Level<T>& L = J.L;
  const typename cvec<T>::type* __restrict__ u = J.u;
  const typename cvec<T>::type* __restrict__ f = J.f;
  const long base = (long)pb * L.es[B] + (long)pc * L.es[C] + (long)p * L.es[A];
  {
    int q[3];
    q[A] = p; q[B] = pb; q[C] = pc;
    const cxd rho = ld<T>(f, A * L.nc + base) - apply_row<T, A>(L, u, q[A], q[B], q[C], base);
    put(c, 8, rho.re);
    put(c, 9, rho.im);
  }
  if (p >= 1) {
    int q[3];
    cxd g;
    const long ob0 = base - L.es[B], oc0 = base - L.es[C];
    q[A] = p; q[B] = pb - 1; q[C] = pc;
    g = ld<T>(f, B * L.nc + ob0) - apply_row<T, B>(L, u, q[B], q[C], q[A], ob0);
    put(c, 0, g.re); put(c, 1, g.im);
    q[B] = pb;
    g = ld<T>(f, B * L.nc + base) - apply_row<T, B>(L, u, q[B], q[C], q[A], base);
    put(c, 2, g.re); put(c, 3, g.im);
    q[C] = pc - 1;
    g = ld<T>(f, C * L.nc + oc0) - apply_row<T, C>(L, u, q[C], q[A], q[B], oc0);
    put(c, 4, g.re); put(c, 5, g.im);
    q[C] = pc;
    g = ld<T>(f, C * L.nc + base) - apply_row<T, C>(L, u, q[C], q[A], q[B], base);
    put(c, 6, g.re); put(c, 7, g.im);
  }
}

// one of the five values of that record: the residual of perpendicular edge
// k = 0..3 or of the along-line edge (k = 4)
template <typename T, int A>
__device__ __forceinline__ cxd node_rhs_row(const LineJob<T>& J, int pb, int pc, int p, int k) {
  constexpr int B = (A + 1) % 3, C = (A + 2) % 3;
  const Level<T>& L = J.L;
  const typename cvec<T>::type* __restrict__ u = J.u;
  const typename cvec<T>::type* __restrict__ f = J.f;
  if (k == 0) pb--;
  if (k == 2) pc--;
  const long o = (long)pb * L.es[B] + (long)pc * L.es[C] + (long)p * L.es[A];
  if (k < 2) return ld<T>(f, B * L.nc + o) - apply_row<T, B>(L, u, pb, pc, p, o);
  if (k < 4) return ld<T>(f, C * L.nc + o) - apply_row<T, C>(L, u, pc, p, pb, o);
  return ld<T>(f, A * L.nc + o) - apply_row<T, A>(L, u, p, pb, pc, o);
}

// the records of node p of a line into its chunked scratch records
template <typename T>
__device__ __forceinline__ void store_rhs_rec(const LineJob<T>& J, int line, int p, long nl,
                                              const Ch<ScrRec<T>> (&c)[schunks<ScrRec<T>>()]) {
  using R = ScrRec<T>;
  constexpr int SC = schunks<R>(), V = Ch<R>::V;
  Ch<R>* rec = reinterpret_cast<Ch<R>*>(J.scr) + line + (long)p * SC * nl;
  if (p >= 1) {
#pragma unroll
    for (int k = 0; k < SC; k++) rec[k * nl] = c[k];
  } else {
    rec[(8 / V) * nl] = c[8 / V];   // node 0: rho_0 only (values 8, 9: one chunk)
  }
}

template <typename T, int A>
__device__ __forceinline__ void node_rhs(const LineJob<T>& J, int line, int pb, int pc, int p, long nl) {
  using R = ScrRec<T>;
  constexpr int SC = schunks<R>(), V = Ch<R>::V;
  Ch<R> c[SC] = {};
  node_rhs_rec<T, A>(J, pb, pc, p, c);
  store_rhs_rec<T>(J, line, p, nl, c);
}

// Right-hand sides of consecutive nodes of one line, marching along it.
// The five rows of a node read 30 distinct values of u; 13 of them are read
// again by node p + 1 (the same (b, c) offsets one node further back), so the
// march carries those and loads 17 per node (with f and sigma-bar of the five
// rows), against about 40 loads per node when each node is built on its own.
// A column (k, db, dc) is component (A + k) % 3 at offsets db, dc along the
// perpendicular axes B, C; the window holds it at da = lo..hi along the line.
struct MarchCol {
  int k, db, dc, lo, hi;
};
constexpr MarchCol kMarch[] = {
    {0, -1, 0, -1, 0},  {0, 0, -1, -1, 0}, {0, 0, 0, -1, 0}, {0, 0, 1, -1, 0}, {0, 1, 0, -1, 0},
    {1, -1, -1, 0, 0},  {1, -1, 0, -1, 1}, {1, -1, 1, 0, 0}, {1, 0, -1, 0, 0}, {1, 0, 0, -1, 1},
    {1, 0, 1, 0, 0},    {2, -1, -1, 0, 0}, {2, -1, 0, 0, 0}, {2, 0, -1, -1, 1}, {2, 0, 0, -1, 1},
    {2, 1, -1, 0, 0},   {2, 1, 0, 0, 0}};
constexpr int kMarchCols = sizeof(kMarch) / sizeof(kMarch[0]);
constexpr int march_col(int k, int db, int dc) {
  for (int i = 0; i < kMarchCols; i++)
    if (kMarch[i].k == k && kMarch[i].db == db && kMarch[i].dc == dc) return i;
  return -1;
}
template <int I>
struct ColIdx {
  static constexpr int value = I;
};
template <typename F, int... I>
__device__ __forceinline__ void each_col(const F& f, std::integer_sequence<int, I...>) {
  (f(ColIdx<I>{}), ...);
}
template <typename F>
__device__ __forceinline__ void each_col(const F& f) {
  each_col(f, std::make_integer_sequence<int, kMarchCols>{});
}

struct MarchWin {
  cxd v[kMarchCols][3];   // [column][da + 1]
  // the value at (da, db, dc) from the node; a position the table lacks
  // does not compile
  template <int K, int DA, int DB, int DC>
  __device__ __forceinline__ cxd at() const {
    constexpr int c = march_col(K, DB, DC);
    static_assert(c >= 0 && DA >= kMarch[c].lo && DA <= kMarch[c].hi, "position outside the march window");
    return v[c][DA + 1];
  }
};

// value KK of row X (0: its own component, 1 and 2 the next ones
// cyclically) at offsets (dx, dy, dz) along the row's axes X, X+1, X+2, for
// the row of the edge at offsets (0, RB, RC) from the node; everything in
// the line frame (0 = A, 1 = B, 2 = C)
template <int X, int RB, int RC, int KK, int dx, int dy, int dz>
__device__ __forceinline__ cxd win_val(const MarchWin& w) {
  constexpr int Y = (X + 1) % 3, Z = (X + 2) % 3;
  constexpr int da = (X == 0 ? dx : 0) + (Y == 0 ? dy : 0) + (Z == 0 ? dz : 0);
  constexpr int db = RB + (X == 1 ? dx : 0) + (Y == 1 ? dy : 0) + (Z == 1 ? dz : 0);
  constexpr int dc = RC + (X == 2 ? dx : 0) + (Y == 2 ? dy : 0) + (Z == 2 ? dz : 0);
  return w.at<(X + KK) % 3, da, db, dc>();
}
// the thirteen values of that row in row_arith's order
template <int X, int RB, int RC>
__device__ __forceinline__ void win_row(const MarchWin& w, cxd (&v)[13]) {
  v[0] = win_val<X, RB, RC, 0, 0, 0, 0>(w);
  v[1] = win_val<X, RB, RC, 1, 1, 0, 0>(w);
  v[2] = win_val<X, RB, RC, 1, 0, 0, 0>(w);
  v[3] = win_val<X, RB, RC, 0, 0, 1, 0>(w);
  v[4] = win_val<X, RB, RC, 1, 1, -1, 0>(w);
  v[5] = win_val<X, RB, RC, 1, 0, -1, 0>(w);
  v[6] = win_val<X, RB, RC, 0, 0, -1, 0>(w);
  v[7] = win_val<X, RB, RC, 0, 0, 0, 1>(w);
  v[8] = win_val<X, RB, RC, 2, 1, 0, 0>(w);
  v[9] = win_val<X, RB, RC, 2, 0, 0, 0>(w);
  v[10] = win_val<X, RB, RC, 0, 0, 0, -1>(w);
  v[11] = win_val<X, RB, RC, 2, 1, 0, -1>(w);
  v[12] = win_val<X, RB, RC, 2, 0, 0, -1>(w);
}

// the records of nodes p0 .. p1-1 of the line at (pb, pc) of job J, handed
// to sink(p, c) in order; equal, value for value, to node_rhs_rec's (the
// rows' arithmetic is row_arith in both).  Every position read lies in the
// level: nodes -1 .. N along the line are read only where node_rhs_rec reads
// them (da = -1 from node 1 on).
template <typename T, int A, typename RS = ScrRec<T>, typename Sink>
__device__ __forceinline__ void line_rhs_march(const LineJob<T>& J, int pb, int pc, int p0, int p1,
                                               const Sink& sink) {
  constexpr int B = (A + 1) % 3, C = (A + 2) % 3;
  const Level<T>& L = J.L;
  const typename cvec<T>::type* __restrict__ u = J.u;
  const typename cvec<T>::type* __restrict__ f = J.f;
  const long sa = L.es[A], sb = L.es[B], sc = L.es[C], nc = L.nc;
  // geometry of the perpendicular axes: fixed along the line
  const double iwb = L.IW[B][pb], iwbm = L.IW[B][pb - 1], hb = L.H[B][pb], wb = L.W[B][pb], wbm = L.W[B][pb - 1];
  const double iwc = L.IW[C][pc], iwcm = L.IW[C][pc - 1], hc = L.H[C][pc], wc = L.W[C][pc], wcm = L.W[C][pc - 1];
  // column ic (a compile-time index) at the node at flat index o, into the
  // window slot of da (compile-time too)
  auto load_col = [&](MarchWin& w, auto ic, auto dai, long o) {
    constexpr int ci = decltype(ic)::value, da = decltype(dai)::value;
    constexpr MarchCol m = kMarch[ci];
    w.v[ci][da + 1] = ld<T>(u, (long)((A + m.k) % 3) * nc + o + m.db * sb + m.dc * sc);
  };
  MarchWin w;
  long o = (long)pb * sb + (long)pc * sc + (long)p0 * sa;
  // the slots of da = -1 of a run from node 0 are never read (rows B and C
  // start at node 1, after a shift); they take node 0's values so that every
  // slot is written unconditionally and the window stays in registers
  const long om = p0 >= 1 ? o - sa : o;
  each_col([&](auto ic) {
    constexpr MarchCol m = kMarch[decltype(ic)::value];
    if constexpr (m.lo < 0) load_col(w, ic, ColIdx<-1>{}, om);
    load_col(w, ic, ColIdx<0>{}, o);
    if constexpr (m.hi > 0) load_col(w, ic, ColIdx<1>{}, o + sa);
  });
  double iwa_m = p0 >= 1 ? L.IW[A][p0 - 1] : 0.0;
  for (int p = p0; p < p1; p++, o += sa) {
    const double iwa = L.IW[A][p], wa = L.W[A][p], ha = L.H[A][p];
    Ch<RS> c[schunks<RS>()] = {};
    cxd v[13];
    {
      // rho_p: row A of the node, local indices (p, pb, pc)
      win_row<0, 0, 0>(w, v);
      const RowGeo g{iwa, iwb, iwbm, iwc, iwcm, hc, hb, wa, L.omu * (double)L.sbar[(long)A * nc + o]};
      const cxd rho = ld<T>(f, (long)A * nc + o) - row_arith(v, g);
      put(c, 8, rho.re);
      put(c, 9, rho.im);
    }
    if (p >= 1) {
      cxd g;
      // row B at pb - 1 and at pb: local indices (pb', pc, p)
      win_row<1, -1, 0>(w, v);
      g = ld<T>(f, (long)B * nc + o - sb) -
          row_arith(v, RowGeo{iwbm, iwc, iwcm, iwa, iwa_m, ha, hc, wbm, L.omu * (double)L.sbar[(long)B * nc + o - sb]});
      put(c, 0, g.re); put(c, 1, g.im);
      win_row<1, 0, 0>(w, v);
      g = ld<T>(f, (long)B * nc + o) -
          row_arith(v, RowGeo{iwb, iwc, iwcm, iwa, iwa_m, ha, hc, wb, L.omu * (double)L.sbar[(long)B * nc + o]});
      put(c, 2, g.re); put(c, 3, g.im);
      // row C at pc - 1 and at pc: local indices (pc', p, pb)
      win_row<2, 0, -1>(w, v);
      g = ld<T>(f, (long)C * nc + o - sc) -
          row_arith(v, RowGeo{iwcm, iwa, iwa_m, iwb, iwbm, hb, ha, wcm, L.omu * (double)L.sbar[(long)C * nc + o - sc]});
      put(c, 4, g.re); put(c, 5, g.im);
      win_row<2, 0, 0>(w, v);
      g = ld<T>(f, (long)C * nc + o) -
          row_arith(v, RowGeo{iwc, iwa, iwa_m, iwb, iwbm, hb, ha, wc, L.omu * (double)L.sbar[(long)C * nc + o]});
      put(c, 6, g.re); put(c, 7, g.im);
    }
    sink(p, c);
    if (p + 1 < p1) {
      // node p + 1: shift the window back one node and load its leading values
      each_col([&](auto ic) {
        constexpr int ci = decltype(ic)::value;
        constexpr MarchCol m = kMarch[ci];
        if constexpr (m.lo < 0) w.v[ci][0] = w.v[ci][1];
        if constexpr (m.hi > 0) {
          w.v[ci][1] = w.v[ci][2];
          load_col(w, ic, ColIdx<1>{}, o + 2 * sa);
        } else {
          load_col(w, ic, ColIdx<0>{}, o + sa);
        }
      });
    }
    iwa_m = iwa;
  }
}

template <typename T, int A>
__global__ void __launch_bounds__(256, EMMI_LINE_RHS_MIN_WAVES) k_line_rhs(LinePack<T> P) {
  const LineJob<T>& J = P.job[blockIdx.y];
  const long nl = (long)J.nlo * J.nhi;
  const int N = J.L.n[A];
  const long t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (t >= nl * N) return;
  const unsigned pu = (unsigned)t / (unsigned)nl;   // fewer than 2^32 nodes per launch
  const int p = (int)pu;
  const int line = (int)((unsigned)t - pu * (unsigned)nl);
  int pb, pc;
  line_of<T, A>(J, line, pb, pc);
  node_rhs<T, A>(J, line, pb, pc, p, nl);
}

// The same records built by marching (line_rhs_march): a thread per run of
// `run` consecutive nodes of a line, lines fastest (y and z lines, whose
// neighbours lie side by side along x)
template <typename T, int A>
__global__ void __launch_bounds__(256) k_line_rhs_run(LinePack<T> P, int run) {
  const LineJob<T>& J = P.job[blockIdx.y];
  const long nl = (long)J.nlo * J.nhi;
  const int N = J.L.n[A];
  const long nruns = (N + run - 1) / run;
  const long t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (t >= nl * nruns) return;
  const int r = (int)(t / nl), line = (int)(t - (long)r * nl);
  const int p0 = r * run, p1 = min(N, p0 + run);
  int pb, pc;
  line_of<T, A>(J, line, pb, pc);
  line_rhs_march<T, A>(J, pb, pc, p0, p1, [&](int p, const Ch<ScrRec<T>>(&c)[schunks<ScrRec<T>>()]) {
    store_rhs_rec<T>(J, line, p, nl, c);
  });
}

// Right-hand sides for lines along x (axis 0): consecutive lines lie in
// different x rows, so a thread per (node, line) with lines fastest would
// load one cache line per lane.  A block takes a tile of 16 nodes x 16 lines,
// computes with nodes fastest (loads contiguous along x) and transposes the
// records through LDS so the stores run along the lines.
constexpr int XT = 16;

template <typename T>
__global__ void __launch_bounds__(256, EMMI_LINE_RHS_MIN_WAVES) k_line_rhs_x(LinePack<T> P, int nlb) {
  constexpr int A = 0, B = 1, C = 2;
  __shared__ double tile[SREC][XT][XT + 1];
  const LineJob<T>& J = P.job[blockIdx.y];
  const Level<T>& L = J.L;
  const long nl = (long)J.nlo * J.nhi;
  const int N = L.n[A];
  // XCD-aware order: each XCD takes a contiguous range of tiles (a slab of
  // nodes over all lines), so the rows that neighbouring line tiles share
  // are fetched into one L2 (in dispatch order they land on different XCDs
  // and the level-0 launch fetched 2.4x its bytes)
  const long bl = xcd_block(blockIdx.x, gridDim.x);
  const int lb = (int)(bl % nlb), pbk = (int)(bl / nlb);
  const long l0 = (long)lb * XT;
  const int p0 = pbk * XT;
  if (l0 >= nl || p0 >= N) return;   // uniform over the block
  {
    const int pl = threadIdx.x % XT, ll = threadIdx.x / XT;
    const int p = p0 + pl;
    const long line = l0 + ll;
    double v[SREC];
#pragma unroll
    for (int k = 0; k < SREC; k++) v[k] = 0.0;
    if (p < N && line < nl) {
      int pb, pc;
      line_of<T, A>(J, (int)line, pb, pc);
      const typename cvec<T>::type* __restrict__ u = J.u;
      const typename cvec<T>::type* __restrict__ f = J.f;
      const long base = (long)pb * L.es[B] + (long)pc * L.es[C] + (long)p * L.es[A];
      int q[3];
      q[A] = p; q[B] = pb; q[C] = pc;
      const cxd rho = ld<T>(f, A * L.nc + base) - apply_row<T, A>(L, u, q[A], q[B], q[C], base);
      v[8] = rho.re;
      v[9] = rho.im;
      if (p >= 1) {
        cxd g;
        const long ob0 = base - L.es[B], oc0 = base - L.es[C];
        q[B] = pb - 1;
        g = ld<T>(f, B * L.nc + ob0) - apply_row<T, B>(L, u, q[B], q[C], q[A], ob0);
        v[0] = g.re; v[1] = g.im;
        q[B] = pb;
        g = ld<T>(f, B * L.nc + base) - apply_row<T, B>(L, u, q[B], q[C], q[A], base);
        v[2] = g.re; v[3] = g.im;
        q[C] = pc - 1;
        g = ld<T>(f, C * L.nc + oc0) - apply_row<T, C>(L, u, q[C], q[A], q[B], oc0);
        v[4] = g.re; v[5] = g.im;
        q[C] = pc;
        g = ld<T>(f, C * L.nc + base) - apply_row<T, C>(L, u, q[C], q[A], q[B], base);
        v[6] = g.re; v[7] = g.im;
      }
#pragma unroll
      for (int k = 0; k < SREC; k++) tile[k][pl][ll] = v[k];
    }
  }
  __syncthreads();
  {
    const int ll = threadIdx.x % XT, pl = threadIdx.x / XT;
    const int p = p0 + pl;
    const long line = l0 + ll;
    if (p < N && line < nl) {
      using R = ScrRec<T>;
      constexpr int SC = schunks<R>(), V = Ch<R>::V;
      Ch<R> c[SC] = {};
#pragma unroll
      for (int k = 0; k < SREC; k++) put(c, k, tile[k][pl][ll]);
      Ch<R>* rec = reinterpret_cast<Ch<R>*>(J.scr) + line + (long)p * SC * nl;
      if (p >= 1) {
#pragma unroll
        for (int k = 0; k < SC; k++) rec[k * nl] = c[k];
      } else {
        rec[(8 / V) * nl] = c[8 / V];
      }
    }
  }
}

// t = B z for the coupling B = diag(l) + v v^T rd of two neighbouring nodes
template <typename T, int A>
__device__ __forceinline__ void bmul(const LineGeo<T, A>& G, const cxd (&z)[4], double iWe, cxd rd, cxd (&t)[4]) {
  const double l[4] = {-G.Wb0 * G.Hc * iWe, -G.Wb1 * G.Hc * iWe, -G.Wc0 * G.Hb * iWe, -G.Wc1 * G.Hb * iWe};
  const cxd vz = z[0] * G.v[0] + z[1] * G.v[1] + z[2] * G.v[2] + z[3] * G.v[3];
#pragma unroll
  for (int i = 0; i < 4; i++) t[i] = z[i] * l[i] + (vz * rd) * G.v[i];
}

template <typename R, int NC>
__device__ __forceinline__ cxd cval(const Ch<R> (&c)[NC], int k) { return cxd(val(c, k), val(c, k + 1)); }

// Lines along x (axis 0) lie in different x rows, so a wave updating u node
// by node would write 64 scattered 8-byte values per store, and the L2
// evicts those partly written lines: the substitution along x wrote 2.7x the
// bytes of the other axes.  Instead it leaves each node's corrections in the
// node's line record (its z values are dead by then; values 0,1: the
// along-line edge, 2..9: the four node edges) and k_line_solve_x_apply adds
// them to u with the lanes running along x.
template <typename RS>
__device__ __forceinline__ void put_corr(Ch<RS>* __restrict__ rec, long stride, cxd ea, const cxd (&ap)[4]) {
  constexpr int SC = schunks<RS>();
  Ch<RS> c[SC] = {};
  put(c, 0, ea.re);
  put(c, 1, ea.im);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    put(c, 2 + 2 * i, ap[i].re);
    put(c, 3 + 2 * i, ap[i].im);
  }
#pragma unroll
  for (int k = 0; k < SC; k++) rec[k * stride] = c[k];
}

// u += the corrections left in the line records by k_line_solve<T, 0>: a
// block takes 16 nodes x 16 lines, reads the records with lines fastest and
// updates u through an LDS transpose with nodes fastest.  Node m = N/2 (its
// node edges are updated by the substitution itself) and node 0 hold no
// correction; the along-line edge of node p is p below m and p-1 above.
template <typename T>
__global__ void __launch_bounds__(XT * XT) k_line_solve_x_apply(LinePack<T> P, int nlb) {
  constexpr int A = 0;
  using RS = ScrRec<T>;
  constexpr int SC = schunks<RS>();
  __shared__ double tile[SREC][XT][XT + 1];
  const LineJob<T>& J = P.job[blockIdx.y];
  const Level<T>& L = J.L;
  const long nl = (long)J.nlo * J.nhi;
  const int N = L.n[A], m = N / 2;
  const int lb = blockIdx.x % nlb, pbk = blockIdx.x / nlb;
  const long l0 = (long)lb * XT;
  const int p0 = pbk * XT;
  if (l0 >= nl || p0 >= N) return;   // uniform over the block
  {
    const int ll = threadIdx.x % XT, pl = threadIdx.x / XT;
    const int p = p0 + pl;
    const long line = l0 + ll;
    if (p < N && line < nl && p >= 1 && p != m) {
      const Ch<RS>* rec = reinterpret_cast<const Ch<RS>*>(J.scr) + line + (long)p * SC * nl;
      Ch<RS> c[SC];
#pragma unroll
      for (int k = 0; k < SC; k++) c[k] = rec[k * nl];
#pragma unroll
      for (int k = 0; k < SREC; k++) tile[k][pl][ll] = val(c, k);
    }
  }
  __syncthreads();
  {
    const int pl = threadIdx.x % XT, ll = threadIdx.x / XT;
    const int p = p0 + pl;
    const long line = l0 + ll;
    if (p < N && line < nl && p >= 1 && p != m) {
      int pb, pc;
      line_of<T, A>(J, (int)line, pb, pc);
      const LineGeo<T, A> G(L, pb, pc);
      typename cvec<T>::type* __restrict__ u = J.u;
      const long o = (long)p * G.sa;
      const long ea = G.oa + (long)(p < m ? p : p - 1) * G.sa;
      st<T>(u, ea, ld<T>(u, ea) + cxd(tile[0][pl][ll], tile[1][pl][ll]));
      const long offs[4] = {G.ob0, G.ob1, G.oc0, G.oc1};
#pragma unroll
      for (int i = 0; i < 4; i++)
        st<T>(u, offs[i] + o, ld<T>(u, offs[i] + o) + cxd(tile[2 + 2 * i][pl][ll], tile[3 + 2 * i][pl][ll]));
    }
  }
}

// Block substitution of the lines of one colour on the twisted factors
// (k_line_factor).  A block of 128 threads takes 64 lines: wave 0 ("top")
// eliminates nodes 1..m-1 downwards and wave 1 ("bottom") nodes M..m+1
// upwards at the same time,
//   top     z_p = W_p^-1 (g_p - B_p z_{p-1})
//   bottom  z_p = U_p^-1 (g_p - B_{p+1} z_{p+1}),
// the waves exchange B_m z_{m-1} and B_{m+1} z_{m+1} through LDS, both solve
// the meeting node x_m = S_m^-1 (g_m - B_m z_{m-1} - B_{m+1} z_{m+1}), and
// each substitutes back over its half,
//   top     x_p = z_p - W_p^-1 B_{p+1} x_{p+1}     p = m-1..1
//   bottom  x_p = z_p - U_p^-1 B_p x_{p-1}         p = m+1..M,
// updating the along-line edges dE_a(e) = q_e + v.(x_{e+1} - x_e) / d_e
// (top: edges 0..m-1, bottom: m..N-1; q_e = rho_e / d_e) and the node
// edges.  g_p = sigma_p + v (q_{p-1} - q_p).  Each wave keeps the chunks of
// its next D nodes in flight in a register ring; ring loads past the end of
// a half are clamped into the line and never used.  The forward passes
// overwrite sigma_p with z_p.
template <typename T, int A>
__global__ void __launch_bounds__(128) k_line_solve(LinePack<T> P) {
  using E = typename cvec<T>::type;
  using RF = FacRec<T>;
  using RS = ScrRec<T>;
  constexpr int FC = fchunks<RF>(), SC = schunks<RS>(), VF = Ch<RF>::V, VS = Ch<RS>::V, D = ring_depth<T>();
  constexpr int ZC = 8 / VS;    // chunks holding values 0..7 (sigma, then z)
  constexpr int CD = 20 / VF;   // factor chunk holding 1/d (values 20, 21)
  constexpr int CQ = 8 / VS;    // record chunk holding rho (values 8, 9)
  __shared__ double xch[2][8][64];
  const LineJob<T>& J = P.job[blockIdx.y];
  const Level<T>& L = J.L;
  const int N = L.n[A];
  if (N < 2) return;   // uniform over the block: no interior node
  const int M = N - 1, m = N / 2;
  const int lane = threadIdx.x & 63, side = threadIdx.x >> 6;
  const int line = blockIdx.x * 64 + lane;
  int pb = 0, pc = 0;
  const bool live = line_of<T, A>(J, line, pb, pc);
  LineGeo<T, A> G;
  if (live) G.init(L, pb, pc);
  const long stride = (long)J.nlo * J.nhi;
  const HalfOrder O(N);
  const FacLine<T, A> F(J, O, line);
  const long fs = F.cs;
  auto fnode = [&](int p) -> const Ch<RF>* { return F.at(O.node(p)); };   // the node's inverse, 1/d of its inner edge
  auto fedge = [&](int e) { return F.at(O.edge(e))[CD * fs]; };           // 1/d of an edge
  Ch<RS>* __restrict__ scr = reinterpret_cast<Ch<RS>*>(J.scr) + line;
  E* __restrict__ u = J.u;
  const double* __restrict__ iw = L.IW[A];
  const long sstep = (long)SC * stride;
  const long off_u[5] = {G.oa, G.ob0, G.ob1, G.oc0, G.oc1};

  // D nodes ahead are in flight: the load for node p + D goes into the slot
  // node p - 1 used, so a slot is never copied before it is refilled
  constexpr int R = D + 1;
  Ch<RF> rf[R][FC];
  Ch<RS> rs[R][SC];
  double riw[R];
  cxd tm[4];   // this half's coupling term at the meeting node
#pragma unroll
  for (int i = 0; i < 4; i++) tm[i] = cxd(0, 0);

  // ---------------- forward elimination ----------------
  if (live && side == 0) {
    const int last = m - 1;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int pn = max(min(1 + d, last), 1);
      load_node(rf[d], fnode(pn), fs);
      load_node(rs[d], scr + pn * sstep, stride);
      riw[d] = iw[pn - 1];
    }
    const Ch<RF> f0 = fedge(0);
    const Ch<RS> s0 = scr[CQ * stride];
    cxd rd_prev((double)f0.v[20 % VF], (double)f0.v[21 % VF]);
    cxd q_prev = cxd((double)s0.v[8 % VS], (double)s0.v[9 % VS]) * rd_prev;
    cxd z[4];
    auto step = [&](const int p, const int d) {
      const Ch<RF>(&cf)[FC] = rf[d];
      const Ch<RS>(&cr)[SC] = rs[d];
      const double iWe = (double)riw[d];
      {
        const int pn = min(p + D, last), dn = (d + D) % R;
        load_node(rf[dn], fnode(pn), fs);
        load_node(rs[dn], scr + pn * sstep, stride);
        riw[dn] = iw[pn - 1];
      }
      const cxd rd = cval(cf, 20);
      const cxd q = cval(cr, 8) * rd;
      const cxd dq = q_prev - q;
      cxd g[4];
#pragma unroll
      for (int i = 0; i < 4; i++) g[i] = cval(cr, 2 * i) + dq * G.v[i];
      if (p >= 2) {
        cxd t[4];
        bmul(G, z, iWe, rd_prev, t);
#pragma unroll
        for (int i = 0; i < 4; i++) g[i] -= t[i];
      }
      symv(cf, g, z);
      Ch<RS> zc[SC] = {};
#pragma unroll
      for (int i = 0; i < 4; i++) { put(zc, 2 * i, z[i].re); put(zc, 2 * i + 1, z[i].im); }
      Ch<RS>* sp = scr + p * sstep;
#pragma unroll
      for (int k = 0; k < ZC; k++) sp[k * stride] = zc[k];
      rd_prev = rd;
      q_prev = q;
    };
    // whole groups of R nodes without a guard per node (guards inside the
    // group make the register allocator copy the ring), then the rest
    int p0 = 1;
    for (; p0 + (R - 1) <= last; p0 += R) {
#pragma unroll
      for (int d = 0; d < R; d++) step(p0 + d, d);
    }
#pragma unroll
    for (int d = 0; d < R - 1; d++)
      if (p0 + d <= last) step(p0 + d, d);
    if (m >= 2) bmul(G, z, (double)iw[m - 1], rd_prev, tm);   // B_m z_{m-1}
  } else if (live) {
    // ring entries also carry rho_{p-1} of the node above and 1/d_p
    Ch<RF> rdn[R];
    Ch<RS> rqn[R];
    const int last = m + 1;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int pn = min(max(M - d, last), M);
      load_node(rf[d], fnode(pn), fs);
      load_node(rs[d], scr + pn * sstep, stride);
      rdn[d] = fedge(pn);
      rqn[d] = scr[(pn - 1) * sstep + CQ * stride];
      riw[d] = iw[pn];
    }
    cxd zn[4], rd_last(0, 0);
    auto step = [&](const int p, const int d) {
      const Ch<RF>(&cf)[FC] = rf[d];
      const Ch<RS>(&cr)[SC] = rs[d];
      const Ch<RF>& cdp = rdn[d];
      const Ch<RS>& cqm = rqn[d];
      const double iWe = (double)riw[d];
      {
        const int pn = max(p - D, last), dn = (d + D) % R;
        load_node(rf[dn], fnode(pn), fs);
        load_node(rs[dn], scr + pn * sstep, stride);
        rdn[dn] = fedge(pn);
        rqn[dn] = scr[(pn - 1) * sstep + CQ * stride];
        riw[dn] = iw[pn];
      }
      const cxd rd((double)cdp.v[20 % VF], (double)cdp.v[21 % VF]);
      const cxd q = cval(cr, 8) * rd;
      const cxd rdm = cval(cf, 20);
      const cxd qm = cxd((double)cqm.v[8 % VS], (double)cqm.v[9 % VS]) * rdm;
      const cxd dq = qm - q;
      cxd g[4];
#pragma unroll
      for (int i = 0; i < 4; i++) g[i] = cval(cr, 2 * i) + dq * G.v[i];
      if (p <= M - 1) {
        cxd t[4];
        bmul(G, zn, iWe, rd, t);
#pragma unroll
        for (int i = 0; i < 4; i++) g[i] -= t[i];
      }
      symv(cf, g, zn);
      Ch<RS> zc[SC] = {};
#pragma unroll
      for (int i = 0; i < 4; i++) { put(zc, 2 * i, zn[i].re); put(zc, 2 * i + 1, zn[i].im); }
      Ch<RS>* sp = scr + p * sstep;
#pragma unroll
      for (int k = 0; k < ZC; k++) sp[k * stride] = zc[k];
      rd_last = rdm;   // 1/d_{p-1}: after the loop, 1/d_m
    };
    // whole groups of R nodes without a guard per node (guards inside the
    // group make the register allocator copy the ring), then the rest
    int p0 = M;
    for (; p0 - (R - 1) >= last; p0 -= R) {
#pragma unroll
      for (int d = 0; d < R; d++) step(p0 - d, d);
    }
#pragma unroll
    for (int d = 0; d < R - 1; d++)
      if (p0 - d >= last) step(p0 - d, d);
    if (m + 1 <= M) bmul(G, zn, (double)iw[m], rd_last, tm);   // B_{m+1} z_{m+1}
  }

  // ---------------- meeting node ----------------
#pragma unroll
  for (int i = 0; i < 4; i++) {
    xch[side][2 * i][lane] = tm[i].re;
    xch[side][2 * i + 1][lane] = tm[i].im;
  }
  __syncthreads();
  if (!live) return;
  cxd xm[4], qmid, rdmid;
  {
    Ch<RF> cf[FC];
          Ch<RS> cr[SC];
    load_node(cf, fnode(m), fs);
    load_node(cr, scr + m * sstep, stride);
    const Ch<RF> cdm = fedge(m - 1), cdp = fedge(m);
    const Ch<RS> cqm = scr[(m - 1) * sstep + CQ * stride];
    rdmid = cxd((double)cdp.v[20 % VF], (double)cdp.v[21 % VF]);
    qmid = cval(cr, 8) * rdmid;
    const cxd rdm((double)cdm.v[20 % VF], (double)cdm.v[21 % VF]);
    const cxd dq = cxd((double)cqm.v[8 % VS], (double)cqm.v[9 % VS]) * rdm - qmid;
    cxd g[4];
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const cxd ttop(xch[0][2 * i][lane], xch[0][2 * i + 1][lane]);
      const cxd tbot(xch[1][2 * i][lane], xch[1][2 * i + 1][lane]);
      g[i] = ((cval(cr, 2 * i) + dq * G.v[i]) - ttop) - tbot;
    }
    symv(cf, g, xm);
  }

  // ---------------- back substitution ----------------
  E ru[R][5];
  if (side == 0) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const long o = off_u[i + 1] + (long)m * G.sa;
      st<T>(u, o, ld<T>(u, o) + xm[i]);
    }
    const int last = m - 1;
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int pn = max(last - d, 1);
      load_node(rf[d], fnode(pn), fs);
      load_node(rs[d], scr + pn * sstep, stride);
      riw[d] = iw[pn];
      if constexpr (A != 0) {
#pragma unroll
        for (int k = 0; k < 5; k++) ru[d][k] = u[off_u[k] + (long)pn * G.sa];
      }
    }
    cxd an[4];   // x_{p+1}
#pragma unroll
    for (int i = 0; i < 4; i++) an[i] = xm[i];
    auto step = [&](const int p, const int d) {
      const Ch<RF>(&cf)[FC] = rf[d];
      const Ch<RS>(&cr)[SC] = rs[d];
      const E(&cu)[5] = ru[d];
      const double iWe = (double)riw[d];
      {
        const int pn = max(p - D, 1), dn = (d + D) % R;
        load_node(rf[dn], fnode(pn), fs);
        load_node(rs[dn], scr + pn * sstep, stride);
        riw[dn] = iw[pn];
        if constexpr (A != 0) {
#pragma unroll
          for (int k = 0; k < 5; k++) ru[dn][k] = u[off_u[k] + (long)pn * G.sa];
        }
      }
      const cxd rd = cval(cf, 20);
      const cxd q = cval(cr, 8) * rd;
      cxd t[4], wt[4], ap[4];
      bmul(G, an, iWe, rd, t);
      symv(cf, t, wt);
#pragma unroll
      for (int i = 0; i < 4; i++) ap[i] = cval(cr, 2 * i) - wt[i];
      cxd dv(0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) dv += (an[i] - ap[i]) * G.v[i];
      if constexpr (A == 0) {
        put_corr(scr + p * sstep, stride, q + dv * rd, ap);
      } else {
        const long o = (long)p * G.sa;
        st<T>(u, G.oa + o, cxd((double)cu[0].x, (double)cu[0].y) + (q + dv * rd));
#pragma unroll
        for (int i = 0; i < 4; i++)
          st<T>(u, off_u[i + 1] + o, cxd((double)cu[i + 1].x, (double)cu[i + 1].y) + ap[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) an[i] = ap[i];
    };
    // whole groups of R nodes without a guard per node (guards inside the
    // group make the register allocator copy the ring), then the rest
    int p0 = last;
    for (; p0 - (R - 1) >= 1; p0 -= R) {
#pragma unroll
      for (int d = 0; d < R; d++) step(p0 - d, d);
    }
#pragma unroll
    for (int d = 0; d < R - 1; d++)
      if (p0 - d >= 1) step(p0 - d, d);
    // along-line edge 0, between the boundary node and node 1
    const Ch<RF> f0 = fedge(0);
    const Ch<RS> s0 = scr[CQ * stride];
    const cxd rd0((double)f0.v[20 % VF], (double)f0.v[21 % VF]);
    const cxd q0 = cxd((double)s0.v[8 % VS], (double)s0.v[9 % VS]) * rd0;
    cxd dv(0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) dv += an[i] * G.v[i];
    st<T>(u, G.oa, ld<T>(u, G.oa) + (q0 + dv * rd0));
  } else {
    const int last = m + 1;
    Ch<RF> rdn[R];   // 1/d_p of the ring nodes
#pragma unroll
    for (int d = 0; d < D; d++) {
      const int pn = min(last + d, M);
      load_node(rf[d], fnode(pn), fs);
      rdn[d] = fedge(pn);
      load_node(rs[d], scr + pn * sstep, stride);
      riw[d] = iw[pn - 1];
      if constexpr (A != 0) {
        ru[d][0] = u[G.oa + (long)(pn - 1) * G.sa];
#pragma unroll
        for (int k = 1; k < 5; k++) ru[d][k] = u[off_u[k] + (long)pn * G.sa];
      }
    }
    cxd xp[4];   // x_{p-1}
#pragma unroll
    for (int i = 0; i < 4; i++) xp[i] = xm[i];
    cxd rdm = rdmid, qm = qmid;   // 1/d and q of edge p-1
    auto step = [&](const int p, const int d) {
      const Ch<RF>(&cf)[FC] = rf[d];
      const Ch<RS>(&cr)[SC] = rs[d];
      const E(&cu)[5] = ru[d];
      const double iWe = (double)riw[d];
      {
        const int pn = min(p + D, M), dn = (d + D) % R;
        load_node(rf[dn], fnode(pn), fs);
        rdn[dn] = fedge(pn);
        load_node(rs[dn], scr + pn * sstep, stride);
        riw[dn] = iw[pn - 1];
        if constexpr (A != 0) {
          ru[dn][0] = u[G.oa + (long)(pn - 1) * G.sa];
#pragma unroll
          for (int k = 1; k < 5; k++) ru[dn][k] = u[off_u[k] + (long)pn * G.sa];
        }
      }
      const cxd rd((double)rdn[d].v[20 % VF], (double)rdn[d].v[21 % VF]);
      const cxd q = cval(cr, 8) * rd;
      cxd t[4], wt[4], ap[4];
      bmul(G, xp, iWe, rdm, t);
      symv(cf, t, wt);
#pragma unroll
      for (int i = 0; i < 4; i++) ap[i] = cval(cr, 2 * i) - wt[i];
      cxd dv(0, 0);
#pragma unroll
      for (int i = 0; i < 4; i++) dv += (ap[i] - xp[i]) * G.v[i];
      if constexpr (A == 0) {
        put_corr(scr + p * sstep, stride, qm + dv * rdm, ap);
      } else {
        const long o = (long)p * G.sa;
        st<T>(u, G.oa + o - G.sa, cxd((double)cu[0].x, (double)cu[0].y) + (qm + dv * rdm));
#pragma unroll
        for (int i = 0; i < 4; i++)
          st<T>(u, off_u[i + 1] + o, cxd((double)cu[i + 1].x, (double)cu[i + 1].y) + ap[i]);
      }
#pragma unroll
      for (int i = 0; i < 4; i++) xp[i] = ap[i];
      rdm = rd;
      qm = q;
    };
    // whole groups of R nodes without a guard per node (guards inside the
    // group make the register allocator copy the ring), then the rest
    int p0 = last;
    for (; p0 + (R - 1) <= M; p0 += R) {
#pragma unroll
      for (int d = 0; d < R; d++) step(p0 + d, d);
    }
#pragma unroll
    for (int d = 0; d < R - 1; d++)
      if (p0 + d <= M) step(p0 + d, d);
    // along-line edge M = N-1, between node M and the boundary node
    cxd dv(0, 0);
#pragma unroll
    for (int i = 0; i < 4; i++) dv += (cxd(0, 0) - xp[i]) * G.v[i];
    const long o = G.oa + (long)M * G.sa;
    st<T>(u, o, ld<T>(u, o) + (qm + dv * rdm));
  }
}

// ---------------------------------------------------------------------------
// substitution on the FP64 matrix cores
// ---------------------------------------------------------------------------
// One launch per colour: a block takes LPB neighbouring lines, builds their
// residual records in LDS with all its threads, substitutes with 16 lanes per
// line half, and adds the corrections to u with all its threads again.
//
// v_mfma_f64_4x4x4_4b multiplies four 4x4 pairs at once, with lanes
//     A[i][k] at i + 4 b + 16 k,  B[k][j] at j + 4 b + 16 k,
//     D[i][j] at j + 4 b + 16 i          (b = 0..3: the pair),
// so a product's D is the next product's B without any exchange.  The pairs
// are the two halves (b / 2) of two lines (b % 2): a wave runs both chains of
// its two lines with one instruction stream, since the bottom half is the top
// half mirrored (the sign of v changes, nothing else).  Column j % 2 of B and
// D holds the real (0) and imaginary (1) parts of a node vector (columns 2
// and 3 repeat 0 and 1), a complex product M y is
//     Re M [y.re, y.im] + Im M [-y.im, y.re]
// -- two matrix instructions and one exchange of neighbouring lanes -- and A
// holds the node's 4x4 matrices, symmetric, one complex entry per lane.
// A node of the forward pass is y = g - B z, z = W^-1 y (three matrix
// instructions, the chain), one of the back pass x = z - W^-1 B x' (three) and
// the along-line edge q + v.(x' - x) / d (one, off the chain).
//
// Why: four lanes per line half on the vector units took 120 (forward) and
// 160 (back) instructions and about 0.45 us a node, two substituting waves per
// CU; a step here takes 35 and 44 instructions around a chain of about 150 cycles
// (62 ns).  Blocks of eight lines keep their records in 80 KiB of LDS at 128
// nodes (in FP64; FP32-storage cycles round sigma, rho and z to FP32), so two blocks and eight
// substituting waves share a CU.  Launches with few lines are bound by the
// chain of N / 2 nodes, large ones by the two reads of the factor records and
// the stencil traffic (128 nodes: about 5 TB/s).  Per launch of a colour, four
// lanes per half and cyclic reduction for single lines -> here: 128 nodes,
// FP64, one right-hand side 137 -> 107 us along y and z, 145 -> 83 along x;
// FP32, three 245 -> 225 and 280 -> 196; 96 nodes, FP32, eight 370 -> 248 and
// 330 -> 218; 64 nodes, FP64, one 37 -> 24; 16 nodes 12.5 -> 9.5; one line of 96
// nodes, eight right-hand sides 26 -> 16.
// LDS of a line: 2 T edges (1 complex), 2 T - 1 node vectors (4 complex) and
// room for one more, which the last step's read of the node after next meets
__host__ __device__ __forceinline__ int line_m_bytes(int n) { return 160 * HalfOrder(n).T; }
static int line_m_lpb(int n) { return 8 * line_m_bytes(n) <= CU_LDS ? 8 : 2; }
static bool line_m_fits(int n) { return 2 * line_m_bytes(n) <= CU_LDS; }
// lines whose records are in memory: lines of a block, nodes in flight per half
constexpr int LONG_LPB = 8, LONG_RING = 8;

// (re, im) -> (-im, re) across the columns of a node vector; sg flips the
// sign of the even columns
__device__ __forceinline__ double mswap(double x, unsigned sg) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0xB1, 0xF, 0xF, true);          // quad_perm [1,0,3,2]
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0xB1, 0xF, 0xF, true);
  return __longlong_as_double(((long long)(int)((unsigned)hi ^ sg) << 32) | (unsigned int)lo);
}
// the other half's value (pairs b and b ^ 2: eight lanes on in the row of 16)
__device__ __forceinline__ double mpeer(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_mov_dpp((int)b, 0x128, 0xF, 0xF, true);         // row_ror:8
  const int hi = __builtin_amdgcn_mov_dpp((int)(b >> 32), 0x128, 0xF, 0xF, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}
__device__ __forceinline__ double mma(double a, double b, double c) {
  return __builtin_amdgcn_mfma_f64_4x4x4f64(a, b, c, 0, 0, 0);
}
// a value of the line records, rounded to the cycle's precision
template <typename T>
__device__ __forceinline__ double rec_val(double x) {
  return (double)(ScrRec<T>)x;
}
// ends a node of the unrolled passes, and before that sets its reload of the
// ring apart: left to itself the scheduler gathers the off-chain products of a
// whole group at its start, and waits there for every load of the ring, or
// issues a reload before the last use of its slot, into registers of its own
// that are copied back (and waited for) at the end of the group
__device__ __forceinline__ void node_end() { __builtin_amdgcn_sched_barrier(0); }

// One lane of the substitution of two lines by a wave (see above).  ST: lines
// side by side in the block's records (the stride between a line's slots).
// MEM: these records are in memory, in the cycle's precision, and the back pass
// adds to u itself; the ring holds a node's part of them beside its factor
// records, as a read of memory takes the time of many nodes.
template <typename T, int A, int D, int ST, bool MEM>
struct HalfLane {
  static constexpr int XS = 8 * ST, QS = 2 * ST;   // doubles between the slots of a line
  static constexpr int RB = fchunks<double>() * 16;   // bytes of a factor record
  int row, j, side, jr;
  unsigned sg;            // sign of the swapped operand's even columns
  double vr, vs, ncl;     // v (entry (j, row) of an A operand whose rows are all v); v of this half; -l W_a
  const char* fb;         // factor records of the wave's lines from a uniform base,
  unsigned fw, fr, fm;    // node d of the current group at a constant offset
  const double* iwa;
  int e0, de, last, TT;   // inner edge of node t: e0 + de t
  bool exact;             // z is kept in FP64 (a single line: the coarsest level)
  double *xq, *qa, *xm;   // LDS: vector component and edge of node t of the half, meeting node
  int qx;                 // from the component jr to the other one
  double2 rw[D], rr[D], wm;
  double ri[D];
  // MEM: sigma (then z), rho and u (node edge, inner edge) of the node
  ScrRec<T> rs[D], ra_[D], rb_[D], *xr, *qr, *xmr;
  T un[D], ue[D], *u0, *ue0, *um;
  long su, sue;
  int t1;                 // first node of the half that is not padding (the boundary node)

  __device__ __forceinline__ HalfLane() {
    const int lane = threadIdx.x & 63;
    row = lane >> 4;
    j = lane & 3;
    side = (lane >> 3) & 1;
    jr = j & 1;
  }
  // 1 for the lanes of the wave's second line
  __device__ __forceinline__ int second() const { return (threadIdx.x >> 2) & 1; }
  // line (pb, pc), the `dl`-th of the wave's lines, whose first is line
  // `first` of the colour; x0, q0: the line's first slots in LDS
  __device__ __forceinline__ void init(const Level<T>& L, const HalfOrder& O, int pb, int pc, const double* fac,
                                       int first, int dl, bool exact_, double2* x0, double2* q0) {
    const LineGeo<T, A> G(L, pb, pc);
    const double h = row < 2 ? G.Hc : G.Hb;
    vr = (row & 1) ? -h : h;
    vs = side ? -vr : vr;
    ncl = row == 0 ? G.Wb0 * G.Hc : row == 1 ? G.Wb1 * G.Hc : row == 2 ? G.Wc0 * G.Hb : G.Wc1 * G.Hb;
    sg = jr ? 0u : 0x80000000u;
    TT = O.T;
    exact = exact_;
    fb = reinterpret_cast<const char*>(fac) + (long)first * O.records() * RB;
    const unsigned fl = (unsigned)(dl * O.records() * RB), sym = 16 * symidx(j, row);
    fw = fl + side * TT * RB + sym;
    fr = fl + side * TT * RB + 160;
    fm = fl + 2 * TT * RB + sym;
    // t - o on top, N + ob - 1 - t below (clamped: the padding's value meets z = 0)
    iwa = L.IW[A];
    e0 = side ? O.N + O.ob - 1 : -O.o;
    de = side ? -1 : 1;
    last = O.N - 1;
    if constexpr (!MEM) {
      xq = reinterpret_cast<double*>(x0) + (side * (TT - 1) - 1) * XS + 2 * row + jr;
      xm = reinterpret_cast<double*>(x0) + (2 * TT - 2) * XS + 2 * row + jr;
      qa = reinterpret_cast<double*>(q0) + side * TT * QS + jr;
    } else {
      xq = xm = qa = nullptr;   // init_mem
    }
    qx = 1 - 2 * jr;
  }
  // MEM: the records of the line and the u of node 0 of the half
  __device__ __forceinline__ void init_mem(const Level<T>& L, const HalfOrder& O, int pb, int pc, ScrRec<T>* x0,
                                           ScrRec<T>* q0, typename cvec<T>::type* u) {
    const LineGeo<T, A> G(L, pb, pc);
    xr = x0 + (side * (TT - 1) - 1) * XS + 2 * row + jr;
    xmr = x0 + (2 * TT - 2) * XS + 2 * row + jr;
    qr = q0 + side * TT * QS + jr;
    t1 = side ? O.ob : O.o;
    su = (side ? -2 : 2) * G.sa;
    T* uc = reinterpret_cast<T*>(u) + jr;
    u0 = uc + 2 * (row == 0 ? G.ob0 : row == 1 ? G.ob1 : row == 2 ? G.oc0 : G.oc1);
    um = u0 + 2 * O.m * G.sa;
    u0 += side ? 2L * (O.N + O.ob) * G.sa : -2L * O.o * G.sa;
    ue0 = uc + 2 * (G.oa + (long)e0 * G.sa);
  }
  // (node 0 has no vector: the value before it is not used)
  __device__ __forceinline__ void load_rec(int d, int t) {
    rs[d] = xr[(long)t * XS];
    ra_[d] = qr[(long)t * QS];
    rb_[d] = qr[(long)t * QS + qx];
  }
  __device__ __forceinline__ void load_u(int d, int t) {   // the padding reads the boundary's
    const long tc = max(t, t1);
    un[d] = u0[tc * su];
    ue[d] = ue0[tc * su];
  }
  __device__ __forceinline__ void load(int d, const char* base, int t) {   // base: record t - d
    rw[d] = *reinterpret_cast<const double2*>(base + d * RB + fw);
    rr[d] = *reinterpret_cast<const double2*>(base + d * RB + fr);
    ri[d] = iwa[min((unsigned)(e0 + de * t), (unsigned)last)];
    if constexpr (MEM) load_rec(d, t);
  }
  __device__ __forceinline__ void first_loads() {
#pragma unroll
    for (int d = 0; d < D; d++) load(d, fb, d);
    wm = *reinterpret_cast<const double2*>(fb + fm);
  }
  // q = rho / d of an edge, component jr
  __device__ __forceinline__ double qval(double ra, double rb, double2 rd) const {
    const double s = __longlong_as_double(__double_as_longlong(rd.y) ^ ((unsigned long long)sg << 32));
    return fma(rb, s, ra * rd.x);
  }
  // both passes, on the records that first_loads() has under way
  __device__ __forceinline__ void run() {
    int t0 = 0;   // first node of the group
    // Software pipeline: a node's step runs its chain on operands prepared in
    // the step before, and prepares the next node's (coupling -B, right-hand
    // side g) and reads the LDS of the one after.
    double z = 0.0, q, sig, ra, rb;
    auto zrec = [&](double v) { return exact ? v : rec_val<T>(v); };
    // -B = -diag(l) - (v / d) v^T towards the node before, g of the node.  B all
    // but cancels on the node's gradient, which W^-1 amplifies in air: v.z is
    // summed first (one matrix instruction, rows all v) and then scaled, as an
    // explicit B would round every entry on its own.
    double nl1, vre, vim, g;
    auto couple = [&](int d) {
      nl1 = ncl * ri[d];
      vre = -vr * rr[d].x;
      vim = -vr * rr[d].y;
    };
    auto bsub = [&](double v, double g0) {   // g0 - B v
      const double sv = mma(vr, v, 0.0);
      return fma(vim, mswap(sv, sg), fma(vre, sv, fma(nl1, v, g0)));
    };
    auto fnext = [&](int d) {   // operands of the node after d (of group slot d)
      couple(d);
      if constexpr (MEM) {
        sig = rs[(d + 1) % D];
        ra = ra_[(d + 1) % D];
        rb = rb_[(d + 1) % D];
      }
      const double q1 = qval(ra, rb, rr[(d + 1) % D]);
      g = fma(vs, q - q1, sig);
      q = q1;
    };
    auto fread = [&](int d) {   // LDS of node d
      if constexpr (MEM) return;
      sig = xq[d * XS];
      ra = qa[d * QS];
      rb = qa[d * QS + qx];
    };
    auto fstep = [&](int d) {
      const double y = bsub(z, g);
      z = mma(rw[d].x, y, 0.0);
      z = mma(rw[d].y, mswap(y, sg), z);
      fnext(d);
      fread(d + 2);
      if constexpr (MEM) {
        rs[d] = (ScrRec<T>)z;
        xr[(long)(t0 + d) * XS] = rs[d];
      } else {
        xq[d * XS] = zrec(z);
      }
    };
    // the first node of a half (boundary or padding) only hands its inner
    // edge on
    q = MEM ? qval(ra_[0], rb_[0], rr[0]) : qval(qa[0], qa[qx], rr[0]);
    fread(1);
    fnext(0);
    fread(2);
    node_end();
    if (TT > D) {
      load(0, fb + D * RB, D);
      node_end();
#pragma unroll
      for (int d = 1; d < D; d++) {
        fstep(d);
        node_end();
        load(d, fb + D * RB, D + d);
        node_end();
      }
      for (t0 = D; t0 < TT - D; t0 += D) {
        xq += D * XS; qa += D * QS; fb += D * RB;
#pragma unroll
        for (int d = 0; d < D; d++) {
          fstep(d);
          node_end();
          load(d, fb + D * RB, t0 + D + d);
          node_end();
        }
      }
      // the last group's records stay for the back pass
      xq += D * XS; qa += D * QS; fb += D * RB;
      if constexpr (MEM) {
#pragma unroll
        for (int d = 0; d < D; d++) load_u(d, t0 + d);
      }
      fstep(0);
      node_end();
    }
#pragma unroll
    for (int d = 1; d < D; d++) {
      fstep(d);
      node_end();
    }

    // meeting node: x_m = S_m^-1 (g_m - B_m z_{m-1} - B_{m+1} z_{m+1})
    double x;
    {
      const double ql = MEM ? qval(ra_[D - 1], rb_[D - 1], rr[D - 1])
                            : qval(qa[(D - 1) * QS], qa[(D - 1) * QS + qx], rr[D - 1]);
      double y = bsub(z, vs * ql);
      y = (MEM ? (double)*xmr : *xm) + (y + mpeer(y));
      x = mma(wm.x, y, 0.0);
      x = mma(wm.y, mswap(y, sg), x);
      if constexpr (!MEM) *xm = x;
      else if (side == 0 && j < 2) *um = (T)((double)*um + x);
    }
    sig = zrec(z);
    // the along-line edge of a node follows one step later, off the chain
    double dx = 0.0, ere = 0.0, eim = 0.0, eq = 0.0;
    auto edge = [&](double* to, int t, int k) {   // q + v.dx / d; k: the node's slot of the ring
      const double sv = mma(vs, dx, 0.0), de_ = fma(eim, mswap(sv, sg), fma(ere, sv, eq));
      if constexpr (!MEM) *to = de_;
      else if (t >= t1 && t < TT && row == 0 && j < 2) ue0[t * su] = (T)((double)ue[k] + de_);
    };
    auto bedge = [&](int d) {   // operands of that edge
      ere = rr[d].x;
      eim = rr[d].y;
      eq = MEM ? qval(ra_[d], rb_[d], rr[d]) : qval(ra, rb, rr[d]);
    };
    // (from the slot before the group, as LDS offsets are not negative)
    double *xb = xq - XS, *qb = qa - QS;
    auto bread = [&](int d) {   // rho of node d's inner edge
      if constexpr (MEM) return;
      ra = qb[(d + 1) * QS];
      rb = qb[(d + 1) * QS + qx];
    };
    // to: where the pending edge goes
    auto bstep = [&](int d, double* to) {
      const double y = bsub(x, 0.0);
      double xp = mma(rw[d].x, y, MEM ? rs[d] : sig);
      xp = mma(rw[d].y, mswap(y, sg), xp);
      if constexpr (!MEM) sig = xb[d * XS];
      edge(to, t0 + d + 1, (d + 1) % D);
      bedge(d);
      bread(d - 1);
      couple((d + D - 1) % D);
      dx = x - xp;
      if constexpr (!MEM) xb[(d + 1) * XS] = xp;
      else if (t0 + d > t1 && j < 2) u0[(t0 + d) * su] = (T)((double)un[d] + xp);
      x = xp;
    };
    couple(D - 1);
    bread(D - 1);
    // no edge is pending at first: that write lands on the edge whose rho has
    // just been read and which the next step writes
    double* qe = qb + D * QS;
    for (; t0 > 0; t0 -= D) {
#pragma unroll
      for (int d = D - 1; d >= 0; d--) {
        bstep(d, d == D - 1 ? qe : qb + (d + 2) * QS);
        node_end();
        // a slot is reloaded one step after its node: that node's edge is
        // still pending until then
        if (d == D - 1) {
          load(0, fb, t0);
          if constexpr (MEM) load_u(0, t0);
        } else {
          load(d + 1, fb - D * RB, t0 - D + d + 1);
          if constexpr (MEM) load_u(d + 1, t0 - D + d + 1);
        }
        node_end();
      }
      qe = qb + QS;
      xb -= D * XS; qb -= D * QS; fb -= D * RB;
    }
#pragma unroll
    for (int d = D - 1; d >= 1; d--) {
      bstep(d, d == D - 1 ? qe : qb + (d + 2) * QS);
      node_end();
      if (d == D - 1) {
        load(0, fb, 0);
        if constexpr (MEM) load_u(0, 0);
      }
      node_end();
    }
    edge(qb + 2 * QS, 1, 1);
    // the first node's correction is zero: its inner edge alone
    bedge(0);
    dx = x;
    edge(qb + QS, 0, 0);
  }
};

// D = line_ring(N): nodes of factor records in flight per half.  MODE: how the
// residual records are built -- M_MARCH by marching along the lines, M_NODES
// node by node, M_SHORT the same for blocks of at most a node per thread,
// whose launch is a chain of memory latencies: it loads its first factor
// records and the u that it will update ahead of the residual phase.
enum { M_NODES = 0, M_MARCH = 1, M_SHORT = 2 };
template <typename T, int A, int LPB, int D, int MODE>
__global__ void __launch_bounds__(32 * LPB, 2) k_line_solve_m(LinePack<T> P) {
  constexpr int BT = 32 * LPB, SC = schunks<double>();
  extern __shared__ double2 mlds[];
  const LineJob<T>& J = P.job[blockIdx.y];
  const Level<T>& L = J.L;
  const int N = L.n[A];
  const int nl = J.nlo * J.nhi;
  const int l0 = (int)xcd_block(blockIdx.x, gridDim.x) * LPB;
  if (N < 2 || l0 >= nl) return;   // uniform over the block
  const HalfOrder O(N);
  const int T2 = 2 * O.T, TT = O.T;
  const int nle = min(LPB, nl - l0);   // lines of this block
  // edges: rho, then dE, in the order of the records; node vectors: sigma,
  // then z, then x, in the same order without each half's first (boundary or
  // padding) record.  Neighbouring threads of the first and last phase walk
  // along x, so x lines lie one after another and other lines side by side.
  double2* __restrict__ Q = mlds;
  double2* __restrict__ X = mlds + T2 * LPB;
  auto qslot = [&](int t2, int l) { return A == 0 ? l * T2 + t2 : t2 * LPB + l; };
  auto xslot = [&](int s, int l) { return 4 * (A == 0 ? l * (T2 - 1) + s : s * LPB + l); };
  // slot of the vector of record r (r = 0 and T have none)
  auto xrec = [&](int r) { return r - 1 - (r > TT ? 1 : 0); };

  // ---------------- the lane of the substitution ----------------
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const bool live = 2 * wave < nle;   // uniform over the wave
  HalfLane<T, A, D, A == 0 ? 1 : LPB, false> H;
  {
    // a wave without a second line runs its first line twice
    const int l = live ? min(2 * wave + H.second(), nle - 1) : 0, l2 = live ? 2 * wave : 0;
    int pb, pc;
    line_of<T, A>(J, l0 + l, pb, pc);
    H.init(L, O, pb, pc, J.fac, l0 + l2, l - l2, nl == 1, X + xslot(0, l), Q + qslot(0, l));
  }
  if constexpr (MODE == M_SHORT) H.first_loads();

  // ---------------- residual records ----------------
  auto put_rec = [&](int p, int l, const Ch<double>(&c)[SC]) {
    Q[qslot(O.edge(p), l)] = make_double2(rec_val<T>(c[4].v[0]), rec_val<T>(c[4].v[1]));
    if (p >= 1) {
      double2* x = X + xslot(xrec(O.node(p)), l);
#pragma unroll
      for (int i = 0; i < 4; i++) x[i] = make_double2(rec_val<T>(c[i].v[0]), rec_val<T>(c[i].v[1]));
    }
  };
  // padding and boundary records
  if (O.o > 0) {
    const double2 zz = make_double2(0.0, 0.0);
    for (int idx = threadIdx.x; idx < LPB * (O.o + 1); idx += BT) {
      const int l = idx % LPB, t = idx / LPB;
      if (t < O.o) Q[qslot(t, l)] = zz;
      if (t < O.ob) Q[qslot(TT + t, l)] = zz;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (t >= 1) X[xslot(t - 1, l) + i] = zz;
        if (t >= 1 && t <= O.ob) X[xslot(TT - 1 + t - 1, l) + i] = zz;
      }
    }
  }
  const int nn = nle * N;
  auto node_of = [&](int idx, int& l, int& p) {
    l = A == 0 ? idx / N : idx % nle;
    p = A == 0 ? idx % N : idx / nle;
  };
  if constexpr (MODE == M_MARCH) {
    // runs of consecutive nodes marching along the line, lines fastest
    constexpr int CH = BT / LPB;
    const int l = (int)threadIdx.x % LPB, ch = (int)threadIdx.x / LPB;
    const int run = (N + CH - 1) / CH;
    const int p0 = ch * run, p1 = min(N, p0 + run);
    if (l < nle && p0 < p1) {
      int pb, pc;
      line_of<T, A>(J, l0 + l, pb, pc);
      line_rhs_march<T, A, double>(J, pb, pc, p0, p1, [&](int p, const Ch<double>(&c)[SC]) { put_rec(p, l, c); });
    }
  } else if (MODE == M_SHORT && 4 * nn <= BT) {
    // few nodes: a thread per row (rows in the order of the records, rho last)
    for (int idx = threadIdx.x; idx < 5 * nn; idx += BT) {
      const int k = idx / nn;
      int l, p, pb, pc;
      node_of(idx - k * nn, l, p);
      line_of<T, A>(J, l0 + l, pb, pc);
      if (k == 4 || p >= 1) {
        const cxd r = node_rhs_row<T, A>(J, pb, pc, p, k);
        double2* to = k == 4 ? Q + qslot(O.edge(p), l) : X + xslot(xrec(O.node(p)), l) + k;
        *to = make_double2(rec_val<T>(r.re), rec_val<T>(r.im));
      }
    }
  } else {
    for (int idx = threadIdx.x; idx < nn; idx += BT) {
      int l, p, pb, pc;
      node_of(idx, l, p);
      line_of<T, A>(J, l0 + l, pb, pc);
      Ch<double> c[SC] = {};
      node_rhs_rec<T, A>(J, pb, pc, p, c);
      put_rec(p, l, c);
    }
  }
  typename cvec<T>::type* __restrict__ u = J.u;
  typename cvec<T>::type uv[5];
  long uo[5];
  auto u_of = [&](int idx, int& l, int& p) {
    constexpr int B = (A + 1) % 3, C = (A + 2) % 3;
    int pb, pc;
    node_of(idx, l, p);
    line_of<T, A>(J, l0 + l, pb, pc);
    const long o = (long)pb * L.es[B] + (long)pc * L.es[C] + (long)p * L.es[A];
    uo[0] = A * L.nc + o;
    uo[1] = B * L.nc + o - L.es[B];
    uo[2] = B * L.nc + o;
    uo[3] = C * L.nc + o - L.es[C];
    uo[4] = C * L.nc + o;
#pragma unroll
    for (int i = 0; i < 5; i++) uv[i] = u[i == 0 || p >= 1 ? uo[i] : uo[0]];
  };
  int ul = 0, up = 0;
  if (MODE == M_SHORT && (int)threadIdx.x < nn) u_of(threadIdx.x, ul, up);
  __syncthreads();

  // ---------------- substitution ----------------
  if (live) {
    if constexpr (MODE != M_SHORT) H.first_loads();
    H.run();
  }
  __syncthreads();

  // ---------------- u += corrections ----------------
  for (int idx = threadIdx.x; idx < nn; idx += BT) {
    if (MODE != M_SHORT) u_of(idx, ul, up);
    auto add = [&](int i, double2 d) { st<T>(u, uo[i], cxd((double)uv[i].x, (double)uv[i].y) + cxd(d.x, d.y)); };
    add(0, Q[qslot(O.edge(up), ul)]);
    if (up >= 1) {
      const double2* x = X + xslot(xrec(O.node(up)), ul);
#pragma unroll
      for (int i = 0; i < 4; i++) add(i + 1, x[i]);
    }
  }
}

// Long lines: the same substitution with the line records in memory (J.scr),
// in two launches: residual records; substitution and u += corrections.  The
// records of x lines lie line after line; those of y and z lines lie side by
// side, eight lines together.
//
// What bounds it: with many lines the traffic (both passes read the factor
// records, 352 bytes a node; the line records are written twice and read twice,
// 288 bytes in FP64; u), for few the chain.  One launch of a colour, four lanes
// per line half -> here: 64 x 64 lines of 1100 nodes, FP64, along z 950 -> 518
// us, along x 1199 -> 518; FP32 752 -> 315 and 1028 -> 391; 128 x 128 lines 1289
// -> 1290 and 1483 -> 1312, FP32 936 -> 821 and 1287 -> 1024; a single line 590
// -> 172.  All in one launch, with the records in FP64 and the update of u as a
// phase of its own, took 621, 534, 527 and 482 us (64 x 64); three waves per
// SIMD and four nodes in flight measured level.
template <typename T, int A>
struct LongLine {
  using R = ScrRec<T>;
  static constexpr int ST = A == 0 ? 1 : LONG_LPB;   // stride between a line's slots
  R *Q, *X;   // edges (2 values) and node vectors (8 values), as in k_line_solve_m
  __device__ __forceinline__ LongLine(const LineJob<T>& J, const HalfOrder& O, int line) {
    const long per = 20L * O.T;   // values of a line
    if constexpr (A == 0) {
      Q = J.scr + line * per;
      X = Q + 4 * O.T;
    } else {
      const int l = line % LONG_LPB;
      R* base = J.scr + (line - l) * per;
      Q = base + 2 * l;
      X = base + 4 * O.T * LONG_LPB + 8 * l;
    }
  }
  __device__ __forceinline__ typename cvec<R>::type* edge(int t) const {
    return reinterpret_cast<typename cvec<R>::type*>(Q + 2L * ST * t);
  }
  // vector of record r (r = 0 and T have none)
  __device__ __forceinline__ typename cvec<R>::type* vec(const HalfOrder& O, int r) const {
    return reinterpret_cast<typename cvec<R>::type*>(X + 8L * ST * (r - 1 - (r > O.T ? 1 : 0)));
  }
};

// residual records: a thread per run of nodes of a line, lines fastest
// (marching) along y and z, nodes fastest (runs of one) along x
template <typename T, int A>
__global__ void __launch_bounds__(256) k_line_long_rhs(LinePack<T> P, int run) {
  constexpr int SC = schunks<double>();
  const LineJob<T>& J = P.job[blockIdx.y];
  const int N = J.L.n[A];
  const long nl = (long)J.nlo * J.nhi, nr = (N + run - 1) / run;
  const long t = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  if (N < 2 || t >= nl * nr) return;
  const int line = (int)(A == 0 ? t / nr : t % nl), p0 = (int)(A == 0 ? t % nr : t / nl) * run, p1 = min(N, p0 + run);
  int pb, pc;
  line_of<T, A>(J, line, pb, pc);
  const HalfOrder O(N);
  const LongLine<T, A> R(J, O, line);
  auto put_rec = [&](int p, const Ch<double>(&c)[SC]) {
    st<T>(R.edge(O.edge(p)), 0, cxd(c[4].v[0], c[4].v[1]));
    if (p >= 1) {
#pragma unroll
      for (int i = 0; i < 4; i++) st<T>(R.vec(O, O.node(p)), i, cxd(c[i].v[0], c[i].v[1]));
    }
  };
  if constexpr (A == 0) {
    Ch<double> c[SC] = {};
    node_rhs_rec<T, A>(J, pb, pc, p0, c);
    put_rec(p0, c);
  } else {
    line_rhs_march<T, A, double>(J, pb, pc, p0, p1, put_rec);
  }
  if (p0 == 0) {   // padding and boundary records
    const cxd zz(0.0, 0.0);
    for (int q = 0; q <= O.o; q++) {
      if (q < O.o) st<T>(R.edge(q), 0, zz);
      if (q < O.ob) st<T>(R.edge(O.T + q), 0, zz);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        if (q >= 1) st<T>(R.vec(O, q), i, zz);
        if (q >= 1 && q <= O.ob) st<T>(R.vec(O, O.T + q), i, zz);
      }
    }
  }
}

template <typename T, int A>
__global__ void __launch_bounds__(32 * LONG_LPB, 2) k_line_long_solve(LinePack<T> P) {
  const LineJob<T>& J = P.job[blockIdx.y];
  const int N = J.L.n[A], nl = J.nlo * J.nhi;
  const int l2 = (int)xcd_block(blockIdx.x, gridDim.x) * LONG_LPB + 2 * __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  if (N < 2 || l2 >= nl) return;   // uniform over the wave
  const HalfOrder O(N);
  HalfLane<T, A, LONG_RING, LongLine<T, A>::ST, true> H;
  // a wave without a second line runs its first line twice
  const int line = min(l2 + H.second(), nl - 1);
  int pb, pc;
  line_of<T, A>(J, line, pb, pc);
  const LongLine<T, A> R(J, O, line);
  H.init(J.L, O, pb, pc, J.fac, l2, line - l2, false, nullptr, nullptr);
  H.init_mem(J.L, O, pb, pc, R.X, R.Q, J.u);
  H.first_loads();
  H.run();
}

// ---------------------------------------------------------------------------
// host side
// ---------------------------------------------------------------------------
void line_colour_counts(const int* n, int a, int colour, int* nlo, int* nhi) {
  const int b = (a + 1) % 3, c = (a + 2) % 3;
  const int cb = colour & 1, cc = (colour >> 1) & 1;
  auto cnt = [](int m, int par) { const int s = par ? 1 : 2; return m - 1 >= s ? (m - 1 - s) / 2 + 1 : 0; };
  const int nbv = cnt(n[b], cb), ncv = cnt(n[c], cc);
  if (b < c) { *nlo = nbv; *nhi = ncv; } else { *nlo = ncv; *nhi = nbv; }
}

// Lines of more than 256 nodes have their records in LDS two lines at a time,
// at most six lines (three waves) a CU: with many lines their
// residual and update phases no longer fill the chip.  Per launch of a colour in
// LDS and in memory, along z: 64 x 64 lines (1024 a colour) of 512 nodes FP64
// 165 and 209 us, FP32 127 and 132; of 1024 nodes 589 and 439, 512 and 275;
// 96 x 96 of 288 nodes 232 and 278, 180 and 166; of 512 nodes 513 and 501, 423
// and 312; 128 x 128 of 288 nodes 378 and 363, 300 and 216.  Along x, where the
// LDS form loads and stores u along the lines, 128 x 128 of 512 nodes 530 and
// 649, 494 and 475; 96 x 96 of 1024 nodes 1146 and 1019, 1131 and 829.
LineRoute line_route(int esize, int axis, int njobs, const int* cells, const long* lines, bool one_lane) {
  if (one_lane || njobs < 1) return LINE_ROUTE_ONE_LANE;
  const int N = cells[0];
  double nodes = 0;
  for (int j = 0; j < njobs; j++) {
    if (cells[j] != N || line_across(esize, axis, N, lines[j])) return LINE_ROUTE_ONE_LANE;
    nodes += (double)N * (double)lines[j];
  }
  const bool many = N > 256 && nodes > 0.9e6 && (axis != 0 || N > 512);
  return line_m_fits(N) && !many ? LINE_ROUTE_MATRIX : LINE_ROUTE_MATRIX_MEM;
}

static int g_line_kernel = 0;

LineRoute line_route_now(int esize, int axis, int njobs, const int* cells, const long* lines) {
  return line_route(esize, axis, njobs, cells, lines, g_line_kernel == 1);
}

int set_line_kernel(int mode) {
  if (mode < 0 || mode > 4) return -1;
  const int prev = g_line_kernel;
  g_line_kernel = mode;
  return prev;
}

// The autotuner's table: the substitution choice measured fastest for a
// launch shape.  Process-wide (every solver on the device shares it) and
// consulted only in the automatic mode (set_line_kernel(0)).
struct TunedLine {
  int choice;
  double us_choice, us_rule;
};
static std::map<LineShape, TunedLine> g_tuned;
static std::mutex g_tuned_mu;

template <typename T>
LineShape line_shape(const LinePack<T>& P, int axis) {
  LineShape k{(int)sizeof(T), axis, 0, 0, P.njobs};
  for (int j = 0; j < P.njobs; j++) {
    k.n = std::max(k.n, P.job[j].L.n[axis]);
    k.nl = std::max(k.nl, (long)P.job[j].nlo * P.job[j].nhi);
  }
  return k;
}

static int tuned_choice(const LineShape& k) {
  std::lock_guard<std::mutex> g(g_tuned_mu);
  const auto it = g_tuned.find(k);
  return it == g_tuned.end() ? LINE_RULE : it->second.choice;
}

void set_line_choice(const LineShape& k, int choice, double us_choice, double us_rule) {
  std::lock_guard<std::mutex> g(g_tuned_mu);
  g_tuned[k] = TunedLine{choice, us_choice, us_rule};
}

bool has_line_choice(const LineShape& k) {
  std::lock_guard<std::mutex> g(g_tuned_mu);
  return g_tuned.count(k) != 0;
}

void clear_line_choices() {
  std::lock_guard<std::mutex> g(g_tuned_mu);
  g_tuned.clear();
}

int line_choices(int* out, double* us, int maxn) {
  std::lock_guard<std::mutex> g(g_tuned_mu);
  int i = 0;
  for (const auto& kv : g_tuned) {
    if (i < maxn) {
      const LineShape& k = kv.first;
      const int row[7] = {k.esize, k.axis, k.n, (int)std::min<long>(k.nl, INT32_MAX), k.njobs, kv.second.choice, 0};
      for (int c = 0; c < 6; c++) out[6 * i + c] = row[c];
      us[2 * i] = kv.second.us_choice;
      us[2 * i + 1] = kv.second.us_rule;
    }
    i++;
  }
  return i;
}

bool line_needs_scratch(int esize, const int* n, int axis) {
  {
    std::lock_guard<std::mutex> g(g_tuned_mu);
    for (const auto& kv : g_tuned)
      if (kv.second.choice == LINE_ONE_LANE) return true;
  }
  for (int colour = 0; colour < 4; colour++) {
    int nlo, nhi, cells[LINE_PACK_MAX];
    long lines[LINE_PACK_MAX];
    line_colour_counts(n, axis, colour, &nlo, &nhi);
    std::fill(cells, cells + LINE_PACK_MAX, n[axis]);
    std::fill(lines, lines + LINE_PACK_MAX, (long)nlo * nhi);
    if (line_route_now(esize, axis, LINE_PACK_MAX, cells, lines) != LINE_ROUTE_MATRIX) return true;
  }
  return false;
}

static size_t chunks_of(int values, size_t esize) {
  const size_t v = 16 / esize;
  return (values + v - 1) / v;
}

size_t line_factor_bytes(const int* n, int a, int colour, size_t esize) {
  int nlo, nhi;
  line_colour_counts(n, a, colour, &nlo, &nhi);
  return (size_t)nlo * nhi * (size_t)HalfOrder(n[a]).records() * chunks_of(FREC, esize) * 16;
}

size_t line_scratch_bytes(const int* n, int a, int colour, size_t esize) {
  int nlo, nhi;
  line_colour_counts(n, a, colour, &nlo, &nhi);
  const size_t one_lane = (size_t)nlo * nhi * (size_t)n[a] * chunks_of(SREC, esize) * 16;
  if (n[a] <= 256) return one_lane;   // always in the LDS
  const size_t blocks = ((size_t)nlo * nhi + LONG_LPB - 1) / LONG_LPB;
  return std::max(one_lane, blocks * LONG_LPB * 20 * HalfOrder(n[a]).T * esize);
}

// A launch; when timing is on, its events are recorded by the dispatch itself
// (hipExtLaunchKernelGGL), so their elapsed time is the kernel's alone.
// bytes = {compulsory, layout} of the launch
struct Bytes {
  double comp, layout;
};

template <typename K, typename... Args>
static void launch_timed(K kernel, dim3 g, dim3 b, hipStream_t s, int cls, Bytes bytes, Args... args) {
  hipEvent_t e0, e1;
  timing::kernel_events(cls, bytes.comp, &e0, &e1, bytes.layout);
  if (e0) hipExtLaunchKernelGGL(kernel, g, b, 0, s, e0, e1, 0, args...);
  else hipLaunchKernelGGL(kernel, g, b, 0, s, args...);
}

// the same with dynamic LDS
template <typename K, typename... Args>
static void launch_lds(K kernel, dim3 g, dim3 b, size_t lds, hipStream_t s, int cls, Bytes bytes, Args... args) {
  if (lds > 64 * 1024 && allow_lds(reinterpret_cast<const void*>(kernel)) != hipSuccess)
    throw std::runtime_error("a line kernel was refused its LDS");
  hipEvent_t e0, e1;
  timing::kernel_events(cls, bytes.comp, &e0, &e1, bytes.layout);
  if (e0) hipExtLaunchKernelGGL(kernel, g, b, lds, s, e0, e1, 0, args...);
  else hipLaunchKernelGGL(kernel, g, b, lds, s, args...);
}

// the matrix-core substitution: lines per block by what the LDS holds, the
// ring by the length of a half
template <typename T, int A>
static void launch_line_m_axis(const LinePack<T>& P, bool mem, int maxl, int maxna, hipStream_t s, Bytes by) {
  const bool by_node = g_line_kernel == 3;   // residual records node by node (for tests)
  if (mem) {
    const int run = A == 0 || maxl < 64 || by_node ? 1 : 8;
    auto blocks = [&](long n, int per) { return dim3((unsigned)((n + per - 1) / per), P.njobs); };
    launch_timed(k_line_long_rhs<T, A>, blocks((long)maxl * ((maxna + run - 1) / run), 256), dim3(256), s, timing::LINE_RHS,
                 Bytes{0.0, 0.0}, P, run);
    launch_timed(k_line_long_solve<T, A>, blocks(maxl, LONG_LPB), dim3(32 * LONG_LPB), s, timing::LINE, by, P);
    return;
  }
  const int lpb = line_m_lpb(maxna), D = line_ring(maxna);
  const dim3 g((unsigned)((maxl + lpb - 1) / lpb), P.njobs), b(32 * lpb);
  const size_t lds = (size_t)lpb * line_m_bytes(maxna);
  auto go = [&](auto kernel) { launch_lds(kernel, g, b, lds, s, timing::LINE, by, P); };
  // Along y and z, lines of 64 nodes and more are marched by runs of N / 32
  // nodes (128 nodes, per launch of a colour: 120 -> 107 us FP64 with one
  // right-hand side, 252 -> 224 FP32 with three); a launch with few lines would
  // leave most threads of its block without a run (one line of 96 nodes: 23 us
  // marched, 16 node by node).
  if constexpr (A != 0) {
    if (D == 8 && maxna >= 64 && maxl > 4 && !by_node) {
      if (lpb == 2) go(k_line_solve_m<T, A, 2, 8, M_MARCH>);
      else go(k_line_solve_m<T, A, 8, 8, M_MARCH>);
      return;
    }
  }
  if (lpb == 2) {
    go(k_line_solve_m<T, A, 2, 8, M_NODES>);   // (more than 256 nodes: groups of eight)
  } else if (maxna <= 32 && D < 8 && (long)g.x * P.njobs <= 256 && !by_node) {
    // at most a block per CU: the look-ahead costs FP32 launches along y and z
    // their third wave per SIMD (163 -> 197 to 220 registers; 192 x 192 lines of 4
    // nodes 11.6 -> 13.1 us, of 12 22.2 -> 25.6; FP64 and x keep two, 14.9 -> 13.1).
    // Within the limit, node by node -> ahead: 64 x 64 lines of 4 nodes FP64
    // 5.9 -> 5.3 us, FP32 6.3 -> 5.5, of 6 6.7 -> 6.1 and 6.9 -> 6.2, of 8 6.4 ->
    // 6.7 and 6.6 -> 6.8, of 12 to 28 within 3%
    if (D == 4) go(k_line_solve_m<T, A, 8, 4, M_SHORT>);
    else go(k_line_solve_m<T, A, 8, 2, M_SHORT>);
  } else {
    if (D == 8) go(k_line_solve_m<T, A, 8, 8, M_NODES>);
    else if (D == 4) go(k_line_solve_m<T, A, 8, 4, M_NODES>);
    else go(k_line_solve_m<T, A, 8, 2, M_NODES>);
  }
}
template <typename T>
static void launch_line_m(const LinePack<T>& P, int axis, bool mem, int maxl, int maxna, hipStream_t s, Bytes by) {
  if (axis == 0) launch_line_m_axis<T, 0>(P, mem, maxl, maxna, s, by);
  else if (axis == 1) launch_line_m_axis<T, 1>(P, mem, maxl, maxna, s, by);
  else launch_line_m_axis<T, 2>(P, mem, maxl, maxna, s, by);
}

template <typename T>
static void launch_pack(const LinePack<T>& P, int axis, bool factor, hipStream_t s, int choice = LINE_RULE) {
  int maxl = 0;
  long maxnodes = 0;
  double rhs_bytes = 0, solve_bytes = 0, rec_bytes = 0, scr_bytes = 0, comp = 0;
  const double es = sizeof(typename cvec<T>::type), cs = sizeof(T);
  for (int j = 0; j < P.njobs; j++) {
    // compulsory bytes of one colour: a quarter of a full sweep's
    // 3 Ne s + 3 Nc c (u read and written, f read, sbar read)
    const Level<T>& L = P.job[j].L;
    comp += 0.25 * (3.0 * 3.0 * (double)L.nc * es + 3.0 * (double)L.n[0] * L.n[1] * L.n[2] * cs);
    const long nl = (long)P.job[j].nlo * P.job[j].nhi;
    const int na = P.job[j].L.n[axis];
    if (nl > maxl) maxl = (int)nl;
    if (nl * na > maxnodes) maxnodes = nl * na;
    const double rows = (double)nl * (5.0 * na - 4.0);
    // right-hand sides: the colour's rows read f and sigma-bar once, u is
    // read once over the level
    rhs_bytes += rows * (es + cs) + 3.0 * (double)P.job[j].L.nc * es;
    // substitution: factors read by both passes, the rows of u read and written
    solve_bytes += (double)nl * na * 2.0 * FREC * sizeof(FacRec<T>) + rows * 2.0 * es;
    // records in memory: written, read by both passes, z written by the first
    rec_bytes += (double)nl * na * SREC * sizeof(ScrRec<T>);
    scr_bytes += (double)nl * na * (2.0 * SREC + 8.0) * sizeof(ScrRec<T>);
  }
  if (maxl == 0 || P.njobs == 0) return;
  int maxna = 0, cells[LINE_PACK_MAX];
  long lines[LINE_PACK_MAX];
  for (int j = 0; j < P.njobs; j++) {
    cells[j] = P.job[j].L.n[axis];
    lines[j] = (long)P.job[j].nlo * P.job[j].nhi;
    maxna = std::max(maxna, cells[j]);
  }
  if (factor) {
    const dim3 g((maxl + 63) / 64, P.njobs), b(64);
    timing::Scope ts(timing::OTHER, s, 0);
    bool by_line = true;
    for (int j = 0; j < P.njobs; j++) by_line = by_line && !line_across(sizeof(T), axis, cells[j], lines[j]);
    auto go = [&](auto kernel) { hipLaunchKernelGGL(kernel, g, b, 0, s, P); };
    if (axis == 0) by_line ? go(k_line_factor<T, 0, true>) : go(k_line_factor<T, 0, false>);
    else if (axis == 1) by_line ? go(k_line_factor<T, 1, true>) : go(k_line_factor<T, 1, false>);
    else by_line ? go(k_line_factor<T, 2, true>) : go(k_line_factor<T, 2, false>);
    return;
  }
  if (choice == LINE_RULE && g_line_kernel == 0) choice = tuned_choice(line_shape(P, axis));
  const bool one_lane = choice == LINE_ONE_LANE || (choice == LINE_RULE && g_line_kernel == 1);
  bool scr = true;
  for (int j = 0; j < P.njobs; j++) scr = scr && P.job[j].scr;
  const LineRoute route = line_route(sizeof(T), axis, P.njobs, cells, lines, one_lane && scr);
  if (route != LINE_ROUTE_MATRIX && !scr) throw std::runtime_error("a line sweep without its records in memory");
  if (route != LINE_ROUTE_ONE_LANE) {
    const bool mem = route == LINE_ROUTE_MATRIX_MEM;
    launch_line_m<T>(P, axis, mem, maxl, maxna, s, Bytes{comp, rhs_bytes + solve_bytes + (mem ? rec_bytes + scr_bytes : 0.0)});
    return;
  }
  rhs_bytes += rec_bytes;
  solve_bytes += scr_bytes;
  if (axis == 0) {
    int maxn = 0;
    for (int j = 0; j < P.njobs; j++) maxn = std::max(maxn, P.job[j].L.n[0]);
    const int nlb = (maxl + XT - 1) / XT, npb = (maxn + XT - 1) / XT;
    const dim3 g((unsigned)(nlb * npb), P.njobs), b(XT * XT);
    launch_timed(k_line_rhs_x<T>, g, b, s, timing::LINE_RHS, Bytes{0.0, rhs_bytes}, P, nlb);
  } else if (maxna >= 64) {
    // lines of 64 nodes and more march
    constexpr int run = 8;
    const long nth = (long)maxl * ((maxna + run - 1) / run);
    const dim3 g((unsigned)((nth + 255) / 256), P.njobs), b(256);
    if (axis == 1) launch_timed(k_line_rhs_run<T, 1>, g, b, s, timing::LINE_RHS, Bytes{0.0, rhs_bytes}, P, run);
    else launch_timed(k_line_rhs_run<T, 2>, g, b, s, timing::LINE_RHS, Bytes{0.0, rhs_bytes}, P, run);
  } else {
    const dim3 g((unsigned)((maxnodes + 255) / 256), P.njobs), b(256);
    if (axis == 1) launch_timed(k_line_rhs<T, 1>, g, b, s, timing::LINE_RHS, Bytes{0.0, rhs_bytes}, P);
    else launch_timed(k_line_rhs<T, 2>, g, b, s, timing::LINE_RHS, Bytes{0.0, rhs_bytes}, P);
  }
  {
    const dim3 g((maxl + 63) / 64, P.njobs), b(128);
    if (axis == 0) {
      // the substitution's algorithmic bytes include the update of u, which
      // the second kernel makes (counted once, with the substitution)
      int maxn = 0;
      for (int j = 0; j < P.njobs; j++) maxn = std::max(maxn, P.job[j].L.n[0]);
      const int nlb = (maxl + XT - 1) / XT, npb = (maxn + XT - 1) / XT;
      launch_timed(k_line_solve<T, 0>, g, b, s, timing::LINE, Bytes{comp, solve_bytes}, P);
      launch_timed(k_line_solve_x_apply<T>, dim3((unsigned)(nlb * npb), P.njobs), dim3(XT * XT), s, timing::LINE,
                   Bytes{0.0, 0.0}, P, nlb);
    } else if (axis == 1) launch_timed(k_line_solve<T, 1>, g, b, s, timing::LINE, Bytes{comp, solve_bytes}, P);
    else launch_timed(k_line_solve<T, 2>, g, b, s, timing::LINE, Bytes{comp, solve_bytes}, P);
  }
}

template <typename T>
void launch_line_factor(const LinePack<T>& P, int axis, hipStream_t s) { launch_pack<T>(P, axis, true, s); }
template <typename T>
void launch_line_solve(const LinePack<T>& P, int axis, hipStream_t s) { launch_pack<T>(P, axis, false, s); }
template <typename T>
void launch_line_solve_as(const LinePack<T>& P, int axis, int choice, hipStream_t s) {
  launch_pack<T>(P, axis, false, s, choice);
}
template void launch_line_factor<double>(const LinePack<double>&, int, hipStream_t);
template void launch_line_factor<float>(const LinePack<float>&, int, hipStream_t);
template void launch_line_solve<double>(const LinePack<double>&, int, hipStream_t);
template void launch_line_solve<float>(const LinePack<float>&, int, hipStream_t);
template void launch_line_solve_as<double>(const LinePack<double>&, int, int, hipStream_t);
template void launch_line_solve_as<float>(const LinePack<float>&, int, int, hipStream_t);
template LineShape line_shape<double>(const LinePack<double>&, int);
template LineShape line_shape<float>(const LinePack<float>&, int);

}  // namespace emmi
