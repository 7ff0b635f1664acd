// tensor.hip -- spherical tensor operators (rank > 0) and the scalar-tensor
// commutator [G, T] with its BCH series on the device: allocate_tensor and
// tensor_elem (basic_IMSRG.f90:644-907, 1504-1641), TS_commutator_111 ..
// _222_ph (TS_commutators.f90:10-1849), the tensor Pandya transform
// (calculate_single_pandya, cross_coupled.f90:1416-1634) and BCH_TENSOR
// (IMSRG_MAGNUS.f90:389-465).
//
// Layout.  A tensor operator of rank R (doubled) and parity change dpar is one
// FP64 buffer [E0 | pad][F: nsp x nsp row-major][V]: F holds f_tensor_elem(a, b)
// for every orbit pair (the (hole, particle) entries are the herm-phased
// (particle, hole) ones), V holds, per tensor block (J1 <= J2, Tz, P1) in the
// reference's order, the FULL n1 x n2 row-major matrix between the scalar
// channels (J1, Tz, P1) and (J2, Tz, P1 + dpar/2): rows and columns are the
// channels' pair lists [pp | ph | hh] of the scalar layout, so the nine
// reference sub-blocks tgam(1..9) tile it and every 222_pp_hh product is a
// plain GEMM against the scalar full channel blocks of G.
//
// Kernels.  Lists of weights for 122 and 212, gathers by classes of orbit
// quadruples for the tensor Pandya matrices and the ph recoupling, one wavefront
// per output for the other one-body terms, FP64 MFMA for the products (the
// pp/hh ladders and the two Pandya products of each cross-coupled block).  The
// ph recoupling is a gather: every stored output element sums, over the
// sixteen index patterns through which TS_commutator_222_ph scatters into it
// and over the cross-coupled (J3, J4) blocks, the 9j-weighted product entries
// that pass the reference's |W| > 1e-6 test.
#include <hip/hip_runtime.h>

#include <atomic>
#include <cfloat>
#include <cmath>
#include <cstring>
#include <utility>

#include "devfun.hpp"
#include "engine_internal.hpp"

using namespace imsrg;

namespace {

// ---------------------------------------------------------------- device view
struct DevTensor {
  int rank, dpar, nblk, ncc, nJ, nh, hx, nhole, npart;
  long long nelem;              // tensor V elements
  const int *holes, *parts;
  const int *J1, *J2, *q1, *q2, *n1, *n2;
  const long long *off;           // per tensor block: V offset
  const int *bidx;                // [((J1/2)*nJ + J2/2)*6 + (Tz+1)*2 + P1] -> block (J1 <= J2) or -1
  const int *ccol;                // [(scalar Pandya block * nsp + p) * nsp + h] -> column of (p,h)
  const double *x6, *s6;
  const double *n9;               // 9j table of the ph recoupling and the tensor Pandya (k_fill9j)
  int nd;                         // rank/2 + 1: J4 - J3 and J2 - J1 steps the table holds
  // the ph recoupling's orbit quadruples x0|x1<<8|x2<<16|x3<<24 (x0 <= x1,
  // x2 <= x3, with stored outputs), class by class (the (l,j,tz) groups of the
  // four orbits), and its work items (first quadruple, 1..kPhQ quadruples of
  // one class)
  const unsigned *quads;
  const struct PhChunkT *qchunk;
  int nqchunk, nqpad;             // items; rounded up to whole runs of 64 on 8 XCDs
  // [(p * nsp + h) * nJ + J/2]: row of the ordered pair in its Pandya block and
  // the row's place in group order, or -1
  const int *crow, *cpos;
  const int *prow;                // [(a * nsp + b) * nJ + J/2], a <= b: row of the pair in its channel, or -1
  const struct OutBlk *oblk;      // [(J1/2 * nd + (J2-J1)/2) * 6 + (Tz+1)*2 + P1]: tensor blocks
  const struct CcBlk *cblk;       // [((Tz + 2*P) * nJ + J3/2) * nd + (J4-J3)/2]: cross-coupled product blocks
  // the orbits i the tensor's one-body part couples to orbit x (same tz, l + dpar/2
  // of the same parity, triangle (ji, jx, R)): part[pstart[x] .. pstart[x+1]),
  // each i | ji << 8
  const int *pstart, *part;
  // group order of the rows inside each scalar Pandya block, by the (l,j,tz)
  // groups of their two orbits (zero rows last): entry i is the block-local row
  // in place i.  CCR, Wx and Wy keep their columns so: the entries that
  // quadruples of one class read then share cache lines
  const int *rperm;
  long long f_off, v_off;
};

// a cross-coupled product block: offset of W (negative: none) and its row length
struct alignas(16) CcBlk {
  long long wo;
  int rl4, pad;
};

// a tensor block: offset in V (negative: none) and its columns
struct alignas(16) OutBlk {
  long long off;
  int n2, pad;
};

// up to kPhQ quadruples of one class: the first's position, the four orbits'
// 2j a byte each, their parities of l (bits 0-3) and tz > 0 (bits 4-7), count
struct alignas(16) PhChunkT {
  unsigned first, jv, lt;
  int n;
};

// A product C (M x N, row-major, ldc) = sum of nseg segments alpha * A * B
// with A(m,k) = X[asrc][a_off + m*a_rs + k*a_cs], B(k,n) = X[bsrc][b_off + k*b_rs + n*b_cs];
// with nseg2 a second one, into C2, from the segments after them.
struct TSeg {
  long long a_off, b_off;
  int K, a_rs, a_cs, b_rs, b_cs, asrc, bsrc;
  double alpha;
};
struct TProb {
  int M, N, ldc, nseg, nseg2, c;
  long long c_off;
  TSeg seg[4];
};
struct TGemm {
  const double *x[4];  // operands
  double *c[2];        // C by the problem's c; C2 is c[1]
  double *res;         // += C - C2 (null: not)
};

// {J1 J2 R; j4 j5 j6} with J1, J2 integer (doubled), j4 up to jmax + R, j5, j6 of the basis
__device__ __forceinline__ double tx6(const DevTensor &T, int J1, int J2, int j4, int j5, int j6) {
  return T.x6[((((size_t)(J1 >> 1) * T.nJ + (J2 >> 1)) * T.hx + (j4 >> 1)) * T.nh + (j5 >> 1)) * T.nh + (j6 >> 1)];
}
// {c d J2; b x J4}: c, d, b of the basis, x up to jmax + R
__device__ __forceinline__ double ts6(const DevTensor &T, int c, int d, int J2, int b, int x, int J4) {
  return T.s6[(((((size_t)(c >> 1) * T.nh + (d >> 1)) * T.nJ + (J2 >> 1)) * T.nh + (b >> 1)) * T.hx + (x >> 1)) *
                  T.nJ + (J4 >> 1)];
}
// ninej (basic_IMSRG.f90:4290-4308): {a b J1; c d J2; J3 J4 R} from three 6j per x
__device__ inline double t9j(const DevTensor &T, int a, int b, int J1, int c, int d, int J2, int J3, int J4) {
  const int R = T.rank;
  const int xmin = max(max(abs(J2 - b), abs(a - R)), abs(J4 - c));
  const int xmax = min(min(J2 + b, a + R), J4 + c);
  double sm = 0.0;
  for (int x = xmin; x <= xmax; x += 2)
    sm -= (x + 1.0) * tx6(T, J1, J2, x, a, b) * ts6(T, c, d, J2, b, x, J4) * tx6(T, J3, J4, x, a, c);
  return sm;
}

// The 9j symbols of the ph recoupling and the tensor Pandya transform, {j1 j2 J3;
// j3 j4 J4; J1 J2 R} with J3 <= J4 <= J3 + R and J1 <= J2 <= J1 + R, tabulated
// once per tensor space: index (((((((k1*nh + k2)*nh + k3)*nh + k4)*nJ + J3/2)*nd + (J4-J3)/2)*nJ + J1/2)*nd + (J2-J1)/2
// zeros past the table: a lane's pair of outputs may start up to a wavefront's
// width of pairs past its row
constexpr int kN9Pad = 256;
__global__ void k_fill9j(DevTensor T, double *__restrict__ n9, long long n) {
  const long long e = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= n) return;
  long long u = e;
  const int d2 = (int)(u % T.nd); u /= T.nd;
  const int J1 = 2 * (int)(u % T.nJ); u /= T.nJ;
  const int d4 = (int)(u % T.nd); u /= T.nd;
  const int J3 = 2 * (int)(u % T.nJ); u /= T.nJ;
  const int k4 = (int)(u % T.nh); u /= T.nh;
  const int k3 = (int)(u % T.nh); u /= T.nh;
  const int k2 = (int)(u % T.nh); u /= T.nh;
  const int k1 = (int)u;
  const int J4 = J3 + 2 * d4, J2 = J1 + 2 * d2, JM2 = 2 * (T.nJ - 1);
  n9[e] = (J4 <= JM2 && J2 <= JM2) ? t9j(T, 2 * k1 + 1, 2 * k2 + 1, J3, 2 * k3 + 1, 2 * k4 + 1, J4, J1, J2) : 0.0;
}

// tensor_elem (basic_IMSRG.f90:1504-1641): position in V of T^{J1x J2x}_{ax bx,
// cx dx} and the factor applied to the stored value (switch phase, exchange
// phase, sqrt 2), with every table read made (indices in range whatever the
// tests say) and no early return: an element the tensor does not hold gets
// position 0 and factor 0.  For batches whose loads should be in flight
// together.  chan: the caller's test that the pairs' parities (with the
// tensor's) and Tz match; j*x the orbits' 2j.
__device__ inline long long t_pos_all(const DevLayout &L, const DevTensor &T, int herm, int ax, int bx, int cx, int dx,
                                      int jax, int jbx, int jcx, int jdx, int J1x, int J2x, bool chan, double &pre) {
  const bool sw = J1x > J2x;
  const int a = sw ? cx : ax, b = sw ? dx : bx, c = sw ? ax : cx, d = sw ? bx : dx;
  const int ja = sw ? jcx : jax, jb = sw ? jdx : jbx, jc = sw ? jax : jcx, jd = sw ? jbx : jdx;
  const int J1 = sw ? J2x : J1x, J2 = sw ? J1x : J2x;
  const int P = (L.l[a] + L.l[b]) & 1, T2 = L.tz[a] + L.tz[b];
  const int q = T.bidx[((J1 >> 1) * T.nJ + (J2 >> 1)) * 6 + (T2 / 2 + 1) * 2 + P];
  const int r = dpos(L, J1, min(a, b), max(a, b)), s = dpos(L, J2, min(c, d), max(c, d));
  const int qc = max(q, 0);
  const long long o = T.off[qc];
  const int n2 = T.n2[qc];
  double f = sw ? (double)(sgnp((J2 - J1) >> 1) * herm) : 1.0;
  f *= a > b ? (double)sgnp(1 + ((ja + jb - J1) >> 1)) : (a == b ? M_SQRT2 : 1.0);
  f *= c > d ? (double)sgnp(1 + ((jc + jd - J2) >> 1)) : (c == d ? M_SQRT2 : 1.0);
  const bool ok = chan && dtri(J1, J2, T.rank) && dtri(ja, jb, J1) && dtri(jc, jd, J2) && q >= 0 && (r | s) >= 0;
  pre = ok ? f : 0.0;
  return ok ? o + (long long)r * n2 + s : 0;
}
// ---------------------------------------------------------------- one-body terms
// TS_commutator_111 (TS_commutators.f90:10-55; overwrites the one-body part), _121
// (:58-303), _211 (:307-552) and _221 (:809-1067; these add to it).  LF: the
// scalar operator's one-body matrix, RF the tensor's.  One workgroup per
// upper output (p,q): (hole, hole), (particle, particle), (particle, hole).
// 111 is the matrix commutator, each class in the stored entries the reference
// reads; the other three, for outputs that the tensor's selection rules allow,
// add to the upper entry, and the lower one becomes herm (-1)^((jp-jq)/2) times
// it (diagonal included, after each term), as each reference routine leaves it;
// (hole, particle) entries are derived.  The terms, flattened over the intermediate
// orbits and the first angular momentum with the 2 rank + 1 second ones the
// tensor couples to it, are spread over the threads.
//
// What bounds it: the latency of a term's dependent lookups.  A wavefront per
// output with a lane per intermediate orbit, a launch per term, took 0.07 +
// 0.40 ms at 90 orbits, rank 4, 20 + 89 us at 30 orbits, rank 2; this kernel
// 0.12 ms and 11 us.
constexpr int kTfThreads = 512;
enum { kTf111 = 1, kTf121 = 2, kTf221 = 4, kTf211 = 8 };
__global__ __launch_bounds__(kTfThreads) void k_t_f(DevLayout L, DevTensor T, int terms, const double *__restrict__ LF,
                                                    const double *__restrict__ RF, const double *__restrict__ RV,
                                                    const double *__restrict__ gcc, const double *__restrict__ W1,
                                                    const double *__restrict__ W2, double *__restrict__ F, int hL,
                                                    int hR, int hres) {
  __shared__ double sh[5][kTfThreads / 64];
  const int tid = threadIdx.x, p = L.ob_p[blockIdx.x], q = L.ob_q[blockIdx.x], n = L.nsp, R = T.rank;
  const int jp = L.jj[p], jq = L.jj[q], lp = L.l[p], lq = L.l[q];
  const bool allowed = (lq & 1) == ((lp + (T.dpar >> 1)) & 1) && L.tz[q] == L.tz[p] && dtri(jq, jp, R);
  const int cp = L.con[p], cq = L.con[q];
  if (!(terms & kTf111) && !allowed) return;
  // 111's upper entry, and the lower one where 111 alone sets it; 121, 221, 211
  double up = 0.0, dn = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  if (terms & kTf111) {
    const double ph = sgnp((jp - jq) >> 1);
    auto lf = [&](int a, int b) { return LF[(size_t)a * n + b]; };
    auto rf = [&](int a, int b) { return RF[(size_t)a * n + b]; };
    for (int k = tid; k < n; k += kTfThreads) {
      const bool hole = L.con[k] != 0;
      if (cp != cq) {
        up += lf(p, k) * rf(k, q) - rf(p, k) * lf(k, q);
      } else if (cp) {
        // hh: Lhh Rhh + hL Lph^T Rph - (hL hR ph) (Lhh Rhh)^T - (hR ph) (Lph^T Rph)^T
        const double x = hole ? lf(p, k) * rf(k, q) : lf(k, p) * rf(k, q) * hL;
        const double y = hole ? lf(q, k) * rf(k, p) : lf(k, q) * rf(k, p) * hL;
        const double f = hL * hR * ph;
        up += x - y * f;
        dn += y - x * f;
      } else {
        // pp: (hR ph) Lph Rph^T + Lpp Rpp - hL (Lph Rph^T)^T - (hL hR ph) (Lpp Rpp)^T
        const double f = hR * ph;
        const double x = hole ? lf(p, k) * rf(q, k) * f : lf(p, k) * rf(k, q);
        const double y = hole ? lf(q, k) * rf(p, k) * f : lf(q, k) * rf(k, p);
        up += x - y * (hL * f);
        dn += y - x * (hL * f);
      }
    }
  }
  const int nd2 = 2 * T.nd - 1;
  if (allowed && (terms & kTf121)) {
    const int K = jp + 1;  // J1 values of (a,p), at most
    for (int t = tid; t < L.nphp * K * nd2; t += kTfThreads) {
      const int d = t % nd2, v = t / nd2, k = v % K, u = v / K;
      const int a = L.php_a[u], i = L.php_i[u], ji = L.jj[i];  // ja = ji
      const int J1 = abs(ji - jp) + 2 * k, J2 = J1 + 2 * (d - (T.nd - 1));
      if (J1 > ji + jp || J2 < abs(ji - jq) || J2 > ji + jq || J1 + J2 < R) continue;
      double f1, f2;
      const long long p1 = t_pos_all(L, T, hR, a, p, i, q, ji, jp, ji, jq, J1, J2, true, f1);
      const long long p2 = t_pos_all(L, T, hR, i, p, a, q, ji, jp, ji, jq, J1, J2, true, f2);
      s1 += LF[(size_t)a * n + i] * (hL * f1 * RV[p1] - f2 * RV[p2]) * sqrt((J1 + 1.0) * (J2 + 1.0)) *
            sgnp((J1 >> 1) + ((R + jq + ji) >> 1)) * tx6(T, J1, J2, jq, jp, ji);
    }
  }
  if (allowed && (terms & kTf221)) {
    // over every orbit c, holes with W1 and particles with W2: J2 < J1 reads
    // W(cq, cp; J2 J1) (the lower half, by herm), J2 >= J1 W(cp, cq; J1 J2).
    // The pairs' channel matches the output's, which passed the tensor's tests.
    const int K = jp + 1;
    for (int t = tid; t < n * K * nd2; t += kTfThreads) {
      const int d = t % nd2, v = t / nd2, k = v % K, c = v / K, jc = L.jj[c];
      const int J1 = abs(jc - jp) + 2 * k, J2 = J1 + 2 * (d - (T.nd - 1));
      if (J1 > jc + jp || J2 < abs(jc - jq) || J2 > jc + jq || J1 + J2 < R) continue;
      const bool lo = J2 < J1;
      double f;
      const long long pos = lo ? t_pos_all(L, T, hR, c, q, c, p, jc, jq, jc, jp, J2, J1, true, f)
                               : t_pos_all(L, T, hR, c, p, c, q, jc, jp, jc, jq, J1, J2, true, f);
      const double co = sqrt((J1 + 1.0) * (J2 + 1.0)) * tx6(T, J1, J2, jq, jp, jc) * sgnp((jc + jq + R) >> 1);
      s2 += (lo ? -co * sgnp(J2 >> 1) * (hL * hR) : co * sgnp(J1 >> 1)) * f * (L.con[c] ? W1 : W2)[pos];
    }
  }
  if (allowed && (terms & kTf211)) {
    const int PAR = (lp + lq) & 1;
    const int qx = (R >> 1) + 2 * PAR * (L.jtot_max + 1);  // Pandya block (J = R, Tz = 0, PAR)
    const int rpq = L.ccrow[((size_t)qx * n + p) * n + q], rqp = L.ccrow[((size_t)qx * n + q) * n + p];
    const long long base = L.ccoff[qx];
    const int rlen = L.ccrlen[qx];
    const double inv = 1.0 / sqrt(R + 1.0);
    const double c1 = sgnp((jp - jq + R) >> 1), c2 = (double)(hR * hL * sgnp(R >> 1));
    if (rpq >= 0 && rqp >= 0)
      for (int u = tid; u < T.npart * T.nhole; u += kTfThreads) {
        const int a = T.parts[u / T.nhole], i = T.holes[u % T.nhole];
        if (((L.l[a] + L.l[i]) & 1) != ((T.dpar >> 1) & 1) || L.tz[i] != L.tz[a] || !dtri(L.jj[a], L.jj[i], R)) continue;
        const int col = T.ccol[((size_t)qx * n + a) * n + i];
        if (col < 0) continue;
        s3 += RF[(size_t)a * n + i] *
              (c1 * gcc[base + (long long)col * rlen + rpq] - c2 * gcc[base + (long long)col * rlen + rqp]) * inv;
      }
  }
  const double part[5] = {wave_sum(up), wave_sum(dn), wave_sum(s1), wave_sum(s2), wave_sum(s3)};
  if ((tid & 63) == 0)
    for (int v = 0; v < 5; v++) sh[v][tid >> 6] = part[v];
  __syncthreads();
  if (tid) return;
  double sum[5];
  for (int v = 0; v < 5; v++) {
    sum[v] = 0.0;
    for (int k = 0; k < kTfThreads / 64; k++) sum[v] += sh[v][k];
  }
  const size_t pq = (size_t)p * n + q, qp = (size_t)q * n + p;
  double v = (terms & kTf111) ? sum[0] : F[pq];
  const bool others = allowed && (terms & ~kTf111);
  if (others)
    for (int k = 0; k < 3; k++)
      if (terms & (kTf121 << k)) {
        v += sum[2 + k];
        if (p == q) v *= hres;
      }
  F[pq] = v;
  if (cp != cq)
    F[qp] = v * hres * sgnp((jq - jp) >> 1);  // (hole, particle): f_tensor_elem's phase
  else if (p != q)
    F[qp] = others ? v * hres * sgnp((jp - jq) >> 1) : sum[1];
}

// ---------------------------------------------------------------- two-body gathers
// TS_commutator_122 (TS_commutators.f90:555-663; overwrites every element) and
// _212 (:666-806; accumulates).  Per output (ab|cd; J1 J2) of a block q, over
// the orbits i of the (l,j,tz) group of a, b, c, d:
//   +LF(a,i) T(ib,cd)  +LF(b,i) T(ai,cd)  -LF(i,c) T(ab,id)  -LF(i,d) T(ab,ci)
// and over the orbits i the tensor's one-body part couples to a, b, d, c:
//   -{J1 J2 R; ji ja jb} RF(a,i) v(ib,cd;J2) (-1)^((ja+jb-J2)/2)
//   +{J1 J2 R; ji jb ja} RF(b,i) v(ia,cd;J2) (-1)^((J1+J2)/2)
//   +{J1 J2 R; jd ji jc} RF(i,d) v(ab,ci;J1) (-1)^((jc+jd-J1)/2)
//   -{J1 J2 R; jc ji jd} RF(i,c) v(ab,di;J1) (-1)^((J1+J2)/2)
// (times sqrt((J1+1)(J2+1)) (-1)^(R/2)): a sparse matrix over (ab) times rows
// of T's block and of G's block at J2, plus rows of T's block and of G's block
// at J1 times a sparse matrix over (cd).  Which entries exist is fixed with the
// tensor space; k_t_lists writes their weights once per commutator (every
// phase, 6j and pair norm; two lists per pair and block, against pair squared
// outputs), k_t_1body then does one multiply-add per entry and output.
//
// Rows go in groups of up to eight of the same or neighbouring (l,j,tz)
// classes: the rows of one class name the same partner rows of T and two
// thirds the same of G, so a group keeps one list of partner rows, each with
// the eight rows' weights.
struct TList {
  long long base;  // columns: weight of entry e at base + 64 e; rows: destination of entry e in rdst[base + e]
  int q, idx, side, n;
};
// ng row groups from g0 of block q
struct TItem {
  int q, g0, ng, pad;
};
// a row group's partner list (n entries from base), or the lists of 64
// columns (n entries each, entry e of column c at base + 64 e + c)
struct TSlice {
  long long base, n;
};
struct TLists {
  const TList *lists;
  const TItem *items;
  const TSlice *groups, *cols;
  const int *cbase;            // first entry of cols of a block
  const int *grow;             // rows of a group, eight entries, the last ones repeated
  const int *rsrc;             // partner row of T's block (>= 0) or of G's block at J2 (~row)
  const int *rdst;             // where a row's entry lies in rw, or -1
  const unsigned short *cp;    // column lists: position in [T's row | G's row at J1]
  double *rw, *cw;             // weights: rw[8 * entry + row of the group], cw by columns
  int nlist, nitem;
  unsigned lds;                // of k_t_1body
};
constexpr int kT1Threads = 768;
constexpr int kT1Lds = 163840;  // LDS of a workgroup at most

// The weight of an entry that an output does not have: it adds nothing, and no
// weight of a term is -0.  Where a sum is not finite it is made again without
// such entries, since 0 times an infinite element is not 0.
constexpr double kAbsent = -0.0;
__device__ __forceinline__ bool absent(double w) { return w == 0.0 && std::signbit(w); }

// one wavefront per list, a lane per entry
__global__ __launch_bounds__(64) void k_t_lists(DevLayout L, DevTensor T, TLists W, const double *__restrict__ LF,
                                                const double *__restrict__ RF, int do122, int do212) {
  const TList li = W.lists[blockIdx.x];
  const int q = li.q, n = L.nsp, R = T.rank, J1 = T.J1[q], J2 = T.J2[q];
  const int pr = L.pbase[li.side ? T.q2[q] : T.q1[q]] + li.idx;
  const int a = L.pair_a[pr], b = L.pair_b[pr], ja = L.jj[a], jb = L.jj[b];
  const double dab = a == b ? M_SQRT1_2 : 1.0;
  const double *x6 = T.x6 + (((size_t)(J1 >> 1) * T.nJ + (J2 >> 1)) * T.hx) * T.nh * T.nh;  // {J1 J2 R; . . .}
  auto six = [&](int j4, int j5, int j6) { return x6[((size_t)(j4 >> 1) * T.nh + (j5 >> 1)) * T.nh + (j6 >> 1)]; };
  const int g1 = L.grp_of[a], g2 = L.grp_of[b], c1 = L.grp_cnt[g1], c2 = L.grp_cnt[g2];
  const int p1 = T.pstart[a], m1 = T.pstart[a + 1] - p1, p2 = T.pstart[b], m2 = T.pstart[b + 1] - p2;
  const double n212 = sqrt((J1 + 1.0) * (J2 + 1.0)) * sgnp(R >> 1);
  for (int e = threadIdx.x; e < li.n; e += 64) {
    double w = kAbsent;
    if (e < c1 + c2) {
      // i for a (with o = b) or for b (o = a)
      const bool fa = e < c1;
      const int i = L.grp_list[fa ? L.grp_start[g1] + e : L.grp_start[g2] + e - c1];
      const int x = fa ? a : b, o = fa ? b : a, ji = L.jj[i], jo = L.jj[o], J = li.side ? J2 : J1;
      // the pair is (i,o) when i stands for a, (o,i) when for b
      const bool swp = fa ? i > o : o > i;
      const double f = swp ? (double)sgnp(1 + ((ji + jo - J) >> 1)) : (i == o ? M_SQRT2 : 1.0);
      if (do122) w = (li.side ? -f * LF[(size_t)i * n + x] * dab : f * LF[(size_t)x * n + i] * dab) + 0.0;
    } else if (e < c1 + c2 + m1 + m2) {
      const int k = e - c1 - c2;
      const bool fa = k < m1;
      const int pi = T.part[fa ? p1 + k : p2 + k - m1], i = pi & 255, ji = pi >> 8;
      const int x = fa ? a : b, o = fa ? b : a, jo = L.jj[o], J = li.side ? J1 : J2;
      // rows: v(i o, cd; J2); columns: v(ab, o i; J1)
      const bool swp = li.side ? o > i : i > o;
      const double f = swp ? (double)sgnp(1 + ((ji + jo - J) >> 1)) : (i == o ? M_SQRT2 : 1.0);
      if (do212) {
        double sx, sg;
        if (!li.side) {
          sx = fa ? six(ji, ja, jb) : six(ji, jb, ja);
          sg = fa ? -(double)sgnp((ja + jb - J2) >> 1) : (double)sgnp((J1 + J2) >> 1);
        } else {  // (a, b) are the reference's (c, d)
          sx = fa ? six(ja, ji, jb) : six(jb, ji, ja);
          sg = fa ? -(double)sgnp((J1 + J2) >> 1) : (double)sgnp((ja + jb - J1) >> 1);
        }
        w = sg * sx * f * (li.side ? RF[(size_t)i * n + x] : RF[(size_t)x * n + i]) * n212 * dab + 0.0;
      }
    }
    if (li.side) {
      W.cw[li.base + 64LL * e] = W.cp[li.base + 64LL * e] == 0xffff ? kAbsent : w;
    } else {
      const int d = W.rdst[li.base + e];
      if (d >= 0) W.rw[d] = w;
    }
  }
}

// A workgroup takes row groups of a block and stages T's and G's rows in LDS,
// where the column lists gather from them, with the groups' partner lists; a
// wavefront computes a group x 64 columns, so that a column list's entry and a
// partner row, read once, serve eight outputs.  Eight partner rows' reads are
// in flight.  Bound by those reads (L2-resident blocks) and the LDS gathers.  A
// thread per output with a pair lookup, an F entry and a 6j per term took
// 0.95 + 3.1 ms for the two commutators at 90 orbits, rank 4 (20 M outputs);
// this kernel 1.0 ms with a partner list per row, 0.66 ms with one per
// group (and a block on one XCD), 0.58 without spills: asked for six wavefronts a
// SIMD the compiler stores 44 bytes a lane, asked for four it needs 80 registers
// and six fit all the same.  The next batch of either list read ahead: 0.73.
// k_t_lists 0.09 ms.
__global__ __launch_bounds__(kT1Threads, 4) void k_t_1body(DevLayout L, DevTensor T, TLists W,
                                                        const double *__restrict__ GV, const double *__restrict__ RV,
                                                        double *__restrict__ OV, int add) {
  extern __shared__ double rows[];
  const TItem it = W.items[blockIdx.x];
  if (it.ng == 0) return;
  const int q = it.q, n2 = T.n2[q], q1 = T.q1[q], q2 = T.q2[q], d1 = L.bdim[q1], ld = (n2 + d1) | 1;
  const double *Tq = RV + T.off[q], *V1 = GV + L.boff[q1], *V2 = GV + L.boff[q2];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const TSlice *gs = W.groups + it.g0;
  const int *grow = W.grow + 8 * it.g0;
  // LDS: 8 rows a group (a repeated row is staged once), the weights, the partner rows
  const long long b0 = gs[0].base;
  const int len = (int)(gs[it.ng - 1].base - b0 + gs[it.ng - 1].n);
  int nst = 0;  // rows before the group's
  for (int g = 0; g < it.ng; g++) {
    const int gn = grow[8 * g + 7] >> 24;  // the group's rows, kept with its last entry
    for (int j = wave; j < gn; j += kT1Threads / 64) {
      const int r = grow[8 * g + j] & 0xffffff;
      const double *t = Tq + (long long)r * n2, *v = V1 + (long long)r * d1;
      double *d = rows + (nst + j) * ld;
      for (int k = lane; k < n2; k += 64) d[k] = t[k];
      for (int k = lane; k < d1; k += 64) d[n2 + k] = v[k];
    }
    nst += gn;
  }
  double *lw = rows + ((nst * ld + 1) & ~1);
  int *lr = reinterpret_cast<int *>(lw + 8 * len);
  for (int k = threadIdx.x; k < 8 * len; k += kT1Threads) lw[k] = W.rw[8 * b0 + k];
  for (int k = threadIdx.x; k < len; k += kT1Threads) lr[k] = W.rsrc[b0 + k];
  __syncthreads();
  const int nch = (n2 + 63) >> 6, nu = nch * it.ng;
  for (int u = wave; u < nu; u += kT1Threads / 64) {
    const int ch = u % nch, g = u / nch;
    const int s = ch * 64 + lane, sc = min(s, n2 - 1);
    double acc[8];
#pragma unroll
    for (int j = 0; j < 8; j++) acc[j] = 0.0;
    const int l0 = (int)(gs[g].base - b0), l1 = l0 + (int)gs[g].n;
    for (int e = l0; e < l1; e += 8) {  // the list's length is a multiple of 8
      double v[8];
#pragma unroll
      for (int k = 0; k < 8; k++) {
        const int r = __builtin_amdgcn_readfirstlane(lr[e + k]);
        v[k] = (r >= 0 ? Tq + (long long)r * n2 : V2 + (long long)~r * n2)[sc];
      }
#pragma unroll
      for (int k = 0; k < 8; k++)
#pragma unroll
        for (int j = 0; j < 8; j++) acc[j] = fma(lw[8 * (e + k) + j], v[k], acc[j]);
    }
    int st = 0;
    for (int k = 0; k < g; k++) st += grow[8 * k + 7] >> 24;
    const int gn = grow[8 * g + 7] >> 24;
    const double *row0 = rows + st * ld;
    const TSlice sl = W.cols[W.cbase[q] + ch];
    // four entries of a column list in flight (their number is a multiple of 4)
    for (int e = 0; e < (int)sl.n; e += 4) {
      double w[4];
      int p[4];
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const long long o = sl.base + (long long)(e + v) * 64 + lane;
        w[v] = W.cw[o];
        p[v] = W.cp[o];
      }
#pragma unroll
      for (int v = 0; v < 4; v++) {
        const int pv = p[v] == 0xffff ? 0 : p[v];
#pragma unroll
        for (int j = 0; j < 8; j++) acc[j] = fma(w[v], row0[min(j, gn - 1) * ld + pv], acc[j]);
      }
    }
    bool finite = true;
#pragma unroll
    for (int j = 0; j < 8; j++) finite = finite && fabs(acc[j]) <= DBL_MAX;
    if (s < n2 && finite) {
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (j < gn) {
          double *o = OV + T.off[q] + (long long)(grow[8 * g + j] & 0xffffff) * n2 + s;
          *o = add ? *o + acc[j] : acc[j];
        }
    } else if (s < n2) {
      // (everything read again here, so that the loops above keep their registers)
#pragma unroll 1
      for (int j = 0; j < grow[8 * g + 7] >> 24; j++) {
        double sum = 0.0;
#pragma unroll 1
        for (int e = (int)(gs[g].base - b0); e < (int)(gs[g].base - b0 + gs[g].n); e++) {
          const int r = lr[e];
          if (!absent(lw[8 * e + j]))
            sum = fma(lw[8 * e + j], (r >= 0 ? Tq + (long long)r * n2 : V2 + (long long)~r * n2)[s], sum);
        }
#pragma unroll 1
        for (int e = 0; e < (int)W.cols[W.cbase[q] + ch].n; e++) {
          const long long o = W.cols[W.cbase[q] + ch].base + (long long)e * 64 + lane;
          if (!absent(W.cw[o])) sum = fma(W.cw[o], rows[(st + j) * ld + W.cp[o]], sum);
        }
        double *o = OV + T.off[q] + (long long)(grow[8 * g + j] & 0xffffff) * n2 + s;
        *o = add ? *o + sum : sum;
      }
    }
  }
}

// The scalar Pandya matrices with each column's rows in group order: the right
// operand of Wy
__global__ void k_gcc_order(DevLayout L, DevTensor T, const double *__restrict__ gcc, double *__restrict__ out) {
  const int col = blockIdx.x, q = L.cccol_q[col], rl = L.ccrlen[q];
  const long long o = L.ccoff[q] + (long long)(col - L.cccbase[q]) * rl;
  const int *ix = T.rperm + L.ccrbase[q];
  for (int i = threadIdx.x; i < rl; i += 256) out[o + i] = gcc[o + ix[i]];
}

// The ph recoupling of TS_commutator_222_ph (TS_commutators.f90:1459-1849) as
// a gather by orbit quadruple (x0 <= x1 | x2 <= x3).  The reference adds every
// product entry W(IX = (d,a) at J3, JX = (c,b) at J4) (Wx or Wy) into up to
// 16 x (J1, J2) outputs; read backwards, an output (x0 x1 | x2 x3; J1 J2)
// receives entries through sixteen patterns: the source orbits (a,b,c,d) as a
// permutation of x, the orbit-order condition of the reference's branch, one
// of four 9j argument orders, a phase and a herm factor.  The entries a
// quadruple's outputs read, over the slots (pattern, J3, J4), do not depend on
// the outputs' (J1, J2), and the weights do not depend on the orbits' radial
// numbers: quadruples of the same four (l,j,tz) groups share slots, weights
// and outputs' (J1, J2).  See k_t222ph.
//
// The sixteen patterns (TS_commutators.f90:1562-1849): the output receives
// W(d,a;c,b) times P * 9j * sign * herm, P = sqrt((2J1+1)(2J2+1)(2J3+1)(2J4+1)),
// ph34 = (-1)^((J3+J4)/2), abcd = (-1)^((ja+jb+jc+jd)/2), all angular momenta doubled.
//  k  W   output = V^{J1 J2} of   branch          9j {. . J3; . . J4; J1 J2 R}   factor
//  0  Wx  (a,b,c,d)               b>=a, d>=c       (ja jd | jb jc)   (-1)^((jb+jd+J2)/2) ph34 hL
//  1  Wx  (c,d,a,b)               b>=a, d>=c       (jd ja | jc jb)  -(-1)^((jc+ja+J1+R)/2) hR
//  2  Wx  (a,b,d,c)               b>=a, d<c        (ja jd | jb jc)   (-1)^((jb+jc)/2) ph34 hL
//  3  Wx  (d,c,a,b)               b>=a, d<c        (jd ja | jc jb)   (-1)^((ja-jd+R)/2) hR
//  4  Wx  (b,a,c,d)               b<a, d>=c        (ja jd | jb jc)   (-1)^((ja+jd+J1+J2)/2) ph34 hL
//  5  Wx  (c,d,b,a)               b<a, d>=c        (jd ja | jc jb)   (-1)^((jc-jb+J1+J2+R)/2) hR
//  6  Wx  (b,a,d,c)               b<a, d<c         (ja jd | jb jc)   (-1)^((ja+jc+J1)/2) ph34 hL
//  7  Wx  (d,c,b,a)               b<a, d<c         (jd ja | jc jb)   (-1)^((jb-jd+J2+R)/2) hR
//  8  Wy  (d,b,c,a)               b>=d, a>=c       (jd ja | jb jc)   (-1)^((jc+ja+J2)/2) hL
//  9  Wy  (c,a,d,b)               b>=d, a>=c       (ja jd | jc jb)   (-1)^((jd-jb+J1+R)/2) ph34 hR
// 10  Wy  (d,b,a,c)               b>=d, a<c        (jd ja | jb jc)  -hL
// 11  Wy  (a,c,d,b)               b>=d, a<c        (ja jd | jc jb)   abcd ph34 (-1)^(R/2) hR
// 12  Wy  (b,d,c,a)               b<d, a>=c        (jd ja | jb jc)  -abcd (-1)^((J1+J2)/2) hL
// 13  Wy  (c,a,b,d)               b<d, a>=c        (ja jd | jc jb)   (-1)^((J1+J2+R)/2) ph34 hR
// 14  Wy  (b,d,a,c)               b<d, a<c         (jd ja | jb jc)   (-1)^((jb+jd+J1)/2) hL
// 15  Wy  (a,c,b,d)               b<d, a<c         (ja jd | jc jb)   (-1)^((ja-jc+J2+R)/2) ph34 hR
// Matching the output (x0 x1 | x2 x3) to the k-th form gives (a,b,c,d) as a
// permutation of x (the packed tables ia..id below) and turns the branch into
// x0 < x1 and / or x2 < x3; no Wy where J3 = J4 (the reference skips it).
// the patterns' (a, b, c, d) as indices into (x0, x1, x2, x3), two bits each,
// pattern k in bits 2k..2k+1, and their branch conditions (1: x0 < x1,
// 2: x2 < x3, 3: both)
constexpr unsigned kPhIa = 0x2727DD88u, kPhIb = 0x88DD88DDu, kPhIc = 0x72727272u, kPhId = 0xDD882727u;
constexpr unsigned kPhCond = 0xF960F960u;
constexpr int kPhQ = 8;    // quadruples of one class per workgroup
constexpr int kPhU = 2;    // slots whose 9j a lane reads together
constexpr int kPhB = 32;   // slots a workgroup weights at a time

// The sums of the recoupling and the tensor Pandya transform: a quadruple's
// outputs o = (J - Jlo)/2 * nd + (J' - J)/2 over up to 128 consecutive o, each
// the sum over slots of weight[slot][quadruple] * 9j[slot][o], for kPhQ
// quadruples of one class at once.  The table's fastest indices are the
// outputs' (J, J'), so a slot's 9j are one contiguous run: groups of lanes as
// wide as half the outputs take a slot each, a lane two neighbouring outputs.
struct Recouple {
  int wsh, G, grp, ol;
  unsigned flip;  // bit 4u + ab: the sign of output u's phase, ab a slot's flags (J/2, J'/2)
  double acc[kPhQ][2];

  // outputs from o0 on, nout of them in all; x / nd = x * ndinv >> 16
  __device__ __forceinline__ void begin(int lane, int o0, int nout, int Jlo, int nd, int ndinv) {
    const int nh2 = (min(nout - o0, 128) + 1) >> 1;  // lanes a group needs
    wsh = nh2 <= 4 ? 2 : nh2 <= 8 ? 3 : nh2 <= 16 ? 4 : nh2 <= 32 ? 5 : 6;
    G = 64 >> wsh;
    grp = lane >> wsh;
    ol = o0 + 2 * (lane & ((1 << wsh) - 1));
    flip = 0;
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int oq = ((ol + u) * ndinv) >> 16;
      const unsigned e1 = ((Jlo >> 1) + oq) & 1, e2 = (e1 + (ol + u - oq * nd)) & 1;
      flip |= (e1 << 1 | e2 << 2 | (e1 ^ e2) << 3) << (4 * u);
    }
#pragma unroll
    for (int q = 0; q < kPhQ; q++) acc[q][0] = acc[q][1] = 0.0;
  }
  // count slots: weights cs (row count: zeros), 9j rows sb9 (flags in the top two bits) from n9
  __device__ __forceinline__ void add(const double *__restrict__ n9, const double (*cs)[kPhQ], const unsigned *sb9,
                                      int count) {
    for (int t0 = grp; t0 < count; t0 += kPhU * G) {
      dpair_t v[kPhU];
      unsigned ab[kPhU];
#pragma unroll
      for (int u = 0; u < kPhU; u++) {
        const unsigned b = sb9[min(t0 + u * G, count)];
        v[u] = *reinterpret_cast<const dpair_t *>(n9 + (b & 0x3fffffffu));
        ab[u] = b >> 30;
      }
#pragma unroll
      for (int u = 0; u < kPhU; u++) {
        __builtin_amdgcn_sched_barrier(0);  // one slot's row from LDS at a time: registers
        const double f0 = ((flip >> ab[u]) & 1) ? -v[u].x : v[u].x;
        const double f1 = ((flip >> (4 + ab[u])) & 1) ? -v[u].y : v[u].y;
        const double *cq = cs[min(t0 + u * G, count)];
#pragma unroll
        for (int q = 0; q < kPhQ; q++) {
          const double c = cq[q];
          acc[q][0] = fma(f0, c, acc[q][0]);
          acc[q][1] = fma(f1, c, acc[q][1]);
        }
      }
    }
  }
  // the groups' sums; each group is left with nown quadruples from q0 (mine
  // false: another group holds the same one)
  __device__ __forceinline__ void reduce(int lane, int &q0, int &nown, bool &mine) {
    q0 = 0;
    nown = kPhQ;
#pragma unroll
    for (int st = 0; st < 3; st++) {
      if (wsh > 5 - st) break;
      const int half = kPhQ >> (st + 1);
      const bool up = (lane >> (5 - st)) & 1;
#pragma unroll
      for (int i = 0; i < half; i++)
#pragma unroll
        for (int u = 0; u < 2; u++) {
          const double give = up ? acc[i][u] : acc[i + half][u], keep = up ? acc[i + half][u] : acc[i][u];
          acc[i][u] = keep + __shfl_xor(give, 32 >> st);
        }
      if (up) q0 += half;
      nown = half;
    }
    mine = true;
    if (wsh == 2) {  // 16 groups for 8 quadruples
#pragma unroll
      for (int u = 0; u < 2; u++) acc[0][u] += __shfl_xor(acc[0][u], 4);
      mine = !(lane & 4);
    }
  }
};
// Runs of 64 class-ordered items per XCD, in turn: its L2 keeps the 9j rows
// and entries that neighbouring items share, and the classes of high j, with
// the most slots, spread over all XCDs.  bid of npad (a multiple of 512), the
// heavy classes first
__device__ __forceinline__ int class_item(int bid, int npad) {
  const int b = npad - 1 - bid, i8 = b >> 3;
  return ((i8 >> 6) << 9) + ((b & 7) << 6) + (i8 & 63);
}

// The tensor Pandya matrices of the cross-coupled blocks (calculate_single_pandya,
// cross_coupled.f90:1416-1634): CCX (rows: ordered pairs (a,b) at J3 in the
// scalar Pandya row order, columns: (p,h) at J4) and CCR (rows: (p,h) at J3,
// columns: ordered pairs (b,a) at J4 in group order).  Both are, for orbits
// (u,v,x,y) = (a,h,b,p) or (h,a,p,b), the sum over (J', J'') of
//   -(-1)^(J''/2) sqrt((J'+1)(J''+1)(J3+1)(J4+1)) {u v J'; x y J''; J3 J4 R}
//   T^{J' J''}(u v, y x) (-1)^((jv+jx+J4)/2), times (-1)^((jp+jh)/2) in CCR
// in row (u,x) at J3 and column (y,v) at J4.  The entries T that a quadruple
// reads do not depend on (J3, J4): gathered once, as in the recoupling, by
// classes of quadruples.  (J', J'') with J' > J'' exchanges the first two
// rows of the 9j, which the table holds for J' <= J'' only.
//
// One thread per element, with a 9j and five table reads per term, took
// 3.8 ms for both matrices at 90 orbits, rank 4 (16 M elements), 100 us at 30
// orbits, rank 2; this kernel 0.55 ms and 20 us.
struct TPan {
  const unsigned *quads;  // u | v<<8 | x<<16 | y<<24
  const PhChunkT *chunks;
  int nchunk, npad;
  const int *rtab, *ctab;     // row of the pair (u,x) or (x,u), column of (y,v), by pair, J fastest
  const struct CcBlk *blk;    // the matrices, as DevTensor::cblk
  double *out;
};
struct PanSeg {
  double c;
  long long off;  // of the tensor block
  unsigned b9;    // 9j table row | 3 << 30 where (-1)^((J3+J4)/2) applies
  int n2;         // its row length
  unsigned code;  // J'/2 | J''/2 << 8 | (J' > J'') << 16
};
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(5))) void k_t_pandya(
    DevLayout L, DevTensor T, TPan P0, TPan P1, const double *__restrict__ RV, int hR) {
  __shared__ PanSeg seg[kPhB + 64];
  __shared__ alignas(16) double cs[kPhB + 1][kPhQ];
  __shared__ unsigned sb9[kPhB + 1];
  const int mode = (int)blockIdx.x >= P0.npad;
  const TPan P = mode ? P1 : P0;
  const int item = class_item((int)blockIdx.x - (mode ? P0.npad : 0), P.npad);
  if (item >= P.nchunk) return;
  const int lane = threadIdx.x, quad = lane & (kPhQ - 1);
  const PhChunkT ch = P.chunks[item];
  const int nq = ch.n, R = T.rank, n = L.nsp, nd = T.nd, nJ = T.nJ, h = T.nh, nd2 = 2 * nd - 1;
  const unsigned code = P.quads[ch.first + min(quad, nq - 1)];  // the lane's quadruple
  const int u = code & 255, v = (code >> 8) & 255, x = (code >> 16) & 255, y = (int)(code >> 24);
  const int ju = ch.jv & 255, jv = (ch.jv >> 8) & 255, jx = (ch.jv >> 16) & 255, jy = (int)(ch.jv >> 24);
  const unsigned lt = ch.lt;  // bits 0-3: l of u, v, x, y; 4-7: tz
  const int Tzq = (int)((lt >> 4) & 1) + (int)((lt >> 5) & 1);
  const int Puv = (lt ^ (lt >> 1)) & 1, Pyx = ((lt >> 2) ^ (lt >> 3)) & 1;
  const int ndinv = 65536 / nd + 1, nd2inv = 65536 / nd2 + 1;  // exact for x <= 32 nd2 + 128, nd2 <= 50
  // the lane's pairs in the channels' order, and what an exchange does
  const int puv = (min(u, v) * n + max(u, v)) * nJ, pyx = (min(x, y) * n + max(x, y)) * nJ;
  const double fq = (u == v ? M_SQRT2 : 1.0) * (x == y ? M_SQRT2 : 1.0);
  const unsigned b9a = (unsigned)((((ju >> 1) * h + (jv >> 1)) * h + (jx >> 1)) * h + (jy >> 1));
  const unsigned b9b = (unsigned)((((jx >> 1) * h + (jy >> 1)) * h + (ju >> 1)) * h + (jv >> 1));
  const int Jlo = abs(ju - jx), nout = (min(ju, jx) + 1) * nd;  // J3 of the row pair
  const int J1lo = abs(ju - jv), nslot = (min(ju, jv) + 1) * nd2;
  Recouple rc;
  for (int o0 = 0; o0 < nout; o0 += 128) {
    rc.begin(lane, o0, nout, Jlo, nd, ndinv);
    const double *n9 = T.n9 + (size_t)(Jlo >> 1) * nd + rc.ol;
    int nseg = 0;
    for (int s0 = 0; s0 < nslot || nseg > 0;) {
      // the slots (J', J'') that exist, until kPhB wait or none is left
      while (nseg < kPhB && s0 < nslot) {
        const int s = s0 + lane, r = min(s, nslot - 1), rq = (r * nd2inv) >> 16;
        const int Ja = J1lo + 2 * rq, Jb = Ja + 2 * (r - rq * nd2 - (nd - 1));
        bool ok = s < nslot && Jb >= abs(jx - jy) && Jb <= jx + jy && Ja + Jb >= R;
        const bool sw = Ja > Jb;
        const int lo = sw ? Jb : Ja, dJ = abs(Jb - Ja);
        OutBlk ob{-1, 0, 0};
        if (ok) ob = T.oblk[((lo >> 1) * nd + (dJ >> 1)) * 6 + Tzq * 2 + (sw ? Pyx : Puv)];
        ok = ok && ob.off >= 0;
        const unsigned long long m = __ballot(ok);
        if (ok) {
          PanSeg g;
          g.c = -sgnp(Jb >> 1) * sqrt((Ja + 1.0) * (Jb + 1.0));
          if (sw) g.c *= sgnp((dJ >> 1) + ((ju + jv + Ja + jx + jy + Jb + R) >> 1)) * hR;
          g.off = ob.off;
          g.n2 = ob.n2;
          g.b9 = (((sw ? b9b : b9a) * nJ + (lo >> 1)) * nd + (dJ >> 1)) * (unsigned)(nJ * nd) | (sw ? 3u << 30 : 0u);
          g.code = (unsigned)(Ja >> 1) | (unsigned)(Jb >> 1) << 8 | (sw ? 1u << 16 : 0u);
          seg[nseg + __popcll(m & ((1ull << lane) - 1ull))] = g;
        }
        nseg += __popcll(m);
        s0 += 64;
      }
      // none may be left: the reads below then take this for slot 0 (leaving the
      // loop here instead costs the compiler 39 more spilled registers)
      if (lane == 0 && nseg == 0) seg[0].code = 0;
      __syncthreads();
      const int nb = min(nseg, kPhB);
      {
        int ix[4], jx_[4];
        double w[4];
        auto slot = [&](int k) -> const PanSeg & { return seg[min(8 * k + (lane >> 3), max(nb - 1, 0))]; };
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const unsigned gc = slot(k).code;
          ix[k] = T.prow[puv + (int)(gc & 31)];
          jx_[k] = T.prow[pyx + (int)((gc >> 8) & 31)];
          if (8 * k + (lane >> 3) >= nb || quad >= nq) ix[k] = -1;
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const bool sw = (slot(k).code >> 16) & 1;
          w[k] = 0.0;
          if ((ix[k] | jx_[k]) >= 0)
            w[k] = RV[slot(k).off + (long long)(sw ? jx_[k] : ix[k]) * slot(k).n2 + (sw ? ix[k] : jx_[k])];
        }
#pragma unroll
        for (int k = 0; k < 4; k++) {
          const int pos = 8 * k + (lane >> 3);
          if (pos < nb) {
            const unsigned gc = slot(k).code;
            // a pair read against its order: (-1)^(1 + (j + j' - J)/2)
            int e = 0;
            if (u > v) e += 1 + ((ju + jv) >> 1) - (int)(gc & 31);
            if (y > x) e += 1 + ((jx + jy) >> 1) - (int)((gc >> 8) & 31);
            const double c = slot(k).c * w[k] * fq;
            cs[pos][quad] = (e & 1) ? -c : c;
            if (quad == 0) sb9[pos] = slot(k).b9;
          }
        }
      }
      if (lane < kPhQ) cs[nb][lane] = 0.0;  // what the last round reads past the end
      if (lane == kPhQ) sb9[nb] = 0;
      // the slots that wait move to the front
      nseg -= nb;
      const double mc = seg[kPhB + lane].c;
      const long long mw = seg[kPhB + lane].off;
      const unsigned mb = seg[kPhB + lane].b9, mo = seg[kPhB + lane].code;
      const int mn = seg[kPhB + lane].n2;
      __syncthreads();
      if (lane < nseg) {
        seg[lane].c = mc;
        seg[lane].off = mw;
        seg[lane].b9 = mb;
        seg[lane].code = mo;
        seg[lane].n2 = mn;
      }
      rc.add(n9, cs, sb9, nb);
      __syncthreads();
    }
    int q0, nown;
    bool mine;
    rc.reduce(lane, q0, nown, mine);
    const int ol = rc.ol, oq0 = (ol * ndinv) >> 16, oq1 = ((ol + 1) * ndinv) >> 16;
    const int J3o[2] = {Jlo + 2 * oq0, Jlo + 2 * oq1};
    const int J4o[2] = {J3o[0] + 2 * (ol - oq0 * nd), J3o[1] + 2 * (ol + 1 - oq1 * nd)};
    CcBlk ob[2];
    double nrm[2];
#pragma unroll
    for (int k = 0; k < 2; k++) {
      const int J3 = J3o[k], J4 = J4o[k];
      const bool val = mine && ol + k < nout && ol + k < o0 + 128 && J4 >= abs(jy - jv) && J4 <= jy + jv;
      const unsigned dl = lt ^ (lt >> 2);  // l and tz of u against x
      ob[k] = P.blk[val ? ((int)(((dl >> 4) & 1) + 2 * (dl & 1)) * nJ + (J3 >> 1)) * nd + ((J4 - J3) >> 1) : 0];
      if (!val) ob[k].wo = -1;
      nrm[k] = sqrt((J3 + 1.0) * (J4 + 1.0)) * sgnp(((jv + jx + J4) >> 1) + (mode ? (ju + jx) >> 1 : 0));
    }
#pragma unroll
    for (int i = 0; i < kPhQ; i++) {
      if (i >= nown) break;
      const unsigned cd = (unsigned)__shfl((int)code, q0 + i);
      const int cu = cd & 255, cv = (cd >> 8) & 255, cx = (cd >> 16) & 255, cy = (int)(cd >> 24);
      const int *p1 = P.rtab + (mode ? cx * n + cu : cu * n + cx) * nJ, *p2 = P.ctab + (cy * n + cv) * nJ;
#pragma unroll
      for (int k = 0; k < 2; k++)
        if (q0 + i < nq && ob[k].wo >= 0) {
          const int r = p1[J3o[k] >> 1], c = p2[J4o[k] >> 1];
          if ((r | c) >= 0) P.out[ob[k].wo + (long long)r * ob[k].rl4 + c] = rc.acc[i][k] * nrm[k];
        }
    }
  }
}

struct PhPat {
  double cs;     // sign * herm
  unsigned b9;   // 9j table index of the four orbits' 2j
  int start;     // first slot
  int j3;        // first J3 of its run
  int flags;     // Tz | parity of the J3 pairs << 1 | ab << 3 | ph34 << 5 | lowest J4 << 6 | highest << 18
};
struct PhSeg {
  double c;       // sign * herm * phase(J3,J4) * sqrt((2J3+1)(2J4+1))
  long long w;    // offset of the slot's product block << 24 | its row length
  unsigned b9;    // 9j table row without the (J1, J2) part | ab << 30
  unsigned code;  // pattern | J3/2 << 4 | J4/2 << 12
};
// One wavefront takes up to kPhQ quadruples of one class, kPhB slots at a time:
//   1. one lane per slot finds the slots that exist (J4's triangle, no Wy at
//      J3 = J4), their (J3, J4) weights and product blocks;
//   2. lanes (slot, quadruple) read the product entries, rows and columns from
//      per-pair tables (a quadruple's run over J3 is contiguous there); the
//      entries that pass the reference's |W| > 1e-6 test go weighted to LDS,
//      slots with no entry left are dropped;
//   3. the slots are summed into the outputs (Recouple).
// What bounds it: the entries' reads (W is two products of 0.85 GB at 90 orbits, rank 2) and the
// index arithmetic around them.  One wavefront per quadruple with a lane per
// slot read a 9j cache line per (slot, output): 7.7 ms there (2.6 M
// quadruples, 256 M slots, 3 G slot-outputs); this form 2.8 ms, 5.3 before
// the columns of W went into class order.
// W: Wx, then Wy wsize doubles on
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(4))) void k_t222ph(DevLayout L, DevTensor T, const double *__restrict__ W,
    long long wsize, double *__restrict__ OV, int hL, int hR) {
  __shared__ PhPat pat[16];
  __shared__ PhSeg seg[kPhB + 64];
  __shared__ ushort2 base[16][kPhQ];  // per pattern and quadruple: the orbit pairs (d,a) and (c,b)
  __shared__ alignas(16) double cs[kPhB + 1][kPhQ];
  __shared__ unsigned sb9[kPhB + 1];
  const int item = class_item(blockIdx.x, T.nqpad);
  if (item >= T.nqchunk) return;
  const int lane = threadIdx.x;
  const PhChunkT ch = T.qchunk[item];
  const int nq = ch.n, R = T.rank, n = L.nsp, JM = L.jtot_max, nd = T.nd, nJ = T.nJ, h = T.nh;
  const int quad = lane & (kPhQ - 1);
  const unsigned code = T.quads[ch.first + min(quad, nq - 1)];  // the lane's quadruple
  // the pattern conditions the lane's quadruple fails (1: x0 < x1, 2: x2 < x3)
  const unsigned drop = ((code & 255) == ((code >> 8) & 255) ? 1u : 0u) |
                        (((code >> 16) & 255) == code >> 24 ? 2u : 0u);
#pragma unroll
  for (int u = 0; u < 2; u++) {
    const int k = 8 * u + (lane >> 3);
    auto orb = [&](unsigned tbl) { return (int)((code >> (8 * ((tbl >> (2 * k)) & 3))) & 255); };
    base[k][quad] = make_ushort2((unsigned short)(orb(kPhId) * n + orb(kPhIa)),
                                 (unsigned short)(orb(kPhIc) * n + orb(kPhIb)));
  }
  const int j0 = ch.jv & 255, j1 = (ch.jv >> 8) & 255, j2 = (ch.jv >> 16) & 255, j3 = (int)(ch.jv >> 24);
  int nslot;
  {
    const int k = lane & 15;
    auto orb = [&](unsigned tbl) { return (int)((tbl >> (2 * k)) & 3); };
    const int oa = orb(kPhIa), ob = orb(kPhIb), oc = orb(kPhIc), od = orb(kPhId);
    const int ja = (ch.jv >> (8 * oa)) & 255, jb = (ch.jv >> (8 * ob)) & 255;
    const int jc = (ch.jv >> (8 * oc)) & 255, jd = (ch.jv >> (8 * od)) & 255;
    const unsigned lt = ch.lt, ad_ = (lt >> oa) ^ (lt >> od), bc_ = (lt >> ob) ^ (lt >> oc);  // l, tz differences
    const int Tz = (ad_ >> 4) & 1, PAR = ad_ & 1, PAR2 = PAR ^ ((T.dpar >> 1) & 1);
    const bool ok = (int)(bc_ & 1) == PAR2 && (int)((bc_ >> 4) & 1) == Tz;
    // constant sign exponent (halves), J1/J2 flags and the (J3,J4) phase of each pattern
    // (TS_commutators.f90:1562-1849)
    int e = 0, ab = 0;
    double sg = 1.0;
    const int abcd = (ja + jb + jc + jd) >> 1;
    switch (k) {
      case 0: e = (jb + jd) >> 1; ab = 2; break;
      case 1: e = (jc + ja + R) >> 1; ab = 1; sg = -1.0; break;
      case 2: e = (jb + jc) >> 1; break;
      case 3: e = (ja - jd + R) >> 1; break;
      case 4: e = (ja + jd) >> 1; ab = 3; break;
      case 5: e = (jc - jb + R) >> 1; ab = 3; break;
      case 6: e = (ja + jc) >> 1; ab = 1; break;
      case 7: e = (jb - jd + R) >> 1; ab = 2; break;
      case 8: e = (jc + ja) >> 1; ab = 2; break;
      case 9: e = (jd - jb + R) >> 1; ab = 1; break;
      case 10: sg = -1.0; break;
      case 11: e = abcd + (R >> 1); break;
      case 12: e = abcd; ab = 3; sg = -1.0; break;
      case 13: e = R >> 1; ab = 3; break;
      case 14: e = (jb + jd) >> 1; ab = 1; break;
      default: e = (ja - jc + R) >> 1; ab = 2; break;
    }
    const bool ph34 = (k < 8) ? !(k & 1) : (k & 1);
    // the 9j argument order of the pattern: (ja,jd | jb,jc), (jd,ja | jc,jb), (jd,ja | jb,jc), (ja,jd | jc,jb)
    const int var = (k < 8) ? (k & 1) : 2 + (k & 1);
    const bool ad = var == 0 || var == 3, bc = var == 0 || var == 2;
    const int len = ok ? (((jd + ja - abs(jd - ja)) >> 1) + 1) * nd : 0;  // slots (J3 of |jd-ja| .. jd+ja, J4 - J3)
    int end = len;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const int v = __shfl_up(end, o, 16);
      if (k >= o) end += v;
    }
    nslot = __shfl(end, 15, 64);
    if (lane < 16) {
      PhPat p;
      p.cs = sg * sgnp(e) * ((k & 1) ? hR : hL);
      p.b9 = (unsigned)(((((ad ? ja : jd) >> 1) * h + ((ad ? jd : ja) >> 1)) * h + ((bc ? jb : jc) >> 1)) * h +
                        ((bc ? jc : jb) >> 1));
      p.start = end - len;
      p.j3 = abs(jd - ja);
      p.flags = Tz | PAR << 1 | ab << 3 | (ph34 ? 32 : 0) | abs(jc - jb) << 6 | (jc + jb) << 18;
      pat[k] = p;
    }
  }
  // outputs (x0 x1 | x2 x3; J1 <= J2): o = (J1 - |j0-j1|)/2 * nd + (J2 - J1)/2
  const int Jlo = abs(j0 - j1), nout = (min(j0, j1) + 1) * nd;
  const int Tzq = ((ch.lt >> 4) & 1) + ((ch.lt >> 5) & 1), P1 = (ch.lt ^ (ch.lt >> 1)) & 1;
  const double thr = (double)1e-6f;
  const int ndinv = 65536 / nd + 1;  // x / nd, exact for x <= 32 nd + 128, nd <= 50
  auto div = [&](int x) { return (x * ndinv) >> 16; };
  __syncthreads();
  Recouple rc;
  for (int o0 = 0; o0 < nout; o0 += 128) {
    rc.begin(lane, o0, nout, Jlo, nd, ndinv);
    const int ol = rc.ol;
    const double *n9 = T.n9 + (size_t)(Jlo >> 1) * nd + ol;
    int k = 0, nseg = 0;  // a lane's pattern: its slot only grows, so k carries over
    for (int s0 = 0; s0 < nslot || nseg > 0;) {
      // 1: the slots that exist, until kPhB wait or none is left
      while (nseg < kPhB && s0 < nslot) {
        const int s = min(s0 + lane, nslot - 1);
        while (k < 15 && pat[k + 1].start <= s) k++;
        const PhPat p = pat[k];
        const int r = s - p.start, rq = div(r), J3 = p.j3 + 2 * rq, J4 = J3 + 2 * (r - rq * nd);
        bool ok = s0 + lane < nslot && J4 <= 2 * JM && J3 + J4 >= R && J4 >= ((p.flags >> 6) & 4095) &&
                  J4 <= (p.flags >> 18) && (k < 8 || J4 != J3);
        CcBlk bk{-1, 0, 0};
        if (ok) bk = T.cblk[((p.flags & 3) * nJ + (J3 >> 1)) * nd + ((J4 - J3) >> 1)];
        ok = ok && bk.wo >= 0;
        const unsigned long long m = __ballot(ok);
        if (ok) {
          PhSeg g;
          // Wx carries LCC%herm (TS_commutators.f90:1506)
          g.c = (k < 8 ? p.cs * hL : p.cs) * ((p.flags & 32) ? (double)sgnp((J3 + J4) >> 1) : 1.0) *
                sqrt((J3 + 1.0) * (J4 + 1.0));
          g.w = (bk.wo + (k < 8 ? 0 : wsize)) << 24 | bk.rl4;
          g.b9 = ((p.b9 * nJ + (J3 >> 1)) * nd + ((J4 - J3) >> 1)) * (unsigned)(nJ * nd) |
                 (unsigned)((p.flags >> 3) & 3) << 30;
          g.code = (unsigned)k | (unsigned)(J3 >> 1) << 4 | (unsigned)(J4 >> 1) << 12;
          seg[nseg + __popcll(m & ((1ull << lane) - 1ull))] = g;
        }
        nseg += __popcll(m);
        s0 += 64;
      }
      __syncthreads();
      // 2: the entries of the first kPhB
      const int nb = min(nseg, kPhB);
      if (nb == 0) break;  // the scan found no further slot: there is none to read below
      int count = 0;
      {
        double w[4];
        int ix[4], jx[4];
        auto slot = [&](int u) -> const PhSeg & { return seg[min(8 * u + (lane >> 3), nb - 1)]; };
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const unsigned gc = slot(u).code;
          const int kk = gc & 15;
          const ushort2 bs = base[kk][quad];
          ix[u] = T.crow[bs.x * nJ + (int)((gc >> 4) & 255)];
          jx[u] = T.cpos[bs.y * nJ + (int)(gc >> 12)];
          // the branch condition of the reference
          if (8 * u + (lane >> 3) >= nb || quad >= nq || ((kPhCond >> (2 * kk)) & drop)) jx[u] = -1;
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          w[u] = 0.0;
          const long long gw = slot(u).w;
          if ((ix[u] | jx[u]) >= 0) w[u] = W[(gw >> 24) + (long long)ix[u] * (int)(gw & 0xffffff) + jx[u]];
        }
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const bool live = fabs(w[u]) > thr;
          // one bit per slot of 8 lanes: some quadruple's entry passes
          unsigned long long m = __ballot(live);
          m |= m >> 4;
          m |= m >> 2;
          m |= m >> 1;
          m &= 0x0101010101010101ull;
          const int sub8 = lane & 56;
          if ((m >> sub8) & 1) {
            const int pos = count + __popcll(m & ((1ull << sub8) - 1ull));
            cs[pos][quad] = live ? slot(u).c * w[u] : 0.0;
            if (quad == 0) sb9[pos] = slot(u).b9;
          }
          count += __popcll(m);
        }
      }
      if (lane < kPhQ) cs[count][lane] = 0.0;  // what the last round reads past the end
      if (lane == kPhQ) sb9[count] = 0;
      // the slots that wait move to the front
      nseg -= nb;
      const double mc = seg[kPhB + lane].c;
      const long long mw = seg[kPhB + lane].w;
      const unsigned mb = seg[kPhB + lane].b9, mo = seg[kPhB + lane].code;
      __syncthreads();
      if (lane < nseg) {
        seg[lane].c = mc;
        seg[lane].w = mw;
        seg[lane].b9 = mb;
        seg[lane].code = mo;
      }
      rc.add(n9, cs, sb9, count);  // 3
      __syncthreads();
    }
    // each group writes its share of the quadruples, with one add per element
    // and no wait for the old value
    int q0, nown;
    bool mine;
    rc.reduce(lane, q0, nown, mine);
    const int oq0 = div(ol), oq1 = div(ol + 1);
    const int J1o[2] = {Jlo + 2 * oq0, Jlo + 2 * oq1};
    const int J2o[2] = {J1o[0] + 2 * (ol - oq0 * nd), J1o[1] + 2 * (ol + 1 - oq1 * nd)};
    OutBlk ob[2];
    double nrm[2];
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int J1 = J1o[u], J2 = J2o[u];
      const bool val = mine && ol + u < nout && ol + u < o0 + 128 && J2 >= abs(j2 - j3) && J2 <= j2 + j3 && J1 + J2 >= R;
      ob[u] = T.oblk[val ? (((J1 >> 1) * nd + ((J2 - J1) >> 1)) * 6 + Tzq * 2 + P1) : 0];
      if (!val) ob[u].off = -1;
      nrm[u] = sqrt((J1 + 1.0) * (J2 + 1.0));
    }
#pragma unroll
    for (int i = 0; i < kPhQ; i++) {
      if (i >= nown) break;
      const unsigned cd = (unsigned)__shfl((int)code, q0 + i);
      const int x0 = cd & 255, x1 = (cd >> 8) & 255, x2 = (cd >> 16) & 255, x3 = (int)(cd >> 24);
      const int *p1 = T.prow + (x0 * n + x1) * nJ, *p2 = T.prow + (x2 * n + x3) * nJ;
      const double f = (x0 == x1 ? M_SQRT2 : 1.0) * (x2 == x3 ? M_SQRT2 : 1.0);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int e1 = J1o[u] >> 1, e2 = J2o[u] >> 1;
        if (q0 + i < nq && ob[u].off >= 0 && !(x0 == x1 && (e1 & 1)) && !(x2 == x3 && (e2 & 1))) {
          const int r = p1[e1], sc = p2[e2];
          if ((r | sc) >= 0)
            unsafeAtomicAdd(OV + ob[u].off + (long long)r * ob[u].n2 + sc, rc.acc[i][u] * nrm[u] * f);
        }
      }
    }
  }
}

// ---------------------------------------------------------------- products
// 64 x 64 tiles, 4 waves of 32 x 32 on v_mfma_f64_16x16x4; tiles (problem, tile row, tile column).
// Matrix-core bound in large bases (59 TF/s over a commutator's products at 90
// orbits, rank 4).  The pp and hh ladders of a tile in one workgroup: the hh
// product's short K follows the pp product's without a launch, and RES takes
// their difference here, not in two more passes over three operators.
__global__ __launch_bounds__(256) void k_tgemm(const TProb *__restrict__ probs, const int4 *__restrict__ tiles,
                                               int ntiles, TGemm X) {
  const int t = blockIdx.x;
  if (t >= ntiles) return;
  const int4 tl = tiles[t];
  const TProb &p = probs[tl.x];
  const int m0 = tl.y * 64, n0 = tl.z * 64;
  __shared__ double As[16][65], Bs[16][65];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave >> 1, wn = wave & 1;
  double4_t acc[2][2];
  for (int i = 0; i < 2; i++)
    for (int j = 0; j < 2; j++) acc[i][j] = (double4_t){0.0, 0.0, 0.0, 0.0};
  // each thread stages 4 elements of A and 4 of B per K step of 16; the next
  // step's elements are loaded into registers (clamped to the operand, so
  // every load is unconditional and the eight stay in flight together) while
  // the current step runs on the matrix cores
  // v_mfma_f64_16x16x4: row lane/16 + 4v, column lane%16; W2 - W1 needs W1 again, which
  // this thread wrote
  auto store = [&](double *C, bool diff) {
    for (int ti = 0; ti < 2; ti++)
      for (int tj = 0; tj < 2; tj++)
        for (int v = 0; v < 4; v++) {
          const int row = m0 + wm * 32 + ti * 16 + (lane >> 4) + 4 * v, col = n0 + wn * 32 + tj * 16 + (lane & 15);
          if (row >= p.M || col >= p.N) continue;
          const long long o = p.c_off + (long long)row * p.ldc + col;
          C[o] = acc[ti][tj][v];
          if (diff) X.res[o] += X.c[p.c][o] - acc[ti][tj][v];
          acc[ti][tj][v] = 0.0;
        }
  };
  for (int sgi = 0; sgi < p.nseg + p.nseg2; sgi++) {
    if (sgi == p.nseg) store(X.c[p.c], false);
    const TSeg sg = p.seg[sgi];
    if (sg.K <= 0) continue;
    const double *Ap = X.x[sg.asrc] + sg.a_off, *Bp = X.x[sg.bsrc] + sg.b_off;
    const bool arow = sg.a_cs == 1, brow = sg.b_cs == 1;
    int am[4], ak[4], bn[4], bk[4];  // element (row/column, k) of each staged value in the tile
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const int e = tid + 256 * u;
      am[u] = arow ? e >> 4 : e & 63;
      ak[u] = arow ? e & 15 : e >> 6;
      bn[u] = brow ? e & 63 : e >> 4;
      bk[u] = brow ? e >> 6 : e & 15;
    }
    double ra[4], rb[4];
    auto gload = [&](int k0) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int m = min(m0 + am[u], p.M - 1), k = min(k0 + ak[u], sg.K - 1);
        const int n = min(n0 + bn[u], p.N - 1), k2 = min(k0 + bk[u], sg.K - 1);
        ra[u] = Ap[(long long)m * sg.a_rs + (long long)k * sg.a_cs];
        rb[u] = Bp[(long long)k2 * sg.b_rs + (long long)n * sg.b_cs];
      }
    };
    gload(0);
    for (int k0 = 0; k0 < sg.K; k0 += 16) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        As[ak[u]][am[u]] = (m0 + am[u] < p.M && k0 + ak[u] < sg.K) ? sg.alpha * ra[u] : 0.0;
        Bs[bk[u]][bn[u]] = (n0 + bn[u] < p.N && k0 + bk[u] < sg.K) ? rb[u] : 0.0;
      }
      __syncthreads();
      gload(k0 + 16);  // past the end: clamped reloads, never used
#pragma unroll
      for (int kq = 0; kq < 4; kq++) {
        const int k = kq * 4 + (lane >> 4);
        const double a0 = As[k][wm * 32 + (lane & 15)], a1 = As[k][wm * 32 + 16 + (lane & 15)];
        const double b0 = Bs[k][wn * 32 + (lane & 15)], b1 = Bs[k][wn * 32 + 16 + (lane & 15)];
        acc[0][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, acc[0][0], 0, 0, 0);
        acc[0][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b1, acc[0][1], 0, 0, 0);
        acc[1][0] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b0, acc[1][0], 0, 0, 0);
        acc[1][1] = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, b1, acc[1][1], 0, 0, 0);
      }
      __syncthreads();
    }
  }
  store(p.nseg2 ? X.c[1] : X.c[p.c], p.nseg2 && X.res);
}

// One term of BCH_TENSOR's series and its norm: HS += coef X (HS null: the norm
// only), and mat_frob_norm of X (basic_IMSRG.f90:3921-3952): fhh^2 + 2 fph^2 +
// fpp^2 + sum over blocks (1 if J1 = J2, else 2) x block^2.  A workgroup per
// run of one block's elements; k_t_norm adds the runs' sums and writes the result
// to host memory, where the host waits for it.
struct TRun {
  long long off;  // into the operator
  int n, w;       // elements, weight; w 0: the one-body matrix
};
struct TNorm {
  double v;
  int seq;
};
__global__ __launch_bounds__(256) void k_t_step(DevLayout L, const TRun *__restrict__ runs,
                                                const double *__restrict__ X, double *__restrict__ HS, double coef,
                                                double *__restrict__ part) {
  __shared__ double sh[256];
  const TRun r = runs[blockIdx.x];
  double s = 0.0;
  if (r.w) {
#pragma unroll 4
    for (int e = threadIdx.x; e < r.n; e += 256) {
      const double v = X[r.off + e];
      if (HS) HS[r.off + e] += coef * v;
      s += v * v;
    }
    s *= r.w;
  } else {
    for (int e = threadIdx.x; e < r.n; e += 256) {
      const double v = X[r.off + e];
      const int a = e / L.nsp, b = e % L.nsp;
      if (HS) HS[r.off + e] += coef * v;
      if (L.con[a] == L.con[b]) s += v * v;
      else if (L.con[a] == 0) s += 2.0 * v * v;  // (particle, hole); (hole, particle) is derived
    }
  }
  s = block_sum256(s, sh);
  if (threadIdx.x == 0) part[blockIdx.x] = s;
}
__global__ __launch_bounds__(256) void k_t_norm(const double *__restrict__ part, int n, TNorm *out, int seq) {
  __shared__ double sh[256];
  double s = 0.0;
  for (int k = threadIdx.x; k < n; k += 256) s += part[k];
  s = block_sum256(s, sh);
  if (threadIdx.x == 0) {
    out->v = s;
    __threadfence_system();
    __hip_atomic_store(&out->seq, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
  }
}

}  // namespace

// ---------------------------------------------------------------- host side
struct TensorSpace {
  int rank = 0, dpar = 0, nblk = 0, ncc = 0, hx = 0;
  std::vector<int> J1, J2, q1, q2, n1, n2, bidx;
  std::vector<long long> off;
  long long vsize = 0, v_off = 0, op_size = 0, neq = 0, nelem = 0;
  std::vector<int> cJ3, cJ4, cq3, cq4, ccol;
  std::vector<long long> xoff, roff, woff;
  long long xsize = 0, rsize = 0, wsize = 0;
  std::vector<double> x6, s6;
  long long n9size = 0;
  PackTables pack{};
  double *pack_d = nullptr;
  DevTensor dt{};
  TLists lists{};
  TPan pan[2]{};  // CCX, CCR
  double *gcc = nullptr, *gccp = nullptr, *ccx = nullptr, *ccr = nullptr, *wx = nullptr, *wy = nullptr;
  double *w1 = nullptr, *w2 = nullptr, *part = nullptr;
  const TRun *runs = nullptr;
  int nrun = 0, seq = 0;
  TNorm *norm = nullptr;   // host memory
  OpPool bch;              // BCH_TENSOR's two work operators, in one buffer, kept up to kBchKeep bytes
  const TProb *pp_probs = nullptr, *cc_probs = nullptr;
  const int4 *pp_tiles = nullptr, *cc_tiles = nullptr;
  int n_pp_tiles = 0, n_cc_tiles = 0;
  ~TensorSpace() {
    if (norm) (void)hipHostFree(norm);
  }
};

struct imsrg_tensor_s {
  imsrg_ctx_s *ctx = nullptr;
  TensorSpace *ts = nullptr;
  double *d = nullptr;
  int herm = 1;
};

static long long align32(long long x) { return (x + 31) & ~31LL; }

static void add_tiles(int pi, int M, int N, std::vector<int4> &tiles) {
  for (int i = 0; i < (M + 63) / 64; i++)
    for (int j = 0; j < (N + 63) / 64; j++) tiles.push_back(make_int4(pi, i, j, 0));
}

static int tspace_build(imsrg_ctx_s *c, int rank, int dpar, TensorSpace &S) {
  const Layout &Ly = c->lay;
  const int JM = Ly.jtot_max, nJ = Ly.nJ, nsp = Ly.nsp, nh = Ly.nhalf;
  S.rank = rank;
  S.dpar = dpar;
  const int dp = (dpar >> 1) & 1;
  // tensor blocks, allocate_tensor's order (basic_IMSRG.f90:690-770)
  S.bidx.assign((size_t)nJ * nJ * 6, -1);
  long long off = 0, el = 0;
  for (int J1 = 0; J1 <= 2 * JM; J1 += 2)
    for (int J2 = std::max(std::abs(J1 - rank), J1); J2 <= J1 + rank; J2 += 2)
      for (int Tz = -1; Tz <= 1; Tz++)
        for (int P1 = 0; P1 <= 1; P1++) {
          const int q = (int)S.J1.size();
          const bool live = J2 <= 2 * JM;
          const int b1 = live ? 3 * J1 + 2 * (Tz + 1) + P1 : -1;
          const int b2 = live ? 3 * J2 + 2 * (Tz + 1) + (P1 ^ dp) : -1;
          S.J1.push_back(J1);
          S.J2.push_back(J2);
          S.q1.push_back(b1);
          S.q2.push_back(b2);
          const int m1 = live ? Ly.bdim[b1] : 0, m2 = live ? Ly.bdim[b2] : 0;
          S.n1.push_back(m1);
          S.n2.push_back(m2);
          S.off.push_back(off);
          off = align32(off + (long long)m1 * m2);
          el += (long long)m1 * m2;
          if (live) S.bidx[((size_t)(J1 >> 1) * nJ + (J2 >> 1)) * 6 + (Tz + 1) * 2 + P1] = q;
        }
  S.nblk = (int)S.J1.size();
  S.nelem = el;
  S.vsize = off;
  S.v_off = align32(Ly.f_off + (long long)nsp * nsp);
  S.op_size = S.v_off + S.vsize;
  S.neq = 1 + (long long)Ly.nhole * Ly.nhole + (long long)Ly.npart * Ly.npart + (long long)Ly.npart * Ly.nhole + el;
  // cross-coupled tensor blocks (allocate_small_tensor_CCMAT, cross_coupled.f90:498-700):
  // J3, J4 >= J3 within rank, |Tz|, parity of the J3 pairs
  long long xo = 0, ro = 0, wo = 0;
  for (int J3 = 0; J3 <= 2 * JM; J3 += 2)
    for (int J4 = std::max(std::abs(J3 - rank), J3); J4 <= std::min(J3 + rank, 2 * JM); J4 += 2)
      for (int Tz = 0; Tz <= 1; Tz++)
        for (int P = 0; P <= 1; P++) {
          const int q3 = (J3 >> 1) + Tz * (JM + 1) + 2 * P * (JM + 1);
          const int q4 = (J4 >> 1) + Tz * (JM + 1) + 2 * (P ^ dp) * (JM + 1);
          S.cJ3.push_back(J3);
          S.cJ4.push_back(J4);
          S.cq3.push_back(q3);
          S.cq4.push_back(q4);
          const long long r3 = Ly.ccrlen[q3], r4 = Ly.ccrlen[q4], nb3 = Ly.ccnph[q3], nb4 = Ly.ccnph[q4];
          S.xoff.push_back(xo);
          S.roff.push_back(ro);
          S.woff.push_back(wo);
          xo = align32(xo + r3 * nb4);
          ro = align32(ro + nb3 * r4);
          wo = align32(wo + r3 * r4);
        }
  S.ncc = (int)S.cJ3.size();
  S.xsize = xo;
  S.rsize = ro;
  S.wsize = wo;
  // column of (p,h) inside each scalar Pandya block
  S.ccol.assign((size_t)Ly.ncc * nsp * nsp, -1);
  for (int q = 0; q < Ly.ncc; q++)
    for (int k = Ly.cccbase[q]; k < Ly.cccbase[q + 1]; k++)
      S.ccol[((size_t)q * nsp + Ly.cccol_p[k]) * nsp + Ly.cccol_h[k]] = k - Ly.cccbase[q];
  // 6j tables of the tensor terms (xxxsixj, store_6j_3halfint, basic_IMSRG.f90:2291-2370, 2558-2595)
  S.hx = (JM + rank + 1) / 2;
  const int hx = S.hx;
  S.x6.assign((size_t)nJ * nJ * hx * nh * nh, 0.0);
  for (int a1 = 0; a1 < nJ; a1++)
    for (int a2 = 0; a2 < nJ; a2++) {
      if (!(2 * a2 <= 2 * a1 + rank && 2 * a2 >= std::abs(2 * a1 - rank))) continue;
      for (int i4 = 0; i4 < hx; i4++)
        for (int i5 = 0; i5 < nh; i5++)
          for (int i6 = 0; i6 < nh; i6++)
            S.x6[((((size_t)a1 * nJ + a2) * hx + i4) * nh + i5) * nh + i6] =
                racah6j(2 * a1, 2 * a2, rank, 2 * i4 + 1, 2 * i5 + 1, 2 * i6 + 1);
    }
  S.s6.assign((size_t)nh * nh * nJ * nh * hx * nJ, 0.0);
  for (int i1 = 0; i1 < nh; i1++)
    for (int i2 = 0; i2 < nh; i2++)
      for (int a3 = 0; a3 < nJ; a3++) {
        if (!(2 * a3 <= 2 * i1 + 1 + 2 * i2 + 1 && 2 * a3 >= std::abs(2 * i1 - 2 * i2))) continue;
        for (int i4 = 0; i4 < nh; i4++)
          for (int i5 = 0; i5 < hx; i5++)
            for (int a6 = 0; a6 < nJ; a6++)
              S.s6[(((((size_t)i1 * nh + i2) * nJ + a3) * nh + i4) * hx + i5) * nJ + a6] =
                  racah6j(2 * i1 + 1, 2 * i2 + 1, 2 * a3, 2 * i4 + 1, 2 * i5 + 1, 2 * a6);
      }
  // device tables
  DevTensor &D = S.dt;
  D.rank = rank; D.dpar = dpar; D.nblk = S.nblk; D.ncc = S.ncc; D.nJ = nJ; D.nh = nh; D.hx = hx;
  D.nhole = Ly.nhole; D.npart = Ly.npart; D.nelem = S.nelem;
  D.f_off = Ly.f_off; D.v_off = S.v_off;
#define TUP(vec, field) \
  if (upload_table(c, vec, &D.field) != 0) return IMSRG_ENOMEM
  TUP(Ly.holes, holes); TUP(Ly.parts, parts);
  TUP(S.J1, J1); TUP(S.J2, J2); TUP(S.q1, q1); TUP(S.q2, q2); TUP(S.n1, n1); TUP(S.n2, n2);
  TUP(S.off, off); TUP(S.bidx, bidx);
  TUP(S.ccol, ccol); TUP(S.x6, x6); TUP(S.s6, s6);
  std::vector<int> rperm, rpos;  // Pandya rows in group order, and each row's place in it
  {
    rperm.resize(Ly.ccrbase[Ly.ncc]);
    rpos.resize(Ly.ccrbase[Ly.ncc]);
    for (int q = 0; q < Ly.ncc; q++) {
      const int r0 = Ly.ccrbase[q], nr = Ly.ccrlen[q];
      std::vector<int> ix(nr);
      auto rkey = [&](int g) {
        const int a = Ly.ccrow_a[r0 + g], b = Ly.ccrow_b[r0 + g];
        return a < 0 ? std::make_pair(1 << 20, 0) : std::make_pair(Ly.grp_of[a], Ly.grp_of[b]);
      };
      for (int g = 0; g < nr; g++) ix[g] = g;
      std::stable_sort(ix.begin(), ix.end(), [&](int x, int y) {
        const auto kx = rkey(x), ky = rkey(y);
        if (kx != ky) return kx < ky;
        return std::make_pair(Ly.ccrow_a[r0 + x], Ly.ccrow_b[r0 + x]) <
               std::make_pair(Ly.ccrow_a[r0 + y], Ly.ccrow_b[r0 + y]);
      });
      std::copy(ix.begin(), ix.end(), rperm.begin() + r0);
      for (int i = 0; i < nr; i++) rpos[r0 + ix[i]] = i;
    }
    TUP(rperm, rperm);
  }
  std::vector<int> pstart_h, part_h;  // the orbits the tensor's one-body part couples
  {
    std::vector<int> &ps = pstart_h, &pl = part_h;
    ps.assign(nsp + 1, 0);
    for (int x = 0; x < nsp; x++) {
      ps[x] = (int)pl.size();
      for (int i = 0; i < nsp; i++)
        if (Ly.tz[i] == Ly.tz[x] && ((Ly.l[i] + dp) & 1) == (Ly.l[x] & 1) && std::abs(Ly.jj[i] - Ly.jj[x]) <= rank &&
            rank <= Ly.jj[i] + Ly.jj[x])
          pl.push_back(i | Ly.jj[i] << 8);
    }
    ps[nsp] = (int)pl.size();
    if (pl.empty()) pl.push_back(0);  // a readable entry for the clamped loads
    TUP(ps, pstart);
    TUP(pl, part);
  }
#undef TUP
  // 9j table of the recoupling and the tensor Pandya transform (up to 4 GiB:
  // rank 2 to emax=14, rank 3 to emax=12)
  D.nd = rank / 2 + 1;
  {
    const long long n9 = (long long)nh * nh * nh * nh * nJ * nJ * D.nd * D.nd;
    if (n9 > (1LL << 29)) return fail(IMSRG_EINVAL, "tensor rank too large for the 9j table at this basis");
    double *t9 = nullptr;
    if (dalloc(c, n9 + kN9Pad, &t9)) return IMSRG_ENOMEM;
    launch_fill(c->stream, t9 + n9, kN9Pad, 0.0);
    hipLaunchKernelGGL(k_fill9j, dim3((unsigned)((n9 + 255) / 256)), dim3(256), 0, c->stream, D, t9, n9);
    D.n9 = t9;
    S.n9size = n9;
  }
  // orbit quadruples of the recoupling gather (k_t222ph): row pair x0 <= x1,
  // column pair x2 <= x3, with at least one stored output (orbits packed in 8
  // bits), by the (l,j,tz) groups of the four orbits
  if (nsp > 256) return fail(IMSRG_EINVAL, "tensor operators need at most 256 orbits");
  {
    std::vector<unsigned> quads;
    std::vector<PhChunkT> chunks;
    const int ng = (int)Ly.grp_start.size();
    auto orbits = [&](int g, int &cnt) {
      cnt = Ly.grp_cnt[g];
      return Ly.grp_list.data() + Ly.grp_start[g];
    };
    for (int g0 = 0; g0 < ng; g0++)
      for (int g1 = 0; g1 < ng; g1++) {
        int c0, c1;
        const int *o0 = orbits(g0, c0), *o1 = orbits(g1, c1);
        std::vector<std::pair<int, int>> bra;
        for (int i = 0; i < c0; i++)
          for (int j = 0; j < c1; j++)
            if (o0[i] <= o1[j]) bra.push_back({o0[i], o1[j]});
        if (bra.empty()) continue;
        const int y0 = o0[0], y1 = o1[0], j0 = Ly.jj[y0], j1 = Ly.jj[y1];
        const int t1 = Ly.tz[y0] + Ly.tz[y1], p1 = (Ly.l[y0] + Ly.l[y1]) & 1;
        for (int g2 = 0; g2 < ng; g2++)
          for (int g3 = 0; g3 < ng; g3++) {
            int c2, c3;
            const int *o2 = orbits(g2, c2), *o3 = orbits(g3, c3);
            if (Ly.tz[o2[0]] + Ly.tz[o3[0]] != t1 || ((Ly.l[o2[0]] + Ly.l[o3[0]]) & 1) != (p1 ^ dp)) continue;
            const int j2 = Ly.jj[o2[0]], j3 = Ly.jj[o3[0]];
            bool any[4] = {false, false, false, false};  // [x0 == x1][x2 == x3]
            for (int J1 = std::abs(j0 - j1); J1 <= j0 + j1; J1 += 2)
              for (int J2 = std::max(J1, std::abs(j2 - j3)); J2 <= std::min(j2 + j3, J1 + rank); J2 += 2)
                if (J1 + J2 >= rank)
                  for (int k = 0; k < 4; k++)
                    any[k] |= !((k & 2) && ((J1 >> 1) & 1)) && !((k & 1) && ((J2 >> 1) & 1));
            if (!any[0]) continue;
            const size_t first = quads.size();
            for (const auto &x : bra)
              for (int i = 0; i < c2; i++)
                for (int j = 0; j < c3; j++)
                  if (o2[i] <= o3[j] && any[(x.first == x.second) * 2 + (o2[i] == o3[j])])
                    quads.push_back((unsigned)x.first | (unsigned)x.second << 8 | (unsigned)o2[i] << 16 |
                                    (unsigned)o3[j] << 24);
            unsigned lt = 0;
            const int ys[4] = {y0, y1, o2[0], o3[0]};
            for (int i = 0; i < 4; i++) lt |= (unsigned)(Ly.l[ys[i]] & 1) << i | (unsigned)(Ly.tz[ys[i]] > 0) << (4 + i);
            const unsigned jv = (unsigned)j0 | (unsigned)j1 << 8 | (unsigned)j2 << 16 | (unsigned)j3 << 24;
            for (size_t k = first; k < quads.size(); k += kPhQ)
              chunks.push_back(PhChunkT{(unsigned)k, jv, lt, (int)std::min<size_t>(kPhQ, quads.size() - k)});
          }
      }
    if (quads.empty()) quads.push_back(0);
    D.nqchunk = (int)chunks.size();
    D.nqpad = (D.nqchunk + 511) & ~511;
    if (chunks.empty()) chunks.push_back(PhChunkT{0, 0, 0, 1});
    if (upload_table(c, quads, &D.quads) != 0 || upload_table(c, chunks, &D.qchunk) != 0) return IMSRG_ENOMEM;
    // rows by pair, J fastest
    std::vector<int> crow((size_t)nsp * nsp * nJ, -1), cpos(crow), prow(crow);
    for (int a = 0; a < nsp; a++)
      for (int b = 0; b < nsp; b++)
        for (int J = 0; J < nJ; J++) {
          const int Tz = std::abs(Ly.tz[a] - Ly.tz[b]) >> 1, P = (Ly.l[a] + Ly.l[b]) & 1;
          const int q = J + Tz * (JM + 1) + 2 * P * (JM + 1);
          const int r = Ly.ccrow[((size_t)q * nsp + a) * nsp + b];
          crow[((size_t)a * nsp + b) * nJ + J] = r;
          if (r >= 0) cpos[((size_t)a * nsp + b) * nJ + J] = rpos[Ly.ccrbase[q] + r];
          prow[((size_t)a * nsp + b) * nJ + J] = Ly.pidx[((size_t)J * nsp + a) * nsp + b];
        }
    std::vector<CcBlk> cblk((size_t)4 * nJ * D.nd, CcBlk{-1, 0, 0});
    for (int x = 0; x < S.ncc; x++) {
      const int q3 = S.cq3[x], Tz = (q3 / (JM + 1)) & 1, P = q3 / (2 * (JM + 1));
      cblk[((size_t)(Tz + 2 * P) * nJ + (S.cJ3[x] >> 1)) * D.nd + ((S.cJ4[x] - S.cJ3[x]) >> 1)] =
          CcBlk{S.woff[x], Ly.ccrlen[S.cq4[x]], 0};
    }
    std::vector<OutBlk> oblk((size_t)6 * nJ * D.nd, OutBlk{-1, 0, 0});
    for (int q = 0; q < S.nblk; q++)
      if (S.q1[q] >= 0)
        oblk[((size_t)(S.J1[q] >> 1) * D.nd + ((S.J2[q] - S.J1[q]) >> 1)) * 6 + S.q1[q] % 6] = OutBlk{S.off[q], S.n2[q], 0};
    if (upload_table(c, oblk, &D.oblk) != 0) return IMSRG_ENOMEM;
    if (upload_table(c, crow, &D.crow) != 0 || upload_table(c, cpos, &D.cpos) != 0 || upload_table(c, prow, &D.prow) != 0 ||
        upload_table(c, cblk, &D.cblk) != 0)
      return IMSRG_ENOMEM;
  }
  // quadruples of the tensor Pandya matrices, by class: (u,v,x,y) = (a,h,b,p)
  // of CCX, (h,a,p,b) of CCR, h a hole, p a particle, a and b any
  {
    const int ng = (int)Ly.grp_start.size();
    std::vector<std::vector<int>> of[3];  // a group's orbits, holes, particles
    for (auto &o : of) o.resize(ng);
    for (int g = 0; g < ng; g++)
      for (int k = 0; k < Ly.grp_cnt[g]; k++) {
        const int x = Ly.grp_list[Ly.grp_start[g] + k];
        of[0][g].push_back(x);
        of[Ly.con[x] ? 1 : 2][g].push_back(x);
      }
    auto gj = [&](int g) { return Ly.jj[Ly.grp_list[Ly.grp_start[g]]]; };
    auto gl = [&](int g) { return Ly.l[Ly.grp_list[Ly.grp_start[g]]] & 1; };
    auto gt = [&](int g) { return Ly.tz[Ly.grp_list[Ly.grp_start[g]]] > 0 ? 1 : 0; };
    std::vector<int> pcol((size_t)nsp * nsp * nJ, -1);
    for (int q = 0; q < Ly.ncc; q++)
      for (int k = Ly.cccbase[q]; k < Ly.cccbase[q + 1]; k++)
        pcol[((size_t)Ly.cccol_p[k] * nsp + Ly.cccol_h[k]) * nJ + Ly.ccJ[q] / 2] = k - Ly.cccbase[q];
    const int *dpcol = nullptr;
    if (upload_table(c, pcol, &dpcol) != 0) return IMSRG_ENOMEM;
    for (int mode = 0; mode < 2; mode++) {
      TPan &P = S.pan[mode];
      const auto &fu = of[mode ? 1 : 0], &fv = of[mode ? 0 : 1], &fx = of[mode ? 2 : 0], &fy = of[mode ? 0 : 2];
      std::vector<unsigned> quads;
      std::vector<PhChunkT> chunks;
      for (int u = 0; u < ng; u++)
        for (int v = 0; v < ng; v++) {
          if (fu[u].empty() || fv[v].empty()) continue;
          for (int x = 0; x < ng; x++)
            for (int y = 0; y < ng; y++) {
              if (fx[x].empty() || fy[y].empty()) continue;
              if ((gl(u) ^ gl(v)) != (gl(x) ^ gl(y) ^ dp) || gt(u) + gt(v) != gt(x) + gt(y)) continue;
              const int ju = gj(u), jv = gj(v), jx = gj(x), jy = gj(y);
              bool any = false;  // some (J3 of (u,x), J4 of (v,y)) with a block
              for (int J3 = std::abs(ju - jx); J3 <= ju + jx && !any; J3 += 2)
                for (int J4 = std::max(J3, std::abs(jv - jy)); J4 <= std::min(jv + jy, J3 + rank); J4 += 2)
                  any |= J3 + J4 >= rank;
              if (!any) continue;
              const size_t first = quads.size();
              for (int a : fu[u])
                for (int b : fv[v])
                  for (int e : fx[x])
                    for (int f : fy[y])
                      quads.push_back((unsigned)a | (unsigned)b << 8 | (unsigned)e << 16 | (unsigned)f << 24);
              const unsigned jc = (unsigned)ju | (unsigned)jv << 8 | (unsigned)jx << 16 | (unsigned)jy << 24;
              const unsigned lt = (unsigned)(gl(u) | gl(v) << 1 | gl(x) << 2 | gl(y) << 3 | gt(u) << 4 | gt(v) << 5 |
                                             gt(x) << 6 | gt(y) << 7);
              for (size_t k = first; k < quads.size(); k += kPhQ)
                chunks.push_back(PhChunkT{(unsigned)k, jc, lt, (int)std::min<size_t>(kPhQ, quads.size() - k)});
            }
        }
      P.nchunk = (int)chunks.size();
      P.npad = (P.nchunk + 511) & ~511;
      if (chunks.empty()) continue;
      // the matrices by (Tz, parity) of the J3 pair and (J3, J4)
      std::vector<CcBlk> blk((size_t)4 * nJ * D.nd, CcBlk{-1, 0, 0});
      for (int i = 0; i < S.ncc; i++) {
        const int q3 = S.cq3[i], Tz = (q3 / (JM + 1)) & 1, Pr = q3 / (2 * (JM + 1));
        blk[((size_t)(Tz + 2 * Pr) * nJ + (S.cJ3[i] >> 1)) * D.nd + ((S.cJ4[i] - S.cJ3[i]) >> 1)] =
            mode ? CcBlk{S.roff[i], Ly.ccrlen[S.cq4[i]], 0} : CcBlk{S.xoff[i], Ly.ccnph[S.cq4[i]], 0};
      }
      if (upload_table(c, quads, &P.quads) != 0 || upload_table(c, chunks, &P.chunks) != 0 ||
          upload_table(c, blk, &P.blk) != 0)
        return IMSRG_ENOMEM;
      P.rtab = mode ? dpcol : D.crow;
      P.ctab = mode ? D.cpos : dpcol;
    }
  }
  // lists and work items of k_t_lists, k_t_1body
  {
    std::vector<TList> lists;
    std::vector<TItem> items;
    std::vector<TSlice> groups, cols;
    std::vector<int> cbase(S.nblk, 0), grow, rsrc, rdst;
    std::vector<unsigned short> cp;
    std::vector<long long> cost(S.nblk, 0);
    unsigned lds = 0;
    int maxdim = 1;
    for (int q = 0; q < Ly.nblocks; q++) maxdim = std::max(maxdim, Ly.bdim[q]);
    // the partner pairs of pair p (block of J1 for side 0, of J2 for side 1), in
    // k_t_lists' order: its position in T's block or (g) in G's, or -1
    auto partners = [&](int p, int side, int J1, int J2, auto &&put) {
      const int a = Ly.pair_a[p], b = Ly.pair_b[p];
      auto pos = [&](int i, int o, int J) {
        return Ly.pidx[((size_t)(J >> 1) * nsp + std::min(i, o)) * nsp + std::max(i, o)];
      };
      int e = 0;
      for (int w = 0; w < 2; w++) {
        const int x = w ? b : a, o = w ? a : b, g = Ly.grp_of[x], J = side ? J2 : J1;
        const bool tri = J <= Ly.jj[x] + Ly.jj[o] && J >= std::abs(Ly.jj[x] - Ly.jj[o]);
        for (int k = 0; k < Ly.grp_cnt[g]; k++)
          put(e++, w, false, tri ? pos(Ly.grp_list[Ly.grp_start[g] + k], o, J) : -1);
      }
      for (int w = 0; w < 2; w++) {
        const int x = w ? b : a, o = w ? a : b;
        for (int k = pstart_h[x]; k < pstart_h[x + 1]; k++) put(e++, w, true, pos(part_h[k] & 255, o, side ? J1 : J2));
      }
      return e;
    };
    std::vector<int> seen(4 * (size_t)maxdim, -1), slot(4 * (size_t)maxdim), ix;
    for (int q = 0; q < S.nblk; q++) {
      const int m1 = S.n1[q], m2 = S.n2[q];
      if (m1 == 0 || m2 == 0) continue;
      const int b1 = S.q1[q], p1 = Ly.pbase[b1], p2 = Ly.pbase[S.q2[q]], J1 = S.J1[q], J2 = S.J2[q];
      const long long ld = (m2 + Ly.bdim[b1]) | 1;
      // rows in class order, in groups of up to eight (fewer where eight rows
      // take more than half of the LDS): whole classes, or parts of one
      const int cap = (int)std::max<long long>(1, std::min<long long>(8, 9000 / ld));
      auto key = [&](int r) { return std::make_pair(Ly.grp_of[Ly.pair_a[p1 + r]], Ly.grp_of[Ly.pair_b[p1 + r]]); };
      ix.resize(m1);
      for (int r = 0; r < m1; r++) ix[r] = r;
      std::stable_sort(ix.begin(), ix.end(), [&](int x, int y) { return key(x) < key(y); });
      const int gfirst = (int)groups.size();
      std::vector<int> gsize;
      for (int r = 0; r < m1;) {
        int n = 0;
        while (r + n < m1 && n < cap) {
          int m = 1;  // the next class
          while (r + n + m < m1 && key(ix[r + n + m]) == key(ix[r + n])) m++;
          if (n > 0 && n + m > cap) break;
          n += std::min(m, cap - n);
        }
        const int gid = (int)groups.size();
        const long long base = (long long)rsrc.size();
        for (int j = 0; j < 8; j++) grow.push_back(ix[r + std::min(j, n - 1)]);
        grow.back() |= n << 24;
        for (int j = 0; j < n; j++) {
          lists.push_back(TList{(long long)rdst.size(), q, ix[r + j], 0, 0});
          lists.back().n = partners(p1 + ix[r + j], 0, J1, J2, [&](int, int w, bool g, int t) {
            if (t < 0) {
              rdst.push_back(-1);
              return;
            }
            const size_t k = ((size_t)(g ? 2 : 0) + w) * maxdim + t;
            if (seen[k] != gid) {
              seen[k] = gid;
              slot[k] = (int)rsrc.size();
              rsrc.push_back(g ? ~t : t);
            }
            rdst.push_back(8 * slot[k] + j);
          });
        }
        while (((long long)rsrc.size() - base) % 8 != 0) rsrc.push_back(0);  // absent
        groups.push_back(TSlice{base, (long long)rsrc.size() - base});
        gsize.push_back(n);
        r += n;
      }
      if (rsrc.size() >= (1u << 28)) return fail(IMSRG_EINVAL, "tensor blocks too many for the one-body terms' lists");
      cbase[q] = (int)cols.size();
      for (int c0 = 0; c0 < m2; c0 += 64) {
        const long long base = (long long)cp.size();
        int n = 0;
        for (int k = c0; k < std::min(m2, c0 + 64); k++) n = std::max(n, partners(p2 + k, 1, J1, J2, [](int, int, bool, int) {}));
        n = (n + 3) & ~3;
        cp.resize(base + 64LL * n, 0xffff);
        for (int k = c0; k < std::min(m2, c0 + 64); k++) {
          lists.push_back(TList{base + k - c0, q, k, 1, 0});
          lists.back().n = partners(p2 + k, 1, J1, J2, [&](int e, int, bool g, int t) {
            if (t >= 0) cp[base + 64LL * e + k - c0] = (unsigned short)(g ? m2 + t : t);
          });
        }
        cols.push_back(TSlice{base, n});
      }
      // groups per workgroup: at least eight units of work (a group x 64
      // columns) for its wavefronts, in half of the LDS
      const int ng = m2 > 384 ? 1 : m2 > 192 ? 2 : 4;
      for (int g = gfirst; g < (int)groups.size();) {
        long long e = 0, nr = 0, bytes = 0;
        int k = 0;
        while (k < ng && g + k < (int)groups.size()) {
          const long long e1 = e + groups[g + k].n, nr1 = nr + gsize[g + k - gfirst];
          const long long by = 8 * ((nr1 * ld + 1) & ~1LL) + 68 * e1;
          if (k > 0 && by > 81920) break;
          e = e1;
          nr = nr1;
          bytes = by;
          k++;
        }
        items.push_back(TItem{q, g, k, 0});
        cost[q] += nr * m2;
        lds = (unsigned)std::max<long long>(lds, bytes);
        g += k;
      }
    }
    if (lds > kT1Lds) return fail(IMSRG_EINVAL, "tensor blocks too wide for the one-body terms' workgroups");
    // a block's workgroups on one XCD (workgroup i runs on XCD i % 8), whose L2
    // keeps its rows: blocks in order of size, each to the least loaded XCD
    {
      std::vector<int> order;
      std::vector<std::vector<TItem>> of(S.nblk), queue(8);
      for (const TItem &it : items) of[it.q].push_back(it);
      for (int q = 0; q < S.nblk; q++)
        if (cost[q] > 0) order.push_back(q);
      std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return cost[x] > cost[y]; });
      long long load[8] = {0};
      size_t n = 0;
      for (int q : order) {
        const int x = (int)(std::min_element(load, load + 8) - load);
        load[x] += cost[q];
        queue[x].insert(queue[x].end(), of[q].begin(), of[q].end());
        n = std::max(n, queue[x].size());
      }
      items.assign(8 * n, TItem{0, 0, 0, 0});
      for (int x = 0; x < 8; x++)
        for (size_t i = 0; i < queue[x].size(); i++) items[8 * i + x] = queue[x][i];
    }
    TLists &W = S.lists;
    W.nlist = (int)lists.size();
    W.nitem = (int)items.size();
    W.lds = lds;
    if (W.nlist > 0) {
      if (upload_table(c, lists, &W.lists) != 0 || upload_table(c, items, &W.items) != 0 ||
          upload_table(c, groups, &W.groups) != 0 || upload_table(c, cols, &W.cols) != 0 ||
          upload_table(c, cbase, &W.cbase) != 0 || upload_table(c, grow, &W.grow) != 0 ||
          upload_table(c, rsrc, &W.rsrc) != 0 || upload_table(c, rdst, &W.rdst) != 0 ||
          upload_table(c, cp, &W.cp) != 0)
        return IMSRG_ENOMEM;
      const long long nr = 8LL * rsrc.size(), nc = (long long)cp.size();
      if (dalloc(c, nr, &W.rw) || dalloc(c, nc, &W.cw)) return IMSRG_ENOMEM;
      launch_fill(c->stream, W.rw, nr, kAbsent);  // the weights no list writes stay so
      launch_fill(c->stream, W.cw, nc, kAbsent);
      if (lds > 65536)
        // (the kernel's limit in the whole process: the most any space may take, not this one's)
        HIPCHK(hipFuncSetAttribute((const void *)k_t_1body, hipFuncAttributeMaxDynamicSharedMemorySize, kT1Lds));
    }
  }
  // products: the pp and hh ladders per tensor block (W1, W2); operand 0: G's V, 1: T's V
  {
    std::vector<TProb> pr;
    std::vector<int4> tiles;
    for (int q = 0; q < S.nblk; q++) {
      const int m1 = S.n1[q], m2 = S.n2[q];
      if (m1 == 0 || m2 == 0) continue;
      const int b1 = S.q1[q], b2 = S.q2[q];
      const int np1 = Ly.bnp[b1], nb1 = Ly.bnb[b1], nh1 = Ly.bnh[b1];
      const int np2 = Ly.bnp[b2], nb2 = Ly.bnb[b2], nh2 = Ly.bnh[b2];
      TProb p{};
      p.M = m1; p.N = m2; p.ldc = m2; p.nseg = p.nseg2 = 2; p.c_off = S.off[q];
      for (int w = 0; w < 2; w++) {  // w 0: pp intermediate, 1: hh
        const int k1 = w ? np1 + nb1 : 0, K1 = w ? nh1 : np1, k2 = w ? np2 + nb2 : 0, K2 = w ? nh2 : np2;
        // G(J1)[:, k] T[k, :] - T[:, k] G(J2)[k, :]
        p.seg[2 * w] = TSeg{Ly.boff[b1] + k1, S.off[q] + (long long)k1 * m2, K1, m1, 1, m2, 1, 0, 1, 1.0};
        p.seg[2 * w + 1] = TSeg{S.off[q] + k2, Ly.boff[b2] + (long long)k2 * m2, K2, m2, 1, m2, 1, 1, 0, -1.0};
      }
      pr.push_back(p);
      add_tiles((int)pr.size() - 1, m1, m2, tiles);
    }
    if (upload_table(c, pr, &S.pp_probs) != 0 || upload_table(c, tiles, &S.pp_tiles) != 0) return IMSRG_ENOMEM;
    S.n_pp_tiles = (int)tiles.size();
  }
  // the two Pandya products per cross-coupled block (TS_commutator_222_ph, TS_commutators.f90:1496-1521):
  // alpha carries 1/sqrt(J3+1) and 1/sqrt(J4+1); the herm of G that the reference also folds into Wx
  // is applied where k_t222ph reads Wx, so these tables serve every G
  {
    std::vector<TProb> pr;
    std::vector<int4> tiles;
    for (int x = 0; x < S.ncc; x++) {
      const int q3 = S.cq3[x], q4 = S.cq4[x];
      const int r3 = Ly.ccrlen[q3], r4 = Ly.ccrlen[q4], nb3 = Ly.ccnph[q3], nb4 = Ly.ccnph[q4];
      if (r3 == 0 || r4 == 0) continue;
      TProb px{};  // Wx = LCC(J3) CCR / sqrt(J3+1): operand 0 the Pandya matrices of G, 1 CCR (2 CCX, 3 G's in group order)
      px.M = r3; px.N = r4; px.ldc = r4; px.c_off = S.woff[x];
      px.nseg = nb3 > 0 ? 1 : 0;
      px.seg[0] = TSeg{Ly.ccoff[q3], S.roff[x], nb3, 1, r3, r4, 1, 0, 1, 1.0 / std::sqrt(S.cJ3[x] + 1.0)};
      pr.push_back(px);
      add_tiles((int)pr.size() - 1, r3, r4, tiles);
      TProb py{};  // Wy = CCX LCC(J4)^T / sqrt(J4+1)
      py.M = r3; py.N = r4; py.ldc = r4; py.c_off = S.woff[x]; py.c = 1;
      py.nseg = (nb4 > 0 && S.cJ3[x] != S.cJ4[x]) ? 1 : 0;
      py.seg[0] = TSeg{S.xoff[x], Ly.ccoff[q4], nb4, nb4, 1, r4, 1, 2, 3, 1.0 / std::sqrt(S.cJ4[x] + 1.0)};
      pr.push_back(py);
      add_tiles((int)pr.size() - 1, r3, r4, tiles);
    }
    if (upload_table(c, pr, &S.cc_probs) != 0 || upload_table(c, tiles, &S.cc_tiles) != 0) return IMSRG_ENOMEM;
    S.n_cc_tiles = (int)tiles.size();
  }
  // workspaces
  if (dalloc(c, Ly.ccsize, &S.gcc) || dalloc(c, Ly.ccsize, &S.gccp) || dalloc(c, S.xsize, &S.ccx) || dalloc(c, S.rsize, &S.ccr) ||
      dalloc(c, 2 * S.wsize, &S.wx) || dalloc(c, S.vsize, &S.w1) ||
      dalloc(c, S.vsize, &S.w2))
    return IMSRG_ENOMEM;
  // entries that the selection rules exclude are never written
  launch_fill(c->stream, S.ccx, S.xsize, 0.0);
  launch_fill(c->stream, S.ccr, S.rsize, 0.0);
  S.pan[0].out = S.ccx;
  S.pan[1].out = S.ccr;
  launch_fill(c->stream, S.w1, S.vsize, 0.0);
  launch_fill(c->stream, S.w2, S.vsize, 0.0);
  S.wy = S.wx + S.wsize;
  launch_fill(c->stream, S.wx, 2 * S.wsize, 0.0);
  {
    std::vector<TRun> runs(1, TRun{Ly.f_off, nsp * nsp, 0});
    constexpr int run = 2048;
    for (int q = 0; q < S.nblk; q++) {
      const long long m = (long long)S.n1[q] * S.n2[q];
      for (long long k = 0; k < m; k += run)
        runs.push_back(TRun{S.v_off + S.off[q] + k, (int)std::min<long long>(run, m - k), S.J1[q] == S.J2[q] ? 1 : 2});
    }
    S.nrun = (int)runs.size();
    if (upload_table(c, runs, &S.runs) != 0 || dalloc(c, S.nrun, &S.part)) return IMSRG_ENOMEM;
  }
  HIPCHK(hipHostMalloc((void **)&S.norm, sizeof(TNorm)));
  S.norm->seq = 0;
  return 0;
}

static int tspace_get(imsrg_ctx_s *c, int rank, int dpar, TensorSpace **out) {
  auto key = std::make_pair(rank, dpar);
  auto it = c->tspaces.find(key);
  if (it != c->tspaces.end()) {
    *out = it->second.get();
    return 0;
  }
  auto S = std::make_shared<TensorSpace>();
  const int rc = tspace_build(c, rank, dpar, *S);
  if (rc != 0) return rc;
  c->tspaces[key] = S;
  *out = S.get();
  return 0;
}

// ---------------------------------------------------------------- C ABI

int imsrg_tensor_create(imsrg_ctx c, int rank, int dpar, int herm, imsrg_tensor *out) {
  if (!c || !out) return fail(IMSRG_EINVAL, "null argument");
  if (c->nbatch != 1) return fail(IMSRG_EINVAL, "tensor operators need a single-instance context");
  if (rank <= 0 || (rank & 1)) return fail(IMSRG_EINVAL, "rank must be doubled and positive (2 lambda)");
  if (dpar != 0 && dpar != 2) return fail(IMSRG_EINVAL, "dpar must be 0 or 2 (doubled)");
  if (herm != 1 && herm != -1) return fail(IMSRG_EINVAL, "herm must be +1 or -1");
  TensorSpace *S = nullptr;
  if (int rc = tspace_get(c, rank, dpar, &S)) return rc;
  imsrg_tensor_s *t = new imsrg_tensor_s;
  t->ctx = c;
  t->ts = S;
  t->herm = herm;
  if (dev_malloc((void **)&t->d, sizeof(double) * S->op_size) != hipSuccess) {
    delete t;
    return fail(IMSRG_ENOMEM, "hipMalloc tensor operator failed");
  }
  launch_fill(c->stream, t->d, S->op_size, 0.0);
  *out = t;
  return 0;
}

int imsrg_tensor_destroy(imsrg_tensor t) {
  if (!t) return 0;
  (void)hipStreamSynchronize(t->ctx->stream);
  (void)hipFree(t->d);
  delete t;
  return 0;
}

int64_t imsrg_tensor_neq(imsrg_tensor t) { return t ? t->ts->neq : -1; }
int imsrg_tensor_set_herm(imsrg_tensor t, int herm) {
  if (!t || (herm != 1 && herm != -1)) return fail(IMSRG_EINVAL, "bad argument");
  t->herm = herm;
  return 0;
}
int imsrg_tensor_get_herm(imsrg_tensor t, int *herm) {
  if (!t || !herm) return fail(IMSRG_EINVAL, "null argument");
  *herm = t->herm;
  return 0;
}

// stream <-> device (see the header for the stream order): the pack tables and
// their device buffer, made on first use
static int tpack_setup(imsrg_ctx_s *c, TensorSpace &S) {
  if (S.pack_d) return 0;
  const Layout &Ly = c->lay;
  std::vector<int> head(1, 0), mir(1, -1);
  std::vector<double> sgn(1, 1.0);
  const int n = Ly.nsp, f = (int)Ly.f_off;
  auto put = [&](int i, int j, bool m) {
    head.push_back(f + i * n + j);
    mir.push_back(m ? f + j * n + i : -1);
    sgn.push_back(((Ly.jj[j] - Ly.jj[i]) / 2) & 1 ? -1.0 : 1.0);
  };
  for (int j : Ly.holes)
    for (int i : Ly.holes) put(i, j, false);
  for (int j : Ly.parts)
    for (int i : Ly.parts) put(i, j, false);
  for (int j : Ly.holes)
    for (int i : Ly.parts) put(i, j, true);
  std::vector<PackSeg> segs;
  long long k = (long long)head.size();
  static const int sea1[9] = {0, 0, 0, 1, 2, 1, 2, 1, 2}, sea2[9] = {0, 1, 2, 1, 2, 2, 0, 0, 1};
  for (int q = 0; q < S.nblk; q++) {
    const int m1 = S.n1[q], m2 = S.n2[q];
    if (m1 == 0 || m2 == 0) continue;
    const int b1 = S.q1[q], b2 = S.q2[q];
    const int s1[4] = {0, Ly.bnp[b1], Ly.bnp[b1] + Ly.bnb[b1], m1};
    const int s2[4] = {0, Ly.bnp[b2], Ly.bnp[b2] + Ly.bnb[b2], m2};
    for (int g = 0; g < 9; g++) {
      const int r0 = s1[sea1[g]], nr = s1[sea1[g] + 1] - r0, c0 = s2[sea2[g]], nc = s2[sea2[g] + 1] - c0;
      if (nr == 0 || nc == 0) continue;
      segs.push_back(PackSeg{S.v_off + S.off[q] + (long long)r0 * m2 + c0, k, -1, nr, nc, m2, 0});
      k += (long long)nr * nc;
    }
  }
  if (k != S.neq) return fail(IMSRG_EINVAL, "tensor stream tables do not cover the stream");
  int rc = pack_tables(c, segs, head, mir, sgn, &S.pack);
  if (!rc) rc = dalloc(c, S.neq, &S.pack_d);
  return rc;
}

int imsrg_tensor_upload(imsrg_tensor t, const double *vec, int64_t n) {
  if (!t || !vec) return fail(IMSRG_EINVAL, "null argument");
  TensorSpace &S = *t->ts;
  imsrg_ctx_s *c = t->ctx;
  if (n != S.neq) return fail(IMSRG_EINVAL, "tensor stream length " + std::to_string(n) + " != " + std::to_string(S.neq));
  if (int rc = tpack_setup(c, S)) return rc;
  if (int rc = stream_to_dev(c, vec, n, S.pack_d)) return rc;
  launch_unpack(c->stream, S.pack, S.pack_d, 0, t->d, 0, (double)t->herm, 1);
  HIPCHK(hipGetLastError());
  return 0;
}

int imsrg_tensor_download(imsrg_tensor t, double *vec, int64_t n) {
  if (!t || !vec) return fail(IMSRG_EINVAL, "null argument");
  TensorSpace &S = *t->ts;
  imsrg_ctx_s *c = t->ctx;
  if (n != S.neq) return fail(IMSRG_EINVAL, "tensor stream length " + std::to_string(n) + " != " + std::to_string(S.neq));
  if (int rc = tpack_setup(c, S)) return rc;
  launch_pack(c->stream, S.pack, t->d, 0, S.pack_d, 0, 1);
  HIPCHK(hipGetLastError());
  return stream_to_host(c, S.pack_d, n, vec);
}

static int same_space(imsrg_tensor a, imsrg_tensor b) {
  if (!a || !b) return fail(IMSRG_EINVAL, "null argument");
  if (a->ts != b->ts || a->ctx != b->ctx) return fail(IMSRG_EINVAL, "tensors of different rank, parity or context");
  return 0;
}

int imsrg_tensor_copy(imsrg_tensor src, imsrg_tensor dst) {
  if (int rc = same_space(src, dst)) return rc;
  HIPCHK(hipMemcpyAsync(dst->d, src->d, sizeof(double) * src->ts->op_size, hipMemcpyDeviceToDevice, src->ctx->stream));
  dst->herm = src->herm;
  return 0;
}

int imsrg_tensor_clear(imsrg_tensor t) {
  if (!t) return fail(IMSRG_EINVAL, "null argument");
  launch_fill(t->ctx->stream, t->d, t->ts->op_size, 0.0);
  return 0;
}

int imsrg_tensor_add(imsrg_tensor A, double ax, imsrg_tensor B, double bx, imsrg_tensor C) {
  if (int rc = same_space(A, B)) return rc;
  if (int rc = same_space(A, C)) return rc;
  launch_axpby(A->ctx->stream, A->ts->op_size, ax, A->d, bx, B->d, C->d, nullptr, 1, 0);
  return 0;
}

// ||X|| (and HS += coef X first), read from host memory as the kernel writes it
static int tstep(imsrg_ctx_s *c, TensorSpace &S, const double *X, double *HS, double coef, double *out) {
  S.seq = S.seq == (1 << 30) ? 1 : S.seq + 1;
  hipLaunchKernelGGL(k_t_step, dim3(S.nrun), dim3(256), 0, c->stream, c->dl, S.runs, X, HS, coef, S.part);
  hipLaunchKernelGGL(k_t_norm, dim3(1), dim3(256), 0, c->stream, (const double *)S.part, S.nrun, S.norm, S.seq);
  HIPCHK(hipGetLastError());
  const volatile int *seq = &S.norm->seq;
  for (long long spin = 1; *seq != S.seq; spin++) {
    if (spin % 4096) continue;
    const hipError_t e = hipStreamQuery(c->stream);
    if (e == hipErrorNotReady || (e == hipSuccess && *seq == S.seq)) continue;
    return fail(IMSRG_EDEVICE, std::string("tensor norm: ") + hipGetErrorString(e));
  }
  std::atomic_thread_fence(std::memory_order_acquire);
  *out = std::sqrt(*(const volatile double *)&S.norm->v);
  return 0;
}

int imsrg_tensor_norm(imsrg_tensor t, double *out) {
  if (!t || !out) return fail(IMSRG_EINVAL, "null argument");
  return tstep(t->ctx, *t->ts, t->d, nullptr, 0.0, out);
}

// [G, T] into RES in BCH_TENSOR's call order (IMSRG_MAGNUS.f90:427-446):
// 111 (overwrites the one-body part), 121, 122 (overwrites the two-body
// part), 212, 222_pp_hh, 221, 211, 222_ph; the others accumulate, so the
// one-body terms run together once the ladder products and G's Pandya matrices
// are there.  221 reads the ladder products, computed here whenever it is
// asked for.  Gd:
// the scalar operator's buffer (may be null when only 211 / 222_ph run on
// Pandya matrices already in S.gcc, gcc_ready).
static int ts_comm(imsrg_ctx_s *c, const double *Gd, int hG, imsrg_tensor T, imsrg_tensor RES, unsigned mask,
                   bool gcc_ready) {
  TensorSpace &S = *T->ts;
  const DevLayout &L = c->dl;
  const DevTensor &D = S.dt;
  hipStream_t s = c->stream;
  const int hL = hG, hR = T->herm, hres = RES->herm;
  const double *GF = Gd ? Gd + c->lay.f_off : nullptr, *GV = Gd ? Gd + c->lay.v_off : nullptr;
  const double *RF = T->d + c->lay.f_off, *RV = T->d + S.v_off;
  double *OF = RES->d + c->lay.f_off, *OV = RES->d + S.v_off;
  if (!Gd && (mask & ~(IMSRG_TS211 | IMSRG_TS222PH))) return fail(IMSRG_EINVAL, "terms need the scalar operator");
  if (S.lists.nlist > 0 && (mask & (IMSRG_TS122 | IMSRG_TS212))) {
    hipLaunchKernelGGL(k_t_lists, dim3(S.lists.nlist), dim3(64), 0, s, L, D, S.lists, GF, RF,
                       (mask & IMSRG_TS122) != 0, (mask & IMSRG_TS212) != 0);
    hipLaunchKernelGGL(k_t_1body, dim3(S.lists.nitem), dim3(kT1Threads), S.lists.lds, s, L, D, S.lists, GV, RV, OV,
                       !(mask & IMSRG_TS122));
  }
  if ((mask & (IMSRG_TS222PPHH | IMSRG_TS221)) && S.n_pp_tiles > 0)
    hipLaunchKernelGGL(k_tgemm, dim3(S.n_pp_tiles), dim3(256), 0, s, S.pp_probs, S.pp_tiles, S.n_pp_tiles,
                       TGemm{{GV, RV, nullptr, nullptr}, {S.w1, S.w2}, (mask & IMSRG_TS222PPHH) ? OV : nullptr});
  if ((mask & (IMSRG_TS211 | IMSRG_TS222PH)) && !gcc_ready) launch_pandya(s, L, Gd, S.gcc, nullptr, 1);
  const int one = ((mask & IMSRG_TS111) ? kTf111 : 0) | ((mask & IMSRG_TS121) ? kTf121 : 0) |
                  ((mask & IMSRG_TS221) ? kTf221 : 0) | ((mask & IMSRG_TS211) ? kTf211 : 0);
  if (one)
    hipLaunchKernelGGL(k_t_f, dim3(L.nob), dim3(kTfThreads), 0, s, L, D, one, GF, RF, RV, (const double *)S.gcc,
                       (const double *)S.w1, (const double *)S.w2, OF, hL, hR, hres);
  if ((mask & IMSRG_TS222PH) && S.nelem > 0) {
    if (L.nccol > 0)
      hipLaunchKernelGGL(k_gcc_order, dim3(L.nccol), dim3(256), 0, s, L, D, (const double *)S.gcc, S.gccp);
    if (S.pan[0].npad + S.pan[1].npad > 0)
      hipLaunchKernelGGL(k_t_pandya, dim3(S.pan[0].npad + S.pan[1].npad), dim3(64), 0, s, L, D, S.pan[0], S.pan[1],
                         RV, hR);
    if (S.n_cc_tiles > 0)
      hipLaunchKernelGGL(k_tgemm, dim3(S.n_cc_tiles), dim3(256), 0, s, S.cc_probs, S.cc_tiles, S.n_cc_tiles,
                         TGemm{{S.gcc, S.ccr, S.ccx, S.gccp}, {S.wx, S.wy}, nullptr});
    if (D.nqchunk > 0)
      hipLaunchKernelGGL(k_t222ph, dim3(D.nqpad), dim3(64), 0, s, L, D, (const double *)S.wx, S.wsize, OV, hL, hR);
  }
  HIPCHK(hipGetLastError());
  return 0;
}

int imsrg_tensor_commutator(imsrg_op G, imsrg_tensor T, imsrg_tensor RES, unsigned mask) {
  if (!G || !T || !RES) return fail(IMSRG_EINVAL, "null argument");
  if (int rc = same_space(T, RES)) return rc;
  if (G->ctx != T->ctx) return fail(IMSRG_EINVAL, "G and T belong to different contexts");
  if (T == RES) return fail(IMSRG_EINVAL, "RES must differ from T");
  return ts_comm(G->ctx, G->d, G->herm, T, RES, mask, false);
}

int imsrg_tensor_commutator_cc(imsrg_tensor T, const double *gcc, int hG, int64_t n, imsrg_tensor RES,
                               unsigned mask) {
  if (!T || !gcc || !RES) return fail(IMSRG_EINVAL, "null argument");
  if (int rc = same_space(T, RES)) return rc;
  if (T == RES) return fail(IMSRG_EINVAL, "RES must differ from T");
  if (hG != 1 && hG != -1) return fail(IMSRG_EINVAL, "herm must be +1 or -1");
  if (mask & ~(IMSRG_TS211 | IMSRG_TS222PH)) return fail(IMSRG_EINVAL, "only 211 and 222_ph run on Pandya matrices");
  imsrg_ctx_s *c = T->ctx;
  if (n != imsrg_cross_coupled_size(c)) return fail(IMSRG_EINVAL, "Pandya stream size mismatch");
  // the reference's row order (all ordered pairs, first orbit major) into the
  // device's paired rows; the zero rows stay zero
  const Layout &Ly = c->lay;
  std::vector<double> img(Ly.ccsize, 0.0);
  int64_t o = 0;
  for (int q = 0; q < Ly.ncc; q++) {
    const int rr = Ly.ccrlen_ref[q], rd = Ly.ccrlen[q], nb = Ly.ccnph[q];
    const int *ref = Ly.ccref.data() + Ly.ccrefbase[q];
    for (int col = 0; col < nb; col++)
      for (int r = 0; r < rr; r++) img[Ly.ccoff[q] + (int64_t)col * rd + ref[r]] = gcc[o++];
  }
  HIPCHK(hipMemcpyAsync(T->ts->gcc, img.data(), sizeof(double) * Ly.ccsize, hipMemcpyHostToDevice, c->stream));
  const int rc = ts_comm(c, nullptr, hG, T, RES, mask, true);
  HIPCHK(hipStreamSynchronize(c->stream));  // img is a local buffer
  return rc;
}

int imsrg_tensor_ladders(imsrg_op G, imsrg_tensor T, imsrg_tensor W1, imsrg_tensor W2) {
  if (!G || !T || !W1 || !W2) return fail(IMSRG_EINVAL, "null argument");
  if (int rc = same_space(T, W1)) return rc;
  if (int rc = same_space(T, W2)) return rc;
  if (G->ctx != T->ctx) return fail(IMSRG_EINVAL, "G and T belong to different contexts");
  imsrg_ctx_s *c = T->ctx;
  TensorSpace &S = *T->ts;
  hipStream_t s = c->stream;
  const double *GV = G->d + c->lay.v_off, *RV = T->d + S.v_off;
  launch_fill(s, W1->d, S.op_size, 0.0);
  launch_fill(s, W2->d, S.op_size, 0.0);
  if (S.n_pp_tiles > 0)
    hipLaunchKernelGGL(k_tgemm, dim3(S.n_pp_tiles), dim3(256), 0, s, S.pp_probs, S.pp_tiles, S.n_pp_tiles,
                       TGemm{{GV, RV, nullptr, nullptr}, {W1->d + S.v_off, W2->d + S.v_off}, nullptr});
  HIPCHK(hipGetLastError());
  return 0;
}

int imsrg_tensor_commutator_221(imsrg_tensor W1, imsrg_tensor W2, int pm, imsrg_tensor RES) {
  if (!W1 || !W2 || !RES) return fail(IMSRG_EINVAL, "null argument");
  if (int rc = same_space(W1, RES)) return rc;
  if (int rc = same_space(W2, RES)) return rc;
  if (pm != 1 && pm != -1) return fail(IMSRG_EINVAL, "pm must be +1 or -1");
  imsrg_ctx_s *c = RES->ctx;
  TensorSpace &S = *RES->ts;
  double *OF = RES->d + c->lay.f_off;
  hipLaunchKernelGGL(k_t_f, dim3(c->dl.nob), dim3(kTfThreads), 0, c->stream, c->dl, S.dt, (int)kTf221,
                     (const double *)nullptr, (const double *)nullptr, (const double *)nullptr, (const double *)nullptr,
                     (const double *)(W1->d + S.v_off), (const double *)(W2->d + S.v_off), OF, pm, 1, RES->herm);
  HIPCHK(hipGetLastError());
  return 0;
}

// BCH_TENSOR: HS += sum of the nested commutators [G, .. [G, HS]] / n! until
// ||ad^n|| / n! < conv.  The nested commutators alternate between two work
// operators; the first reads HS itself, which only changes after it.  All of a
// work operator's one- and two-body elements are overwritten by 111 and 122.
static constexpr long long kBchKeep = 1LL << 30;
int imsrg_bch_tensor(imsrg_op G, imsrg_tensor HS, int *nterms) {
  if (!G || !HS) return fail(IMSRG_EINVAL, "null argument");
  imsrg_ctx_s *c = HS->ctx;
  if (G->ctx != c) return fail(IMSRG_EINVAL, "G and HS belong to different contexts");
  TensorSpace &S = *HS->ts;
  const long long bytes = 2LL * (long long)sizeof(double) * S.op_size;
  double *buf = S.bch.take();
  if (!buf) {
    if (dev_malloc((void **)&buf, bytes) != hipSuccess) return fail(IMSRG_ENOMEM, "hipMalloc BCH_TENSOR workspace failed");
    launch_fill(c->stream, buf, 2 * S.op_size, 0.0);
  }
  imsrg_tensor_s W[2];
  for (int k = 0; k < 2; k++) {
    W[k].ctx = c;
    W[k].ts = &S;
    W[k].d = buf + k * S.op_size;
    W[k].herm = HS->herm;  // copy_sq_op keeps HS's herm (IMSRG_MAGNUS.f90:419-422)
  }
  const double conv = (double)1e-6f;  // real(8), parameter :: conv = 1e-6
  double coef = 1.0;
  int n = 0, rc = 0;
  imsrg_tensor AD = HS;
  for (int iw = 2; iw <= 30; iw++) {
    coef = coef / (iw - 1.0);
    imsrg_tensor INT2 = &W[iw & 1];
    if ((rc = ts_comm(c, G->d, G->herm, AD, INT2, IMSRG_TSALL, false))) break;
    n++;
    double nrm = 0.0;
    if ((rc = tstep(c, S, INT2->d, HS->d, coef, &nrm))) break;
    if (nrm * coef < conv) break;
    AD = INT2;
  }
  if (bytes > kBchKeep || rc != 0 || !S.bch.give(buf, bytes)) {
    (void)hipStreamSynchronize(c->stream);
    (void)hipFree(buf);
  }
  if (nterms) *nterms = n;
  return rc;
}

