// adjoint.hip -- transpose of the IMSRG(2) commutator in its second operand.
//
// For fixed P and a cotangent C (herm hC = -hP*hY) these kernels accumulate
//   Ybar = d <C, [P, Y]> / dY
// where <A, B> is the Frobenius product over the full device layout
// (E0, the full one-body matrix, every channel block in full).  Each term is
// the exact transpose of its forward kernel in kernels.hip, term by term:
// gathers become scatters (FP64 atomics), the 222 products become products
// with the transposed operands.  The caller projects Ybar onto operators of
// hermiticity hY afterwards.  By antisymmetry of the commutator,
// d <C, [X, Y]> / dX = -Ybar(P = Y).
#include <hip/hip_runtime.h>

#include "comm_dev.hpp"
#include "device.hpp"

namespace imsrg {

// cotangent of one-body output (p,q) of the ob list: the forward kernel writes
// F(p,q) = val and F(q,p) = hC*val (diagonal: val, or 0 for hC = -1)
__device__ __forceinline__ double ob_cot(const DevLayout &L, const double *CF, int p, int q, int hC) {
  const int N = L.nsp;
  if (p != q) return CF[p * N + q] + hC * CF[q * N + p];
  return hC == 1 ? CF[p * N + p] : 0.0;
}

// ---- projection onto hermiticity h: X <- (I + h I^T)/2 on F and every block;
// E0 <- 0 unless keep_e0 (I's).  Workgroup b: mirror tile b, or (b = nmirror)
// the one-body part and E0.  I and X may be the same operator.
__device__ __forceinline__ void project_tile(const DevLayout &L, int b, const double *I, double *X, int h, int keep_e0,
                                             double (*U)[33], double (*W)[33]) {
  if (b == L.nmirror) {  // one-body part and E0
    const int N = L.nsp;
    const double *G = I + L.f_off;
    double *F = X + L.f_off;
    for (int t = threadIdx.x; t < N * N; t += 256) {
      const int a = t / N, c = t % N;
      if (a < c) {
        const double u = G[a * N + c], v = G[c * N + a];
        F[a * N + c] = 0.5 * (u + h * v);
        F[c * N + a] = 0.5 * (v + h * u);
      } else if (a == c) {
        F[t] = h == -1 ? 0.0 : G[t];
      }
    }
    if (threadIdx.x == 0) X[0] = keep_e0 ? I[0] : 0.0;
    return;
  }
  const int4 t = L.mirror_tiles[b];
  const int q = t.x, dim = L.bdim[q];
  const double *IV = I + L.v_off + L.boff[q];
  double *OV = X + L.v_off + L.boff[q];
  const int r0 = t.y * 32, c0 = t.z * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx;
    U[k][tx] = (r < dim && c < dim) ? IV[(long long)r * dim + c] : 0.0;
    const int r2 = c0 + k, c2 = r0 + tx;
    W[k][tx] = (r2 < dim && c2 < dim) ? IV[(long long)r2 * dim + c2] : 0.0;
  }
  __syncthreads();
  const bool diag = t.y == t.z;
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx;  // upper element (r, c); its mirror is W[tx][k]
    if (r < dim && c < dim && (!diag || k <= tx)) {
      const double v = 0.5 * (U[k][tx] + h * W[tx][k]);
      OV[(long long)r * dim + c] = (diag && k == tx && h == -1) ? 0.0 : v;
    }
    const int r2 = c0 + k, c2 = r0 + tx;  // lower element (r2, c2); its mirror is U[tx][k]
    if (r2 < dim && c2 < dim && (!diag || tx < k)) OV[(long long)r2 * dim + c2] = h * (0.5 * (U[tx][k] + h * W[k][tx]));
  }
}
__global__ __launch_bounds__(256) void k_project(DevLayout L, double *X, int h, int keep_e0) {
  __shared__ double U[32][33], W[32][33];
  project_tile(L, blockIdx.x, X, X, h, keep_e0, U, W);
}

// The kernels are lists of workgroups of different kinds, launched in seven
// steps (they were sixteen launches and one more per Pandya block, most of them
// shorter than the 5 us a launch costs the host):
//   k_adj_a  C projected; Y, the J' cotangents and the Z cotangent cleared; Pandya of P
//   k_adj_b  E0, one-body and 122 terms into Y; Q = P C; J' cotangents
//   k_adj_c  222_pp_hh from Q into Y; Z cotangent from the J' ones
//   k_adj_d  Sbar from the Z cotangent
//   k_adj_e  Ybar_CC^T = P_CC^T Sbar^T
//   k_adj_f  transpose of the Pandya transform into Y
//   k_project (caller's hermiticity)
// What bounds a call now is FP64 atomics (steps b, c, f) and, in small bases,
// seven dependent launches.  Per call, separate kernels / these, in us: emax 2
// 127 / 34, emax 4 276 / 67, emax 5 474 / 128, emax 6 865 / 285, emax 8 4327 / 2260.

// ---- E0 terms: 110 (commutators.f90:10-33) and 220 (:399-432); workgroup b < nblocks: block b
__device__ __forceinline__ void adj_e0(const DevLayout &L, const double *__restrict__ P, const double *__restrict__ C,
                                       double *__restrict__ Y, int hP, int hY, unsigned mask, int b) {
  const double e = C[0];
  if (e == 0.0) return;
  if (b < L.nblocks) {
    if (!(mask & T220) || hP * hY != -1) return;
    const int np = L.bnp[b], nb = L.bnb[b], nh = L.bnh[b], dim = L.bdim[b];
    const double *A = P + L.v_off + L.boff[b];
    double *YV = Y + L.v_off + L.boff[b];
    const double w = -2.0 * (L.bJ[b] + 1) * hY * e;
    for (int t = threadIdx.x; t < np * nh; t += 256) {
      const int ix = t / nh, jx = t % nh;
      const long long o = (long long)ix * dim + np + nb + jx;
      atomicAdd(YV + o, w * A[o]);
    }
  } else {
    if (!(mask & T110)) return;
    const int N = L.nsp;
    const double *FP = P + L.f_off;
    double *YF = Y + L.f_off;
    for (int t = threadIdx.x; t < N * N; t += 256) {
      const int a = t / N, i = t % N;
      if (L.con[a] != 0 || L.con[i] != 1) continue;
      atomicAdd(YF + t, e * FP[t] * (double)(hP - hY) * (L.jj[i] + 1));
    }
  }
}

// ---- one-body outputs.  111 (commutators.f90:36-80): one wavefront per output t
__device__ __forceinline__ void adj_111(const DevLayout &L, const double *__restrict__ P, const double *__restrict__ C,
                                        double *__restrict__ Y, int hC, int t) {
  const int p = L.ob_p[t], q = L.ob_q[t], N = L.nsp;
  const double c = ob_cot(L, C + L.f_off, p, q, hC);
  if (c == 0.0) return;
  const double *FP = P + L.f_off;
  double *YF = Y + L.f_off;
  // val = sum_k P(p,k) Y(k,q) - Y(p,k) P(k,q)
  for (int k = threadIdx.x & 63; k < N; k += 64) {
    const double x = c * FP[p * N + k], y = c * FP[k * N + q];
    if (x != 0.0) atomicAdd(YF + k * N + q, x);
    if (y != 0.0) atomicAdd(YF + p * N + k, -y);
  }
}
// 121 (:83-280) and 221 (:435-578) of the same-(l,j,tz) output sp.  Work item i
// of an output: i < N orbit i of 221, one J per wavefront round, lanes over
// the pairs; from N on, 256 terms of 121.
__device__ __forceinline__ void adj_121_221(const DevLayout &L, const double *__restrict__ P,
                                            const double *__restrict__ C, double *__restrict__ Y, int hP, int hY,
                                            int hC, unsigned mask, int sp, int i) {
  const int t = L.same_ob[sp], p = L.ob_p[t], q = L.ob_q[t], N = L.nsp, MJ = L.nJ;
  const double c = ob_cot(L, C + L.f_off, p, q, hC);
  if (c == 0.0) return;
  const double *FP = P + L.f_off, *VP = P + L.v_off;
  double *YF = Y + L.f_off, *YV = Y + L.v_off;
  const double w0 = c / (L.jj[p] + 1.0);
  if (i >= N) {
    if (!(mask & T121)) return;
    const int it = (i - N) * 256 + (int)threadIdx.x, jq = L.jj[q];
    if (it >= L.nphp * MJ) return;
    const int e = it / MJ, m = it - e * MJ;
    const int a = L.php_a[e], h = L.php_i[e], ji = L.jj[h];
    const int JT = abs(ji - jq) + 2 * m;
    if (JT > ji + jq) return;
    const double g = w0 * (JT + 1), fp = FP[a * N + h];
    // + FP(a,i) (hP v_Y(a,p,i,q) - v_Y(i,p,a,q)) - FY(a,i) (hY v_P(a,p,i,q) - v_P(i,p,a,q))
    double f1, f2;
    const long long o1 = dv_pos(L, a, p, h, q, JT, f1), o2 = dv_pos(L, h, p, a, q, JT, f2);
    const double v1 = o1 >= 0 ? VP[o1] * f1 : 0.0, v2 = o2 >= 0 ? VP[o2] * f2 : 0.0;
    if (o1 >= 0) atomicAdd(YV + o1, g * fp * hP * f1);
    if (o2 >= 0) atomicAdd(YV + o2, -g * fp * f2);
    atomicAdd(YF + a * N + h, -g * (hY * v1 - v2));
    return;
  }
  if (!(mask & T221)) return;
  // val += sum_c,J (J+1)/(2j_p+1) pre * sum_{k} (P(r,k) Y(k,s) - Y(r,k) P(k,s)),
  // r = (c,p), s = (c,q); k over pp pairs for a hole c, hh pairs for a particle c
  const int cc = i, jc = L.jj[cc], jp = L.jj[p], wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int Pq = (L.l[cc] + L.l[p]) & 1, T2 = L.tz[cc] + L.tz[p];
  for (int JT = abs(jc - jp) + 2 * wave; JT <= jc + jp; JT += 8) {
    const int qb = 3 * JT + 2 * (T2 / 2 + 1) + Pq;
    const int r = dpos(L, JT, min(cc, p), max(cc, p)), s = dpos(L, JT, min(cc, q), max(cc, q));
    if ((r | s) < 0) continue;
    double pre = cc > p ? (double)sgnp(1 + ((jc + jp - JT) >> 1)) : cc == p ? M_SQRT2 : 1.0;
    pre *= cc > q ? (double)sgnp(1 + ((jc + jp - JT) >> 1)) : cc == q ? M_SQRT2 : 1.0;
    const long long bo = L.boff[qb];
    const int dim = L.bdim[qb];
    const int k0 = L.con[cc] ? 0 : L.bnp[qb] + L.bnb[qb], k1 = L.con[cc] ? L.bnp[qb] : dim;
    const double g = w0 * (JT + 1) * pre;
    const double *Pb = VP + bo;
    double *Yb = YV + bo;
    for (int k = k0 + lane; k < k1; k += 64) {
      atomicAdd(Yb + (long long)k * dim + s, g * Pb[(long long)r * dim + k]);
      atomicAdd(Yb + (long long)r * dim + k, -g * Pb[(long long)k * dim + s]);
    }
  }
}

// ---- 122: RES = M + hC M^T, M(r,s) = sum_{e in nb(r)} c_e [fP(x,i) Y(r_e,s) - fY(x,i) P(r_e,s)].
// With C of hermiticity hC the cotangent of M is Mbar = C + hC C^T = 2C (diagonal (1+hC) C).
// One workgroup per row, a neighbour entry per wavefront.
__device__ __forceinline__ void adj_122(const DevLayout &L, const double *__restrict__ P, const double *__restrict__ C,
                                        double *__restrict__ Y, int hC, int r) {
  const int q = L.pair_q[r], rl = r - L.pbase[q], dim = L.bdim[q], N = L.nsp, lane = threadIdx.x & 63;
  const long long bo = L.v_off + L.boff[q];
  const double *PV = P + bo, *CV = C + bo + (long long)rl * dim;
  double *YV = Y + bo;
  const double *FP = P + L.f_off;
  double *YF = Y + L.f_off;
  for (int e = L.nb_start[r] + (int)(threadIdx.x >> 6); e < L.nb_start[r + 1]; e += 4) {
    const long long pe = L.nb_pos[e];
    const int xi = L.nb_x[e] * N + L.nb_i[e];
    const double ce = L.nb_coef[e], w = ce * FP[xi];
    double dot = 0.0;
    for (int s = lane; s < dim; s += 64) {
      const double mb = (s == rl) ? (1.0 + hC) * CV[s] : 2.0 * CV[s];
      if (w != 0.0) atomicAdd(YV + pe * dim + s, w * mb);
      dot += PV[pe * dim + s] * mb;
    }
    dot = wave_sum(dot);
    if (lane == 0 && dot != 0.0) atomicAdd(YF + xi, -ce * dot);
  }
}

// ---- 222_pp_hh: C = P D Y - Y D P  =>  Ybar(r,s) += hP d_r Q(r,s) - hC d_s Q(s,r), Q = P C;
// a 32 x 32 tile pair, Q's two tiles through LDS
__device__ __forceinline__ void adj_pphh(const DevLayout &L, const int4 t, const double *__restrict__ Q,
                                         double *__restrict__ Y, int hP, int hC, double (*U)[33], double (*W)[33]) {
  const int q = t.x, dim = L.bdim[q], np = L.bnp[q], nh0 = L.bnp[q] + L.bnb[q];
  const double *Qb = Q + L.boff[q];
  double *Yb = Y + L.v_off + L.boff[q];
  const int r0 = t.y * 32, c0 = t.z * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  auto sg = [&](int r) { return r < np ? 1.0 : r >= nh0 ? -1.0 : 0.0; };
  for (int k = ty; k < 32; k += 8) {
    U[k][tx] = r0 + k < dim && c0 + tx < dim ? Qb[(long long)(r0 + k) * dim + c0 + tx] : 0.0;
    W[k][tx] = c0 + k < dim && r0 + tx < dim ? Qb[(long long)(c0 + k) * dim + r0 + tx] : 0.0;
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    const int r = r0 + k, c = c0 + tx, r2 = c0 + k, c2 = r0 + tx;
    if (r < dim && c < dim) Yb[(long long)r * dim + c] += hP * sg(r) * U[k][tx] - hC * sg(c) * W[tx][k];
    if (t.y != t.z && r2 < dim && c2 < dim)
      Yb[(long long)r2 * dim + c2] += hP * sg(r2) * W[k][tx] - hC * sg(c2) * U[tx][k];
  }
}

// ---- 222_ph, step 1: cotangents of the J' terms (transpose of k_ph_apply):
// one wavefront per work item of up to 64 outputs, four lanes an output
__device__ __forceinline__ void adj_ph_apply(const DevLayout &L, const PhChunk h, const double *__restrict__ C,
                                             double *__restrict__ Tbar, int hC) {
  const int lane = threadIdx.x & 63, g = lane >> 2, sub = lane & 3;
  const double *CV = C + h.vrow;
  const unsigned long long *desc = L.ph_desc + h.dbase;
  const double *S6 = L.ap6_val + h.b0;
  const double pre = h.half ? .70710678118 : 1.0;
#pragma unroll
  for (int u = 0; u < 4; u++) {
    const int o = g + 16 * u;
    if (o >= h.n) continue;
    // the forward writes the upper element and its mirror herm * value; a row's
    // first element is its diagonal one when the item starts there (h.diag)
    const double cv = CV[o], ob = (h.diag && o == 0) ? ((hC == 1) ? cv : 0.0) : 2.0 * cv;
    int toff, n1, n, o1, o2;
    double g1, g2, pre2;
    ph_decode(desc[o], toff, n1, n, o1, o2, g1, g2, pre2);
    const double w = ob * pre * pre2;
    if (w == 0.0) continue;
    double *T = Tbar + h.tbase + toff;
    for (int m = sub; m < n; m += 4) {
      const double x = w * ph_coef(S6, m, n, n1, o1, o2, g1, g2);
      if (x != 0.0) atomicAdd(T + m, x);
    }
  }
}

// ---- 222_ph, step 2: cotangent of Z (transpose of k_ph_terms), term t
__device__ __forceinline__ void adj_ph_term(const DevLayout &L, const double *__restrict__ Tbar,
                                            double *__restrict__ Zbar, double sigma, long long t) {
  if (t >= L.nphterm) return;
  const double v = Tbar[t];
  if (v == 0.0) return;
  const unsigned tc = L.ph_terms[t];
  if (tc == 0xFFFFFFFFu) return;  // padding term
  const unsigned code = L.ph_quads[tc >> 6];
  const int side = (tc >> 5) & 1, m = tc & 31;
  const int i = code >> 24, j = (code >> 16) & 255, k = (code >> 8) & 255, l = code & 255;
  const int N = L.nsp, JTM1 = L.jtot_max + 1;
  const int ji = L.jj[i], jj = L.jj[j], jk = L.jj[k], jl = L.jj[l];
  const double ph = sgnp((ji + jj + jk + jl) >> 1);
  // (a, b | c, d) = (k, i | l, j) on side 0, (k, j | l, i) on side 1
  const int b = side ? j : i, d = side ? i : j, jb = side ? jj : ji, jd = side ? ji : jj;
  const int Tz = abs(L.tz[b] - L.tz[k]) / 2, P = (L.l[b] + L.l[k]) % 2;
  const int JP = max(abs(jd - jl), abs(jb - jk)) + 2 * m;
  const int qx = (JP >> 1) + Tz * JTM1 + 2 * P * JTM1;
  const int *rowt = L.ccrow + (size_t)qx * N * N;
  const int kb = rowt[k * N + b], bk = rowt[b * N + k], ld = rowt[l * N + d], dl = rowt[d * N + l];
  if ((kb | bk | ld | dl) < 0) return;
  const long long rl = L.ccrlen[qx];
  double *Zq = Zbar + L.cwoff[qx];
  if (side == 0) {
    atomicAdd(Zq + kb * rl + dl, v);
    atomicAdd(Zq + bk * rl + ld, ph * sigma * v);
  } else {
    atomicAdd(Zq + bk * rl + ld, sigma * v);
    atomicAdd(Zq + kb * rl + dl, ph * v);
  }
}

// Step a.  Workgroups: tiles of C (and its one-body part), Pandya columns of P, clears.
__global__ __launch_bounds__(256) void k_adj_a(DevLayout L, AdjArgs A) {
  extern __shared__ double lds[];
  int b = blockIdx.x;
  if (b < L.nccol * A.ph) {
    pandya_col<false>(L, A.P, A.ccP, b, lds);
    return;
  }
  b -= L.nccol * A.ph;
  if (b <= L.nmirror) {
    project_tile(L, b, A.Cin, A.C, A.hC, 1, reinterpret_cast<double(*)[33]>(lds),
                 reinterpret_cast<double(*)[33]>(lds + 32 * 33));
    return;
  }
  b -= L.nmirror + 1;
  const long long n0 = L.op_size, n1 = A.ph ? L.nphterm : 0, n2 = A.ph ? L.cwsize : 0, st = 256LL * A.nfill;
  for (long long i = 256LL * b + threadIdx.x; i < n0 + n1 + n2; i += st) {
    if (i < n0) A.Y[i] = 0.0;
    else if (i < n0 + n1) A.T[i - n0] = 0.0;
    else A.Z[i - n0 - n1] = 0.0;
  }
}
__global__ __launch_bounds__(256) void k_adj_b(DevLayout L, AdjArgs A) {
  __shared__ SplitSmem S;
  int b = blockIdx.x;
  if (b < A.n_pp) {
    const int4 tl = A.pp_tiles[b];
    plain_tile(A.pp_probs[tl.x], tl.y * 32, tl.z * 32, A.P + L.v_off, A.C + L.v_off, A.Q, S);
    return;
  }
  b -= A.n_pp;
  if (b < A.n_ob) {  // the longest chains first
    const int per = L.nsp + (L.nphp * L.nJ + 255) / 256;
    adj_121_221(L, A.P, A.C, A.Y, A.hP, A.hY, A.hC, A.mask, b / per, b % per);
    return;
  }
  b -= A.n_ob;
  if (b < A.n_122) {
    adj_122(L, A.P, A.C, A.Y, A.hC, b);
    return;
  }
  b -= A.n_122;
  if (b < A.n_ap) {
    const int i = 4 * b + (int)(threadIdx.x >> 6);
    if (i < A.n_chunks) adj_ph_apply(L, L.ph_chunks[i], A.C, A.T, A.hC);
    return;
  }
  b -= A.n_ap;
  if (b < A.n_111) {
    const int t = 4 * b + (int)(threadIdx.x >> 6);
    if (t < L.nob) adj_111(L, A.P, A.C, A.Y, A.hC, t);
    return;
  }
  adj_e0(L, A.P, A.C, A.Y, A.hP, A.hY, A.mask, b - A.n_111);
}
__global__ __launch_bounds__(256) void k_adj_c(DevLayout L, AdjArgs A) {
  __shared__ double U[32][33], W[32][33];
  int b = blockIdx.x;
  const int npp = A.n_pp ? L.nmirror : 0;
  if (b < npp) {
    adj_pphh(L, L.mirror_tiles[b], A.Q, A.Y, A.hP, A.hC, U, W);
    return;
  }
  adj_ph_term(L, A.T, A.Z, (double)(-A.hP * A.hY), (long long)(b - npp) * 256 + threadIdx.x);
}
// step d: Sbar^T = hP Zbar - hY Zbar^T in place, a 32 x 32 tile pair of one Pandya block
__global__ __launch_bounds__(256) void k_adj_d(DevLayout L, const int4 *__restrict__ tiles, double *__restrict__ Z,
                                               int hP, int hY) {
  __shared__ double U[32][33], W[32][33];
  const int4 t = tiles[blockIdx.x];
  const int r = L.ccrlen[t.x], a0 = t.y * 32, b0 = t.z * 32, tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
  double *Zq = Z + L.cwoff[t.x];
  for (int k = ty; k < 32; k += 8) {
    U[k][tx] = a0 + k < r && b0 + tx < r ? Zq[(long long)(a0 + k) * r + b0 + tx] : 0.0;
    W[k][tx] = b0 + k < r && a0 + tx < r ? Zq[(long long)(b0 + k) * r + a0 + tx] : 0.0;
  }
  __syncthreads();
  for (int k = ty; k < 32; k += 8) {
    if (a0 + k < r && b0 + tx < r) Zq[(long long)(a0 + k) * r + b0 + tx] = hP * U[k][tx] - hY * W[tx][k];
    if (t.y != t.z && b0 + k < r && a0 + tx < r)
      Zq[(long long)(b0 + k) * r + a0 + tx] = hP * W[k][tx] - hY * U[tx][k];
  }
}
__global__ __launch_bounds__(256) void k_adj_e(const GemmProb *__restrict__ probs, const int4 *__restrict__ tiles,
                                               const double *__restrict__ A, const double *__restrict__ B,
                                               double *__restrict__ C) {
  __shared__ SplitSmem S;
  const int4 tl = tiles[blockIdx.x];
  plain_tile(probs[tl.x], tl.y * 32, tl.z * 32, A, B, C, S);
}
__global__ __launch_bounds__(256) void k_adj_f(DevLayout L, const double *__restrict__ ccb, double *__restrict__ Y) {
  extern __shared__ double lds[];
  pandya_col<true>(L, Y, ccb, blockIdx.x, lds);
}
// ---- generator transpose: build_gs_white / build_gs_atan (generators.f90:4-106, 163-266)
// eta = g(h, Eden) with g = h/E (kind 0) or atan(2h/E)/2 (kind 1), written at
// (a,i) and (i,a) = -eta; with the cotangent ebar of that pair the pieces are
//   Hbar(h) += ebar dg/dh,  Ebar = ebar dg/dE  -> f diagonals and V elements of E.
__device__ __forceinline__ void gen_derivs(double h, double E, int kind, double &dh, double &dE) {
  if (kind == 0) {
    dh = 1.0 / E;
    dE = -h / (E * E);
  } else {
    const double x = 2.0 * h / E, w = 1.0 / (1.0 + x * x);
    dh = w / E;
    dE = -w * h / (E * E);
  }
}
__global__ void k_adj_eta_onebody(DevLayout L, const double *__restrict__ H, const double *__restrict__ Eb,
                                  double *__restrict__ Hb, int kind) {
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= L.nphp) return;
  const int a = L.php_a[e], i = L.php_i[e], N = L.nsp, ji = L.jj[i];
  const double *V = H + L.v_off, *F = H + L.f_off;
  double Eden = 0.0;
  for (int JT = 0; JT <= 2 * ji; JT += 2) Eden = Eden - (JT + 1) * dv(L, V, a, i, a, i, JT);
  Eden = Eden / (ji + 1.0) / (ji + 1.0);
  Eden = Eden + F[a * N + a] - F[i * N + i];
  const double h = F[a * N + i];
  const double eb = Eb[L.f_off + a * N + i] - Eb[L.f_off + i * N + a];
  if (eb == 0.0) return;
  double dh, dE;
  gen_derivs(h, Eden, kind, dh, dE);
  const double EbarD = eb * dE;
  double *HF = Hb + L.f_off, *HV = Hb + L.v_off;
  atomicAdd(HF + a * N + i, eb * dh);
  atomicAdd(HF + a * N + a, EbarD);
  atomicAdd(HF + i * N + i, -EbarD);
  for (int JT = 0; JT <= 2 * ji; JT += 2) {
    double pre;
    const long long o = dv_pos(L, a, i, a, i, JT, pre);
    if (o >= 0) atomicAdd(HV + o, -EbarD * (JT + 1) / ((ji + 1.0) * (ji + 1.0)) * pre);
  }
}
// two-body part: Ebar of every pphh element goes to the f diagonals and, through
// the J-averaged monopoles, into mbar (nsp x nsp) for k_adj_monopole
__global__ __launch_bounds__(256) void k_adj_eta_twobody(DevLayout L, const double *__restrict__ H,
                                                         const double *__restrict__ mono,
                                                         const double *__restrict__ Eb, double *__restrict__ Hb,
                                                         double *__restrict__ mbar, int kind) {
  const int q = blockIdx.x;
  const int np = L.bnp[q], nb = L.bnb[q], nh = L.bnh[q], dim = L.bdim[q], base = L.pbase[q], N = L.nsp;
  const double *F = H + L.f_off;
  const double *Vh = H + L.v_off + L.boff[q];
  const double *Vb = Eb + L.v_off + L.boff[q];
  double *HV = Hb + L.v_off + L.boff[q], *HF = Hb + L.f_off;
  for (int e = threadIdx.x; e < np * nh; e += 256) {
    const int ix = e / nh, jx = e % nh;
    const int a = L.pair_a[base + ix], b = L.pair_b[base + ix];
    const int i = L.pair_a[base + np + nb + jx], j = L.pair_b[base + np + nb + jx];
    const long long o = (long long)ix * dim + np + nb + jx, oT = (long long)(np + nb + jx) * dim + ix;
    const double eb = Vb[o] - Vb[oT];
    if (eb == 0.0) continue;
    const double Eden = mono[a * N + b] + mono[i * N + j] - mono[a * N + i] - mono[a * N + j] - mono[i * N + b] -
                        mono[j * N + b] + F[a * N + a] + F[b * N + b] - F[i * N + i] - F[j * N + j];
    double dh, dE;
    gen_derivs(Vh[o], Eden, kind, dh, dE);
    const double EbarD = eb * dE;
    HV[o] += eb * dh;  // each pphh element is written by one thread
    atomicAdd(HF + a * N + a, EbarD);
    atomicAdd(HF + b * N + b, EbarD);
    atomicAdd(HF + i * N + i, -EbarD);
    atomicAdd(HF + j * N + j, -EbarD);
    atomicAdd(mbar + a * N + b, EbarD);
    atomicAdd(mbar + i * N + j, EbarD);
    atomicAdd(mbar + a * N + i, -EbarD);
    atomicAdd(mbar + a * N + j, -EbarD);
    atomicAdd(mbar + i * N + b, -EbarD);
    atomicAdd(mbar + j * N + b, -EbarD);
  }
}
// mono(a,b) = sum_J (2J+1) v(ab,ab;J) / ((2ja+1)(2jb+1))  (twobody_monopole, basic_IMSRG.f90:2031-2046)
__global__ void k_adj_monopole(DevLayout L, const double *__restrict__ mbar, double *__restrict__ Hb) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  const int N = L.nsp;
  if (t >= N * N) return;
  const double m = mbar[t];
  if (m == 0.0) return;
  const int a = t / N, b = t % N, ja = L.jj[a], jb = L.jj[b];
  for (int JT = abs(ja - jb); JT <= ja + jb; JT += 2) {
    double pre;
    const long long o = dv_pos(L, a, b, a, b, JT, pre);
    if (o >= 0) atomicAdd(Hb + L.v_off + o, m * (JT + 1) / ((ja + 1.0) * (jb + 1.0)) * pre);
  }
}

// ---- normal-ordering transpose (normal_order, basic_IMSRG.f90:2375-2506)
// forward: E0 = sum_h (2j_h+1) f_hh + 1/2 sum_{hh',J} (2J+1) v(hh',hh';J);
// f(a,b) += sum_{h,J} (2J+1)/(2j_a+1) v(ah,bh;J) for the (a,b) of the one-body
// list with equal (l,j,tz) (f(b,a) mirrored); V unchanged.  Hb starts as a
// copy of the output cotangent Cb.
__global__ void k_adj_no_f(DevLayout L, const double *__restrict__ Cb, double *__restrict__ Hb, int herm) {
  const int t = blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= L.nob) return;
  const int a = L.ob_p[t], b = L.ob_q[t], N = L.nsp;
  if (!same_ljt(L, a, b)) return;
  const double *CF = Cb + L.f_off;
  double *HF = Hb + L.f_off;
  // output (a,b) = T(a,b) + sum; output (b,a) = herm * output(a,b) overwrites T(b,a)
  const double c = (a != b) ? CF[a * N + b] + herm * CF[b * N + a] : CF[a * N + a];
  HF[a * N + b] = c;
  if (a != b) HF[b * N + a] = 0.0;
  for (int ii = 0; ii < N; ii++) {
    if (L.con[ii] != 1) continue;
    for (int JT = abs(L.jj[ii] - L.jj[a]); JT <= L.jj[ii] + L.jj[a]; JT += 2) {
      double pre;
      const long long o = dv_pos(L, a, ii, b, ii, JT, pre);
      if (o >= 0) atomicAdd(Hb + L.v_off + o, c * (JT + 1.0) / (L.jj[a] + 1) * pre);
    }
  }
}
__global__ __launch_bounds__(256) void k_adj_no_e0(DevLayout L, const double *__restrict__ Cb, double *__restrict__ Hb) {
  const double e = Cb[0];
  const int N = L.nsp;
  if (e != 0.0)
    for (int t = threadIdx.x; t < N * N; t += 256) {
      const int i = t / N, j = t % N;
      if (L.con[i] * L.con[j] == 0) continue;
      if (i == j) atomicAdd(Hb + L.f_off + i * N + i, e * (L.jj[i] + 1));
      for (int JT = abs(L.jj[i] - L.jj[j]); JT <= L.jj[i] + L.jj[j]; JT += 2) {
        double pre;
        const long long o = dv_pos(L, i, j, i, j, JT, pre);
        if (o >= 0) atomicAdd(Hb + L.v_off + o, 0.5 * e * (JT + 1) * pre);
      }
    }
}

void launch_adj_generator(hipStream_t s, const DevLayout &L, const double *H, const double *mono,
                          const double *Eb, double *Hb, double *mbar, int kind) {
  launch_fill(s, mbar, (long long)L.nsp * L.nsp, 0.0);
  if (L.nphp > 0)
    hipLaunchKernelGGL(k_adj_eta_onebody, dim3((L.nphp + 63) / 64), dim3(64), 0, s, L, H, Eb, Hb, kind);
  hipLaunchKernelGGL(k_adj_eta_twobody, dim3(L.nblocks), dim3(256), 0, s, L, H, mono, Eb, Hb, mbar, kind);
  const int n = L.nsp * L.nsp;
  hipLaunchKernelGGL(k_adj_monopole, dim3((n + 255) / 256), dim3(256), 0, s, L, mbar, Hb);
}
void launch_adj_normal_order(hipStream_t s, const DevLayout &L, const double *Cb, double *Hb, int herm) {
  if (L.nob > 0) hipLaunchKernelGGL(k_adj_no_f, dim3((L.nob + 63) / 64), dim3(64), 0, s, L, Cb, Hb, herm);
  hipLaunchKernelGGL(k_adj_no_e0, dim3(1), dim3(256), 0, s, L, Cb, Hb);
}

// ---------------------------------------------------------------- launchers
void launch_project(hipStream_t s, const DevLayout &L, double *X, int h, int keep_e0) {
  hipLaunchKernelGGL(k_project, dim3(L.nmirror + 1), dim3(256), 0, s, L, X, h, keep_e0);
}
// lets the kernels that stage Pandya tables take more than 64 KiB of dynamic LDS
hipError_t adjoint_allow_lds(size_t bytes) {
  const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(&k_adj_a),
                                           hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
  return e != hipSuccess ? e
                         : hipFuncSetAttribute(reinterpret_cast<const void *>(&k_adj_f),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}
void launch_adjoint(hipStream_t s, const DevLayout &L, AdjArgs A) {
  A.ph = (A.mask & T222PH) && L.nccol > 0 ? 1 : 0;
  if (!(A.mask & T222PPHH)) A.n_pp = 0;
  const bool ap = A.ph && L.nphterm > 0 && A.n_chunks > 0;
  A.n_ob = (A.mask & (T121 | T221)) ? L.nsame * (L.nsp + (L.nphp * L.nJ + 255) / 256) : 0;
  A.n_122 = (A.mask & T122) ? L.npairs : 0;
  A.n_ap = ap ? (A.n_chunks + 3) / 4 : 0;
  A.n_111 = (A.mask & T111) ? (L.nob + 3) / 4 : 0;
  const long long nz = L.op_size + (A.ph ? L.nphterm + L.cwsize : 0);
  A.nfill = (int)std::min<long long>(4096, (nz + 1023) / 1024);
  const size_t lds = std::max(pandya_lds_bytes(L), 2 * 32 * 33 * sizeof(double));
  hipLaunchKernelGGL(k_adj_a, dim3(L.nccol * A.ph + L.nmirror + 1 + A.nfill), dim3(256), lds, s, L, A);
  const int ne0 = (A.mask & (T110 | T220)) ? L.nblocks + 1 : 0;
  const int nb = A.n_pp + A.n_ob + A.n_122 + A.n_ap + A.n_111 + ne0;
  if (nb > 0) hipLaunchKernelGGL(k_adj_b, dim3(nb), dim3(256), 0, s, L, A);
  const unsigned nc = (A.n_pp ? L.nmirror : 0) + (ap ? (unsigned)((L.nphterm + 255) / 256) : 0);
  if (nc > 0) hipLaunchKernelGGL(k_adj_c, dim3(nc), dim3(256), 0, s, L, A);
  if (A.ph) {
    if (A.n_sbt > 0) hipLaunchKernelGGL(k_adj_d, dim3(A.n_sbt), dim3(256), 0, s, L, A.sbt_tiles, A.Z, A.hP, A.hY);
    if (A.n_ph > 0)
      hipLaunchKernelGGL(k_adj_e, dim3(A.n_ph), dim3(256), 0, s, A.ph_probs, A.ph_tiles, (const double *)A.ccP,
                         (const double *)A.Z, A.ccY);
    hipLaunchKernelGGL(k_adj_f, dim3(L.nccol), dim3(256), pandya_lds_bytes(L), s, L, (const double *)A.ccY, A.Y);
  }
  launch_project(s, L, A.Y, A.hY, 0);
}

}  // namespace imsrg
