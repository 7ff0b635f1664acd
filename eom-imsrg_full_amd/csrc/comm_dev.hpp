// comm_dev.hpp -- device pieces of the commutator that its kernels and their
// transposes share: the Pandya column, the ph sums' descriptors, the FP64 products.
#pragma once
#include <type_traits>

#include "devfun.hpp"

namespace imsrg {

// calculate_cross_coupled (cross_coupled.f90:1190-1300): one workgroup per
// Pandya column (p,h), threads over rows (a,b); output column-major per block.
// Everything a term needs except the operator element itself is staged in
// LDS once per column: the 6j slice {jp jh JC; ja jb J'}, the pair positions
// of (h,a) and (p,b) in every J' block, block offsets and sizes, and the
// orbit quantum numbers, so each J' term does a single global load.
// ADJ: the transpose, for a cotangent of the column in cc: every term adds its
// weight times the entry to the operator's element (FP64 atomics).
template <bool ADJ>
__device__ __forceinline__ void pandya_col(const DevLayout &L, std::conditional_t<ADJ, double, const double> *__restrict__ op,
                                           std::conditional_t<ADJ, const double, double> *__restrict__ cc, int col,
                                           double *pan_lds) {
  const int q1 = L.cccol_q[col];
  const int c = col - L.cccbase[q1];
  const int p = L.cccol_p[col], h = L.cccol_h[col];
  const int JC = L.ccJ[q1], rlen = L.ccrlen[q1];
  const int jp = L.jj[p], jh = L.jj[h], lp = L.l[p], lh = L.l[h], tp = L.tz[p], th = L.tz[h];
  auto *V = op + L.v_off;
  auto *out = cc + L.ccoff[q1] + (long long)c * rlen;
  const double sq = sqrt(JC + 1.0);
  const int N = L.nsp, h6 = L.nhalf, nJ = L.nJ, nsl = h6 * h6 * nJ, NB = L.nblocks;
  const size_t NN = (size_t)N * N;
  double *S6 = pan_lds;
  long long *BO = reinterpret_cast<long long *>(S6 + nsl);
  int *BD = reinterpret_cast<int *>(BO + NB);
  int *OQ = BD + NB;                           // jj | l << 8 | (2tz + 1) << 16
  // [J'/2][a]: position of pair (h,a) in block J'; [J'/2][b]: of pair (p,b)
  // (16 bits: positions below 2^15, -1 absent; the smaller list lets eight
  // wavefronts per SIMD stay resident)
  short *PR = reinterpret_cast<short *>(OQ + N);
  short *PS = PR + nJ * N;
  {
    // every staging load of a batch is issued before the first LDS store, so
    // a thread waits for one memory latency per batch, not one per element
    const double *six0 = L.sixj + (((size_t)(jp >> 1) * h6 + (jh >> 1)) * nJ + (JC >> 1)) * (size_t)nsl;
    for (int e0 = 0; e0 < nsl; e0 += 256 * 8) {
      double v[8];
#pragma unroll
      for (int u = 0; u < 8; u++) v[u] = six0[min(e0 + (int)threadIdx.x + 256 * u, nsl - 1)];  // off any branch
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int e = e0 + (int)threadIdx.x + 256 * u;
        if (e < nsl) S6[e] = v[u];
      }
    }
    for (int e = threadIdx.x; e < NB; e += 256) {
      BO[e] = L.boff[e];
      BD[e] = L.bdim[e];
    }
    for (int e0 = 0; e0 < nJ * N; e0 += 256 * 8) {
      int vr[8], vs[8];
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int e = min(e0 + (int)threadIdx.x + 256 * u, nJ * N - 1);  // off any branch
        const int J2 = e / N, x = e - J2 * N;
        const int *pj = L.pidx + (size_t)J2 * NN;
        vr[u] = pj[h > x ? x * N + h : h * N + x];
        vs[u] = pj[p > x ? x * N + p : p * N + x];
      }
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const int e = e0 + (int)threadIdx.x + 256 * u;
        if (e < nJ * N) {
          PR[e] = (short)vr[u];
          PS[e] = (short)vs[u];
        }
      }
    }
    for (int e = threadIdx.x; e < N; e += 256) OQ[e] = L.jj[e] | (L.l[e] << 8) | ((L.tz[e] + 1) << 16);
  }
  __syncthreads();
  // the next row's orbits are loaded while the current row's terms are summed
  const int *rowa = L.ccrow_a + L.ccrbase[q1], *rowb = L.ccrow_b + L.ccrbase[q1];
  int a_next = -1, b_next = -1;
  if ((int)threadIdx.x < rlen) {
    a_next = rowa[threadIdx.x];
    b_next = rowb[threadIdx.x];
  }
  for (int r = threadIdx.x; r < rlen; r += blockDim.x) {
    const int a = a_next, b = b_next;
    if (r + (int)blockDim.x < rlen) {
      a_next = rowa[r + blockDim.x];
      b_next = rowb[r + blockDim.x];
    }
    if (a < 0) {  // zero row that makes the row count even
      if constexpr (!ADJ) out[r] = 0.0;
      continue;
    }
    const int qa = OQ[a], qbb = OQ[b];
    const int ja = qa & 255, jb = qbb & 255, la = (qa >> 8) & 255, lb = (qbb >> 8) & 255;
    const int ta = (qa >> 16) - 1, tb = (qbb >> 16) - 1;
    double val = 0.0;
    if constexpr (ADJ) val = out[r];
    if ((((la + lh) & 1) == ((lb + lp) & 1)) && (ta + th == tb + tp)) {
      const int Jmin = max(abs(jp - jb), abs(ja - jh));
      const int Jmax = min(jp + jb, ja + jh);
      // v_elem(h,a,p,b;J'): bra pair (h,a), ket pair (p,b), block (J', T2, P)
      const int qb = 2 * ((th + ta) / 2 + 1) + ((lh + la) & 1);
      const bool sw1 = h > a, sw2 = p > b;
      const double *six = S6 + ((ja >> 1) * h6 + (jb >> 1)) * nJ;
      double sm = 0.0;
      // eight J' terms a batch; the element offsets and weights first (a J'
      // past Jmax, or an element the block does not hold, reads element 0
      // with weight 0), then the eight gathers, none of them on a branch, so
      // they are in flight together
      for (int J0 = Jmin; J0 <= Jmax; J0 += 16) {
        long long off[8];
        double w[8];
        unsigned held = 0;  // bit u: the block holds the element
#pragma unroll
        for (int u = 0; u < 8; u++) {
          const int JT = min(J0 + 2 * u, Jmax);
          const int rr = PR[(JT >> 1) * N + a], ss = PS[(JT >> 1) * N + b], q = 3 * JT + qb;
          double pre = 1.0;
          if (sw1) pre = sgnp(1 + ((jh + ja - JT) >> 1));
          else if (h == a) pre = pre * M_SQRT2;
          if (sw2) pre = pre * sgnp(1 + ((jp + jb - JT) >> 1));
          else if (p == b) pre = pre * M_SQRT2;
          const bool ok = J0 + 2 * u <= Jmax && (rr | ss) >= 0;
          off[u] = ok ? BO[q] + (long long)rr * BD[q] + ss : 0;
          w[u] = ok ? pre * (double)(sgnp(JT >> 1) * (JT + 1)) * six[JT >> 1] : 0.0;
          held |= (unsigned)ok << u;
        }
        if constexpr (ADJ) {
          const double g0 = val * sgnp((jh + jb + JC) >> 1) * sq;
#pragma unroll
          for (int u = 0; u < 8; u++)
            if ((held >> u & 1) && g0 * w[u] != 0.0) atomicAdd(V + off[u], g0 * w[u]);
        } else {
          double vv[8];
#pragma unroll
          for (int u = 0; u < 8; u++) vv[u] = V[off[u]];
#pragma unroll
          for (int u = 0; u < 8; u++) sm = sm + w[u] * vv[u];
        }
      }
      if constexpr (!ADJ) val = sm * sgnp((jh + jb + JC) >> 1) * sq;
    }
    if constexpr (!ADJ) out[r] = val;
  }
}

// ---- descriptors of the ph sums (k_ph_apply)
__device__ __forceinline__ void ph_decode(unsigned long long d, int &toff, int &n1, int &n, int &o1, int &o2,
                                          double &g1, double &g2, double &pre2) {
  toff = (int)(d & 0x7FFFFFull);
  n1 = (int)((d >> 23) & 31);
  n = n1 + (int)((d >> 28) & 31);
  o1 = (int)((d >> 33) & 4095);
  o2 = (int)((d >> 45) & 4095) - n1;
  g1 = ((d >> 57) & 1) ? (((d >> 58) & 1) ? -1.0 : 1.0) : 0.0;
  g2 = ((d >> 59) & 1) ? 1.0 : 0.0;
  pre2 = ((d >> 60) & 1) ? .70710678118 : 1.0;
}
// 6j weight of term m of an output (0 past its run); index 0 when unused
__device__ __forceinline__ double ph_coef(const double *S6, int m, int n, int n1, int o1, int o2, double g1,
                                          double g2) {
  const bool s1 = m < n1, in = m < n;
  const int e = in ? (s1 ? o1 + m : o2 + m) : 0;
  return (in ? (s1 ? g1 : g2) : 0.0) * S6[e];
}

// ---- FP64 products, one 32 x 32 output tile per wavefront, operands straight
// from L1/L2 into registers: no LDS staging, no barriers.  The segments come in
// pairs over one K range, X0 X1 and X1 X0; a K chunk of 8 of a pair is eight
// 16-byte loads a lane and 16 v_mfma_f64_16x16x4 (1024 matrix-core cycles).
// The loop body is straight-line (every load made, clamped past the range), so
// the next chunk's loads stay in flight under this chunk's products, and four
// wavefronts share a SIMD.  A lane's 16 bytes are two neighbours of a K row of
// B (and of A when A is K-major): the tile's even and odd columns (rows) are
// its two 16-wide sub-tiles; or, for a row-major A, two neighbouring k of one
// row, with the K rows of B taken in the same order (k = 2 g + t in step t).
// Rows and columns past M are read clamped and never stored; k past the range
// is zeroed on both sides.  M is the leading dimension of every operand.
// NW = 4: the four wavefronts of a workgroup share one tile, each taking every
// fourth K chunk, and add their sums through LDS: a tile's K chain is a quarter
// as long, which is the time in small bases and the tail of the schedule in
// large ones.  Measured alone, in us (64 x 64 tiles of LDS slabs, the form
// before / a quadrant a wavefront / four wavefronts a tile): pp/hh emax 4 17 / - / 7,
// emax 6 43 / 25 / 20, 16 x emax 6 233 / 263 / 234, emax 7 73 / 55 / 48, emax 8
// 168 / 162 / 145 (37 TF/s); Pandya product emax 4 9.6 / 7.5 / 5.0, emax 6
// 20.5 / 15.9 / 18.0, 16 x emax 6 202 / 162 / 221, emax 8 177 / 147 (44 TF/s) / 165.
// Hence pp/hh always shares, the Pandya product while the basis' two-body part
// holds at most 3e5 elements (emax 5); the choice is the basis', so a batch has
// its instances' bits.
struct WFrag {
  dpair_t a[2][2], b[2][2];  // [segment of the pair][A: sub-tile or step, B: step]
};
template <bool Z, int NW>
__device__ __forceinline__ void wave_pair(const SegDesc &d0, const SegDesc &d1, int M, const double *__restrict__ X0,
                                          const double *__restrict__ X1, double g0, double g1, int m0, int n0, int w,
                                          double4_t acc[2][2]) {
  const int K = d0.K, lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4;
  if (8 * w >= K) return;
  const double sg0 = d0.sign * g0, sg1 = d1.sign * g1;
  const double *A0 = X0 + d0.a_off, *B0 = X1 + d0.b_off, *A1 = X1 + d1.a_off, *B1 = X0 + d1.b_off;
  // columns 2c, 2c + 1 of the tile (an odd M's last column is read with the
  // element after it, which the block's padding or next row holds)
  const int nc = n0 + 2 * c < M ? n0 + 2 * c : 0;
  const int mc = Z ? (m0 + 2 * c < M ? m0 + 2 * c : 0) : 0;
  const int r0 = Z ? 0 : min(m0 + c, M - 1) * M, r1 = Z ? 0 : min(m0 + 16 + c, M - 1) * M;
  auto fetch = [&](WFrag &f, int k) {
    if (Z) {
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const int o = min(k + 4 * t + g, K - 1) * M;
        f.a[0][t] = *(const dpair_t *)(A0 + (o + mc));
        f.b[0][t] = *(const dpair_t *)(B0 + (o + nc));
        f.a[1][t] = *(const dpair_t *)(A1 + (o + mc));
        f.b[1][t] = *(const dpair_t *)(B1 + (o + nc));
      }
    } else {
      // (a pair whose second k is past the range reads the element after it)
      const int kp = min(k + 2 * g, K - 1);
      f.a[0][0] = *(const dpair_t *)(A0 + (r0 + kp));
      f.a[0][1] = *(const dpair_t *)(A0 + (r1 + kp));
      f.a[1][0] = *(const dpair_t *)(A1 + (r0 + kp));
      f.a[1][1] = *(const dpair_t *)(A1 + (r1 + kp));
#pragma unroll
      for (int t = 0; t < 2; t++) {
        const int o = min(k + 2 * g + t, K - 1) * M + nc;
        f.b[0][t] = *(const dpair_t *)(B0 + o);
        f.b[1][t] = *(const dpair_t *)(B1 + o);
      }
    }
  };
  auto product = [&](WFrag &f, int k) {
    if (K - k < 8) {
#pragma unroll
      for (int t = 0; t < 2; t++)
        if (k + (Z ? 4 * t + g : 2 * g + t) >= K) {
#pragma unroll
          for (int q = 0; q < 2; q++) {
            f.b[q][t] = (dpair_t){0.0, 0.0};
            if (Z) f.a[q][t] = (dpair_t){0.0, 0.0};
            else f.a[q][0][t] = f.a[q][1][t] = 0.0;
          }
        }
    }
#pragma unroll
    for (int q = 0; q < 2; q++) {
      f.a[q][0] *= q ? sg1 : sg0;
      f.a[q][1] *= q ? sg1 : sg0;
#pragma unroll
      for (int t = 0; t < 2; t++)
#pragma unroll
        for (int ti = 0; ti < 2; ti++)
#pragma unroll
          for (int tj = 0; tj < 2; tj++)
            acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(Z ? f.a[q][t][ti] : f.a[q][ti][t], f.b[q][t][tj],
                                                               acc[ti][tj], 0, 0, 0);
    }
  };
  constexpr int S = 8 * NW;
  WFrag f0, f1;
  fetch(f0, 8 * w);
  for (int k = 8 * w; k < K; k += 2 * S) {
    fetch(f1, k + S);
    product(f0, k);
    if (k + S >= K) break;
    fetch(f0, k + 2 * S);
    product(f1, k + S);
  }
}
// segments [s0, s1) of a problem, which are pairs
template <bool Z, int NW>
__device__ __forceinline__ void wave_segments(const SegProb &p, int s0, int s1, const double *__restrict__ X0,
                                              const double *__restrict__ X1, double g0, double g1, int m0, int n0,
                                              int w, double4_t acc[2][2]) {
  for (int s = s0; s < s1; s += 2)
    wave_pair<Z, NW>(p.seg[s], p.seg[s + 1], p.M, X0, X1, g0, g1, m0, n0, w, acc);
}
// C tile = A B, A row-major (lda), B K-major (ldb), one 32 x 32 tile for four
// wavefronts as above, summed through LDS; reads and writes stay inside
// M x K, K x N and M x N except the neighbour an odd K's or N's last 16-byte
// pair takes (in a channel block: its padding or next row).
struct alignas(16) SplitSmem {  // (read and written in pairs)
  double s[4][32][34];
};
__device__ __forceinline__ void plain_tile(const GemmProb &p, int m0, int n0, const double *__restrict__ A,
                                           const double *__restrict__ B, double *__restrict__ C, SplitSmem &S) {
  const int lane = threadIdx.x & 63, c = lane & 15, g = lane >> 4, K = p.K;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const double *Ap = A + p.a_off, *Bp = B + p.b_off;
  const int nc = n0 + 2 * c < p.N ? n0 + 2 * c : 0, kl = (K & 1) ? K - 1 : K - 2;
  const int r0 = min(m0 + c, p.M - 1) * p.lda, r1 = min(m0 + 16 + c, p.M - 1) * p.lda;
  double4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) acc[i][j] = (double4_t){0.0, 0.0, 0.0, 0.0};
  struct Frag {
    dpair_t a[2], b[2];
  };
  auto fetch = [&](Frag &f, int k) {
    const int kp = min(k + 2 * g, kl);
    f.a[0] = *(const dpair_t *)(Ap + (r0 + kp));
    f.a[1] = *(const dpair_t *)(Ap + (r1 + kp));
#pragma unroll
    for (int t = 0; t < 2; t++) f.b[t] = *(const dpair_t *)(Bp + (min(k + 2 * g + t, K - 1) * p.ldb + nc));
  };
  auto product = [&](Frag &f, int k) {
    if (K - k < 8) {
#pragma unroll
      for (int t = 0; t < 2; t++)
        if (k + 2 * g + t >= K) {
          f.b[t] = (dpair_t){0.0, 0.0};
          f.a[0][t] = f.a[1][t] = 0.0;
        }
    }
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
      for (int ti = 0; ti < 2; ti++)
#pragma unroll
        for (int tj = 0; tj < 2; tj++)
          acc[ti][tj] = __builtin_amdgcn_mfma_f64_16x16x4f64(f.a[ti][t], f.b[t][tj], acc[ti][tj], 0, 0, 0);
  };
  if (8 * wave < K) {
    Frag f0, f1;
    fetch(f0, 8 * wave);
    for (int k = 8 * wave; k < K; k += 64) {
      fetch(f1, k + 32);
      product(f0, k);
      if (k + 32 >= K) break;
      fetch(f0, k + 64);
      product(f1, k + 32);
    }
  }
  __syncthreads();
#pragma unroll
  for (int ti = 0; ti < 2; ti++)
#pragma unroll
    for (int v = 0; v < 4; v++)
      *(double2 *)&S.s[wave][16 * ti + g + 4 * v][2 * c] = make_double2(acc[ti][0][v], acc[ti][1][v]);
  __syncthreads();
  const int u = threadIdx.x >> 4, w = threadIdx.x & 15;
#pragma unroll
  for (int i = 0; i < 2; i++)
#pragma unroll
    for (int j = 0; j < 2; j++) {
      const int row = m0 + 2 * u + i, col = n0 + 2 * w + j;
      double x = 0.0;
#pragma unroll
      for (int k = 0; k < 4; k++) x += S.s[k][2 * u + i][2 * w + j];
      if (row < p.M && col < p.N) C[p.c_off + (long long)row * p.ldc + col] = x;
    }
}

}  // namespace imsrg
