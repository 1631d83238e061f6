// Interstitial (IPW) part of the wave-function products by FFT convolution,
// replacing the FFTW path of wavefproducts.f:576-758 (plans fft.f:90-93).
//
// Reference (SUBTYPE 2, noinv, fullpw optional):
//   phi1(r) = conjg(FFT_bwd(c1)(r) / sqrt(vol)) [* theta(r)]    (:624-633)
//   psi2(r) = FFT_bwd(c2)(r) / nnfft                             (:658-665)
//   cprod(b2,b1,k,ig) = FFT_fwd(phi1*psi2)(imati.(Gm_ig - g_k) mod nfft)
//                                                                (:670-684)
// with FFT_bwd = sum_G c(G) e^{+2 pi i G.r/N}, FFT_fwd = sum_r p(r)
// e^{-2 pi i G.r/N}, both unnormalised (FFTW BACKWARD / FORWARD).
//
// Every transform here is a pruned separable DFT evaluated as FP64 complex
// MFMA products on v_mfma_f64_16x16x4f64.  Wave-function coefficients live
// in a 16^3 box of Fourier components (-8..7 per axis), so the backward
// transform starts from that box and the forward transform only produces
// the box (then gathers the mixed-basis IPWs):
//   pw_inverse  (one workgroup per state, waves take z planes):
//     U(gx,gy) = sum_gz e^{+i..gz z} C(gz,gy,gx)           (VALU, from LDS)
//     V(gx,y)  = U x E2         (MFMA, K = 16 gy)
//     psi(y,x) = V^T x E1       (MFMA, K = 16 gx) -> grid, scaled
//   pw_pair_xy (one wave per pair (b1,b2), workgroup = 4 b1 sharing b2):
//     R^T(y,gx) = (phi1*psi2)(y,x) x F1(x,gx)   (MFMA, K = N1)
//     Q(gy,gx)  = F2(gy,y) x R^T(y,gx)          (MFMA, K = N2)  -> slab
//   pw_pair_z  (one workgroup per pair):
//     cprod(t, ig) = sum_z e^{-i..gz z} Q_z(gy,gx) at the IPW's box point.
// The accumulator layout of one MFMA (column j = lane%16, rows lane/16+4r)
// is exactly the operand layout the next MFMA needs, so no transposes go
// through LDS between passes.
// Square planes (N1 = N2) of the usual FFT sizes take kernels of their own,
// pw_states_kernel and pw_pair_square_kernel below, for up to 16 k points per
// launch.
#include <algorithm>
#include <cmath>
#include <vector>

#include "plan.hpp"

namespace {

constexpr int NT = 256;

__device__ inline double2 twid(long m, int N, double sign) {
  long r = m % N;
  if (r < 0) r += N;
  double s, c;
  sincospi(2.0 * (double)r / (double)N, &s, &c);
  return make_double2(c, sign * s);
}

__device__ inline double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

// acc += a * b (complex, one 16x16x4 MFMA step)
__device__ inline void cmfma(d4_t &ar, d4_t &ai, double2 a, double2 b) {
  ar = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, ar, 0, 0, 0);
  ar = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, ar, 0, 0, 0);
  ai = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, ai, 0, 0, 0);
  ai = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, ai, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// Backward transform of states: s < nA -> (kA, bandA+s) as phi1, else
// (kB, bandB+s-nA) as psi2.  grids[s] is N3 x N2 x N1 (x fastest).
template <int NB>
__global__ __launch_bounds__(NT) void pw_inverse_kernel(
    const double2 *__restrict__ cpw, int maxgpt, int nband, const int *__restrict__ gidx,
    const int *__restrict__ ngpt, int kA, int bandA, int nA, int kB, int bandB, int N1, int N2,
    int N3, double scaleA, double scaleB, const double2 *__restrict__ step,
    double2 *__restrict__ grids) {
  __shared__ double Cr[PW_BOX * PW_BOX * PW_BOX], Ci[PW_BOX * PW_BOX * PW_BOX];
  __shared__ double2 tz[64][PW_BOX];  // N3 <= 64
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  const int s = blockIdx.x;
  const bool occ = s < nA;
  const int kq = occ ? kA : kB;
  const int band = occ ? bandA + s : bandB + (s - nA);
  for (int e = tid; e < PW_BOX * PW_BOX * PW_BOX; e += NT) {
    Cr[e] = 0.0;
    Ci[e] = 0.0;
  }
  for (int e = tid; e < N3 * PW_BOX; e += NT) {
    const int z = e / PW_BOX, g = e % PW_BOX;
    tz[z][g] = twid((long)(g - PW_OFF) * z, N3, +1.0);
  }
  __syncthreads();
  const int ng = ngpt[kq];
  const double2 *c = cpw + (long)maxgpt * (band + (long)nband * kq);
  const int *gi = gidx + (long)maxgpt * kq;
  for (int ig = tid; ig < ng; ig += NT) {
    const int b = gi[ig];
    Cr[b] = c[ig].x;
    Ci[b] = c[ig].y;
  }
  __syncthreads();

  // constant MFMA operands: E2(gy, y) and E1(gx, x), lane layout B[k][j]
  double2 E2[NB][4], E1[NB][4];
#pragma unroll
  for (int b = 0; b < NB; b++)
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      const int g = 4 * kk + lk - PW_OFF, j = 16 * b + lr;
      E2[b][kk] = j < N2 ? twid((long)g * j, N2, +1.0) : make_double2(0.0, 0.0);
      E1[b][kk] = j < N1 ? twid((long)g * j, N1, +1.0) : make_double2(0.0, 0.0);
    }

  const long NN = (long)N1 * N2 * N3;
  double2 *out = grids + (long)s * NN;
  const double scale = occ ? scaleA : scaleB;
  for (int z = wv; z < N3; z += NT / 64) {
    double2 U[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      const int gy = 4 * kk + lk;
      double ur = 0.0, ui = 0.0;
#pragma unroll 4
      for (int gz = 0; gz < PW_BOX; gz++) {
        const double2 t = tz[z][gz];
        const int b = gz * PW_BOX * PW_BOX + gy * PW_BOX + lr;
        const double cr = Cr[b], ci = Ci[b];
        ur += t.x * cr - t.y * ci;
        ui += t.x * ci + t.y * cr;
      }
      U[kk] = make_double2(ur, ui);
    }
    // y and x passes; for grids of up to 32 points per axis with three real
    // MFMAs per complex product (Gauss): t1 = ar.br, t2 = ai.bi,
    // t3 = (ar + ai)(br + bi); re = t1 - t2, im = t3 - t1 - t2.  Larger grids
    // keep four (the third accumulators would cost the second wave per SIMD).
    constexpr bool M3 = NB <= 2;
#pragma unroll
    for (int mb = 0; mb < NB; mb++) {
      if (16 * mb >= N2) continue;
      d4_t vr = {0, 0, 0, 0}, vi = {0, 0, 0, 0}, vs = {0, 0, 0, 0};
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {
        const double2 u = U[kk], e = E2[mb][kk];
        if (M3) {
          vr = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x, e.x, vr, 0, 0, 0);
          vi = __builtin_amdgcn_mfma_f64_16x16x4f64(u.y, e.y, vi, 0, 0, 0);
          vs = __builtin_amdgcn_mfma_f64_16x16x4f64(u.x + u.y, e.x + e.y, vs, 0, 0, 0);
        } else {
          cmfma(vr, vi, u, e);
        }
      }
      const d4_t yr = M3 ? vr - vi : vr, yi = M3 ? vs - vr - vi : vi;
#pragma unroll
      for (int nb = 0; nb < NB; nb++) {
        if (16 * nb >= N1) continue;
        d4_t tr = {0, 0, 0, 0}, ti = {0, 0, 0, 0}, ts = {0, 0, 0, 0};
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          const double2 e = E1[nb][kk];
          if (M3) {
            tr = __builtin_amdgcn_mfma_f64_16x16x4f64(yr[kk], e.x, tr, 0, 0, 0);
            ti = __builtin_amdgcn_mfma_f64_16x16x4f64(yi[kk], e.y, ti, 0, 0, 0);
            ts = __builtin_amdgcn_mfma_f64_16x16x4f64(yr[kk] + yi[kk], e.x + e.y, ts, 0, 0, 0);
          } else {
            cmfma(tr, ti, make_double2(yr[kk], yi[kk]), e);
          }
        }
        const d4_t orr = M3 ? tr - ti : tr, oi = M3 ? ts - tr - ti : ti;
        const int x = 16 * nb + lr;
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int y = 16 * mb + lk + 4 * r;
          if (x < N1 && y < N2) {
            const long g = x + (long)N1 * (y + (long)N2 * z);
            double2 v = make_double2(orr[r], oi[r]);
            if (occ) {
              v = make_double2(v.x * scale, -v.y * scale);
              if (step) v = cmul(v, step[g]);  // fullpw: conj(psi1)/sqrt(vol) * theta
            } else {
              v.x *= scale;
              v.y *= scale;
            }
            out[g] = v;
          }
        }
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Forward passes x and y of the products of pairs (b1, b2).
// grids: [0, nocc) phi1 of the occupied states, [nocc, nocc+nunocc) psi2.
// slab[(b1*nunocc + b2)][z][gy][gx], 16 x 16 per plane.
template <int NB>
__global__ __launch_bounds__(NT) void pw_pair_xy_kernel(const double2 *__restrict__ grids,
                                                        int nocc, int nunocc, int N1, int N2,
                                                        int N3, double2 *__restrict__ slab) {
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  const int b2 = blockIdx.x;
  const int b1 = blockIdx.y * (NT / 64) + wv;
  if (b1 >= nocc) return;  // whole wave; this kernel has no workgroup barrier
  const long NN = (long)N1 * N2 * N3;
  const double2 *p1 = grids + (long)b1 * NN;
  const double2 *p2 = grids + (long)(nocc + b2) * NN;
  double2 *S = slab + ((long)b1 * nunocc + b2) * N3 * PW_BOX * PW_BOX;
  constexpr int KX = 4 * NB;  // x steps (N1 <= 16*NB)
  double2 F1[KX], F2[KX];
#pragma unroll
  for (int kk = 0; kk < KX; kk++) {
    const int x = 4 * kk + lk;  // B[k = x][j = gx]
    F1[kk] = x < N1 ? twid((long)(lr - PW_OFF) * x, N1, -1.0) : make_double2(0.0, 0.0);
    const int y = 4 * kk + lk;  // A[i = gy][k = y]
    F2[kk] = y < N2 ? twid((long)(lr - PW_OFF) * y, N2, -1.0) : make_double2(0.0, 0.0);
  }
  for (int z = 0; z < N3; z++) {
    d4_t xr[NB], xi[NB];
#pragma unroll
    for (int mb = 0; mb < NB; mb++) {
      xr[mb] = d4_t{0, 0, 0, 0};
      xi[mb] = d4_t{0, 0, 0, 0};
      if (16 * mb >= N2) continue;
      const int y = 16 * mb + lr;
#pragma unroll
      for (int kk = 0; kk < KX; kk++) {
        if (4 * kk < N1) {  // wave-uniform guard (keeps the loop unrollable)
          const int x = 4 * kk + lk;
          double2 a = make_double2(0.0, 0.0);
          if (x < N1 && y < N2) {
            const long g = x + (long)N1 * (y + (long)N2 * z);
            a = cmul(p1[g], p2[g]);
          }
          cmfma(xr[mb], xi[mb], a, F1[kk]);
        }
      }
    }
    d4_t qr = {0, 0, 0, 0}, qi = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < KX; kk++)
      if (4 * kk < N2) cmfma(qr, qi, F2[kk], make_double2(xr[kk / 4][kk % 4], xi[kk / 4][kk % 4]));
    double2 *Sz = S + (long)z * PW_BOX * PW_BOX;
#pragma unroll
    for (int r = 0; r < 4; r++) Sz[(lk + 4 * r) * PW_BOX + lr] = make_double2(qr[r], qi[r]);
  }
}

// Fused forward transform of the products of pairs (b1, b2): passes x and y
// on MFMA as in pw_pair_xy_kernel, then per plane the 16x16 result goes
// through a per-wave LDS tile into the z pass, accumulated directly at the
// mixed-basis IPWs each lane owns (ig = lane + 64 j), with twiddles
// e^{-2 pi i gz z/N3} from an LDS table.  No slab round trip through HBM.
// Requires ngptm <= 64*PW_FOUT.
constexpr int PW_FOUT = 16;
template <int NB>
__global__ __launch_bounds__(NT) void pw_pair_fused_kernel(
    const double2 *__restrict__ grids, int nocc, int nunocc, int N1, int N2, int N3,
    const int *__restrict__ oidx, int ngptm, double2 *__restrict__ M, long ldm, long t0, int col0) {
  constexpr int KX = 4 * NB;
  __shared__ double2 tz[64][PW_BOX];               // e^{-2 pi i (g-8) z/N3}
  __shared__ double2 Qs[NT / 64][PW_BOX * PW_BOX];  // per-wave plane result
  // MFMA operands of the x and y passes, per lane: e^{-2 pi i (lr-8) x/N}
  // with x = 4kk + lk (kept in LDS rather than registers, for occupancy)
  __shared__ double2 F1s[KX][64], F2s[KX][64];
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  for (int e = tid; e < N3 * PW_BOX; e += NT) {
    const int z = e / PW_BOX, g = e % PW_BOX;
    tz[z][g] = twid((long)(g - PW_OFF) * z, N3, -1.0);
  }
  for (int e = tid; e < KX * 64; e += NT) {
    const int kk = e >> 6, ln = e & 63, x = 4 * kk + (ln >> 4), g = (ln & 15) - PW_OFF;
    F1s[kk][ln] = x < N1 ? twid((long)g * x, N1, -1.0) : make_double2(0.0, 0.0);
    F2s[kk][ln] = x < N2 ? twid((long)g * x, N2, -1.0) : make_double2(0.0, 0.0);
  }
  __syncthreads();
  const int b2 = blockIdx.x;
  const int b1 = blockIdx.y * (NT / 64) + wv;
  if (b1 >= nocc) return;  // whole wave; no workgroup barrier after this point
  const long NN = (long)N1 * N2 * N3;
  const double2 *p1 = grids + (long)b1 * NN;
  const double2 *p2 = grids + (long)(nocc + b2) * NN;
  int ob[PW_FOUT];
  double2 acc[PW_FOUT];
#pragma unroll
  for (int j = 0; j < PW_FOUT; j++) {
    const int ig = l + 64 * j;
    ob[j] = ig < ngptm ? oidx[ig] : -1;
    acc[j] = make_double2(0.0, 0.0);
  }
  double2 *Q = Qs[wv];
  for (int z = 0; z < N3; z++) {
    d4_t xr[NB], xi[NB];
#pragma unroll
    for (int mb = 0; mb < NB; mb++) {
      xr[mb] = d4_t{0, 0, 0, 0};
      xi[mb] = d4_t{0, 0, 0, 0};
      if (16 * mb >= N2) continue;
      const int y = 16 * mb + lr;
#pragma unroll
      for (int kk = 0; kk < KX; kk++) {
        if (4 * kk < N1) {
          const int x = 4 * kk + lk;
          double2 a = make_double2(0.0, 0.0);
          if (x < N1 && y < N2) {
            const long g = x + (long)N1 * (y + (long)N2 * z);
            a = cmul(p1[g], p2[g]);
          }
          cmfma(xr[mb], xi[mb], a, F1s[kk][l]);
        }
      }
    }
    d4_t qr = {0, 0, 0, 0}, qi = {0, 0, 0, 0};
#pragma unroll
    for (int kk = 0; kk < KX; kk++)
      if (4 * kk < N2) cmfma(qr, qi, F2s[kk][l], make_double2(xr[kk / 4][kk % 4], xi[kk / 4][kk % 4]));
    // Q(gy, gx): lane holds gx = lr, gy = lk + 4r
#pragma unroll
    for (int r = 0; r < 4; r++) Q[(lk + 4 * r) * PW_BOX + lr] = make_double2(qr[r], qi[r]);
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
#pragma unroll
    for (int j = 0; j < PW_FOUT; j++) {
      if (ob[j] >= 0) {
        const double2 t = tz[z][ob[j] >> 8];
        const double2 v = Q[ob[j] & 255];
        acc[j].x += t.x * v.x - t.y * v.y;
        acc[j].y += t.x * v.y + t.y * v.x;
      }
    }
    __builtin_amdgcn_wave_barrier();  // Q is rewritten by the next plane
  }
  double2 *out = M + (t0 + (long)b1 * nunocc + b2) * ldm + col0;
#pragma unroll
  for (int j = 0; j < PW_FOUT; j++) {
    const int ig = l + 64 * j;
    if (ig < ngptm) out[ig] = acc[j];
  }
}

// ---------------------------------------------------------------------------
// The transforms of square planes (N1 = N2 = N): even/odd DFTs on grids stored
// in the order in which the pair kernel's MFMAs read them.
//
// Even/odd form of a DFT between N points and the box frequencies g = -8..7:
// the points are taken in pairs (w, N - w), w = 0 .. NP-1, the point 0 together
// with N/2 (N even) or with itself (N odd).  With s, d the sum and the
// difference of a pair,
//     sum_x p(x) e^{-i a g x} = sum_w cos(a g w) s_w - i sin(a g w) d_w,
// complex values times real coefficients: N/4 steps of two real MFMAs
// instead of N/4 of three (Gauss) or four.  The pair w = 0 of an even N has
// the real coefficients (1 +- (-1)^g)/2 for s and d.
//
// K index of the MFMAs: slot t holds the pairs w = 4t + lk (lk = lane/16), one
// step for s and one for d.  If one or two pairs are left over, a last slot
// has a single step, s in the lanes lk = 0, 1 and d of the same pairs in
// lk = 2, 3; three left over take a slot with lk = 3 at coefficient zero.
template <int N>
struct Pairs {
  static constexpr int NP = (N + 1) / 2, FULL = NP / 4, REM = NP % 4;
  static constexpr int S = FULL + (REM ? 1 : 0);  // slots
  static constexpr bool HALF = REM == 1 || REM == 2;  // the last slot is a single step
  static constexpr int STEPS = 2 * S - (HALF ? 1 : 0);
  __device__ static bool half(int t) { return HALF && t == FULL; }
  __device__ static int pair(int t, int lk) {  // w of slot t (a valid pair where padded)
    const int w = 4 * t + (half(t) ? (lk & 1) : lk);
    return w < NP ? w : NP - 1;
  }
  __device__ static int partner(int w) { return w ? N - w : (N % 2 ? 0 : N / 2); }
  // coefficients of s and d of pair w for frequency g
  __device__ static double2 coef(int w, int g) {
    if (w == 0) {
      if (N % 2) return make_double2(0.5, 0.0);  // s = 2 p(0)
      return g & 1 ? make_double2(0.0, 1.0) : make_double2(1.0, 0.0);
    }
    return twid((long)g * w, N, +1.0);
  }
  // coefficient of step st for lane lk and frequency g
  __device__ static double step_coef(int st, int lk, int g) {
    const int t = st / 2;
    if (4 * t + (half(t) ? (lk & 1) : lk) >= NP) return 0.0;
    const double2 c = coef(pair(t, lk), g);
    return (half(t) ? lk < 2 : st % 2 == 0) ? c.x : c.y;
  }
};

// Partner of plane zp and the coefficients of its pair (runtime N3).
__device__ inline int plane_partner(int zp, int N3) { return zp ? N3 - zp : (N3 % 2 ? 0 : N3 / 2); }
__device__ inline double2 plane_coef(int zp, int g, int N3) {
  if (zp == 0) {
    if (N3 % 2) return make_double2(0.5, 0.0);
    return g & 1 ? make_double2(0.0, 1.0) : make_double2(1.0, 0.0);
  }
  return twid((long)g * zp, N3, +1.0);
}

// Grid of one state: planes in pairs zp (z and its partner), whose 2 S row
// slots of two members each fill S row blocks of 16 rows: row lr of block rb is
// member (lr/4)%2 of the pair w = pair(tt, lr%4), slot 2 rb + lr/8 = S zz + tt of
// plane zz.  Per row block the slots t along x with both members of a pair, 64
// lanes (lk, lr) of 16 bytes each -- one MFMA operand, 1 KB, read by one load:
//     element ((((zp S + rb) S + t) 2 + member) 64 + lane.
// Read in the natural order instead (16 rows of 64 bytes per load, twice that
// for the partners), the pair kernel was bound by the vector L1's line rate.
template <int N>
struct Rows {
  static constexpr int S = Pairs<N>::S;
  __device__ static int plane(int rb, int lr) { return (2 * rb + (lr >> 3)) / S; }
  __device__ static int y(int rb, int lr) {
    const int w = Pairs<N>::pair((2 * rb + (lr >> 3)) % S, lr & 3);
    return (lr >> 2) & 1 ? Pairs<N>::partner(w) : w;
  }
};
__host__ __device__ constexpr int pair_slots(int N) { return ((N + 1) / 2 + 3) / 4; }
__host__ __device__ constexpr long square_grid(int N, int N3) {
  return (long)((N3 + 1) / 2) * pair_slots(N) * pair_slots(N) * 128;
}

// k points of one launch: states at k1 and k2.
constexpr int PW_KMAX = 16;
struct KList {
  int k1[PW_KMAX], k2[PW_KMAX];
};

// frequency of index i = 0..15 in the order 0, 1, .., 7, -8, -1, .., -7
__device__ inline int freq_of(int i) { return i < 8 ? i : (i == 8 ? -8 : 8 - i); }

// Backward transforms of the states of the k points of a launch (blockIdx.y):
// s < nA as phi1 = conj(psi) scaleA [* theta], else as psi2 = psi scaleB, into
// the layout above.  One workgroup per state; a wave takes pairs of planes.
//   z: the box is kept as sums and differences of the frequencies +-gz, so
//      both planes of a pair come from one sweep: C +- i S (VALU, from LDS);
//   y: V(gx, row) with sums and differences over +-gy (real coefficients);
//   x: both points of a pair from C = sum cos V and S = sum sin V, C +- i S.
// Bound by the z pass's VALU and LDS reads and by the 16 bytes per point it
// writes (24^3, 416 states: 28 us per k point, 92 MB).
template <int N>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void pw_states_kernel(
    const double2 *__restrict__ cpw, int maxgpt, int nband, const int *__restrict__ gidx,
    const int *__restrict__ ngpt, KList kl, int bandA, int nA, int bandB, int N3, double scaleA,
    double scaleB, const double2 *__restrict__ step, double2 *__restrict__ grids) {
  using P = Pairs<N>;
  constexpr int S = P::S, XB = (S + 3) / 4;
  constexpr int COL = PW_BOX * PW_BOX;
  __shared__ double2 C[PW_BOX * COL];
  __shared__ double tc[32][17];  // cos of gz = 0..8, then -sin(8), sin(1..7)
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  const int s = blockIdx.x;
  const bool occ = s < nA;
  const int kq = occ ? kl.k1[blockIdx.y] : kl.k2[blockIdx.y];
  const int band = occ ? bandA + s : bandB + (s - nA);
  const int ZP = (N3 + 1) / 2;
  for (int e = tid; e < PW_BOX * COL; e += NT) C[e] = make_double2(0.0, 0.0);
  for (int e = tid; e < ZP * 17; e += NT) {
    const int zp = e / 17, i = e % 17;
    const double2 t = twid((long)(i < 9 ? i : (i == 9 ? 8 : i - 9)) * zp, N3, +1.0);
    tc[zp][i] = i < 9 ? t.x : (i == 9 ? -t.y : t.y);
  }
  __syncthreads();
  const int ng = ngpt[kq];
  const double2 *c = cpw + (long)maxgpt * (band + (long)nband * kq);
  const int *gi = gidx + (long)maxgpt * kq;
  for (int ig = tid; ig < ng; ig += NT) C[gi[ig]] = c[ig];
  __syncthreads();
  {  // per (gy, gx): c_0, sums of +-1..7, c_-8, differences of +-1..7
    double2 v[PW_BOX];
#pragma unroll
    for (int g = 0; g < PW_BOX; g++) v[g] = C[g * COL + tid];
    C[tid] = v[PW_OFF];
    C[8 * COL + tid] = v[0];
#pragma unroll
    for (int g = 1; g < 8; g++) {
      const double2 a = v[PW_OFF + g], b = v[PW_OFF - g];
      C[g * COL + tid] = make_double2(a.x + b.x, a.y + b.y);
      C[(8 + g) * COL + tid] = make_double2(a.x - b.x, a.y - b.y);
    }
  }
  // coefficients.  y: steps cos(a g y) for g = 4 st + lk (st = 0, 1), cos(8 a y)
  // in lane lk = 0, sin(a g y) (lane lk = 0, st = 3: g = 8).
  double ey[S][5], ec[XB][4], es[XB][4];
#pragma unroll
  for (int rb = 0; rb < S; rb++) {
    const int y = Rows<N>::y(rb, lr);
#pragma unroll
    for (int st = 0; st < 2; st++) {
      const double2 t = twid((long)(4 * st + lk) * y, N, +1.0);
      const double2 t8 = twid(8l * y, N, +1.0);
      ey[rb][st] = t.x;
      if (st == 0) ey[rb][2] = lk == 0 ? t8.x : 0.0;
      ey[rb][3 + st] = st == 0 && lk == 0 ? t8.y : t.y;
    }
  }
#pragma unroll
  for (int xb = 0; xb < XB; xb++) {
    const int t = 4 * xb + (lr >> 2) < S ? 4 * xb + (lr >> 2) : S - 1;
#pragma unroll
    for (int kk = 0; kk < 4; kk++) {
      const int w = P::pair(t, lr & 3), g = freq_of(4 * kk + lk);
      // (for an odd N the point 0 is both members)
      const double2 f = N % 2 && w == 0 ? make_double2(1.0, 0.0) : P::coef(w, g);
      ec[xb][kk] = f.x;
      es[xb][kk] = f.y;
    }
  }
  __syncthreads();
  const long GS = square_grid(N, N3);
  double2 *out = grids + ((long)blockIdx.y * gridDim.x + s) * GS;
  const double scale = occ ? scaleA : scaleB;
  const int gxi = freq_of(lr) + PW_OFF;
  const bool real0 = N % 2 == 0 && lk == 0;  // pair w = 0 in slot 0
  for (int zp = wv; zp < ZP; zp += NT / 64) {
    d2_t Uc[4], Us[4];
#pragma unroll
    for (int kk = 0; kk < 4; kk++) Uc[kk] = Us[kk] = d2_t{0.0, 0.0};
    auto at = [&](int e, int kk) {
      return *(const d2_t *)&C[e * COL + (freq_of(4 * kk + lk) + PW_OFF) * PW_BOX + gxi];
    };
    if (zp == 0) {  // planes 0 and N3/2 (or 0 again): sums only, signs (-1)^gz
      const double alt = N3 % 2 ? 1.0 : -1.0;
#pragma unroll
      for (int e = 0; e < 9; e++) {
        const double sg = e & 1 ? alt : 1.0;
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          const d2_t v = at(e, kk);
          Uc[kk] += v;
          Us[kk] += sg * v;
        }
      }
    } else {
#pragma unroll
      for (int e = 0; e < PW_BOX; e++) {
        const double cz = tc[zp][e < 9 ? e : 0], sz = tc[zp][e < 8 ? 0 : e + 1];
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          const d2_t v = at(e, kk);
          if (e < 9) Uc[kk] += cz * v;
          if (e >= 8) Us[kk] += sz * v;
        }
      }
#pragma unroll
      for (int kk = 0; kk < 4; kk++) {  // C + i S, C - i S
        const d2_t a = Uc[kk], b = Us[kk];
        Uc[kk] = d2_t{a.x - b.y, a.y + b.x};
        Us[kk] = d2_t{a.x + b.y, a.y - b.x};
      }
    }
    // operands of the y pass: sums, c_-8, differences (lane lk = 0: g = 0 has
    // no partner and -8 stands for the sine of 8)
    d2_t yo[2][5];
#pragma unroll
    for (int zz = 0; zz < 2; zz++) {
      const d2_t *U = zz ? Us : Uc;
      yo[zz][0] = lk == 0 ? U[0] : U[0] + U[2];
      yo[zz][1] = U[1] + U[3];
      yo[zz][2] = U[2];
      const d2_t d0 = lk == 0 ? -U[2] : U[0] - U[2], d1 = U[1] - U[3];
      yo[zz][3] = d2_t{-d0.y, d0.x};  // i d
      yo[zz][4] = d2_t{-d1.y, d1.x};
    }
#pragma unroll
    for (int rb = 0; rb < S; rb++) {
      // V(gx, row), rows gx = freq_of(lk + 4r)
      d4_t vr, vi;
      auto ypass = [&](int zz) {
        vr = d4_t{0, 0, 0, 0};
        vi = d4_t{0, 0, 0, 0};
#pragma unroll
        for (int st = 0; st < 5; st++) {
          vr = __builtin_amdgcn_mfma_f64_16x16x4f64(yo[zz][st].x, ey[rb][st], vr, 0, 0, 0);
          vi = __builtin_amdgcn_mfma_f64_16x16x4f64(yo[zz][st].y, ey[rb][st], vi, 0, 0, 0);
        }
      };
      const bool mixed = S % 2 == 1 && rb == S / 2;  // rows 0..7 of plane 0, 8..15 of plane 1
      ypass(2 * rb >= S ? 1 : 0);
      if (mixed) {
        const d4_t ar = vr, ai = vi;
        ypass(1);
        vr = lr < 8 ? ar : vr;
        vi = lr < 8 ? ai : vi;
      }
      const int zz = Rows<N>::plane(rb, lr);
#pragma unroll
      for (int xb = 0; xb < XB; xb++) {
        d4_t cr = {0, 0, 0, 0}, ci = {0, 0, 0, 0}, sr = {0, 0, 0, 0}, si = {0, 0, 0, 0};
#pragma unroll
        for (int kk = 0; kk < 4; kk++) {
          cr = __builtin_amdgcn_mfma_f64_16x16x4f64(ec[xb][kk], vr[kk], cr, 0, 0, 0);
          ci = __builtin_amdgcn_mfma_f64_16x16x4f64(ec[xb][kk], vi[kk], ci, 0, 0, 0);
          sr = __builtin_amdgcn_mfma_f64_16x16x4f64(es[xb][kk], vr[kk], sr, 0, 0, 0);
          si = __builtin_amdgcn_mfma_f64_16x16x4f64(es[xb][kk], vi[kk], si, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; r++) {
          const int t = 4 * xb + r;
          if (t >= S) continue;
          // C +- i S, or C +- S for the pair of point 0
          const bool re0 = t == 0 && real0;
          const double dx = re0 ? sr[r] : -si[r], dy = re0 ? si[r] : sr[r];
          double2 p[2] = {make_double2((cr[r] + dx) * scale, (ci[r] + dy) * scale),
                          make_double2((cr[r] - dx) * scale, (ci[r] - dy) * scale)};
#pragma unroll
          for (int m = 0; m < 2; m++) {
            if (occ) {
              p[m].y = -p[m].y;
              if (step) {  // fullpw: conj(psi1)/sqrt(vol) * theta
                const int w = P::pair(t, lk), x = m ? P::partner(w) : w;
                const int z = zz ? plane_partner(zp, N3) : zp;
                p[m] = cmul(p[m], step[x + (long)N * (Rows<N>::y(rb, lr) + (long)N * z)]);
              }
            }
            out[(((long)(zp * S + rb) * S + t) * 2 + m) * 64 + l] = p[m];
          }
        }
      }
    }
  }
}

// Forward transform of the products of pairs (b1, b2) of the k points of a
// launch (blockIdx.y): one wave per pair, four pairs sharing b2 per workgroup.
// Per pair of planes the x pass (two row blocks at a time), the y pass of
// each row block -- its register pairs are the members of a pair of rows,
// which the layout above arranges -- and the sum and difference of the two
// planes, which go through a per-wave LDS tile into the z pass, accumulated
// directly at the mixed-basis IPWs each lane owns (ig = lane + 64 j).
// The next slot's loads are in flight while the current one's MFMAs run.
// Bound by MFMAs and the VALU together (a VALU instruction holds up the FP64
// matrix pipe for four cycles): per pair of planes 126 MFMAs at 36^2, 60 at
// 24^2, where three products per complex step took 216 and 90.
// Requires ngptm <= 64*PW_FOUT.
template <int N>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(2, 2))) void pw_pair_square_kernel(
    const double2 *__restrict__ grids, int nocc, int nunocc, int N3, const int *__restrict__ oidx,
    int ngptm, double2 *__restrict__ M, long ldm, long t0, int col0) {
  using P = Pairs<N>;
  constexpr int S = P::S, NG = (S + 1) / 2;  // row blocks, in groups of two
  constexpr int PL = PW_BOX * PW_BOX;
  extern __shared__ double2 tz[];               // z coefficients, [zp][gz]
  __shared__ double2 Qs[NT / 64][2 * PL];       // per wave: sum, difference of two planes
  __shared__ double Fs[P::STEPS][64];           // coefficients of step st: lane (lk, g)
  const int tid = threadIdx.x, wv = tid >> 6, l = tid & 63, lr = l & 15, lk = l >> 4;
  // Workgroup -> (unoccupied state b2, group of four occupied states): the
  // ngrp workgroups of one b2 get ids that are equal mod 8, so they run on
  // one XCD (ids go round-robin over the 8) and read psi2 through one L2.
  const int ngrp = (nocc + 3) / 4;
  const int xcd = blockIdx.x & 7, r8 = blockIdx.x >> 3;
  const int b2 = (r8 / ngrp) * 8 + xcd, grp = r8 % ngrp;
  if (b2 >= nunocc) return;  // whole workgroup, before any barrier
  const int ZP = (N3 + 1) / 2, ik = blockIdx.y;
  for (int e = tid; e < ZP * PW_BOX; e += NT)
    tz[e] = plane_coef(e / PW_BOX, e % PW_BOX - PW_OFF, N3);
  for (int e = tid; e < P::STEPS * 64; e += NT)
    Fs[e >> 6][e & 63] = P::step_coef(e >> 6, (e & 63) >> 4, (e & 15) - PW_OFF);
  __syncthreads();
  const int b1 = grp * (NT / 64) + __builtin_amdgcn_readfirstlane(wv);
  if (b1 >= nocc) return;  // whole wave; no workgroup barrier after this point
  const long GS = square_grid(N, N3);
  const d2_t *p1 = (const d2_t *)grids + ((long)ik * (nocc + nunocc) + b1) * GS;
  const d2_t *p2 = (const d2_t *)grids + ((long)ik * (nocc + nunocc) + nocc + b2) * GS;
  d2_t acc[PW_FOUT];
  // LDS byte offsets of the outputs: z coefficients (high half, advanced by a
  // row of the table per pair of planes), plane point (low half).  Slots past
  // ngptm take point 0 and are not stored.
  unsigned ob[PW_FOUT];
#pragma unroll
  for (int j = 0; j < PW_FOUT; j++) {
    const int ig = l + 64 * j, o = ig < ngptm ? oidx[(long)ik * ngptm + ig] : 0;
    ob[j] = (unsigned)(o >> 8) << 20 | (unsigned)((wv * 2 * PL + (o & 255)) * 16);
    acc[j] = d2_t{0.0, 0.0};
  }
  double2 *Q = Qs[wv];
  d2_t ca[2][2], cb[2][2];  // [row block of the group][member], both states
  auto load_slot = [&](int zp, int g, int t) __attribute__((always_inline)) {
#pragma unroll
    for (int b = 0; b < 2; b++) {
      if (2 * g + b >= S) continue;
      const long e = ((long)(zp * S + 2 * g + b) * S + t) * 128;
#pragma unroll
      for (int m = 0; m < 2; m++) {
        ca[b][m] = (p1 + e + 64 * m)[(unsigned)l];
        cb[b][m] = (p2 + e + 64 * m)[(unsigned)l];
      }
    }
  };
  // operand of the difference of a pair: -i S (d.x + i d.y) = S (d.y - i d.x),
  // or d itself where the coefficient is real (pair 0 of an even N)
  const bool real0 = N % 2 == 0 && lk == 0;
  auto diff = [&](d2_t u, d2_t v, bool first) __attribute__((always_inline)) {
    const d2_t d = u - v;
    d2_t o = d2_t{d.y, -d.x};
    if (first) o = real0 ? d : o;
    return o;
  };
  load_slot(0, 0, 0);
  for (int zp = 0; zp < ZP; zp++) {
    d4_t qr[2], qi[2];
#pragma unroll
    for (int zz = 0; zz < 2; zz++) {
      qr[zz] = d4_t{0, 0, 0, 0};
      qi[zz] = d4_t{0, 0, 0, 0};
    }
#pragma unroll
    for (int g = 0; g < NG; g++) {
      constexpr int last = S % 2;  // the last group has one row block
      d4_t xr[2], xi[2];
#pragma unroll
      for (int b = 0; b < 2; b++) {
        xr[b] = d4_t{0, 0, 0, 0};
        xi[b] = d4_t{0, 0, 0, 0};
      }
#pragma unroll
      for (int t = 0; t < S; t++) {
        const bool half = P::HALF && t == P::FULL;
        d2_t u[2], v[2];
#pragma unroll
        for (int b = 0; b < 2; b++) {
          if (g == NG - 1 && last && b == 1) continue;
          const d2_t p = ca[b][0], q = cb[b][0], pp = ca[b][1], qq = cb[b][1];
          const d2_t m = d2_t{p.x * q.x - p.y * q.y, p.x * q.y + p.y * q.x};
          const d2_t n = d2_t{pp.x * qq.x - pp.y * qq.y, pp.x * qq.y + pp.y * qq.x};
          u[b] = m + n;
          v[b] = diff(m, n, t == 0);
          if (half) u[b] = lk < 2 ? u[b] : v[b];
        }
        if (t + 1 < S) load_slot(zp, g, t + 1);
        else if (g + 1 < NG) load_slot(zp, g + 1, 0);
        else if (zp + 1 < ZP) load_slot(zp + 1, 0, 0);
        const double f = Fs[2 * t][l], h = half ? 0.0 : Fs[2 * t + 1][l];
#pragma unroll
        for (int b = 0; b < 2; b++) {
          if (g == NG - 1 && last && b == 1) continue;
          xr[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[b].x, f, xr[b], 0, 0, 0);
          xi[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(u[b].y, f, xi[b], 0, 0, 0);
        }
        if (half) continue;
#pragma unroll
        for (int b = 0; b < 2; b++) {
          if (g == NG - 1 && last && b == 1) continue;
          xr[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[b].x, h, xr[b], 0, 0, 0);
          xi[b] = __builtin_amdgcn_mfma_f64_16x16x4f64(v[b].y, h, xi[b], 0, 0, 0);
        }
      }
      // y pass of the group's row slots: lane holds gx = lr
#pragma unroll
      for (int b = 0; b < 2; b++) {
        if (g == NG - 1 && last && b == 1) continue;
#pragma unroll
        for (int h2 = 0; h2 < 2; h2++) {
          const int ps = 2 * (2 * g + b) + h2, zz = ps / S, tt = ps % S, r0 = 2 * h2;
          const bool half = P::HALF && tt == P::FULL;
          const d2_t m = d2_t{xr[b][r0], xi[b][r0]}, n = d2_t{xr[b][r0 + 1], xi[b][r0 + 1]};
          d2_t u = m + n;
          const d2_t v = diff(m, n, tt == 0);
          if (half) u = lk < 2 ? u : v;
          const double f = Fs[2 * tt][l];
          qr[zz] = __builtin_amdgcn_mfma_f64_16x16x4f64(f, u.x, qr[zz], 0, 0, 0);
          qi[zz] = __builtin_amdgcn_mfma_f64_16x16x4f64(f, u.y, qi[zz], 0, 0, 0);
          if (half) continue;
          const double h = Fs[2 * tt + 1][l];
          qr[zz] = __builtin_amdgcn_mfma_f64_16x16x4f64(h, v.x, qr[zz], 0, 0, 0);
          qi[zz] = __builtin_amdgcn_mfma_f64_16x16x4f64(h, v.y, qi[zz], 0, 0, 0);
        }
      }
    }
    // sum and difference operand of the two planes: gx = lr, gy = lk + 4r
    const bool first = zp == 0 && N3 % 2 == 0;
#pragma unroll
    for (int r = 0; r < 4; r++) {
      const double dx = qr[0][r] - qr[1][r], dy = qi[0][r] - qi[1][r];
      Q[(lk + 4 * r) * PW_BOX + lr] = make_double2(qr[0][r] + qr[1][r], qi[0][r] + qi[1][r]);
      Q[PL + (lk + 4 * r) * PW_BOX + lr] = first ? make_double2(dx, dy) : make_double2(dy, -dx);
    }
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    // branch-free, the LDS reads of four outputs in flight together
#pragma unroll
    for (int j0 = 0; j0 < PW_FOUT; j0 += 4) {
      d2_t T[4], V[4], W[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const unsigned o = ob[j0 + j];
        T[j] = *(const d2_t *)((const char *)tz + (o >> 16));
        V[j] = *(const d2_t *)((const char *)Qs + (o & 0xffffu));
        W[j] = *(const d2_t *)((const char *)Qs + PL * 16 + (o & 0xffffu));
        ob[j0 + j] = o + (PW_BOX * 16u << 16);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        d2_t &a = acc[j0 + j];
        a.x = fma(T[j].y, W[j].x, fma(T[j].x, V[j].x, a.x));
        a.y = fma(T[j].y, W[j].y, fma(T[j].x, V[j].y, a.y));
      }
    }
    __builtin_amdgcn_wave_barrier();  // Q is rewritten by the next planes
  }
  d2_t *out = (d2_t *)M + (t0 + ((long)ik * nocc + b1) * nunocc + b2) * ldm + col0;
#pragma unroll
  for (int j = 0; j < PW_FOUT; j++) {
    const int ig = l + 64 * j;
    if (ig < ngptm) out[ig] = acc[j];
  }
}

// Forward pass z and gather of the mixed-basis IPWs (oidx: box index
// gz*256 + gy*16 + gx of imati.(Gm - g_k) per IPW).
__global__ __launch_bounds__(NT) void pw_pair_z_kernel(const double2 *__restrict__ slab,
                                                       int nunocc, int N3,
                                                       const int *__restrict__ oidx, int ngptm,
                                                       double2 *__restrict__ M, long ldm, long t0,
                                                       int col0) {
  __shared__ double2 tz[64][PW_BOX];  // N3 <= 64
  const int tid = threadIdx.x;
  for (int e = tid; e < N3 * PW_BOX; e += NT) {
    const int z = e / PW_BOX, g = e % PW_BOX;
    tz[z][g] = twid((long)(g - PW_OFF) * z, N3, -1.0);
  }
  __syncthreads();
  const long pair = blockIdx.x;  // b1*nunocc + b2
  const double2 *S = slab + pair * N3 * PW_BOX * PW_BOX;
  double2 *out = M + (t0 + pair) * ldm + col0;
  for (int ig = tid; ig < ngptm; ig += NT) {
    const int b = oidx[ig];
    const int gz = b >> 8, gyx = b & 255;
    double ar = 0.0, ai = 0.0;
    for (int z = 0; z < N3; z++) {
      const double2 t = tz[z][gz];
      const double2 v = S[(long)z * PW_BOX * PW_BOX + gyx];
      ar += t.x * v.x - t.y * v.y;
      ai += t.x * v.y + t.y * v.x;
    }
    out[ig] = make_double2(ar, ai);
  }
}

int box_index(const int *imati, const int *v, int &idx, int *gout = nullptr) {
  int g3[3];
  int *g = gout ? gout : g3;
  for (int i = 0; i < 3; i++) {
    g[i] = imati[3 * i] * v[0] + imati[3 * i + 1] * v[1] + imati[3 * i + 2] * v[2];
    if (g[i] < -PW_OFF || g[i] >= PW_BOX - PW_OFF) return 1;
  }
  idx = ((g[2] + PW_OFF) * PW_BOX + (g[1] + PW_OFF)) * PW_BOX + (g[0] + PW_OFF);
  return 0;
}

// The kernels of an N x N plane: the FFT sizes (products of 2, 3, 5, 7) from
// the box's 16 to 48.  Other planes take the general kernels.
struct SquareFn {
  void (*states)(const double2 *, int, int, const int *, const int *, KList, int, int, int, int,
                 double, double, const double2 *, double2 *);
  void (*pair)(const double2 *, int, int, int, const int *, int, double2 *, long, long, int);
};
SquareFn square_kernels(int N) {
  switch (N) {
#define SPX_SQUARE(n) \
  case n: return {pw_states_kernel<n>, pw_pair_square_kernel<n>};
    SPX_SQUARE(16) SPX_SQUARE(18) SPX_SQUARE(20) SPX_SQUARE(21) SPX_SQUARE(24) SPX_SQUARE(25)
    SPX_SQUARE(27) SPX_SQUARE(28) SPX_SQUARE(30) SPX_SQUARE(32) SPX_SQUARE(35) SPX_SQUARE(36)
    SPX_SQUARE(40) SPX_SQUARE(42) SPX_SQUARE(45) SPX_SQUARE(48)
#undef SPX_SQUARE
    default: return {nullptr, nullptr};
  }
}

// Bytes of the grids of one k point if the plan takes the square kernels, or 0.
size_t square_set(const spexhip_plan *p, int nocc, int nunocc) {
  const int N = p->nfft[0];
  if (p->nfft[1] != N || p->ngptm > 64 * PW_FOUT || !square_kernels(N).pair) return 0;
  return sizeof(double2) * (size_t)(nocc + nunocc) * square_grid(N, p->nfft[2]);
}

template <int NB>
int launch_pw(spexhip_ctx *ctx, hipStream_t st, const spexhip_plan *p, const void *cpw, int nband,
              int nk, const int *k1, const int *k2, const int *oidx_dev, int b1lo, int nocc,
              int b2lo, int nunocc, void *M, long ldm, int col0, void *ws) {
  const int N1 = p->nfft[0], N2 = p->nfft[1], N3 = p->nfft[2];
  const long NN = (long)N1 * N2 * N3;
  double2 *grids = (double2 *)ws;
  double2 *slab = grids + (long)(nocc + nunocc) * NN;
  const int *ngpt_dev = p->gidx + (long)p->nkpt * p->maxgpt;
  const double scaleA = 1.0 / std::sqrt(p->vol), scaleB = 1.0 / (double)NN;
  for (int ik = 0; ik < nk; ik++) {
    hipLaunchKernelGGL(pw_inverse_kernel<NB>, dim3(nocc + nunocc), dim3(NT), 0, st,
                       (const double2 *)cpw, p->maxgpt, nband, p->gidx, ngpt_dev, k1[ik], b1lo,
                       nocc, k2[ik], b2lo, N1, N2, N3, scaleA, scaleB, p->step, grids);
    SPX_LAUNCHED(ctx);
    if (p->ngptm <= 64 * PW_FOUT) {
      hipLaunchKernelGGL(pw_pair_fused_kernel<NB>, dim3(nunocc, (nocc + 3) / 4), dim3(NT), 0, st,
                         grids, nocc, nunocc, N1, N2, N3, oidx_dev + (long)ik * p->ngptm, p->ngptm,
                         (double2 *)M, ldm, (long)ik * nocc * nunocc, col0);
      SPX_LAUNCHED(ctx);
      continue;
    }
    hipLaunchKernelGGL(pw_pair_xy_kernel<NB>, dim3(nunocc, (nocc + 3) / 4), dim3(NT), 0, st, grids,
                       nocc, nunocc, N1, N2, N3, slab);
    SPX_LAUNCHED(ctx);
    hipLaunchKernelGGL(pw_pair_z_kernel, dim3(nocc * nunocc), dim3(NT), 0, st, slab, nunocc, N3,
                       oidx_dev + (long)ik * p->ngptm, p->ngptm, (double2 *)M, ldm,
                       (long)ik * nocc * nunocc, col0);
    SPX_LAUNCHED(ctx);
  }
  return SPEXHIP_OK;
}

// Square planes: as many k points per pair of launches as the workspace has
// room for grids (one of the benchmark's k points alone is 1,600 workgroups
// of which 512 run at a time: its last round would leave most CUs idle).
int launch_square(spexhip_ctx *ctx, hipStream_t st, const spexhip_plan *p, const void *cpw,
                  int nband, int nk, const int *k1, const int *k2, const int *oidx_dev, int b1lo,
                  int nocc, int b2lo, int nunocc, void *M, long ldm, int col0, void *ws,
                  int kbatch) {
  const int N = p->nfft[0], N3 = p->nfft[2];
  const SquareFn fn = square_kernels(N);
  const int *ngpt_dev = p->gidx + (long)p->nkpt * p->maxgpt;
  const unsigned ngrp = (nocc + 3) / 4;
  for (int ik = 0; ik < nk; ik += kbatch) {
    const int n = std::min(kbatch, nk - ik);
    KList kl{};
    for (int i = 0; i < n; i++) {
      kl.k1[i] = k1[ik + i];
      kl.k2[i] = k2[ik + i];
    }
    hipLaunchKernelGGL(fn.states, dim3(nocc + nunocc, n), dim3(NT), 0, st, (const double2 *)cpw,
                       p->maxgpt, nband, p->gidx, ngpt_dev, kl, b1lo, nocc, b2lo, N3,
                       1.0 / std::sqrt(p->vol), 1.0 / ((double)N * N * N3), p->step,
                       (double2 *)ws);
    SPX_LAUNCHED(ctx);
    hipLaunchKernelGGL(fn.pair, dim3(((nunocc + 7) / 8) * 8 * ngrp, n), dim3(NT),
                       (size_t)((N3 + 1) / 2) * PW_BOX * sizeof(double2), st, (const double2 *)ws,
                       nocc, nunocc, N3, oidx_dev + (long)ik * p->ngptm, p->ngptm, (double2 *)M,
                       ldm, (long)ik * nocc * nunocc, col0);
    SPX_LAUNCHED(ctx);
  }
  return SPEXHIP_OK;
}

}  // namespace

int spx_pw_plan_build(spexhip_ctx *ctx, const spexhip_pw_desc *d, spexhip_plan *p) {
  p->kind = 2;
  for (int i = 0; i < 3; i++) {
    SPX_CHECK(ctx, d->nfft[i] >= PW_BOX && d->nfft[i] <= 64,
              "pw plan: nfft[%d]=%d outside [16, 64]", i, d->nfft[i]);
    p->nfft[i] = d->nfft[i];
  }
  for (int i = 0; i < 9; i++) p->imati[i] = d->imati[i];
  SPX_CHECK(ctx, d->vol > 0 && d->nkpt > 0 && d->maxgpt > 0 && d->ngptm >= 0 && d->gpt && d->ngpt,
            "pw plan: bad descriptor");
  p->vol = d->vol;
  p->nkpt = d->nkpt;
  p->maxgpt = d->maxgpt;
  p->ngptm = d->ngptm;
  p->ngpt.assign(d->ngpt, d->ngpt + d->nkpt);
  p->gptm.assign(d->gptm, d->gptm + 3 * d->ngptm);
  std::vector<int> tab((size_t)d->nkpt * d->maxgpt + d->nkpt, 0);
  int lo[3] = {PW_BOX, PW_BOX, PW_BOX}, hi[3] = {-PW_BOX, -PW_BOX, -PW_BOX};
  for (int k = 0; k < d->nkpt; k++) {
    SPX_CHECK(ctx, d->ngpt[k] >= 0 && d->ngpt[k] <= d->maxgpt, "pw plan: ngpt[%d] out of range", k);
    for (int ig = 0; ig < d->ngpt[k]; ig++) {
      int idx, g[3];
      if (box_index(p->imati, d->gpt + 3 * ((long)k * d->maxgpt + ig), idx, g))
        return spx_seterr(ctx, SPEXHIP_E_INVALID,
                          "pw plan: G vector %d of k %d outside the -8..7 Fourier box", ig, k);
      tab[(size_t)k * d->maxgpt + ig] = idx;
      for (int i = 0; i < 3; i++) {
        lo[i] = std::min(lo[i], g[i]);
        hi[i] = std::max(hi[i], g[i]);
      }
    }
    tab[(size_t)d->nkpt * d->maxgpt + k] = d->ngpt[k];
  }
  // Without theta the pair product is a pure convolution of two states with
  // Fourier support of width W = hi - lo per axis, i.e. product frequencies
  // in [-W, W]; the outputs lie in the -8..7 box.  On a grid with
  // N >= W + 9 no product frequency aliases onto an output, so the DFT gives
  // the exact convolution -- the same numbers on every such grid, the
  // caller's included.  The plan then uses the smallest such grid (at least
  // the 16-point box); a caller grid that aliases is kept as given.
  // The box holds W <= 15, so that is 24 at most.  Sizes are rounded up to 16,
  // 20 or 24 where that is still below the caller's grid (18 and 21 have square
  // kernels too, but have not been timed against 20 and 24).
  const bool theta = d->step_r || d->step_c;
  if (!theta)
    for (int i = 0; i < 3; i++) {
      int nmin = std::max(PW_BOX, hi[i] >= lo[i] ? hi[i] - lo[i] + PW_OFF + 1 : PW_BOX);
      for (int nice : {16, 20, 24})
        if (nmin <= nice && nice <= p->nfft[i]) {
          nmin = nice;
          break;
        }
      if (p->nfft[i] > nmin) p->nfft[i] = nmin;
    }
  int rc = spx_alloc(ctx, sizeof(int) * tab.size(), (void **)&p->gidx);
  if (rc) return rc;
  p->owned.push_back(p->gidx);
  SPX_HIP(ctx, hipMemcpy(p->gidx, tab.data(), sizeof(int) * tab.size(), hipMemcpyHostToDevice));
  if (theta) {
    const size_t nn = (size_t)p->nfft[0] * p->nfft[1] * p->nfft[2];
    std::vector<double2> th(nn);
    for (size_t i = 0; i < nn; i++)
      th[i] = d->step_c ? make_double2(d->step_c[2 * i], d->step_c[2 * i + 1])
                        : make_double2(d->step_r[i], 0.0);
    rc = spx_alloc(ctx, 16 * nn, (void **)&p->step);
    if (rc) return rc;
    p->owned.push_back(p->step);
    SPX_HIP(ctx, hipMemcpy(p->step, th.data(), 16 * nn, hipMemcpyHostToDevice));
  }
  return SPEXHIP_OK;
}

size_t spx_wfprod_pw_ws_core(const spexhip_plan *p, int nocc, int nunocc);
// Workspace of the synchronous form: grids, then the oidx table.  two: room for
// two k points' grids on square planes where the core has room for two in the
// natural layout but not in the square one's (up to a quarter larger): one k
// point at a time of 8 x 56 states on 36^3 points, 112 workgroups, takes 1.95 ms
// for eight of them, two together 0.99.
static size_t pw_grid_bytes(const spexhip_plan *p, int nocc, int nunocc, bool two) {
  const size_t core = spx_wfprod_pw_ws_core(p, nocc, nunocc), set = square_set(p, nocc, nunocc);
  const size_t plain = 16 * (size_t)(nocc + nunocc) * p->nfft[0] * p->nfft[1] * p->nfft[2];
  return two && set && core >= 2 * plain ? std::max(core, 2 * set) : core;
}
size_t spx_wfprod_pw_ws(const spexhip_plan *p, int nk, int nocc, int nunocc, bool two) {
  return pw_grid_bytes(p, nocc, nunocc, two && nk > 1) + 4 * (size_t)nk * p->ngptm + 256;
}

// Box indices of imati.(Gm - g2(k)) for every packet k and IPW (host).
int spx_pw_oidx(spexhip_ctx *ctx, const spexhip_plan *p, int nk, const int *g2, int *oidx) {
  for (int ik = 0; ik < nk; ik++)
    for (int ig = 0; ig < p->ngptm; ig++) {
      int v[3];
      for (int i = 0; i < 3; i++) v[i] = p->gptm[3 * ig + i] - g2[3 * ik + i];
      int idx;
      if (box_index(p->imati, v, idx))
        return spx_seterr(ctx, SPEXHIP_E_INVALID,
                          "wfprod_pw: IPW %d - umklapp of k %d outside the -8..7 Fourier box", ig, ik);
      oidx[(size_t)ik * p->ngptm + ig] = idx;
    }
  return SPEXHIP_OK;
}

// Workspace without the oidx table.
size_t spx_wfprod_pw_ws_core(const spexhip_plan *p, int nocc, int nunocc) {
  const long NN = (long)p->nfft[0] * p->nfft[1] * p->nfft[2];
  return std::max(square_set(p, nocc, nunocc),
                  16 * ((size_t)(nocc + nunocc) * NN +
                        (size_t)nocc * nunocc * p->nfft[2] * PW_BOX * PW_BOX));
}

// Asynchronous launches (no host synchronisation): k1, k2 are host arrays
// used as launch arguments, oidx_dev a device table from spx_pw_oidx.  ws_bytes:
// of ws where it holds more than the core.
int spx_wfprod_pw_async(spexhip_ctx *ctx, hipStream_t st, const spexhip_plan *p, const void *cpw,
                        int nband, int nk, const int *k1, const int *k2, const int *oidx_dev,
                        int b1lo, int nocc, int b2lo, int nunocc, void *M, long ldm, int col0,
                        void *ws, size_t ws_bytes) {
  for (int ik = 0; ik < nk; ik++)
    SPX_CHECK(ctx, k1[ik] >= 0 && k1[ik] < p->nkpt && k2[ik] >= 0 && k2[ik] < p->nkpt,
              "wfprod_pw: k index out of range");
  if (const size_t set = square_set(p, nocc, nunocc)) {
    const size_t fit = std::max(ws_bytes, spx_wfprod_pw_ws_core(p, nocc, nunocc)) / set;
    return launch_square(ctx, st, p, cpw, nband, nk, k1, k2, oidx_dev, b1lo, nocc, b2lo, nunocc, M,
                         ldm, col0, ws, (int)std::min<size_t>(fit, PW_KMAX));
  }
  const int nbmax = (std::max(p->nfft[0], p->nfft[1]) + 15) / 16;
  switch (nbmax) {
    case 1:
    case 2:
      return launch_pw<2>(ctx, st, p, cpw, nband, nk, k1, k2, oidx_dev, b1lo, nocc, b2lo, nunocc, M, ldm, col0, ws);
    case 3:
      return launch_pw<3>(ctx, st, p, cpw, nband, nk, k1, k2, oidx_dev, b1lo, nocc, b2lo, nunocc, M, ldm, col0, ws);
    default:
      return launch_pw<4>(ctx, st, p, cpw, nband, nk, k1, k2, oidx_dev, b1lo, nocc, b2lo, nunocc, M, ldm, col0, ws);
  }
}

// Synchronous form: builds and uploads the oidx table into the tail of ws.
int spx_wfprod_pw(spexhip_ctx *ctx, hipStream_t st, const spexhip_plan *p, const void *cpw,
                  int nband, int nk, const int *k1, const int *k2, const int *g2, int b1lo,
                  int nocc, int b2lo, int nunocc, void *M, long ldm, int col0, void *ws, bool two) {
  const size_t gb = pw_grid_bytes(p, nocc, nunocc, two && nk > 1);
  std::vector<int> oidx((size_t)nk * p->ngptm);
  int rc = spx_pw_oidx(ctx, p, nk, g2, oidx.data());
  if (rc) return rc;
  int *oidx_dev = (int *)((char *)ws + gb);
  SPX_HIP(ctx, hipMemcpyAsync(oidx_dev, oidx.data(), 4 * oidx.size(), hipMemcpyHostToDevice, st));
  rc = spx_wfprod_pw_async(ctx, st, p, cpw, nband, nk, k1, k2, oidx_dev, b1lo, nocc, b2lo, nunocc,
                           M, ldm, col0, ws, gb);
  SPX_HIP(ctx, hipStreamSynchronize(st));  // oidx is a host temporary
  return rc;
}
