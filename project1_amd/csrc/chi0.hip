// chi0 pair sum as a Hermitian rank-k update on the CDNA4 matrix cores.
//
// Reference: susceptibility.f:1159-1251 (pair loop) with spectral_function,
// HILBERT NONE branch :1780-1788, i.e.
//     susceph(ij,w) += sum_t wghtSr(t,w) * cprod(t,i) * conjg(cprod(t,j)),
// one DDOT of length n per (i<=j, w) in the reference.  Here the same sum
// is C_w = L_w^T conj(M) with L_w(t,I) = wght(t,w) M(t,I), computed per
// 64x64 output tile of the upper triangle with MFMA:
//   * FP64 form: v_mfma_f64_16x16x4f64, 3 real products per complex step
//     (chi0_tile.hpp);
//   * split-FP32 form: both sides are sqrt|D| M on a grid relative to their
//     column maximum, split into an integer part h (<= 10 bits, so h*h and
//     its K-chunk sums are exact in FP32) and an FP32 rest l; h*h goes into
//     one FP32 accumulator, h*l + l*fp32(h+l) into another, both flushed
//     into FP64 accumulators after every K-chunk of 16 transitions
//     (chi0_tile.hpp).  A scale pass (colscale.hpp) reads M once first.
#include <algorithm>
#include <type_traits>

#include "colscale.hpp"
#include "common.hpp"

#include "chi0_tile.hpp"

namespace {

using chi0t::Lds;
using chi0t::Problem;

// The tiles of one call in launch order, and how the last of them are split
// over the transitions: tiles t < full are whole; each of the rest is summed
// in ks parts, which are added in order: by chi0_reduce_kernel from `part`, or,
// where there is no room for them (part null), by one workgroup per tile that
// runs the parts one after the other (chi0_parts_kernel).
struct Split {
  int ntri;      // tiles per frequency
  long full;     // whole tiles
  int rem, ks;   // split tiles, parts of each
  double2 *part; // [rem * ks][TM * TM]
};

constexpr int CT = 64, CK = 16;  // tile edge and K-slice of this file's launches

// Two workgroups (two waves per SIMD) share a CU: one's barrier and LDS
// latencies hide behind the other's MFMAs.  FP64 at 51,200 transitions, 1200
// columns, 12 frequencies: 48.0 ms, FP64 matrix pipe busy 77 % (68.3 ms with
// four products per step and no split of the last round); error against long
// double sums at 409,600 transitions 5e-16 of the norm (2.3e-14 before).

//
// Real-frequency weights: one chain of sums per output over all transitions,
// four products per step.  The inverse of eps at real frequencies carries
// condition numbers beyond 1e5: another order of rounding in chi, though its
// error is smaller (3e-15 against 4e-15), moves eps^-1 by 1e-11 to 5e-10, so
// the results of this form keep their order.  With the parts and three
// products the pair sums take 0.55 ms at 7,040 transitions x 403 columns x 5
// frequencies, like this 0.73 ms (1.27 with the operands staged through
// registers and 140 tiles of 64).
template <int TM, bool COLMAJOR, bool DMA>
__global__ __launch_bounds__(chi0t::NT) __attribute__((amdgpu_waves_per_eu(2))) void chi0_one_kernel(
    Problem P) {
  __shared__ Lds<TM, CK, false> s;
  const long nbt = (P.nb + TM - 1) / TM, ntri = nbt * (nbt + 1) / 2;
  int bi, bj;
  chi0t::tri_index((int)(blockIdx.x % ntri), bi, bj);
  const int w = (int)(blockIdx.x / ntri);
  chi0t::Acc<TM / 32> acc;
  chi0t::tile_sums<TM, CK, COLMAJOR, false, DMA, true>(P, bi, bj, w, 0, (P.n + CK - 1) / CK, s,
                                                       acc);
  chi0t::store_tile<TM, false>(P, bi, bj, w, acc);
}

template <bool COLMAJOR, bool SPLIT, bool DMA>
__global__ __launch_bounds__(chi0t::NT) __attribute__((amdgpu_waves_per_eu(COLMAJOR && SPLIT ? 1 : 2, 2))) void chi0_kernel(
    Problem P, Split S) {
  __shared__ Lds<CT, CK, SPLIT> s;
  const long u = blockIdx.x;
  const long t = u < S.full ? u : S.full + (u - S.full) / S.ks;
  const int w = (int)(t / S.ntri);
  int bi, bj;
  chi0t::tri_index((int)(t % S.ntri), bi, bj);
  chi0t::Acc<CT / 32> acc;
  const long nst = (P.n + CK - 1) / CK;
  if (u < S.full) {
    chi0t::tile_sums<CT, CK, COLMAJOR, SPLIT, DMA>(P, bi, bj, w, 0, nst, s, acc);
    chi0t::store_tile<CT, SPLIT>(P, bi, bj, w, acc);
    return;
  }
  const int p = (int)((u - S.full) % S.ks);
  chi0t::tile_sums<CT, CK, COLMAJOR, SPLIT, DMA>(P, bi, bj, w, nst * p / S.ks,
                                                 nst * (p + 1) / S.ks, s, acc);
  double2 *out = S.part + (u - S.full) * (CT * CT) + threadIdx.x;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 4; r++)
        out[((a * 2 + b) * 4 + r) * chi0t::NT] = make_double2(acc.re[a][b][r], acc.im[a][b][r]);
}

// One workgroup per split tile: the parts in ascending order, then the store
// of a whole tile.
template <bool SPLIT>
__global__ __launch_bounds__(chi0t::NT) void chi0_reduce_kernel(Problem P, Split S) {
  const long t = S.full + blockIdx.x;
  const int w = (int)(t / S.ntri);
  int bi, bj;
  chi0t::tri_index((int)(t % S.ntri), bi, bj);
  const double2 *in = S.part + (long)blockIdx.x * S.ks * (CT * CT) + threadIdx.x;
  chi0t::Acc<CT / 32> acc;
#pragma unroll
  for (int a = 0; a < 2; a++)
#pragma unroll
    for (int b = 0; b < 2; b++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        const int e = ((a * 2 + b) * 4 + r) * chi0t::NT;
        double2 v = in[e];
        for (int p = 1; p < S.ks; p++) {
          const double2 x = in[(long)p * (CT * CT) + e];
          v.x += x.x;
          v.y += x.y;
        }
        acc.re[a][b][r] = v.x;
        acc.im[a][b][r] = v.y;
      }
  chi0t::store_tile<CT, SPLIT>(P, bi, bj, w, acc);
}

// The split tiles without room for their parts: one workgroup per tile, the
// parts in ascending order, the same sums as above.  Both accumulators take the
// registers of one wave per SIMD.  60 tiles of 3,584 transitions: 444 us (145 us
// in 8 parts each, side by side); 196 tiles of 9,045: 1,103 us (995).
template <bool COLMAJOR, bool SPLIT, bool DMA>
__global__ __launch_bounds__(chi0t::NT) __attribute__((amdgpu_waves_per_eu(1, 1))) void
chi0_parts_kernel(Problem P, Split S) {
  __shared__ Lds<CT, CK, SPLIT> s;
  const long t = S.full + blockIdx.x;
  const int w = (int)(t / S.ntri);
  int bi, bj;
  chi0t::tri_index((int)(t % S.ntri), bi, bj);
  const long nst = (P.n + CK - 1) / CK;
  chi0t::Acc<CT / 32> acc, sum;
#pragma unroll 1
  for (int p = 0; p < S.ks; p++) {
    chi0t::tile_sums<CT, CK, COLMAJOR, SPLIT, DMA>(P, bi, bj, w, nst * p / S.ks,
                                                   nst * (p + 1) / S.ks, s, acc);
    if (p == 0) {
      sum = acc;
      continue;
    }
#pragma unroll
    for (int a = 0; a < 2; a++)
#pragma unroll
      for (int b = 0; b < 2; b++) {
        sum.re[a][b] += acc.re[a][b];
        sum.im[a][b] += acc.im[a][b];
      }
  }
  chi0t::store_tile<CT, SPLIT>(P, bi, bj, w, sum);
}

// How a call's tiles are split.  512 workgroups run at once (two per CU,
// 65 KB of LDS each).  Whole rounds of 512 tiles run unsplit; the tiles of
// the last, partial round are cut over the transitions so that they fill it:
// 60 tiles (3,584 transitions, 256 columns, 6 frequencies) took 631 us whole
// and take 144 us in 8 parts each, the reduction included.  A part keeps at
// least 8 K-slices, and 512 parts bound the workspace to 32 MiB.  The rule
// depends on the sizes only and both ways to run the parts add them in the same
// order, so the order of every sum depends on the sizes only.
constexpr int CSLOTS = 512;
Split split_rule(long n, int nb, int nw) {
  const int nbt = (nb + CT - 1) / CT;
  Split S{};
  S.ntri = nbt * (nbt + 1) / 2;
  const long total = (long)S.ntri * nw;
  S.full = total / CSLOTS * CSLOTS;
  S.rem = (int)(total - S.full);
  const long nst = (n + CK - 1) / CK;
  S.ks = S.rem ? (int)std::max(1L, std::min((long)(CSLOTS / S.rem), nst / 8)) : 1;
  if (S.ks == 1) {
    S.full = total;
    S.rem = 0;
  }
  return S;
}
size_t part_bytes(const Split &S) { return 16 * (size_t)S.rem * S.ks * CT * CT; }

// ------------------------------------------------------------ weights --
__global__ void weights_none_kernel(int nk, int nocc, int nunocc,
                                    const double *__restrict__ eo,
                                    const double *__restrict__ eu, int nkpt,
                                    int nsym1, const int *__restrict__ nkpts,
                                    int nw, const double *__restrict__ om,
                                    double *__restrict__ wght) {
  const long n = (long)nk * nocc * nunocc;
  const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const int b2 = (int)(t % nunocc);
  const long r = t / nunocc;
  const int b1 = (int)(r % nocc);
  const int k = (int)(r / nocc);
  const double d = eu[(long)k * nunocc + b2] - eo[(long)k * nocc + b1];
  const double kw = (double)nkpts[k];
  for (int f = 0; f < nw; f++) {
    // same operation order and roundings as the reference expression (no FMA)
#pragma clang fp contract(off)
    const double w = om[f];
    wght[t + n * f] = -2 * d / (w * w + d * d) / nkpt / nsym1 * kw;
  }
}

// ----------------------------------------------------------- packing --
__global__ void pack_upper_kernel(int nb, int nw, const double2 *__restrict__ X,
                                  long ldx, double2 *__restrict__ P) {
  const long npack = (long)nb * (nb + 1) / 2;
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= npack * nw) return;
  const int w = (int)(g / npack);
  const long ij = g - (long)w * npack;
  long j = (long)((sqrt(8.0 * (double)ij + 1.0) - 1.0) * 0.5);
  while ((j + 1) * (j + 2) / 2 <= ij) j++;
  while (j * (j + 1) / 2 > ij) j--;
  const long i = ij - j * (j + 1) / 2;
  P[g] = X[(long)w * ldx * nb + i + ldx * j];
}

__global__ void unpack_kernel(int nb, int nw, const double2 *__restrict__ P,
                              double2 *__restrict__ X, long ldx) {
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g >= (long)nb * nb * nw) return;
  const int w = (int)(g / ((long)nb * nb));
  const long r = g - (long)w * nb * nb;
  const int j = (int)(r / nb), i = (int)(r % nb);
  const long npack = (long)nb * (nb + 1) / 2;
  double2 v;
  if (i <= j) {
    v = P[(long)w * npack + (long)j * (j + 1) / 2 + i];
  } else {
    v = P[(long)w * npack + (long)i * (i + 1) / 2 + j];
    v.y = -v.y;
  }
  X[(long)w * ldx * nb + i + ldx * (long)j] = v;
}

}  // namespace

// One chain per output: tiles of 64, or for row-major M with fewer than 512 of
// them tiles of 32, four times the workgroups (140 tiles of 64: 1.09 -> 0.73 ms).
static void launch_one(hipStream_t st, const Problem &P, int colmajor) {
  auto tiles = [&](int tm) {
    const long nbt = (P.nb + tm - 1) / tm;
    return nbt * (nbt + 1) / 2 * P.nw;
  };
  const bool dma = chi0t::dma_ok(P.M), small = !colmajor && tiles(64) < 512;
  auto kern = colmajor ? (dma ? chi0_one_kernel<64, true, true> : chi0_one_kernel<64, true, false>)
              : small  ? (dma ? chi0_one_kernel<32, false, true> : chi0_one_kernel<32, false, false>)
                       : (dma ? chi0_one_kernel<64, false, true> : chi0_one_kernel<64, false, false>);
  hipLaunchKernelGGL(kern, dim3((unsigned)tiles(small ? 32 : 64)), dim3(chi0t::NT), 0, st, P);
}

static void launch_tiles(hipStream_t st, const Problem &P, const Split &S, int colmajor, int split) {
  const dim3 grid((unsigned)(S.full + (S.part ? (long)S.rem * S.ks : 0))), block(chi0t::NT);
  auto go = [&](auto sp, auto dma) {
    constexpr bool SP = decltype(sp)::value, DMA = decltype(dma)::value;
    if (grid.x && colmajor)
      hipLaunchKernelGGL((chi0_kernel<true, SP, DMA>), grid, block, 0, st, P, S);
    else if (grid.x)
      hipLaunchKernelGGL((chi0_kernel<false, SP, DMA>), grid, block, 0, st, P, S);
    if (!S.rem) return;
    if (S.part)
      hipLaunchKernelGGL(chi0_reduce_kernel<SP>, dim3(S.rem), block, 0, st, P, S);
    else if (colmajor)
      hipLaunchKernelGGL((chi0_parts_kernel<true, SP, DMA>), dim3(S.rem), block, 0, st, P, S);
    else
      hipLaunchKernelGGL((chi0_parts_kernel<false, SP, DMA>), dim3(S.rem), block, 0, st, P, S);
  };
  if (split) go(std::true_type{}, std::false_type{});
  else if (chi0t::dma_ok(P.M)) go(std::false_type{}, std::true_type{});
  else go(std::false_type{}, std::false_type{});
}

// ------------------------------------------------------- column scales --
namespace colscale {

// scale[w][I] via atomicMax on the bit pattern (non-negative doubles order
// like unsigned integers); the caller zeroes scale first.
//
// Transition-major M: one thread per column I and tchunk transitions.  The
// weights of a stage of 64 transitions are the same for every thread: the
// workgroup stages them in LDS (NWP = nw rounded up to 4, rows w >= nw read
// as 0) and each thread reads them back as broadcasts, eight transitions at
// a time.
template <int NWP, bool FROM_D>
__global__ __launch_bounds__(256) void col_scale_kernel(long n, int nb,
                                                        const double2 *__restrict__ M, long ldm,
                                                        int nw, const double *__restrict__ W,
                                                        long tchunk,
                                                        unsigned long long *__restrict__ scale) {
  constexpr int TS = 64;
  __shared__ double ss[NWP][TS];
  const int I = blockIdx.x * blockDim.x + threadIdx.x;
  const bool live = I < nb;
  const long t0 = (long)blockIdx.y * tchunk;
  const long t1 = t0 + tchunk < n ? t0 + tchunk : n;
  double m[NWP];
#pragma unroll
  for (int w = 0; w < NWP; w++) m[w] = 0.0;
  for (long tb = t0; tb < t1; tb += TS) {
    const int len = (int)(t1 - tb < TS ? t1 - tb : TS);
    __syncthreads();  // the previous stage has been read
    for (int e = threadIdx.x; e < NWP * TS; e += blockDim.x) {
      const int w = e / TS, j = e % TS;
      double v = 0.0;
      if (w < nw && j < len) {
        v = W[(long)w * n + tb + j];
        if (FROM_D) v = sqrt(fabs(v));
      }
      ss[w][j] = v;
    }
    __syncthreads();
    if (live) {
      int j0 = 0;
      for (; j0 + 8 <= len; j0 += 8) {  // no branches: eight loads in flight
        double2 v[8];
#pragma unroll
        for (int j = 0; j < 8; j++) v[j] = M[(tb + j0 + j) * ldm + I];
        __builtin_amdgcn_sched_barrier(0);  // keep the eight loads ahead of their uses
        double a[8];
#pragma unroll
        for (int j = 0; j < 8; j++) a[j] = fmax(fabs(v[j].x), fabs(v[j].y));
#pragma unroll
        for (int w = 0; w < NWP; w++) {
          double x = a[0] * ss[w][j0];
#pragma unroll
          for (int j = 1; j < 8; j++) x = fmax(x, a[j] * ss[w][j0 + j]);
          m[w] = fmax(m[w], x);
        }
      }
      for (; j0 < len; j0++) {
        const double2 v = M[(tb + j0) * ldm + I];
        const double a = fmax(fabs(v.x), fabs(v.y));
#pragma unroll
        for (int w = 0; w < NWP; w++) m[w] = fmax(m[w], a * ss[w][j0]);
      }
    }
  }
  if (!live) return;
#pragma unroll
  for (int w = 0; w < NWP; w++)
    if (w < nw) atomicMax(scale + (long)w * nb + I, (unsigned long long)__double_as_longlong(m[w]));
}

// x of the lane `CTRL` rotates to within its row of 16 lanes
template <int CTRL>
__device__ inline double dpp_ror(double x) {
  const long long v = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(v >> 32), CTRL, 0xf, 0xf, true);
  return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Column-major M: a wave takes CS_COLS columns and tchunk transitions, its
// lanes along the transitions, so that loads are contiguous.  A thread per
// column (as above) reads 64 columns 16 bytes at a time: at 9,045
// transitions, 403 columns and 7 frequencies that took 259 us.  Each row of
// 16 lanes reduces by rotations; its first lane updates the maximum.
constexpr int CS_COLS = 4;
template <int NWP, bool FROM_D>
__global__ __launch_bounds__(256) void col_scale_t_kernel(long n, int nb,
                                                          const double2 *__restrict__ M, long ldm,
                                                          int nw, const double *__restrict__ W,
                                                          long tchunk,
                                                          unsigned long long *__restrict__ scale) {
  const int lane = threadIdx.x & 63;
  const int I0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * CS_COLS;
  if (I0 >= nb) return;
  const long t0 = (long)blockIdx.y * tchunk;
  const long t1 = t0 + tchunk < n ? t0 + tchunk : n;
  double m[CS_COLS][NWP];
#pragma unroll
  for (int c = 0; c < CS_COLS; c++)
#pragma unroll
    for (int w = 0; w < NWP; w++) m[c][w] = 0.0;
  for (long t = t0 + lane; t < t1; t += 64) {
    double a[CS_COLS];
#pragma unroll
    for (int c = 0; c < CS_COLS; c++) {
      const int I = I0 + c < nb ? I0 + c : nb - 1;
      const double2 v = M[t + ldm * (long)I];
      a[c] = fmax(fabs(v.x), fabs(v.y));
    }
#pragma unroll
    for (int w = 0; w < NWP; w++) {
      double s = w < nw ? W[(long)w * n + t] : 0.0;
      if (FROM_D) s = sqrt(fabs(s));
#pragma unroll
      for (int c = 0; c < CS_COLS; c++) m[c][w] = fmax(m[c][w], a[c] * s);
    }
  }
#pragma unroll
  for (int c = 0; c < CS_COLS; c++)
#pragma unroll
    for (int w = 0; w < NWP; w++) {
      double x = m[c][w];
      x = fmax(x, dpp_ror<0x128>(x));  // row_ror:8, 4, 2, 1
      x = fmax(x, dpp_ror<0x124>(x));
      x = fmax(x, dpp_ror<0x122>(x));
      x = fmax(x, dpp_ror<0x121>(x));
      if ((lane & 15) == 0 && w < nw && I0 + c < nb)
        atomicMax(scale + (long)w * nb + I0 + c, (unsigned long long)__double_as_longlong(x));
    }
}

__global__ void zero_u64_kernel(unsigned long long *__restrict__ p, long count) {
  const long g = (long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g < count) p[g] = 0ull;
}

}  // namespace colscale

size_t spx_split_ws_bytes(int nb, int nw) { return 8 * (size_t)nb * nw; }

static size_t scale_bytes(int nb, int nw, int precision) {
  return precision == SPEXHIP_PREC_SPLIT_FP32 ? (spx_split_ws_bytes(nb, nw) + 255) & ~(size_t)255 : 0;
}

size_t spx_chi0_ws_bytes(long n, int nb, int nw, int precision) {
  return scale_bytes(nb, nw, precision) + part_bytes(split_rule(n, nb, nw));
}

// Column scales of spexhip_chi0_noalloc_dev: a fixed array in device memory
// (one copy per GPU, held until the process ends) instead of a context
// allocation.  All contexts on a GPU share it, so nothing else goes there: the
// FP64 form uses none of it and overlapping FP64 calls stay independent.  Host
// code never passes `scratch` itself to a kernel (on the host its name is a
// stand-in, not a device address); spx_noalloc_setup looks up the device
// address once per context, with the context's device current, and the entry
// point passes that address.
static __device__ __align__(256) double scratch[SPEXHIP_NOALLOC_MAX_SCALES];

int spx_noalloc_setup(spexhip_ctx *ctx) {
  void *ptr = nullptr;
  SPX_HIP(ctx, hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch)));
  SPX_CHECK(ctx, ptr != nullptr, "no-alloc scratch: null device address");
  ctx->noalloc_scales = ptr;
  return SPEXHIP_OK;
}

int spx_col_scales(spexhip_ctx *ctx, hipStream_t st, long n, int nb, const void *M, long ldm,
                   int colmajor, int nw, const double *W, int from_d, double *scale) {
  const long cnt = (long)nb * nw;
  hipLaunchKernelGGL(colscale::zero_u64_kernel, dim3((unsigned)((cnt + 255) / 256)), dim3(256), 0,
                     st, (unsigned long long *)scale, cnt);
  SPX_LAUNCHED(ctx);
  if (n == 0) return SPEXHIP_OK;
  // Transitions per workgroup: enough workgroups to fill the chip (about
  // 1024), few enough atomics per column (at most 1024 transitions each).  A
  // fixed 1024 left 4 workgroups at 3,584 transitions and 256 columns: 201 us.
  const int gx = colmajor ? (nb + 4 * colscale::CS_COLS - 1) / (4 * colscale::CS_COLS) : (nb + 255) / 256;
  const long tchunk = std::min(1024L, std::max(64L, (n * gx / 1024 + 63) / 64 * 64));
  dim3 grid(gx, (unsigned)((n + tchunk - 1) / tchunk));
  for (int w0 = 0; w0 < nw; w0 += 16) {
    const int g = std::min(16, nw - w0);
    const double *Wg = W + (long)w0 * n;  // rows of n transitions
    unsigned long long *Sg = (unsigned long long *)scale + (long)w0 * nb;
    auto go = [&](auto np, auto fd) {
      constexpr int NWP = decltype(np)::value;
      constexpr bool FD = decltype(fd)::value;
      if (colmajor)
        hipLaunchKernelGGL((colscale::col_scale_t_kernel<NWP, FD>), grid, dim3(256), 0, st, n, nb,
                           (const double2 *)M, ldm, g, Wg, tchunk, Sg);
      else
        hipLaunchKernelGGL((colscale::col_scale_kernel<NWP, FD>), grid, dim3(256), 0, st, n, nb,
                           (const double2 *)M, ldm, g, Wg, tchunk, Sg);
    };
    auto go_nw = [&](auto fd) {
      switch ((g + 3) / 4 * 4) {
        case 4: go(std::integral_constant<int, 4>{}, fd); break;
        case 8: go(std::integral_constant<int, 8>{}, fd); break;
        case 12: go(std::integral_constant<int, 12>{}, fd); break;
        default: go(std::integral_constant<int, 16>{}, fd); break;
      }
    };
    if (from_d) go_nw(std::true_type{});
    else go_nw(std::false_type{});
    SPX_LAUNCHED(ctx);
  }
  return SPEXHIP_OK;
}

int spx_chi0_launch(spexhip_ctx *ctx, hipStream_t st, long n, int nb,
                    const void *M, long ldm, int colmajor, int nw,
                    const void *wght, int precision, double alpha, double beta,
                    void *chi, int ldchi, void *ws, size_t ws_bytes, int how) {
  SPX_CHECK(ctx, n >= 0 && nb > 0 && nw > 0, "chi0: bad sizes n=%ld nb=%d nw=%d", n, nb, nw);
  SPX_CHECK(ctx, ldchi >= nb, "chi0: ldchi=%d < nb=%d", ldchi, nb);
  SPX_CHECK(ctx, colmajor ? ldm >= n : ldm >= nb, "chi0: ldm=%ld too small", ldm);
  SPX_CHECK(ctx, precision == SPEXHIP_PREC_FP64 || precision == SPEXHIP_PREC_SPLIT_FP32 ||
                     precision == SPEXHIP_PREC_OZAKI_INT8,
            "chi0: unknown precision %d", precision);
  if (precision == SPEXHIP_PREC_OZAKI_INT8)
    return spx_chi0_ozaki(ctx, st, n, nb, M, ldm, colmajor, nw, wght, alpha, beta, chi, ldchi,
                          ctx->ozaki_ws_limit);
  const int split = precision == SPEXHIP_PREC_SPLIT_FP32 && n > 0;
  Split S = split_rule(n, nb, nw);
  const bool one = (how & CHI0_ONE) && !split;
  if (one) {
    S.full += S.rem;
    S.rem = 0;
    S.ks = 1;
  }
  const size_t sb = split ? scale_bytes(nb, nw, precision) : 0, pb = part_bytes(S);
  std::unique_lock<std::mutex> own;  // of the context's buffer, until the launches are enqueued
  if (!ws && sb + pb && !(how & CHI0_NO_PARTS)) {
    SPX_CHECK(ctx, !sb || st == ctx->stream, "chi0: split form off the context stream needs a workspace");
    // the context's buffer, whose parts are left out when the budget has no
    // room for them, and off the context stream
    ws_bytes = st == ctx->stream ? sb + pb : 0;
    if (ws_bytes) own = std::unique_lock<std::mutex>(ctx->chi0_mu);
    int rc = ws_bytes ? spx_chi0_buf(ctx, ws_bytes, &ws) : SPEXHIP_OK;
    if (rc == SPEXHIP_E_NOMEM && pb) {
      ws_bytes = sb;
      rc = sb ? spx_chi0_buf(ctx, sb, &ws) : SPEXHIP_OK;
    }
    if (rc) return rc;
  }
  SPX_CHECK(ctx, ws_bytes >= sb, "chi0: workspace too small");
  double *scale = sb ? (double *)ws : nullptr;
  const bool parts = pb && !(how & CHI0_NO_PARTS) && ws_bytes >= sb + pb;
  S.part = parts ? (double2 *)((char *)ws + sb) : nullptr;
  if (split) {
    int rc = spx_col_scales(ctx, st, n, nb, M, ldm, colmajor, nw, (const double *)wght, 1, scale);
    if (rc) return rc;
  }
  Problem P{n, nb, nw, (const double2 *)M, ldm, (const double *)wght, (double2 *)chi,
            (long)ldchi, n == 0 ? 0.0 : alpha, beta, scale};
  if (one) launch_one(st, P, colmajor);
  else launch_tiles(st, P, S, colmajor, split);
  SPX_LAUNCHED(ctx);
  return SPEXHIP_OK;
}

int spx_weights_launch(spexhip_ctx *ctx, hipStream_t st, int nk, int nocc, int nunocc,
                       const void *e_occ, const void *e_unocc, int nkpt, int nsym1,
                       const void *nkpts, int nw, const void *omega, void *wght) {
  const long n = (long)nk * nocc * nunocc;
  if (n == 0) return SPEXHIP_OK;
  const int bs = 256;
  hipLaunchKernelGGL(weights_none_kernel, dim3((n + bs - 1) / bs), dim3(bs), 0, st, nk, nocc,
                     nunocc, (const double *)e_occ, (const double *)e_unocc, nkpt, nsym1,
                     (const int *)nkpts, nw, (const double *)omega, (double *)wght);
  SPX_LAUNCHED(ctx);
  return SPEXHIP_OK;
}

int spx_pack_upper(spexhip_ctx *ctx, hipStream_t st, int nb, int nw, const void *X, long ldx,
                   void *P) {
  const long npack = (long)nb * (nb + 1) / 2;
  const int bs = 256;
  hipLaunchKernelGGL(pack_upper_kernel, dim3((npack * nw + bs - 1) / bs), dim3(bs), 0, st, nb, nw,
                     (const double2 *)X, ldx, (double2 *)P);
  SPX_LAUNCHED(ctx);
  return SPEXHIP_OK;
}

extern "C" {

int spexhip_weights_none_dev(spexhip_ctx *ctx, int nk, int nocc, int nunocc,
                             const void *e_occ, const void *e_unocc, int nkpt,
                             int nsym1, const void *nkpts, int nw,
                             const void *omega, void *wght) {
  if (!ctx) return SPEXHIP_E_INVALID;
  SPX_CHECK(ctx, nk >= 0 && nocc >= 0 && nunocc >= 0 && nw > 0 && nkpt > 0 && nsym1 > 0,
            "weights: bad sizes");
  const long n = (long)nk * nocc * nunocc;
  if (n == 0) return SPEXHIP_OK;
  SPX_CHECK(ctx, spx_owns(ctx, wght, sizeof(double) * n * nw), "weights: output not a context allocation of n*nw doubles");
  SPX_CHECK(ctx, spx_owns(ctx, e_occ, sizeof(double) * nk * nocc) &&
                 spx_owns(ctx, e_unocc, sizeof(double) * nk * nunocc) &&
                 spx_owns(ctx, nkpts, sizeof(int) * nk) &&
                 spx_owns(ctx, omega, sizeof(double) * nw),
            "weights: input not a context allocation of the stated size");
  SPX_HIP(ctx, hipSetDevice(ctx->device));
  const int bs = 256;
  hipLaunchKernelGGL(weights_none_kernel, dim3((n + bs - 1) / bs), dim3(bs), 0, ctx->stream,
                     nk, nocc, nunocc, (const double *)e_occ, (const double *)e_unocc, nkpt,
                     nsym1, (const int *)nkpts, nw, (const double *)omega, (double *)wght);
  SPX_LAUNCHED(ctx);
  return SPEXHIP_OK;
}

int spexhip_chi0_dev(spexhip_ctx *ctx, long n, int nb, const void *M, long ldm,
                     int colmajor, int nw, const void *wght, int precision,
                     double alpha, double beta, void *chi, int ldchi) {
  if (!ctx) return SPEXHIP_E_INVALID;
  SPX_CHECK(ctx, nb > 0 && nw > 0 && n >= 0 && ldchi >= nb, "chi0: bad sizes");
  if (n > 0) {
    const size_t mbytes = colmajor ? 16 * ((size_t)ldm * (nb - 1) + n)
                                   : 16 * ((size_t)ldm * (n - 1) + nb);
    SPX_CHECK(ctx, spx_owns(ctx, M, mbytes), "chi0: M is not a context allocation of the stated shape");
    SPX_CHECK(ctx, spx_owns(ctx, wght, sizeof(double) * n * nw), "chi0: wght is not a context allocation of n*nw doubles");
  }
  SPX_CHECK(ctx, spx_owns(ctx, chi, 16 * ((size_t)ldchi * nb * (nw - 1) + (size_t)ldchi * (nb - 1) + nb)),
            "chi0: chi is not a context allocation of the stated shape");
  SPX_HIP(ctx, hipSetDevice(ctx->device));
  return spx_chi0_launch(ctx, ctx->stream, n, nb, M, ldm, colmajor, nw, wght, precision,
                         alpha, beta, chi, ldchi);
}

int spexhip_chi0_noalloc_dev(spexhip_ctx *ctx, long n, int nb, const void *M, long ldm,
                             int colmajor, int nw, const void *wght, int precision,
                             double alpha, double beta, void *chi, int ldchi) {
  if (!ctx) return SPEXHIP_E_INVALID;
  SPX_CHECK(ctx, precision == SPEXHIP_PREC_FP64 || precision == SPEXHIP_PREC_SPLIT_FP32,
            "chi0_noalloc: precision %d not available without allocation (the Ozaki form "
            "needs a slice workspace; use spexhip_chi0_dev)", precision);
  SPX_CHECK(ctx, nb > 0 && nw > 0 && n >= 0 && ldchi >= nb, "chi0_noalloc: bad sizes");
  SPX_CHECK(ctx, (long)nb * nw <= SPEXHIP_NOALLOC_MAX_SCALES,
            "chi0_noalloc: nb*nw = %ld exceeds the fixed scratch of %d column scales",
            (long)nb * nw, SPEXHIP_NOALLOC_MAX_SCALES);
  SPX_CHECK(ctx, ctx->noalloc_scales != nullptr, "chi0_noalloc: scratch address not set up");
  if (n > 0) {
    const size_t mbytes = colmajor ? 16 * ((size_t)ldm * (nb - 1) + n)
                                   : 16 * ((size_t)ldm * (n - 1) + nb);
    SPX_CHECK(ctx, spx_owns(ctx, M, mbytes), "chi0_noalloc: M is not a context allocation of the stated shape");
    SPX_CHECK(ctx, spx_owns(ctx, wght, sizeof(double) * n * nw), "chi0_noalloc: wght is not a context allocation of n*nw doubles");
  }
  SPX_CHECK(ctx, spx_owns(ctx, chi, 16 * ((size_t)ldchi * nb * (nw - 1) + (size_t)ldchi * (nb - 1) + nb)),
            "chi0_noalloc: chi is not a context allocation of the stated shape");
  SPX_HIP(ctx, hipSetDevice(ctx->device));
  return spx_chi0_launch(ctx, ctx->stream, n, nb, M, ldm, colmajor, nw, wght, precision,
                         alpha, beta, chi, ldchi, ctx->noalloc_scales,
                         sizeof(double) * SPEXHIP_NOALLOC_MAX_SCALES, CHI0_NO_PARTS);
}

int spexhip_pack_upper_d2h(spexhip_ctx *ctx, int nb, int nw, const void *X, int ldx,
                           double *packed, int accumulate) {
  if (!ctx) return SPEXHIP_E_INVALID;
  SPX_CHECK(ctx, nb > 0 && nw > 0 && ldx >= nb && packed, "pack: bad arguments");
  SPX_CHECK(ctx, spx_owns(ctx, X, 16 * ((size_t)ldx * nb * nw)), "pack: X is not a context allocation of the stated shape");
  SPX_HIP(ctx, hipSetDevice(ctx->device));
  const long npack = (long)nb * (nb + 1) / 2;
  const size_t bytes = 16 * (size_t)npack * nw;
  void *P;
  int rc = spx_scratch(ctx, bytes, &P);
  if (rc) return rc;
  const int bs = 256;
  hipLaunchKernelGGL(pack_upper_kernel, dim3((npack * nw + bs - 1) / bs), dim3(bs), 0,
                     ctx->stream, nb, nw, (const double2 *)X, (long)ldx, (double2 *)P);
  SPX_LAUNCHED(ctx);
  if (!accumulate) {
    SPX_HIP(ctx, hipMemcpyAsync(packed, P, bytes, hipMemcpyDeviceToHost, ctx->stream));
    SPX_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return SPEXHIP_OK;
  }
  double *tmp = (double *)malloc(bytes);
  SPX_CHECK(ctx, tmp, "pack: host allocation failed");
  hipError_t e = hipMemcpyAsync(tmp, P, bytes, hipMemcpyDeviceToHost, ctx->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(ctx->stream);
  if (e != hipSuccess) {
    free(tmp);
    return spx_seterr(ctx, SPEXHIP_E_DEVICE, "pack: copy failed: %s", hipGetErrorString(e));
  }
  for (size_t q = 0; q < bytes / 8; q++) packed[q] += tmp[q];
  free(tmp);
  return SPEXHIP_OK;
}

int spexhip_unpack_h2d(spexhip_ctx *ctx, int nb, int nw, const double *packed, void *X,
                       int ldx) {
  if (!ctx) return SPEXHIP_E_INVALID;
  SPX_CHECK(ctx, nb > 0 && nw > 0 && ldx >= nb && packed, "unpack: bad arguments");
  SPX_CHECK(ctx, spx_owns(ctx, X, 16 * ((size_t)ldx * nb * nw)), "unpack: X is not a context allocation of the stated shape");
  SPX_HIP(ctx, hipSetDevice(ctx->device));
  const long npack = (long)nb * (nb + 1) / 2;
  const size_t bytes = 16 * (size_t)npack * nw;
  void *P;
  int rc = spx_scratch(ctx, bytes, &P);
  if (rc) return rc;
  SPX_HIP(ctx, hipMemcpyAsync(P, packed, bytes, hipMemcpyHostToDevice, ctx->stream));
  const int bs = 256;
  const long tot = (long)nb * nb * nw;
  hipLaunchKernelGGL(unpack_kernel, dim3((tot + bs - 1) / bs), dim3(bs), 0, ctx->stream, nb, nw,
                     (const double2 *)P, (double2 *)X, (long)ldx);
  SPX_LAUNCHED(ctx);
  SPX_HIP(ctx, hipStreamSynchronize(ctx->stream));
  return SPEXHIP_OK;
}

int spexhip_susceptibility_none(spexhip_ctx *ctx, long n, int nb, const double *cprod,
                                long ldc, int nw, const double *wght, int precision,
                                double *susceph) {
  if (!ctx) return SPEXHIP_E_INVALID;
  SPX_CHECK(ctx, n >= 0 && nb > 0 && nw > 0 && ldc >= n && susceph, "susceptibility: bad arguments");
  if (n == 0) return SPEXHIP_OK;
  SPX_CHECK(ctx, cprod && wght, "susceptibility: null input");
  SPX_HIP(ctx, hipSetDevice(ctx->device));
  const size_t mb = 16 * (size_t)n * nb, wb = 8 * (size_t)n * nw,
               cb = 16 * (size_t)nb * nb * nw;
  void *dM = nullptr, *dW = nullptr, *dC = nullptr;
  int rc = spx_alloc(ctx, mb, &dM);
  if (!rc) rc = spx_alloc(ctx, wb, &dW);
  if (!rc) rc = spx_alloc(ctx, cb, &dC);
  if (!rc) {
    hipError_t e = hipMemcpy2DAsync(dM, 16 * n, cprod, 16 * ldc, 16 * n, nb,
                                    hipMemcpyHostToDevice, ctx->stream);
    if (e == hipSuccess)
      e = hipMemcpyAsync(dW, wght, wb, hipMemcpyHostToDevice, ctx->stream);
    if (e != hipSuccess)
      rc = spx_seterr(ctx, SPEXHIP_E_DEVICE, "susceptibility: upload failed: %s", hipGetErrorString(e));
  }
  if (!rc)
    rc = spx_chi0_launch(ctx, ctx->stream, n, nb, dM, n, 1, nw, dW, precision, 1.0, 0.0, dC, nb);
  if (!rc) rc = spexhip_pack_upper_d2h(ctx, nb, nw, dC, nb, susceph, 1);
  (void)hipStreamSynchronize(ctx->stream);
  if (dM) spx_free(ctx, dM);
  if (dW) spx_free(ctx, dW);
  if (dC) spx_free(ctx, dC);
  return rc;
}

}  // extern "C"
