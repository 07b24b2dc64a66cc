// bf_weights.hip -- beam weights on the device (replaces calc_weights,
// dsaX_beamformer.cu:420-449): FP64 phase exp(-2 pi i f ang x / c) times the
// calibration, scaled by a power of two per (channel, pol, beam) and written
// as FP16, FP8 E4M3 hi+lo or FP6 E2M3 hi+lo (or hi+mid+lo) MFMA B-operand
// fragments.
#include <stdarg.h>

#include "bf_common.h"

static thread_local char g_err[256];
extern "C" const char *bfk_last_error(void) { return g_err; }
void bfk_set_error(const char *fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}
int bfk_check(hipError_t e, const char *what) {
  if (e == hipSuccess) return 0;
  bfk_set_error("%s: %s", what, hipGetErrorString(e));
  return -3; /* DSAXBF_EHIP */
}

extern "C" size_t bfk_wfrag_bytes(const bfk_dims *d) {
  return (size_t)d->ncal * 2 * d->nbt * d->nkc * 64 * (d->prec == 3 ? 3 * WFRAG_LANE_BYTES / 2 : WFRAG_LANE_BYTES);
}
extern "C" size_t bfk_wscale_bytes(const bfk_dims *d) {
  return (size_t)d->ncal * 2 * d->nbeam_pad * sizeof(float);
}

// The largest k in 0..kmax with m * 2^k <= 7.5 (0 for m = 0).
__device__ static inline int lane_boost(double m, int kmax) {
  if (!(m > 0.0)) return 0;
  int k = (int)floor(log2(7.5 / m));
  k = k < 0 ? 0 : k > kmax ? kmax : k;
  while (k > 0 && ldexp(m, k) > 7.5) k--;
  while (k < kmax && ldexp(m, k + 1) <= 7.5) k++;
  return k;
}

// (_Float16)x, correctly rounded, by way of a float rounded to odd.
__device__ __forceinline__ _Float16 f16_of(double x) {
  const float f = (float)x;
  uint32_t u = __builtin_bit_cast(uint32_t, f);
  u -= fabs((double)f) > fabs(x);
  u |= (double)f != x;
  const uint16_t nan = (uint16_t)(0x7e00u | (u >> 31 << 15));
  return x != x ? __builtin_bit_cast(_Float16, nan) : (_Float16)__builtin_bit_cast(float, u);
}

// The scale puts the largest
// component of the beam's weights in [2^14, 2^15) (FP16) or [128, 256) (FP8),
// or at exactly 7.5, the top of E2M3 (FP6); wscale holds the power factor
// that undoes it and the voltage code's unit (2^-9 for FP8, 1/8 for FP6).
// E2M3 has only two exponent bits, so FP6 also boosts each lane's 32 slots
// (16 antennas of one beam and K step) by the largest power of two that keeps
// them within 7.5, and each further part (lo; or mid, then lo) by the
// largest that keeps the lane's remaining residuals within 7.5; the lane's
// E8M0 MFMA operand scales take them back (their exponents stay >= 0).
//
// One workgroup per weight channel and 32-beam tile.  Its wave w is K step w & 1
// of antenna chunk w >> 1, a lane one lane of the operand: 16 antennas of one beam,
// of both pols, whose phase is the same.  The FP64 sine and cosine bound it, so
// each is computed once and kept in registers, and the threads of a beam meet only for its largest component.  A
// thread per beam and pol computed each sine four times and kept the weights in
// scratch: 384 channels x 64 antennas x 256 beams in FP16 136 us, 40 now; 48 groups of
// them in FP6 202 and 46; 384 x 256 x 1024 in FP8 2.69 and 1.26 ms.  (The phases in
// LDS, 2 wavefronts a SIMD: 83 us.  Conversions of FP64 to FP16 take some 38
// instructions each unless they go by way of a float.)
template <int PREC, int NKC>
__global__ __launch_bounds__(128 * NKC, PREC < 2 ? 4 : 2) void bf_weights_kernel(bfk_dims d, const float *__restrict__ antpos,
                                                         const float *__restrict__ cal,
                                                         const double *__restrict__ freqs,
                                                         const double *__restrict__ theta,
                                                         uint8_t *__restrict__ wfrag,
                                                         float *__restrict__ wscale) {
  constexpr int nt = 128 * NKC;
  __shared__ float4 cw[64 * NKC];           // both pols' (re, im) calibration
  __shared__ float pos[64 * NKC];
  __shared__ double wmax[2][2 * NKC][32];
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = tid >> 6, kc = wave >> 1, s2 = wave & 1;
  const int wc = blockIdx.x / d.nbt, bt = blockIdx.x % d.nbt, b = bt * 32 + n;
  const double f = d.wmode ? freqs[wc] : freqs[wc * 8 + 4];
  const bool live = b < d.nbeam;
  double ang = live ? theta[b] : 0.0;
  if (d.amode) ang = sin(ang);
  const double afac = -2.0 * M_PI * f * ang / 299792458.0;
  const int a0 = kc * 64 + h * 32 + s2 * 16, na = live ? min(16, d.nant - a0) : 0;
  for (int a = tid; a < d.nant; a += nt) {
    cw[a] = ((const float4 *)cal)[(long)a * d.ncal + wc];
    pos[a] = antpos[a];
  }
  __syncthreads();
  double s[16], c[16];
  // the weight of antenna a0 + i, pol q, unscaled
  auto weight = [&](int i, int q, double &wr, double &wi) {
    const float *w = (const float *)&cw[a0 + i] + 2 * q;
    wr = c[i] * w[0] - s[i] * w[1];
    wi = s[i] * w[0] + c[i] * w[1];
  };
  double mx[2] = {0.0, 0.0};
#pragma unroll
  for (int i = 0; i < 16; i++) {
    if (i >= na) continue;
    sincos(afac * (double)pos[a0 + i], &s[i], &c[i]);
#pragma unroll
    for (int q = 0; q < 2; q++) {
      double wr, wi;
      weight(i, q, wr, wi);
      mx[q] = fmax(mx[q], fmax(fabs(wr), fabs(wi)));
    }
  }
#pragma unroll
  for (int q = 0; q < 2; q++) {
    mx[q] = fmax(mx[q], __shfl_xor(mx[q], 32));
    if (h == 0) wmax[q][wave][n] = mx[q];
  }
  __syncthreads();

#pragma unroll 1
  for (int q = 0; q < 2; q++) {
    double m = 0.0;
    for (int w = 0; w < 2 * NKC; w++) m = fmax(m, wmax[q][w][n]);
    int k = 0;
    if (m > 0.0) frexp(m, &k);
    const int e = (PREC == 0 ? 15 : 8) - k;
    double sc = ldexp(1.0, e);
    if (PREC >= 2) sc = m > 0.0 ? 7.5 / m : 1.0;
    const int cq = wc * 2 + q;
    if (tid < 32)
      wscale[(long)cq * d.nbeam_pad + b] = (float)(PREC == 0   ? ldexp(1.0, -2 * e)
                                                   : PREC == 1 ? ldexp(1.0, 18 - 2 * e)
                                                               : 64.0 / (sc * sc));
    auto scaled = [&](int i, double &wr, double &wi) {
      wr = wi = 0.0;
      if (i < na) {
        weight(i, q, wr, wi);
        wr *= sc;
        wi *= sc;
      }
    };
    const long rec0 = (long)(cq * d.nbt + bt) * d.nkc + kc;
    if constexpr (PREC == 0) {
#pragma unroll
      for (int u = 0; u < 4; u++) {
        h8v v;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          double wr, wi;
          scaled(4 * u + i, wr, wi);
          v[(i & 1) + 4 * (i >> 1)] = f16_of(wr);
          v[(i & 1) + 4 * (i >> 1) + 2] = f16_of(wi);
        }
        *(h8v *)(wfrag + ((rec0 * 8 + 4 * s2 + u) * 64 + lane) * 16) = v;
      }
    } else if constexpr (PREC >= 2) {
      constexpr int NPART = PREC == 3 ? 3 : 2;
      double r[32];                     // slot j: Wr (j < 16) or Wi of antenna j % 16
#pragma unroll
      for (int i = 0; i < 16; i++) scaled(i, r[i], r[16 + i]);
      uint8_t *dst = wfrag + ((rec0 * 2 + s2) * NPART * 64 + lane) * 32;
      int ktot = 0;
      uint32_t sexp[3] = {0, 0, 0};
#pragma unroll 1
      for (int pt = 0; pt < NPART; pt++) {
        double rm = 0.0;
#pragma unroll
        for (int j = 0; j < 32; j++) rm = fmax(rm, fabs(r[j]));
        const int kb = lane_boost(rm, 127 - ktot < 60 ? 127 - ktot : 60);
        ktot += kb;
        const uint32_t ex = (uint32_t)(127 - ktot);   // E8M0 scale 2^-ktot of this part
        if (pt == 0) sexp[0] = ex;
        else if (pt == 1) sexp[1] = ex;
        else sexp[2] = ex;
        uint32_t code[6] = {0, 0, 0, 0, 0, 0};
#pragma unroll
        for (int j = 0; j < 32; j++) {
          const double rb = ldexp(r[j], kb);
          const uint32_t c = e2m3_encode(rb);
          r[j] = rb - e2m3_decode(c);
          const int bit = 6 * j, dw = bit >> 5, sh = bit & 31;
          code[dw] |= c << sh;
          if (sh > 26) code[dw + 1] |= c >> (32 - sh);
        }
        *(uint4 *)(dst + pt * 64 * 32) = make_uint4(code[0], code[1], code[2], code[3]);
        *(uint2 *)(dst + pt * 64 * 32 + 16) = make_uint2(code[4], code[5]);
      }
      *(uint2 *)(dst + 24) = make_uint2(sexp[0], sexp[1]);
      *(uint2 *)(dst + 64 * 32 + 24) = make_uint2(NPART == 3 ? sexp[2] : 0u, 0u);
      if (NPART == 3) *(uint2 *)(dst + 2 * 64 * 32 + 24) = make_uint2(0u, 0u);
    } else {
      uint32_t hi[8], lo[8];
#pragma unroll
      for (int u = 0; u < 4; u++) {
        uint32_t hr = 0, hi_i = 0, lr = 0, li = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
          double wr, wi;
          scaled(4 * u + i, wr, wi);
          const uint32_t br = e4m3_encode(wr), bi = e4m3_encode(wi);
          const uint32_t cr = e4m3_encode(wr - e4m3_decode(br));
          const uint32_t ci = e4m3_encode(wi - e4m3_decode(bi));
          hr |= br << (8 * i);  hi_i |= bi << (8 * i);
          lr |= cr << (8 * i);  li |= ci << (8 * i);
        }
        hi[2 * u] = hr; hi[2 * u + 1] = hi_i;
        lo[2 * u] = lr; lo[2 * u + 1] = li;
      }
      uint4 *ph = (uint4 *)(wfrag + ((rec0 * 2 + s2) * 2 * 64 + lane) * 32), *pl = ph + 64 * 2;
      ph[0] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
      ph[1] = make_uint4(hi[4], hi[5], hi[6], hi[7]);
      pl[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      pl[1] = make_uint4(lo[4], lo[5], lo[6], lo[7]);
    }
  }
}

extern "C" int bfk_weights(const bfk_dims *d, const float *d_antpos, const float *d_cal,
                           const double *d_freqs, const double *d_theta, void *d_wfrag,
                           float *d_wscale, void *stream) {
  const dim3 grid(d->ncal * d->nbt), block(128 * d->nkc);
#define WEIGHTS(P, K)                                                                                 \
  hipLaunchKernelGGL((bf_weights_kernel<P, K>), grid, block, 0, (hipStream_t)stream, *d, d_antpos, d_cal, \
                     d_freqs, d_theta, (uint8_t *)d_wfrag, d_wscale)
#define WEIGHTS_NKC(P)              \
  do {                              \
    if (d->nkc == 1) WEIGHTS(P, 1); \
    else if (d->nkc == 2) WEIGHTS(P, 2); \
    else WEIGHTS(P, 4);             \
  } while (0)
  if (d->prec == 0) WEIGHTS_NKC(0);
  else if (d->prec == 1) WEIGHTS_NKC(1);
  else if (d->prec == 2) WEIGHTS_NKC(2);
  else WEIGHTS_NKC(3);
#undef WEIGHTS_NKC
#undef WEIGHTS
  return bfk_check(hipGetLastError(), "bf_weights_kernel");
}
