// bf_aux.hip -- the small kernels around the fused beamformer: antenna
// stuffing (-s) and the incoherent beam (-q), and the per-beam power sums
// the AGC consumes.
#include "bf_common.h"

namespace {
// Sum of the squares of the eight signed nibbles of x.
__device__ __forceinline__ int nib_power(uint32_t x, int acc) { return __builtin_amdgcn_sdot8((int)x, (int)x, acc, false); }
constexpr int STUFF_WAVES = 8;
}  // namespace

// The sums of |d|^2 per output bin, over the bin's packets, 8 channels, 2 times
// and 2 pols: whole numbers.
//  stuff 1: beam b <- antenna ((b/16)%4)*16 + b%16  (dsaX_beamformer.cu:326-337)
//  stuff 2: beam 0 <- sum over all antennas          (dsaX_beamformer.cu:307-323)
// The per-32-sample beam sums in bpart are rewritten for the beams written here.
//
// Reading the voltages bounds it (two instructions a dword), so a wave reads
// whole lines, 16 packets in flight: one workgroup takes one 64-sample block of
// four groups, a wave eight antennas of it at a time, a lane 16 bytes of each
// packet: with antennas outermost (ORDER 0) eight lanes a 128-byte line of four
// groups, with groups outermost 16 lanes the 256 bytes of eight antennas.  Sums are
// kept per four packets, the finest bin.  64 antennas x 384 channels x 4096
// samples (201 MB): 33 us, 6.1 TB/s; with a thread per antenna and 32 bytes of
// each of its packets in turn it took 102.
template <int ORDER>
__global__ __launch_bounds__(64 * STUFF_WAVES) void bf_stuff_kernel(bfk_dims d, const uint8_t *__restrict__ in,
                                                                    const float *__restrict__ scale,
                                                                    uint8_t *__restrict__ out,
                                                                    float *__restrict__ power,
                                                                    float *__restrict__ bpart) {
  constexpr int ABIT = ORDER == 0 ? 3 : 1;   // lane bits: antennas from here on, groups from GBIT, 16-byte half 0
  constexpr int GBIT = ORDER == 0 ? 1 : 4;
  __shared__ __attribute__((aligned(16))) int S[256][4][8];   // [antenna][group][4 packets]
  static_assert(__alignof__(S) == 16, "S is written 16 bytes at a time");
  __shared__ int part[STUFF_WAVES][4][8];
  __shared__ float IB[4][10];                // up to 8 bins, then the two 32-sample halves
  const int nblk = d.nsamp / 64, t64 = blockIdx.x % nblk, g0 = blockIdx.x / nblk * 4;
  const int ng = min(4, d.ngroup - g0);
  const int nbin = 64 / d.tavg, fpb = 8 / nbin;   // bins, and sums of four packets per bin
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int gl = (lane >> GBIT) & 3, al = (lane >> ABIT) & 7;
  const long pstep = (long)d.nant * d.nchan * 4;
  int tot[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  for (int a0 = wave * 8; a0 < d.nant; a0 += 8 * STUFF_WAVES) {
    const int ant = a0 + al;
    const bool in_block = ant < d.nant && gl < ng;    // (other lanes read antenna 0 of the first group again)
    const uint8_t *src = in + chunk_offset(ORDER, (long)t64 * 32, in_block ? ant : 0, in_block ? g0 + gl : g0, d.nant,
                                           d.nchan, d.ngroup) + (lane & 1) * 16;
    int s[8];
#pragma unroll
    for (int hh = 0; hh < 2; hh++) {
      uint4 v[16];
#pragma unroll
      for (int p = 0; p < 16; p++) v[p] = *(const uint4 *)(src + (16 * hh + p) * pstep);
#pragma unroll
      for (int k = 0; k < 4; k++) {
        int x = 0;
#pragma unroll
        for (int p = 4 * k; p < 4 * k + 4; p++)
          x = nib_power(v[p].x, nib_power(v[p].y, nib_power(v[p].z, nib_power(v[p].w, x))));
        s[4 * hh + k] = in_block ? x : 0;
      }
    }
#pragma unroll
    for (int k = 0; k < 8; k++) {
      tot[k] += s[k];
      s[k] += __shfl_xor(s[k], 1);
    }
    if ((lane & 1) == 0) {
      *(int4 *)&S[ant][gl][0] = make_int4(s[0], s[1], s[2], s[3]);
      *(int4 *)&S[ant][gl][4] = make_int4(s[4], s[5], s[6], s[7]);
    }
  }
  // sum of antenna a's fine sums k0 .. k0 + n - 1 (exact in float)
  auto fsum = [&](int a, int g, int k0, int n) {
    int x = 0;
    for (int k = k0; k < k0 + n; k++) x += S[a][g][k];
    return (float)x;
  };
  if (d.stuff == 2) {
#pragma unroll
    for (int k = 0; k < 8; k++) {
      tot[k] += __shfl_xor(tot[k], 1);
#pragma unroll
      for (int m = 0; m < 3; m++) tot[k] += __shfl_xor(tot[k], 1 << (ABIT + m));
      if (al == 0 && (lane & 1) == 0) part[wave][gl][k] = tot[k];
    }
    __syncthreads();
    if (tid < 40) {
      const int g = tid / 10, j = tid % 10, n = j < 8 ? fpb : 4, k0 = j < 8 ? j * fpb : (j - 8) * 4;
      if (j >= 8 || j < nbin) {
        int x = 0;
        for (int w = 0; w < STUFF_WAVES; w++)
          for (int k = k0; k < k0 + n; k++) x += part[w][g][k];
        float y = (float)x;
        if (x > 1 << 24) {                 // not exact in float: rounded antenna by antenna
          y = 0.f;
          for (int a = 0; a < d.nant; a++) y += fsum(a, g, k0, n);
        }
        IB[g][j] = y;
      }
    }
  }
  __syncthreads();
  const int bend = d.stuff == 2 ? 1 : d.nbeam;
  for (int i = tid; i < bend * 4; i += 64 * STUFF_WAVES) {
    const int b = i >> 2, g = i & 3, ant = ((b / 16) % 4) * 16 + b % 16;
    if (g >= ng) continue;
    for (int k = 0; k < nbin; k++) {
      const float x = d.stuff == 2 ? IB[g][k] : (ant < d.nant ? fsum(ant, g, k * fpb, fpb) : 0.f);
      const long idx = out_index(d.layout, d.nout, d.nbeam, d.ngroup, t64 * nbin + k, b, g0 + g);
      if (power) power[idx] = x;
      out[idx] = requant_u8(x, scale[b]);
    }
    for (int hh = 0; hh < 2; hh++)
      bpart[((long)b * 2 * nblk + 2 * t64 + hh) * d.ngroup + g0 + g] =
          d.stuff == 2 ? IB[g][8 + hh] : (ant < d.nant ? fsum(ant, g, 4 * hh, 4) : 0.f);
  }
}

// beam_power[b] = sum over 32-sample units and groups of bpart[b][.][.]
// (badder + calc_allbp, dsaX_beamformer.cu:78-112,482-495).  One workgroup
// per beam, FP32 throughout: each thread sums its strided share in eight
// independent partial sums (all loads of a round issued before the adds),
// the waves reduce with cross-lane swaps and the four wave sums are added in
// LDS, all in a fixed order, so the result is deterministic.
__device__ __forceinline__ void beam_sum(const float *__restrict__ src, int n, float *__restrict__ dst) {
  __shared__ float red[4];
  const int tid = threadIdx.x;
  float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  int i = tid;
  for (; i + 7 * 256 < n; i += 8 * 256) {
    float v[8];
#pragma unroll
    for (int k = 0; k < 8; k++) v[k] = src[i + k * 256];
#pragma unroll
    for (int k = 0; k < 8; k++) acc[k] += v[k];
  }
  for (; i < n; i += 256) acc[0] += src[i];
  float s = ((acc[0] + acc[1]) + (acc[2] + acc[3])) + ((acc[4] + acc[5]) + (acc[6] + acc[7]));
#pragma unroll
  for (int m = 32; m > 0; m >>= 1) s += __shfl_xor(s, m);
  if ((tid & 63) == 0) red[tid >> 6] = s;
  __syncthreads();
  if (tid == 0) *dst = (red[0] + red[1]) + (red[2] + red[3]);
}

__global__ __launch_bounds__(256) void bf_beam_power_kernel(bfk_dims d, const float *__restrict__ bpart,
                                                            float *__restrict__ bp) {
  const int n = (d.nsamp / 32) * d.ngroup;
  beam_sum(bpart + (long)blockIdx.x * n, n, bp + blockIdx.x);
}

// The beam-power sums of every block of a batch in one launch: workgroup B
// is beam B - beam_start[j] of job j, reduced exactly as bf_beam_power_kernel
// does, so the sums are bit-identical to a per-block launch.
__global__ __launch_bounds__(256) void bf_beam_power_batch_kernel(const bfk_bp_job *__restrict__ jobs,
                                                                  const int *__restrict__ beam_start) {
  const int B = blockIdx.x;
  int j = 0;
  while (B >= beam_start[j + 1]) j++;
  const bfk_bp_job &job = jobs[j];
  const int b = B - beam_start[j];
  beam_sum(job.bpart + (long)b * job.n, job.n, job.out + b);
}

extern "C" int bfk_beam_power_batch(const void *d_jobs, const int *d_beam_start, int nbeams_total,
                                    void *stream) {
  if (nbeams_total < 1) return 0;
  hipLaunchKernelGGL(bf_beam_power_batch_kernel, dim3(nbeams_total), dim3(256), 0, (hipStream_t)stream,
                     (const bfk_bp_job *)d_jobs, d_beam_start);
  return bfk_check(hipGetLastError(), "bf_beam_power_batch_kernel");
}

extern "C" int bfk_stuff(const bfk_dims *d, const uint8_t *d_in, const float *d_scale,
                         uint8_t *d_out, float *d_power, float *d_bpart, void *stream) {
  if (d->nant > 256 || d->nsamp % 64 != 0) {
    bfk_set_error("bfk_stuff: unsupported shape nant=%d nsamp=%d", d->nant, d->nsamp);
    return -1;
  }
  const dim3 grid((d->nsamp / 64) * ((d->ngroup + 3) / 4)), block(64 * STUFF_WAVES);
  if (d->order == 0)
    hipLaunchKernelGGL(bf_stuff_kernel<0>, grid, block, 0, (hipStream_t)stream, *d, d_in, d_scale, d_out, d_power, d_bpart);
  else
    hipLaunchKernelGGL(bf_stuff_kernel<1>, grid, block, 0, (hipStream_t)stream, *d, d_in, d_scale, d_out, d_power, d_bpart);
  return bfk_check(hipGetLastError(), "bf_stuff_kernel");
}

extern "C" size_t bfk_bpart_bytes(const bfk_dims *d) {
  return (size_t)d->nbeam * (d->nsamp / 32) * d->ngroup * sizeof(float);
}

extern "C" int bfk_beam_power(const bfk_dims *d, const float *d_bpart, float *d_beam_power,
                              void *stream) {
  hipLaunchKernelGGL(bf_beam_power_kernel, dim3(d->nbeam), dim3(256), 0, (hipStream_t)stream, *d,
                     d_bpart, d_beam_power);
  return bfk_check(hipGetLastError(), "bf_beam_power_kernel");
}
