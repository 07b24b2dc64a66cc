// fl_kernels.hip -- device work of the search-side RFI flagger on a
// [nbeam][ntime][nchan] uint8 filterbank block (gpu_flagger.cu:113-520).
//
// The reference reads the 1 GiB block (64 beams x 16384 times x 1024
// channels) once per statistic: calc_spectrum, calc_varspec, calc_ppspec and
// (as its loop calls it) calc_spectrum again, each with one 32-thread block
// per (beam, channel) walking a column at a stride of 1 KB, after scaley has
// read and written it.  Here:
//
//   fl_stats_kernel   one pass for every statistic, optionally scaling the
//                     block in place first (scaley fused, as a per-channel
//                     table of the 256 byte values built in LDS with the
//                     reference's FP64 formula): a workgroup owns a slab of
//                     256 to 32 of a beam's channels, each lane 4 of them read
//                     as one dword per row (a wave reads 256 contiguous bytes,
//                     or 32 and up of several rows), the 16 waves the 32 time
//                     segments of the reference's threads.  Sums are integers (exact in any order); the
//                     variance comes from exact integer sums (the reference's
//                     float sums differ from it by their rounding, < 1e-5
//                     relative); ppspec keeps the reference's 32-segment
//                     semantics (max over segments of the largest 128-sample
//                     bin mean, minus the minimum over segments 16..31: what
//                     its unsynchronised max-then-min tree leaves in slot 0).
//   fl_flag_ts_kernel one pass that replaces the masked (beam, channel)
//                     columns and sums each row of the flagged block (flag +
//                     make_ts): 16 bytes per lane.
//   fl_masks_kernel, fl_apply_kernel, fl_tsmask_kernel: the block step's masks
//                     and its second pass (scale, flag, row sums).
//   fl_flagts_kernel  the masked (beam, time) rows, channels 128..nchan-129.
//   and elementwise kernels for sumpulse, genrand (own counter-based
//   generator), the noise replacement copy and fix_zspec's median.
#include <stdint.h>

#include "bf_common.h"

namespace {
constexpr int FL_SW = 16;      // waves per stats workgroup
constexpr int FL_NSEG = 32;    // the reference's threads per (beam, channel)
constexpr int FL_TBIN = 128;   // ppspec bin
constexpr double FL_MN = 48.0, FL_SIG = 6.0;
constexpr int FL_RPW = 16;     // loads per wave in fl_flag_ts_kernel
// (unsigned char)(__float2uint_rn(2 * val) / 2): round half to even, the
// saturating conversion (NaN and negatives to 0), halve, keep the low byte.
__device__ inline uint32_t fl_u8(float val) {
  const float r = __builtin_rintf(2.0f * val);
  const uint32_t u = r > 0.f ? (r >= 4294967296.f ? 0xFFFFFFFFu : (uint32_t)r) : 0u;
  return (u >> 1) & 0xFFu;
}

// The replacement byte of flag / flagts: MN * bpwr stored to a byte
// (truncation toward zero, clamped to 0..255, NaN to 0).
__device__ inline uint32_t fl_rep(float bpwr) {
  const double v = FL_MN * (double)bpwr;
  return v > 0. ? (v >= 255. ? 255u : (uint32_t)v) : 0u;
}

// scaley on one byte: (float)fma((double)(x - spec0), SIG / sqrtf(var0), MN).
__device__ inline uint32_t fl_scale(uint32_t x, float s0, double k) {
  const float a = (float)x - s0;
  return fl_u8((float)__builtin_fma((double)a, k, FL_MN));
}

struct FlStats {
  const uint8_t *data;
  uint8_t *wdata;          // scaled block (scaley fused), else NULL
  const float *spec0, *var0;
  const float *spec_in;    // varspec's spectrum argument (NULL: the block's own mean)
  float *spec, *var, *mx, *pp;
  int nb, nt, nc;
};

// A beam's plane as a buffer resource.  The base goes through readfirstlane:
// a resource built from vector registers puts a waterfall loop around every
// load.
__device__ inline __amdgpu_buffer_rsrc_t fl_plane(const uint8_t *data, int bm, size_t plane) {
  const uint64_t base = (uint64_t)(data + (size_t)bm * plane);
  const uint64_t sbase = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)base) |
                         (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(base >> 32)) << 32;
  return buffer_rsrc((const void *)sbase, (uint32_t)plane);
}

// Work item of this workgroup: consecutive items (the slabs of one beam, which
// share its 128-byte lines below 128 channels) run on one XCD.
__device__ inline int fl_item() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }

// scaley as a table: lut[x][channel], the scaled byte of every input byte x for
// each of the slab's W channels, so that the lanes of a row (consecutive channel
// quads) read distinct banks whatever their bytes.  A channel with a nonzero
// mask byte holds the beam's replacement byte for every x instead, which makes
// flagging part of the lookup; channels past the band hold zeros.
template <int W> struct FlLutScratch {
  double k[W];
  float s0[W];
  int fix[W];                    // -1, or the byte of every x
};
template <int W>
__device__ inline void fl_lut_build(uint8_t *lut, FlLutScratch<W> &t, const float *spec0, const float *var0,
                                    const uint8_t *mask, uint32_t rep, int slab, int nc) {
  const int tid = threadIdx.x;
  if (tid < W) {
    const int ch = slab * W + tid;
    t.s0[tid] = ch < nc ? spec0[ch] : 0.f;
    t.k[tid] = ch < nc ? __ddiv_rn(FL_SIG, (double)__fsqrt_rn(var0[ch])) : 0.;
    t.fix[tid] = ch >= nc ? 0 : mask && mask[ch] ? (int)rep : -1;
  }
  __syncthreads();
  constexpr int QPR = W / 4;
  const int q = tid % QPR;
  float s[4];
  double k[4];
  int fix[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    s[j] = t.s0[4 * q + j];
    k[j] = t.k[4 * q + j];
    fix[j] = t.fix[4 * q + j];
  }
  for (int x = tid / QPR; x < 256; x += 1024 / QPR) {
    uint32_t o = 0;
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const uint32_t v = fl_scale((uint32_t)x, s[j], k[j]);
      o |= (fix[j] < 0 ? v : (uint32_t)fix[j]) << (8 * j);
    }
    *(uint32_t *)(lut + x * W + 4 * q) = o;
  }
  __syncthreads();
}

// The four bytes of x (channels c .. c + 3 of the slab) through the table.
template <int W>
__device__ inline uint32_t fl_lut4(const uint8_t *lut, uint32_t x, uint32_t c) {
  uint32_t a[4];
  if constexpr (W == 256) {
    // byte j of x over c's low byte, in one permute
    a[0] = __builtin_amdgcn_perm(x, c, 0x0C0C0400u);
    a[1] = __builtin_amdgcn_perm(x, c, 0x0C0C0500u);
    a[2] = __builtin_amdgcn_perm(x, c, 0x0C0C0600u);
    a[3] = __builtin_amdgcn_perm(x, c, 0x0C0C0700u);
  } else {
#pragma unroll
    for (int j = 0; j < 4; j++) a[j] = ((x >> (8 * j)) & 0xFFu) * W + c;
  }
  return (uint32_t)lut[a[0]] | (uint32_t)lut[a[1] + 1] << 8 | (uint32_t)lut[a[2] + 2] << 16 | (uint32_t)lut[a[3] + 3] << 24;
}
}  // namespace

// Every statistic of a (beam, W-channel slab) in one pass, optionally through
// scaley's table (SCALE) and writing the scaled block (WRITE).  Bound by the
// stream over the block where the grid fills the chip: 64 x 16384 x 1024 takes
// 0.174 ms (6.2 TB/s), 0.468 ms with scaley (4.6 TB/s read and written, a plain
// copy 5.1).  12 x 8192 x 400 takes 16 and 31 us (51 and 102 us on 24 workgroups
// of 256 channels).
//
// 16 waves; W/4 lanes read one row of the slab (a dword each), so a wave's load
// covers RPI = 256/W consecutive rows.  W is 256 where that gives the chip
// enough workgroups, else narrower (flk_stats says where).  Wave w walks
// segments w and w + 16 with PF loads in flight.  Rows are taken four at a time
// and their 4x4 bytes transposed, so that a channel's four samples are one
// dword: its sum is one sad and its sum of squares one dot product, 16 + 8
// instructions for 16 samples where byte-wise sums took 64.  PF = 8 is enough
// where the chip is full (the scaled read-only pass took 0.209 ms with 8 loads a
// wave and 0.220 with 16; 0.186 with non-temporal loads since); with less to do
// more loads a wave draw more.
template <int W, bool NT, bool SCALE, bool WRITE, bool WMAX>
__global__ __launch_bounds__(1024) void fl_stats_kernel(FlStats a) {
  constexpr int LPR = W / 4, RPI = 64 / LPR, TB = FL_TBIN / RPI, PF = W == 256 ? 8 : 16;
  static_assert(TB % PF == 0, "bins end on a prefetch block");
  // the table, and after the pass the waves' sums, in the same LDS
  constexpr int RED = (FL_NSEG + 3 * FL_SW) * W * 4, LUT = SCALE ? 256 * W : 4;
  __shared__ __attribute__((aligned(16))) uint8_t lds[RED > LUT ? RED : LUT];
  __shared__ FlLutScratch<SCALE ? W : 1> lt;
  uint8_t *lut = lds;
  const int nslab = (a.nc + W - 1) / W;
  const int item = fl_item();
  if (item >= a.nb * nslab) return;            // the whole workgroup
  const int bm = item / nslab, slab = item % nslab;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), lane = threadIdx.x & 63;
  const int cl = (lane & (LPR - 1)) * 4, rg = lane / LPR;
  const int c0 = slab * W + cl;
  const bool live = c0 < a.nc;
  const int per = a.nt / FL_NSEG, n1 = per / RPI, n2 = 2 * n1;   // loads per segment, per wave
  const size_t plane = (size_t)a.nt * a.nc;
  const __amdgpu_buffer_rsrc_t rin = fl_plane(a.data, bm, plane);
  // (non-live lanes read zeros past the plane's end, and their stores there are
  // dropped: the rows need no branch)
  const __amdgpu_buffer_rsrc_t rout = WRITE ? fl_plane(a.wdata, bm, plane) : rin;
  const uint32_t vo = live ? (uint32_t)rg * (uint32_t)a.nc + (uint32_t)c0 : 0x80000000u;
  // byte offset of the rows of load i (the last ones are re-read past the end)
  auto row = [&](int i) {
    i = min(i, n2 - 1);
    const int seg = i < n1 ? w : w + FL_SW, r = seg * per + (i < n1 ? i : i - n1) * RPI;
    return (uint32_t)r * (uint32_t)a.nc;
  };
  uint32_t buf[PF];
#pragma unroll
  for (int d = 0; d < PF; d++) buf[d] = __builtin_amdgcn_raw_buffer_load_b32(rin, vo, row(d), (NT ? 2 : 0));
  if constexpr (SCALE)
    fl_lut_build<W>(lut, lt, a.spec0 + (size_t)bm * a.nc, a.var0 + (size_t)bm * a.nc, nullptr, 0, slab, a.nc);
  uint32_t S[4] = {0, 0, 0, 0}, Q[4] = {0, 0, 0, 0}, bs[4] = {0, 0, 0, 0};
  uint32_t cm[2][4] = {{0, 0, 0, 0}, {0, 0, 0, 0}}, Me = 0, Mo = 0;
#pragma unroll
  for (int h = 0; h < 2; h++) {
    for (int i0 = h * n1; i0 < (h + 1) * n1; i0 += PF) {
#pragma unroll
      for (int d = 0; d < PF; d += 4) {
        uint32_t x[4];
#pragma unroll
        for (int r = 0; r < 4; r++) {
          x[r] = buf[d + r];
          // (every lane: cl + 3 < W keeps a non-live lane's lookups in the
          // table, and its statistics are never written)
          if (SCALE) x[r] = fl_lut4<W>(lut, x[r], (uint32_t)cl);
          if (WRITE) __builtin_amdgcn_raw_buffer_store_b32(x[r], rout, vo, row(i0 + d + r), (NT ? 2 : 0));
          if (WMAX) {
            typedef unsigned short us2 __attribute__((ext_vector_type(2)));
            const uint32_t e = x[r] & 0x00FF00FFu, o = (x[r] >> 8) & 0x00FF00FFu;
            Me = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2, Me), __builtin_bit_cast(us2, e)));
            Mo = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(us2, Mo), __builtin_bit_cast(us2, o)));
          }
        }
        const uint32_t l01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u), h01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u);
        const uint32_t l23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u), h23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
        const uint32_t t[4] = {__builtin_amdgcn_perm(l23, l01, 0x05040100u), __builtin_amdgcn_perm(l23, l01, 0x07060302u),
                               __builtin_amdgcn_perm(h23, h01, 0x05040100u), __builtin_amdgcn_perm(h23, h01, 0x07060302u)};
#pragma unroll
        for (int j = 0; j < 4; j++) {
          bs[j] = __builtin_amdgcn_sad_u8(t[j], 0u, bs[j]);
          Q[j] = __builtin_amdgcn_udot4(t[j], t[j], Q[j], false);
        }
        // the next loads into these registers once their values are dead: a
        // load issued earlier needs other registers, and the loop then rotates
        // registers whose loads are still in flight
#pragma unroll
        for (int r = 0; r < 4; r++)
          buf[d + r] = __builtin_amdgcn_raw_buffer_load_b32(rin, vo, row(i0 + PF + d + r), (NT ? 2 : 0));
        __builtin_amdgcn_sched_barrier(0);
      }
      if (((i0 - h * n1 + PF) & (TB - 1)) == 0) {          // end of a 128-sample bin
#pragma unroll
        for (int j = 0; j < 4; j++) {
#pragma unroll
          for (int o = LPR; o < 64; o <<= 1) bs[j] += __shfl_xor(bs[j], o, 64);
          S[j] += bs[j];
          cm[h][j] = max(cm[h][j], bs[j]);
          bs[j] = 0;
        }
      }
    }
  }
  uint32_t M[4] = {Me & 0xFFFFu, Mo & 0xFFFFu, Me >> 16, Mo >> 16};
#pragma unroll
  for (int j = 0; j < 4; j++)
#pragma unroll
    for (int o = LPR; o < 64; o <<= 1) {
      Q[j] += __shfl_xor(Q[j], o, 64);
      if (WMAX) M[j] = max(M[j], (uint32_t)__shfl_xor(M[j], o, 64));
    }
  uint32_t *lc = (uint32_t *)lds;                                          // [segment][W]: largest bin sum
  uint32_t *ls = lc + FL_NSEG * W, *lq = ls + FL_SW * W, *lm = lq + FL_SW * W;   // [wave][W]
  if (SCALE) __syncthreads();                                              // every wave is done with the table
  if (rg == 0) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      lc[w * W + cl + j] = cm[0][j];
      lc[(w + FL_SW) * W + cl + j] = cm[1][j];
      ls[w * W + cl + j] = S[j];
      lq[w * W + cl + j] = Q[j];
      if (WMAX) lm[w * W + cl + j] = M[j];
    }
  }
  __syncthreads();
  const int c = threadIdx.x, ch = slab * W + c;
  if (c >= W || ch >= a.nc) return;
  uint64_t St = 0, Qt = 0;
  uint32_t Mt = 0, cmax = 0, cmin = 0xFFFFFFFFu;
  for (int v = 0; v < FL_SW; v++) {
    St += ls[v * W + c];
    Qt += lq[v * W + c];
    if (WMAX) Mt = max(Mt, lm[v * W + c]);
  }
  for (int s = 0; s < FL_NSEG; s++) {
    cmax = max(cmax, lc[s * W + c]);
    if (s >= FL_NSEG / 2) cmin = min(cmin, lc[s * W + c]);
  }
  const size_t i = (size_t)bm * a.nc + ch;
  const double n = (double)a.nt;
  const float sp = (float)__ddiv_rn((double)St, n);
  if (a.spec) a.spec[i] = sp;
  if (a.var) {
    // sum (x - s)^2 = [(n Q - S^2) + (S - s n)^2] / n, exact up to its last
    // rounding when s is the mean
    const double s = (double)(a.spec_in ? a.spec_in[i] : sp);
    const double dl = __dsub_rn((double)St, __dmul_rn(s, n));
    const int64_t q = (int64_t)a.nt * (int64_t)Qt - (int64_t)St * (int64_t)St;
    const double num = __dadd_rn((double)q, __dmul_rn(dl, dl));
    a.var[i] = (float)__ddiv_rn(__ddiv_rn(num, n), n);
  }
  if (WMAX) a.mx[i] = (float)Mt;
  if (a.pp) a.pp[i] = (float)cmax / (float)FL_TBIN - (float)cmin / (float)FL_TBIN;
}

// ---- the block step's second pass ---------------------------------------------
namespace {
// Value of the lane whose number differs in bit O.
template <int O> __device__ inline uint32_t fl_xor_lane(uint32_t v) {
  if constexpr (O == 1) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0xB1, 0xF, 0xF, true);        // quad_perm 1,0,3,2
  else if constexpr (O == 2) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x4E, 0xF, 0xF, true);   // quad_perm 2,3,0,1
  else if constexpr (O == 4) return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, 0x101F);
  else return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x128, 0xF, 0xF, true);                        // O == 8: row_ror 8
}
// a summed over the lane pairs of bit O in the lanes with the bit clear, b in
// those with it set.
template <int O> __device__ inline uint32_t fl_fold(uint32_t a, uint32_t b, int lane) {
  if constexpr (O == 32) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    return r[0] + r[1];
  } else if constexpr (O == 16) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    return r[0] + r[1];
  } else {
    const bool up = lane & O;
    return (up ? b : a) + fl_xor_lane<O>(up ? a : b);
  }
}
// Sums of 16 rows over the LPR lanes of a row: rs[i] is this lane's share of
// row i (any 8 lanes' shares below 2^16), the result two rows' sums packed,
// rows 2k and 2k + 1 for k = (lane % LPR) / (LPR / 8).  Each fold halves both
// the rows a lane carries and the lanes that share them: 26 instructions for 16
// rows of 64 lanes, where a cross-lane sum per row takes 96.
template <int LPR> __device__ inline uint32_t fl_row_sums(const uint32_t (&rs)[16], int lane) {
  uint32_t p[8], q[4], r[2], v;
#pragma unroll
  for (int k = 0; k < 8; k++) p[k] = rs[2 * k] | rs[2 * k + 1] << 16;
#pragma unroll
  for (int k = 0; k < 4; k++) q[k] = fl_fold<LPR / 2>(p[k], p[k + 4], lane);
#pragma unroll
  for (int k = 0; k < 2; k++) r[k] = fl_fold<LPR / 4>(q[k], q[k + 2], lane);
  v = fl_fold<LPR / 8>(r[0], r[1], lane);
  if constexpr (LPR == 64) v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x141, 0xF, 0xF, true);   // row_half_mirror
  if constexpr (LPR >= 32) v += fl_xor_lane<2>(v);
  if constexpr (LPR >= 16) v += fl_xor_lane<1>(v);
  return v;
}

struct FlApply {
  uint8_t *data;
  const float *spec0, *var0;
  const uint8_t *mask;
  const float *bpwr;
  uint16_t *part;              // [beam][slab][time] row sums of the slab, or NULL
  const double *bsum;          // per-beam sums of the spectrum
  int *ran, *h_ran;            // set to 1 by a pass that ran, else 0 (device and host)
  float prev;                  // total power of the last block, and the jump that
  float jump;                  // has the block replaced instead
  int force;
  int nb, nt, nc;
};
}  // namespace

// scaley, flag and the row sums of make_ts in one pass in place, after the
// masks: the statistics come from a pass that only read the raw block, so the
// scaled block is written once and never read back.  64 x 16384 x 1024: the
// read-only pass and this one move 3 GiB where scaley + flag moved 4.
// Bound by the stream over the block (read and written).
//
// A workgroup takes a (beam, W-channel slab), its 16 waves a sixteenth of the
// times each; rows and prefetch as in fl_stats_kernel.  The masked channels are
// part of the table.  The slab's row sums (at most 256 * 255) go out as 16 bits.
// The pass leaves the block alone when the total power has jumped: the block is
// then replaced by noise, and the host, which sums the spectrum in the
// reference's order meanwhile, has the last word (force, or the noise).
template <int W, bool NT>
__global__ __launch_bounds__(1024) void fl_apply_kernel(FlApply a) {
  constexpr int LPR = W / 4, RPI = 64 / LPR, PF = 16;
  __shared__ __attribute__((aligned(16))) uint8_t lut[256 * W];
  __shared__ FlLutScratch<W> lt;
  const int nslab = (a.nc + W - 1) / W;
  const int item = fl_item();
  const int lane = threadIdx.x & 63;
  bool go = true;
  if (!a.force) {
    double e = 0.;
    for (int b = lane; b < a.nb; b += 64) e += a.bsum[b];
    for (int o = 32; o > 0; o >>= 1) e += __shfl_xor(e, o, 64);
    go = !(fabs(e - (double)a.prev) / (double)a.prev >= (double)a.jump);
  }
  if (blockIdx.x == 0 && threadIdx.x == 0) *a.ran = *a.h_ran = go;
  if (!go || item >= a.nb * nslab) return;       // the whole workgroup
  const int bm = item / nslab, slab = item % nslab;
  const int w = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int cl = (lane & (LPR - 1)) * 4, rg = lane / LPR;
  const int c0 = slab * W + cl;
  const int n = a.nt / 16 / RPI;                 // loads of this wave
  const uint32_t r0 = (uint32_t)w * (uint32_t)(a.nt / 16);
  const size_t plane = (size_t)a.nt * a.nc;
  const __amdgpu_buffer_rsrc_t rsrc = fl_plane(a.data, bm, plane);
  // (lanes past the band: zeros in, zeros from the table, stores dropped)
  const uint32_t vo = c0 < a.nc ? (uint32_t)rg * (uint32_t)a.nc + (uint32_t)c0 : 0x80000000u;
  auto row = [&](int i) { return (r0 + (uint32_t)(min(i, n - 1) * RPI)) * (uint32_t)a.nc; };
  uint32_t buf[PF];
#pragma unroll
  for (int d = 0; d < PF; d++) buf[d] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, vo, row(d), (NT ? 2 : 0));
  fl_lut_build<W>(lut, lt, a.spec0 + (size_t)bm * a.nc, a.var0 + (size_t)bm * a.nc, a.mask + (size_t)bm * a.nc,
                  fl_rep(a.bpwr[bm]), slab, a.nc);
  uint16_t *part = a.part ? a.part + (size_t)item * a.nt : nullptr;
  for (int i0 = 0; i0 < n; i0 += PF) {
    uint32_t rs[PF];
#pragma unroll
    for (int d = 0; d < PF; d++) {
      const uint32_t x = fl_lut4<W>(lut, buf[d], (uint32_t)cl);
      __builtin_amdgcn_raw_buffer_store_b32(x, rsrc, vo, row(i0 + d), (NT ? 2 : 0));
      rs[d] = __builtin_amdgcn_sad_u8(x, 0u, 0u);
      // (past the end this wave's last row again, into registers that are not used)
      buf[d] = __builtin_amdgcn_raw_buffer_load_b32(rsrc, vo, row(i0 + PF + d), (NT ? 2 : 0));
      __builtin_amdgcn_sched_barrier(0);
    }
    if (part) {
      const uint32_t v = fl_row_sums<LPR>(rs, lane);
      const int l = lane & (LPR - 1), k = l / (LPR / 8);
      if (l % (LPR / 8) == 0) {
        const uint32_t t = r0 + (uint32_t)((i0 + 2 * k) * RPI + rg);
        if constexpr (RPI == 1) {
          *(uint32_t *)(part + t) = v;           // t is even
        } else {
          part[t] = (uint16_t)v;
          part[t + RPI] = (uint16_t)(v >> 16);
        }
      }
    }
  }
}

// ---- the masks ------------------------------------------------------------------
namespace {
constexpr int FL_ZERO = 128, FL_FILT = 21, FL_FBIN = 8;   // band edge, median window, simple_channflag bin
constexpr int FL_LDSN = 4096;                             // values of one selection kept in LDS

// Floats in order as unsigned numbers (finite values).
__device__ inline uint32_t fl_key(float v) {
  const uint32_t u = __builtin_bit_cast(uint32_t, v);
  return u ^ ((uint32_t)((int)u >> 31) | 0x80000000u);
}
__device__ inline float fl_unkey(uint32_t k) {
  return __builtin_bit_cast(float, k & 0x80000000u ? k ^ 0x80000000u : ~k);
}

// The k-th smallest (from 0) of the n keys get(i), for every thread of a team
// of four waves.  The keys' range is cut into at most 256 bins of a power of two
// and the one that holds the k-th taken as the next range: four rounds at most.
// (One bit a round, counted by one wave or by all of them, took 9 us for 768
// keys: few waves issue an instruction only every eight cycles or so.)  Every
// thread of the workgroup calls it (it has barriers), teams with data and FlSel
// of their own.
struct alignas(16) FlSel {
  uint32_t hist[256];
  uint32_t lo[4], hi[4];             // per wave, then the range in [0]
  uint32_t k;
};
static_assert(alignof(FlSel) == 16, "hist is read 16 bytes at a time, in every element of an array");
template <class G> __device__ inline uint32_t fl_kth(G get, int n, int k, int tid, FlSel &t) {
  const int lane = tid & 63;
  uint32_t lo = 0xFFFFFFFFu, hi = 0;
  for (int i = tid; i < n; i += 256) {
    const uint32_t x = get(i);
    lo = min(lo, x);
    hi = max(hi, x);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    lo = min(lo, (uint32_t)__shfl_xor((int)lo, o, 64));
    hi = max(hi, (uint32_t)__shfl_xor((int)hi, o, 64));
  }
  __syncthreads();                   // the last call's reads
  if (lane == 0) {
    t.lo[tid >> 6] = lo;
    t.hi[tid >> 6] = hi;
  }
  t.hist[tid] = 0;
  __syncthreads();
  lo = min(min(t.lo[0], t.lo[1]), min(t.lo[2], t.lo[3]));
  hi = max(max(t.hi[0], t.hi[1]), max(t.hi[2], t.hi[3]));
  uint32_t uk = (uint32_t)k;
#pragma unroll 1
  for (int r = 0; r < 4; r++) {
    const int width = 32 - __builtin_clz((hi - lo) | 1u), s = width > 8 ? width - 8 : 0;
    for (int i = tid; i < n; i += 256) {
      const uint32_t x = get(i);
      if (x >= lo && x <= hi) atomicAdd(&t.hist[(x - lo) >> s], 1u);
    }
    __syncthreads();
    if (tid < 64) {
      const uint4 c = *(const uint4 *)&t.hist[4 * lane];
      uint32_t sum = c.x + c.y + c.z + c.w;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t v = (uint32_t)__shfl_up((int)sum, o, 64);
        if (lane >= o) sum += v;
      }
      // the first lane whose running count passes k, and its bin
      const int at = __ffsll((unsigned long long)__ballot(sum > uk)) - 1;
      if (lane == at) {
        uint32_t e = sum - (c.x + c.y + c.z + c.w), bin = 4 * lane;
        if (uk >= e + c.x) { e += c.x; bin++; if (uk >= e + c.y) { e += c.y; bin++; if (uk >= e + c.z) { e += c.z; bin++; } } }
        t.k = uk - e;
        t.lo[0] = lo + (bin << s);
        t.hi[0] = min(hi, lo + (bin << s) + ((1u << s) - 1));
      }
    }
    __syncthreads();
    lo = t.lo[0];
    hi = t.hi[0];
    uk = t.k;
    t.hist[tid] = 0;
    __syncthreads();
  }
  return lo;
}

// Median of 21 values: of 12 the smallest and the largest are dropped and the
// next value joins, until three are left (92 exchanges; no value can be the
// median once it is the extreme of more than half of them).
__device__ inline float fl_median21(const float *w) {
  float a[12];
#pragma unroll
  for (int i = 0; i < 12; i++) a[i] = w[i];
#pragma unroll
  for (int n = 12; n > 3; n--) {
    auto order = [&](int i, int j) {
      const float lo = fminf(a[i], a[j]), hi = fmaxf(a[i], a[j]);
      a[i] = lo;
      a[j] = hi;
    };
#pragma unroll
    for (int i = 0; i < n / 2; i++) order(i, n - 1 - i);
#pragma unroll
    for (int i = 1; i < (n + 1) / 2; i++) order(0, i);          // the smallest to the front
#pragma unroll
    for (int i = n / 2; i < n - 1; i++) order(i, n - 1);        // the largest to the back
    a[0] = w[24 - n];                                           // n = 12: w[12], ..., n = 4: w[20]
  }
  return __builtin_amdgcn_fmed3f(a[0], a[1], a[2]);
}

struct FlMasks {
  const float *spec, *var, *pp;
  float *big;                   // [3][beam][nchan - 256] where that is above FL_LDSN, else NULL
  uint8_t *mask;                // [beam][channel], 0 or 1
  int *h_nmask;                 // per beam (host)
  float *h_spec;                // the spectrum for the host
  double *bsum;
  float *bpwr;                  // calc_bpwr's levels, or NULL to leave them
  float thr[3];                 // channflag of spec and of var, simple_channflag of pp (over sqrt(FBIN))
  int nb, nc, nperm;
  int perm[64];
};
}  // namespace

// channflag on spec and var, simple_channflag on pp (gpu_flagger.cu:557-660),
// and the count of the flagged channels: workgroup (beam, 0), a team of four
// waves per statistic.  Every float and double operation of the reference's CPU
// code, in its order; medians are selections, so which equal element is taken
// does not matter.  Workgroup (beam, 1): the spectrum to the host, its sum, and
// calc_bpwr.  64 beams x 1024 channels: 20-30 us (a spread of the writes to host
// memory) for what took the host, with the copies both ways, about 0.6 ms.
// Bound by its barriers and the latency of few waves.
__global__ __launch_bounds__(768) void fl_masks_kernel(FlMasks a) {
  __shared__ float val[3][FL_LDSN];
  __shared__ FlSel sel[3];
  __shared__ uint32_t cnt[12];
  __shared__ double red[12];
  const int bm = blockIdx.x, tid = threadIdx.x;
  const size_t at = (size_t)bm * a.nc;
  if (blockIdx.y == 1) {
    double s = 0.;
    for (int c = tid; c < a.nc; c += 768) {
      const float v = a.spec[at + c];
      a.h_spec[at + c] = v;
      s += (double)v;
    }
    for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    if ((tid & 63) == 0) red[tid >> 6] = s;
    __syncthreads();
    if (tid == 0) {
      for (int k = 1; k < 12; k++) s += red[k];
      a.bsum[bm] = s;
    }
    if (!a.bpwr) return;
    // calc_bpwr's float sum in channel order, a stretch of the row at a time
    float f = 0.f;
    for (int c0 = 0; c0 < a.nc; c0 += FL_LDSN) {
      const int m = min(FL_LDSN, a.nc - c0);
      __syncthreads();
      for (int c = tid; c < m; c += 768) val[0][c] = a.spec[at + c0 + c];
      __syncthreads();
      if (tid == 0) {
#pragma unroll 16
        for (int c = 0; c < m; c++) f = __fadd_rn(f, val[0][c]);
      }
    }
    if (tid == 0) a.bpwr[bm] = (float)__ddiv_rn(__ddiv_rn((double)f, (double)(a.nc - 2 * FL_ZERO)), FL_MN);
    return;
  }
  const int team = tid >> 8, tt = tid & 255;
  const int nin = a.nc - 2 * FL_ZERO;
  uint8_t *mask = a.mask + at;
  for (int c = tid; c < a.nc; c += 768) mask[c] = 0;
  const float *row = (team == 0 ? a.spec : team == 1 ? a.var : a.pp) + at + FL_ZERO;
  float *v = nin <= FL_LDSN ? val[team] : a.big + ((size_t)team * a.nb + bm) * nin;
  for (int j = tt; j < nin; j += 256) {
    float x = row[j];
    if (team < 2) {
      float w[FL_FILT];
      const float *src = row + min(j, nin - FL_FILT);
#pragma unroll
      for (int i = 0; i < FL_FILT; i++) w[i] = src[i];
      x = __fsub_rn(x, fl_median21(w));
    }
    v[j] = x;
  }
  __syncthreads();
  const int k = (nin + 1) / 2 - 1;
  const float med = fl_unkey(fl_kth([&](int i) { return fl_key(v[i]); }, nin, k, tt, sel[team]));
  const float mad = fl_unkey(fl_kth([&](int i) { return fl_key(fabsf(__fsub_rn(v[i], med))); }, nin, k, tt, sel[team]));
  const float lim = __fmul_rn(a.thr[team], mad);
  // (teams that set the same byte store the same value)
  if (team < 2) {
    for (int j = tt; j < nin; j += 256)
      if (v[j] > lim || v[j] < -lim) mask[FL_ZERO + j] = 1;
    if (tid < a.nperm && a.perm[tid] >= FL_ZERO && a.perm[tid] < a.nc - FL_ZERO) mask[a.perm[tid]] = 1;
  } else {
    for (int j = tt; j < nin - FL_FBIN; j += 256) {
      float s = 0.f;
#pragma unroll
      for (int i = 0; i < FL_FBIN; i++) s = __fadd_rn(s, v[j]);       // the same element FBIN times
      if ((float)__dsub_rn((double)s * (1. / FL_FBIN), (double)med) > lim) mask[FL_ZERO + j] = 1;
    }
  }
  __syncthreads();
  uint32_t m = 0;
  for (int c = tid; c < a.nc; c += 768) m += mask[c];
  for (int o = 32; o > 0; o >>= 1) m += __shfl_xor(m, o, 64);
  if ((tid & 63) == 0) cnt[tid >> 6] = m;
  __syncthreads();
  if (tid == 0) {
    for (int i = 1; i < 12; i++) m += cnt[i];
    a.h_nmask[bm] = (int)m;
  }
}

namespace {
struct FlTsMask {
  const uint16_t *part;         // fl_apply_kernel's row sums, or NULL: ts holds the series
  float *ts;
  int *idx, *n_ts, *h_nts;      // per beam: flagged rows (beam * ntime + time), their count (device and host)
  const int *ran;               // fl_apply_kernel's flag, or NULL
  float thr;
  int nb, nt, nc, nslab;
};
}  // namespace

// make_ts's division and simple_tsflag (gpu_flagger.cu:413-452,662-700): a
// workgroup per beam, the series' median and MAD over its first ntime/16
// samples, and the list of its flagged rows.  (The four teams of four waves
// each select the same values; the order of the list does not matter.)  64 x
// 16384: 23 us, bound by the latency of 64 workgroups.
__global__ __launch_bounds__(1024) void fl_tsmask_kernel(FlTsMask a) {
  __shared__ float val[FL_LDSN];
  __shared__ FlSel sel[4];
  __shared__ uint32_t nf;
  const int bm = blockIdx.x, tid = threadIdx.x, tt = tid & 255, team = tid >> 8;
  const int nm = a.nt / 16;
  float *ts = a.ts + (size_t)bm * a.nt;
  const bool live = !a.ran || *a.ran;
  if (tid == 0) nf = 0;
  if (!live) {                                   // the whole grid
    if (tid == 0) a.n_ts[bm] = a.h_nts[bm] = 0;
    return;
  }
  if (a.part) {
    const uint16_t *p = a.part + (size_t)bm * a.nslab * a.nt;
    const double rnc = __ddiv_rn(1., (double)a.nc);
#pragma unroll 2
    for (int t = tid * 4; t < a.nt; t += 4096) {
      uint32_t s[4] = {0, 0, 0, 0};
#pragma unroll 4
      for (int k = 0; k < a.nslab; k++) {
        const uint2 v = *(const uint2 *)(p + (size_t)k * a.nt + t);
        s[0] += v.x & 0xFFFFu;
        s[1] += v.x >> 16;
        s[2] += v.y & 0xFFFFu;
        s[3] += v.y >> 16;
      }
      // s / nc by its reciprocal and one exact remainder: a quotient that a
      // double holds comes out exact, another one within an ulp of a double,
      // which is far nearer than a float's rounding boundary can be
      float f[4];
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const double d = (double)s[j], q = d * rnc;
        f[j] = (float)__builtin_fma(__builtin_fma(-q, (double)a.nc, d), rnc, q);
      }
      *(float4 *)(ts + t) = make_float4(f[0], f[1], f[2], f[3]);
    }
    __syncthreads();
  }
  const float *v = ts;
  if (nm <= FL_LDSN) {
    for (int t = tid; t < nm; t += 1024) val[t] = ts[t];
    v = val;
  }
  __syncthreads();
  const int k = (nm + 1) / 2 - 1;
  const float med = fl_unkey(fl_kth([&](int i) { return fl_key(v[i]); }, nm, k, tt, sel[team]));
  const float mad = fl_unkey(fl_kth([&](int i) { return fl_key(fabsf(__fsub_rn(v[i], med))); }, nm, k, tt, sel[team]));
  const float lim = __fmul_rn(a.thr, mad);
  int *idx = a.idx + (size_t)bm * a.nt;
#pragma unroll 4
  for (int t = tid * 4; t < a.nt; t += 4096) {
    const float4 f = *(const float4 *)(ts + t);
    const float x[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (__fsub_rn(x[j], med) > lim) idx[atomicAdd(&nf, 1u)] = bm * a.nt + t + j;
  }
  __syncthreads();
  if (tid == 0) a.n_ts[bm] = a.h_nts[bm] = (int)nf;
}

// bytes != 0 -> 0xFF, == 0 -> 0x00
__device__ inline uint32_t fl_bytemask(uint32_t x) {
  x |= (x >> 4) & 0x0F0F0F0Fu;
  x |= (x >> 2) & 0x33333333u;
  x |= (x >> 1) & 0x55555555u;
  return (x & 0x01010101u) * 0xFFu;
}

// Sums of 16 rows over the LPR lanes of a row, for the lane's row
// (lane % LPR) / (LPR / 16): as fl_row_sums, in 32 bits.
template <int LPR> __device__ inline uint32_t fl_row_sums32(const uint32_t (&rs)[FL_RPW], int lane) {
  static_assert(FL_RPW == 16 && LPR >= 16, "four folds");
  uint32_t p[8], q[4], r[2], v;
#pragma unroll
  for (int k = 0; k < 8; k++) p[k] = fl_fold<LPR / 2>(rs[k], rs[k + 8], lane);
#pragma unroll
  for (int k = 0; k < 4; k++) q[k] = fl_fold<LPR / 4>(p[k], p[k + 4], lane);
#pragma unroll
  for (int k = 0; k < 2; k++) r[k] = fl_fold<LPR / 8>(q[k], q[k + 2], lane);
  v = fl_fold<LPR / 16>(r[0], r[1], lane);
  if constexpr (LPR == 64) v += fl_xor_lane<2>(v);
  if constexpr (LPR >= 32) v += fl_xor_lane<1>(v);
  return v;
}

// Replace the masked columns (mask[bm][ch] != 0) with the beam's byte and,
// when ts is given, write ts[bm][t] = (sum over channels of the flagged row)
// / nchan.  LPR lanes read a row, 16 bytes each (64, or 32 and 16 for rows of
// fewer 16-byte chunks, so that lanes are not idle: make_ts of 12 x 8192 x 400
// takes 8 us where a wave per row took 16), a wave FL_RPW loads of 64/LPR rows each.
// A lane stores its chunk when the chunk holds a masked column, or, when at
// least a quarter of the wave's chunks do, every lane stores (unchanged chunks
// are written back as read): on the 64 x 16384 x 1024 block, 5 % of columns
// masked at random touch every line of a row, and whole rows then take
// 0.382 ms against 0.430 ms as scattered chunks, while 0.5 % at random or a
// 64-channel band run faster as chunks (0.305 and 0.271 ms, against 0.414
// whole).  (Row sums by a cross-lane sum per row: 0.425 ms with 5 %.)
template <int LPR, bool MASK>
__global__ __launch_bounds__(256) void fl_flag_ts_kernel(uint8_t *data, const uint8_t *mask,
                                                         const float *bpwr, float *ts, int nb, int nt,
                                                         int nc) {
  constexpr int RPI = 64 / LPR;                // rows per load
  const int lane = threadIdx.x & 63, l = lane & (LPR - 1), rg = lane / LPR;
  const long gw = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  const int wpb = nt / (FL_RPW * RPI);         // waves per beam
  if (gw >= (long)nb * wpb) return;            // the whole wave leaves together
  const int bm = (int)(gw / wpb), t0 = (int)(gw % wpb) * FL_RPW * RPI;
  const int nq = nc / 16;                      // 16-byte chunks per row
  const uint32_t rep = MASK ? fl_rep(bpwr[bm]) * 0x01010101u : 0u;
  uint32_t rs[FL_RPW];
#pragma unroll
  for (int r = 0; r < FL_RPW; r++) rs[r] = 0;
  for (int q = l; q - l < nq; q += LPR) {
    if (q >= nq) break;
    uint4 m = make_uint4(0, 0, 0, 0);
    if (MASK) {
      m = *(const uint4 *)(mask + (size_t)bm * nc + 16 * q);
      m = make_uint4(fl_bytemask(m.x), fl_bytemask(m.y), fl_bytemask(m.z), fl_bytemask(m.w));
    }
    const bool own = (m.x | m.y | m.z | m.w) != 0;
    // (both ballots in every active lane: under `own ||` they would run only
    // in the lanes whose chunk is clean)
    const bool whole = 4 * __popcll(__ballot(own)) >= __popcll(__ballot(1));
    const bool any = MASK && (own || whole);
#pragma unroll
    for (int r = 0; r < FL_RPW; r++) {
      uint4 *pv = (uint4 *)(data + ((size_t)bm * nt + t0 + r * RPI + rg) * nc + 16 * q);
      uint4 v = *pv;
      if (any) {
        v.x = (v.x & ~m.x) | (rep & m.x);
        v.y = (v.y & ~m.y) | (rep & m.y);
        v.z = (v.z & ~m.z) | (rep & m.z);
        v.w = (v.w & ~m.w) | (rep & m.w);
        *pv = v;
      }
      uint32_t s = __builtin_amdgcn_sad_u8(v.x, 0u, rs[r]);
      s = __builtin_amdgcn_sad_u8(v.y, 0u, s);
      s = __builtin_amdgcn_sad_u8(v.z, 0u, s);
      rs[r] = __builtin_amdgcn_sad_u8(v.w, 0u, s);
    }
  }
  if (ts) {
    const uint32_t s = fl_row_sums32<LPR>(rs, lane);
    if (l % (LPR / 16) == 0)
      ts[(size_t)bm * nt + t0 + l / (LPR / 16) * RPI + rg] = (float)__ddiv_rn((double)s, (double)nc);
  }
}

// flagts (gpu_flagger.cu:478-494): row midx[i] = bm * ntime + t, channels
// 128 .. nchan-129 set to the beam's byte.  A wave per listed row.
__global__ __launch_bounds__(256) void fl_flagts_kernel(uint8_t *data, const int *midx, int n,
                                                        const float *bpwr, int nb, int nt, int nc) {
  const int lane = threadIdx.x & 63;
  const long i = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (i >= n) return;
  const int m = midx[i];
  if (m < 0 || m >= nb * nt) return;
  const int bm = m / nt;
  const uint32_t rep = fl_rep(bpwr[bm]) * 0x01010101u;
  uint8_t *row = data + (size_t)m * nc;
  for (int q = 8 + lane; q < nc / 16 - 8; q += 64) *(uint4 *)(row + 16 * q) = make_uint4(rep, rep, rep, rep);
}

// flagts on fl_tsmask_kernel's lists: blockIdx.x the beam, the waves of the
// beam's gridDim.y workgroups a row each in turn.
__global__ __launch_bounds__(256) void fl_flagts_list_kernel(uint8_t *data, const int *idx, const int *n_ts,
                                                             const float *bpwr, int nt, int nc) {
  const int bm = blockIdx.x, lane = threadIdx.x & 63;
  const int n = n_ts[bm];
  const uint32_t rep = fl_rep(bpwr[bm]) * 0x01010101u;
  for (int i = blockIdx.y * 4 + (threadIdx.x >> 6); i < n; i += gridDim.y * 4) {
    uint8_t *row = data + (size_t)idx[(size_t)bm * nt + i] * nc;
    for (int q = 8 + lane; q < nc / 16 - 8; q += 64) *(uint4 *)(row + 16 * q) = make_uint4(rep, rep, rep, rep);
  }
}

// flag (gpu_flagger.cu:458-474): column midx[i] = bm * nchan + ch, every time.  3 %
// of the columns of 12 x 8192 x 400 take 10 us, but 16 after scaley in 32-channel
// slabs, also some ms after it (10 after it in 256-channel slabs, which take 71 us
// longer): what state of the caches the narrow slabs leave was not looked into.
__global__ __launch_bounds__(256) void fl_flag_cols_kernel(uint8_t *data, const int *midx, int n,
                                                           const float *bpwr, int nb, int nt, int nc) {
  const int i = blockIdx.y;
  const int t = blockIdx.x * 256 + threadIdx.x;
  if (i >= n || t >= nt) return;
  const int m = midx[i];
  if (m < 0 || m >= nb * nc) return;
  const int bm = m / nc, ch = m % nc;
  data[((size_t)bm * nt + t) * nc + ch] = (uint8_t)fl_rep(bpwr[bm]);
}

// sumpulse (gpu_flagger.cu:398-406): 4 bytes per thread, a tail thread for
// the last n % 4.
__global__ __launch_bounds__(256) void fl_sumpulse_kernel(uint8_t *data, const float *summand, size_t n) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i + 4 <= n) {
    const uint32_t x = *(const uint32_t *)(data + i);
    const float4 s = *(const float4 *)(summand + i);
    *(uint32_t *)(data + i) = fl_u8((float)(x & 0xFF) + s.x) | fl_u8((float)((x >> 8) & 0xFF) + s.y) << 8 |
                              fl_u8((float)((x >> 16) & 0xFF) + s.z) << 16 | fl_u8((float)(x >> 24) + s.w) << 24;
  } else {
    for (size_t j = i; j < n; j++) data[j] = (uint8_t)fl_u8((float)data[j] + summand[j]);
  }
}

__device__ inline uint64_t fl_mix(uint64_t z) {
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

// genrand (gpu_flagger.cu:499-520) with a counter-based generator: element i
// from the splitmix64 finaliser of (seed * 2^32 + i), uniforms
// (32-bit half % 16384) / 16384, Box-Muller in FP64.
__global__ __launch_bounds__(256) void fl_genrand_kernel(uint8_t *rep, size_t n, uint32_t seed) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint64_t r = fl_mix(((uint64_t)seed << 32) + i);
  const double u1 = (double)((uint32_t)r % 16384u) / 16384.0;
  const double u2 = (double)((uint32_t)(r >> 32) % 16384u) / 16384.0;
  const double va = sqrt(-2.0 * log(u1)) * cos(2.0 * M_PI * u2);
  rep[i] = (uint8_t)fl_u8((float)__builtin_fma(va, FL_SIG, FL_MN));
}

// Every beam of the block replaced by the [ntime][nchan] noise block
// (the reference's per-beam device copies, gpu_flagger.cu:1319-1320,1356-1358).
__global__ __launch_bounds__(256) void fl_noise_kernel(uint8_t *data, const uint8_t *rep, size_t per_beam,
                                                       int nb) {
  const size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * 16;
  if (i >= per_beam) return;
  const uint4 v = *(const uint4 *)(rep + i);
  for (int b = 0; b < nb; b++) *(uint4 *)(data + (size_t)b * per_beam + i) = v;
}

// fix_zspec (gpu_flagger.cu:113-168): entry i of s0 / v0 becomes the value
// among the naver stacked blocks with exactly naver/2 others <= it; with no
// such value (ties) entry i keeps block 0's.
__global__ __launch_bounds__(256) void fl_fix_zspec_kernel(float *s0, float *v0, int nbc, int naver) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i >= nbc) return;
  const int place = naver / 2;
  for (int h = 0; h < 2; h++) {
    float *a = h ? v0 : s0;
    float pick = a[i];
    for (int t = 0; t < naver; t++) {
      const float x = a[(size_t)t * nbc + i];
      int ct = 0;
      for (int k = 0; k < naver; k++) ct += (k != t && a[(size_t)k * nbc + i] <= x);
      if (ct == place) pick = x;
    }
    a[i] = pick;
  }
}

// ---- launchers --------------------------------------------------------------

static bool fl_shape_ok(int nb, int nt, int nc, const char *who) {
  if (nb < 1 || nt < 4096 || nt % 4096 || nc < 16 || nc % 16 || (long)nb * nt > (1L << 30) / 16 ||
      (long)nt * nc >= (1L << 31)) {
    bfk_set_error("%s: shape %d x %d x %d unsupported (ntime a multiple of 4096, nchan of 16)", who, nb,
                  nt, nc);
    return false;
  }
  return true;
}

// Channels per slab of the block-wide passes: the widest that still gives more
// than half the CUs a workgroup.  Wide slabs read whole cache lines (64 x 16384
// x 1024 scaley: 256, 128, 64 and 32 channels take 475, 498, 540 and 693 us),
// but few workgroups cannot draw the bandwidth (12 x 8192 x 400: 105, 62, 37
// and 31 us; 8 x 8192 x 1024, where 64 channels give just half: 118, 80, 64 and 54;
// 30 x 16384 x 640: 249, 160, 214 and 271; a step of 20 x 16384 x 400: 64 and 32
// channels, 140 and 260 workgroups, 170 and 214).
static int fl_slab_width(int nb, int nc) {
  int w = 256;
  while (w > 32 && (long)nb * ((nc + w - 1) / w) <= 128) w >>= 1;
  return w;
}

// Whether the slab passes read and write the block non-temporally: where the rows
// of slabs of 128 channels or more are whole 128-byte lines (64 x 16384 x 1008, the
// scaley loop 1170 us and 1425 non-temporal) and the block is larger than the
// Infinity Cache, from which the next pass reads a smaller one; a block that scaley
// has written it reads in part from there up to about twice its size.  us of three
// blocks in turn, without and with: steps 64 x 16384 x 1024 787 and 707, 24 x 12288 x
// 896 (264 MB) 269 and 251, 49 x 4096 x 768 (154 MB) 182 and 175 but 154 and 176 one
// at a time; loops 1209 and 1127, 206 and 271, 138 and 165.
static bool fl_nontemporal(int nb, int nt, int nc, bool scaley) {
  return nc % 128 == 0 && (long)nb * nt * nc > (scaley ? 500000000L : 250000000L);
}

template <int W, bool NT>
static void fl_stats_launch(const FlStats &a, dim3 grid, dim3 block, hipStream_t s) {
  if (a.spec0 && !a.wdata) {
    hipLaunchKernelGGL((fl_stats_kernel<W, NT, true, false, false>), grid, block, 0, s, a);
  } else if (a.wdata) {
    if (a.mx) hipLaunchKernelGGL((fl_stats_kernel<W, NT, true, true, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fl_stats_kernel<W, NT, true, true, false>), grid, block, 0, s, a);
  } else {
    if (a.mx) hipLaunchKernelGGL((fl_stats_kernel<W, NT, false, false, true>), grid, block, 0, s, a);
    else hipLaunchKernelGGL((fl_stats_kernel<W, NT, false, false, false>), grid, block, 0, s, a);
  }
}

static int fl_stats_any(const FlStats &a, const char *who, void *stream) {
  if (!fl_shape_ok(a.nb, a.nt, a.nc, who)) return -1;
  const int w = fl_slab_width(a.nb, a.nc);
  const int items = a.nb * ((a.nc + w - 1) / w);
  const dim3 grid((items + 7) / 8 * 8), block(64 * FL_SW);
  hipStream_t s = (hipStream_t)stream;
  const bool nt = fl_nontemporal(a.nb, a.nt, a.nc, a.wdata != NULL);
  if (w == 256 && nt) fl_stats_launch<256, true>(a, grid, block, s);
  else if (w == 256) fl_stats_launch<256, false>(a, grid, block, s);
  else if (w == 128 && nt) fl_stats_launch<128, true>(a, grid, block, s);
  else if (w == 128) fl_stats_launch<128, false>(a, grid, block, s);
  else if (w == 64) fl_stats_launch<64, false>(a, grid, block, s);
  else fl_stats_launch<32, false>(a, grid, block, s);
  return bfk_check(hipGetLastError(), "fl_stats_kernel");
}

extern "C" int flk_stats(const uint8_t *d_data, uint8_t *d_scaled, const float *d_spec0, const float *d_var0,
                         const float *d_spec_in, float *d_spec, float *d_var, float *d_max, float *d_pp,
                         int nb, int nt, int nc, void *stream) {
  if (d_scaled && (!d_spec0 || !d_var0)) {
    bfk_set_error("flk_stats: scaling needs spec0 and var0");
    return -1;
  }
  const FlStats a{d_data, d_scaled, d_scaled ? d_spec0 : NULL, d_scaled ? d_var0 : NULL, d_spec_in, d_spec, d_var,
                  d_max,  d_pp,     nb, nt, nc};
  return fl_stats_any(a, "flk_stats", stream);
}

// The statistics that the scaled block will have; the block is only read.
extern "C" int flk_stats_scaled(const uint8_t *d_data, const float *d_spec0, const float *d_var0, float *d_spec,
                                float *d_var, float *d_pp, int nb, int nt, int nc, void *stream) {
  const FlStats a{d_data, NULL, d_spec0, d_var0, NULL, d_spec, d_var, NULL, d_pp, nb, nt, nc};
  return fl_stats_any(a, "flk_stats_scaled", stream);
}

extern "C" size_t flk_masks_big_bytes(int nb, int nc) {
  const int nin = nc - 2 * FL_ZERO;
  return nin > FL_LDSN ? (size_t)3 * nb * nin * sizeof(float) : 0;
}

extern "C" int flk_masks(const float *d_spec, const float *d_var, const float *d_pp, float *d_big, uint8_t *d_mask,
                         int *h_nmask, float *h_spec, double *d_bsum, float *d_bpwr, float thresh, const int *perm,
                         int nperm, int nb, int nc, void *stream) {
  if (nb < 1 || nc < 2 * FL_ZERO + FL_FILT || nperm < 0 || nperm > 64 || (flk_masks_big_bytes(nb, nc) && !d_big)) {
    bfk_set_error("flk_masks: %d beams x %d channels, %d permanent", nb, nc, nperm);
    return -1;
  }
  FlMasks a;
  a.spec = d_spec;
  a.var = d_var;
  a.pp = d_pp;
  a.big = d_big;
  a.mask = d_mask;
  a.h_nmask = h_nmask;
  a.h_spec = h_spec;
  a.bsum = d_bsum;
  a.bpwr = d_bpwr;
  a.thr[0] = thresh;
  a.thr[1] = (float)((double)thresh + 0.5);
  a.thr[2] = (float)(thresh / sqrt(1. * FL_FBIN));
  a.nb = nb;
  a.nc = nc;
  a.nperm = nperm;
  for (int i = 0; i < 64; i++) a.perm[i] = i < nperm ? perm[i] : 0;
  hipLaunchKernelGGL(fl_masks_kernel, dim3(nb, 2), dim3(768), 0, (hipStream_t)stream, a);
  return bfk_check(hipGetLastError(), "fl_masks_kernel");
}

extern "C" size_t flk_part_bytes(int nb, int nt, int nc) {
  const int w = fl_slab_width(nb, nc);
  return (size_t)nb * ((nc + w - 1) / w) * nt * sizeof(uint16_t);
}

extern "C" int flk_apply(uint8_t *d_data, const float *d_spec0, const float *d_var0, const uint8_t *d_mask,
                         const float *d_bpwr, uint16_t *d_part, const double *d_bsum, int *d_ran, int *h_ran, float prev,
                         float jump, int force, int nb, int nt, int nc, void *stream) {
  if (!fl_shape_ok(nb, nt, nc, "flk_apply")) return -1;
  const FlApply a{d_data, d_spec0, d_var0, d_mask, d_bpwr, d_part, d_bsum, d_ran, h_ran, prev, jump, force, nb, nt, nc};
  const int w = fl_slab_width(nb, nc);
  const int items = nb * ((nc + w - 1) / w);
  const dim3 grid((items + 7) / 8 * 8), block(1024);
  hipStream_t s = (hipStream_t)stream;
#define FL_APPLY(W, NT) hipLaunchKernelGGL((fl_apply_kernel<W, NT>), grid, block, 0, s, a)
  const bool nontemporal = fl_nontemporal(nb, nt, nc, false);
  if (w == 256 && nontemporal) FL_APPLY(256, true);
  else if (w == 256) FL_APPLY(256, false);
  else if (w == 128 && nontemporal) FL_APPLY(128, true);
  else if (w == 128) FL_APPLY(128, false);
  else if (w == 64) FL_APPLY(64, false);
  else FL_APPLY(32, false);
#undef FL_APPLY
  return bfk_check(hipGetLastError(), "fl_apply_kernel");
}

// simple_tsflag of the series (from fl_apply's row sums, or d_ts itself with
// d_part NULL) and flagts of the rows it finds.
extern "C" int flk_tsmask_flagts(uint8_t *d_data, const uint16_t *d_part, float *d_ts, int *d_idx, int *d_nts, int *h_nts,
                                 const int *d_ran, const float *d_bpwr, float thr, int nb, int nt, int nc, void *stream) {
  if (!fl_shape_ok(nb, nt, nc, "flk_tsmask_flagts")) return -1;
  const int w = fl_slab_width(nb, nc);
  const FlTsMask a{d_part, d_ts, d_idx, d_nts, h_nts, d_ran, thr, nb, nt, nc, (nc + w - 1) / w};
  hipStream_t s = (hipStream_t)stream;
  hipLaunchKernelGGL(fl_tsmask_kernel, dim3(nb), dim3(1024), 0, s, a);
  hipLaunchKernelGGL(fl_flagts_list_kernel, dim3(nb, 16), dim3(256), 0, s, d_data, d_idx, d_nts, d_bpwr, nt, nc);
  return bfk_check(hipGetLastError(), "fl_tsmask_kernel");
}

extern "C" int flk_flag_ts(uint8_t *d_data, const uint8_t *d_mask, const float *d_bpwr, float *d_ts, int nb,
                           int nt, int nc, void *stream) {
  if (!fl_shape_ok(nb, nt, nc, "flk_flag_ts")) return -1;
  // lanes per row: no more than the row has 16-byte chunks, in powers of two
  const int lpr = nc > 512 ? 64 : nc > 256 ? 32 : 16;
  const long waves = (long)nb * (nt / (FL_RPW * (64 / lpr)));
  const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
  hipStream_t s = (hipStream_t)stream;
#define FL_FLAG_TS(L)                                                                                       \
  do {                                                                                                      \
    if (d_mask) hipLaunchKernelGGL((fl_flag_ts_kernel<L, true>), grid, block, 0, s, d_data, d_mask, d_bpwr, \
                                   d_ts, nb, nt, nc);                                                       \
    else hipLaunchKernelGGL((fl_flag_ts_kernel<L, false>), grid, block, 0, s, d_data, d_mask, d_bpwr, d_ts, \
                            nb, nt, nc);                                                                    \
  } while (0)
  if (lpr == 64) FL_FLAG_TS(64);
  else if (lpr == 32) FL_FLAG_TS(32);
  else FL_FLAG_TS(16);
#undef FL_FLAG_TS
  return bfk_check(hipGetLastError(), "fl_flag_ts_kernel");
}

extern "C" int flk_flagts(uint8_t *d_data, const int *d_midx, int n, const float *d_bpwr, int nb, int nt, int nc,
                          void *stream) {
  if (!fl_shape_ok(nb, nt, nc, "flk_flagts")) return -1;
  if (n <= 0) return 0;
  hipLaunchKernelGGL(fl_flagts_kernel, dim3((n + 3) / 4), dim3(256), 0, (hipStream_t)stream, d_data, d_midx, n,
                     d_bpwr, nb, nt, nc);
  return bfk_check(hipGetLastError(), "fl_flagts_kernel");
}

extern "C" int flk_flag_cols(uint8_t *d_data, const int *d_midx, int n, const float *d_bpwr, int nb, int nt,
                             int nc, void *stream) {
  if (!fl_shape_ok(nb, nt, nc, "flk_flag_cols")) return -1;
  if (n <= 0) return 0;
  if (n > 65535 * 16) {
    bfk_set_error("flk_flag_cols: %d columns", n);
    return -1;
  }
  for (int i0 = 0; i0 < n; i0 += 65535) {
    const int k = n - i0 < 65535 ? n - i0 : 65535;
    hipLaunchKernelGGL(fl_flag_cols_kernel, dim3((nt + 255) / 256, k), dim3(256), 0, (hipStream_t)stream,
                       d_data, d_midx + i0, k, d_bpwr, nb, nt, nc);
  }
  return bfk_check(hipGetLastError(), "fl_flag_cols_kernel");
}

extern "C" int flk_sumpulse(uint8_t *d_data, const float *d_summand, size_t n, void *stream) {
  if (n == 0) return 0;
  const size_t threads = (n + 3) / 4;
  hipLaunchKernelGGL(fl_sumpulse_kernel, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, d_data, d_summand, n);
  return bfk_check(hipGetLastError(), "fl_sumpulse_kernel");
}

extern "C" int flk_genrand(uint8_t *d_rep, size_t n, uint32_t seed, void *stream) {
  if (n == 0) return 0;
  hipLaunchKernelGGL(fl_genrand_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream,
                     d_rep, n, seed);
  return bfk_check(hipGetLastError(), "fl_genrand_kernel");
}

extern "C" int flk_noise(uint8_t *d_data, const uint8_t *d_rep, int nb, int nt, int nc, void *stream) {
  if (!fl_shape_ok(nb, nt, nc, "flk_noise")) return -1;
  const size_t per = (size_t)nt * nc;
  hipLaunchKernelGGL(fl_noise_kernel, dim3((unsigned)((per / 16 + 255) / 256)), dim3(256), 0,
                     (hipStream_t)stream, d_data, d_rep, per, nb);
  return bfk_check(hipGetLastError(), "fl_noise_kernel");
}

extern "C" int flk_fix_zspec(float *d_s0, float *d_v0, int nbc, int naver, void *stream) {
  if (nbc < 1 || naver < 1) {
    bfk_set_error("flk_fix_zspec: %d entries x %d blocks", nbc, naver);
    return -1;
  }
  hipLaunchKernelGGL(fl_fix_zspec_kernel, dim3((nbc + 255) / 256), dim3(256), 0, (hipStream_t)stream, d_s0, d_v0,
                     nbc, naver);
  return bfk_check(hipGetLastError(), "fl_fix_zspec_kernel");
}
