// bf_spread.hip -- the "spread" schedule of the fused beamformer, for blocks
// whose tiles do not fill the chip: one 16-wave workgroup per (8-channel group,
// 64 samples, a few 32-beam tiles), a wave per (channel, pol).
//
// Reference path: src/dsaX_beamformer.cu promoter (:170-193), beamformer
// (:267-416), badder (:78-112) and adder (:120-158), fused into one launch.
//
// Why.  The classic and shared tiles take their 16 (channel, pol) steps one
// after another in each wave.  A block of 8 such tiles (64 antennas x 16
// channels x 128 samples -> 256 beams) keeps 8 of 256 CUs busy for 38 us, and
// every block below about 500 tiles takes that long.  Here the 16 steps of a
// tile run in 16 waves and the 32-beam tiles in different workgroups: the same
// block is 32 workgroups of one step per wave and takes 7 us, bound by latencies
// (staging, weights, one chain, the sums), or 11 with the beam powers, whose own
// launch takes 4.  56 channels x 512 samples x 200
// antennas -> 128 beams, FP8: 106 -> 32 us.  A full chip prefers the other
// schedules, whose waves read a staged or unpacked operand for more beams; the
// rule is in bf_dispatch.hip.
//
// Per workgroup: (a) the voltages are loaded and transposed into LDS rows
// [(channel, pol)][sample][antenna] as in the other schedules; (b) per 32-beam
// tile and 32-sample unit, wave cq runs the MFMA chain of its (channel, pol)
// and sums |B|^2 over its bins, without the weight scale; the sums of the 16
// waves go through LDS, and (c) one wave adds them, scaled, in the order in
// which the tile schedules take the steps.  So each chain, bin sum and the order
// of the powers are those of the other schedules and the results bit-identical.
//
// Rows are 64 bytes per 64 antennas, their 16-byte chunks XOR-swizzled so that
// the 16 lanes of a read phase fall on distinct banks.  More than 128 antennas
// are staged one 32-sample unit at a time (128 KB).
#include "bf_common.h"

namespace {
constexpr int SW = 16, ST = SW * 64;            // waves, threads per workgroup

template <int NKC, int NP> struct Spread {
  static constexpr int NU = NKC == 4 ? 1 : 2;    // units staged together
  static constexpr int RS = 32 * NU;             // staged samples per (channel, pol)
  static constexpr int ROW = 64 * NKC, NCH = ROW / 16;
  static constexpr int SH = NCH == 4 ? 2 : NCH == 8 ? 1 : 0;
  static constexpr int STAGE = 16 * RS * ROW;
  static constexpr int XBUF = 16 * NU * NP * 64;  // floats: [cq][unit][bin][lane]
  static_assert(XBUF >= SW * 64, "the beam power sums reuse it");
  static constexpr int SBUF = 16 * 32;            // floats: [cq][beam] weight scales
  // two exchange buffers where they fit: one barrier per beam tile, else two;
  // the scales beside them where those fit (not 128 or 256 antennas in 8-sample
  // bins, where the adding wave loads them)
  static constexpr int NX = STAGE + 2 * (XBUF + SBUF) * 4 <= 160 * 1024 ? 2 : 1;
  static constexpr bool SX = STAGE + NX * (XBUF + SBUF) * 4 <= 160 * 1024;
  static __device__ __forceinline__ int row(int r, int c) { return r * ROW + ((c ^ ((r >> SH) & (NCH - 1))) << 4); }
};

// One 32-sample unit of one 64-antenna chunk: 32 packed bytes per lane (row n,
// antennas 32h .. 32h + 31) against the wave's weights of 32 beams, in the
// order of the other schedules' chains.  With pf each K step of W is reloaded
// from record wnext right after its last MFMA has issued.
template <int PREC>
__device__ __forceinline__ void spread_unit(f16v &cr, f16v &ci, WFrag<PREC, 1, 1> &W, const uint4 &d0, const uint4 &d1,
                                            const WSrc &src, bool pf, uint32_t wnext) {
  const uint32_t dw[8] = {d0.x, d0.y, d0.z, d0.w, d1.x, d1.y, d1.z, d1.w};
  if constexpr (PREC == 0) {
#pragma unroll
    for (int s = 0; s < 8; s++) {
      h8v are, aim;
      unpack_f16(dw[s], are, aim);
      cr = __builtin_amdgcn_mfma_f32_32x32x16_f16(are, W.w[0][0][s], cr, 0, 0, 0);
      ci = __builtin_amdgcn_mfma_f32_32x32x16_f16(aim, W.w[0][0][s], ci, 0, 0, 0);
      if (pf) W.load_one_rb(src, wnext, 0, s);
    }
  } else {
#pragma unroll
    for (int s2 = 0; s2 < 2; s2++) {
      i8v are, aim;
      if constexpr (PREC == 1) {
#pragma unroll
        for (int u = 0; u < 4; u++) {
          const uint32_t x = dw[4 * s2 + u];
          const uint32_t dr = nib_e4m3(x), di = nib_e4m3(x >> 4);
          are[2 * u] = (int)dr;
          are[2 * u + 1] = (int)(di ^ 0x80808080u);
          aim[2 * u] = (int)di;
          aim[2 * u + 1] = (int)dr;
        }
      } else {
        const uint32_t x[4] = {dw[4 * s2], dw[4 * s2 + 1], dw[4 * s2 + 2], dw[4 * s2 + 3]};
        uint32_t o[6];
        f6_operand(x, o);
        f6_re_im(make_uint4(o[0], o[1], o[2], o[3]), make_uint2(o[4], o[5]), are, aim);
      }
      cr = mfma64<PREC>(are, W.hi[0][0][s2], cr, W.shi(0, 0, s2));
      ci = mfma64<PREC>(aim, W.hi[0][0][s2], ci, W.shi(0, 0, s2));
      if constexpr (PREC == 3) {
        cr = mfma64<PREC>(are, W.mid[0][0][s2], cr, W.smid(0, 0, s2));
        ci = mfma64<PREC>(aim, W.mid[0][0][s2], ci, W.smid(0, 0, s2));
      }
      cr = mfma64<PREC>(are, W.lo[0][0][s2], cr, W.slo(0, 0, s2));
      ci = mfma64<PREC>(aim, W.lo[0][0][s2], ci, W.slo(0, 0, s2));
      if (pf) W.load_one_rb(src, wnext, 0, s2);
    }
  }
}

// The beam power sums of the set's beam tiles bt0 .. bt0 + nbt - 1, as
// bf_beam_power_kernel (bf_aux.hip) adds up to 1792 per-unit sums a beam.  There thread 64 q + l adds sums 64 q + l + 256 k (one
// after another), each wave q its threads' by lane ^ 32, 16, ..., 1, and the four
// waves (0 + 1) + (2 + 3).  Here wave 4 j + q of the workgroup is pass q of beam
// tile j, a lane one beam: half h holds l = 32 h .. 32 h + 31, so the first step
// adds across the halves and the others in registers.  (Which of two values
// comes first does not matter.)  The sums [unit][32 beams] are read in whole lines
// past this XCD's L2, 32 loads in flight; those past the end read as zeros, the
// whole offset being the lane's (a scalar offset past the buffer's size would wrap
// the check).
__device__ __forceinline__ void spread_beam_power(const BfArgs &a, int bt0, int nbt, int wave, int lane, float *lds) {
  constexpr int SC1 = 16;            // agent-scope loads
  const int n = 2 * a.ntblk * a.ngroup, q = wave & 3, h = lane >> 5;
  for (int j0 = 0; j0 < nbt; j0 += 4) {
    const int bt = bt0 + j0 + (wave >> 2);
    float v[32];
#pragma unroll
    for (int l = 0; l < 32; l++) v[l] = 0.f;
    if (j0 + (wave >> 2) < nbt) {
      const __amdgpu_buffer_rsrc_t rs = buffer_rsrc(a.psum + (long)bt * n * 32, (uint32_t)n * 128u);
      for (int k = 0; 64 * q + 256 * k < n; k++)
#pragma unroll
        for (int l = 0; l < 32; l++)
          v[l] += __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(
                                                rs, (uint32_t)(64 * q + 256 * k + 32 * h + l) * 128u + (lane & 31) * 4u,
                                                0, SC1));
    }
#pragma unroll
    for (int l = 0; l < 32; l++) {
      const uint32_t x = __builtin_bit_cast(uint32_t, v[l]);
      const auto s = __builtin_amdgcn_permlane32_swap(x, x, false, false);
      const uint32_t lo = s[0], hi = s[1];       // (bit_cast of s[1] itself takes s[0])
      v[l] = __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
    }
#pragma unroll
    for (int m = 16; m > 0; m >>= 1)
#pragma unroll
      for (int l = 0; l < m; l++) v[l] += v[l + m];
    __syncthreads();
    lds[wave * 64 + lane] = v[0];
    __syncthreads();
    const float *r = lds + (wave & ~3) * 64 + lane;
    const int b = bt * 32 + lane;
    if (q == 0 && lane < 32 && j0 + (wave >> 2) < nbt && b < a.nbeam)
      a.beam_power[b] = (r[0] + r[64]) + (r[128] + r[192]);
  }
}

template <int PREC> __device__ __forceinline__ void spread_load(WFrag<PREC, 1, 1> &W, const WSrc &src, uint32_t w) {
#pragma unroll
  for (int s = 0; s < (PREC == 0 ? 8 : 2); s++) W.load_one_rb(src, w, 0, s);
}

}  // namespace

// Workgroups are ordered beam sets fastest, so that those that read the same
// voltages run together on one XCD, then gw groups, time blocks and the rest of
// the groups.  nbw: beam tiles per workgroup; pol_outer: the powers summed over the channels
// of pol 0 and then of pol 1, else pol fastest.
template <int PREC, int TAVG, int NKC>
__global__ __launch_bounds__(ST) void bf_spread_kernel(BfArgs a, int nbw, int pol_outer, int gw) {
  constexpr int NP = TAVG <= 32 ? 32 / TAVG : 1, VPB = 16 / NP;
  using S = Spread<NKC, NP>;
  __shared__ __attribute__((aligned(16))) uint8_t stage[S::STAGE];
  __shared__ float xch[S::NX][S::XBUF + (S::SX ? S::SBUF : 0)];
  const int live_bt = (a.nbeam + 31) / 32, nset = (live_bt + nbw - 1) / nbw;
  const int L = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (L >= nset * a.ngroup * a.ntblk) return;
  TileId t;
  const int bt0 = L % nset * nbw, nbt = min(nbw, live_bt - bt0);
  const int gt = L / nset, slab = gt / (gw * a.ntblk), in_slab = gt % (gw * a.ntblk);
  const int w = min(gw, a.ngroup - slab * gw);           // groups of this slab
  t.g = slab * gw + in_slab % w;
  t.tblk = in_slab / w;
  t.bset = 0;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int cq = __builtin_amdgcn_readfirstlane(tid >> 6);

  WSrc src;
  src.rw = buffer_rsrc(a.wfrag, a.wfrag_bytes);
  src.rs = buffer_rsrc(a.wscale, a.wscale_bytes);
  src.vl = (uint32_t)lane * (PREC == 0 ? 16u : 32u);
  src.vn4 = (uint32_t)n * 4u;
  const uint32_t wrow = (uint32_t)weight_row(a, t.g, cq);
  // weight record of beam tile i (of this workgroup), antenna chunk kc
  auto wrec = [&](int i, int kc) { return (wrow * a.nbt + bt0 + i) * NKC + kc; };

  // (a) the unit-independent part of a staging task: 4 antennas x 4 channels of
  // one packet (16 bytes of each antenna's 32-byte chunk)
  const __amdgpu_buffer_rsrc_t rin = buffer_rsrc(a.in, a.in_bytes);
  constexpr int NTASK = 16 * S::NU * 16 * NKC * 2, TPT = NTASK / ST;   // packets x antenna quads x halves
  static_assert(NTASK % ST == 0, "whole staging tasks per thread");
  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  auto stage_units = [&](int u0) {
    u4 x[TPT][4];
#pragma unroll
    for (int k = 0; k < TPT; k++) {
      const int task = tid + k * ST, hf = task & 1, aq = (task >> 1) % (16 * NKC), pl = (task >> 1) / (16 * NKC);
      const long p = (long)t.tblk * PCU + u0 * 16 + pl;
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const int ant = aq * 4 + j;
        // padding antennas read past the block's end: the buffer returns zeros
        const uint32_t off = ant < a.nant ? (uint32_t)chunk_offset(a.order, p, ant, t.g, a.nant, a.nchan, a.ngroup) + hf * 16
                                          : 0x80000000u;
        x[k][j] = __builtin_amdgcn_raw_buffer_load_b128(rin, off, 0, 0);
      }
    }
    return [=](uint8_t *dst) {
#pragma unroll
      for (int k = 0; k < TPT; k++) {
        const int task = tid + k * ST, hf = task & 1, aq = (task >> 1) % (16 * NKC), pl = (task >> 1) / (16 * NKC);
        const int c = aq >> 2, w = (aq & 3) * 4;
#pragma unroll
        for (int ci = 0; ci < 4; ci++) {
          const uint32_t l01 = __builtin_amdgcn_perm(x[k][1][ci], x[k][0][ci], 0x05010400u);
          const uint32_t h01 = __builtin_amdgcn_perm(x[k][1][ci], x[k][0][ci], 0x07030602u);
          const uint32_t l23 = __builtin_amdgcn_perm(x[k][3][ci], x[k][2][ci], 0x05010400u);
          const uint32_t h23 = __builtin_amdgcn_perm(x[k][3][ci], x[k][2][ci], 0x07030602u);
          const int r0 = ((hf * 4 + ci) * 2) * S::RS + 2 * pl, r1 = r0 + S::RS;
          *(uint32_t *)(dst + S::row(r0, c) + w) = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
          *(uint32_t *)(dst + S::row(r1, c) + w) = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
          *(uint32_t *)(dst + S::row(r0 + 1, c) + w) = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
          *(uint32_t *)(dst + S::row(r1 + 1, c) + w) = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
        }
      }
    };
  };

  WFrag<PREC, 1, 1> W;
  float part[2][1][NP];                          // in the adding waves
  // (a copy of the lane number that the compiler cannot see through: addresses
  // made from it stay in the adding branch instead of in registers across the
  // chains.  Up to 64 antennas nothing then spills, up to 128 one to three
  // registers in five of the kernels.  Above, where 64 registers of weights are
  // prefetched beside 32 accumulators and 16 waves leave 128 in all, 8 to 44
  // do, 36 to 164 bytes a lane, most with 8-sample bins)
  auto hide = [](int v) {
    asm volatile("" : "+v"(v));
    return v;
  };
  // (c) one wave adds the sums of unit u of beam tile i into part[p]
  auto add = [&](int i, int u, int p, const float *x, int ln) {
    const int n = ln & 31;
#pragma unroll
    for (int j = 0; j < NP; j++) part[p][0][j] = 0.f;
    float sc[16];
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const int c = pol_outer ? 2 * (k & 7) + (k >> 3) : k;
      if constexpr (S::SX) {
        sc[k] = x[S::XBUF + c * 32 + n];
      } else {
        const uint32_t so = ((uint32_t)weight_row(a, t.g, c) * a.nbeam_pad + (bt0 + i) * 32) * 4u;
        sc[k] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src.rs, src.vn4, so, 0));
      }
    }
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const int c = pol_outer ? 2 * (k & 7) + (k >> 3) : k;
#pragma unroll
      for (int j = 0; j < NP; j++)
        part[p][0][j] =
            __builtin_fmaf(x[((c * S::NU + (S::NU == 2 ? u : 0)) * NP + j) * 64 + ln], sc[k], part[p][0][j]);
    }
  };
  auto chain = [&](int i, int u) {
    float *x = xch[S::NX == 2 ? i & 1 : 0];
    if constexpr (S::SX) {
      if (u == 0 || S::NU == 1) {
        const uint32_t so = (wrow * a.nbeam_pad + (bt0 + i) * 32) * 4u;
        const float sc = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(src.rs, src.vn4, so, 0));
        if (h == 0) x[S::XBUF + cq * 32 + n] = sc;
      }
    }
    f16v cr = (f16v){}, ci = (f16v){};
#pragma unroll
    for (int kc = 0; kc < NKC; kc++) {
      const int r = cq * S::RS + (S::NU == 2 ? u * 32 : 0) + n;
      const uint4 d0 = *(const uint4 *)(stage + S::row(r, kc * 4 + h * 2));
      const uint4 d1 = *(const uint4 *)(stage + S::row(r, kc * 4 + h * 2 + 1));
      // the next chunk's weights, or the next unit's or beam tile's first (the
      // last step reloads its own); one chunk serves both units
      const bool last = kc == NKC - 1;
      const bool pf = NKC > 1 || u == 1;
      const int ni = !last || (NKC > 1 && u == 0 && S::NU == 2) ? i : min(i + 1, nbt - 1);
      spread_unit<PREC>(cr, ci, W, d0, d1, src, pf, wrec(ni, last ? 0 : kc + 1));
      __builtin_amdgcn_sched_barrier(0);       // (the next chunk's operands would spill, more than does)
    }
#pragma unroll
    for (int j = 0; j < NP; j++) {
      float s0 = 0.f, s1 = 0.f, s2 = 0.f, s3 = 0.f;
#pragma unroll
      for (int v = j * VPB; v < (j + 1) * VPB; v += 2) {
        s0 = __builtin_fmaf(cr[v], cr[v], s0);
        s1 = __builtin_fmaf(ci[v], ci[v], s1);
        s2 = __builtin_fmaf(cr[v + 1], cr[v + 1], s2);
        s3 = __builtin_fmaf(ci[v + 1], ci[v + 1], s3);
      }
      x[((cq * S::NU + (S::NU == 2 ? u : 0)) * NP + j) * 64 + lane] = (s0 + s1) + (s2 + s3);
    }
  };

  if constexpr (S::NU == 2) {
    {
      auto store = stage_units(0);
      if (NKC == 1) spread_load<PREC>(W, src, wrec(0, 0));
      store(stage);
      if (NKC > 1) spread_load<PREC>(W, src, wrec(0, 0));
    }
    __syncthreads();
    for (int i = 0; i < nbt; i++) {
#pragma unroll
      for (int u = 0; u < 2; u++) chain(i, u);
      __syncthreads();
      const float *x = xch[S::NX == 2 ? i & 1 : 0];
      if (TAVG == 64) {                                  // one bin, of both units
        if (cq == (i & 15)) {
          const int ln = hide(lane);
          add(i, 0, 0, x, ln);
          add(i, 1, 1, x, ln);
          tile_output<TAVG, 1, true>(a, t, bt0 + i, ln & 31, ln >> 5, part, 0, 2);
        }
      } else if (cq >> 1 == (i & 7)) {
        const int ln = hide(lane);
        add(i, cq & 1, 0, x, ln);
        tile_output<TAVG, 1, true>(a, t, bt0 + i, ln & 31, ln >> 5, part, cq & 1, 1);
      }
      if (S::NX == 1 && i + 1 < nbt) __syncthreads();   // before the buffer is written again
    }
  } else {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      {
        auto store = stage_units(u);
        spread_load<PREC>(W, src, wrec(0, 0));
        if (u) __syncthreads();                         // the first unit's rows are read
        store(stage);
      }
      __syncthreads();
      for (int i = 0; i < nbt; i++) {
        chain(i, u);
        __syncthreads();
        if (cq == i) {
          const int ln = hide(lane);
          add(i, u, u, xch[S::NX == 2 ? i & 1 : 0], ln);
          if (u) tile_output<TAVG, 1, true>(a, t, bt0 + i, ln & 31, ln >> 5, part, 0, 2);
        }
        if (S::NX == 1) __syncthreads();                // before the buffer is written again
      }
      if (S::NX == 2) __syncthreads();
    }
  }
  // (d) the last workgroup of the beam set to finish sums its beams' powers.  The
  // partial sums are agent-scope stores and loads, past the XCDs' L2s; every
  // wave waits for its own stores before the barrier, so they are all performed
  // when the workgroup is counted.  (Fences instead write back and invalidate the
  // XCD's L2 once a workgroup: 56 channels x 512 samples -> 128 beams 24 us
  // alone and 18 among others, against 16 and 6.3.)
  if (!a.beam_power) return;
  unsigned *last = (unsigned *)xch[0];           // (free once every wave is past its sums)
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid == 0) {
    const unsigned total = (unsigned)(a.ngroup * a.ntblk);
    *last = atomicInc(a.count + L % nset, total - 1) == total - 1;
  }
  __syncthreads();
  if (!*last) return;
  __syncthreads();                               // (`last` is read)
  spread_beam_power(a, bt0, nbt, cq, lane, xch[0]);
}

template <int PREC, int NKC>
static void spread_launch(int tavg, dim3 grid, hipStream_t s, const BfArgs &a, int nbw, int pol_outer, int gw) {
  switch (tavg) {
    case 8:  hipLaunchKernelGGL((bf_spread_kernel<PREC, 8, NKC>), grid, dim3(ST), 0, s, a, nbw, pol_outer, gw); break;
    case 16: hipLaunchKernelGGL((bf_spread_kernel<PREC, 16, NKC>), grid, dim3(ST), 0, s, a, nbw, pol_outer, gw); break;
    case 32: hipLaunchKernelGGL((bf_spread_kernel<PREC, 32, NKC>), grid, dim3(ST), 0, s, a, nbw, pol_outer, gw); break;
    default: hipLaunchKernelGGL((bf_spread_kernel<PREC, 64, NKC>), grid, dim3(ST), 0, s, a, nbw, pol_outer, gw); break;
  }
}

// Where the launch sums the beam powers: up to one chain (64 antennas) per CU.
// There a second launch is what bounds a run of blocks (us among others, two
// launches and one; 64 antennas unless said: 8 channels x 64 samples -> 32 beams
// 6.5 and 4.0, 8 x 4096 -> 64 8.3 and 5.0, 24 x 3520 -> 30 8.2 and 6.6, 56 x 512 ->
// 128 6.8 and 6.3, 16 x 512 -> 300 8.1 and 6.2, 100 antennas 24 x 256 -> 64 8.1 and
// 5.1), against up to 1.1 us more for a block alone (11.1 and 12.2 at the 300
// beams).  Beyond it the last workgroup's sums cost what the launch did (56 x 512
// -> 256 12.7 and 12.9, FP6x3 14.4 and 14.9; 100 antennas 88 x 448 -> 125 15.9 and
// 16.5).
extern "C" size_t bfk_psum_bytes(const bfk_dims *d) {
  const long live_bt = (d->nbeam + 31) / 32, chains = live_bt * d->ngroup * (d->nsamp / TCU) * d->nkc;
  return chains <= 256 && live_bt <= BFK_COUNTS ? (BFK_COUNTS + live_bt * 32 * (d->nsamp / 32) * d->ngroup) * sizeof(float) : 0;
}

extern "C" int bfk_beamform_spread(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag, const float *d_wscale,
                                   const float *d_scale, uint8_t *d_out, float *d_power, float *d_bpart,
                                   float *d_beam_power, void *d_psum, int nbw, int pol_outer, void *stream) {
  if (d_beam_power && (!d_psum || !bfk_psum_bytes(d))) {
    bfk_set_error("bfk_beamform_spread: no sums of %d beams x %d units here", d->nbeam, d->nsamp / 32 * d->ngroup);
    return -1;
  }
  if (d->nant_pad != 64 * d->nkc || (d->nkc != 1 && d->nkc != 2 && d->nkc != 4) || d->nsamp % TCU || nbw < 1 || nbw > SW ||
      (d->prec == 3 && d->nkc > 2)) {
    bfk_set_error("bfk_beamform_spread: nant_pad=%d nsamp=%d nbw=%d", d->nant_pad, d->nsamp, nbw);
    return -1;
  }
  BfArgs a = bf_make_args(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, 32);
  a.beam_power = d_beam_power;
  a.count = (unsigned *)d_psum;
  a.psum = (float *)d_psum + BFK_COUNTS;
  const int nset = ((d->nbeam + 31) / 32 + nbw - 1) / nbw;
  const dim3 grid((unsigned)((nset * d->ngroup * a.ntblk + 7) / 8 * 8));
  hipStream_t s = (hipStream_t)stream;
  // Groups side by side: four read whole 128-byte input lines together, but the
  // 32 workgroups of an XCD should leave four time blocks or more to each
  // fine-weight row (of a 56-channel x 512-sample block: 200 antennas -> 256 beams
  // in 4 sets, 1, 2 and 4 groups 52, 54 and 70 us; 128 beams in one set 70, 70
  // and 71; 256 channels x 2048 samples, 64 antennas -> 128 beams in one set 109,
  // 92 and 87 us).
  int gw = 4;
  while (gw > 1 && d->wmode != 0 && nset * gw > 8) gw >>= 1;
#define SPREAD(P)                                                             \
  do {                                                                        \
    if (d->nkc == 1) spread_launch<P, 1>(d->tavg, grid, s, a, nbw, pol_outer, gw); \
    else spread_launch<P, 2>(d->tavg, grid, s, a, nbw, pol_outer, gw);            \
  } while (0)
#define SPREAD4(P)                                                            \
  do {                                                                        \
    if (d->nkc == 4) spread_launch<P, 4>(d->tavg, grid, s, a, nbw, pol_outer, gw); \
    else SPREAD(P);                                                           \
  } while (0)
  if (d->prec == 0) SPREAD4(0);
  else if (d->prec == 1) SPREAD4(1);
  else if (d->prec == 2) SPREAD4(2);
  else SPREAD(3);
#undef SPREAD4
#undef SPREAD
  return bfk_check(hipGetLastError(), "bf_spread_kernel");
}
