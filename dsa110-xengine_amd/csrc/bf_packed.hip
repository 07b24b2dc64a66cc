// bf_packed.hip -- large blocks of 65 to 256 antennas: the voltages are first
// repacked, antennas innermost, and the beamforming workgroups of eight waves (one
// 32-beam tile each) then take 128 samples of a group at a time.
//
// Reference path: src/dsaX_beamformer.cu promoter (:170-193), beamformer
// (:267-416), badder (:78-112) and adder (:120-158).
//
// Why.  A wave's weights of one (channel, pol) are 16 (128 antennas) or 32 KB, read
// anew by every workgroup; straight from the input a workgroup of 64 samples reads
// its voltages 8 or 16 bytes at a time out of 128-byte lines, as many bytes
// through the L1 as the weights.  Together they filled it (256 antennas -> 1024
// beams in FP8: L2 to L1 16.5 TB/s, matrix cores 47 % busy).  Repacked, a (channel,
// pol) of 128 samples is one contiguous 16 or 32 KB, which costs one more pass
// over the block, and one channel in LDS at a time leaves room for 128 samples,
// which halves the weights' bytes too.  256 antennas x 384 channels x 4096 samples ->
// 1024 beams in FP8, fine weights: 6.13 -> 4.62 ms alone, 7.24 -> 4.77 among other
// blocks (0.32 of it the repacking); 100 x 200 x 2112 -> 300 in three-part FP6: 0.65
// -> 0.34 and 0.52 -> 0.31, of which the short last set is a third.
//
// The operands, chains and detection are those of bf_shared8.hip, in its order,
// so the results are bit for bit its.
#include "bf_shared8_tile.h"

namespace {
constexpr int TP = 2 * TCU;                // samples of a tile
template <int V> struct IntC { static constexpr int value = V; };

template <int PREC, int NKC> struct P8 {
  static constexpr int ROW = S8<NKC>::ROW;
  static constexpr int CQB = TP * ROW;                        // packed bytes of a (channel, pol) of one tile
  static constexpr int NLD = CQB / 16 / NT8;                  // 16-byte loads of it per thread
  static constexpr int GU = PREC == 0 ? 1 : 2, NG = 4 / GU;   // units per A_re buffer, buffers per (channel, pol)
  static constexpr int ABUF = PREC == 0 ? S8<NKC>::UNIT16 : 2 * S8<NKC>::UNIT8;
};
}  // namespace

// Packed voltages [group][128 samples][channel, pol][sample][antenna], one byte
// each, 64 NKC antennas (those past nant zero), samples past the last one zero;
// the 16-byte chunks of a row XORed with the row as in srow8.  A thread takes the
// 16-byte half of the 32-byte chunks of 16 antennas of one packet; its stores
// write 128 bytes of a row with those of the other 16-antenna chunks.  A workgroup
// takes eight packets of four groups: whole 128-byte lines with antennas outermost.  805 + 805 MB in 315 us, 5.1 TB/s,
// which is a large copy's rate (a group a workgroup: 400 us).
template <int NKC>
__global__ __launch_bounds__(256) void bf_pack_kernel(BfArgs a, int nb2, uint8_t *__restrict__ packed) {
  using S = S8<NKC>;
  constexpr int PPW = 256 / (8 * S::NCH);                     // packets of a workgroup at a time
  const int L = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int piece = L & 3, tb = (L >> 2) % (nb2 * 2);         // 8 packets of a 64-sample block
  const int tid = threadIdx.x, half = tid & 1, g = (L >> 2) / (nb2 * 2) * 4 + ((tid >> 1) & 3);
  const int c = (tid >> 3) % S::NCH, p0 = piece * 8 + tid / (8 * S::NCH);
  if (g >= a.ngroup) return;
  uint8_t *dst = packed + ((long)(g * nb2 + (tb >> 1)) * 16 * TP + (tb & 1) * TCU) * S::ROW;
#pragma unroll 1
  for (int pl = p0; pl < piece * 8 + 8; pl += PPW) {
    uint4 v[16];
#pragma unroll
    for (int i = 0; i < 16; i++) {
      v[i] = make_uint4(0, 0, 0, 0);
      if (tb < a.ntblk && c * 16 + i < a.nant)
        v[i] = *(const uint4 *)(a.in + chunk_offset(a.order, (long)tb * PCU + pl, c * 16 + i, g, a.nant, a.nchan, a.ngroup) +
                                half * 16);
    }
#pragma unroll
    for (int ch = 0; ch < 4; ch++) {
      uint32_t o[4][4];                                       // [time * 2 + pol][antenna quad]
#pragma unroll
      for (int k = 0; k < 4; k++) {
        uint32_t x[4];
#pragma unroll
        for (int j = 0; j < 4; j++) {
          const uint4 &u = v[4 * k + j];
          x[j] = ch == 0 ? u.x : ch == 1 ? u.y : ch == 2 ? u.z : u.w;
        }
        const uint32_t l01 = __builtin_amdgcn_perm(x[1], x[0], 0x05010400u), h01 = __builtin_amdgcn_perm(x[1], x[0], 0x07030602u);
        const uint32_t l23 = __builtin_amdgcn_perm(x[3], x[2], 0x05010400u), h23 = __builtin_amdgcn_perm(x[3], x[2], 0x07030602u);
        o[0][k] = __builtin_amdgcn_perm(l23, l01, 0x05040100u);
        o[1][k] = __builtin_amdgcn_perm(l23, l01, 0x07060302u);
        o[2][k] = __builtin_amdgcn_perm(h23, h01, 0x05040100u);
        o[3][k] = __builtin_amdgcn_perm(h23, h01, 0x07060302u);
      }
#pragma unroll
      for (int tp = 0; tp < 4; tp++) {
        const int cq = (half * 4 + ch) * 2 + (tp & 1), r = 2 * pl + (tp >> 1);
        *(uint4 *)(dst + (long)cq * TP * S::ROW + srow8<NKC>(r, c)) = make_uint4(o[tp][0], o[tp][1], o[tp][2], o[tp][3]);
      }
    }
  }
}

// A workgroup's beam set: 8 / SPLIT tiles of 32 beams from bt0, each taken by SPLIT
// waves, which share the tile's four 32-sample units.
struct PSet {
  int bt0, split;
};
// Set i of `live` beam tiles: eights, then what remains: up to 2 tiles on four waves
// each, 3 and 4 on two, more as an eight (140 beams, five tiles, as one such set, or as
// four and one: 256 antennas x 384 channels x 2048 samples in FP8 276 and 333 us among
// other blocks, in FP16 321 and 431).
__host__ __device__ inline PSet packed_set(int live, int i) {
  const int full = live / 8, rem = live % 8;
  return {i * 8, i < full || rem > 4 ? 1 : rem <= 2 ? 4 : 2};
}
__host__ __device__ inline int packed_sets(int live) { return (live + 7) / 8; }

template <int PREC, int TAVG, int NKC, int SPLIT>
__device__ __forceinline__ void packed_tile(const BfArgs &a, TileId t, int tb2, int nb2, int bt0, const uint8_t *packed,
                                            uint8_t (&stage)[2][P8<PREC, NKC>::CQB],
                                            uint8_t (&abuf)[2][P8<PREC, NKC>::ABUF]) {
  using P = P8<PREC, NKC>;
  constexpr int NP = TAVG <= 32 ? 32 / TAVG : 1, NL = 4 / SPLIT, NBT = NW8 / SPLIT;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int tile = wave % NBT, share = wave / NBT;   // this wave's beam tile, and which of its SPLIT waves it is
  const int btw = bt0 + tile;
  const bool live = btw * 32 < a.nbeam;              // (a wave without beams only stages and unpacks)

  typedef uint32_t u4 __attribute__((ext_vector_type(4)));
  const u4 *src = (const u4 *)(packed + (long)(t.g * nb2 + tb2) * 16 * P::CQB) + tid;
  u4 r0, r1, r2, r3;                                 // a (channel, pol)'s voltages in flight (two with 128 antennas)
  auto load = [&](int cq) __attribute__((always_inline)) {
    const u4 *p = src + (long)cq * (P::CQB / 16);
    r0 = p[0];
    r1 = p[NT8];
    if constexpr (P::NLD == 4) {
      r2 = p[2 * NT8];
      r3 = p[3 * NT8];
    }
  };
  auto store = [&](int cq) __attribute__((always_inline)) {
    u4 *p = (u4 *)stage[cq & 1] + tid;
    p[0] = r0;
    p[NT8] = r1;
    if constexpr (P::NLD == 4) {
      p[2 * NT8] = r2;
      p[3 * NT8] = r3;
    }
  };
  // A_re of buffer gr of the (channel, pol) staged in st
  auto unpack = [&](const uint8_t *st, int gr, uint8_t *ab) __attribute__((always_inline)) {
    if constexpr (PREC == 0) unpack8_f16<NKC>(st, ab, gr, tid);
    else if constexpr (PREC == 1) unpack8_f8<NKC>(st, ab, gr, tid);
    else unpack8_f6<NKC>(st, ab, gr, tid);
  };

  load(0);
  WFrag<PREC, 1, NKC> W;
  if (live) {
    const long wr = weight_row(a, t.g, 0);
    W.load(a.wfrag, a.wscale, wr * a.nbt + btw, wr * a.nbeam_pad + btw * 32, lane, lane & 31);
  }
  store(0);
  load(1);
  float part[NL][1][NP];                             // of this wave's units
#pragma unroll
  for (int i = 0; i < NL; i++)
#pragma unroll
    for (int j = 0; j < NP; j++) part[i][0][j] = 0.f;
  __syncthreads();
  unpack(stage[0], 0, abuf[0]);
  store(1);
  __syncthreads();

#pragma unroll 1
  for (int cq = 0; cq < 16; cq++) {
    const long wn = weight_row(a, t.g, cq < 15 ? cq + 1 : cq);
    // unit k of the buffer ab, the wave's l-th of this (channel, pol)
    auto unit = [&](const uint8_t *ab, int k, auto l) __attribute__((always_inline)) {
      constexpr int LU = decltype(l)::value;
      Acc<1> A;
      unit8w<PREC, NKC, LU == NL - 1>(A, W, ab + k * (PREC == 0 ? 0 : S8<NKC>::UNIT8), lane, a.wfrag,
                                      LU == NL - 1 ? wn * a.nbt + btw : 0);
      detect<TAVG>(A, W.sc, part[LU]);
      if (LU == NL - 1) W.load_scale(a.wscale, wn * a.nbeam_pad + btw * 32, lane & 31);
    };
    auto buffer = [&](auto g) __attribute__((always_inline)) {
      constexpr int gr = decltype(g)::value;
      // stage[cq & 1] is free from the last buffer on, stage[(cq + 1) & 1] until
      // then: (channel, pol) cq + 2 is loaded here and stored a buffer later
      if (gr == P::NG - 1 && cq + 2 < 16) load(cq + 2);
      if (gr == 0 && cq > 0 && cq < 15) store(cq + 1);
      if (gr < P::NG - 1) unpack(stage[cq & 1], gr + 1, abuf[(gr + 1) & 1]);
      else if (cq < 15) unpack(stage[(cq + 1) & 1], 0, abuf[0]);
      const uint8_t *ab = abuf[gr & 1];
      if (live) {
        if constexpr (P::GU == 2) {
          if constexpr (SPLIT == 1) {
            unit(ab, 0, IntC<2 * gr>());
            unit(ab, 1, IntC<2 * gr + 1>());
          } else if constexpr (SPLIT == 2) {
            unit(ab, share, IntC<gr>());
          } else {
            if (share >> 1 == gr) unit(ab, share & 1, IntC<0>());
          }
        } else {
          if (share == gr % SPLIT) unit(ab, 0, IntC<gr / SPLIT>());
        }
      }
      __syncthreads();
    };
    buffer(IntC<0>());
    buffer(IntC<1>());
    if constexpr (P::NG == 4) {
      buffer(IntC<2>());
      buffer(IntC<3>());
    }
  }

  float all[2][2][1][NP];                            // [64-sample block][unit]
  if constexpr (SPLIT > 1) {
    // wave tile + NBT * share holds units share, share + SPLIT of beam tile `tile`
    float *x = (float *)abuf;
    static_assert(NW8 * NL * NP * 256 <= sizeof(abuf), "the sums of every wave");
#pragma unroll
    for (int i = 0; i < NL; i++)
#pragma unroll
      for (int j = 0; j < NP; j++) x[((wave * NL + i) * NP + j) * 64 + lane] = part[i][0][j];
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < NP; j++)
        all[u >> 1][u & 1][0][j] = x[(((tile + NBT * (u % SPLIT)) * NL + u / SPLIT) * NP + j) * 64 + lane];
  } else {
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
      for (int j = 0; j < NP; j++) all[u >> 1][u & 1][0][j] = part[u % NL][0][j];
  }
  if (!live || share > 0) return;
#pragma unroll
  for (int i = 0; i < 2; i++) {
    t.tblk = tb2 * 2 + i;
    if (t.tblk < a.ntblk) tile_output<TAVG>(a, t, btw, lane & 31, lane >> 5, all[i], 0, 2);
  }
}

template <int PREC, int TAVG, int NKC>
__global__ __launch_bounds__(NT8) __attribute__((amdgpu_waves_per_eu(2, 2)))
void bf_packed_kernel(BfArgs a, int nb2, const uint8_t *__restrict__ packed) {
  using P = P8<PREC, NKC>;
  __shared__ __attribute__((aligned(16))) uint8_t stage[2][P::CQB];
  __shared__ __attribute__((aligned(16))) uint8_t abuf[2][P::ABUF];
  // One beam set after another, the short, split ones last; within a set tiles of one
  // group are consecutive on an XCD, so that they read the same weights at about the
  // same time.
  const int n8 = (nb2 * a.ngroup + 7) / 8, wg = blockIdx.x % (8 * n8);
  const int L = (wg & 7) * n8 + (wg >> 3);
  if (L >= nb2 * a.ngroup) return;
  const int tb2 = L % nb2;
  const PSet set = packed_set((a.nbeam + 31) / 32, blockIdx.x / (8 * n8));
  TileId t;
  t.g = L / nb2;
  t.bset = 0;
  if (set.split == 1) packed_tile<PREC, TAVG, NKC, 1>(a, t, tb2, nb2, set.bt0, packed, stage, abuf);
  else if (set.split == 2) packed_tile<PREC, TAVG, NKC, 2>(a, t, tb2, nb2, set.bt0, packed, stage, abuf);
  else packed_tile<PREC, TAVG, NKC, 4>(a, t, tb2, nb2, set.bt0, packed, stage, abuf);
}

// ---- host side --------------------------------------------------------------

extern "C" int bfk_packed_sets(int live) { return packed_sets(live); }
extern "C" int bfk_packed_split(int live, int set) { return packed_set(live, set).split; }

extern "C" size_t bfk_packed_bytes(const bfk_dims *d) {
  if ((d->nkc != 2 && d->nkc != 4) || (d->prec == 3 && d->nkc != 2)) return 0;
  return (size_t)((d->nsamp + TP - 1) / TP) * d->ngroup * 16 * TP * d->nant_pad;
}

template <int PREC, int NKC>
static void packed_launch(int tavg, dim3 grid, hipStream_t s, const BfArgs &a, int nb2, const uint8_t *packed) {
  switch (tavg) {
    case 8:  hipLaunchKernelGGL((bf_packed_kernel<PREC, 8, NKC>), grid, dim3(NT8), 0, s, a, nb2, packed); break;
    case 16: hipLaunchKernelGGL((bf_packed_kernel<PREC, 16, NKC>), grid, dim3(NT8), 0, s, a, nb2, packed); break;
    case 32: hipLaunchKernelGGL((bf_packed_kernel<PREC, 32, NKC>), grid, dim3(NT8), 0, s, a, nb2, packed); break;
    default: hipLaunchKernelGGL((bf_packed_kernel<PREC, 64, NKC>), grid, dim3(NT8), 0, s, a, nb2, packed); break;
  }
}

extern "C" int bfk_beamform_packed(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag, const float *d_wscale,
                                   const float *d_scale, uint8_t *d_out, float *d_power, float *d_bpart, void *d_packed,
                                   void *stream) {
  if (!bfk_packed_bytes(d) || !d_packed || d->nant_pad != 64 * d->nkc || d->nsamp % TCU || d->nbeam_pad % BSET8) {
    bfk_set_error("bfk_beamform_packed: nant_pad=%d nsamp=%d buffer %p", d->nant_pad, d->nsamp, d_packed);
    return -1;
  }
  const BfArgs a = bf_make_args(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, BSET8);
  const int nb2 = (d->nsamp + TP - 1) / TP;
  const dim3 pgrid((d->ngroup + 3) / 4 * nb2 * 8), grid((nb2 * d->ngroup + 7) / 8 * 8 * packed_sets((d->nbeam + 31) / 32));
  hipStream_t s = (hipStream_t)stream;
  uint8_t *packed = (uint8_t *)d_packed;
  if (d->nkc == 2) hipLaunchKernelGGL(bf_pack_kernel<2>, pgrid, dim3(256), 0, s, a, nb2, packed);
  else hipLaunchKernelGGL(bf_pack_kernel<4>, pgrid, dim3(256), 0, s, a, nb2, packed);
  if (int rc = bfk_check(hipGetLastError(), "bf_pack_kernel")) return rc;
#define PACKED(P, K) packed_launch<P, K>(d->tavg, grid, s, a, nb2, packed)
  if (d->nkc == 2) {
    if (d->prec == 0) PACKED(0, 2);
    else if (d->prec == 1) PACKED(1, 2);
    else if (d->prec == 2) PACKED(2, 2);
    else PACKED(3, 2);
  } else {
    if (d->prec == 0) PACKED(0, 4);
    else if (d->prec == 1) PACKED(1, 4);
    else PACKED(2, 4);
  }
#undef PACKED
  return bfk_check(hipGetLastError(), "bf_packed_kernel");
}
