// xc_corr.hip -- the correlator X-engine on the beamformer's 4-bit input:
// for every channel and pol, the visibility of each antenna pair (i, j <= i)
// summed over the block, on int8 matrix cores.
//
// Reference: src/dsaX_bfCorr.cu dcorrelator (:472-569): the block
// [packet][antenna][channel][2 times][2 pols] is transposed and unpacked to
// FP16 planes in HBM (:316-356), four strided batched FP16 GEMMs per
// (channel, time, pol) form C = r r^T + i i^T and C' = r i^T - i r^T with FP16
// accumulation (:512-556), and two more kernels transpose and gather the
// upper triangle into [baseline][channel][pol][re, im] (:366-457).
//
// Here:
//   - Up to 64 antennas, where that pays (bfk_xcorr_use_fused), one kernel reads the
//     block itself (xc_fused_kernel below); else:
//   - xc_turn_kernel turns the packed block, still one byte (4-bit re, 4-bit
//     im) per sample, into (channel, pol) planes [channel*2 + pol][antenna]
//     [sample]: each lane reads one channel's 4-byte words of 64 packets
//     (32 lanes cover a 128-byte run of 32 channels) and writes its 128-byte
//     row segment.
//   - xc_kernel: one wave per ((channel, pol), share of the triangle, time
//     slice); waves are independent (no LDS, no barriers).  Per 64 samples a
//     lane loads 32 contiguous bytes of each antenna block its tiles read.
//   - Operands are int8: a 4-bit sample v is taken as u = v + 8 = nibble ^ 8
//     in 0..15 (masks, no conversion), so the matrix op sums products of
//     small non-negative integers in int32, exactly.  Lane (n, h) of an
//     operand holds antenna 32J + n and 8 samples as 16 K slots X = [ur | ui];
//     W = [ui | -ur] (-u is representable).  Re' = X_j . X_i and
//     Im' = X_j . W_i; with the per-antenna sums S = sum (ur + ui) and
//     E = sum (ur - ui) over the N samples, the visibilities of v = u - 8 are
//     Re V(j, i) = Re' - 8 S_j - 8 S_i + 128 N and
//     Im V(j, i) = Im' - 8 E_j + 8 E_i, integers, exact in FP32 below 2^24.
//   - With several time slices each slice writes its partial triangle and
//     xc_reduce_kernel adds them (exact).
#include "bf_common.h"

namespace {
constexpr int XU = 64;                    // samples per unit
constexpr int XUP = XU / 2;               // packets per unit
constexpr int TCH = 32;                   // channels per turn workgroup (one 128-byte run)
constexpr int XPD = 2;                    // units of voltages in flight per wave

struct XcArgs {
  const uint8_t *in;                      // (channel, pol) planes [channel*2 + pol][antenna][sample]
  float *out;                             // visibilities, or slice partials
  int nant, nchan, npkt, nslice;
  uint32_t in_bytes;
  long slice_floats;
};
typedef int i4v __attribute__((ext_vector_type(4)));
typedef int i16v __attribute__((ext_vector_type(16)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
}  // namespace

// The block to (channel, pol) planes, unit-blocked: plane pq = channel*2 + pol,
// unit u (64 samples), antenna a: 64 bytes at ((pq * nunit + u) * nant + a) * 64.
// Workgroup = (unit, 16 antennas, 32 channels).  (1) Its 512 (packet, antenna)
// 128-byte runs of 32 channels, 16 bytes a lane, go to LDS as words
// [antenna][channel][packet] (row pitch 34 words: a wave's stores, lanes over
// (16-byte piece, packet), fall on 64 distinct banks).  (2) Each lane builds
// 16 bytes (8 packets) of one (channel, pol) of one antenna with byte
// permutes and stores them; four lanes cover an antenna's 64-byte segment.
constexpr int TA16 = 16, TPS = 34;
__global__ __launch_bounds__(256) void xc_turn_kernel(const uint8_t *__restrict__ in, uint8_t *__restrict__ turn,
                                                      int nant, int nchan, int npkt, int order, uint32_t in_bytes) {
  __shared__ uint32_t lds[TA16 * TCH * TPS];
  const int ncb = (nchan + TCH - 1) / TCH, nunit = npkt / XUP;
  const long w = blockIdx.x;
  const int u = (int)(w % nunit), cb = (int)((w / nunit) % ncb), ab = (int)(w / ((long)nunit * ncb));
  const int tid = threadIdx.x;
  const int ngroup = nchan / 8;
  const __amdgpu_buffer_rsrc_t rin = buffer_rsrc(in, in_bytes);
  // (1) piece i = tid + 256k: quad = i & 7 (channels 4 quad .. + 3), packet
  // (i >> 3 & 7) + 8 (i >> 10), antenna (i >> 6) & 15
  uint4 v[16];
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const int i = tid + 256 * k, quad = i & 7, pl = ((i >> 3) & 7) + 8 * (i >> 10), al = (i >> 6) & 15;
    const int c = cb * TCH + 4 * quad, ant = ab * TA16 + al, p = u * XUP + pl;
    const uint32_t off = c < nchan && ant < nant
                             ? (uint32_t)(chunk_offset(order, p, ant, c >> 3, nant, nchan, ngroup) + (c & 7) * 4)
                             : 0x80000000u;
    typedef uint32_t u4 __attribute__((ext_vector_type(4)));
    const u4 x = __builtin_amdgcn_raw_buffer_load_b128(rin, off, 0, 0);
    v[k] = make_uint4(x.x, x.y, x.z, x.w);
  }
#pragma unroll
  for (int k = 0; k < 16; k++) {
    const int i = tid + 256 * k, quad = i & 7, pl = ((i >> 3) & 7) + 8 * (i >> 10), al = (i >> 6) & 15;
    uint32_t *r = lds + (al * TCH + 4 * quad) * TPS + pl;
    r[0] = v[k].x;
    r[TPS] = v[k].y;
    r[2 * TPS] = v[k].z;
    r[3 * TPS] = v[k].w;
  }
  __syncthreads();
  // (2) piece i = tid + 256k: 16 bytes (packets 8 (i & 3) .. + 7) of channel
  // (i >> 2) & 31, pol (i >> 7) & 1, antenna k; word (p, a, c) = bytes
  // [t0 q0, t0 q1, t1 q0, t1 q1]
#pragma unroll 4
  for (int k = 0; k < 16; k++) {
    const int i = tid + 256 * k, pc = i & 3, cl = (i >> 2) & 31, q = (i >> 7) & 1;
    const int c = cb * TCH + cl, ant = ab * TA16 + k;
    if (c >= nchan || ant >= nant) continue;
    const uint32_t *r = lds + (k * TCH + cl) * TPS + 8 * pc;
    const uint2 w0 = *(const uint2 *)r, w1 = *(const uint2 *)(r + 2), w2 = *(const uint2 *)(r + 4),
                w3 = *(const uint2 *)(r + 6);
    const uint32_t sel = q ? 0x07050301u : 0x06040200u;
    const uint4 o = make_uint4(__builtin_amdgcn_perm(w0.y, w0.x, sel), __builtin_amdgcn_perm(w1.y, w1.x, sel),
                               __builtin_amdgcn_perm(w2.y, w2.x, sel), __builtin_amdgcn_perm(w3.y, w3.x, sel));
    *(uint4 *)(turn + ((long)((2 * c + q) * nunit + u) * nant + ant) * XU + 16 * pc) = o;
  }
}

// The triangle's 32x32 tiles (J <= I) in column-major order, (0,0), (0,1),
// (1,1), (0,2), ..., and the share of them that wave part P of NS takes: in
// this order the first shares need fewer antenna blocks (96 antennas, two
// shares: blocks 0-1 with two W operands, and blocks 0-2 with one, where
// row-major order gives 3 + 3 and 2 + 2).
namespace {
template <int NB> constexpr int ntile() { return NB * (NB + 1) / 2; }
template <int NB> constexpr int tile_j(int t) {
  int k = 0;
  for (int I = 0; I < NB; I++)
    for (int J = 0; J <= I; J++, k++)
      if (k == t) return J;
  return -1;
}
template <int NB> constexpr int tile_i(int t) {
  int k = 0;
  for (int I = 0; I < NB; I++)
    for (int J = 0; J <= I; J++, k++)
      if (k == t) return I;
  return -1;
}
template <int NB, int NS, int P> constexpr int tile_lo() { return P * ntile<NB>() / NS; }
template <int NB, int NS, int P> constexpr int tile_hi() { return (P + 1) * ntile<NB>() / NS; }
template <int NB, int NS> constexpr int tiles_max() {
  int m = 0;
  for (int P = 0; P < NS; P++) {
    const int n = (P + 1) * ntile<NB>() / NS - P * ntile<NB>() / NS;
    m = n > m ? n : m;
  }
  return m;
}
// block b is read by a tile of the share: as a row block (X) or a column block (X and W)
template <int NB, int NS, int P> constexpr bool reads(int b) {
  for (int t = tile_lo<NB, NS, P>(); t < tile_hi<NB, NS, P>(); t++)
    if (tile_j<NB>(t) == b || tile_i<NB>(t) == b) return true;
  return false;
}
template <int NB, int NS, int P> constexpr bool is_col(int b) {
  for (int t = tile_lo<NB, NS, P>(); t < tile_hi<NB, NS, P>(); t++)
    if (tile_i<NB>(t) == b) return true;
  return false;
}

// Share P of one (channel, pol) plane over units [ub, ub + nunit).
template <int NB, int NS, int P, int PD>
__device__ __forceinline__ void xc_share(const XcArgs &a, int pq, int ub, int nunit, float *out, int lane) {
  constexpr int T0 = tile_lo<NB, NS, P>(), T1 = tile_hi<NB, NS, P>(), NTW = tiles_max<NB, NS>();
  const int n = lane & 31, h = lane >> 5;
  const int nsamp = 2 * a.npkt;
  const __amdgpu_buffer_rsrc_t rin = buffer_rsrc(a.in, a.in_bytes);
  // lane part of each block's offset in a unit (sentinel for padding
  // antennas: zeros); unit u of the plane starts at (pq * nunit + u) * nant * 64
  const int ntot = nsamp / XU;
  uint32_t off[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    const int ant = 32 * b + n;
    off[b] = ant < a.nant ? (uint32_t)(ant * XU + 32 * h) : 0x80000000u;
  }
  // (units past the slice read at offset in_bytes and up, which the buffer's
  // range check answers with zeros: every pass of the loop below issues the
  // same loads, so each unit waits only for its own)
  auto load = [&](int u, uint32_t (&r)[NB][8]) {
    const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane(
        u < nunit ? (int)(((long)pq * ntot + ub + u) * a.nant * XU) : (int)a.in_bytes);
#pragma unroll
    for (int b = 0; b < NB; b++) {
      if (!reads<NB, NS, P>(b)) continue;
      const u4v v0 = __builtin_amdgcn_raw_buffer_load_b128(rin, off[b], so, 0);
      const u4v v1 = __builtin_amdgcn_raw_buffer_load_b128(rin, off[b] + 16, so, 0);
      r[b][0] = v0.x; r[b][1] = v0.y; r[b][2] = v0.z; r[b][3] = v0.w;
      r[b][4] = v1.x; r[b][5] = v1.y; r[b][6] = v1.z; r[b][7] = v1.w;
    }
  };
  i16v accr[NTW], acci[NTW];
#pragma unroll
  for (int t = 0; t < NTW; t++) { accr[t] = (i16v){}; acci[t] = (i16v){}; }
  uint32_t sr[NB], si[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) sr[b] = si[b] = 0;

  // four 16-sample K steps per unit: lane half h takes samples 32h + 8s .. + 7
  auto compute = [&](const uint32_t (&r)[NB][8]) {
#pragma unroll
    for (int st = 0; st < 4; st++) {
      i4v X[NB], W[NB];
#pragma unroll
      for (int b = 0; b < NB; b++) {
        if (!reads<NB, NS, P>(b)) continue;
        const uint32_t y0 = r[b][2 * st] ^ 0x88888888u, y1 = r[b][2 * st + 1] ^ 0x88888888u;
        const uint32_t ur0 = y0 & 0x0F0F0F0Fu, ur1 = y1 & 0x0F0F0F0Fu;
        const uint32_t ui0 = (y0 >> 4) & 0x0F0F0F0Fu, ui1 = (y1 >> 4) & 0x0F0F0F0Fu;
        sr[b] = __builtin_amdgcn_sad_u8(ur0, 0u, sr[b]);
        sr[b] = __builtin_amdgcn_sad_u8(ur1, 0u, sr[b]);
        si[b] = __builtin_amdgcn_sad_u8(ui0, 0u, si[b]);
        si[b] = __builtin_amdgcn_sad_u8(ui1, 0u, si[b]);
        X[b] = (i4v){(int)ur0, (int)ur1, (int)ui0, (int)ui1};
        if (is_col<NB, NS, P>(b)) {
          // -u bytewise, borrow-free: (0x80 - u) ^ 0x80 for u in 0..15
          const uint32_t nr0 = (0x80808080u - ur0) ^ 0x80808080u, nr1 = (0x80808080u - ur1) ^ 0x80808080u;
          W[b] = (i4v){(int)ui0, (int)ui1, (int)nr0, (int)nr1};
        }
      }
#pragma unroll
      for (int t = T0; t < T1; t++) {
        const int J = tile_j<NB>(t), I = tile_i<NB>(t);
        accr[t - T0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(X[J], X[I], accr[t - T0], 0, 0, 0);
        acci[t - T0] = __builtin_amdgcn_mfma_i32_32x32x32_i8(X[J], W[I], acci[t - T0], 0, 0, 0);
      }
    }
  };

  uint32_t r[PD][NB][8];
  // in unit order, as the loop issues them
#pragma unroll
  for (int k = 0; k < PD; k++) {
    load(k, r[k]);
    __builtin_amdgcn_sched_barrier(0);
  }
  // whole rounds of PD units, then the rest
  int u0 = 0;
  for (; u0 + PD <= nunit; u0 += PD) {
#pragma unroll
    for (int k = 0; k < PD; k++) {
      compute(r[k]);
      load(u0 + k + PD, r[k]);
      // (the loads stay here: sunk below the next units' work, they would be
      // waited for with those units')
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int k = 0; k < PD - 1; k++)
    if (u0 + k < nunit) compute(r[k]);

  // per-antenna sums over both lane halves: S = sum (ur + ui), E = sum (ur - ui)
  int S[NB], E[NB];
#pragma unroll
  for (int b = 0; b < NB; b++) {
    S[b] = E[b] = 0;
    if (!reads<NB, NS, P>(b)) continue;
    const int s0 = (int)(sr[b] + si[b]), e0 = (int)sr[b] - (int)si[b];
    S[b] = s0 + __shfl_xor(s0, 32, 64);
    E[b] = e0 + __shfl_xor(e0, 32, 64);
  }
  const int N128 = 128 * nunit * XU;
  // lane (n, h) of tile (J, I) holds column i = 32I + n and rows
  // j = 32J + 8(v/4) + 4h + v%4
  const int pol = pq & 1, ch = pq >> 1;
#pragma unroll
  for (int t = T0; t < T1; t++) {
    const int J = tile_j<NB>(t), I = tile_i<NB>(t);
    const int ii = 32 * I + n;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int jl = 8 * (v >> 2) + 4 * h + (v & 3), jj = 32 * J + jl;
      const int Sj = __shfl(S[J], jl, 64), Ej = __shfl(E[J], jl, 64);
      if (ii < a.nant && jj <= ii) {
        const long bl = (long)ii * (ii + 1) / 2 + jj;
        const int re = accr[t - T0][v] - 8 * Sj - 8 * S[I] + N128;
        const int im = acci[t - T0][v] - 8 * Ej + 8 * E[I];
        *(float2 *)(out + ((bl * a.nchan + ch) * 2 + pol) * 2) = make_float2((float)re, (float)im);
      }
    }
  }
}
}  // namespace

// Share `part` of NS (a wave-uniform branch to the share's own code).
template <int NB, int NS, int P, int PD>
__device__ __forceinline__ void xc_share_of(int part, const XcArgs &a, int pq, int ub, int nunit, float *out,
                                            int lane) {
  if constexpr (P + 1 < NS) {
    if (part != P) {
      xc_share_of<NB, NS, P + 1, PD>(part, a, pq, ub, nunit, out, lane);
      return;
    }
  }
  xc_share<NB, NS, P, PD>(a, pq, ub, nunit, out, lane);
}

// NB antenna blocks of 32, NS waves per (channel, pol) plane, PD units of
// voltages in flight.  Wave g of the grid: share g % NS of plane (g / NS) %
// nplane of slice g / (NS nplane); the NS shares of a plane are neighbours in
// one workgroup or the next (same XCD: blockIdx is spread round-robin, so
// workgroup P takes work item (P % 8) * (grid / 8) + P / 8).
template <int NB, int NS, int PD>
__global__ __launch_bounds__(256) void xc_kernel(XcArgs a) {
  const int P = blockIdx.x;
  const int L = (P & 7) * (gridDim.x >> 3) + (P >> 3);
  const int lane = threadIdx.x & 63;
  // wave-uniform (a scalar): the plane's offset goes in the loads' scalar offset
  const int gw = L * 4 + __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int nplane = 2 * a.nchan;
  // (readfirstlane: the runtime division leaves its result in vector registers)
  const int part = gw % NS;
  const int pq = __builtin_amdgcn_readfirstlane((gw / NS) % nplane);
  const int slice = __builtin_amdgcn_readfirstlane(gw / (NS * nplane));
  if (slice >= a.nslice) return;          // whole waves; nothing below synchronises
  const int ntot = a.npkt / XUP;
  const int ub = (int)((long)ntot * slice / a.nslice), nunit = (int)((long)ntot * (slice + 1) / a.nslice) - ub;
  float *out = a.out + slice * a.slice_floats;
  xc_share_of<NB, NS, 0, PD>(part, a, pq, ub, nunit, out, lane);
}

// Up to 64 antennas the correlation reads the block itself.  The samples of a
// (channel, pol) may enter the sums in any order, so the words of four packets
// become the operands' eight samples by byte permutes, with no turned copy of the
// block: one workgroup takes CH channels (16 or 32 bytes of each packet and
// antenna), a thread four packets of one antenna and four channels, and stages
// [channel][four packets][antenna][pol][8 samples] in LDS, double-buffered per 32
// packets with two more units in flight; a wave takes one (channel, pol) of 33 to 64
// antennas or one channel of up to 32.  Workgroups that share 128-byte lines are
// neighbours on one XCD.  64 antennas x 384 channels x 4096 samples with groups
// outermost: 127 -> 51 us (201 MB, 3.9 TB/s), with antennas outermost 129 -> 91.  (Three
// units in flight: the same, and scratch up to 32 antennas.)
namespace {
constexpr int XF = 512;                   // threads
}  // namespace

template <int NB, int CH>
__global__ __launch_bounds__(XF, NB == 1 ? 4 : 2) void xc_fused_kernel(XcArgs a, int order) {
  constexpr int NA = 32 * NB, NT = NB * (NB + 1) / 2, NPOL = CH / 4;   // pols of a wave
  static_assert(NA * 8 * (CH / 4) == XF, "one staging task per thread and unit");
  __shared__ uint4 lds[2][CH * 8 * NA];
  const int P = blockIdx.x, nq = a.nchan / CH;
  const int L = (P & 7) * (gridDim.x >> 3) + (P >> 3);
  if (L >= nq * a.nslice) return;
  const int c0 = L % nq * CH, slice = L / nq;
  const int ntot = a.npkt / XUP;
  const int ub = (int)((long)ntot * slice / a.nslice), nunit = (int)((long)ntot * (slice + 1) / a.nslice) - ub;
  const int tid = threadIdx.x, lane = tid & 63, n = lane & 31, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);

  // staging task: antenna ant, packets 4 wave .. + 3 of the unit, channels c0 + 4 half .. + 3
  const int ant = CH == 4 ? lane : n, half = CH == 4 ? 0 : h;
  const __amdgpu_buffer_rsrc_t rin = buffer_rsrc(a.in, a.in_bytes);
  uint32_t off[4];
#pragma unroll
  for (int k = 0; k < 4; k++)
    off[k] = ant < a.nant ? (uint32_t)(chunk_offset(order, 4 * wave + k, ant, c0 >> 3, a.nant, a.nchan, a.nchan / 8) +
                                       ((c0 & 7) + 4 * half) * 4)
                          : 0x80000000u;
  // (units past the slice read at offset in_bytes and up, which the buffer's range
  // check answers with zeros)
  auto load = [&](int u, u4v (&r)[4]) __attribute__((always_inline)) {
    const uint32_t so = (uint32_t)__builtin_amdgcn_readfirstlane(
        u < nunit ? (int)((long)(ub + u) * XUP * a.nant * a.nchan * 4) : (int)a.in_bytes);
#pragma unroll
    for (int k = 0; k < 4; k++) r[k] = __builtin_amdgcn_raw_buffer_load_b128(rin, off[k], so, 0);
  };
  auto store = [&](uint4 *st, const u4v (&r)[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 4; c++)
      st[((4 * half + c) * 8 + wave) * NA + ant] =
          make_uint4(__builtin_amdgcn_perm(r[1][c], r[0][c], 0x06040200u), __builtin_amdgcn_perm(r[3][c], r[2][c], 0x06040200u),
                     __builtin_amdgcn_perm(r[1][c], r[0][c], 0x07050301u), __builtin_amdgcn_perm(r[3][c], r[2][c], 0x07050301u));
  };

  const int cw = NPOL == 1 ? wave >> 1 : wave, q0 = NPOL == 1 ? wave & 1 : 0;   // this wave's channel and first pol
  i16v accr[NPOL][NT], acci[NPOL][NT];
  uint32_t sr[NPOL][NB], si[NPOL][NB];
#pragma unroll
  for (int q = 0; q < NPOL; q++) {
#pragma unroll
    for (int t = 0; t < NT; t++) { accr[q][t] = (i16v){}; acci[q][t] = (i16v){}; }
#pragma unroll
    for (int b = 0; b < NB; b++) sr[q][b] = si[q][b] = 0;
  }
  auto compute = [&](const uint4 *st) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; s++) {
#pragma unroll
      for (int q = 0; q < NPOL; q++) {
        i4v X[NB], W[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) {
          const uint2 r = ((const uint2 *)(st + (cw * 8 + 2 * s + h) * NA + 32 * b + n))[q0 + q];
          const uint32_t y0 = r.x ^ 0x88888888u, y1 = r.y ^ 0x88888888u;
          const uint32_t ur0 = y0 & 0x0F0F0F0Fu, ur1 = y1 & 0x0F0F0F0Fu;
          const uint32_t ui0 = (y0 >> 4) & 0x0F0F0F0Fu, ui1 = (y1 >> 4) & 0x0F0F0F0Fu;
          sr[q][b] = __builtin_amdgcn_sad_u8(ur1, 0u, __builtin_amdgcn_sad_u8(ur0, 0u, sr[q][b]));
          si[q][b] = __builtin_amdgcn_sad_u8(ui1, 0u, __builtin_amdgcn_sad_u8(ui0, 0u, si[q][b]));
          X[b] = (i4v){(int)ur0, (int)ur1, (int)ui0, (int)ui1};
          const uint32_t nr0 = (0x80808080u - ur0) ^ 0x80808080u, nr1 = (0x80808080u - ur1) ^ 0x80808080u;
          W[b] = (i4v){(int)ui0, (int)ui1, (int)nr0, (int)nr1};
        }
#pragma unroll
        for (int t = 0; t < NT; t++) {
          const int J = tile_j<NB>(t), I = tile_i<NB>(t);
          accr[q][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(X[J], X[I], accr[q][t], 0, 0, 0);
          acci[q][t] = __builtin_amdgcn_mfma_i32_32x32x32_i8(X[J], W[I], acci[q][t], 0, 0, 0);
        }
      }
    }
  };

  u4v ra[4], rb[4];                         // units u + 1 and u + 2, in flight while unit u is computed
  load(0, ra);
  load(1, rb);
  store(lds[0], ra);
  load(2, ra);
  __syncthreads();
#pragma unroll 1
  for (int u = 0; u < nunit; u += 2) {
    store(lds[1], rb);
    load(u + 3, rb);
    __builtin_amdgcn_sched_barrier(0);
    compute(lds[0]);
    __syncthreads();
    if (u + 1 >= nunit) break;
    store(lds[0], ra);
    load(u + 4, ra);
    __builtin_amdgcn_sched_barrier(0);
    compute(lds[1]);
    __syncthreads();
  }

  // The sums leave by way of LDS, eight rows of a tile at a time, so that the CH
  // channels' visibilities of a baseline (64 or 128 bytes) are written together; a
  // pitch of one entry more than a baseline has spreads them over the banks.
  constexpr int E8 = 2 * CH, PITCH = E8 + 1, NBUF = CH == 4 ? 2 : 1;
  static_assert(NBUF * 256 * PITCH * sizeof(float2) <= sizeof(lds), "the rows in transit");
  float2 *vis = (float2 *)(a.out + slice * a.slice_floats);
  const int N128 = 128 * nunit * XU;
  int S[NPOL][NB], E[NPOL][NB];
#pragma unroll
  for (int q = 0; q < NPOL; q++)
#pragma unroll
    for (int b = 0; b < NB; b++) {
      const int s0 = (int)(sr[q][b] + si[q][b]), e0 = (int)sr[q][b] - (int)si[q][b];
      S[q][b] = s0 + __shfl_xor(s0, 32, 64);
      E[q][b] = e0 + __shfl_xor(e0, 32, 64);
    }
  int turn = 0;
#pragma unroll
  for (int t = 0; t < NT; t++) {
    const int J = tile_j<NB>(t), I = tile_i<NB>(t);
#pragma unroll
    for (int m = 0; m < 4; m++) {
      if (32 * J + 8 * m >= a.nant || 32 * I >= a.nant) continue;
      float2 *buf = (float2 *)lds + (NBUF == 2 ? (turn++ & 1) : 0) * 256 * PITCH;
#pragma unroll
      for (int q = 0; q < NPOL; q++)
#pragma unroll
        for (int x = 0; x < 4; x++) {
          const int v = 4 * m + x, row = 4 * h + x, jl = 8 * m + row;
          const int Sj = __shfl(S[q][J], jl, 64), Ej = __shfl(E[q][J], jl, 64);
          const int re = accr[q][t][v] - 8 * Sj - 8 * S[q][I] + N128;
          const int im = acci[q][t][v] - 8 * Ej + 8 * E[q][I];
          buf[(row * 32 + n) * PITCH + cw * 2 + q0 + q] = make_float2((float)re, (float)im);
        }
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 256 * E8 / XF; k++) {
        const int e = tid + k * XF, i = 32 * I + (e / E8) % 32, j = 32 * J + 8 * m + e / E8 / 32;
        if (i < a.nant && j <= i)
          vis[((long)i * (i + 1) / 2 + j) * a.nchan * 2 + c0 * 2 + e % E8] = buf[(e / E8) * PITCH + e % E8];
      }
      if (NBUF == 1) __syncthreads();
    }
  }
}

extern "C" size_t bfk_xcorr_vis_bytes(int nant, int nchan) {
  return (size_t)nant * (nant + 1) / 2 * nchan * 2 * 2 * sizeof(float);
}

// Sum of the slice partials (integer-valued floats: exact in any order).
__global__ __launch_bounds__(256) void xc_reduce_kernel(const float4 *__restrict__ part, float4 *__restrict__ vis,
                                                        long n4, int nslice) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  float4 s = part[i];
  for (int k = 1; k < nslice; k++) {
    const float4 v = part[k * n4 + i];
    s.x += v.x; s.y += v.y; s.z += v.z; s.w += v.w;
  }
  vis[i] = s;
}

// Slices of the block's time for a shape: one when the (channel, pol) planes
// alone give about a wave per SIMD (2 nchan planes x 2 waves >= 1024; measured
// on the 384-channel block: 1, 2, 4 and 8 slices took 0.235, 0.254, 0.299 and
// 0.409 ms: the partial sums' traffic outweighs the extra waves), else enough
// for that, with at least 8 units (512 samples) per slice.
extern "C" int bfk_xcorr_default_slices(int nchan, int npkt) {
  const int nunit = npkt / XUP;
  int s = nchan >= 256 ? 1 : (256 + nchan - 1) / nchan;
  if (s > nunit / 8) s = nunit / 8;
  return s < 1 ? 1 : s;
}

extern "C" size_t bfk_xcorr_part_bytes(int nant, int nchan, int nslice) {
  return nslice > 1 ? (size_t)nslice * bfk_xcorr_vis_bytes(nant, nchan) : 0;
}

// The turned path or the fused kernel, and the latter's time slices, by modelled
// times in us: of a block alone on one stream, and among others (three plans in turn,
// where the launches themselves take 3.75, 6.6 and 9.4 for one, two and three).  Fitted
// to 469 shapes of 8 to 64 antennas, 8 to 384 channels and 64 to 4096 samples in one to
// 24 slices each, near the faster ones to 3 % (5 % above 32 antennas with antennas
// outermost).
//   fused: a workgroup per 8 channels (4 above 32 antennas) and slice; a base and some
//     per 8 antennas, then a time per 32 packets.  Up to 32 antennas two share a CU.
//     With antennas outermost a 128-byte line serves eight workgroups of one XCD, if
//     the XCD has whole eights.  Several slices: the sum of their partials.
//   turned: bytes, the units of a wave's slice, visibilities, and again the sum.
struct XcCost {
  float alone, among;
};
static float vis_mb(int nant, int nchan) { return 8e-6f * (float)nant * (float)(nant + 1) * (float)nchan; }
static XcCost xc_fused_cost(int nant, int nchan, int npkt, int order, int slices) {
  //                               base  /8 ant  /unit  + /antenna  MB    sum  /slice  /MB
  static const float c[2][2][8] = {{{3.31f, .864f, .75f, .012f, .521f, 1.36f, .235f, 0.f},
                                    {2.78f, 1.05f, .849f, .003f, .258f, 1.45f, .24f, .147f}},
                                   {{5.83f, .285f, .474f, .02f, .314f, 1.78f, .218f, .174f},
                                    {4.76f, .57f, .982f, .003f, .181f, 1.44f, .241f, .213f}}};
  const float(&p)[8] = c[nant > 32][order];
  const int sets = nchan / (nant <= 32 ? 8 : 4), wgs = sets * slices, room = nant <= 32 ? 512 : 256;
  const int units = (npkt / XUP + slices - 1) / slices;
  const float mb = 4e-6f * (float)npkt * (float)nant * (float)nchan, vis = vis_mb(nant, nchan) * (float)slices;
  float unit = p[2] + p[3] * (float)nant;
  if (nant <= 32 && wgs > 256) unit *= 1.8f;
  if (nant > 32 && order == 0 && nchan > 32 && wgs % 64 && wgs % (8 * sets)) unit *= 1.12f;
  const float once = p[0] + p[1] * (float)((nant + 7) / 8), chain = unit * (float)units;
  const float sum = slices > 1 ? p[5] + p[6] * (float)slices + p[7] * vis : 0.f;
  const float alone = fmaxf(once + (float)((wgs + room - 1) / room) * chain, mb / 4.3f) + p[4] * vis + sum;
  const float share = (once + chain) * (float)wgs / (float)room + (slices > 1 ? p[7] * vis : 0.f);
  return {alone, fmaxf(fmaxf(slices > 1 ? 6.6f : 3.75f, alone / 2.75f), fmaxf(share, mb / 4.3f))};
}
static XcCost xc_turned_cost(int nant, int nchan, int npkt, int order) {
  //                               base   MB     /unit  /8 ant  vis MB  sum
  static const float c[2][2][6] = {{{6.27f, .354f, .235f, .298f, .619f, 2.26f}, {6.32f, .266f, .25f, .275f, .815f, 2.61f}},
                                   {{7.87f, .453f, .311f, .091f, .41f, 1.98f}, {7.46f, .407f, .333f, .17f, .323f, 2.58f}}};
  const float(&p)[6] = c[nant > 32][order];
  const int slices = bfk_xcorr_default_slices(nchan, npkt), units = (npkt / XUP + slices - 1) / slices;
  const float mb = 4e-6f * (float)npkt * (float)nant * (float)nchan, vis = vis_mb(nant, nchan);
  const float alone = p[0] + p[1] * mb + p[2] * (float)units + p[3] * (float)((nant + 7) / 8) + p[4] * vis * (float)slices +
                      (slices > 1 ? p[5] : 0.f);
  return {alone, fmaxf(slices > 1 ? 9.4f : 6.5f, fmaxf(alone / 2.3f, .66f * mb + .25f * vis))};
}
// The fused kernel's slices that make the product of its times least, none of them
// above `most`; 0 where there are none, or the kernel cannot run: above 64 antennas, or
// with sums that FP32 may not hold.
static int xc_slices(int nant, int nchan, int npkt, int order, XcCost most) {
  if (nant > 64 || npkt > 65536) return 0;
  const int room = (nant <= 32 ? 512 : 256) / (nchan / (nant <= 32 ? 8 : 4));
  int best = 0;
  float least = 0.f;
  for (int s = 1; s <= 32 && s <= npkt / XUP && (s == 1 || s <= room); s++) {
    const XcCost f = xc_fused_cost(nant, nchan, npkt, order, s);
    if (f.alone > most.alone || f.among > most.among || (best && f.alone * f.among >= least)) continue;
    least = f.alone * f.among;
    best = s;
  }
  return best;
}
extern "C" int bfk_xcorr_fused_slices(int nant, int nchan, int npkt, int order) {
  return xc_slices(nant, nchan, npkt, order, {1e9f, 1e9f});
}
// The slices in which the fused kernel takes the turned path's place, or 0: where its
// time among others is no longer, that of a block alone, with the 11 us of a launch and
// its wait beside the kernels, at most 3 to 4 % longer (5 % shorter above 32 antennas
// with antennas outermost, where the model errs by more), and their product 5 % less.
// In the 207 of the shapes that it picks a block alone takes 0.48 to 1.12 times the
// turned path's time (mean 0.95, over 1.05 in 7), one among others 0.64.  us alone and among others,
// turned and fused: 64 antennas x 384 channels x 4096 samples, antennas outermost 127/143
// and 87/92, groups outermost 130/145 and 57/52; 63 x 48 x 2048, groups outermost 21.4/12.4
// and 23.0/8.3 (with the launch and wait 32.6 and 34.3); 8 x 328 x 128 7.2/6.8 and 6.0/3.8.
// Left turned: 60 x 16 x 128 10.0/6.6 and 12.1/4.2, 32 x 32 x 1088 12.8/9.6 and 15.0/6.6, 64
// x 128 x 1024 with antennas outermost 23.4/15.8 and 27.6/14.1.
extern "C" int bfk_xcorr_use_fused(int nant, int nchan, int npkt, int order) {
  static const float longer[2][2] = {{1.03f, 1.03f}, {.95f, 1.04f}};
  const XcCost t = xc_turned_cost(nant, nchan, npkt, order);
  const int s = xc_slices(nant, nchan, npkt, order, {longer[nant > 32][order] * (t.alone + 11.f) - 11.f, t.among});
  if (!s) return 0;
  const XcCost f = xc_fused_cost(nant, nchan, npkt, order, s);
  return f.alone * f.among < .95f * t.alone * t.among ? s : 0;
}

// nfused: 0, or the slices in which the fused kernel runs.  d_part:
// bfk_xcorr_part_bytes of its slices, or of nslice; d_turn: the input's size, not used
// by the fused kernel.
extern "C" int bfk_xcorr(int nant, int nchan, int npkt, int order, const uint8_t *d_in, uint8_t *d_turn,
                         float *d_part, int nslice, int nfused, float *d_vis, void *stream) {
  if (nant < 1 || nant > 96 || nchan < 8 || nchan % 8 || npkt < XUP || npkt % XUP || order < 0 || order > 1) {
    bfk_set_error("bfk_xcorr: unsupported shape nant=%d nchan=%d npkt=%d order=%d", nant, nchan, npkt, order);
    return -1;
  }
  if ((size_t)npkt * nant * nchan * 4 > 0x7fffffffu) {
    bfk_set_error("bfk_xcorr: block above 2 GiB");
    return -1;
  }
  if (nfused && (nant > 64 || npkt > 65536 || nfused < 0 || nfused > npkt / XUP || (nfused > 1 && !d_part))) {
    bfk_set_error("bfk_xcorr: %d slices of the fused kernel (partials %p)", nfused, (void *)d_part);
    return -1;
  }
  if (nslice < 1 || nslice > npkt / XUP || (!nfused && ((nslice > 1 && !d_part) || !d_turn))) {
    bfk_set_error("bfk_xcorr: %d slices of %d units (partials %p)", nslice, npkt / XUP, (void *)d_part);
    return -1;
  }
  hipStream_t s = (hipStream_t)stream;
  const uint32_t in_bytes = (uint32_t)((size_t)npkt * nant * nchan * 4);
  const long n4 = (long)(bfk_xcorr_vis_bytes(nant, nchan) / sizeof(float4));
  if (nfused) {
    XcArgs a;
    a.in = d_in;
    a.out = nfused > 1 ? d_part : d_vis;
    a.nant = nant;
    a.nchan = nchan;
    a.npkt = npkt;
    a.nslice = nfused;
    a.in_bytes = in_bytes;
    a.slice_floats = 4 * n4;
    const int ch = nant <= 32 ? 8 : 4;
    const dim3 grid((unsigned)((nchan / ch * nfused + 7) / 8 * 8));
    if (ch == 8) hipLaunchKernelGGL((xc_fused_kernel<1, 8>), grid, dim3(XF), 0, s, a, order);
    else hipLaunchKernelGGL((xc_fused_kernel<2, 4>), grid, dim3(XF), 0, s, a, order);
    if (nfused > 1)
      hipLaunchKernelGGL(xc_reduce_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s, (const float4 *)d_part,
                         (float4 *)d_vis, n4, nfused);
    return bfk_check(hipGetLastError(), "xc_fused_kernel");
  }
  const long nturn = (long)(npkt / XUP) * ((nchan + TCH - 1) / TCH) * ((nant + TA16 - 1) / TA16);
  hipLaunchKernelGGL(xc_turn_kernel, dim3((unsigned)nturn), dim3(256), 0, s, d_in, d_turn, nant, nchan, npkt, order,
                     in_bytes);
  XcArgs a;
  a.in = d_turn;
  a.out = nslice > 1 ? d_part : d_vis;
  a.nant = nant;
  a.nchan = nchan;
  a.npkt = npkt;
  a.nslice = nslice;
  a.in_bytes = in_bytes;
  a.slice_floats = (long)(bfk_xcorr_vis_bytes(nant, nchan) / sizeof(float));
  // two waves per plane above 32 antennas (measured on the 96-antenna block,
  // whole block: one, two, three and six waves per plane took 0.242, 0.238,
  // 0.249 and 0.259 ms; more waves per SIMD do not pay for the duplicated
  // loads and conversions.  With each unit waiting for its own loads: two
  // waves 0.222 ms, three 0.252 ms, or 0.266 ms held to 168 registers for
  // three waves per SIMD; XPD = 3 0.229 ms)
  const int ns = nant <= 32 ? 1 : 2;
  const long nwave = (long)ns * 2 * nchan * nslice;
  const dim3 grid((unsigned)(((nwave + 3) / 4 + 7) / 8 * 8)), block(256);
  if (nant <= 32) hipLaunchKernelGGL((xc_kernel<1, 1, XPD>), grid, block, 0, s, a);
  else if (nant <= 64) hipLaunchKernelGGL((xc_kernel<2, 2, XPD>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((xc_kernel<3, 2, XPD>), grid, block, 0, s, a);
  if (nslice > 1) {
    hipLaunchKernelGGL(xc_reduce_kernel, dim3((unsigned)((n4 + 255) / 256)), dim3(256), 0, s,
                       (const float4 *)d_part, (float4 *)d_vis, n4, nslice);
  }
  return bfk_check(hipGetLastError(), "xc_kernel");
}
