// bf_shared8_tile.h -- the parts of a workgroup of eight waves for 65 to 256
// antennas that bf_shared8.hip and bf_packed.hip share: staged rows, the unpack
// into MFMA operands, and the MFMA chains of a wave's 32-beam tile.
#pragma once
#include "bf_common.h"

namespace {
constexpr int NW8 = 8, NT8 = NW8 * 64;     // waves, threads per workgroup
constexpr int BSET8 = NW8 * 32;            // beams per tile
constexpr int STAGE8 = 64 * 1024;          // one channel sub-step, any NKC

template <int NKC> struct S8 {
  static constexpr int NCI = 8 / NKC;           // channels per sub-step
  static constexpr int CQS = 2 * NCI;           // (channel, pol) per sub-step
  static constexpr int ROW = 64 * NKC;          // staged row bytes (antennas)
  static constexpr int NCH = ROW / 16;          // 16-byte chunks per row
  static constexpr int TPT = PCU * 16 * NKC / NT8;   // staging tasks per thread (= NKC)
  static constexpr int UNIT16 = NKC * 8 * 64 * 16;    // FP16 A_re bytes per unit
  static constexpr int UNIT8 = NKC * 2 * 64 * 32;     // FP8 A_re bytes per unit
};

// Byte offset of 16-byte chunk c of staged row r (chunks XORed with the row).
template <int NKC>
__device__ __forceinline__ int srow8(int r, int c) {
  return r * S8<NKC>::ROW + ((c ^ (r & (S8<NKC>::NCH - 1))) << 4);
}

// FP16 A_re of unit u (= 2*cql + tt) of the sub-step: K step S = kc*8 + s of
// lane l at (S*64 + l)*16.  Thread t covers lane t & 63 and the NKC steps
// (t >> 6)*NKC ...: 4*NKC packed bytes of one row, read in one piece.
template <int NKC>
__device__ __forceinline__ void unpack8_f16(const uint8_t *stage, uint8_t *abuf, int u, int tid) {
  const int li = tid & 63, n = li & 31, h = li >> 5, q = tid >> 6;
  const int r = (u >> 1) * TCU + (u & 1) * 32 + n;
  const int S0 = q * NKC, kc = S0 >> 3, s0 = S0 & 7;
  const int byte = kc * 64 + h * 32 + 4 * s0;           // first antenna of the piece
  const uint8_t *src = stage + srow8<NKC>(r, byte >> 4) + (byte & 15);
  uint32_t x[NKC];
  if constexpr (NKC == 4) {
    const uint4 v = *(const uint4 *)src;
    x[0] = v.x; x[1] = v.y; x[2] = v.z; x[3] = v.w;
  } else {
    const uint2 v = *(const uint2 *)src;
    x[0] = v.x; x[1] = v.y;
  }
#pragma unroll
  for (int i = 0; i < NKC; i++) {
    h8v re, im;
    unpack_f16(x[i], re, im);
    *(h8v *)(abuf + ((S0 + i) * 64 + li) * 16) = re;
  }
}

// FP8 A_re of both units of sub-step (channel, pol) cql: unit tt, chunk kc,
// step s2, lane l: record C = (tt*NKC + kc)*2 + s2, its 32 bytes in two
// 16-byte planes, half hl at ((C*2 + hl)*64 + l)*16 (16-byte lane stride:
// conflict-free).  Thread t covers lane t & 63 and NKC/2 of the records.
template <int NKC>
__device__ __forceinline__ void unpack8_f8(const uint8_t *stage, uint8_t *abuf, int cql, int tid) {
  const int li = tid & 63, n = li & 31, h = li >> 5, q = tid >> 6;
#pragma unroll
  for (int i = 0; i < NKC / 2; i++) {
    const int C = q * (NKC / 2) + i, tt = C / (2 * NKC), kc = (C >> 1) % NKC, s2 = C & 1;
    const int r = cql * TCU + tt * 32 + n;
    const uint4 v = *(const uint4 *)(stage + srow8<NKC>(r, kc * 4 + h * 2 + s2));
    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[8];
#pragma unroll
    for (int k = 0; k < 4; k++) {
      o[2 * k] = nib_e4m3(x[k]);
      o[2 * k + 1] = nib_e4m3(x[k] >> 4) ^ 0x80808080u;
    }
    uint8_t *p = abuf + ((C * 2) * 64 + li) * 16;
    *(uint4 *)p = make_uint4(o[0], o[1], o[2], o[3]);
    *(uint4 *)(p + 64 * 16) = make_uint4(o[4], o[5], o[6], o[7]);
  }
}

// FP6 A_re, the record layout of unpack8_f8: six dwords per lane, dwords 0..3
// in plane 0 and 4..5 in the first half of plane 1's 16-byte lane slot.
template <int NKC>
__device__ __forceinline__ void unpack8_f6(const uint8_t *stage, uint8_t *abuf, int cql, int tid) {
  const int li = tid & 63, n = li & 31, h = li >> 5, q = tid >> 6;
#pragma unroll
  for (int i = 0; i < NKC / 2; i++) {
    const int C = q * (NKC / 2) + i, tt = C / (2 * NKC), kc = (C >> 1) % NKC, s2 = C & 1;
    const int r = cql * TCU + tt * 32 + n;
    const uint4 v = *(const uint4 *)(stage + srow8<NKC>(r, kc * 4 + h * 2 + s2));
    const uint32_t x[4] = {v.x, v.y, v.z, v.w};
    uint32_t o[6];
    f6_operand(x, o);
    uint8_t *p = abuf + ((C * 2) * 64 + li) * 16;
    *(uint4 *)p = make_uint4(o[0], o[1], o[2], o[3]);
    *(uint2 *)(p + 64 * 16) = make_uint2(o[4], o[5]);
  }
}

// One unit from LDS A_re: gemm_unit's MFMA chains (one beam tile), A_im
// derived.  With PF, each K step of W is reloaded from row wnext right after
// its last MFMA has issued (rolling prefetch, pinned by scheduling barriers
// that VALU, SALU and LDS work may still cross).
template <int PREC, int NKC, bool PF>
__device__ __forceinline__ void unit8w(Acc<1> &A, WFrag<PREC, 1, NKC> &W, const uint8_t *unit, int lane,
                                       const uint8_t *wfrag, long wnext) {
  __builtin_amdgcn_s_setprio(1);
  A.r[0] = (f16v){};
  A.i[0] = (f16v){};
#pragma unroll
  for (int kc = 0; kc < NKC; kc++) {
    if constexpr (PREC == 0) {
#pragma unroll
      for (int s = 0; s < 8; s++) {
        const uint4 r = *(const uint4 *)(unit + ((kc * 8 + s) * 64 + lane) * 16);
        // A_re = [Dr0,Dr1,-Di0,-Di1,Dr2,Dr3,-Di2,-Di3] -> A_im = [Di0,Di1,Dr0,Dr1,...]
        const uint4 m = make_uint4(r.y ^ 0x80008000u, r.x, r.w ^ 0x80008000u, r.z);
        A.r[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, r), W.w[0][kc][s], A.r[0], 0, 0, 0);
        A.i[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(h8v, m), W.w[0][kc][s], A.i[0], 0, 0, 0);
        if constexpr (PF) {
          __builtin_amdgcn_sched_barrier(0x386);
          W.load_k(wfrag, wnext, 0, kc, s, lane);
          __builtin_amdgcn_sched_barrier(0x386);
        }
      }
    } else {
#pragma unroll
      for (int s2 = 0; s2 < 2; s2++) {
        const uint8_t *src = unit + (((kc * 2 + s2) * 2) * 64 + lane) * 16;
        i8v are, aim;
        if constexpr (PREC == 1) {
          const uint4 r0 = *(const uint4 *)src, r1 = *(const uint4 *)(src + 64 * 16);
          // A_re dwords [Dr, -Di] per 4 antennas -> A_im [Di, Dr]
          are = (i8v){(int)r0.x, (int)r0.y, (int)r0.z, (int)r0.w, (int)r1.x, (int)r1.y, (int)r1.z, (int)r1.w};
          aim = (i8v){(int)(r0.y ^ 0x80808080u), (int)r0.x, (int)(r0.w ^ 0x80808080u), (int)r0.z,
                      (int)(r1.y ^ 0x80808080u), (int)r1.x, (int)(r1.w ^ 0x80808080u), (int)r1.z};
        } else {
          f6_re_im(*(const uint4 *)src, *(const uint2 *)(src + 64 * 16), are, aim);
        }
        A.r[0] = mfma64<PREC>(are, W.hi[0][kc][s2], A.r[0], W.shi(0, kc, s2));
        A.i[0] = mfma64<PREC>(aim, W.hi[0][kc][s2], A.i[0], W.shi(0, kc, s2));
        if constexpr (PREC == 3) {
          A.r[0] = mfma64<PREC>(are, W.mid[0][kc][s2], A.r[0], W.smid(0, kc, s2));
          A.i[0] = mfma64<PREC>(aim, W.mid[0][kc][s2], A.i[0], W.smid(0, kc, s2));
        }
        A.r[0] = mfma64<PREC>(are, W.lo[0][kc][s2], A.r[0], W.slo(0, kc, s2));
        A.i[0] = mfma64<PREC>(aim, W.lo[0][kc][s2], A.i[0], W.slo(0, kc, s2));
        if constexpr (PF) {
          __builtin_amdgcn_sched_barrier(0x386);
          W.load_k(wfrag, wnext, 0, kc, s2, lane);
          __builtin_amdgcn_sched_barrier(0x386);
        }
      }
    }
  }
  __builtin_amdgcn_s_setprio(0);
}
}  // namespace
