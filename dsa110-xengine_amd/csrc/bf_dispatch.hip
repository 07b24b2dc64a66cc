// bf_dispatch.hip -- the fused beamformer's launch arguments and the
// dispatch to its schedules (classic: bf_classic.hip; shared: bf_shared.hip
// to 64 antennas, bf_shared8.hip above).
//
// Reference path: src/dsaX_beamformer.cu promoter (:170-193), beamformer
// (:267-416), badder (:78-112) and adder (:120-158).  The reference runs five
// launches per 32-sample "int" (640 per block) and keeps unpacked FP16 planes
// and FP32 partial powers in HBM between them.  Here one kernel does, per
// tile (one 8-channel output group x 64 samples x a set of beams):
//   (a) the packed 4-bit block is loaded in coalesced 32-byte chunks and
//       transposed into [channel][pol][sample][antenna] rows in LDS;
//   (b) per (channel, pol) a complex GEMM in the real 4M form on
//       v_mfma_f32_32x32x16_f16 (FP16) or v_mfma_f32_32x32x64_f8f6f4
//       (FP8 E4M3 or FP6 E2M3 voltages x split weights), FP32 accumulation;
//   (c) |B|^2, the sums over 2 pols x 8 channels x tavg samples, scaling and
//       the uint8 requantisation in registers, with no HBM round trip.
//
// GEMM orientation: rows (M) = samples, columns (N) = beams, K = antennas x
// {re, im}.  Each lane of a 32x32 accumulator holds one beam column and 16
// sample rows, so the time average is an in-lane sum plus one cross-lane add.
// The complex structure sits on the voltage side: with B-operand K-slots
// [Wr, Wi], the real part uses A = [Dr, -Di] and the imaginary part
// A = [Di, Dr]; weights are stored once.
#include "bf_common.h"

BfArgs bf_make_args(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag,
                    const float *d_wscale, const float *d_scale, uint8_t *d_out, float *d_power,
                    float *d_bpart, int bset_beams) {
  BfArgs a;
  a.in = d_in;
  a.wfrag = (const uint8_t *)d_wfrag;
  a.wscale = d_wscale;
  a.scale = d_scale;
  a.out = d_out;
  a.power = d_power;
  a.bpart = d_bpart;
  a.nant = d->nant;
  a.nchan = d->nchan;
  a.ngroup = d->ngroup;
  a.nbeam = d->nbeam;
  a.nbeam_pad = d->nbeam_pad;
  a.nbt = d->nbt;
  a.wmode = d->wmode;
  a.order = d->order;
  a.ntblk = d->nsamp / TCU;
  a.nbsets = (d->nbeam + bset_beams - 1) / bset_beams;   // beams past nbeam: zero weights, no output
  a.ntiles = a.nbsets * d->ngroup * a.ntblk;
  a.layout = d->layout;
  a.nout = d->nout;
  a.tiles_per_xcd = (a.ntiles + 7) / 8;
  a.pstride = (uint32_t)d->nant * d->nchan * 4;
  a.astride = d->order == 0 ? (uint32_t)d->nchan * 4 : 32u;
  a.gstride = d->order == 0 ? 32u : (uint32_t)d->nant * 32;
  a.in_bytes = (uint32_t)((size_t)d->npkt * d->nant * d->nchan * 4);
  a.wfrag_bytes = (uint32_t)bfk_wfrag_bytes(d);
  a.wscale_bytes = (uint32_t)bfk_wscale_bytes(d);
  a.split = 0;
  a.beam_power = a.psum = NULL;
  a.count = NULL;
  return a;
}

extern "C" int bfk_beamform_classic(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag,
                                    const float *d_wscale, const float *d_scale, uint8_t *d_out,
                                    float *d_power, float *d_bpart, void *stream);
extern "C" int bfk_beamform_shared(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag,
                                   const float *d_wscale, const float *d_scale, uint8_t *d_out,
                                   float *d_power, float *d_bpart, int in_order, void *stream);
extern "C" int bfk_beamform_shared8(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag,
                                   const float *d_wscale, const float *d_scale, uint8_t *d_out,
                                   float *d_power, float *d_bpart, void *stream);

extern "C" int bfk_beamform_spread(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag, const float *d_wscale,
                                   const float *d_scale, uint8_t *d_out, float *d_power, float *d_bpart, float *d_beam_power, void *d_psum,
                                   int nbw, int pol_outer, void *stream);

extern "C" int bfk_beamform_packed(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag, const float *d_wscale,
                                   const float *d_scale, uint8_t *d_out, float *d_power, float *d_bpart, void *d_packed,
                                   void *stream);
// beam sets of `live` beam tiles, and the waves that share a beam tile in one
extern "C" int bfk_packed_sets(int live);
extern "C" int bfk_packed_split(int live, int set);
extern "C" int bfk_classic_beams(int variant, int nkc);

// Spread tiles or the plan's variant (bf_launch.h), by the times below in us,
// measured on blocks of 8 to 384 channels, 64 to 4096 samples and 20 to 1024
// beams.
//   spread: one workgroup per CU, t0 + t1 per 32-beam tile (FP6 three-part 13 %
//     more), in rounds of 256; the beam tiles are dealt evenly to the sets.
//   the variants: the 256-, 128- or 64-beam tiles of up to 64 antennas run two
//     workgroups a CU (t1 with one each at most, t2 once most have two, per512 in
//     the steady state), the 8-wave tiles of more antennas one (per round of 256).
// A block alone takes `alone`; where several streams have blocks in flight (three
// were measured), a pass takes `among`: a third of that latency, or its share of
// the chip.  Spread tiles run where neither is longer, with the set size that
// makes their product least.  E.g. 56 channels x 512 samples -> 256 beams of 64
// antennas FP16: alone 41 -> 18 us, among others 16 -> 12.5; 100 antennas FP8: 55
// -> 26 alone but 19 -> 22 among others, left alone.  Past one round, fine weights
// of more than 64 antennas no longer share their rows in an XCD's L2 (825 tiles,
// 300 beams FP6 three-part: 538 -> 395 alone, 500 -> 690 among others).
struct TileTimes {
  float t1, t2, per512;
};
struct TileCost {
  float alone, among;
};
static TileCost variant_cost(const bfk_dims *d) {
  const int k = d->nkc == 1 ? 0 : d->nkc == 2 ? 1 : 2;
  const bool group = d->wmode == 0;
  int beams = bfk_classic_beams(d->variant, d->nkc);
  if (d->variant == BFK_VAR_SHARED_256) beams = 256;
  const long n = (long)(d->nsamp / TCU) * d->ngroup * ((d->nbeam + beams - 1) / beams);
  if (beams == 256 && d->nkc > 1) {
    static const float per[2][2][4] = {{{68, 57, 49.5f, 70}, {66, 57, 48.5f, 67}}, {{150, 133, 126, 0}, {143, 123, 110, 0}}};
    const float p = per[k - 1][group][d->prec], alone = (float)((n + 255) / 256) * p;
    return {alone, fmaxf(alone / 3, (float)n * p / 256)};
  }
  static const TileTimes shared[2][4] = {{{38, 53, 58}, {33, 49, 52}, {31, 38, 43}, {39, 52, 59}},
                                         {{36, 50, 54}, {28, 43, 44}, {22, 34, 35}, {26, 42, 46}}};
  static const TileTimes half[3] = {{22, 42, 37}, {48, 87, 70}, {133, 256, 185}};      // 128 beams
  static const TileTimes quarter[3] = {{17, 33, 26}, {35, 67, 45}, {106, 222, 137}};   // 64 beams
  TileTimes t = beams == 256 ? shared[group][d->prec] : beams == 128 ? half[k] : quarter[k];
  if (beams == 256 && d->nbeam <= 128) {            // one beam tile a wave (64 x 384 x 2048 -> 100, FP6: 112 -> 85)
    t.t1 *= 0.7f;
    t.t2 *= 0.7f;
    t.per512 *= 0.7f;
  }
  const float steady = (float)n * t.per512 / 512;
  const float alone = n <= 256   ? t.t1
                      : n <= 512 ? beams == 256 ? t.t2 : fminf(t.t2, t.t1 + (t.t2 - t.t1) * (float)(n - 256) / 192)
                                 : fmaxf(t.t2, steady);
  return {alone, fmaxf(alone / 3, steady)};
}
// Whether spread tiles of nbw beam tiles a workgroup, of modelled times s, hold up
// against the variant's v: with both corrected by what 1250 blocks that the model gave
// spread tiles took, neither may be longer (among others 3 % less).  By real over
// modelled times, to 9-15 %: the antennas of the last chunk, the share of the CUs in
// the first round and, for the variant, antennas outermost in it, for spread tiles
// 8-sample bins.  Without it the variant was over 5 % faster for 15 of them alone and
// for 64 among others (193 antennas x 40 channels x 512 samples -> 325 beams FP8, fine
// weights, 98/35 us against 95/52); with it for none and 14 of 1098, and of 450 other
// blocks for none and 10, which take about half the time alone.  (Below 9 us blocks
// among others are bound by their launches.)
static bool spread_holds(const bfk_dims *d, int nbw, const TileCost &s, const TileCost &v) {
  static const float variant[3][2][4] = {{{.95f, .04f, -.05f, .06f}, {1.18f, .19f, -.42f, .06f}},
                                         {{.78f, .08f, .08f, .12f}, {.88f, .13f, -.01f, .13f}},
                                         {{.66f, .07f, .16f, .2f}, {.81f, .39f, .06f, .29f}}};
  static const float spread[3][2][4] = {{{1.2f, .05f, -.05f, .13f}, {1.08f, .23f, -.11f, .1f}},
                                        {{1.06f, .18f, -.05f, .11f}, {.84f, .22f, .14f, .08f}},
                                        {{.75f, .22f, .25f, .2f}, {.86f, .29f, .11f, .18f}}};
  const int k = d->nkc == 1 ? 0 : d->nkc == 2 ? 1 : 2;
  const int beams = d->variant == BFK_VAR_SHARED_256 ? 256 : bfk_classic_beams(d->variant, d->nkc);
  const float tiles = (float)(d->nsamp / TCU) * (float)d->ngroup, na = (float)d->nant / (float)d->nant_pad - .75f;
  const float fv = fminf(tiles * (float)((d->nbeam + beams - 1) / beams) / 256, 1.f);
  const float fs = fminf(tiles * (float)(((d->nbeam + 31) / 32 + nbw - 1) / nbw) / 256, 1.f);
  auto real = [&](const float(&c)[4], float model, float fill, float last) {
    return model * (c[0] + c[1] * na + c[2] * fill + c[3] * last);
  };
  const float ov = d->order == 0 ? fv : 0.f, bins = d->tavg == 8 ? 1.f : 0.f;
  if (real(spread[k][0], s.alone, fs, bins) > real(variant[k][0], v.alone, fv, ov)) return false;
  const float among = s.among > 9 ? real(spread[k][1], s.among, fs, bins) : s.among;
  const float most = v.among > 9 ? real(variant[k][1], v.among, fv, ov) : v.among;
  return fmaxf(among, 6.6f) * 1.03f <= fmaxf(most, 6.6f * 1.03f);
}
static int spread_tiles(const bfk_dims *d, TileCost *cost) {
  static const float t0[3][2] = {{4.5f, 4.6f}, {5.5f, 5.f}, {17.5f, 16.f}}, t1[3][2] = {{3.9f, 3.6f}, {7.6f, 7.4f}, {15.f, 14.f}};
  const int k = d->nkc == 1 ? 0 : d->nkc == 2 ? 1 : 2;
  const bool group = d->wmode == 0;
  const long ntile = (long)(d->nsamp / TCU) * d->ngroup;
  const int live = (d->nbeam + 31) / 32;
  const TileCost v = variant_cost(d);
  float best = 0.f;
  int tiles = 0;
  TileCost pick = {0.f, 0.f};
  for (int nset = (live + 15) / 16; nset <= live; nset++) {
    const int nbw = (live + nset - 1) / nset;
    const long wgs = ntile * nset, rounds = (wgs + 255) / 256;
    if (!group && rounds > (d->nkc == 1 ? 2 : 1)) break;
    const float wg = t0[k][group] + nbw * t1[k][group] * (d->prec == 3 ? 1.13f : 1.f);
    // (blocks in flight together contend for the weights' bytes)
    const float share = group || d->nkc == 1 ? 1.05f : d->prec == 3 ? 1.5f : 1.25f;
    const float alone = rounds * wg, among = fmaxf(alone / 3, (float)wgs * wg / 256 * share);
    if (alone * 1.08f > v.alone || among > v.among) continue;
    if (!tiles || alone * among < best) {
      best = alone * among;
      tiles = nbw;
      pick = {alone, among};
    }
  }
  if (!tiles || !spread_holds(d, tiles, pick, v)) return 0;
  *cost = pick;
  return tiles;
}
extern "C" int bfk_spread_tiles(const bfk_dims *d) {
  TileCost c;
  return spread_tiles(d, &c);
}

// Whether a block of more than 64 antennas is repacked (bf_packed.hip), by the us
// of its workgroups of 8, 4 and 2 beam tiles (one per CU) and the repacking at 5.1
// TB/s, against the spread tiles or the variant: where the product of the two
// times (see above) is 5 % less and neither is more than 5 % longer.  256 antennas
// gain at whole sets of eight beam tiles (256 channels x 4096 samples -> 256 beams,
// fine weights, alone and among others: FP8 1096/1211 -> 947/920, FP6 1058/1253 ->
// 830/793), 128 antennas only with fine weights (FP6 three-part 582/751 ->
// 558/536; FP8 489/542 -> 492/452; group weights, which stay in the L2, 466/457 and
// 481/439), two beam tiles hardly (256 antennas, group weights FP8: 98/101 and
// 131/117).
static TileCost packed_cost(const bfk_dims *d) {
  static const float per[2][2][3][4] = {
      {{{112, 92, 74, 110}, {64, 53, 47, 70}, {56, 32, 29, 43}}, {{110, 88, 70, 100}, {62, 48, 41, 60}, {55, 30, 27, 39}}},
      {{{222, 182, 152, 0}, {135, 117, 104, 0}, {110, 70, 66, 0}}, {{214, 175, 138, 0}, {130, 104, 90, 0}, {115, 68, 62, 0}}}};
  const float(&p)[3][4] = per[d->nkc == 4][d->wmode == 0];
  // (an XCD with the most tiles of each set, on its 32 CUs)
  const long tiles = ((long)((d->nsamp + 2 * TCU - 1) / (2 * TCU)) * d->ngroup + 7) / 8;
  const int live = (d->nbeam + 31) / 32, nset = bfk_packed_sets(live);
  // the sets one after another, each workgroup on the CU that is free first: up to
  // 8 times at which CUs become free (more are taken as the last)
  struct {
    float at;
    long n;
  } cu[9] = {{0.f, 32}};
  int ncu = 1;
  float sum = 0.f, end = 0.f;
  for (int i = 0; i < nset; i++) {
    const int split = bfk_packed_split(live, i);
    const float t = p[split == 1 ? 0 : split == 2 ? 1 : 2][d->prec] *
                    (split == 1 && live < 8 * i + 8 ? 0.28f + 0.09f * (float)(live - 8 * i) : 1.f);
    sum += t;
    for (long n = tiles; n > 0;) {
      if (ncu == 1 && n >= 32) {
        cu[0].at += t * (float)(n / 32);
        end = fmaxf(end, cu[0].at);
        n %= 32;
        continue;
      }
      const long k = n < cu[0].n ? n : cu[0].n;
      const float at = cu[0].at + t;
      end = fmaxf(end, at);
      n -= k;
      cu[0].n -= k;
      if (!cu[0].n) {
        ncu--;
        for (int j = 0; j < ncu; j++) cu[j] = cu[j + 1];
      }
      int j = ncu;
      for (; j > 0 && cu[j - 1].at > at; j--) cu[j] = cu[j - 1];
      if (j > 0 && (ncu == 8 || cu[j - 1].at == at)) {
        cu[j - 1].n += k;
        for (; j < ncu; j++) cu[j] = cu[j + 1];
      } else {
        cu[j].at = at;
        cu[j].n = k;
        ncu++;
      }
    }
  }
  const float pack = 2.f * d->nsamp * d->nchan * (d->nant + d->nant_pad) / 5.1e6f, share = sum * (float)tiles / 32;
  const float alone = pack + 5 + end;
  return {alone, fmaxf(alone / 3, share + pack)};
}
static bool packed_holds(const bfk_dims *d, float less) {
  if (d->pinned || !bfk_packed_bytes(d) || !bfk_variant_supported(d, d->variant)) return false;
  // (256-beam tiles: fine weights contend for the L2 among others; zeros take the
  // place of missing beam tiles, and five of eight this part of the time)
  static const float contend[4] = {1.05f, 1.1f, 1.25f, 1.27f};
  static const float five[2][4] = {{0.87f, 0.9f, 0.85f, 0.95f}, {0.67f, 0.74f, 0.81f, 0.8f}};
  TileCost v = variant_cost(d);
  if (d->variant == BFK_VAR_SHARED_256) {
    const bool group = d->wmode == 0;
    const int live = (d->nbeam + 31) / 32, nset = (live + 7) / 8;
    const float part = 1.f - (1.f - five[group][d->prec]) / 3 * (float)(8 * nset - live) / (float)nset;
    v.alone *= part;
    v.among *= part * (group ? 1.f : contend[d->prec]);
  }
  v.alone *= less;
  v.among *= less;
  spread_tiles(d, &v);
  const TileCost k = packed_cost(d);
  return k.alone < 1.05f * v.alone && k.among < 1.05f * v.among && k.alone * k.among < 0.95f * v.alone * v.among;
}
extern "C" int bfk_use_packed(const bfk_dims *d) {
  return !d->pinned && bfk_packed_bytes(d) && bfk_variant_supported(d, d->variant);
}
// With groups outermost eight antennas' chunks are together and the variant wastes less
// of its lines: 256-beam tiles take 0.9 of their times above, classic ones 0.78.  Of 380
// blocks that the times above chose, with the chip's 256 CUs for an XCD's 32, 13 were 5
// to 56 % slower repacked, alone or among others, all of this order (67 antennas x 120
// channels x 1536 samples -> 100 beams in FP8 56/37 and 72/42 us, 195 x 304 x 1600 -> 58
// 206/188 and 249/220; 119 x 112 x 704 -> 706 in FP6, 33 workgroups on an XCD's CUs,
// 92/80 and 143/76).  None of the 354 left is, and the others were 1.02 and 0.88.
extern "C" int bfk_pack_block(const bfk_dims *d) {
  return packed_holds(d, d->order == 0 ? 1.f : d->variant == BFK_VAR_SHARED_256 ? 0.9f : 0.78f);
}

extern "C" int bfk_variant_supported(const bfk_dims *d, int v) {
  if (d->nant_pad != 64 * d->nkc || (d->nkc != 1 && d->nkc != 2 && d->nkc != 4)) return 0;
  if (d->prec == 3 && d->nkc > 2) return 0;          // three-part FP6: up to 128 antennas
  if (d->prec >= 2) return v == BFK_VAR_SHARED_256;   // FP6: shared tiles only
  if (v == BFK_VAR_SHARED_256) return 1;       // 4-wave tiles to 64 antennas, 8-wave above
  return bfk_classic_beams(v, d->nkc) > 0;
}

// FP8 blocks of 65 to 128 beams that the 128-beam classic tiles would take run shared
// tiles of one beam tile a wave, in the same order (64 antennas x 384 channels x 2048
// samples -> 100 beams, fine weights 97/106 -> 92/99 us alone and among other blocks;
// x 4096 -> 128, group weights 188/206 -> 176/190; FP16 103/108 with either).
static bool short_shared(const bfk_dims *d) {
  return !d->pinned && d->variant == BFK_VAR_CLASSIC_128S && d->prec == 1 && d->nkc == 1 && d->nbeam > 64 && d->nbeam <= 128;
}
extern "C" int bfk_unset_differs(const bfk_dims *d) { return bfk_spread_tiles(d) || short_shared(d); }

extern "C" int bfk_beamform(const bfk_dims *d, const uint8_t *d_in, const void *d_wfrag,
                            const float *d_wscale, const float *d_scale, uint8_t *d_out,
                            float *d_power, float *d_bpart, float *d_beam_power, void *d_psum,
                            int *summed, void *d_packed, void *stream) {
  *summed = 0;
  // buffer offsets are 32-bit
  if ((size_t)d->npkt * d->nant * d->nchan * 4 > 0x7fffffffu || bfk_wfrag_bytes(d) > 0x7fffffffu) {
    bfk_set_error("bfk_beamform: block or weights above 2 GiB");
    return -1;
  }
  if (!bfk_variant_supported(d, d->variant)) {
    bfk_set_error("bfk_beamform: variant %d cannot run this shape (nant_pad %d)", d->variant, d->nant_pad);
    return -1;
  }
  if (d_packed)
    return bfk_beamform_packed(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, d_packed, stream);
  if (const int nbw = d->pinned ? 0 : bfk_spread_tiles(d)) {
    // the order in which the variant adds the (channel, pol) powers: the shared
    // tiles take group weights pol-outer, except the two-part splits from 32
    // samples a bin on (bf_shared.hip)
    const int pol_outer = d->variant == BFK_VAR_SHARED_256 && d->nkc == 1 && d->wmode == 0 &&
                          !((d->prec == 1 || d->prec == 2) && d->tavg >= 32);
    if (!d_psum || !bfk_psum_bytes(d)) d_beam_power = NULL;
    *summed = d_beam_power != NULL;
    return bfk_beamform_spread(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, d_beam_power, d_psum,
                               nbw, pol_outer, stream);
  }
  if (short_shared(d))
    return bfk_beamform_shared(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, 1, stream);
  if (d->variant == BFK_VAR_SHARED_256)
    return d->nkc == 1 ? bfk_beamform_shared(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, 0, stream)
                       : bfk_beamform_shared8(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, stream);
  return bfk_beamform_classic(d, d_in, d_wfrag, d_wscale, d_scale, d_out, d_power, d_bpart, stream);
}
