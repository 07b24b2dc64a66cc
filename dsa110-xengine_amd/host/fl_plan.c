/*
 * fl_plan.c -- the flagger's device entry points and the plan that runs one
 * block of the flagger loop (C, HIP runtime C API).
 *
 * Replaces gpu_flagger.cu:1233-1460.  Per block the reference launches
 * scaley, calc_spectrum, calc_varspec, calc_spectrum (its "maxspec"),
 * calc_ppspec, flag, make_ts and flagts -- five full reads of the 1 GiB block
 * and two writes -- with blocking copies of every statistic between them.
 * The plan runs two passes over the block -- one that only reads it, for the
 * statistics of the scaled block, and one that scales, flags and sums its rows
 * in place -- plus flagts on the masked rows.  The masks are made on the device
 * between them; the host only sums the spectrum (the total power, in the
 * reference's order) while the second pass runs.
 */
#include <hip/hip_runtime_api.h>
#include <math.h>
#include <stdlib.h>
#include <string.h>

#include "../csrc/bf_launch.h"
#include "bf_internal.h"
#include "dsaxfl.h"

int flk_stats(const uint8_t *d_data, uint8_t *d_scaled, const float *d_spec0, const float *d_var0,
              const float *d_spec_in, float *d_spec, float *d_var, float *d_max, float *d_pp, int nb, int nt,
              int nc, void *stream);
int flk_stats_scaled(const uint8_t *d_data, const float *d_spec0, const float *d_var0, float *d_spec, float *d_var,
                     float *d_pp, int nb, int nt, int nc, void *stream);
size_t flk_masks_big_bytes(int nb, int nc);
int flk_masks(const float *d_spec, const float *d_var, const float *d_pp, float *d_big, uint8_t *d_mask, int *h_nmask,
              float *h_spec, double *d_bsum, float *d_bpwr, float thresh, const int *perm, int nperm, int nb, int nc,
              void *stream);
size_t flk_part_bytes(int nb, int nt, int nc);
int flk_apply(uint8_t *d_data, const float *d_spec0, const float *d_var0, const uint8_t *d_mask, const float *d_bpwr,
              uint16_t *d_part, const double *d_bsum, int *d_ran, int *h_ran, float prev, float jump, int force, int nb,
              int nt, int nc, void *stream);
int flk_tsmask_flagts(uint8_t *d_data, const uint16_t *d_part, float *d_ts, int *d_idx, int *d_nts, int *h_nts,
                      const int *d_ran, const float *d_bpwr, float thr, int nb, int nt, int nc, void *stream);
int flk_flag_ts(uint8_t *d_data, const uint8_t *d_mask, const float *d_bpwr, float *d_ts, int nb, int nt, int nc,
                void *stream);
int flk_flagts(uint8_t *d_data, const int *d_midx, int n, const float *d_bpwr, int nb, int nt, int nc,
               void *stream);
int flk_flag_cols(uint8_t *d_data, const int *d_midx, int n, const float *d_bpwr, int nb, int nt, int nc,
                  void *stream);
int flk_sumpulse(uint8_t *d_data, const float *d_summand, size_t n, void *stream);
int flk_genrand(uint8_t *d_rep, size_t n, uint32_t seed, void *stream);
int flk_noise(uint8_t *d_data, const uint8_t *d_rep, int nb, int nt, int nc, void *stream);
int flk_fix_zspec(float *d_s0, float *d_v0, int nbc, int naver, void *stream);

/* launcher codes: -1 a shape or argument the kernels do not take, -3 a HIP
   launch error */
#define KCALL(expr)                                                                    \
  do {                                                                                 \
    dsaxbf_clear_error();                                                              \
    int rc_ = (expr);                                                                  \
    if (rc_) return dsaxbf_fail(rc_ == -3 ? DSAXBF_EHIP : DSAXBF_EINVAL, "%s", bfk_last_error()); \
  } while (0)

static int nonnull(const void *p) { return p != NULL; }

/* ---- device entry points ------------------------------------------------ */

int dsaxfl_stats(const uint8_t *d_data, int nb, int nt, int nc, const float *d_spec_in, float *d_spec,
                 float *d_var, float *d_max, float *d_pp, void *stream) {
  if (!nonnull(d_data)) return dsaxbf_fail(DSAXBF_EINVAL, "NULL block");
  KCALL(flk_stats(d_data, NULL, NULL, NULL, d_spec_in, d_spec, d_var, d_max, d_pp, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_scaley(uint8_t *d_data, int nb, int nt, int nc, const float *d_spec0, const float *d_var0,
                  float *d_spec, float *d_var, float *d_max, float *d_pp, void *stream) {
  if (!d_data || !d_spec0 || !d_var0) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  KCALL(flk_stats(d_data, d_data, d_spec0, d_var0, NULL, d_spec, d_var, d_max, d_pp, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_make_ts(const uint8_t *d_data, int nb, int nt, int nc, float *d_ts, void *stream) {
  if (!d_data || !d_ts) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  /* no mask: the block is only read */
  KCALL(flk_flag_ts((uint8_t *)d_data, NULL, NULL, d_ts, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_flag(uint8_t *d_data, int nb, int nt, int nc, const int *d_midx, int n_mask, const float *d_bpwr,
                void *stream) {
  if (!d_data || (n_mask > 0 && (!d_midx || !d_bpwr))) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  if (n_mask < 0 || (long)n_mask > (long)nb * nc) return dsaxbf_fail(DSAXBF_EINVAL, "n_mask=%d", n_mask);
  KCALL(flk_flag_cols(d_data, d_midx, n_mask, d_bpwr, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_flag_mask(uint8_t *d_data, int nb, int nt, int nc, const uint8_t *d_mask, const float *d_bpwr,
                     float *d_ts, void *stream) {
  if (!d_data || !d_mask || !d_bpwr) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  KCALL(flk_flag_ts(d_data, d_mask, d_bpwr, d_ts, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_flagts(uint8_t *d_data, int nb, int nt, int nc, const int *d_midx, int n_mask, const float *d_bpwr,
                  void *stream) {
  if (!d_data || (n_mask > 0 && (!d_midx || !d_bpwr))) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  if (n_mask < 0 || (long)n_mask > (long)nb * nt) return dsaxbf_fail(DSAXBF_EINVAL, "n_mask=%d", n_mask);
  KCALL(flk_flagts(d_data, d_midx, n_mask, d_bpwr, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_sumpulse(uint8_t *d_data, size_t n, const float *d_summand, void *stream) {
  if (!d_data || !d_summand) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  KCALL(flk_sumpulse(d_data, d_summand, n, stream));
  return DSAXBF_OK;
}

int dsaxfl_genrand(uint8_t *d_repval, size_t n, uint32_t seed, void *stream) {
  if (!d_repval) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  KCALL(flk_genrand(d_repval, n, seed, stream));
  return DSAXBF_OK;
}

int dsaxfl_noise(uint8_t *d_data, int nb, int nt, int nc, const uint8_t *d_repval, void *stream) {
  if (!d_data || !d_repval) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  KCALL(flk_noise(d_data, d_repval, nb, nt, nc, stream));
  return DSAXBF_OK;
}

int dsaxfl_fix_zspec(float *d_s0, float *d_v0, int nbc, int naver, void *stream) {
  if (!d_s0 || !d_v0) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  KCALL(flk_fix_zspec(d_s0, d_v0, nbc, naver, stream));
  return DSAXBF_OK;
}

/* ---- plan ------------------------------------------------------------------ */

struct dsaxfl_plan {
  dsaxfl_config cfg;
  hipStream_t stream;
  hipEvent_t masked;               /* the masks and the host's spectrum are there */
  float *d_spec0, *d_var0, *d_spec, *d_var, *d_pp, *d_ts, *d_bpwr, *d_big;
  uint8_t *d_mask, *d_repval;
  uint16_t *d_part;                /* row sums of each slab of channels */
  double *d_bsum;                  /* per-beam sums of the spectrum, then d_nts and d_ran */
  int *d_tsidx, *d_nts, *d_ran;
  float *h_spec, *h_var;           /* pinned; after h_spec's values */
  int *h_nmask, *h_nts, *h_ran;    /* those that the kernels write */
  float prev_tpwr;
  int have_ref;
};

void dsaxfl_config_default(dsaxfl_config *c) {
  if (!c) return;
  memset(c, 0, sizeof(*c));
  c->nbeam = DSAXFL_NBEAMS;
  c->ntime = DSAXFL_NTIMES;
  c->nchan = DSAXFL_NCHAN;
  c->thresh = 5.0f;
  c->tsthresh = 10.0f;
  c->mod_thresh = 0.0005f;
  c->nperm = 1;
  c->perm[0] = 10;
  c->seed = 1;
}

void dsaxfl_destroy(dsaxfl_plan *p) {
  if (!p) return;
  hipSetDevice(p->cfg.device);
  if (p->stream) hipStreamSynchronize(p->stream);
  hipFree(p->d_spec0);
  hipFree(p->d_var0);
  hipFree(p->d_spec);
  hipFree(p->d_var);
  hipFree(p->d_pp);
  hipFree(p->d_ts);
  hipFree(p->d_bpwr);
  hipFree(p->d_mask);
  hipFree(p->d_repval);
  hipFree(p->d_tsidx);
  hipFree(p->d_big);
  hipFree(p->d_part);
  hipFree(p->d_bsum);
  hipHostFree(p->h_spec);
  hipHostFree(p->h_var);
  if (p->masked) hipEventDestroy(p->masked);
  if (p->stream) hipStreamDestroy(p->stream);
  free(p);
}

void *dsaxfl_get_stream(dsaxfl_plan *p) { return p ? (void *)p->stream : NULL; }

int dsaxfl_create(dsaxfl_plan **out, const dsaxfl_config *cfg) {
  dsaxbf_clear_error();
  if (!out || !cfg) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  *out = NULL;
  const int nb = cfg->nbeam, nt = cfg->ntime, nc = cfg->nchan;
  if (nb < 1 || nt < 4096 || nt % 4096 || nc % 16 || nc <= 2 * DSAXFL_ZERO_CHANNELS + 21 ||
      (long)nb * nt * nc > (1L << 34) || (long)nt * nc >= (1L << 31))
    return dsaxbf_fail(DSAXBF_EINVAL,
                       "shape %d x %d x %d: ntime a multiple of 4096, nchan a multiple of 16 above 277", nb, nt,
                       nc);
  if (cfg->nperm < 0 || cfg->nperm > 64) return dsaxbf_fail(DSAXBF_EINVAL, "nperm=%d outside 0..64", cfg->nperm);
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || cfg->device < 0 || cfg->device >= ndev)
    return dsaxbf_fail(DSAXBF_ENODEV, "no HIP device %d (found %d)", cfg->device, ndev);
  if (hipSetDevice(cfg->device) != hipSuccess) return dsaxbf_fail(DSAXBF_EHIP, "hipSetDevice");
  dsaxfl_plan *p = calloc(1, sizeof(*p));
  if (!p) return dsaxbf_fail(DSAXBF_ENOMEM, "host allocation failed");
  p->cfg = *cfg;
  const size_t nbc = (size_t)nb * nc, nbt = (size_t)nb * nt;
  hipError_t e = hipStreamCreateWithFlags(&p->stream, hipStreamNonBlocking);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_spec0, nbc * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_var0, nbc * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_spec, nbc * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_var, nbc * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_pp, nbc * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_ts, nbt * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_bpwr, (size_t)nb * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_mask, nbc);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_repval, (size_t)nt * nc);
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_tsidx, nbt * 4);
  if (e == hipSuccess) e = hipHostMalloc((void **)&p->h_spec, nbc * 4 + (2 * (size_t)nb + 1) * sizeof(int), 0);
  if (e == hipSuccess) e = hipHostMalloc((void **)&p->h_var, nbc * 4, 0);
  if (e == hipSuccess && flk_masks_big_bytes(nb, nc)) e = hipMalloc((void **)&p->d_big, flk_masks_big_bytes(nb, nc));
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_part, flk_part_bytes(nb, nt, nc));
  if (e == hipSuccess) e = hipMalloc((void **)&p->d_bsum, nb * sizeof(double) + (nb + 1) * sizeof(int));
  if (e == hipSuccess) e = hipEventCreateWithFlags(&p->masked, hipEventDisableTiming);
  if (e != hipSuccess) {
    dsaxfl_destroy(p);
    return dsaxbf_fail(DSAXBF_ENOMEM, "flagger allocation failed: %s", hipGetErrorString(e));
  }
  p->d_nts = (int *)(p->d_bsum + nb);
  p->d_ran = p->d_nts + nb;
  p->h_nmask = (int *)(p->h_spec + nbc);
  p->h_nts = p->h_nmask + nb;
  p->h_ran = p->h_nts + nb;
  for (int b = 0; b < nb; b++) p->h_spec[b] = 1.f;       /* bpwr, gpu_flagger.cu:1234 */
  e = hipMemcpyAsync(p->d_bpwr, p->h_spec, (size_t)nb * 4, hipMemcpyHostToDevice, p->stream);
  int rc = e == hipSuccess ? flk_genrand(p->d_repval, (size_t)nt * nc, cfg->seed, p->stream) : -1;
  if (rc == 0) e = hipStreamSynchronize(p->stream);
  if (e != hipSuccess || rc) {
    dsaxfl_destroy(p);
    return dsaxbf_fail(DSAXBF_EHIP, "flagger set-up: %s", e != hipSuccess ? hipGetErrorString(e) : bfk_last_error());
  }
  *out = p;
  return DSAXBF_OK;
}

int dsaxfl_set_reference(dsaxfl_plan *p, const float *h_spec0, const float *h_var0) {
  if (!p || !h_spec0 || !h_var0) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  const size_t n = (size_t)p->cfg.nbeam * p->cfg.nchan * 4;
  hipError_t e = hipMemcpyAsync(p->d_spec0, h_spec0, n, hipMemcpyHostToDevice, p->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(p->d_var0, h_var0, n, hipMemcpyHostToDevice, p->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(p->stream);
  if (e != hipSuccess) return dsaxbf_fail(DSAXBF_EHIP, "reference upload: %s", hipGetErrorString(e));
  p->have_ref = 1;
  return DSAXBF_OK;
}

int dsaxfl_get_reference(dsaxfl_plan *p, float *h_spec0, float *h_var0) {
  if (!p || !h_spec0 || !h_var0) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  if (!p->have_ref) return dsaxbf_fail(DSAXBF_ESTATE, "no reference spectra yet");
  const size_t n = (size_t)p->cfg.nbeam * p->cfg.nchan * 4;
  hipError_t e = hipMemcpyAsync(h_spec0, p->d_spec0, n, hipMemcpyDeviceToHost, p->stream);
  if (e == hipSuccess) e = hipMemcpyAsync(h_var0, p->d_var0, n, hipMemcpyDeviceToHost, p->stream);
  if (e == hipSuccess) e = hipStreamSynchronize(p->stream);
  if (e != hipSuccess) return dsaxbf_fail(DSAXBF_EHIP, "reference download: %s", hipGetErrorString(e));
  return DSAXBF_OK;
}

int dsaxfl_calibrate(dsaxfl_plan *p, const uint8_t *const *d_blocks, int naver) {
  dsaxbf_clear_error();
  if (!p || !d_blocks) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  if (naver < 1 || naver > 16) return dsaxbf_fail(DSAXBF_EINVAL, "naver=%d outside 1..16", naver);
  if (hipSetDevice(p->cfg.device) != hipSuccess) return dsaxbf_fail(DSAXBF_EHIP, "hipSetDevice");
  const int nb = p->cfg.nbeam, nt = p->cfg.ntime, nc = p->cfg.nchan;
  const size_t nbc = (size_t)nb * nc;
  float *d_s = NULL, *d_v = NULL;
  hipError_t e = hipMalloc((void **)&d_s, nbc * naver * 4);
  if (e == hipSuccess) e = hipMalloc((void **)&d_v, nbc * naver * 4);
  int rc = DSAXBF_OK;
  if (e != hipSuccess) rc = dsaxbf_fail(DSAXBF_ENOMEM, "calibration buffers: %s", hipGetErrorString(e));
  for (int k = 0; k < naver && rc == DSAXBF_OK; k++) {
    if (!d_blocks[k]) rc = dsaxbf_fail(DSAXBF_EINVAL, "block %d is NULL", k);
    else if (flk_stats(d_blocks[k], NULL, NULL, NULL, NULL, d_s + k * nbc, d_v + k * nbc, NULL, NULL, nb, nt, nc,
                       p->stream))
      rc = dsaxbf_fail(DSAXBF_EHIP, "%s", bfk_last_error());
  }
  if (rc == DSAXBF_OK && naver > 1 && flk_fix_zspec(d_s, d_v, (int)nbc, naver, p->stream))
    rc = dsaxbf_fail(DSAXBF_EHIP, "%s", bfk_last_error());
  if (rc == DSAXBF_OK) {
    e = hipMemcpyAsync(p->h_spec, d_s, nbc * 4, hipMemcpyDeviceToHost, p->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(p->h_var, d_v, nbc * 4, hipMemcpyDeviceToHost, p->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(p->stream);
    if (e != hipSuccess) rc = dsaxbf_fail(DSAXBF_EHIP, "calibration: %s", hipGetErrorString(e));
  }
  hipFree(d_s);
  hipFree(d_v);
  if (rc) return rc;
  dsaxfl_median_calc(p->h_spec, nb, nc);
  dsaxfl_median_calc(p->h_var, nb, nc);
  rc = dsaxfl_set_reference(p, p->h_spec, p->h_var);
  p->prev_tpwr = 0.f;
  return rc;
}

int dsaxfl_set_total_power(dsaxfl_plan *p, float prev_tpwr) {
  if (!p) return dsaxbf_fail(DSAXBF_EINVAL, "NULL plan");
  p->prev_tpwr = prev_tpwr;
  return DSAXBF_OK;
}

#define HCALL(expr, what)                                                                 \
  do {                                                                                    \
    hipError_t e_ = (expr);                                                               \
    if (e_ != hipSuccess) return dsaxbf_fail(DSAXBF_EHIP, "%s: %s", what, hipGetErrorString(e_)); \
  } while (0)
#define FCALL(expr)                                                                     \
  do {                                                                                  \
    int rc_ = (expr);                                                                   \
    if (rc_) return dsaxbf_fail(rc_ == -3 ? DSAXBF_EHIP : DSAXBF_EINVAL, "%s", bfk_last_error()); \
  } while (0)

/* The second pass and the time masks; force: whatever the device makes of the
 * total power. */
static int apply(dsaxfl_plan *p, uint8_t *d_data, int force) {
  const dsaxfl_config *c = &p->cfg;
  const int nb = c->nbeam, nt = c->ntime, nc = c->nchan;
  uint16_t *d_part = c->tsflag ? p->d_part : NULL;
  FCALL(flk_apply(d_data, p->d_spec0, p->d_var0, p->d_mask, p->d_bpwr, d_part, p->d_bsum, p->d_ran, p->h_ran,
                  p->prev_tpwr, c->mod_thresh, force, nb, nt, nc, p->stream));
  if (d_part)
    FCALL(flk_tsmask_flagts(d_data, d_part, p->d_ts, p->d_tsidx, p->d_nts, p->h_nts, p->d_ran, p->d_bpwr, c->tsthresh,
                            nb, nt, nc, p->stream));
  return DSAXBF_OK;
}

int dsaxfl_step(dsaxfl_plan *p, uint8_t *d_data, dsaxfl_step_info *info) {
  dsaxbf_clear_error();
  if (!p || !d_data) return dsaxbf_fail(DSAXBF_EINVAL, "NULL argument");
  if (!p->have_ref) return dsaxbf_fail(DSAXBF_ESTATE, "step before dsaxfl_set_reference / dsaxfl_calibrate");
  HCALL(hipSetDevice(p->cfg.device), "hipSetDevice");
  const dsaxfl_config *c = &p->cfg;
  const int nb = c->nbeam, nt = c->ntime, nc = c->nchan;
  const size_t nbc = (size_t)nb * nc;
  hipStream_t s = p->stream;
  int rc;
  /* spectrum, varspec and ppspec of the scaled block, which is not written yet */
  FCALL(flk_stats_scaled(d_data, p->d_spec0, p->d_var0, p->d_spec, p->d_var, p->d_pp, nb, nt, nc, s));
  /* channflag on spectrum - oldspec (oldspec is never updated from zero in
     the reference), on varspec at thresh + 0.5 and on its "maxspec" (a
     second calc_spectrum: the same mask again); simple_channflag on ppspec */
  FCALL(flk_masks(p->d_spec, p->d_var, p->d_pp, p->d_big, p->d_mask, p->h_nmask, p->h_spec, p->d_bsum,
                  c->pwr ? p->d_bpwr : NULL, c->thresh, c->perm, c->nperm, nb, nc, s));
  HCALL(hipEventRecord(p->masked, s), "masks");
  /* the rest of the step before its total power is known here: the device has
     a sum of its own to go by, and the block is replaced or the pass run after
     all where the sum in the reference's order says otherwise */
  if (c->mkrand) FCALL(flk_noise(d_data, p->d_repval, nb, nt, nc, s));
  else if ((rc = apply(p, d_data, 0))) return rc;
  HCALL(hipEventSynchronize(p->masked), "statistics");
  float tpwr = 0.f;
  for (size_t i = 0; i < nbc; i++) tpwr += p->h_spec[i];
  dsaxfl_step_info inf = {tpwr, 0, -1, -1};
  if (fabs(tpwr - p->prev_tpwr) / p->prev_tpwr >= c->mod_thresh) {
    inf.replaced = 1;
    if (!c->mkrand) FCALL(flk_noise(d_data, p->d_repval, nb, nt, nc, s));
    HCALL(hipStreamSynchronize(s), "flagger step");
  } else {
    if (c->mkrand && c->tsflag) {
      FCALL(flk_flag_ts(d_data, NULL, p->d_bpwr, p->d_ts, nb, nt, nc, s));
      FCALL(flk_tsmask_flagts(d_data, NULL, p->d_ts, p->d_tsidx, p->d_nts, p->h_nts, NULL, p->d_bpwr, c->tsthresh, nb,
                              nt, nc, s));
    }
    HCALL(hipStreamSynchronize(s), "flagger step");
    if (!c->mkrand && !*p->h_ran) {
      if ((rc = apply(p, d_data, 1))) return rc;
      HCALL(hipStreamSynchronize(s), "flagger step");
    }
    inf.n_mask = inf.n_tsmask = 0;
    for (int b = 0; b < nb; b++) {
      inf.n_mask += p->h_nmask[b];
      if (c->tsflag) inf.n_tsmask += p->h_nts[b];
    }
  }
  p->prev_tpwr = tpwr;
  if (info) *info = inf;
  return DSAXBF_OK;
}
