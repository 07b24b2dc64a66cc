"""The rules that pick a kernel for a shape, which the host evaluates: what they may
answer, over the ranges that the entry points take.  No GPU."""
import ctypes as C
import random

import pytest


def dims(cfg, pinned=0):
    """The library's bfk_dims (csrc/bf_launch.h) of a plan whose variant nobody picked."""
    pad = 64 if cfg.nant <= 64 else 128 if cfg.nant <= 128 else 256
    bpad = (cfg.nbeam + 255) // 256 * 256
    variant = 5 if cfg.nbeam > 128 or cfg.precision >= 2 else (2 if pad == 64 else 3) if cfg.nbeam > 64 else 4
    return (C.c_int * 21)(cfg.nant, pad, pad // 64, cfg.nchan, cfg.nchan // 8, cfg.npkt, 2 * cfg.npkt, cfg.nbeam, bpad, bpad // 32,
                          cfg.tavg, 2 * cfg.npkt // cfg.tavg, cfg.ncal, cfg.weight_mode, cfg.angle_mode, cfg.precision,
                          cfg.input_order, 0, variant, cfg.output_layout, pinned)


def psum_bytes(bf, cfg):
    f = bf.lib.bfk_psum_bytes
    f.restype = C.c_size_t
    return f(dims(cfg))


# Blocks that run spread tiles: antennas, channels, packets, beams, precision, fine weights, the
# 32-beam tiles that a workgroup takes, and whether the launch sums the beam powers itself.  Every
# precision and weight mode with one, two, three and more tiles, with and without the sums (which
# occur up to three), up to 64 antennas; with two and more at 65 to 128 and 129 to 256.
SPREAD = [
    (35, 184, 384, 11, 0, 0, 1, 0), (55, 144, 96, 11, 0, 0, 1, 1), (43, 32, 288, 365, 0, 0, 2, 0),
    (20, 64, 224, 111, 0, 0, 2, 1), (62, 88, 224, 267, 0, 0, 3, 0), (35, 80, 256, 70, 0, 0, 3, 1),
    (46, 184, 352, 158, 0, 0, 5, 0), (38, 184, 384, 1, 0, 1, 1, 0), (24, 72, 64, 233, 0, 1, 1, 1),
    (53, 96, 96, 354, 0, 1, 2, 0), (50, 120, 256, 60, 0, 1, 2, 1), (49, 112, 192, 134, 0, 1, 3, 0),
    (54, 128, 160, 71, 0, 1, 3, 1), (34, 168, 352, 299, 0, 1, 10, 0), (26, 184, 384, 20, 1, 0, 1, 0),
    (54, 32, 320, 158, 1, 0, 1, 1), (26, 160, 96, 177, 1, 0, 2, 0), (60, 184, 128, 56, 1, 0, 2, 1),
    (53, 64, 384, 90, 1, 0, 3, 0), (25, 160, 128, 89, 1, 0, 3, 1), (62, 40, 320, 194, 1, 0, 4, 0),
    (23, 184, 384, 16, 1, 1, 1, 0), (59, 32, 256, 31, 1, 1, 1, 1), (21, 72, 256, 133, 1, 1, 2, 0),
    (24, 184, 160, 46, 1, 1, 2, 1), (64, 72, 288, 188, 1, 1, 3, 0), (31, 120, 160, 90, 1, 1, 3, 1),
    (24, 80, 288, 299, 1, 1, 5, 0), (25, 192, 384, 7, 2, 0, 1, 0), (47, 56, 128, 15, 2, 0, 1, 1),
    (43, 40, 288, 190, 2, 0, 2, 0), (31, 88, 288, 47, 2, 0, 2, 1), (32, 72, 128, 287, 2, 0, 3, 0),
    (36, 136, 96, 150, 2, 0, 3, 1), (23, 48, 224, 231, 2, 0, 4, 0), (28, 192, 384, 19, 2, 1, 1, 0),
    (34, 16, 288, 69, 2, 1, 1, 1), (24, 160, 96, 170, 2, 1, 2, 0), (20, 120, 256, 43, 2, 1, 2, 1),
    (53, 176, 64, 284, 2, 1, 3, 0), (61, 48, 384, 81, 2, 1, 3, 1), (61, 104, 128, 281, 2, 1, 5, 0),
    (37, 184, 384, 25, 3, 0, 1, 0), (25, 72, 64, 74, 3, 0, 1, 1), (51, 144, 256, 33, 3, 0, 2, 0),
    (33, 88, 352, 34, 3, 0, 2, 1), (21, 24, 384, 283, 3, 0, 3, 0), (28, 56, 320, 70, 3, 0, 3, 1),
    (64, 120, 96, 200, 3, 0, 4, 0), (25, 192, 384, 29, 3, 1, 1, 0), (36, 80, 32, 75, 3, 1, 1, 1),
    (58, 64, 192, 164, 3, 1, 2, 0), (51, 56, 288, 102, 3, 1, 2, 1), (57, 120, 352, 75, 3, 1, 3, 0),
    (21, 96, 224, 70, 3, 1, 3, 1), (45, 192, 128, 103, 3, 1, 4, 0), (70, 32, 288, 232, 0, 0, 2, 0),
    (80, 184, 96, 219, 0, 0, 4, 0), (67, 96, 160, 145, 0, 1, 2, 0), (82, 120, 128, 383, 0, 1, 4, 0),
    (90, 144, 64, 356, 1, 0, 2, 0), (127, 176, 128, 319, 1, 0, 5, 0), (75, 176, 64, 199, 1, 1, 2, 0),
    (91, 80, 160, 220, 1, 1, 4, 0), (66, 144, 256, 52, 2, 0, 2, 0), (65, 120, 320, 346, 2, 0, 11, 0),
    (84, 192, 96, 127, 2, 1, 2, 0), (97, 48, 192, 315, 2, 1, 5, 0), (68, 56, 128, 348, 3, 0, 2, 0),
    (81, 168, 160, 271, 3, 0, 5, 0), (76, 152, 64, 205, 3, 1, 2, 0), (114, 136, 128, 165, 3, 1, 6, 0),
    (176, 64, 256, 214, 0, 0, 2, 0), (158, 144, 128, 308, 0, 0, 5, 0), (179, 88, 128, 248, 0, 1, 2, 0),
    (167, 112, 160, 319, 0, 1, 5, 0), (155, 24, 352, 242, 1, 0, 2, 0), (167, 72, 224, 211, 1, 0, 4, 0),
    (147, 32, 192, 366, 1, 1, 2, 0), (176, 56, 192, 313, 1, 1, 5, 0), (162, 24, 256, 324, 2, 0, 2, 0),
    (158, 88, 160, 199, 2, 0, 4, 0), (145, 16, 384, 360, 2, 1, 2, 0), (178, 64, 160, 366, 2, 1, 6, 0),
]


@pytest.mark.parametrize("nant,nchan,npkt,nbeam,prec,fine,tiles,sums", SPREAD)
def test_spread_tiles_a_workgroup(bf, nant, nchan, npkt, nbeam, prec, fine, tiles, sums):
    """The table's blocks run spread tiles of as many beam tiles a workgroup as it says;
    a plan whose variant is set runs that."""
    cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=32, precision=prec, weight_mode=fine)
    assert bf.lib.bfk_spread_tiles(dims(cfg)) == tiles
    assert bool(psum_bytes(bf, cfg)) == bool(sums)
    assert bf.lib.bfk_unset_differs(dims(cfg))


@pytest.mark.parametrize("nbeam", [65, 96, 128])
@pytest.mark.parametrize("fine", [0, 1])
def test_fp8_blocks_of_65_to_128_beams_run_no_spread_tiles(bf, nbeam, fine):
    """60 antennas x 256 channels x 1280 samples in FP8 to 65 to 128 beams: shared tiles
    in the variant's place, not spread ones."""
    cfg = bf.config(nant=60, nchan=256, npkt=640, nbeam=nbeam, tavg=32, precision=1, weight_mode=fine)
    assert bf.lib.bfk_spread_tiles(dims(cfg)) == 0 and bf.lib.bfk_unset_differs(dims(cfg))


@pytest.mark.parametrize("seed", range(4))
def test_correlator_slices_are_within_the_block_and_the_chip(bf, seed):
    """bfk_xcorr_use_fused gives 0 or slices in which the kernel that reads the block can
    run: no more than the units of 32 packets, and with several no more workgroups than
    run at once; none above 64 antennas or 65536 packets.  Wherever it gives slices,
    bfk_xcorr_fused_slices (the best ones, whichever path is faster) does."""
    rng = random.Random(seed)
    for _ in range(3000):
        nant, order = rng.randint(1, 96), rng.randint(0, 1)
        nchan, npkt = 8 * rng.choice([1, 2, 3, 6, 13, 48, 200, rng.randint(1, 512)]), 32 * rng.choice([1, 2, 3, 64, 2048, 2049, rng.randint(1, 4000)])
        use, best = (f(nant, nchan, npkt, order) for f in (bf.lib.bfk_xcorr_use_fused, bf.lib.bfk_xcorr_fused_slices))
        if nant > 64 or npkt > 65536:
            assert use == best == 0
            continue
        assert best >= 1
        for s in (use, best):
            assert 0 <= s <= min(32, npkt // 32)
            assert s <= 1 or nchan // (8 if nant <= 32 else 4) * s <= (512 if nant <= 32 else 256)


@pytest.mark.parametrize("nant,nchan,npkt,order,fused", [
    (64, 384, 2048, 1, 1), (64, 384, 2048, 0, 1), (32, 384, 2048, 0, 1), (61, 264, 128, 1, 1), (14, 8, 64, 0, 1),   # both times shorter
    (60, 16, 64, 0, 0), (11, 32, 224, 0, 0), (32, 32, 544, 0, 0), (28, 104, 416, 0, 0), (64, 128, 512, 0, 0)])      # a block alone a tenth longer
def test_correlator_route_by_both_times(bf, nant, nchan, npkt, order, fused):
    """Shapes timed well on one side of the rule: a block alone and one among others,
    the turned path and the kernel that reads the block."""
    assert bool(bf.lib.bfk_xcorr_use_fused(nant, nchan, npkt, order)) == bool(fused)
