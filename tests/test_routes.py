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
# 32-beam tiles that a workgroup takes, and whether the launch sums the beam powers itself; in all
# bins and both input orders.  Each precision and weight mode with one, two, three and more tiles,
# with and without the sums (which occur up to three), up to 64 antennas; with two and more at 65
# to 128 and 129 to 256 (as far as there are such blocks of up to 20 MB).
SPREAD = [
    (23, 264, 384, 27, 0, 0, 1, 0), (61, 56, 480, 19, 0, 0, 1, 1), (35, 88, 64, 399, 0, 0, 2, 0),
    (34, 112, 288, 58, 0, 0, 2, 1), (26, 56, 384, 149, 0, 0, 3, 0), (58, 56, 352, 77, 0, 0, 3, 1),
    (46, 72, 352, 158, 0, 0, 5, 0), (45, 288, 320, 13, 0, 1, 1, 0), (21, 56, 224, 134, 0, 1, 1, 1),
    (40, 16, 448, 290, 0, 1, 2, 0), (25, 240, 64, 105, 0, 1, 2, 1), (44, 168, 64, 325, 0, 1, 3, 0),
    (61, 112, 224, 148, 0, 1, 5, 0), (40, 192, 576, 20, 1, 0, 1, 0), (55, 24, 32, 65, 1, 0, 1, 1),
    (32, 40, 224, 226, 1, 0, 2, 0), (25, 96, 160, 119, 1, 0, 2, 1), (47, 56, 160, 324, 1, 0, 3, 0),
    (22, 96, 224, 93, 1, 0, 3, 1), (30, 304, 32, 351, 1, 0, 4, 0), (31, 144, 608, 7, 1, 1, 1, 0),
    (21, 8, 128, 270, 1, 1, 1, 1), (30, 72, 96, 325, 1, 1, 2, 0), (42, 160, 96, 111, 1, 1, 2, 1),
    (34, 128, 96, 259, 1, 1, 3, 0), (45, 224, 64, 255, 1, 1, 4, 0), (60, 304, 224, 21, 2, 0, 1, 0),
    (33, 16, 288, 109, 2, 0, 1, 1), (28, 32, 288, 243, 2, 0, 2, 0), (43, 64, 96, 305, 2, 0, 2, 1),
    (22, 64, 128, 282, 2, 0, 3, 0), (58, 24, 544, 151, 2, 0, 3, 1), (29, 168, 640, 16, 2, 1, 1, 0),
    (47, 64, 96, 208, 2, 1, 1, 1), (48, 232, 32, 308, 2, 1, 2, 0), (25, 32, 448, 115, 2, 1, 2, 1),
    (26, 96, 96, 349, 2, 1, 3, 0), (45, 152, 96, 199, 2, 1, 4, 0), (38, 256, 384, 10, 3, 0, 1, 0),
    (25, 136, 96, 74, 3, 0, 1, 1), (36, 304, 32, 198, 3, 0, 2, 0), (43, 40, 640, 35, 3, 0, 2, 1),
    (46, 304, 32, 285, 3, 0, 3, 0), (34, 160, 640, 30, 3, 1, 1, 0), (52, 112, 64, 45, 3, 1, 1, 1),
    (51, 24, 352, 368, 3, 1, 2, 0), (64, 168, 96, 113, 3, 1, 2, 1), (60, 160, 160, 70, 3, 1, 3, 0),
    (21, 96, 224, 90, 3, 1, 3, 1), (26, 48, 512, 136, 3, 1, 5, 0), (86, 24, 288, 322, 0, 0, 2, 0),
    (106, 200, 192, 136, 0, 0, 5, 0), (96, 128, 96, 175, 0, 1, 2, 0), (105, 72, 544, 317, 0, 1, 10, 0),
    (113, 56, 128, 303, 1, 0, 2, 0), (78, 312, 160, 159, 1, 0, 5, 0), (72, 128, 96, 189, 1, 1, 2, 0),
    (76, 160, 384, 264, 1, 1, 9, 0), (72, 96, 448, 38, 2, 0, 2, 0), (102, 96, 416, 99, 2, 0, 4, 0),
    (123, 88, 96, 253, 2, 1, 2, 0), (68, 40, 224, 315, 3, 0, 2, 0), (95, 288, 128, 141, 3, 0, 5, 0),
    (122, 64, 192, 167, 3, 1, 2, 0), (94, 88, 192, 152, 3, 1, 5, 0), (218, 192, 96, 113, 0, 0, 2, 0),
    (130, 136, 256, 399, 0, 0, 13, 0), (143, 24, 256, 338, 0, 1, 2, 0), (248, 48, 384, 302, 0, 1, 5, 0),
    (212, 296, 32, 219, 1, 0, 2, 0), (147, 176, 192, 307, 1, 0, 10, 0), (198, 208, 32, 315, 1, 1, 2, 0),
    (135, 96, 384, 271, 1, 1, 9, 0), (150, 40, 416, 97, 2, 0, 2, 0), (143, 208, 160, 271, 2, 0, 9, 0),
    (242, 88, 128, 177, 2, 1, 2, 0),
]


@pytest.mark.parametrize("nant,nchan,npkt,nbeam,prec,fine,tiles,sums", SPREAD)
def test_spread_tiles_a_workgroup(bf, nant, nchan, npkt, nbeam, prec, fine, tiles, sums):
    """The table's blocks run spread tiles of as many beam tiles a workgroup as it says;
    a plan whose variant is set runs that."""
    for tavg in (8, 16, 32, 64):
        for order in (0, 1):
            cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=tavg, precision=prec, weight_mode=fine,
                            input_order=order)
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


@pytest.mark.parametrize("nant,nchan,npkt,nbeam,prec,fine,tavg,order", [
    (217, 168, 128, 245, 0, 0, 8, 1), (193, 40, 256, 325, 1, 1, 32, 1), (28, 120, 896, 64, 1, 1, 32, 0), (26, 224, 224, 57, 1, 1, 64, 0),
    (131, 344, 32, 789, 0, 1, 64, 1), (197, 240, 96, 631, 0, 1, 8, 1), (60, 384, 1856, 60, 3, 0, 16, 0), (56, 328, 384, 47, 1, 0, 16, 0)])
def test_blocks_whose_variant_is_faster_run_no_spread_tiles(bf, nant, nchan, npkt, nbeam, prec, fine, tavg, order):
    """Blocks that took 10 to 50 % longer in spread tiles, alone or among others."""
    cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=tavg, precision=prec, weight_mode=fine, input_order=order)
    assert bf.lib.bfk_spread_tiles(dims(cfg)) == 0


# Blocks that are repacked, in all bins: antennas, channels, packets, beams, precision, fine weights,
# input order.  Each precision and order at 65 to 128 and 129 to 256 antennas with one, two, three or
# four, five to seven, and eight 32-beam tiles in the last set.
PACKS = [
    (73, 144, 736, 538, 0, 1, 0), (109, 128, 544, 314, 0, 1, 0), (70, 104, 736, 343, 0, 1, 0),
    (75, 176, 320, 418, 0, 1, 0), (69, 144, 832, 487, 0, 1, 0), (69, 192, 512, 524, 0, 1, 1),
    (112, 56, 1184, 307, 0, 1, 1), (102, 152, 288, 590, 0, 1, 1), (66, 112, 608, 159, 0, 1, 1),
    (106, 88, 608, 529, 1, 0, 0), (84, 88, 768, 294, 1, 1, 0), (78, 168, 416, 382, 1, 1, 0),
    (86, 104, 768, 204, 1, 0, 0), (105, 160, 288, 511, 1, 1, 0), (74, 120, 768, 525, 1, 0, 1),
    (95, 88, 992, 317, 1, 0, 1), (76, 112, 800, 582, 1, 1, 1), (96, 152, 512, 398, 1, 1, 1),
    (65, 120, 896, 484, 1, 0, 1), (115, 56, 416, 520, 2, 1, 0), (67, 48, 832, 292, 2, 0, 0),
    (75, 64, 544, 592, 2, 0, 0), (73, 176, 512, 216, 2, 1, 0), (69, 96, 608, 486, 2, 0, 0),
    (76, 152, 672, 528, 2, 0, 1), (106, 176, 320, 575, 2, 1, 1), (66, 104, 672, 356, 2, 0, 1),
    (70, 112, 992, 464, 2, 1, 1), (97, 152, 256, 507, 2, 1, 1), (65, 144, 736, 261, 3, 1, 0),
    (100, 96, 736, 573, 3, 0, 0), (95, 144, 256, 583, 3, 1, 0), (90, 64, 1120, 174, 3, 1, 0),
    (96, 192, 224, 510, 3, 0, 0), (107, 72, 832, 543, 3, 0, 1), (128, 192, 128, 552, 3, 1, 1),
    (78, 40, 896, 356, 3, 1, 1), (99, 160, 448, 148, 3, 1, 1), (80, 144, 736, 231, 3, 1, 1),
    (180, 64, 704, 525, 0, 0, 0), (155, 40, 960, 568, 0, 1, 0), (140, 48, 960, 581, 0, 1, 0),
    (199, 80, 512, 467, 0, 1, 0), (133, 32, 1088, 488, 0, 0, 0), (143, 96, 416, 524, 0, 1, 1),
    (148, 152, 224, 552, 0, 1, 1), (151, 168, 288, 595, 0, 1, 1), (136, 136, 256, 451, 0, 1, 1),
    (140, 80, 480, 504, 0, 0, 1), (194, 184, 224, 536, 1, 1, 0), (194, 40, 896, 567, 1, 0, 0),
    (205, 112, 320, 110, 1, 1, 0), (136, 80, 448, 452, 1, 0, 0), (148, 152, 256, 489, 1, 1, 0),
    (211, 32, 1216, 540, 1, 1, 1), (166, 56, 896, 545, 1, 1, 1), (133, 56, 1088, 363, 1, 1, 1),
    (153, 48, 768, 418, 1, 1, 1), (144, 32, 1056, 484, 1, 0, 1), (160, 80, 352, 533, 2, 1, 0),
    (239, 56, 608, 547, 2, 0, 0), (146, 96, 288, 593, 2, 1, 0), (148, 64, 768, 415, 2, 0, 0),
    (177, 96, 384, 482, 2, 1, 0), (183, 64, 704, 537, 2, 1, 1), (142, 168, 224, 308, 2, 1, 1),
    (190, 64, 384, 594, 2, 0, 1), (162, 32, 1120, 391, 2, 0, 1), (130, 40, 864, 490, 2, 1, 1),
]


@pytest.mark.parametrize("nant,nchan,npkt,nbeam,prec,fine,order", PACKS)
def test_repacked_blocks(bf, nant, nchan, npkt, nbeam, prec, fine, order):
    """The table's blocks are repacked; a plan whose variant is set runs that."""
    for tavg in (8, 16, 32, 64):
        cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=tavg, precision=prec, weight_mode=fine, input_order=order)
        assert bf.lib.bfk_pack_block(dims(cfg)) and not bf.lib.bfk_pack_block(dims(cfg, 1))


@pytest.mark.parametrize("nant,nchan,npkt,nbeam,prec,fine,packs", [
    (67, 120, 768, 100, 1, 0, 0), (130, 64, 512, 100, 1, 1, 0), (195, 304, 800, 58, 1, 1, 0), (162, 336, 224, 40, 1, 1, 0), (119, 112, 352, 706, 2, 0, 0),
    (67, 104, 640, 1, 3, 1, 1), (129, 72, 480, 400, 1, 0, 1), (256, 384, 2048, 1024, 1, 1, 1)])
def test_blocks_with_groups_outermost_are_repacked_where_that_is_faster(bf, nant, nchan, npkt, nbeam, prec, fine, packs):
    """Blocks timed both ways in the order of dsaX_split -r, whose lines the variants
    waste less of: those that took up to 56 % longer alone, or 48 % among others,
    repacked stay as they are."""
    cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=32, precision=prec, weight_mode=fine, input_order=1)
    assert bool(bf.lib.bfk_pack_block(dims(cfg))) == bool(packs)
    assert bf.lib.bfk_use_packed(dims(cfg))
