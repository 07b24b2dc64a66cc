"""The rules that pick a kernel for a shape, which the host evaluates: what they may
answer, over the ranges that the entry points take.  No GPU."""
import random

import pytest


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
