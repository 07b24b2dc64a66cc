"""Blocks of every route of the spread tiles and the repacked ones on the GPU
(tests/test_routes.py has the tables and checks on the CPU which route each takes)."""
import numpy as np
import pytest

from test_routes import PACKS, SPREAD, dims

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tavg", [8, 16, 32, 64])
def test_spread_tiles_of_one_to_many_beam_tiles_have_the_variants_bits(bf, tavg):
    """One, two, three and more beam tiles a workgroup, with and without the sums of the
    beam powers in the launch, at each antenna chunk count, precision and weight mode:
    output, power and beam power equal the pinned variant's bit for bit, for two blocks
    one after another.  (Each block of the table at two of the four bins.)"""
    for i, (nant, nchan, npkt, nbeam, prec, fine, tiles, sums) in enumerate(SPREAD):
        if (i + tavg.bit_length()) % 2:
            continue
        print(f"spread tavg={tavg} {nant}x{nchan}x{npkt}->{nbeam} prec={prec} fine={fine} tiles={tiles} sums={sums}", flush=True)
        cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=tavg, precision=prec, weight_mode=fine,
                        angle_mode=bf.ANGLE_SIN, input_order=(i >> 1) & 1, output_layout=(i >> 2) & 1)
        assert bf.lib.bfk_spread_tiles(dims(cfg)) == tiles and bf.lib.bfk_spread_tiles(dims(cfg)) > 0
        antpos, cal, theta = bf.synth_geometry(nant, cfg.ncal, nbeam, 3 + i)
        scale = np.full(nbeam, 2e-3 / nant, np.float32)
        plans = [bf.Plan(cfg), bf.Plan(cfg)]
        for plan in plans:
            plan.set_weights(antpos, cal, bf.reference_freqs(1498.75, nchan), theta)
        plans[1].variant = plans[1].variant
        for seed in (i, i + 1):
            block = np.random.default_rng(seed).integers(0, 256, bf.input_bytes(cfg), dtype=np.uint8)
            got = [plan.process_block(block, scale, want_power=True, want_beam_power=True) for plan in plans]
            for a, b in zip(*got):
                assert np.array_equal(a, b)
        for plan in plans:
            plan.close()


@pytest.mark.parametrize("tavg", [8, 16, 32, 64])
def test_repacked_blocks_have_the_variants_bits(bf, tavg):
    """Every size of the last beam set, both chunk counts, input orders and output
    layouts: output, power and beam power equal the pinned variant's bit for bit.
    (Each block of the table at two of the four bins.)"""
    for i, (nant, nchan, npkt, nbeam, prec, fine, order) in enumerate(PACKS):
        if (i + tavg.bit_length()) % 2:
            continue
        print(f"packed tavg={tavg} {nant}x{nchan}x{npkt}->{nbeam} prec={prec} fine={fine} order={order}", flush=True)
        cfg = bf.config(nant=nant, nchan=nchan, npkt=npkt, nbeam=nbeam, tavg=tavg, precision=prec, weight_mode=fine,
                        angle_mode=bf.ANGLE_SIN, input_order=order, output_layout=(i >> 1) & 1)
        assert bf.lib.bfk_pack_block(dims(cfg))
        antpos, cal, theta = bf.synth_geometry(nant, cfg.ncal, nbeam, 3 + i)
        block = np.random.default_rng(i).integers(0, 256, bf.input_bytes(cfg), dtype=np.uint8)
        got = []
        for pin in (False, True):
            plan = bf.Plan(cfg)
            plan.set_weights(antpos, cal, bf.reference_freqs(1498.75, nchan), theta)
            if pin:
                plan.variant = plan.variant
            got.append(plan.process_block(block, np.full(nbeam, 2e-3 / nant, np.float32), want_power=True, want_beam_power=True))
            plan.close()
        for a, b in zip(*got):
            assert np.array_equal(a, b)
