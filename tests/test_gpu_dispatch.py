"""The kernel variants that a call's sizes and options choose, each at the edges of
its range, against the FP64 oracle or the general path."""

import numpy as np
import pytest

from common import C1_SMALL, Mirror, from_starfile, write_starfile

pytestmark = pytest.mark.gpu


def say(msg):
    print(msg, flush=True)


def make(params, irs=False, **extra):
    from irs_amd.microlensing.IPM.ipm import IPM
    from irs_amd.microlensing.IRS.irs import IRS
    kw = dict(params, write_stars=False, write_maps=False, write_histograms=False)
    kw.update(extra)
    m = (IRS if irs else IPM)(**kw)
    m.run()
    return m


@pytest.mark.parametrize("rect", [False, True])
def test_irs_parity_windows(oracle, rect, tmp_path):
    """Parity counts share the words of a block's LDS window, which is flushed every
    512 rows: tiles below, at and above that height, of linear and of general smooth
    matter, in both precisions, against the oracle's rays (2 rays may differ, as for
    every FP64 ray map: one lands within 1e-12 of a pixel edge)."""
    # a star file: the float library returns its own field rounded to float
    field = dict(C1_SMALL, rectangular=rect, num_rays_y=9)
    stars = write_starfile(oracle, tmp_path / "stars.bin", field, seed=7)
    params = dict(from_starfile(field, tmp_path / "stars.bin"), expansion_order=16, write_parities=True)
    ref = None
    for precision, th in ((0, 0), (0, 511), (1, 512), (0, 513), (1, 1100), (0, 3)):
        say(f"[irs windows] rect {rect}, precision {precision}, tile_rows {th}")
        m = make(params, irs=True, precision=precision, tile_rows=th)
        if ref is None:
            ref = Mirror(oracle, m, stars=stars).irs_map(parities=True)
        assert m.num_rays_received == ref[3] == m.num_rays.sum()
        for got, want in zip((m.num_rays, m.num_rays_minima, m.num_rays_saddles), ref):
            assert np.abs(got.astype(np.int64) - want).sum() <= 2
        m.close()


@pytest.mark.parametrize("general", [False, True])
def test_batch_tiles_and_pieces(general):
    """The last tiles of a batch go out in pieces of eight rows: tile heights below
    a piece, one piece, and with a remainder, at few and many resident blocks, for
    batches of linear smooth matter and with one general instance, against the
    instances' single maps (FP32 summation order only, the bound of the batched
    parity test)."""
    from irs_amd.microlensing.IPM.batch import IPMBatch, draw_instances
    from irs_amd.microlensing.IPM.ipm import IPM
    params = draw_instances(3, seed=5, sides=(64, 96), star_range=(1.5e3, 3.0e3), num_rays_y=3)
    if general:
        params[1]["rectangular"] = True
    objs, refs = [], []
    for p in params:
        m = IPM(**p)
        m.run()
        refs.append(m.magnifications.astype(np.float64))
        objs.append(m)
    for tile_h, blocks in ((1, 1), (8, 16), (20, 12), (63, 2), (300, 16)):
        say(f"[batch pieces] general {general}, tile_h {tile_h}, blocks/CU {blocks}")
        batch = IPMBatch()
        batch.set_tuning(tile_h, blocks)
        for m in objs:
            batch.add(m)
        h = batch.run()
        for m, ref, counts in zip(objs, refs, h):
            e = np.abs(m.magnifications - ref) / np.maximum(ref, 1e-3 * ref.max())
            assert np.max(e) < 2e-5
            assert counts.sum() == ref.size
        batch.close()
    for m in objs:
        m.close()
