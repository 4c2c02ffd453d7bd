"""The kernel variants that a call's sizes and options choose, each at the edges of
its range, against the FP64 oracle or the general path."""

import ctypes
import os

import numpy as np
import pytest

from common import C1_SMALL, Mirror, from_starfile, write_starfile

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


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


def free_memory(lib):
    """Bytes of device memory left, through the HIP runtime that the engine library is linked with."""
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def late_work(m):
    """Wide triangles and rows that the last shot left for later launches."""
    return m.lib.get_late_triangles(m.obj), m.lib.get_late_rows(m.obj)


@pytest.mark.parametrize("parities", [False, True])
@pytest.mark.parametrize("pixels,rays,half,least", [(40, 2, 6.0, (0, 1)), (301, 1, 6.0, (1, 1)), (700, 4, 6.0, (1, 1)),
                                                    (2500, 1, 6.0, (65536, 1)), (3000, 4, 10.0, (65536, 32768))])
def test_work_left_for_later_launches(parities, pixels, rays, half, least):
    """A single map leaves wide triangles and rows of many triangles for two launches
    of their own, up to the lists' lengths; a batch shoots every tile whole. Small and
    odd maps, one that fills the list of triangles and one that fills both: the same map
    from both. Each pixel is two FP32 sums of at most some 300 terms in another order,
    300 * 2^-24 < 2e-5 of the pixel (of the mean, below it, for the residue of the runs)."""
    from irs_amd.microlensing.IPM.batch import IPMBatch
    from irs_amd.microlensing.IPM.ipm import IPM
    params = dict(C1_SMALL, half_length_y1=half, half_length_y2=half, num_pixels_y1=pixels, num_pixels_y2=pixels,
                  num_rays_y=rays)
    whole = IPM(**params)
    whole.prepare()
    whole.build()
    batch = IPMBatch()
    batch.set_tuning(64, 16)
    batch.add(whole)
    batch.run()
    m = make(params, write_parities=parities)
    ref = whole.magnifications.astype(np.float64)
    err = np.abs(m.magnifications - ref) / np.maximum(ref, ref.mean())
    say(f"[later] {pixels} pixels, {rays} rays, parities {parities}: {err.max():.1e}, {late_work(m)} left")
    assert all(got >= n for got, n in zip(late_work(m), least))
    assert ref.mean() > 0 and err.max() < 2e-5
    m.close()
    whole.close()


@pytest.mark.parametrize("double", [True, False])
@pytest.mark.parametrize("pixels,rays,rect", [(301, 1, False), (301, 1, True), (700, 4, False)])
def test_later_launches_keep_the_parities(oracle, tmp_path, double, pixels, rays, rect):
    """Triangles and rows shot by the later launches land in the map of their parity: total,
    minima and saddles each against the oracle's, for both value types, linear and general
    smooth matter, with and without parity maps. FP64 corners differ by rounding, which moves
    a pixel by 1e-8 at most over 3e8 cells (whole-map parity tests); mixed ones to the bounds
    of the mixed parity test, and the flux of a map by the few triangles whose area is zero to
    FP32 (less than 1e-6 of all; half of the wide ones would be 1e-5 or more)."""
    field = dict(C1_SMALL, half_length_y1=6.0, half_length_y2=6.0, num_pixels_y1=pixels, num_pixels_y2=pixels, num_rays_y=rays,
                 rectangular=rect)
    stars = write_starfile(oracle, tmp_path / "stars.bin", field, seed=11, margin=1.2)
    params = dict(from_starfile(field, tmp_path / "stars.bin"), expansion_order=16, is_double=double)
    m = make(params, write_parities=True)
    triangles, rows = late_work(m)
    assert triangles > 0 and (rows == 0 if rect else rows > 0)   # a rectangular sheet's rows stay with their tile
    ref = Mirror(oracle, m, stars=stars).ipm_map(parities=True)[:3]
    plain = make(params)
    mean = ref[0].mean()
    for what, got, want in zip(("total", "minima", "saddles", "plain"), (m.magnifications, m.magnifications_minima,
                               m.magnifications_saddles, plain.magnifications), (*ref, ref[0])):
        e = np.abs(got - want) / np.maximum(want, mean)
        flux = abs(got.sum(dtype=np.float64) - want.sum()) / ref[0].sum()
        say(f"[later {what}] {pixels} pixels, rect {rect}, double {double}: max {e.max():.1e}, p99 {np.percentile(e, 99):.1e}, "
            f"flux {flux:.1e}")
        if double:
            assert e.max() < 1e-7 and flux < 1e-10
        else:
            assert np.median(e) < 1e-4 and np.percentile(e, 99) < 1e-2 and flux < 1e-5
    m.close()
    plain.close()


def write_field(path, stars, radius):
    with open(path, "wb") as fh:
        np.array([len(stars), 0], dtype=np.int32).tofile(fh)
        np.array([radius, 0.0, 1.0]).tofile(fh)
        np.ascontiguousarray(stars, dtype=np.float64).tofile(fh)


def disk(rng, n, radius, centre=(0.0, 0.0)):
    r, t = radius * np.sqrt(rng.random(n)), 2 * np.pi * rng.random(n)
    return np.stack([centre[0] + r * np.cos(t), centre[1] + r * np.sin(t)], axis=1)


def built(path, stars, order, mode=3):
    """A built double-precision object over `stars` in a disk of radius 40."""
    from irs_amd.microlensing.IPM.ipm import IPM
    write_field(path, stars, 40.0)
    m = IPM(kappa_tot=0.3, shear=0.3, light_loss=0.01, starfile=str(path), half_length_y1=0.5, half_length_y2=0.5,
            num_pixels_y1=16, num_pixels_y2=16, is_double=True, expansion_order=order, m2l_mode=mode)
    m.prepare()
    m.build()
    return m


def coefficient_errors(m, tree):
    for which in ("multipole", "local"):
        g, o = m.export_coeffs(which), tree.coeffs(which)
        yield which, np.max(np.abs(g - o) / np.maximum(np.max(np.abs(o), axis=1, keepdims=True), 1e-300))


@pytest.mark.parametrize("n,cluster", [(1, 0), (32, 0), (33, 0), (300, 0), (3000, 0), (16384, 0), (16385, 0), (60000, 0),
                                       (250000, 0), (2000, 1500), (2000, 20000)])
def test_trees_of_every_split_path(oracle, tmp_path, n, cluster):
    """A level is split by one block per node of 64, 256 or 1024 threads, or device-wide
    above 16384 stars in a node, its nodes ranked by one block or, above 32768 of them,
    by a device-wide scan; M2L runs one or two column tiles per block. The leaf tables hold
    an entry per leaf, numbered as the levels are split: points in the first leaf, the last and
    a few thousand others deflect as in the oracle's tree (the parity tests' bound). Even fields and
    fields with a cluster a few thousandths wide: the oracle's tree bit for bit, its
    coefficients to FP64 rounding (the bound of the parity tests)."""
    rng = np.random.default_rng(n + cluster)
    xy = np.concatenate([disk(rng, n, 39.0), disk(rng, cluster, 2e-3, (3.1, -7.3))])
    stars = np.concatenate([xy, np.full((len(xy), 1), 16.0 / len(xy))], axis=1)
    say(f"[tree] {n} stars, {cluster} in a cluster")
    m = built(tmp_path / "stars.bin", stars, 12)
    tree = oracle.Tree(stars, m.root_half_length)
    for got, want in zip(m.export_tree(), tree.export()):
        np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(m.stars, tree.stars())
    tree.fmm(12)
    for which, err in coefficient_errors(m, tree):
        say(f"[tree] {which}: {err:.1e}")
        assert err < 1e-11, which
    geom, info, _ = m.export_tree()
    leaves = geom[info[:, 2] < 0]
    assert m.lib.get_num_leaves(m.obj) == len(leaves)
    some = leaves[np.unique(np.linspace(0, len(leaves) - 1, 4000).astype(int))]
    z = some[:, 0] + 0.3 * some[:, 2] + 1j * (some[:, 1] - 0.4 * some[:, 2])
    lens = oracle.make_lens(m.kappa_tot, m.shear, m.theta_star, m.kappa_star, (40.0, 0.0), 0, 1, m.lib.get_taylor_smooth(m.obj))
    want, _ = tree.deflect(lens, z)
    err = np.abs(m.deflect(z) - want)
    say(f"[tree] {len(leaves)} leaves, deflections of {len(z)}: {err.max():.1e}")
    assert err.max() < 1e-10
    m.close()


@pytest.mark.parametrize("n", [1, 15, 255, 256, 257, 4096, 4097, 70000])
def test_star_moments_of_every_count(tmp_path, n):
    """A block sums 16 of 256 interleaved chains, 16 stars of each at a time: fields with
    fewer stars than chains, at a round's edges and of many rounds, masses over five
    decades. The terms of a sum add in n / 256 + 8 steps of an ulp and log is good to
    one, so 1e-12 of the sum of the terms' magnitudes holds for every n here."""
    rng = np.random.default_rng(n)
    mass = 10.0 ** rng.uniform(-4, 1, n)
    mass *= 16.0 / mass.sum()
    m = built(tmp_path / "stars.bin", np.column_stack([disk(rng, n, 39.0), mass]), 8)
    logs = mass * mass * np.log(mass)
    for got, terms in ((m.lib.get_mean_mass_actual(m.obj), mass), (m.lib.get_mean_mass2_actual(m.obj), mass * mass),
                       (m.lib.get_mean_mass2_ln_mass_actual(m.obj), logs)):
        assert abs(got - terms.mean()) <= 1e-12 * np.abs(terms).mean()
    assert m.lib.get_m_lower_actual(m.obj) == mass.min() and m.lib.get_m_upper_actual(m.obj) == mass.max()
    m.close()


@pytest.mark.parametrize("order", [1, 3, 7, 8, 15, 16, 23, 24, 31])
def test_fmm_at_the_edges_of_its_matrix_sizes(oracle, tmp_path, order):
    """The stacked M2L matrices are padded to 16, 32, 48 or 64: the first and last order
    of each, by recurrences, FP64 and FP32 MFMA, and with two column tiles per block.
    FP64 to rounding; FP32 to single precision of the products (the parity tests' bounds)."""
    rng = np.random.default_rng(order)
    for n, modes in ((3000, (0, 3, 2)), (60000, (3,))):
        stars = np.concatenate([disk(rng, n, 39.0), np.full((n, 1), 16.0 / n)], axis=1)
        tree = None
        for mode in modes:
            m = built(tmp_path / "stars.bin", stars, order, mode)
            if tree is None:
                tree = oracle.Tree(stars, m.root_half_length)
                tree.fmm(order)
            for which, err in coefficient_errors(m, tree):
                say(f"[fmm] {n} stars, order {order}, m2l_mode {mode}, {which}: {err:.1e}")
                assert err < (2e-5 if mode == 2 else 1e-11)
            m.close()


@pytest.mark.parametrize("irs,double", [(False, False), (False, True), (True, False)])
@pytest.mark.parametrize("n1,n2", [(1, 1), (128, 128), (129, 127), (400, 300)])
def test_histograms_inside_and_past_the_window(tmp_path, irs, double, n1, n2):
    """Blocks of at least 16384 pixels count the first 8192 bins of both histograms in LDS:
    maps of less than, exactly and several blocks, whose bright pixels and ray counts lie
    past the window. Every bin of the files against numpy's count of the returned maps."""
    prefix = str(tmp_path) + "/"
    m = make(dict(kappa_tot=0.45, shear=0.45, kappa_star=0.36, mass_function="equal"), irs=irs, half_length_y1=0.02 * n1,
             half_length_y2=0.02 * n2, num_pixels_y1=n1, num_pixels_y2=n2, num_rays_y=900 if irs else 4, light_loss=0.01,
             random_seed=5, expansion_order=12, write_parities=True, write_histograms=True, outfile_prefix=prefix,
             **({"is_double": double} if not irs else {}))
    check_histograms(m, prefix, irs)
    m.close()


def check_histograms(m, prefix, irs):
    """Every bin of the saved histograms against numpy's count of the returned maps."""
    m.save()
    maps = (m.num_rays, m.num_rays_minima, m.num_rays_saddles) if irs else (
        m.magnifications, m.magnifications_minima, m.magnifications_saddles)
    for suffix, mp in zip(("", "_minima", "_saddles"), maps):
        v = np.asarray(mp, dtype=np.float64).ravel()
        kinds = [("numrays_numpixels" if irs else "mags_numpixels", v if irs else 1000.0 * v)]
        if not irs:
            kinds.append(("log_mags_numpixels", 1000.0 * np.log10(v[v > 0])))
        for kind, x in kinds:
            t = np.trunc(x)
            u, c = np.unique((t + np.where(np.abs(x - t) >= 0.5, np.sign(x), 0.0)).astype(np.int64), return_counts=True)
            got = np.loadtxt(prefix + ("irs_" if irs else "ipm_") + kind + suffix + ".txt", dtype=np.int64, ndmin=2)
            np.testing.assert_array_equal(got, np.column_stack([u, c]), err_msg=kind + suffix)
            say(f"[hist] {kind}{suffix}: {len(u)} bins up to {u[-1]}")


@pytest.mark.parametrize("irs", [False, True])
def test_histograms_of_wide_ranges(tmp_path, irs):
    """One star images the pixel behind it into a ring, thousands of times the others: histograms
    of millions of bins, counted map by map; and the memory they took is given back."""
    from irs_amd.microlensing.IPM.ipm import IPM
    from irs_amd.microlensing.IRS.irs import IRS
    path = tmp_path / "stars.bin"
    write_field(path, np.array([[0.0, 0.0, 1.0]]), 40.0)
    prefix = str(tmp_path) + "/"
    kw = dict(kappa_tot=1.0 / 1600, shear=0.0, starfile=str(path), light_loss=4e-4, half_length_y1=0.3, half_length_y2=0.3,
              num_pixels_y1=501, num_pixels_y2=501, num_rays_y=1000 if irs else 30, expansion_order=8, write_parities=True,
              outfile_prefix=prefix)
    m = (IRS if irs else IPM)(**kw, write_stars=False, write_maps=False, write_histograms=True)
    m.prepare()
    m.build()
    m.shoot()
    before = free_memory(m.lib)
    m.finish()
    held = before - free_memory(m.lib)
    bins = float((m.num_rays if irs else 1000 * m.magnifications).max())
    say(f"[hist wide] irs {irs}: {bins:.3g} bins, {held >> 20} MB held")
    assert bins > 1 << 20 and held < 8 << 20
    check_histograms(m, prefix, irs)
    m.close()


def test_critical_curves_beside_other_work(tmp_path):
    """Chains of two objects and of two processes on the device at once, with a map being
    shot beside them: blocks that are not all resident give way, and the roots stay the same."""
    import subprocess
    import sys
    import threading
    from irs_amd.microlensing.CCF.ccf import CCF
    from irs_amd.microlensing.IPM.ipm import IPM
    code = ("import sys; sys.path.insert(0, {root!r})\n"
            "import numpy as np\n"
            "from irs_amd.microlensing.CCF.ccf import CCF\n"
            "for k in range(3):\n"
            "    c = CCF(kappa_tot=0.3, shear=0.3, kappa_star=0.27, num_stars=600, num_phi=12, random_seed=3, write_stars=False)\n"
            "    c.run()\n"
            "np.save({out!r}, c.critical_curves)\n").format(root=ROOT, out=str(tmp_path / "other.npy"))

    def curves():
        c = CCF(kappa_tot=0.3, shear=0.3, kappa_star=0.27, num_stars=600, num_phi=12, random_seed=3, write_stars=False)
        c.run()
        out = c.critical_curves.copy()
        c.close()
        return out

    alone = curves()
    say("[ccf] beside another process, another object and a map")
    other = subprocess.Popen([sys.executable, "-c", code])
    results = []
    threads = [threading.Thread(target=lambda: results.append(curves())) for _ in range(3)]
    m = IPM(kappa_tot=0.45, shear=0.4, kappa_star=0.36, half_length_y1=5, half_length_y2=5, num_pixels_y1=1000,
            num_pixels_y2=1000, num_rays_y=16, random_seed=2, write_histograms=False)
    threads.append(threading.Thread(target=m.run))
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert other.wait(timeout=100) == 0
    m.close()
    for r in results + [np.load(tmp_path / "other.npy")]:
        np.testing.assert_array_equal(r, alone)
    assert len(results) == 3


@pytest.mark.parametrize("stars,phases,branches,exact", [(1, 4, 1, False), (2, 4, 2, True), (5, 600, 300, False),
                                                         (1024, 2, 1, False), (1025, 2, 1, False), (1100, 2, 1, False),
                                                         (2100, 2, 1, False), (1300, 2, 1, True)])
def test_critical_curve_chains(stars, phases, branches, exact):
    """Chains of one block and of many, more chains than the device holds at once (600),
    the last field that a block holds (1024 stars, 2048 roots) and larger ones, which take
    a launch per iteration, linear and general smooth matter:
    every root solves the critical-curve equation by direct sums (1/mu below 1e-6, as in
    the oracle tests) and the roots of a phase are distinct."""
    from irs_amd.microlensing.CCF.ccf import CCF
    from oracle import ccf as OC
    from scipy.spatial import cKDTree
    say(f"[ccf] {stars} stars, {phases} phases, {branches} branches, exact sheet {exact}")
    # one star on one branch cannot leave the line its starting roots lie on: use two there
    branches = max(branches, 2) if stars == 1 else branches
    kw = dict(kappa_tot=0.3, shear=0.3, kappa_star=0.27, num_stars=stars, num_phi=phases, num_branches=branches, random_seed=7,
              approx=not exact, write_stars=False)
    c, single = CCF(**kw), CCF(**kw)
    c.run()
    # the path that a busy device takes, one iteration per launch: the same roots bit for bit
    single.lib.set_resident_chains(single.obj, 0)
    single.run()
    np.testing.assert_array_equal(single.critical_curves, c.critical_curves)
    single.close()
    # blocks that give up on each other after one look, which starts the chains again: the same
    for polls in (0, 1, 20):
        impatient = CCF(**kw)
        impatient.lib.set_chain_polls(impatient.obj, polls)
        impatient.run()
        np.testing.assert_array_equal(impatient.critical_curves, c.critical_curves)
        impatient.close()
    prob = OC.Problem(c.stars, 0.3, 0.3, 1.0, 0.27, c.corner, approx=int(not exact))
    z = c.critical_curves[..., 0] + 1j * c.critical_curves[..., 1]
    half = phases // (2 * branches)
    phi = np.array([[np.pi / branches + 2 * np.pi * b / branches + (k - half) * 2 * np.pi / phases for k in range(2 * half + 1)]
                    for b in range(branches)])
    assert np.nanmax(prob.inv_mu_error(z, np.tile(phi, (c.num_roots, 1)))) < 1e-6
    for b in range(0, branches, max(1, branches // 3)):
        r = z[b::branches, 0]
        d, _ = cKDTree(np.column_stack([r.real, r.imag])).query(np.column_stack([r.real, r.imag]), k=2)
        assert d[:, 1].min() > 1e-8
    c.close()


@pytest.mark.parametrize("batch,n", [(16, 16), (48, 100), (240, 256)])
def test_surrogate_batches_and_requests(batch, n):
    """One block per 16 rows: batches of one, several and fifteen blocks, whose epochs
    leave rows over, against an epoch made of single steps (the same kernels in the same
    order: equal); and requests through pinned memory (up to 256 rows) and through device
    buffers, padded or not, against the FP64 network (the bound of the gradient test)."""
    from irs_amd.microlensing.Surrogate import surrogate as S
    from oracle import mlp
    rng = np.random.default_rng(batch)
    x, t = rng.normal(size=(n, 6)), rng.random((n, 128)) + 0.1
    s = S.HistogramSurrogate(max_batch=256, seed=4)
    p0 = s.params()
    losses = s.fit(x, t, epochs=2, batch=batch)
    trained = s.params()
    s.set_params(p0)
    order, step, steps = np.random.default_rng(0), 0, 2 * (n // batch)
    for ep in range(2):
        perm, tot = order.permutation(n).astype(np.int32), 0.0
        for b0 in range(0, n - batch + 1, batch):
            rows = np.ascontiguousarray(perm[b0:b0 + batch])
            tot += S.lib.surrogate_train_step(s.obj, rows.ctypes.data_as(ctypes.POINTER(ctypes.c_int)), batch,
                                              2e-3 * 0.5 * (1 + np.cos(np.pi * step / steps)), 1e-4)
            step += 1
        assert tot / (n // batch) == losses[ep]
    np.testing.assert_array_equal(s.params(), trained)
    for rows in (1, 15, 16, 17, 255, 256, 257, 300):
        q = rng.normal(size=(rows, 6))
        got = s.predict(q)
        want, _, _ = mlp.forward(s.params().astype(np.float64), s._inputs(q).astype(np.float64), bf16_ops=True)
        say(f"[surrogate] batch {batch}, request of {rows}: {np.max(np.abs(got - want)):.1e}")
        assert np.max(np.abs(got - want)) < 1e-4
    s.close()


@pytest.mark.parametrize("rect", [False, True])
def test_deflections_of_mixed_waves(oracle, tmp_path, rect):
    """A wave of points serves two shared leaves, then its other lanes one by one: waves
    of one leaf, of two, of three and of 64, partial waves, and points outside the root
    box, for linear and general smooth matter: the deflection and magnification of a point
    do not depend on its neighbours, and match the oracle (the parity tests' bounds)."""
    from irs_amd.microlensing.IPM.ipm import IPM
    field = dict(C1_SMALL, rectangular=rect)
    stars = write_starfile(oracle, tmp_path / "stars.bin", field, seed=9)
    m = IPM(**from_starfile(field, tmp_path / "stars.bin"), is_double=True, expansion_order=16)
    m.run()
    tree = Mirror(oracle, m, stars=stars)
    rng = np.random.default_rng(2)
    far = 2.0 * m.root_half_length
    spots = np.array([0.1 + 0.2j, 9.3 - 4.1j, -7.7 + 11.2j])
    waves = [np.repeat(spots[:k], 64 // k + 1)[:64] + 1e-3 * (rng.random(64) + 1j * rng.random(64)) for k in (1, 2, 3)]
    waves.append(20 * (rng.random(64) - 0.5) + 40j * (rng.random(64) - 0.5))
    waves.append(np.where(np.arange(64) % 3 == 0, far * np.exp(2j * np.pi * rng.random(64)), waves[3]))
    z = np.concatenate(waves)
    w, mu = m.deflect(z, want_mu=True)
    one = [m.deflect(z[k:k + 1], want_mu=True) for k in range(len(z))]
    assert np.max(np.abs(w - np.array([o[0][0] for o in one]))) <= 1e-13 * np.max(np.abs(w))
    np.testing.assert_allclose(mu, [o[1][0] for o in one], rtol=1e-9)
    for n in (1, 63, 65, 127):
        np.testing.assert_allclose(m.deflect(z[:n]), w[:n], rtol=0, atol=1e-13 * np.max(np.abs(w)))
    inside = np.concatenate(waves[:4])
    ref = tree.tree.deflect(tree.lens, inside)
    ref = ref[0] if isinstance(ref, tuple) else ref
    assert np.max(np.abs(w[:256] - ref)) < 1e-10
    m.close()


def astroids(rng, curves, spread, size):
    """Closed clockwise curves around centres uniform in a box of half-lengths `spread`."""
    t = -np.linspace(0, 2 * np.pi, 60)
    t[-1] = t[0]
    return (rng.uniform(-spread[0], spread[0], (curves, 1)) + 1j * rng.uniform(-spread[1], spread[1], (curves, 1)) +
            size * np.exp(2j * np.pi * rng.random((curves, 1))) * (np.cos(t) ** 3 + 1j * np.sin(t) ** 3))


def check_crossings(tmp_path, rows, npx, over_sample, path):
    """A run over the curves `rows` takes the given path (0 grid, 1 lists, 2 lists that overflow)
    and gives the oracle's counts and histogram."""
    from irs_amd.microlensing.NCC.ncc import NCC
    from oracle import ncc as ON
    with open(tmp_path / "ccf_caustics.bin", "wb") as fh:
        np.array(rows.shape, dtype=np.int32).tofile(fh)
        np.ascontiguousarray(rows, dtype=np.complex128).tofile(fh)
    prefix = str(tmp_path) + "/"
    n = NCC(infile_prefix=prefix, outfile_prefix=prefix, num_pixels_y1=npx[0], num_pixels_y2=npx[1], over_sample=over_sample,
            write_maps=False)
    n.run()
    say(f"[ncc lists] {npx}, over_sample {over_sample}, {len(rows)} curves: path {n.lib.get_crossing_path(n.obj)}")
    want = ON.ncc_map(rows, (0.0, 0.0), (5.0, 5.0), npx, over_sample)
    np.testing.assert_array_equal(n.num_caustic_crossings, want)
    n.save()
    u, c = np.unique(want, return_counts=True)
    np.testing.assert_array_equal(np.loadtxt(prefix + "ncc_ncc_numpixels.txt", dtype=np.int64, ndmin=2), np.column_stack([u, c]))
    assert n.lib.get_crossing_path(n.obj) == path
    n.close()


@pytest.mark.parametrize("npx,over_sample,curves", [((1, 1), 0, 3), ((7, 5), 0, 40), ((301, 9), 0, 40), ((64, 33), 1, 40),
                                                    ((4095, 3), 0, 20), ((2048, 3), 1, 20), ((2049, 3), 1, 20), ((1025, 3), 3, 20),
                                                    ((1024, 3), 2, 20), ((8192, 2), 0, 20), ((8193, 2), 0, 20), ((4096, 3), 1, 20),
                                                    ((2048, 3), 2, 20), ((1024, 3), 3, 20),
                                                    ((4100, 2), 2, 20), ((8193, 2), 1, 20), ((8193, 2), 2, 10), ((20, 6), 8, 8)])
def test_crossing_lists(tmp_path, npx, over_sample, curves):
    """Crossings go to a list per sub-pixel row, and the waves of a workgroup sum a row each
    in LDS: odd and even widths, one to 256 sub-pixels a pixel, the first and last width of
    each variant, and grids too wide for lists, against the oracle: identical counts and
    histogram."""
    rng = np.random.default_rng(curves + over_sample)
    rows = astroids(rng, curves, (4, 4), np.exp(rng.normal(0.0, 0.5, (curves, 1))))
    check_crossings(tmp_path, rows, npx, over_sample, 1 if npx[0] << over_sample <= 8192 else 0)


@pytest.mark.parametrize("npx,over_sample,curves,height,size,path", [((40, 30), 1, 4000, 4, 1.0, 0), ((100, 100), 0, 900, 4, 1.0, 1),
                                                                     ((600, 2100), 0, 3000, 0.005, 0.05, 2),
                                                                     ((64, 700), 2, 3000, 0.005, 0.05, 2), ((1, 3000), 0, 30, 4, 1.0, 1)])
def test_crossings_of_dense_networks(tmp_path, npx, over_sample, curves, height, size, path):
    """Networks with more crossings a row than lists are good for go to the grid at once, narrow
    maps have room for many, curves heaped on a few rows overflow lists that the mean allowed (all
    waves then stop and the grid takes over), and one column: the oracle's counts and histogram on
    each path."""
    rng = np.random.default_rng(curves)
    check_crossings(tmp_path, astroids(rng, curves, (4, height), size), npx, over_sample, path)


@pytest.mark.parametrize("heaped", [False, True])
@pytest.mark.parametrize("npx", [(1023, 512), (1024, 512), (1025, 513), (1500, 1201)])
def test_crossing_histograms(tmp_path, npx, heaped):
    """Maps of 2^19 pixels or more with at most 64 values are counted in a column per lane, all
    others in shared bins: below, at and above that size, with pixels left over in a block, of few
    values and (curves heaped on one place) of more than 64: the oracle's counts and histogram."""
    rng = np.random.default_rng(npx[0])
    curves = astroids(rng, 200 if heaped else 30, (0.3, 0.3) if heaped else (4, 4), 1.0)
    check_crossings(tmp_path, curves, npx, 0, 1)


def test_overflowed_lists_make_room(tmp_path):
    """The memory check counts the grid: lists that overflowed are freed before it is allocated,
    so that a map which passes the check fits. 512 x 131072 sub-pixels, 256 MB either way."""
    from irs_amd.microlensing.NCC.ncc import NCC
    rows = astroids(np.random.default_rng(1), 3000, (4, 0.005), 0.01)
    with open(tmp_path / "ccf_caustics.bin", "wb") as fh:
        np.array(rows.shape, dtype=np.int32).tofile(fh)
        np.ascontiguousarray(rows, dtype=np.complex128).tofile(fh)
    n = NCC(infile_prefix=str(tmp_path) + "/", num_pixels_y1=32, num_pixels_y2=8192, over_sample=4, write_maps=False)
    warm = NCC(infile_prefix=str(tmp_path) + "/", num_pixels_y1=32, num_pixels_y2=32, write_maps=False)
    warm.run()
    before = free_memory(n.lib)
    n.run()
    held = before - free_memory(n.lib)
    warm.close()
    say(f"[ncc memory] path {n.lib.get_crossing_path(n.obj)}, {held >> 20} MB held")
    assert n.lib.get_crossing_path(n.obj) == 2 and n.num_caustic_crossings.max() > 0
    assert held < 384 << 20
    n.close()
    # the same of an object whose lists sufficed for its first run
    with open(tmp_path / "ccf_caustics.bin", "wb") as fh:
        np.array([1, rows.shape[1]], dtype=np.int32).tofile(fh)
        np.ascontiguousarray(rows[:1], dtype=np.complex128).tofile(fh)
    n = NCC(infile_prefix=str(tmp_path) + "/", num_pixels_y1=32, num_pixels_y2=8192, over_sample=4, write_maps=False)
    before = free_memory(n.lib)
    n.run()
    assert n.lib.get_crossing_path(n.obj) == 1
    with open(tmp_path / "ccf_caustics.bin", "wb") as fh:
        np.array(rows.shape, dtype=np.int32).tofile(fh)
        np.ascontiguousarray(rows, dtype=np.complex128).tofile(fh)
    n.run()
    held = before - free_memory(n.lib)
    say(f"[ncc memory] second run: path {n.lib.get_crossing_path(n.obj)}, {held >> 20} MB held")
    assert held < 384 << 20
    n.close()


def test_failed_crossings_leave_zeros(tmp_path):
    """A run that fails on the device (an over-sampled grid past its memory) leaves a map of zeros,
    the first time and after a run that held counts, never what memory happened to hold."""
    from irs_amd.microlensing.NCC.ncc import NCC
    rows = astroids(np.random.default_rng(1), 50, (1, 1), 1.0)
    with open(tmp_path / "ccf_caustics.bin", "wb") as fh:
        np.array(rows.shape, dtype=np.int32).tofile(fh)
        np.ascontiguousarray(rows, dtype=np.complex128).tofile(fh)
    for first in (True, False):
        n = NCC(infile_prefix=str(tmp_path) + "/", num_pixels_y1=300, num_pixels_y2=200, over_sample=0, write_maps=False)
        if not first:
            n.run()
            assert n.num_caustic_crossings.max() > 0
        n.over_sample = 12
        with pytest.raises(Exception, match="Error running NCC"):
            n.run()
        counts = np.ctypeslib.as_array(n.lib.get_num_crossings(n.obj), shape=(200, 300))
        assert not counts.any()
        n.close()


@pytest.mark.parametrize("n", [262143, 262144, 262145, 600001])
def test_star_fields_come_back_in_pieces(tmp_path, n):
    """Stars return through a buffer of 2^18 rows: fields of less than one piece, one, and
    several with a remainder come back whole, and what the device keeps for it stays small."""
    from irs_amd.microlensing.IPM.ipm import IPM
    rng = np.random.default_rng(n)
    stars = np.column_stack([disk(rng, n, 39.0), rng.uniform(0.5, 1.5, n) * 16.0 / n])
    write_field(tmp_path / "stars.bin", stars, 40.0)
    m = IPM(kappa_tot=0.3, shear=0.3, light_loss=0.01, starfile=str(tmp_path / "stars.bin"), half_length_y1=0.5, half_length_y2=0.5,
            num_pixels_y1=16, num_pixels_y2=16, is_double=True, expansion_order=3)
    m.prepare()
    assert m.lib.ipm_build(m.obj, 0)
    before = free_memory(m.lib)
    got = np.ctypeslib.as_array(m.lib.get_stars(m.obj), shape=(n, 3)).copy()
    held = before - free_memory(m.lib)
    say(f"[stars] {n}: {held >> 20} MB held")
    np.testing.assert_array_equal(got[np.lexsort(got.T)], stars[np.lexsort(stars.T)])
    assert held <= 8 << 20
    m.close()


def test_large_deflection_calls_give_their_memory_back(tmp_path):
    """The points of a call stay on the device for the next one up to 2^21 of them; a call of more
    frees them, and both give the same deflections."""
    rng = np.random.default_rng(5)
    m = built(tmp_path / "stars.bin", np.column_stack([disk(rng, 500, 39.0), np.full(500, 16.0 / 500)]), 8)
    z = 20 * (rng.random((1 << 21) + 1) - 0.5) + 1j * (rng.random((1 << 21) + 1) - 0.5)
    m.deflect(z[:10])
    before = free_memory(m.lib)
    w = m.deflect(z)
    assert before - free_memory(m.lib) < 8 << 20
    np.testing.assert_array_equal(m.deflect(z[:-1]), w[:-1])
    m.close()


@pytest.mark.parametrize("n", [0, -1, -16, -20, -31, -40])
def test_timed_request_without_rows_is_refused(n):
    """No rows to time, and counts below none, give the error value."""
    from irs_amd.microlensing.Surrogate import surrogate as S
    s = S.HistogramSurrogate(max_batch=64, seed=1)
    x = np.zeros((1, 6), dtype=np.float32)
    assert S.lib.surrogate_time_predict(s.obj, x.ctypes.data_as(ctypes.POINTER(ctypes.c_float)), n, 3) == -1.0
    assert s.seconds_per_histogram(x) > 0
    s.close()
