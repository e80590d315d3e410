"""GPU thermal Monte Carlo: parity with the FP64 oracle (same Philox streams,
same epoch schedule), bitwise reproducibility, closed forms, error paths."""
import numpy as np
import pytest

import oracle
from pdspy_amd import configs, rt
from tests.helpers import dT_stats, oracle_arrays

pytestmark = pytest.mark.gpu


def _gpu_T(arr, nphot, seed, **opts):
    dm = rt.DeviceModel(arr)
    st = dm.thermal(nphot, seed, count_visits=1, **opts)
    T, vis = dm.temperature(with_visits=True)
    return T, vis, st


def test_thermal_matches_oracle_disk():
    # 1e6 packets: independent seeds of the oracle already differ by median
    # 0.14 %, p99 5.2 % here; the same seed shares most packet histories
    print("case: disk 32x32, 1e6 packets, seed 7", flush=True)
    arr = oracle_arrays(configs.disk_c1(nr=32, nt=32))
    n = 1000000
    Tg, vg, sg = _gpu_T(arr, n, 7, max_events=20000)
    To, vo, so = oracle.thermal(arr, n, seed=7, max_events=20000, lagged=True)
    med, p99, ncell = dT_stats(To, Tg, vo)
    print("median %.2e p99 %.2e cells %d" % (med, p99, ncell))
    assert ncell > 500
    assert med <= 0.01 and p99 <= 0.05
    assert sg["n_epochs"] == so["n_epochs"]
    assert abs(int(vg.sum()) - int(vo.sum())) <= 0.01 * vo.sum()
    for k in ("n_abs", "n_scat", "n_cross"):
        assert sg[k] == pytest.approx(so[k], rel=0.02), k
    assert sg["n_escape"] + sg["n_killed"] == n


def test_thermal_matches_oracle_disk_envelope_two_species():
    print("case: disk+envelope 48x24, 5e4 packets, seed 1", flush=True)
    arr = oracle_arrays(configs.disk_envelope(nr=48, nt=24))
    n = 50000
    Tg, vg, sg = _gpu_T(arr, n, 1, max_events=20000)
    To, vo, so = oracle.thermal(arr, n, seed=1, max_events=20000, lagged=True)
    med, p99, ncell = dT_stats(To, Tg, vo)
    print("median %.2e p99 %.2e cells %d" % (med, p99, ncell))
    assert med <= 0.01 and p99 <= 0.05
    # species share one opacity: equal temperatures wherever both are present
    both = (arr["rho"][0].ravel() > 0) & (arr["rho"][1].ravel() > 0)
    assert np.array_equal(Tg[0][both], Tg[1][both])


def test_thermal_matches_oracle_two_absorption_groups():
    """Disk and envelope with different dust (as pdspy's fits have them): two
    absorption groups, the (2 species, 2 groups) kernel variant."""
    print("case: disk+envelope 48x24, distinct dust, 5e4 packets, seed 2", flush=True)
    arr = oracle_arrays(configs.disk_envelope(nr=48, nt=24))
    lam = arr["lam_um"]
    arr["kabs"] = np.array(arr["kabs"], dtype=float)
    arr["ksca"] = np.array(arr["ksca"], dtype=float)
    arr["kabs"][0] = np.where(lam > 1.0, 1e3 * lam ** -0.6, 1e3)   # grown grains in the disk
    arr["ksca"][0] = 2.0 * arr["kabs"][0]
    n = 50000
    Tg, vg, sg = _gpu_T(arr, n, 2, max_events=20000)
    To, vo, so = oracle.thermal(arr, n, seed=2, max_events=20000, lagged=True)
    med, p99, ncell = dT_stats(To, Tg, vo)
    print("median %.2e p99 %.2e cells %d" % (med, p99, ncell))
    assert med <= 0.01 and p99 <= 0.05
    both = (arr["rho"][0].ravel() > 0) & (arr["rho"][1].ravel() > 0)
    assert both.sum() > 100 and not np.array_equal(Tg[0][both], Tg[1][both])


def test_thermal_hg_3d_matches_oracle():
    print("case: 3D spiral 16x8x8 HG g=0.6, 2e4 packets", flush=True)
    arr = oracle_arrays(configs.spiral_3d(nr=16, nt=8, nphi=8))
    n = 20000
    Tg, vg, sg = _gpu_T(arr, n, 2, max_events=20000)
    To, vo, so = oracle.thermal(arr, n, seed=2, max_events=20000, lagged=True)
    med, p99, ncell = dT_stats(To, Tg, vo)
    print("median %.2e p99 %.2e cells %d" % (med, p99, ncell))
    assert med <= 0.01 and p99 <= 0.05


def test_thermal_mrw_matches_oracle():
    print("case: disk+envelope 64x32 MRW, 1.5e5 packets, seed 4", flush=True)
    arr = oracle_arrays(configs.disk_envelope(nr=64, nt=32))
    n = 150000
    Tg, vg, sg = _gpu_T(arr, n, 4, max_events=1000000, mrw=1)
    To, vo, so = oracle.thermal(arr, n, seed=4, max_events=1000000, lagged=True, mrw=True)
    med, p99, ncell = dT_stats(To, Tg, vo)
    print("median %.2e p99 %.2e cells %d  mrw steps gpu %d oracle %d"
          % (med, p99, ncell, sg["n_mrw"], so["n_mrw"]))
    assert med <= 0.01 and p99 <= 0.05
    assert sg["n_mrw"] == pytest.approx(so["n_mrw"], rel=0.05)
    assert sg["n_killed"] == 0


def test_thermal_bitwise_reproducible_across_launch_shapes():
    print("case: determinism disk 24x24, 3e4 packets", flush=True)
    arr = oracle_arrays(configs.disk_c1(nr=24, nt=24))
    dm = rt.DeviceModel(arr)
    out = []
    for bs, bpc, fc in [(256, 0, 0), (256, 0, 0), (64, 1, 0), (128, 3, 0), (256, 0, 1)]:
        dm.thermal(30000, 9, max_events=20000, block_size=bs, blocks_per_cu=bpc,
                   free_cus_per_xcd=fc)
        out.append(dm.temperature())
    for T in out[1:]:
        assert np.array_equal(T, out[0])
    dm.thermal(30000, 10, max_events=20000)
    assert not np.array_equal(dm.temperature(), out[0])


def test_thermal_thin_shell_closed_form_gpu():
    from tests.test_oracle import _thin_shell_model, _star_lum
    m = _thin_shell_model()
    T, vis, st = _gpu_T(m, 400000, 4)
    L = _star_lum(m["lam_um"], 1.392e11, 4000.0)
    assert st["lum"] == pytest.approx(L, rel=1e-9)
    rw = m["rw"]
    for i in range(4):
        e = L * 10.0 * (rw[i + 1] - rw[i]) / (4.0 / 3.0 * np.pi * (rw[i + 1] ** 3 - rw[i] ** 3))
        lo, hi = 1.0, 3000.0
        for _ in range(80):
            mid = np.sqrt(lo * hi)
            if oracle.emis_per_gram(np.full(100, 10.0), m["lam_um"], mid) < e:
                lo = mid
            else:
                hi = mid
        Tc = T[0].reshape(4, 4)[:, i]
        assert np.all(np.abs(Tc / lo - 1) < 5e-3), (i, Tc, lo)


def test_thermal_event_cap_kills_and_counts():
    arr = oracle_arrays(configs.disk_c1(nr=16, nt=16))
    T, vis, st = _gpu_T(arr, 5000, 3, max_events=10)
    assert st["n_killed"] > 0
    assert st["n_killed"] + st["n_escape"] == 5000


def test_thermal_watchdog_returns_error_not_hang():
    arr = oracle_arrays(configs.disk_c1(nr=16, nt=16))
    dm = rt.DeviceModel(arr)
    from pdspy_amd._lib import RTError
    with pytest.raises(RTError) as e:
        dm.thermal(2000000, 0, max_events=1000000, max_seconds=1e-4)
    assert e.value.code == -4


def test_model_api_fills_grid_temperature():
    m = configs.disk_envelope(nr=32, nt=16)
    st = rt.run_thermal(m, nphot=20000, iseed=5, max_events=20000, return_stats=True,
                        modified_random_walk=False, setthreads=8, verbose=False)
    assert len(m.grid.temperature) == 2
    for T, d in zip(m.grid.temperature, m.grid.density):
        assert T.shape == d.shape and T.dtype == np.float64
        assert np.all(T[d > 0] > 0) or np.mean(T[d > 0] > 0) > 0.9
    assert st["n_escape"] + st["n_killed"] == 20000


def test_invalid_inputs_rejected():
    from pdspy_amd._lib import RTError
    arr = oracle_arrays(configs.disk_c1(nr=8, nt=8))
    bad = dict(arr)
    bad["rho"] = arr["rho"].copy()
    bad["rho"][0, 0, 0, 0] = np.nan
    with pytest.raises(RTError):
        rt.DeviceModel(bad)
    bad = dict(arr)
    bad["rw"] = arr["rw"][::-1].copy()
    with pytest.raises(RTError):
        rt.DeviceModel(bad)


def test_device_density_generator_matches_host_builders():
    # the disk + Ulrich envelope builders on the device against the host ones
    # (scipy brenth for mu0, numpy trapezoids); includes r < Rc cells where the
    # cubic for mu0 has three real roots
    print("case: device density generator vs host builders", flush=True)
    cases = [dict(nr=256, nt=128, mdisk=1e-3, plrho=1.75, plh=1.25, menv=0.1),
             dict(nr=32, nt=16, nphi=6, mdisk=2e-4, plrho=1.5, plh=1.15, menv=0.03),
             dict(nr=64, nt=64, mdisk=3e-5, plrho=1.2, plh=1.05, menv=2e-3, rcent=20.0),
             dict(nr=128, nt=64, mdisk=8e-3, plrho=2.6, plh=1.3, menv=0.25, rcent=120.0)]
    for c in cases:
        host = configs.disk_envelope(**c)
        m = rt.DeviceModel(rt.model_arrays(configs.disk_envelope(
            nr=c["nr"], nt=c["nt"], nphi=c.get("nphi", 1)).grid))
        comps = configs.disk_envelope_components(
            mdisk=c["mdisk"], plrho=c["plrho"], plh=c["plh"], menv=c["menv"],
            rcent=c.get("rcent", 50.0))
        # two stream-ordered generations in a row with no wait between them
        # (the components travel by value): the second one's densities stay
        m.generate_density(configs.disk_envelope_components(
            mdisk=5e-2, plrho=1.0, plh=1.0, menv=1e-4, rcent=10.0))
        m.generate_density(comps)
        got = m.rho_device().cpu().numpy().astype(np.float64)
        want = rt.model_arrays(host.grid)["rho"].reshape(m.nspec, m.ncell).astype(np.float32)
        want = want.astype(np.float64)
        assert got.shape == want.shape
        assert np.array_equal(got > 0, want > 0), c
        rel = np.abs(got - want) / np.maximum(want, 1e-300)
        assert rel.max() <= 2e-7, (c, rel.max())


@pytest.mark.parametrize("max_events,slice_events", [
    (1, 10000), (4, 10000), (5, 10000), (12, 10000), (68, 10000), (69, 10000), (70, 10000),
    (133, 10000), (1000, 10000), (1000, 9), (1000, 10), (1000, 64), (1000, 65), (1000, 73)])
def test_walk_inside_a_thick_cell_counts_every_interaction(max_events, slice_events):
    """Two packets in a cell of optical depth 1e9: neither can leave, so each
    interacts exactly max_events times, wherever a walk of up to 64
    interactions ends (the cap, a slice's last interaction), and every tally
    add is counted once: the temperature equals that of a batch of the same
    run, whose slots and waves are laid out differently, bit for bit."""
    print("case: thick cell, max_events %d, slice %d" % (max_events, slice_events), flush=True)
    arr = oracle_arrays(configs.disk_c1(nr=4, nt=2))
    arr["rho"] = np.full(arr["rho"].shape, 1e-4)
    dm = rt.DeviceModel(arr)
    st = dm.thermal(2, 5, max_events=max_events, slice_events=slice_events)
    assert st["n_killed"] == 2 and st["n_escape"] == 0
    assert st["n_events"] == 2 * max_events == st["n_abs"] + st["n_scat"]
    T = dm.temperature()
    other = rt.DeviceModel(arr)
    b = rt.Batch([other, dm])
    b.thermal([2, 2], [5, 5], max_events=max_events, slice_events=slice_events)
    assert np.array_equal(other.temperature(), T) and np.array_equal(dm.temperature(), T)


@pytest.mark.parametrize("model", ["one group", "two groups", "modified walk", "forward"])
def test_walks_leave_a_run_as_it_is(model):
    """16000 packets in waves of 62 (64-lane blocks, one per CU: a wave looks for walks
    only near the end) and of four and fewer (the default): the interactions
    replayed in walks are the loop's own, so the temperatures and the counts are
    equal bit for bit -- isotropic with one and two absorption groups, with the
    modified random walk, and with forward scattering."""
    print("case: walks, %s" % model, flush=True)
    if model == "forward":
        arr = oracle_arrays(configs.spiral_3d(nr=12, nt=8, nphi=6))
    else:
        arr = oracle_arrays(configs.disk_envelope(nr=24, nt=16))
    if model == "two groups":
        lam = arr["lam_um"]
        arr["kabs"] = np.array(arr["kabs"], dtype=float)
        arr["kabs"][0] = np.where(lam > 1.0, 1e3 * lam ** -0.6, 1e3)
    dm = rt.DeviceModel(arr)
    out = []
    for bs, bpc in [(64, 1), (256, 0)]:
        st = dm.thermal(16000, 3, max_events=20000, block_size=bs, blocks_per_cu=bpc,
                        mrw=1 if model == "modified walk" else 0)
        out.append((dm.temperature(), [st[k] for k in ("n_cross", "n_abs", "n_scat", "n_events",
                                                       "n_escape", "n_killed", "n_mrw")]))
    assert out[0][1] == out[1][1]
    assert np.array_equal(out[0][0], out[1][0])


@pytest.mark.parametrize("model", ["one group", "two groups", "forward"])
@pytest.mark.parametrize("max_events", [69, 133, 1000, 20000])
def test_walk_inside_a_thick_cell_tallies_what_the_loop_does(model, max_events):
    """A walk needs more than eight interactions left in the packet's slice, so with
    slices of eight there are none.  In a run's first epoch a slice only decides
    which slot a deposit goes to: the temperatures, which come from every deposit of
    two packets in cells of optical depth 1e6, and the counts are equal bit for bit
    with walks and without."""
    print("case: thick cell against the loop, %s, max_events %d" % (model, max_events), flush=True)
    if model == "forward":
        arr = oracle_arrays(configs.spiral_3d(nr=4, nt=4, nphi=3))
    else:
        arr = oracle_arrays(configs.disk_envelope(nr=4, nt=2))
    if model == "two groups":
        lam = arr["lam_um"]
        arr["kabs"] = np.array(arr["kabs"], dtype=float)
        arr["kabs"][0] = np.where(lam > 1.0, 1e3 * lam ** -0.6, 1e3)
    # (at 1e9 the adds, in units of 2^-28 of the largest, would round to 0)
    k = np.asarray(arr["kabs"]).max()
    arr["rho"] = np.broadcast_to(1e6 / (k * np.diff(arr["rw"])), arr["rho"].shape).copy()
    out = []
    for slice_events in (8, 10000):
        dm = rt.DeviceModel(arr)
        st = dm.thermal(2, 5, max_events=max_events, slice_events=slice_events)
        assert st["n_epochs"] == 1 and st["n_killed"] == 2
        assert st["n_events"] == 2 * max_events == st["n_abs"] + st["n_scat"]
        out.append((dm.temperature(), [st[k] for k in ("n_cross", "n_abs", "n_scat")]))
    assert out[0][1] == out[1][1] and np.array_equal(out[0][0], out[1][0])
    assert out[0][0].max() > 0
    # the batched instances' walks (the one-group one has its packets in memory meanwhile)
    dms = [rt.DeviceModel(arr) for _ in range(2)]
    st = rt.Batch(dms).thermal([2, 2], [5, 5], max_events=max_events)
    for dm, s in zip(dms, st):
        assert [s[k] for k in ("n_cross", "n_abs", "n_scat")] == out[0][1]
        assert np.array_equal(dm.temperature(), out[0][0])
