"""The PCG by sectors (csrc/sect.hip) against the general iteration (TDGL_HIP_SECT=0) and the oracle, and the
inputs it leaves to the general iteration.  Needs a HIP device."""
import numpy as np
import pytest

from cases import compare_states, mgb2, seed_state
from juliatdgl_amd.scheme import Grid, box_masks, make_stepper
from juliatdgl_amd.state import seeded_state

pytestmark = pytest.mark.gpu


def _run(st, s0, H, HJ, n, monkeypatch, sect, calls=1):
    from juliatdgl_amd.hip import HipStepper, device_count
    if device_count() < 1:
        pytest.fail("no HIP device visible")
    if sect:
        monkeypatch.delenv("TDGL_HIP_SECT", raising=False)
    else:
        monkeypatch.setenv("TDGL_HIP_SECT", "0")
    d = HipStepper(st)
    try:
        d.upload(s0)
        for _ in range(calls):
            d.step(n, H, HJ)
        d.profile(True)
        d.step(1, H, HJ)
        took = d.profile_get()["pcg_sectors"][0]
        d.profile(False)
        return d.download(), took, d.stats()
    finally:
        d.close()


def _core(errs):
    return max(v for k, v in errs.items() if not k.startswith(("U", "V")))


# nodes per axis n = cells + 2 buf - 1: three nodes, odd and even counts, half extents at and past whole
# 16-point tiles (31, 32 | 33, 34 nodes), one to three z tiles (half 16, 17, 33, 46), each elements-a-thread instance
# (2, 4, 6, 8, 10, 11 x 512), more ghosts than threads (90 x 4 half nodes), the largest sector (40 x 46 nodes), and y tiles
# in rounds: 5 and 6 a wave of 12 x 3, 7 x 5 and 21 x 2
SIZES = [(2, 2, 2, 1), (5, 4, 3, 2), (9, 13, 8, 2), (20, 12, 28, 2), (17, 29, 30, 2), (33, 30, 31, 2), (34, 31, 29, 2), (12, 60, 28, 2),
         (6, 28, 62, 2), (70, 66, 13, 2), (4, 92, 32, 2), (4, 120, 36, 2),
         (4, 140, 44, 2), (3, 177, 5, 2), (9, 76, 88, 2), (3, 360, 14, 2), (4, 220, 30, 2), (2, 640, 5, 2)]


@pytest.mark.parametrize("nx,ny,nz,buf", SIZES)
def test_sectors_match_the_general_iteration(nx, ny, nz, buf, monkeypatch):
    """Both solve to ||r|| <= tol ||b||, so their increments differ by at most 2 tol ||b|| / min D a step (min D =
    0.01): 2e-10 of ||b|| at tol 1e-12, 1.4e-9 in the seven steps' sum; the bound is 1e-8 of each field's scale.  Seven
    steps launched and replayed, the iterations at most a quarter and two a step more."""
    gr = Grid.make(nx, ny, nz, dx=0.5, buf=buf)
    st = make_stepper(mgb2(), gr, box_masks(gr), sigma_vac=0.01, pcg_tol=1e-12)
    H, HJ = 0.03, st.selffield(0.3)
    s0 = seeded_state(st.model, st.grid, st.masks, H, seed=nx)
    print(f"[gpu] sectors {nx}x{ny}x{nz} buf {buf}", flush=True)
    a, na, sa = _run(st, s0, H, HJ, 3, monkeypatch, True, calls=2)
    b, nb, sb = _run(st, s0, H, HJ, 3, monkeypatch, False, calls=2)
    assert (na, nb) == (1, 0)
    errs = compare_states(a, b)
    print(f"    worst {_core(errs):.2e}, iterations {sa['pcg_iters']} / {sb['pcg_iters']}", flush=True)
    assert _core(errs) <= 1e-8, errs
    assert sa["pcg_iters"] <= sb["pcg_iters"] + sb["pcg_iters"] // 4 + 2 * sb["steps"]
    assert sa["rollbacks"] == 0


def test_refinement_goes_by_sectors(monkeypatch):
    """pcg_refine where the sectors apply, against its Float32 inner solves: the bound of
    test_sectors_match_the_general_iteration."""
    gr = Grid.make(33, 20, 9, dx=0.5, buf=2)
    st = make_stepper(mgb2(), gr, box_masks(gr), sigma_vac=0.01, pcg_tol=1e-12, pcg_refine=True)
    H, HJ = 0.03, st.selffield(0.3)
    s0 = seeded_state(st.model, st.grid, st.masks, H, seed=4)
    a, na, _ = _run(st, s0, H, HJ, 3, monkeypatch, True, calls=2)
    b, nb, _ = _run(st, s0, H, HJ, 3, monkeypatch, False, calls=2)
    assert (na, nb) == (1, 0)
    errs = compare_states(a, b)
    assert _core(errs) <= 1e-8, errs


def test_sectors_repeat_to_the_bit(monkeypatch):
    """The sums of a sector run in a fixed order: two handles give the same bits, replayed or launched."""
    gr = Grid.make(33, 20, 9, dx=0.5, buf=2)
    st = make_stepper(mgb2(), gr, box_masks(gr), sigma_vac=0.01)
    H, HJ = 0.03, st.selffield(0.3)
    s0 = seeded_state(st.model, st.grid, st.masks, H, seed=4)
    a, _, _ = _run(st, s0, H, HJ, 5, monkeypatch, True, calls=3)
    monkeypatch.setenv("TDGL_HIP_GRAPH", "0")
    b, _, _ = _run(st, s0, H, HJ, 5, monkeypatch, True, calls=3)
    for (k, x), (_, y) in zip(a.arrays(), b.arrays()):
        assert np.array_equal(x, y), k


@pytest.mark.parametrize("what", ["x", "y", "z", "values", "large"])
def test_other_conductivities_take_the_general_iteration(what, monkeypatch):
    """D that varies along x, is not its own mirror image along y or z, takes more than 16 values, or planes
    whose sectors do not fit a workgroup (75 x 38 nodes): the general iteration runs, and agrees with the
    oracle on the small grid."""
    from oracle.oracle import Oracle
    big = what == "large"
    gr = Grid.make(6, 134, 60, dx=0.5, buf=8) if big else Grid.make(20, 13, 6, dx=0.5, buf=2)
    st = make_stepper(mgb2(), gr, box_masks(gr), sigma_vac=0.01, pcg_tol=1e-12)
    if not big:
        D = [np.array(x, order="F") for x in st.D]
        if what == "x":
            D[0][7] *= 0.5
        elif what == "y":
            D[1][:, 3] *= 0.5
        elif what == "z":
            D[2][:, :, 2] *= 0.5
        else:
            j = np.arange(D[0].shape[1])
            D[0] *= (1 + 0.01 * np.minimum(j, j[::-1]))[None, :, None] * (1 + 0.003 * np.minimum(np.arange(gr.Nz + 1),
                                                                          np.arange(gr.Nz + 1)[::-1]))[None, None]
        st.D = tuple(D)
    H, HJ = 0.03, st.selffield(0.3)
    s0 = seeded_state(st.model, st.grid, st.masks, H, seed=2)
    got, took, _ = _run(st, s0, H, HJ, 1 if big else 5, monkeypatch, True)
    assert took == 0
    if not big:
        o = Oracle(st)
        o.set_state(s0)
        o.step(6, H, HJ)
        errs = compare_states(got, o.get_state())
        assert _core(errs) <= 1e-10, errs


@pytest.mark.parametrize("tol,maxit,bound", [(1e-8, 500, 2e-6), (1e-12, 500, 2e-10), (1e-12, 3, 1.0)])
def test_sectors_match_the_oracle(tol, maxit, bound, monkeypatch):
    """Against the oracle's PCG on a wedge-free box with even node counts, and with the iterations limited to
    three: each sector stops there, and the step goes on.  Two solutions within tol ||b|| differ by at most
    2 tol ||b|| / min D (min D = 0.01), and the steps' ||b|| add up to the field's scale: 200 tol."""
    from oracle.oracle import Oracle
    gr = Grid.make(27, 13, 7, dx=0.5, buf=2)
    st = make_stepper(mgb2(), gr, box_masks(gr), sigma_vac=0.01, pcg_tol=tol, pcg_maxit=maxit)
    s0, _, H, HJ = seed_state(st, warm_steps=0)
    got, took, stt = _run(st, s0, H, HJ, 9, monkeypatch, True)
    assert took == 1
    if maxit == 3:
        assert stt["last_iters"] <= 3 and all(np.isfinite(g).all() for g in got.G)
        return
    o = Oracle(st)
    o.set_state(s0)
    o.step(10, H, HJ)
    errs = compare_states(got, o.get_state())
    print(f"[gpu] sectors against the oracle, tol {tol:g}: {_core(errs):.2e}", flush=True)
    assert _core(errs) <= bound, errs


@pytest.mark.parametrize("nx,ny,nz", [(200, 110, 34), (200, 250, 4), (8, 640, 5), (16, 60, 88)])
def test_sectors_are_no_slower_than_the_general_iteration(nx, ny, nz, monkeypatch):
    """Planes of three to six y tiles a wave: a step by sectors takes no longer than the general iteration's (half of it,
    measured; the best of four calls a side)."""
    from juliatdgl_amd.hip import HipStepper
    gr = Grid.make(nx, ny, nz, dx=0.5, buf=2)
    best = {}
    for sect in ("0", None):
        if sect:
            monkeypatch.setenv("TDGL_HIP_SECT", sect)
        else:
            monkeypatch.delenv("TDGL_HIP_SECT", raising=False)
        st = make_stepper(mgb2(), gr, box_masks(gr), sigma_vac=0.01)
        d = HipStepper(st)
        d.upload(seeded_state(st.model, st.grid, st.masks, 0.03, seed=1))
        ms = []
        for _ in range(6):
            t = d.stats()["device_ms"]
            d.step(6, 0.03, st.selffield(0.3))
            ms.append((d.stats()["device_ms"] - t) / 6)
        d.close()
        best[sect] = min(ms[2:])
    print(f"[gpu] {nx}x{ny}x{nz}: general {1e3 * best['0']:.0f} us a step, sectors {1e3 * best[None]:.0f}", flush=True)
    assert best[None] <= best["0"]


def test_sectors_are_no_further_from_the_solution(monkeypatch):
    """Six cycles of 96x48x24 cells with a wedge: the fields are no further from those of an all-FP64 solve to 1e-13 than
    the general iteration's, by either path of its preconditioner (2.3e-9 against 2.5e-9 and 7.1e-9, measured)."""
    from juliatdgl_amd.hip import HipStepper
    from juliatdgl_amd.scheme import two_band, wedge_masks
    gr = Grid.make(96, 48, 24, dx=0.5, buf=2)
    H = 0.03

    def run(env, **kw):
        for k, v in env.items():
            monkeypatch.setenv(k, v)
        st = make_stepper(two_band(xi_ratio=4.0, kappa=2.0), gr, wedge_masks(gr), sigma_vac=0.01, **kw)
        d = HipStepper(st)
        for k in env:
            monkeypatch.delenv(k)
        d.upload(seeded_state(st.model, gr, st.masks, H, seed=3))
        for _ in range(6):
            d.step(40, H, st.selffield(0.3))
        out = d.download()
        d.close()
        return out
    print("[gpu] sectors, distance from the solution, 96x48x24", flush=True)
    ref = run({}, pcg_fast=False, pcg_f32=False, pcg_tol=1e-13)

    def off(s):
        return max(np.linalg.norm((a - b).ravel()) / np.linalg.norm(b.ravel()) for (_, a), (_, b) in zip(s.arrays(), ref.arrays())
                   if np.any(b))
    sect = off(run({}))
    general = [off(run({"TDGL_HIP_SECT": "0", "TDGL_HIP_FOLD": f})) for f in ("1", "0")]
    print(f"    sectors {sect:.2e}, folds {general[0]:.2e}, full length {general[1]:.2e}", flush=True)
    assert sect <= min(general)
