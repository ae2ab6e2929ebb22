"""The separable solve by sectors (k_sect_sep; TDGL_HIP_SECT=1: also below the sizes it is chosen at) against the
solve it replaces (TDGL_HIP_SECT=0), and batched against alone.  Needs a HIP device."""
import numpy as np
import pytest

from cases import compare_states, mgb2
from juliatdgl_amd.scheme import Grid, box_masks, make_stepper
from juliatdgl_amd.state import seeded_state

pytestmark = pytest.mark.gpu


def _steppers(sizes):
    from juliatdgl_amd.hip import HipStepper, device_count
    if device_count() < 1:
        pytest.fail("no HIP device visible")
    out = []
    for nx, ny, nz in sizes:
        gr = Grid.make(nx, ny, nz, dx=0.5)
        st = make_stepper(mgb2(), gr, box_masks(gr))
        d = HipStepper(st)
        d.upload(seeded_state(st.model, st.grid, st.masks, 0.03, seed=nx))
        out.append((st, d))
    return out


# nodes n = cells + 1 an axis: one and two tiles past a whole number along y, both parities of each count, one to
# three z tiles (2, 16, 17, 33 half nodes), the least z (3 nodes), more than four y tiles a wave
SIZES = [(160, 7, 2), (161, 8, 3), (9, 96, 31), (10, 127, 33), (5, 129, 20), (6, 98, 64), (4, 223, 62)]


@pytest.mark.parametrize("size", SIZES)
def test_sectors_match_the_transforms(size, monkeypatch):
    """Five steps: both sides are FP64 products of at most 256 terms a pass, 1e-14 of the field's scale a solve;
    the bound is 1e-12."""
    print(f"[gpu] separable solve by sectors {size}", flush=True)
    res = []
    for sect in (True, False):
        monkeypatch.setenv("TDGL_HIP_SECT", "1" if sect else "0")
        (st, d), = _steppers([size])
        d.step(3, 0.03, st.selffield(0.3))
        d.profile(True)
        d.step(2, 0.03, st.selffield(0.3))
        pr = d.profile_get()
        d.profile(False)
        res.append((d.download(), pr["sep_transform_f64"][0], pr["sep_fold"][0]))
        d.close()
    assert res[0][1:] == (4, 0)
    assert any(not np.array_equal(u, v) for (_, u), (_, v) in zip(res[0][0].arrays(), res[1][0].arrays()))  # two routes
    errs = compare_states(res[0][0], res[1][0])
    worst = max(v for k, v in errs.items() if not k.startswith(("U", "V")))
    print(f"    worst {worst:.2e}", flush=True)
    assert worst <= 1e-12, errs


@pytest.mark.parametrize("sizes", [[(161, 8, 3), (10, 127, 33), (4, 223, 62)], [(40, 240, 20), (20, 12, 6)]])
def test_batched_sectors(sizes, monkeypatch):
    """A batch of sectors leaves each run where its own steps do, to the bit; beside a run whose own step takes the
    planes all take the single-axis passes, the same values to rounding."""
    from juliatdgl_amd.hip import HipBatch
    if len(sizes) == 3:
        monkeypatch.setenv("TDGL_HIP_SECT", "1")
    print(f"[gpu] batched separable sectors {sizes}", flush=True)
    H, alone, got = 0.03, [], []
    for st, d in _steppers(sizes):
        d.step(4, H, st.selffield(0.3))
        alone.append(d.download())
        d.close()
    runs = _steppers(sizes)
    b = HipBatch([d for _, d in runs])
    b.step(4, np.full(len(runs), H), np.array([st.selffield(0.3) for st, _ in runs]))
    got = [d.download() for _, d in runs]
    b.close()
    for x, y in zip(alone, got):
        if len(sizes) == 3:
            for (k, u), (_, v) in zip(x.arrays(), y.arrays()):
                assert np.array_equal(u, v), k
        else:
            errs = compare_states(x, y)
            assert max(v for k, v in errs.items() if not k.startswith(("U", "V"))) <= 1e-12, errs
    for _, d in runs:
        d.close()


@pytest.mark.parametrize("graph", ["1", "0"])
@pytest.mark.parametrize("sizes,paths", [([(170, 100, 30), (170, 100, 20), (60, 200, 14)], [2, 1, 2]),
                                         ([(256, 128, 20), (200, 100, 24)], [1, 1])])
def test_batched_sectors_beside_folds(sizes, paths, graph, monkeypatch):
    """Wide runs, some by sectors and some by the folded transforms (the last two on different kernels of them), in one
    batch, replayed or launched from the host: each is where its own steps leave it, to the bit."""
    from juliatdgl_amd.hip import HipBatch
    H = 0.03
    monkeypatch.setenv("TDGL_HIP_GRAPH", graph)
    print(f"[gpu] batched sectors beside folds {sizes}", flush=True)
    alone = []
    for st, d in _steppers(sizes):
        d.step(4, H, st.selffield(0.3))
        alone.append((d.download(), d.stats()["folded"]))
        d.close()
    assert [f for _, f in alone] == paths
    runs = _steppers(sizes)
    b = HipBatch([d for _, d in runs])
    for _ in range(2):
        b.step(2, np.full(len(runs), H), np.array([st.selffield(0.3) for st, _ in runs]))
    got = [d.download() for _, d in runs]
    b.close()
    for _, d in runs:
        d.close()
    for (x, _), y in zip(alone, got):
        for (k, u), (_, v) in zip(x.arrays(), y.arrays()):
            assert np.array_equal(u, v), k


@pytest.mark.parametrize("size,by_sectors", [((4, 128, 64), False), ((10, 128, 64), False), ((6, 170, 80), False),
                                             ((11, 128, 64), True), ((4, 128, 40), True), ((60, 200, 14), True)])
def test_few_sectors_keep_the_planes(size, by_sectors):
    """Deep planes, which the folds do not take, go by sectors from 48 workgroups on (12 nodes along x); where the folds
    are the other way, at any width."""
    (_, d), = _steppers([size])
    folded = d.stats()["folded"]
    d.close()
    assert (folded == 2) == by_sectors, folded
