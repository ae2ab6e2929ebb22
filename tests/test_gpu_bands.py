"""The bands' stages and the field pass (k_bands), and the curl, the ghosts and the noise clock
(k_curl_ghosts), in common launches against a launch each (TDGL_HIP_MERGE=0): the same bits.  Needs a HIP device."""
import numpy as np
import pytest

from cases import make_case, seed_state

pytestmark = pytest.mark.gpu


def _case(name):
    if not name.startswith("noise"):
        st, _ = make_case(name)
        s0, pcg, H, HJ = seed_state(st)
        return st, s0, pcg, H, HJ
    from juliatdgl_amd.sweep import RunSpec, state_of, stepper_of
    # 65 x 5 nodes across: one node past a block's width, one row past its height
    spec = RunSpec(0, 66, 6, 4, 0.4, hole=1.0, noise=1e-3, bands=int(name[-1]))
    st = stepper_of(spec)
    return st, state_of(spec, st), None, spec.H, st.selffield(spec.J)


@pytest.mark.parametrize("name", ["production", "no_extrap", "rkl", "hard", "explicit", "explicit_padding", "three_aniso", "three_frustrated",
                                  "kwt10", "kwt10_pcg", "qp_two", "qp_three", "open", "noise2", "noise3"])
def test_merged_bands_give_the_same_bits(name, monkeypatch):
    from juliatdgl_amd.hip import HipStepper, device_count
    if device_count() < 1:
        pytest.fail("no HIP device visible")
    st, s0, pcg, H, HJ = _case(name)
    outs = []
    for v in ("0", "1"):
        print(f"[gpu] TDGL_HIP_MERGE={v}: {name}", flush=True)
        monkeypatch.setenv("TDGL_HIP_MERGE", v)
        d = HipStepper(st)
        try:
            d.upload(s0)
            if pcg is not None:
                d.set_pcg(pcg)
            for _ in range(3):
                d.step(5, H, HJ)
            outs.append(d.download())
        finally:
            d.close()
    for (k, a), (_, b) in zip(outs[0].arrays(), outs[1].arrays()):
        assert np.array_equal(a, b), k


@pytest.mark.parametrize("name,own", [("kwt10_pcg", 40), ("kwt10", 40), ("production", 0), ("euler_substeps", 0)])
def test_bands_in_turn_share_their_work_arrays(name, own, monkeypatch):
    """A second band's own W, W2 (32 B a node) and frame rate (8 B) are there only where the bands step side by side:
    with TDGL_HIP_MERGE=0 one set serves all."""
    from juliatdgl_amd.hip import HipStepper
    st, _ = make_case(name)
    print(f"[gpu] work arrays of {name}", flush=True)
    held = {}
    for v in ("0", "1"):
        monkeypatch.setenv("TDGL_HIP_MERGE", v)
        d = HipStepper(st)
        held[v] = d.stats()["device_bytes"]
        d.close()
    nodes = (st.grid.Nx + 1) * (st.grid.Ny + 1) * (st.grid.Nz + 1)
    extra = held["1"] - held["0"]
    print(f"    {extra} B more side by side ({extra / nodes:.1f} a node)", flush=True)
    assert extra >= own * nodes if own else extra == 0
