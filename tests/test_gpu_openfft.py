"""The line FFTs of the open boundary (k_fft) against the oracle's direct sum, at padded lengths of every
radix and at line counts that leave a block's last lines empty.  Needs a HIP device."""
import numpy as np
import pytest

from juliatdgl_amd.scheme import Grid, box_masks, make_stepper
from juliatdgl_amd.state import initial_state
from test_oracle_open import _two_band

pytestmark = pytest.mark.gpu


# cells; one more on each side: links n = cells + 2 and nodes n = cells + 3 along an axis, padded to the next
# 2^a 3^b 5^c >= 2n - 1
@pytest.mark.parametrize("cells", [(12, 6, 4),      # 27, 30 | 15, 18 | 12, 15
                                   (2, 3, 13),      # 8, 9 | 9, 12 | 30, 32: short lines, 64 a block
                                   (41, 5, 3),      # 90, 90 | 15, 15 | 9, 12
                                   (119, 4, 2),     # 243: 3s only
                                   (310, 3, 2),     # 625: 5s only
                                   (1021, 3, 2)])   # 2048: the longest line, one a block
def test_line_ffts_against_the_direct_sum(cells):
    """h_δ after its first recomputation.  Both sides round θ_δ by a few ulp of its maximum times the
    logarithm of the padded size, 1e-12 of it at most; a face is four links over dx²."""
    from oracle.oracle import Oracle
    from juliatdgl_amd.hip import HipStepper, device_count
    if device_count() < 1:
        pytest.fail("no HIP device visible")
    md = _two_band()
    gr = Grid.make(*cells, dx=0.5)
    st = make_stepper(md, gr, box_masks(gr), selffield_bc="open", open_every=0.05)
    s0 = initial_state(md, gr, st.masks, 0.03)
    HJ = st.selffield(0.3)
    o = Oracle(st)
    o.set_state(s0)
    o.step(1, 0.03, HJ)
    theta, _ = o.open_fields()
    _, _, want = o.open_state()
    print(f"[gpu] open line FFTs: {cells}", flush=True)
    d = HipStepper(st)
    try:
        d.upload(s0)
        d.step(1, 0.03, HJ)
        cnt, _, got = d.get_open()
    finally:
        d.close()
    tol = 4e-12 * max(np.max(np.abs(t)) for t in theta) / 0.5 ** 2
    assert max(np.max(np.abs(w)) for w in want) > 1e3 * tol
    for a, b in zip(got, want):
        assert np.max(np.abs(a - b)) <= tol
