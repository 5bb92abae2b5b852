"""Copies between host and device memory: page-locked slots up to 256 KiB, the runtime's staging above."""

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w", [1, 16383, 16384, 16385, 70001])
@pytest.mark.parametrize("locked", [False, True])
def test_planar_round_trip_is_exact_on_both_sides_of_the_slot_size(w, locked):
    from zenjpegai_amd import nn

    eng = nn.Engine(0, "f32")
    rng = np.random.default_rng(w)
    # Every slot in turn and the first ones again. (Each call waits for its own copy, so no slot is taken
    # while it is still being read.)
    xs = [torch.from_numpy(rng.standard_normal((4, 1, w)).astype(np.float32)) for _ in range(7)]
    if locked:
        xs = [x.pin_memory() for x in xs]
    xs = [x.numpy() for x in xs]
    ts = [nn.BTensor.from_planar(eng, x) for x in xs]
    for x, t in zip(xs, ts):
        np.testing.assert_array_equal(t.to_planar(), x)
    eng.close()
