"""The plane packer against its definition, element by element."""

import numpy as np
import pytest

from metalfish_amd import backend


@pytest.mark.parametrize("batch", [1, 3, 17])
def test_pack_planes_definition(batch):
    """Masks and values of planes holding zeros of both signs, NaN, infinities
    and denormals, each square of a plane in turn the first one set."""
    rng = np.random.default_rng(batch)
    planes = np.zeros((batch, 112, 64), np.float32)
    odd = np.array([1.0, -0.0, np.nan, np.inf, 1e-45, -2.5, 0.0], np.float32)
    for b in range(batch):
        for p in range(112):
            first = (b * 112 + p) % 65
            planes[b, p, first:] = rng.choice(odd, 64 - first)
    masks, values = backend.pack_planes(planes)
    for b in range(batch):
        for p in range(112):
            v = planes[b, p]
            if (p < 104 and p % 13 == 12) or p in (106, 107) or p >= 109:
                mask = (1 << 64) - 1 if v[0] != 0 else 0
                value = v[0]
            else:
                on = np.flatnonzero(v != 0)
                mask = sum(1 << int(s) for s in on)
                value = v[on[0]] if on.size else np.float32(0)
            assert int(masks[b, p]) == mask, (b, p)
            assert np.float32(values[b, p]).tobytes() == np.float32(value).tobytes(), (b, p)
