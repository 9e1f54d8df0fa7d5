"""Learned compression of a batch with fields too thin to hold a judged cell, odd
sizes and gains that call for fallback: counts and critical points."""
import numpy as np
import pytest
import torch

import cpsz_amd as cz
from cpsz_amd.synth import field_2d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bias", [0.0, 7.5], ids=["no-gain", "gain"])
def test_batch_of_odd_fields(bias):
    shapes = [(3, 50), (64, 97), (40, 3), (1, 7), (5, 33), (97, 131)]
    p = cz.learn_init_params(5)
    p[-1 - 128:] = 0
    p[-1] = bias  # the same gain everywhere
    dev = [tuple(torch.from_numpy(np.ascontiguousarray(x, np.float32)).cuda() for x in field_2d(*s, 60 + k))
           for k, s in enumerate(shapes)]
    torch.cuda.synchronize()
    base, off, size, rounds, boosted, fell = cz.compress_2d_learned_batch_dev(
        [(u.data_ptr(), v.data_ptr(), *s) for (u, v), s in zip(dev, shapes)], 0.1, p)
    n = sum(a * b for a, b in shapes)
    assert boosted == (n if bias else 0) and fell <= boosted and (bias == 0 or rounds > 1) and (rounds == 1) == (fell == 0)
    out = [tuple(torch.zeros(s, device="cuda") for _ in range(2)) for s in shapes]
    torch.cuda.synchronize()
    cz.decompress_2d_batch_dev([(base + int(o), int(k)) for o, k in zip(off, size)], shapes,
                               [(u.data_ptr(), v.data_ptr()) for u, v in out])
    for (u, v), (x, y), s in zip(dev, out, shapes):
        for judge in (cz.critical_points_2d_dev, cz.critical_points_2d_sos_dev):
            for a, b in zip(judge(u.data_ptr(), v.data_ptr(), *s), judge(x.data_ptr(), y.data_ptr(), *s)):
                assert np.array_equal(a, b)
