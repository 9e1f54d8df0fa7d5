"""The 3D bounds in strips of different lengths: a field alone (short strips, all
resident at once) against the oracle, and against copies of it in batches that
call for longer ones, last strips of a single plane included."""
import ctypes as C

import numpy as np
import pytest
import torch

import cpsz_amd as cz
from _libs import load_oracle
from cpsz_amd.synth import field_3d

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,count", [((33, 47, 66), 48), ((17, 16, 64), 200), ((2, 31, 127), 3)], ids=str)
def test_strip_lengths(shape, count):
    print(f"[strips3d] {shape} x {count}", flush=True)
    U, V, W = (np.ascontiguousarray(a, np.float32) for a in field_3d(*shape, 11))
    want = load_oracle().compress_3d(U, V, W, 0.05)
    assert np.array_equal(cz.sz_compress_cp_preserve_3d_offline_log(U, V, W, 0.05), want)
    d = [torch.from_numpy(a).cuda() for a in (U, V, W)]
    torch.cuda.synchronize()
    base, off, size = cz.compress_3d_batch_dev([(*(x.data_ptr() for x in d), *shape)] * count, 0.05)
    for k in (0, count // 2, count - 1):
        got = np.empty(int(size[k]), np.uint8)
        C.CDLL("libamdhip64.so").hipMemcpy(C.c_void_p(got.ctypes.data), C.c_void_p(base + int(off[k])),
                                           C.c_size_t(got.size), 2)
        assert np.array_equal(got, want)
