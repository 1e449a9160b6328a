"""The batch's state copies between the callers' buffers and its pools: exact
for any cell count and any 4-byte alignment of the callers' buffers."""
import ctypes

import pytest
import torch

from cardiax_amd import _lib, solve
from cardiax_amd.params import PARAMSET_3

pytestmark = pytest.mark.gpu

SHAPES = [(3, 3), (5, 7), (64, 64), (33, 31), (128, 130)]


@pytest.mark.parametrize("shift", [0, 1, 2, 3])
@pytest.mark.parametrize("steps", [0, 1, 3])
def test_batch_state_round_trip(gpu, shift, steps):
    """Buffers `shift` floats off a 256-byte boundary; 0 steps return the
    state as it was, more equal each simulation's own solve."""
    L = _lib.lib()
    g = torch.Generator().manual_seed(shift)
    arr = (_lib.FkSim * len(SHAPES))()
    keep, refs = [], []
    for d, (H, W) in zip(arr, SHAPES):
        n = H * W
        fields = []
        for _ in range(3):
            buf = torch.full((n + 8,), 7.0, device=gpu)
            buf[shift:shift + n] = torch.rand(n, generator=g).to(gpu)
            fields.append(buf)
        D = torch.full((H, W), 1e-3, device=gpu)
        st = [x[shift:shift + n].reshape(H, W).clone() for x in fields]
        refs.append(solve._forward_euler(st, 0, steps, PARAMSET_3, D, [], 0.01, 0.01))
        d.params = _lib.make_params(PARAMSET_3)
        d.D = D.data_ptr()
        d.v, d.w, d.u = (x.data_ptr() + 4 * shift for x in fields)
        d.H, d.W, d.n_stimuli, d.t, d.dt, d.dx = H, W, 0, 0.0, 0.01, 0.01
        keep.append((fields, D))
    h = ctypes.c_void_p()
    s = torch.cuda.current_stream().cuda_stream
    torch.cuda.synchronize()
    _lib.check(L.fk_batch_create(arr, len(SHAPES), ctypes.byref(h)))
    try:
        _lib.check(L.fk_batch_run(h, steps, 1, s))
        torch.cuda.synchronize()
        for (H, W), (fields, _), ref in zip(SHAPES, keep, refs):
            for buf, r in zip(fields, ref):
                assert torch.equal(buf[shift:shift + H * W].reshape(H, W), r)
                assert (buf[:shift] == 7.0).all() and (buf[shift + H * W:] == 7.0).all()
    finally:
        _lib.check(L.fk_batch_destroy(h))
