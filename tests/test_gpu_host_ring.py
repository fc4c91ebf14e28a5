"""The host-pointer forward copies through a ring of pinned slots: at one column, at arrays
that straddle slots, and at more slots than the ring has, with and without padding columns,
its outputs and diagnostics are the device entry point's bit for bit and the caller's
padding columns stay as they were."""
import ctypes as C

import numpy as np
import pytest

from uwshcu_amd import _capi
from uwshcu_amd.generator import make_chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pcols,ncol,pver,ncnst", [(1, 1, 30, 0), (513, 513, 30, 5), (700, 513, 35, 3),
                                                  (4096, 4096, 35, 3), (4099, 4096, 35, 3)])
def test_host_forward_equals_device_forward(pcols, ncol, pver, ncnst):
    import torch
    from uwshcu_amd import device
    ch = make_chunk(ncol, pver, ncnst, seed=79)
    ctx = device.Context(0)
    inp = device.chunk_to_device(ch, "cuda:0")
    want = ctx.alloc_outputs(ncol, pver, ncnst, diag=True)
    cush = inp["cush"].clone()
    ctx.forward_into(inp, want, cush, dt=ch.dt)
    ctx.check()
    # without constituents there is no trten (the wrapper's tensor is a placeholder)
    want = {k: v.cpu().numpy() for k, v in want.items() if ncnst or k != "trten"}
    want["cush"] = cush.cpu().numpy()

    def padded(v, fill):
        w = np.full(v.shape[:-1] + (pcols,), fill, dtype=v.dtype)
        w[..., :ncol] = v
        return w

    arrays = {k: padded(np.ascontiguousarray(v), 1.0) for k, v in ch.fields.items()}
    got = {k: np.full(v.shape[:-1] + (pcols,), -7, dtype=v.dtype) for k, v in want.items() if k != "cush"}
    got["cush"] = padded(ch.fields["cush"], -7.0)
    arrays.update(got)
    arrays.setdefault("trten", np.zeros(1))
    bad = C.c_int(-1)
    print(f"[host] {pcols}/{ncol}x{pver}x{ncnst}", flush=True)
    for _ in range(2):                      # the second call finds the slots used
        got["cush"][:ncol] = ch.fields["cush"]
        rc = _capi.lib().uwshcu_forward_host(
            ctx._h, _capi.FP64, C.byref(_capi.default_params()), pcols, ncol, pver, ncnst, C.c_double(ch.dt),
            *[C.c_void_p(arrays[k].ctypes.data) for k in _capi.ARRAY_ARGS],
            C.c_void_p(got["diag"].ctypes.data), C.byref(bad))
        assert rc == 0, (rc, bad.value)
        for k, v in want.items():
            np.testing.assert_array_equal(got[k][..., :ncol], v, err_msg=k)
            assert (got[k][..., ncol:] == -7).all(), k
    ctx.close()
