"""The allocation-free forward at the largest chunks that its scratch admits, and one
wavefront of columns: the lists, saved scalars and records of its split launch must fit
their own scratch there, and every output and diagnostic must equal the allocating entry
point's bit for bit."""
import numpy as np
import pytest

from uwshcu_amd import _capi
from uwshcu_amd.generator import make_chunk

from test_zz_no_alloc import _host, _run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pver,ncnst,full", [(35, 3, True), (72, 10, True), (3, 0, True), (30, 0, False)])
def test_noalloc_equals_forward_device_at_the_scratch_limit(pver, ncnst, full):
    import torch
    from uwshcu_amd import device
    ncol = _capi.NOALLOC_SCRATCH_BYTES // _capi.workspace_bytes_per_column(pver, ncnst) // 64 * 64 if full else 1
    ch = make_chunk(ncol, pver, ncnst, seed=75, ptop=100.0 if pver > 60 else 200.0)
    ctx = device.Context(0)
    got = []
    for noalloc in (False, True):
        fn, args, out, cush, _inputs = _run(ctx, ch, noalloc)
        print(f"[noalloc] {ncol}x{pver}x{ncnst} noalloc={noalloc}", flush=True)
        assert fn(*args) == 0
        torch.cuda.synchronize()
        got.append(_host(out, cush))
    assert ctx.status()[0] == 0
    for k, v in got[0].items():
        np.testing.assert_array_equal(got[1][k], v, err_msg=k)
    ctx.close()
