"""Launch batching under a workspace limit: a chunk that the limit holds runs in one launch
whatever its size, one that it does not hold runs in several; every way of cutting it gives
the portable-math oracle's bits."""
import numpy as np
import pytest

import oracle
from uwshcu_amd import _capi
from uwshcu_amd.generator import make_chunk

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ncol,limit_cols", [(1, 64), (63, 64), (65, 65), (200, 200), (200, 256), (200, 199), (321, 128),
                                             (129, 1)])
def test_batches_give_the_oracle_bits(ncol, limit_cols):
    import torch
    from uwshcu_amd import device
    ch = make_chunk(ncol, 30, 5, seed=17)
    per_col = _capi.workspace_bytes_per_column(30, 5)
    ctx = device.Context(0, workspace_limit=per_col * limit_cols)
    out = ctx.compute_uwshcu_inv(device.chunk_to_device(ch, "cuda:0"), dt=ch.dt, diag=True)
    torch.cuda.synchronize()
    ref, diag, rc, _ = oracle.run(ch, nthreads=8, portable=True)
    assert rc == 0
    np.testing.assert_array_equal(out["diag"].cpu().numpy().T, diag)
    for k, v in ref.items():
        np.testing.assert_array_equal(out[k].cpu().numpy(), v, err_msg=k)
    ctx.close()


@pytest.mark.parametrize("limit_cols", [64, 192, 256, 320])
def test_mixed_batches_equal_one_launch(limit_cols):
    """The mixed mode's recompute runs over a list that ends inside a batch, after batches of
    other sizes left their lists and marks in the same storage."""
    import torch
    from uwshcu_amd import device
    ch = make_chunk(700, 30, 5, seed=18, inversion_frac=0.1)
    inp = device.chunk_to_device(ch, "cuda:0")
    res = []
    for limit in (None, _capi.workspace_bytes_per_column(30, 5) * limit_cols):
        ctx = device.Context(0, workspace_limit=limit)
        ctx.set_mixed_tolerance(1e-13)       # many columns fail the check and are recomputed
        out = ctx.compute_uwshcu_inv(inp, dt=ch.dt, precision=_capi.MIXED, diag=True)
        torch.cuda.synchronize()
        res.append((ctx.mixed_recomputed(), {k: v.cpu().numpy() for k, v in out.items()}))
        ctx.close()
    assert res[0][0] == res[1][0] > 0
    for k, v in res[0][1].items():
        np.testing.assert_array_equal(res[1][1][k], v, err_msg=k)
