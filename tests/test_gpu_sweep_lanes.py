"""The adjoint's backward sweep at every number of columns per wavefront (8, 16, 32, 64,
chosen by the launch's size) and at incomplete wavefronts: a column's gradients are the
host sweep's, bit for bit, whichever columns share its wavefront."""
import numpy as np
import pytest

import hostemu
from uwshcu_amd.generator import make_chunk

pytestmark = pytest.mark.gpu

GRADS = ("t0", "qv0", "u0", "v0", "tke")
DISTINCT = 61


@pytest.mark.parametrize("ncol", [1, 61, 8193, 16385, 32769])
def test_sweep_gradients_do_not_depend_on_the_launch(ncol):
    import torch
    from uwshcu_amd import device
    ch = make_chunk(DISTINCT, 20, 4, seed=23, inversion_frac=0.1)
    rng = np.random.default_rng(3)
    cot = {k: rng.normal(0.0, 1.0, (20, DISTINCT)) for k in ("sten", "qvten", "cufrc")}
    cot["trten"] = rng.normal(0.0, 1.0, (4, 20, DISTINCT))
    cot["precip"] = rng.normal(0.0, 1.0, DISTINCT)
    _, want, _, _ = hostemu.adjoint(ch, cot)
    at = torch.arange(ncol, device="cuda:0") % DISTINCT

    def tiled(v):
        return torch.from_numpy(np.ascontiguousarray(v)).to("cuda:0")[..., at].contiguous()

    ctx = device.Context(0, workspace_limit=64 << 30)
    inp = {k: tiled(v) for k, v in ch.fields.items()}
    out = ctx.alloc_outputs(ncol, 20, 4)
    grads = {k: torch.zeros_like(inp[k]) for k in GRADS}
    grads["par_col"] = torch.zeros((3, ncol), dtype=torch.float64, device="cuda:0")
    ctx.adjoint_into(inp, out, inp["cush"].clone(), {k: tiled(v) for k, v in cot.items()}, grads, dt=ch.dt)
    ctx.check()
    want["par_col"] = want["par"]
    for k in GRADS + ("par_col",):
        np.testing.assert_array_equal(grads[k].cpu().numpy(), want[k][..., at.cpu().numpy()], err_msg=k)
    ctx.close()
