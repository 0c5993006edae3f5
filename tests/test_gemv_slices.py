"""2..8 activation rows against few, long weight rows: K slices that a second launch adds up (plain, with silu * up in front,
with the residual add behind); shapes whose last slice, last step and last row tile are partly filled."""
import numpy as np
import pytest

import oracle
from lattice_amd import backend, synth
from util import REL_TOL, rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    b = backend.HipQ4Backend(0)
    yield b
    b.close()


@pytest.mark.parametrize("n,k,batch", [(5, 9216, 3), (1000, 9248, 8), (129, 17408, 4), (63, 10240 + 32, 5)])
def test_plain_slices(be, n, k, batch):
    import torch
    print(f"slices n={n} k={k} batch={batch}", flush=True)
    wq = synth.q4_weight(n, k, seed=n)
    x = synth.activations(batch, k, seed=2)
    y = torch.full((batch + 1, n), float("nan"), dtype=torch.float32, device="cuda")
    be.gemv_batch(torch.from_numpy(x).cuda(), be.upload_q4_blocks(wq), y, batch, n, k)
    got = y.cpu().numpy()
    assert np.all(np.isnan(got[batch])) and rel_err(got[:batch], oracle.gemm_f32(x, wq, n, k)) <= REL_TOL


@pytest.mark.parametrize("n,k,batch", [(130, 5152, 8), (4096, 4128, 3), (72, 6144, 5)])
@pytest.mark.parametrize("silu,with_y", [(True, True), (True, False), (False, True)])
def test_fused_slices(be, n, k, batch, silu, with_y):
    import torch
    print(f"fused slices n={n} k={k} batch={batch} silu={silu}", flush=True)
    dev = lambda a: torch.from_numpy(a).cuda()
    wq = synth.q4_weight(n, k, seed=k)
    x = synth.activations(batch, 2 * k if silu else k, seed=3)
    r0 = synth.activations(batch, n, seed=4)
    res, out = dev(r0.copy()), torch.full((batch, n), float("nan"), device="cuda")
    y = torch.full((batch, n), float("nan"), device="cuda") if with_y else None
    be.dispatch_matmul_fused(dev(x), be.upload_q4_blocks(wq), y, n, k, silu_mul=silu, add_residual=(res, out), batch=batch)
    want = oracle.gemm_f32(oracle.silu_mul(x) if silu else x, wq, n, k)
    if with_y:
        assert rel_err(y.cpu().numpy(), want) <= REL_TOL
        assert np.array_equal(res.cpu().numpy(), r0 + y.cpu().numpy())
    assert rel_err(res.cpu().numpy(), r0 + want) <= REL_TOL
    assert np.array_equal(out.cpu().numpy(), res.cpu().numpy())
