"""The integer matrix-core GEMV where its weights, rows and chunks end: matrices that end with their buffer inside a unit of 16
rows x 256 weights, rows that start on any boundary, more units than a wave keeps in flight, several tiles a workgroup."""
import os

import numpy as np
import pytest

import oracle
from lattice_amd import backend, synth
from util import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def i8():
    old = os.environ.get("LQ4_GEMV_I8")
    os.environ["LQ4_GEMV_I8"] = "2"  # every shape that it can hold
    try:
        b = backend.HipQ4Backend(0)
    finally:
        if old is None:
            del os.environ["LQ4_GEMV_I8"]
        else:
            os.environ["LQ4_GEMV_I8"] = old
    yield b
    b.close()


@pytest.mark.parametrize("lead", [0, 20])
@pytest.mark.parametrize("n,k", [(1, 32), (3, 160), (16, 224), (17, 256), (31, 288), (40, 1056), (33, 2048), (19, 2304), (24, 4128),
                                 (4097, 1024), (8200, 1184), (12289, 2080), (300, 6944),
                                 (32763, 1184), (28700, 2080), (65530, 224)])  # one column of chunks beside eight tiles
@pytest.mark.parametrize("batch", [2, 4, 5, 8])
def test_rows_end_with_the_buffer(i8, lead, n, k, batch):
    import torch
    print(f"i8 row ends n={n} k={k} batch={batch} lead={lead}", flush=True)
    wq = synth.q4_weight(n, k, seed=n)
    qw = i8.wrap_device_blocks(torch.from_numpy(np.concatenate([np.zeros(lead, np.uint8), np.frombuffer(bytes(wq), np.uint8)])).cuda())
    x = synth.activations(batch, k, seed=k)
    y = torch.full((batch + 1, n), float("nan"), device="cuda")
    i8.gemv_batch(torch.from_numpy(x).cuda(), qw, y, batch, n, k, qw_extra_offset=lead)
    got = y.cpu().numpy()
    # (the bars of the kernel's other tests: f32 sums over activations of 24 and of 16 bits below their block's maximum)
    assert np.all(np.isnan(got[batch])) and rel_err(got[:batch], oracle.gemm_f32(x, wq, n, k)) <= (5e-6 if batch <= 4 else 1e-4)


@pytest.mark.parametrize("n,k,rank,dt", [(40, 1056, 16, np.float16), (40, 1056, 5, np.float32), (2000, 2336, 32, np.float16), (70, 4128, 64, np.float32)])
@pytest.mark.parametrize("batch", [3, 8])
def test_factors_computed_by_the_launch(i8, n, k, rank, dt, batch):
    """Producers of A . x: rows of A that are no whole number of their steps, both adapter types, ranks with and without eights."""
    import torch
    print(f"i8 factors n={n} k={k} rank={rank} batch={batch}", flush=True)
    wq = synth.q4_weight(n, k, seed=n)
    a, b = synth.lora_pair(rank, k, n, seed=rank, dtype=dt)
    x = synth.activations(batch, k, seed=4)
    qw, dx = i8.upload_q4_blocks(wq), torch.from_numpy(x).cuda()
    y = torch.full((batch, n), float("nan"), device="cuda")
    i8.load_lora_adapter([backend.LoraLayerData(0, {"v_proj": (a, b)})], scale=2.0)
    try:
        before = i8.path_counters()
        i8.gemv_batch(dx, qw, y, batch, n, k, layer_idx=0, module="v_proj")
        assert i8.path_counters()["lora_a"] == before["lora_a"]
    finally:
        i8.unload_lora_adapter()
    want = oracle.lora_apply(a.astype(np.float32), b.astype(np.float32), 2.0, x, oracle.gemm_f32(x, wq, n, k))
    assert rel_err(y.cpu().numpy(), want) <= (5e-6 if batch <= 4 else 1e-4)
