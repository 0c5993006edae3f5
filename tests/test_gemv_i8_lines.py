"""Which kernel serves 2..8 rows: both sides of the lines between the integer matrix-core GEMV and the others, plain, fused and several
views at once, against the oracle and against a context that is told which to take."""
import os

import numpy as np
import pytest

import oracle
from lattice_amd import backend, synth
from util import REL_TOL, rel_err

pytestmark = pytest.mark.gpu


def context(which):
    old = os.environ.get("LQ4_GEMV_I8")
    os.environ["LQ4_GEMV_I8"] = which
    try:
        return backend.HipQ4Backend(0)
    finally:
        if old is None:
            del os.environ["LQ4_GEMV_I8"]
        else:
            os.environ["LQ4_GEMV_I8"] = old


@pytest.fixture(scope="module")
def contexts():
    c = {w: context(w) for w in ("0", "1", "2")}  # never, by the rule, wherever it can be held
    yield c
    for b in c.values():
        b.close()


@pytest.mark.parametrize("n,k,batch,served", [
    (2048, 2048, 2, False), (2560, 2048, 2, True), (4096, 2016, 2, False), (4097, 2048, 2, False), (7168, 2048, 2, True), (10256, 2304, 2, False),
    (4096, 2048, 3, True), (511, 2080, 3, False), (1024, 2816, 3, True), (1023, 2816, 3, False), (2560, 5120, 4, True), (2560, 5152, 4, False),
    (5120, 992, 4, False), (5120, 1024, 4, True), (12304, 4128, 4, False), (1536, 2848, 6, False), (1536, 2848, 7, True), (5120, 2560, 5, False),
    (6144, 2560, 5, True), (8192, 3072, 5, True), (65552, 1024, 8, True),
    (10240, 2304, 2, True), (12288, 2048, 2, True), (12304, 2048, 2, True), (12288, 2080, 2, False), (12288, 2560, 2, False), (12288, 2816, 2, True), (14336, 2304, 2, True),
    (20480, 2560, 2, False), (16384, 2784, 2, True)])
def test_lines(contexts, n, k, batch, served):
    import torch
    print(f"i8 lines n={n} k={k} batch={batch}", flush=True)
    wq = synth.q4_weight(n, k, seed=n)
    x = synth.activations(batch, k, seed=k)
    dx, got = torch.from_numpy(x).cuda(), {}
    for w, be in contexts.items():
        y = torch.full((batch, n), float("nan"), device="cuda")
        be.gemv_batch(dx, be.upload_q4_blocks(wq), y, batch, n, k)
        got[w] = y.cpu().numpy()
    want = oracle.gemm_f32(x, wq, n, k)
    assert rel_err(got["1"], want) <= REL_TOL
    assert np.array_equal(got["1"], got["2" if served else "0"]) and not np.array_equal(got["0"], got["2"])
    # more rows than f16 keeps, never fewer: the new route is at least as close as the old one
    assert not served or rel_err(got["2"], want) <= max(rel_err(got["0"], want), 5e-6)


@pytest.mark.parametrize("rank", [0, 16])
@pytest.mark.parametrize("k,shapes,batch", [(4096, (4096, 1024, 1024), 3), (2560, (2560, 512, 512), 8), (3072, (3072, 48, 16), 5), (5120, (5120, 128, 128), 2)])
def test_views_at_once(contexts, k, shapes, batch, rank):
    import torch
    print(f"i8 views k={k} shapes={shapes} batch={batch} rank={rank}", flush=True)
    x = synth.activations(batch, k, seed=3)
    dx = torch.from_numpy(x).cuda()
    ws = [synth.q4_weight(n, k, seed=n + i) for i, n in enumerate(shapes)]
    names = [f"p{i}" for i in range(len(shapes))]
    pairs = {m: synth.lora_pair(rank, k, n, seed=n, tag=m) for m, n in zip(names, shapes)} if rank else {}
    be = contexts["1"]
    kw = {}
    if rank:
        be.load_lora_adapter([backend.LoraLayerData(0, pairs)], scale=2.0)
        kw = dict(layer_idx=0)
    try:
        ys = [torch.full((batch, n), float("nan"), device="cuda") for n in shapes]
        be.gemv_multi(dx, [(be.upload_q4_blocks(w), n, y, m) for w, n, y, m in zip(ws, shapes, ys, names)], batch, k, **kw)
    finally:
        be.unload_lora_adapter()
    for w, n, y, m in zip(ws, shapes, ys, names):
        want = oracle.gemm_f32(x, w, n, k)
        if rank:
            a, b = pairs[m]
            want = oracle.lora_apply(a.astype(np.float32), b.astype(np.float32), 2.0, x, want)
        assert rel_err(y.cpu().numpy(), want) <= REL_TOL, m
