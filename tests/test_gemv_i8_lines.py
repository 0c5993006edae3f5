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


@pytest.mark.parametrize("n,k,batch,served", [(4096, 4096, 3, True), (12304, 4128, 4, False), (6144, 2560, 5, True), (5120, 2560, 5, False),
                                              (1536, 2848, 7, True), (1536, 2848, 6, False)])
def test_lines_behind_a_norm(contexts, n, k, batch, served):
    """What lq4_gemv_fused_batch leaves of a call once the norm is a launch of its own (more than 64 KB of rows and deltas) is a plain
    product, by the same lines."""
    import torch
    print(f"i8 lines fused n={n} k={k} batch={batch}", flush=True)
    wq = synth.q4_weight(n, k, seed=n)
    x, delta, gamma = synth.activations(batch, k, seed=k), synth.activations(batch, k, seed=k + 2), synth.activations(1, k, seed=k + 1)[0] * 0.1
    (dx, dd, dg), got = (torch.from_numpy(t).cuda() for t in (x, delta, gamma)), {}
    for w, be in contexts.items():
        y = torch.full((batch, n), float("nan"), device="cuda")
        be.dispatch_matmul_fused(None, be.upload_q4_blocks(wq), y, n, k, norm=(dx, dd, dg, 1e-6, torch.empty_like(dx)), batch=batch)
        got[w] = y.cpu().numpy()
    x = x.astype(np.float64) + delta
    normed = (x / np.sqrt(np.mean(x ** 2, axis=1, keepdims=True) + 1e-6) * (1 + gamma.astype(np.float64))).astype(np.float32)
    assert rel_err(got["1"], oracle.gemm_f32(normed, wq, n, k)) <= REL_TOL
    assert np.array_equal(got["1"], got["2" if served else "0"]) and not np.array_equal(got["0"], got["2"])


@pytest.mark.parametrize("rank", [0, 16])
@pytest.mark.parametrize("k,shapes,batch,at_once", [
    (4096, (4096, 1024, 1024), 3, True), (2560, (2560, 512, 512), 8, False), (3072, (3072, 48, 16), 5, True), (5120, (5120, 128, 128), 2, False),
    (2048, (2048, 512, 512), 2, True),     # up to 4096 rows of K up to 2048 from two rows on, unlike one matrix
    (4096, (2048, 512, 512), 2, True), (2048, (3072, 512, 528), 2, False),  # two rows: 2560..4096 rows together
    (2560, (4096, 1024, 1024), 5, True),  # five and more: by how busy the waves are
    (5152, (2560, 512, 512), 4, False), (2560, (4096, 1024, 1032), 8, False)])  # K; a view that is no whole number of tiles
def test_views_at_once(contexts, k, shapes, batch, at_once, rank):
    """By the sum of the views' rows, with and without adapters; elsewhere each view by its own."""
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
        before = be.path_counters()["gemv_multi"]
        ys = [torch.full((batch, n), float("nan"), device="cuda") for n in shapes]
        be.gemv_multi(dx, [(be.upload_q4_blocks(w), n, y, m) for w, n, y, m in zip(ws, shapes, ys, names)], batch, k, **kw)
        assert be.path_counters()["gemv_multi"] - before == int(at_once)
    finally:
        be.unload_lora_adapter()
    for w, n, y, m in zip(ws, shapes, ys, names):
        want = oracle.gemm_f32(x, w, n, k)
        if rank:
            a, b = pairs[m]
            want = oracle.lora_apply(a.astype(np.float32), b.astype(np.float32), 2.0, x, want)
        assert rel_err(y.cpu().numpy(), want) <= REL_TOL, m
