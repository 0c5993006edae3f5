"""The few-token GEMM above 128 tokens: the edges of its token groups, row tiles and K steps, the three formats, both sides of its
lines, and a capture whose scratch just holds the packed activations."""
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


def weights(be, fmt, n, k):
    src = np.random.default_rng(n + k).normal(scale=0.05, size=(n, k)).astype(np.float32)
    if fmt == "q4":
        wq = synth.q4_weight(n, k, seed=n)
        return be.upload_q4_blocks(wq), oracle.dequantize(wq, n * k).reshape(n, k), be.dispatch_gemm
    if fmt == "q8":
        wq = oracle.q8_quantize_rows(src)
        return be.upload_q8_blocks(wq), oracle.q8_dequantize(wq, n * k).reshape(n, k), be.dispatch_gemm_q8
    wq = oracle.q3_quantize_rows(src)
    return be.upload_q3_blocks(wq), oracle.q3_dequantize(wq, n * k).reshape(n, k), be.dispatch_gemm_q3


# tokens, rows, K, served by the few-token kernel
@pytest.mark.parametrize("fmt", ["q4", "q8", "q3"])
@pytest.mark.parametrize("xdt", [np.float16, np.float32])
@pytest.mark.parametrize("m,n,k,few", [(129, 17, 256, False), (129, 17, 1056, True), (129, 513, 1056, True), (176, 1023, 1184, True), (256, 130, 2080, True), (257, 47, 288, False), (257, 47, 800, True),
                                       (500, 512, 1056, True), (512, 33, 4064, True), (769, 250, 544, False), (769, 250, 1056, True), (912, 272, 1056, True), (1024, 256, 1056, True),
                                       (1025, 64, 512, False), (192, 100, 224, False), (256, 6160, 1056, False), (1024, 520, 2080, False)])
def test_edges_and_lines(be, fmt, m, n, k, few, xdt):
    import torch
    print(f"few-token wide {fmt} m={m} n={n} k={k} x={np.dtype(xdt).name}", flush=True)
    qw, deq, call = weights(be, fmt, n, k)
    x = synth.activations(m, k, seed=3, dtype=xdt)
    dx, got = torch.from_numpy(x).cuda(), {}
    try:
        for which in (0, 2):  # by the rule, the weights-in-registers kernel
            y = torch.full((m + 1, n), float("nan"), device="cuda")
            be.set_gemm_kernel(which)
            call(dx, 0, qw, y, 0, m, n, k)
            got[which] = y.cpu().numpy()
    finally:
        be.set_gemm_kernel(0)
    want = x.astype(np.float32) @ deq.T
    for v in got.values():
        assert np.all(np.isnan(v[m])) and rel_err(v[:m], want) <= REL_TOL
    if fmt == "q4":  # (forced above 128 tokens too; for the siblings up to there only)
        y = torch.full((m, n), float("nan"), device="cuda")
        be.set_gemm_kernel(3)
        try:
            call(dx, 0, qw, y, 0, m, n, k)
        finally:
            be.set_gemm_kernel(0)
        assert np.array_equal(got[0][:m], y.cpu().numpy()) == few


@pytest.mark.parametrize("m,n,k,few", [(128, 4096, 8192, True), (65, 2080, 8192, True), (128, 4096, 8224, False), (128, 2049, 14336, False)])
def test_lines_up_to_128(be, m, n, k, few):
    import torch
    print(f"few-token lines m={m} n={n} k={k}", flush=True)
    qw, deq, call = weights(be, "q4", n, k)
    x = synth.activations(m, k, seed=3, dtype=np.float16)
    dx, got = torch.from_numpy(x).cuda(), {}
    try:
        for which in (0, 3):
            y = torch.full((m, n), float("nan"), device="cuda")
            be.set_gemm_kernel(which)
            call(dx, 0, qw, y, 0, m, n, k)
            got[which] = y.cpu().numpy()
    finally:
        be.set_gemm_kernel(0)
    assert rel_err(got[0], x.astype(np.float32) @ deq.T) <= REL_TOL
    assert np.array_equal(got[0], got[3]) == few


@pytest.mark.parametrize("m,n,k", [(100, 2048, 2048), (512, 512, 1024)])
def test_capture_with_scratch_for_the_packed_activations(m, n, k):
    """Reserved scratch comes in whole MiB; the packed activations of the second shape fill one.  (Less of it, and none:
    test_few_token_context.py.)"""
    import torch
    print(f"few-token capture m={m} n={n} k={k}", flush=True)
    be = backend.HipQ4Backend(0)
    wq = synth.q4_weight(n, k, seed=2)
    x = synth.activations(m, k, seed=2, dtype=np.float16)
    qw, dx, y = be.upload_q4_blocks(wq), torch.from_numpy(x).cuda(), torch.empty((m, n), device="cuda")
    want = x.astype(np.float32) @ oracle.dequantize(wq, n * k).reshape(n, k).T
    be.reserve_scratch(1 << 16)
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            be.dispatch_gemm(dx, 0, qw, y, 0, m, n, k)
    got = []
    for _ in range(2):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got.append(y.cpu().numpy())
        assert rel_err(got[-1], want) <= REL_TOL
    be.set_gemm_kernel(3)
    be.dispatch_gemm(dx, 0, qw, y, 0, m, n, k)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], y.cpu().numpy())
    del qw
    be.close()
