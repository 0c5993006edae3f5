"""The tile shapes of the weights-in-registers GEMM: one shape (M, N) per tile at which the schedule takes it, its last
token and row tiles partly filled, K with and without a partly filled last step, all formats and activation types."""
import numpy as np
import pytest

import oracle
from lattice_amd import backend, synth
from util import REL_TOL, rel_err

pytestmark = pytest.mark.gpu

# 128 x 128, 96 x 192, 112 x 192, 128 x 192, 96 x 256 and 128 x 256 tokens x rows
SHAPES = [(201, 515), (777, 5119), (1790, 3070), (2039, 3060), (1530, 4090), (2040, 4095)]


@pytest.fixture(scope="module")
def be():
    b = backend.HipQ4Backend(0)
    yield b
    b.close()


@pytest.mark.parametrize("m,n", SHAPES)
@pytest.mark.parametrize("fmt,k,xdt", [("q4", 160, "f16"), ("q4", 96, "f32"), ("q8", 160, "f32"), ("q8", 192, "f16"), ("q8", 512, "f16"),
                                       ("q3", 416, "f16"), ("q3", 128, "f32")])
def test_tiles_match_the_dequantised_product(be, m, n, fmt, k, xdt):
    import torch
    print(f"gemm tiles {fmt} m={m} n={n} k={k} x={xdt}", flush=True)
    if fmt == "q4":
        wq = synth.q4_weight(n, k, seed=m)
        deq, qw, call = oracle.dequantize(wq, n * k), be.upload_q4_blocks(wq), be.dispatch_gemm
    else:
        src = np.random.default_rng(m + k).normal(scale=0.05, size=(n, k)).astype(np.float32)
        if fmt == "q8":
            wq = oracle.q8_quantize_rows(src)
            deq, qw, call = oracle.q8_dequantize(wq, n * k), be.upload_q8_blocks(wq), be.dispatch_gemm_q8
        else:
            wq = oracle.q3_quantize_rows(src)
            deq, qw, call = oracle.q3_dequantize(wq, n * k), be.upload_q3_blocks(wq), be.dispatch_gemm_q3
    x = synth.activations(m, k, seed=3, dtype=np.float16 if xdt == "f16" else np.float32)
    y = torch.full((m + 1, n), float("nan"), dtype=torch.float32, device="cuda")
    be.set_gemm_kernel(2)
    try:
        call(torch.from_numpy(x).cuda(), 0, qw, y, 0, m, n, k)
    finally:
        be.set_gemm_kernel(0)
    got = y.cpu().numpy()
    assert np.all(np.isnan(got[m])) and np.all(np.isfinite(got[:m]))
    assert rel_err(got[:m], x.astype(np.float32) @ deq.reshape(n, k).T) <= REL_TOL
