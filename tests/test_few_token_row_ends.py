"""The few-token GEMM's weights come in 16-byte pieces of rows: matrices that end inside a piece or inside a step, with the end of
the buffer right behind them, rows that start on any boundary their format allows, fewer rows than a row tile."""
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


@pytest.mark.parametrize("fmt,lead", [("q4", 0), ("q4", 20), ("q8", 0), ("q8", 34), ("q3", 0), ("q3", 16)])
@pytest.mark.parametrize("m,n,k", [(17, 1, 32), (20, 3, 64), (33, 17, 96), (128, 47, 160), (50, 33, 1056), (24, 4097, 224), (64, 31, 2048),
                                   (20, 17, 32), (40, 33, 32), (18, 16, 96), (96, 300, 3104)])  # (a tile in front of the last that cannot load whole steps either)
def test_rows_end_with_the_buffer(be, fmt, lead, m, n, k):
    import torch
    print(f"few-token row ends {fmt} lead={lead} m={m} n={n} k={k}", flush=True)
    src = np.random.default_rng(n + k).normal(scale=0.05, size=(n, k)).astype(np.float32)
    if fmt == "q4":
        wq = synth.q4_weight(n, k, seed=n)
        deq, call = oracle.dequantize(wq, n * k), be._x.lq4_gemm
    elif fmt == "q8":
        wq = oracle.q8_quantize_rows(src)
        deq, call = oracle.q8_dequantize(wq, n * k), be._x.lq4_gemm_q8
    else:
        wq = oracle.q3_quantize_rows(src)
        deq, call = oracle.q3_dequantize(wq, n * k), be._x.lq4_gemm_q3
    wq = np.frombuffer(bytes(wq), np.uint8)
    qw = be.wrap_device_blocks(torch.from_numpy(np.concatenate([np.zeros(lead, np.uint8), wq])).cuda())
    x = synth.activations(m, k, seed=5, dtype=np.float16)
    dx, y = torch.from_numpy(x).cuda(), torch.full((m + 1, n), float("nan"), device="cuda")
    extra = (None, 0.0) if fmt == "q4" else ()
    call(be._c, qw.handle, lead, n, k, dx.data_ptr(), backend.LQ4_F16, m, y.data_ptr(), *extra, be._current_stream(be.device))
    got = y.cpu().numpy()
    assert np.all(np.isnan(got[m])) and rel_err(got[:m], x.astype(np.float32) @ deq.reshape(n, k).T) <= REL_TOL
