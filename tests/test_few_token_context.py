"""What the few-token GEMM takes of the context: products that the large tiles run whole, without any scratch, stay theirs above 128
tokens and beside the lines of 33..128, so that the call is the same on a new context, under capture and after scratch has grown."""
import numpy as np
import pytest

import oracle
from lattice_amd import backend, synth
from util import REL_TOL, rel_err

pytestmark = pytest.mark.gpu


def blocks(fmt, n, k):
    src = np.random.default_rng(n + k).normal(scale=0.05, size=(n, k)).astype(np.float32)
    if fmt == "q4":
        wq = synth.q4_weight(n, k, seed=n)
        return wq, oracle.dequantize(wq, n * k).reshape(n, k)
    if fmt == "q8":
        wq = oracle.q8_quantize_rows(src)
        return wq, oracle.q8_dequantize(wq, n * k).reshape(n, k)
    wq = oracle.q3_quantize_rows(src)
    return wq, oracle.q3_dequantize(wq, n * k).reshape(n, k)


def caller(be, fmt, wq):
    upload = {"q4": be.upload_q4_blocks, "q8": be.upload_q8_blocks, "q3": be.upload_q3_blocks}[fmt]
    call = {"q4": be.dispatch_gemm, "q8": be.dispatch_gemm_q8, "q3": be.dispatch_gemm_q3}[fmt]
    qw = upload(wq)
    return lambda dx, y, m, n, k: call(dx, 0, qw, y, 0, m, n, k)


def captured(call, y):
    """`call` captured; its output after two replays with the stream's own work between them."""
    import torch
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        with torch.cuda.graph(graph, stream=stream):
            call()
    got = []
    for _ in range(2):
        y.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got.append(y.cpu().numpy())
    assert np.array_equal(*got)
    return got[0]


# (the second half: shapes beside them that do go to the few-token kernel, as K slices of theirs would need more scratch)
@pytest.mark.parametrize("fmt,m,n,k,xdt,whole", [
    ("q4", 129, 64, 256, np.float16, True), ("q4", 160, 2048, 384, np.float32, True), ("q4", 256, 6160, 1024, np.float32, True),
    ("q4", 40, 20196, 1152, np.float16, True), ("q4", 104, 16003, 1088, np.float32, True),
    ("q8", 104, 8106, 64, np.float16, True), ("q8", 54, 15475, 736, np.float16, True), ("q8", 315, 834, 352, np.float32, True),
    ("q3", 96, 6760, 480, np.float16, True), ("q3", 299, 152, 352, np.float32, True),
    ("q4", 129, 64, 1056, np.float16, False), ("q8", 104, 2000, 1024, np.float16, False), ("q3", 299, 152, 1056, np.float32, False)])
def test_products_without_scratch_stay_without(fmt, m, n, k, xdt, whole):
    import torch
    print(f"without scratch {fmt} m={m} n={n} k={k} x={np.dtype(xdt).name}", flush=True)
    be = backend.HipQ4Backend(0)
    wq, deq = blocks(fmt, n, k)
    call = caller(be, fmt, wq)
    x = synth.activations(m, k, seed=3, dtype=xdt)
    dx, y = torch.from_numpy(x).cuda(), torch.empty((m, n), device="cuda")
    want = x.astype(np.float32) @ deq.T
    if whole:
        first = captured(lambda: call(dx, y, m, n, k), y)
        assert rel_err(first, want) <= REL_TOL
    be.reserve_scratch(64 << 20)
    call(dx, y, m, n, k)
    got = y.cpu().numpy()
    assert rel_err(got, want) <= REL_TOL
    if whole:
        assert np.array_equal(first, got)  # the same kernel, with scratch at hand or not
    elif m > 128 or fmt == "q4":
        be.set_gemm_kernel(2)
        call(dx, y, m, n, k)
        assert not np.array_equal(got, y.cpu().numpy())
    del call
    be.close()
