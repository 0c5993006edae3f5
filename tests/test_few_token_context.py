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


def many(be, wqs, n, k, m):
    qws = [be.upload_q4_blocks(wq) for wq in wqs]
    return lambda dx, ys: be.gemv_multi(dx, [(q, n, y, None) for q, y in zip(qws, ys)], m, k)


# shapes of the few-token kernel whose large tiles are whole (nothing reserved), or whose K slices fit where the packed
# activations do not
@pytest.mark.parametrize("fmt,m,n,k,reserve", [("q4", 17, 2048, 352, 0), ("q4", 100, 512, 352, 0), ("q4", 160, 128, 8192, 2 << 20), ("q8", 40, 1024, 352, 0),
                                               ("q3", 120, 512, 256, 0), ("multi", 40, 512, 352, 0), ("multi", 128, 128, 8192, 1 << 20)])
def test_capture_takes_the_large_tiles_where_only_their_scratch_fits(fmt, m, n, k, reserve):
    import torch
    print(f"few-token capture {fmt} m={m} n={n} k={k}", flush=True)
    be = backend.HipQ4Backend(0)
    wq, deq = blocks("q4" if fmt == "multi" else fmt, n, k)
    x = synth.activations(m, k, seed=2)
    dx = torch.from_numpy(x).cuda()
    y, other = (torch.empty((m, n), device="cuda") for _ in range(2))
    if fmt == "multi":
        both = many(be, [wq, wq], n, k, m)
        go = lambda: both(dx, (y, other))  # noqa: E731
    else:
        call = caller(be, fmt, wq)
        go = lambda: call(dx, y, m, n, k)  # noqa: E731
    if reserve:
        be.reserve_scratch(reserve)
    if fmt in ("q8", "q3"):
        # (up to 32 rows always, above by the lines: there a forced kernel does not hold, the large tiles are what a capture takes)
        got = captured(go, y)
        assert rel_err(got, x @ deq.T) <= REL_TOL
        go()
        assert not np.array_equal(got, y.cpu().numpy())
    else:
        got = captured(go, y)
        assert rel_err(got, x @ deq.T) <= REL_TOL
        be.set_gemm_kernel(2)
        go()
        assert np.array_equal(got, y.cpu().numpy())
        be.set_gemm_kernel(0)
        go()
        assert not np.array_equal(got, y.cpu().numpy())
    go = call = both = None
    be.close()


@pytest.mark.parametrize("fmt,m,n,k,rank,need", [("q4", 100, 2048, 2048, 0, 7 * 16 * 4096), ("q4", 100, 2048, 2048, 32, 7 * 16 * 4096), ("q8", 100, 1024, 2048, 0, 7 * 16 * 4096),
                                                 ("multi", 64, 1024, 2048, 0, 4 * 16 * 4096)])
def test_capture_that_fits_neither_names_the_packed_activations(fmt, m, n, k, rank, need):
    """K slices of the large tiles would take several times the bytes of the packed activations (need: token groups x K steps x 4 KB)."""
    import torch
    print(f"few-token refused {fmt} m={m} n={n} k={k} rank={rank}", flush=True)
    be = backend.HipQ4Backend(0)
    wq, _ = blocks("q4" if fmt == "multi" else fmt, n, k)
    dx = torch.from_numpy(synth.activations(m, k, seed=2)).cuda()
    y, other = (torch.empty((m, n), device="cuda") for _ in range(2))
    kw = {}
    if rank:
        be.load_lora_adapter([backend.LoraLayerData(0, {"q_proj": synth.lora_pair(rank, k, n, seed=3)})], scale=2.0)
        kw = dict(layer_idx=0, module="q_proj")
    if fmt == "multi":
        both = many(be, [wq, wq], n, k, m)
        go = lambda: both(dx, (y, other))  # noqa: E731
    elif rank:
        qw = be.upload_q4_blocks(wq)
        go = lambda: be.dispatch_gemm(dx, 0, qw, y, 0, m, n, k, **kw)  # noqa: E731
    else:
        call = caller(be, fmt, wq)
        go = lambda: call(dx, y, m, n, k)  # noqa: E731
    stream, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    with pytest.raises(backend.Q4Error, match=f"to {need} bytes"):
        with torch.cuda.stream(stream):
            with torch.cuda.graph(graph, stream=stream):
                go()
    be.reserve_scratch(need)
    assert np.all(np.isfinite(captured(go, y)))  # and what it names is enough
    go = call = both = qw = None
    be.close()


def test_the_shared_expert_works_in_the_scratch_anyway():
    """A product that the large tiles would run whole (hidden 1408 x 576 and 1152 x 1408 at 174 tokens), inside a call that works in the
    context's scratch and is ordered by it: the few-token kernel's bits; of the plain call, the large tiles'."""
    import torch
    print("few-token context shared expert", flush=True)
    be = backend.HipQ4Backend(0)
    try:
        tokens, hidden, inter = 174, 1408, 576
        gu, dn = synth.q4_weight(2 * inter, hidden, seed=1), synth.q4_weight(hidden, inter, seed=2)
        x, sg = synth.activations(tokens, hidden, seed=3), synth.activations(1, hidden, seed=4)[0] / hidden ** 0.5
        qgu, qdn, dx, dsg = be.upload_q4_blocks(gu), be.upload_q4_blocks(dn), torch.from_numpy(x).cuda(), torch.from_numpy(sg).cuda()
        got, plain = {}, {}
        for which in (0, 2, 3):
            be.set_gemm_kernel(which)
            y, z = torch.zeros((tokens, hidden), device="cuda"), torch.empty((tokens, hidden), device="cuda")
            be.moe_shared_expert(qgu, qdn, dsg, inter, hidden, dx, y)
            be.dispatch_gemm(dx[:, :inter].contiguous(), 0, qdn, z, 0, tokens, hidden, inter)
            got[which], plain[which] = y.cpu().numpy(), z.cpu().numpy()
        assert rel_err(got[0], oracle.moe_shared_expert(gu, dn, sg, inter, hidden, x, np.zeros_like(got[0]))) <= REL_TOL
        assert np.array_equal(got[0], got[3]) and not np.array_equal(got[0], got[2])
        assert np.array_equal(plain[0], plain[2]) and not np.array_equal(plain[0], plain[3])
    finally:
        be.close()
