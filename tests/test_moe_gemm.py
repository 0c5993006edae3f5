"""The grouped GEMM of the MoE path (many tokens per expert) against the oracle at the sizes where its tiles end: pairs per
expert around 32 and 64, rows of a number of blocks that is not a multiple of a step (4) or of a pair of steps (8), outputs
that do not fill a workgroup's chunk, a shared expert narrower and wider than the routed ones."""
import numpy as np
import pytest

import oracle
from lattice_amd import backend, synth
from util import rel_err

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def be():
    return backend.HipQ4Backend(0)


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("cfg", [dict(e=1, inter=128, shared=128, hidden=128, tokens=31, top_k=1),
                                 dict(e=1, inter=160, shared=128, hidden=224, tokens=33, top_k=1),    # 5 and 7 blocks a row
                                 dict(e=2, inter=192, shared=288, hidden=544, tokens=64, top_k=2),    # 6, 9 and 17 blocks
                                 dict(e=3, inter=288, shared=160, hidden=1056, tokens=65, top_k=3),   # every expert: 65 pairs
                                 dict(e=7, inter=512, shared=1024, hidden=2048, tokens=120, top_k=4),
                                 dict(e=2, inter=1056, shared=128, hidden=256, tokens=512, top_k=2)])
def test_moe_grouped_gemm_matches_oracle(be, cfg):
    import torch
    e_, inter, sh, hidden, tokens, top_k = (cfg[k] for k in ("e", "inter", "shared", "hidden", "tokens", "top_k"))
    print(f"moe grouped gemm {cfg}", flush=True)
    gu = synth.q4_weight(e_ * 2 * inter, hidden, seed=9, tag="gu", symmetric_bias=False)
    dn = synth.q4_weight(e_ * hidden, inter, seed=9, tag="dn", symmetric_bias=False)
    sgu, sdn = synth.q4_weight(2 * sh, hidden, seed=9, tag="sgu"), synth.q4_weight(hidden, sh, seed=9, tag="sdn")
    x, lg = synth.activations(tokens, hidden, seed=9), synth.router_logits(tokens, e_, seed=9)
    x[1] = 0.0
    x[2] *= 1e12
    x[3] *= 1e-6
    sg = (np.random.default_rng(9).normal(size=hidden) * (2.0 / np.sqrt(hidden))).astype(np.float32)
    q = [be.upload_q4_blocks(b) for b in (gu, dn, sgu, sdn)]
    y = torch.full((tokens, hidden), float("nan"), dtype=torch.float32, device="cuda")

    ids, wts, _ = oracle.moe_route(lg, top_k)
    want = oracle.moe_ffn(gu, dn, e_, inter, hidden, x, ids, wts, f64=True)
    want = oracle.moe_shared_expert(sgu, sdn, sg, sh, hidden, x, want, f64=True)
    be.moe_ffn(dev(lg), q[0], q[1], e_, top_k, inter, q[2], q[3], dev(sg), sh, hidden, dev(x), y)
    got = y.cpu().numpy()
    rows = [r for r in range(tokens) if r != 2]
    assert rel_err(got[rows], want[rows]) <= 2e-6 and rel_err(got[2], want[2]) <= 2e-5 and rel_err(got[3], want[3]) <= 2e-5

    # the routed experts alone, with slots that no expert fills; an infinity spoils its own token only
    if e_ > 1:
        ids[0, top_k - 1], ids[tokens - 1, 0] = -1, e_ + 1
    x[5, 7] = np.inf
    y.fill_(float("nan"))
    be.moe_experts(q[0], q[1], e_, inter, hidden, dev(x), dev(ids), dev(wts), y)
    want = oracle.moe_ffn(gu, dn, e_, inter, hidden, x, ids, wts, f64=True)
    got = y.cpu().numpy()
    rows = [r for r in range(tokens) if r not in (2, 5)]
    assert rel_err(got[rows], want[rows]) <= 2e-6 and np.isnan(got[5]).all()
