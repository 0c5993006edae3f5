"""The first launches of a process from several threads at once: the table of kernel handles is filled by whoever comes first."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

CHILD = """
import threading
import numpy as np
import torch
import oracle
from lattice_amd import backend, synth
from util import REL_TOL, rel_err

shapes = [(256, 256), (512, 2048), (4096, 1024), (300, 544)]
work = []
for i in range(8):
    n, k = shapes[i % 4]
    x, wq = synth.activations(64, k, seed=i), synth.q4_weight(n, k, seed=i % 4)
    be = backend.HipQ4Backend(0)
    work.append((n, k, x, wq, be, be.upload_q4_blocks(wq), torch.from_numpy(x).cuda(), torch.cuda.Stream()))
torch.cuda.synchronize()
start, got = threading.Barrier(8), [[] for _ in range(8)]

def go(i):
    n, k, x, wq, be, qw, dx, stream = work[i]
    start.wait()
    with torch.cuda.stream(stream):
        for batch in (1, 3, 8, 24, 64):
            y = torch.empty(batch, n, device="cuda")
            if batch <= 16:
                be.gemv_batch(dx[:batch], qw, y, batch, n, k)
            else:
                be.dispatch_gemm(dx[:batch], 0, qw, y, 0, batch, n, k)
            got[i].append((batch, y))
    stream.synchronize()

threads = [threading.Thread(target=go, args=(i,)) for i in range(8)]
for t in threads:
    t.start()
for t in threads:
    t.join()
for (n, k, x, wq, *_), ys in zip(work, got):
    assert len(ys) == 5
    for batch, y in ys:
        e = rel_err(y.cpu().numpy(), oracle.gemm_f32(x[:batch], wq, n, k))
        assert e <= REL_TOL, (n, k, batch, e)
print("eight threads done", flush=True)
"""


def test_first_launches_from_eight_threads():
    here = os.path.dirname(os.path.abspath(__file__))
    env = dict(os.environ, PYTHONPATH=os.pathsep.join([os.path.dirname(here), here]))
    done = subprocess.run([sys.executable, "-c", CHILD], env=env, capture_output=True, text=True, timeout=100)
    assert done.returncode == 0 and "eight threads done" in done.stdout, done.stdout + done.stderr
