"""What the compiler made of the loads that kernels issue by hand: read from the built library, no GPU needed.

The integer matrix-core GEMV loads activations and adapter factors through inline assembly, which returns a register that the compiler
believes filled, and waits for them through inline assembly further down.  A copy or a spill in between would carry old data; no
result on the GPU would show it reliably.  And where the compiler believes loads of its own pending on registers of the product, it
waits for everything in flight in front of every unit.  The few-token GEMM's weights go into LDS by hand, beside operands that the
compiler loads and waits for: its waits count from where those stand among the others, and must not empty the queue."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from lattice_amd import build

OBJDUMP = shutil.which("llvm-objdump", path="/opt/rocm/llvm/bin:" + os.environ.get("PATH", ""))
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def code_objects(path):
    data = open(path, "rb").read()
    pos = data.find(BUNDLE)
    while pos >= 0:
        count, = struct.unpack_from("<Q", data, pos + len(BUNDLE))
        at = pos + len(BUNDLE) + 8
        for _ in range(count):
            off, size, length = struct.unpack_from("<QQQ", data, at)
            if b"gfx950" in data[at + 24:at + 24 + length]:
                yield data[pos + off:pos + off + size]
            at += 24 + length
        pos = data.find(BUNDLE, pos + 1)


def instantiations(kernel, tmp):
    """{name: [(address, text)]}"""
    if not OBJDUMP:
        pytest.skip("no llvm-objdump")
    if not os.path.exists(build.LIB):
        build.build()
    out = {}
    for i, obj in enumerate(code_objects(build.LIB)):
        if kernel.encode() not in obj:
            continue
        f = tmp / f"{i}.co"
        f.write_bytes(obj)
        name = None
        for line in subprocess.run([OBJDUMP, "-d", str(f)], capture_output=True, text=True, check=True).stdout.splitlines():
            head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
            if head:
                name = head[1] if kernel in head[1] else None
            elif name and "//" in line:
                text, _, note = line.partition("//")
                out.setdefault(name, []).append((int(note.split(":")[0], 16), text.strip()))
    return out


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """Of the integer matrix-core GEMV."""
    out = instantiations("gemv_q4_i8", tmp_path_factory.mktemp("i8"))
    assert len(out) == 64
    return out


@pytest.fixture(scope="module")
def few_token(tmp_path_factory):
    out = instantiations("gemm_q4_skinny", tmp_path_factory.mktemp("skinny"))
    assert len(out) == 48
    return out


def successors(ins):
    index = {a: i for i, (a, _) in enumerate(ins)}
    out = []
    for i, (a, text) in enumerate(ins):
        m = re.match(r"s_(c?)branch\w*\s+(\d+)", text)
        if m:
            offset = int(m[2]) - (65536 if int(m[2]) >= 32768 else 0)
            out.append([index[a + 4 + 4 * offset]] + ([i + 1] if m[1] else []))
        else:
            out.append([] if text.startswith("s_endpgm") or i + 1 == len(ins) else [i + 1])
    return out


def registers(text):
    out = set()
    for m in re.finditer(r"\b([va])(?:(\d+)\b|\[(\d+):(\d+)\])", text):
        first, last = (int(m[2]),) * 2 if m[2] else (int(m[3]), int(m[4]))
        out.update(m[1] + str(r) for r in range(first, last + 1))
    return out


def vmcnt(text):
    m = re.match(r"s_waitcnt .*vmcnt\((\d+)\)", text)
    return int(m[1]) if m else None


def test_nothing_touches_a_register_between_its_load_and_a_wait(kernels):
    """On no path through the code.  (A choice of waits by the number of units in flight is a chain of branches around them, in flags
    that this does not follow: entering the chain counts as waiting.)"""
    loads = 0
    for name, ins in kernels.items():
        waits = [i for i, (_, t) in enumerate(ins) if vmcnt(t) is not None]
        waited = {j for a, b in zip(waits, waits[1:] + [len(ins) * 2]) for j in (range(a, b + 1) if b - a < 24 else [a])}
        follow, state, work = successors(ins), [None] * len(ins), [0]
        state[0] = frozenset()
        while work:
            i = work.pop()
            text, flight = ins[i][1], state[i]
            by_hand = text.startswith("global_load_dwordx4") and i and ins[i - 1][1] == "s_nop 4"
            touched = registers(text.partition(",")[2] if text.startswith("global_load") else text)
            assert i in waited or not touched & flight, (name, hex(ins[i][0]), text)
            if i in waited:
                flight = frozenset()
            if by_hand:
                loads += 1
                flight = flight | registers(text.split(",")[0])
            for j in follow[i]:
                if state[j] is None or not flight <= state[j]:
                    state[j] = flight if state[j] is None else flight | state[j]
                    work.append(j)
    assert loads > 64


def test_scalar_addresses_of_loads_by_hand_are_settled(kernels, few_token):
    """Five wait states between a vector instruction that writes a scalar register and the load that reads it: the compiler counts
    them for its own instructions only."""
    writes = re.compile(r"v_(?:readlane|readfirstlane)_b32\S*\s+(s\d+)|v_cmp\S+\s+(s\[\d+:\d+\])")
    for name, ins in (kernels | few_token).items():
        for i, (a, text) in enumerate(ins):
            m = re.match(r"global_load\S*\s.*(s\[(\d+):(\d+)\])", text)
            if m and name in few_token and "_lds_" not in text:
                continue  # the compiler's own
            if not m:
                continue
            base, states, j = {f"s{r}" for r in range(int(m[2]), int(m[3]) + 1)}, 0, i - 1
            while j >= 0 and states < 5:
                w = writes.match(ins[j][1])
                assert not (w and (w[1] in base or w[2] == m[1])), (name, hex(a), ins[j][1], text)
                nop = re.match(r"s_nop (\d+)", ins[j][1])
                states += int(nop[1]) + 1 if nop else 1
                j -= 1


def test_the_product_waits_for_no_load_but_by_hand(kernels):
    """In the straight-line code of a unit's product: four blocks' matrix instructions twice, from its LDS reads on."""
    for name, ins in kernels.items():
        targets = {j for f in successors(ins) if len(f) != 1 for j in f} | {f[0] for i, f in enumerate(successors(ins)) if len(f) == 1 and f[0] != i + 1}
        products = [i for i, (_, t) in enumerate(ins) if t.startswith("v_mfma_i32")]
        assert len(products) == 8, name
        start = products[0]
        while start not in targets and not ins[start - 1][1].startswith(("s_branch", "s_cbranch")):
            start -= 1
        waits = [t for _, t in ins[start:products[-1]] if vmcnt(t) is not None]
        assert not waits, (name, waits)


def test_the_few_token_loop_keeps_two_units_in_flight(few_token):
    """The loop over K, two units a round: each unit's product, then the packed operands of the unit two places on, then its weights;
    in front of a product a wait by hand that leaves what was requested behind the unit, and none of the compiler's that leaves less
    than the next unit's operands."""
    for name, ins in few_token.items():
        rt, fmt, ntg = (int(v) for v in re.search(r"skinnyILi(\d)ELi(\d)ELi(\d)E", name).groups())
        bodies = []
        for i, follow in enumerate(successors(ins)):
            for j in follow:
                body = [t for _, t in ins[j:i + 1]]
                if j <= i and sum(t.startswith("v_mfma") for t in body) == 8 * rt * ntg and any("_lds_" in t for t in body):
                    bodies.append(body)
        body = min(bodies, key=len)
        kind = {"v_mfma": "M", "global_load_lds": "D", "global_load": "L"}
        runs = []
        for t in body:
            k = next((v for p, v in kind.items() if t.startswith(p)), None)
            if k:
                runs[-1:] = [(k, runs[-1][1] + 1)] if runs and runs[-1][0] == k else runs[-1:] + [(k, 1)]
        if runs[0][0] == runs[-1][0]:
            runs[0] = (runs[0][0], runs[0][1] + runs.pop()[1])
        order = "".join(k for k, _ in runs)
        assert order in ("MLDMLD", "LDMLDM", "DMLDML"), (name, runs)
        assert [c for k, c in runs if k == "M"] == [4 * rt * ntg] * 2 and [c for k, c in runs if k == "L"] == [4 * ntg] * 2, (name, runs)
        loads = -(-16 * rt * (5, 9, 4)[fmt] // 64)
        waits = [vmcnt(t) for t in body if vmcnt(t) is not None]
        assert waits.count(loads + 4 * ntg) >= 2 and min(waits) >= 4 * ntg, (name, waits)
