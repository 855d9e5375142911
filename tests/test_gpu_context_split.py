"""The split prefill launch (keys of a block shared out over workgroups, then
merged) against the float64 oracle, at the shapes where its cuts can go wrong:
one block over many workgroups, cuts between blocks, segments and heads,
segments without queries or prefix, padded groups and narrow heads, partial
last blocks, and parts whose maxima lie far apart."""

import numpy as np
import pytest
import torch

from akv_amd import _lib, context_attention as ca
from test_gpu_context_attention import TOL, _case, _run

pytestmark = pytest.mark.gpu


def _split(hq, hkv, d, q_lens, p_lens):
    return _lib.load().akv_context_attention_split_bytes(len(q_lens), hq, hkv, d, -1, sum(q_lens), max(q_lens),
                                                         sum(p_lens)) > 0


CASES = [
    # d, hq, hkv, queries, prefixes, cap
    (64, 8, 1, [3], [5000], 0.0),  # one short block over every workgroup it can feed
    (64, 64, 8, [200], [2500], 0.0),  # full blocks and a short last one
    (64, 16, 2, [1, 0, 300, 33], [4000, 10, 0, 1500], 0.0),  # no queries / no prefix
    (64, 32, 4, [64, 128, 65], [1024, 896, 1025], 0.0),  # blocks and tiles exactly full, and one past
    (128, 32, 8, [33, 257, 64], [1500, 700, 64], 0.0),
    (128, 4, 1, [1], [3000], 0.0),
    (64, 3, 3, [700], [1100], 0.0),  # group 1: 512-token blocks
    (128, 28, 4, [40, 9], [1300, 2000], 0.0),  # padded group
    (96, 24, 8, [50], [1800], 20.0),  # padded group, narrow head, cap
    (32, 8, 1, [17, 90], [2100, 5], 0.0),
]


@pytest.mark.parametrize("d,hq,hkv,q_lens,p_lens,cap", CASES)
@pytest.mark.parametrize("with_sinks,out_dtype", [(False, torch.float32), (True, torch.bfloat16)])
def test_split_matches_oracle(device, d, hq, hkv, q_lens, p_lens, cap, with_sinks, out_dtype):
    assert _split(hq, hkv, d, q_lens, p_lens)
    c = _case(device, hq, hkv, d, q_lens, p_lens, seed=d + hq + len(q_lens), slots=sum(p_lens) + 8)
    sinks = (torch.randn(hq, generator=torch.Generator().manual_seed(5)) * 2).to(device) if with_sinks else None
    print(f"split d={d} hq={hq} hkv={hkv} q={q_lens} p={p_lens} cap={cap} sinks={with_sinks}", flush=True)
    got, want = _run(device, c, window=-1, positions=False, sinks=sinks, out_dtype=out_dtype, scale=d ** -0.5,
                     logit_cap=cap)
    assert np.abs(got - want).max() <= TOL


@pytest.mark.parametrize("d,hq,hkv", [(64, 8, 1), (128, 8, 2)])
@pytest.mark.parametrize("step", [-300.0, -60.0, 30.0, 70.0, 300.0])
def test_split_parts_far_apart(device, d, hq, hkv, step):
    """Scores that step by ``step`` (log2 domain) every 500 prefix keys, so
    the parts' maxima differ by up to thousands: the merge keeps the largest
    part and drops what underflows beside it."""
    q_lens, p_lens = [20], [3000]
    assert _split(hq, hkv, d, q_lens, p_lens)
    c = _case(device, hq, hkv, d, q_lens, p_lens, seed=int(step) + 400, slots=4000)
    rng = np.random.default_rng(3)
    c["idx"] = (rng.permutation(3999)[:3000] + 1).astype(np.int32)
    c["q"][..., 0] = 8.0
    unit = d ** -0.5 * 1.4426950408889634 * 8.0
    for j in range(0, 3000, 500):
        c["kp"][torch.from_numpy(c["idx"][j:j + 500]).long(), :, 0] = step * (j // 500) / unit
    c["dev"]["q"], c["dev"]["kp"] = c["q"].to(device), c["kp"].to(device)
    print(f"split parts far apart d={d} step={step}", flush=True)
    got, want = _run(device, c, window=-1, positions=False, sinks=None, out_dtype=torch.float32, scale=d ** -0.5)
    assert np.isfinite(got).all()
    assert np.abs(got - want).max() <= TOL


@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("idx,ind,pos", [(torch.int32, torch.int64, torch.int64), (torch.int64, torch.int32, torch.int32),
                                         (torch.int64, torch.int64, None)])
@pytest.mark.parametrize("segments", [1, 7, 64])
def test_split_matches_plain(device, monkeypatch, d, idx, ind, pos, segments):
    """The split launch against the plain one over index and position types,
    strided queries, K/V, pools and outputs, and up to 64 segments (the last
    lane of its plan); the two differ by the rounding of their sums."""
    rng = np.random.default_rng(segments + d)
    q_lens = rng.integers(0, 90, segments)
    q_lens[0] = 37
    p_lens = rng.integers(0, 300, segments) + (4000 // segments)
    hq, hkv, nq, slots = 16, 2, int(q_lens.sum()), int(p_lens.sum()) + 8
    g = torch.Generator().manual_seed(d)

    def strided(n, heads):  # a view into wider rows
        t = torch.randn((n, heads + 1, d), generator=g).to(torch.bfloat16).to(device)
        return t[:, 1:]

    q, ke, ve, kp, vp = strided(nq, hq), strided(nq, hkv), strided(nq, hkv), strided(slots, hkv), strided(slots, hkv)
    indices = torch.from_numpy(rng.permutation(slots - 1)[: p_lens.sum()] + 1).to(idx).to(device)
    qo = torch.from_numpy(np.concatenate(([0], np.cumsum(q_lens)))).to(ind).to(device)
    kv = torch.from_numpy(np.concatenate(([0], np.cumsum(p_lens)))).to(ind).to(device)
    qp = kpos = None
    if pos is not None:
        qp = torch.arange(nq, dtype=pos, device=device) + 100000
        kpos = torch.arange(int(p_lens.sum()), dtype=pos, device=device)
    workspace = torch.empty(70 << 20, dtype=torch.uint8, device=device)  # more than either head_dim needs

    def run(split):
        monkeypatch.setattr(ca, "_split_workspace", lambda *a: workspace if split else None)
        out = torch.full((nq, hq + 2, d), 7.0, dtype=torch.float32, device=device)
        ca.extend_attention_fwd(q, ke, ve, out[:, 1:-1], kp, vp, qo, kv, indices, None, True, None, int(q_lens.max()),
                                context_q_positions=qp, context_kv_positions=kpos)
        torch.cuda.synchronize()
        assert (out[:, 0] == 7).all() and (out[:, -1] == 7).all()
        return out[:, 1:-1]

    got, want = run(True), run(False)
    # both round the weights to bf16 (2^-9) against a different maximum, so an
    # output differs by at most 2 x 2^-9 of the values' size (below 5)
    assert (got - want).abs().max() <= 2e-2


@pytest.mark.parametrize("d,hq,hkv", [(64, 16, 2), (128, 28, 4)])
@pytest.mark.parametrize("shift", [0, 1, 2, 5, 8])
def test_any_workspace(device, monkeypatch, d, hq, hkv, shift):
    """As many workgroups as the workspace holds parts for, from one up."""
    q_lens, p_lens = [200, 0, 33], [3000, 10, 1100]
    whole = 8 * (32768 + 2 * (512 if d == 64 else 256)) + 32  # two parts and a cut, per workgroup
    workspace = torch.full(((whole << shift) + 64,), 255, dtype=torch.uint8, device=device)
    monkeypatch.setattr(ca, "_split_workspace", lambda *a: workspace[: whole << shift])
    c = _case(device, hq, hkv, d, q_lens, p_lens, seed=shift)
    print(f"split workspace d={d} shift={shift}", flush=True)
    got, want = _run(device, c, window=-1, positions=False, sinks=None, out_dtype=torch.float32, scale=d ** -0.5)
    assert np.abs(got - want).max() <= TOL
    assert (workspace[whole << shift:] == 255).all()


def test_without_memory_the_plain_launch_runs(device, monkeypatch):
    q_lens, p_lens = [40], [3000]
    assert _split(16, 2, 64, q_lens, p_lens)
    c = _case(device, 16, 2, 64, q_lens, p_lens, seed=1)

    def run():
        return _run(device, c, window=-1, positions=False, sinks=None, out_dtype=torch.float32, scale=0.125)

    with monkeypatch.context() as m:
        m.setattr(ca, "_split_workspace", lambda *a: None)
        plain, want = run()
    empty, asked = torch.empty, []

    def no_memory(*args, dtype=None, **kw):
        if dtype is torch.uint8:
            asked.append(args)
            raise torch.OutOfMemoryError("no memory for the workspace")
        return empty(*args, dtype=dtype, **kw)

    monkeypatch.setattr(torch, "empty", no_memory)
    got, _ = run()
    assert len(asked) == 1
    assert (got == plain).all()
    assert np.abs(got - want).max() <= TOL


@pytest.mark.parametrize("d,hq,hkv", [(64, 64, 8), (128, 32, 8)])
def test_split_in_a_graph(device, d, hq, hkv):
    """Replays with other inputs in the same buffers, eager calls between them."""
    q_lens, p_lens = [70, 9], [2500, 900]
    assert _split(hq, hkv, d, q_lens, p_lens)
    nq, slots = sum(q_lens), sum(p_lens) + 8
    rng = np.random.default_rng(d)
    g = torch.Generator(device=device).manual_seed(d)
    q, ke, ve, kp, vp = (torch.empty((n, h, d), dtype=torch.bfloat16, device=device)
                         for n, h in ((nq, hq), (nq, hkv), (nq, hkv), (slots, hkv), (slots, hkv)))
    idx = torch.from_numpy((rng.permutation(slots - 1)[: sum(p_lens)] + 1).astype(np.int32)).to(device)
    qo = torch.tensor([0, 70, 79], dtype=torch.int32, device=device)
    kv = torch.tensor([0, 2500, 3400], dtype=torch.int32, device=device)
    out, eager = (torch.zeros((nq, hq, d), dtype=torch.bfloat16, device=device) for _ in range(2))

    def call(o):
        ca.extend_attention_fwd(q, ke, ve, o, kp, vp, qo, kv, idx, None, True, None, max(q_lens))

    def refill():
        for t in (q, ke, ve, kp, vp):
            t.normal_(generator=g)

    refill()
    call(eager)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(out)
    for _ in range(4):
        refill()
        call(eager)
        junk = torch.full((80 << 20,), 255, dtype=torch.uint8, device=device)  # where eager workspaces were
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
        del junk


# heads, head_dim, queries, prefixes; the last two fill a round of full blocks
@pytest.mark.parametrize("hq,hkv,d,q_lens,p_lens", [(16, 2, 64, [300, 17], [900, 40]), (32, 1, 64, [65, 9], [700, 20]),
                                                    (128, 1, 64, [7, 33], [600, 530]), (14, 2, 32, [130, 1], [20, 600]),
                                                    (64, 8, 64, [64] * 32, [30] * 32), (64, 8, 32, [63] * 32, [70] * 32)])
@pytest.mark.parametrize("positions", [True, False])
@pytest.mark.parametrize("window", [1, 256, 511, 512, 513, 700])
def test_windows_at_the_block_size_rule(device, hq, hkv, d, q_lens, p_lens, window, positions):
    """Blocks of a quarter of the rows (down to one token) where the window
    and the batch call for them, full blocks otherwise."""
    c = _case(device, hq, hkv, d, q_lens, p_lens, seed=window)
    got, want = _run(device, c, window=window, positions=positions, sinks=None, out_dtype=torch.float32, scale=0.125)
    assert np.abs(got - want).max() <= TOL


@pytest.mark.parametrize("window", [-1, 128, 600])
def test_without_the_queries_count(device, monkeypatch, window):
    """The entry that is not told how many queries the segments hold."""
    lib = _lib.load()

    class Unsized:
        akv_context_attention_split_bytes = staticmethod(lambda *a: 0)
        akv_context_attention_sized = staticmethod(lambda *a: lib.akv_context_attention(*a[:-2], a[-1]))

    monkeypatch.setattr(ca._lib, "calls", lambda: Unsized)
    c = _case(device, 16, 2, 64, [300, 17, 90], [900, 40, 300], seed=window + 2)
    got, want = _run(device, c, window=window, positions=True, sinks=None, out_dtype=torch.bfloat16, scale=0.125)
    assert np.abs(got - want).max() <= TOL


@pytest.mark.parametrize("positions", [True, False])
# the first visible key near the prefix's end, inside it, and at its start
@pytest.mark.parametrize("window", [1, 128, 500, 3000, 9000, 100000])
@pytest.mark.parametrize("d", [64, 128])
def test_windows_over_long_prefixes(device, d, window, positions):
    """Searches of two and three rounds for the first visible key."""
    c = _case(device, 8, 1, d, [20, 5, 70], [20000, 4097, 4095], seed=window, slots=24000)
    got, want = _run(device, c, window=window, positions=positions, sinks=None, out_dtype=torch.float32, scale=d ** -0.5)
    assert np.abs(got - want).max() <= TOL
