"""Decode attention at the edges of a workgroup's passes: one, two and four
passes of 256 keys per chunk, requests that end inside, at and past each of
them, bounds far from the longest request, unaligned queries, and an infinite
V row in the last key's place."""

import numpy as np
import pytest
import torch

from akv_amd import attention
from oracle import attention as oat

pytestmark = pytest.mark.gpu

TOL = 2e-2  # abs, bf16 weights: as the other decode checks
LENGTHS = [0, 1, 63, 64, 65, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 2049, 3000]


def _f32(t):
    return t.detach().float().cpu().numpy()


@pytest.mark.parametrize("head_dim", [64, 128])
# the bounds allow 1, 2 and 4 passes for these 16 x 8 heads
@pytest.mark.parametrize("max_len", [3000, 10000, 40000])
@pytest.mark.parametrize("aligned", [True, False])
def test_passes_match_oracle(device, head_dim, max_len, aligned):
    g = torch.Generator().manual_seed(head_dim + max_len)
    rng = np.random.default_rng(max_len)
    slots, hq, hkv, B = 4000, 64, 8, len(LENGTHS)
    k = torch.randn((slots, hkv, head_dim), generator=g).to(torch.bfloat16).to(device)
    v = torch.randn((slots, hkv, head_dim), generator=g).to(torch.bfloat16).to(device)
    q = torch.empty(B * hq * head_dim + 1, dtype=torch.bfloat16, device=device)[0 if aligned else 1:]
    q = q[: B * hq * head_dim].view(B, hq, head_dim)
    q.copy_(torch.randn((B, hq, head_dim), generator=g))
    indptr = np.concatenate(([0], np.cumsum(LENGTHS))).astype(np.int32)
    idx = rng.integers(1, slots, size=indptr[-1]).astype(np.int32)
    sinks = torch.randn(hq, generator=g).to(device)
    out = torch.full((B, hq, head_dim), 7.0, dtype=torch.float32, device=device)
    print(f"decode passes d={head_dim} max_len={max_len} aligned={aligned}", flush=True)
    attention.decode_attention(q, k, v, torch.from_numpy(indptr).to(device), torch.from_numpy(idx).to(device), out,
                               scale=head_dim ** -0.5, max_len=max_len, sinks=sinks)
    torch.cuda.synchronize()
    got, kk, vv, qq = _f32(out), _f32(k), _f32(v), _f32(q)
    for b, n in enumerate(LENGTHS):
        sel = idx[indptr[b]: indptr[b + 1]]
        err = np.abs(got[b] - oat.decode_attention(qq[b], kk[sel], vv[sel], head_dim ** -0.5, _f32(sinks))).max()
        assert err <= TOL, f"request {b} (len {n}) max err {err}"


@pytest.mark.parametrize("head_dim,hq,hkv", [(64, 64, 64), (128, 64, 32)])
# keys of all requests times KV heads, over 512: 2048 take two passes, 4096 four
@pytest.mark.parametrize("passes", [1, 2, 4])
# the longest request, a bound of few chunks (requests before heads in the
# grid), and one of many more than the batch fills
@pytest.mark.parametrize("bound", [None, 3500, 70000])
def test_passes_of_the_batch(device, head_dim, hq, hkv, passes, bound):
    """Lengths at the edges of a chunk of ``passes`` passes and of its equal
    shares; the batch's keys, not the bound, say how many passes there are."""
    edge = 256 * passes
    lengths = [0, 1, 63, 255, 257, 511, 512, 513, edge - 1, edge, edge + 1, 2 * edge - 1, 2 * edge + 1, 3 * edge - 65,
               3 * edge + 64, 3000]
    need = {1: 0, 2: 2048, 4: 4096}[passes] * 512
    while sum(lengths) * hkv < need:
        lengths.append(min(2600 + len(lengths), -(-(need - sum(lengths) * hkv) // hkv)))
    assert {1: 0, 2: 2048, 4: 4096}[passes] <= sum(lengths) * hkv // 512 < {1: 2048, 2: 4096, 4: 1 << 30}[passes]
    g = torch.Generator().manual_seed(head_dim + passes)
    rng = np.random.default_rng(passes)
    slots, B = 4000, len(lengths)
    k = torch.randn((slots, hkv, head_dim), generator=g).to(torch.bfloat16).to(device)
    v = torch.randn((slots, hkv, head_dim), generator=g).to(torch.bfloat16).to(device)
    q = torch.randn((B, hq, head_dim), generator=g).to(torch.bfloat16).to(device)
    indptr = np.concatenate(([0], np.cumsum(lengths))).astype(np.int32)
    idx = rng.integers(1, slots, size=indptr[-1]).astype(np.int32)
    out = torch.full((B, hq, head_dim), 7.0, dtype=torch.float32, device=device)
    print(f"decode batch passes={passes} d={head_dim} bound={bound}", flush=True)
    attention.decode_attention(q, k, v, torch.from_numpy(indptr).to(device), torch.from_numpy(idx).to(device), out,
                               scale=head_dim ** -0.5, max_len=bound or max(lengths))
    torch.cuda.synchronize()
    got, kk, vv, qq = _f32(out), _f32(k), _f32(v), _f32(q)
    for b, n in enumerate(lengths):
        sel = idx[indptr[b]: indptr[b + 1]]
        err = np.abs(got[b] - oat.decode_attention(qq[b], kk[sel], vv[sel], head_dim ** -0.5, None)).max()
        assert err <= TOL, f"request {b} (len {n}) max err {err}"


@pytest.mark.parametrize("head_dim", [64, 128])
@pytest.mark.parametrize("n", [1, 5, 130, 700])
def test_infinite_last_value_stays_infinite(device, head_dim, n):
    """Nothing past a request's last key is multiplied with that key's V row:
    an infinite value there gives infinity, not NaN."""
    g = torch.Generator().manual_seed(n)
    k = torch.randn((n + 1, 1, head_dim), generator=g).to(torch.bfloat16).to(device)
    v = torch.randn((n + 1, 1, head_dim), generator=g).to(torch.bfloat16).to(device)
    v[n, 0, 3] = float("inf")
    q = torch.randn((1, 8, head_dim), generator=g).to(torch.bfloat16).to(device)
    out = torch.zeros((1, 8, head_dim), dtype=torch.float32, device=device)
    attention.decode_attention(q, k, v, torch.tensor([0, n], dtype=torch.int32, device=device),
                               torch.arange(1, n + 1, dtype=torch.int32, device=device), out,
                               scale=head_dim ** -0.5, max_len=n)
    torch.cuda.synchronize()
    assert torch.isposinf(out[0, :, 3]).all()
    assert torch.isfinite(torch.cat((out[0, :, :3], out[0, :, 4:]), dim=1)).all()
