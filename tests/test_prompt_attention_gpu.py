"""Attention of portions of prompts, 32 rows a wave, at the edges of its tiles
and in every width, against float64.

Tolerance: scores are fp32 and exact to some 2^-20; weights and results are
rounded to bf16, each off by 2^-9 / sqrt(3) of itself in the mean, and a result
is about the root of the sum of its squared terms: sqrt(2 / 3) 2^-9 or 1.6e-3
of the root mean square; twice that is allowed.
"""
import pytest
import torch

from hybrid_common import meta_for, rows_of
from ollamamq_amd.ops import interface as ops

pytestmark = pytest.mark.gpu
CLOSE = 3.2e-3


def _hip():
    from ollamamq_amd.ops import hip
    hip.require()
    return hip


def _rel(got, want):
    return ((got.double() - want).square().mean()
            / want.square().mean()).sqrt().item()


def _attend(q, k, v, scale, pos, lo, sink=None):
    """q [n, D] at positions pos, keys from lo on; float64, one head."""
    s = q.double() @ k.double().T * scale
    j = torch.arange(k.shape[0], device=q.device)
    s = s.masked_fill((j > pos[:, None]) | (j < lo[:, None]), -torch.inf)
    if sink is not None:
        s = torch.cat((s, sink.double().expand(len(s), 1)), 1)
    return torch.softmax(s, 1)[:, :k.shape[0]] @ v.double()


def _first(pos, window, chunk):
    if window:
        return (pos - window + 1).clamp(min=0)
    return pos - pos % chunk if chunk else pos * 0


@pytest.mark.parametrize("rows", [128, 256])
@pytest.mark.parametrize("H,G,D,V,page", [
    (8, 2, 128, 128, 16), (7, 1, 64, 64, 8), (6, 3, 128, 64, 32),
    (3, 3, 64, 128, 16), (4, 2, 72, 40, 16), (5, 1, 33, 100, 4),
    (8, 2, 128, 128, 2)])
@pytest.mark.parametrize("window,chunk,scale", [
    (0, 0, 0.1), (1, 0, 0.1), (70, 0, 0.1), (0, 50, 0.1), (0, 0, -0.1),
    (0, 0, 1e-30)])
def test_paged(rows, H, G, D, V, page, window, chunk, scale, monkeypatch):
    """Portions of several sequences, one after tokens it has seen before,
    with sinks; the most negative scores, and equal ones."""
    from ollamamq_amd.engine import HybridCache
    from ollamamq_amd.engine.kvcache import RunStore
    hip = _hip()
    monkeypatch.setattr(hip._lib, "softmax_rows", lambda *a: rows)
    g = torch.Generator(device="cuda").manual_seed(4)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    new, kv = [9, 64, 131, 65], [9, 200, 131, 129]
    cache = HybridCache([RunStore(kv=(G, D, V))], page_size=page,
                        n_pages=600 // page + 8, max_slots=4, max_ctx=256,
                        device="cuda", dtype=torch.bfloat16)
    sink = torch.randn(H, generator=g, device="cuda")
    w = ops.SoftmaxAttn(H, G, D, V, scale, sink, window, chunk=chunk)
    slots = [cache.alloc_slot() for _ in new]
    q, k, v = rand(sum(new), H, D), rand(4, 200, G, D), rand(4, 200, G, V)
    qp = torch.zeros(sum(new), H, cache.key_pool[0].shape[3],
                     device="cuda").bfloat16()
    qp[..., :D] = q
    want, at = [], 0
    for i, (n, have) in enumerate(zip(new, kv)):
        cache.ensure(slots[i], have)
        pages = cache.page_table[slots[i], :-(-have // page)].long()
        for pool, x in ((cache.key_pool[0], k), (cache.value_pool[0], v)):
            full = torch.zeros(len(pages) * page, G, pool.shape[3],
                               device="cuda").bfloat16()
            full[:have, :, :x.shape[3]] = x[i, :have]
            pool[pages] = full.view(-1, page, G, pool.shape[3]).transpose(1, 2)
        pos = torch.arange(have - n, have, device="cuda")
        want.append(torch.stack([_attend(
            q[at:at + n, h], k[i, :have, h * G // H], v[i, :have, h * G // H],
            scale, pos, _first(pos, window, chunk), sink[h])
            for h in range(H)], 1))
        at += n
    sl, pos = rows_of("cuda", slots, new, kv)
    got = ops.softmax_attention(qp, cache, 0, w, sl, pos,
                                meta_for("cuda", slots, new, kv))
    want = torch.cat(want)
    assert _rel(got.view_as(want), want) < CLOSE


@pytest.mark.parametrize("D,E,V", [
    (128, 64, 128), (120, 72, 50), (96, 64, 64), (64, 64, 128), (128, 0, 64),
    (32, 16, 128), (48, 16, 64), (33, 10, 30), (20, 7, 128), (100, 66, 64)])
@pytest.mark.parametrize("window", [0, 1, 70])
@pytest.mark.parametrize("scale", [0.1, -0.1])
def test_expanded(D, E, V, window, scale):
    """Contiguous keys with a shared part and transposed values, in tiles of
    which the last is not full."""
    hip, H = _hip(), 3
    QT = hip._lib.flash_rows(0, D + E, V)
    g = torch.Generator(device="cuda").manual_seed(5)
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda").bfloat16()
    new, kv = [33, 300, 64], [33, 400, 190]
    place = [0, 64, 64 + 448]                       # whole groups of 64 keys
    n_kv = 64 + 448 + 192
    k, kr, vt = rand(n_kv, H * D), rand(n_kv, E + 8), rand(H * V, n_kv)
    q, gate = rand(sum(new), H * (D + E)), rand(sum(new), H * V + 8)
    out = torch.zeros(sum(new), H, V, device="cuda").bfloat16()
    tiles, want, at = [], [], 0
    for n, have, kv0 in zip(new, kv, place):
        tiles += [(at + t, have - n + t, min(QT, n - t), kv0)
                  for t in range(0, n, QT)]
        pos = torch.arange(have - n, have, device="cuda")
        rows = slice(kv0, kv0 + have)
        want.append(torch.stack([_attend(
            q[at:at + n].unflatten(1, (H, -1))[:, h],
            torch.cat((k[rows, h * D:(h + 1) * D], kr[rows, :E]), 1),
            vt[h * V:(h + 1) * V, rows].T, scale, pos, _first(pos, window, 0))
            for h in range(H)], 1))
        at += n
    want = torch.cat(want) * gate[:, 8:].double().sigmoid().unflatten(
        1, (H, V))
    tl = torch.tensor(tiles, dtype=torch.int32, device="cuda")
    p = hip._p
    def launch(frag):
        hip._check(hip._lib.flash_attn(
            0, p(out), p(q), p(k), p(kr if E else None), p(vt), p(gate),
            gate.stride(0), 8, p(tl), len(tiles), H, D, E, V, q.stride(0),
            kr.stride(0), n_kv, scale, window, frag, hip._stream()),
            "flash_attn")

    launch(0)
    assert _rel(out, want) < CLOSE
    if H * V % 64 == 0:
        plain, T = out, out.shape[0]
        out = torch.zeros(-(-T // 32) * 32, H * V, device="cuda").bfloat16()
        launch(1)
        out = out.view(-1, H * V // 64, 4, 2, 32, 8).permute(0, 4, 1, 2, 3, 5)
        assert torch.equal(out.reshape(-1, H, V)[:T], plain)


def test_largest_weight_is_exact():
    """Rows whose maximum grows by less than 8 octaves after their first 64
    keys, at a key that alone has the value: the largest weight is 1, so what
    is left is the result's rounding to bf16, of 8 bits: half a unit, 2^-8 of
    it at most, and fp32's."""
    hip, n, D = _hip(), 128, 128
    g = torch.Generator(device="cuda").manual_seed(6)
    peak = 3.5 + 1.9 * torch.rand(n, generator=g, device="cuda")
    mass = 1 + torch.rand(n, generator=g, device="cuda")
    q, vt = torch.diag(peak).bfloat16(), torch.diag(mass).bfloat16()
    k = torch.eye(n, device="cuda").bfloat16()
    out = torch.zeros(n, D, device="cuda").bfloat16()
    tile = torch.tensor([[0, 0, n, 0]], dtype=torch.int32, device="cuda")
    p = hip._p
    hip._check(hip._lib.flash_attn(
        0, p(out), p(q), p(k), None, p(vt), None, 0, 0, p(tile), 1, 1, D, 0,
        D, D, 0, n, 1.0, 0, 0, hip._stream()), "flash_attn")
    pos = torch.arange(n, device="cuda")
    want = _attend(q, k, vt.T, 1.0, pos, pos * 0).diag()
    off = (out.diag().double() - want).abs() / want
    assert off.max().item() < 2 ** -8 * 1.01
