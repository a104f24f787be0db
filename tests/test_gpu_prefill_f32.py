"""The f32 pool's prefill kernels (32-row wavefront tiles with two key halves at head dims 64 and
128, 16-row ones at 256 and for sequences of up to 128 keys) at the edges of their tiles, against
the oracle.

Tolerance: an operand x is kept as bf16 hi + lo (relative error 2^-17), the lo.lo product is
dropped (2^-16 of |q_i k_i|), so a score moves by at most e = 2^-15 scale sum_i |q_i k_i|, a
softmax weight by a factor within exp(+-2 e), and the weights' and values' own splits add
2^-15: |out - ref| <= (exp(2 e) - 1 + 2^-15) max |v| + f32 rounding (2^-20 max |v|).
"""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from tests.gpu_util import device, to_dev
from tests.test_gpu_prefill_paged import Chunk

pytestmark = pytest.mark.gpu


def _bound(q, k, v):
    hq, hkv, d = q.shape[1], k.shape[1], q.shape[2]
    kk = np.abs(k[:, np.arange(hq) % hkv].astype(np.float64))  # modulo head map
    e = 2.0 ** -15 * np.einsum("nhd,lhd->nlh", np.abs(q.astype(np.float64)), kk).max() / np.sqrt(d)
    return (np.expm1(2 * e) + 2.0 ** -15 + 2.0 ** -20) * np.abs(v).max()


def _check(c, out, rows, k=None, v=None):
    q, kr, vr = c.prepared(f32=True)
    k, v = (kr if k is None else k), (vr if v is None else v)
    for i in rows:
        ref = orc.attn_decode(q[i], k[:c.prev + i + 1], v[:c.prev + i + 1])
        err, tol = float(np.abs(out[i] - ref).max()), _bound(q[i:i + 1], k[:c.prev + i + 1], v)
        assert err <= tol, f"row {i}: max-abs {err} > {tol}"


# rows around the 32-row groups and the 32 / 64 / 128-row blocks of 4, 2 and 1 heads a workgroup;
# histories at and beside tiles, so that a key half holds no key of some rows
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 2), (3, 3), (5, 2)])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("prev,n", [(0, 31), (0, 33), (31, 1), (63, 66), (64, 127), (97, 129)])
def test_f32_prefill_tile_edges(prev, n, hq, hkv, d):
    c = Chunk(np.random.default_rng(prev * 131 + n + hq + d), prev, n, hq, hkv, d)
    out = c.gpu(device(), pool_dtype=torch.float32)
    _check(c, out, sorted({0, n // 2, n - 1} | {r for r in (31, 32, 63, 64, 127, 128) if r < n}))


# 128 keys in all pick the 16-row kernel at every head dim, 129 the 32-row one at 64 and 128
@pytest.mark.parametrize("hq,hkv", [(8, 2), (3, 3), (5, 2)])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("prev,n", [(0, 1), (0, 16), (0, 17), (0, 128), (0, 129), (127, 1), (128, 1), (95, 33),
                                    (96, 33), (50, 64)])
def test_f32_prefill_short_sequences(prev, n, hq, hkv, d):
    c = Chunk(np.random.default_rng(prev * 17 + n + hq + d), prev, n, hq, hkv, d)
    out = c.gpu(device(), pool_dtype=torch.float32)
    _check(c, out, sorted({0, n // 2, n - 1} | {r for r in (15, 16, 31, 32, 127) if r < n}))


@pytest.mark.parametrize("d", [64, 128, 256])
def test_f32_prefill_max_rises_late(d):
    """Scores that outgrow the running max tile after tile."""
    c = Chunk(np.random.default_rng(d), 0, 200, 4, 2, d)
    c.k *= np.linspace(0.2, 4.0, 200, dtype=np.float32)[:, None, None]
    out = c.gpu(device(), pool_dtype=torch.float32)
    _check(c, out, [0, 31, 63, 64, 130, 199])


@pytest.mark.parametrize("late", [70, 150, 190])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_f32_prefill_largest_weight_is_exact(d, late):
    """One key ahead of two in the first tile (one a key half) by less than 2^8, the rest far
    behind: its weight is exactly 1 in the products too.  Scores and values are exact here, so
    what is left is the rounding of the scaled scores below 8 (2^-22 each), an exponential, the
    sum of three and the division (2^-23 each): 2^-20; a weight kept as bf16 hi + lo is off by
    up to 2^-17."""
    from powerinfer_x64_amd import runtime as rt
    dev = device()
    n, prev = 45, 200
    a = 1 + np.arange(n) / 128.0  # 8 bits
    q, k, v = np.zeros((n, 2, d), np.float32), np.zeros((1, prev + n, 1, d), np.float32), np.zeros((1, prev + n, 1, d), np.float32)
    q[:, :, 0] = a[:, None]
    k[0, :, 0, 0] = -64
    k[0, [5, 40], 0, 0] = 0
    k[0, late, 0, 0] = 4
    v[0, late] = 1
    pages = (prev + n + 15) // 16
    pt = to_dev(np.random.default_rng(d).permutation(pages).astype(np.int32)[None])
    pool = rt.KvPool(dev, pages, 1, d, dtype=torch.float32)
    pool.append(to_dev(k), to_dev(v), pt, torch.zeros(1, dtype=torch.int32, device="cuda"))
    out = rt.attn_prefill_paged(dev, to_dev(q), pool, pt[0].contiguous(), prev, scale=1.0).cpu().numpy()
    w = np.exp(4 * a)
    assert float(np.abs(out / (w / (w + 2))[:, None, None] - 1).max()) <= 2.0 ** -20


# history, chunk and the pages made invalid: inside and at the edges of the 32-key halves and the
# 32 / 64-key tiles, whole tiles (first, last), the chunk's own pages, and every page of a row
@pytest.mark.parametrize("ksplit", ["1", "3"])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("prev,n,bad", [(150, 40, (3, 9)), (150, 40, (4, 5, 6, 7, 11)), (0, 100, (0, 1)),
                                        (200, 70, (0, 1, 2, 3, 12, 13, 16)), (37, 60, tuple(range(6)))])
def test_f32_prefill_pages_outside_the_pool_hold_no_tokens(monkeypatch, prev, n, bad, d, ksplit):
    """Page-table entries outside [0, n_pages) hold no tokens, as for the decode and the f16
    prefill: their keys are left out of the softmax, and a row with no other key gets zeros."""
    from powerinfer_x64_amd import runtime as rt
    dev = device()
    monkeypatch.setenv("PI_PREFILL_KSPLIT", ksplit)
    c = Chunk(np.random.default_rng(d + prev), prev, n, 4, 2, d)
    c.gpu(dev, pool_dtype=torch.float32)
    q, k, v = c.prepared(f32=True)
    row, keep = c.row.copy(), np.ones(prev + n, bool)
    for i, p in enumerate(bad):
        row[p] = (-1, c.n_pages, c.n_pages + 3, -7)[i % 4]
        keep[16 * p:16 * p + 16] = False
    out = rt.attn_prefill_paged(dev, to_dev(q), c.pool, to_dev(row), prev).cpu().numpy()
    dec = rt.attn_decode(dev, to_dev(q), c.pool, to_dev(np.tile(row, (n, 1))),
                         to_dev(np.arange(prev + 1, prev + n + 1, dtype=np.int32))).cpu().numpy()
    for i in range(n):
        m = keep[:prev + i + 1]
        kk, vv = k[:prev + i + 1][m], v[:prev + i + 1][m]
        if not m.any():
            assert not out[i].any() and not dec[i].any(), f"row {i} has no keys"
            continue
        ref, tol = orc.attn_decode(q[i], kk, vv), _bound(q[i:i + 1], kk, v)
        assert float(np.abs(out[i] - ref).max()) <= tol, f"row {i}"
        assert float(np.abs(out[i] - dec[i]).max()) <= 2 * tol, f"row {i} against the decode"


@pytest.mark.parametrize("ksplit", ["2", "3", "4"])
@pytest.mark.parametrize("prev,n,hq,hkv,d", [(0, 300, 4, 1, 64), (500, 130, 3, 3, 128), (1000, 33, 5, 2, 128),
                                             (64, 257, 8, 4, 256), (2000, 16, 16, 2, 256)])
def test_f32_prefill_key_splits(monkeypatch, prev, n, hq, hkv, d, ksplit):
    """Forced key splits: pieces of the longest blocks, short blocks whole, pieces that hold no key
    of a row, through the layer's gated step as well as the paged entry."""
    from powerinfer_x64_amd import runtime as rt
    dev = device()
    c = Chunk(np.random.default_rng(prev + n + d), prev, n, hq, hkv, d)
    monkeypatch.setenv("PI_PREFILL_KSPLIT", ksplit)
    out = c.gpu(dev, pool_dtype=torch.float32)
    _check(c, out, sorted({0, 1, 31, n // 2, n - 1} & set(range(n))))
    if prev == 0:
        g = np.random.default_rng(1).standard_normal((n, hq, d)).astype(np.float32)
        got = []
        for k in (ksplit, "1"):
            monkeypatch.setenv("PI_PREFILL_KSPLIT", k)
            layer = rt.AttnLayer(dev, n, hq, hkv, d, torch.float32, rope_base=c.theta)
            got.append(layer.forward_dev(*(to_dev(x) for x in (c.q, c.k, c.v, g))))
        assert float((got[0] - got[1]).abs().max()) <= 2.0 ** -18 * float(np.abs(c.v).max())


def test_f32_prefill_automatic_split_and_capture():
    """Few queries over a long history: the launch splits by itself, and not under capture; the
    replays equal the eager unsplit call bit for bit."""
    import os
    from powerinfer_x64_amd import runtime as rt
    dev = device()
    c = Chunk(np.random.default_rng(7), 3000, 20, 8, 2, 128)
    out = c.gpu(dev, pool_dtype=torch.float32)
    _check(c, out, [0, 7, 19])
    q = to_dev(c.prepared(f32=True)[0])
    os.environ["PI_PREFILL_KSPLIT"] = "1"
    try:
        ref = rt.attn_prefill_paged(dev, q, c.pool, c.row_dev, c.prev)
    finally:
        del os.environ["PI_PREFILL_KSPLIT"]
    o = torch.zeros_like(ref)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        rt.attn_prefill_paged(dev, q, c.pool, c.row_dev, c.prev, out=o)
    for _ in range(3):
        o.zero_()
        rt.attn_prefill_paged(dev, q, c.pool, c.row_dev, c.prev)  # eager work between replays
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(o, ref)
