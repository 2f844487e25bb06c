"""The row-packed attention kernel (csrc/attention_rows.hip): few query rows
per KV head, keys dealt to waves and, with a workspace, to workgroups.

Bar: max|o - o_cpu| / max|o_cpu| <= 2e-3 (f16; the fp16 parity bound) and
4e-4 (f32 results: f16 probabilities) against the oracle. Cases with a
workspace run twice on it (re-armed counters).
"""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def rand(g, *shape):
    return torch.randn(*shape, generator=g).half()


def family(pkg, q, k, v, o, causal=False, mask=None):
    """The kernel that the wrapper's call of these operands runs."""
    a = pkg.AttentionArgs(
        q=q.data_ptr(), k=k.data_ptr(), v=v.data_ptr(), o=o.data_ptr(),
        batch=q.shape[0], heads=q.shape[1], kv_heads=k.shape[1],
        seq_q=q.shape[2], seq_kv=k.shape[2], head_dim=q.shape[3],
        head_dim_v=v.shape[3], scale=0.1,
        flags=((pkg.CAUSAL if causal else 0) |
               (pkg.ATTENTION_OUT_F32 if o.dtype == torch.float32 else 0) |
               (pkg.ATTENTION_MASK if mask is not None else 0)))
    for f, t in (("q", q), ("k", k), ("v", v), ("o", o)):
        getattr(a.strides, f)[:] = list(t.stride()[:3])
    if mask is not None:
        m = mask.expand(q.shape[0], q.shape[1], q.shape[2], k.shape[2])
        a.mask = m.data_ptr()
        a.mask_strides[:] = list(m.stride())
    return pkg.classify_attention(a)


def run(pkg, oracle, b, h, hk, sq, skv, d, dv, causal=False, mask=None,
        out_f32=False, seed=0, cache=0, twice=True, bound=None,
        rows_only=False):
    g = torch.Generator().manual_seed(seed)
    q = rand(g, b, h, sq, d)
    k = rand(g, b, hk, skv + cache, d)
    v = rand(g, b, hk, skv + cache, dv)
    dt = torch.float32 if out_f32 else torch.float16
    kd, vd = k.cuda()[:, :, :skv], v.cuda()[:, :, :skv]
    # o is laid out [B, S, H, D], with canary columns
    for _ in range(2 if twice else 1):
        buf = torch.full((b, sq, h, dv + 8), 99.0, dtype=dt, device="cuda")
        o = buf[..., :dv].permute(0, 2, 1, 3)
        qd, md = q.cuda(), None if mask is None else mask.cuda()
        if rows_only:
            assert family(pkg, qd, kd, vd, o, causal,
                          md) == pkg.ATTENTION_FAMILY_ROWS
        pkg.attention(qd, kd, vd, o, causal=causal, mask=md)
        got = o.cpu().numpy()
        assert bool((buf[..., dv:] == 99).all()), "write past the head dim"
        ref = oracle.attention(
            q.numpy(), k[:, :, :skv].contiguous().numpy(),
            v[:, :, :skv].contiguous().numpy(), scale=d ** -0.5,
            causal=causal, out_f32=out_f32,
            mask=None if mask is None else
            mask.expand(b, h, sq, skv).contiguous().numpy())
        ref = ref.astype(np.float32)
        assert np.isfinite(got).all()
        err = oracle.fp16_parity(got, ref)
        assert err <= (bound or (4e-4 if out_f32 else 2e-3)), err
    return got


def need(pkg, b, h, hk, sq, skv, d, dv, flags=0):
    return pkg._attention_workspace_need(b, h, hk, sq, skv, d, dv, flags)


# (most of these are the row-packed kernel's, some of the few-key and causal
# ones another's) edges: one key, blocks of 32 keys and 16 / 32 rows, a key block for some
# waves only, head dims short of their bucket, split and unsplit
@pytest.mark.parametrize("b,h,hk,sq,skv,d,dv", [
    (1, 8, 1, 1, 2048, 128, 128), (2, 8, 2, 1, 3001, 64, 64),
    (1, 6, 2, 5, 1023, 80, 80), (1, 4, 4, 3, 4097, 40, 40),
    (1, 16, 1, 2, 777, 192, 128), (1, 3, 3, 33, 33, 256, 256),
    (1, 2, 1, 16, 300, 8, 24), (2, 9, 3, 200, 200, 64, 64),
    (1, 4, 1, 31, 31, 96, 128)])
@pytest.mark.parametrize("causal", [False, True])
def test_rows_shapes(pkg, oracle, dev, b, h, hk, sq, skv, d, dv, causal):
    print(f"rows {b} {h} {hk} {sq} {skv} {d} {dv} {causal}", flush=True)
    run(pkg, oracle, b, h, hk, sq, skv, d, dv, causal, cache=5,
        out_f32=sq == 5)


@pytest.mark.parametrize("out_f32", [False, True])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("sq,d,dv", [
    (sq, d, dv) for sq in (3, 37)
    for d, dv in ((64, 56), (40, 64), (128, 120), (104, 72), (256, 200),
                  (136, 248))])
def test_rows_instances(pkg, oracle, dev, sq, d, dv, masked, out_f32):
    """Every instance: 16- and 32-row tiles of each head-dim bucket, head dims
    short of it and apart, with and without a mask, f16 and f32 out, keys
    split over workgroups or (777 keys at 37 queries) not."""
    skv = 777 if sq == 37 else 1500
    print(f"rows instance {sq} {skv} {d} {dv} {masked} {out_f32}", flush=True)
    mask = None
    if masked:
        g = torch.Generator().manual_seed(d)
        mask = torch.randn(sq, skv, generator=g).half()
        mask[torch.rand(sq, skv, generator=g) < 0.2] = -float("inf")
    run(pkg, oracle, 1, 4, 1, sq, skv, d, dv, mask=mask, out_f32=out_f32,
        seed=d + dv, rows_only=True)


def test_rows_route_and_split(pkg):
    """One query over a long cache splits its keys; a long prompt does not
    come here."""
    assert need(pkg, 4, 32, 8, 1, 3001, 128, 128) > 256 * 1024
    assert need(pkg, 1, 32, 32, 2048, 2048, 128, 128, pkg.CAUSAL) == 0


@pytest.mark.parametrize("skv", [4, 5, 7, 63, 777])
@pytest.mark.parametrize("kind", ["random", "hidden_rows", "lowest"])
def test_rows_masks(pkg, oracle, dev, skv, kind):
    g = torch.Generator().manual_seed(skv)
    sq = 37
    m = torch.randn(sq, skv, generator=g).half()
    if kind == "random":
        m[torch.rand(sq, skv, generator=g) < 0.3] = -float("inf")
    elif kind == "hidden_rows":
        m[::3] = -float("inf")
    else:  # the lowest f16 hides keys and, in some rows, all of them
        m[torch.rand(sq, skv, generator=g) < 0.3] = -65504.0
        m[1::4] = -65504.0
    # a row hidden by the lowest f16 throughout: its scores are rounded at
    # 65504's f32 spacing (2^-8; 2^-7 in the log2 units of the fused kernel,
    # which takes 4 keys), half of it on either side: 4e-3 of a weight each
    got = run(pkg, oracle, 2, 6, 2, sq, skv, 64, 64, mask=m, twice=False,
              seed=skv, bound=8e-3 if kind == "lowest" else None)
    if kind == "hidden_rows":
        assert bool((got[:, :, ::3] == 0).all())


def test_rows_infinities(pkg, dev):
    """A NaN or infinite value reaches the rows that see it and no others; a
    +inf score makes its row NaN (inf - inf, as in torch's softmax and the
    other kernels)."""
    g = torch.Generator().manual_seed(3)
    q, k = rand(g, 1, 4, 3, 64).cuda(), rand(g, 1, 1, 1500, 64).cuda()
    v = rand(g, 1, 1, 1500, 64).cuda()
    q[0, 2, 1, 5] = float("nan")
    o = pkg.attention(q, k, v, causal=False)
    bad = torch.isnan(o).all(-1)[0]
    assert bool(bad[2, 1]) and int(bad.sum()) == 1
    # +inf scores: q . k overflows to +inf where q has an infinity and k is
    # positive, to -inf where k is negative
    q[0, 2, 1, 5] = float("inf")
    o = pkg.attention(q, k, v, causal=False)
    bad = torch.isnan(o).all(-1)[0]
    assert bool(bad[2, 1]) and int(bad.sum()) == 1
    assert bool(torch.isfinite(o[0][~bad]).all())
    q[0, 2, 1, 5] = 0
    v[0, 0, 7, 11] = float("inf")
    o = pkg.attention(q, k, v, causal=False)
    assert bool(torch.isinf(o[..., 11]).all())
    assert bool(torch.isfinite(o[..., :11]).all())
    # a key past the filled part of the cache is not read into any row
    v[0, 0, 7, 11] = 0
    k[0, 0, 1400:] = float("nan")
    v[0, 0, 1400:] = float("nan")
    o = pkg.attention(q, k[:, :, :1400], v[:, :, :1400], causal=False)
    assert bool(torch.isfinite(o).all())


@pytest.mark.parametrize("kernel", ["ROWS", "FUSED"])
def test_hidden_non_finite_values(pkg, dev, kernel):
    """Under the causal mask a key's NaN or infinity in K stays out of the
    rows that do not see it. One in V is multiplied by their weight of 0, so
    it spreads to rows of its own tile (rows of one 32-row tile on the
    row-packed kernel, of one 128-row block on the fused one), in its own
    column and to no earlier tile."""
    b, h, s, d = (1, 4, 192, 64) if kernel == "ROWS" else (2, 32, 600, 64)
    g = torch.Generator().manual_seed(4)
    q, k, v = (rand(g, b, h, s, d).cuda() for _ in range(3))
    assert family(pkg, q, k, v, torch.empty_like(q), True) == getattr(
        pkg, "ATTENTION_FAMILY_" + kernel)
    tile = 32 if kernel == "ROWS" else 128
    key = s // 2 + 3
    want = pkg.attention(q, k, v).float()

    def same(got, ref):
        # a row's maximum may have been moved at another block: rounding
        return bool(((got.float() - ref).abs() <= 2e-3 * ref.abs().max()).all())

    for bad in (float("nan"), float("inf")):
        k2, v2 = k.clone(), v.clone()
        k2[0, 1, key, 7] = bad
        o = pkg.attention(q, k2, v)
        assert same(o[0, 1, :key], want[0, 1, :key])
        assert bool(torch.isnan(o[0, 1, key:]).any())
        v2[0, 1, key, 11] = bad
        o = pkg.attention(q, k, v2)
        first = key // tile * tile
        assert same(o[0, 1, :first], want[0, 1, :first])
        assert bool((~torch.isfinite(o[0, 1, key:, 11])).all())
        o[0, 1, :, 11] = want[0, 1, :, 11].half()
        assert same(o, want)


def test_rows_with_less_workspace(pkg, oracle, dev):
    """The same call with no workspace, a short one and all it can use: the
    same values within the rounding of the probabilities."""
    g = torch.Generator().manual_seed(9)
    q, k = rand(g, 1, 8, 1, 128).cuda(), rand(g, 1, 2, 4000, 128).cuda()
    v = rand(g, 1, 2, 4000, 128).cuda()
    lib, st = pkg.library(), torch.cuda.current_stream().cuda_stream
    full = need(pkg, 1, 8, 2, 1, 4000, 128, 128)
    assert full > 0
    outs = []
    for size in (0, 256 * 1024, (256 << 10) + 40000, full):
        o = torch.full((1, 8, 1, 128), 9.0, dtype=torch.float16,
                       device="cuda")
        ws = torch.zeros(max(size, 1), dtype=torch.uint8, device="cuda")
        a = pkg.AttentionArgs(q=q.data_ptr(), k=k.data_ptr(),
                              v=v.data_ptr(), o=o.data_ptr(), batch=1,
                              heads=8, kv_heads=2, seq_q=1, seq_kv=4000,
                              head_dim=128, head_dim_v=128,
                              scale=128 ** -0.5)
        for f, t in (("q", q), ("k", k), ("v", v), ("o", o)):
            getattr(a.strides, f)[:] = list(t.stride()[:3])
        assert lib.iree_mi355x_attention_with_workspace(
            ctypes.byref(a), ws.data_ptr() if size else None, size,
            st) == pkg.OK
        outs.append(o.float())
        torch.cuda.synchronize()
        assert int(ws[:256 * 1024].sum()) == 0
    for o in outs[1:]:
        err = (o - outs[0]).abs().max() / outs[0].abs().max()
        assert float(err) <= 2e-3


def test_rows_misaligned_fused_layout_stays_refused(pkg, dev):
    """Head dims 64 and 128 without a mask demand 16-byte rows, also where
    the row-packed kernel would take the call."""
    q = torch.randn(1, 8, 1, 128, device=dev).half()
    buf = torch.randn(1, 2, 4000, 129, device=dev).half()
    k = buf[..., 1:]
    with pytest.raises(pkg.MI355XError) as e:
        pkg.attention(q, k, k, causal=False)
    assert e.value.status == pkg.MISALIGNED
    # a head dim of 40 has no such demand
    q, k = q[..., :40], buf[..., 1:41]
    o = pkg.attention(q, k, k, causal=False)
    ref = torch.nn.functional.scaled_dot_product_attention(
        q.cpu().float(), k.cpu().float().repeat_interleave(4, 1),
        k.cpu().float().repeat_interleave(4, 1))
    assert float((o.cpu().float() - ref).abs().max() / ref.abs().max()) < 2e-3


def test_rows_under_capture(pkg, dev):
    """Captured on a stream with no workspace: runs unsplit; replays agree."""
    g = torch.Generator().manual_seed(5)
    q, k = rand(g, 2, 8, 1, 64).cuda(), rand(g, 2, 2, 3000, 64).cuda()
    v = rand(g, 2, 2, 3000, 64).cuda()
    want = pkg.attention(q, k, v, causal=False).float()
    o = torch.zeros(2, 8, 1, 64, dtype=torch.float16, device=dev)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        pkg.attention(q, k, v, o, causal=False)
    for _ in range(3):
        o.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert float((o.float() - want).abs().max() / want.abs().max()) < 2e-3
