"""The general matmul (csrc/gemm_ragged.hip): any extents, strides, alignment
and layout, f16 with f16 / f32 results, int8 and W8A16, with and without a K
split.

Bars: int8 results are exact; f16 and W8A16 ones max|y - y_cpu| / max|y_cpu|
<= 2e-3 (the fp16 parity bound) against the oracle, f32 ones 1e-5 (f32 sums of
at most 777 products). Operands are views into NaN-filled (int8: random)
buffers, outputs views into filled ones: nothing outside a view is used or
written.
"""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

BOUND = {"f16": 2e-3, "f32": 1e-5, "w8a16": 2e-3}

# edges of the 64x64 tile, of a 16-byte load and of a K stage (64 f16, 128
# int8), and the smallest of everything
SHAPES = [(1, 1, 1), (2, 3, 5), (7, 17, 9), (16, 8, 15), (63, 65, 64),
          (64, 64, 128), (65, 63, 129), (127, 129, 63), (128, 128, 200),
          (129, 127, 257), (5, 1030, 777), (300, 72, 130)]


def view_in(rows, cols, t, fill, pad, lead):
    """`t` as a [rows, cols] view whose rows are `pad` elements further apart
    than their length and which starts `lead` elements into its buffer."""
    buf = torch.full((lead + rows * (cols + pad),), fill, dtype=t.dtype)
    if t.dtype == torch.int8:
        buf = torch.randint(-128, 128, buf.shape, dtype=torch.int8)
    v = torch.as_strided(buf, (rows, cols), (cols + pad, 1), lead)
    v.copy_(t)
    d = buf.cuda()
    return torch.as_strided(d, (rows, cols), (cols + pad, 1), lead)


def operands(kind, at, bt, m, n, k, pad, lead):
    g = torch.Generator().manual_seed(m * 7919 + n * 31 + k)

    def f16(r, c):
        return torch.randn(r, c, generator=g).half()

    def i8(r, c):
        return torch.randint(-128, 128, (r, c), generator=g).to(torch.int8)

    a = (i8 if kind == "i8" else f16)(*((k, m) if at else (m, k)))
    b = (i8 if kind in ("i8", "w8a16") else f16)(*((n, k) if bt else (k, n)))
    nan = float("nan")
    da = view_in(*a.shape, a, 0 if kind == "i8" else nan, pad, lead)
    db = view_in(*b.shape, b, 0 if b.dtype == torch.int8 else nan, pad, lead)
    return a, b, da, db


def run(pkg, kind, at, bt, da, db, scale, m, n, c):
    if kind == "w8a16":
        pkg.quantized_matmul(da, db, scale, c, w_transposed=bt)
    else:
        pkg.matmul(da, db, c, a_transposed=at, b_transposed=bt,
                   out_dtype=c.dtype)


def output(kind, m, n):
    dt = {"i8": torch.int32, "f32": torch.float32}.get(kind, torch.float16)
    buf = torch.full((m + 2, n + 5), 77, dtype=dt, device="cuda")
    return buf, buf[1:m + 1, :n]


def check(oracle, kind, at, bt, a, b, scale, buf, m, n):
    full = buf.cpu()
    c = full[1:m + 1, :n].numpy().copy()
    full[1:m + 1, :n] = 77
    assert bool((full == 77).all()), "write outside the output view"
    an, bn = a.numpy(), b.numpy()
    if kind == "i8":
        assert np.array_equal(c, oracle.matmul_i8(an, bn, b_transposed=bt))
        return
    if kind == "w8a16":
        ref = oracle.w8a16(an, np.ascontiguousarray(bn.T) if bt else bn,
                           scale.numpy())
    else:
        ref = oracle.matmul_f16(np.ascontiguousarray(an.T) if at else an, bn,
                                b_transposed=bt, out_f32=kind == "f32")
    assert np.isfinite(c).all()
    assert oracle.fp16_parity(c, ref) <= BOUND[kind]


FORMS = [(kind, at, bt) for kind in ("f16", "f32", "i8", "w8a16")
         for at in (False, True) for bt in (False, True)
         if not (at and kind in ("i8", "w8a16"))]


@pytest.mark.parametrize("kind,at,bt", FORMS)
def test_general_edges(pkg, oracle, dev, kind, at, bt):
    for i, (m, n, k) in enumerate(SHAPES):
        pad, lead = ((0, 0), (1, 1), (5, 3), (8, 8))[i % 4]
        print(f"{kind} at={at} bt={bt} {m}x{n}x{k} pad={pad}", flush=True)
        a, b, da, db = operands(kind, at, bt, m, n, k, pad, lead)
        scale = (torch.rand(n) * 0.019 + 0.001).half()
        buf, c = output(kind, m, n)
        run(pkg, kind, at, bt, da, db, scale.cuda(), m, n, c)
        check(oracle, kind, at, bt, a, b, scale, buf, m, n)


# (tile, M, N, K, split): edges of the larger tiles, whose K loop, fragment
# counts, swizzles and split sums are their own: one row or column past a tile
# and one short of it, K tails of one and two elements, one stage and many
WIDE = [("64x128", 641, 4737, 65, False), ("64x128", 1281, 2305, 130, False),
        ("128x128", 1025, 4735, 65, False), ("128x128", 1153, 3329, 130, False),
        ("64x128", 129, 4097, 2689, True), ("64x128", 257, 3329, 1700, True),
        ("64x128", 131, 4405, 4867, True),
        ("128x128", 385, 4737, 4099, True), ("128x128", 1281, 1601, 4099, True)]
TYPES = {"f16": (0, 0, 0), "f32": (0, 0, 3), "i8": (1, 1, 2),
         "w8a16": (0, 1, 0)}


def wide_plan(pkg, kind, at, bt, m, n, k, workspace=None):
    return pkg.plan(pkg.make_desc(
        *TYPES[kind], m, n, k,
        (pkg.B_TRANSPOSED if bt else 0) | (pkg.A_TRANSPOSED if at else 0),
        has_scale=kind == "w8a16", aligned=False), workspace)


def in_64_bits(kind, at, bt, da, db, scale):
    """The product in float64 (exact for int8)."""
    a = (da.t() if at else da).double().contiguous()
    b = (db.t() if bt else db).double().contiguous()
    c = torch.mm(a, b)
    return c * scale.double() if kind == "w8a16" else c


@pytest.mark.parametrize("kind,at,bt", FORMS)
def test_general_wide_tiles(pkg, dev, kind, at, bt):
    ran = set()
    for i, (tile, m, n, k, split) in enumerate(WIDE):
        p = wide_plan(pkg, kind, at, bt, m, n, k)
        if (not p.config_name.endswith(b"_" + tile.encode())
                or (p.splits > 1) != split):
            continue
        ran.add((tile, split))
        pad, lead = ((1, 1), (5, 3), (8, 8))[i % 3]
        print(f"{kind} at={at} bt={bt} {m}x{n}x{k} "
              f"{p.config_name.decode()} x{p.splits}", flush=True)
        _, _, da, db = operands(kind, at, bt, m, n, k, pad, lead)
        scale = (torch.rand(n) * 0.019 + 0.001).half().cuda()
        ref = in_64_bits(kind, at, bt, da, db, scale)
        for _ in range(2 if split else 1):  # the counters are re-armed
            buf, c = output(kind, m, n)
            run(pkg, kind, at, bt, da, db, scale, m, n, c)
            got = c.double()
            c.fill_(77)
            assert bool((buf == 77).all()), "write outside the output view"
            if kind == "i8":
                assert torch.equal(got, ref)
            else:
                # f32 sums of up to 4099 products: 2e-5
                err = float((got - ref).abs().max() / ref.abs().max())
                assert err <= (2e-5 if kind == "f32" else BOUND[kind]), err
    assert ran == {(t, s) for t in ("64x128", "128x128")
                   for s in (False, True)}


@pytest.mark.parametrize("m,n,k,tile", [(641, 4737, 65, "64x128"),
                                        (1153, 3329, 130, "128x128"),
                                        (129, 4097, 2689, "64x128"),
                                        (385, 4737, 4099, "128x128")])
@pytest.mark.parametrize("bt", [False, True])
def test_general_wide_tiles_epilogue(pkg, dev, m, n, k, tile, bt):
    """C += gate * gelu(x W + bias) from the larger tiles, whole and split, at
    odd pitches."""
    p = wide_plan(pkg, "f16", False, bt, m, n, k)
    assert p.config_name.endswith(b"_" + tile.encode())
    g = torch.Generator(device=dev).manual_seed(m)

    def rand(*shape):
        return torch.randn(*shape, generator=g, device=dev).half()

    x, w = rand(m, k), (rand(*((n, k) if bt else (k, n))) / k ** 0.5)
    bias, mul, init = rand(n), rand(m, n + 3)[:, :n], rand(m + 2, n + 5)
    buf = init.clone()
    c = buf[1:m + 1, :n]
    pkg.batch_matmul(x[None], w[None], c[None], bias=bias,
                     activation="gelu_tanh", multiplier=mul[None],
                     accumulate=True, b_transposed=bt)
    v = torch.mm(x.double(), (w.t() if bt else w).double().contiguous())
    v = torch.nn.functional.gelu(v + bias.double(), approximate="tanh")
    ref = init[1:m + 1, :n].double() + mul.double() * v
    assert float((c.double() - ref).abs().max() / ref.abs().max()) <= 2e-3
    buf[1:m + 1, :n] = init[1:m + 1, :n]
    assert torch.equal(buf, init), "write outside the output view"


def test_general_without_the_first_pick_s_workspace(pkg, dev):
    """An aligned shape whose plan does not split runs with no workspace,
    where the split tiles that are ranked first would need one."""
    m, n, k = 300, 11008, 4096
    g = torch.Generator(device=dev).manual_seed(2)
    a = torch.randn(m, k, generator=g, device=dev).half()
    b = torch.randn(n, k, generator=g, device=dev).half()
    c = torch.empty(m, n, dtype=torch.float16, device=dev)
    p = pkg.plan(pkg.make_desc(0, 0, 0, m, n, k, pkg.B_TRANSPOSED))
    assert p.family == pkg.FAMILY_GENERAL and p.workspace_bytes == 0
    assert pkg.library().iree_mi355x_matmul_f16(
        a.data_ptr(), b.data_ptr(), c.data_ptr(), m, n, k, k, k, n,
        pkg.B_TRANSPOSED, None, 0,
        torch.cuda.current_stream().cuda_stream) == pkg.OK, pkg.last_error()
    ref = torch.mm(a.double(), b.double().t().contiguous())
    assert float((c.double() - ref).abs().max() / ref.abs().max()) <= 2e-3


@pytest.mark.parametrize("kind,at,bt", FORMS)
def test_general_wide_pitch(pkg, oracle, dev, kind, at, bt):
    """Rows 8 MiB apart: the lane offsets of a tile pass 32 bits."""
    m, n, k = 5, 20, 24
    a, b, _, _ = operands(kind, at, bt, m, n, k, 0, 0)
    pitch = 8 << 20

    def wide(t):
        buf = torch.zeros((t.shape[0] - 1) * pitch + t.shape[1],
                          dtype=t.dtype, device="cuda")
        v = torch.as_strided(buf, tuple(t.shape), (pitch, 1))
        v.copy_(t)
        return v

    scale = (torch.rand(n) * 0.019 + 0.001).half()
    buf, c = output(kind, m, n)
    run(pkg, kind, at, bt, wide(a), wide(b), scale.cuda(), m, n, c)
    check(oracle, kind, at, bt, a, b, scale, buf, m, n)


@pytest.mark.parametrize("kind,bt", [("f16", False), ("f32", True),
                                     ("i8", True), ("w8a16", True)])
def test_general_split_and_no_workspace(pkg, oracle, dev, kind, bt):
    """A shape whose plan splits K, twice on one workspace (the counters are
    re-armed), and without a workspace, where it runs unsplit."""
    m, n, k = 65, 200, 4100
    a, b, da, db = operands(kind, False, bt, m, n, k, 1, 1)
    scale = (torch.rand(n) * 0.019 + 0.001).half()
    ds = scale.cuda()
    types = {"f16": (0, 0, 0), "f32": (0, 0, 3), "i8": (1, 1, 2),
             "w8a16": (0, 1, 0)}[kind]
    p = pkg.plan(pkg.make_desc(*types, m, n, k, 1 if bt else 0,
                               has_scale=kind == "w8a16", aligned=False))
    assert p.family == pkg.FAMILY_GENERAL and p.splits > 1
    for _ in range(2):
        buf, c = output(kind, m, n)
        run(pkg, kind, False, bt, da, db, ds, m, n, c)
        if kind == "f32":  # 4100 products: 2e-5
            ref = oracle.matmul_f16(a.numpy(), b.numpy(), b_transposed=bt,
                                    out_f32=True)
            assert oracle.fp16_parity(c.cpu().numpy(), ref) <= 2e-5
        else:
            check(oracle, kind, False, bt, a, b, scale, buf, m, n)
    split = c.clone()
    c.fill_(77)
    lib, st = pkg.library(), torch.cuda.current_stream().cuda_stream
    flags = (1 if bt else 0) | (pkg.OUT_F32 if kind == "f32" else 0)
    if kind == "w8a16":
        rc = lib.iree_mi355x_w8a16_matmul(
            da.data_ptr(), db.data_ptr(), ds.data_ptr(), c.data_ptr(), m, n,
            k, da.stride(0), db.stride(0), c.stride(0), flags, None, 0, st)
    else:
        fn = (lib.iree_mi355x_matmul_i8 if kind == "i8"
              else lib.iree_mi355x_matmul_f16)
        rc = fn(da.data_ptr(), db.data_ptr(), c.data_ptr(), m, n, k,
                da.stride(0), db.stride(0), c.stride(0), flags, None, 0, st)
    assert rc == pkg.OK, pkg.last_error()
    if kind == "i8":
        assert torch.equal(c, split)
    else:
        err = (c.double() - split.double()).abs().max() / split.abs().max()
        assert float(err) <= (2e-5 if kind == "f32" else 2e-3)


@pytest.mark.parametrize("act", ["none", "relu", "gelu_tanh", "silu"])
@pytest.mark.parametrize("shape", [(3, 65, 67, 70), (2, 130, 129, 1030)])
def test_general_batched_epilogue(pkg, oracle, dev, act, shape):
    z, m, n, k = shape
    g = torch.Generator().manual_seed(m + n)
    x = torch.randn(z, m, k, generator=g).half()
    w = (torch.randn(z, k, n, generator=g) / k ** 0.5).half()
    bias = torch.randn(n, generator=g).half()
    mul = torch.randn(z, m, n, generator=g).half()
    init = torch.randn(z, m, n, generator=g).half()
    c = init.cuda()
    pkg.batch_matmul(x.cuda(), w.cuda(), c, bias=bias.cuda(), activation=act,
                     multiplier=mul.cuda(), accumulate=True)
    v = torch.matmul(x.double(), w.double()) + bias.double()
    v = {"none": lambda t: t, "relu": torch.relu,
         "gelu_tanh": lambda t: torch.nn.functional.gelu(
             t, approximate="tanh"),
         "silu": torch.nn.functional.silu}[act](v)
    ref = init.double() + mul.double() * v
    err = (c.cpu().double() - ref).abs().max() / ref.abs().max()
    assert float(err) <= 2e-3


def test_general_zero_k(pkg, dev):
    """K = 0 writes the epilogue of an empty sum, and C_init if it adds."""
    a = torch.empty(70, 0, dtype=torch.float16, device=dev)
    b = torch.empty(0, 33, dtype=torch.float16, device=dev)
    assert bool((pkg.matmul(a, b) == 0).all())
    c = torch.full((70, 33), 3.0, dtype=torch.float16, device=dev)
    pkg.matmul(a, b, c, accumulate=True)
    assert bool((c == 3).all())


def test_general_under_capture(pkg, oracle, dev):
    """A split shape captured on a stream that has no workspace runs unsplit,
    as it did before it could split; replays agree with the eager result."""
    m, n, k = 33, 130, 2050
    a, b, da, db = operands("f16", False, False, m, n, k, 1, 1)
    eager = pkg.matmul(da, db)
    s = torch.cuda.Stream()
    c = torch.zeros(m, n, dtype=torch.float16, device=dev)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        pkg.matmul(da, db, c)
    for _ in range(3):
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        ref = oracle.matmul_f16(a.numpy(), b.numpy())
        assert oracle.fp16_parity(c.cpu().numpy(), ref) <= 2e-3
    assert oracle.fp16_parity(eager.cpu().numpy(), ref) <= 2e-3


@pytest.mark.parametrize("op", ["matmul", "attention"])
def test_captured_calls_leave_the_stream_workspace_alone(pkg, dev, op):
    """Captured on a stream whose workspace a warm-up call has filled: the
    graph runs without it, so it may replay beside other work. Its counters
    are spoilt before the replays, which a call that counts on them would
    not survive."""
    g = torch.Generator().manual_seed(6)
    if op == "matmul":
        a, b = (torch.randn(*s, generator=g).half().to(dev)
                for s in ((33, 2050), (2050, 130)))
        c = torch.zeros(33, 130, dtype=torch.float16, device=dev)

        def call():
            pkg.matmul(a, b, c)
    else:
        q, k, v = (torch.randn(*s, generator=g).half().to(dev)
                   for s in ((2, 8, 1, 64), (2, 2, 3000, 64), (2, 2, 3000, 64)))
        c = torch.zeros(2, 8, 1, 64, dtype=torch.float16, device=dev)

        def call():
            pkg.attention(q, k, v, c, causal=False)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        call()
    torch.cuda.synchronize()
    want = c.float()
    ws, size = pkg._FLAT_WORKSPACES[dev.index or 0, s.cuda_stream]
    buf = pkg._STREAM_WORKSPACES[dev.index or 0, s.cuda_stream, None][-1]
    assert buf.data_ptr() == ws and size == buf.numel()
    assert int(buf[256 << 10:].count_nonzero()) > 0  # the warm-up split
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=s):
        call()
    buf[:256 << 10].fill_(1)
    for _ in range(3):
        c.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert float((c.float() - want).abs().max() / want.abs().max()) < 2e-3
    assert bool((buf[:256 << 10] == 1).all())
    buf[:256 << 10].zero_()
    torch.cuda.synchronize()
