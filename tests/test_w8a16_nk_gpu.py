"""W8A16 with weights stored [N,K] on the macro-tiles (csrc/gemm.hip, kBW8T):
every tile the planner picks, at one K stage, a stage count below and above
the LDS ring's depth, whole and ragged last row tiles, padded rows and a K
split.

Bar: max|y - y_ref| / max|y_ref| <= 2e-3 (the fp16 parity bound) against the
product in float64; results are f32 sums rounded once to f16, 5e-4 of their own
size at most.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


CASES = [
    ("w8a16_tn_256x256x64_w2x4_s3", 2048, 7168, 64),
    ("w8a16_tn_256x256x64_w2x4_s3", 1024, 11008, 320),
    ("w8a16_tn_128x256x64_w2x4_s4", 2048, 4096, 64),
    ("w8a16_tn_128x256x64_w2x4_s4", 1024, 7168, 192),
    ("w8a16_tn_128x256x64_w2x4_s4", 512, 11008, 4096),
    ("w8a16_tn_128x256x64_w2x4_s4_sk", 513, 8192, 1024),
    ("w8a16_tn_128x256x64_w2x4_s4_sk", 600, 7168, 448),
    ("w8a16_tn_128x256x64_w2x4_s4_sk", 600, 4096, 11008),  # 3 splits
    ("w8a16_tn_128x128x64_w2x2_s3_sk", 512, 8192, 1024),
    ("w8a16_tn_128x128x64_w2x2_s3_sk", 513, 4096, 2048),
    ("w8a16_tn_64x128x64_w2x2_s4_sk", 129, 7168, 1536),
]


def planned(pkg, m, n, k):
    return pkg.plan(pkg.make_desc(0, 1, 0, m, n, k, pkg.B_TRANSPOSED,
                                  has_scale=True))


def operands(m, n, k, pad):
    """x, w and scale; rows of x and w `pad` bytes apart beyond their length,
    the gap NaN (w: random)."""
    g = torch.Generator().manual_seed(m * 7919 + n * 31 + k)
    x = torch.full((m, k + pad // 2), float("nan"), dtype=torch.float16)
    x[:, :k] = torch.randn(m, k, generator=g).half()
    w = torch.randint(-128, 128, (n, k + pad), generator=g).to(torch.int8)
    scale = (torch.rand(n, generator=g) * 0.019 + 0.001).half()
    return x.cuda()[:, :k], w.cuda()[:, :k], scale.cuda()


def check(c, buf, x, w, scale):
    m, n = c.shape
    ref = torch.mm(x.double(), w.double().t().contiguous()) * scale.double()
    err = (c.double() - ref).abs().max() / ref.abs().max()
    assert float(err) <= 2e-3
    full = buf.clone()
    full[1:m + 1, :n] = 77
    assert bool((full == 77).all()), "write outside the output view"


@pytest.mark.parametrize("ldc_pad", [0, 8, 5])
@pytest.mark.parametrize("config,m,n,k", CASES)
def test_tiles(pkg, dev, config, m, n, k, ldc_pad):
    p = planned(pkg, m, n, k)
    assert p.config_name.decode() == config
    print(config, m, n, k, ldc_pad, flush=True)
    x, w, scale = operands(m, n, k, 16 * (ldc_pad != 0))
    buf = torch.full((m + 2, n + ldc_pad), 77, dtype=torch.float16,
                     device=dev)
    c = buf[1:m + 1, :n]
    for _ in range(2):  # a split's counters are re-armed
        c.fill_(77)
        pkg.quantized_matmul(x, w, scale, c, w_transposed=True)
        check(c, buf, x, w, scale)


def run_without_workspace(pkg, x, w, scale, c):
    (m, k), n = x.shape, w.shape[0]
    rc = pkg.library().iree_mi355x_w8a16_matmul(
        x.data_ptr(), w.data_ptr(), scale.data_ptr(), c.data_ptr(), m, n, k,
        x.stride(0), w.stride(0), c.stride(0), pkg.B_TRANSPOSED, None, 0,
        torch.cuda.current_stream().cuda_stream)
    assert rc == pkg.OK, pkg.last_error()


@pytest.mark.parametrize("m,n,k,with_ws,without", [
    (600, 4096, 11008, "w8a16_tn_128x256x64_w2x4_s4_sk",
     "w8a16_tn_128x128x64_w2x2_s3_sk"),
    (5, 4096, 4096, "general_w8a16_tn", "gemv_rowdot_w8a16_r5"),
    (7, 1000, 1008, "general_w8a16_tn", "gemv_rowdot_w8a16_r7"),
    (16, 4096, 4096, "general_w8a16_tn", "gemv_rowdot_w8a16_r16"),
    (3, 300, 11008, "general_w8a16_tn", "gemv_rowdot_w8a16_r3"),
    (8, 128, 128, "general_w8a16_tn", "general_w8a16_tn"),
])
def test_with_and_without_workspace(pkg, dev, m, n, k, with_ws, without):
    print(m, n, k, flush=True)
    desc = pkg.make_desc(0, 1, 0, m, n, k, pkg.B_TRANSPOSED, has_scale=True)
    assert pkg.plan(desc).config_name.decode() == with_ws
    assert pkg.plan(desc, 0).config_name.decode() == without
    x, w, scale = operands(m, n, k, 16)
    for run in (lambda c: pkg.quantized_matmul(x, w, scale, c,
                                               w_transposed=True),
                lambda c: run_without_workspace(pkg, x, w, scale, c)):
        buf = torch.full((m + 2, n + 8), 77, dtype=torch.float16, device=dev)
        c = buf[1:m + 1, :n]
        for _ in range(2):
            c.fill_(77)
            run(c)
            check(c, buf, x, w, scale)
