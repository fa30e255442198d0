"""The stock path in fp32 (dfq_qmm_fallback for promoted dtypes, fp32 arrays, 2-bit codes and
groups the one-dtype kernels do not take), at the edges of its tiles and steps, against fp64."""
import numpy as np
import pytest

from gpu_util import announce, download
from oracle.qmm_oracle import pack

pytestmark = pytest.mark.gpu

# (M, N, K, bits, gs, x dtype, scale dtype): one row tile and its remainders, ragged N, K below, at
# and past a whole round of 16 waves for either step, odd 32s of K; then grids of more than 256
# workgroups, which take two and four row tiles, and outputs few enough for the per-element kernel;
# last, one dtype over a long K, which the product and the GEMV leave to this kernel
CASES = [
    (1, 1, 32, 4, 32, "f32", "bf16"), (16, 17, 512, 4, 64, "f32", "bf16"),
    (17, 40, 544, 2, 32, "f32", "f16"), (32, 16, 2048, 8, 128, "bf16", "f16"),
    (33, 31, 2080, 4, 32, "f16", "bf16"), (64, 65, 4128, 2, 96, "bf16", "f32"),
    (65, 33, 1984, 8, 64, "f32", "f32"), (6, 4096, 4096, 4, 64, "f32", "bf16"),
    (5, 70, 6144, 8, 512, "f32", "bf16"), (3, 50, 96, 8, 96, "f32", "f16"),
    (130, 20, 4096, 4, 128, "f16", "f32"), (7, 90, 640, 2, 64, "bf16", "bf16"),
    (5, 40, 1056, 4, 32, "f32", "bf16"),
    (32, 2070, 544, 4, 32, "f32", "bf16"), (31, 2080, 2080, 8, 32, "bf16", "f16"),
    (65, 1400, 160, 2, 32, "f32", "f16"), (129, 1391, 2080, 4, 32, "f16", "bf16"),
    (3, 33, 1024, 2, 64, "bf16", "bf16"), (4, 60, 768, 8, 64, "f32", "f16"),
    (8, 256, 1536, 4, 32, "f16", "f32"),
    (9, 40, 8192, 8, 128, "bf16", "bf16"), (16, 33, 8224, 4, 32, "f16", "f16"),
    (32, 17, 17408, 4, 64, "bf16", "bf16"), (1, 40, 40960, 4, 64, "bf16", "bf16"),
    (4, 21, 24576, 8, 128, "f16", "f16"),
]


@pytest.mark.parametrize("case", CASES)
def test_matches_fp64(ctx, case):
    """|y - y64| <= (K / 16 + 24) 2^-24 sum |x| (|s| q + |b|): the longest chain of roundings an
    output meets (a wave's quarter of its products, their tree, the weight's own), + the output's
    rounding where it is 16-bit."""
    import torch
    M, N, K, bits, gs, xdt, sdt = case
    DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
    rng = np.random.default_rng(M + N + K)
    codes = rng.integers(0, 1 << bits, size=(N, K), dtype=np.uint8)
    t = lambda a, d: torch.from_numpy(a.astype(np.float32)).to(DT[d]).cuda()
    x = t(rng.normal(size=(M, K)), xdt)
    s = t(np.abs(rng.normal(size=(N, K // gs))) * 0.02, sdt)
    b = t(rng.normal(size=(N, K // gs)) * 0.05, sdt)
    lb = t(rng.normal(size=N), sdt)
    w = torch.from_numpy(pack(codes, bits).view(np.int32)).cuda()
    announce(f"stock fp32 {case}")
    y = ctx.fallback(x, w, s, b, bits, gs, lbias=lb)
    assert y.dtype == (DT[xdt] if xdt == sdt else torch.float32)
    rep = lambda a: np.repeat(a.double().cpu().numpy(), gs, axis=1)
    xd, ld = x.double().cpu().numpy(), lb.double().cpu().numpy()
    ref = xd @ (codes * rep(s) + rep(b)).T + ld
    S = np.abs(xd) @ (codes * rep(s) + np.abs(rep(b))).T + np.abs(ld)
    bound = (K / 16 + 24) * 2.0 ** -24 * S
    if y.dtype != torch.float32:
        bound = bound + 2.0 ** -8 * np.abs(ref)
    assert (np.abs(download(y) - ref) <= bound).all()


def test_padding_lanes_add_nothing(ctx):
    """Infinities in one row and one column stay there: rows and columns past the edge repeat
    the last, and lanes past K add zeros."""
    import torch
    M, N, K = 5, 20, 96
    rng = np.random.default_rng(3)
    w = torch.from_numpy(pack(rng.integers(0, 16, size=(N, K), dtype=np.uint8), 4)
                         .view(np.int32)).cuda()
    x = torch.ones(M, K, device="cuda")
    s = torch.full((N, K // 32), 0.5, dtype=torch.bfloat16, device="cuda")
    b = torch.ones_like(s)
    announce("stock fp32 infinities")
    want = ctx.fallback(x, w, s, b, 4, 32)
    x[M - 1, K - 1] = float("inf")
    b[N - 1, 2] = float("inf")
    y = ctx.fallback(x, w, s, b, 4, 32)
    assert torch.equal(y[:-1, :-1], want[:-1, :-1])
    assert torch.isinf(y[-1]).all() and torch.isinf(y[:, -1]).all()


@pytest.mark.parametrize("M,N,K", [(65, 1400, 544), (32, 2080, 2080), (200, 16, 4128)])
def test_rows_do_not_depend_on_how_many_there_are(ctx, M, N, K):
    """One, two and four row tiles a workgroup add the same products in the same order."""
    import torch
    rng = np.random.default_rng(M)
    w = torch.from_numpy(pack(rng.integers(0, 16, size=(N, K), dtype=np.uint8), 4)
                         .view(np.int32)).cuda()
    x = torch.from_numpy(rng.normal(size=(M, K)).astype(np.float32)).cuda()
    s = torch.full((N, K // 32), 0.5, dtype=torch.bfloat16, device="cuda")
    b = torch.full_like(s, -3.75)
    announce(f"stock fp32 rows M={M} N={N} K={K}")
    y = ctx.fallback(x, w, s, b, 4, 32)
    few = ctx.fallback(x[:9].contiguous(), w, s, b, 4, 32)
    assert torch.equal(y[:9], few)
