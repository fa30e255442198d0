"""The stock path's many-row matrix product (dfq_qmm_fallback above 8 rows, one 16-bit dtype).

Pinned two ways, in every format and at the edges of every tile:

* bit-exact one-hot rows: with x[m] = e_k, power-of-two scales and small integer biases every
  term of the factored form is exact, so y must equal the oracle's dequant bit for bit;
* against the fp64 oracle, elementwise: the output's rounding plus the fp32 sums' bound.
"""
import numpy as np
import pytest

from gpu_util import announce, download, to_dev16, upload
from onehot import exact_case
from oracle.qmm_oracle import BF16, F16, make_case, pack, to_bits

pytestmark = pytest.mark.gpu

FORMATS = [(bits, gs, dt) for bits in (4, 8) for gs in (32, 64, 128) for dt in (BF16, F16)]
# (rows, columns) that take each tile of the dispatch on 256 CUs, with ragged edges: 32 x 64 in
# four K slices (twice), 32 x 128 and 64 x 128 in two, 64 x 128, 96 x 128, 128 x 128 (96 x 128 in
# groups of 32)
TILES = [(9, 37), (33, 130), (32, 17000), (64, 16397), (385, 9001), (65, 16397), (400, 14001)]


@pytest.mark.parametrize("bits,gs,dt", FORMATS)
def test_one_hot_rows_are_exact(ctx, bits, gs, dt):
    import torch
    K = 11 * gs if gs != 128 else 5 * gs   # a ragged line, step (group 32) and slice of K
    N = 77
    w, sb, bb, deq = exact_case(N, K, bits, gs, dt, seed=bits * 100 + gs + dt)
    wd = torch.from_numpy(w.view(np.int32)).cuda()
    sd, bd = to_dev16(sb, dt), to_dev16(bb, dt)
    x = torch.eye(K, dtype=torch.bfloat16 if dt == BF16 else torch.float16, device="cuda")
    announce(f"stock gemm one-hot bits={bits} gs={gs} dt={dt} K={K}")
    y = ctx.fallback(x, wd, sd, bd, bits, gs)
    torch.cuda.synchronize()
    got = y.view(torch.int16).cpu().numpy().view(np.uint16)
    assert np.array_equal(got, to_bits(deq.T, dt))


@pytest.mark.parametrize("bits,gs,dt", FORMATS)
@pytest.mark.parametrize("M,N", TILES)
def test_matches_oracle(ctx, oracle, M, N, bits, gs, dt):
    """|y - y64| <= u_out |y64| + (K + 8) 2^-24 S, S = sum |x| (|s| (MAGIC + q_max) + |b|): one
    output rounding and at most K + 8 roundings of sums no larger than S (MAGIC 16 at bf16
    4-bit, 0 otherwise), + one unit of the smallest fp16."""
    K = {32: 352, 64: 704, 128: 640}[gs] if N < 6000 else 3 * gs
    c = make_case(M, N, K, bits=bits, gs=gs, xdt=dt, seed=M + N + bits, lbias=(M % 2 == 1))
    x, w, s, b, lb = upload(c)
    announce(f"stock gemm M={M} N={N} K={K} bits={bits} gs={gs} dt={dt}")
    y = download(ctx.fallback(x, w, s, b, bits, gs, lbias=lb))
    ref = oracle.qmm_f64(c)
    top = (1 << bits) - 1 + (16 if bits == 4 and dt == BF16 else 0)
    wmax = np.repeat(np.abs(download(s)) * top + np.abs(download(b)), gs, axis=1)
    S = np.abs(download(x)) @ wmax.T + (0 if lb is None else np.abs(download(lb)))
    u = 2.0 ** -8 if dt == BF16 else 2.0 ** -11  # half a unit of 8 and 11 significant bits
    bound = u * np.abs(ref) + (K + 8) * 2.0 ** -24 * S + 2.0 ** -24
    bad = np.argwhere(~(np.abs(y - ref) <= bound))
    assert bad.size == 0, (len(bad), bad[0], y[tuple(bad[0])], ref[tuple(bad[0])])


def dequantised(w, s, b, bits, gs):
    """Rows of the weight in float64, on the GPU."""
    import torch
    per = 32 // bits
    q = torch.stack([(w >> (bits * t)) & ((1 << bits) - 1) for t in range(per)], 2)
    q = q.reshape(w.shape[0], -1, gs).double()
    return (q * s.double()[:, :, None] + b.double()[:, :, None]).reshape(w.shape[0], -1)


@pytest.mark.parametrize("bits,gs,dt", FORMATS)
@pytest.mark.parametrize("M,N", TILES)
@pytest.mark.parametrize("ragged", [False, True])
def test_every_tile_over_many_lines_and_slices(ctx, M, N, bits, gs, dt, ragged):
    """38 to 40 steps of 64 k: every slice of K has work, code and scale buffers and X sets are
    used again in each, with whole lines of scales (vector loads, groups of 32 and 64) and with a
    last line, set and step that are not whole.  Against float64 at the first and last columns and
    a sample, with the bound of test_matches_oracle; and a row's bits depend on that row alone,
    among calls of as many rows."""
    import torch
    K = {32: 2464, 64: 2496, 128: 2432}[gs] if ragged else 2560
    tdt = torch.bfloat16 if dt == BF16 else torch.float16
    g = torch.Generator(device="cuda").manual_seed(M + N + bits + gs + dt)
    w = torch.randint(-2**31, 2**31, (N, K * bits // 32), dtype=torch.int64, device="cuda",
                      generator=g).to(torch.int32)
    r = lambda *size: torch.randn(*size, device="cuda", generator=g)
    s, b = (r(N, K // gs) * 0.02).to(tdt), (r(N, K // gs) * 0.1).to(tdt)
    x, lb = r(M, K).to(tdt), r(N).to(tdt)
    announce(f"stock gemm tiles M={M} N={N} K={K} bits={bits} gs={gs} dt={dt}")
    y = ctx.fallback(x, w, s, b, bits, gs, lbias=lb).double()
    c = torch.cat([torch.arange(min(N, 40)), torch.randint(0, N, (200,)),
                   torch.arange(max(0, N - 140), N)]).cuda()
    ref = x.double() @ dequantised(w[c], s[c], b[c], bits, gs).t().contiguous() + lb[c].double()
    top = (1 << bits) - 1 + (16 if bits == 4 and dt == BF16 else 0)
    wmax = (s[c].double().abs() * top + b[c].double().abs()).repeat_interleave(gs, 1)
    S = x.double().abs() @ wmax.t().contiguous() + lb[c].double().abs()
    u = 2.0 ** -8 if dt == BF16 else 2.0 ** -11
    bound = u * ref.abs() + (K + 8) * 2.0 ** -24 * S + 2.0 ** -24
    bad = ((y[:, c] - ref).abs() > bound).nonzero().cpu()
    assert len(bad) == 0 and bool(torch.isfinite(y).all()), (len(bad), bad[:3])
    x[1:] = r(M - 1, K).to(tdt)
    assert torch.equal(ctx.fallback(x, w, s, b, bits, gs, lbias=lb)[0].double(), y[0])


@pytest.mark.parametrize("bits,gs,dt", FORMATS)
@pytest.mark.parametrize("M,N", TILES)
def test_one_hot_rows_are_exact_in_every_tile(ctx, M, N, bits, gs, dt):
    """M positions of K over all slices, lines and steps, 53 weight rows repeated over N."""
    import torch
    K = {32: 2464, 64: 2496, 128: 2432}[gs]
    w, sb, bb, deq = exact_case(53, K, bits, gs, dt, seed=bits * 10 + gs + dt)
    n = np.arange(N) % 53
    k = np.concatenate([[0, K - 1], np.linspace(1, K - 2, M - 2).astype(int)])
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a).view(np.int16)).cuda()
    tdt = torch.bfloat16 if dt == BF16 else torch.float16
    wd = torch.from_numpy(w.view(np.int32)).cuda()[torch.from_numpy(n).cuda()].contiguous()
    sd, bd = (dev(a)[torch.from_numpy(n).cuda()].contiguous().view(tdt) for a in (sb, bb))
    x = torch.zeros(M, K, dtype=tdt, device="cuda")
    x[torch.arange(M), torch.from_numpy(k)] = 1.0
    announce(f"stock gemm one-hot tiles M={M} N={N} bits={bits} gs={gs} dt={dt}")
    y = ctx.fallback(x, wd, sd, bd, bits, gs)
    want = dev(to_bits(deq[:, k].T, dt))[:, torch.from_numpy(n).cuda()]
    assert torch.equal(y.view(torch.int16), want)


def test_rows_past_the_gemvs_limit_in_k_and_misaligned_scales(ctx, oracle):
    """A long K, and scales that are not aligned for a line's vector load, which are read one by
    one: the same bits."""
    import torch
    c = make_case(40, 40, 32768, bits=4, gs=64, seed=5)
    x, w, s, b, _ = upload(c)
    assert ctx.stock_gemv_launches(3, 40, 32768, 4, 64) == 0
    announce("stock gemm long K")
    y = ctx.fallback(x, w, s, b, 4, 64)
    buf = torch.empty(2 * s.numel() + 1, dtype=s.dtype, device="cuda")
    s2 = buf[1:1 + s.numel()].view(s.shape).copy_(s)
    y2 = ctx.fallback(x, w, s2, b, 4, 64)
    torch.cuda.synchronize()
    ref = oracle.qmm_f64(c)
    assert np.abs(download(y) - ref).max() <= 2.0 ** -8 * np.abs(ref).max()
    assert torch.equal(y.view(torch.int16), y2.view(torch.int16))


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("one_sign", [False, True])
def test_four_bit_sums_are_no_further_off_than_the_gemvs(ctx, gs, dt, one_sign):
    """Sums that are exactly 0, so that the output's rounding does not hide theirs: every group of
    x meets codes q with bias -j s and codes 15 - q with bias -(15 - j) s, in shuffled order.  The
    outputs are the sums' own errors, and the matrix product's are no larger (root mean square)
    than the GEMV's on the same inputs, in a tile of four slices of K and in one of none."""
    import torch
    K, rng = 2560, np.random.default_rng(gs + dt)
    G, tdt = K // gs, torch.bfloat16 if dt == BF16 else torch.float16
    for M, N in ((16, 300), (400, 14001)):
        q = rng.integers(0, 16, size=(N, G // 2, gs), dtype=np.uint8)
        s = rng.integers(8, 16, size=(N, G // 2)) * 2.0 ** -13
        j = rng.integers(5, 11, size=(N, G // 2))  # (four bits by four: exact in either dtype)
        x = rng.normal(size=(M, G // 2, gs))
        perm = rng.permutation(G)
        twice = lambda a, b: np.concatenate([a, b], 1)[:, perm]
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float32)).to(tdt).cuda()
        w = pack(twice(q, 15 - q).reshape(N, K), 4)
        w = torch.from_numpy(w.view(np.int32)).cuda()
        sd, bd = t(twice(s, s)), t(twice(-s * j, -s * (15 - j)))
        xd = t(twice(np.abs(x) if one_sign else x, np.abs(x) if one_sign else x).reshape(M, K))
        announce(f"stock gemm precision gs={gs} dt={dt} one_sign={one_sign} M={M}")
        rms = lambda y: y.double().pow(2).mean().sqrt().item()
        got = rms(ctx.fallback(xd, w, sd, bd, 4, gs))
        gemv = rms(ctx.fallback(xd[:8].contiguous(), w, sd, bd, 4, gs))
        assert 0 < got <= gemv, (M, got / gemv)


@pytest.mark.parametrize("dt", [BF16, F16])
def test_an_infinite_activation_stays_in_its_row(ctx, dt):
    """8-bit codes and biases above zero: the row with the infinity is infinite, as the fp64
    product has it, and no other row changes."""
    import torch
    c = make_case(20, 40, 512, bits=8, gs=64, xdt=dt, seed=2)
    x, w, s, b, _ = upload(c)
    b, w = b.abs() + 0.5, w | 0x01010101  # (a code of 0 times infinity is NaN)
    announce(f"stock gemm infinity dt={dt}")
    want = ctx.fallback(x, w, s, b, 8, 64)
    x[7, 100] = float("inf")
    y = ctx.fallback(x, w, s, b, 8, 64)
    torch.cuda.synchronize()
    keep = [r for r in range(20) if r != 7]
    assert torch.equal(y[keep].view(torch.int16), want[keep].view(torch.int16))
    assert (y[7] == float("inf")).all()


def classes_case(M, N, K, bits, gs, dt, seed, positive=False):
    """MLX-style weights: s > 0 and b the group's minimum, below zero (above it and no code of 0
    if `positive`); returns tensors and the dequantised weight."""
    import torch
    rng = np.random.default_rng(seed)
    tdt = torch.bfloat16 if dt == BF16 else torch.float16
    top = (1 << bits) - 1
    codes = rng.integers(1 if positive else 0, top + 1, size=(N, K), dtype=np.uint8)
    t = lambda a: torch.from_numpy(a.astype(np.float32)).to(tdt).cuda()
    s = t(rng.uniform(0.5, 1.5, size=(N, K // gs)) / top)
    b = t(rng.uniform(0.3, 0.7, size=(N, K // gs)) * (1 if positive else -1))
    x = t(rng.normal(size=(M, K)))
    w = torch.from_numpy(pack(codes, bits).view(np.int32)).cuda()
    rep = lambda a: np.repeat(a.double().cpu().numpy(), gs, axis=1)
    return x, w, s, b, codes * rep(s) + rep(b)


@pytest.mark.parametrize("bits,gs,dt", FORMATS)
def test_an_infinite_activation_never_gives_the_wrong_sign(ctx, bits, gs, dt):
    """Biases below zero, as quantised weights have: s P and b X are infinities of either sign, so
    the factored form gives NaN where the weight's sign cannot be told, as the GEMV does, and
    never an infinity that the weight does not give."""
    import torch
    K = 11 * gs if gs != 128 else 5 * gs
    x, w, s, b, deq = classes_case(20, 70, K, bits, gs, dt, seed=bits + gs)
    announce(f"stock gemm infinity, negative biases bits={bits} gs={gs} dt={dt}")
    want = ctx.fallback(x, w, s, b, bits, gs)
    hit = {5: (3, 1.0), 7: (gs + 1, -1.0), 11: (K - 1, 1.0)}
    for m, (k, sign) in hit.items():
        x[m, k] = sign * float("inf")
    y = ctx.fallback(x, w, s, b, bits, gs)
    gemv = ctx.fallback(x[4:12].contiguous(), w, s, b, bits, gs)
    torch.cuda.synchronize()
    keep = [r for r in range(20) if r not in hit]
    assert torch.equal(y[keep].view(torch.int16), want[keep].view(torch.int16))
    for m, (k, sign) in hit.items():
        got, few = download(y[m:m + 1])[0], download(gemv[m - 4:m - 3])[0]
        right = np.sign(deq[:, k]) * sign * np.inf
        assert not np.isfinite(got).any()
        assert (np.isnan(got) | (got == right)).all()
        assert (np.isnan(few) | ~np.isnan(got)).all()  # no NaN where the GEMV has none


@pytest.mark.parametrize("bits,gs,dt", [f for f in FORMATS if f[0] == 8 or f[2] == F16])
@pytest.mark.parametrize("M,N", [(47, 40), (47, 17000), (400, 9001)])
def test_an_infinity_stays_one_in_every_group(ctx, M, N, bits, gs, dt):
    """Weights above zero, an infinity in each row at another place: every output is +inf, also
    where the last groups of a slice of K are fewer than an X product takes."""
    import torch
    K = 2944 if gs == 128 else 3008  # 46 or 47 steps of 64 k
    x, w, s, b, _ = classes_case(M, N, K, bits, gs, dt, seed=M + gs, positive=True)
    x[torch.arange(M), (torch.arange(M) * (64 if M < 64 else 8) + 5) % K] = float("inf")
    announce(f"stock gemm infinity by group M={M} N={N} bits={bits} gs={gs} dt={dt}")
    y = ctx.fallback(x, w, s, b, bits, gs)
    bad = (y != float("inf")).nonzero().cpu()
    assert len(bad) == 0, (len(bad), bad[0])


@pytest.mark.parametrize("bits,gs,dt", FORMATS)
def test_an_infinite_bias_gives_infinities(ctx, bits, gs, dt):
    """Positive activations whose group sums are short numbers (no low parts): the column of an
    infinite bias is infinite, as the GEMV has it, and no other column changes."""
    import torch
    K = 11 * gs if gs != 128 else 5 * gs
    x, w, s, b, _ = classes_case(20, 70, K, bits, gs, dt, seed=bits + gs)
    x.fill_(0.5)
    announce(f"stock gemm infinite bias bits={bits} gs={gs} dt={dt}")
    want = ctx.fallback(x, w, s, b, bits, gs)
    hit = {3: (0, 1.0), 40: (K // gs - 1, -1.0), 69: (2, 1.0)}
    for n, (g, sign) in hit.items():
        b[n, g] = sign * float("inf")
    y = ctx.fallback(x, w, s, b, bits, gs)
    gemv = ctx.fallback(x[:8].contiguous(), w, s, b, bits, gs)
    torch.cuda.synchronize()
    keep = [n for n in range(70) if n not in hit]
    assert torch.equal(y[:, keep].view(torch.int16), want[:, keep].view(torch.int16))
    for n, (_, sign) in hit.items():
        assert (gemv[:, n] == sign * float("inf")).all()
        assert (y[:, n] == sign * float("inf")).all(), n


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("M,N", [(1, 8), (3, 1000), (257, 24), (333, 4096)])
def test_silu_mul_by_pieces_equals_by_elements(ctx, M, N, dt):
    """Rows of whole 16-byte pieces go eight elements a thread; arrays two bytes off that
    alignment go one by one: the same values, bit for bit."""
    import torch
    tdt = torch.bfloat16 if dt == "bf16" else torch.float16
    buf = torch.randn(2 * M * N + 1, device="cuda", dtype=torch.float32).mul_(3).to(tdt)
    odd = buf[1:].view(M, 2 * N)
    announce(f"silu_mul pieces {dt} M={M} N={N}")
    h = ctx.silu_mul(odd.clone())
    h_odd = ctx.silu_mul(odd)
    torch.cuda.synchronize()
    assert torch.equal(h.view(torch.int16), h_odd.view(torch.int16))
