"""GPU parity of the batched projection qd_gemm_nt (the prefill GEMM) in both
modes, and of the engine's MFMA prefill mode.

Bars:
  * QD_GEMM_EXACT: every row bit-exact against the oracle's decode-order GEMV
    (and against its projection + residual), i.e. the same bits as the decode
    step computes token by token;
  * QD_GEMM_MFMA: fp16 x fp16 products are exact in fp32 and the matrix cores
    sum them in fp32 in their own order, so each output is within one fp16 ulp
    of the float64 sum plus the fp32 summation bound k * 2^-23 * sum|x w|
    (with a residual: plus one more fp16 rounding);
  * engine, MFMA prefill: the KV rows differ from exact prefill only by that
    summation order, so the next step's logits agree closely; decode steps
    themselves are unchanged.
"""
import numpy as np
import pytest
import torch

from common import model_kv_fp64, model_tensors, normal_f16, ulp16
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def qdiy():
    import qdiy as m
    torch.cuda.set_device(0)
    m.load()
    return m


def _same(a, b):
    return np.array_equal(np.asarray(a).view(np.uint16), np.asarray(b).view(np.uint16))


def _dev(a):
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (37, 100, 520), (127, 6144, 2048), (256, 2048, 5504),
                                   (45, 4104, 1544), (300, 4100, 2000)])
@pytest.mark.parametrize("with_res", [False, True])
def test_exact_mode_is_the_decode_gemv(qdiy, m, n, k, with_res):
    """Exact-mode rows against the oracle's decode GEMV, bit for bit: one token on the
    two-row kernel, the others on the fp32 matrix instructions.  (45, 4104, 1544) has a
    last chunk of K of one lane and a ragged last tile in both directions; (300, 4100,
    2000) more than 256 tokens; (256, 2048, 5504) the widest K of the 1.8B shape.  The
    rows checked straddle the 16- and 32-token tiles."""
    rng = np.random.default_rng(m * 1000 + n + k + with_res)
    x, W, R = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (m, n))
    y = torch.zeros(m * n, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k,
                 residual=_dev(R.reshape(-1)) if with_res else None, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    rows = sorted({i for i in (0, 1, 7, 8, 31, 32, 63, 64, m // 2, m - 2, m - 1) if 0 <= i < m})
    for i in rows:
        if with_res:
            want = oracle.proj_residual(x[i], W.reshape(-1), R[i], n, k)
        else:
            want = oracle.gemv(x[i], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)
        assert _same(got[i], want), f"row {i}"


@pytest.mark.parametrize("m,n,k", [
    # the two-row kernel's last token count and the matrix instructions' first
    (4, 33, 72), (5, 33, 72),
    # edges of the 16 x 16 and 32 x 32 output tiles in both directions
    (15, 16, 512), (16, 17, 520), (17, 31, 1032), (31, 33, 1000), (33, 32, 2056), (65, 65, 64),
    # K: one class, a group of classes partly filled, whole groups without a last
    # chunk, the widest (from one token on the matrix instructions)
    (9, 40, 8), (40, 40, 440), (70, 48, 1536), (3, 40, 8192), (100, 50, 7176),
    # 32 x 32 tiles: several rounds of a device's workgroups
    (520, 1100, 136)])
@pytest.mark.parametrize("with_res", [False, True])
def test_exact_mode_tile_edges(qdiy, m, n, k, with_res):
    """Every output of the exact mode where its tiles, its last chunk of K or its
    choice of kernel change, bit for bit; x and y rows padded, y at an odd element
    offset (no 8-byte stores) without a residual."""
    rng = np.random.default_rng(m * 77 + n + k + with_res)
    ldx, ldy, off = k + 8, n + (4 if with_res else 3), 0 if with_res else 1
    x, W = normal_f16(rng, (m, ldx)), normal_f16(rng, (n, k), 0.02)
    R = normal_f16(rng, (m, ldy))
    y = torch.full((off + m * ldy + 8,), 9.0, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y[off:], m, n, k, ldx=ldx, ldy=ldy,
                 residual=_dev(R.reshape(-1)) if with_res else None, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    out = y.cpu().numpy()
    got = out[off:off + m * ldy].reshape(m, ldy)
    assert np.all(got[:, n:] == np.float16(9.0)) and np.all(out[:off] == 9.0) and np.all(out[off + m * ldy:] == 9.0)
    for i in range(m):
        if with_res:
            want = oracle.proj_residual(x[i, :k], W.reshape(-1), R[i, :n], n, k)
        else:
            want = oracle.gemv(x[i, :k], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)
        assert _same(got[i, :n], want), f"row {i}"


def test_exact_mode_infinities_stay_in_their_row(qdiy):
    """An infinity in one token's or weight's row (next to the last chunk, whose elements
    past K belong to the following row) reaches that row's outputs only, with the
    oracle's infinities and NaNs."""
    m, n, k = 40, 48, 456
    rng = np.random.default_rng(5)
    x, W = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02)
    x[7, 0], x[20, k - 1], W[33, 0], W[11, 448] = np.inf, -np.inf, np.inf, np.nan
    y = torch.zeros(m * n, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    with np.errstate(invalid="ignore"):
        want = np.stack([oracle.gemv(x[i], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64) for i in range(m)])
    nan = np.isnan(want)
    assert np.array_equal(np.isnan(got), nan) and nan.any() and np.isinf(want).any()
    assert np.array_equal(got.view(np.uint16)[~nan], want.view(np.uint16)[~nan])


def test_exact_mode_far_apart_rows(qdiy):
    """Token rows 2^26 elements apart, beyond the matrix kernel's 32-bit lane offsets,
    take the two-row kernel: the same bits."""
    m, n, k, ldx = 6, 64, 264, 1 << 26
    rng = np.random.default_rng(6)
    x, W = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02)
    far = torch.empty((m - 1) * ldx + k, dtype=torch.float16, device="cuda")
    for i in range(m):
        far[i * ldx:i * ldx + k] = _dev(x[i])
    y = torch.zeros(m * n, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(far, _dev(W.reshape(-1)), y, m, n, k, ldx=ldx, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    for i in range(m):
        assert _same(got[i], oracle.gemv(x[i], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)), f"row {i}"


@pytest.mark.parametrize("k", [1544, 2048, 4104, 5504, 6152, 7168, 7176, 8192])
@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("with_res", [False, True])
def test_exact_mode_two_row_kernel(qdiy, m, k, with_res):
    """Up to 4 tokens, every output bit for bit: the two-row kernel with 4 to 16 chunks of K
    per lane, whole and ragged, with its next tile's loads in flight (up to 11 chunks) and
    without, eight and (from K = 7169) four waves per workgroup; odd and even tokens, an odd
    last row, padded x and y rows."""
    n, ldx, pad = 37, k + 8, 3
    rng = np.random.default_rng(17 * m + k + with_res)
    x, W, R = normal_f16(rng, (m, ldx)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (m, n + pad))
    y = torch.full((m * (n + pad) + 8,), 9.0, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k, ldx=ldx, ldy=n + pad,
                 residual=_dev(R.reshape(-1)) if with_res else None, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    out = y.cpu().numpy()
    got = out[:m * (n + pad)].reshape(m, n + pad)
    assert np.all(got[:, n:] == 9.0) and np.all(out[m * (n + pad):] == 9.0)
    for i in range(m):
        if with_res:
            want = oracle.proj_residual(x[i, :k], W.reshape(-1), R[i, :n], n, k)
        else:
            want = oracle.gemv(x[i, :k], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)
        assert _same(got[i, :n], want), f"row {i}"


@pytest.mark.parametrize("m,n,k", [
    # both sides of the two-row kernel's ranges: few weight rows, and more than 32 per CU
    # (8192 at 256)
    (5, 1, 264), (6, 128, 5632), (5, 128, 5640), (6, 129, 5632), (5, 77, 256), (7, 99, 1000),
    (6, 8192, 264), (5, 8193, 136), (6, 8211, 1024), (5, 8193, 1032), (6, 8200, 128),
    (8, 8193, 512), (7, 8203, 264), (8, 8193, 520), (7, 8193, 256), (9, 8193, 512)])
@pytest.mark.parametrize("with_res", [False, True])
def test_exact_mode_five_to_eight_tokens(qdiy, m, n, k, with_res):
    """5 to 9 tokens on either kernel: every output bit for bit, nothing past a row."""
    pad = 5
    rng = np.random.default_rng(31 * m + n + k + with_res)
    x, W, R = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (m, n + pad))
    y = torch.full((m, n + pad), 9.0, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y.view(-1), m, n, k, ldy=n + pad,
                 residual=_dev(R.reshape(-1)) if with_res else None, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    got = y.cpu().numpy()
    assert np.all(got[:, n:] == 9.0)
    for i in range(m):
        if with_res:
            want = oracle.proj_residual(x[i], W.reshape(-1), R[i, :n], n, k)
        else:
            want = oracle.gemv(x[i], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)
        assert _same(got[i, :n], want), f"row {i}"


@pytest.mark.parametrize("n", [2048, 2049])
def test_exact_mode_wide_rows_change_kernel(qdiy, n):
    """K > 7168: up to 2048 weight rows on the two-row kernel, more on the matrix
    instructions (256 compute units): the same bits."""
    m, k = 2, 7176
    rng = np.random.default_rng(n)
    x, W = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02)
    y = torch.zeros(m * n, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    for i in range(m):
        assert _same(got[i], oracle.gemv(x[i], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)), f"row {i}"


@pytest.mark.parametrize("m,k", [(41, 264), (34, 2048), (37, 6152), (35, 8192)])
def test_exact_mode_far_apart_rows_past_a_token_block(qdiy, m, k):
    """More than 32 token rows 2^26 elements apart: the two-row kernel's second block of
    tokens and its later tiles, with and without its prefetch."""
    n, ldx = 24, 1 << 26
    rng = np.random.default_rng(m + k)
    x, W = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02)
    far = torch.empty((m - 1) * ldx + k, dtype=torch.float16, device="cuda")
    for i in range(m):
        far[i * ldx:i * ldx + k] = _dev(x[i])
    y = torch.zeros(m * n, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(far, _dev(W.reshape(-1)), y, m, n, k, ldx=ldx, mode=qdiy.GEMM_EXACT)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, n)
    for i in range(m):
        assert _same(got[i], oracle.gemv(x[i], W.reshape(-1), n, k, 0, oracle.ORDER_WAVE64)), f"row {i}"


@pytest.mark.parametrize("m,n,k", [(1, 64, 64), (37, 100, 512), (127, 6144, 2048), (256, 2048, 5504),
                                   (200, 5504, 2048),
                                   # from 128 rows: the 64 x 64 tile where a 128 x 128 grid would
                                   # leave most CUs idle (ragged m and n, a partial group of four
                                   # outputs at n = 130), the 128 x 128 ring tile, and the 192 x 256
                                   # ring tile where its grid covers the CUs (ragged rows of W at
                                   # n = 6000, ragged tokens at m = 1800)
                                   (600, 130, 512), (1024, 2048, 5504), (512, 6144, 2048),
                                   (2048, 6144, 2048), (2048, 6000, 2048), (1800, 6144, 1024),
                                   # the 192 x 256 tile with 1, 2, 3 and 17 K tiles of 64 (its two
                                   # stages never fill, fill once, or end on an odd tile)
                                   (2048, 6144, 64), (2048, 6144, 128), (2048, 6000, 192),
                                   (1800, 6144, 1088)])
@pytest.mark.parametrize("with_res", [False, True])
def test_mfma_mode_within_fp32_summation_bound(qdiy, m, n, k, with_res):
    rng = np.random.default_rng(7 * m + n + k + with_res)
    x, W, R = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (m, n))
    y = torch.full((m * n + 64,), 9.0, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k,
                 residual=_dev(R.reshape(-1)) if with_res else None, mode=qdiy.GEMM_MFMA)
    torch.cuda.synchronize()
    out = y.cpu().numpy()
    assert np.all(out[m * n:] == np.float16(9.0)), "write past the end of y"
    got = out[:m * n].reshape(m, n).astype(np.float64)
    x64, W64 = x.astype(np.float64), W.astype(np.float64)
    s = x64 @ W64.T
    bound = k * 2.0 ** -23 * (np.abs(x64) @ np.abs(W64).T)
    if with_res:
        h = s.astype(np.float16).astype(np.float64)
        want = R.astype(np.float64) + h
        tol = ulp16(want) + ulp16(h) + bound + ulp16(s)
    else:
        want, tol = s, ulp16(s) + bound
    assert np.all(np.abs(got - want) <= tol), float(np.max(np.abs(got - want) - tol))


@pytest.mark.parametrize("m,n,k", [
    # 32 x 16 and 32 x 32 tiles, K over eight waves: fewer K tiles than waves, a wave
    # with one more than another, ragged rows and tokens
    (1, 32, 64), (16, 33, 64 * 7), (17, 31, 64 * 9), (33, 2050, 64 * 17), (100, 2048, 64 * 11),
    # 32 x 64 tiles in two K groups: odd and even K tiles, one alone; ragged tokens
    (63, 6144, 64), (49, 6112, 64 * 3), (64, 6100, 64 * 8),
    # 64 x 64 and 64 x 128 tiles (two rounds and one of a device's workgroups)
    (90, 6000, 64 * 5), (100, 11008, 64 * 3), (127, 11000, 64 * 2), (128, 10950, 64),
    # from 128 tokens where the ring tiles would leave CUs idle
    (200, 1024, 64 * 6), (140, 520, 64 * 13)])
@pytest.mark.parametrize("form", ["plain", "residual", "swiglu"])
def test_mfma_short_prompt_tiles(qdiy, m, n, k, form):
    """The short-prompt shapes of both matrix-core products at their edges, with padded x
    rows and y at an odd element offset (no 8-byte stores) when m is odd; nothing is
    written outside y's rows.  Bounds as in the tests around this one."""
    rng = np.random.default_rng(3 * m + n + k)
    ldx, off, pad = k + 8, m % 2, 0 if m % 2 else 4
    ldy = n + pad
    if form == "swiglu":
        n = max(1, n // 2)                              # two W rows per output: the same tiles
        ldy = n + pad
    x, W, W2 = normal_f16(rng, (m, ldx)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (n, k), 0.02)
    R = normal_f16(rng, (m, ldy))
    y = torch.full((off + m * ldy + 8,), 9.0, dtype=torch.float16, device="cuda")
    if form == "swiglu":
        qdiy.gemm_swiglu(_dev(x.reshape(-1)), _dev(W.reshape(-1)), _dev(W2.reshape(-1)), y[off:], m, n, k, ldx=ldx,
                         ldy=ldy)
    else:
        qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y[off:], m, n, k, ldx=ldx, ldy=ldy,
                     residual=_dev(R.reshape(-1)) if form == "residual" else None, mode=qdiy.GEMM_MFMA)
    torch.cuda.synchronize()
    out = y.cpu().numpy()
    rows = out[off:off + m * ldy].reshape(m, ldy)
    assert np.all(rows[:, n:] == 9.0) and np.all(out[:off] == 9.0) and np.all(out[off + m * ldy:] == 9.0)
    got = rows[:, :n].astype(np.float64)
    x64 = x[:, :k].astype(np.float64)
    s, bs = x64 @ W.astype(np.float64).T, k * 2.0 ** -23 * (np.abs(x64) @ np.abs(W.astype(np.float64)).T)
    if form == "plain":
        want, tol = s, ulp16(s) + bs
    elif form == "residual":
        h = s.astype(np.float16).astype(np.float64)
        want = R[:, :n].astype(np.float64) + h
        tol = ulp16(want) + ulp16(h) + bs + ulp16(s)
    else:
        u, bu = x64 @ W2.astype(np.float64).T, k * 2.0 ** -23 * (np.abs(x64) @ np.abs(W2.astype(np.float64)).T)
        g16, u16 = s.astype(np.float16).astype(np.float64), u.astype(np.float16).astype(np.float64)
        silu = u16 / (1.0 + np.exp(-u16))
        want = g16 * silu
        tol = np.abs(silu) * (ulp16(g16) + bs) + np.abs(g16) * 1.1 * (ulp16(u16) + bu) + 2 * ulp16(want)
    assert np.all(np.abs(got - want) <= tol), float(np.max(np.abs(got - want) - tol))


@pytest.mark.parametrize("m,n,k", [
    # short K, where a round's fixed part decides: 64 x 64 tiles in one and several rounds,
    # 32 x 64 tiles from two K tiles on, 64 x 128 tiles over many rows
    (9, 20000, 64), (33, 8190, 128), (63, 6144, 128), (65, 20010, 256), (127, 11000, 64),
    # one K tile: with a residual the 32 x 64 tile, whose second K group then has none
    (63, 6144, 64), (50, 6000, 64)])
@pytest.mark.parametrize("form", ["plain", "residual", "swiglu"])
def test_mfma_short_prompt_tiles_short_k(qdiy, m, n, k, form):
    """The tiles of the test above where K is short."""
    test_mfma_short_prompt_tiles(qdiy, m, n, k, form)


@pytest.mark.parametrize("m,n,k", [(231, 9979, 192), (303, 8703, 64), (403, 5123, 448), (34, 9183, 128)])
@pytest.mark.parametrize("form", ["plain", "residual", "swiglu"])
def test_mfma_short_prompt_tiles_unaligned_rows(qdiy, m, n, k, form):
    """Rows of y an odd number of elements apart: where that moves the choice of the tile."""
    test_mfma_short_prompt_tiles(qdiy, m, n, k, form)


@pytest.mark.parametrize("m,n,k,ldy", [(37, 100, 512, 100), (127, 1368, 2048, 1368),
                                        # from 128 rows: the 64 x 64 tile (n = 130, a strided
                                        # output), the 128 x 128 ring tile (a ragged last tile at
                                        # n = 1000; 512 x 5504), the 192 x 256 ring tile (2048 x
                                        # 5504: a last tile of 32 of its 96 outputs)
                                        (600, 130, 512, 136), (1000, 1000, 1024, 1000),
                                        (512, 5504, 2048, 5504), (2048, 5504, 2048, 5504),
                                        # the 192 x 256 tile over 3 K tiles, ragged tokens
                                        (1900, 5504, 192, 5504)])
def test_gemm_swiglu_within_bound(qdiy, m, n, k, ldy):
    """qd_gemm_swiglu: gate and up GEMMs on the matrix cores with the SwiGLU in the
    epilogue.  Each act is half(g * silu(u)) of g and u the fp16 roundings of
    fp32 sums; those may round to the neighbour of the float64 sum's fp16
    value when the fp32 sum lies within its summation bound of the boundary,
    so act is within the propagated bound of half(g64) * silu(half(u64)):
    |silu(u)| (ulp(g) + bound_g) + |g| 1.1 (ulp(u) + bound_u) + 2 ulp(act)."""
    rng = np.random.default_rng(31 * m + n + k)
    x = normal_f16(rng, (m, k))
    W1, W2 = normal_f16(rng, (n, k), 0.03), normal_f16(rng, (n, k), 0.03)
    act = torch.full((m * ldy + 64,), 9.0, dtype=torch.float16, device="cuda")
    qdiy.gemm_swiglu(_dev(x.reshape(-1)), _dev(W1.reshape(-1)), _dev(W2.reshape(-1)), act, m, n, k,
                     ldy=ldy)
    torch.cuda.synchronize()
    out = act.cpu().numpy()
    assert np.all(out[(m - 1) * ldy + n:] == np.float16(9.0)), "write past the last row"
    got = np.stack([out[i * ldy:i * ldy + n] for i in range(m)]).astype(np.float64)
    if ldy > n:
        gaps = np.stack([out[i * ldy + n:(i + 1) * ldy] for i in range(m - 1)])
        assert np.all(gaps == np.float16(9.0)), "write between rows"
    x64, W1d, W2d = x.astype(np.float64), W1.astype(np.float64), W2.astype(np.float64)
    g, u = x64 @ W1d.T, x64 @ W2d.T
    ax = np.abs(x64)
    bg, bu = k * 2.0 ** -23 * (ax @ np.abs(W1d).T), k * 2.0 ** -23 * (ax @ np.abs(W2d).T)
    gh = g.astype(np.float16).astype(np.float64)
    uh = u.astype(np.float16).astype(np.float64)
    silu = uh / (1.0 + np.exp(-uh))
    want = gh * silu
    tol = np.abs(silu) * (ulp16(gh) + bg) + np.abs(gh) * 1.1 * (ulp16(uh) + bu) + 2 * ulp16(want)
    err = np.abs(got - want)
    assert np.all(err <= tol), (float(np.max(err - tol)), np.unravel_index(np.argmax(err - tol), err.shape))
    # the bound is tight enough to see a swapped gate and up
    swapped = uh * (gh / (1.0 + np.exp(-gh)))
    assert np.mean(np.abs(swapped - got) > tol) > 0.5


@pytest.mark.parametrize("seed", range(16))
def test_mfma_random_shapes(qdiy, seed):
    """Seeded random m (both sides of the 128-row ring-tile threshold and of the
    64-token tile), n (ragged against 64), k (a multiple of 64 up to 6144, so the
    K-tile rings wrap several times or run short of their stages), row strides
    and the residual form of qd_gemm_nt, then qd_gemm_swiglu at the same m:
    every output within the bounds of the fixed-shape tests."""
    rng = np.random.default_rng(52000 + seed)
    m = int(rng.integers(1, 130)) if rng.random() < 0.6 else int(rng.integers(130, 700))
    n = int(rng.integers(1, 700))
    k = 64 * int(rng.integers(1, 97))
    ldy = n + int(rng.integers(0, 9))
    with_res = bool(rng.random() < 0.5)
    x, W, R = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (m, n))
    y = torch.full((m * ldy + 64,), 9.0, dtype=torch.float16, device="cuda")
    if with_res:
        yv = y[:m * ldy].view(m, ldy)
        yv[:, :n] = torch.from_numpy(R).cuda()
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k, residual=y if with_res else None,
                 mode=qdiy.GEMM_MFMA, ldy=ldy)
    torch.cuda.synchronize()
    out = y.cpu().numpy()
    assert np.all(out[m * ldy:] == np.float16(9.0)), "write past the end of y"
    rows = out[:m * ldy].reshape(m, ldy)
    if ldy > n:
        assert np.all(rows[:, n:] == np.float16(9.0)), "write into a row's padding"
    got = rows[:, :n].astype(np.float64)
    x64, W64 = x.astype(np.float64), W.astype(np.float64)
    s = x64 @ W64.T
    bound = k * 2.0 ** -23 * (np.abs(x64) @ np.abs(W64).T)
    if with_res:
        h = s.astype(np.float16).astype(np.float64)
        want = R.astype(np.float64) + h
        tol = ulp16(want) + ulp16(h) + bound + ulp16(s)
    else:
        want, tol = s, ulp16(s) + bound
    assert np.all(np.abs(got - want) <= tol), (m, n, k, ldy, with_res, float(np.max(np.abs(got - want) - tol)))
    # gate and up with the SwiGLU epilogue at the same m (ldy = n)
    W1, W2 = normal_f16(rng, (n, k), 0.03), normal_f16(rng, (n, k), 0.03)
    act = torch.full((m * n + 64,), 9.0, dtype=torch.float16, device="cuda")
    qdiy.gemm_swiglu(_dev(x.reshape(-1)), _dev(W1.reshape(-1)), _dev(W2.reshape(-1)), act, m, n, k)
    torch.cuda.synchronize()
    a = act.cpu().numpy()
    assert np.all(a[m * n:] == np.float16(9.0)), "write past the last row"
    got = a[:m * n].reshape(m, n).astype(np.float64)
    W1d, W2d = W1.astype(np.float64), W2.astype(np.float64)
    g, u = x64 @ W1d.T, x64 @ W2d.T
    ax = np.abs(x64)
    bg, bu = k * 2.0 ** -23 * (ax @ np.abs(W1d).T), k * 2.0 ** -23 * (ax @ np.abs(W2d).T)
    gh, uh = g.astype(np.float16).astype(np.float64), u.astype(np.float16).astype(np.float64)
    silu = uh / (1.0 + np.exp(-uh))
    want = gh * silu
    tol = np.abs(silu) * (ulp16(gh) + bg) + np.abs(gh) * 1.1 * (ulp16(uh) + bu) + 2 * ulp16(want)
    assert np.all(np.abs(got - want) <= tol), (m, n, k, float(np.max(np.abs(got - want) - tol)))


def test_gemm_nt_rejects_bad_arguments(qdiy):
    x = torch.zeros(4 * 96, dtype=torch.float16, device="cuda")
    w = torch.zeros(16 * 96, dtype=torch.float16, device="cuda")
    y = torch.zeros(4 * 16, dtype=torch.float16, device="cuda")
    with pytest.raises(qdiy.QdError, match="multiple of 64"):
        qdiy.gemm_nt(x, w, y, 4, 16, 96, mode=qdiy.GEMM_MFMA)
    with pytest.raises(qdiy.QdError, match="unknown mode"):
        qdiy.gemm_nt(x, w, y, 4, 16, 96, mode=7)
    big = torch.zeros(4096, dtype=torch.float16, device="cuda")
    with pytest.raises(qdiy.QdError, match="overlaps"):
        qdiy.gemm_nt(big[:4 * 64], w, big[128:128 + 4 * 16], 4, 16, 64)
    qdiy.gemm_nt(x, w, y, 4, 16, 64, mode=qdiy.GEMM_MFMA, ldx=96)     # strided x is fine
    torch.cuda.synchronize()


def test_mfma_large_m_unaligned_output_and_in_place_residual(qdiy):
    """m >= 512 with y rows an odd number of elements apart (the 64 x 64 tile
    takes it: the ring tiles store 8 bytes at a time) and with the residual
    added in place: both within the fp32 summation bound."""
    m, n, k = 640, 96, 256
    rng = np.random.default_rng(3)
    x, W, R = normal_f16(rng, (m, k)), normal_f16(rng, (n, k), 0.02), normal_f16(rng, (m, n))
    x64, W64 = x.astype(np.float64), W.astype(np.float64)
    s = x64 @ W64.T
    bound = k * 2.0 ** -23 * (np.abs(x64) @ np.abs(W64).T)
    ldy = n + 1
    y = torch.zeros(m * ldy, dtype=torch.float16, device="cuda")
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), y, m, n, k, mode=qdiy.GEMM_MFMA, ldy=ldy)
    torch.cuda.synchronize()
    got = y.cpu().numpy().reshape(m, ldy)[:, :n].astype(np.float64)
    assert np.all(np.abs(got - s) <= ulp16(s) + bound)
    yr = _dev(R.reshape(-1))
    qdiy.gemm_nt(_dev(x.reshape(-1)), _dev(W.reshape(-1)), yr, m, n, k, residual=yr, mode=qdiy.GEMM_MFMA)
    torch.cuda.synchronize()
    got = yr.cpu().numpy().reshape(m, n).astype(np.float64)
    h = s.astype(np.float16).astype(np.float64)
    want = R.astype(np.float64) + h
    assert np.all(np.abs(got - want) <= ulp16(want) + ulp16(h) + bound + ulp16(s))


@pytest.mark.parametrize("hidden,inter,n_prompt", [(512, 1368, 100), (512, 1368, 300), (2048, 5504, 300),
                                                  (512, 1408, 700)])
def test_engine_mfma_prefill(qdiy, hidden, inter, n_prompt):
    """MFMA prefill against exact prefill on the same prompt (with c_proj exact
    where inter is not a multiple of 64): the next step's logits agree to the
    fp32-order difference, and plain decode steps are bit-identical in both
    modes.  Gate/up is one launch with the SwiGLU epilogue; at hidden 2048 and 299
    tokens o_proj and c_proj share K out inside short tiles' workgroups."""
    cfg = qdiy.model_cfg(vocab_size=512, hidden_size=hidden, num_layers=2, num_heads=hidden // 128,
                         intermediate_size=inter, max_seqlen=n_prompt + 20)
    img = qdiy.random_model_image(cfg, 41 + hidden, 0.03, nthreads=8)
    prompt = [int(t) for t in np.random.default_rng(hidden).integers(0, 512, n_prompt)]
    res, kv = {}, {}
    with qdiy.Engine(image=img) as eng:
        for mode in (qdiy.GEMM_EXACT, qdiy.GEMM_MFMA):
            eng.set_prefill_mode(mode)
            eng.reset()
            pos = eng.prefill(prompt[:-1])
            kv[mode] = [eng.kv_rows(layer, 0, pos) for layer in range(cfg.num_layers)]
            eng.step(prompt[-1], pos)
            prefilled = eng.logits().astype(np.float64)
            eng.reset()
            eng.step(prompt[0], 0)                     # no prefill: decode kernels only
            res[mode] = (prefilled, eng.logits())
    exact, mfma = res[qdiy.GEMM_EXACT], res[qdiy.GEMM_MFMA]
    assert _same(exact[1], mfma[1]), "decode steps must not depend on the prefill mode"
    d = np.abs(exact[0] - mfma[0])
    assert float(np.max(d)) <= 0.02 * float(np.max(np.abs(exact[0]))) + 0.01, float(np.max(d))
    assert float(np.corrcoef(exact[0], mfma[0])[0, 1]) > 0.999
    # The KV rows the prefill leaves, against a float64 recomputation of the prompt.
    n = len(prompt) - 1
    m = model_tensors(img)
    ref_k, ref_v, term_k, term_v = model_kv_fp64(m, prompt[:-1], terms=True)
    bad_k, _ = model_kv_fp64(m, prompt[:-1], mutate="rope_sign")
    kv_terms = {"K": term_k, "V": term_v}
    for layer in range(cfg.num_layers):
        for mode in (qdiy.GEMM_EXACT, qdiy.GEMM_MFMA):
            k, v = kv[mode][layer]
            for name, got, ref in (("K", k, ref_k[layer]), ("V", v, ref_v[layer])):
                err = np.abs(got.astype(np.float64) - ref)
                scale = np.max(np.abs(ref), axis=1, keepdims=True)
                if layer == 0:
                    # fp16 roundings of the normalised input, the QKV sums, the bias add and
                    # the rotation, each within an ulp of values at most the row's scale
                    tol = 4 * ulp16(scale) + 2.0 ** -10 * kv_terms[name][layer]
                else:
                    # plus what the first layer's fp16 activations and attention carry over
                    tol = 0.01 * scale
                assert np.all(err <= tol), (layer, mode, name, float(np.max(err - tol)))
        if layer == 0:
            k0 = kv[qdiy.GEMM_MFMA][0][0].astype(np.float64)
            assert np.mean(np.abs(k0 - bad_k[0]) > 4 * ulp16(np.max(np.abs(bad_k[0])))) > 0.3


@pytest.mark.parametrize("inter,tokens", [(5504, 1024), (5440, 899), (64, 1000)])
def test_engine_mfma_prefill_two_slices_of_k(qdiy, inter, tokens):
    """Hidden 2048 with 897 to 1024 tokens: o_proj and c_proj have 128 tiles of 128 x 128,
    half the compute units, and run as two slices of K with a fold launch.  86 K tiles; 85
    (slices of 43 and 42) with 3 rows in the last token tile; a single one, which no slice can
    share.  What the second layer's KV rows see of both products is no further from float64
    than in the exact mode (the two differ by the order of fp32 sums alone)."""
    cfg = qdiy.model_cfg(vocab_size=512, hidden_size=2048, num_layers=2, num_heads=16,
                         intermediate_size=inter, max_seqlen=tokens + 8)
    img = qdiy.random_model_image(cfg, 43 + inter, 0.03, nthreads=8)
    prompt = [int(t) for t in np.random.default_rng(tokens).integers(0, 512, tokens)]
    kv = {}
    with qdiy.Engine(image=img) as eng:
        for mode in (qdiy.GEMM_EXACT, qdiy.GEMM_MFMA):
            eng.set_prefill_mode(mode)
            eng.reset()
            eng.prefill(prompt)
            kv[mode] = [a.astype(np.float64) for a in eng.kv_rows(1, 0, tokens)]
    ref_k, ref_v = model_kv_fp64(model_tensors(img), prompt)
    for i, ref in enumerate((ref_k[1], ref_v[1])):
        scale = np.max(np.abs(ref), axis=1, keepdims=True)
        err = {mode: np.abs(kv[mode][i] - ref) for mode in kv}
        assert np.all(err[qdiy.GEMM_MFMA] <= 0.01 * scale), float(np.max(err[qdiy.GEMM_MFMA] / scale))
        rms = {mode: np.sqrt(np.mean(err[mode] ** 2, axis=1)) for mode in kv}     # per token
        assert np.all(rms[qdiy.GEMM_MFMA] <= 2 * rms[qdiy.GEMM_EXACT])


def test_engine_mfma_prefill_two_passes(qdiy):
    """A 2300-token prompt: the MFMA mode runs it as passes of 2048 and 251 tokens (the
    second pass's attention starts at position 2048, over the first pass's KV rows), the
    exact mode as passes of 256. The next step's logits agree as above, and switching the
    mode back and forth keeps both working."""
    cfg = qdiy.model_cfg(vocab_size=512, hidden_size=512, num_layers=2, num_heads=4,
                         intermediate_size=1408, max_seqlen=2400)
    img = qdiy.random_model_image(cfg, 77, 0.03, nthreads=8)
    prompt = [int(t) for t in np.random.default_rng(2300).integers(0, 512, 2300)]
    logits = {}
    with qdiy.Engine(image=img) as eng:
        for mode in (qdiy.GEMM_MFMA, qdiy.GEMM_EXACT, qdiy.GEMM_MFMA):
            eng.set_prefill_mode(mode)
            eng.reset()
            pos = eng.prefill(prompt[:-1])
            assert pos == len(prompt) - 1
            eng.step(prompt[-1], pos)
            got = eng.logits().astype(np.float64)
            if mode in logits:
                assert _same(logits[mode], got), "the same mode must repeat bit for bit"
            logits[mode] = got
    exact, mfma = logits[qdiy.GEMM_EXACT], logits[qdiy.GEMM_MFMA]
    assert np.all(np.isfinite(mfma))
    d = np.abs(exact - mfma)
    assert float(np.max(d)) <= 0.02 * float(np.max(np.abs(exact))) + 0.01, float(np.max(d))
    assert float(np.corrcoef(exact, mfma)[0, 1]) > 0.999
