"""The prefill GEMM's group and wide tiles at the edges of their tiles: k that
leaves a remainder of every pipeline length, rows and tokens one past a tile,
rows that are no multiple of the four a store covers, every format and X / Y
type -- against the oracle's bit-exact f16 weights times the f16-rounded X in
float64.  fp32 Y: 1e-5 normwise (fp32 accumulation of at most 4096 products
of 11-bit operands: 4096^0.5 * 2^-24 is 4e-6); f16 Y: one rounding, 2^-11."""
import numpy as np
import pytest

import oracle
from cima_amd import gguf, nf4, synth
from cima_amd.hip import gemm_plan

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 2, 3, 6, 7, 8, 12, 13, 14, 23
FORMATS = [Q8_0, Q4_0, Q4_1, Q5_0, Q5_1, Q4_K, Q5_K, Q6_K, IQ4_XS]
# rows x tokens of every tile kind (128 x 128 instead of 64 x 128 for f32 X)
TILES = [(16, 16), (32, 16), (64, 32), (64, 64), (64, 128), (128, 256), (256, 256)]
TDT = {gguf.DT_F32: torch.float32, gguf.DT_F16: torch.float16, gguf.DT_BF16: torch.bfloat16}
F32, F16, BF16 = gguf.DT_F32, gguf.DT_F16, gguf.DT_BF16


def rel(a, b):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    return float(np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-300))


def operands(t, m, n, k, xd, offset=0):
    """Device x, device w at `offset` bytes past an aligned address, and the float64 product."""
    w = synth.weights(t, 300 + t, 0.02, n, k)
    raw = torch.zeros(w.size + offset, dtype=torch.uint8, device="cuda")
    raw[offset:] = torch.from_numpy(w.reshape(-1)).cuda()
    x = torch.from_numpy(synth.normal(301 + m, 1.0, m * k).reshape(m, k)).to(TDT[xd]).cuda()
    x16 = x.float().cpu().numpy().astype(np.float16).astype(np.float64)
    w16 = oracle.f16_bits_to_f32(oracle.dequant(t, w.reshape(-1), n * k)).reshape(n, k)
    return x, raw[offset:], x16 @ w16.astype(np.float64).T


def check(hip, t, m, n, k, xd, yd, tile=0, slab=None, offset=0, plan=(0, 0, 0), ops=None):
    x, w, want = ops or operands(t, m, n, k, xd, offset)
    ldy = n + 3
    y = torch.full((m, ldy), 7.0, dtype=TDT[yd], device="cuda")
    hip.set_gemm_tile(tile)
    hip.set_gemm_plan(*plan)
    try:
        if slab is None:
            hip.gguf_gemm(t, x, w, y, m, n, k, ldy, xd, yd)
        else:
            hip.gguf_gemm_slab(t, x, w, y, m, n, k, slab, ldy=ldy, x_dtype=xd, y_dtype=yd)
    finally:
        hip.set_gemm_tile(0)
        hip.set_gemm_plan(0, 0, 0)
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    assert rel(got[:, :n], want) <= (1e-5 if yd == F32 else 2.0 ** -11), (t, m, n, k, xd, yd, tile, plan)
    assert np.all(got[:, n:] == 7.0), "wrote past n"
    return y


@pytest.mark.parametrize("tile", [32, 64, 128, 256])
@pytest.mark.parametrize("k", [256, 512, 768, 1280, 2304])
def test_every_k_remainder(hip, tile, k):
    """4, 8, 12, 20 and 36 stages: whole rounds of the k groups' pipelines,
    fewer than one, and one to three stages over."""
    for xd, yd in ((BF16, F32), (F16, F16), (F32, F32)):
        check(hip, Q4_K, 70, 130, k, xd, yd, tile)


@pytest.mark.parametrize("tile", [32, 64, 128, 256])
@pytest.mark.parametrize("k", [64, 128, 192, 320, 832])
def test_every_k_remainder_32_element_blocks(hip, tile, k):
    """1, 2, 3, 5 and 13 stages: groups without a stage, odd unit counts."""
    for xd, yd in ((BF16, F32), (F16, F16), (F32, F32)):
        check(hip, Q8_0, 70, 130, k, xd, yd, tile)


@pytest.mark.parametrize("t", FORMATS)
@pytest.mark.parametrize("m, n", [(17, 1), (33, 63), (65, 65), (129, 129), (257, 258), (300, 67)])
def test_row_and_token_edges(hip, t, m, n):
    """Whatever tile is planned (the 16- and 32-token ones, at these few
    rows) at ragged rows and tokens."""
    check(hip, t, m, n, 512, BF16, F32)
    check(hip, t, m, n, 512, F16, F16)


@pytest.mark.parametrize("t", FORMATS)
@pytest.mark.parametrize("rows, tokens", TILES)
def test_edges_of_every_tile(hip, t, rows, tokens):
    """Every tile kind and format at rows and tokens one past a tile and one
    short of it, a row count the four-row stores do not divide among them."""
    for m, n in ((tokens + 1, rows + 1), (tokens - 1, 2 * rows - 1)):
        for xd, yd in ((BF16, F32), (F16, F16), (F32, F32)):
            check(hip, t, m, n, 512, xd, yd, plan=(rows, tokens, 0))


@pytest.mark.parametrize("k", [64, 128, 192, 320, 832])
def test_every_k_remainder_of_the_square_tile(hip, k):
    """The 256 x 256 tile at 1, 2, 3, 5 and 13 stages: no pair of weight
    units, whole pairs, one stage over."""
    for xd, yd in ((BF16, F32), (F16, F16)):
        check(hip, Q8_0, 70, 130, k, xd, yd, plan=(256, 256, 0))


@pytest.mark.parametrize("rows, tokens", TILES)
@pytest.mark.parametrize("bs", [64, 48])
def test_bitsandbytes_on_every_tile(hip, rows, tokens, bs):
    """NF4 decoded in the tiles (blocksize 64) and f16 weights decoded into
    the slab first (48), one past every tile."""
    m, n, k = tokens + 1, rows + 1, 768
    rng = np.random.default_rng(rows + tokens)
    packed = rng.integers(0, 256, n * k // 2, dtype=np.uint8)
    absmax = (rng.random(n * k // bs) + 0.01).astype(np.float32)
    w16 = oracle.f16_bits_to_f32(oracle.nf4_dequant(packed, absmax, nf4.NF4_CODE, n * k, bs)).reshape(n, k)
    p, a, q = (torch.from_numpy(v.copy()).cuda() for v in (packed, absmax, nf4.NF4_CODE))
    slab = torch.empty(hip.nf4_slab_bytes(m, n, k), dtype=torch.uint8, device="cuda")
    for xd, yd in ((BF16, F32), (F16, F16), (F32, F32)):
        x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(TDT[xd]).cuda()
        y = torch.full((m, n), float("nan"), dtype=TDT[yd], device="cuda")
        hip.set_gemm_plan(rows, tokens)
        try:
            hip.nf4_gemm_slab(x, p, a, q, y, m, n, k, bs, slab)
        finally:
            hip.set_gemm_plan(0, 0)
        torch.cuda.synchronize()
        want = x.float().cpu().numpy().astype(np.float16).astype(np.float64) @ w16.astype(np.float64).T
        assert rel(y.float().cpu().numpy(), want) <= (1e-5 if yd == F32 else 2.0 ** -11), (xd, yd)


@pytest.mark.parametrize("m", [13, 32, 40, 100, 140, 600, 2100])
@pytest.mark.parametrize("k", [768, 320])
def test_f16_slices_sum_alike(hip, m, k):
    """Weights decoded into the slab a slice at a time: slices of whatever size
    the slab holds, the last one short, take tiles by their own rows, and Y has
    the bits of one slice of all rows."""
    n, bs = 1030, 48 if k % 48 == 0 else 80
    rng = np.random.default_rng(m + k)
    p, a, q = (torch.from_numpy(v).cuda() for v in (rng.integers(0, 256, n * k // 2, dtype=np.uint8),
                                                    (rng.random(-(-n * k // bs)) + 0.01).astype(np.float32),
                                                    nf4.NF4_CODE.copy()))
    for xd, yd in ((BF16, F32), (F16, F16), (F32, F32)):
        x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(TDT[xd]).cuda()
        ys = []
        for rows in (n, 512, 130, 24):
            slab = torch.empty(2 * rows * k, dtype=torch.uint8, device="cuda")
            ys.append(torch.full((m, n), float("nan"), dtype=TDT[yd], device="cuda"))
            hip.nf4_gemm_slab(x, p, a, q, ys[-1], m, n, k, bs, slab)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(ys[0]).all()) and all(torch.equal(y, ys[0]) for y in ys[1:]), (xd, yd)


@pytest.mark.parametrize("t", [Q8_0, Q4_0, Q5_0, Q6_K])
@pytest.mark.parametrize("tile", [16, 32, 64, 128, 256])
def test_weights_two_bytes_off_a_word(hip, t, tile):
    """Formats read as aligned words at 2-byte alignment: the packed weight
    2 bytes past a word boundary gives the bits of an aligned one."""
    a = check(hip, t, 40, 96, 512, F16, F32, tile)
    b = check(hip, t, 40, 96, 512, F16, F32, tile, offset=2)
    assert torch.equal(a, b)


@pytest.mark.parametrize("t, k", [(Q4_K, 256), (Q8_0, 192), (Q6_K, 512), (Q5_K, 256)])
@pytest.mark.parametrize("xd, yd", [(BF16, F32), (F16, F16)])
def test_square_wide_tile(hip, t, k, xd, yd):
    """The 256 x 256 tile, planned where it saves a round of workgroups:
    ragged rows and tokens, whole and odd numbers of stages."""
    assert gemm_plan(t, 300, 32770, k, xd) == (256, 256, 1)
    check(hip, t, 300, 32770, k, xd, yd)


@pytest.mark.parametrize("t, m, n, k", [(Q4_K, 100, 512, 4096), (Q6_K, 33, 130, 4096), (Q8_0, 70, 256, 2048)])
@pytest.mark.parametrize("yd", [F32, F16])
def test_k_split_of_the_group_tiles(hip, t, m, n, k, yd):
    """With a slab, narrow weights are planned split along k over workgroups:
    within the bars, and bit-identical run to run."""
    slab = torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
    assert gemm_plan(t, m, n, k, BF16, slab.numel())[2] > 1
    a = check(hip, t, m, n, k, BF16, yd, slab=slab)
    b = check(hip, t, m, n, k, BF16, yd, slab=slab)
    assert torch.equal(a, b)


@pytest.mark.parametrize("t, k", [(Q4_K, 2304), (Q6_K, 4096), (Q8_0, 2176)])
@pytest.mark.parametrize("rows, tokens", [(16, 16), (32, 16), (64, 32), (64, 64), (64, 128)])
@pytest.mark.parametrize("xd", [BF16, F16, F32])
def test_k_split_of_every_tile(hip, t, k, rows, tokens, xd):
    """Two and four ranges of k (34, 36 and 64 stages of 64: even, odd and
    whole-round shares of a split) on every tile that splits, at rows and
    tokens one past a tile: within the bars, the partial tiles in the slab
    (as many as the split) and nothing past them, the same bits run to
    run; against the unsplit product only the order of the sum differs."""
    m, n = tokens + 1, rows + 1
    ops = operands(t, m, n, k, xd)
    for ks in (2, 4):
        stages = k // 128 if tokens == 16 else k // 64
        split = stages % ks == 0 and stages // ks >= (4 if tokens == 16 else 8) and k % (128 if tokens == 16 else 64) == 0
        need = 4 * ks * m * n
        for yd in (F32, F16):
            slab = torch.full((need + 4096,), 0x5A, dtype=torch.uint8, device="cuda")
            a = check(hip, t, m, n, k, xd, yd, slab=slab, plan=(rows, tokens, ks), ops=ops)
            if tokens != 16 or k % 128 == 0:
                assert bool((slab[:need] != 0x5A).any()) == split, (ks, split)
                if split:  # the last partial tile is the last that is written
                    assert bool((slab[need - 4 * m * n:need] != 0x5A).any())
            assert bool((slab[need:] == 0x5A).all()), "wrote past the partial tiles"
            b = check(hip, t, m, n, k, xd, yd, slab=slab, plan=(rows, tokens, ks), ops=ops)
            assert torch.equal(a, b)
            u = check(hip, t, m, n, k, xd, yd, plan=(rows, tokens, 1), ops=ops)
            assert rel(a.float().cpu().numpy(), u.float().cpu().numpy()) <= (1e-6 if yd == F32 else 2.0 ** -11)
            # a slab one byte short of the partials is left alone
            short = torch.full((need - 1,), 0x5A, dtype=torch.uint8, device="cuda")
            v = check(hip, t, m, n, k, xd, yd, slab=short, plan=(rows, tokens, ks), ops=ops)
            if tokens != 16 or k % 128 == 0:
                assert torch.equal(v, u) and bool((short == 0x5A).all())


@pytest.mark.parametrize("t, m, n, k, xd, plan", [(Q6_K, 100, 4096, 14336, F16, (64, 128)),
                                                  (Q4_K, 60, 4096, 14336, BF16, (64, 64)),
                                                  (Q4_K, 100, 14336, 4096, F32, (128, 128))])
def test_planned_k_split_of_the_wide_group_tiles(hip, t, m, n, k, xd, plan):
    """Shapes of real layers that plan the 64- and 128-token tiles split, f32
    X's two k groups among them, on 256 sampled rows."""
    slab = torch.zeros(32 << 20, dtype=torch.uint8, device="cuda")
    assert gemm_plan(t, m, n, k, xd, slab.numel())[:2] == plan and gemm_plan(t, m, n, k, xd, slab.numel())[2] > 1
    w = synth.weights(t, 300 + t, 0.02, n, k)
    x = torch.from_numpy(synth.normal(301 + m, 1.0, m * k).reshape(m, k)).to(TDT[xd]).cuda()
    y = torch.empty((m, n), device="cuda")
    hip.gguf_gemm_slab(t, x, torch.from_numpy(w.reshape(-1)).cuda(), y, m, n, k, slab, x_dtype=xd, y_dtype=F32)
    torch.cuda.synchronize()
    rows = np.random.default_rng(m).choice(n, 256, replace=False)
    w16 = oracle.f16_bits_to_f32(oracle.dequant(t, np.stack([w.reshape(n, -1)[r] for r in rows]).reshape(-1), 256 * k))
    want = x.float().cpu().numpy().astype(np.float16).astype(np.float64) @ w16.reshape(256, k).astype(np.float64).T
    assert rel(y.cpu().numpy()[:, rows], want) <= 1e-5
    assert bool((slab != 0).any())


@pytest.mark.parametrize("t", [Q4_K, Q5_K, IQ4_XS, 0], ids=["q4_k", "q5_k", "iq4_xs", "nf4"])
@pytest.mark.parametrize("n, k", [(8225, 256), (8225, 768), (8225, 1280), (8225, 2048), (24617, 2048)])
def test_32_row_tiles_of_full_and_low_grids(hip, t, n, k):
    """The 32-row tiles decode in one go at two and four workgroups per CU
    where k is a multiple of 2048 (258 and 770 row tiles; NF4 at four, any k)
    and in parts otherwise (slices of 4096 rows, at most 128 tiles): the same
    bits."""
    m, bs = 13, 64
    rng = np.random.default_rng(k)
    if t:
        w = torch.from_numpy(synth.weights(t, 300 + t, 0.02, n, k).reshape(n, -1)).cuda()
    else:
        w = torch.from_numpy(rng.integers(0, 256, (n, k // 2), dtype=np.uint8)).cuda()
        absmax = torch.from_numpy((rng.random((n, k // bs)) + 0.01).astype(np.float32)).cuda()
        qmap = torch.from_numpy(nf4.NF4_CODE.copy()).cuda()
        slab = torch.empty(1 << 20, dtype=torch.uint8, device="cuda")

    def mul(x, r0, r1, yd):
        y = torch.full((m, r1 - r0), float("nan"), dtype=TDT[yd], device="cuda")
        if t:
            hip.gguf_gemm(t, x, w[r0:r1], y, m, r1 - r0, k)
        else:
            hip.nf4_gemm_slab(x, w[r0:r1], absmax[r0:r1], qmap, y, m, r1 - r0, k, bs, slab)
        return y

    hip.set_gemm_plan(32, 16)
    try:
        for xd, yd in ((BF16, F32), (F16, F16), (F32, F32)):
            x = torch.from_numpy(rng.standard_normal((m, k)).astype(np.float32)).to(TDT[xd]).cuda()
            whole = mul(x, 0, n, yd)
            parts = torch.cat([mul(x, r, min(r + 4096, n), yd) for r in range(0, n, 4096)], 1)
            torch.cuda.synchronize()
            assert torch.equal(whole, parts) and bool(torch.isfinite(whole).all()), (xd, yd)
    finally:
        hip.set_gemm_plan(0, 0)
