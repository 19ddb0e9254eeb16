"""The prefill GEMM's group and wide tiles at the edges of their tiles: k that
leaves a remainder of every pipeline length, rows and tokens one past a tile,
rows that are no multiple of the four a store covers, every format and X / Y
type -- against the oracle's bit-exact f16 weights times the f16-rounded X in
float64.  fp32 Y: 1e-5 normwise (fp32 accumulation of at most 4096 products
of 11-bit operands: 4096^0.5 * 2^-24 is 4e-6); f16 Y: one rounding, 2^-11."""
import numpy as np
import pytest

import oracle
from cima_amd import gguf, synth

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

Q4_0, Q4_1, Q5_0, Q5_1, Q8_0, Q4_K, Q5_K, Q6_K, IQ4_XS = 2, 3, 6, 7, 8, 12, 13, 14, 23
FORMATS = [Q8_0, Q4_0, Q4_1, Q5_0, Q5_1, Q4_K, Q5_K, Q6_K, IQ4_XS]
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


def check(hip, t, m, n, k, xd, yd, tile=0, slab=None, offset=0):
    x, w, want = operands(t, m, n, k, xd, offset)
    ldy = n + 3
    y = torch.full((m, ldy), 7.0, dtype=TDT[yd], device="cuda")
    hip.set_gemm_tile(tile)
    try:
        if slab is None:
            hip.gguf_gemm(t, x, w, y, m, n, k, ldy, xd, yd)
        else:
            hip.gguf_gemm_slab(t, x, w, y, m, n, k, slab, ldy=ldy, x_dtype=xd, y_dtype=yd)
    finally:
        hip.set_gemm_tile(0)
    torch.cuda.synchronize()
    got = y.float().cpu().numpy()
    assert rel(got[:, :n], want) <= (1e-5 if yd == F32 else 2.0 ** -11), (t, m, n, k, xd, yd, tile)
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
    """The planned tile at rows and tokens one past (or short of) a tile."""
    check(hip, t, m, n, 512, BF16, F32)
    check(hip, t, m, n, 512, F16, F16)


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
    check(hip, t, 300, 32770, k, xd, yd)


@pytest.mark.parametrize("t, m, n, k", [(Q4_K, 100, 512, 4096), (Q6_K, 33, 130, 4096), (Q8_0, 70, 256, 2048),
                                        (Q4_K, 32, 1024, 4096)])
@pytest.mark.parametrize("yd", [F32, F16])
def test_k_split_of_the_group_tiles(hip, t, m, n, k, yd):
    """With a slab, narrow weights split along k over workgroups: within the
    bars, and bit-identical run to run."""
    slab = torch.empty(32 << 20, dtype=torch.uint8, device="cuda")
    a = check(hip, t, m, n, k, BF16, yd, slab=slab)
    b = check(hip, t, m, n, k, BF16, yd, slab=slab)
    assert torch.equal(a, b)
