"""The planner of the prefill products, asked without a device (cima_hip_gemm_plan
on 256 compute units)."""
import ctypes

import pytest

from cima_amd import gguf, hip

F32, F16, BF16 = gguf.DT_F32, gguf.DT_F16, gguf.DT_BF16
SLAB = 32 << 20
TILES = {(16, 16), (32, 16), (64, 32), (64, 64), (64, 128), (128, 128), (128, 256), (256, 256)}


@pytest.mark.parametrize("t", [0] + [int(f) for f in gguf.DType])
@pytest.mark.parametrize("xd", [F32, F16, BF16])
def test_every_plan_can_run(t, xd):
    """A built tile, 16-token tiles only for k % 128 == 0, 256 x 256 not for f32
    X, a split only into ranges the tile takes and the slab holds."""
    for m in (1, 16, 17, 32, 33, 64, 65, 100, 128, 129, 256, 300, 700, 2048, 5000):
        for n in (1, 63, 300, 1024, 4096, 14336, 128256):
            for k in (256, 768, 4096, 14336) + (() if t in (12, 13, 14, 23) else (64, 192, 832)):
                for slab in (0, 1 << 16, SLAB):
                    rows, tokens, ks = hip.gemm_plan(t, m, n, k, xd, slab)
                    assert (rows, tokens) in TILES
                    assert (rows, tokens) != ((256, 256) if xd == F32 else (128, 128))
                    assert (rows, tokens) != (64, 128) or xd != F32
                    assert tokens != 16 or k % 128 == 0
                    stages, least = (k // 128, 4) if tokens == 16 else (k // 64, 8)
                    assert ks == 1 or (ks in (2, 4) and tokens <= 128 and stages % ks == 0 and stages // ks >= least
                                       and 4 * ks * m * n <= slab)


@pytest.mark.parametrize("t, m, n, k, xd, slab, plan", [
    (12, 16, 1024, 4096, BF16, SLAB, (16, 16, 4)),   # 7.9 us; unsplit 9.1
    (12, 16, 1024, 4096, F32, SLAB, (16, 16, 4)),    # 9.3; unsplit 12.9
    (12, 16, 512, 2048, BF16, SLAB, (16, 16, 1)),    # 6.1; four ranges 6.6
    (13, 16, 896, 4864, F16, SLAB, (16, 16, 2)),     # 9.4; 64 x 32 in four 12.4
    (14, 24, 896, 4864, F16, SLAB, (16, 16, 2)),     # 64 x 32 in four 16.8 against 14.7
    (3, 32, 4864, 896, F32, 0, (32, 16, 1)),         # 7.0; 16-row tiles 11.0
    (0, 32, 4864, 896, F32, 0, (32, 16, 1)),         # 8.2; 16-row tiles 11.8
    (12, 16, 14336, 4096, BF16, SLAB, (32, 16, 1)),  # 16.5
    (12, 32, 14336, 4096, BF16, SLAB, (64, 32, 1)),  # 21.6; 16-token tiles 33.0
    (12, 16, 4096, 14336, BF16, 0, (16, 16, 1))])    # 26.6; 32-row tiles 42.6
def test_few_tokens_take_the_measured_plan(t, m, n, k, xd, slab, plan):
    """Up to 32 tokens a plan by the CUs' fill stands unless another is clearly
    cheaper (measured on MI355X, cold, us)."""
    assert hip.gemm_plan(t, m, n, k, xd, slab) == plan


@pytest.mark.parametrize("xd", [F32, F16, BF16])
def test_slices_are_planned_by_their_rows(xd):
    """f16 weights of 14336 x 4096 in slices of 4096 rows: at least a quarter of
    the 256 compute units at work up to 64 tokens, over half beyond 200 (planned
    for the whole weight, the 256-token tiles left 32 workgroups at 300
    tokens); every slab size sums alike."""
    for m in (16, 64, 200, 300, 700):
        rows, tokens, ks = hip.gemm_plan(1, m, 14336, 4096, xd, SLAB)
        assert ks == 1 and -(-4096 // rows) * -(-m // tokens) >= (64 if m <= 64 else 128 if m != 700 else 96)
        alike = {t for t in TILES if [t[1] == 16, t[1] == 256, t == (128, 128)] ==
                 [tokens == 16, tokens == 256, (rows, tokens) == (128, 128)]}
        assert all(hip.gemm_plan(1, m, 14336, 4096, xd, s)[:2] in alike
                   for s in (8192, 100 << 10, 1 << 20, SLAB, 1 << 30))
    with pytest.raises(hip.EngineError):
        hip.gemm_plan(1, 16, 14336, 4096, xd, 8191)


def test_refusals():
    for bad in ((0, 16, 16, 256), (256, 0, 16, 256), (256, 16, 16, 100), (256, 16, 16, -256)):
        cu, m, n, k = bad
        with pytest.raises(hip.EngineError):
            hip.gemm_plan(12, m, n, k, F16, 0, cu)
    with pytest.raises(hip.EngineError):
        hip.gemm_plan(99, 16, 16, 256, F16)
    with pytest.raises(hip.EngineError):
        hip.gemm_plan(12, 16, 16, 256, 7)
    L = hip.load_library()
    assert L.cima_hip_gemm_plan(256, 12, 16, 16, 256, F16, 0, None, None, ctypes.byref(ctypes.c_int())) == hip.E_INVALID
    assert L.cima_hip_set_gemm_plan(None, 64, 64, 1) == hip.E_NOT_INIT
