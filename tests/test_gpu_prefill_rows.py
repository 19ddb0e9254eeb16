"""RMSNorm and RoPE over several rows at the edges of their wide paths: word
counts around a thread's registers, rows and pointers that only the
element-wise path takes, head counts around a workgroup's."""
import numpy as np
import pytest

from oracle import decode as od

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def dev(a, offset=0):
    """a on the device as f16, `offset` elements past an aligned address."""
    t = torch.zeros(a.size + offset, dtype=torch.float16, device="cuda")
    t[offset:] = torch.from_numpy(np.ascontiguousarray(a, np.float16).reshape(-1)).cuda()
    return t[offset:]


@pytest.mark.parametrize("n, offset", [(8, 0), (248, 0), (256, 0), (1000, 0), (2048, 0), (2056, 0), (8192, 0),
                                       (8200, 0), (100, 0), (4096, 1)])
@pytest.mark.parametrize("unit", [False, True])
def test_rmsnorm_rows(hip, n, offset, unit):
    """Within two f16 steps of float64 (one rounding, and the inverse root
    mean square in fp32 can move a value across a rounding boundary)."""
    rows = 3
    r = np.random.default_rng(n)
    x = (r.normal(size=(rows, n)) * np.array([[1], [300], [20000]])).astype(np.float16)
    w = r.normal(1, 0.1, size=n).astype(np.float16)
    y = dev(np.zeros((rows, n)), offset)
    hip.rmsnorm(dev(x, offset), None if unit else dev(w, offset), y, rows, n, 1e-5)
    torch.cuda.synchronize()
    xs = np.clip(x.astype(np.float64), -65000, 65000)
    want = xs / np.sqrt((xs * xs).mean(1, keepdims=True) + 1e-5) * (1.0 if unit else w.astype(np.float64))
    got = y.cpu().numpy().astype(np.float64).reshape(rows, n)
    assert np.all(np.abs(got - want) <= 2 * np.spacing(np.abs(want).astype(np.float16)).astype(np.float64))


@pytest.mark.parametrize("heads, dim, nfreqs", [(1, 64, 32), (15, 64, 32), (16, 128, 64), (17, 128, 64), (33, 32, 10),
                                                (2, 256, 128)])
@pytest.mark.parametrize("rows", [5, 205])
def test_rope_head_counts(hip, heads, dim, nfreqs, rows):
    """Every head of every row rotates once, by a head or by up to 16 heads a
    workgroup (from 3072 heads on): against the oracle row by row (fp32 sine
    and cosine of fp32 angles below 2000 rad: absolute 2e-3)."""
    pos = 1000
    x = np.random.default_rng(heads).normal(size=(rows, heads, dim)).astype(np.float16)
    t = dev(x)
    hip.rope(t, rows, heads, dim, pos, 1e4, nfreqs)
    torch.cuda.synchronize()
    got = t.cpu().numpy().reshape(rows, heads, dim).astype(np.float64)
    for i in range(rows):
        want = od.rope(x[i:i + 1], pos + i, 1e4, nfreqs=nfreqs)[0].astype(np.float64)
        assert np.abs(got[i] - want).max() <= 2e-3
