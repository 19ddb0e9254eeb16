"""The merge of split-attention partials in a launch of its own: the kernel at
every count of chunks around its batches and groups, and the decode step of
models whose partials are large enough to take that route."""
import numpy as np
import pytest

from cima_amd.decoder import DecoderConfig, DeviceDecoder, synthetic_kv, synthetic_model
from oracle import decode as od

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [64, 128])
@pytest.mark.parametrize("seq, window", [(1, 0), (16, 0), (17, 0), (127, 0), (128, 0), (129, 0), (384, 0), (385, 0),
                                         (1024, 0), (1025, 0), (2100, 0), (2100, 33), (2100, 700)])
def test_attn_reduce_chunk_counts(hip, dim, seq, window):
    """1 to 132 chunks of 16 positions against the merge in float64; chunks
    outside the live range hold NaN and must not be read into the result.
    One f16 rounding (2^-11) of a sum whose weights carry fp32 exponentials
    (a few 2^-23 each)."""
    heads, csz, max_seq = 5, 16, 2112
    nch = max_seq // csz
    r = np.random.default_rng(seq + dim)
    part = np.full((heads, nch, dim + 2), np.nan, np.float32)
    c0, active = (max(0, seq - window) // csz if window else 0), -(-seq // csz)
    live = slice(c0, active)
    part[:, live, 0] = r.normal(size=(heads, active - c0)) * 4
    part[:, live, 1] = r.uniform(1, 16, size=(heads, active - c0))
    part[:, live, 2:] = r.normal(size=(heads, active - c0, dim)) * part[:, live, 1:2]
    if active - c0 > 1:  # a chunk with nothing unmasked carries no weight, the first one too
        part[:, c0 + seq % 2, 0], part[:, c0 + seq % 2, 1:] = -np.inf, 0
    out = torch.empty((heads, dim), dtype=torch.float16, device="cuda")
    hip.attn_reduce(torch.from_numpy(part).cuda(), out, heads, dim, csz, nch, seq, max_seq, window)
    torch.cuda.synchronize()
    p = part[:, live].astype(np.float64)
    w = np.exp(p[:, :, 0] - p[:, :, 0].max(1, keepdims=True))
    want = (w[..., None] * p[:, :, 2:]).sum(1) / (w * p[:, :, 1]).sum(1)[:, None]
    got = out.float().cpu().numpy()
    assert np.all(np.abs(got - want) <= 2.0 ** -11 * np.abs(want) + 2e-6), np.abs(got - want).max()


@pytest.mark.parametrize("head_dim, q_heads, kv_heads, max_seq, chunk, window",
                         [(64, 16, 4, 2048, 64, 0), (128, 8, 2, 2048, 64, 0), (64, 16, 4, 2048, 64, 150)])
def test_decode_step_merging_apart(hip, head_dim, q_heads, kv_heads, max_seq, chunk, window):
    """Partials past 128 KB: the step merges them in their own launch; the
    logits of steps early and late in the cache against the oracle (2
    sqrt(layers) 1e-3, the decode steps' end-to-end bar)."""
    cfg = DecoderConfig(n_layers=2, hidden=512, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, ffn=512,
                        vocab=1000, max_seq=max_seq, attn_chunk=chunk, window=window)
    assert q_heads * (max_seq // chunk) * (head_dim + 2) * 4 > 128 << 10
    m = synthetic_model(cfg, seed=6)
    d = DeviceDecoder(hip, m)
    for ctx_len in (0, 1000):
        kvs = [synthetic_kv(cfg, i, ctx_len) for i in range(cfg.n_layers)]
        for i, (kc, vc) in enumerate(kvs):
            d.load_kv(i, kc, vc)
        om = dict(cfg=dict(hidden=cfg.hidden, q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, ffn=cfg.ffn,
                           vocab=cfg.vocab, rope_theta=cfg.rope_theta, rms_eps=cfg.rms_eps, type=int(cfg.ggml_type),
                           embed_type=int(m.embed_type), head_type=int(m.head_type)),
                  embed=m.embed, head=m.head, final_norm=m.final_norm,
                  layers=[dict(L, k_cache=kv[0].copy(), v_cache=kv[1].copy()) for L, kv in zip(m.layers, kvs)])
        d.set_state(17, ctx_len)
        d.step()
        torch.cuda.synchronize()
        want, _ = od.decode_step(om, 17, ctx_len)
        got = d.logits.float().cpu().numpy().astype(np.float64)
        want = want.astype(np.float64)
        assert np.linalg.norm(got - want) / np.linalg.norm(want) <= 2.0 * np.sqrt(2) * 1e-3
        assert d.position() == ctx_len + 1


def test_merging_apart_replays_as_eager(hip):
    """The step with its merge launch, captured once: every replay equals an
    eager step of a second decoder in the same state."""
    cfg = DecoderConfig(n_layers=2, hidden=512, q_heads=16, kv_heads=4, head_dim=64, ffn=512, vocab=1000, max_seq=2048,
                        attn_chunk=64)
    m = synthetic_model(cfg, seed=8)
    eager, graph = DeviceDecoder(hip, m), DeviceDecoder(hip, m)
    for d in (eager, graph):
        for i in range(cfg.n_layers):
            d.load_kv(i, *synthetic_kv(cfg, i, 700))
        d.set_state(3, 700)
    graph.capture()
    for s in range(4):
        eager.step()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(eager.logits, graph.logits), s
        assert eager.token() == graph.token() and graph.position() == 701 + s
