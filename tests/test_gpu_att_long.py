"""Attention over contexts past 1024 positions (the scores of a kv head's
query heads together, the values by chunks of 256) against the oracle, bit
for bit, prompt batches and decode steps. The rotary table is the identity
and each input lies on a circle, so a position's score runs with its angle:
flat rows, rows that rise or fall over many binades, a late peak."""
import numpy as np
import pytest

from oracle.model import Config, Stage
from test_gpu_fused_stage import coded_model, make_stage, oracle_generate, same_bits
from test_gpu_stage_seqs import seqs_generate

pytestmark = pytest.mark.gpu

T = 1400
ANGLES = {
    "flat": lambda t: 0 * t,
    "rising": lambda t: np.pi * (1 - t / T),
    "falling": lambda t: np.pi * t / T,
    "late peak": lambda t: np.where(t == T - 150, 0.0, np.pi * 0.9),
    "random": lambda t: np.random.default_rng(1).uniform(0, 2 * np.pi, t.size),
}


@pytest.mark.parametrize("heads,kv_heads,hd", [(4, 2, 128), (2, 2, 128), (4, 1, 64), (3, 3, 32)])
@pytest.mark.parametrize("scale", [3e-4, 6e-3])
def test_long_context_rows(dev, heads, kv_heads, hd, scale):
    c = Config(dim=96, hidden=64, layers=1, heads=heads, kv_heads=kv_heads, head_dim=hd, vocab=50, seq_len=T + 4,
               dtype="q8_0")
    m = coded_model(c, 21, scale / 2, scale * 2)
    half = hd // 2
    m.rope = lambda n: (np.ones(n * half, np.float32), np.zeros(n * half, np.float32))
    rng = np.random.default_rng(5)
    a, b = rng.normal(0, 1, (2, c.dim)).astype(np.float32)
    for name, angle in ANGLES.items():
        if hd < 128 and name not in ("rising", "random"):
            continue
        th = angle(np.arange(T)).astype(np.float32)[:, None]
        xs = np.concatenate([np.cos(th) * a + np.sin(th) * b, np.stack([a, b, a + b])]).astype(np.float32)
        cpu = Stage(m, T + 4)
        want = np.stack([cpu.forward(x.copy(), t) for t, x in enumerate(xs)])
        st, mats = make_stage(dev, m, T + 4)
        try:
            got = np.concatenate([st.forward(xs[:T], 0)] + [st.forward(xs[t], t) for t in range(T, T + 3)])
            for t in range(T + 3):
                same_bits(got[t], want[t], f"{name}, position {t}")
        finally:
            st.free()
            for mt in mats:
                mt.free()
    assert dev.used == 0


# (a context of 4100: a prompt's values past 1024 positions by the kernel of
# the decode steps, else by two workgroups a CU)
@pytest.mark.parametrize("heads,kv_heads,hd,ctx", [(4, 2, 128, 1200), (4, 2, 128, 4100), (4, 1, 64, 1200)])
def test_infinity_and_nan_rows(dev, heads, kv_heads, hd, ctx):
    """A position whose activations hold an infinity (its key and value are
    NaNs): the positions before it are untouched, those after it as the
    oracle's, in a prompt and in decode steps."""
    c = Config(dim=96, hidden=64, layers=1, heads=heads, kv_heads=kv_heads, head_dim=hd, vocab=50, seq_len=ctx,
               dtype="q8_0")
    m = coded_model(c, 21, 1e-3, 1e-2)
    rng = np.random.default_rng(5)
    xs = rng.normal(0, 1, (1110, c.dim)).astype(np.float32)
    xs[1100, 7] = np.inf
    cpu = Stage(m, 1200)
    want = np.stack([cpu.forward(x.copy(), t) for t, x in enumerate(xs)])
    st, mats = make_stage(dev, m, ctx)
    try:
        got = np.concatenate([st.forward(xs[:1105], 0)] + [st.forward(xs[t], t) for t in range(1105, 1110)])
        for t in range(1110):
            same_bits(got[t], want[t], f"position {t}")
    finally:
        st.free()
        for mt in mats:
            mt.free()
    assert dev.used == 0


@pytest.mark.parametrize("heads,kv_heads,hd,ctx,lens", [
    (4, 2, 128, 1300, (1100, 3, 1, 40)), (4, 2, 128, 1300, (1022, 3, 1, 40)), (4, 2, 64, 1300, (1100, 3, 1, 40)),
    (4, 2, 64, 1300, (1022, 3, 1, 40)), (8, 2, 128, 4100, (1100, 3, 1, 40, 7, 200, 64, 2, 1022))])
def test_sequences_of_a_long_context(dev, heads, kv_heads, hd, ctx, lens):
    """Sequences side by side in a long context: each one's position and
    caches, a prompt past 1024 positions (no batches shared), one whose steps
    cross them, and more values workgroups than CUs."""
    c = Config(dim=96, hidden=64, layers=1, heads=heads, kv_heads=kv_heads, head_dim=hd, vocab=50, seq_len=ctx,
               dtype="q8_0")
    m = coded_model(c, 22, 1e-3, 1e-2)
    rng = np.random.default_rng(6)
    prompts = [[int(t) for t in rng.integers(0, c.vocab, n)] for n in lens]
    steps = 6
    lg, toks = seqs_generate(dev, m, prompts, steps, ctx)
    for z, p in enumerate(prompts):
        want_t, want_l = oracle_generate(m, p, steps, ctx)
        for k in range(steps):
            same_bits(lg[k, z], want_l[k], f"sequence {z} (prompt {len(p)}), step {k}")
        assert toks[z] == want_t, f"sequence {z} tokens"
    assert dev.used == 0
