"""Attention over contexts past 1024 positions (the scores of a kv head's
query heads together, the values by chunks of 256) against the oracle, bit
for bit, prompt batches and decode steps. The rotary table is the identity
and each input lies on a circle, so a position's score runs with its angle:
flat rows, rows that rise or fall over many binades, a late peak."""
import numpy as np
import pytest

from oracle.model import Config, Stage
from test_gpu_fused_stage import coded_model, make_stage, same_bits

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
