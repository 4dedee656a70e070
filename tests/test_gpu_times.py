"""Kernel times beside each other: of the same work where a configuration
does not add any (a longer context, a padded slice), and of less work
against more. Each is the profiler's time of a call's launches, the least of
several calls; the bounds leave half of the difference that the right launch
makes."""
import numpy as np
import pytest

import rkhip
from oracle.model import Config
from test_gpu_fused_stage import coded_model, make_stage, upload_layers

pytestmark = pytest.mark.gpu


def profile(dev, run):
    """{kernel: (launches, ms)} of run()."""
    dev.profile_start()
    try:
        run()
    finally:
        prof = dev.profile_stop()
    return prof


def least_ms(dev, run, kernel, calls=7):
    return min(profile(dev, run)[kernel][1] for _ in range(calls))


@pytest.mark.parametrize("transposed", [0, 1])
def test_tensor_positions_past_k_cost_nothing(dev, transposed):
    """2048 x k x 2048 float32: a slice of 8 positions against a whole one."""
    n = 2048
    arena = dev.arena(2 * n * 64 + n * n, 64)
    try:
        def run(k):
            dev._check(rkhip.lib().rk_tensor_matmul_device(dev.h, rkhip.TENSOR_F32, transposed, n, k, n,
                                                           arena.device_ptr(0), arena.device_ptr(64 * n),
                                                           arena.device_ptr(128 * n), None))

        ms = {k: least_ms(dev, lambda: [run(k) for _ in range(10)], "tensor_matmul_f32") for k in (8, 64)}
    finally:
        arena.free()
    assert ms[8] < 0.8 * ms[64], ms


@pytest.mark.parametrize("kind,rows,cols,n,inside", [
    (rkhip.FP8, 4096, 1024, 3, True), (rkhip.FP8, 64, 65536, 1, False), (rkhip.FP8, 16384, 4096, 1, False),
    (rkhip.FP4, 4096, 1024, 2, True), (rkhip.FP4, 64, 1024, 3, False), (rkhip.FP4, 64, 65536, 1, False),
    (rkhip.FP4, 32768, 4096, 1, False)])
def test_block_scaled_products_quantize_where_it_pays(dev, kind, rows, cols, n, inside):
    """The input's quantize launch, by the weights that would quantize it
    again: inside the products for the smaller calls only."""
    w = np.zeros(rows * cols // (1 if kind == rkhip.FP8 else 2), np.uint8)
    s = np.full((rows + 31) // 32 * (cols // 32) if kind == rkhip.FP8 else rows * cols // 32, 120, np.uint8)
    ms = [dev.upload_mx(kind, rows, cols, w, s) for _ in range(n)]
    try:
        prof = profile(dev, lambda: dev.matvecs(ms, np.ones(cols, np.float32)))
    finally:
        for m in ms:
            m.free()
    assert ("act_fp8" in prof) == (not inside), prof


@pytest.mark.parametrize("kind", [rkhip.BF16, rkhip.F32])
def test_narrow_dense_rows(dev, kind):
    """128000 rows of 32 values against as many of 512."""
    ms = {}
    for cols in (32, 512):
        m = dev.upload(kind, 128000, cols, np.zeros(128000 * cols, np.uint16 if kind == rkhip.BF16 else np.float32))
        arena = dev.arena(cols + 128000, 64)
        try:
            name = "matvec_bf16" if kind == rkhip.BF16 else "matvec_f32"
            ms[cols] = least_ms(dev, lambda: dev.matvecs_device([m], [arena.device_ptr(cols)], arena.device_ptr(0), cols),
                                name)
        finally:
            arena.free()
            m.free()
    assert ms[32] < 0.75 * ms[512], ms


def test_shared_prompts_scores_do_not_grow_with_the_context(dev):
    """Heads of 64: a scores workgroup for each position up to the furthest
    prompt's, not up to the context."""
    c = Config(dim=64, hidden=64, layers=1, heads=32, kv_heads=2, head_dim=64, vocab=50, seq_len=8192, dtype="q8_0")
    m = coded_model(c, 5, 1e-3, 1e-2)
    prompts = [[int(t) for t in np.random.default_rng(z).integers(0, c.vocab, 17)] for z in range(8)]
    ms = {}
    for ctx in (256, 8192):
        layers, mats = upload_layers(dev, m)
        emb = dev.upload(m.embed.kind, m.embed.rows, m.embed.cols, m.embed.q, m.embed.scales)
        cos, sin = m.rope(ctx)
        st = rkhip.Stage(dev, c.dim, c.hidden, c.heads, c.kv_heads, ctx, layers, cos, sin, head_dim=c.head_dim,
                         norm_eps=float(c.eps()), seqs=len(prompts))
        try:
            st.set_head(emb, emb, m.rms_final)
            st.seqs_start(prompts)
            ms[ctx] = least_ms(dev, lambda: st.seqs_start(prompts), "att_scores")
        finally:
            st.free()
            emb.free()
            for mt in mats:
                mt.free()
    assert ms[8192] < 2 * ms[256], ms


@pytest.mark.parametrize("heads,kv_heads,hd", [(16, 1, 128), (32, 8, 128), (32, 8, 64)])
def test_early_positions_of_a_long_context(dev, heads, kv_heads, hd):
    """A decode step at position 40: its attention's scores and values in a
    context of 4096 positions against one of 1024."""
    c = Config(dim=64, hidden=64, layers=1, heads=heads, kv_heads=kv_heads, head_dim=hd, vocab=50, seq_len=4096,
               dtype="q8_0")
    m = coded_model(c, 5, 1e-3, 1e-2)
    xs = np.random.default_rng(1).normal(0, 1, (41, c.dim)).astype(np.float32)
    ms = {}
    for ctx in (1024, 4096):
        st, mats = make_stage(dev, m, ctx)
        try:
            st.forward(xs[:40], 0)
            p = [profile(dev, lambda: st.forward(xs[40:], 40)) for _ in range(25)]
            ms[ctx] = {k: min(x[k][1] for x in p) for k in p[0] if k.startswith("att_")}
        finally:
            st.free()
            for mt in mats:
                mt.free()
    for k in ms[1024].keys() & ms[4096].keys():
        assert ms[4096][k] < 1.25 * ms[1024][k], (k, ms)


def test_prompt_past_1024_positions_two_workgroups_a_cu(dev):
    """A prompt's values past 1024 positions: a context whose weights leave a
    CU room for two workgroups, against one that does not."""
    c = Config(dim=64, hidden=64, layers=1, heads=16, kv_heads=4, head_dim=128, vocab=50, seq_len=8192, dtype="q8_0")
    m = coded_model(c, 5, 1e-3, 1e-2)
    xs = np.random.default_rng(1).normal(0, 1, (1400, c.dim)).astype(np.float32)
    ms = {}
    for ctx in (2048, 8192):
        st, mats = make_stage(dev, m, ctx)
        try:
            st.forward(xs[:1200], 0)
            ms[ctx] = least_ms(dev, lambda: st.forward(xs[1200:], 1200), "att_values")
        finally:
            st.free()
            for mt in mats:
                mt.free()
    assert ms[2048] < 0.9 * ms[8192], ms
