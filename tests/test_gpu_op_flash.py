"""The tile-parallel launches of the operator-level flash attention (ops 14 and 17) over
many tiles against the oracle, at the tile counts around where they take over, head_dims
and groups at the edges of their loops, saturating keys and values, and contexts where the
running maximum rises at every tile."""
import numpy as np
import pytest

from oracle import orc
import workloads
from helpers import accel_shape

pytestmark = pytest.mark.gpu

SPECS = {  # head_dim, query heads per KV head
    "d128g8": workloads.ShapeSpec("d128g8", 64, 2048, 256, 1, 16, 2, 2048, 0.1, 0.3),
    "d64g2": workloads.ShapeSpec("d64g2", 64, 256, 256, 1, 4, 2, 2048, 0.1, 0.3),
    "d48g5": workloads.ShapeSpec("d48g5", 64, 480, 256, 1, 10, 2, 2048, 0.1, 0.3),
    "d16g16": workloads.ShapeSpec("d16g16", 64, 256, 256, 1, 16, 1, 2048, 0.1, 0.3),
    "d112g3": workloads.ShapeSpec("d112g3", 64, 336, 256, 1, 3, 1, 2048, 0.1, 0.3),
}


def _cache(rng, n, d, kind):
    if kind == "saturating":
        k = rng.integers(-32768, 32768, size=(n, d))
        v = rng.integers(-32768, 32768, size=(n, d))
    else:
        k = rng.normal(size=(n, d)) * 256
        v = rng.normal(size=(n, d)) * 400
        if kind == "rising":  # scores grow with the position
            k = k * 0.1 + np.arange(n)[:, None] * 0.3
    return [np.clip(np.round(x), -32768, 32767).astype(np.int16) for x in (k, v)]


@pytest.mark.parametrize("name,kind,n", [
    ("d128g8", "plain", 129), ("d128g8", "plain", 128), ("d128g8", "saturating", 700),
    ("d128g8", "rising", 1999), ("d64g2", "plain", 513), ("d64g2", "rising", 1030),
    ("d48g5", "plain", 200), ("d48g5", "saturating", 321), ("d16g16", "plain", 640),
    ("d112g3", "saturating", 450)])
def test_flash_and_prefill_block(name, kind, n):
    import llm_accel
    spec = SPECS[name]
    g, d, hk = spec.heads // spec.kv_heads, spec.head_dim, spec.kv_heads
    rng = np.random.default_rng(n + d)
    rows = [_cache(rng, n + 8, d, kind) for _ in range(hk)]
    q = np.clip(np.round(rng.normal(size=(hk, 8, g, d)) * (300 if kind != "rising" else 20)
                         + (0 if kind != "rising" else 40)), -32768, 32767).astype(np.int16)
    if kind == "saturating":
        q[0, 0] = -32768
        rows[0][0][5] = -32768  # every bank of this score reaches 2^31
    print(f"case {name} {kind} n={n}", flush=True)
    with llm_accel.Accelerator(accel_shape(spec)) as a:
        for h in range(hk):
            a.kv_write(0, h, 0, *rows[h])
        if g <= 8:  # op 14's rows are the group's heads, at most 8
            got, _ = a.run_attention(llm_accel.OP_ATTN_FLASH, q[:, 0], position=n - 1)
        for h in range(hk if g <= 8 else 0):
            want = orc.attention(q[h, 0], rows[h][0][:n], rows[h][1][:n], semantics=2)
            assert np.array_equal(got[h], want), f"op 14 head {h}"
        for t0, tokens in ((0, 8), (3, 1)):
            got, _ = a.run_prefill_attention_block(q[:, :tokens], n - 1 + t0, tokens)
            for h in range(hk):
                for t in range(tokens):
                    e = n + t0 + t
                    want = orc.attention(q[h, t], rows[h][0][:e], rows[h][1][:e], semantics=0)
                    assert np.array_equal(got[h, t], want), f"op 17 head {h} token {t}"
