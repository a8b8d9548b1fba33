"""The layer-major prompt path of llm_generate (csrc/prefill.hip) against the
block-by-block prompt, bit for bit: sampled tokens, every K/V row, both hidden
pairs and the report's counts, over row counts at the edges of the 32-row pieces,
64-position tiles and 64- / 128-row workgroup tiles, ragged block sizes, head_dims
that fill the matrix cores' operands and that do not, 12-bit weights with and
without corrections, 16-bit weights, and saturating queries, keys and values; prompts
that run in several parts; and once against the oracle's block by block replay.  Every
comparison checks from the launch counts that the two requests took the two paths."""
import sys

import numpy as np
import pytest

import workloads
from helpers import accel_shape, oracle_from_synthetic, oracle_shape

pytestmark = pytest.mark.gpu

# (vocab, hidden, inter, heads, KV heads): head_dim 64, 128, 48, 32 and 16
D64 = workloads.ShapeSpec("d64", 512, 256, 688, 2, 4, 2, 1200, 0.25, 0.5)
D128 = workloads.ShapeSpec("d128", 512, 1024, 1300, 2, 8, 2, 1200, 0.125, 0.3)
D48 = workloads.ShapeSpec("d48", 512, 480, 1300, 2, 10, 2, 1200, 0.125, 0.3)
D32 = workloads.ShapeSpec("d32", 512, 192, 260, 2, 6, 3, 1200, 0.25, 0.5)
D16 = workloads.ShapeSpec("d16", 512, 128, 132, 2, 8, 8, 1200, 0.25, 0.5)


def _say(msg):
    print(msg, flush=True)
    sys.stdout.flush()


class Model:
    """Arrays of a SyntheticModel with weights planted or replaced."""

    def __init__(self, spec, kind):
        self.synth = workloads.SyntheticModel(spec)
        rng = np.random.default_rng(91)
        self.emb = self.synth.embedding()
        for layer in range(spec.layers):
            for proj in range(7):
                w = self.synth.weight(layer, proj)
                n, k = w.shape
                if kind == "corrections":
                    for r in (0, 1, n // 2, n - 1):
                        cols = rng.choice(k, size=4, replace=False)
                        w[r, cols] = rng.choice([-32768, -2049, 2048, 30000], size=4)
                elif kind == "wide":
                    w[rng.random(w.shape) < 0.02] = 4095
                    w[0, :6] = [32767, -32768, 32640, 32767, -2049, 2048]
        if kind == "saturating":  # q, k, v past the Q4.12 operand's range
            for proj in range(3):
                self.synth.weight(0, proj)[:] = rng.integers(-2048, 2048, size=self.synth.weight(0, proj).shape)
        if kind == "extreme":
            # every query and key element of layer 0 the lowest value: at
            # position 0 each bank's sum is exactly 2^31
            self.emb = np.abs(self.emb) + 64
            for proj in range(2):
                self.synth.weight(0, proj)[:] = -2048

    def weight(self, layer, proj):
        return self.synth.weight(layer, proj)

    def norms(self):
        return self.synth.norms()


def _request(monkeypatch, spec, model, prompt, block, gen, layer_major):
    import llm_accel
    monkeypatch.setenv("LLM_ACCEL_PROMPT", "1" if layer_major else "0")
    with llm_accel.Accelerator(accel_shape(spec)) as a:
        a.load_model(model)
        a.load_lm_head(model.emb)
        for pair in (0, 1):  # rows that no block writes stay what they were
            a.upload(pair, np.full((8, spec.hidden), 7 + pair, np.int16))
        a.kernel_timing(True)
        toks, st = a.generate(model.emb, prompt, block, spec.layers, gen)
        parts = a.kernel_stats()["rope"][0] / spec.layers  # a launch of this path only
        a.kernel_timing(False)
        kv = [a.kv_read(layer, h, 0, len(prompt)) for layer in range(spec.layers)
              for h in range(spec.kv_heads)]
        pairs = [a.download(p, 8) for p in (0, 1)]
        # the next tasks find the state a block left
        a.task(18, 0, 1, len(prompt), 1, 0)
        more = a.download(0, 8)
    counts = {k: v for k, v in st.items() if not k.endswith("ms")}
    return toks, kv, pairs, more, counts, parts


def _compare(monkeypatch, spec, kind, n, block, gen=1, parts=1):
    model = Model(spec, kind)
    rng = np.random.default_rng(n)
    prompt = [int(t) for t in rng.integers(0, spec.vocab, size=n)]
    _say(f"case {spec.name} {kind} P{n} B{block}")
    want = _request(monkeypatch, spec, model, prompt, block, gen, False)
    got = _request(monkeypatch, spec, model, prompt, block, gen, True)
    assert got[0] == want[0], "tokens"
    for i, ((k0, v0), (k1, v1)) in enumerate(zip(want[1], got[1])):
        assert np.array_equal(k0, k1), f"K rows {i}: {np.argwhere(k0 != k1)[:3]}"
        assert np.array_equal(v0, v1), f"V rows {i}"
    for p in (0, 1):
        assert np.array_equal(got[2][p], want[2][p]), \
            f"pair {p}: {np.argwhere(got[2][p] != want[2][p])[:3]}"
    assert np.array_equal(got[3], want[3])
    assert got[4] == want[4]
    assert want[5] == 0 and got[5] == parts


@pytest.mark.parametrize("n,block", [(4, 1), (5, 1), (31, 8), (33, 5), (64, 8), (65, 8), (127, 3),
                                     (129, 8), (200, 7)])
def test_row_counts(monkeypatch, n, block):
    # four rows one by one stay in blocks
    _compare(monkeypatch, D64, "plain", n, block, parts=0 if (n, block) == (4, 1) else 1)


@pytest.mark.parametrize("spec", [D128, D48, D32, D16], ids=lambda s: s.name)
@pytest.mark.parametrize("n,block", [(26, 8), (193, 6)])
def test_head_dims(monkeypatch, spec, n, block):
    _compare(monkeypatch, spec, "plain", n, block, gen=3)


@pytest.mark.parametrize("kind", ["corrections", "wide", "saturating", "extreme"])
@pytest.mark.parametrize("spec", [D64, D128, D48], ids=lambda s: s.name)
def test_weights_and_saturation(monkeypatch, spec, kind):
    _compare(monkeypatch, spec, kind, 131, 8)


def test_long_prompt(monkeypatch):
    _compare(monkeypatch, D128, "plain", 1100, 8)


# Prompts of more rows than run at a time (2,048, or the multiple of the block below):
# later parts read the earlier rows' K/V pages, share a page with them where the block
# does not divide 64, and may be shorter than a block.
LONG64 = workloads.ShapeSpec("long64", 512, 256, 688, 2, 4, 2, 4300, 0.25, 0.5)
LONG128 = workloads.ShapeSpec("long128", 512, 512, 700, 1, 4, 2, 4300, 0.125, 0.3)
LONG48 = workloads.ShapeSpec("long48", 512, 480, 700, 1, 10, 2, 4300, 0.125, 0.3)


@pytest.mark.parametrize("spec,kind,n,block,parts", [
    (LONG64, "plain", 2048, 8, 1), (LONG64, "plain", 2049, 8, 2), (LONG64, "saturating", 2056, 8, 2),
    (LONG64, "plain", 2047, 5, 1), (LONG64, "plain", 2049, 5, 2),
    (LONG64, "corrections", 2100, 5, 2), (LONG64, "wide", 2051, 7, 2),
    (LONG64, "plain", 4200, 8, 3), (LONG128, "plain", 2100, 5, 2), (LONG128, "saturating", 4100, 3, 3),
    (LONG128, "extreme", 2081, 7, 2), (LONG48, "plain", 2075, 6, 2), (LONG48, "saturating", 2300, 8, 2)],
    ids=lambda v: getattr(v, "name", str(v)))
def test_prompts_in_parts(monkeypatch, spec, kind, n, block, parts):
    _compare(monkeypatch, spec, kind, n, block, gen=2, parts=parts)


# Shapes whose products have more tiles than workgroups, which then take several in
# turn: gate|up with one and three 128-input steps per tile (even and odd numbers of
# steps leave the buffers' parity either way), and down with K in four parts.
TURN1 = workloads.ShapeSpec("turn1", 512, 128, 6016, 1, 4, 2, 1200, 0.25, 0.5)
TURN3 = workloads.ShapeSpec("turn3", 512, 384, 4004, 1, 6, 2, 1200, 0.125, 0.3)
TURNP = workloads.ShapeSpec("turnp", 512, 1152, 4096, 1, 18, 2, 1200, 0.125, 0.3)


@pytest.mark.parametrize("spec,kind,n", [
    (TURN1, "plain", 700), (TURN1, "wide", 641), (TURN3, "plain", 769),
    (TURN3, "corrections", 650), (TURNP, "plain", 600)],
    ids=lambda v: getattr(v, "name", str(v)))
def test_tiles_in_turn(monkeypatch, spec, kind, n):
    _compare(monkeypatch, spec, kind, n, 8)


# K in two, four and eight parts for up to 64 rows, of unequal lengths: 40, 21 and 11
# steps of down, 9 of Q|K|V and O.
SPLIT40 = workloads.ShapeSpec("split40", 512, 256, 5100, 1, 4, 2, 1200, 0.25, 0.5)
SPLIT21 = workloads.ShapeSpec("split21", 512, 1152, 2600, 1, 18, 2, 1200, 0.125, 0.3)
SPLIT11 = workloads.ShapeSpec("split11", 512, 128, 1300, 1, 4, 2, 1200, 0.25, 0.5)


@pytest.mark.parametrize("kind", ["plain", "wide", "corrections"])
@pytest.mark.parametrize("spec,n", [(SPLIT40, 32), (SPLIT40, 51), (SPLIT21, 25),
                                    (SPLIT21, 64), (SPLIT11, 30)],
                         ids=lambda v: getattr(v, "name", str(v)))
def test_split_products(monkeypatch, spec, n, kind):
    _compare(monkeypatch, spec, kind, n, 4)


@pytest.mark.parametrize("kind,n,block,layered", [
    ("plain", 24, 8, False), ("plain", 25, 8, True), ("plain", 4, 1, False), ("plain", 5, 1, True),
    ("one corrected", 25, 8, True), ("corrections", 32, 8, False), ("corrections", 33, 8, True),
    ("corrections", 5, 1, False), ("corrections", 6, 1, True), ("wide", 40, 8, False),
    ("wide", 41, 8, True), ("wide", 6, 1, False), ("wide", 7, 1, True)])
def test_where_it_begins(monkeypatch, kind, n, block, layered):
    """The blocks from which a prompt runs layer by layer: more where the weights need
    corrections in most launches, or 16 bits, as each is where it becomes the faster way."""
    import llm_accel
    monkeypatch.setenv("LLM_ACCEL_PROMPT", "1")
    model = Model(D64, "plain" if kind == "one corrected" else kind)
    if kind == "one corrected":
        model.weight(0, 6)[3, 5] = 3000
    with llm_accel.Accelerator(accel_shape(D64)) as a:
        a.load_model(model)
        a.kernel_timing(True)
        a.generate(model.emb, list(range(n)), block, D64.layers, 0)
        assert a.kernel_stats()["rope"][0] == (D64.layers if layered else 0)


def test_prompts_that_outgrow_the_workspace(monkeypatch):
    """One context, prompts of growing and falling length: each is the first work on a
    workspace that has just been allocated, or runs in a larger one."""
    import llm_accel
    spec = D128
    model = Model(spec, "plain")
    rng = np.random.default_rng(23)
    prompts = [[int(t) for t in rng.integers(0, spec.vocab, size=n)] for n in (40, 300, 1100, 90)]
    got = {}
    for mode in ("0", "1"):
        monkeypatch.setenv("LLM_ACCEL_PROMPT", mode)
        with llm_accel.Accelerator(accel_shape(spec)) as a:
            a.load_model(model)
            a.load_lm_head(model.emb)
            for prompt in prompts:
                toks, _ = a.generate(model.emb, prompt, 8, spec.layers, 2)
                kv = [a.kv_read(layer, h, 0, len(prompt)) for layer in range(spec.layers)
                      for h in range(spec.kv_heads)]
                got.setdefault(mode, []).append((toks, a.download(0, 8), a.download(1, 8), kv))
    for n, (want, have) in zip(map(len, prompts), zip(got["0"], got["1"])):
        assert have[0] == want[0], n
        assert np.array_equal(have[1], want[1]) and np.array_equal(have[2], want[2]), n
        for i, ((k0, v0), (k1, v1)) in enumerate(zip(want[3], have[3])):
            assert np.array_equal(k0, k1) and np.array_equal(v0, v1), (n, i)


def _bounded(monkeypatch, spec, model, prompts, block, limit):
    """One context whose prompt buffers may take `limit` bytes (None: any): per prompt
    its token, pairs, K/V rows and how often a layer ran over rows of it (0: in blocks)."""
    import llm_accel
    monkeypatch.setenv("LLM_ACCEL_PROMPT", "1")
    monkeypatch.delenv("LLM_ACCEL_PROMPT_BYTES", raising=False)
    if limit is not None:
        monkeypatch.setenv("LLM_ACCEL_PROMPT_BYTES", str(int(limit)))
    out = []
    with llm_accel.Accelerator(accel_shape(spec)) as a:
        a.load_model(model)
        a.load_lm_head(model.emb)
        for prompt in prompts:
            a.kernel_timing(True)
            toks, _ = a.generate(model.emb, prompt, block, spec.layers, 1)
            times = a.kernel_stats()["rope"][0]
            assert times % spec.layers == 0
            kv = [a.kv_read(layer, h, 0, len(prompt)) for layer in range(spec.layers)
                  for h in range(spec.kv_heads)]
            out.append((toks, a.download(0, 8), a.download(1, 8), kv, times // spec.layers))
    return out


@pytest.mark.parametrize("block", [8, 7])
def test_no_room_for_the_workspace(monkeypatch, block):
    """A workspace that cannot be had in full: fewer rows at a time, at last the prompt
    in blocks; the same results, and no error."""
    spec, model = D64, Model(D64, "plain")
    prompt = [int(t) for t in np.random.default_rng(31).integers(0, spec.vocab, size=1100)]
    want, = _bounded(monkeypatch, spec, model, [prompt], block, None)
    assert want[4] == 1
    seen = []
    for limit in (41e6, 37e6, 35.9e6, 35.2e6, 30e6, 0):
        got, = _bounded(monkeypatch, spec, model, [prompt], block, limit)
        _say(f"case blocks of {block}, workspace of {limit / 1e6:.1f} MB: {got[4]} parts")
        assert got[0] == want[0]
        assert np.array_equal(got[1], want[1]) and np.array_equal(got[2], want[2])
        for i, ((k0, v0), (k1, v1)) in enumerate(zip(want[3], got[3])):
            assert np.array_equal(k0, k1) and np.array_equal(v0, v1), i
        seen.append(got[4])
    assert seen[0] > 1 and seen[:4] == sorted(set(seen[:4])) and seen[4:] == [0, 0], seen


def test_workspace_that_cannot_grow(monkeypatch):
    """A longer prompt than the buffers in hand, and no room for larger ones: it runs in
    those, and so does the next."""
    spec, model = D64, Model(D64, "plain")
    rng = np.random.default_rng(37)
    prompts = [[int(t) for t in rng.integers(0, spec.vocab, size=n)] for n in (100, 500, 90)]
    want = _bounded(monkeypatch, spec, model, prompts, 8, None)
    got = _bounded(monkeypatch, spec, model, prompts, 8, 35.2e6)
    assert [w[4] for w in want] == [1, 1, 1] and [g[4] for g in got] == [1, 4, 1]
    for w, g in zip(want, got):
        assert g[0] == w[0] and np.array_equal(g[1], w[1]) and np.array_equal(g[2], w[2])
        for (k0, v0), (k1, v1) in zip(w[3], g[3]):
            assert np.array_equal(k0, k1) and np.array_equal(v0, v1)


def test_oracle_replay(monkeypatch):
    """Hidden pairs and K/V rows of a prompt over three tiles against the
    oracle's task by task replay."""
    import llm_accel
    spec, n, block = D64, 139, 8
    model = Model(spec, "corrections")
    prompt = [int(t) for t in np.random.default_rng(5).integers(0, spec.vocab, size=n)]
    om = oracle_from_synthetic(model, oracle_shape(spec))
    kv = om.new_kv()
    for b0 in range(0, n, block):
        h = model.emb[prompt[b0:b0 + block]].copy()
        for layer in range(spec.layers):
            _, h, _ = om.task(kv, 18, layer, h, b0)
            _, h, _ = om.task(kv, 19, layer, h, b0)
    _, fin, _ = om.task(kv, 20, 0, h, b0)
    with llm_accel.Accelerator(accel_shape(spec)) as a:
        a.load_model(model)
        a.generate(model.emb, prompt, block, spec.layers, 0)
        rows = n - b0
        assert np.array_equal(a.download(1, rows), h)
        assert np.array_equal(a.download(0, rows), fin)
        for layer in range(spec.layers):
            for hd in range(spec.kv_heads):
                k, v = a.kv_read(layer, hd, 0, n)
                assert np.array_equal(k, kv[0][layer, hd, :n]), f"K {layer} {hd}"
                assert np.array_equal(v, kv[1][layer, hd, :n]), f"V {layer} {hd}"
