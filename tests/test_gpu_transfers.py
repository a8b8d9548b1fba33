"""Rows and ports between host and device (copy kernels over pinned staging): sizes that
end within a 16-byte piece or a workgroup, uploads that follow one another, fill the
staging or overtake running tasks, and projections that read their rows from the port or
from elsewhere."""
import numpy as np
import pytest

import workloads
from helpers import accel_shape, oracle_from_synthetic, oracle_shape
from oracle import orc

pytestmark = pytest.mark.gpu

SPEC = workloads.ShapeSpec("transfers", 512, 256, 688, 1, 4, 2, 256, 0.25, 0.5)


@pytest.fixture(scope="module")
def ctx():
    import llm_accel
    synth = workloads.SyntheticModel(SPEC)
    with llm_accel.Accelerator(accel_shape(SPEC)) as acc:
        acc.load_model(synth)
        yield synth, acc


def _ints(rng, shape):
    return rng.integers(-32768, 32768, size=shape).astype(np.int16)


def test_port_sizes(ctx):
    import llm_accel
    _, acc = ctx
    rng = np.random.default_rng(1)
    for n in (1, 7, 8, 9, 2047, 2048, 2049, 8 * 688):
        whole = _ints(rng, 8 * 688)
        acc.port_write(llm_accel.PORT_IN, whole)
        acc.port_write(llm_accel.PORT_IN, whole[:n] ^ 1)
        assert np.array_equal(acc.port_read(llm_accel.PORT_IN, n), whole[:n] ^ 1), n
        # nothing past the written values changes
        got = acc.port_read(llm_accel.PORT_IN, whole.size)
        assert np.array_equal(got[n:], whole[n:]), n


@pytest.mark.parametrize("rows", [1, 3, 8])
def test_uploads_in_a_row(ctx, rows):
    """More uploads than the staging holds, none read in between; then an upload behind
    a running task that reads the rows before it."""
    synth, acc = ctx
    rng = np.random.default_rng(rows)
    last = {}
    for i in range(24):
        last[i % 2] = _ints(rng, (rows, SPEC.hidden))
        acc.upload(i % 2, last[i % 2])
    for pair, want in last.items():
        assert np.array_equal(acc.download(pair, rows), want)
    h = synth.hidden_rows(rows)
    om = oracle_from_synthetic(synth, oracle_shape(SPEC))
    _, want, _ = om.task(om.new_kv(), 18, 0, h, 0)
    acc.upload(1, h)
    acc.task(18, 0, rows, 0, 1, 0)
    acc.upload(1, last[1])
    assert np.array_equal(acc.download(0, rows), want)
    assert np.array_equal(acc.download(1, rows), last[1])


@pytest.mark.parametrize("rows", [1, 2, 5, 8])
def test_projection_rows_from_anywhere(ctx, rows):
    """Rows in the in port (read in place), in another port, at an address that is no
    multiple of 16 bytes, and overwritten by the result."""
    import llm_accel as L
    synth, acc = ctx
    x = _ints(np.random.default_rng(rows), (rows, SPEC.hidden))
    want = orc.projection(x, synth.weight(0, 3))
    p_in, p_aux, p_out = (acc.port(p)[0] for p in (L.PORT_IN, L.PORT_AUX, L.PORT_OUT))
    for port, src, shift, dst in ((L.PORT_IN, p_in, 0, p_out), (L.PORT_AUX, p_aux, 0, p_out),
                                  (L.PORT_IN, p_in, 1, p_out), (L.PORT_IN, p_in, 0, p_in)):
        acc.port_write(port, np.concatenate([np.full(shift, 77, np.int16), x.reshape(-1)]))
        _, st = acc.op(L.OP_O_PROJECTION, 0, rows, 0, 0, in_ptr=src + 2 * shift, out_ptr=dst)
        assert st.code == 0
        got = acc.port_read(L.PORT_OUT if dst == p_out else L.PORT_IN, want.size)
        assert np.array_equal(got.reshape(want.shape), want), (port, shift, dst == p_in)
