"""Rows and ports between host and device (copy kernels over pinned staging): sizes that
end within a 16-byte piece or a workgroup, uploads that follow one another, fill the
staging or overtake running tasks, projections that read their rows from the port or
from elsewhere, and copies that are complete once an address is in the caller's hands."""
import ctypes

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


class _Memory:
    """Copies through the HIP runtime that the library links, on the null stream: the
    context's stream does not wait for it, nor it for the context's."""

    def __init__(self):
        self.rt = ctypes.CDLL("libamdhip64.so.7")

    def read(self, dev, n):
        a = np.zeros(n, np.int16)
        assert self.rt.hipMemcpy(a.ctypes.data_as(ctypes.c_void_p), ctypes.c_void_p(dev),
                                 ctypes.c_size_t(2 * n), 2) == 0
        return a

    def write(self, dev, a):
        a = np.ascontiguousarray(a)
        assert self.rt.hipMemcpy(ctypes.c_void_p(dev), a.ctypes.data_as(ctypes.c_void_p),
                                 ctypes.c_size_t(a.nbytes), 1) == 0


@pytest.mark.parametrize("stream_out", [False, True])
def test_copies_are_complete_when_an_address_is_handed_out(stream_out):
    """Uploads and port writes under way when the address is asked for the first time:
    what another stream reads through it is the new rows, and what it writes through it
    stays.  Then the same with the address in hand, and with the stream in hand."""
    import llm_accel as L
    hidden, inter, pairs = 2048, 11008, 10
    rng = np.random.default_rng(11 + stream_out)
    mem = _Memory()
    with L.Accelerator(L.Shape(64, hidden, inter, 1, 16, 2, 64, 1e6), num_pairs=pairs) as acc:
        if stream_out:
            assert L.lib().llm_stream(acc._ctx)
        for p in range(1, pairs):
            for again in range(2):  # the first time the address leaves, then with it known
                acc.sync()
                rows = [_ints(rng, (8, hidden)) for _ in range(4)]
                for i in range(8):  # copies that the last one stands behind
                    acc.upload(0, rows[i % 3])
                acc.upload(p, rows[3])
                ptr = L.lib().llm_pair_device_ptr(acc._ctx, p)
                assert np.array_equal(mem.read(ptr, rows[3].size), rows[3].reshape(-1)), (p, again)
                acc.upload(p, rows[0])
                if not again:
                    ptr = L.lib().llm_pair_device_ptr(acc._ctx, p)
                mem.write(ptr, rows[1])
                assert np.array_equal(acc.download(p, 8), rows[1]), (p, again)
        n = 8 * inter
        for port in (L.PORT_IN, L.PORT_AUX, L.PORT_OUT):
            x, y = _ints(rng, n), _ints(rng, n)
            acc.sync()
            acc.port_write(port, y)
            acc.port_write(port, x)
            dev, _ = acc.port(port)
            assert np.array_equal(mem.read(dev, n), x), port
            acc.port_write(port, y)
            mem.write(dev, x)
            assert np.array_equal(acc.port_read(port, n), x), port


def test_first_writes_of_new_buffers():
    """Rows and ports written as the first thing that happens to their memory, which the
    allocation's fill with zeros must not overtake: large contexts, whose fills take long."""
    import llm_accel as L
    rng = np.random.default_rng(17)
    for _ in range(4):
        rows, port = _ints(rng, (8, 2048)), _ints(rng, 8 * 11008)
        with L.Accelerator(L.Shape(64, 2048, 11008, 1, 16, 2, 16384, 1e6), num_pairs=64) as acc:
            acc.upload(63, rows)
            acc.port_write(L.PORT_OUT, port)
            acc.sync()
            assert np.array_equal(acc.download(63, 8), rows)
            assert np.array_equal(acc.port_read(L.PORT_OUT, port.size), port)
