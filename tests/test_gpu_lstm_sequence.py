"""A whole LSTM sequence in one launch (tfcc_rocm_lstm_sequence_f32) against the oracle's recurrence: every configuration of
the kernel at the edges of its range of units and rows, one and two directions, on several streams at once, and with a
wait that is over at once, so that the launch behind it computes the sequence."""
import ctypes as C
import threading

import numpy as np
import pytest

import oracle_lib as O
from conftest import rel_fro

pytestmark = pytest.mark.gpu


def setup(T, seq, batch, length, hidden, directions, seed=0):
    rng = np.random.default_rng(seq * 100 + batch * 10 + hidden + seed)
    u = lambda *s: (rng.uniform(-1, 1, s) / np.sqrt(hidden)).astype(np.float32)
    x = rng.standard_normal((seq, batch, length)).astype(np.float32)
    sets = [dict(ik=u(length, 4 * hidden), sk=u(hidden, 4 * hidden), bias=u(4 * hidden), ih=u(batch, hidden), ic=u(batch, hidden))
            for _ in range(directions)]
    return x, sets


def launch(pkg, T, x, sets, backward, wait_us=20000, stream=None, spread=False):
    import torch
    seq, batch, _ = x.shape
    hidden = sets[0]["ih"].shape[1]
    d = pkg.LstmSequenceDesc()
    d.seq, d.batch, d.units, d.directions, d.forget, d.wait_us = seq, batch, hidden, len(sets), 0.0, wait_us
    need = pkg.lib().tfcc_rocm_lstm_sequence_workspace(batch, hidden, len(sets))
    keep = [torch.randint(0, 255, (need,), dtype=torch.uint8, device="cuda")]  # no particular contents
    d.workspace, d.workspace_bytes = keep[0].data_ptr(), need
    outs = []
    for i, s in enumerate(sets):
        dev = {k: T.t(v) for k, v in s.items()}
        values = pkg.blas_matmul(T.t(x.reshape(seq * batch, -1)), dev["ik"])
        out, h, c = torch.empty((seq, batch, hidden), device="cuda"), torch.empty((batch, hidden), device="cuda"), torch.empty((batch, hidden), device="cuda")
        keep += [dev, values]
        d.x[i], d.kernel[i], d.bias[i], d.h0[i], d.c0[i] = (t.data_ptr() for t in (values, dev["sk"], dev["bias"], dev["ih"], dev["ic"]))
        d.out[i], d.h[i], d.c[i], d.backward[i] = out.data_ptr(), h.data_ptr(), c.data_ptr(), int(backward[i])
        outs.append((out, h, c))
    torch.cuda.synchronize()
    call = pkg.lib().tfcc_rocm_lstm_sequence_f32_spread if spread else pkg.lib().tfcc_rocm_lstm_sequence_f32
    pkg.check(call(stream, C.byref(d)))
    return outs, keep


def gave_up(T, keep):
    """the word by which the workgroups tell the launch behind them to compute the sequence"""
    return int(T.n(keep[0])[-64:-60].view(np.uint32)[0])


def compare(T, outs, x, sets, backward):
    for (out, h, c), s, back in zip(outs, sets, backward):
        want = O.lstm_sequence(x, s["ik"], s["sk"], s["bias"], s["ih"], s["ic"], back)
        for got, w in zip((out, h, c), want):
            assert rel_fro(T.n(got), w.astype(np.float64)) <= 1e-5


@pytest.mark.parametrize("seq,batch,hidden,directions", [
    (1, 1, 1, 1), (2, 1, 3, 2), (3, 2, 255, 2), (4, 3, 256, 2), (5, 4, 257, 2), (3, 5, 511, 1), (4, 8, 512, 2),   # rows 1 to 16, units
    (3, 9, 513, 2), (3, 12, 700, 1), (3, 13, 1023, 2), (4, 16, 1024, 2), (64, 4, 512, 2), (7, 16, 200, 2), (9, 1, 1000, 2)])
def test_sequence_against_the_oracle(pkg, T, seq, batch, hidden, directions):
    print("lstm sequence", seq, batch, hidden, directions, flush=True)
    x, sets = setup(T, seq, batch, 40, hidden, directions)
    backward = (False, True)[:directions]
    outs, keep = launch(pkg, T, x, sets, backward)
    compare(T, outs, x, sets, backward)
    assert gave_up(T, keep) == 0
    again, keep2 = launch(pkg, T, x, sets, backward)
    assert gave_up(T, keep2) == 0
    for a, b in zip(outs, again):
        for p, q in zip(a, b):
            assert np.array_equal(T.n(p), T.n(q))


@pytest.mark.parametrize("seq,batch,hidden,directions", [
    (1, 4, 256, 2), (2, 5, 257, 2), (3, 7, 512, 2), (4, 9, 513, 2), (5, 13, 768, 2), (6, 16, 767, 1), (9, 15, 249, 2),
    (11, 8, 505, 1), (8, 9, 769, 1), (13, 11, 745, 2), (7, 1, 768, 1), (10, 10, 8, 1)])
def test_rows_dealt_out_to_xcds(pkg, T, seq, batch, hidden, directions):
    """up to 768 units: one to four rows to an XCD with fewer in the last group, units that do not fill a workgroup or a
    lane's four k, sequences around the four steps whose inputs are fetched together; twice, with the same bits"""
    print("lstm rows", seq, batch, hidden, directions, flush=True)
    x, sets = setup(T, seq, batch, 24, hidden, directions)
    backward = (True, False)[:directions]
    outs, keep = launch(pkg, T, x, sets, backward)
    compare(T, outs, x, sets, backward)
    assert gave_up(T, keep) == 0
    again, keep = launch(pkg, T, x, sets, backward)
    for a, b in zip(outs, again):
        for p, q in zip(a, b):
            assert np.array_equal(T.n(p), T.n(q))


@pytest.mark.parametrize("seq,batch,hidden,directions", [
    (1, 4, 256, 2), (2, 5, 257, 2), (3, 7, 512, 2), (9, 13, 768, 2), (6, 16, 767, 1), (40, 15, 249, 2), (11, 1, 65, 1)])
def test_rows_whose_workgroups_share_no_xcd(pkg, T, seq, batch, hidden, directions):
    """The workgroups of a group side by side, so on all XCDs: they find that out from the first step's words, and h goes through
    memory from then on.  The same bits as with a group on one XCD, and not by way of the launch behind."""
    print("lstm spread", seq, batch, hidden, directions, flush=True)
    x, sets = setup(T, seq, batch, 24, hidden, directions)
    backward = (True, False)[:directions]
    outs, keep = launch(pkg, T, x, sets, backward, spread=True)
    compare(T, outs, x, sets, backward)
    assert gave_up(T, keep) == 0
    together, keep = launch(pkg, T, x, sets, backward)
    assert gave_up(T, keep) == 0
    for a, b in zip(outs, together):
        for p, q in zip(a, b):
            assert np.array_equal(T.n(p), T.n(q))


@pytest.mark.parametrize("seq,batch,hidden", [(5, 3, 96), (4, 12, 600), (1, 1, 5), (3, 16, 1024)])
def test_a_wait_that_is_over_at_once(pkg, T, seq, batch, hidden):
    x, sets = setup(T, seq, batch, 24, hidden, 2)
    outs, keep = launch(pkg, T, x, sets, (False, True), wait_us=0)
    compare(T, outs, x, sets, (False, True))
    assert gave_up(T, keep) == 1


def test_limits(pkg, T):
    lib = pkg.lib()
    assert lib.tfcc_rocm_lstm_sequence_workspace(17, 64, 2) == 0 and lib.tfcc_rocm_lstm_sequence_workspace(1, 1025, 2) == 0
    d = pkg.LstmSequenceDesc()
    d.seq, d.batch, d.units, d.directions = 1, 1, 8, 1
    assert lib.tfcc_rocm_lstm_sequence_f32(None, C.byref(d)) == 1


def test_several_threads_and_streams(pkg, T):
    import torch
    x, sets = setup(T, 20, 4, 32, 512, 2)
    errors = []

    def work():
        try:
            for _ in range(5):
                stream = torch.cuda.Stream()
                outs, keep = launch(pkg, T, x, sets, (False, True), stream=stream.cuda_stream)
                torch.cuda.synchronize()
                compare(T, outs, x, sets, (False, True))
                pkg.check(pkg.lib().tfcc_rocm_stream_release(stream.cuda_stream))
        except BaseException as e:  # noqa: B036
            errors.append(e)

    threads = [threading.Thread(target=work) for _ in range(3)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors


def test_beside_a_capture_after_the_null_stream(pkg, T):
    """The null stream may not be asked, waited for or recorded on while a graph is being recorded elsewhere."""
    import torch
    x, sets = setup(T, 6, 3, 16, 300, 2)
    lib, prepared = pkg.lib(), []

    class Held:  # launch() up to the call itself, which comes while the graph is being recorded
        def __getattr__(self, name):
            return (lambda stream, d: prepared.append(d) or 0) if name == "tfcc_rocm_lstm_sequence_f32" else getattr(lib, name)

    class Package:
        LstmSequenceDesc, blas_matmul, check, lib = pkg.LstmSequenceDesc, staticmethod(pkg.blas_matmul), staticmethod(pkg.check), staticmethod(Held)

    runs = [launch(Package, T, x, sets, (False, True)) for _ in range(4)]
    call, recorded, other, graph = lib.tfcc_rocm_lstm_sequence_f32, C.c_void_p(), C.c_void_p(), C.c_void_p()
    for stream in (recorded, other):
        pkg.check(lib.tfcc_rocm_stream_create(C.byref(stream)))
    status = [call(other, prepared[0]), call(None, prepared[1])]  # the null stream had the last turn
    torch.cuda.synchronize()
    t = torch.zeros(64, dtype=torch.uint8, device="cuda")
    torch.cuda.synchronize()
    pkg.check(lib.tfcc_rocm_stream_begin_capture(recorded))  # of a stream that the null stream waits for
    pkg.check(lib.tfcc_rocm_fill_async(recorded, t.data_ptr(), 7, 1, 64))
    status.append(call(other, prepared[2]))
    pkg.check(lib.tfcc_rocm_stream_end_capture(recorded, C.byref(graph)))
    torch.cuda.synchronize()
    status.append(call(None, prepared[3]))
    pkg.check(lib.tfcc_rocm_graph_launch(graph, recorded))
    torch.cuda.synchronize()
    assert (t == 7).all()
    pkg.check(lib.tfcc_rocm_graph_destroy(graph))
    for stream in (recorded, other):
        pkg.check(lib.tfcc_rocm_stream_destroy(stream))
    assert status == [0, 0, 0, 0], lib.tfcc_rocm_last_error_string()
    for outs, keep in runs:
        compare(T, outs, x, sets, (False, True))


def test_after_a_stream_that_is_gone(pkg, T):
    import torch
    hip = C.CDLL("libamdhip64.so")
    x, sets = setup(T, 5, 2, 16, 128, 2)
    for _ in range(3):
        raw = C.c_void_p()
        assert hip.hipStreamCreate(C.byref(raw)) == 0
        outs, keep = launch(pkg, T, x, sets, (False, True), stream=raw)
        assert hip.hipStreamSynchronize(raw) == 0 and hip.hipStreamDestroy(raw) == 0  # not through the library
        compare(T, outs, x, sets, (False, True))
        outs, keep = launch(pkg, T, x, sets, (False, True))
        torch.cuda.synchronize()
        compare(T, outs, x, sets, (False, True))


@pytest.mark.parametrize("function,low,high", [("tanh", -0.65, 0.65), ("tanh", 0.5, 0.8), ("tanh", -4.0, 4.0), ("tanh", -12.0, 12.0), ("sigmoid", -1.0, 1.0),
                                               ("sigmoid", -4.0, 4.0), ("sigmoid", 0.0, 20.0), ("sigmoid", -20.0, -4.0), ("sigmoid", -87.0, 0.0)])
def test_functions_of_the_cell(pkg, T, function, low, high):
    """One step with a state kernel of zeros leaves tanh(x) (gates i open, f shut) or sigmoid(x) (c gate 0, state 1) in c.  No
    further from float64 than the step kernel with the library's functions, which the reference's formulas call."""
    import torch
    lib, batch, units = pkg.lib(), 16, 1024
    v = np.random.default_rng(int(abs(high) * 8 + abs(low))).uniform(low, high, (batch, units)).astype(np.float32)
    x = np.zeros((batch, 4, units), np.float32)
    x[:, 0], x[:, 3] = 40.0, 40.0
    x[:, 1], x[:, 2] = (v, -200.0) if function == "tanh" else (0.0, v)
    t = {k: T.t(a) for k, a in dict(x=x.reshape(batch, -1), kernel=np.zeros((units, 4 * units), np.float32), bias=np.zeros(4 * units, np.float32),
                                    h0=np.zeros((batch, units), np.float32), h=np.zeros((batch, 4 * units), np.float32),
                                    c0=np.full((batch, units), 0.0 if function == "tanh" else 1.0, np.float32)).items()}
    got, library, h, out = (torch.empty((batch, units), device="cuda") for _ in range(4))
    d = pkg.LstmSequenceDesc()
    d.seq, d.batch, d.units, d.directions, d.wait_us = 1, batch, units, 1, 20000
    need = lib.tfcc_rocm_lstm_sequence_workspace(batch, units, 1)
    workspace = torch.empty(need, dtype=torch.uint8, device="cuda")
    d.workspace, d.workspace_bytes = workspace.data_ptr(), need
    d.x[0], d.kernel[0], d.bias[0], d.h0[0], d.c0[0] = (t[k].data_ptr() for k in ("x", "kernel", "bias", "h0", "c0"))
    d.out[0], d.h[0], d.c[0] = out.data_ptr(), h.data_ptr(), got.data_ptr()
    pkg.check(lib.tfcc_rocm_lstm_sequence_f32(None, C.byref(d)))
    pkg.check(lib.tfcc_rocm_lstm_cell_f32(None, batch, units, t["c0"].data_ptr(), t["x"].data_ptr(), t["h"].data_ptr(), t["bias"].data_ptr(), 0.0,
                                          h.data_ptr(), library.data_ptr()))
    wide = v.astype(np.float64)
    want = np.tanh(wide) if function == "tanh" else 1.0 / (1.0 + np.exp(-wide))
    unit = np.spacing(np.abs(want).astype(np.float32)).astype(np.float64)
    ours, theirs = (np.abs(T.n(r).astype(np.float64) - want) / unit for r in (got, library))
    print(function, low, high, "largest %.3f mean %.4f, library %.3f %.4f" % (ours.max(), ours.mean(), theirs.max(), theirs.mean()))
    # (a hundredth for what the choice of inputs does to a mean, a tenth for the largest of 16384)
    assert ours.max() <= theirs.max() + 0.1 and ours.mean() <= theirs.mean() + 0.01


@pytest.mark.parametrize("seq,batch,hidden", [(9, 2, 257), (11, 6, 510), (10, 12, 512), (9, 12, 1024), (13, 5, 601), (70, 4, 514)])
def test_words_without_a_number(pkg, T, seq, batch, hidden):
    """more than 256 units: the four sets of words in turn, and values that look like a word nobody has written"""
    x, sets = setup(T, seq, batch, 40, hidden, 2)
    outs, keep = launch(pkg, T, x, sets, (False, True))
    compare(T, outs, x, sets, (False, True))
    assert gave_up(T, keep) == 0
    sets[0]["ih"].view(np.uint32)[-1, :] = 0xffffffff
    outs, keep = launch(pkg, T, x, sets, (False, True))
    assert gave_up(T, keep) == 0
    assert np.isnan(T.n(outs[0][0])[:, -1]).all()
    want = O.lstm_sequence(x[:, :-1], sets[0]["ik"], sets[0]["sk"], sets[0]["bias"], sets[0]["ih"][:-1], sets[0]["ic"][:-1], False)
    for got, w in zip(outs[0], want):
        assert rel_fro(T.n(got)[..., :-1, :], w.astype(np.float64)) <= 1e-5
