"""Model.run on numpy arrays: what it takes and returns equals the message form (run_serialized), at the sizes where its
transfers change course, and its outputs stay valid for as long as they are held."""
import collections
import gc
import importlib
import types

import numpy as np
import pytest

NP = [np.float32, np.float64, np.int8, np.uint8, np.int16, np.uint16, np.int32, np.uint32, np.int64, np.uint64]


@pytest.fixture(scope="module")
def mf(pkg):
    return importlib.import_module("wechat_tfcc_amd.modelfile")


@pytest.fixture(scope="module")
def rt(pkg):
    return importlib.import_module("wechat_tfcc_amd.runtime_api")


def copies(mf, rt, specs, host):
    """a model that hands its inputs back: specs = [(dtype code, shape)]"""
    g = mf.GraphBuilder("copies")
    for i, (dtype, shape) in enumerate(specs):
        x = g.input("x%d" % i, dtype, list(shape))
        y = g._symbol("y%d" % i, dtype, mf.VARIABLE, list(shape))
        g.node("base.Identity", [x], [y])
        g.output(y)
    return rt.Model(mf.write_model([g], g.name), host=host)


def values(rng, dtype, shape):
    if np.dtype(dtype).kind == "f":
        return rng.standard_normal(shape).astype(dtype)
    info = np.iinfo(dtype)
    return rng.integers(info.min, info.max, shape, dtype=dtype, endpoint=True)


def round_trip(mf, rt, shapes, host):
    rng = np.random.default_rng(len(shapes))
    specs = [(mf.DTYPE_OF[np.dtype(NP[i % len(NP)])], s) for i, s in enumerate(shapes)]
    model = copies(mf, rt, specs, host)
    inputs = {"x%d" % i: values(rng, NP[i % len(NP)], s) for i, s in enumerate(shapes)}
    out = model.run(inputs)
    message = mf.decode_outputs(model.run_serialized(mf.encode_inputs(inputs)))
    assert list(out) == list(message) == ["y%d" % i for i in range(len(shapes))]
    for i in range(len(shapes)):
        got = out["y%d" % i]
        assert got.dtype == inputs["x%d" % i].dtype and got.flags.writeable and got.flags.c_contiguous
        assert np.array_equal(got, inputs["x%d" % i]) and np.array_equal(message["y%d" % i], got)


def test_every_type_on_the_host_device(mf, rt):
    round_trip(mf, rt, [(3,), (2, 3), (1,), (5,), (7, 1), (2, 2, 2), (9,), (4,), (3, 3), (2,)], True)


def test_what_is_not_an_input_raises(mf, rt):
    model = copies(mf, rt, [(mf.FLOAT, (2, 2))], True)
    with pytest.raises(KeyError):
        model.run({"x0": np.zeros((2, 2), np.float16)})
    with pytest.raises(KeyError):
        model.run({"x0": np.zeros((2, 2), ">f4")})
    with pytest.raises(rt.RuntimeError_):
        model.run({"nobody": np.zeros((2, 2), np.float32)})
    with pytest.raises(rt.RuntimeError_):
        model.run({"x0\0": np.zeros((2, 2), np.float32)})
    with pytest.raises(rt.RuntimeError_, match="type not match"):
        model.run({"x0": np.zeros((2, 2), np.float64)})
    view = np.arange(8, dtype=np.float32).reshape(4, 2)[::2]  # not contiguous
    assert np.array_equal(model.run({"x0": view})["y0"], view)


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [
    [(1,)], [(3,), (5,), (1,), (4093,)],                     # bytes that are no multiple of 16
    [(4096,)], [(4097,)],                                    # one workgroup's 16 KB, and one element more
    [(65536,)], [(65537,)],                                  # the first staged chunk of 256 KB
    [((8 << 20) // 4 + 77,)], [(1 << 20,), (1 << 19,), (777,)],  # more than the staging block holds
    [(i + 1,) for i in range(17)],                           # more pieces than one launch takes
])
def test_sizes_where_the_transfers_change(mf, rt, dev, shapes):
    round_trip(mf, rt, shapes, False)


@pytest.mark.gpu
@pytest.mark.parametrize("shapes", [
    [(1023,)], [(1024,), (1025,)],                                     # one workgroup's 4 KB
    [((384 << 10) // 4,)], [((384 << 10) // 4 + 1,)],                  # up to here in, which is the first chunk, and a float more
    [(77,), ((384 << 10) // 4,), ((768 << 10) // 4 + 3,), (5,)],       # chunks that end inside an input and hold the next
    [((1536 << 10) // 4,)], [((1536 << 10) // 4 - 8,), (9,)],          # and out, in one piece and in two
])
def test_sizes_where_a_workgroup_takes_more(mf, rt, dev, shapes):
    round_trip(mf, rt, shapes, False)


def test_any_mapping_is_taken(mf, rt):
    model = copies(mf, rt, [(mf.FLOAT, (2,)), (mf.INT32, (3,))], True)
    want = {"x0": np.array([1, 2], np.float32), "x1": np.array([3, 4, 5], np.int32)}

    class Items:
        def items(self):
            return ([k, v] for k, v in want.items())

    for arrays in (want, collections.OrderedDict(want), types.MappingProxyType(want), collections.UserDict(want),
                   collections.ChainMap({"x0": want["x0"]}, {"x1": want["x1"]}), Items()):
        out = model.run(arrays)
        assert np.array_equal(out["y0"], want["x0"]) and np.array_equal(out["y1"], want["x1"])
    with pytest.raises(AttributeError):
        model.run([("x0", want["x0"])])

    class Pairs:
        def items(self):
            return [("x0",)]

    with pytest.raises(ValueError):
        model.run(Pairs())


def test_a_kept_output_does_not_hold_the_others(mf, rt):
    # a run hands out 64 MB beside three numbers; sixteen of the small ones together hold none of the large
    def resident():
        with open("/proc/self/statm") as f:
            return int(f.read().split()[1]) * 4096
    n = 16 << 20
    model = copies(mf, rt, [(mf.FLOAT, (n,)), (mf.FLOAT, (3,))], True)
    inputs = {"x0": np.ones(n, np.float32), "x1": np.arange(3, dtype=np.float32)}
    held = [model.run(inputs)["y1"]]
    before = resident()
    for _ in range(16):
        held.append(model.run(inputs)["y1"])
    assert resident() - before < 4 * inputs["x0"].nbytes
    model.close()
    assert all((h == [0, 1, 2]).all() for h in held)


@pytest.mark.gpu
def test_pinned_outputs_kept_alone_leave_the_bound_to_others(mf, rt, dev):
    # 40 MB beside three numbers: blocks of 64 MB, of which the process-wide bound admits four
    n = 10 << 20
    model = copies(mf, rt, [(mf.FLOAT, (n,)), (mf.FLOAT, (3,))], False)
    held = []
    for i in range(8):
        out = model.run({"x0": np.full(n, i, np.float32), "x1": np.full(3, i, np.float32)})
        assert (out["y0"] == i).all()
        held.append(out["y1"])
    assert all((h == i).all() for i, h in enumerate(held))


@pytest.mark.gpu
def test_outputs_outlive_the_model_and_later_runs(mf, rt, dev):
    # 9 MB each: blocks of 16 MB, of which the process-wide bound admits sixteen; the runs beyond it get ordinary memory
    n = (9 << 20) // 4
    model = copies(mf, rt, [(mf.FLOAT, (n,))], False)
    held = []
    for i in range(20):
        held.append(model.run({"x0": np.full(n, i, np.float32)})["y0"])
    model.close()
    for i, y in enumerate(held):
        assert (y == i).all()
    del held
    gc.collect()
