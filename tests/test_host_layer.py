"""Runs the C++ test driver of the host-side TFCC layer (tests/cpp/host_tests.cpp).  The CPU part
exercises Shape / Variable / View / FlexAllocator and the argument checks on a host-memory device;
the GPU part runs the reference's data / blas / quantization cases on the ROCm device."""
import os
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
DRIVER = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "host_tests")


def _sig(v):
    return 1 / (1 + np.exp(-v))


def write_named_test_data(path, seed=5):
    """An .npz named the way tfcc/test/python/createtestdata.py names the reference's test data
    ("<package>/<case>/<i>/<key>", "<package>/<case>/__count__"), holding LSTM-cell cases made with the formulas of
    tfcc/test/python/testcase/rnn/lstmcell.py:31-44 (forget bias 1) and dense-layer cases (matmul + bias), with the
    expectations formed in float64."""
    rng = np.random.default_rng(seed)
    u = lambda *s: rng.uniform(-1.0, 1.0, s).astype(np.float32)  # noqa: E731
    data = {}
    cases = [(1, 64, 64), (4, 300, 100), (3, 130, 511)]
    data["rnn/lstmcell/__count__"] = np.asarray([len(cases)], np.int32)
    for i, (batch, units, input_size) in enumerate(cases):
        inputs, kernel, bias, h, cs = u(batch, input_size), u(input_size + units, units * 4), u(units * 4), \
            u(batch, units), u(batch, units)
        xh = np.concatenate((inputs, h), axis=1).astype(np.float64) @ kernel.astype(np.float64) + bias
        gi, ci, f, o = np.split(xh, 4, axis=1)
        next_cs = np.tanh(ci) * _sig(gi) + cs * _sig(f + 1)
        expect = np.tanh(next_cs) * _sig(o)
        prefix = "rnn/lstmcell/%d/" % i
        data.update({prefix + "units": np.asarray([units], np.int32), prefix + "inputs": inputs, prefix + "h": h,
                     prefix + "cs": cs, prefix + "lstm_cell/kernel": kernel, prefix + "lstm_cell/bias": bias,
                     prefix + "ecs": next_cs.astype(np.float32), prefix + "expect": expect.astype(np.float32)})
    # tfcc/test/python/testcase/rnn/grucell.py:31-56 and pytorchgrucell.py:24-60
    cases = [(1, 64, 64), (4, 130, 75), (9, 96, 200)]
    data["rnn/grucell/__count__"] = np.asarray([len(cases)], np.int32)
    data["rnn/pytorch_grucell/__count__"] = np.asarray([len(cases)], np.int32)
    for i, (batch, units, input_size) in enumerate(cases):
        inputs, state = u(batch, input_size), u(batch, units)
        g_kernel, g_bias = u(input_size + units, units * 2), u(units * 2)
        c_kernel, c_bias = u(input_size + units, units), u(units)
        value = _sig(np.concatenate((inputs, state), axis=1).astype(np.float64) @ g_kernel + g_bias)
        r, upd = np.split(value, 2, axis=1)
        cand = np.tanh(np.concatenate((inputs, r * state), axis=1) @ c_kernel.astype(np.float64) + c_bias)
        prefix = "rnn/grucell/%d/" % i
        data.update({prefix + "units": np.asarray([units], np.int32), prefix + "inputs": inputs, prefix + "state": state,
                     prefix + "gru_cell/gates/kernel": g_kernel, prefix + "gru_cell/gates/bias": g_bias,
                     prefix + "gru_cell/candidate/kernel": c_kernel, prefix + "gru_cell/candidate/bias": c_bias,
                     prefix + "expect": (upd * state + (1 - upd) * cand).astype(np.float32)})
        ci_kernel, ci_bias, ch_kernel, ch_bias = u(input_size, units), u(units), u(units, units), u(units)
        r, z = value[:, :units], value[:, units:]
        ni = inputs.astype(np.float64) @ ci_kernel + ci_bias
        nh = state.astype(np.float64) @ ch_kernel + ch_bias
        n = np.tanh(ni + r * nh)
        prefix = "rnn/pytorch_grucell/%d/" % i
        data.update({prefix + "units": np.asarray([units], np.int32), prefix + "inputs": inputs, prefix + "state": state,
                     prefix + "gru_cell/weight_gates": g_kernel, prefix + "gru_cell/bias_gates": g_bias,
                     prefix + "gru_cell/weight_candidate_i": ci_kernel, prefix + "gru_cell/bias_candidate_i": ci_bias,
                     prefix + "gru_cell/weight_candidate_h": ch_kernel, prefix + "gru_cell/bias_candidate_h": ch_bias,
                     prefix + "expect": (n + z * (state - n)).astype(np.float32)})
    cases = [((5, 70), 33), ((2, 3, 768), 3072), ((1, 512), 2048), ((2, 2, 9, 40), 17)]
    data["layer/dense/__count__"] = np.asarray([len(cases)], np.int32)
    for i, (shape, units) in enumerate(cases):
        inputs, kernel, bias, w, b = u(*shape), u(shape[-1], units), u(units), u(shape[-1], units), u(units)
        prefix = "layer/dense/%d/" % i
        x64 = inputs.astype(np.float64)
        data.update({prefix + "units": np.asarray([units], np.int32), prefix + "inputs": inputs,
                     prefix + "dense/kernel": kernel, prefix + "dense/bias": bias, prefix + "other/w": w,
                     prefix + "other/b": b, prefix + "expect": (x64 @ kernel + bias).astype(np.float32),
                     prefix + "expect_nobias": (x64 @ kernel).astype(np.float32),
                     prefix + "expect_other": (x64 @ w + b).astype(np.float32)})
    np.savez(path, **data)


def _run(mode, data=None):
    if not os.path.exists(DRIVER):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "csrc")])
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host")])
    res = subprocess.run([DRIVER, mode] + ([data] if data else []), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=300)
    print(res.stdout)
    assert res.returncode == 0, res.stdout[-4000:]
    assert "0 failures" in res.stdout


def test_host_layer_framework_cpu(tmp_path):
    write_named_test_data(str(tmp_path / "named.npz"))
    _run("cpu", str(tmp_path / "named.npz"))


@pytest.mark.gpu
def test_host_layer_gpu(tmp_path):
    write_named_test_data(str(tmp_path / "named.npz"))
    _run("gpu", str(tmp_path / "named.npz"))


def test_copy_offsets_stay_inside_their_operands():
    """The HBM -> LDS copies that carry a slab's offset in the unchecked scalar offset: every (lane offset, scalar
    offset) pair the int8 256 x 256 kernel and the fp32 one-wavefront-per-SIMD kernel can issue on ragged shapes,
    enumerated on the host with the kernels' own offset functions (tests/cpp/copy_offset_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "copy_offset_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/copy_offset_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "copy offsets ok" in res.stdout, res.stdout[-2000:]


def test_gemv_workspace_bookkeeping():
    """Per-stream workspaces of the skinny quantized matmul: kept across calls, never freed while a recorded launch
    may use them, no growth while allocation is not allowed, cleared after a failed launch, released per stream
    (tests/cpp/gemv_workspace_tests.cpp with a counting allocator)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "gemv_workspace_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/gemv_workspace_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "bookkeeping ok" in res.stdout, res.stdout[-2000:]


def test_how_the_k_of_skinny_quantized_products_is_dealt_out():
    """A launch without a workspace keeps a short K in one part (tests/cpp/gemv_wide_plan_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "gemv_wide_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/gemv_wide_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_lstm_sequences_that_do_not_fit_on_the_gpu_are_left_to_the_steps():
    """A GPU with fewer CUs than the launch has workgroups: no workspace, so no launch (tests/cpp/lstm_plan_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "lstm_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/lstm_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_how_the_k_of_fp32_products_is_dealt_out():
    """The limits of the plan, the memory in which splits meet among them (tests/cpp/sgemm_deal_plan_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "sgemm_deal_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/sgemm_deal_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_which_fp32_products_share_a_k():
    """The limits of the rule, and that the plan of the other kernel is worked out once (tests/cpp/sgemm_skinny_plan_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "sgemm_skinny_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/sgemm_skinny_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_which_fp32_products_run_on_the_bf16_matrix_cores():
    """The limits of the rule, and that B given transposed goes where B as stored goes (tests/cpp/sgemm_split_plan_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "sgemm_split_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/sgemm_split_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_which_small_quantized_products_are_shared():
    """The limits of the rule (tests/cpp/qgemm_small_plan_tests.cpp): both sides of its line as measured, and that the memory the
    workgroups meet in is large enough for whatever they share."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "qgemm_small_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/qgemm_small_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_words_of_the_one_launch_quantize():
    """No word of an earlier call, and none that nobody has written, is taken for this call's (tests/cpp/quantize_exchange_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "quantize_exchange_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/quantize_exchange_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_where_uploads_are_cut():
    """Every piece begins on a line, whatever the sizes of the inputs in front of it (tests/cpp/upload_cut_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "upload_cut_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/upload_cut_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]


def test_which_attention_kernel_takes_a_call():
    """Both sides of the rule's lines, and no more threads than a launch may have (tests/cpp/attention_plan_tests.cpp)."""
    exe = os.path.join(ROOT, "wechat-tfcc_amd", "host", "build", "attention_plan_tests")
    if not os.path.exists(exe):
        subprocess.check_call(["make", "-C", os.path.join(ROOT, "wechat-tfcc_amd", "host"), "build/attention_plan_tests"])
    res = subprocess.run([exe], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
    assert res.returncode == 0 and "all passed" in res.stdout, res.stdout[-2000:]
