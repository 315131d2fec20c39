"""The builtin functions that hand torch tensors to the operators (diopi_amd/csrc/rt/torch_binding.cpp): what they refuse, and
that calls without a context keep the order of torch's current stream, whatever the thread, stream or graph."""
import os
import subprocess
import sys
import threading

import pytest
import torch

from diopi_amd import functions as F
from diopi_amd import runtime as rt
from diopi_amd import workloads as W
from tests.helpers import assert_bit_equal

DEV = "cuda"


def test_arguments_that_are_no_tensors_of_a_known_type():
    ops = rt.torch_ops()
    assert all(hasattr(ops, name) for name in rt.OPERATOR_SYMBOLS)
    x, w = torch.ones(2, 4), torch.ones(4)
    with pytest.raises(TypeError, match="unsupported dtype"):
        F.rms_norm(x.to(torch.complex64), (4,), w, None, 1e-6)
    with pytest.raises(TypeError, match="torch.Tensor or None"):
        F.rms_norm(x, (4,), [1.0] * 4, None, 1e-6)
    with pytest.raises(TypeError, match="expected 8 arguments"):
        ops.diopiRMSNorm(None, x)
    with pytest.raises(rt.DiopiException, match="device memory"):  # a host tensor, no stream asked for
        F.rms_norm(x, (4,), w, None, 1e-6)
    with pytest.raises(rt.DiopiException, match="null handle"):
        F.rms_norm_backward([None], x, w, None, (4,), 1e-6, inv_rms=torch.ones(2))
    with pytest.raises(rt.DiopiException, match="rank 9"):
        F.destindex_copy_kv(torch.ones([1] * 9), torch.zeros(1, dtype=torch.int32), torch.ones([1] * 9))


def test_a_closed_context_is_refused():
    ctx = rt.Context(own_stream=True)
    ctx.close()
    with pytest.raises(rt.DiopiException):
        F.rms_norm(torch.ones(2, 4), (4,), torch.ones(4), None, 1e-6, ctx=ctx)


def test_a_build_of_the_c_libraries_alone(tmp_path):
    for path in (rt.RT_LIB_PATH, rt.IMPL_LIB_PATH):
        os.symlink(path, tmp_path / os.path.basename(path))
    code = ("import torch; from diopi_amd import functions as F, runtime as rt\n"
            "try: F.rms_norm(torch.ones(2, 4), (4,), torch.ones(4), None, 1e-6)\n"
            "except rt.DiopiException as e: print(e)")
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", code], cwd=root, env=dict(os.environ, DIOPI_AMD_LIB_DIR=str(tmp_path)), capture_output=True, text=True, timeout=100)
    assert "device memory" in res.stdout, res.stderr[-2000:]


def test_the_c_libraries_are_made_without_python(tmp_path):
    """`make all` asks for nothing that needs torch's headers or Python's."""
    csrc = os.path.join(os.path.dirname(os.path.abspath(rt.__file__)), "csrc")
    res = subprocess.run(["make", "-C", csrc, "-n", "-B", "all"], capture_output=True, text=True, timeout=100)
    assert res.returncode == 0 and "libdiopi_impl.so" in res.stdout
    assert "torch" not in res.stdout and "python" not in res.stdout.lower()


def _step(w, x, go, weight):
    """Three operators that take scratch, without a context."""
    inv = torch.rsqrt((x * x).mean(-1) + 1e-6)
    grads = F.rms_norm_backward([go], x, weight, None, (x.shape[1],), 1e-6, inv_rms=inv)
    logits = torch.zeros(w["H"], w["total_len"], dtype=w["dtype"], device=DEV)
    F.token_attention(w["q"], w["k_cache"], logits, w["b_loc"], w["b_start_loc"], w["b_seq_len"], w["max_input_len"])
    out = torch.zeros_like(w["q"])
    F.token_softmax_reducev(logits, w["v_cache"], out, w["b_loc"], w["b_start_loc"], w["b_seq_len"], w["max_input_len"], 0)
    return grads["input"], grads["weight"], logits, out


def _inputs(seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    w = W._decode(DEV, seed, torch.float16, 3, 8, 2, 128, 16000, 2500, 5000, 3)  # ranges of several work-groups: partial sums in scratch
    return w, torch.randn(700, 512, device=DEV, generator=g), torch.randn(700, 512, device=DEV, generator=g), torch.rand(512, device=DEV, generator=g)


@pytest.mark.gpu
def test_calls_without_a_context_from_two_threads_on_their_own_streams():
    inputs = [_inputs(21), _inputs(22)]
    want = [[t.clone() for t in _step(*i)] for i in inputs]
    torch.cuda.synchronize()
    got, errors = [None, None], []

    def worker(n):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(10):
                    got[n] = _step(*inputs[n])
                torch.cuda.current_stream().synchronize()
        except Exception as e:  # surfaced in the main thread
            errors.append(e)

    threads = [threading.Thread(target=worker, args=(n,)) for n in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for n in range(2):
        for a, b, name in zip(got[n], want[n], ("grad_input", "grad_weight", "logits", "decode out")):
            assert_bit_equal(a, b, f"thread {n}: {name}")


@pytest.mark.gpu
def test_calls_without_a_context_in_a_hip_graph():
    args = _inputs(23)
    _step(*args)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        held = _step(*args)
    g = torch.Generator(device=DEV).manual_seed(24)
    for replay in range(3):
        args[0]["q"].copy_(torch.randn(args[0]["q"].shape, device=DEV, generator=g))
        args[1].copy_(torch.randn(args[1].shape, device=DEV, generator=g))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        got = [t.clone() for t in held]
        want = _step(*args)
        for a, b, name in zip(got, want, ("grad_input", "grad_weight", "logits", "decode out")):
            assert_bit_equal(a, b, f"replay {replay}: {name}")


@pytest.mark.gpu
def test_context_on_torchs_default_stream():
    """Its handle is null: the operator still runs behind what torch has queued there, and torch behind the operator."""
    ctx = rt.Context(stream=torch.cuda.default_stream())
    a = torch.randn(4096, 4096, device=DEV)
    cache, dest = torch.zeros(4, 1, 64, device=DEV), torch.tensor([1], dtype=torch.int32, device=DEV)
    row = torch.zeros(1, 1, 64, device=DEV)
    torch.cuda.synchronize()
    for n in range(1, 6):
        for _ in range(20):  # some milliseconds of work in front of the row that the operator reads
            a = a @ a * 1e-2
        row.copy_((a[:1, :64] * 0 + n).view(1, 1, 64))
        F.destindex_copy_kv(row, dest, cache, ctx=ctx)
        seen = cache.clone()
        assert float(seen[1, 0, 0]) == n and float(seen[1, 0, 63]) == n
    ctx.close()


def _long_call():
    """Attention that takes milliseconds, without a context."""
    q = torch.randn(1, 8192, 16, 128, device=DEV).half()
    F.flash_attention(q, q, q, None, 0.0, None, False)
    torch.cuda.synchronize()
    return lambda: F.flash_attention(q, q, q, None, 0.0, None, False)


@pytest.mark.gpu
def test_the_default_context_stands_for_calls_without_a_context():
    ctx, call = rt.default_context(), _long_call()
    torch_events, events = [torch.cuda.Event(enable_timing=True) for _ in range(2)], [rt.Event() for _ in range(2)]
    torch_events[0].record()
    events[0].record(ctx)
    for _ in range(5):
        call()
    events[1].record(ctx)
    torch_events[1].record()
    torch.cuda.synchronize()
    whole = torch_events[0].elapsed_time(torch_events[1])
    assert 0.5 * whole <= events[0].elapsed_ms(events[1]) <= 1.01 * whole + 0.1, whole  # host gaps are on both sides
    # calls on another stream, waited for outside of it
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        for _ in range(20):
            call()
    assert not stream.query()  # tens of milliseconds of work
    ctx.synchronize()
    assert stream.query()
    # their scratch: partial sums of two ranges for three sequences and eight heads of 128
    _step(*_inputs(25))
    assert ctx.scratch_peak >= 3 * 2 * 8 * 130 * 4


@pytest.mark.gpu
def test_the_ctypes_route_gives_the_same(monkeypatch):
    args = _inputs(26)
    want = _step(*args)
    x = torch.randn(300, 4, 64, device=DEV).half()
    cu = torch.tensor([0, 100, 300], dtype=torch.int32, device=DEV)
    attend = lambda: (F.flash_attention_varlen(x, x, x, cu, cu, None, 200, 200, 0.0, None, True), F.GLOBAL_STATE["flash_attention_varlen_softmax_lse"])
    hidden, weight = torch.randn(2, 256, device=DEV).half(), torch.randn(256, 768, device=DEV).half() * 0.05
    caches, lens = [torch.zeros(1, 2, 2, 33, 128, device=DEV).half() for _ in range(2)], torch.tensor([3, 9], dtype=torch.int32, device=DEV)
    fused = lambda: F.fused_decoder_attention_inp(hidden.clone(), weight, None, None, 0, *caches, None, 32 - lens, lens, 33, 0, 2, 2, 128, 33, 128, 10000.0)
    want += attend() + (fused(),)
    torch.cuda.synchronize()
    monkeypatch.setattr(rt, "_torch_ops", rt._CtypesOps())
    for n, (a, b) in enumerate(zip(_step(*args) + attend() + (fused(),), want)):
        assert_bit_equal(a, b, f"output {n}")
