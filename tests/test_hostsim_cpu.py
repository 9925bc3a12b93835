"""The library's host runtime and the benchmark's drivers on the CPU, under AddressSanitizer and
UndefinedBehaviorSanitizer, against a host-memory simulation of the HIP runtime
(tests/hostsim/hip_sim.cpp, built as libamdhip64.so.7) with launch stubs in place of the kernels
(tests/hostsim/launch_stubs.cpp). Every launch names the device ranges its kernel would touch; the
simulation checks them against the live allocations when the launch executes, which for a
captured launch is every graph replay, so a buffer freed while a graph still names it, or smaller
than a launch assumes, fails the run. The bench legs run as they do on the GPU box: C5's 26
layers with 64 per-token graphs (the leg during which one profiled run once ended in a
segmentation fault), and the default bench line with every other leg. Kernels do not run, so no
figure here means anything; the test is about host code and lifetimes."""

import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _runtime(name):
    out = subprocess.run(["g++", f"-print-file-name={name}"], capture_output=True, text=True)
    path = out.stdout.strip()
    return path if os.path.isabs(path) and os.path.exists(path) else None


@pytest.fixture(scope="module")
def sim(tmp_path_factory):
    if shutil.which("g++") is None or _runtime("libasan.so") is None:
        pytest.skip("needs g++ with AddressSanitizer")
    d = tmp_path_factory.mktemp("hostsim")
    flags = ["-std=c++17", "-O1", "-g", "-fPIC", "-shared", "-fno-omit-frame-pointer",
             "-I", os.path.join(ROOT, "tests", "hostsim")]
    runtime = d / "libamdhip64.so.7"
    build = subprocess.run(["g++", *flags, "-fsanitize=address",
                            os.path.join(ROOT, "tests", "hostsim", "hip_sim.cpp"),
                            "-Wl,-soname,libamdhip64.so.7", "-o", str(runtime)],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    lib = d / "libjmodels_attn_hostsim.so"
    build = subprocess.run(["g++", *flags, "-fsanitize=address,undefined",
                            "-I", os.path.join(ROOT, "include"),
                            "-I", os.path.join(ROOT, "models_amd", "csrc"),
                            os.path.join(ROOT, "models_amd", "csrc", "jma_runtime.cpp"),
                            os.path.join(ROOT, "tests", "hostsim", "launch_stubs.cpp"),
                            f"-L{d}", "-l:libamdhip64.so.7", f"-Wl,-rpath,{d}", "-o", str(lib)],
                           capture_output=True, text=True)
    assert build.returncode == 0, build.stderr
    env = dict(os.environ)
    env.update({
        "LD_LIBRARY_PATH": str(d),
        "LD_PRELOAD": " ".join(p for p in (_runtime("libasan.so"), _runtime("libubsan.so")) if p),
        "ASAN_OPTIONS": "detect_leaks=0",
        "UBSAN_OPTIONS": "print_stacktrace=1:halt_on_error=1",
        "MODELS_HIP_ATTENTION_LIBRARY": str(lib),
        "PYTHONUNBUFFERED": "1",
    })
    return env


def _bench(env, *args, timeout=900):
    run = subprocess.run([sys.executable, os.path.join(ROOT, "bench.py"), *args], cwd=ROOT, env=env,
                         capture_output=True, text=True, timeout=timeout)
    out = run.stdout + run.stderr
    assert run.returncode == 0, out[-4000:]
    assert "hipsim:" in out and " 0 errors" in out, out[-4000:]
    assert "AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
    return run.stdout


def test_c5_leg_lifetimes(sim):
    """bench.py --c5-only: the cache filled layer by layer, 64 eager tokens, 64 per-token graphs
    (30 launches each: 22 sliding layers, 4 global layers with their reduce launch) replayed after
    warm-up, then graphs destroyed, buffers freed and the cache closed, as on the GPU box."""
    out = _bench(sim, "--c5-only")
    assert '"c5_us_per_token"' in out


def test_default_bench_line(sim):
    """The default bench line (every leg but the CPU baseline, 2 timed steps): C2, C1, C3, the
    other prefills and decode layers, C4, C5 and the projections, ending in the JSON line."""
    out = _bench(sim, "--steps", "2", "--warmup", "1", "--no-cpu", timeout=1500)
    assert '"metric"' in out and '"roofline"' in out


def _python(env, code):
    run = subprocess.run([sys.executable, "-c", code], cwd=ROOT, env=env, capture_output=True, text=True,
                         timeout=300)
    out = run.stdout + run.stderr
    assert run.returncode == 0 and " 0 errors" in out, out[-4000:]
    assert "AddressSanitizer" not in out and "runtime error" not in out, out[-4000:]
    return run.stdout


def test_synchronize_waits_for_null_stream_fills(sim):
    """A caller's hipMemset on the null stream is over once jmodels_attn_context_synchronize returns:
    the context's non-blocking stream alone would not wait for it."""
    _python(sim, """
import ctypes
from models_amd import attention as A, hip_runtime as rt
with A.HipAttentionLibrary(0) as hip:
    d = rt.DeviceArray(64)
    rt.check(rt.hip().hipMemset(d.ptr, 0, d.nbytes), "hipMemset")
    assert any(ctypes.string_at(d.ptr, d.nbytes)), "the fill has not run yet"
    hip.synchronize()
    assert not any(ctypes.string_at(d.ptr, d.nbytes)), "the fill was not waited for"
""")


def test_projection_scratch(sim):
    """A prefill-sized projection holds scratch for what its formats keep of the activations (32-element
    formats 2 1/16 bytes each, K-quants up to 4 9/64, with 31 rows of 65536 inputs to spare), so that a
    captured call of no more activations than the eager one before it does not have to grow it; where
    so much cannot be allocated it takes what the call itself needs, and a captured call that fits runs."""
    _python(sim, """
import ctypes
import numpy as np
from models_amd import attention as A, hip_runtime as rt
live = rt.hip().hipsim_live_bytes
live.restype = ctypes.c_size_t
largest = lambda n: rt.hip().hipsim_largest_allocation(ctypes.c_size_t(n))
Q8_0, Q4_K, Q6_K = A.WEIGHTS_Q8_0, A.WEIGHTS_Q4_K, A.WEIGHTS_Q6_K
sizes = {Q8_0: (34, 32), Q4_K: (144, 256), Q6_K: (210, 256)}

def call(hip, formats, batch, cols):
    ws = [rt.DeviceArray(cols // sizes[f][1] * sizes[f][0], np.uint8) for f in formats]
    hip.quantized_grouped_matmul_device(formats, [w.ptr for w in ws], [w.nbytes for w in ws], [1] * len(ws),
                                        x.ptr, x.count, out.ptr, out.count, batch, cols)

def captured(hip, *args):
    g = rt.Graph(hip.stream(), lambda: call(hip, *args))
    g.destroy()

n, spare = 4096 * 8192, 31 * 65536
x, out = rt.DeviceArray(n), rt.DeviceArray(4 * 8192)
for fmt, per in ((Q8_0, 2 + 1 / 16), (Q4_K, 4 + 9 / 64), (Q6_K, 4 + 9 / 64)):
    with A.HipAttentionLibrary(0) as hip:
        before = live()
        call(hip, [fmt], 4096, 8192)
        held = live() - before
        assert n * per <= held <= (n + spare) * per + 4096, (fmt, held / n)
        if fmt != Q8_0:
            call(hip, [Q4_K, Q6_K], 4096, 8192)
            call(hip, [Q6_K, Q4_K], 4095, 8192)
            call(hip, [Q4_K], 511, 65536)
            assert live() - before == held, "a call of no more activations grew the scratch"
for fmt, other, per in ((Q4_K, Q6_K, 2 + 9 / 64), (Q6_K, Q4_K, 2 + 1 / 64), (Q8_0, Q8_0, 2 + 1 / 16)):
    with A.HipAttentionLibrary(0) as hip:
        before = live()
        largest(int(n * per) + 4096)  # not the whole preference
        for _ in range(2):
            call(hip, [fmt], 4096, 8192)
            assert live() - before <= n * per + 4096, "more than the call itself needs"
        captured(hip, [fmt], 4096, 8192)
        if other != fmt:
            try:
                captured(hip, [fmt, other], 4096, 8192)
                raise AssertionError("captured past its scratch")
            except A.AttentionStatusError as e:
                assert "NOT_CAPTURABLE" in str(e), e
        largest(2 ** 62)
x = rt.DeviceArray(32 * 4096)
with A.HipAttentionLibrary(0) as hip:
    call(hip, [Q8_0], 32, 4096)
    before = live()
    captured(hip, [Q4_K, Q6_K], 16, 8192)
    captured(hip, [Q6_K], 17, 7680)
    assert live() == before, "a call of no more activations grew the scratch"
""")


def test_projection_past_one_launch_is_refused_first(sim):
    """A product whose grid would pass 2^32 threads, or whose batch the calls' limit, is refused as an
    invalid shape before its activations are quantized. (The buffers' claimed sizes pass the size checks;
    nothing is ever read from them.)"""
    _python(sim, """
import ctypes
from models_amd import attention as A, hip_runtime as rt
launches = rt.hip().hipsim_launches
launches.restype = ctypes.c_long
x = rt.DeviceArray(64 * 32)
with A.HipAttentionLibrary(0) as hip:
    for batch, rows in ((16, 0xFFFFFF00), (64, 0xFFFFFF00), (65535 * 64 + 1, 32)):
        try:
            hip.quantized_matmul_device(A.WEIGHTS_Q4_0, x.ptr, rows * 18, x.ptr, batch * 32, x.ptr, batch * rows,
                                        batch, rows, 32)
        except A.AttentionStatusError as e:
            assert "INVALID_SHAPE" in str(e), e
        else:
            raise AssertionError("not refused")
        assert launches() == 0
""")
