"""The host side of uploads without a GPU: what happens when threads or memory cannot be had, and what several callers of one
uploader see.  Each test runs in a process of its own with tests/native/host_stub.c preloaded, so that HIP's memory calls work
on ordinary memory and can be told to fail."""
import os
import subprocess
import sys
import textwrap

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, threading
import numpy as np
import tcbnn_amd
from tcbnn_amd import _lib, device, layers
L = _lib.lib
stub = C.CDLL(STUB)
def knob(name, value):
    C.c_int.in_dll(stub, "stub_" + name).value = value
def allocations():
    return C.c_int.in_dll(stub, "stub_allocations").value
for name in ("hipMalloc", "hipHostMalloc", "hipFree", "hipHostFree", "hipMemcpy", "hipMemset"):
    getattr(stub, name).argtypes = getattr(_lib.hip, name).argtypes
device.hip = stub
r = np.random.default_rng(1)
def floats(n):
    return r.standard_normal(n).astype(np.float32)
def uploader(nbytes, staged=0):
    p = C.c_void_p(0)
    assert L.tcbnn_uploader_create(nbytes, staged, C.byref(p)) == 0, L.tcbnn_last_error()
    return p
"""


@pytest.fixture(scope="module")
def run(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("native") / "host_stub.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", "-o", so, os.path.join(ROOT, "tests/native/host_stub.c"), "-ldl"], check=True)

    preload = ":".join([so] + [v for v in [os.environ.get("LD_PRELOAD")] if v])
    env = dict(os.environ, LD_PRELOAD=preload, PYTHONPATH=ROOT, OMP_NUM_THREADS="1", OPENBLAS_NUM_THREADS="1")

    def go(body):
        code = "STUB = %r\n" % so + PRELUDE + textwrap.dedent(body) + "\nprint('done')\n"
        p = subprocess.run([sys.executable, "-c", code], env=env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=240)
        assert p.returncode == 0 and p.stdout.strip().endswith("done"), "exit %d: %s" % (p.returncode, p.stdout[-2000:])
    go.env, go.stub = env, so
    return go


def test_new_batches_through_the_cpp_layer(run, tmp_path):
    exe, lib = str(tmp_path / "layer_uploads"), os.path.join(ROOT, "tcbnn_amd")
    subprocess.run(["g++", "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-o", exe,
                    os.path.join(ROOT, "tests/native/layer_uploads.cpp"), run.stub, "-L" + lib, "-ltcbnn_hip", "-L/opt/rocm/lib", "-lamdhip64",
                    "-pthread", "-Wl,-rpath," + lib, "-Wl,-rpath,/opt/rocm/lib", "-w"],
                   check=True)
    p = subprocess.run([exe], env=run.env, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=240)
    assert p.returncode == 0 and p.stdout.strip() == "done", "exit %d: %s" % (p.returncode, p.stdout[-2000:])


@pytest.mark.parametrize("left", [0, 1, 3])
def test_fewer_threads_than_asked_for_are_enough(run, left):
    """A thread that cannot be created, the first or a later one, costs speed and nothing else."""
    run("""
    knob("threads_left", %d)
    x = floats((3 << 20) + 5)
    u = uploader(x.nbytes, 1)
    y, most = np.empty_like(x), C.c_float(0)
    assert L.tcbnn_upload_stage(u, x.ctypes.data, x.size, C.byref(most)) == 0 and L.tcbnn_upload_commit(u, y.ctypes.data) == 0
    assert np.array_equal(x, y) and most.value == np.abs(x).max()
    L.tcbnn_uploader_destroy(u)
    assert L.tcbnn_host_abs_max(x.ctypes.data, x.size) == np.abs(x).max()
    im = floats((12, 3, 9, 9))
    bound = L.tcbnn_inconv_residual_bound_of_input(im.ctypes.data, 12, 9, 9, 9, 9, 9, 9, 0)
    most = np.abs(im.astype(np.float64)).sum((1, 2, 3)).max()
    assert most <= bound <= most * 1.001 + 2
    """ % left)


def test_a_failed_or_refused_stage_leaves_nothing_to_commit(run):
    """Staging overwrites what was staged before: after a stage that failed on the way there is nothing to commit."""
    run("""
    x, z = floats(3 << 20), floats(3 << 20)     # 12 MiB: goes on to the device copy chunk by chunk
    u = uploader(x.nbytes, 1)
    y, most = np.zeros_like(x), C.c_float(0)
    assert L.tcbnn_upload_stage(u, x.ctypes.data, x.size, C.byref(most)) == 0
    knob("copies_left", 1)
    assert L.tcbnn_upload_stage(u, z.ctypes.data, z.size, C.byref(most)) == -3
    knob("copies_left", -1)
    assert L.tcbnn_upload_commit(u, y.ctypes.data) == -1 and not y.any()
    assert L.tcbnn_upload_stage(u, z.ctypes.data, z.size, C.byref(most)) == 0 and L.tcbnn_upload_commit(u, y.ctypes.data) == 0
    assert np.array_equal(y, z)
    L.tcbnn_uploader_destroy(u)
    assert allocations() == 0
    """)


def test_two_threads_with_new_batches_for_one_layer(run):
    """set_input from two threads: each batch is staged, judged and committed as a whole, one after the other."""
    run("""
    n = 3 * 20 * 20 * 8
    layer = layers.InConv128LayerParam("Conv1", 20, 20, 3, 3, 3, 64, 8, save_residual=True)
    layer.input_gpu = device.DeviceBuffer.zeros(4 * n)
    layer._uploads = device.InputUploads(staged=True)
    class Residual:
        bound, format, channels, readers = 2000, _lib.RES_I12, 64, []
    layer.output_residual_gpu = Residual()
    layers._residual_bound_limit = lambda buf: 2047
    first = [floats(n), floats(n)]
    for x in first:
        layer.set_input(x)
    assert layer._uploads.uploader is not None
    staged = threading.Barrier(2, timeout=2)
    stage = device.Uploader.stage
    def stage_and_wait(self, arr):
        most = stage(self, arr)
        try:
            staged.wait()                        # lets the other thread stage too, where it can
        except threading.BrokenBarrierError:
            pass
        return most
    device.Uploader.stage = stage_and_wait
    failed = []
    def call(x):
        try:
            layer.set_input(x)
        except Exception as e:
            failed.append(e)
    threads = [threading.Thread(target=call, args=(x,)) for x in first]
    [t.start() for t in threads]; [t.join() for t in threads]
    assert not failed, failed
    got = layer.input_gpu.to_numpy(np.float32, (n,))
    assert any(np.array_equal(got, x) for x in first)
    """)


def test_two_threads_downloading_through_one_pinned_buffer(run):
    run("""
    import time
    a, b = device.DeviceBuffer.from_numpy(floats(1000)), device.DeviceBuffer.from_numpy(floats(1000))
    host = device.Downloads()
    for _ in range(2):
        assert np.array_equal(host.get(a, np.float32, (1000,)), a.to_numpy(np.float32, (1000,)))
    assert host.pinned is not None
    class Slow:
        def __getattr__(self, name):
            return getattr(stub, name)
        def hipMemcpy(self, *args):
            rc = stub.hipMemcpy(*args)
            time.sleep(0.05)
            return rc
    device.hip = Slow()
    got = {}
    def call(i, src):
        got[i] = host.get(src, np.float32, (1000,))
    threads = [threading.Thread(target=call, args=(i, s)) for i, s in enumerate((a, b))]
    [t.start() for t in threads]; [t.join() for t in threads]
    assert np.array_equal(got[0], a.to_numpy(np.float32, (1000,))) and np.array_equal(got[1], b.to_numpy(np.float32, (1000,)))
    """)


def test_the_first_batch_and_result_allocate_nothing_and_the_second_can_do_without(run):
    """set_input and the results of a layer: pinned memory, a staging copy and threads are made for the second batch or
    result, and where they cannot be had everything goes on as it began; a refused batch leaves the buffer alone."""
    run("""
    n = 3 * 224 * 224 * 8                        # 4.8 MB: staged on the device
    class Residual:
        format, channels, readers = _lib.RES_I12, 64, []
    def layer_of(save):
        layer = layers.InConv128LayerParam("Conv1", 224, 224, 3, 3, 3, 64, 8, save_residual=save)
        layer.input_gpu = device.DeviceBuffer.zeros(4 * n)
        layer._uploads = device.InputUploads(staged=save)
        layer.output_residual_gpu = Residual()
        layer.output_residual_gpu.bound = 2000
        return layer
    layers._residual_bound_limit = lambda buf: 2047
    layers._raise_residual_bound = lambda buf, bound: None
    held = lambda layer: layer.input_gpu.to_numpy(np.float32, (n,))
    for what in (None, "host_mallocs_left", "mallocs_left", "threads_left"):
        for save in (False, True):
            layer = layer_of(save)
            before = allocations()
            x = floats(n)
            layer.set_input(x)
            assert np.array_equal(held(layer), x) and allocations() == before
            if what:
                knob(what, 0)
            for _ in range(3):
                x = floats(n)
                layer.set_input(x)
                assert np.array_equal(held(layer), x)
            if save:
                try:
                    layer.set_input(floats(n) * 1000)
                    raise SystemExit("not refused")
                except _lib.TcbnnError:
                    assert np.array_equal(held(layer), x)
            if what in ("host_mallocs_left", "mallocs_left") and (save or what == "host_mallocs_left"):
                assert layer._uploads.uploader is None and allocations() == before
            if what:
                knob(what, -1)
            layer._uploads.free()
            assert allocations() == before
            layer.input_gpu.free()
    src = device.DeviceBuffer.from_numpy(floats(100))
    before = allocations()
    for left in (-1, 0):
        out = device.Downloads()
        knob("host_mallocs_left", left)
        for k in range(3):
            assert np.array_equal(out.get(src, np.float32, (100,)), src.to_numpy(np.float32, (100,)))
            assert allocations() == before + (1 if k and left else 0)
        out.free()
        knob("host_mallocs_left", -1)
    """)
