"""Small device results in host memory (csrc/copyout.hip) and the memory eager runs reuse (runtime/device_cache.cc)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    return gpu_util


@pytest.fixture(scope="module")
def vm(g):
    import importlib
    return importlib.import_module(g.pkg.__name__ + ".chxvm")


@pytest.mark.parametrize("n", [1, 15, 16, 17, 4095, 65536, 512 * 1024 - 1, 512 * 1024, 512 * 1024 + 1])
@pytest.mark.parametrize("offset", [0, 3])
def test_copy_to_host(g, n, offset):
    src = torch.arange(n + 8, device="cuda", dtype=torch.int64).remainder(251).to(torch.uint8)
    torch.cuda.synchronize()
    got = np.full(n + 2, 255, np.uint8)
    for _ in range(3):
        got[1:n + 1] = 254
        g.capi.check(g.capi.lib().chx_hip_memcpy_d2h(ctypes.c_void_p(got.ctypes.data + 1), ctypes.c_void_p(src.data_ptr() + offset), ctypes.c_size_t(n), None))
        np.testing.assert_array_equal(got[1:n + 1], (np.arange(n) + offset) % 251)
    assert got[0] == 255 and got[-1] == 255


def scaling_program(g, vm, shape):
    """y = relu(2 * x), z = y + x: values that are freed inside the run, two results."""
    b = vm.ProgramBuilder()
    x = b.input("x", "float32", shape)
    two = b.constant(np.full((1,), 2, np.float32))
    t = b.Mul(x, two)
    y = b.Relu(t)
    b.Free(t)
    b.output("y", y)
    b.output("z", b.Add(y, x))
    return vm.Program(b.serialize())


# results that fit the host block together, and results that do not
@pytest.mark.parametrize("elements", [5, 1000, 70000])
def test_runs_of_alternating_programs_and_sizes(g, vm, elements):
    rng = np.random.default_rng(elements)
    progs = [scaling_program(g, vm, (elements,)) for _ in range(2)]
    for i in range(6):
        n = elements + 100 * (i % 3)
        x = rng.standard_normal(n).astype(np.float32)
        out = progs[i % 2].run({"x": g.dev(x)})
        np.testing.assert_array_equal(out["y"], np.maximum(2 * x, 0))
        np.testing.assert_array_equal(out["z"], np.maximum(2 * x, 0) + x)


@pytest.mark.parametrize("elements", [1000, 70000])
@pytest.mark.parametrize("own_stream", [True, False])
def test_replay_results_follow_every_launch(g, vm, elements, own_stream):
    prog = scaling_program(g, vm, (elements,))
    x = torch.zeros(elements, device="cuda")
    replay = prog.capture({"x": x})
    stream = torch.cuda.Stream()
    for i in range(5):
        torch.cuda.synchronize()
        x.fill_(i - 2.0)
        torch.cuda.synchronize()
        if own_stream:
            replay.launch()
            replay.synchronize()
        else:
            replay.launch(ctypes.c_void_p(stream.cuda_stream))
            stream.synchronize()
        if i != 1:  # a launch whose results the host does not read
            out = replay.outputs()
            assert (out["y"] == max(2 * (i - 2.0), 0)).all() and (out["z"] == max(2 * (i - 2.0), 0) + i - 2.0).all()
    replay.close()


def test_threads_running_one_program_get_their_own_results(g, vm):
    import threading
    prog, wrong = scaling_program(g, vm, (3000,)), []

    def work(k):
        x = np.full(3000, float(k), np.float32)
        xd = g.dev(x)
        torch.cuda.synchronize()
        for _ in range(200):
            out = prog.run({"x": xd})
            if not ((out["y"] == 2 * k).all() and (out["z"] == 3 * k).all()):
                wrong.append(k)

    threads = [threading.Thread(target=work, args=(k,)) for k in range(1, 5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
