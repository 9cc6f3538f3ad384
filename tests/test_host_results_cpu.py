"""Results on the host (runtime/chxvm_capi.cc, csrc/copyout.hip) and the memory eager runs reuse, without a GPU."""
import ctypes
import os
import sys
import threading
import time

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["two_threads_of_one_program", "memory_of_each_device", "sources_of_the_result_copy", "launches_do_not_wait"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def run_to_host(host, program, inputs):
    rt = host.chxvm.runtime()
    out = ctypes.c_void_p()
    assert rt.chxvm_program_run_to_host(program, *host.names_and(inputs), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
    return out


def host_copy(host, out, i, nbytes):
    p = host.chxvm.runtime().chxvm_outputs_host(out, i)
    return ctypes.string_at(p, nbytes) if p else None


def copying_program(host):
    b = host.chxvm.ProgramBuilder()
    b.output("y", b.input("x", "uint8", [64]))
    return host.program(b)


def wait_until(condition):
    end = time.time() + 20
    while not condition():
        assert time.time() < end
        time.sleep(0.001)


def two_threads_of_one_program(host):
    """One thread's run waits for its results while another thread's run of the same program starts and ends."""
    program, got = copying_program(host), {}

    def run(name):
        x = host.tensor("uint8", (64,))
        host.bytes(x.data, bytes([ord(name)]) * 64)
        out = run_to_host(host, program, {"x": x})
        got[name] = host_copy(host, out, 0, 64)
        host.chxvm.runtime().chxvm_outputs_destroy(out)

    for size in range(3):  # (also with blocks that earlier runs have left)
        host.hh.hh_hold(1)
        a = threading.Thread(target=run, args="a")
        a.start()
        wait_until(lambda: host.hh.hh_held() >= 1)
        b = threading.Thread(target=run, args="b")
        b.start()
        b.join(20)
        assert not b.is_alive()
        host.hh.hh_release()
        a.join(20)
        assert got == {"a": b"a" * 64, "b": b"b" * 64}


def memory_of_each_device(host):
    """Runs on two devices in turn: every array lies on the device of its run, whatever earlier runs have left."""
    rt, b = host.chxvm.runtime(), host.chxvm.ProgramBuilder()
    x = b.input("x", "float32", [64])
    t = b.QuantizeLinear(x, b.scalar(0.5, "float32"), b.scalar(3, "uint8"))
    b.output("y", b.DequantizeLinear(t, b.scalar(0.25, "float32"), b.scalar(3, "uint8")))
    b.Free(t)
    program, held = host.program(b), []
    for device in (0, 1, 1, 0, 1):
        host.check(host.lib.chx_hip_init(device))
        x = host.tensor("float32", (64,))
        out, y = ctypes.c_void_p(), host.capi.Tensor()
        assert rt.chxvm_program_run(program, *host.names_and({"x": x}), 0, ctypes.byref(out)) == 0, rt.chxvm_last_error()
        assert rt.chxvm_outputs_get(out, 0, ctypes.byref(y)) == 0
        assert host.device_of(y.data) == device
        held.append((device, out, y.data))
        if len(held) == 2:
            # given up while the other device is current: waiting for that one would not do, so the block is not kept
            device, out, data = held.pop(0)
            host.check(host.lib.chx_hip_init(1 - device))
            rt.chxvm_outputs_destroy(out)
            assert host.device_of(data) == -2


def sources_of_the_result_copy(host):
    """The kernel that copies results reads memory of its own device only: every other source is the runtime's copy, as it
    was before there was the kernel."""
    lib, n = host.lib, 1000
    here = host.malloc(n)
    host.check(lib.chx_hip_init(1))
    there, stream_there = host.malloc(n), host.stream()
    host.check(lib.chx_hip_init(0))
    pinned, elsewhere = ctypes.c_void_p(), ctypes.create_string_buffer(n)
    assert host.hh.hipHostMalloc(ctypes.byref(pinned), ctypes.c_size_t(n), 0) == 0
    pageable = ctypes.addressof(elsewhere)
    got = ctypes.create_string_buffer(n)
    for src, stream, kernel in [(here, None, True), (there, None, False), (pinned.value, None, False), (pageable, None, False), (here, stream_there, False),
                                (there, stream_there, False)]:
        host.clear()
        host.bytes(src, bytes(range(250)) * 4)
        ctypes.memset(got, 0, n)
        host.check(lib.chx_hip_memcpy_d2h(got, ctypes.c_void_p(src), ctypes.c_size_t(n), stream))
        assert got.raw == bytes(range(250)) * 4
        assert any("copy_out_kernel" in k for k in host.launches()) == kernel, (src, stream)
    # a program whose output is its input, wherever that lies
    rt, program = host.chxvm.runtime(), copying_program(host)
    for src in (here, there, pinned.value, pageable):
        out = run_to_host(host, program, {"x": host.tensor("uint8", (64,), base=src)})
        assert (host_copy(host, out, 0, 64) is not None) == (src == here)
        rt.chxvm_outputs_destroy(out)
    # a block of device 0 does not serve device 1's launches
    block = ctypes.c_void_p()
    host.check(lib.chx_hip_copyout_create(ctypes.c_size_t(64), ctypes.byref(block)))
    host.check(lib.chx_hip_init(1))
    rc = lib.chx_hip_copyout_enqueue(block, (ctypes.c_void_p * 1)(there), (ctypes.c_size_t * 1)(64), 1, None)
    assert rc == host.capi.EUNSUPPORTED


def launches_do_not_wait(host):
    """A replay's launches only enqueue, whatever is still on its way to the host, and those whose results nobody asks for
    send nothing."""
    rt, replay, program = host.chxvm.runtime(), ctypes.c_void_p(), copying_program(host)
    x = host.tensor("uint8", (64,))
    assert rt.chxvm_program_capture(program, *host.names_and({"x": x}), ctypes.byref(replay)) == 0, rt.chxvm_last_error()
    rt.chxvm_replay_outputs.restype = ctypes.c_void_p
    outputs, streams = ctypes.c_void_p(rt.chxvm_replay_outputs(replay)), [None, host.stream(), host.stream()]
    refill = lambda v: host.bytes(x.data, bytes([v]) * 64)

    def launch(stream=None):
        rcs = []
        thread = threading.Thread(target=lambda: rcs.append(rt.chxvm_replay_launch(replay, stream)))
        host.clear()
        thread.start()
        thread.join(10)
        assert rcs == [0], "a launch waits"
        return sum("copy_out_kernel" in k for k in host.launches())

    assert launch() == 0 and launch() == 0
    assert host_copy(host, outputs, 0, 64) is None  # (the caller copies them from the device)
    for i in range(3):  # read after every launch: every launch sends its results
        refill(i)
        assert launch(streams[i]) == 1 and host_copy(host, outputs, 0, 64) == bytes([i]) * 64
    host.hh.hh_hold(1)
    assert launch() == 1
    for s in streams + streams:
        assert launch(s) == 0
    host.hh.hh_release()
    refill(77)
    assert launch() == 0
    assert host_copy(host, outputs, 0, 64) is None  # the block holds an older launch's
    refill(78)
    assert launch() == 1 and host_copy(host, outputs, 0, 64) == bytes([78]) * 64
    rt.chxvm_replay_destroy(replay)


if __name__ == "__main__":
    host_hip.main(globals())
