"""What the kernels of a recorded run address stays where it is until the recording is gone, without a GPU."""
import ctypes

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["program_destroyed_first", "replay_destroyed_first"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def recording(host):
    """A float32 layer whose weights the kernel reads where they lie, as a program and a recording of it."""
    import numpy as np
    b = host.chxvm.ProgramBuilder()
    x = b.input("x", "float32", [8, 64])
    b.output("y", b.MatMul(x, b.constant(np.ones((64, 96), np.float32))))
    rt, program, replay = host.chxvm.runtime(), host.program(b), ctypes.c_void_p()
    assert rt.chxvm_program_capture(program, *host.names_and({"x": host.tensor("float32", (8, 64))}), ctypes.byref(replay)) == 0, rt.chxvm_last_error()
    host.clear()
    return rt, program, replay


def program_destroyed_first(host):
    rt, program, replay = recording(host)
    rt.chxvm_program_destroy(program)
    assert not host.log(), host.log()
    assert rt.chxvm_replay_launch(replay, None) == 0 and rt.chxvm_replay_synchronize(replay) == 0
    rt.chxvm_replay_destroy(replay)
    assert "hipFree" in host.log()
    waits = [i for i, line in enumerate(host.log()) if line.startswith("hipDeviceSynchronize")]
    assert waits and "hipFree" in host.log()[waits[-1]:]  # (the constants, behind everything)


def replay_destroyed_first(host):
    rt, program, replay = recording(host)
    rt.chxvm_replay_destroy(replay)
    host.clear()
    rt.chxvm_program_destroy(program)
    assert "hipFree" in host.log()


if __name__ == "__main__":
    host_hip.main(globals())
