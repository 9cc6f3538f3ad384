"""Inverted residual blocks as one launch (csrc/inverted_residual.hip): whole networks, every block's output bit for bit
against the oracle's convolutions and sums."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def g():
    import gpu_util
    gpu_util.capi.init(0)
    return gpu_util


@pytest.fixture(scope="module")
def vm(g):
    return importlib.import_module(g.pkg.__name__ + ".chxvm")


def check(g, vm, oracle, model, keep, blocks):
    """Through Program.run and a recording of it, in which the input changes."""
    wl = g.pkg.workloads
    prog = vm.Program(wl.program_to_chxvm(model, vm, g.pkg.ops, keep=keep).serialize())
    prog.set_option("qlinearconv_bias", "onnx_int32")
    x = torch.from_numpy(model["input"]).cuda()
    before = vm.counter("inverted_residuals")
    got = prog.run({"x": x})
    assert vm.counter("inverted_residuals") - before == blocks
    oracle.set_threads(16)
    try:
        for i in range(2):
            ref = wl.run_reference(model, oracle, model["input"][::-1] if i else model["input"], keep=set(keep))
            if i:
                replay = prog.capture({"x": x})
                x.copy_(torch.from_numpy(model["input"][::-1].copy()))
                torch.cuda.synchronize()
                for _ in range(3):
                    replay.launch()
                    replay.synchronize()
                    again = prog.run({"x": x})
                got = replay.outputs()
                for name in keep:
                    np.testing.assert_array_equal(again[name], ref[name], err_msg=name)
            for name in keep:
                np.testing.assert_array_equal(got[name], ref[name], err_msg="%d %s" % (i, name))
    finally:
        oracle.set_threads(1)
    replay.close()
    prog.close()


def block_outputs(model):
    """The last value of every block: a sum, or the result of a projection that no sum reads."""
    program = model["program"]
    read_by_sum = {v for ins in program if ins[0] in ("Add", "AddRelu") for v in ins[2:4]}
    names = [ins[1] for ins in program if ins[0] == "Add"]
    return names


# image: what the first block sees is half of it; (expansion, channels, repeats, stride)
@pytest.mark.parametrize("batch,image,blocks,stem", [
    (2, 64, ((1, 16, 1, 1), (6, 24, 2, 2), (6, 32, 1, 2)), 32),                  # 16 -> 96 channels, a pixel of one chunk
    (3, 30, ((1, 8, 1, 1), (6, 40, 2, 1), (3, 48, 2, 2)), 24),                   # 15x15 and 8x8: odd rows, odd chunks
    (130, 14, ((6, 64, 1, 1), (6, 96, 1, 1), (6, 160, 2, 2), (6, 320, 1, 1)), 32),  # 7x7 and 4x4, two tiles of channels for a wavefront
    (1, 14, ((6, 64, 1, 1), (6, 96, 2, 1), (6, 256, 1, 2)), 32),                 # eight tiles of channels and few rows
    (5, 2, ((6, 32, 2, 1),), 32),                                                # one pixel
    (2, 6, ((2, 17, 2, 1), (5, 33, 1, 2)), 20),                                  # 3x3, channels that are no multiple of anything
    (2, 226, ((6, 24, 2, 1),), 16),                                              # 113 columns
])
def test_networks(g, vm, oracle, batch, image, blocks, stem):
    model = g.pkg.workloads.build_mobilenetv2(batch=batch, image=image, seed=batch + image, blocks=blocks, stem=stem, head=64, classes=10)
    count = sum(n for t, _, n, _ in blocks if t != 1)
    check(g, vm, oracle, model, ["logits"] + block_outputs(model), count)


@pytest.mark.parametrize("batch", [1, 40, 80])
def test_full_size(g, vm, oracle, batch):
    """All blocks of the network at the sizes it is used at, on few and on many images."""
    model = g.pkg.workloads.build_mobilenetv2(batch=batch, seed=11)
    wl = g.pkg.workloads
    prog = vm.Program(wl.program_to_chxvm(model, vm, g.pkg.ops, keep=["logits"] + block_outputs(model)).serialize())
    prog.set_option("qlinearconv_bias", "onnx_int32")
    got = prog.run({"x": torch.from_numpy(model["input"]).cuda()})
    picks = [0] if batch == 1 else [0, batch // 2, batch - 1]
    oracle.set_threads(16)
    try:
        ref = wl.run_reference(model, oracle, model["input"][picks], keep=set(got))
    finally:
        oracle.set_threads(1)
    for name in got:
        np.testing.assert_array_equal(got[name][picks], ref[name], err_msg=name)
    prog.close()
