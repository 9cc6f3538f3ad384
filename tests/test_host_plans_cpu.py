"""Which kernels the entry points of csrc/contract_api.hip launch, and on what memory, without a GPU."""
import ctypes

import pytest

import host_hip


@pytest.fixture(scope="module")
def host_so(tmp_path_factory):
    return host_hip.build(tmp_path_factory.mktemp("host_hip"))


@pytest.mark.parametrize("case", ["one_plan_on_dense_images_and_crops"])
def test_case(host_so, case):
    host_hip.run_case(host_so, __file__, case)


def one_plan_on_dense_images_and_crops(host):
    """A measured configuration is for the strides it was measured on: the pixel-streaming kernel takes dense images only."""
    n, c, h, w = 8, 64, 32, 32
    dense, crop = host.channels_last("uint8", (n, c, h, w)), host.tensor("uint8", (n, c, h, w), [36 * 40 * c, 1, 40 * c, c])
    rows = host.tensor("uint8", (n, c, h, w), [36 * w * c, 1, w * c, c])
    y = host.channels_last("uint8", (n, 64, h, w))
    host.hh.hh_prefer(b"conv_point_kernel")
    for order in ([dense, crop, rows, dense], [crop, dense, rows], [rows, dense, crop]):
        plan = host.plan(64, c, 1)
        for x in order:
            host.check(host.plan_run(plan, x, y))  # measures
            host.clear()
            host.check(host.plan_run(plan, x, y))
            assert len(host.launches()) == 1 and ("conv_point_kernel" in host.launches()[0]) == (x is dense)
        host.lib.chx_hip_qconv_plan_destroy(plan)
    # one image whose rows alone lie apart, on a plan of its own: what other plans have measured is shared
    dense, apart = host.channels_last("uint8", (1, c, 96, 96)), host.tensor("uint8", (1, c, 96, 96), [96 * 96 * c, 1, 100 * c, c])
    y = host.channels_last("uint8", (1, 64, 96, 96))
    for x in (dense, apart, dense):
        plan = host.plan(64, c, 1)
        host.check(host.plan_run(plan, x, y))


if __name__ == "__main__":
    host_hip.main(globals())
