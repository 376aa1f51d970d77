"""The index arithmetic of the fused widening + depthwise launch, on the host: the library's own plan and the kernel's own walk, over
frames, strides, paddings and shared workgroups (tests/host/ir_cells.cpp says what is checked)."""
import subprocess

import numpy as np
import pytest

from helpers import host_check


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = host_check("ir_cells", tmp_path_factory.mktemp("ir"))

    def run(N, H, W, K, C, stride, pad, first=None):
        """pad: (top, bottom, left, right); first: (window, stride, channels), unpadded, its image as large as its windows need.
        -> images per workgroup"""
        OH, OW = (H + pad[0] + pad[1] - 3) // stride + 1, (W + pad[2] + pad[3] - 3) // stride + 1
        args = [N, H, W, K, C, OH, OW, stride, pad[0], pad[2]]
        if first:
            k, s, c = first
            args += [k, s, 0, 0, (H - 1) * s + k, (W - 1) * s + k, c, k]
        done = subprocess.run([exe] + [str(a) for a in args], stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=120)
        assert done.returncode == 0, (args, done.stdout)
        return int(done.stdout)

    return run


# windows that stop short of the image's last row, in workgroups of several images
SHORT = [((300, 8, 8, 16, 256, 2, (0, 0, 0, 0)), 2), ((256, 14, 14, 96, 576, 2, (0, 0, 0, 0)), 4), ((300, 7, 7, 16, 256, 2, (1, 0, 1, 1)), 2)]


# segments that make more rows than the last of them has, in strips that are shorter than the others, and where that took a launch past 64 KB of LDS
DEEP = [(600, 34, 5, 16, 272, 1, (1, 1, 1, 1)), (300, 66, 3, 32, 272, 2, (1, 1, 1, 1)), (1, 64, 1, 16, 32, 1, (1, 1, 1, 1)), (1, 131, 1, 16, 32, 2, (1, 1, 1, 1)), (1, 11, 3, 16, 32, 2, (1, 1, 1, 1)),
        (1, 5, 65, 16, 32, 1, (1, 1, 1, 1)), (1, 5, 640, 16, 32, 1, (1, 1, 1, 1)), (1, 300, 16, 16, 32, 1, (1, 1, 1, 1)), (259, 13, 14, 96, 592, 1, (1, 1, 1, 1)), (66, 2, 1, 64, 1040, 1, (1, 1, 1, 1))]


@pytest.mark.parametrize("case", DEEP, ids=lambda c: "x".join(str(v) for v in c[:6]))
def test_rows_below_the_strip(check, case):
    check(*case)


@pytest.mark.parametrize("runs", [False, True])
@pytest.mark.parametrize("case,images", SHORT, ids=["8x8_s2", "14x14_s2", "7x7_s2_top"])
def test_rows_no_window_reaches(check, case, images, runs):
    shared = check(*case, first=(3, 1, 3) if runs else None)
    assert shared >= images, "the case is about images that share a workgroup"


@pytest.mark.parametrize("case,images", [
    ((32, 14, 14, 64, 384, 1, (1, 1, 1, 1)), 2), ((256, 14, 14, 64, 384, 1, (1, 1, 1, 1)), 4), ((256, 7, 7, 160, 960, 1, (1, 1, 1, 1)), 11), ((54, 16, 16, 32, 192, 2, (0, 1, 0, 1)), 2),
    ((12, 10, 10, 96, 576, 1, (1, 1, 1, 1)), 1), ((1, 14, 14, 96, 576, 1, (1, 1, 1, 1)), 1),
], ids=["14x14_b32", "14x14_b256", "7x7_b256", "16x16_b54", "10x10_b12", "14x14_b1"])
def test_images_by_the_estimate(check, case, images):
    """As many images a workgroup as are measured ahead: two where strips of one image had been cut in two."""
    assert check(*case) == images


def test_drawn_geometries(check):
    rng = np.random.default_rng(11)
    shared = 0
    for _ in range(200):
        H, W = int(rng.integers(1, 24)), int(rng.integers(1, 40))
        pad = tuple(int(v) for v in rng.integers(0, 3, size=4))
        stride = int(rng.integers(1, 3))
        if H + pad[0] + pad[1] < 3 or W + pad[2] + pad[3] < 3:
            continue
        # what the planner asks too: no window starts behind the image
        if (H + pad[0] + pad[1] - 3) // stride * stride - pad[0] >= H or (W + pad[2] + pad[3] - 3) // stride * stride - pad[2] >= W:
            continue
        K = int(rng.choice([16, 48, 64, 160]))
        first = (int(rng.integers(1, 5)), int(rng.integers(1, 3)), int(rng.integers(1, 5))) if rng.integers(0, 3) == 0 else None
        if first and first[0] * first[2] > 16:
            continue
        shared += check(int(rng.choice([1, 40, 300, 1100])), H, W, K, int(rng.choice([16, 80, 256, 576])), stride, pad, first) > 1
    assert shared >= 20
