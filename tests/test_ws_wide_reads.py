"""The watershed's classification takes four pixels in a row by wide loads where they stay inside the marker
and colour planes.  On the CPU: the rule that decides it (nscale_amd/csrc/ws_rules.hpp), against the elements and
bytes that the wide path touches, over every group of every small plane.  On the GPU: planes of one column or
row that take the wide path, equal to the oracle's cv::watershed."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests._lib import ROOT, o_cv_watershed

PROGRAM = r"""
#include <cstdio>
#include "ws_rules.hpp"
int main() {
    int bad = 0, wide = 0;
    for (int W = 1; W <= 40; ++W)
        for (int H = 1; H <= 40; ++H) {
            const int N = W * H;
            for (int i0 = 0; i0 < N; i0 += 4) {
                if (!nsc::classify_wide(i0, W, N)) continue;
                ++wide;
                const int px[6][2] = {{i0 - W, i0 - W + 4}, {i0 + W, i0 + W + 4}, {i0 - 1, i0 + 5}, {0, 0}, {0, 0}, {0, 0}};
                const int by[4][2] = {{3 * i0 - 4, 3 * i0}, {3 * i0, 3 * i0 + 16}, {3 * (i0 - W), 3 * (i0 - W) + 12},
                                      {3 * (i0 + W), 3 * (i0 + W) + 12}};
                bool in = true;
                for (auto& r : px) in = in && r[0] >= 0 && r[1] <= N;
                for (auto& r : by) in = in && r[0] >= 0 && r[1] <= 3 * N;
                if (!in && bad++ < 5) std::printf("W %d H %d i0 %d\n", W, H, i0);
            }
        }
    std::printf("%d of %d groups leave a plane\n", bad, wide);
    return bad || wide < 10000;
}
"""


def test_wide_groups_stay_inside_the_planes(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    src = tmp_path / "rule.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-I", os.path.join(ROOT, "nscale_amd", "csrc"), "-o", str(tmp_path / "rule"), str(src)],
                   check=True)
    r = subprocess.run([str(tmp_path / "rule")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(9, 1), (13, 1), (17, 1), (1, 9), (1, 17), (9, 2), (2, 9)])
def test_thin_planes_match_the_oracle(shape):
    torch = pytest.importorskip("torch")
    from nscale_amd import gpu
    for seed in range(4):
        rng = np.random.default_rng(seed)
        bgr = rng.integers(0, 4, shape + (3,)).astype(np.uint8) * 60
        m = np.where(rng.random(shape) < 0.3, rng.integers(1, 4, shape), 0).astype(np.int32)
        print("thin plane", shape, seed, flush=True)
        got = gpu.cv_watershed(torch.from_numpy(bgr).cuda(), torch.from_numpy(m).cuda()).cpu().numpy()
        assert np.array_equal(got, o_cv_watershed(bgr, m))
