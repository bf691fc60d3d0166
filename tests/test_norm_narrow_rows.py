"""Normalization of images whose rows are apart (crops): groups of four pixels numbered over the rows.  On the CPU: the
rule that finds a group's row (nscale_amd/csrc/normalize_rules.hpp) against division.  On the GPU: crops
of every small width give the bytes and the statistics that the same pixels give without gaps."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from tests._lib import ROOT

PROGRAM = r"""
#include <cstdio>
#include <random>
#include "normalize_rules.hpp"
int main() {
    std::mt19937_64 rng(1);
    long long bad = 0, n = 0;
    auto one = [&](unsigned long long q, unsigned long long d) {
        ++n;
        if (nsc::row_of(q, nsc::row_magic(d)) != q / d && bad++ < 5) std::printf("%llu / %llu\n", q, d);
    };
    for (unsigned long long d = 1; d <= 300; ++d)
        for (unsigned long long q = 0; q < 3000; ++q) one(q, d);
    for (int k = 0; k < 2000000; ++k) {
        const unsigned long long d = 1 + (rng() >> 35 >> rng() % 29), top = (1ull << 35) / d + 1;
        const unsigned long long y = rng() % top, q = y * d;
        if (q >= 1ull << 35) continue;
        one(q, d);
        one(q + d - 1, d);
        if (q) one(q - 1, d);
    }
    std::printf("%lld of %lld\n", bad, n);
    return bad != 0 || n < 5000000;
}
"""


def test_row_of_a_group(tmp_path):
    if shutil.which("g++") is None:
        pytest.skip("no host compiler")
    src = tmp_path / "rule.cpp"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", os.path.join(ROOT, "nscale_amd", "csrc"), "-o", str(tmp_path / "rule"), str(src)],
                   check=True)
    r = subprocess.run([str(tmp_path / "rule")], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("w", [1, 2, 3, 4, 5, 7, 8, 63, 100, 255, 257, 513, 2047, 2049])
def test_crops_match_their_copies(w):
    torch = pytest.importorskip("torch")
    from nscale_amd import gpu
    from nscale_amd.synth import synth_he
    h = 77
    big = torch.from_numpy(synth_he(h + 2, w + 9, w)).cuda()
    mean, std = (-0.4, 0.06, 0.03), (0.2, 0.03, 0.02)
    for x0 in (0, 1, 6):
        crop = big[1:1 + h, x0:x0 + w]
        print("crop", w, x0, flush=True)
        dense = crop.contiguous()
        m0, s0, n0 = gpu.normalization_target_parameters(dense)
        m1, s1, n1 = gpu.normalization_target_parameters(crop)
        # sums of doubles in another order, rounded to float once
        assert n0 == n1 and np.allclose(m0, m1, rtol=1e-6, atol=0, equal_nan=True)
        assert np.allclose(s0, s1, rtol=1e-5, atol=1e-7, equal_nan=True)
        if n0 < 2:
            continue
        a = gpu.normalization(dense, mean, std)
        b = gpu.normalization(crop, mean, std)
        # the statistics may differ in their last float bit, which moves a value by far less than a level
        assert int((a.int() - b.int()).abs().max()) <= 1
        same = big.clone()
        inner = same[1:1 + h, x0:x0 + w]
        gpu.normalization(inner, mean, std, out=inner)
        assert torch.equal(inner, b)
        same[1:1 + h, x0:x0 + w] = crop
        assert torch.equal(same, big)
