"""gelu_erf (clarus_amd/csrc/common.hpp), the GELU of every epilogue and gate: the fit on the CPU, the kernel's values on
the GPU."""
from __future__ import annotations

import os
import re

import numpy as np
import pytest
import torch
from scipy.special import ndtr

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "clarus_amd", "csrc", "common.hpp")
FIT = 3.3e-8  # of max(Phi(-a), 1e-2), with the coefficients as fp32 holds them


def test_gelu_fit():
    """Phi(-a) = exp(-a^2 / 2) N(a) / D(a) with the source's coefficients, in 64 bits, within the bounds it states."""
    with open(SRC) as f:
        body = f.read().split("gelu_erf(float x) {")[1].split("}")[0]
    coef = [[float(np.float32(v)) for v in re.findall(r"([0-9.]+)f\b", line)]
            for line in body.splitlines() if line.strip().startswith("const float n") or line.strip().startswith("const float d")]
    assert [len(c) for c in coef] == [4, 5]
    a = np.linspace(0, 20, 400001)
    got = np.exp(-a * a / 2) * np.polyval(coef[0], a) / np.polyval(coef[1], a)
    ref = ndtr(-a)
    assert (np.abs(got - ref) / np.maximum(ref, 1e-2)).max() <= FIT
    assert np.abs(got - ref).max() <= 6.5e-9
    for most, rel in ((3, 5e-8), (4, 8.1e-7), (6, 1.65e-5), (10, 1.25e-4)):
        assert np.abs(got / ref - 1)[a <= most].max() <= rel


@pytest.fixture(scope="module")
def hip_f32(gpu_device):
    from clarus_amd.hip_ops import HipOps
    return HipOps(torch.float32, gpu_device)


@pytest.mark.gpu
@pytest.mark.parametrize("c", [256, 264])
def test_gelu_values(c, hip_f32):
    """GELU of single values: images of one pixel through a depthwise conv whose only tap is a centre of 1, on the tiled and
    the per-pixel kernel. Phi(-a) is off by the fit and by fp32 steps: 2 a^2 half-ulps from the exponent's argument, 8 from the
    rest of its product; then two roundings of the result. Below 2^-120, exp2 may flush to 0."""
    from clarus_amd import _lib
    x = torch.cat([torch.linspace(-14, 14, 97 * 88), torch.tensor([0.0, -0.0, 1e-30, -1e-30, 20.5, -20.5, 3e38, -3e38])])
    special = torch.tensor([float("inf"), float("-inf"), float("nan")])
    full = torch.cat([x, special, torch.zeros(-(len(x) + 3) % c)]).view(-1, 1, 1, c)
    tap = torch.zeros(c, 1, 3, 3)
    tap[:, 0, 1, 1] = 1
    got = hip_f32.dwconv(full.cuda(), tap.cuda(), None, act="gelu")
    assert _lib.last_kernel().startswith("dw_tile_kernel" if c <= 256 else "dwconv3x3_kernel"), _lib.last_kernel()
    got = got.cpu().flatten()
    v = x.double().numpy()
    phi, ref = ndtr(-np.abs(v)), v * ndtr(v)
    bound = np.abs(v) * (FIT * np.maximum(phi, 1e-2) + phi * 2.0 ** -24 * (8 + 2 * v * v)) + 2.0 ** -23 * np.abs(ref) + 2.0 ** -120
    bad = np.abs(got[:len(v)].double().numpy() - ref) > bound
    assert not bad.any(), (v[bad][:5], got[:len(v)].numpy()[bad][:5], ref[bad][:5])
    inf, minus, nan = got[len(v):len(v) + 3]
    assert inf == float("inf") and torch.isnan(minus) and torch.isnan(nan)  # as torch.nn.functional.gelu
