"""GROUP_NORM and NORM with their chains on the device against the oracle's
restatement of norm.cc (the same statistics in the same precisions), and
against float64 for the normalisation itself."""

import numpy as np
import pytest
import torch

import oracle_lib as orc
import sdhip
from helpers import dev, normal, rng, uniform, unwritten

# Fused and apart within 1e-6 of the largest output, as the reference's
# fusion tests hold them (ops_test.cc:567-637); the statistics here are the
# reference's own, so the outputs agree to a few units in the last place.
CLOSE = 1e-6


def chain_ref(y, gamma, beta, silu):
    out = y * gamma
    out = out + beta
    if silu:
        out = orc.silu(out)
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("shape,groups,eps,silu", [
    ((2, 64, 20, 36), 32, 1e-6, True),     # ops_test.cc:1062-1075
    ((1, 30, 7, 13), 10, 1e-5, True),      # rows of no multiple of eight
    ((2, 1280, 8, 8), 32, 1e-5, True),     # cfg3a's GroupNorm + SiLU
    ((2, 1280, 32, 32), 32, 1e-5, True),   # cfg3b's
    ((1, 30, 7, 13), 7, 1e-5, False),      # groups of ceil(30/7) = 5 channels, the last of none
    ((1, 128, 128, 128), 32, 1e-6, True),  # groups of many slices
])
def test_group_norm(gpu, shape, groups, eps, silu):
    r = rng(sum(shape) + groups)
    x = uniform(r, shape, 3.0)
    c = shape[1]
    gamma = normal(r, (1, c, 1, 1), 1.0, 0.1)
    beta = normal(r, (1, c, 1, 1), 0.0, 0.1)
    x_d, g_d, b_d = dev(x, gpu), dev(gamma, gpu), dev(beta, gpu)
    y = unwritten(shape, gpu)
    steps = [("mul", g_d), ("add", b_d)] + ([("silu", None)] if silu else [])
    sdhip.group_norm(x_d, y, groups, eps, sdhip.epilogue(steps))
    torch.cuda.synchronize()
    want = chain_ref(orc.group_norm(x, groups, eps), gamma, beta, silu)
    got = y.cpu().numpy()
    assert np.isfinite(got).all()
    diff = np.abs(got - want).max() / np.abs(want).max()
    print(f"group_norm {shape}/{groups}: {diff:.3g} of the largest")
    assert diff <= CLOSE


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 64, 32, 32), (1, 30, 7, 13)])
def test_group_norm_operand_per_position(gpu, shape):
    """A chain operand that varies along the rows (a residual of the output's
    shape, and one broadcast over channels): the per-element path."""
    r = rng(7 + sum(shape))
    x = uniform(r, shape, 2.0)
    res = uniform(r, shape, 1.0)
    rows = uniform(r, (1, 1, shape[2], shape[3]), 1.0)
    x_d, res_d, rows_d = dev(x, gpu), dev(res, gpu), dev(rows, gpu)
    y = unwritten(shape, gpu)
    sdhip.group_norm(x_d, y, 16 if shape[1] % 16 == 0 else 10, 1e-5,
                     sdhip.epilogue([("add", res_d), ("mul", rows_d)]))
    torch.cuda.synchronize()
    want = (orc.group_norm(x, 16 if shape[1] % 16 == 0 else 10, 1e-5) + res) * rows
    got = y.cpu().numpy()
    diff = np.abs(got - want).max() / np.abs(want).max()
    print(f"group_norm per position {shape}: {diff:.3g}")
    assert diff <= CLOSE


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(2, 77, 320), (2, 988, 1280), (3, 5, 33)])
def test_norm(gpu, shape):
    r = rng(sum(shape))
    x = uniform(r, shape, 3.0)
    n = shape[-1]
    gamma = normal(r, (n,), 1.0, 0.1)
    beta = normal(r, (n,), 0.0, 0.1)
    x_d, g_d, b_d = dev(x, gpu), dev(gamma, gpu), dev(beta, gpu)
    y = unwritten(shape, gpu)
    sdhip.norm(x_d, y, 1e-5, sdhip.epilogue([("mul", g_d), ("add", b_d)]))
    torch.cuda.synchronize()
    want = chain_ref(orc.norm(x, 1e-5), gamma, beta, False)
    got = y.cpu().numpy()
    diff = np.abs(got - want).max() / np.abs(want).max()
    print(f"norm {shape}: {diff:.3g} of the largest")
    assert diff <= CLOSE


@pytest.mark.gpu
@pytest.mark.parametrize("shape,view", [((2, 50, 4), False), ((1, 7, 2048), False), ((1, 9, 2052), False),
                                        ((2, 300, 640), True), ((3, 33, 1280), True), ((2, 64, 320), False),
                                        ((1, 7, 128), False), ((2, 33, 200), True), ((2, 65, 320), True),
                                        ((1, 5, 324), True), ((2, 33, 600), False)],
                         ids=lambda v: "x".join(map(str, v)) if isinstance(v, tuple) else str(v))
def test_norm_rows_and_operands(gpu, shape, view):
    """NORM over rows of 4 .. 2048 numbers a float4 at a time (up to 320:
    four rows a wave, 16 lanes each, row counts no multiple of four among
    them; 2052: the general form), the input a view whose rows lie further apart where
    `view`; the chain a per-column scale, a residual of the output's shape
    starting one number past a 16-byte boundary (read a number at a time), a
    per-row scale (broadcast along the row) and the SiLU."""
    r = rng(sum(shape) + view)
    n = shape[-1]
    full = uniform(r, shape[:-1] + (n + 8,), 3.0)
    x = np.ascontiguousarray(full[..., :n])
    gamma = normal(r, (n,), 1.0, 0.1)
    res_full = uniform(r, shape[:-1] + (n + 4,), 1.0)
    res = np.ascontiguousarray(res_full[..., 1:n + 1])
    per_row = normal(r, shape[:-1] + (1,), 1.0, 0.5)
    x_d = dev(full, gpu)[..., :n] if view else dev(x, gpu)
    g_d, pr_d = dev(gamma, gpu), dev(per_row, gpu)
    r_d = dev(res_full, gpu)[..., 1:n + 1]
    y = unwritten(shape, gpu)
    sdhip.norm(x_d, y, 1e-5, sdhip.epilogue([("mul", g_d), ("add", r_d), ("mul", pr_d), ("silu", None)]))
    torch.cuda.synchronize()
    want = orc.silu((orc.norm(x, 1e-5) * gamma + res) * per_row)
    got = y.cpu().numpy()
    diff = np.abs(got - want).max() / np.abs(want).max()
    print(f"norm {shape} view={view}: {diff:.3g} of the largest")
    assert diff <= CLOSE


@pytest.mark.gpu
@pytest.mark.parametrize("shape,groups,offset", [
    ((1, 32, 256, 256), 1, 0),     # one group: more slices than a wave has lanes
    ((2, 34, 65, 67), 2, 0),       # planes of no multiple of 4, the last slice short
    ((1, 48, 64, 64), 3, 1),       # rows that start between quads
    ((1, 4, 512, 512), 2, 0),      # slices read twice
])
def test_group_norm_slices(gpu, shape, groups, offset):
    """Groups of several slices whose means differ by hundreds of their
    deviations: the squares about each slice's own mean, put together, against
    float64.  A number of 1000 is rounded by 3e-5 in single precision and the
    mean likewise; over the group's deviation, about 300, that is 2e-7."""
    r = rng(sum(shape) + groups)
    n = int(np.prod(shape))
    x = (np.linspace(-500.0, 500.0, n) + r.standard_normal(n)).astype(np.float32).reshape(shape)
    flat = torch.empty(n + 4, device=gpu)
    x_d = flat[offset:offset + n].view(shape)
    x_d.copy_(torch.from_numpy(x))
    y = unwritten(shape, gpu)
    sdhip.group_norm(x_d, y, groups, 1e-5)
    torch.cuda.synchronize()
    want = torch.nn.functional.group_norm(torch.from_numpy(x).double(), groups, eps=1e-5).numpy()
    diff = np.abs(y.cpu().numpy() - want).max()
    print(f"group_norm slices {shape}/{groups}: {diff:.3g}")
    assert diff <= 1e-6


@pytest.mark.gpu
@pytest.mark.parametrize("shape,groups,offset", [
    ((1, 64, 256, 256), 32, 0),    # a slice's numbers held in registers
    ((1, 6, 301, 211), 3, 1),      # read twice, between quads
])
def test_group_norm_of_great_numbers(gpu, shape, groups, offset):
    """Numbers of +-1.5e19, whose squares about the group's mean (near 0) fit
    single precision and, in slices that lie off it, about the slice's own mean
    (+-7.5e18) do not.  Against float64: the difference, the scale and their
    product round once each, outputs up to 1.2."""
    r = rng(sum(shape))
    n = int(np.prod(shape))
    share = np.where(np.arange(n) // (n // groups // 2) % 2 == 0, 0.75, 0.25)  # halves of a group
    x = np.where(r.random(n) < share, np.float32(-1.5e19), np.float32(1.5e19)).astype(np.float32).reshape(shape)
    flat = torch.empty(n + 4, device=gpu)
    x_d = flat[offset:offset + n].view(shape)
    x_d.copy_(torch.from_numpy(x))
    y = unwritten(shape, gpu)
    sdhip.group_norm(x_d, y, groups, 1e-5)
    torch.cuda.synchronize()
    want = torch.nn.functional.group_norm(torch.from_numpy(x).double(), groups, eps=1e-5).numpy()
    diff = np.abs(y.cpu().numpy() - want).max()
    print(f"group_norm of great numbers {shape}/{groups}: {diff:.3g}")
    assert diff <= 1e-6
