"""RMSNorm, residual_add and silu_multiply on the device against float64, at
the widths and counts where the 16-byte forms change (one value short of, at
and past whole quads, register rounds and workgroups), from pointers that are
only float-aligned, and in place; RMSNorm's sums in one order at every width."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

PAD = 1  # floats before each tensor: every pointer is 4-byte aligned only


def _put(qk, a):
    buf = qk.DeviceBuffer(4 * (a.size + 2 * PAD))
    buf.upload(np.concatenate([np.full(PAD, 7.0, np.float32), a.ravel(), np.full(PAD, 7.0, np.float32)]))
    return buf, buf.ptr + 4 * PAD


def _get(qk, buf, n):
    qk.synchronize()
    got = buf.download(np.float32)
    assert got[0] == 7.0 and got[n + PAD] == 7.0, "wrote outside the tensor"
    return got[PAD:n + PAD].astype(np.float64)


@pytest.mark.parametrize("width", [1, 4, 255, 1020, 1024, 1028, 2048, 2560, 2562, 3076, 4096, 4100, 8192, 8196])
@pytest.mark.parametrize("rows", [1, 3])
def test_rms_norm(gpu, width, rows):
    rng = np.random.default_rng(width + rows)
    x = (rng.standard_normal((rows, width)) * 10.0 ** rng.integers(-3, 4, (rows, 1))).astype(np.float32)
    scale = rng.standard_normal(width).astype(np.float32)
    bx, px = _put(gpu, x)
    bs, ps = _put(gpu, scale)
    bo, po = _put(gpu, np.zeros_like(x))
    gpu.rms_norm(px, ps, po, rows, width, 1e-6)
    x64 = x.astype(np.float64)
    want = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-6) * scale
    # the sum's roundings (a chain of at most width / 256 + 12 adds, halved by
    # the root), rsqrtf (2 ulp), the division, and two products: relative, per element
    bound = ((width / 256 + 12) / 2 + 6) * 2.0 ** -24
    got = _get(gpu, bo, x.size).reshape(rows, width)
    assert np.all(np.abs(got - want) <= bound * np.abs(want))
    gpu.rms_norm(px, ps, px, rows, width, 1e-6)  # in place
    assert np.array_equal(_get(gpu, bx, x.size).reshape(rows, width), got)


@pytest.mark.parametrize("width", [1, 255, 1000, 1024, 2048, 2560, 2562, 4096, 8192])
def test_rms_norm_sums_in_one_order_at_every_width(gpu, width):
    """A row and the same row padded with zeros to 4^k times its width, past
    the one-pass form: the sum is the same if its order is, the mean, eps and
    1 / root scale by powers of two, so the outputs differ by 2^k exactly."""
    rng = np.random.default_rng(width)
    rows, eps = 64, 2.0 ** -20
    k = 1
    while width * 4 ** k <= 8192:
        k += 1
    wide = width * 4 ** k
    x = rng.standard_normal((rows, width)).astype(np.float32)
    scale = rng.standard_normal(width).astype(np.float32)
    xw, sw = np.zeros((rows, wide), np.float32), np.zeros(wide, np.float32)
    xw[:, :width], sw[:width] = x, scale
    got = []
    for xi, si, w, e in ((x, scale, width, eps), (xw, sw, wide, eps / 4 ** k)):
        bx, px = _put(gpu, xi)
        bs, ps = _put(gpu, si)
        bo, po = _put(gpu, np.zeros_like(xi))
        gpu.rms_norm(px, ps, po, rows, w, e)
        got.append(_get(gpu, bo, xi.size).reshape(rows, w)[:, :width])
    assert np.array_equal(got[0] * 2 ** k, got[1])


@pytest.mark.parametrize("count", [1, 3, 4, 1023, 1024, 1027, 20480, 1024 * 16384 + 5])
def test_residual_add_and_silu(gpu, count):
    rng = np.random.default_rng(count)
    a = rng.standard_normal(count, dtype=np.float32) * 4
    b = rng.standard_normal(count, dtype=np.float32)
    ba, pa = _put(gpu, a)
    bb, pb = _put(gpu, b)
    bo, po = _put(gpu, np.zeros_like(a))
    gpu.silu_multiply(pa, pb, po, count)
    a64 = a.astype(np.float64)
    want = a64 / (1 + np.exp(-a64)) * b
    # expf within 2 ulp, the sum, the division (2.5 ulp) and the product: 8 roundings
    assert np.all(np.abs(_get(gpu, bo, count) - want) <= 8 * 2.0 ** -23 * np.abs(want))
    gpu.residual_add(pa, pb, count)
    assert np.array_equal(_get(gpu, ba, count), (a + b).astype(np.float64))
