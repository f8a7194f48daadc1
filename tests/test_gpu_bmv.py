"""The batched mat-vec (csrc/bmv.hip) on one matrix of few rows a workgroup,
too wide for the whole-share form: Q4_K tiles straight from memory, Q6_K tiles
through LDS slots, from fp32 and from Q8 blocks, at the edges of its range
(rows per workgroup, superblock counts, activation rows, the first shape past
it), against the oracle's product."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14
SEED = 20261501


@pytest.mark.parametrize("qtype,K,N,M,takes", [
    (Q4, 9728, 2560, 3, True), (Q4, 9728, 2561, 8, True), (Q4, 9728, 4096, 4, True), (Q4, 9728, 4097, 5, False),
    (Q4, 12288, 700, 8, True), (Q4, 9728, 2560, 2, False),
    (Q6, 9728, 2560, 3, True), (Q6, 9728, 2561, 4, True), (Q6, 9728, 2560, 5, True), (Q6, 9728, 2816, 8, True),
    (Q6, 9984, 257, 7, True), (Q6, 9728, 3329, 8, False), (Q6, 9728, 2560, 2, False),
])
def test_one_wide_matrix(gpu, oracle, qtype, K, N, M, takes):
    w_host = oracle.synth_superblocks(qtype, N, K, SEED + N, 0.01, 0.01)
    w = gpu.DeviceBuffer.from_array(w_host)
    x = oracle.synth_normal(M * K, SEED + M)
    xd = gpu.DeviceBuffer.from_array(x)
    y = gpu.DeviceBuffer.from_array(np.full(M * N + 2, 123.0, np.float32))
    gpu.matmul(xd, w, qtype, K, N, y, M, y_offset=4)
    gpu.synchronize()
    launch = gpu.last_launch()
    print(f"[case] type={qtype} K={K} N={N} M={M} launch {launch}", flush=True)
    assert launch.startswith("bmv_kernel") == takes
    out = y.download(np.float32)
    assert out[0] == 123.0 and out[-1] == 123.0
    got = out[1:-1].reshape(M, N)
    # fp32 sums of exact integer dots: the bar of the other mat-vec tests
    ref = oracle.reference_product(x, w_host, qtype, K, N).reshape(M, N)
    assert oracle.row_norm_error(got, ref) <= 1e-5
    if takes:  # the same codes and scales from Q8 blocks: the same bits
        q8 = gpu.DeviceBuffer(M * K // 32 * gpu.Q8_BLOCK_BYTES)
        gpu.quantize_q8(xd, M, K, q8)
        gpu.matmul_q8(q8, w, qtype, K, N, y, M)
        gpu.synchronize()
        assert gpu.last_launch().startswith("bmv_kernel")
        assert np.array_equal(y.download(np.float32)[:M * N].reshape(M, N), got)
