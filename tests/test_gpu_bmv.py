"""The batched mat-vec (csrc/bmv.hip) on one matrix of few rows a workgroup,
too wide for the whole-share form: Q4_K tiles straight from memory, Q6_K tiles
through LDS slots, from fp32 and from Q8 blocks, at the edges of its range
(rows per workgroup, superblock counts, activation rows, the first shape past
it), against the oracle's product."""
from __future__ import annotations

import numpy as np
import pytest

from test_bmv_layout import plan

pytestmark = pytest.mark.gpu

Q4, Q6 = 12, 14
SEED = 20261501


def check_plan(launch, rows, types, K, M, takes):
    """The launch is the one the CPU model of the indices checks."""
    cfg = plan(rows, types, K, 0, M)
    assert (cfg is not None) == takes
    if takes:
        kind = types[0] if len(types) == 1 else 0
        assert launch == f"bmv_kernel<{kind},0,{cfg[1]},{cfg[2]},0> grid={sum(cfg[0])}"


@pytest.mark.parametrize("qtype,K,N,M,takes", [
    (Q4, 9728, 2560, 3, True), (Q4, 9728, 2561, 8, True), (Q4, 9728, 4096, 4, True), (Q4, 9728, 4097, 5, False),
    (Q4, 12288, 700, 8, True), (Q4, 9728, 2560, 2, False), (Q4, 8192, 4096, 2, True), (Q4, 5888, 17, 2, True),
    (Q4, 8448, 300, 2, False), (Q6, 5888, 300, 2, False),
    (Q6, 9728, 2560, 3, True), (Q6, 9728, 2561, 4, True), (Q6, 9728, 2560, 5, True), (Q6, 9728, 2816, 8, True),
    (Q6, 9984, 257, 7, True), (Q6, 9728, 3329, 8, False), (Q6, 9728, 2560, 2, False),
    # M = 3, 4: to K = 8192, or above 8 rows a CU; M = 8, and 7 to K = 8192: above 3 rows a CU
    (Q6, 8192, 257, 4, True), (Q6, 8448, 2048, 3, False), (Q6, 8448, 2049, 4, True), (Q6, 5120, 768, 8, False),
    (Q6, 5120, 769, 8, True), (Q6, 5888, 257, 7, False), (Q6, 8448, 257, 7, True), (Q6, 5888, 257, 6, True),
    # LDS without room for the runs: 5 tiles on a wave for 3, 16 for 3, 53 for 4
    (Q6, 10240, 2560, 4, False), (Q6, 10240, 2560, 5, True), (Q6, 12288, 1024, 3, False), (Q6, 12288, 1024, 8, False),
    (Q4, 13568, 300, 3, False), (Q4, 13056, 300, 3, True),
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
    check_plan(launch, [N], [qtype], K, M, takes)
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


@pytest.mark.parametrize("K,shapes,M,takes", [
    (2560, [(Q4, 4096), (Q4, 1024), (Q6, 1024)], 3, True),   # q, k and v of both types
    (2560, [(Q4, 4096), (Q4, 1024), (Q6, 1024)], 8, True),
    (2560, [(Q4, 4096), (Q4, 1024), (Q4, 1024)], 2, True),   # all Q4_K: from M = 2
    (2560, [(Q4, 4096), (Q4, 1024), (Q4, 1024)], 7, True),
    (2560, [(Q4, 4096), (Q4, 1024), (Q6, 1024)], 2, False),
    (2560, [(Q6, 1700), (Q4, 33), (Q6, 1560), (Q4, 17)], 5, True),   # 13 rows of Q6_K a workgroup
    (2560, [(Q6, 1700), (Q4, 33), (Q6, 1700), (Q4, 17)], 5, False),  # past the CUs
    (1280, [(Q4, 8160), (Q4, 32)], 5, False),                # under 9 superblocks a row
    (2560, [(Q4, 8160), (Q4, 32)], 4, True),                 # 256 workgroups of 32 rows
    (2560, [(Q4, 8160), (Q4, 33)], 4, False),
    (2048, [(Q4, 4096), (Q4, 1024), (Q4, 1024)], 8, False),  # 8 superblocks a row, and 9
    (2304, [(Q4, 4096), (Q4, 1024), (Q4, 1024)], 2, True),
    (4096, [(Q4, 4096), (Q4, 1024), (Q4, 1024)], 2, True),   # 8 divides the superblocks: 24 rows a CU
    (4096, [(Q4, 4096), (Q4, 2048), (Q4, 33)], 4, False),
    (4096, [(Q4, 4096), (Q4, 2048), (Q4, 33)], 5, True),
    (6144, [(Q4, 4096), (Q4, 1024)], 3, True),               # past K = 4096: 20
    (6144, [(Q4, 4096), (Q4, 1024), (Q4, 33)], 3, False),
    (4096, [(Q4, 2048), (Q4, 512), (Q6, 512)], 3, False),    # and not both types
    (4352, [(Q4, 2048), (Q4, 512), (Q6, 512)], 3, True),
    (4352, [(Q4, 1024), (Q4, 512), (Q6, 512)], 3, False),    # both types: above 8 rows a CU
    (4352, [(Q4, 1024), (Q4, 513), (Q6, 512)], 4, True),
    (4352, [(Q4, 1024), (Q4, 512), (Q6, 512)], 5, True),
    (2560, [(Q4, 2048), (Q4, 1024), (Q6, 1024)], 3, False),  # below K = 3328: 16
    (2560, [(Q4, 2048), (Q4, 1025), (Q6, 1024)], 4, True),
    (3328, [(Q4, 2048), (Q4, 1024), (Q6, 1024)], 3, True),
    (4352, [(Q6, 700), (Q6, 700)], 3, True),                 # one type
    (8448, [(Q6, 700), (Q6, 700)], 4, False),
    (6400, [(Q4, 4096), (Q4, 1024)], 2, True),               # M = 2: the last K
    (6656, [(Q4, 4096), (Q4, 1024)], 2, False),
    (8192, [(Q4, 2048), (Q4, 2048)], 2, True),
    (8448, [(Q4, 2048), (Q4, 2048)], 2, False),
])
def test_several_matrices(gpu, oracle, K, shapes, M, takes):
    """One launch of 2..4 matrices on fp32 activations against the oracle's
    products, at the row counts where its plan ends (256 CUs)."""
    hosts = [oracle.synth_superblocks(q, N, K, SEED + 7 * i + N, 0.01, 0.01) for i, (q, N) in enumerate(shapes)]
    ws = [gpu.DeviceBuffer.from_array(h) for h in hosts]
    x = oracle.synth_normal(M * K, SEED + 60 + M)
    xd = gpu.DeviceBuffer.from_array(x)
    ys = [gpu.DeviceBuffer.from_array(np.full(M * N + 1, 123.0, np.float32)) for _, N in shapes]
    gpu.matmul_segments(xd, M, K, [(w, q, N, y) for w, (q, N), y in zip(ws, shapes, ys)])
    gpu.synchronize()
    launch = gpu.last_launch()
    print(f"[case] K={K} {shapes} M={M} launch {launch}", flush=True)
    assert launch.startswith("bmv_kernel") == takes
    check_plan(launch, [N for _, N in shapes], [q for q, _ in shapes], K, M, takes)
    for h, (q, N), y in zip(hosts, shapes, ys):
        out = y.download(np.float32)
        assert out[-1] == 123.0
        ref = oracle.reference_product(x, h, q, K, N).reshape(M, N)
        assert oracle.row_norm_error(out[:-1].reshape(M, N), ref) <= 1e-5


@pytest.mark.parametrize("K,N,M,ranges", [(8192, 4096, 8, 16), (8192, 4095, 8, 16), (9728, 4096, 3, 13)])
def test_runs_of_a_share_of_sixteen_rows(gpu, oracle, K, N, M, ranges):
    """256 CUs of exactly 16 rows are one row group each, planned like those of
    15 and 16: as many runs as the waves need."""
    w_host = oracle.synth_superblocks(Q4, N, K, SEED + 80, 0.01, 0.01)
    w = gpu.DeviceBuffer.from_array(w_host)
    x = oracle.synth_normal(M * K, SEED + 81)
    xd = gpu.DeviceBuffer.from_array(x)
    y = gpu.DeviceBuffer(4 * M * N)
    gpu.matmul(xd, w, Q4, K, N, y, M)
    gpu.synchronize()
    print(f"[case] K={K} N={N} M={M} launch {gpu.last_launch()}", flush=True)
    assert gpu.last_launch() == f"bmv_kernel<12,0,{ranges},1,0> grid=256"
    ref = oracle.reference_product(x, w_host, Q4, K, N).reshape(M, N)
    assert oracle.row_norm_error(y.download(np.float32).reshape(M, N), ref) <= 1e-5
