"""The aggregation kernel's row window, stage and zero stretches at their edges.

A wave reads its rows 64 at a time into an LDS window and their nonzeros 256
at a time into an LDS stage (csrc/spmm_mean.hip).  The graphs here put what
can go wrong on those edges: 63, 64 and 65 rows of a degree, stretches of
empty rows that end before, at and after a window's end, chunks that begin
inside a stage and end outside it, hub rows of 255, 256, 257 and 513
nonzeros, degrees on both sides of the length at which a chunk runs on all
slots (2 to 64, by the width), and runs of one task and of the whole graph.
Tolerance: the parity contract, 1e-6 + 1e-5 |ref| (32-bit sums of at most
600 terms in another order stay below 600 * 2^-24 = 3.6e-5 of the sum of
magnitudes; the mean of uniform features is compared at 1e-5 relative and
1e-6 absolute, above the 3e-8 that is measured).
"""
import numpy as np
import pytest

import oracle
from conftest import SKEWED_COSTS
from cwlb_amd import capi, synth, workloads
from test_gpu_spmm import check, custom_graph, run_gpu

pytestmark = pytest.mark.gpu

DEGREES = {
    "windows": [1] * 63 + [2] * 64 + [3] * 65 + [5] * 129,
    "empty1": [0] + [4] * 70,
    "empty63": [0] * 63 + [1, 7, 33],
    "empty64": [0] * 64 + [2] * 3,
    "empty65": [0] * 65 + [17] * 20 + [255, 256, 257],
    "empty200": [0] * 200 + [1] * 5 + [513, 600],
    "all_empty": [0] * 130,
    "stage": [31, 32, 33] * 12 + [63, 64, 65] * 3 + [100] * 4 + [255, 256, 257, 513],
    "slots": sorted([1, 2, 3, 4, 7, 8, 9, 15, 16, 17, 31, 32, 33] * 5),
}


def graph(name):
    rng = np.random.default_rng(sum(name.encode()))
    degs = np.array(DEGREES[name])
    n = len(degs)
    h_rows = max(n, 700)
    rp = np.concatenate([[0], np.cumsum(degs)])
    ci = np.concatenate([np.sort(rng.choice(h_rows, d, replace=False)) for d in degs] +
                        [np.zeros(0, np.int64)])
    return custom_graph(rp, ci, 1.0 - rng.random(len(ci), dtype=np.float32)), h_rows


@pytest.mark.parametrize("K", [1, 2, 3, 4, 5, 6, 7, 18, 32, 50, 75, 96, 128, 253, 257, 600, 1027, 1028, 2050])
@pytest.mark.parametrize("name", list(DEGREES))
def test_window_edges(gpu_ctx, name, K):
    g, h_rows = graph(name)
    H = synth.features(h_rows, K, 11)
    for S in (5, 300):
        p = workloads.prepare(g, SKEWED_COSTS, S)
        ref = oracle.spmm_mean_f32(p.row_ptr, p.col_idx, p.val, p.origin, H, p.tasks)
        empty = p.origin[np.diff(p.row_ptr) == 0]
        for m in (1, 0, 1 << 20):
            gpu_ctx.set_schedule(m, 0)
            try:
                # A NaN-filled C: every row is written; with the empty rows
                # kept, those alone are left.
                got, _ = run_gpu(gpu_ctx, p, H, large_k=K > 1024)
                check(got, ref)
                kept, _ = run_gpu(gpu_ctx, p, H, flags=capi.KEEP_EMPTY_ROWS, large_k=K > 1024)
            finally:
                gpu_ctx.set_schedule(0, 0)
            want = ref.copy()
            want[empty] = np.nan
            check(kept, want)
