"""Column phases over the band-by-band copy of the feature matrix.

Where a feature slice's rows are not whole 128-byte lines and the graph
gathers each feature row often enough, a phased call gathers from a padded
copy of H (csrc/col_phases.hip).  Widths and slice counts with and without
one, phase counts that divide the feature rows and that do not (64 phases of
200 rows), chains that begin and end inside a row (those rows come from H
itself), a column outside the feature matrix, and several windows' worth of
rows in one run.  Tolerance: the parity contract (32-bit sums of at most 150
terms, band by band).
"""
import dataclasses

import numpy as np
import pytest
import torch

import oracle
from conftest import SKEWED_COSTS
from cwlb_amd import capi, synth, workloads
from test_gpu_spmm import check, custom_graph, dev, run_gpu

pytestmark = pytest.mark.gpu

N, H_ROWS = 300, 200


def graph(rng):
    degs = np.concatenate([rng.integers(40, 60, N - 60), [0] * 20, [1] * 20, [150] * 20])
    rp = np.concatenate([[0], np.cumsum(degs)])
    ci = np.concatenate([np.sort(rng.choice(H_ROWS, d, replace=False)) for d in degs])
    assert len(ci) >= 32 * H_ROWS  # the copy's rule
    return custom_graph(rp, ci, 1.0 - rng.random(len(ci), dtype=np.float32))


@pytest.fixture
def phased(gpu_ctx):
    yield gpu_ctx
    gpu_ctx.set_schedule(0, 0)
    gpu_ctx.set_column_phases(0)
    gpu_ctx.set_lane_tiling(0)


@pytest.mark.parametrize("K", [4, 20, 64, 100, 128, 300, 600])
@pytest.mark.parametrize("SL", [1, 2, 4, 8])
def test_phase_copy(phased, K, SL, rng):
    g = graph(rng)
    H = synth.features(H_ROWS, K, 3)
    for S in (7, 200):
        p = workloads.prepare(g, SKEWED_COSTS, S)
        ref = oracle.spmm_mean_f32(p.row_ptr, p.col_idx, p.val, p.origin, H, p.tasks)
        for P, m, tiling in ((2, 0, 1), (3, 1, 2), (16, 16, 2), (64, 1 << 20, 1)):
            phased.set_schedule(m, SL)
            phased.set_column_phases(P)
            phased.set_lane_tiling(tiling)
            got, _ = run_gpu(phased, p, H)
            check(got, ref)


def test_partial_chain_and_bad_column(phased, rng):
    g = graph(rng)
    K = 100
    H = synth.features(H_ROWS, K, 5)
    p = workloads.prepare(g, SKEWED_COSTS, 7)
    phased.set_schedule(8, 4)
    phased.set_column_phases(16)
    inside = [i for i, t in enumerate(p.tasks) if t[2] > 0]
    part = dataclasses.replace(p, tasks=p.tasks[inside[3]:inside[-4]])
    ref = oracle.spmm_mean_f32(p.row_ptr, p.col_idx, p.val, p.origin, H, part.tasks)
    got, _ = run_gpu(phased, part, H, flags=capi.ZERO_OUTPUT, c_fill=7.0)
    check(got, ref)
    bad = p.col_idx.copy()
    bad[len(bad) // 2] = H_ROWS
    C = torch.zeros((N, K), device="cuda")
    with pytest.raises(capi.CwlbError) as e:
        phased.spmm(dev(p.row_ptr), dev(bad), dev(p.val), dev(p.origin), N, p.nnz, dev(H), H_ROWS,
                    K, dev(np.ascontiguousarray(p.tasks, np.int32).reshape(-1)), len(p.tasks), C)
    assert e.value.status == capi.INVALID_ARG
