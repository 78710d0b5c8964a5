"""The GPU reordering's row copies at the edges of their splits.

Rows of at most 64 entries are copied 64 rows to a wave, longer ones in
chunks of 4,096 entries that may begin and end inside a row
(csrc/reorder.hip): degrees of 63, 64 and 65, row counts around a wave and a
work-group, hub rows shorter and longer than a chunk, graphs of one kind of
row only, and one context for graphs of falling and growing size.  The
permutation, the offsets and every entry are the host reordering's, exactly.
"""
import numpy as np
import pytest

from cwlb_amd import capi

pytestmark = pytest.mark.gpu

DEGREES = {
    "one_row": [7],
    "one_long": [65],
    "edge": [63, 64, 65] * 50 + [0] * 30,
    "chunks": [4095, 4096, 4097, 8192, 64, 65, 1] * 3,
    "hub": [50_000] + [1] * 300 + [0] * 100,
    "rows63": [3] * 63,
    "rows64": [64] * 64,
    "rows65": [65] * 65,
    "rows255": [2] * 255,
    "rows257": [1] * 257,
    "all_empty": [0] * 129,
    "tail_empty": [70] * 5 + [0] * 200,
}


@pytest.mark.parametrize("name", list(DEGREES))
def test_row_copies(gpu_ctx, name):
    import torch
    rng = np.random.default_rng(sum(name.encode()))
    d = rng.permutation(DEGREES[name])
    rp = np.concatenate([[0], np.cumsum(d)]).astype(np.int32)
    nnz = int(rp[-1])
    ci = rng.integers(0, 1 << 30, nnz).astype(np.int32)
    val = rng.random(nnz, dtype=np.float32)
    want = capi.reorder_by_degree(rp, ci, val)
    dev = lambda a: torch.from_numpy(a if a.size else np.zeros(1, a.dtype)).cuda()  # noqa: E731
    out = [torch.full((max(len(w), 1) + 1,), -7, dtype=torch.float32 if w.dtype == np.float32
                      else torch.int32, device="cuda") for w in want]
    gpu_ctx.reorder_device(len(d), nnz, dev(rp), dev(ci), dev(val), *out)
    for w, o in zip(want, out):
        got = o.cpu().numpy()
        assert np.array_equal(got[:len(w)], w) and got[-1] == -7
