"""The single-launch step's long form (FusedStepKernel<true, 512>): batches
whose largest request has 257 to 512 candidates, against the oracle, at the
edges of its eight candidate slots, of its selection forms and of the rule
that picks it."""
import numpy as np
import pytest

import _oracle as orc

pytestmark = pytest.mark.gpu

H, D = 32, 128
E = H * D


def check(gpu, counts, ps, k, edit=None, seed=0, fused=1):
    """One step over requests of counts[r] pages of ps tokens."""
    rng = np.random.default_rng(seed + sum(counts) + k)
    cap, B = sum(counts), len(counts)
    keys, values = (rng.standard_normal((cap, ps, E), dtype=np.float32) for _ in range(2))
    queries = rng.standard_normal((B, E), dtype=np.float32)
    offsets = np.concatenate([[0], np.cumsum(counts)]).astype(np.int32)
    ids = rng.permutation(cap).astype(np.int32)
    if edit is not None:
        edit(rng, keys, queries, offsets, ids)
    tokens = np.full(cap, ps, np.int32)
    pool = gpu.DevicePagePool(H, D, ps, cap)
    pool.upload_pages(np.arange(cap), tokens, np.arange(cap, dtype=np.int64) * ps * E, keys, values)
    with gpu.SparseContext(pool, k, B, cap, B * k) as ctx:
        got = ctx.run_batch(queries, offsets, ids, output_mode=gpu.OUTPUT_OUTPUTS, want_ids=True)
        info = ctx.last_launch()
        again = ctx.run_batch(queries, offsets, ids, output_mode=gpu.OUTPUT_OUTPUTS, want_ids=True)
    pool.close()
    assert info["fused"] == fused and info["wide"] == 1 - fused, info
    summ = orc.pool_summaries(keys, tokens, E)
    _, selected, outs = orc.sparse_batch(queries, keys, values, summ, tokens, offsets, ids, H, D,
                                         ps, k)
    for r in range(B):
        assert got["selected"][r].tolist() == selected[r].tolist(), r
        assert again["selected"][r].tolist() == selected[r].tolist(), r
    assert orc.max_abs_diff(got["outputs"], outs) <= 1e-4
    assert np.array_equal(got["outputs"].view(np.uint32), again["outputs"].view(np.uint32))


@pytest.mark.parametrize("counts,ps,k,fused", [
    ([257, 1, 64, 65, 0, 300], 16, 8, 1),         # the form's first candidate count
    ([512, 511, 449, 448, 385, 384, 320], 1, 32, 1),  # every slot count, one-wave selection
    ([512, 33, 256, 130, 321, 5], 1, 33, 1),      # ballot ranks
    ([500, 64, 512, 63, 257, 400, 3, 2, 1], 4, 64, 1),   # the most members; k above counts
    ([300] * 40, 1, 1, 1),                        # eight heads per workgroup
    ([513, 20, 20, 20, 20, 20], 1, 8, 0),         # one candidate too many: the wide step
    ([300, 20, 20, 20, 20, 20], 1, 65, 0),        # too many members
    ([300, 20, 20, 20, 20, 20], 16, 17, 0),       # too many tokens
    ([300, 20, 20, 20, 20], 1, 8, 0),             # too few requests
    ([340] * 6, 4, 33, 1),                        # more than 128 tokens: few pages on average
    ([341] + [340] * 5, 4, 33, 0),                # one more
    ([341] * 6, 4, 32, 1),
    ([512] + [224] * 8, 4, 33, 1),
    ([512] + [224] * 7 + [225], 4, 33, 0),
    ([300] * 16, 4, 33, 1),
])
def test_long_form_matches_oracle(gpu, counts, ps, k, fused):
    check(gpu, counts, ps, k, fused=fused)


@pytest.mark.parametrize("k", [8, 40])
@pytest.mark.parametrize("kind", ["near", "equal", "zero_query"])
def test_long_form_settles_open_intervals(gpu, k, kind):
    def edit(rng, keys, queries, offsets, ids):
        mine = ids[offsets[2]:offsets[3]]
        if kind == "zero_query":
            queries[2] = 0.0
            return
        order = mine[np.argsort(-(keys[mine, 0] @ queries[2]), kind="stable")]
        for j in (k - 1, k + 1, 0):   # pairs across the line, below it and at the top
            keys[order[j + 1]] = keys[order[j]]
            if kind == "near":
                keys[order[j + 1], 0, 5] = np.nextafter(keys[order[j + 1], 0, 5], np.float32(9))

    check(gpu, [40, 257, 500, 300, 10, 512], 1, k, edit, seed=3)
