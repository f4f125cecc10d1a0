"""The certified score kernel for any E that is a multiple of 64
(ScoreBoundGenericKernel): every interval holds the exact sequential score, and
the selection is the oracle's, at the edges of its rows of 256 products, of the
pages a wave takes and of the query's place in LDS (64 KiB, E = 16384)."""
import numpy as np
import pytest

import _oracle as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,D,ps,k,lengths", [
    (1, 64, 1, 5, [2048, 1901, 1] + [2047] * 8),  # a quarter row; waves of 2 pages
    (3, 64, 2, 7, [70, 3]),                 # E = 192
    (4, 64, 2, 7, [130]),                   # E = 256: one whole row
    (5, 64, 2, 7, [130, 64]),               # E = 320: a row and a quarter
    (16, 128, 4, 9, [900, 17]),             # E = 2048: two steps of four rows
    (65, 64, 2, 3, [41, 8]),                # E = 4160: a quarter row in its own step
    (128, 128, 1, 3, [9, 5]),               # E = 16384: the largest query in LDS
    (129, 128, 1, 3, [9, 5]),               # E = 16512: read from memory
])
def test_bounds_hold_and_select_like_the_oracle(gpu, H, D, ps, k, lengths):
    batch = gpu.SyntheticBatch(H, D, ps, lengths, seed=H * D + len(lengths))
    E, B, total = H * D, len(lengths), batch.total_candidates
    pool = gpu.DevicePagePool(H, D, ps, batch.capacity)
    batch.upload(pool)
    empty = int(batch.cand_ids[0])
    pool.mark_free([empty])  # a page holding no tokens: an all-zero summary
    counts = batch.token_counts.copy()
    counts[empty] = 0
    summ = np.zeros((batch.capacity, E), np.float32)
    live = batch.live_page_ids()[1:]
    summ[live] = orc.pool_summaries(batch.key_pool, counts, E, live)
    with gpu.SparseContext(pool, k, B, total, B * k) as ctx:
        cert = ctx.run_batch(batch.queries, batch.cand_offsets, batch.cand_ids,
                             output_mode=gpu.OUTPUT_OUTPUTS, want_ids=True)
        mid, lo, hi = ctx.score_bounds(total)
        exact = ctx.run_batch(batch.queries, batch.cand_offsets, batch.cand_ids)
    assert np.all(lo <= exact["scores"]) and np.all(exact["scores"] <= hi)
    assert np.all(lo <= mid) and np.all(mid <= hi)
    scores, selected, outs = orc.sparse_batch(
        batch.queries, batch.key_pool, batch.value_pool, summ, counts, batch.cand_offsets,
        batch.cand_ids, H, D, ps, k)
    assert np.array_equal(exact["scores"].view(np.uint32), scores.view(np.uint32))
    for r in range(B):
        assert cert["selected"][r].tolist() == selected[r].tolist()
    assert orc.max_abs_diff(cert["outputs"], outs) <= 1e-4
    pool.close()


def test_device_queries_need_no_alignment(gpu):
    """A device step's queries at a 4-byte offset: the same ids and bits."""
    import torch
    H, D, ps, k = 8, 96, 4, 5
    batch = gpu.SyntheticBatch(H, D, ps, [900, 33], seed=2)
    E, total = H * D, batch.total_candidates
    pool = gpu.DevicePagePool(H, D, ps, batch.capacity)
    batch.upload(pool)
    offs, ids = (torch.from_numpy(a).cuda() for a in (batch.cand_offsets, batch.cand_ids))
    results = []
    with gpu.SparseContext(pool, k, 2, total, 2 * k) as ctx:
        for shift in (0, 1):
            room = torch.zeros(2 * E + 4, device="cuda")
            room[shift:shift + 2 * E] = torch.from_numpy(batch.queries.reshape(-1)).cuda()
            out = torch.zeros(2, E, device="cuda")
            sel = torch.full((2, k), -1, dtype=torch.int32, device="cuda")
            torch.cuda.synchronize()
            ctx.run_batch_device(2, total, batch.max_candidates, room.data_ptr() + 4 * shift,
                                 offs.data_ptr(), ids.data_ptr(), out.data_ptr(), 0,
                                 sel.data_ptr())
            ctx.device_status()
            results.append((out.cpu().numpy().view(np.uint32), sel.cpu().numpy()))
    assert np.array_equal(results[0][0], results[1][0])
    assert np.array_equal(results[0][1], results[1][1])
    pool.close()
