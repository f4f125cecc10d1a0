"""The certified select for 257 to 8192 candidates per request
(SelectCertifiedKernel), its helper workgroups, and the exact kernels that
finish the requests it leaves undecided: ids equal to the oracle's, scores and
counts included."""
import numpy as np
import pytest

import _oracle as orc

pytestmark = pytest.mark.gpu


def run(gpu, keys, values, queries, offsets, ids, H, D, k):
    """One step (page size 1) and the oracle's ids and outputs."""
    cap, E, B = len(keys), H * D, len(queries)
    pool = gpu.DevicePagePool(H, D, 1, cap)
    all_ids = np.arange(cap, dtype=np.int32)
    ones = np.ones(cap, np.int32)
    pool.upload_pages(all_ids, ones, all_ids.astype(np.int64) * E, keys, values)
    with gpu.SparseContext(pool, k, B, len(ids), B * max(1, k)) as ctx:
        got = ctx.run_batch(queries, offsets, ids, output_mode=gpu.OUTPUT_OUTPUTS, want_ids=True)
        info = ctx.last_launch()
        chained = ctx.exact_rescored_pages()
    pool.close()
    summ = orc.pool_summaries(keys.reshape(cap, 1, E), ones, E)
    _, selected, outs = orc.sparse_batch(queries, keys.reshape(cap, 1, E),
                                         values.reshape(cap, 1, E), summ, ones, offsets, ids, H,
                                         D, 1, k)
    for r in range(B):
        assert got["selected"][r].tolist() == selected[r].tolist(), r
    assert orc.max_abs_diff(got["outputs"], outs) <= 1e-4
    return info, chained


@pytest.mark.parametrize("H,D,n,k", [
    (1, 64, [2049, 5], 1),
    (4, 64, [4096, 0, 300], 64),         # four candidates per thread
    (4, 64, [4097, 2048], 7),            # eight
    (3, 64, [8192, 8191], 1024),         # E = 192: no refinement; the most members
    (4, 64, [2000, 257], 257),           # up to 2048: sets of a pass of 256 and a bit more
    (4, 64, [2048, 600], 513),
    (4, 64, [2500], 1025),               # more members: the exact path
    (32, 128, [2600, 2100], 64),         # E = 4096: the float score passes
])
def test_random_batches(gpu, H, D, n, k):
    rng = np.random.default_rng(sum(n) + k)
    cap, E = max(n), H * D
    keys, values = (rng.standard_normal((cap, E)).astype(np.float32) for _ in range(2))
    queries = rng.standard_normal((len(n), E)).astype(np.float32)
    offsets = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    ids = np.concatenate([rng.permutation(cap)[:c] for c in n]).astype(np.int32)
    info, _ = run(gpu, keys, values, queries, offsets, ids, H, D, k)
    assert info["certified"] == (1 if k <= 1024 else 0)
    assert info["fused"] == 0 and info["wide"] == 0
    if H * D == 4096:  # the float score passes' launch: 224 workgroups, whole passes of 8
        per = -(-sum(n) // (224 * 8)) * 8
        assert info["score_pages_per_group"] == per == 24
        assert info["grid"] == len(n) * -(-max(n) // per)


@pytest.mark.parametrize("kind", ["near", "pairs", "many_equal", "zero_query", "infinite"])
def test_open_intervals(gpu, kind):
    """Near ties are refined or chained; ties beyond the flag list go to the
    exact kernels, for that request only."""
    rng = np.random.default_rng(5)
    H, D, k, n = 4, 64, 48, 3000
    E = H * D
    keys, values = (rng.standard_normal((n, E)).astype(np.float32) for _ in range(2))
    queries = rng.standard_normal((2, E)).astype(np.float32)
    order = np.argsort(-(keys @ queries[0]))
    if kind == "near":           # the 48th and 49th differ in one product's last bits
        keys[order[k]] = keys[order[k - 1]]
        keys[order[k], 7] = np.nextafter(keys[order[k], 7], np.float32(9))
    elif kind == "pairs":        # 40 pairs of equal pages around the boundary
        for j in range(k - 40, k + 40, 2):
            keys[order[j + 1]] = keys[order[j]]
    elif kind == "many_equal":   # more open candidates than the flag list holds
        keys[order[10:700]] = keys[order[10]]
    elif kind == "zero_query":
        queries[0] = 0.0
    else:
        keys[order[5], 3] = np.inf
        queries[0, 3] = 1.0
    offsets = np.array([0, n, 2 * n], np.int32)
    ids = np.concatenate([rng.permutation(n), rng.permutation(n)]).astype(np.int32)
    if kind == "infinite":
        queries[1, 3] = 0.5      # both finite-or-inf, no NaN: the order is defined
    _, chained = run(gpu, keys, values, queries, offsets, ids, H, D, k)
    if kind == "pairs":
        assert chained > 0
    if kind in ("many_equal", "zero_query"):
        # every page of the deferred request, and the other request's, if any
        assert n <= chained <= n + 64
    else:
        assert chained <= 2 * 128


def test_scores_of_a_device_step_stay_exact(gpu):
    import torch
    rng = np.random.default_rng(9)
    H, D, n, k = 4, 64, 2500, 8
    E = H * D
    keys, values = (rng.standard_normal((n, E)).astype(np.float32) for _ in range(2))
    query = rng.standard_normal((1, E)).astype(np.float32)
    pool = gpu.DevicePagePool(H, D, 1, n)
    ids = np.arange(n, dtype=np.int32)
    pool.upload_pages(ids, np.ones(n, np.int32), ids.astype(np.int64) * E, keys, values)
    dev = [torch.from_numpy(a).cuda() for a in (query, np.array([0, n], np.int32), ids)]
    out, scores = torch.zeros(1, E, device="cuda"), torch.zeros(n, device="cuda")
    want, _, _ = orc.sparse_batch(query, keys.reshape(n, 1, E), values.reshape(n, 1, E), keys,
                                  np.ones(n, np.int32), np.array([0, n], np.int32), ids, H, D, 1,
                                  k)
    with gpu.SparseContext(pool, k, 1, n, k) as ctx:
        torch.cuda.synchronize()
        ctx.run_batch_device(1, n, n, *[t.data_ptr() for t in dev], out.data_ptr(),
                             scores.data_ptr())
        ctx.device_status()
        assert np.array_equal(scores.cpu().numpy().view(np.uint32), want.view(np.uint32))
        # a request longer than the step was told selects nothing and is reported
        ctx.run_batch_device(1, n, 2100, *[t.data_ptr() for t in dev], out.data_ptr())
        with pytest.raises(gpu.InvalidArgument):
            ctx.device_status()
        assert not out.cpu().numpy().any()
    pool.close()


@pytest.mark.parametrize("n", [40, 300, 2100])
def test_a_chain_that_overflows(gpu, n):
    """A page whose fp32 chain passes the float range and stays infinite, though
    its sum is 0, scores above a page of a large finite score."""
    H, D, k = 4, 64, 1
    E = H * D
    rng = np.random.default_rng(n)
    keys, values = (rng.standard_normal((n, E)).astype(np.float32) for _ in range(2))
    summ = keys.copy()
    summ[7] = 0.0
    summ[7, 0] = 8e35
    summ[11] = 0.0
    summ[11, :4] = 3e38, 3e38, -3e38, -3e38
    query, ones, ids = np.ones((1, E), np.float32), np.ones(n, np.int32), np.arange(n, dtype=np.int32)
    offsets = np.array([0, n], np.int32)
    with gpu.DevicePagePool(H, D, 1, n) as pool:
        pool.upload_pages(ids, ones, ids.astype(np.int64) * E, keys, values, summ)
        with gpu.SparseContext(pool, k, 1, n, k) as ctx:
            got = ctx.run_batch(query, offsets, ids, output_mode=gpu.OUTPUT_OUTPUTS,
                                want_ids=True)
            assert ctx.last_launch()["certified"] == 1
    _, want, outs = orc.sparse_batch(query, keys.reshape(n, 1, E), values.reshape(n, 1, E), summ,
                                     ones, offsets, ids, H, D, 1, k)
    assert want[0].tolist() == [11]
    assert got["selected"][0].tolist() == [11]
    assert orc.max_abs_diff(got["outputs"], outs) <= 1e-4


@pytest.mark.parametrize("n", [[8192, 8192], [8192, 8191, 2], [8192, 1, 8191, 8192, 5]])
def test_exact_scores_of_many_pages(gpu, n):
    """Either side of the 16384 pages up to which exact scores come from the
    chains kernel."""
    H, D, k = 1, 64, 3
    E, cap = H * D, 8192
    rng = np.random.default_rng(len(n))
    keys, values = (rng.standard_normal((cap, E)).astype(np.float32) for _ in range(2))
    queries = rng.standard_normal((len(n), E)).astype(np.float32)
    offsets = np.concatenate([[0], np.cumsum(n)]).astype(np.int32)
    ids = np.concatenate([rng.permutation(cap)[:c] for c in n]).astype(np.int32)
    ones, all_ids = np.ones(cap, np.int32), np.arange(cap, dtype=np.int32)
    with gpu.DevicePagePool(H, D, 1, cap) as pool:
        pool.upload_pages(all_ids, ones, all_ids.astype(np.int64) * E, keys, values)
        with gpu.SparseContext(pool, k, len(n), len(ids), len(n) * k) as ctx:
            got = ctx.run_batch(queries, offsets, ids)
    scores, selected, _ = orc.sparse_batch(queries, keys.reshape(cap, 1, E),
                                           values.reshape(cap, 1, E), keys, ones, offsets, ids,
                                           H, D, 1, k)
    assert np.array_equal(got["scores"].view(np.uint32), scores.view(np.uint32))
    for r in range(len(n)):
        assert got["selected"][r].tolist() == selected[r].tolist(), r


def open_positions(mid, lo, hi, ids, k):
    """How many candidates the first-pass intervals leave open: members whose
    interval meets another's that can still be selected, and outsiders that meet
    a member's."""
    order = np.lexsort((ids, -mid))
    members, others = order[:k], order[k:]
    others = others[hi[others] >= lo[members].min()]
    some = np.concatenate([members, others])
    meets = (lo[some][:, None] <= hi[some]) & (lo[some] <= hi[some][:, None])
    np.fill_diagonal(meets, False)
    return int(meets[:k].any(1).sum() + meets[k:, :k].any(1).sum())


@pytest.mark.parametrize("batch,n,near,k", [
    (1, 300, 20, 12),   # more than the 8 that the selecting workgroup refines itself
    (3, 1900, 40, 40),
    (1, 2300, 12, 5),   # beyond 2048 candidates
    (2, 8192, 50, 30),
])
def test_helpers_refine_the_open_pages(gpu, batch, n, near, k):
    """near pages whose first-pass intervals overlap and whose refined ones do
    not: the helper workgroups settle them without an exact chain.  Where every
    wait for them gives up, the same pages take the chain and the ids stay."""
    H, D = 8, 128
    E = H * D
    rng = np.random.default_rng(n)
    scale = 1.0 / np.sqrt(np.float32(D))
    query = np.repeat(rng.standard_normal((1, E)).astype(np.float32), batch, axis=0)
    m = int(np.argmax(np.abs(query)))
    base = (0.2 * query[0] + 0.25 * rng.standard_normal(E)).astype(np.float32)
    summ = (0.25 * rng.standard_normal((n, E))).astype(np.float32)
    for j in range(near):
        summ[j] = base
        summ[j, m] += np.float32(j * 1e-4 / (query[0, m] * scale))
    keys, values = (rng.standard_normal((n, E)).astype(np.float32) for _ in range(2))
    ones, all_ids = np.ones(n, np.int32), np.arange(n, dtype=np.int32)
    ids = np.concatenate([rng.permutation(n) for _ in range(batch)]).astype(np.int32)
    offsets = np.arange(0, (batch + 1) * n, n, dtype=np.int32)
    _, want, outs = orc.sparse_batch(query, keys.reshape(n, 1, E), values.reshape(n, 1, E), summ,
                                     ones, offsets, ids, H, D, 1, k)
    with gpu.DevicePagePool(H, D, 1, n) as pool:
        pool.upload_pages(all_ids, ones, all_ids.astype(np.int64) * E, keys, values, summ)
        with gpu.SparseContext(pool, k, batch, batch * n, batch * k) as ctx:
            def step():
                got = ctx.run_batch(query, offsets, ids, output_mode=gpu.OUTPUT_OUTPUTS,
                                    want_ids=True)
                for r in range(batch):
                    assert got["selected"][r].tolist() == want[r].tolist(), r
                assert orc.max_abs_diff(got["outputs"], outs) <= 1e-4
                return ctx.exact_rescored_pages(reset=True)

            chained = step()
            info = ctx.last_launch()
            assert info["certified"] == 1 and info["fused"] == 0 and info["wide"] == 0
            bounds = [np.split(a, batch) for a in (*ctx.score_bounds(batch * n), ids)]
            opened = [open_positions(*request, k) for request in zip(*bounds)]
            print(f"[helpers] n={n} open={opened} chained={chained}", flush=True)
            assert all(8 < o <= 64 for o in opened) and chained == 0
            ctx.set_wait_limit(1 << 17, True)
            assert step() == sum(opened)
            ctx.set_wait_limit(1)
            assert step() <= sum(opened)   # (a helper may be that quick)
            ctx.set_wait_limit(1 << 17)
            assert step() == 0
