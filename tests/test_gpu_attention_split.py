"""Attention whose heads are spread over several workgroups (attention.hip):
pieces at their edges, the scratch left clean for the next launch, launches on
several streams and from several threads, and a captured step.

Tolerance: outputs within 1e-4 of the oracle, the path's bar.  The rounding
bound behind it: a logit is a dot of D <= 256 products summed in fp32 along
paths of at most D/LPT + 6 additions, so its error is below
26 * 2^-24 * sum|q_i k_i| / sqrt(D) (about 1.6e-5 for N(0, 1) rows at D = 256),
and an output moves by at most twice that times the largest |value| (about 5)
in the worst case.  Merging pieces adds one exponential and one product per
piece, the same as merging waves.
"""
import threading
import time

import numpy as np
import pytest

import _oracle as orc

pytestmark = pytest.mark.gpu


def make_pool(gpu, H, D, ps, lengths, seed):
    batch = gpu.SyntheticBatch(H, D, ps, lengths, seed=seed)
    pool = gpu.DevicePagePool(H, D, ps, batch.capacity)
    batch.upload(pool)
    return batch, pool


@pytest.mark.parametrize("H,D,ps,lengths", [
    (2, 128, 16, [1, 0, 127, 128, 129, 384, 385, 3000]),  # steps of 128 slots, 3 and 4 of them
    (2, 128, 1, [700, 256, 257]),       # one token per page: several tiles of 256 entries
    (4, 128, 48, [5000, 49]),           # pieces that start inside a page
    (1, 64, 16, [767, 768, 769, 9000]),
    (3, 80, 16, [1300, 1]),             # 128-slot steps, 6 merge groups
    (3, 96, 16, [2000, 17]),
    (2, 256, 16, [600, 1025]),          # two merge groups
    (2, 32, 16, [900]),                 # no float4 lane split: one workgroup per head
])
def test_dense_pieces_match_oracle(gpu, H, D, ps, lengths):
    import torch
    batch, pool = make_pool(gpu, H, D, ps, lengths, seed=sum(lengths) + D)
    want = orc.dense_batch(batch.queries, batch.key_pool, batch.value_pool, batch.token_counts,
                           batch.cand_offsets, batch.cand_ids, H, D, ps)
    dev = [torch.from_numpy(a).cuda() for a in (batch.queries, batch.cand_offsets,
                                                batch.cand_ids)]
    outs = [torch.full((len(lengths), H * D), 7.0, device="cuda") for _ in range(6)]
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    torch.cuda.synchronize()
    # back to back, the streams in turn: one scratch, launches in order
    for i, out in enumerate(outs):
        gpu.dense_run_batch_device(pool, len(lengths), *[t.data_ptr() for t in dev],
                                   out.data_ptr(), streams[i % 2].cuda_stream)
    torch.cuda.synchronize()
    host, _ = gpu.dense_run_batch(pool, batch.queries, batch.cand_offsets, batch.cand_ids)
    assert orc.max_abs_diff(host, np.asarray(want).reshape(host.shape)) <= 1e-4
    for out in outs:
        assert np.array_equal(out.cpu().numpy().view(np.uint32), host.view(np.uint32))
    pool.close()


def dense_inputs(H, D, ps, lengths, seed):
    """One pool's list of device batches: its requests with other queries."""
    import torch
    rng = np.random.default_rng(seed)
    return [torch.from_numpy(rng.standard_normal((len(lengths), H * D)).astype(np.float32)).cuda()
            for _ in range(6)]


def test_steps_on_many_streams_and_threads(gpu):
    """Six host threads, each with a stream of its own (more than there are
    scratches of streams), enqueue split steps on one pool at once: the bits of
    the steps one after the other."""
    import torch
    H, D, ps, lengths = 4, 128, 16, [6000, 1700]
    batch, pool = make_pool(gpu, H, D, ps, lengths, seed=31)
    queries = dense_inputs(H, D, ps, lengths, 32)
    offs, ids = (torch.from_numpy(a).cuda() for a in (batch.cand_offsets, batch.cand_ids))
    streams = [torch.cuda.Stream() for _ in queries]
    outs = [[torch.zeros(2, H * D, device="cuda") for _ in range(25)] for _ in queries]
    torch.cuda.synchronize()

    def step(i, out):
        gpu.dense_run_batch_device(pool, 2, queries[i].data_ptr(), offs.data_ptr(),
                                   ids.data_ptr(), out.data_ptr(), streams[i].cuda_stream)

    want = []
    for i in range(len(queries)):
        out = torch.zeros(2, H * D, device="cuda")
        torch.cuda.synchronize()
        step(i, out)
        torch.cuda.synchronize()
        want.append(out.cpu().numpy().view(np.uint32))
    start = threading.Barrier(len(queries))

    def run(i):
        start.wait()
        for out in outs[i]:
            step(i, out)

    threads = [threading.Thread(target=run, args=(i,)) for i in range(len(queries))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    for i, mine in enumerate(outs):
        for out in mine:
            assert np.array_equal(out.cpu().numpy().view(np.uint32), want[i]), i
    pool.close()


def test_a_stream_does_not_wait_for_another_streams_step(gpu):
    import torch
    H, D, ps, lengths = 4, 128, 16, [6000]
    batch, pool = make_pool(gpu, H, D, ps, lengths, seed=33)
    query = dense_inputs(H, D, ps, lengths, 34)[0]
    offs, ids = (torch.from_numpy(a).cuda() for a in (batch.cand_offsets, batch.cand_ids))
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    out = {s: torch.zeros(1, H * D, device="cuda") for s in (a, b)}
    scratch = torch.zeros(64, device="cuda")
    torch.cuda.synchronize()

    def step(s):
        gpu.dense_run_batch_device(pool, 1, query.data_ptr(), offs.data_ptr(), ids.data_ptr(),
                                   out[s].data_ptr(), s.cuda_stream)

    def b_ends_first(work):
        begin = time.perf_counter()
        with torch.cuda.stream(a):
            torch.cuda._sleep(200_000_000)
        step(a)
        work()
        b.synchronize()
        b_took = time.perf_counter() - begin
        a.synchronize()
        a_took = time.perf_counter() - begin
        print(f"[streams] a {a_took * 1e3:.2f} ms, b {b_took * 1e3:.2f} ms", flush=True)
        return b_took < a_took / 2

    def plain():
        with torch.cuda.stream(b):
            scratch.add_(1.0)

    step(a)
    step(b)
    plain()
    torch.cuda.synchronize()
    if not b_ends_first(plain):
        pytest.skip("the two streams share a hardware queue")
    assert b_ends_first(lambda: step(b))
    assert torch.equal(out[a], out[b])
    pool.close()


@pytest.mark.parametrize("H,D,lengths,whole", [
    (8, 128, [700] * 30, True),              # 240 even heads load the chip
    (8, 128, [1100] * 35, False),            # 280: a few CUs would run two
    (2, 128, [300] * 70, True),              # more requests than lanes, short lists
    (2, 64, [769] + [5] * 6, False),         # one request past three steps
    (4, 64, [900] * 32, True),
    (2, 128, [100] * 69 + [3000], False),    # the tail, in the second 64 requests
])
def test_where_heads_are_split(gpu, H, D, lengths, whole):
    """Even batches stay unsplit (the captured step's bits); a long tail is
    split, and either way the outputs are the oracle's."""
    import torch
    ps, B = 16, len(lengths)
    batch, pool = make_pool(gpu, H, D, ps, lengths, seed=B + H)
    want = orc.dense_batch(batch.queries, batch.key_pool, batch.value_pool, batch.token_counts,
                           batch.cand_offsets, batch.cand_ids, H, D, ps)
    dev = [torch.from_numpy(a).cuda() for a in (batch.queries, batch.cand_offsets,
                                                batch.cand_ids)]
    eager, captured = (torch.full((B, H * D), 7.0, device="cuda") for _ in range(2))
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    gpu.dense_run_batch_device(pool, B, *[t.data_ptr() for t in dev], eager.data_ptr(),
                               side.cuda_stream)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        gpu.dense_run_batch_device(pool, B, *[t.data_ptr() for t in dev], captured.data_ptr(),
                                   side.cuda_stream)
    graph.replay()
    torch.cuda.synchronize()
    host, _ = gpu.dense_run_batch(pool, batch.queries, batch.cand_offsets, batch.cand_ids)
    eager = eager.cpu().numpy()
    assert orc.max_abs_diff(eager, np.asarray(want).reshape(eager.shape)) <= 1e-4
    assert np.array_equal(host.view(np.uint32), eager.view(np.uint32))
    same = np.array_equal(eager.view(np.uint32), captured.cpu().numpy().view(np.uint32))
    assert same == whole
    pool.close()


@pytest.mark.parametrize("bad", [np.nan, -np.inf])
def test_nonfinite_keys_of_whole_pieces(gpu, bad):
    """Pieces (of 128 slots here) whose logits are all NaN or -inf: the output
    is NaN, or what the other tokens give, as of an unsplit head (the captured
    step)."""
    import torch
    H, D, ps, lengths = 2, 128, 16, [3000, 3000, 500]
    batch = gpu.SyntheticBatch(H, D, ps, lengths, seed=21)
    keys = batch.key_pool.reshape(batch.capacity, ps, H, D)
    queries = np.abs(batch.queries) + np.float32(0.1)  # (with -inf keys: logits of -inf)
    offs, ids = batch.cand_offsets, batch.cand_ids
    keys[ids[offs[0] + 64:offs[0] + 80], :, 0] = bad   # request 0, head 0: slots 1024-1279
    keys[ids[offs[0] + 80], :8, 1] = -np.inf           # head 1: a piece's first eight
    keys[ids[offs[1]:offs[2]], :, 1] = bad             # request 1, head 1: every slot
    pool = gpu.DevicePagePool(H, D, ps, batch.capacity)
    batch.upload(pool)
    dev = [torch.from_numpy(np.ascontiguousarray(a)).cuda() for a in (queries, offs, ids)]
    split, whole = (torch.full((3, H * D), 7.0, device="cuda") for _ in range(2))
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    gpu.dense_run_batch_device(pool, 3, *[t.data_ptr() for t in dev], split.data_ptr(),
                               side.cuda_stream)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        gpu.dense_run_batch_device(pool, 3, *[t.data_ptr() for t in dev], whole.data_ptr(),
                                   side.cuda_stream)
    graph.replay()
    torch.cuda.synchronize()
    split, whole = (t.cpu().numpy().reshape(3, H, D) for t in (split, whole))
    assert np.isnan(whole[0, 0]).all() == np.isnan(bad) and not whole[1, 1].any()
    assert np.array_equal(np.isnan(split), np.isnan(whole))
    ok = ~np.isnan(whole)
    assert np.abs(split[ok] - whole[ok]).max() <= 1e-4
    pool.close()


def test_captured_dense_step(gpu):
    import torch
    H, D, ps = 2, 128, 16
    batch, pool = make_pool(gpu, H, D, ps, [1500, 40], seed=3)
    want = orc.dense_batch(batch.queries, batch.key_pool, batch.value_pool, batch.token_counts,
                           batch.cand_offsets, batch.cand_ids, H, D, ps)
    dev = [torch.from_numpy(a).cuda() for a in (batch.queries, batch.cand_offsets,
                                                batch.cand_ids)]
    out = torch.zeros(2, H * D, device="cuda")
    side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=side):
        gpu.dense_run_batch_device(pool, 2, *[t.data_ptr() for t in dev], out.data_ptr(),
                                   side.cuda_stream)
    for _ in range(3):
        out.fill_(7.0)
        graph.replay()
        torch.cuda.synchronize()
        assert orc.max_abs_diff(out.cpu().numpy(),
                                np.asarray(want).reshape(2, H * D)) <= 1e-4
    pool.close()


def test_sparse_step_with_pieces_eager_and_captured(gpu):
    """Lists of up to 40 x 16 slots (five steps) of a few heads: the sparse
    step's attention in pieces, the same bits from a graph's replays."""
    import torch
    H, D, ps, k = 8, 128, 16, 40
    lengths = [2100, 90, 700]
    batch, pool = make_pool(gpu, H, D, ps, lengths, seed=11)
    summ = orc.pool_summaries(batch.key_pool, batch.token_counts, H * D)
    rng = np.random.default_rng(12)
    sets = [batch.queries, rng.standard_normal(batch.queries.shape).astype(np.float32)]
    offs, ids = (torch.from_numpy(a).cuda() for a in (batch.cand_offsets, batch.cand_ids))
    q = torch.zeros(3, H * D, device="cuda")
    out = torch.zeros(3, H * D, device="cuda")
    total, most = batch.total_candidates, batch.max_candidates
    with gpu.SparseContext(pool, k, 3, total, 3 * k) as ctx:
        def step(stream):
            ctx.run_batch_device(3, total, most, q.data_ptr(), offs.data_ptr(), ids.data_ptr(),
                                 out.data_ptr(), stream=stream)

        main = torch.cuda.Stream()
        eager = []
        for qs in sets:
            q.copy_(torch.from_numpy(qs))
            torch.cuda.synchronize()
            step(main.cuda_stream)
            torch.cuda.synchronize()
            eager.append(out.cpu().numpy().copy())
            _, _, want = orc.sparse_batch(qs, batch.key_pool, batch.value_pool, summ,
                                          batch.token_counts, batch.cand_offsets,
                                          batch.cand_ids, H, D, ps, k)
            assert orc.max_abs_diff(eager[-1], want) <= 1e-4
        side, graph = torch.cuda.Stream(), torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=side):
            step(side.cuda_stream)
        for i in (1, 0, 1):
            q.copy_(torch.from_numpy(sets[i]))
            out.fill_(7.0)
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert np.array_equal(out.cpu().numpy().view(np.uint32), eager[i].view(np.uint32))
        ctx.device_status()
    pool.close()


def test_a_merge_that_gives_up_is_reported_and_recovers(gpu):
    """Every wait of the merge gives up (it polls for a tag nobody writes): the
    split requests' outputs are zeros and the step reports it; what it left in
    the scratch is not taken for the next step's."""
    import torch
    H, D, ps, k = 8, 128, 16, 40
    batch, pool = make_pool(gpu, H, D, ps, [2100, 90, 700], seed=13)
    dev = [torch.from_numpy(a).cuda() for a in (batch.queries, batch.cand_offsets,
                                                batch.cand_ids)]
    other = torch.from_numpy(np.ascontiguousarray(batch.queries[::-1])).cuda()
    total, most = batch.total_candidates, batch.max_candidates
    with gpu.SparseContext(pool, k, 3, total, 3 * k) as ctx:
        def step(queries):
            out = torch.full((3, H * D), 7.0, device="cuda")
            torch.cuda.synchronize()
            ctx.run_batch_device(3, total, most, queries.data_ptr(), dev[1].data_ptr(),
                                 dev[2].data_ptr(), out.data_ptr())
            torch.cuda.synchronize()
            return out.cpu().numpy()

        good, turned = step(dev[0]), step(other)
        ctx.device_status()
        ctx.set_wait_limit(4, True)
        late = step(other)
        with pytest.raises(gpu.DsdError, match="timed out"):
            ctx.device_status()
        assert not late[0].any() and not late[2].any()  # 640 slots each
        assert np.array_equal(late[1].view(np.uint32), turned[1].view(np.uint32))  # one piece
        ctx.set_wait_limit(1 << 17, False)
        for queries, want in ((dev[0], good), (other, turned)):
            assert np.array_equal(step(queries).view(np.uint32), want.view(np.uint32))
        ctx.device_status()
    pool.close()


@pytest.mark.parametrize("H,D,batch,k", [
    (2, 64, 2, 8), (2, 64, 2, 9),         # 128 and 144 slots: one chunk in flight, four
    (8, 64, 64, 16), (8, 64, 64, 65),     # 512 heads: 256 and 1040 slots
    (2, 80, 2, 8), (2, 80, 2, 9),         # four waves, eight
])
def test_sparse_lists_by_length(gpu, H, D, batch, k):
    """Either side of the list lengths that choose the kernel's form."""
    ps = 16
    lengths = [k * ps + 37] + [ps * (k // 2) + r for r in range(batch - 1)]
    batch_, pool = make_pool(gpu, H, D, ps, lengths, seed=D + k)
    summ = orc.pool_summaries(batch_.key_pool, batch_.token_counts, H * D)
    with gpu.SparseContext(pool, k, batch, batch_.total_candidates, batch * k) as ctx:
        got = ctx.run_batch(batch_.queries, batch_.cand_offsets, batch_.cand_ids,
                            output_mode=gpu.OUTPUT_OUTPUTS, want_ids=True)
    _, selected, outs = orc.sparse_batch(batch_.queries, batch_.key_pool, batch_.value_pool, summ,
                                         batch_.token_counts, batch_.cand_offsets,
                                         batch_.cand_ids, H, D, ps, k)
    for r in range(batch):
        assert got["selected"][r].tolist() == selected[r].tolist(), r
    assert orc.max_abs_diff(got["outputs"], outs) <= 1e-4
    pool.close()
