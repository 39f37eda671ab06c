"""The torch-facing operators of infinicore_amd.ops (argument order of the reference's Python ops)."""
import pytest
import torch

from infinicore_amd import workloads

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_paged_attention_and_caching_through_the_python_operators(oracle):
    from infinicore_amd import ops

    cfg = workloads.DecodeConfig("ops", torch.bfloat16, 4, 32, 8, 128, 16, 10, 1500, seed=77)
    inp = workloads.make_decode_inputs(cfg)
    q, k, v, bt, sl = [t.to(DEV) for t in (inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens)]
    want = oracle.paged_attention(inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens, inp.scale).float()
    for _ in range(2):  # second call hits the plan cache
        got = ops.paged_attention(q, k, v, bt, sl, None, inp.scale)
        torch.cuda.synchronize()
        assert torch.all((got.float().cpu() - want).abs() <= 1e-2 + 2e-3 * want.abs())
    out = torch.empty_like(q)
    assert ops.paged_attention(q, k, v, bt, sl, scale=inp.scale, out=out) is out

    # one decode step: append one token per sequence with paged_caching, lengths grow by one
    new_k = torch.randn(4, 8, 128, device=DEV).to(torch.bfloat16)
    new_v = torch.randn(4, 8, 128, device=DEV).to(torch.bfloat16)
    slots = torch.stack([bt[s, int(sl[s]) // 16] * 16 + int(sl[s]) % 16 for s in range(4)])
    room = torch.tensor([int(sl[s]) // 16 < ((int(sl[s]) + 15) // 16) for s in range(4)])
    slots = torch.where(room.to(DEV), slots, torch.full_like(slots, -1))  # no free row in the last page: skip
    k_ret, v_ret = ops.paged_caching(k, v, new_k, new_v, slots)
    assert k_ret is k and v_ret is v
    k_want, v_want = oracle.paged_caching(inp.k_cache.clone(), inp.v_cache.clone(), new_k.cpu(), new_v.cpu(), slots.cpu())
    torch.cuda.synchronize()
    assert torch.equal(k.cpu().view(torch.int16), k_want.view(torch.int16))
    assert torch.equal(v.cpu().view(torch.int16), v_want.view(torch.int16))
    ops.clear_plan_cache()


def test_operators_refuse_host_tensors():
    from infinicore_amd import ops

    t = torch.zeros(1, 1, 128, dtype=torch.float16)
    with pytest.raises(ValueError):
        ops.paged_attention(t, t, t, t, t)


def test_a_query_without_dimensions_is_refused_by_the_operator():
    from infinicore_amd import ops

    kc = torch.zeros(4, 2, 16, 64, dtype=torch.float16, device=DEV)
    bt, sl = torch.zeros(1, 2, dtype=torch.int64, device=DEV), torch.ones(1, dtype=torch.int64, device=DEV)
    with pytest.raises(RuntimeError) as refused:
        ops.paged_attention(torch.zeros((), dtype=torch.float16, device=DEV), kc, kc, bt, sl)
    assert hasattr(refused.value, "status")


def test_plans_by_metadata_stream_and_thread(oracle):
    """More shapes than the cache keeps, called again after their plans went; strided queries of one shape; several
    threads on streams of their own at once."""
    import threading

    from infinicore_amd import ops

    cfg = workloads.DecodeConfig("plans", torch.float16, 3, 8, 2, 64, 16, 200, 700, seed=5)
    inp = workloads.make_decode_inputs(cfg)
    q, k, v, bt, sl = [t.to(DEV) for t in (inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens)]
    want = oracle.paged_attention(inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens, inp.scale).float()

    def check(got):
        assert torch.all((got.float().cpu() - want).abs() <= 1e-2 + 2e-3 * want.abs())

    ops.clear_plan_cache()
    for width in [*range(bt.shape[1], bt.shape[1] + 120), bt.shape[1]]:
        table = torch.zeros(3, width, dtype=bt.dtype, device=DEV)
        table[:, :bt.shape[1]] = bt
        check(ops.paged_attention(q, k, v, table, sl, None, inp.scale))
    assert ops._native.size() == 100
    wide = torch.zeros(3, 8, 128, dtype=q.dtype, device=DEV)
    wide[..., :64] = q
    check(ops.paged_attention(wide[..., :64], k, v, bt, sl, None, inp.scale))

    failures = []
    torch.cuda.synchronize()

    def work():
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for _ in range(20):
                    check(ops.paged_attention(q, k, v, bt, sl, None, inp.scale))
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    threads = [threading.Thread(target=work) for _ in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures
    with pytest.raises(RuntimeError) as refused:
        ops.paged_attention(q, k, v, bt, sl.to(torch.float32), None, inp.scale)
    assert hasattr(refused.value, "status")
    ops.clear_plan_cache()
    assert ops._native.size() == 0


# ---- scratch: a call's own ---------------------------------------------------------------------------------------

def split_prefill(seed, new=5, total=3000, width=None):
    """A prefill whose row blocks are split, so that it needs scratch: two sequences of a few tokens over a long history."""
    cfg = workloads.PrefillConfig("scratch", torch.bfloat16, 2, 32, 8, 128, 16, new, new, total - new, total - new, seed=seed)
    inp = workloads.make_prefill_inputs(cfg)
    if width is not None:
        inp.block_tables = torch.nn.functional.pad(inp.block_tables, (0, width - inp.block_tables.shape[1]))
    return inp, [t.to(DEV) for t in (inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens, inp.cum_seq_lens_q)]


def test_calls_of_one_plan_at_once_do_not_share_scratch():
    """Two threads in the same call on one stream. Stand-ins for the library's entry points (no kernel runs) hold both
    threads inside a prefill and note the scratch each was given; of two decode calls only one may be inside at a time."""
    import ctypes
    import threading
    import time

    from infinicore_amd import libinfiniop as lib
    from infinicore_amd import ops

    inp, dev = split_prefill(1)
    q = dev[0][:2].contiguous()
    meet, seen = threading.Barrier(2, timeout=30), []
    inside, most = [], []
    void = ctypes.c_void_p

    @ctypes.CFUNCTYPE(ctypes.c_int, void, void, ctypes.c_size_t, *([void] * 9))
    def prefill(descriptor, workspace, size, *rest):
        seen.append((workspace, size))
        meet.wait()
        return 0

    @ctypes.CFUNCTYPE(ctypes.c_int, void, void, ctypes.c_size_t, *([void] * 8))
    def decode(descriptor, workspace, size, *rest):
        assert workspace and size
        inside.append(0)
        time.sleep(0.05)
        most.append(len(inside))
        inside.pop()
        return 0

    def setup(functions):
        ops._native.setup(tuple(ctypes.cast(f, void).value for f in functions),
                          ctypes.cast(lib.LIBINFINIRT.infinirtSetDevice, void).value, int(lib.InfiniDevice.AMD),
                          ops._PLAN_CACHE_CAPACITY)

    def twice(call):
        threads = [threading.Thread(target=call) for _ in range(2)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()

    real = {name: getattr(lib.LIBINFINIOP, name) for name in ops._RUN}
    ops.clear_plan_cache()
    try:
        setup({**real, "infiniopPagedAttention": decode, "infiniopPagedAttentionPrefill": prefill}.values())
        twice(lambda: ops.paged_attention_prefill(*dev, None, inp.scale))
        twice(lambda: ops.paged_attention(q, *dev[1:5], None, inp.scale))
    finally:
        setup(real.values())
        ops.clear_plan_cache()
    (a, size), (b, _) = seen
    assert size > 0 and a and b and (a + size <= b or b + size <= a)
    assert most == [1, 1]


def test_threads_on_one_stream(oracle):
    """Different inputs of one shape, each thread's results its own: split prefill and decode merged by a second kernel."""
    import threading

    from infinicore_amd import ops

    jobs = []
    for seed in range(4):
        inp, dev = split_prefill(20 + seed)
        want = oracle.paged_attention_prefill(inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens,
                                              inp.cum_seq_lens_q, inp.scale).float()
        last = inp.cum_seq_lens_q[1:] - 1  # the sequences' last tokens as a decode
        jobs.append((inp, dev, want, dev[0][last.to(DEV)].contiguous(), want[last]))
    failures = []

    def work(inp, dev, want, q, want_decode):
        try:
            for _ in range(40):
                got = ops.paged_attention_prefill(*dev, None, inp.scale)
                one = ops.paged_attention(q, *dev[1:5], None, inp.scale)
                for x, y in ((got, want), (one, want_decode)):
                    assert torch.all((x.float().cpu() - y).abs() <= 1e-2 + 8e-3 * y.abs())
        except BaseException as e:  # noqa: BLE001
            failures.append(e)

    torch.cuda.synchronize()
    threads = [threading.Thread(target=work, args=job) for job in jobs]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not failures, failures


def test_prefill_plans_hold_no_device_memory():
    from infinicore_amd import ops

    ops.clear_plan_cache()
    inp, dev = split_prefill(3)
    tables = [torch.nn.functional.pad(dev[3], (0, extra)) for extra in range(40)]
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    for table in tables:
        ops.paged_attention_prefill(*dev[:3], table, *dev[4:], None, inp.scale)
    torch.cuda.synchronize()
    assert ops._native.size() == 40
    assert torch.cuda.memory_allocated() == before
    ops.clear_plan_cache()


def test_captured_call_outlives_its_plan(oracle):
    """A graph over a split prefill and a cut decode, replayed after their plans went and their memory would be in use
    again: the same results, and nothing else written."""
    from infinicore_amd import ops

    inp, dev = split_prefill(4)
    want = oracle.paged_attention_prefill(inp.q, inp.k_cache, inp.v_cache, inp.block_tables, inp.seq_lens, inp.cum_seq_lens_q,
                                          inp.scale).float()
    last = inp.cum_seq_lens_q[1:] - 1
    q = dev[0][last.to(DEV)].contiguous()
    out, one = torch.empty_like(dev[0]), torch.empty_like(q)
    stream = torch.cuda.Stream()
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        ops.paged_attention_prefill(*dev, None, inp.scale, out=out)
        ops.paged_attention(q, *dev[1:5], None, inp.scale, out=one)
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            ops.paged_attention_prefill(*dev, None, inp.scale, out=out)
            ops.paged_attention(q, *dev[1:5], None, inp.scale, out=one)
    with torch.cuda.stream(stream):
        for width in range(dev[3].shape[1] + 1, dev[3].shape[1] + 1 + ops._PLAN_CACHE_CAPACITY + 5):
            ops.paged_attention_prefill(*dev[:3], torch.nn.functional.pad(dev[3], (0, width - dev[3].shape[1])), *dev[4:], None,
                                        inp.scale)
    ops.clear_plan_cache()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):  # memory of all sizes of that stream, as later tensors of a program would take it
        others = [torch.full((n,), 0x55, dtype=torch.uint8, device=DEV) for n in [1 << 20] * 64 + [8 << 20] * 16 + [40 << 20] * 4]
    torch.cuda.synchronize()
    for _ in range(3):
        out.zero_(), one.zero_()
        torch.cuda.synchronize()
        graph.replay()
        ops.paged_attention_prefill(*dev, None, inp.scale)  # the same shape on another stream beside the replay
        torch.cuda.synchronize()
        for x, y in ((out, want), (one, want[last])):
            assert torch.all((x.float().cpu() - y).abs() <= 1e-2 + 8e-3 * y.abs())
        assert all(bool((t == 0x55).all()) for t in others)
