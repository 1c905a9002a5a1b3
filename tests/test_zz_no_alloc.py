"""The decode entry point that allocates nothing (weed_hip_kv_decode_attn_noalloc) against weed_hip_kv_decode_attn.

Both run the same kernels with the same work partition, so their outputs must be identical bit for bit; the first is
also held to the attention tolerance against the CPU checker.  Two calls in a row share the library's static workspace,
the second with a smaller input, so stale contents of the first would show.
"""
import numpy as np
import pytest

from gpu_helpers import assert_attn_close, coder_specs, dev, export
from weed_amd import workloads

pytestmark = pytest.mark.gpu


def _cache(gpu, oracle, wl, seed):
    K, V, q = wl.tensors()
    rng = np.random.default_rng(seed)
    d = wl.head_dim
    Rk = oracle.orthonormalize_columns(rng.normal(size=d * d).astype(np.float32))
    Rv = oracle.orthonormalize_columns(rng.normal(size=d * d).astype(np.float32))
    cache = gpu.KVCache(gpu.KV_LLOYDMAX, wl.n_seq, wl.n_kv_heads, d, wl.max_len, wl.k_bits, wl.v_bits, wl.k_sign,
                        wl.v_sign)
    cache.set_rotations(dev(Rk), dev(Rv))
    Kd, Vd = dev(K), dev(V)
    for s, L in enumerate(wl.lens):
        cache.encode_append(Kd[s:s + 1, :, :L], Vd[s:s + 1, :, :L], seq_begin=s, rotate=1)
    return cache, q, Rk, Rv


def _both(gpu, cache, q, flags):
    import torch
    qd = dev(q)
    ref = torch.zeros_like(qd)
    out = torch.full_like(qd, float("nan"))
    cache.decode_attn(qd, ref, gqa_mapping=gpu.GQA_BLOCKED, flags=flags)
    cache.decode_attn_noalloc(qd, out, gqa_mapping=gpu.GQA_BLOCKED, flags=flags)
    gpu.sync()
    return ref.cpu().numpy(), out.cpu().numpy()


def test_noalloc_matches_decode_attn_on_two_calls_in_a_row(gpu, oracle):
    flags = gpu.ATTN_ROTATE_Q | gpu.ATTN_UNROTATE_OUT
    # first call: 6 ragged sequences, long enough for several context splits per region
    big = workloads.Workload("noalloc_a", 6, 16, 4, 128, [1500, 700, 2048, 64, 1, 999], 3, 4, 0, 0, 21)
    cache_a, q_a, Rk, Rv = _cache(gpu, oracle, big, 5)
    ref_a, out_a = _both(gpu, cache_a, q_a, flags)
    assert np.array_equal(ref_a, out_a), "first call differs from weed_hip_kv_decode_attn"
    kspec, vspec = coder_specs(oracle, cache_a)
    kf, ka = export(cache_a, 0, big.max_len)
    vf, va = export(cache_a, 1, big.max_len)
    want = oracle.decode_attn(kspec, vspec, kf, ka, vf, va, q_a, big.lens, gqa_weed=False, Rk=Rk, Rv=Rv)
    assert_attn_close(out_a, want, "noalloc first call vs checker")
    # second call, smaller in every dimension: it reuses the workspace the first one left behind
    small = workloads.Workload("noalloc_b", 2, 4, 2, 64, [130, 37], 2, 3, 1, 0, 22)
    cache_b, q_b, Rk2, Rv2 = _cache(gpu, oracle, small, 6)
    ref_b, out_b = _both(gpu, cache_b, q_b, flags)
    assert np.array_equal(ref_b, out_b), "second (smaller) call differs from weed_hip_kv_decode_attn"
    kspec, vspec = coder_specs(oracle, cache_b)
    kf, ka = export(cache_b, 0, small.max_len)
    vf, va = export(cache_b, 1, small.max_len)
    want = oracle.decode_attn(kspec, vspec, kf, ka, vf, va, q_b, small.lens, gqa_weed=False, Rk=Rk2, Rv=Rv2)
    assert_attn_close(out_b, want, "noalloc second call vs checker")
    # and the first shape again after the small one
    ref_c, out_c = _both(gpu, cache_a, q_a, flags)
    assert np.array_equal(ref_c, out_c) and np.array_equal(out_c, out_a)
    cache_a.close()
    cache_b.close()


def test_noalloc_head_dim_256_whole_regions_per_workgroup(gpu, oracle):
    """A batch of equal sequences at head_dim 256, which is one kernel (the workgroups rotate their queries and merge
    their partials themselves): the same bits from both entry points, and the checker's values."""
    flags = gpu.ATTN_ROTATE_Q | gpu.ATTN_UNROTATE_OUT
    wl = workloads.Workload("noalloc_256", 4, 8, 2, 256, [1024] * 4, 3, 4, 0, 0, 23)
    cache, q, Rk, Rv = _cache(gpu, oracle, wl, 7)
    try:
        gpu.decode_tuning(32)
        ref, out = _both(gpu, cache, q, flags)
    finally:
        gpu.decode_tuning()
    assert np.array_equal(ref, out)
    kspec, vspec = coder_specs(oracle, cache)
    kf, ka = export(cache, 0, wl.max_len)
    vf, va = export(cache, 1, wl.max_len)
    want = oracle.decode_attn(kspec, vspec, kf, ka, vf, va, q, wl.lens, gqa_weed=False, Rk=Rk, Rv=Rv)
    assert_attn_close(out, want, "noalloc at head_dim 256 vs checker")
    cache.close()


def test_noalloc_refuses_shapes_beyond_its_workspace(gpu):
    import torch
    # 1024 sequences x 64 heads x 128: the rotated queries alone are 32 MiB, the size of the static workspace
    cache = gpu.KVCache(gpu.KV_LLOYDMAX, 1024, 4, 128, 64, 3, 4)
    K = torch.randn((1024, 4, 64, 128), device="cuda")
    cache.encode_append(K, K)
    q = torch.randn((1024, 64, 128), device="cuda")
    out = torch.zeros_like(q)
    with pytest.raises(gpu.WeedHipError) as err:
        cache.decode_attn_noalloc(q, out, gqa_mapping=gpu.GQA_BLOCKED, flags=0)
    assert err.value.code == gpu.EINVAL and "static scratch" in str(err.value)
    cache.decode_attn(q, out, gqa_mapping=gpu.GQA_BLOCKED, flags=0)  # the allocating entry point takes it
    gpu.sync()
    assert bool(torch.isfinite(out).all())
    cache.close()


def _long_cache(gpu, S, Hkv, tokens, room):
    """A cache of S sequences with room for `room` tokens, and what appends `tokens` normal ones to each."""
    import torch
    cache = gpu.KVCache(gpu.KV_LLOYDMAX, S, Hkv, 128, room, 3, 4)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(S + tokens)

    def append(n):
        k, v = (torch.randn((S, Hkv, n, 128), generator=gen, device="cuda") for _ in range(2))
        torch.cuda.synchronize()
        cache.encode_append(k, v, rotate=0)
        gpu.sync()

    append(tokens)
    return cache, append


def test_noalloc_takes_what_the_passes_leave_room_for(gpu):
    """256 heads on one KV head over blocks enough to share their unpacking, which needs a workspace of 40 MB where the passes
    take 28: within the static workspace, so both entry points take the call, with the same bits."""
    import torch
    cache, _ = _long_cache(gpu, 16, 1, 22100, 22100)
    q = torch.randn((16, 256, 128), device="cuda")
    ref, out = torch.zeros_like(q), torch.full_like(q, float("nan"))
    torch.cuda.synchronize()
    cache.decode_attn(q, ref, gqa_mapping=gpu.GQA_BLOCKED, flags=0)
    cache.decode_attn_noalloc(q, out, gqa_mapping=gpu.GQA_BLOCKED, flags=0)
    gpu.sync()
    assert bool(torch.isfinite(ref).all()) and torch.equal(ref, out)
    cache.close()


def test_a_captured_chunk_keeps_to_the_workspace_it_finds(gpu):
    """A chunk whose cache has grown, since its workspace was allocated, past where chunks share the unpacking, which takes more
    of it: captured and replayed in what is there; eager calls afterwards let it grow, and agree."""
    import torch
    S, Hkv, T, Hq = 2, 8, 64, 32
    cache, append = _long_cache(gpu, S, Hkv, 21000, 22100)
    q = torch.randn((S, T, Hq, 128), device="cuda")
    warm, out, eager = torch.zeros_like(q), torch.full_like(q, float("nan")), torch.zeros_like(q)
    torch.cuda.synchronize()
    cache.decode_attn_chunk(q, warm, gqa_mapping=gpu.GQA_BLOCKED, flags=0)
    append(1100)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
        cache.decode_attn_chunk(q, out, gqa_mapping=gpu.GQA_BLOCKED, flags=0)
    first = None
    for _ in range(3):
        out.fill_(float("nan"))
        graph.replay()
        gpu.sync()
        first = out.clone() if first is None else first
        assert torch.equal(out, first)
    del graph
    cache.decode_attn_chunk(q, eager, gqa_mapping=gpu.GQA_BLOCKED, flags=0)
    gpu.sync()
    # (8e-6: the bound of test_chunks_that_share_the_unpacking)
    assert float((first - eager).double().norm() / eager.double().norm()) <= 8e-6
    cache.close()


@pytest.mark.parametrize("n_seq,ctx", [(1, 2048), (8, 1024), (3, 1000)])
def test_noalloc_call_replayed_from_a_graph(gpu, oracle, n_seq, ctx):
    """The allocation-free entry point under graph capture: the captured call is one kernel whose workgroups count
    their arrivals per region and leave the counters at zero, so every replay must give the bits of the eager call,
    also with eager calls of another shape in between."""
    import torch
    flags = gpu.ATTN_ROTATE_Q | gpu.ATTN_UNROTATE_OUT
    wl = workloads.Workload("graph", n_seq, 8, 2, 128, [ctx] * n_seq, 3, 4, 0, 0, 31)
    cache, q, _, _ = _cache(gpu, oracle, wl, 9)
    other = workloads.Workload("graph_b", 2, 4, 2, 64, [130, 37], 2, 3, 1, 0, 32)
    cache_b, q_b, _, _ = _cache(gpu, oracle, other, 10)
    qd, qb = dev(q), dev(q_b)
    eager = torch.zeros_like(qd)
    cache.decode_attn_noalloc(qd, eager, gqa_mapping=gpu.GQA_BLOCKED, flags=flags)
    gpu.sync()
    out = torch.full_like(qd, float("nan"))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
        cache.decode_attn_noalloc(qd, out, gqa_mapping=gpu.GQA_BLOCKED, flags=flags)
    for _ in range(4):
        out.fill_(float("nan"))
        graph.replay()
        gpu.sync()
        assert np.array_equal(out.cpu().numpy(), eager.cpu().numpy())
        ob = torch.zeros_like(qb)
        cache_b.decode_attn_noalloc(qb, ob, gqa_mapping=gpu.GQA_BLOCKED, flags=flags)
        gpu.sync()
    cache.close()
    cache_b.close()


@pytest.mark.parametrize("M,N,K", [(232, 768, 768), (20, 600, 301), (131, 130, 515)])
def test_short_products_in_a_graph_need_no_scratch(gpu, M, N, K):
    """Products of fewer than 1024 k, whose k ranges go through a scratch buffer outside a capture: a captured one must
    not hold that buffer's address, so it stays right after a larger product has replaced it."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(K)
    a = torch.randn((K, M), generator=gen, device="cuda").t()
    b = torch.randn((N, K), generator=gen, device="cuda").t()
    want = a.double() @ b.double()
    bound = 4 * 1.2e-7 * (a.double().abs() @ b.double().abs())  # as the dense products' tests
    out = torch.zeros((N, M), device="cuda").t()
    gpu.matmul(a, b, out)
    gpu.sync()
    assert bool(((out.double() - want).abs() <= bound).all())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
        gpu.matmul(a, b, out)
    big_a = torch.randn((4096, 1024), generator=gen, device="cuda").t()
    big_b, big = torch.randn((1024, big_a.shape[1]), generator=gen, device="cuda").t(), torch.zeros((1024, 1024), device="cuda")
    for _ in range(4):
        gpu.matmul(big_a, big_b, big)
        out.fill_(float("nan"))
        graph.replay()
        gpu.sync()
        assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("warm", [False, True])
def test_products_in_a_graph_outlive_the_scratch_they_were_captured_with(gpu, warm):
    """Captured before the library has any scratch, products run without; captured after the same call has run, they use what
    is there.  Either way the replays stay right after a larger product has taken a larger scratch: 17 to 64 rows on and off
    the 16-byte grid, few whole and ragged tiles, k short and long."""
    import torch
    shapes = [(20, 600, 512), (32, 22001, 1025), (33, 2048, 2050), (64, 1024, 2048), (256, 512, 2048), (203, 301, 1030),
              (40, 300, 4097)]
    gen = torch.Generator(device="cuda")
    gen.manual_seed(77)
    gpu.shutdown()
    gpu.check(gpu.load().weed_hip_init(0))
    gpu.use_torch_stream(torch.cuda.current_stream())
    work = []
    for M, N, K in shapes:
        a = torch.randn((K, M), generator=gen, device="cuda").t()
        b = torch.randn((N, K), generator=gen, device="cuda").t()
        out = torch.zeros((N, M), device="cuda").t()
        bound = 4 * 1.2e-7 * (a.double().abs() @ b.double().abs())  # as the dense products' tests
        work.append((a, b, out, a.double() @ b.double(), bound))
    torch.cuda.synchronize()
    if warm:
        for a, b, out, _, _ in work:
            gpu.matmul(a, b, out)
        gpu.sync()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
        for a, b, out, _, _ in work:
            gpu.matmul(a, b, out)
    for i in range(4):
        # 512 rows in up to 64 k ranges: more scratch than anything before, every pass another number of columns
        N = 512 << i
        big_a, big_b = torch.randn((16384, 512), generator=gen, device="cuda").t(), torch.randn((N, 16384), generator=gen, device="cuda").t()
        big = torch.zeros((N, 512), device="cuda").t()
        gpu.matmul(big_a, big_b, big)
        for _, _, out, _, _ in work:
            out.fill_(float("nan"))
        graph.replay()
        gpu.sync()
        for (M, N, K), (_, _, out, want, bound) in zip(shapes, work):
            assert bool(((out.double() - want).abs() <= bound).all()), (M, N, K, i)


# Captured products of 2^30 multiply-adds and more: k ranges of either tile, on and off the 16-byte grid, strips, and whole tiles of 256,
# with what of the scratch that SCRATCH_BEFORE leaves they find room for (see test_matmul_plan_cpu.py).
LARGE_IN_A_GRAPH = [(512, 4096, 4096), (2708, 920, 1500), (1001, 4096, 4096), (1030, 4096, 4096), (4096, 4096, 544)]
SCRATCH_BEFORE = (640, 1024, 4096)


@pytest.mark.parametrize("scratch", ["none", "some", "all"])
def test_large_products_in_a_graph_keep_to_the_scratch_they_find(gpu, scratch):
    """Captured before the library has any scratch, with less of it than their plans ask for, and with all of it: right on every
    replay, also after eager calls that took a larger one."""
    import torch
    gen = torch.Generator(device="cuda")
    gen.manual_seed(78)
    gpu.shutdown()
    gpu.check(gpu.load().weed_hip_init(0))
    gpu.use_torch_stream(torch.cuda.current_stream())

    def product(M, N, K):
        a = torch.randn((K, M), generator=gen, device="cuda").t()
        b = torch.randn((N, K), generator=gen, device="cuda").t()
        return a, b, torch.zeros((N, M), device="cuda").t()

    work = [product(*shape) for shape in LARGE_IN_A_GRAPH]
    before, beside = product(*SCRATCH_BEFORE), product(1024, 2048, 8192)
    for a, b, out in work if scratch == "all" else [before] if scratch == "some" else []:
        gpu.matmul(a, b, out)
    gpu.sync()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=torch.cuda.current_stream()):
        for a, b, out in work:
            gpu.matmul(a, b, out)
    wants = [(a.double().contiguous() @ b.double().contiguous(), a.double().abs().contiguous() @ b.double().abs().contiguous()) for a, b, _ in work]
    for i in range(4):
        for _, _, out in work:
            out.fill_(float("nan"))
        graph.replay()
        gpu.sync()
        for shape, (_, _, out), (want, scale) in zip(LARGE_IN_A_GRAPH, work, wants):
            assert float(((out.double() - want).abs() / scale).max()) <= 4 * 1.2e-7, (shape, i)  # as the dense products' tests
        gpu.matmul(*beside)
        gpu.sync()
