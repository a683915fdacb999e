"""GPU: the library's launches can be captured into a HIP graph and replayed.

A serving loop captures one decode step and replays it while the device-side lengths, block
table and activations change underneath.  That works only if a call does nothing but launch
kernels once its workspaces have their size: no allocation, no memset node, no host round
trip.  Every replay is checked against the same call made eagerly on copies of the inputs.
"""

import pytest
import torch

from pypto_amd import workloads
from pypto_amd.runtime import decoder_layer_decode, decoder_layer_decode_w16, ffn_block, ffn_swiglu, paged_attention, projection

pytestmark = pytest.mark.gpu


def _cuda(args, keep_host=()):
    return [a.cuda() if isinstance(a, torch.Tensor) and i not in keep_host else a for i, a in enumerate(args)]


def _capture(worker, program, args, stream):
    """Warm-up call (sizes the workspaces), then the same call recorded into a graph."""
    with torch.cuda.stream(stream):
        with worker.register(program) as h:
            h(*args, stream=stream.cuda_stream)
        stream.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            with worker.register(program) as h:
                h(*args, stream=stream.cuda_stream)
    return graph


@pytest.mark.parametrize("batch", [6, 40])
def test_decoder_layer_replays_follow_growing_sequences(worker, batch):
    """Batch 6 takes the skinny projections, batch 40 the tiled GEMMs whose k-split slabs feed the
    RoPE and RMSNorm kernels directly (a scratch area of their own)."""
    if batch == 6:
        ctxs = [100, 1, 250, 33, 60, 129]  # four more tokens stay inside each last block
    else:
        g0 = torch.Generator().manual_seed(21)
        ctxs = (torch.randint(0, 5, (batch,), generator=g0) * 64 + torch.randint(1, 59, (batch,), generator=g0)).tolist()
    inp = workloads.decoder_layer_inputs(batch=batch, hidden=1024, num_heads=8, kv_head_num=2, head_dim=128,
                                         intermediate=2816, block_size=64, context_lens=ctxs, seed=11)
    args = _cuda(inp.args())
    hidden, seq_lens, key_cache, value_cache, out = args[0], args[1], args[3], args[4], args[19]
    assert out.shape == hidden.shape
    stream = torch.cuda.Stream()
    # eager twin on its own copies of everything the step writes
    twin = list(args)
    for i in (0, 1, 3, 4, 19):
        twin[i] = args[i].clone()
    graph = _capture(worker, decoder_layer_decode, args, stream)
    # the warm-up and the capture's own (unexecuted) call left the caches one step ahead of the twin
    with worker.register(decoder_layer_decode) as h:
        h(*twin)
    worker.sync()
    g = torch.Generator(device="cuda").manual_seed(5)
    for step in range(4):
        # next decode step: one more token per sequence, new activations
        new_hidden = torch.randn(hidden.shape, generator=g, device="cuda").to(hidden.dtype)
        for a in (args, twin):
            a[0].copy_(new_hidden)
            a[1].add_(1)
        torch.cuda.synchronize()
        graph.replay()
        with worker.register(decoder_layer_decode) as h:
            h(*twin)
        torch.cuda.synchronize()
        assert torch.isfinite(out.float()).all()
        assert torch.equal(out, twin[19]), f"replay {step} differs from the eager step"
        assert torch.equal(key_cache, twin[3]) and torch.equal(value_cache, twin[4])
    assert int(seq_lens[0]) == ctxs[0] + 4


def test_attention_and_ffn_replays(worker):
    att = workloads.paged_attention_inputs(batch=4, num_heads=16, kv_head_num=4, head_dim=128, block_size=64,
                                           context_lens=[300, 40, 1, 680], ctx_range=(1, 1024), seed=3)
    a_args = _cuda(att.args(), keep_host=(6,))
    ffn = workloads.ffn_inputs(tokens=200, hidden=1024, intermediate=2816, seed=4)
    f_args = _cuda((ffn.x, ffn.gamma, ffn.w_gate, ffn.w_up, ffn.w_down, ffn.out, ffn.eps))
    stream = torch.cuda.Stream()
    # The FFN call after the attention capture needs a larger scratch buffer than the one the
    # attention launches were recorded with: the outgrown buffer must stay allocated.
    ga = _capture(worker, paged_attention, a_args, stream)
    gf = _capture(worker, ffn_block, f_args, stream)
    for step in range(3):
        a_args[4].add_(5)                       # longer contexts, still inside each sequence's last block
        f_args[0].mul_(0.5)
        a_args[5].fill_(float("nan"))
        f_args[5].fill_(float("nan"))
        torch.cuda.synchronize()
        ga.replay()
        gf.replay()
        torch.cuda.synchronize()
        got_a, got_f = a_args[5].clone(), f_args[5].clone()
        with worker.register(paged_attention) as h:
            h(*a_args)
        with worker.register(ffn_block) as h:
            h(*f_args)
        worker.sync()
        assert torch.equal(got_a, a_args[5]), f"attention replay {step}"
        assert torch.equal(got_f, f_args[5]), f"ffn replay {step}"


def test_a_skinny_projection_sizes_its_scratch_for_every_batch(worker):
    """One eager call is what a caller owes before it captures: the scratch it leaves must do for the other
    batch sizes of the shape, since it cannot grow under capture."""
    held = worker.get_option("workspace_bytes")
    k, n = 32, (held // (4 * 32) // 128 + 512) * 128  # partial sums of 32 rows beyond everything held so far
    x = torch.randn((32, k), device="cuda").to(torch.bfloat16)
    w = torch.randn((k, n), device="cuda", dtype=torch.bfloat16)
    out = torch.empty((32, n), device="cuda")
    with worker.register(projection) as h:
        h(x[:1], w, out[:1])
        sized = worker.get_option("workspace_bytes")
        assert sized > held
        h(x, w, out)
    worker.sync()
    assert worker.get_option("workspace_bytes") == sized


@pytest.mark.parametrize("hidden,inter", [(512, 1024), (512, 3520), (40, 96)])  # narrow tiles; skinny projections; no k for those
@pytest.mark.parametrize("norm", [False, True])
def test_an_ffn_call_sizes_its_scratch_for_up_to_32_tokens(worker, hidden, inter, norm):
    """One eager call of one token, then a capture of 32 of the same block: whichever form its products take."""
    _without_scratch(worker)
    f = workloads.ffn_inputs(tokens=32, hidden=hidden, intermediate=inter, with_norm=norm, seed=hidden, device="cuda")

    def call(h, tokens, out, **kw):
        h(f.x[:tokens], *((f.gamma,) if norm else ()), f.w_gate, f.w_up, f.w_down, out, *((f.eps,) if norm else ()), **kw)

    got = torch.full_like(f.out, float("nan"))
    stream = torch.cuda.Stream()
    with worker.register(ffn_block if norm else ffn_swiglu) as h:
        call(h, 1, f.out[:1])
        worker.sync()
        held = worker.get_option("workspace_bytes")
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call(h, 32, got, stream=stream.cuda_stream)
        assert worker.get_option("workspace_bytes") == held
        call(h, 32, f.out)
        worker.sync()
        for _ in range(3):
            got.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(got, f.out)
            call(h, 1, torch.empty_like(f.out[:1]))


def _replays_agree(worker, graph, outputs, eager, again):
    """Three replays against an eager call that may take another form: bf16 outputs apart by two units in the norm."""
    for _ in range(3):
        for t in outputs:
            t.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        for t, want in zip(outputs, eager):
            assert ((t.double() - want.double()).norm() / want.double().norm()).item() < 2.0 ** -7
        again()


def test_streamed_forms_do_not_grow_their_scratch_under_capture(worker):
    """A block and a layer of some tens of rows whose streamed form needs more scratch than is held, the tiled one not: captured tiled.  (The
    slabs of the streamed products fit: an earlier call of another shape left room for them.)"""
    _without_scratch(worker)
    f = workloads.ffn_inputs(tokens=96, hidden=64, intermediate=8192, with_norm=False, out_dtype=torch.bfloat16, seed=1, device="cuda")
    wide = workloads.ffn_inputs(tokens=96, hidden=16384, intermediate=64, with_norm=False, out_dtype=torch.bfloat16, seed=2, device="cuda")
    d = workloads.decoder_layer_inputs(batch=33, hidden=64, num_heads=1, kv_head_num=1, intermediate=8192, block_size=64, context=40, seed=3,
                                       device="cuda", int8_weights=False, weight_std=None)
    stream = torch.cuda.Stream()
    with worker.register(ffn_swiglu) as h, worker.register(decoder_layer_decode_w16) as layer:
        wide_args, f_args = ((g.x, g.w_gate, g.w_up, g.w_down, g.out) for g in (wide, f))
        try:
            worker.set_option("gemm_stream", 0)
            layer(*d.args())  # attention's scratch and the tiled layer's
            worker.set_option("gemm_stream", 2)
            h(*f_args)
            worker.sync()
            held = worker.get_option("workspace_bytes")
            graphs = [torch.cuda.CUDAGraph() for _ in range(2)]
            with torch.cuda.graph(graphs[0], stream=stream):
                h(*wide_args, stream=stream.cuda_stream)
            with torch.cuda.graph(graphs[1], stream=stream):
                layer(*d.args(), stream=stream.cuda_stream)
            assert worker.get_option("workspace_bytes") == held
            for call, args in ((h, wide_args), (layer, d.args())):  # the streamed forms, not captured
                call(*args)
                worker.sync()
                assert worker.get_option("workspace_bytes") > held
                held = worker.get_option("workspace_bytes")
        finally:
            worker.set_option("gemm_stream", 1)
        _replays_agree(worker, graphs[0], [wide.out], [wide.out.clone()], lambda: h(*f_args))
        _replays_agree(worker, graphs[1], [d.out], [d.out.clone()], lambda: h(*f_args))


def _without_scratch(worker):
    """The library's scratch areas are given back, as in a process that has just started."""
    torch.cuda.synchronize()
    worker.close()
    worker.init()
    assert worker.get_option("workspace_bytes") == 0


@pytest.mark.parametrize("hi", [100, 1500, 8000])
@pytest.mark.parametrize("fp8", [False, True])
def test_an_attention_call_sizes_its_scratch_for_smaller_batches(worker, fp8, hi):
    """One eager call is what a caller owes before it captures, whatever form that call took: here a workgroup per pair or one
    partition, without partials of its own."""
    _without_scratch(worker)

    def call(batch):
        inp = workloads.paged_attention_inputs(batch=batch, num_heads=32, kv_head_num=8, context_lens=[hi] * batch, ctx_range=(1, hi), fp8_kv=fp8,
                                               seed=batch, device="cuda")
        with worker.register(paged_attention) as h:
            h(*inp.args())
        worker.sync()
        return worker.get_option("workspace_bytes")

    sized = call(32)
    assert sized > 0
    for batch in (31, 30, 17, 13, 9, 8, 5, 3, 2, 1):
        assert call(batch) == sized, batch


def test_an_eager_attention_call_leaves_another_streams_capture_alone(worker):
    """The room it makes for smaller batches is its own affair: a capture that is going on elsewhere ends and replays as recorded."""
    inp = workloads.paged_attention_inputs(batch=32, num_heads=32, kv_head_num=8, context_lens=[300] * 32, ctx_range=(1, 300), seed=9, device="cuda")
    with worker.register(paged_attention) as h:
        h(*inp.args())  # (loads the kernels)
    _without_scratch(worker)
    x = torch.zeros(64, device="cuda")
    recorded, eager = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    worker.set_option("attn_autotune", 0)
    try:
        with worker.register(paged_attention) as h:
            with torch.cuda.graph(graph, stream=recorded):
                x.add_(1.0)
                h(*inp.args(), stream=eager.cuda_stream)
                x.mul_(2.0)
            worker.sync()
            got = inp.out.clone()
            h(*inp.args())
            worker.sync()
    finally:
        worker.set_option("attn_autotune", 1)
    assert torch.equal(got, inp.out) and bool(got.isfinite().all())
    for step in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert bool((x == 2.0 ** (step + 2) - 2.0).all())


@pytest.mark.parametrize("ctx,d", [(100, 128), (250, 256)])
def test_a_captured_attention_call_without_scratch_takes_whole_blocks(worker, ctx, d):
    """Nothing ran before the capture, so there is no room for partials: the graph holds the call on whole blocks, bit for bit."""
    inp = workloads.paged_attention_inputs(batch=1, num_heads=8, kv_head_num=8, head_dim=d, block_size=256, context_lens=[ctx], ctx_range=(1, 256), seed=ctx,
                                           device="cuda")
    args = inp.args()
    with worker.register(paged_attention) as h:
        worker.set_option("attn_tokens_per_partition", 256)
        try:
            h(*args)
        finally:
            worker.set_option("attn_tokens_per_partition", 0)
        worker.sync()
        want = inp.out.clone()
        h(*args)  # (loads the kernels of the cut form)
        worker.sync()
    _without_scratch(worker)
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with worker.register(paged_attention) as h:
        with torch.cuda.graph(graph, stream=stream):
            h(*args, stream=stream.cuda_stream)
    assert worker.get_option("workspace_bytes") == 0
    for _ in range(3):
        inp.out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(inp.out, want)


@pytest.mark.parametrize("kind", ["e4m3", "16-bit"])
def test_a_split_product_is_captured_unsplit_when_its_slabs_do_not_fit(worker, kind):
    """No eager call of the split form before the capture: the graph holds the unsplit product, bit for bit, and the
    scratch has not grown."""
    from pypto_amd import _lib
    from pypto_amd.runtime import _dtype_code

    lib, bf16 = _lib.load(), _dtype_code(torch.bfloat16)
    k, n = 2048, 2048
    m = worker.get_option("workspace_bytes") // (16 * 2 * 4 * n) + 256  # 8 splits' slabs: beyond half of everything held
    m *= 2
    g = torch.Generator(device="cuda").manual_seed(m)
    x, wg, wu = (torch.randn(s, generator=g, device="cuda") for s in ((m, k), (k, n), (k, n)))
    out, want = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    one = torch.ones(max(m, n), device="cuda")
    if kind == "e4m3":
        x, wg, wu = (t.to(torch.float8_e4m3fn) for t in (x, wg.t().contiguous(), wu.t().contiguous()))
    else:
        x, wg, wu = (t.to(torch.bfloat16) for t in (x, wg, wu))

    def call(dst, stream):
        if kind == "e4m3":
            _lib.check(lib.pto_hip_gate_up_swiglu_fp8(x.data_ptr(), one.data_ptr(), wg.data_ptr(), one.data_ptr(), wu.data_ptr(),
                                                      one.data_ptr(), dst.data_ptr(), m, k, n, bf16, stream.cuda_stream))
        else:
            _lib.check(lib.pto_hip_gate_up_swiglu(x.data_ptr(), wg.data_ptr(), wu.data_ptr(), dst.data_ptr(), m, k, n, bf16,
                                                  stream.cuda_stream))

    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    worker.set_option("gemm_variant", 5)
    try:
        worker.set_option("gemm_splits", 1)
        call(want, stream)
        stream.synchronize()
        held = worker.get_option("workspace_bytes")
        worker.set_option("gemm_splits", 8)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            call(out, stream)
    finally:
        worker.set_option("gemm_variant", 0)
        worker.set_option("gemm_splits", 0)
    assert worker.get_option("workspace_bytes") == held
    for _ in range(3):
        out.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)
