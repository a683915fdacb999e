"""Skinny projections of up to four rows that make their activations themselves (skinny.h): the bits of the separate launches."""

import pytest
import torch

from pypto_amd import runtime, workloads

pytestmark = pytest.mark.gpu


def _run(worker, program, args, outputs, fuse):
    """The outputs of one call and the sources its projections took, its caches put back afterwards."""
    before = [t.clone() for t in outputs]
    worker.set_option("skinny_fuse", fuse)
    try:
        with worker.register(program) as h:
            for _ in range(2):  # (the second call may take another launch shape of the attention: the same bits)
                for t, b in zip(outputs, before):
                    t.copy_(b)
                h(*args)
        worker.sync()
        took = worker.get_option("skinny_fused")
    finally:
        worker.set_option("skinny_fuse", 7)
    got = [t.clone() for t in outputs]
    for t, b in zip(outputs, before):
        t.copy_(b)
    return got, took


def _same(a, b):
    return all(torch.equal(x.view(torch.uint8), y.view(torch.uint8)) for x, y in zip(a, b))


# hidden with a half last step and without, shares of one and several pieces; head_dim 128 and 256; one partition, up to 8, up
# to 40 and more (which keeps its merge launch); an empty sequence beside long ones; 8 and 16 codes a lane.  The calls are not measured: a
# measured call keeps its merge launch.  takes: the sources that the dispatch takes
@pytest.mark.parametrize("batch,hidden,heads,kv_heads,head_dim,inter,block,lens,int8,e4m3,wide,takes", [
    (1, 4096, 32, 8, 128, 14336, 128, [2049], True, False, 1, 7), (2, 1040, 8, 2, 128, 2064, 64, [1, 700], True, False, 1, 7),
    (4, 1040, 8, 1, 128, 2064, 64, [0, 33, 1300, 2500], False, False, 1, 3), (3, 512, 4, 4, 256, 1040, 128, [400, 0, 3000], False, False, 1, 7),
    (1, 2048, 8, 2, 256, 4096, 64, [1111], True, True, 1, 7), (4, 2048, 16, 4, 128, 5632, 128, [600, 599, 1, 128], False, False, 1, 3),
    (2, 2048, 16, 4, 128, 5632, 128, [600, 5000], True, True, 2, 3), (1, 48, 2, 1, 128, 80, 16, [17], True, False, 1, 3),
    (1, 8192, 64, 8, 128, 8192, 128, [900], True, False, 2, 3), (1, 2048, 8, 2, 256, 4096, 64, [450], False, False, 1, 7),
    (1, 2048, 8, 2, 256, 4096, 64, [5000], True, False, 1, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_decoder_layer_has_the_bits_of_separate_launches(worker, batch, hidden, heads, kv_heads, head_dim, inter, block, lens, int8, e4m3, wide, takes, dtype):
    d = workloads.decoder_layer_inputs(batch=batch, hidden=hidden, num_heads=heads, kv_head_num=kv_heads, head_dim=head_dim, intermediate=inter,
                                       block_size=block, context_lens=lens, dtype=dtype, seed=hidden + batch, device="cuda", int8_weights=int8,
                                       weight_std=None)
    args, outputs = d.args(), [d.out, d.key_cache, d.value_cache]
    if e4m3:
        from perf.cases import _quantised
        kc, ks = _quantised(d.key_cache, kv_heads, block)
        vc, vs = _quantised(d.value_cache, kv_heads, block)
        args, outputs = args[:3] + (kc, vc, ks, vs) + args[5:], [d.out, kc, vc, ks, vs]
        program = runtime.decoder_layer_decode_fp8kv if int8 else runtime.decoder_layer_decode_w16_fp8kv
    else:
        program = runtime.decoder_layer_decode if int8 else runtime.decoder_layer_decode_w16
    worker.set_option("w8a16_wide", wide)
    worker.set_option("attn_autotune", 0)
    try:
        ref, none = _run(worker, program, args, outputs, 0)
        assert bool(ref[0].isfinite().all()) and none == 0
        for fuse in (1, 2, 4, 7):
            got, took = _run(worker, program, args, outputs, fuse)
            assert _same(got, ref), fuse
            assert took == fuse & takes, fuse
    finally:
        worker.set_option("attn_autotune", 1)
        worker.set_option("w8a16_wide", 1)


@pytest.mark.parametrize("hidden,heads,lens,int8", [(4096, 32, [2049], True), (2048, 16, [1500, 900], False)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_measured_and_settled_calls_have_the_same_bits(worker, hidden, heads, lens, int8, dtype):
    """The calls that measure a signature merge its partitions in a launch, the later ones inside the o projection."""
    d = workloads.decoder_layer_inputs(batch=len(lens), hidden=hidden, num_heads=heads, kv_head_num=heads // 4, intermediate=3 * hidden, block_size=128,
                                       context_lens=lens, dtype=dtype, seed=5, device="cuda", int8_weights=int8, weight_std=None)
    worker.set_option("attn_autotune", 0)  # forget what earlier tests settled
    worker.set_option("attn_autotune", 1)
    outs, merged = [], []
    with worker.register(runtime.decoder_layer_decode if int8 else runtime.decoder_layer_decode_w16) as h:
        for _ in range(32):
            h(*d.args())
            worker.sync()
            outs.append(d.out.clone())
            merged.append(bool(worker.get_option("skinny_fused") & 4))
    assert not merged[0] and merged[-1]
    assert all(torch.equal(o, outs[0]) for o in outs)


@pytest.mark.parametrize("tokens,hidden,inter", [(1, 4096, 11008), (2, 1040, 4112), (3, 2048, 5632), (4, 1024, 3072), (4, 8192, 2048), (1, 48, 40000), (1, 4096, 16384), (2, 4096, 16384),
                                                 (1, 2496, 8448), (2, 2560, 8448)])  # the pair's channels have two or three partial sums
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_ffn_block_has_the_bits_of_separate_launches(worker, tokens, hidden, inter, dtype):
    f = workloads.ffn_inputs(tokens=tokens, hidden=hidden, intermediate=inter, dtype=dtype, seed=tokens, device="cuda")
    args = (f.x, f.gamma, f.w_gate, f.w_up, f.w_down, f.out, f.eps)
    worker.set_option("gemm_narrow", -1)
    try:
        ref, none = _run(worker, runtime.ffn_block, args, [f.out], 0)
        assert none == 0
        seen = 0
        for fuse in (1, 2, 7):
            got, took = _run(worker, runtime.ffn_block, args, [f.out], fuse)
            assert _same(got, ref), fuse
            seen |= took
        assert seen
    finally:
        worker.set_option("gemm_narrow", 0)


@pytest.mark.parametrize("tokens", [1, 4, 7, 32])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_step_that_ends_inside_keeps_infinities_apart(worker, tokens, dtype):
    """k of 48 and 1040: the last 32-row step repeats 16 rows, and an infinite weight among them must not become NaN.  With and without a norm (of
    ones: ones), the projections' own activations and given ones; SiLU(8) is nearly 8, so that h is finite but for its infinite channels."""
    hidden, inter = 48, 1040
    x, gamma = torch.ones(tokens, hidden, dtype=dtype, device="cuda"), torch.ones(1, hidden, device="cuda")
    wg = torch.full((hidden, inter), 8.0 / hidden, dtype=dtype, device="cuda")
    wd = torch.full((inter, hidden), 1.0 / inter, dtype=dtype, device="cuda")
    wu_inf, wd_inf = wg.clone(), wd.clone()
    wu_inf[-32, 3] = wd_inf[-32, 0] = wd_inf[-1, -1] = float("inf")
    out = torch.zeros(tokens, hidden, dtype=torch.float32, device="cuda")
    worker.set_option("gemm_narrow", -1)
    try:
        for fuse in (0, 7):
            worker.set_option("skinny_fuse", fuse)
            for program, gamma_arg, eps in ((runtime.ffn_swiglu, (), ()), (runtime.ffn_block, (gamma,), (1e-6,))):
                with worker.register(program) as h:
                    def call(wu, wd):
                        out.fill_(float("nan"))
                        h(x, *gamma_arg, wg, wu, wd, out, *eps)
                        worker.sync()
                        return out.clone()

                    assert bool(call(wg, wd).isfinite().all())
                    got = call(wg, wd_inf)
                    assert bool((got[:, 0] == float("inf")).all()) and bool((got[:, -1] == float("inf")).all()) and bool(got[:, 1:-1].isfinite().all())
                    assert bool((call(wu_inf, wd) == float("inf")).all())
    finally:
        worker.set_option("gemm_narrow", 0)
        worker.set_option("skinny_fuse", 7)


def test_replays_of_a_captured_layer(worker):
    """Recorded after one eager call, replayed between eager calls that use the same scratch."""
    d = workloads.decoder_layer_inputs(batch=1, hidden=2048, num_heads=16, kv_head_num=4, intermediate=5632, context_lens=[700], seed=3, device="cuda")
    big = workloads.decoder_layer_inputs(batch=8, hidden=2048, num_heads=16, kv_head_num=4, intermediate=5632, context=900, seed=4, device="cuda")
    want = _run(worker, runtime.decoder_layer_decode, d.args(), [d.out, d.key_cache, d.value_cache], 0)[0]
    stream = torch.cuda.Stream()
    with worker.register(runtime.decoder_layer_decode) as h:
        with torch.cuda.stream(stream):
            h(*d.args(), stream=stream.cuda_stream)
            stream.synchronize()
            graph = torch.cuda.CUDAGraph()
            graph.capture_begin()
            h(*d.args(), stream=stream.cuda_stream)
            graph.capture_end()
            assert worker.get_option("skinny_fused") & 4
            for _ in range(3):
                d.out.zero_()
                graph.replay()
                stream.synchronize()
                assert torch.equal(d.out, want[0]) and torch.equal(d.key_cache, want[1]) and torch.equal(d.value_cache, want[2])
                h(*big.args(), stream=stream.cuda_stream)
                stream.synchronize()
