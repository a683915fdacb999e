"""Projections of 33 to 96 rows that stream their weights (stream_rows.h), inside decoder layers and FFN blocks."""

import ctypes as C

import pytest
import torch

import oracle
from pypto_amd import _lib, runtime, workloads

pytestmark = pytest.mark.gpu


def _error(got, want):
    return ((got.double() - want.double()).norm() / want.double().norm()).item()


# row groups of 16 full and not, 3, 4 and 6 of them; k that ends inside a 32-row step, fewer steps than wavefronts, columns
# that end inside a slab and inside a matrix of a pair
@pytest.mark.parametrize("batch", [33, 48, 49, 64, 65, 96])
@pytest.mark.parametrize("hidden,heads,kv_heads,inter,int8,dtype", [
    (512, 4, 2, 1040, True, torch.float16), (1040, 8, 1, 2064, True, torch.bfloat16), (1040, 8, 1, 2064, False, torch.bfloat16),
    (48, 2, 1, 80, False, torch.float16), (2048, 5, 5, 4112, False, torch.float16), (4096, 32, 8, 1344, True, torch.bfloat16)])
def test_decoder_layer_streamed_beside_tiled(worker, batch, hidden, heads, kv_heads, inter, int8, dtype):
    """Both are fp32 sums of the same products, rounded to the activation type at the same places: they differ by what a sum in another
    order moves across a rounding boundary, under two units of the type in the norm (2^-8 bf16, 2^-11 fp16)."""
    lens = [1 + (37 * i) % 130 for i in range(batch)]
    d = workloads.decoder_layer_inputs(batch=batch, hidden=hidden, num_heads=heads, kv_head_num=kv_heads, intermediate=inter, block_size=64,
                                       context_lens=lens, dtype=dtype, seed=batch, device="cuda", int8_weights=int8, weight_std=None)
    before = d.key_cache.clone(), d.value_cache.clone()
    program = runtime.decoder_layer_decode if int8 else runtime.decoder_layer_decode_w16
    got = []
    try:
        for stream in (0, 2, 2):
            worker.set_option("gemm_stream", stream)
            d.key_cache.copy_(before[0])
            d.value_cache.copy_(before[1])
            d.out.fill_(float("nan"))
            with worker.register(program) as h:
                h(*d.args())
            worker.sync()
            got.append((d.out.clone(), d.key_cache.clone(), d.value_cache.clone()))
    finally:
        worker.set_option("gemm_stream", 1)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert all(torch.equal(a, b) for a, b in zip(got[1], got[2]))
    for a, b in zip(got[1], got[0]):
        assert bool(a.isfinite().all()) and _error(a, b) < 2 * unit


@pytest.mark.parametrize("tokens,hidden,inter", [(33, 1040, 4112), (64, 2048, 1032), (90, 48, 200), (96, 4096, 11008)])
@pytest.mark.parametrize("out_dtype", [torch.float32, torch.bfloat16])
def test_ffn_block_streamed_against_the_oracle(worker, tokens, hidden, inter, out_dtype):
    f = workloads.ffn_inputs(tokens=tokens, hidden=hidden, intermediate=inter, out_dtype=out_dtype, seed=tokens, device="cuda")
    buf = torch.full((tokens * hidden + 1024,), -77.0, dtype=out_dtype, device="cuda")
    out = buf[512:512 + tokens * hidden].view(tokens, hidden)
    worker.set_option("gemm_stream", 2)
    try:
        with worker.register(runtime.ffn_block) as h:
            h(f.x, f.gamma, f.w_gate, f.w_up, f.w_down, out, f.eps)
        worker.sync()
    finally:
        worker.set_option("gemm_stream", 1)
    ref = oracle.ffn_block(f.x.cpu(), f.gamma.cpu(), f.w_gate.cpu(), f.w_up.cpu(), f.w_down.cpu(), f.eps)
    runtime.validate_golden({"out": out.cpu().float()}, {"out": ref.float()}, rtol=2e-2, atol=1e-2)
    assert bool((buf[:512] == -77.0).all()) and bool((buf[512 + tokens * hidden:] == -77.0).all())


@pytest.mark.parametrize("tokens,hidden,inter", [(33, 1040, 4112), (47, 264, 1032), (65, 48, 200), (96, 20488, 512)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_ffn_without_a_norm_streamed_beside_tiled(worker, tokens, hidden, inter, dtype):
    """The copy into the blocked layout moves values as they are (rows beyond the norm's limit too): the two routes differ by the order of
    fp32 sums and, through it, by single roundings of h to 16 bits, of which a sum over `inter` averages most."""
    f = workloads.ffn_inputs(tokens=tokens, hidden=hidden, intermediate=inter, dtype=dtype, with_norm=False, out_dtype=torch.float32, seed=tokens, device="cuda")
    got = {}
    try:
        for stream in (0, 2):
            worker.set_option("gemm_stream", stream)
            f.out.fill_(float("nan"))
            with worker.register(runtime.ffn_swiglu) as h:
                h(f.x, f.w_gate, f.w_up, f.w_down, f.out)
            worker.sync()
            got[stream] = f.out.clone()
    finally:
        worker.set_option("gemm_stream", 1)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert bool(got[2].isfinite().all()) and _error(got[2], got[0]) < unit


@pytest.mark.parametrize("tokens,hidden,inter", [(33, 40, 264), (64, 1032, 48), (96, 264, 1048)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_a_step_that_ends_inside_keeps_infinities_apart(worker, tokens, hidden, inter, dtype):
    """The last step of a k that is no multiple of 32 repeats rows: an infinite weight among them must not become NaN.  The gate is one on
    every channel (SiLU(8) is nearly 8, an infinite gate stays infinite), so that h is finite and positive but for its infinite channels."""
    x = torch.ones(tokens, hidden, dtype=dtype, device="cuda")
    wg = torch.full((hidden, inter), 8.0 / hidden, dtype=dtype, device="cuda")
    wu, wd = wg.clone(), torch.full((inter, hidden), 1.0 / inter, dtype=dtype, device="cuda")
    out = torch.zeros(tokens, hidden, dtype=torch.float32, device="cuda")

    def call(wu, wd):
        out.fill_(float("nan"))
        h(x, wg, wu, wd, out)
        worker.sync()
        return out.clone()

    worker.set_option("gemm_stream", 2)
    try:
        with worker.register(runtime.ffn_swiglu) as h:
            assert bool(call(wu, wd).isfinite().all())
            wd_inf = wd.clone()
            wd_inf[-32, 0] = wd_inf[-1, -1] = float("inf")
            got = call(wu, wd_inf)
            assert bool((got[:, 0] == float("inf")).all()) and bool((got[:, -1] == float("inf")).all()) and bool(got[:, 1:-1].isfinite().all())
            wu_inf = wu.clone()
            wu_inf[-32, 3] = float("inf")
            assert bool((call(wu_inf, wd) == float("inf")).all())
    finally:
        worker.set_option("gemm_stream", 1)


def test_replays_of_a_captured_block(worker):
    """Recorded after one eager call; every replay, between eager calls that use the same scratch, gives its result."""
    small = workloads.ffn_inputs(tokens=40, hidden=4096, intermediate=11008, seed=1, device="cuda")
    torch.cuda.synchronize()  # the inputs are made on another stream than the call's
    with worker.register(runtime.ffn_block) as h:
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            h(small.x, small.gamma, small.w_gate, small.w_up, small.w_down, small.out, small.eps, stream=stream.cuda_stream)
            stream.synchronize()
            want = small.out.clone()
            graph = torch.cuda.CUDAGraph()
            graph.capture_begin()
            h(small.x, small.gamma, small.w_gate, small.w_up, small.w_down, small.out, small.eps, stream=stream.cuda_stream)
            graph.capture_end()
            for _ in range(3):
                small.out.zero_()
                graph.replay()
                stream.synchronize()
                assert torch.equal(small.out, want)
                h(small.x, small.gamma, small.w_gate, small.w_up, small.w_down, torch.empty_like(small.out), small.eps, stream=stream.cuda_stream)
                stream.synchronize()


class _LayerArgs(C.Structure):
    """PtoHipDecoderLayerArgs (programs refuse misaligned tensors by themselves, callers of the C interface do not)."""

    POINTERS = ("hidden_states seq_lens block_table key_cache value_cache rope_cos rope_sin gamma_in gamma_post wqkv_q wqkv_s wo_q wo_s wg_q wg_s "
                "wu_q wu_s wd_q wd_s out").split()
    SIZES = "batch hidden num_heads kv_head_num head_dim intermediate block_size max_num_blocks_per_req max_pos pool_rows".split()
    _fields_ = ([(n, C.c_void_p) for n in POINTERS] + [(n, C.c_int64) for n in SIZES] + [("eps", C.c_float)] +
                [(n, C.c_int32) for n in ("dtype", "kv_dtype", "rope_table_width")] + [("k_scale", C.c_void_p), ("v_scale", C.c_void_p)])


# the o projection with its finish and norm in one kernel (whose scale may start anywhere), and apart
@pytest.mark.parametrize("hidden,name", [(512, "wg_s"), (512, "wu_s"), (512, "wd_s"), (512, "out"), (8208, "wo_s"), (8208, "hidden_states")])
def test_a_streamed_layer_refuses_what_the_tiled_one_refuses(worker, hidden, name):
    """An operand that starts four bytes off a 16-byte boundary: the same refusal in both forms, and none where all are aligned."""
    d = workloads.decoder_layer_inputs(batch=40, hidden=hidden, num_heads=2, kv_head_num=1, intermediate=1040, block_size=64, context=50, seed=1,
                                       device="cuda", int8_weights=True, weight_std=None)
    tensors = dict(zip(_LayerArgs.POINTERS, d.args()))
    t = tensors[name]
    moved = torch.cat([t.flatten()[:4 // t.element_size()], t.flatten()])[4 // t.element_size():]
    assert moved.data_ptr() % 16 == 4
    lib, said = _lib.load(), []

    def call(**kw):
        a = _LayerArgs(**{n: t.data_ptr() for n, t in {**tensors, **kw}.items()}, batch=40, hidden=hidden, num_heads=2, kv_head_num=1, head_dim=128,
                       intermediate=1040, block_size=64, max_num_blocks_per_req=d.block_table.numel() // 40, max_pos=d.rope_cos.shape[0],
                       pool_rows=d.key_cache.shape[0], eps=d.eps, dtype=runtime._dtype_code(torch.bfloat16))
        _lib.check(lib.pto_hip_decoder_layer_decode(C.byref(a), None))

    try:
        for stream in (0, 2):
            worker.set_option("gemm_stream", stream)
            call()
            with pytest.raises(ValueError, match="misaligned") as refused:
                call(**{name: moved})
            worker.sync()
            said.append(str(refused.value))
    finally:
        worker.set_option("gemm_stream", 1)
    assert said[0] == said[1]
