"""The products of a small call (narrow_gemm.h) in every tile, against the oracle, between guarded operands."""

import pytest
import torch

import oracle
from pypto_amd.runtime import ffn_block, gate_up_swiglu, projection, projection_residual, validate_golden

pytestmark = pytest.mark.gpu
TILES = (1, 2, 3, 4)


def _between(shape, dtype, fill):
    """A tensor with 512 elements of `fill` on either side (16-byte aligned for every type used)."""
    n = shape[0] * shape[1]
    buf = torch.full((1024 + n,), fill, dtype=dtype, device="cuda")
    return buf, buf[512:512 + n].view(shape)


# rows and columns at, below and above every tile's; k below one step of all eight wavefronts, 1 to 5 steps a wavefront with and
# without a step that ends inside, and past the steps that are requested at once
@pytest.mark.parametrize("m,k,n", [(1, 32, 8), (15, 40, 32), (17, 264, 40), (16, 256, 64), (64, 512, 72), (65, 776, 56), (33, 1024, 136),
                                   (48, 1032, 264), (63, 1288, 128), (129, 2080, 96)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_every_tile_gives_the_product_and_stays_inside_its_operands(worker, m, k, n, dtype):
    g = torch.Generator(device="cuda").manual_seed(m * k + n)
    (_, x), (_, w), (_, wu) = (_between(s, dtype, float("nan")) for s in ((m, k), (k, n), (k, n)))
    x.copy_(torch.randn((m, k), generator=g, device="cuda") / k ** 0.5)
    w.copy_(torch.randn((k, n), generator=g, device="cuda"))
    wu.copy_(torch.randn((k, n), generator=g, device="cuda"))
    res = torch.randn((m, n), generator=g, device="cuda")
    ref, ref_up = oracle.projection(x.cpu(), w.cpu()), oracle.projection(x.cpu(), wu.cpu())
    both = oracle.swiglu(ref, ref_up)
    tol16 = 1e-2 if dtype == torch.bfloat16 else 2e-3
    try:
        for tile in TILES:
            worker.set_option("gemm_narrow", tile)
            for program, args, out_dtype, want, tol in ((projection, (x, w), torch.float32, ref, 2e-3), (projection, (x, w), dtype, ref, tol16),
                                                        (projection_residual, (x, w, res), torch.float32, ref + res.cpu(), 2e-3),
                                                        (gate_up_swiglu, (x, w, wu), dtype, both, tol16)):
                if m <= 32 and k * n * (2 if program is gate_up_swiglu else 1) > 1600000:
                    continue  # the skinny form has these
                buf, out = _between((m, n), out_dtype, -77.0)
                with worker.register(program) as h:
                    h(*args, out)
                worker.sync()
                validate_golden({"out": out.cpu().float()}, {"out": want.float()}, rtol=tol, atol=tol)
                assert bool((buf[:512] == -77.0).all()) and bool((buf[512 + m * n:] == -77.0).all()), (tile, program.name)
    finally:
        worker.set_option("gemm_narrow", 0)


@pytest.mark.parametrize("k", [40, 264, 520, 1032])
def test_a_step_that_ends_inside_keeps_infinities_apart(worker, k):
    """The last step of a k that is no multiple of 32 repeats rows: an infinite weight among them must not become NaN."""
    m, n = 33, 40
    x = torch.ones(m, k, dtype=torch.bfloat16)
    w = torch.zeros(k, n, dtype=torch.bfloat16)
    w[-32, 0] = w[-1, -1] = float("inf")
    try:
        for tile in TILES:
            worker.set_option("gemm_narrow", tile)
            out = torch.zeros(m, n)
            with worker.register(projection) as h:
                h(x, w, out)
            assert bool((out[:, 0] == float("inf")).all()) and bool((out[:, -1] == float("inf")).all()), tile
            assert bool((out[:, 1:-1] == 0.0).all()), tile
    finally:
        worker.set_option("gemm_narrow", 0)


@pytest.mark.parametrize("tokens", [1, 32, 33, 128, 500])
def test_small_block_against_the_tiled_and_skinny_forms(worker, tokens):
    """The block as it is dispatched, with its norm, beside the same block with the form switched off: both are fp32 sums of
    the same products and h is rounded once, so they differ by the order of the sums (an ulp of h where that crosses a rounding
    boundary: 2^-8 of h, a 512th of the 1024 terms' sum)."""
    from pypto_amd import workloads
    f = workloads.ffn_inputs(tokens=tokens, hidden=512, intermediate=1024, seed=tokens, device="cuda")
    got = []
    try:
        for narrow in (0, -1):
            worker.set_option("gemm_narrow", narrow)
            out = torch.zeros_like(f.out)
            with worker.register(ffn_block) as h:
                h(f.x, f.gamma, f.w_gate, f.w_up, f.w_down, out, f.eps)
            worker.sync()
            got.append(out.double())
    finally:
        worker.set_option("gemm_narrow", 0)
    assert ((got[0] - got[1]).norm() / got[1].norm()).item() < 2.0 ** -9


@pytest.mark.parametrize("k,n", [(512, 512), (1024, 256)])
@pytest.mark.parametrize("m", [1, 17, 32])
@pytest.mark.parametrize("program", [projection, gate_up_swiglu])
def test_a_result_laid_over_its_operand(worker, m, k, n, program):
    """Up to 32 rows a result may lie where the activations do: the small-call form would write them while other workgroups still read, so
    such a call takes the form with a finish of its own, and has its bits."""
    g = torch.Generator(device="cuda").manual_seed(m + n)
    x = (torch.randn((m, k), generator=g, device="cuda") / k ** 0.5).to(torch.bfloat16)
    w = tuple(torch.randn((k, n), generator=g, device="cuda").to(torch.bfloat16) for _ in range(1 if program is projection else 2))
    with worker.register(program) as h:
        want = torch.zeros((m, n), dtype=torch.bfloat16, device="cuda")
        worker.set_option("gemm_narrow", -1)
        try:
            h(x, *w, want)
        finally:
            worker.set_option("gemm_narrow", 0)
        for _ in range(8):
            buf = x.clone()
            over = buf.flatten()[:m * n].view(m, n)
            h(buf, *w, over)
            worker.sync()
            assert torch.equal(over, want)


@pytest.mark.parametrize("program,m,more,k,n", [(projection, 8, 40, 2048, 1024), (gate_up_swiglu, 8, 40, 1024, 1024), (ffn_block, 8, 100, 1024, 1024),
                                                (ffn_block, 40, 100, 4096, 11008)])
def test_a_tile_asked_for_is_taken_whatever_the_rows(worker, program, m, more, k, n):
    """Shapes that the skinny form (up to 32 rows) and the streams (33 to 96) have by default: with a tile forced, a row has the bits that it has
    in a call of more rows, which only the small-call form gives."""
    from pypto_amd import workloads
    f = workloads.ffn_inputs(tokens=more, hidden=k, intermediate=n, out_dtype=torch.float32, seed=m, device="cuda")
    weights = {projection: (f.w_gate,), gate_up_swiglu: (f.w_gate, f.w_up), ffn_block: (f.w_gate, f.w_up, f.w_down)}[program]
    width, out_dtype = (k if program is ffn_block else n), torch.bfloat16 if program is gate_up_swiglu else torch.float32
    got = {}
    try:
        for tile in (0, 3):
            worker.set_option("gemm_narrow", tile)
            for rows in (m, more):
                out = torch.full((rows, width), float("nan"), dtype=out_dtype, device="cuda")
                with worker.register(program) as h:
                    h(*((f.x[:rows], f.gamma) if program is ffn_block else (f.x[:rows],)), *weights, out, *((f.eps,) if program is ffn_block else ()))
                worker.sync()
                got[tile, rows] = out
    finally:
        worker.set_option("gemm_narrow", 0)
    assert torch.equal(got[3, m], got[3, more][:m])
    assert not torch.equal(got[3, m], got[0, m])
