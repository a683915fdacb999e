"""The e4m3 products of a small call (narrow_gemm8.h) in every tile, against exact sums and against the tiled GEMM."""

import pytest
import torch

from pypto_amd import _lib
from pypto_amd.runtime import _dtype_code

pytestmark = pytest.mark.gpu
F8 = torch.float8_e4m3fn
NAN8 = 0x7F


def _codes(rows, cols, values):
    """e4m3 codes [rows, cols] with 512 bytes of NaN on either side."""
    buf = torch.full((1024 + rows * cols,), NAN8, dtype=torch.uint8, device="cuda")
    view = buf[512:512 + rows * cols].view(rows, cols)
    view.copy_(values.to(F8).view(torch.uint8))
    return view


def _run(lib, x, sx, w, sw, w2, sw2, m, k, n, dtype):
    buf = torch.full((256 + m * n,), 7.0, dtype=dtype, device="cuda")
    out = buf[128:128 + m * n].view(m, n)
    if w2 is None:
        rc = lib.pto_hip_projection_fp8(x.data_ptr(), sx.data_ptr(), w.data_ptr(), sw.data_ptr(), out.data_ptr(), m, k, n, _dtype_code(dtype), 0)
    else:
        rc = lib.pto_hip_gate_up_swiglu_fp8(x.data_ptr(), sx.data_ptr(), w.data_ptr(), sw.data_ptr(), w2.data_ptr(), sw2.data_ptr(),
                                            out.data_ptr(), m, k, n, _dtype_code(dtype), 0)
    _lib.check(rc)
    torch.cuda.synchronize()
    assert (buf[:128] == 7).all() and (buf[128 + m * n:] == 7).all()
    return out


# rows and channels at, below and above every tile's; 1 step of 128 codes to past a full pipeline of eight wavefronts, with
# wavefronts that have none
SHAPES = [(1, 128, 4), (15, 384, 20), (16, 512, 16), (17, 640, 36), (33, 1024, 32), (64, 1152, 64), (65, 2816, 100), (130, 4224, 48), (63, 11008, 12)]


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_every_tile_is_exact_on_whole_numbers_and_stays_inside(worker, m, k, n):
    """Whole numbers up to 8 and scales that are powers of two: every partial sum is below 2^24 (64 * 11008), so fp32 sums
    in any order are exact; a pair's SwiGLU is then the tiled GEMM's to the bit."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(m + k + n)
    num = lambda rows: torch.randint(-8, 9, (rows, k), generator=g).float()
    scale = lambda rows: 2.0 ** torch.randint(-9, -6, (rows,), generator=g).float()
    xf, wf, uf, sxf, swf, suf = num(m), num(n), num(n), scale(m), scale(n), scale(n)
    x, w, u = _codes(m, k, xf), _codes(n, k, wf), _codes(n, k, uf)
    sx, sw, su = sxf.cuda(), swf.cuda(), suf.cuda()
    want = (xf.double() @ wf.double().t()) * sxf.double()[:, None] * swf.double()[None, :]
    try:
        worker.set_option("gemm_narrow", -1)
        tiled = {d: _run(lib, x, sx, w, sw, u, su, m, k, n, d) for d in (torch.bfloat16, torch.float16)}
        for tile in (1, 2, 3):
            worker.set_option("gemm_narrow", tile)
            for d in (torch.float32, torch.bfloat16, torch.float16):
                got = _run(lib, x, sx, w, sw, None, None, m, k, n, d)
                assert torch.equal(got.cpu(), want.float().to(d)), (tile, d)
            for d in tiled:
                assert torch.equal(_run(lib, x, sx, w, sw, u, su, m, k, n, d), tiled[d]), (tile, d)
    finally:
        worker.set_option("gemm_narrow", 0)


@pytest.mark.parametrize("m,k,n", [(24, 2816, 96), (130, 4096, 256)])
def test_error_is_no_larger_than_the_tiled_form(worker, m, k, n):
    """Against 64 bits, in norm; 1.1: two orders of the same fp32 sums."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(3)
    xf, wf = torch.randn((m, k), generator=g).to(F8).float(), torch.randn((n, k), generator=g).to(F8).float()
    x, w = _codes(m, k, xf), _codes(n, k, wf)
    sx, sw = torch.rand(m, generator=g) * 0.05 + 0.01, torch.rand(n, generator=g) * 0.02 + 0.01
    want = (xf.double() @ wf.double().t()) * sx.double()[:, None] * sw.double()[None, :]
    err = {}
    try:
        for tile in (-1, 1, 2, 3):
            worker.set_option("gemm_narrow", tile)
            got = _run(lib, x, sx.cuda(), w, sw.cuda(), None, None, m, k, n, torch.float32)
            err[tile] = ((got.cpu().double() - want).norm() / want.norm()).item()
    finally:
        worker.set_option("gemm_narrow", 0)
    assert max(err[1], err[2], err[3]) <= 1.1 * err[-1], err


@pytest.mark.parametrize("m,k,n,dual", [(1, 512, 256, False), (17, 512, 256, False), (32, 4096, 256, False), (8, 4096, 2048, False),
                                        (17, 256, 128, True), (8, 2048, 512, True)])
def test_a_result_laid_over_its_codes(worker, m, k, n, dual):
    """A product whose tiled form has one tile of channels, or k splits that are summed behind it, may write its result over its codes; the
    small-call form would write them while other workgroups still read.  Such a call has the tiled form's bits."""
    lib = _lib.load()
    g = torch.Generator().manual_seed(m + n)
    codes = lambda rows: _codes(rows, k, torch.randn((rows, k), generator=g))
    x, w, u = codes(m), codes(n), codes(n) if dual else None
    sx, sw, su = (torch.rand(rows, generator=g).cuda() * 0.05 + 0.01 for rows in (m, n, n))
    program = lib.pto_hip_gate_up_swiglu_fp8 if dual else lib.pto_hip_projection_fp8
    weights = (w.data_ptr(), sw.data_ptr()) + ((u.data_ptr(), su.data_ptr()) if dual else ())
    try:
        worker.set_option("gemm_narrow", -1)
        want = _run(lib, x, sx, w, sw, u, su, m, k, n, torch.bfloat16)
    finally:
        worker.set_option("gemm_narrow", 0)
    for _ in range(8):
        buf = x.clone().flatten()
        _lib.check(program(buf.data_ptr(), sx.data_ptr(), *weights, buf.data_ptr(), m, k, n, _dtype_code(torch.bfloat16), 0))
        torch.cuda.synchronize()
        assert torch.equal(buf[:m * n * 2].view(torch.bfloat16).view(m, n), want)
