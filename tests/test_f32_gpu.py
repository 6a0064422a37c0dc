"""fp32 products at the edges of their tiles: few rows (K shared by the waves), tiles with remainders, every count of K steps, grouped rows."""
import ctypes as C

import pytest
import torch

from moondream_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 16, 17, 33, 64, 65, 130])
@pytest.mark.parametrize("n,k", [(64, 64), (192, 128), (320, 192), (64, 1472)])
@pytest.mark.parametrize("bias", [False, True])
def test_product(m, n, k, bias):
    lib = _lib.load()
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a, w, b = (torch.randn(*s, generator=g, device="cuda") for s in ((m, k + 8), (n, k), (n,)))
    for ldc in (n, n + 3):  # rows that 16-byte stores can and cannot take
        c = torch.full((m, ldc), 7.0, device="cuda")
        lin = _lib.MdLinear()
        lin.w, lin.b, lin.n, lin.k, lin.n_pad, lin.k_pad = w.data_ptr(), b.data_ptr() if bias else None, n, k, n, k
        _lib.check(lib.md_gemm_f32(a.data_ptr(), k + 8, C.byref(lin), c.data_ptr(), ldc, m, torch.cuda.current_stream().cuda_stream), "md_gemm_f32")
        want = a[:, :k].double() @ w.double().t() + (b.double() if bias else 0)
        # k products of rounding error 2^-24 each, added in fp32
        bound = (a[:, :k].abs().double() @ w.abs().double().t() + b.abs().double()) * (k + 1) * 2.0 ** -24
        assert bool(((c[:, :n].double() - want).abs() <= bound).all()) and bool((c[:, n:] == 7).all())
