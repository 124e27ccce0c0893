"""The FP8 GEMMs at the edges of their tiles, of the split kernel's K split and of the dispatch."""
import pytest
import torch

from oracle import quant as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


# (M, N, K): M around 16, 32 and 64 rows; N with a part tile (and not a multiple of 4 or 16);
# one k-step, fewer k-steps than wavefronts and splits of unequal length, all on the split kernel;
# one part tile of activation rows or of weight rows on the large tiles; sizes of large tiles that
# run on 128 x 128 or on the previous 256 x 192 tiles where y's rows rule the large ones out
SIZES = [(1, 16, 128), (1, 6144, 2560), (2, 20, 256), (15, 48, 384), (16, 2560, 9728), (17, 33, 640), (32, 80, 1152),
         (33, 6144, 2560), (49, 130, 256), (64, 1008, 1024), (65, 2560, 4096), (129, 200, 896), (255, 19456, 256),
         (257, 19456, 256), (300, 1024, 1024), (512, 6144, 640), (1023, 192, 384), (1024, 192, 384), (1025, 208, 384),
         (65, 19456, 256), (129, 17280, 384), (200, 19456, 256), (239, 19456, 256), (20000, 128, 2560),
         (257, 16501, 640), (400, 14500, 512), (513, 11000, 512), (1300, 4800, 512)]


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("pad", [0, 6])
def test_fp8_gemm_tiles_and_splits(M, N, K, pad):
    """fp32 products of exact e4m3 values in another order, then one rounding to bf16: within
    half a bf16 ulp (8 significant bits: at most 2^-8 of the value) plus K * 2^-24 of the sum of |products|, which bounds
    any order of fp32 additions. Output rows at a stride past N (pad, not a multiple of 4)
    leave the padding alone."""
    from kernels import _lib as L
    print(f"[case] fp8 split M={M} N={N} K={K} pad={pad}", flush=True)
    g = torch.Generator().manual_seed(M * 31 + N + K)
    xq, xs = O.fp8_quantize_activation(torch.randn(M, K, generator=g).to(torch.bfloat16))
    w = O.fp8_quantize((torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16))
    xd, wd = xq.to(DEV), w["qweight"].to(DEV)
    xsd, wsd = xs.reshape(-1).to(DEV), w["scale"].to(DEV)
    y = torch.full((M, N + pad), 7.0, dtype=torch.bfloat16, device=DEV)
    L.call("miq_fp8_gemm", L.ptr(xd), L.ptr(xsd), L.ptr(wd), L.ptr(wsd), L.ptr(y), N + pad, M, N, K, L.stream(y.device))
    x64, w64 = xd.double(), wd.double()
    s = xsd.double()[:, None] * wsd.double()[None, :]
    want, mag = (x64 @ w64.t()) * s, (x64.abs() @ w64.abs().t()) * s
    bound = (2.0 ** -8 + 2.0 ** -22) * want.abs() + K * 2.0 ** -24 * mag + 1e-30
    assert ((y[:, :N].double() - want).abs() <= bound).all()
    assert (y[:, N:] == 7.0).all()


def test_fp8_gemm_repeats_bit_for_bit():
    """The wavefronts' partial sums are added in a fixed order."""
    from kernels import quant_ops as ops
    print("[case] fp8 split repeat", flush=True)
    g = torch.Generator().manual_seed(5)
    xq, xs = O.fp8_quantize_activation(torch.randn(40, 2560, generator=g).to(torch.bfloat16))
    w = O.fp8_quantize((torch.randn(6144, 2560, generator=g) * 0.02).to(torch.bfloat16))
    args = [t.to(DEV) for t in (xq, xs, w["qweight"], w["scale"])]
    first = ops.fp8_gemm(*args)
    for _ in range(3):
        assert torch.equal(ops.fp8_gemm(*args), first)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("shape,N,K", [((1,), 64, 128), ((3, 7), 96, 640), ((2, 600), 192, 256)])
def test_fp8_linear_in_one_call_equals_two(shape, N, K, dtype):
    """miq_fp8_linear = miq_fp8_quantize_rows + miq_fp8_gemm, byte for byte, for contiguous,
    row-strided and misaligned (last-dim offset) activations."""
    from engine.quantization import get_method
    from kernels import quant_ops as ops
    print(f"[case] fp8 linear {shape} N={N} K={K} {dtype}", flush=True)
    g = torch.Generator().manual_seed(K + N)
    w = {k: v.to(DEV) for k, v in O.fp8_quantize((torch.randn(N, K, generator=g) * 0.02).to(torch.bfloat16)).items()}
    m = get_method("fp8", device=DEV)
    wide = torch.randn(*shape, K + 9, generator=g).to(dtype).to(DEV)
    for x in (wide[..., :K].contiguous(), wide[..., :K], wide[..., 3:3 + K]):
        q, s = ops.fp8_quantize_rows(x.reshape(-1, K))
        want = ops.fp8_gemm(q, s, w["qweight"], w["scale"]).to(dtype).reshape(*shape, N)
        got = m.linear(x, **w)
        assert got.dtype == dtype and got.shape == want.shape and torch.equal(got, want)
