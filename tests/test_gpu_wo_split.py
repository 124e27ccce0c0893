"""The INT8 split kernel for decode batches at the edges of its tiles, its K split and its
dispatch range."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"

# M around one to four 16-row tiles and several of them; N from one 16-row tile to the widths whose
# plans take two to five tiles per workgroup, with part workgroups; K of one k-step (three of
# four wavefronts have none), of unequal shares, of more steps than are in flight, and from 32
# steps up (eight wavefronts)
SIZES = [(1, 16, 128), (5, 48, 128), (16, 1024, 256), (17, 8208, 128), (24, 10000, 256), (33, 12288, 256),
         (48, 19456, 128), (64, 19440, 256), (64, 16384, 128), (49, 6144, 640), (64, 2560, 4096), (16, 2560, 4224),
         (40, 1040, 9728), (65, 272, 1152), (100, 4096, 640), (200, 1024, 1024), (256, 48, 2560)]


def _data(M, N, K, sdt, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    x = torch.randn(M, K + 8, generator=g, device=DEV).bfloat16()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) * 0.01 + 1e-4).to(sdt)
    return x, q, s


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float16, torch.float32])
def test_w8a16_split(M, N, K, sdt, miq_env):
    """Against 64 bits: K * 2^-24 of the sum of |products| for any order of fp32 additions, and
    the two bf16 roundings of bf16(bf16(acc) * bf16(s)), 2^-8 of the value each. Activations with
    a row stride past K, output rows at strides that take and that rule out 8-byte stores; the
    padding stays untouched and a second call gives the same bytes."""
    from kernels import _lib as L
    miq_env("MIQ_WO_SPLIT", "1")
    print(f"[case] w8a16 split M={M} N={N} K={K} {sdt}", flush=True)
    x, q, s = _data(M, N, K, sdt, M + N + K)
    ws = L.wo_workspace(x.device, L.load().miq_wo_gemm_workspace_bytes(M, N, K, 8))
    x64, q64, s64 = x[:, :K].double(), q.double(), s.bfloat16().double()
    want, mag = (x64 @ q64.t()) * s64, (x64.abs() @ q64.abs().t()) * s64
    bound = (2.0 ** -7 + 2.0 ** -15) * want.abs() + K * 2.0 ** -24 * mag + 1e-30
    for pad in (0, 4, 3):
        ys = []
        for _ in range(2):
            y = torch.full((M, N + pad), 7.0, dtype=torch.bfloat16, device=DEV)
            L.call("miq_w8a16_gemm", L.ptr(x), x.stride(0), L.ptr(q), L.ptr(s), L.dtype_code(sdt), L.ptr(y), N + pad,
                   M, N, K, L.ptr(ws), ws.numel(), L.stream(x.device))
            ys.append(y)
        assert ((ys[0][:, :N].double() - want).abs() <= bound).all()
        assert (ys[0][:, N:] == 7.0).all() and torch.equal(*ys)


@pytest.mark.parametrize("M,N,K,split", [(64, 2560, 4096, True), (8, 6144, 2560, True), (8, 19456, 2560, False),
                                         (4, 6144, 2560, False), (128, 1024, 1024, True), (128, 19456, 2560, False),
                                         # one, two and three tiles per CU; a vocabulary's projection
                                         (64, 20480, 512, True), (64, 24576, 512, True), (48, 32768, 1024, True),
                                         (64, 40960, 512, False), (64, 40960, 4096, True), (17, 49152, 512, False),
                                         (32, 50304, 2048, False),
                                         # a deep K on narrow tiles; five to seven rows; past 64 rows
                                         (40, 6144, 14336, False), (17, 8192, 4096, True), (16, 2560, 12288, False),
                                         (12, 2560, 9728, True), (5, 6144, 1024, False), (6, 6144, 1024, True),
                                         (96, 12288, 512, False), (96, 12288, 2560, True)])
def test_w8a16_split_is_the_planned_kernel(M, N, K, split, miq_env):
    """Both sides of the dispatch's lines: the call gives the bytes of the kernel the rule names."""
    from kernels import quant_ops as ops
    print(f"[case] w8a16 split plan M={M} N={N} K={K}", flush=True)
    x, q, s = _data(M, N, K, torch.bfloat16, 5)
    x = x[:, :K].contiguous()
    y = ops.w8a16_linear(x, q, s)
    miq_env("MIQ_WO_SPLIT", "1" if split else "0")
    assert torch.equal(ops.w8a16_linear(x, q, s), y)
