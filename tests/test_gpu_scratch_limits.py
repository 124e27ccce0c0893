"""Kernels that need less or more scratch than others for the same call: the size that a call may
bring stays what the older kernels need, and a call that brings just that runs on those."""
import pytest
import torch

from oracle import quant as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("routed", [True, False])
def test_int8_moe_takes_the_streaming_kernels_scratch(routed, miq_env):
    from kernels import _lib as L
    from kernels.fused_moe import fused_moe_int8, moe_align
    print(f"[case] int8 moe small workspace routed={routed}", flush=True)
    E, H, I, T, k = 8, 256, 128, 200, 2
    g = torch.Generator().manual_seed(51)
    gu = O.int8_quantize((torch.randn(E, 2 * I, H, generator=g) * 0.02).bfloat16())
    dn = O.int8_quantize((torch.randn(E, H, I, generator=g) * 0.02).bfloat16())
    gq, gs, dq, ds = (x.to(DEV) for x in (gu["qweight"], gu["scale"], dn["qweight"], dn["scale"]))
    hidden = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(DEV)
    w = torch.rand(T, k, generator=g).bfloat16().to(DEV)
    miq_env("MIQ_MOE_BLOCK", "1")
    full = L.load().miq_moe_workspace_bytes(T, k, E, H, I)
    miq_env("MIQ_MOE_BLOCK", "0")
    small = L.load().miq_moe_workspace_bytes(T, k, E, H, I)
    want = fused_moe_int8(hidden, idx, w, gq, gs, dq, ds)
    miq_env("MIQ_MOE_BLOCK", "1")
    assert small < full
    ws = torch.empty(small, dtype=torch.uint8, device=DEV)
    got = torch.empty_like(want)
    args = (L.ptr(hidden), T, H, I, E, k, L.ptr(gq), L.ptr(gs), L.ptr(dq), L.ptr(ds), L.dtype_code(gs.dtype),
            L.ptr(w), L.dtype_code(w.dtype))
    tail = (L.ptr(ws), small, L.ptr(got), L.stream(hidden.device))
    if routed:
        L.call("miq_w8a16_moe_routed", *args, L.ptr(idx), L.dtype_code(idx.dtype), *tail)
    else:
        L.call("miq_w8a16_moe", *args, *(L.ptr(t) for t in moe_align(idx, E, 16)), *tail)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,N,K", [(64, 6144, 2560), (17, 2560, 4096)])
def test_int8_gemm_without_workspace_is_still_refused(M, N, K):
    from kernels import _lib as L
    print(f"[case] w8a16 without a workspace M={M} N={N} K={K}", flush=True)
    x = torch.zeros(M, K, dtype=torch.bfloat16, device=DEV)
    q, s = torch.zeros(N, K, dtype=torch.int8, device=DEV), torch.ones(N, device=DEV)
    y = torch.empty(M, N, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(RuntimeError, match="workspace"):
        L.call("miq_w8a16_gemm", L.ptr(x), K, L.ptr(q), L.ptr(s), L.MIQ_F32, L.ptr(y), N, M, N, K, None, 0,
               L.stream(x.device))
