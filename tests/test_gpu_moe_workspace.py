"""How much scratch memory the fused MoE layers ask for."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("kind", ["int4", "int8", "fp8"])
def test_only_int8_layers_ask_for_the_block_layout(kind, miq_env, monkeypatch):
    from engine.quantization import get_method
    from kernels import _lib as L
    from kernels.fused_moe import fused_moe_fp8, fused_moe_int4, fused_moe_int8
    print(f"[case] moe workspace {kind}", flush=True)
    miq_env("MIQ_MOE_BLOCK", "1")
    E, H, I, T, k = 8, 256, 128, 300, 2
    g = torch.Generator().manual_seed(61)
    m = get_method({"int4": "int4_wo", "int8": "int8_wo", "fp8": "fp8"}[kind], device=DEV, group_size=128)
    gu = m.quantize((torch.randn(E, 2 * I, H, generator=g) * 0.02).bfloat16().to(DEV))
    dn = m.quantize((torch.randn(E, H, I, generator=g) * 0.02).bfloat16().to(DEV))
    hidden = torch.randn(T, H, generator=g).bfloat16().to(DEV)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)]).to(DEV)
    w = torch.rand(T, k, generator=g).bfloat16().to(DEV)
    sizes, call = [], L.call

    def spy(name, *args):
        if "moe" in name:
            sizes.append(args[-3])  # (.., workspace, workspace_bytes, out, stream)
        return call(name, *args)

    monkeypatch.setattr(L, "call", spy)
    args = (gu["qweight"], gu["scale"], dn["qweight"], dn["scale"])
    if kind == "int4":
        fused_moe_int4(hidden, idx, w, args[0], args[1], gu["zero"], args[2], args[3], dn["zero"])
    else:
        (fused_moe_int8 if kind == "int8" else fused_moe_fp8)(hidden, idx, w, *args)
    least, block = (f(T, k, E, H, I) for f in (L.load().miq_moe_min_workspace_bytes, L.load().miq_moe_workspace_bytes))
    assert least < block and sizes == [block if kind == "int8" else least]
