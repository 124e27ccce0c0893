"""Layouts of the fused MoE kernels at the sizes where they change, vs the CPU oracle."""
import pytest
import torch

from oracle import moe as MO
from oracle import quant as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _routed(T, H, E, k, seed):
    g = torch.Generator().manual_seed(seed)
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16)
    router = (torch.randn(E, H, generator=g) * 0.02).to(torch.bfloat16)
    w, idx = torch.topk(torch.softmax(hidden.float() @ router.float().t(), dim=-1), k, dim=-1)
    return hidden, w.to(torch.bfloat16), idx


@pytest.mark.parametrize("T,H,I,E,k", [(20, 1536, 512, 4, 2), (17, 512, 1536, 5, 2), (16, 2048, 2048, 3, 1),
                                       (400, 1536, 512, 4, 2), (300, 512, 1536, 5, 2), (200, 2048, 2048, 3, 1)])
@pytest.mark.parametrize("sym", [False, True])
def test_int4_scales_from_registers(T, H, I, E, k, sym):
    """Rows of 4, 12 and 16 groups in four-wavefront workgroups (few tokens, with zero points) and
    in eight-wavefront ones: every group's scale (and
    zero) word comes from the lane that loaded it. The groups' scales differ by powers of
    two, so a word taken from a wrong lane or slot moves the output far past the bound,
    which is the fused INT4 layer's (fp32 sums in another order, bf16 roundings alike)."""
    from kernels.fused_moe import fused_moe_int4
    print(f"[case] int4 moe register scales T={T} H={H} I={I} E={E} k={k} sym={sym}", flush=True)
    g = torch.Generator().manual_seed(17)
    steps = lambda K: (2.0 ** -(torch.arange(K) // 128 % 5).float())  # noqa: E731
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.04 * steps(H)).to(torch.bfloat16)
    wdn = (torch.randn(E, H, I, generator=g) * 0.04 * steps(I)).to(torch.bfloat16)
    qf = O.int4_quantize_symmetric if sym else O.int4_quantize
    gu, dn = qf(wgu, 128), qf(wdn, 128)
    hidden, w, idx = _routed(T, H, E, k, seed=18)
    want = MO.int4_experts_reference(hidden, gu, dn, w, idx)
    got = fused_moe_int4(hidden.to(DEV), idx.to(DEV), w.to(DEV), gu["qweight"].to(DEV), gu["scale"].to(DEV),
                         None if sym else gu["zero"].to(DEV), dn["qweight"].to(DEV), dn["scale"].to(DEV),
                         None if sym else dn["zero"].to(DEV)).float().cpu()
    assert ((got - want).norm() / want.norm()).item() < 2e-2
    assert ((got - want).abs() <= 1e-2 + 2e-2 * want.abs()).all()


@pytest.mark.parametrize("k", [1, 2, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("H", [128, 2048, 2176])
def test_combine_order_of_many_tokens(k, H):
    """The combine of large batches adds a token's slots in the same order as that of small
    ones (bf16 after every addition, so another order gives other bytes): a call of 256 or 300
    tokens equals calls of at most 100, with slots out of range for some tokens."""
    from kernels.fused_moe import fused_moe_int4
    print(f"[case] combine order k={k} H={H}", flush=True)
    E, I = 20, 128
    g = torch.Generator().manual_seed(23)
    gu = O.int4_quantize_symmetric((torch.randn(E, 2 * I, H, generator=g) * 0.05).bfloat16(), 128)
    dn = O.int4_quantize_symmetric((torch.randn(E, H, I, generator=g) * 0.05).bfloat16(), 128)
    gq, gs, dq, ds = (x.to(DEV) for x in (gu["qweight"], gu["scale"], dn["qweight"], dn["scale"]))
    hidden = torch.randn(300, H, generator=g).bfloat16().to(DEV)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(300)])
    idx[::7, 0] = E
    idx, w = idx.to(DEV), torch.rand(300, k, generator=g).bfloat16().to(DEV)
    call = lambda a, b: fused_moe_int4(hidden[a:b], idx[a:b], w[a:b], gq, gs, None, dq, ds, None)  # noqa: E731
    want = torch.cat([call(a, a + 100) for a in (0, 100, 200)])
    assert torch.equal(call(0, 300), want)
    assert torch.equal(call(0, 256), want[:256])
