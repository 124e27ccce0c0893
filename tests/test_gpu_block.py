"""The INT8 block GEMMs (long prefill linears and expert GEMMs over many tokens) at the edges of
their tiles and of their dispatch range."""
import pytest
import torch

from oracle import moe as MO
from oracle import quant as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


# M of one row and of one 32-row fragment and one more (with the prefill kernels' own limit of 65 rows
# lowered), below, at and past one half block (128 rows), one block (256) and two; N with part blocks of
# 256 and part wavefronts of 64; K of two, four and ten stages; 130 blocks (a last round that is
# not halved would need more than 256) and 260 (one full round and four halved blocks)
LINEAR = [(1, 16, 128), (33, 272, 640), (65, 48, 128), (128, 256, 256), (129, 272, 640), (255, 512, 128), (256, 64, 256),
          (257, 528, 128), (600, 1040, 640), (300, 16640, 128), (1030, 13312, 128)]


@pytest.mark.parametrize("M,N,K", LINEAR)
@pytest.mark.parametrize("sdt", [torch.bfloat16, torch.float16, torch.float32])
def test_w8a16_block(M, N, K, sdt, miq_env):
    """Against 64 bits: K * 2^-24 of the sum of |products| for any order of fp32 additions, and
    the two bf16 roundings of bf16(bf16(acc) * bf16(s)), 2^-8 of the value each (the scale's own
    rounding to bf16 is part of the formula). Activations with a row stride past K, output rows
    at strides that take and that rule out 16-byte stores; the padding stays untouched."""
    from kernels import _lib as L
    miq_env("MIQ_WO_BLOCK", "1")
    miq_env("MIQ_WO_PREFILL_MIN_M", "1")
    print(f"[case] w8a16 block M={M} N={N} K={K} {sdt}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(M + N + K)
    x = torch.randn(M, K + 8, generator=g, device=DEV).bfloat16()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) * 0.01 + 1e-4).to(sdt)
    ws = L.wo_workspace(x.device, L.load().miq_wo_gemm_workspace_bytes(M, N, K, 8))
    x64, q64, s64 = x[:, :K].double(), q.double(), s.bfloat16().double()
    want, mag = (x64 @ q64.t()) * s64, (x64.abs() @ q64.abs().t()) * s64
    bound = (2.0 ** -7 + 2.0 ** -15) * want.abs() + K * 2.0 ** -24 * mag + 1e-30
    for pad in (0, 8, 3):
        y = torch.full((M, N + pad), 7.0, dtype=torch.bfloat16, device=DEV)
        L.call("miq_w8a16_gemm", L.ptr(x), x.stride(0), L.ptr(q), L.ptr(s), L.dtype_code(sdt), L.ptr(y), N + pad,
               M, N, K, L.ptr(ws), ws.numel(), L.stream(x.device))
        assert ((y[:, :N].double() - want).abs() <= bound).all()
        assert (y[:, N:] == 7.0).all()


@pytest.mark.parametrize("M,N,K,block", [(2048, 19456, 2560, True), (1000, 6144, 2560, True), (200, 2560, 9728, False),
                                         (450, 6144, 4096, False), (512, 6144, 2560, True)])
def test_w8a16_block_is_the_planned_kernel(M, N, K, block, miq_env):
    """The dispatch rule on both sides of its line: the call gives the bytes of the kernel that
    the rule names."""
    from kernels import quant_ops as ops
    print(f"[case] w8a16 block plan M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device=DEV).manual_seed(1)
    x = torch.randn(M, K, generator=g, device=DEV).bfloat16()
    q = torch.randint(-127, 128, (N, K), generator=g, device=DEV, dtype=torch.int8)
    s = (torch.rand(N, generator=g, device=DEV) * 0.01).bfloat16()
    y = ops.w8a16_linear(x, q, s)
    miq_env("MIQ_WO_BLOCK", "1" if block else "0")
    assert torch.equal(ops.w8a16_linear(x, q, s), y)


def _layer(E, H, I, seed):
    g = torch.Generator().manual_seed(seed)
    wgu = (torch.randn(E, 2 * I, H, generator=g) * 0.02).to(torch.bfloat16)
    wdn = (torch.randn(E, H, I, generator=g) * 0.02).to(torch.bfloat16)
    return O.int8_quantize(wgu), O.int8_quantize(wdn), g


def _run(hidden, idx, w, gu, dn):
    from kernels.fused_moe import fused_moe_int8
    return fused_moe_int8(hidden.to(DEV), idx.to(DEV), w.to(DEV), gu["qweight"].to(DEV), gu["scale"].to(DEV),
                          dn["qweight"].to(DEV), dn["scale"].to(DEV)).float().cpu()


# rows per expert from none to several tiles of 160: counts[e] tokens take expert e in slot 0
COUNTS = [[1, 0, 32, 33], [31, 160, 161, 0], [0, 0, 0, 1], [330, 64, 65, 96], [128, 129, 5, 320]]


@pytest.mark.parametrize("counts", COUNTS)
@pytest.mark.parametrize("H,I", [(128, 128), (640, 384), (1024, 256)])
@pytest.mark.parametrize("wdtype,ids", [(torch.bfloat16, torch.int64), (torch.float32, torch.int32)])
def test_int8_moe_block(counts, H, I, wdtype, ids, miq_env):
    """The block expert GEMMs against the reference loop (modules.py:55-75) with the reference's
    own int8 linear: the same bf16 roundings, fp32 sums in another order, so the bound is the
    streaming kernels'. Experts without pairs, of one row, of whole and part row tiles and of
    several tiles; a second slot that is out of range for some tokens; part column blocks."""
    miq_env("MIQ_MOE_BLOCK", "1")
    print(f"[case] int8 moe block counts={counts} H={H} I={I} {wdtype} {ids}", flush=True)
    E, T = len(counts), sum(counts)
    gu, dn, g = _layer(E, H, I, seed=41)
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16)
    first = torch.repeat_interleave(torch.arange(E), torch.tensor(counts))[torch.randperm(T, generator=g)]
    second = (first + 1 + torch.randint(0, E - 1, (T,), generator=g)) % E
    second[::5] = E
    idx = torch.stack((second, first), dim=1).to(ids)
    w = torch.rand(T, 2, generator=g).to(wdtype)
    loop = MO.quant_experts_loop(hidden, O.int8_linear, gu, dn, idx.long(), w, E).float()
    got = _run(hidden, idx, w, gu, dn)
    assert ((got - loop).norm() / loop.norm()).item() < 1e-2
    assert ((got - loop).abs() <= 1e-2 + 2e-2 * loop.abs()).all()


@pytest.mark.parametrize("T,E,k,H,I,planned", [(65, 8, 2, 256, 128, False), (700, 40, 3, 256, 128, False),
                                               (1100, 8, 8, 256, 128, False), (40, 300, 4, 256, 128, False),
                                               (1500, 300, 4, 256, 128, True), (600, 16, 8, 1024, 512, True)])
def test_int8_moe_block_equals_streaming(T, E, k, H, I, planned, miq_env):
    """More experts than a wavefront or than threads per segment, more than 128 chunks of pairs
    (T = 1100, k = 8), and the dispatch rule's default on both sides of its line: block and
    streaming kernels place the same pairs, so tokens agree to the layer's bound, and repeated
    calls to the byte."""
    print(f"[case] int8 moe block vs streaming T={T} E={E} k={k} H={H} I={I}", flush=True)
    gu, dn, g = _layer(E, H, I, seed=43)
    hidden = torch.randn(T, H, generator=g).to(torch.bfloat16)
    idx = torch.stack([torch.randperm(E, generator=g)[:k] for _ in range(T)])
    w = torch.rand(T, k, generator=g).to(torch.bfloat16)
    default = _run(hidden, idx, w, gu, dn)
    miq_env("MIQ_MOE_BLOCK", "0")
    stream = _run(hidden, idx, w, gu, dn)
    miq_env("MIQ_MOE_BLOCK", "1")
    block = _run(hidden, idx, w, gu, dn)
    assert torch.equal(block, _run(hidden, idx, w, gu, dn))
    assert torch.equal(default, block if planned else stream) and not torch.equal(block, stream)
    assert ((block - stream).abs() <= 1e-2 + 2e-2 * stream.abs()).all()
