"""The merge of the partitions of paged decode attention, at the partition counts where its
loops end: none, one, the most that one thread per column holds (4, 8 and 16) and one more, a
workgroup's rows in flight (64) and one more, and past the 512 partitions whose weights are
formed at once.

Each head puts about half of its probability on one token of one partition, so a partition that
is left out, added twice or given another's weight moves that head's output by about half a
value; the bound is that of the rounding: probabilities and the result are rounded to bf16
(unit roundoff 2^-8 each), so |err| <= 2^-7 sum p |v| plus the fp32 accumulation."""
import pytest
import torch

from oracle import attention as A

pytestmark = pytest.mark.gpu
DEV = "cuda"
H, D, PAGE, PART = 8, 128, 16, 128


@pytest.mark.parametrize("lens", [[0, 3, 128], [0, 1, 129, 385, 512], [0, 129, 513], [1, 500, 1024], [0, 1025, 300],
                                  [0, 1, 127, 128, 129, 2047, 2048], [0, 5, 128 * 16 + 1, 128 * 64, 128 * 64 + 1],
                                  [128 * 16 + 1, 0], [128 * 511 + 3, 130], [128 * 519 + 3, 0],
                                  [0, 2049, 128 * 33] + [129] * 125])
@pytest.mark.parametrize("unaligned", [False, True])
def test_merge_adds_every_partition_once(lens, unaligned):
    from kernels import _lib as L
    print(f"[case] merge {lens} unaligned={unaligned}", flush=True)
    g = torch.Generator().manual_seed(len(lens))
    B, pages = len(lens), [-(-n // PAGE) for n in lens]
    total = sum(pages) + 1
    k = torch.zeros(total * PAGE, H, D, dtype=torch.bfloat16)
    v = torch.randn(total * PAGE, H, D, generator=g).bfloat16()
    table = torch.zeros(B, max(max(pages), 1), dtype=torch.int32)
    first = 0
    for b, n in enumerate(lens):
        table[b, :pages[b]] = torch.arange(first, first + pages[b])
        parts = -(-n // PART)
        for h, part in enumerate([0, 1, 15, 16, 63, 64, parts // 2, parts - 1]):
            if n:  # (logit log n: as much weight as all other tokens of the context together)
                at = min(min(part, parts - 1) * PART + 7 * h, n - 1)
                k[first * PAGE + at, h] = torch.log(torch.tensor(float(n))) / D ** 0.5
        first += pages[b]
    q = torch.ones(B, H, D, dtype=torch.bfloat16)
    sl = torch.tensor(lens, dtype=torch.int32)
    live = [b for b, n in enumerate(lens) if n]
    want = A.paged_decode_reference(q[live], k, v, table[live], sl[live], PAGE, D ** -0.5).float()
    mag = A.paged_decode_reference(q[live], k, v.abs(), table[live], sl[live], PAGE, D ** -0.5).float()

    parts = -(-max(lens) // PART)
    qd, kd, vd, td, sd = (x.to(DEV) for x in (q, k, v, table, sl))
    o = torch.full((B * H * parts * D + 1,), float("nan"), device=DEV)[int(unaligned):]  # (one float further on)
    lse = torch.full((B * H * parts,), float("nan"), device=DEV)
    got = torch.empty(B, H, D, dtype=torch.bfloat16, device=DEV)
    L.call("miq_paged_decode", L.ptr(qd), H * D, D, L.ptr(kd), L.ptr(vd), L.dtype_code(kd.dtype), H * D, D,
           None, None, L.MIQ_F32, 0, 0, L.ptr(td), td.stride(0), L.ptr(sd), B, H, H, D, PAGE, D ** -0.5, PART, parts,
           L.ptr(o), L.ptr(lse), L.ptr(got), H * D, D, L.stream(qd.device))
    got = got.cpu().float()
    assert torch.isfinite(got).all()
    for b, n in enumerate(lens):
        if n == 0:
            assert torch.count_nonzero(got[b]) == 0
    err = (got[live] - want).abs()
    assert (err <= 2.0 ** -7 * mag + 1e-5).all(), (err - 2.0 ** -7 * mag).max().item()
