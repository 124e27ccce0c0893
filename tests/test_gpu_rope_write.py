"""KVCache.write_rotated: the one-launch kernel against the formula and KVCache.write."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("kind", ["fp8", "int8"])
@pytest.mark.parametrize("model_dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("T,heads,kv", [(1, 32, 8), (5, 3, 1), (257, 16, 16), (2, 7, 2)])
@pytest.mark.parametrize("strided", [False, True])
def test_rope_kv_write_is_bit_exact(kind, model_dtype, T, heads, kv, strided):
    """Rotated queries, codes and scales equal the torch formula's followed by the two KV writes,
    bit for bit (bf16 and fp32 cache scales); q, k and v as slices of one projection too; rows
    of zeros and of one huge value, and an infinity in a query, a key and a value head (whose
    scale is infinite and whose codes are those of x / inf and, at the infinity, of NaN)."""
    from engine.core.kv_cache import KVCache, rotate_half
    print(f"[case] rope kv write {kind} {model_dtype} T={T} heads={heads} kv={kv} strided={strided}", flush=True)
    g = torch.Generator().manual_seed(T * 100 + heads)
    D = 128
    qkv = torch.randn(T, heads + 2 * kv, D, generator=g).bfloat16().to(DEV)
    qkv[0, heads] = 0
    qkv[-1, -1, 5] = 3e38
    qkv[-1, 0, 7] = float("inf")
    qkv[T // 2, heads, 3] = float("-inf")
    qkv[T // 2, heads + kv, 9] = float("inf")
    q, k, v = qkv.split([heads, kv, kv], dim=1)
    if not strided:
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    ang = torch.randn(T, 1, D, generator=g) * 3
    cos, sin = ang.cos().bfloat16().to(DEV), ang.sin().bfloat16().to(DEV)
    slots = torch.randperm(T + 40, generator=g)[:T].to(DEV)
    got, want = (KVCache("paged", 2, kv, D, (T + 56) // 16 * 16, model_dtype, DEV, block_size=16, kv_dtype=kind)
                 for _ in range(2))
    out = got.write_rotated(1, slots, q, k, v, cos, sin)
    ref = q * cos + rotate_half(q) * sin
    want.write(1, slots, k * cos + rotate_half(k) * sin, v)
    bits = lambda t: t.contiguous().view(torch.int16)  # noqa: E731
    assert out.shape == ref.shape and torch.equal(out.isnan(), ref.isnan())
    assert torch.equal(bits(out)[~ref.isnan()], bits(ref)[~ref.isnan()])
    for a, b in ((got.k, want.k), (got.v, want.v)):
        assert torch.equal(a.view(torch.uint8), b.view(torch.uint8))
    assert torch.equal(got.k_scale, want.k_scale) and torch.equal(got.v_scale, want.v_scale)


def test_a_replaced_write_is_called():
    """A write() of a subclass or set on the cache object gets k rotated and v."""
    from engine.core.kv_cache import KVCache, rotate_half
    print("[case] rope kv write, replaced write", flush=True)
    calls = []

    class Own(KVCache):
        def write(self, layer, slots, k, v):
            calls.append((k, v))

    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(3, n, 128, generator=g).bfloat16().to(DEV) for n in (4, 2, 2))
    ang = torch.randn(3, 1, 128, generator=g)
    cos, sin = ang.cos().bfloat16().to(DEV), ang.sin().bfloat16().to(DEV)
    slots = torch.tensor([4, 0, 9], device=DEV)
    args = ("paged", 1, 2, 128, 16, torch.bfloat16, DEV, 16, 0.01, "fp8")
    spied = KVCache(*args)
    spied.write = lambda layer, slots, k, v: calls.append((k, v))
    for cache in (Own(*args), spied):
        out = cache.write_rotated(0, slots, q, k, v, cos, sin)
        assert torch.equal(out, q * cos + rotate_half(q) * sin)
    assert len(calls) == 2
    for got_k, got_v in calls:
        assert torch.equal(got_k, k * cos + rotate_half(k) * sin) and torch.equal(got_v, v)


def test_other_forms_take_the_formula():
    """fp32 activations, a head size other than 128 and a bf16 cache: the torch formula and
    KVCache.write."""
    from engine.core.kv_cache import KVCache, rotate_half
    print("[case] rope kv write, other forms", flush=True)
    for D, dtype, kind in ((64, torch.bfloat16, "fp8"), (128, torch.float32, "int8"), (128, torch.bfloat16, None)):
        g = torch.Generator().manual_seed(D)
        q, k, v = (torch.randn(3, n, D, generator=g).to(dtype).to(DEV) for n in (4, 2, 2))
        ang = torch.randn(3, 1, D, generator=g)
        cos, sin = ang.cos().to(dtype).to(DEV), ang.sin().to(dtype).to(DEV)
        slots = torch.tensor([4, 0, 9], device=DEV)
        got, want = (KVCache("paged", 1, 2, D, 16, torch.bfloat16, DEV, block_size=16, kv_dtype=kind) for _ in range(2))
        out = got.write_rotated(0, slots, q, k, v, cos, sin)
        want.write(0, slots, k * cos + rotate_half(k) * sin, v)
        assert torch.equal(out, q * cos + rotate_half(q) * sin)
        assert torch.equal(got.k.view(torch.uint8), want.k.view(torch.uint8))
        assert torch.equal(got.v.view(torch.uint8), want.v.view(torch.uint8))
