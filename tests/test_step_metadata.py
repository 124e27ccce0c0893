"""BatchMetadata's index tensors on the CPU, against the tensors formed one request at a time."""
import pytest
import torch

from engine.core.kv_cache import CacheBookkeeping, make_allocator, pack_block_tables
from engine.core.model_runner import BatchMetadata, Request


class Cache(CacheBookkeeping):
    def __init__(self, mode, capacity=512, block_size=4):
        self.mode, self.block_size = mode, block_size
        self.allocator = make_allocator(mode, capacity, block_size)


class Other(Cache):
    """A cache with its own slots()."""

    def slots(self, req, start, end):
        return super().slots(req, start, end) + 1000


def requests(cache, lengths, seed):
    g = torch.Generator().manual_seed(seed)
    out = []
    for i, n in enumerate(lengths):
        ids = torch.randint(0, 1000, (n,), generator=g).tolist()
        cut = max(1, n - i % 3)  # the last tokens are generated ones
        r = Request(ids[:cut], 8, rid=i)
        r.output_ids = ids[cut:]
        assert cache.admit(r, 64) is not None and cache.ensure(r, n)
        out.append(r)
    return out


@pytest.mark.parametrize("mode", ["paged", "contiguous"])
@pytest.mark.parametrize("kind", [Cache, Other])
@pytest.mark.parametrize("starts", [[4, 8, 16, 0, 10], [4, 0, 3, 0, 10], [0, 0, 0, 0, 0], [4, 8, 16, 0, 9]])
@pytest.mark.parametrize("backend", ["triton", "sdpa"])
def test_indexes_equal_the_per_request_ones(mode, kind, starts, backend):
    """Decode rows only, prompts only and both; tables of odd and even length in front of the
    context lengths; a one-token prompt (start 0) is a prefill."""
    lengths = [5, 9, 17, 1, 11]
    cache = kind(mode)
    chunks = [(r, s, n) for r, s, n in zip(requests(cache, lengths, seed=3), starts, lengths)]
    meta = BatchMetadata(chunks, cache, "cpu", backend)
    assert meta.input_ids.tolist() == [t for r, s, e in chunks for t in r.all_ids[s:e]]
    assert torch.equal(meta.positions, torch.cat([torch.arange(s, e) for _, s, e in chunks]))
    assert torch.equal(meta.write_slots, torch.cat([cache.slots(r, s, e) for r, s, e in chunks]))
    rows = torch.tensor([e - s for _, s, e in chunks]).cumsum(0) - 1
    assert torch.equal(meta.last_rows, rows) and meta.num_tokens == int(rows[-1]) + 1
    decode = [i for i, (_, s, e) in enumerate(chunks) if e - s == 1 and s > 0]
    assert meta.decode_rows.tolist() == [int(rows[i]) for i in decode]
    assert meta.all_decode == (len(decode) == len(chunks)) and len(meta.prefill) == len(chunks) - len(decode)
    for t in (meta.input_ids, meta.positions, meta.write_slots, meta.last_rows, meta.decode_rows):
        assert t.dtype == torch.int64
    if backend == "triton" and decode:
        want = cache.decode_tables([(chunks[i][0], chunks[i][2]) for i in decode], "cpu")
        table, lens, page, longest, splits = meta.decode_tables
        assert table.dtype == lens.dtype == torch.int32 and table.is_contiguous()
        assert torch.equal(table, want[0]) and torch.equal(lens, want[1])
        assert (page, longest, splits) == (want[2], want[3], None)
    else:
        assert meta.decode_tables is None


@pytest.mark.parametrize("mode", ["paged", "contiguous"])
def test_prompts_stay_tensors(mode, monkeypatch):
    """The slots and positions of a prompt or a longer chunk never become Python integers (which
    takes longer than the rest of the metadata), next to decode rows either."""
    cache = Cache(mode)
    chunks = [(r, s, n) for r, s, n in zip(requests(cache, [9, 30, 17, 1], seed=5), [8, 0, 5, 0], [9, 30, 17, 1])]

    def refuse(tensor):
        raise AssertionError(f"{tensor.numel()} values to Python")

    with monkeypatch.context() as patch:
        patch.setattr(torch.Tensor, "tolist", refuse)
        meta = BatchMetadata(chunks, cache, "cpu")
    assert torch.equal(meta.positions, torch.cat([torch.arange(s, e) for _, s, e in chunks]))
    assert torch.equal(meta.write_slots, torch.cat([cache.slots(r, s, e) for r, s, e in chunks]))
    for (first, n, start, context), (r, s, e) in zip(meta.prefill, chunks[1:]):
        assert (n, start) == (e - s, s) and torch.equal(context, cache.slots(r, 0, e))


def test_a_step_without_chunks_is_refused():
    with pytest.raises((RuntimeError, ValueError), match="non-empty"):
        BatchMetadata([], Cache("paged"), "cpu")


def test_slots_of_another_width_are_taken():
    """A cache's own slots() may give 32-bit values."""
    class Narrow(Cache):
        def slots(self, req, start, end):
            return super().slots(req, start, end).int()

    cache = Narrow("paged")
    chunks = [(r, s, n) for r, s, n in zip(requests(cache, [9, 30], seed=5), [8, 0], [9, 30])]
    meta = BatchMetadata(chunks, cache, "cpu")
    assert meta.write_slots.dtype == torch.int64
    assert meta.write_slots.tolist() == [t for r, s, e in chunks for t in cache.slots(r, s, e).tolist()]


@pytest.mark.parametrize("where", ["slots", "decode_tables", "allocator", "allocator_class"])
def test_replaced_methods_are_asked(where):
    """A slots() or decode_tables() set on the cache object, a slots() set on its allocator, and
    an allocator of another class are used for decode rows too."""
    cache = Cache("paged")
    plain_slots, plain_tables = cache.slots, cache.decode_tables
    if where == "slots":
        cache.slots = lambda req, start, end: plain_slots(req, start, end) + 1000
    elif where == "decode_tables":
        cache.decode_tables = lambda entries, device: ("tables", entries, device, 7)
    elif where == "allocator":
        inner = cache.allocator.slots
        cache.allocator.slots = lambda req, start, end: inner(req, start, end) + 1000
    else:
        class Shifted:  # (no slot(), as an allocator may lack it)
            def __init__(self, own):
                self.own, self.tables, self.block_size, self.blocks_for = own, own.tables, own.block_size, own.blocks_for

            def __getattr__(self, name):
                if name == "slot":
                    raise AttributeError(name)
                return getattr(self.own, name)

            def slots(self, req, start, end):
                return self.own.slots(req, start, end) + 1000

        cache.allocator = Shifted(cache.allocator)
    chunks = [(r, n - 1, n) for r, n in zip(requests(cache, [5, 9], seed=7), [5, 9])]
    meta = BatchMetadata(chunks, cache, "cpu")
    assert meta.write_slots.tolist() == [cache.slots(r, s, e).item() for r, s, e in chunks]
    assert (int(meta.write_slots[0]) >= 1000) == (where != "decode_tables")
    if where == "decode_tables":
        assert meta.decode_tables[0] == "tables" and meta.decode_tables[3] == 7
    else:
        assert torch.equal(meta.decode_tables[0], plain_tables([(r, e) for r, _, e in chunks], "cpu")[0])


def test_tables_do_not_alias_the_allocator():
    """The packed tables are copies: growing a request later leaves an older step's table alone."""
    lists = [[3, 1], [2]]
    table, lens = pack_block_tables(lists, [7, 2], "cpu")
    lists[0][0] = 9
    assert table.tolist() == [[3, 1], [2, 0]] and lens.tolist() == [7, 2]
