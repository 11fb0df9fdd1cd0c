"""GPU: a ragged batch of requests in one launch installs exactly what per-request launches do.

Each request of the batch has its own source slots, block-table pages,
positions and prefix (windows). The batch writes every row bit-identically
to one ``map_install`` per request (the per-request path is pinned against
the oracle by the fused-install parity tests), leaves every other row
untouched, and flags rows an index places outside a pool without writing
them.
"""

from __future__ import annotations

import pytest
import torch

from cachebridge_amd import synthetic
from cachebridge_amd.online.blocks import map_install_batch
from cachebridge_amd.plan import RequestSpan
from cachebridge_amd.pool import PagedKVPool, pool_rows

pytestmark = pytest.mark.gpu


def _shape(name, tokens, layers):
    sh = synthetic.shape(name, tokens=tokens)
    if layers is not None:
        sh.target_layers = layers
        if sh.windows is not None:
            sh.windows = [None if w is None else 1024 for w in sh.windows[:layers]]
            sh.target_theta = sh.target_theta[:layers]
    return sh


def _batch(lengths, positions, prefixes, pages_total, seed):
    """Spans over one concatenated source-slot vector and one concatenated block table."""
    g = torch.Generator().manual_seed(seed)
    order = torch.randperm(pages_total, generator=g).to(torch.int32)
    spans, src, entry = [], 0, 0
    for n, p, pre in zip(lengths, positions, prefixes):
        spans.append(RequestSpan(src, entry * 16, n, p, pre))
        src += n
        entry += (n + 15) // 16
    assert entry <= pages_total
    return spans, order[:max(entry, 1)].contiguous()


def _target_like(pool, fill="zeros"):
    return PagedKVPool(layer_num=pool.layer_num, pages=pool.pages, head_num=pool.head_num,
                       head_dim=pool.head_dim, page_size=pool.page_size, dtype=pool.dtype,
                       device=pool.device, fill=fill)


@pytest.mark.parametrize("name,layers,lengths,positions,prefixes", [
    ("tp4", 6, [1, 15, 0, 16, 17, 300, 1000, 2500], [0, 0, 0, 3, 40, 0, 77, 0], [0] * 8),
    ("toy", None, [5, 64, 200, 33], [0, 10, 0, 100], [0, 0, 0, 0]),
    ("gemma", 12, [200, 1500, 700, 2100], [0, 0, 500, 0], [0, 0, 2000, 0]),
])
def test_batch_equals_per_request_installs(name, layers, lengths, positions, prefixes):
    print(f"batch {name} layers={layers} lengths={lengths}", flush=True)
    sh = _shape(name, sum(lengths), layers)
    pages = sum((n + 15) // 16 for n in lengths) * 2
    h = synthetic.make_handoff(sh, target_pages=pages, fill_target="zeros")
    spans, bt = _batch(lengths, positions, prefixes, pages, seed=11)
    check_batch_equals_single(h, spans, bt.to(h.target_pool.device))


def _streamed(plan):
    """Whether the plan's last launch was the streaming kernel's: a workgroup per CU."""
    return plan.last_split()[1] == torch.cuda.get_device_properties(0).multi_processor_count // 8 * 8


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("windows", [None, [None, 40, 300]])
def test_batch_equals_per_request_installs_at_head_dim_64(dtype, windows):
    """Batches long enough for the streaming kernel (shorter ones take another),
    whose requests alone are short ones."""
    print(f"batch D=64 {dtype} windows={windows}", flush=True)
    lt, lengths = 12, [700, 33, 0, 1200, 16, 1500]
    sh = synthetic.Shape("batch64", 8, 2, lt, 4, 64, sum(lengths), dtype, [],
                         target_theta=1e6 if windows is None else [1e6 if windows[l % 3] is None else 1e4
                                                                   for l in range(lt)],
                         windows=windows and [windows[l % 3] for l in range(lt)], seed=51)
    pages = sum((n + 15) // 16 for n in lengths) * 2
    h = synthetic.make_handoff(sh, target_pages=pages, fill_target="zeros")
    spans, bt = _batch(lengths, [0, 3, 0, 77, 0, 0], [0] * 6, pages, seed=17)
    map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool, spans,
                      block_table=bt.to(h.target_pool.device), page_size=16)
    assert _streamed(h.mapper.plan)
    check_batch_equals_single(h, spans, bt.to(h.target_pool.device))


def check_batch_equals_single(h, spans, bt):
    """One batched launch over ``spans`` against one ``map_install`` per request."""
    map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool, spans,
                      block_table=bt, page_size=16)
    assert h.mapper.plan.read_errors() == 0
    single = _target_like(h.target_pool)
    for sp in spans:
        if sp.num_tokens == 0:
            continue
        e = sp.target_offset // 16
        src = pool_rows(h.source_pool, index=h.source_slots, index_offset=sp.source_offset,
                        tokens=sp.num_tokens)
        tgt = pool_rows(single, block_table=bt[e:e + (sp.num_tokens + 15) // 16], page_size=16,
                        tokens=sp.num_tokens)
        h.mapper.map_install(src, tgt, num_tokens=sp.num_tokens, position_start=sp.position_start,
                             prefix_length=sp.prefix_length)
    torch.cuda.synchronize()
    assert h.mapper.plan.read_errors() == 0
    assert torch.equal(h.target_pool.k_data, single.k_data)
    assert torch.equal(h.target_pool.v_data, single.v_data)
    # the batch wrote the last token of every request that some layer keeps
    # (so the comparison is not between two all-zero pools)
    for sp in spans:
        if sp.num_tokens and _some_layer_keeps_last_token(h.shape, sp):
            u = sp.target_offset + sp.num_tokens - 1
            row = int(bt[u // 16]) * 16 + u % 16
            assert h.target_pool.v_data[:, row].abs().sum() > 0


def _some_layer_keeps_last_token(sh, sp):
    """A layer without a window keeps every token; a window W keeps the last W - 1 of the prefix."""
    prefix = sp.prefix_length or sp.position_start + sp.num_tokens
    last = sp.position_start + sp.num_tokens - 1
    return any(w is None or last >= prefix - (w - 1) for w in (sh.windows or [None]))


@pytest.mark.parametrize("windows", [[40, 300, 40, 300, 90], [300, 40, None, 40, 300]])
@pytest.mark.parametrize("tokens", [100, 200, 600])
def test_support_classes_without_tokens(windows, tokens):
    """Early blocks of a long prefix at support 4: windows that have not opened
    keep no token, alone or before and after classes that do."""
    print(f"support batch windows={windows} tokens={tokens}", flush=True)
    sh = synthetic.Shape("closed_windows", 9, 3, 5, 3, 128, 2 * tokens, torch.bfloat16, [], target_theta=1e6,
                         windows=windows, head_map="identity", target_pages=256, seed=43, support=4)
    h = synthetic.make_handoff(sh, fill_target="zeros")
    pages = h.target_pool.pages
    for prefixes in ([tokens + 45, tokens + 100], [tokens + 120, 0], [4096, 4096]):
        h.target_pool.k_data.zero_()
        h.target_pool.v_data.zero_()
        spans, bt = _batch([tokens, tokens], [0, 0], prefixes, pages, seed=13)
        check_batch_equals_single(h, spans, bt.to(h.target_pool.device))
        kept = torch.zeros(5, h.target_pool.size, dtype=torch.bool)
        for sp, prefix in zip(spans, prefixes):
            for layer, window in enumerate(windows):
                first = 0 if window is None else min(tokens, max(0, (prefix or tokens) - (window - 1)))
                u = torch.arange(first, tokens) + sp.target_offset
                kept[layer, bt[u // 16].long() * 16 + u % 16] = True
        written = (h.target_pool.v_data != 0).flatten(2).any(2).cpu()
        assert torch.equal(written, kept), prefixes


@pytest.mark.parametrize("layers,lengths", [(2, [40, 56]), (32, [500, 400])])
def test_batch_flags_out_of_range_rows_and_skips_them(layers, lengths):
    """In a batch of the short kernel and in one of the streaming kernel."""
    pages = sum((n + 15) // 16 for n in lengths) + 9
    sh = _shape("tp4", sum(lengths), layers)
    h = synthetic.make_handoff(sh, target_pages=pages, fill_target="zeros")
    spans, bt = _batch(lengths, [0, 0], [0, 0], pages, seed=3)
    bt = bt.to(h.target_pool.device)
    bad = bt.clone()
    bad[1] = h.target_pool.pages + 5  # request 0's second page lies beyond the pool
    map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool, spans,
                      block_table=bad, page_size=16)
    assert h.mapper.plan.read_errors() & 2
    assert _streamed(h.mapper.plan) == (layers == 32)
    good = _target_like(h.target_pool)
    # request 0 without its tokens 16..31 (the bad page): those rows are not written
    ok = [spans[0]._replace(num_tokens=16),
          RequestSpan(spans[0].source_offset + 32, spans[0].target_offset + 32, lengths[0] - 32, 32, lengths[0]),
          spans[1]]
    map_install_batch(h.mapper, h.source_pool, h.source_slots, good, ok, block_table=bt,
                      page_size=16)
    assert h.mapper.plan.read_errors() == 0
    assert torch.equal(h.target_pool.k_data, good.k_data)
    assert torch.equal(h.target_pool.v_data, good.v_data)


def test_batch_rejects_bad_requests_before_launch():
    sh = _shape("tp4", 64, 2)
    h = synthetic.make_handoff(sh, target_pages=16, fill_target="zeros")
    spans, bt = _batch([32, 32], [0, 0], [0, 0], 16, seed=5)
    bt = bt.to(h.target_pool.device)
    with pytest.raises(ValueError, match="positions"):
        map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool,
                          [spans[0]._replace(position_start=h.mapper.plan.max_positions - 8)],
                          block_table=bt, page_size=16)
    with pytest.raises(ValueError, match="source_indices"):
        map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool,
                          [spans[1]._replace(source_offset=40)], block_table=bt, page_size=16)
    with pytest.raises(ValueError, match="block table"):
        map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool,
                          [spans[1]._replace(target_offset=16 * 16)], block_table=bt, page_size=16)
    with pytest.raises(ValueError, match="prefix_length"):
        map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool,
                          [spans[0]._replace(prefix_length=10)], block_table=bt, page_size=16)
    torch.cuda.synchronize()
    assert int(h.target_pool.k_data.abs().sum()) == 0  # nothing was written
    map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool, [],
                      block_table=bt, page_size=16)  # an empty batch is a no-op
