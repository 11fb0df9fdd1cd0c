"""GPU: short requests take a kernel of their own whose rows are bit-identical.

The streaming kernel (forced by an explicit ``tokens_per_workgroup``) and the
short-request kernel (the default at these lengths) must write the same bits:
at the edges of the 16-token sub-tiles, 64-token rounds and workgroup chunks,
with windows, per-layer thetas, slot vectors, batches and rows out of range.
"""

from __future__ import annotations

import pytest
import torch

from cachebridge_amd import synthetic
from cachebridge_amd.online.blocks import map_install_batch, map_install_block
from cachebridge_amd.plan import RequestSpan

pytestmark = pytest.mark.gpu


def _handoff(dim, dtype, tokens, windows=None, target_theta=1e6):
    lt = 5
    sh = synthetic.Shape(f"short{dim}", 6, 3, lt, 3, dim, tokens, dtype, [0, 2, 3, 5], source_theta=1e6,
                         target_theta=target_theta, windows=windows, target_pages=2 * (tokens // 16 + 2), seed=31 + dim)
    return synthetic.make_handoff(sh, fill_target="zeros")


def _pools(h, run):
    pool = h.target_pool
    pool.k_data.fill_(0.25)
    pool.v_data.fill_(0.25)
    run()
    torch.cuda.synchronize()
    assert h.mapper.plan.read_errors() == 0
    return pool.k_data.clone(), pool.v_data.clone()


@pytest.mark.parametrize("dim,dtype", [(128, torch.bfloat16), (64, torch.bfloat16), (64, torch.float32)])
@pytest.mark.parametrize("tokens", [1, 15, 16, 17, 63, 64, 65, 127, 129, 513, 700])
def test_short_rows_equal_streaming_rows(dim, dtype, tokens):
    print(f"short D={dim} {dtype} T={tokens}", flush=True)
    windows = [None, 40, None, 40, 2] if tokens % 2 else None
    h = _handoff(dim, dtype, tokens, windows, [1e6, 1e4, 1e6, 1e4, 1e6])
    short = _pools(h, h.run)
    chunks, groups = h.mapper.plan.last_split()
    assert chunks == 0
    stream = _pools(h, lambda: h.run(tokens_per_workgroup=512))
    assert torch.equal(short[0], stream[0]) and torch.equal(short[1], stream[1])
    assert bool((short[0] != 0.25).any())


@pytest.mark.parametrize("tokens,window,prefix,items", [
    (200, 64, 0, 40 * 4 + 216),       # few long jobs: round by round
    (400, 64, 0, 40 * 7 + 216),
    (600, 128, 0, None),              # more rounds than the chip holds: the streaming kernel
    (2000, 64, 0, None),
    (600, 1024, 5000, 40 * 10),       # windows that have not opened: 12 chunks a global job fill the chip
    (1500, 1024, 5000, 40 * 12),
])
def test_unequal_window_classes(tokens, window, prefix, items):
    """Which kernel maps a request whose window classes keep unequal token
    counts, and that its rows are the streaming kernel's."""
    print(f"unequal classes T={tokens} window={window} prefix={prefix}", flush=True)
    windows = [None if l % 6 == 5 else window for l in range(64)]
    sh = synthetic.Shape("unequal", 6, 2, 64, 2, 64, tokens, torch.bfloat16, [0, 2, 3, 5], source_theta=1e6,
                         target_theta=[1e6 if w is None else 1e4 for w in windows], windows=windows,
                         target_pages=tokens // 16 + 2, seed=37)
    h = synthetic.make_handoff(sh, fill_target="zeros")

    def run(cap):
        map_install_block(h.mapper, h.source_pool, h.source_slots, h.target_pool, start=0, stop=tokens,
                          block_table=h.block_table, page_size=16, prefix_length=prefix, tokens_per_workgroup=cap)

    got = _pools(h, lambda: run(0))
    groups = h.mapper.plan.last_split()[1]
    cus = torch.cuda.get_device_properties(0).multi_processor_count // 8 * 8
    stream = _pools(h, lambda: run(512))
    assert torch.equal(got[0], stream[0]) and torch.equal(got[1], stream[1])
    assert groups == (cus if items is None else -(-items // 8) * 8), groups


@pytest.mark.parametrize("tokens,prefix,windows", [
    (900, 1300, [None, 40, 300, 600]),    # two closed windows at the end, one open in between
    (900, 1100, [None, 40, 300, 150]),    # two closed ones between others
    (900, 940, [500, 40, 300, 150]),      # one closed at the start
    (900, 5000, [None, 40, 300, 600]),
])
@pytest.mark.parametrize("lt", [12, 64])
def test_streaming_line_steps_over_closed_windows(lt, tokens, prefix, windows):
    """Early blocks of a prefix at the streaming kernel: the rows are the short
    kernel's wherever the classes without tokens lie (at 64 layers, a gap of
    one or two classes is long enough for a launch on either side of it)."""
    print(f"closed windows={windows} prefix={prefix} layers={lt}", flush=True)
    sh = synthetic.Shape("closed", 6, 3, lt, 3, 64, tokens, torch.bfloat16, [0, 2, 3, 5], source_theta=1e6,
                         target_theta=[1e6 if windows[l % 4] is None else 1e4 for l in range(lt)],
                         windows=[windows[l % 4] for l in range(lt)], target_pages=tokens // 16 + 2, seed=39)
    h = synthetic.make_handoff(sh, fill_target="zeros")

    def run(block, cap):
        for start in range(0, tokens, block):
            map_install_block(h.mapper, h.source_pool, h.source_slots, h.target_pool, start=start, stop=start + block,
                              block_table=h.block_table, page_size=16, prefix_length=prefix, tokens_per_workgroup=cap)

    short = _pools(h, lambda: run(100, 0))
    cus = torch.cuda.get_device_properties(0).multi_processor_count // 8 * 8
    assert h.mapper.plan.last_split()[1] != cus  # (the streaming kernel's grid)
    stream = _pools(h, lambda: run(tokens, 16))
    assert torch.equal(short[0], stream[0]) and torch.equal(short[1], stream[1])
    assert bool((stream[1] != 0.25).any())


def test_closed_windows_cost_next_to_nothing():
    """The launch of a target whose windows have not opened against one of its
    global layers alone (10 of 62): about the same work. Walking the 832 units
    without tokens had taken 5 to 10 times as long."""
    print("time of closed windows", flush=True)
    times = {}
    for lt, windows in ((62, [None if l % 6 == 5 else 1024 for l in range(62)]), (10, None)):
        sh = synthetic.Shape("closed", 6, 4, lt, 16, 64, 1500, torch.bfloat16, [0, 2, 3, 5], target_theta=1e6,
                             windows=windows, target_pages=96, seed=40)
        h = synthetic.make_handoff(sh, fill_target="zeros")
        for _ in range(2):  # the first turn warms up
            start, stop = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            torch.cuda._sleep(2_000_000)
            start.record()
            for _ in range(20):
                map_install_block(h.mapper, h.source_pool, h.source_slots, h.target_pool, start=0, stop=1500,
                                  block_table=h.block_table, page_size=16, prefix_length=9000)
            stop.record()
            torch.cuda.synchronize()
            times[lt] = start.elapsed_time(stop)
    assert times[62] <= 2 * times[10], times


def test_short_batch_equals_per_request_rows():
    """Ragged requests (one empty, one inside its prefix) in one short launch."""
    print("short batch", flush=True)
    lengths, starts = [37, 0, 16, 90], [0, 0, 100, 7]
    h = _handoff(128, torch.bfloat16, sum(lengths), [None, 40, None, 40, 2])
    need = [(n + 15) // 16 for n in lengths]
    bt = torch.randperm(h.target_pool.pages, generator=torch.Generator().manual_seed(3))[:sum(need)].to(torch.int32).cuda()
    spans, off, entry = [], 0, 0
    for n, p, k in zip(lengths, starts, need):
        spans.append(RequestSpan(off, entry * 16, n, p, 0))
        off, entry = off + n, entry + k

    def each():
        for sp, k in zip(spans, need):
            if sp.num_tokens:
                map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool, [sp], block_table=bt, page_size=16)

    got = _pools(h, lambda: map_install_batch(h.mapper, h.source_pool, h.source_slots, h.target_pool, spans,
                                              block_table=bt, page_size=16))
    want = _pools(h, each)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])


def test_rows_out_of_range_are_flagged_not_written():
    print("short rows out of range", flush=True)
    h = _handoff(128, torch.bfloat16, 50)
    slots = torch.arange(50, dtype=torch.int64, device="cuda")
    good = _pools(h, lambda: map_install_block(h.mapper, h.source_pool, h.source_slots, h.target_pool, start=0, stop=50,
                                               target_indices=slots))
    bad_slots, bad_source = slots.clone(), h.source_slots.clone()
    bad_slots[3] = h.target_pool.size
    bad_slots[40] = -1
    bad_source[20] = h.source_pool.size
    pool = h.target_pool
    pool.k_data.fill_(0.25)
    pool.v_data.fill_(0.25)
    map_install_block(h.mapper, h.source_pool, bad_source, pool, start=0, stop=50, target_indices=bad_slots)
    assert h.mapper.plan.read_errors() == 3
    for got, want in zip((pool.k_data, pool.v_data), good):
        want = want.clone()
        want[:, [3, 20, 40]] = 0.25
        assert torch.equal(got, want)


@pytest.mark.parametrize("windows", [None, [None, 300, None, 40, 2]])
def test_support_rows_do_not_depend_on_the_request_length(windows):
    """Support maps: waves without tokens, last blocks of every wave count and
    unequal token chunks per job, against the rows of one long request."""
    print(f"support lengths windows={windows}", flush=True)
    sh = synthetic.Shape("support_lengths", 9, 3, 5, 3, 128, 700, torch.bfloat16, [], target_theta=1e6,
                         windows=windows, head_map="identity", target_pages=128, seed=41, support=4)
    h = synthetic.make_handoff(sh, fill_target="zeros")
    pool = h.target_pool
    slots = torch.randperm(pool.size, generator=torch.Generator().manual_seed(2))[:700].cuda()

    def rows(start, stop):
        pool.k_data.fill_(0.25)
        pool.v_data.fill_(0.25)
        map_install_block(h.mapper, h.source_pool, h.source_slots, pool, start=start, stop=stop, target_indices=slots,
                          prefix_length=700)
        torch.cuda.synchronize()
        assert h.mapper.plan.read_errors() == 0
        return pool.k_data[:, slots].clone(), pool.v_data[:, slots].clone(), pool.k_data.clone()

    whole = rows(0, 700)
    for start, n in [(0, 1), (0, 31), (5, 32), (0, 33), (0, 96), (400, 224), (400, 225), (400, 256), (0, 257), (389, 311),
                     (100, 513)]:
        got = rows(start, start + n)
        for a, b in zip(got[:2], whole[:2]):
            assert torch.equal(a[:, start:start + n], b[:, start:start + n]), (start, n)
            assert bool((a[:, :start] == 0.25).all()) and bool((a[:, start + n:] == 0.25).all()), (start, n)
        outside = torch.ones(pool.size, dtype=torch.bool, device="cuda")
        outside[slots] = False
        assert bool((got[2][:, outside] == 0.25).all())
