"""The work this framework does for its users, as cases that can be timed and compared.

A case names a handoff geometry (source layers x KV heads -> target layers x
KV heads, head_dim, support size, dtype), the request's tokens and the public
entry point that maps it:

- ``install``:   ``map_install_block``, source pool rows straight into target
                 pool pages (block table) or slots (page size 1);
- ``batch``:     ``map_install_batch``, a ragged cohort of requests at once;
- ``delivered``: ``SelectedBlockDelivery`` + ``map_install_delivered``, a
                 history that arrives in 2048-token blocks;
- ``page``:      ``HeadwiseMapper.map_page``, one dense page in and out;
- ``delta``:     ``transform_delta_state``, the recurrent memory of a hybrid
                 model's linear-attention layers.

Maps are N(0, 1/(s D)), biases N(0, 0.01), source rows N(0, 1) times a
lognormal scale per channel, pages drawn from a shuffled free list.
"""

from __future__ import annotations

import math
import random

import torch

from cachebridge_amd.architectures import transform_delta_state
from cachebridge_amd.layouts import gemma_layer_types, head_assignment, mapper_windows
from cachebridge_amd.mapper import HeadwiseMapper
from cachebridge_amd.online.blocks import map_install_batch, map_install_block
from cachebridge_amd.online.delivery import SelectedBlockDelivery, map_install_delivered
from cachebridge_amd.plan import RequestSpan
from cachebridge_amd.pool import PagedKVPool

PAGE = 16
BLOCK = 2048
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
SELECTED = 16  # source layers a support-1 mapper reads


def _handoff(op, tokens, *, source=(40, 2), target=(64, 2), head_dim=128, support=1, dtype="bf16",
             window=0, slots=False, **more):
    return dict(op=op, tokens=tokens, source_layers=source[0], source_heads=source[1],
                target_layers=target[0], target_heads=target[1], head_dim=head_dim, support=support,
                dtype=dtype, window=window, slots=slots, **more)


def _delta(layers, heads, k, v, kp, vp):
    return dict(op="delta", layers=layers, heads=heads, k=k, v=v, kp=kp, vp=vp)


def listed():
    named = [
        # One tensor-parallel rank's share of a 40-layer -> 64-layer handoff:
        # the benchmark's own step, an ordinary prompt.
        ("share 4096", _handoff("install", 4096)),
        # The same share for a short prompt: the smallest call.
        ("share 37", _handoff("install", 37)),
        # The whole model on one GPU.
        ("whole 4096", _handoff("install", 4096, source=(40, 8), target=(64, 8))),
        # A target with sliding-window layers (5 local : 1 global) and twice
        # the source's KV heads, long history.
        ("windows 8192", _handoff("install", 8192, source=(40, 8), target=(62, 16), window=1024)),
        # The shipped recipe: every target head maps eight source rows.
        ("support8 4096", _handoff("install", 4096, support=8)),
        # The recipe for a short prompt.
        ("support8 311", _handoff("install", 311, support=8)),
        # An admitted cohort of ragged requests in one launch.
        ("cohort 16", _handoff("batch", 2048, requests=16)),
        # A history delivered block by block, the last block ragged.
        ("delivered 6000", _handoff("delivered", 6000)),
        # Head size 256 (the smaller sliding-window models).
        ("dim256 2048", _handoff("install", 2048, source=(34, 4), target=(48, 8), head_dim=256, window=1024)),
        # A pool in half precision, token slots instead of pages.
        ("fp16 1000", _handoff("install", 1000, dtype="fp16", slots=True)),
        # The dense page interface in fp32 at the small-model shape.
        ("page fp32 250", _handoff("page", 250, source=(8, 2), target=(12, 2), head_dim=64, dtype="fp32")),
        # Recurrent states of 48 linear-attention layers of 32 heads.
        ("delta 48x32", _delta(48, 32, 128, 128, 128, 128)),
    ]
    return [dict(case, name=name) for name, case in named]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    family = rng.choice(["share", "share", "whole", "windows", "support", "support", "batch", "delivered",
                         "dim256", "half", "page", "delta"])
    if family == "share":
        return _handoff("install", _log_uniform(rng, 16, 16384), head_dim=rng.choice([64, 128, 128]),
                        slots=rng.random() < 0.3)
    if family == "whole":
        return _handoff("install", _log_uniform(rng, 16, 4096), source=(40, 8), target=(64, 8))
    if family == "windows":
        return _handoff("install", _log_uniform(rng, 64, 8192), source=(40, 8), target=(62, 16),
                        window=rng.choice([512, 1024]))
    if family == "support":
        return _handoff("install", _log_uniform(rng, 16, 4096), head_dim=rng.choice([64, 128, 128]),
                        support=rng.choice([2, 4, 8, 8]))
    if family == "batch":
        return _handoff("batch", rng.choice([512, 1024, 2048]), requests=rng.randint(2, 16))
    if family == "delivered":
        return _handoff("delivered", _log_uniform(rng, 100, 12000))
    if family == "dim256":
        return _handoff("install", _log_uniform(rng, 16, 2048), source=(34, 4), target=(48, 8), head_dim=256,
                        window=rng.choice([0, 1024]), support=rng.choice([1, 1, 2]))
    if family == "half":
        return _handoff("install", _log_uniform(rng, 16, 2000), head_dim=rng.choice([64, 96, 128]), dtype="fp16",
                        support=rng.choice([1, 1, 4]), slots=rng.random() < 0.5)
    if family == "page":
        return _handoff("page", _log_uniform(rng, 16, 4096), source=(8, 2), target=(12, 2),
                        head_dim=rng.choice([64, 128]), dtype=rng.choice(["fp32", "fp32", "bf16"]))
    k, v = rng.choice([64, 128, 128]), rng.choice([64, 128, 128, 256])
    kp, vp = rng.choice([(k, v), (128, 128), (64, 128)])
    return _delta(rng.randint(1, 24), rng.choice([16, 32]), k, v, kp, vp)


# ---------------------------------------------------------------------------
# Geometry that follows from a case
# ---------------------------------------------------------------------------


def _windows(case):
    """Per target layer: sliding window or None."""
    if not case["window"]:
        return [None] * case["target_layers"]
    return mapper_windows(gemma_layer_types(case["target_layers"]), case["window"])


def _target_thetas(case):
    return [1e6 if w is None else 1e4 for w in _windows(case)]


def _lengths(case):
    """Tokens of each request."""
    if case["op"] != "batch":
        return [case["tokens"]]
    r = random.Random(1000 * case["requests"] + case["tokens"])
    return [max(64, min(8192, round(case["tokens"] * math.exp(0.5 * r.gauss(0, 1)))))
            for _ in range(case["requests"])]


def _kept(case, n, window):
    return n if window is None else min(n, window - 1)


def _selected(case):
    count = min(case["source_layers"], SELECTED)
    return [round(i * (case["source_layers"] - 1) / (count - 1)) for i in range(count)]


def _assignment(case, g):
    """Source (layer, head) of every target (layer, head): ``[Lt, Ht, s]`` each."""
    lt, ht, s = case["target_layers"], case["target_heads"], case["support"]
    ls, hs = case["source_layers"], case["source_heads"]
    if s == 1:
        sel = torch.tensor(_selected(case))
        layer = sel[torch.randint(0, len(sel), (lt, ht, 1), generator=g)]
    else:  # the depth-matched layer and its neighbours, shared by a layer's heads
        rows = []
        for l in range(lt):
            c = round(l * (ls - 1) / (lt - 1))
            near = [x for x in range(max(0, c - 12), min(ls, c + 13)) if x != c]
            pick = torch.randperm(len(near), generator=g)[: s - 1].tolist()
            rows.append([c] + [near[i] for i in pick])
        layer = torch.tensor(rows)[:, None, :].expand(lt, ht, s).clone()
    if hs == ht and s > 1:
        head = torch.arange(ht).view(1, ht, 1).expand(lt, ht, s).clone()
    elif hs != ht:  # two target heads per source head
        heads = head_assignment(hs, ht, [h * hs // ht for h in range(ht)])
        head = torch.tensor(heads).view(1, ht, 1).expand(lt, ht, s).clone()
    else:
        head = torch.randint(0, hs, (lt, ht, 1), generator=g)
    return layer, head


def _distinct_pairs(case):
    """Source (layer, head) pairs that a handoff reads, about."""
    lt, ht, s = case["target_layers"], case["target_heads"], case["support"]
    if s > 1:
        return min(case["source_layers"] * case["source_heads"], lt * ht * s)
    pairs = min(case["source_layers"], SELECTED) * case["source_heads"]
    return round(pairs * (1 - (1 - 1 / pairs) ** (lt * ht)))


# ---------------------------------------------------------------------------
# Inputs
# ---------------------------------------------------------------------------


def _rows(shape, scale, dtype, g):
    """Source rows N(0, 1) times the channel scale, layer by layer."""
    out = torch.empty(shape, dtype=dtype, device="cuda")
    for part in out.unbind(0):
        part.copy_(torch.randn(part.shape, generator=g, device="cuda").mul_(scale))
    return out


def _prepare_handoff(case, seed):
    cpu = torch.Generator().manual_seed(seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    lt, ht, s, d = case["target_layers"], case["target_heads"], case["support"], case["head_dim"]
    dtype = DTYPES[case["dtype"]]
    layer, head = _assignment(case, cpu)
    std = 1 / math.sqrt(s * d)
    maps = {"k_weight": torch.randn(lt, ht, s * d, d, generator=g, device="cuda") * std,
            "v_weight": torch.randn(lt, ht, s * d, d, generator=g, device="cuda") * std,
            "k_bias": torch.randn(lt, ht, d, generator=g, device="cuda") * 0.1,
            "v_bias": torch.randn(lt, ht, d, generator=g, device="cuda") * 0.1}
    mapper = HeadwiseMapper.from_assignment(
        assign_layer=layer, assign_head=head, source_rope_theta=1e6, target_rope_theta=_target_thetas(case),
        windows=_windows(case), dtype=dtype, device="cuda", max_positions=16384, **maps)
    scale = torch.exp(torch.randn(d, generator=cpu) * 0.5).cuda()
    state = dict(case=case, mapper=mapper, maps=maps, layer=layer, head=head)
    if case["op"] == "page":
        state["position"] = 128
        state["page"] = _rows((2, case["source_layers"], case["tokens"], case["source_heads"], d), scale, dtype, g)
        return state
    lengths = _lengths(case)
    pages = [-(-n // PAGE) for n in lengths]
    need = sum(pages)
    source = PagedKVPool(layer_num=case["source_layers"], pages=2 * need, head_num=case["source_heads"],
                         head_dim=d, page_size=PAGE, dtype=dtype, device="cuda")
    for data in (source.k_data, source.v_data):
        data.copy_(_rows(data.shape, scale, dtype, g))
    target = PagedKVPool(layer_num=lt, pages=2 * need, head_num=ht, head_dim=d, page_size=PAGE, dtype=dtype,
                         device="cuda", fill="zeros")
    table = [torch.randperm(2 * need, generator=cpu)[:need] for _ in range(2)]  # source, target pages
    slots, spans, entry, token = [[], []], [], 0, 0
    for n, k in zip(lengths, pages):
        t = torch.arange(n)
        for side in range(2):
            slots[side].append(table[side][entry + t // PAGE] * PAGE + t % PAGE)
        spans.append(RequestSpan(token, entry * PAGE, n))
        entry, token = entry + k, token + n
    state.update(source=source, target=target, spans=spans, lengths=lengths,
                 source_slots=torch.cat(slots[0]).to(torch.int32).cuda(),
                 target_slots=torch.cat(slots[1]).cuda(), block_table=table[1].to(torch.int32).cuda())
    if case["op"] == "delivered":
        state["delivery"] = SelectedBlockDelivery(source, state["source_slots"], layers=mapper.source_layers,
                                                  block_tokens=BLOCK)
    return state


def prepare(case, seed):
    if case["op"] != "delta":
        return _prepare_handoff(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed)
    lead = (case["layers"], case["heads"])
    return dict(case=case,
                state=torch.randn(*lead, case["k"], case["v"], generator=g, device="cuda"),
                key=torch.randn(*lead, case["k"], case["kp"], generator=g, device="cuda") / math.sqrt(case["k"]),
                value=torch.randn(*lead, case["v"], case["vp"], generator=g, device="cuda") / math.sqrt(case["v"]))


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "delta":
        return {"state": transform_delta_state(state["state"], state["key"], state["value"])}
    if op == "page":
        return {"page": state["mapper"].map_page(state["page"], position_start=state["position"],
                                                 output_device="cuda")}
    mapper, target = state["mapper"], state["target"]
    if op == "batch":
        map_install_batch(mapper, state["source"], state["source_slots"], target, state["spans"],
                          block_table=state["block_table"], page_size=PAGE)
    elif op == "delivered":
        delivery = state["delivery"]
        for i, start in enumerate(range(0, case["tokens"], BLOCK)):
            delivery.deliver(i % 2, start, min(start + BLOCK, case["tokens"]))
            map_install_delivered(mapper, delivery, i % 2, target, block_table=state["block_table"],
                                  page_size=PAGE, prefix_length=case["tokens"])
    elif case["slots"]:
        map_install_block(mapper, state["source"], state["source_slots"], target, start=0, stop=case["tokens"],
                          target_indices=state["target_slots"])
    else:
        map_install_block(mapper, state["source"], state["source_slots"], target, start=0, stop=case["tokens"],
                          block_table=state["block_table"], page_size=PAGE)
    return {"k": target.k_data, "v": target.v_data}


def work(case):
    """Mapped rows written once, the distinct source rows, the fp32 maps and a token index read once."""
    if case["op"] == "delta":
        n = case["layers"] * case["heads"]
        k, v, kp, vp = case["k"], case["v"], case["kp"], case["vp"]
        return {"bytes": 4 * n * (k * v + k * kp + v * vp + kp * vp), "flops": 2 * n * (kp * k * v + kp * v * vp)}
    e, d, s = DTYPES[case["dtype"]].itemsize, case["head_dim"], case["support"]
    tokens = sum(_lengths(case))
    kept = sum(_kept(case, n, w) for n in _lengths(case) for w in _windows(case))
    maps = 2 * case["target_layers"] * case["target_heads"] * (s * d * d + d)
    rows = 2 * e * d * (kept * case["target_heads"] + _distinct_pairs(case) * tokens)
    return {"bytes": rows + 4 * maps + 8 * tokens, "flops": 4 * kept * case["target_heads"] * s * d * d}


def tolerance(case):
    # About four times what the outputs differ by from the 64-bit result: the
    # rounding to the pool's dtype (bf16, fp16), or fp32 sums.
    if case["op"] == "delta":
        return {"rel": 1.2e-6, "max": 2e-5}
    return {"bf16": {"rel": 6.6e-3, "max": 1.6e-2}, "fp16": {"rel": 8.5e-4, "max": 2e-3},
            "fp32": {"rel": 8e-7, "max": 2e-5}}[case["dtype"]]


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------


def _rotation(positions, d, theta):
    """cos and sin ``[tokens, 1, D/2]``; models compute the angle itself in fp32."""
    inverse = 1.0 / (theta ** (torch.arange(0, d, 2).float() / d))
    angle = (positions.float()[:, None] * inverse).double().cuda()
    return angle.cos()[:, None], angle.sin()[:, None]


def _map_layer(state, kind, rows, positions, layer, theta):
    """``rows(source layer) -> [n, Hs, D]`` mapped for one target layer: fp64 ``[n, Ht, D]``."""
    case, d = state["case"], state["case"]["head_dim"]
    half = d // 2
    source, head = state["layer"][layer], state["head"][layer]  # [Ht, s]
    x = []
    for k in range(case["support"]):
        x.append(torch.stack([rows(int(source[h, k]))[:, int(head[h, k])] for h in range(case["target_heads"])], 1))
    x = torch.stack(x, 2).double()  # [n, Ht, s, D]
    if kind == "k":
        c, s = (t[:, :, None] for t in _rotation(positions, d, 1e6))
        x1, x2 = x[..., :half], x[..., half:]
        x = torch.cat((x1 * c + x2 * s, x2 * c - x1 * s), -1)
    w = state["maps"][kind + "_weight"][layer].double()
    y = torch.bmm(x.flatten(2).transpose(0, 1).contiguous(), w).transpose(0, 1)
    y = y + state["maps"][kind + "_bias"][layer].double()
    if kind == "k":
        c, s = _rotation(positions, d, theta)
        y1, y2 = y[..., :half], y[..., half:]
        y = torch.cat((y1 * c - y2 * s, y2 * c + y1 * s), -1)
    return y


def exact(case, seed):
    state = prepare(case, seed)
    if case["op"] == "delta":
        u, a, b = (state[k].double().flatten(0, 1) for k in ("state", "key", "value"))
        out = torch.bmm(torch.bmm(a.transpose(1, 2).contiguous(), u), b)
        return {"state": out.unflatten(0, (case["layers"], case["heads"]))}
    thetas, windows = _target_thetas(case), _windows(case)
    if case["op"] == "page":
        page = state["page"]
        positions = torch.arange(case["tokens"]) + state["position"]
        return {"page": torch.stack([torch.stack([
            _map_layer(state, kind, lambda l, i=i: page[i, l], positions, layer, thetas[layer])
            for layer in range(case["target_layers"])]) for i, kind in enumerate("kv")])}
    out = {}
    for kind in "kv":
        pool = state["source"].k_data if kind == "k" else state["source"].v_data
        target = state["target"].k_data if kind == "k" else state["target"].v_data
        out[kind] = torch.zeros(target.shape, dtype=torch.float64, device="cuda")
        for layer in range(case["target_layers"]):
            begin = 0
            for n in state["lengths"]:
                first = n - _kept(case, n, windows[layer])
                take = slice(begin + first, begin + n)
                src, dst = state["source_slots"][take].long(), state["target_slots"][take]
                out[kind][layer][dst] = _map_layer(state, kind, lambda l: pool[l][src], torch.arange(first, n),
                                                   layer, thetas[layer])
                begin += n
    return out
