"""The dispatch workloads whose speed this repository answers for.

One pass is one call of the framework as a program makes it: an expert-parallel
dispatch of this GPU's share (eager, or the replay of a captured graph) in the
default mode, in which the caller's stream waits for the result, or the FP8 wire
codec.  The GPU is rank 0; the other ranks are the host threads of
``buffer.peers`` on the same pinned rings, started once and serving epoch after
epoch, as the processes of the other GPUs would.

A case is a dict of plain values:

``path``      "eager", "graph" (captured dispatch that derives its routing anew in
              every replay), "replay" (captured dispatch on a cached layout) or
              "codec" (``quantize_fp8`` followed by ``dequantize_fp8``)
``tokens``    tokens of every source rank; with ``ragged`` every source has another
              number of its own between a half and all of it
``hidden``, ``topk``, ``experts``, ``world``   the model's and the world's sizes
``fp8``       E4M3FN wire with one scale per token instead of BF16
``routing``   "uniform", or "hotspot": 20 % of the experts take 80 % of the routes
``expand``    expert-major rows, or one row per token ("unique" layout)
``fuse``      expand while receiving, or with the expand kernel behind the transport
``align``     alignment of every expert's rows, with zeroed gaps where it is above 1
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path("pcie-ep_amd").resolve())
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

from pcie_ep import HostStagedConfig, HostStagedEPBuffer  # noqa: E402
from pcie_ep.quantization import dequantize_fp8, quantize_fp8  # noqa: E402

_DEFAULTS = {"path": "eager", "tokens": 128, "ragged": False, "hidden": 7168, "topk": 8, "experts": 256, "world": 8, "fp8": False,
             "routing": "uniform", "expand": True, "fuse": True, "align": 1}


def _case(name: str | None = None, **values):
    case = dict(_DEFAULTS, **values)
    return dict({"name": name}, **case) if name else case


def listed():
    return [
        # One decoding step of a small batch: latency and launches, no bandwidth.
        _case("decode_16", tokens=16),
        # The same in a serving loop: graph with fresh routes in every replay, FP8 on the wire.
        _case("decode_graph_64_fp8", path="graph", tokens=64, fp8=True),
        # A decoding step whose rows go into a grouped matrix product with 128-row tiles.
        _case("decode_96_aligned", tokens=96, align=128),
        # A full decoding batch replayed on a fixed routing plan.
        _case("decode_replay_128", path="replay", tokens=128),
        # A chunk of a prefill, every source with another number of tokens.
        _case("chunk_700_ragged", tokens=700, ragged=True),
        # Two ranks that share the experts: half of what a rank sends stays on its GPU.
        _case("pair_1000", tokens=1000, world=2, experts=64, hidden=4096),
        # A narrow model on the FP8 wire whose rows are not whole wire vectors.
        _case("narrow_1536_fp8", tokens=1536, hidden=1000, experts=128, topk=4, fp8=True),
        # An ordinary model width, sixteen ranks.
        _case("wide_world_2048", tokens=2048, hidden=2048, world=16, experts=128, topk=6),
        # Receive without expansion on the FP8 wire: the consumer gathers by itself.
        _case("unique_1024_fp8", tokens=1024, fp8=True, expand=False),
        # Hotspot routing, expansion by a kernel of its own, aligned rows.
        _case("hotspot_3000_expand", tokens=3000, topk=4, routing="hotspot", fuse=False, align=16),
        # The largest prefill the configurations name.
        _case("prefill_8192", tokens=8192),
        # The wire codec on its own, both directions, on a prefill's rows.
        _case("codec_8192", path="codec", tokens=8192),
    ]


def _log_uniform(rng, low: int, high: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    path = rng.choice(["eager", "eager", "eager", "graph", "replay", "codec"])
    hidden = rng.choice([1024, 2048, 2880, 4096, 5120, 7168, 7168, rng.randrange(512, 4097)])
    tokens = _log_uniform(rng, 12, 6000)
    if path == "codec":
        return _case(path=path, tokens=tokens, hidden=hidden, fp8=True)
    world = rng.choice([2, 4, 8, 8, 8, 16])
    tokens = min(tokens, 40_000 // world)  # also with every hotspot on this rank no more than the largest listed case
    experts = world * rng.choice([8, 16, 32])
    topk = rng.choice([2, 4, 6, 8, 8])
    expand = rng.random() < 0.8
    return _case(path=path, tokens=tokens, ragged=rng.random() < 0.3, hidden=hidden, topk=topk, experts=experts, world=world,
                 fp8=rng.random() < 0.4, routing=rng.choice(["uniform", "uniform", "hotspot"]), expand=expand,
                 fuse=not expand or rng.random() < 0.75, align=rng.choice([1, 1, 16, 128]) if expand else 1)


class _State:
    """What a program keeps between dispatches; the pinned rings and the peers' threads go with it."""

    buffer = graph = None

    def __del__(self):
        if self.buffer is not None:
            self.graph = None
            self.buffer.close()


def _payload(generator, tokens: int, hidden: int, heavy_tail: bool, device):
    """Activations: normal, on the FP8 wire with one channel in a hundred fifty times as large."""
    x = torch.randn(tokens, hidden, generator=generator, device=device)
    if heavy_tail:
        x[:, torch.randperm(hidden, generator=generator, device=device)[: max(1, hidden // 100)]] *= 50.0
    return x.to(torch.bfloat16)


def _routes(generator, tokens: int, case, hot, device):
    """Distinct experts per token, softmax weights."""
    scores = torch.rand(tokens, case["experts"], generator=generator, device=device)
    if case["routing"] == "hotspot":
        # Sampling without replacement with weights: the largest of u ** (1 / w).
        weight = torch.full((case["experts"],), 0.2 / (case["experts"] - len(hot)), device=device)
        weight[hot] = 0.8 / len(hot)
        scores = scores.clamp_min(1e-30).log() / weight
    idx = scores.topk(case["topk"], dim=1).indices.contiguous()
    weights = torch.softmax(torch.randn(tokens, case["topk"], generator=generator, device=device), dim=1).contiguous()
    return idx, weights


def _tokens_of(case, rank: int) -> int:
    """Tokens of a source: all of ``tokens``, or, ragged, between a half and all (the same for every seed)."""
    if not case["ragged"]:
        return case["tokens"]
    return case["tokens"] - (rank * 7919 + case["tokens"] * 31) % (case["tokens"] // 2 + 1)


def prepare(case, seed):
    case = dict(_DEFAULTS, **case)
    device = torch.device("cuda")
    generator = torch.Generator(device=device).manual_seed(seed)
    state = _State()
    state.case = case
    if case["path"] == "codec":
        state.x = _payload(generator, case["tokens"], case["hidden"], True, device)
        return state
    hot = torch.randperm(case["experts"], generator=generator, device=device)[: max(1, case["experts"] // 5)]
    world = case["world"]
    graph = case["path"] in ("graph", "replay")
    config = HostStagedConfig(stage=7 if case["fp8"] else 6, wire_dtype="fp8_e4m3" if case["fp8"] else "bf16", channels=32,
                              fuse_receive_expand=case["fuse"], receive_expand_mode="pipelined" if case["fuse"] else "scalar",
                              enable_graph=graph, timeout_ms=60_000)
    buffer = state.buffer = HostStagedEPBuffer(num_max_tokens_per_rank=case["tokens"], hidden=case["hidden"], num_topk=case["topk"],
                                               num_experts=case["experts"], config=config, num_ranks=world, rank=0, peer_threads=4)
    for rank in range(world):
        tokens = _tokens_of(case, rank)
        x = _payload(generator, tokens, case["hidden"], case["fp8"], device)
        idx, weights = _routes(generator, tokens, case, hot, device)
        if rank == 0:
            state.x, state.idx, state.weights = x, idx, weights
        else:
            buffer.peers.set_source(rank, x, idx, weights)
    state.options = {"do_expand": case["expand"]}
    if case["align"] > 1:
        state.options.update(expert_alignment=case["align"], do_zero_padding=True)
    buffer.peers.start(1 << 30)
    buffer.peers.wait_staged()
    if case["path"] == "replay":
        handle = buffer.dispatch(state.x, state.idx, state.weights, **state.options)[3]
        state.graph = buffer.capture_dispatch(state.x, topk_weights=state.weights, handle=buffer.cache_layout(handle), **state.options)
    elif case["path"] == "graph":
        state.graph = buffer.capture_dispatch(state.x, state.idx, state.weights, **state.options)
    # Results have room for the worst routing and a dispatch writes the rows that its routes need: what is behind
    # them is zeroed once, in every result set that the buffer cycles through.
    for result in [run(state) for _ in range(1 if graph else config.output_pool_size)]:
        for name in ("x", "idx", "weights", "source"):
            result[name].zero_()
    torch.cuda.synchronize()
    return state


def run(state):
    if state.case["path"] == "codec":
        codes, scales = quantize_fp8(state.x)
        return {"codes": codes, "scales": scales, "x": dequantize_fp8(codes, scales)}
    if state.graph is not None:
        x, idx, weights, handle, _ = state.graph.replay()
    else:
        x, idx, weights, handle, _ = state.buffer.dispatch(state.x, state.idx, state.weights, **state.options)
    return {"x": x, "idx": idx, "weights": weights, "source": handle.source_meta, "expert_counts": handle.expert_counts,
            "expert_offsets": handle.expert_offsets, "source_offsets": handle.source_offsets, "error": handle.error}


def work(case):
    """Bytes a pass cannot do without: own rows read, rows for other ranks written once to the host ring, rows for this
    rank read once from it, result rows written, each with its routing.  Expected numbers of rows, from the distribution."""
    case = dict(_DEFAULTS, **case)
    hidden = case["hidden"]
    if case["path"] == "codec":
        return {"bytes": case["tokens"] * (hidden * (2 + 1 + 1 + 2) + 8), "flops": 4 * case["tokens"] * hidden}
    world, topk = case["world"], case["topk"]
    own = _tokens_of(case, 0)
    every = sum(_tokens_of(case, rank) for rank in range(world))
    hit = _hit_probability(case)
    received = (every - own) * hit
    local_experts = case["experts"] // world
    result_rows = every * topk / world if case["expand"] else every * hit
    if case["expand"] and case["align"] > 1:
        result_rows += local_experts * (case["align"] - 1) / 2
    wire = hidden * (1 if case["fp8"] else 2)
    bytes_ = own * hidden * 2 + own * wire + received * wire + result_rows * hidden * 2
    bytes_ += every * topk * 12 + result_rows * 36
    flops = 4 * (own + received) * hidden if case["fp8"] else 0
    return {"bytes": int(bytes_), "flops": int(flops)}


def _hit_probability(case) -> float:
    """Probability that a token has at least one of its experts on this rank (distinct experts, one rank's share of them)."""
    experts, local = case["experts"], case["experts"] // case["world"]
    miss = 1.0
    for taken in range(case["topk"]):
        miss *= max(0.0, (experts - local - taken) / (experts - taken))
    return 1.0 - miss


def tolerance(case):
    # Rows are moved, not computed with; the FP8 wire is defined byte for byte (round to nearest even, exact scales).
    return "exact"
