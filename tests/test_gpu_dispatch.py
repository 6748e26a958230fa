"""GPU parity of the full dispatch against the CPU oracle (bit-exact), through
the drop-in Python surface and therefore through the C ABI.

The matrix follows the reference's distributed correctness test
(tests/test_correctness.py:228-262): ring windows Q/L in {(1,1),(2,3),(3,2),
(256,256)}, route patterns random / local / multicast / hotspot / partial /
none, unique and expanded layouts, T in {0, 17, 33, 129 unequal}, alignments
1 / 8 / 16, with and without weights.  The seven other logical ranks are host
threads on the same pinned rings; what they receive from the GPU is captured
and compared too (TX parity).
"""

from __future__ import annotations

import ctypes as C
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from helpers import make_inputs, run_dispatch, verify_captured, verify_dispatch
from pcie_ep import _native

pytestmark = pytest.mark.gpu

WORLD, EXPERTS, TOPK = 8, 256, 8


def make_buffer(world=WORLD, rank=0, tmax=129, hidden=7168, topk=TOPK, experts=EXPERTS, **config):
    from pcie_ep import HostStagedConfig, HostStagedEPBuffer

    config.setdefault("timeout_ms", 5000)
    extra = {key: config.pop(key) for key in ("tx_waves", "rx_waves", "peer_threads", "worker_groups", "staging_numa_node", "comm_stream_cus") if key in config}
    return HostStagedEPBuffer(num_max_tokens_per_rank=tmax, hidden=hidden, num_topk=topk, num_experts=experts,
                              config=HostStagedConfig(**config), num_ranks=world, rank=rank, **extra)


def check_case(buffer, label, tokens, pattern="random", expand=True, alignment=1, weights=True, seed=7, capture=True,
               hidden=None, topk=None, experts=None, world=None, fp8=False, gaussian=False):
    world = world or buffer.num_ranks
    hidden, topk, experts = hidden or buffer.hidden, topk or buffer.num_topk, experts or buffer.num_experts
    print(f"case: {label} pattern={pattern} tokens={tokens} expand={expand} alignment={alignment} weights={weights} seed={seed}", flush=True)
    inputs = make_inputs(world, tokens, hidden, experts, topk, pattern, seed=seed, gaussian=gaussian)
    result, _ = run_dispatch(buffer, inputs, expand=expand, alignment=alignment, zero_padding=expand, with_weights=weights, capture=capture)
    summary = verify_dispatch(result, inputs, buffer.rank_idx, world, experts, topk, expand, alignment, expand, with_weights=weights, fp8_wire=fp8)
    if capture:
        verify_captured(buffer.peers, inputs, buffer.rank_idx, world, experts, topk, fp8_wire=fp8, with_weights=weights)
    return summary


def test_cpu_plumbing_configuration():
    """8 logical ranks, T=64, H=512 BF16 N(0,1), 16 experts (2 per rank), top-2,
    softmax weights, BF16 wire, expand on."""
    with make_buffer(tmax=64, hidden=512, topk=2, experts=16, channels=4) as buffer:
        summary = check_case(buffer, "plumbing", [64] * 8, gaussian=True, seed=1)
        assert summary["expanded"] > 0
        check_case(buffer, "plumbing-unique", [64] * 8, expand=False, gaussian=True, seed=1)


@pytest.mark.parametrize("slots,descriptors", [(1, 1), (2, 3), (3, 2), (256, 256)])
def test_ring_windows_and_patterns(slots, descriptors):
    """Tiny rings force slot reuse, descriptor credit waits and tail drains."""
    with make_buffer(payload_slots=slots, descriptor_slots=descriptors, channels=2, hidden=1024) as buffer:
        for pattern in ("random", "local", "multicast", "hotspot", "partial", "none"):
            for expand in (False, True):
                check_case(buffer, f"Q{slots}L{descriptors}", [17] * 8, pattern, expand)
        check_case(buffer, "empty", [0] * 8)
        check_case(buffer, "unequal", [0] + [max(1, 129 - r * 3) for r in range(1, 8)])
        check_case(buffer, "aligned16", [33] * 8, alignment=16)
        for i in range(6):
            check_case(buffer, "repeat", [3 + i % 5] * 8, expand=bool(i % 2), alignment=8, seed=100 + i)
        check_case(buffer, "no-weights", [5] * 8, "multicast", weights=False)


def test_full_hidden_32_channels():
    with make_buffer(channels=32) as buffer:
        check_case(buffer, "h7168", [129] * 8)
        check_case(buffer, "h7168-unique", [129] * 8, expand=False, seed=9)
        check_case(buffer, "h7168-gpu-empty", [0] + [129] * 7, seed=10)


def test_lopsided_send_receive_ratios():
    """A payload wavefront chooses its direction by the rows left to send and to
    receive: the extremes (nothing to receive, nothing to send, hundreds of rows
    one way against a handful the other way) must end like any other dispatch,
    also with rings that wrap many times and with the default launch shape."""
    with make_buffer(tmax=1500, channels=8, hidden=1024, payload_slots=16, descriptor_slots=16) as buffer:
        check_case(buffer, "send-only", [1500] + [0] * 7, capture=True)
        check_case(buffer, "receive-only", [0] + [1500] * 7)
        check_case(buffer, "send-heavy", [1500] + [3] * 7, capture=True, seed=21)
        check_case(buffer, "receive-heavy", [2] + [1500] * 7, capture=True, seed=22)
        check_case(buffer, "send-heavy-multicast", [1500] + [1] * 7, "multicast", expand=False, seed=23)
        check_case(buffer, "one-source", [40, 0, 0, 1500, 0, 0, 0, 0], seed=24)
    with make_buffer(tmax=1500, channels=8, hidden=1024, stage=7, wire_dtype="fp8_e4m3") as buffer:
        check_case(buffer, "fp8-send-heavy", [1500] + [5] * 7, capture=True, seed=25, fp8=True)
        check_case(buffer, "fp8-receive-heavy", [4] + [1500] * 7, seed=26, fp8=True)


def test_parity_while_other_traffic_saturates_the_link():
    """Ordering mistakes on the host link only show when it is busy (the hand-off
    litmus has the numbers): tiny rings, so that every slot, descriptor entry and
    ACK word is reused dozens of times per dispatch, both wires and both layouts,
    while kernel-driven copies keep both directions of the link saturated."""
    from pcie_ep import litmus

    with litmus.link_traffic():
        with make_buffer(tmax=700, channels=4, hidden=2048, payload_slots=2, descriptor_slots=1) as buffer:
            for repeat in range(4):
                check_case(buffer, "busy-link", [700, 650, 1, 700, 0, 333, 700, 700], expand=bool(repeat % 2), seed=40 + repeat)
        with make_buffer(tmax=300, channels=32, hidden=7168, payload_slots=3, descriptor_slots=2, stage=7, wire_dtype="fp8_e4m3") as buffer:
            for repeat in range(3):
                check_case(buffer, "busy-link-fp8", [300] * 8, "multicast" if repeat == 1 else "random", seed=50 + repeat, fp8=True)


@pytest.mark.parametrize("rank", [3, 7])
def test_other_local_rank(rank):
    with make_buffer(rank=rank, channels=3, hidden=512, payload_slots=4, descriptor_slots=4) as buffer:
        check_case(buffer, f"rank{rank}", [40] * 8)
        check_case(buffer, f"rank{rank}-unique", [40] * 8, expand=False, alignment=1)


@pytest.mark.parametrize("hidden", [129, 24, 8, 1])
def test_odd_hidden_sizes(hidden):
    """Rows that are not a multiple of 16 bytes take the scalar path."""
    with make_buffer(hidden=hidden, channels=2, payload_slots=3, descriptor_slots=3) as buffer:
        check_case(buffer, f"h{hidden}", [37] * 8)
        check_case(buffer, f"h{hidden}-unique", [37] * 8, expand=False)


def test_small_world_and_topk_shapes():
    with make_buffer(world=2, tmax=50, hidden=256, topk=4, experts=8, channels=1, payload_slots=2, descriptor_slots=2) as buffer:
        check_case(buffer, "p2", [50, 31])
    with make_buffer(world=16, tmax=20, hidden=64, topk=32, experts=64, channels=5) as buffer:
        check_case(buffer, "p16k32", [20] * 16)
        check_case(buffer, "p16k32-unique", [20] * 16, expand=False)
    with make_buffer(world=1, tmax=16, hidden=64, topk=2, experts=4, channels=2) as buffer:
        check_case(buffer, "p1", [16], capture=False)


def test_large_hidden_multi_pass():
    """A row longer than one register pass (16 KiB) is moved in several passes."""
    with make_buffer(hidden=12288, tmax=20, channels=2) as buffer:
        check_case(buffer, "h12288", [20] * 8)


def test_wave_counts():
    for tx_waves, rx_waves, helpers in ((1, 1, -1), (4, 6, 3), (2, 2, 192)):
        with make_buffer(hidden=512, channels=4, payload_slots=2, descriptor_slots=2, tx_waves=tx_waves, rx_waves=rx_waves,
                         worker_groups=helpers) as buffer:
            check_case(buffer, f"tx{tx_waves}rx{rx_waves}h{helpers}", [60] * 8)


def test_multi_chunk_layout_with_ragged_token_counts():
    """The layout kernel cuts tokens into chunks of 1024 (one workgroup each) and
    chains their totals; token counts that are not multiples of the chunk, differ
    per rank, or leave the last chunk nearly empty must give the same ordinals."""
    with make_buffer(tmax=3100, hidden=128, channels=7, payload_slots=32, descriptor_slots=16) as buffer:
        check_case(buffer, "chunks-ragged", [2500, 3100, 1025, 1, 0, 2048, 1023, 3000], capture=True)
        check_case(buffer, "chunks-1025", [1025] * 8, expand=False, seed=12)
        check_case(buffer, "chunks-partial", [3071] * 8, "partial", alignment=16, seed=13)


def test_many_experts_narrow_chunks():
    """With 4096 experts the per-chunk LDS tables only fit two wavefronts of
    tokens, so a few hundred tokens already span several chained chunks."""
    with make_buffer(world=16, tmax=700, hidden=64, topk=8, experts=4096, channels=3, payload_slots=8, descriptor_slots=8) as buffer:
        check_case(buffer, "e4096", [700, 129, 128, 127, 1, 0, 300, 650] * 2)
        check_case(buffer, "e4096-unique", [333] * 16, expand=False, seed=21)


def test_separate_expand_with_more_padding_work_than_rows():
    """Many local experts and a pool of a few rows: the stand-alone expand's grid is
    then sized by the alignment gaps it zeroes, not by the rows, and the workgroups
    beyond the pool must not touch it (128 local experts, a pool of 10 rows)."""
    with make_buffer(world=2, tmax=5, hidden=256, topk=4, experts=256, channels=3, payload_slots=4, descriptor_slots=4,
                     fuse_receive_expand=False, receive_expand_mode="scalar") as buffer:
        check_case(buffer, "wide-grid", [5, 3], alignment=16)
        check_case(buffer, "wide-grid-empty", [0, 0], alignment=2, seed=9)
    with make_buffer(world=1, tmax=1, hidden=2048, topk=1, experts=64, channels=2, fuse_receive_expand=False,
                     receive_expand_mode="scalar") as buffer:
        check_case(buffer, "wide-grid-one-row", [1], alignment=256, capture=False)


@pytest.mark.parametrize("fuse", [True, False])
@pytest.mark.parametrize("world,experts,alignment,hidden", [(8, 8, 256, 1024), (2, 128, 128, 264), (2, 130, 2, 129), (1, 200, 64, 2048), (8, 256, 128, 7168)])
def test_alignment_gaps_of_small_batches(world, experts, alignment, hidden, fuse):
    """A few tokens under a wide alignment: nearly every row is a gap row, dealt out over
    all wavefronts that clear them.  One local expert, exactly 64 (one per lane), 65 and
    200 (several groups of lanes), gaps of one row, scalar rows, and no token at all."""
    print(f"case: gaps world={world} experts={experts} alignment={alignment} hidden={hidden} fuse={fuse}", flush=True)
    mode = {} if fuse else {"fuse_receive_expand": False, "receive_expand_mode": "scalar"}
    with make_buffer(world=world, tmax=9, hidden=hidden, topk=4, experts=experts, channels=3, payload_slots=4, descriptor_slots=4, **mode) as buffer:
        check_case(buffer, "gaps", [9, 3, 1, 0, 2, 9, 5, 7][:world], alignment=alignment, capture=world > 1)
        check_case(buffer, "gaps-empty", [0] * world, alignment=alignment, seed=9, capture=world > 1)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hidden", [1, 7, 9, 15, 1000, 1001, 4095, 4097, 8190, 8197])
def test_ragged_rows(hidden, fp8):
    """Rows with something behind their whole vectors, on either wire: 1 to 15 bytes, rows shorter than a
    vector, the rest in the last item of a pass (4095, BF16; 8190, FP8) and alone in a pass of its own (4097 and 8197); expanded
    while receiving, by the expand kernel and not at all, with cleared gap rows between the rows; own
    tokens that start in the middle of a vector."""
    wire = {"stage": 7, "wire_dtype": "fp8_e4m3"} if fp8 else {}
    for mode in ({}, {"fuse_receive_expand": False, "receive_expand_mode": "scalar"}):
        with make_buffer(world=4, tmax=23, hidden=hidden, topk=4, experts=16, channels=2, payload_slots=3, descriptor_slots=3, **wire, **mode) as buffer:
            check_case(buffer, f"ragged-h{hidden}", [23, 17, 0, 5], alignment=16, fp8=fp8)
            if mode:
                continue
            check_case(buffer, f"ragged-h{hidden}-unique", [23, 17, 0, 5], expand=False, seed=9, fp8=fp8)
            inputs = make_inputs(4, [23, 1, 20, 23], hidden, 16, 4, "random", seed=10, gaussian=fp8)
            x, idx, weights = inputs[0]
            flat = torch.zeros(1 + x.numel(), dtype=torch.bfloat16, device="cuda")
            flat[1:] = x.flatten().cuda()
            if hidden % 8:
                shifted = [(flat[1:].view(x.shape), idx.cuda(), weights.cuda())] + inputs[1:]
                result, _ = run_dispatch(buffer, shifted, expand=True, capture=True)
                verify_dispatch(result, inputs, 0, 4, 16, 4, True, 1, False, fp8_wire=fp8)
                verify_captured(buffer.peers, inputs, 0, 4, 16, 4, fp8_wire=fp8)
                del result


@pytest.mark.parametrize("hidden,fp8", [(1000, True), (4095, True), (7169, True), (1001, False), (4095, False)])
def test_ragged_dispatches_fit_four_workgroups_to_a_compute_unit(hidden, fp8):
    """`comm_stream_cus` is admitted by what a unit holds: a dispatch of ragged rows whose workgroups fit 32 units only
    at four to a unit is accepted there, and runs."""
    wire = {"stage": 7, "wire_dtype": "fp8_e4m3"} if fp8 else {}
    with make_buffer(world=4, tmax=40, hidden=hidden, topk=4, experts=16, channels=16, comm_stream_cus=32, **wire) as buffer:
        needed, resident = buffer.runtime.transport_residency(32)
        assert 3 * 32 < needed <= resident
        check_case(buffer, f"ragged-on-32-units-h{hidden}", [40, 9, 40, 33], alignment=16, fp8=fp8)


@pytest.mark.parametrize("experts,hidden,fp8", [(640, 1001, False), (704, 1000, True), (704, 4095, False)])
def test_ragged_dispatches_of_many_experts_fit_four_workgroups_to_a_compute_unit(experts, hidden, fp8):
    """The same where the layout tables of the one-launch prologue fill most of a workgroup's share of the LDS."""
    wire = {"stage": 7, "wire_dtype": "fp8_e4m3"} if fp8 else {}
    with make_buffer(world=16, tmax=40, hidden=hidden, topk=4, experts=experts, channels=32, comm_stream_cus=40, **wire) as buffer:
        needed, resident = buffer.runtime.transport_residency(40)
        assert 3 * 40 < needed <= resident
        check_case(buffer, f"ragged-on-40-units-e{experts}-h{hidden}", [40, 9, 40, 33] + [3] * 12, fp8=fp8)


@pytest.mark.parametrize("hidden,topk,fp8", [(1312, 8, False), (1313, 8, False), (4096, 8, True), (4095, 8, True), (4097, 8, True), (64, 13, False), (64, 14, True)])
def test_short_rows_are_received_in_pairs(hidden, topk, fp8):
    """Both sides of the line up to which a wavefront takes two rows at a time: longest rows, ragged ones that
    fill the last register of a pair's half, and the largest metadata; both layouts.  A wavefront claims its share of the
    tickets that are there, so few wavefronts make the claims large: two of them take claims of eight (pairs of neighbouring
    slots, of two channels and of two sources, and the odd last one) from rings of 64 slots, and what rings of one slot
    hold, where the second row of a claim comes only after the first was acknowledged; four are the smallest ordinary workgroup."""
    wire = {"stage": 7, "wire_dtype": "fp8_e4m3"} if fp8 else {}
    for channels, slots, waves in ((16, 64, 1), (2, 1, 1), (3, 5, 2)):
        with make_buffer(tmax=200, hidden=hidden, topk=topk, channels=channels, payload_slots=slots, descriptor_slots=slots, worker_groups=1,
                         tx_waves=waves, rx_waves=waves, **wire) as buffer:
            tokens = [200] * 8 if slots > 1 else [40, 7, 40, 0, 1, 33, 40, 12]
            check_case(buffer, f"pairs-h{hidden}-k{topk}-s{slots}", tokens, alignment=16, fp8=fp8)
            check_case(buffer, f"pairs-h{hidden}-k{topk}-s{slots}-unique", tokens, expand=False, seed=9, fp8=fp8)


@pytest.mark.parametrize("world,hidden,slots,descriptors,fp8", [(8, 1024, 64, 64, False), (2, 4096, 1, 1, False), (4, 1001, 2, 3, False), (8, 1000, 64, 2, True),
                                                                (8, 7168, 3, 64, True)])
def test_first_rows_of_a_channel_go_ahead_of_the_plan(world, hidden, slots, descriptors, fp8):
    """Up to three tokens of every channel are transmitted without a ticket, where the dispatch before has drained the
    rings: as many as channels, one less and one more, two and three times as many and beyond; tokens among them that
    go nowhere or stay on this rank; rings that hold fewer; a dispatch too large for it (6 MB of rows to come) between.
    Exactly those rows are counted as such, and none behind an epoch that is not known to have drained the rings."""
    wire = {"stage": 7, "wire_dtype": "fp8_e4m3"} if fp8 else {}
    channels = 4
    with make_buffer(world=world, tmax=1000, hidden=hidden, channels=channels, payload_slots=slots, descriptor_slots=descriptors, **wire) as buffer:
        sizes, shape = buffer.runtime.sizes, [C.c_int32() for _ in range(4)]
        _native.check(_native.library().pcie_ep_profile_shape(buffer.runtime.handle, *(C.byref(value) for value in shape)))
        row_bytes = (int(sizes.payload_bytes) + 15) // 16 * 16 + int(sizes.meta_bytes)
        early = channels * min(3, shape[3].value // (2 * channels), (544 << 10) // (channels * row_bytes), slots, descriptors)
        assert early >= channels
        epoch = 0
        for repeat, own in enumerate((3, 4, 5, 8, 13, 40, 1000, 1, 0, 12)):
            tokens = [own] + [max(0, own - 3 * r) for r in range(1, world)]
            too_large = (world - 1) * own * row_bytes > 6 << 20
            assert too_large == (own == 1000)
            for pattern in ("random", "partial", "local", "multicast")[: 1 if too_large else 4]:
                by_hand = repeat in (3, 9) and pattern == "partial"
                if by_hand:
                    buffer.runtime.set_test_epoch(epoch)
                check_case(buffer, f"first-rows-w{world}-h{hidden}", tokens, pattern, expand=repeat % 2 == 0, seed=60 + repeat, fp8=fp8)
                epoch += 1
                idx = make_inputs(world, tokens, hidden, EXPERTS, TOPK, pattern, seed=60 + repeat)[0][1]
                remote = int(((idx >= 0) & (idx // (EXPERTS // world) != 0)).any(dim=1)[:early].sum())
                assert buffer.runtime.early_rows() == (0 if too_large or by_hand else remote, epoch)


def test_profiling_records_count_every_row_of_a_pair():
    """The per-role records (profiling build, a process of its own): rows received and transmitted equal the
    dispatch's statistics, and fewer moves than rows: pairs are taken."""
    program = """
import sys
sys.path[:0] = ["tests", "pcie-ep_amd", "."]
import torch
from helpers import make_inputs, run_dispatch
from test_gpu_dispatch import make_buffer
from pcie_ep import profiling
with make_buffer(tmax=200, hidden=64, channels=4, payload_slots=64, descriptor_slots=64, worker_groups=1, tx_waves=1, rx_waves=1) as buffer:
    result, _ = run_dispatch(buffer, make_inputs(8, [200] * 8, 64, 256, 8))
    records = profiling.read(buffer.runtime)["workers"]
    total = {name: int(records[:, profiling.WORKER.index(name)].sum()) for name in ("items", "tx_rows", "rx_rows")}
    stats = result[3].stats.cpu().tolist()
    assert (total["tx_rows"], total["rx_rows"]) == (stats[0], stats[1]), (total, stats)
    assert total["items"] < 0.75 * stats[1] + stats[0], (total, stats)
    print("counted", total, flush=True)
"""
    run = subprocess.run([sys.executable, "-u", "-c", program], cwd=Path(__file__).resolve().parents[1], env=dict(os.environ, PCIE_EP_PROFILING="1"),
                         capture_output=True, text=True, timeout=100)
    print(run.stdout, run.stderr, flush=True)
    assert run.returncode == 0 and "counted" in run.stdout


def test_numa_bound_staging_segments():
    """The pinned segments can be bound to a NUMA node (the far-node staging of the
    cached-replay configuration); node 0 exists on every box.  Results do not change."""
    from pcie_ep import _native

    node = _native.library().pcie_ep_device_numa_node(0)
    print(f"case: staging on NUMA node 0 (the GPU reports node {node})", flush=True)
    assert node >= -1
    with make_buffer(hidden=1024, channels=4, staging_numa_node=0) as buffer:
        check_case(buffer, "numa0", [65] * 8)
    with pytest.raises(RuntimeError, match="set_mempolicy"):
        make_buffer(hidden=64, channels=1, staging_numa_node=900)


def test_invalid_routes_raise_code_two():
    """Duplicate, < -1 and >= E ids are terminal error 2 (tests/test_integration.py:222-260)."""
    for bad in ([3, 3], [-2, 1], [256, 1]):
        with make_buffer(hidden=64, topk=2, channels=2, timeout_ms=500) as buffer:
            inputs = make_inputs(8, [4] * 8, 64, 256, 2, seed=3)
            inputs[0][1][1] = torch.tensor(bad)
            x, idx, weights = (item.cuda() for item in inputs[0])
            result = buffer.dispatch(x, idx, weights, do_expand=True)
            with pytest.raises(RuntimeError, match="GPU error"):
                buffer.check_errors()
            assert int(result[3].error[0].cpu()) == 2
            with pytest.raises(RuntimeError, match="failed"):
                buffer.dispatch(x, idx, weights, do_expand=True)
