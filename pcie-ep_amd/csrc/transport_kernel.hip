// Channel transport kernel: TX control (+ guardian), RX control (+ receive
// prefixes), TX payload workers and RX/scatter workers, all as single
// wavefronts with their own role.
//
// Replaces advanced_transport_pipelined and its roles
// (csrc/kernels/host_staged/fused_receive.cuh:333-360;
// advanced_dispatch.cuh:287-477 tx_control, :479-625 rx_control, :627-689
// tx_worker; fused_receive.cuh:199-305 producer/consumer) and, for the unique
// layout, advanced_transport (advanced_dispatch.cuh:919-958).
//
// Design for MI355X (64-lane wavefronts, 8 XCDs):
//  * A payload worker is ONE wavefront that owns a whole row: its up to
//    14 x 16-byte loads per lane (896 vectors of a 14 336-byte BF16 row) leave
//    kReadWindow at a time (see there), the row lives in registers, and the same
//    wavefront stores it to every destination expert row.  The staged row is read once; there is no
//    LDS tile and no producer/consumer hand-off (the reference stages through
//    shared memory with 3+3 warps per ticket).
//  * Control wavefronts work on 64 candidates at a time with ballots: TX control
//    derives ring slots and per-destination descriptor ordinals for 64 tokens
//    from popcounts of ballots; RX control probes up to 64/P descriptors per
//    source per iteration instead of one source per iteration.
//  * Work is handed out through two global ticket rings in device memory (one
//    for TX, one for RX).  Control wavefronts only reserve and hand out tickets;
//    the payload workgroups hold payload wavefronts, which claim tickets of ANY
//    channel, so every channel's rows are moved by all payload XCDs.  This matters
//    because the XCDs get unequal shares of the host link: with workers bound to
//    their channel's workgroup, equal work finished in 8.8 ms on the best XCD and
//    12.8 ms on the worst.  It also decouples the bytes in flight (worker
//    wavefronts x row size), which set the latency of every control-path read,
//    from the number of channels.
//  * Which workgroup runs on which XCD is chosen (workgroup id = row * 8 + XCD):
//    two XCDs hold the control class - the epoch begin and the layout chunks of the
//    prologue when it rides in this launch, and per pair of channels one workgroup
//    of transmit controls and one of receive controls, on different XCDs - and six
//    hold the payload class (payload and local-bypass workgroups).  A host read
//    stays in its XCD's memory queues for as long as the link needs for the bytes
//    requested before it, and every other memory operation through that XCD waits
//    behind it: controls that shared an XCD with payload wavefronts saw their
//    tickets and flags arrive tens of microseconds late.
//  * With the prologue in the same launch (one launch per dispatch), the roles
//    here start with the queues not yet reset: one thread per workgroup waits for
//    the epoch begin's word before its role touches them; rows to transmit and the
//    local bypass wait for the plan's word, the transmit controls (which hand out
//    tickets straight from the routes) and the receive side do not.
//  * Workers publish their own descriptors and payload ACKs when their own stores /
//    loads have completed (see settle); control wavefronts only reserve and hand out.
//  * The first tokens of every channel are copied to their slots without ticket or
//    plan, before the first received rows are requested (see direct_row).
//  * A payload wavefront has no fixed direction: before every row it takes the
//    direction that needs it, in proportion to the rows left to send and to
//    receive, so that the writes are spread thinly over the whole dispatch (row
//    writes compete with the read REQUESTS for the upstream half of the link) and
//    both directions end together whatever the routing's send/receive ratio is.
//  * Vector memory operations complete in order: wherever several host words are
//    wanted at once (count mailboxes, ACK arrays), their addresses are computed
//    first and the loads issued in one run, with no other load in between.
//  * Every read from host memory is a whole 16-byte vector per lane (payload, slot
//    metadata, descriptor entries) or a packed word array (ACKs): small scattered
//    reads cost the host link far more than their bytes.
//  * The workgroups after the payload workgroups do the local bypass (own tokens
//    routed to own experts: advanced_copy_local_tokens, advanced_layout.cuh:217-248)
//    and the zeroing of the alignment gaps (:250-265) as soon as the receive
//    prefixes are known, token by token from a shared counter.  That work only
//    touches HBM and runs on compute units the transport leaves idle, so it hides
//    completely behind the host link.  The last role wavefront to end reduces the
//    per-channel statistics (:267-283).  The dispatch needs no kernel after this one.
#include "device_common.h"
#include "launch.h"
#include "prologue_body.h"
#include "row_codec.h"

namespace pcie_ep {

namespace {

constexpr int kScratchDwords = kReceiveScratchDwords;  // per wavefront: slot metadata records (of one or kMaxReceiveBatch rows)
// What a payload wavefront owes the other ends (see Owed): slot ACKs (address, token), then a transmitted row's
// channel, slot, token and descriptor ordinal per endpoint; behind them the words of a direct row's ticket, its scale
// and the wavefront's counters.
constexpr int kTicketWords = int(sizeof(TxEntry) / 4);
constexpr int kOwedRow = 4 * kMaxReceiveBatch, kOwedDescriptors = kOwedRow + 4, kDirectTicket = kOwedDescriptors + kMaxEndpoints;
constexpr int kDirectScale = kDirectTicket + kTicketWords, kOwedCounts = kDirectScale + 1, kOwedDwords = kOwedCounts + 7;

// One of these per wavefront of the workgroup, in the LDS that the launch asks for (transport_lds_bytes), where a workgroup of
// the prologue has its tables.  Sized for the largest workgroup and beside those tables, they took the ragged kernels from
// four workgroups on a compute unit to three from 640 experts on (16 ranks, 32 channels).
struct WaveScratch {
    uint32_t words[kScratchDwords];
    uint32_t owed[kOwedDwords];
};
static_assert(kOwedCounts + 5 <= kOwedDwords && sizeof(WaveScratch) % 16 == 0, "room for every counter, vectors on 16-byte boundaries");

// Local time only: payload workers never scan the host abort flags themselves
// (hundreds of wavefronts doing so would be PCIe traffic of their own); the
// channel's guardian does and raises the channel's abort word.
struct Deadline {
    uint64_t start;
    __device__ explicit Deadline(uint64_t begin) : start(begin) {}
    __device__ __forceinline__ bool expired(const DeviceState& state) const { return now_ticks() - start > progress_timeout_ticks(state); }
};

__device__ __forceinline__ bool aborted(TransportQueues& q) { return device_load(&q.abort.value) != 0; }
__device__ __forceinline__ void raise_abort(TransportQueues& q) { device_store(&q.abort.value, 1u); }

// Prologue inside this launch: a role may touch the queues and the diagnostics once
// the epoch begin has cleared them.  One thread per workgroup polls (hundreds of
// wavefronts polling one word would slow down the very stores they wait for).
// Bounded: an epoch begin that never runs ends the role.
__device__ __forceinline__ bool wait_for_begin(const DeviceState& state, TransportQueues& q) {
    const uint32_t tag = epoch_flag(dispatch_epoch(state));
    const uint64_t start = now_ticks();
    // The word cannot be there in the first microsecond: stay off the memory the clearing goes to.
    __builtin_amdgcn_s_sleep(48);
    while (device_load(&q.begun.value) != tag) {
        if (now_ticks() - start > state.timeout_ticks) return false;
        __builtin_amdgcn_s_sleep(16);
    }
    return true;
}
// ... and read the route plan, or publish a row, once the epoch's verdict is there and every chunk's part of the plan
// is in memory.  The own counts may then still be on their way to the peers: a descriptor can become visible
// before `counts_ready`.  No receiver is misled by that.  A descriptor carries its epoch and ordinal, a slot its
// epoch and token; a transport kernel on the other end copies such a row only behind its gate, when the counts of all sources have been
// requested, and places it by prefixes made of them; a relay worker and an emulated peer take up an epoch when they see its
// `counts_ready`, and only then look at its descriptors.  False when the prologue failed (abort) or never finished (timeout, recorded as
// a ring-progress error).
__device__ __forceinline__ bool wait_for_plan(const DeviceState& state, TransportQueues& q, int lane) {
    if (!state.fused) return true;
    const uint32_t tag = epoch_flag(dispatch_epoch(state));
    const uint64_t start = now_ticks();
    while (true) {
        int verdict = 0;
        if (lane == 0) {
            if (device_load(&q.plan_ready.value) == tag) verdict = 1;
            else if (aborted(q)) verdict = -1;
            else if (now_ticks() - start > progress_timeout_ticks(state)) {
                record_error(state, kErrRingProgressWait);
                raise_abort(q);
                verdict = -1;
            }
        }
        verdict = broadcast_first(verdict);
        if (verdict) return verdict > 0;
        backoff();
    }
}

// Producer side: reserve `count` consecutive tickets (one fetch-add per wavefront).
__device__ __forceinline__ int reserve_tickets(QueueCounter& tail, int count, int lane) {
    uint32_t base = 0;
    if (lane == 0) base = device_add(&tail.value, uint32_t(count));
    return broadcast_first(int(base));
}
__device__ __forceinline__ bool ring_entry_free(const uint64_t* taken, uint64_t epoch, int ticket) {
    const int previous = ticket - kRing;
    return previous < 0 || device_load(taken + previous % kRing) == sequence(epoch, previous);
}

// Consumer side: claim the next tickets, then wait until an entry is complete.
// Returns 1 when available, -1 when there is no such ticket or on abort.
__device__ __forceinline__ int claim_tickets(QueueCounter& head, int count, int lane) {
    uint32_t ticket = 0;
    if (lane == 0) ticket = device_add(&head.value, uint32_t(count));
    return broadcast_first(int(ticket));
}
template <typename BeforeWaiting>
__device__ __forceinline__ int wait_ticket(const DeviceState& state, TransportQueues& q, const uint64_t* ready, QueueCounter& head, int ticket,
                                  uint64_t epoch, int lane, const Deadline& deadline, BeforeWaiting before_waiting) {
    while (true) {
        int action = 0;
        if (lane == 0) {
            if (aborted(q)) action = -1;
            else if (device_load(ready + ticket % kRing) == sequence(epoch, ticket)) action = 1;
            else {
                const int limit = device_load(&head.total), direct = device_load(&head.direct);
                if (limit >= 0 && ticket >= limit - direct) action = -1;
                else if (deadline.expired(state)) {
                    record_error(state, kErrRingProgressWait);
                    raise_abort(q);
                    action = -1;
                }
            }
        }
        action = broadcast_first(action);
        if (action) return action;
        before_waiting();
        backoff();
    }
}

// ---------------------------------------------------------------------------------------
// Receive prefixes (advanced_layout.cuh:94-195).  One wavefront of the grid is
// elected by a device-scope CAS; it waits for every source's counts_ready,
// folds the mailboxes in rank order and publishes a generation-valued READY.
// ---------------------------------------------------------------------------------------
// The producer's first look at every source's counts_ready (lane r: rank r), issued by the
// kernel's entry code before the role is let in; see RxFirstPoll.
struct PrefixFirstLook {
    uint64_t word;
    bool issued;
};
__device__ __forceinline__ PrefixFirstLook prefix_first_look(const DeviceState& state, int lane) {
    const SegmentLayout& z = state.z;
    const int ranks = z.dims.num_ranks;
    PrefixFirstLook look{0, true};
    if (lane < ranks && !(state.fused != 0 && lane == state.local_rank))
        look.word = host_load_global(signal_at(state.seg[lane], z.counts_ready_offset));
    return look;
}

__device__ __forceinline__ bool compute_receive_prefixes(const DeviceState& state, int lane, PrefixFirstLook entry_look PCIE_EP_PROFILE(, RoleProfile& profile)) {
    const SegmentLayout& z = state.z;
    const int ranks = z.dims.num_ranks, local = z.local_experts, channels = z.dims.channels;
    const int me = state.local_rank;
    const uint64_t epoch = dispatch_epoch(state);
    const uint64_t start = now_ticks();
    HealthCheck health(state, start);
    PCIE_EP_PROFILE(profile.first(kProfilePrefixEnterNs);)
    if (lane == 0) {
        state.prefix_tx_timestamps_ns[0] = ticks_to_ns(state, start);
        test_delay(state.prefix_delay);
    }
    // This runs while the payload wavefronts already stream rows, so it keeps to
    // the discipline of the hot path: host words are read with the system-scope
    // policy (never from a GPU cache, so no invalidate is needed), results are
    // written through to device memory (so no cache write-back is needed), and
    // ordering is by waiting for this wavefront's own operations.  A cache
    // write-back here would have to flush the rows the scatter is writing.
    // Once every source's counts are ready, every mailbox word this wavefront needs
    // is requested before the first one is used: one round trip over the host link
    // instead of one per group.  Vector memory operations complete in order, so
    // nothing else may be loaded in between - not even a segment's base address out of the kernel arguments:
    // waiting for that load would wait for every host word requested before it.
    // The addresses are therefore computed first (lane r holds the base of rank
    // r's segment and hands it out by lane shuffle) - before the wait for the
    // sources, where it costs nothing - and the loads follow in one run.
    const char* const lane_segment = state.seg[lane < ranks ? lane : 0];
    // Prologue in the same launch: the own counts are taken from the route plan in
    // device memory once the leader has announced it, not from the own mailbox in
    // host memory; the other sources' words are requested before that wait.
    const bool own_from_plan = state.fused != 0;
    // The first look at every source's counts_ready is requested now; its value is
    // used after the address arithmetic below, which so runs inside its round trip.
    uint64_t first_look = entry_look.word;
    if (!entry_look.issued && lane < ranks && !(own_from_plan && lane == me))
        first_look = host_load_global(signal_at(const_cast<char*>(lane_segment), z.counts_ready_offset));
    const auto segment_of = [&](int rank) {
        const uint64_t bits = reinterpret_cast<uint64_t>(lane_segment);
        return reinterpret_cast<char*>(uint64_t(uint32_t(__shfl(int(uint32_t(bits)), rank))) | uint64_t(uint32_t(__shfl(int(uint32_t(bits >> 32)), rank))) << 32);
    };
    constexpr int kExpectedPerLane = kMaxChannels * kMaxRanks / kWave;
    const int32_t* expected_address[kExpectedPerLane];
#pragma unroll
    for (int i = 0; i < kExpectedPerLane; ++i) {
        const int index = lane + i * kWave;
        const bool valid = index < channels * ranks;
        char* segment = segment_of(valid ? index % ranks : 0);
        expected_address[i] = valid ? mailbox_at(z, segment, me) + 1 + local + index / ranks : nullptr;
        if (own_from_plan && valid && index % ranks == me) expected_address[i] = state.plan_chan_counts + (index / ranks) * ranks + me;
    }
    const int32_t* first_address[kMaxRanks];
#pragma unroll
    for (int source = 0; source < kMaxRanks; ++source) {
        char* segment = segment_of(source < ranks ? source : 0);
        first_address[source] = (source < ranks && lane < local) ? mailbox_at(z, segment, me) + 1 + lane : nullptr;
        if (own_from_plan && source == me && lane < local) first_address[source] = state.plan_counts + ranks + me * local + lane;
    }
    const int32_t* unique_address = lane < ranks ? mailbox_at(z, const_cast<char*>(lane_segment), me) : nullptr;
    if (own_from_plan && lane == me) unique_address = state.plan_counts + me;
    // All sources are polled in parallel, one lane each.
    bool ready = lane >= ranks || (own_from_plan && lane == me) || first_look == epoch;
    while (true) {
        if (__all(ready)) break;
        if (!ready) ready = host_load_global(signal_at(const_cast<char*>(lane_segment), z.counts_ready_offset)) == epoch;
        if (__all(ready)) break;
        if (health.poll(state, lane)) {
            if (lane == 0) record_error(state, kErrCountsReadyWait);
            return false;
        }
        // Nothing will come of this dispatch when the prologue of the same launch has failed.
        if (state.fused && broadcast_first(aborted(*state.queues) ? 1 : 0)) return false;
        backoff();
    }
    wait_memory_ops();
    compiler_barrier();
    PCIE_EP_PROFILE(profile.first(kProfilePrefixCountsReadyNs);)
    // Host words first (every word of the other sources, in one run) ...
    int unique = 0;
    if (unique_address && !(own_from_plan && lane == me)) unique = host_field_load_global(unique_address);
    int expected_values[kExpectedPerLane];
#pragma unroll
    for (int i = 0; i < kExpectedPerLane; ++i)
        expected_values[i] = (expected_address[i] && !(own_from_plan && (lane + i * kWave) % ranks == me)) ? host_field_load_global(expected_address[i]) : 0;
    int first_counts[kMaxRanks];
#pragma unroll
    for (int source = 0; source < kMaxRanks; ++source)
        first_counts[source] = (first_address[source] && !(own_from_plan && source == me)) ? host_field_load_global(first_address[source]) : 0;
    // The reads are on the link (requests leave in issue order): the receive side
    // may now flood it with row reads without delaying these few words.
    compiler_barrier();
    if (lane == 0) device_store(state.receive_prefix_state, epoch | kPrefixRequested);
    compiler_barrier();
    if (own_from_plan) {
        // ... then the own words, out of device memory, once the plan is there.
        if (!wait_for_plan(state, *state.queues, lane)) return false;
        if (lane == me) unique = device_load_global(unique_address);
#pragma unroll
        for (int i = 0; i < kExpectedPerLane; ++i)
            if (expected_address[i] && (lane + i * kWave) % ranks == me) expected_values[i] = device_load_global(expected_address[i]);
#pragma unroll
        for (int source = 0; source < kMaxRanks; ++source)
            if (source == me && first_address[source]) first_counts[source] = device_load_global(first_address[source]);
    }
    // Per-source unique counts -> source_offsets (lane = source).
    int inclusive = unique;
    PCIE_EP_PROFILE(if (__builtin_amdgcn_readfirstlane(inclusive) >= 0) profile.first(kProfilePrefixMailboxNs);)  // the first use of a mailbox word: the reads have returned
    for (int offset = 1; offset < kMaxRanks; offset <<= 1) {
        const int other = __shfl_up(inclusive, offset);
        if (lane >= offset) inclusive += other;
    }
    if (lane < ranks) device_store(state.source_offsets + lane + 1, inclusive);
    if (lane == 0) device_store(state.source_offsets, 0);
    const int total_unique = __shfl(inclusive, ranks - 1);
    // Expert branches: lane = local expert; all sources' loads are issued first.
    int carry_offset = 0;
    int64_t expanded_total = 0;
    for (int begin = 0; begin < local; begin += kWave) {
        const int expert = begin + lane;
        int counts[kMaxRanks];
#pragma unroll
        for (int source = 0; source < kMaxRanks; ++source) {
            if (begin == 0) counts[source] = first_counts[source];
            else if (own_from_plan && source == me) counts[source] = expert < local ? device_load(state.plan_counts + ranks + me * local + expert) : 0;
            else counts[source] = (source < ranks && expert < local) ? host_field_load(mailbox_at(z, state.seg[source], me) + 1 + expert) : 0;
        }
        int running = 0;
#pragma unroll
        for (int source = 0; source < kMaxRanks; ++source) {
            if (source < ranks && expert < local) device_store(state.source_expert_prefix + source * local + expert, running);
            running += counts[source];
        }
        const int padded = (running + state.alignment - 1) / state.alignment * state.alignment;
        int scan = padded;
        for (int offset = 1; offset < kWave; offset <<= 1) {
            const int other = __shfl_up(scan, offset);
            if (lane >= offset) scan += other;
        }
        const int exclusive = carry_offset + scan - padded;
        if (expert < local) {
            device_store(state.expert_counts + expert, running);
            device_store(state.expert_offsets + expert, exclusive);
            device_store(state.expert_prefix + expert, exclusive + running);
            if (expert == local - 1) device_store(state.expert_offsets + local, exclusive + padded);
        }
        carry_offset += __shfl(scan, kWave - 1);
        int sum = running;
        for (int offset = 32; offset > 0; offset >>= 1) sum += __shfl_xor(sum, offset);
        expanded_total += sum;
    }
    // Expected tokens per (channel, source) for this receiver.
#pragma unroll
    for (int i = 0; i < kExpectedPerLane; ++i) {
        const int index = lane + i * kWave;
        if (index < channels * ranks) device_store(state.expected_receive_counts + index, expected_values[i]);
    }
    const int own_unique = __shfl(unique, me);
    if (lane == 0) {
        device_store(state.unique_count, int64_t(total_unique));
        device_store(state.expanded_count, expanded_total);
        // Receive tickets of this dispatch: every unique row of a remote source.
        device_store(&state.queues->rx_head.total, total_unique - own_unique);
    }
    return true;
}

// A source may overwrite its count mailbox for the next epoch once this rank has
// said so.  Every lane has its counts in registers by now (the loads above were
// waited for, wave-wide), so the ACK needs no fence (advanced_layout.cuh:91-93).
__device__ __forceinline__ void acknowledge_counts(const DeviceState& state, int lane) {
    const SegmentLayout& z = state.z;
    wait_memory_ops();
    if (lane < z.dims.num_ranks && lane != state.local_rank && lane != state.counts_ack_skip_source)
        host_field_store(signal_at(state.seg[lane], z.counts_consumed_offset, state.local_rank), dispatch_epoch(state));
}

__device__ __forceinline__ void produce_receive_prefixes(const DeviceState& state, int lane, PrefixFirstLook entry_look PCIE_EP_PROFILE(, RoleProfile& profile));

// One wavefront of the grid (the first RX control to get there) computes the
// receive prefixes; nobody waits here.
__device__ __forceinline__ void elect_receive_prefixes(const DeviceState& state, int lane PCIE_EP_PROFILE(, RoleProfile& profile)) {
    const uint64_t epoch = dispatch_epoch(state);
    int claimed = 0;
    if (lane == 0) {
        unsigned long long expected = 0;
        claimed = atomicCAS(reinterpret_cast<unsigned long long*>(state.receive_prefix_state), expected, epoch) == 0ull;
    }
    if (!broadcast_first(claimed)) return;
    produce_receive_prefixes(state, lane, PrefixFirstLook{0, false} PCIE_EP_PROFILE(, profile));
}

// With payload workgroups of their own, the control workgroups have wavefronts to
// spare (a third one exists with three or more payload wavefronts per workgroup):
// the receive prefixes are then produced by that one (wavefront 2 of
// channel 0's workgroup) and no RX control is held up by them - the channel of an
// elected RX control starts to receive a prefix computation late.
__device__ __forceinline__ bool dedicated_prefix_producer(const DeviceState& state) { return state.worker_groups > 0 && state.tx_waves + state.rx_waves >= 3; }

__device__ __forceinline__ void receive_prefix_role(const DeviceState& state, int lane, PrefixFirstLook entry_look) {
    PCIE_EP_PROFILE(RoleProfile profile(state.clock_khz);)
    if (lane == 0) device_store(state.receive_prefix_state, dispatch_epoch(state));
    produce_receive_prefixes(state, lane, entry_look PCIE_EP_PROFILE(, profile));
    PCIE_EP_PROFILE(profile.save(state.profiling, profile_rows(state.z.dims.channels, state.worker_groups * (state.tx_waves + state.rx_waves)) - 1, lane);)
}

__device__ __forceinline__ void produce_receive_prefixes(const DeviceState& state, int lane, PrefixFirstLook entry_look PCIE_EP_PROFILE(, RoleProfile& profile)) {
    const uint64_t epoch = dispatch_epoch(state);
    const bool success = compute_receive_prefixes(state, lane, entry_look PCIE_EP_PROFILE(, profile));
    // The results were written through; they are complete once this wavefront's
    // stores have been acknowledged.  Local consumers come first, the ACK to the
    // sources (which nobody on this GPU waits for) second.
    wait_memory_ops();
    if (lane == 0) {
        state.prefix_tx_timestamps_ns[1] = ticks_to_ns(state, now_ticks());
        device_store(state.receive_prefix_state + 1, success ? epoch : kPrefixFailed);
    }
    PCIE_EP_PROFILE(profile.first(kProfilePrefixPublishedNs);)
    if (success) acknowledge_counts(state, lane);
}

// 1 once the receive prefixes of this epoch are published, -1 when they never
// will be (their producer failed or the dispatch has an error), 0 otherwise.
// The elected producer owns the timeout; everybody else only reads device flags.
__device__ __forceinline__ int receive_prefix_verdict(const DeviceState& state, uint64_t epoch, int lane) {
    int verdict = 0;
    if (lane == 0) {
        // Relaxed: what the flag guards is read with device-scope loads.
        const uint64_t value = device_load(state.receive_prefix_state + 1);
        if (value == epoch) verdict = 1;
        else if (value == kPrefixFailed || load_error_code(state)) verdict = -1;
    }
    return broadcast_first(verdict);
}

// ---------------------------------------------------------------------------------------
// TX control + guardian
// ---------------------------------------------------------------------------------------
// Destination ranks of a token, straight from its routes: what the plan will say (ids that are out of range count for
// none, a repeated one for the same rank; either ends the dispatch).  Only where the prologue rides in this launch, with
// at most eight routes per token.
__device__ __forceinline__ uint32_t route_destinations(const DeviceState& state, int token) {
    constexpr int kFusedTopk = 8;
    const int topk = state.z.dims.topk, experts = state.z.dims.num_experts, local = state.z.local_experts;
    int64_t raw[kFusedTopk];
#pragma unroll
    for (int branch = 0; branch < kFusedTopk; ++branch) raw[branch] = branch < topk ? state.topk_idx[size_t(token) * topk + branch] : -1;
    uint32_t destinations = 0;
#pragma unroll
    for (int branch = 0; branch < kFusedTopk; ++branch)
        if (raw[branch] >= 0 && raw[branch] < experts) destinations |= 1u << (uint32_t(raw[branch]) / uint32_t(local));
    return destinations;
}

// Entry `ordinal` of the queue that this rank reads `source`'s descriptors from: of another domain's source, the one its
// relay fills for this rank's domain (advanced_common.cuh:237-247).
__device__ __forceinline__ Descriptor* descriptor_of(const DeviceState& state, int channel, int source, int ordinal) {
    const SegmentLayout& z = state.z;
    const int me = state.local_rank;
    return reads_replica(z.dims, source, me) ? replica_descriptor_at(z, state.seg[source], channel, z.dims.rank_domain[me], me, ordinal)
                                             : descriptor_at(z, state.seg[source], channel, me, ordinal);
}

// ---------------------------------------------------------------------------------------
// Direct rows
// ---------------------------------------------------------------------------------------
// The host link is idle until the first received rows are requested, some 10 us into the launch, and once they are, a
// row to be transmitted waits behind them twice: its reads from HBM pass the same queues of its XCD (10 to 20 us where
// an idle machine takes 1.4), and its stores share the link.  The first tokens of every channel are therefore
// transmitted by payload wavefronts that need neither ticket nor plan for it: token t by wavefront t, as it
// enters.  Its place in the rings follows from the routes of the tokens in front of it in its channel.  The
// metadata and the descriptors follow when the plan is there.
//
// As many as the link takes in that time (kDirectBytes), at most kMaxDirectRows of a channel: 64 rows of 14 KB hold the
// first received rows up (cached replay of 128 tokens 186 us per dispatch with 32 of them, 192 with 64), 64 of 8 KB do
// not (4 ranks, 200 tokens of 4096 columns 119 / 110).  And only in a dispatch that receives little (kDirectDispatchBytes,
// by the rows of all other sources): a longer one ends with its receive side whatever the transmit side does, and
// the early rows only delay it (96 aligned tokens, 9.7 MB: 145 us without, 148 with them).
// Us per dispatch without and with: 16 tokens 50.2 / 48.2, 32 75 / 68, 64 of 4096 columns 80 / 73, 24 of 2048 (top-4) 40 / 35,
// 2 ranks with 300 tokens 157 / 138.
constexpr int64_t kDirectBytes = 544 << 10;
constexpr int64_t kDirectDispatchBytes = 6 << 20;
constexpr int kMaxDirectRows = 3;
__device__ __forceinline__ int payload_wavefronts(const DeviceState& state) { return state.worker_groups * (state.tx_waves + state.rx_waves); }
// How many tokens of every channel are direct rows: with the prologue in the launch, payload wavefronts of their own for
// them, and rings that the dispatch before has left drained.
__device__ __forceinline__ int direct_rows_per_channel(const DeviceState& state) {
    const SegmentLayout& z = state.z;
    const int64_t row_bytes = z.meta_offset + z.meta_bytes;
    if (!state.fused || int64_t(z.dims.num_ranks - 1) * state.num_tokens * row_bytes > kDirectDispatchBytes || device_load(state.epoch + kDrainedEpochWord) + 1 != dispatch_epoch(state)) return 0;
    int rows = payload_wavefronts(state) / (2 * z.dims.channels);
    const int most = int(kDirectBytes / (z.dims.channels * row_bytes));
    rows = rows < most ? rows : most;
    rows = rows < kMaxDirectRows ? rows : kMaxDirectRows;
    rows = rows < z.dims.payload_slots ? rows : z.dims.payload_slots;
    return rows < z.dims.descriptor_slots ? rows : z.dims.descriptor_slots;
}
// Destination ranks of a token without the plan of this dispatch.
__device__ __forceinline__ uint32_t early_destinations(const DeviceState& state, int token) {
    return state.fused && !state.reuse_plan ? route_destinations(state, token) : state.plan_mask[token];
}
__device__ __forceinline__ void tx_control(const DeviceState& state, TransportQueues& q, int channel, int lane) {
    const SegmentLayout& z = state.z;
    const int channels = z.dims.channels, me = state.local_rank;
    const int endpoints = z.endpoints;  // destination ranks, then (relay mode) one relay endpoint per domain
    const int slots = z.dims.payload_slots;
    const int stride = (z.dims.max_tokens + channels - 1) / channels;
    char* own = state.seg[me];
    const uint64_t epoch = dispatch_epoch(state);
    const uint64_t start = now_ticks();
    HealthCheck health(state, start, true, channel, channels);
    PCIE_EP_PROFILE(RoleProfile profile(state.clock_khz);)
    if (lane == 0) device_store(state.channel_timestamps_ns + channel * 2, ticks_to_ns(state, start));
    const int tokens = state.num_tokens;
    const int candidates = tokens > channel ? (tokens - channel + channels - 1) / channels : 0;
    const uint64_t below = lanes_below(lane);
    const __amdgpu_buffer_rsrc_t ring = device_resource(q.tx, sizeof(q.tx));
    int produced = 0;
    int reserved[kMaxEndpoints];
#pragma unroll
    for (int endpoint = 0; endpoint < kMaxEndpoints; ++endpoint) reserved[endpoint] = 0;
    const int direct = broadcast_first(direct_rows_per_channel(state));
    bool failed = false;
    int64_t stage_busy = 0, prepared_ahead = 0;

    for (int base = 0; base < candidates && !failed; base += kWave) {
        const int candidate = base + lane;
        const int token = channel + candidate * channels;
        // Where the token is published: its destination ranks, with those of other
        // domains folded into one relay endpoint per domain (advanced_common.cuh:207-225).
        uint32_t destinations = 0;
        if (candidate < candidates) destinations = early_destinations(state, token);
        const uint32_t remote = endpoint_mask_of(z.dims, me, destinations);
        const uint64_t batch = __ballot(remote != 0);
        if (!batch) continue;
        const int ordinal = produced + __popcll(batch & below);
        int my_descriptor[kMaxEndpoints];
#pragma unroll
        for (int endpoint = 0; endpoint < kMaxEndpoints; ++endpoint) {
            my_descriptor[endpoint] = 0;
            if (endpoint < endpoints) {
                const uint64_t hits = __ballot((remote >> endpoint) & 1u);
                my_descriptor[endpoint] = reserved[endpoint] + __popcll(hits & below);
                reserved[endpoint] += __popcll(hits);
            }
        }
        // Ring history: which token occupied ordinal i (needed when a slot is reused).
        if (remote) device_store(state.chan_remote_tokens + size_t(channel) * stride + ordinal, token);
        // The channel's first tokens may be direct rows, which have no ticket.
        const uint64_t ticketed = __ballot(remote != 0 && candidate >= direct);
        int ticket_index = 0;
        if (ticketed) ticket_index = reserve_tickets(q.tx_tail, __popcll(ticketed), lane) + __popcll(ticketed & below);
        else wait_memory_ops();
        // Tickets prepared while an earlier payload of this channel is still in
        // flight: the control path runs ahead of the payload path (the event the
        // reference counts in stats[3]: advanced_dispatch.cuh:384-387).
        if (produced > 0 && broadcast_first(int(device_load(&q.tx_retired[channel].value))) < produced) prepared_ahead += __popcll(batch);
        bool pending = (ticketed >> lane) & 1ull;
        while (true) {
            if (pending && ring_entry_free(q.tx_taken, epoch, ticket_index)) {
                const uint32_t at = uint32_t(ticket_index % kRing) * uint32_t(sizeof(TxEntry));
                device_store_b32(ring, at + 0, uint32_t(token));
                device_store_b32(ring, at + 4, uint32_t(ordinal));
                device_store_b32(ring, at + 8, remote);
                device_store_b32(ring, at + 12, uint32_t(channel));
#pragma unroll
                for (int endpoint = 0; endpoint < kMaxEndpoints; ++endpoint)
                    if (endpoint < endpoints) device_store_b32(ring, at + 16 + 4 * endpoint, uint32_t(my_descriptor[endpoint]));
                // Ring history and the ticket body are complete before the tag.
                wait_memory_ops();
                device_store(q.tx_ready + ticket_index % kRing, sequence(epoch, ticket_index));
                pending = false;
            }
            if (!__any(pending)) break;
            ++stage_busy;
            const bool unhealthy = health.poll(state, lane);
            if (unhealthy || broadcast_first(aborted(q) ? 1 : 0)) {
                // A peer's abort flag or the timeout: raise the kernel-wide abort at
                // once, the workers are spinning on tickets that will never be marked ready.
                if (unhealthy && lane == 0) {
                    record_error(state, kErrRingProgressWait);
                    raise_abort(q);
                }
                failed = true;
                break;
            }
            backoff();
        }
        produced += __popcll(batch);
        PCIE_EP_PROFILE(profile.first(kProfileFirstTicketNs); profile.last(kProfileLastTicketNs);)
    }
    PCIE_EP_PROFILE(profile.values[kProfileItems] = uint64_t(produced);)

    // Wait for the workers, then drain the ACKs of the last ring window: earlier
    // slots were checked when they were reused (advanced_dispatch.cuh:229-285).
    // Lanes poll different (ordinal, destination) pairs in parallel.
    bool drained = failed;
    // Relay mode: every relay flow of the channel, also one without work, must
    // have consumed this epoch's counts and released its replica slots before a
    // later dispatch may overwrite the mailbox (advanced_dispatch.cuh:213-225).
    bool relays_drained = z.dims.domains == 0;
    int drain_ordinal = produced > slots ? produced - slots : 0;
    uint64_t next_drain_poll = 0;
    bool workers_finished = false;
    while (true) {
        if (broadcast_first(aborted(q) ? 1 : 0)) break;
        if (!workers_finished) {
            workers_finished = broadcast_first(int(device_load(&q.tx_retired[channel].value))) >= produced;
            PCIE_EP_PROFILE(if (workers_finished) profile.first(kProfileWorkersDoneNs);)
        }
        if (workers_finished && !drained) {
            // Each pass checks up to kDrainBatch * (64 / endpoints) ordinals of every
            // endpoint; lanes of one endpoint read consecutive ACK words (one 64-byte read
            // per eight slots) and all reads of a pass are on the link before the first
            // is used, so a ring window costs a few round trips, not one per handful of slots.
            // While the channel's receive side is still busy the drain is not what the
            // kernel waits for: it then polls sparingly, so that the small reads do not
            // compete with the row reads for the link.
            const bool receive_busy = broadcast_first(int(device_load(&q.rx_finished[channel].value))) == 0;
            if (!receive_busy || broadcast_first(now_ticks() >= next_drain_poll ? 1 : 0)) {
                PCIE_EP_PROFILE(const uint64_t poll_begin = profile.now(); profile.add(kProfilePolls);)
                constexpr int kDrainBatch = 8;
                const int group = kWave / endpoints;
                const int per_pass = group * kDrainBatch;
                const int endpoint = lane / group;
                // Vector memory operations complete in order: what the ACK addresses depend
                // on (tokens, route masks) is loaded first, the host reads follow in one run.
                uint64_t seen[kDrainBatch], wanted[kDrainBatch];
                const uint64_t* address[kDrainBatch];
#pragma unroll
                for (int batch = 0; batch < kDrainBatch; ++batch) {
                    const int my_ordinal = drain_ordinal + batch * group + lane % group;
                    seen[batch] = wanted[batch] = 0;
                    address[batch] = nullptr;
                    if (endpoint < endpoints && my_ordinal < produced) {
                        const int token = device_load(state.chan_remote_tokens + size_t(channel) * stride + my_ordinal);
                        const uint32_t remote = endpoint_mask_of(z.dims, me, state.plan_mask[token]);
                        if ((remote >> endpoint) & 1u) {
                            wanted[batch] = sequence(epoch, token);
                            address[batch] = ack_at(z, own, channel, my_ordinal % slots, endpoint);
                        }
                    }
                }
                wait_memory_ops();
                compiler_barrier();
#pragma unroll
                for (int batch = 0; batch < kDrainBatch; ++batch)
                    if (address[batch]) seen[batch] = host_load_global(address[batch]);
                int missing_ordinal = 0x7FFFFFFF;
#pragma unroll
                for (int batch = kDrainBatch - 1; batch >= 0; --batch)
                    if (seen[batch] != wanted[batch]) missing_ordinal = drain_ordinal + batch * group + lane % group;
                for (int offset = 32; offset > 0; offset >>= 1) {
                    const int other = __shfl_xor(missing_ordinal, offset);
                    missing_ordinal = other < missing_ordinal ? other : missing_ordinal;
                }
                // Everything before the first miss is done.
                drain_ordinal = missing_ordinal < drain_ordinal + per_pass ? missing_ordinal : drain_ordinal + per_pass;
                if (drain_ordinal >= produced) drained = true;
                else if (missing_ordinal != 0x7FFFFFFF) next_drain_poll = now_ticks() + 20 * state.clock_khz / 1000;
                PCIE_EP_PROFILE(profile.add(kProfilePollSum, profile.now() - poll_begin); if (drained) profile.first(kProfileDrainedNs); else profile.add(kProfilePollMisses);)
            }
        }
        if (workers_finished && drained && !relays_drained) {
            bool done = true;
            if (lane < z.dims.domains) done = host_load(signal_at(own, z.relay_drained_offset, flow_index(z, channel, lane))) == epoch;
            relays_drained = __all(done);
        }
        if (workers_finished && drained && (relays_drained || failed) && broadcast_first(int(device_load(&q.rx_finished[channel].value)))) break;
        // Guardian: this wavefront outlives TX so that a stalled RX still times out.
        PCIE_EP_PROFILE(const uint64_t health_begin = profile.now();)
        const bool unhealthy = health.poll(state, lane);
        PCIE_EP_PROFILE(profile.add(kProfileHealthSum, profile.now() - health_begin);)
        const bool forced = channel == 0 && state.control_abort_after && now_ticks() - start >= state.control_abort_after;
        if (unhealthy || broadcast_first(forced ? 1 : 0)) {
            if (lane == 0) {
                record_error(state, kErrRingProgressWait);
                raise_abort(q);
            }
            break;
        }
        backoff();
    }
    if (lane == 0) {
        atomicAdd(reinterpret_cast<unsigned long long*>(state.channel_stats + channel * kStatFields + kStatRingFull),
                  static_cast<unsigned long long>(stage_busy));
        atomicAdd(reinterpret_cast<unsigned long long*>(state.channel_stats + channel * kStatFields + kStatPreparedAhead),
                  static_cast<unsigned long long>(prepared_ahead));
        // Only this wavefront writes the channel's mapped abort word.
        if (aborted(q)) store_release_system(signal_at(own, z.channel_abort_offset, channel), epoch);
        // Both directions are complete (or aborted): the channel's end time.
        device_store(state.channel_timestamps_ns + channel * 2 + 1, ticks_to_ns(state, now_ticks()));
    }
    PCIE_EP_PROFILE(profile.values[kProfileHealthScans] = uint64_t(health.scans); if (produced == 0) profile.first(kProfileDrainedNs);
                    profile.last(kProfileFinishedNs); profile.save(state.profiling, channel, lane);)
}

// ---------------------------------------------------------------------------------------
// RX control
// ---------------------------------------------------------------------------------------
// The first look of a receive control at its descriptor queues (entry `ahead` of every
// source's queue): the same load as in the first pass of rx_control's loop, issued by
// the kernel's entry code while the role still waits to be let in (the queues it hands
// tickets out through are being reset), so that the round trip over the host link and
// that wait overlap.
struct RxFirstPoll {
    u32x4 published;
    bool issued;
};
// Which descriptor queue a lane of a receive control looks at: up to 64 / P entries ahead in every source's queue.
struct RxLane {
    int lookahead, source, ahead, my_domain;
    bool member, replica;
    __device__ __forceinline__ RxLane(const DeviceState& state, int lane) {
        const SegmentLayout& z = state.z;
        const int ranks = z.dims.num_ranks, me = state.local_rank;
        lookahead = kWave / ranks > 32 ? 32 : kWave / ranks;
        source = lane / lookahead;
        ahead = lane % lookahead;
        member = source < ranks && source != me;
        // A source of another domain is read from the replica ring its relay fills
        // for this rank's domain (advanced_common.cuh:237-247).
        replica = member && reads_replica(z.dims, source, me);
        my_domain = z.dims.domains ? z.dims.rank_domain[me] : 0;
    }
    // Entry `ordinal` of the lane's queue (entry 0 of the own queue for a lane without one: never loaded).
    __device__ __forceinline__ Descriptor* entry(const DeviceState& state, int channel, int ordinal) const {
        return descriptor_of(state, channel, member ? source : state.local_rank, ordinal);
    }
};
__device__ __forceinline__ RxFirstPoll rx_first_poll(const DeviceState& state, int channel, int lane) {
    const RxLane at(state, lane);
    RxFirstPoll poll{{0u, 0u, 0u, 0u}, true};
    if (at.member) poll.published = host_load_b128_at(at.entry(state, channel, at.ahead));
    return poll;
}

__device__ __forceinline__ void rx_control(const DeviceState& state, TransportQueues& q, int channel, int lane, RxFirstPoll first_poll) {
    const SegmentLayout& z = state.z;
    const int ranks = z.dims.num_ranks, me = state.local_rank;
    const uint64_t begin = now_ticks();
    const uint64_t epoch = dispatch_epoch(state);
    PCIE_EP_PROFILE(RoleProfile profile(state.clock_khz);)
    if (!dedicated_prefix_producer(state)) elect_receive_prefixes(state, lane PCIE_EP_PROFILE(, profile));
    // Polling does not wait for the prefixes: a descriptor entry is valid as soon as
    // its tag carries this epoch and the next ordinal, whatever the counts say, so
    // rows are requested from the first microseconds of the kernel on.  The counts
    // (how many rows each source sends on this channel) are only needed to know
    // when to stop; the payload wavefronts wait for the prefixes after they have
    // requested a row, before they compute where it goes.
    const RxLane at(state, lane);
    const int lookahead = at.lookahead, source = at.source, ahead = at.ahead, my_domain = at.my_domain;
    const bool member = at.member, replica = at.replica;
    int expected = member ? 0x7FFFFFFF : 0, total = 0x7FFFFFFF;
    bool counts_known = false, prefix_failed = false;
    const uint64_t below = lanes_below(lane);
    const uint64_t group_mask = (1ull << lookahead) - 1ull;
    const __amdgpu_buffer_rsrc_t ring = device_resource(q.rx, sizeof(q.rx));
    Deadline deadline(begin);
    int consumed = 0, issued = 0;
    int64_t not_ready = 0, ring_waits = 0;
    bool failed = false;
    while (!failed && !prefix_failed) {
        // The pass that consumes the look taken at entry goes straight to it: the abort word and the
        // prefixes' state (two trips to device memory) cannot have anything to say a few microseconds
        // into the launch, and are looked at from the second pass on.
        const bool entry_pass = first_poll.issued && consumed == 0 && issued == 0 && !counts_known;
        if (!entry_pass && broadcast_first(aborted(q) ? 1 : 0)) break;
        if (!counts_known && !entry_pass) {
            const int verdict = receive_prefix_verdict(state, epoch, lane);
            if (verdict < 0) {
                prefix_failed = true;
                break;
            }
            if (verdict > 0) {
                expected = member ? device_load(state.expected_receive_counts + channel * ranks + source) : 0;
                total = ahead == 0 ? expected : 0;
                for (int offset = 32; offset > 0; offset >>= 1) total += __shfl_xor(total, offset);
                counts_known = true;
                PCIE_EP_PROFILE(profile.first(kProfileCountsKnownNs);)
            }
        }
        if (counts_known && issued >= total) break;
        const int ordinal = consumed + ahead;
        const bool want = member && ordinal < expected;
        Descriptor* descriptor = at.entry(state, channel, want ? ordinal : 0);
        // One 16-byte load brings READY together with the slot and token it guards.
        u32x4 published = {0u, 0u, 0u, 0u};
        PCIE_EP_PROFILE(const uint64_t poll_begin = profile.now(); profile.add(kProfilePolls);)
        if (entry_pass) {
            // Nothing has been consumed and the counts are not known: this pass would load exactly what was loaded at entry.
            published = first_poll.published;
            first_poll.issued = false;
        } else if (want) {
            published = host_load_b128_at(descriptor);
        }
        PCIE_EP_PROFILE(profile.add(kProfilePollSum, profile.now() - poll_begin);)
        const bool ready = want && (uint64_t(published[0]) | uint64_t(published[1]) << 32) == sequence(epoch, ordinal);
        const uint64_t ready_lanes = __ballot(ready);
        // Descriptors of one source are consumed in order: accept the leading run.
        const uint64_t group = (ready_lanes >> (source < ranks ? source * lookahead : 0)) & group_mask;
        const int run = __builtin_ctzll(~group | (1ull << lookahead));
        const bool accept = ready && ahead < run;
        const uint64_t accepted = __ballot(accept);
        if (!accepted) {
            PCIE_EP_PROFILE(profile.add(kProfilePollMisses);)
            ++not_ready;
            backoff();
            continue;
        }
        // Slot and token come from the peer (or its relay) and become the base of a
        // host read: a value outside the ring would make the payload wavefront read
        // beyond the pinned segment, which is a memory fault, not a protocol error.
        // Same verdict as a wrong identity: terminal, nothing is ACKed.
        {
            const int named_slot = int(published[2]), named_token = int(published[3]);
            const int ring_slots = replica ? z.dims.replica_slots : z.dims.payload_slots;
            const bool outside = accept && (named_slot < 0 || named_slot >= ring_slots || named_token < 0 || named_token >= z.dims.max_tokens);
            if (__any(outside)) {
                if (lane == 0) {
                    record_error(state, kErrPayloadSequence);
                    raise_abort(q);
                }
                failed = true;
                break;
            }
        }
        const int ticket_index = reserve_tickets(q.rx_tail, __popcll(accepted), lane) + __popcll(accepted & below);
        const int slot = int(published[2]), token = int(published[3]);
        const uint64_t payload_sequence = sequence(epoch, token);
        bool pending = accept;
        while (true) {
            if (pending && ring_entry_free(q.rx_taken, epoch, ticket_index)) {
                const uint32_t at = uint32_t(ticket_index % kRing) * uint32_t(sizeof(RxEntry));
                device_store_b32(ring, at + 0, uint32_t(source));
                device_store_b32(ring, at + 4, uint32_t(slot));
                device_store_b32(ring, at + 8, uint32_t(token));
                device_store_b32(ring, at + 12, uint32_t(channel));
                device_store_b32(ring, at + 16, uint32_t(payload_sequence));
                device_store_b32(ring, at + 20, uint32_t(payload_sequence >> 32));
                device_store_b32(ring, at + 24, uint32_t(issued + __popcll(accepted & below)));
                device_store_b32(ring, at + 28, replica ? 1u : 0u);
                // The ticket body is complete before its tag.
                wait_memory_ops();
                device_store(q.rx_ready + ticket_index % kRing, sequence(epoch, ticket_index));
                pending = false;
            }
            if (!__any(pending)) break;
            ++ring_waits;
            if (broadcast_first((aborted(q) || deadline.expired(state)) ? 1 : 0)) {
                failed = true;
                break;
            }
            backoff();
        }
        issued += __popcll(accepted);
        PCIE_EP_PROFILE(profile.first(kProfileFirstTicketNs); profile.last(kProfileLastTicketNs);)
        // Every accepted entry is captured in a ticket: return the credits, one
        // store per source for the whole run (entries are consumed in order).  The
        // payload ACK and the ticket ring entry are separate resources.
        if (member && ahead == 0 && run > 0 && !failed)
            host_field_store(replica ? replica_credit_at(z, state.seg[source], channel, my_domain, me) : credit_at(z, state.seg[source], channel, me),
                             sequence(epoch, consumed + run - 1));
        if (member) consumed += run;
    }
    if (prefix_failed) {
        if (lane == 0) {
            raise_abort(q);
            device_store(&q.rx_finished[channel].value, 1u);
        }
        PCIE_EP_PROFILE(profile.save(state.profiling, state.z.dims.channels + channel, lane);)
        return;
    }
    // RX is finished when every ticket has been retired by a worker.
    while (true) {
        if (broadcast_first(aborted(q) ? 1 : 0)) break;
        if (broadcast_first(int(device_load(&q.rx_retired[channel].value))) >= issued && issued >= total) break;
        backoff();
    }
    PCIE_EP_PROFILE(profile.first(kProfileWorkersDoneNs); profile.values[kProfileItems] = uint64_t(issued);)
    if (lane == 0) {
        atomicAdd(reinterpret_cast<unsigned long long*>(state.channel_stats + channel * kStatFields + kStatRxNotReady),
                  static_cast<unsigned long long>(not_ready));
        // Column 1 of the receive/expand diagnostic: how many receive tickets of
        // this channel have completed their scatter (fused_receive.cuh:290-294).
        if (state.overlap_diagnostic) state.receive_expand_overlap[channel * 2 + 1] = int64_t(device_load(&q.rx_retired[channel].value));
        atomicAdd(reinterpret_cast<unsigned long long*>(state.channel_stats + channel * kStatFields + kStatRingFull),
                  static_cast<unsigned long long>(ring_waits));
        device_store(&q.rx_finished[channel].value, 1u);
    }
    PCIE_EP_PROFILE(profile.last(kProfileFinishedNs); profile.save(state.profiling, state.z.dims.channels + channel, lane);)
}

// ---------------------------------------------------------------------------------------
// Local bypass, padding and the final reduction
// ---------------------------------------------------------------------------------------
// Every wavefront of the local workgroups claims own tokens 0 .. T-1 one at a time
// until none is left, then (with zero padding on an expanded layout) clears its
// share of the alignment gaps' rows; `wave` is its position among the `waves` of them.
template <bool kVector>
__device__ __forceinline__ void local_rows(const DeviceState& state, TransportQueues& q, int lane, int wave, int waves) {
    const uint64_t epoch = dispatch_epoch(state);
    // Destination rows depend on the receive prefixes of this epoch.
    int ready = 0;
    if (lane == 0) {
        while (true) {
            const uint64_t value = device_load(state.receive_prefix_state + 1);  // what it guards is read with device-scope loads
            if (value == epoch) { ready = 1; break; }
            // The wavefront that computes the prefixes owns the timeout.
            if (value == kPrefixFailed || aborted(q) || load_error_code(state)) break;
            __builtin_amdgcn_s_sleep(48);
        }
    }
    if (!broadcast_first(ready)) return;
    if (!wait_for_plan(state, q, lane)) return;
    while (true) {
        uint32_t claimed = 0;
        if (lane == 0) claimed = aborted(q) ? 0xFFFFFFFFu : device_add(&q.local_head.value, 1u);
        const int item = broadcast_first(int(claimed));
        if (item < 0) return;
        if (item >= state.num_tokens) break;
        if (!local_token_rows<kVector>(state, item, lane)) {
            if (lane == 0) {
                record_error(state, kErrExpandedCapacity);
                raise_abort(q);
            }
            return;
        }
    }
    if (state.expand && state.fuse_expand && state.zero_padding) zero_padding_rows<kVector>(state, wave, waves, lane);
}

// Called by every role wavefront as its last act.  Everything the reduction
// reads was written with device-scope stores or atomics, so waiting for this
// wavefront's own operations is all the ordering the count needs.
__device__ __forceinline__ void finish_role(const DeviceState& state, TransportQueues& q, int lane, uint32_t roles) {
    wait_memory_ops();
    uint32_t earlier = 0;
    if (lane == 0) earlier = device_add(&q.finished.value, 1u);
    if (uint32_t(broadcast_first(int(earlier))) + 1u != roles) return;
    // Last one out: column sums of the per-channel statistics and the span of
    // the channel timestamps.  Done after failures too (the reference launches
    // advanced_reduce_statistics unconditionally).
    // The whole kernel waits for this wavefront: every word is requested before the
    // first is used (lane l reads words l, l + 64, ...), and the sums and the span
    // come out of lane shuffles - two round trips to memory, not one per channel.
    const int channels = state.z.dims.channels;
    constexpr int kStatWordsPerLane = kMaxChannels * kStatFields / kWave;
    int64_t words[kStatWordsPerLane];
#pragma unroll
    for (int i = 0; i < kStatWordsPerLane; ++i) {
        const int word = lane + i * kWave;
        words[i] = word < channels * kStatFields ? device_load(state.channel_stats + word) : 0;
    }
    // Channel c's start and end stamps are words 2c and 2c + 1: lane l takes word l.
    const int64_t stamp = lane < channels * 2 ? device_load(state.channel_timestamps_ns + lane) : 0;
    // kStatFields divides 64: word w belongs to field w % kStatFields whatever i is.
    int64_t sum = 0;
#pragma unroll
    for (int i = 0; i < kStatWordsPerLane; ++i) sum += words[i];
    for (int offset = kStatFields; offset < kWave; offset <<= 1) sum += __shfl_xor(sum, offset);
    if (lane < kStatFields) state.stats[lane] = sum;
    // Even lanes hold start stamps (earliest non-zero wins), odd lanes end stamps (latest wins).
    int64_t span = lane % 2 == 0 && stamp == 0 ? INT64_MAX : stamp;
    for (int offset = 2; offset < kWave; offset <<= 1) {
        const int64_t other = __shfl_xor(span, offset);
        span = lane % 2 == 0 ? (other < span ? other : span) : (other > span ? other : span);
    }
    if (lane == 0) state.transport_timestamps_ns[0] = span == INT64_MAX ? 0 : span;
    if (lane == 1) state.transport_timestamps_ns[1] = span;
    const uint64_t epoch = dispatch_epoch(state);
    // Every own slot has been acknowledged unless the dispatch failed: the next one may write them at once.
    if (lane == 0 && !aborted(q) && load_error_code(state) == 0) state.epoch[kDrainedEpochWord] = epoch;
    // Prologue inside this launch: every workgroup has read the epoch word by now.
    if (lane == 0 && state.fused) *state.epoch = epoch;
}

// ---------------------------------------------------------------------------------------
// TX payload worker
// ---------------------------------------------------------------------------------------
// An instantiation for short rows (receive_batch) has none above kBatchedFp8Columns to hold: holding room for 8192
// columns it kept 9 registers in scratch memory (1500 tokens of 2048 columns, 8 ranks: 362 us per dispatch, 352).
template <bool kFp8, bool kVector, int kRows, typename BeforeStores>
__device__ __forceinline__ float tx_copy_row(const DeviceState& state, const uint16_t* input, __amdgpu_buffer_rsrc_t slot, int lane, BeforeStores before_stores) {
    const int hidden = state.z.dims.hidden;
    constexpr int kGroups = (kRows > 1 ? kBatchedFp8Columns : kPassItems * kWave * 8) / (16 * kWave);
    if constexpr (kFp8) return quantize_row_to_host<kVector, kGroups>(input, slot, hidden, lane, before_stores);
    copy_row_to_host<kVector>(input, slot, hidden, lane, before_stores);
    return 1.0f;
}

// Payload wavefront `order` transmits the payload of its direct row, if it has one, and leaves the words of its ticket and
// behind them the row's scale in `ticket`.  Whether it had one.
template <bool kFp8, bool kVector, int kRows>
__device__ __forceinline__ bool direct_row(const DeviceState& state, uint32_t* ticket, int order, int lane) {
    const SegmentLayout& z = state.z;
    const int channels = z.dims.channels, me = state.local_rank, token = order;
    if (!state.fused || token >= state.num_tokens || token >= channels * kMaxDirectRows || token >= channels * broadcast_first(direct_rows_per_channel(state))) return false;
    // Lane c: the channel's candidate c.
    const int channel = token % channels, candidate = token / channels;
    uint32_t remote = 0;
    if (lane <= candidate) remote = endpoint_mask_of(z.dims, me, early_destinations(state, channel + lane * channels));
    const uint32_t endpoints = uint32_t(__shfl(int(remote), candidate));
    if (endpoints == 0) return false;
    const uint64_t in_front = lanes_below(candidate);
    const int ordinal = __popcll(__ballot(remote != 0) & in_front);
    // Lane 4 + e: descriptor ordinal of endpoint e (TxEntry).
    uint32_t word = lane == 0 ? uint32_t(token) : lane == 1 ? uint32_t(ordinal) : lane == 2 ? endpoints : uint32_t(channel);
    for (int endpoint = 0; endpoint < z.endpoints; ++endpoint) {
        const int before = __popcll(__ballot((remote >> endpoint) & 1u) & in_front);
        if (lane == 4 + endpoint) word = uint32_t(before);
    }
    if (lane < kTicketWords) ticket[lane] = word;
    const float scale = tx_copy_row<kFp8, kVector, kRows>(state, state.x + size_t(token) * z.dims.hidden,
                                                          host_resource(slot_at(z, state.seg[me], channel, ordinal), uint32_t(z.meta_offset)), lane, [] {});
    if (lane == 0) ticket[kTicketWords] = float_bits(scale);
    return true;
}

// What a payload wavefront still owes the other ends of the rows it has moved: a received row's slot ACK (lane r: row
// r's), a transmitted row's descriptors (lane e: endpoint e's) and its retirement.  A store to host memory is
// acknowledged one loaded round trip later, and vector memory operations complete in order: stored as soon as the row has
// been moved, it would hold up every step towards the next row - the look at the queues, the claim, the ticket - by that
// round trip.  The wavefront therefore stores it when it has the next row's ticket and is about to
// touch the link again, or finds that there is no next row, and always before it waits for anybody else.
// The record lies in LDS: in registers it would be alive across the row's vectors.
struct Owed {
    uint32_t* record;
    int acks = 0;       // received rows
    bool row = false;   // a transmitted one
    // Few rows of the direction are left (or nobody knows yet): there may be no next row to put it off to, and the
    // other end is waited for.
    bool prompt = true;
};
// The row's own loads / stores must have completed: every caller is behind a wait_memory_ops() that is behind the row.
__device__ __forceinline__ void settle_acks(const DeviceState& state, Owed& owed, int lane) {
    if (lane < owed.acks) {
        const uint32_t* ack = owed.record + 4 * lane;
        typedef uint64_t __attribute__((address_space(1))) * GlobalWord;
        __hip_atomic_store((GlobalWord)(uint64_t(ack[0]) | uint64_t(ack[1]) << 32), sequence(dispatch_epoch(state), int(ack[2])), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_SYSTEM);
    }
    owed.acks = 0;
}
__device__ __forceinline__ void settle(const DeviceState& state, TransportQueues& q, Owed& owed, int lane) {
    settle_acks(state, owed, lane);
    if (!owed.row) return;
    owed.row = false;
    const int channel = broadcast_first(int(owed.record[kOwedRow]));
    const int ordinal = lane < state.z.endpoints ? int(owed.record[kOwedDescriptors + lane]) : -1;
    if (ordinal >= 0) {
        // READY, slot and token in one 16-byte store: nothing to order inside the entry.
        const uint64_t ready = sequence(dispatch_epoch(state), ordinal);
        host_store_b128_at(descriptor_at(state.z, state.seg[state.local_rank], channel, lane, ordinal),
                           u32x4{uint32_t(ready), uint32_t(ready >> 32), owed.record[kOwedRow + 1], owed.record[kOwedRow + 2]});
    }
    if (lane == 0) {
        if (owed.record[kOwedRow + 3]) state.prefix_tx_timestamps_ns[(channel + 1) * 2 + 1] = ticks_to_ns(state, now_ticks());
        device_add(&q.tx_retired[channel].value, 1u);
    }
}

// Counters a payload wavefront accumulates over the rows it moves, flushed once when it ends (in LDS, as the record above).
enum WorkerCount : int { kCountWrites = 0, kCountDeliveries, kCountPublished, kCountCreditMiss, kCountReads, kWorkerCounts };
__device__ __forceinline__ void count_rows(uint32_t* record, WorkerCount which, int amount, int lane) {
    if (lane == 0) record[kOwedCounts + which] += uint32_t(amount);
}

// Moves the own token of transmit ticket `ticket_index` (already marked ready), or of the direct row whose payload is on
// its way, into its host slot; what publishes it is left to settle().  Returns false when the wavefront must stop.
// One copy of this code serves both: with a second one for direct rows five of the eight kernels kept up to eight
// registers in scratch memory.
template <bool kFp8, bool kVector, int kRows>
__device__ __forceinline__ bool tx_row(const DeviceState& state, TransportQueues& q, uint32_t* scratch, int lane, int ticket_index, bool direct,
                       const Deadline& deadline, Owed& owed, bool& plan_known PCIE_EP_PROFILE(, RoleProfile& profile, bool sampled)) {
    const SegmentLayout& z = state.z;
    const int ranks = z.dims.num_ranks, topk = z.dims.topk, me = state.local_rank;
    const int endpoint_count = z.endpoints;
    const int slots = z.dims.payload_slots, descriptors = z.dims.descriptor_slots;
    const int stride = (z.dims.max_tokens + z.dims.channels - 1) / z.dims.channels;
    char* own = state.seg[me];
    const uint64_t epoch = dispatch_epoch(state);
    const int meta_dwords = z.meta_bytes / 4;
    const __amdgpu_buffer_rsrc_t ring = device_resource(q.tx, sizeof(q.tx));
    {
        // Copy the ticket out of the ring (one dword per lane), then free its entry.
        const uint32_t entry_base = uint32_t(ticket_index % kRing) * uint32_t(sizeof(TxEntry));
        uint32_t word;
        if (direct) {
            word = owed.record[kDirectTicket + (lane < kTicketWords ? lane : 0)];
            if (lane == 0) device_add(reinterpret_cast<uint32_t*>(&q.tx_head.direct), 1u);
        } else {
            word = device_load_b32(ring, entry_base + uint32_t(lane < kTicketWords ? lane : 0) * 4u);
        }
        const int token = __shfl(int(word), 0), ordinal = __shfl(int(word), 1);
        const uint32_t endpoints = uint32_t(__shfl(int(word), 2));
        const int channel = __shfl(int(word), 3);
        const int my_descriptor = __shfl(int(word), 4 + (lane < endpoint_count ? lane : 0));
        if (!direct) {
            wait_memory_ops();
            if (lane == 0) device_store(q.tx_taken + ticket_index % kRing, sequence(epoch, ticket_index));
        }
        const int slot = ordinal % slots;
        const bool targeted = lane < endpoint_count && ((endpoints >> lane) & 1u);
        if (ordinal == 0 && lane == 0) state.prefix_tx_timestamps_ns[(channel + 1) * 2] = ticks_to_ns(state, now_ticks());

        // Flow control: the slot's previous occupant must be ACKed by all its
        // targets and a descriptor entry must have been consumed before reuse
        // (advanced_dispatch.cuh:158-187).  One lane per endpoint.
        bool slot_ok = true, credit_ok = true;
        uint64_t previous_sequence = 0;
        if (!plan_known) {
            // A direct row's payload is on its way; everything else of it, and all of any other row, follows the plan.
            settle(state, q, owed, lane);
            if (!wait_for_plan(state, q, lane)) return false;
            plan_known = true;
        }
        if (ordinal >= slots) {
            const int previous_token = device_load(state.chan_remote_tokens + size_t(channel) * stride + ordinal - slots);
            const uint32_t previous_remote = endpoint_mask_of(z.dims, me, state.plan_mask[previous_token]);
            slot_ok = !(lane < endpoint_count && ((previous_remote >> lane) & 1u));
            previous_sequence = sequence(epoch, previous_token);
        }
        if (targeted && my_descriptor >= descriptors) credit_ok = false;
        bool stop = false;
        PCIE_EP_PROFILE(const uint64_t flow_begin = sampled ? profile.now() : 0;)
        while (true) {
            if (!slot_ok) slot_ok = host_load(ack_at(z, own, channel, slot, lane)) == previous_sequence;
            if (!credit_ok) credit_ok = credit_covers(host_load(credit_at(z, own, channel, lane)), epoch, my_descriptor, descriptors);
            if (__all(slot_ok && credit_ok)) break;
            count_rows(owed.record, kCountCreditMiss, 1, lane);
            settle(state, q, owed, lane);
            if (broadcast_first((aborted(q) || deadline.expired(state)) ? 1 : 0)) {
                stop = true;
                break;
            }
            backoff();
        }
        if (stop) return false;
        compiler_barrier();
        PCIE_EP_PROFILE(const uint64_t copy_begin = sampled ? profile.now() : 0; if (sampled) profile.add(kProfileTxFlowWaitSum, copy_begin - flow_begin);)

        // Slot metadata: composed in this wavefront's LDS scratch, then copied out
        // as consecutive dwords.  Weights are the live ones of this dispatch.
        char* slot_base = slot_at(z, own, channel, slot);
        for (int index = lane; index < meta_dwords; index += kWave) scratch[index] = 0;
        fence_lds();
        if (lane == 0) {
            scratch[0] = uint32_t(token);
            scratch[1] = state.plan_mask[token];
        }
        if (lane < ranks) scratch[kMetaRankOrdinalsOffset / 4 + lane] = uint32_t(state.plan_rank_ord[size_t(token) * ranks + lane]);
        if (lane < topk) {
            scratch[kMetaBranchOffset / 4 + lane] = uint32_t(state.plan_exp_idx[size_t(token) * topk + lane]);
            scratch[kMetaBranchOffset / 4 + topk + lane] = uint32_t(state.plan_exp_ord[size_t(token) * topk + lane]);
            scratch[kMetaBranchOffset / 4 + 2 * topk + lane] =
                float_bits(state.topk_weights ? state.topk_weights[size_t(token) * topk + lane] : 1.0f);
        }
        if (lane == kWave - 1) test_delay(state.tx_delay);
        const __amdgpu_buffer_rsrc_t slot_resource = host_resource(slot_base, uint32_t(z.meta_offset + z.meta_bytes));
        float scale;
        if (direct) scale = bits_float(owed.record[kDirectScale]);
        else scale = tx_copy_row<kFp8, kVector, kRows>(state, state.x + size_t(token) * z.dims.hidden, host_resource(slot_base, uint32_t(z.meta_offset)), lane,
                                                       [&] { settle(state, q, owed, lane); });
        if (lane == 0) scratch[2] = float_bits(scale);
        fence_lds();
        if (lane == meta_dwords - 1 || (lane == kWave - 1 && meta_dwords > kWave)) test_delay(state.metadata_delay);
        for (int index = lane; index < meta_dwords; index += kWave)
            host_store_b32(slot_resource, uint32_t(z.meta_offset + index * 4), scratch[index]);
        // Every lane's payload and metadata stores have been acknowledged before
        // any lane publishes a descriptor (the counters are wave-wide): see settle().
        PCIE_EP_PROFILE(if (sampled) { wait_memory_ops(); profile.add(kProfileTxCopySum, profile.now() - copy_begin); })
        if (lane < endpoint_count) owed.record[kOwedDescriptors + lane] = uint32_t(targeted ? my_descriptor : -1);
        if (lane == 0) {
            owed.record[kOwedRow] = uint32_t(channel);
            owed.record[kOwedRow + 1] = uint32_t(slot);
            owed.record[kOwedRow + 2] = uint32_t(token);
            owed.record[kOwedRow + 3] = ordinal == 0 ? 1u : 0u;
        }
        owed.row = true;
        count_rows(owed.record, kCountWrites, 1, lane);
        // Logical deliveries count destination ranks; a relay endpoint stands for
        // all targeted ranks of its domain with one descriptor.
        count_rows(owed.record, kCountDeliveries, __popc(scratch[1] & ~(1u << me)), lane);
        count_rows(owed.record, kCountPublished, __popc(endpoints), lane);
        fence_lds();  // scratch is reused by the next ticket
        if (owed.prompt) {
            wait_memory_ops();
            settle(state, q, owed, lane);
        }
    }
    return true;
}

// ---------------------------------------------------------------------------------------
// RX + scatter worker
// ---------------------------------------------------------------------------------------
// Loads of a row (1 KB each) that a wavefront has on the link at once.  About 130 KB in flight fill the link; whatever is
// requested beyond that only waits, in queues that the writes, the control's polls and the tickets have to
// pass.  (One wavefront's write of a 14 KB row, beside 188 that read, is acknowledged after 45 us with 14 loads in
// flight each, 37 with 4, 18 with 2.)  Wavefronts are not always reading, so that fewer than 4 cost more than they save:
// us per dispatch with all 14, with 4, with 2, with 1: 700 tokens 647 / 645 / 648 / 661, cached replay of 128 185 / 183 /
// 189 / 193, 2000 tokens hotspot top-4 1645 / 1625 / 1641 / -, 300 tokens on 2 ranks 154 / 150 / 152 / 161.
// It spaces the first pass of a row that is received alone: all of the row up to 8192 columns (4096 of ragged BF16 rows).
// A pass behind the first is requested whole, as are short rows received two at a time.
// Rows on the FP8 wire (7168 columns, 8 ranks) gain while the front and the end of the dispatch count and lose a little in
// long ones, requested whole / spaced: 16 tokens 38.9 / 38.2, 128 103.9 / 103.0, 512 331.7 / 329.6, 2048 1271 / 1269, 8192 4987 / 4999.
constexpr int kReadWindow = 4;
// Reads the rows of receive tickets first_ticket .. first_ticket + count - 1 (already
// marked ready, count <= kRows) from their host slots and stores them to their
// destination rows.  Returns false when the wavefront must stop.
//
// Short rows are not bound by their bytes but by what a row costs the link and the queues whatever its
// length: its ACK, eight bytes in a line of host memory that the source's thread keeps
// fetching (33 ns each: a second store of every ACK adds exactly that), and its claim, an atomic on one word
// (12 ns).  They are therefore taken kRows at a time (receive_batch): consecutive tickets
// are mostly neighbouring slots of one source, so that their ACKs leave as one store.
template <bool kFp8, bool kVector, int kRows>
__device__ __forceinline__ bool rx_rows(const DeviceState& state, TransportQueues& q, uint32_t* scratch, int lane, int first_ticket, int count,
                       Owed& owed, const Deadline& deadline, bool& gate_open, bool& prefixes_known PCIE_EP_PROFILE(, RoleProfile& profile, bool sampled)) {
    const SegmentLayout& z = state.z;
    const int topk = z.dims.topk, me = state.local_rank, local = z.local_experts;
    const int hidden = z.dims.hidden;
    const uint64_t epoch = dispatch_epoch(state);
    const bool scatter = state.expand && state.fuse_expand;
    const __amdgpu_buffer_rsrc_t ring = device_resource(q.rx, sizeof(q.rx));
    constexpr int kEntryWords = int(sizeof(RxEntry) / 4);
    static_assert(kRows * kEntryWords <= kWave, "one lane per ticket word");
    // Lane 8 r + w: word w of row r's ticket.  Rows beyond `count` repeat the first one's ticket; their loads are
    // empty and nothing of theirs is stored.
    const int lane_row = lane / kEntryWords < count ? lane / kEntryWords : 0;
    const uint32_t word = device_load_b32(ring, uint32_t((first_ticket + lane_row) % kRing) * uint32_t(sizeof(RxEntry)) + uint32_t(lane % kEntryWords) * 4u);
    const auto entry = [&](int row, int index) { return __builtin_amdgcn_readlane(int(word), row * kEntryWords + index); };
    int source[kRows], ticket_token[kRows], channel[kRows];
    uint64_t payload_sequence[kRows];
    const char* slot_base[kRows];
    PCIE_EP_PROFILE(profile.first(kProfileFirstEntryNs);)
    // The tickets now live in registers: their ring entries may be reused while
    // this wavefront is still moving the rows.
    wait_memory_ops();
    if (lane < count) device_store(q.rx_taken + (first_ticket + lane) % kRing, sequence(epoch, first_ticket + lane));
    settle(state, q, owed, lane);  // in front of this row's requests and before any wait below
    fence_lds();
    uint32_t* owed_ack = owed.record + 4 * (lane < kRows ? lane : 0);
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        source[r] = entry(r, 0);
        const int slot = entry(r, 1);
        ticket_token[r] = entry(r, 2);
        channel[r] = entry(r, 3);
        payload_sequence[r] = uint64_t(uint32_t(entry(r, 4))) | uint64_t(uint32_t(entry(r, 5))) << 32;
        const bool replica = entry(r, 7) != 0;
        slot_base[r] = replica ? replica_slot_at(z, state.replica_in[source[r]], channel[r], slot) : slot_at(z, state.seg[source[r]], channel[r], slot);
        uint64_t* ack = replica ? replica_ack_at(z, state.seg[source[r]], channel[r], z.dims.rank_domain[me], slot, me)
                                : ack_at(z, state.seg[source[r]], channel[r], slot, me);
        if (lane == r) {
            // (payload_sequence[r] is this token's: checked below.)
            owed_ack[0] = uint32_t(reinterpret_cast<uint64_t>(ack));
            owed_ack[1] = uint32_t(reinterpret_cast<uint64_t>(ack) >> 32);
            owed_ack[2] = uint32_t(ticket_token[r]);
        }
    }
    if (lane == kWave - 1) test_delay(state.rx_delay);
    // Tickets are handed out from the first descriptor on, but no row is requested
    // before the producer of the prefixes has put its reads of the count mailboxes
    // on the link (a few hundred bytes that everything waits for must not queue
    // behind megabytes of row reads).  That producer has seen every source's counts by
    // then.  The prologue of the same launch may still be laying out thousands of own
    // tokens: count stores that leave with rows already in flight are acknowledged some
    // 12 us later than on an idle link (measured), so a peer whose counts came early
    // learns this rank's that much later.  It holds its first rows in registers for as
    // long, with their requests on the link - no link time is lost - and among ranks
    // that start together every gate opens after the last counts have arrived anyway.
    // The wavefront waits here with its tickets read and its addresses computed:
    // the requests leave the moment the gate opens.
    while (!gate_open) {
        int gate = 0;
        if (lane == 0) {
            if (device_load(state.receive_prefix_state) & kPrefixRequested) gate = 1;
            else if (aborted(q) || device_load(state.receive_prefix_state + 1) == kPrefixFailed) gate = -1;
            else if (deadline.expired(state)) {
                record_error(state, kErrRingProgressWait);
                raise_abort(q);
                gate = -1;
            }
        }
        gate = broadcast_first(gate);
        if (gate < 0) return false;
        if (gate > 0) gate_open = true;
        else __builtin_amdgcn_s_sleep(24);
    }
    PCIE_EP_PROFILE(profile.first(kProfileGateOpenNs);)
    // Column 0 of the receive/expand diagnostic: a row's host read starts
    // while an earlier row of the channel has not finished its scatter (the
    // conservative proof point of fused_receive.cuh:216-225; a count, not a time).
    if (state.overlap_diagnostic && lane < count) {
        int my_channel = 0, channel_ordinal = 0;
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            if (lane == r) {
                my_channel = channel[r];
                channel_ordinal = entry(r, 6);
            }
        }
        if (channel_ordinal > 0 && int(device_load(&q.rx_retired[my_channel].value)) < channel_ordinal)
            atomicAdd(reinterpret_cast<unsigned long long*>(state.receive_expand_overlap + my_channel * 2), 1ull);
    }

    PCIE_EP_PROFILE(const uint64_t request_begin = sampled ? profile.now() : 0;)
    // Whole wire vectors of a row, and with a ragged row (any length and any alignment of the destination rows:
    // one more wire vector, of which `rest` bytes of BF16 are stored).  Byte by byte such a row was one host read
    // and one store per element: 1536 tokens of 1000 columns on the FP8 wire, 8 ranks, top-4: 606 -> 315 us per dispatch.
    constexpr int kWireItems = kFp8 ? kPassItems / 2 : kRowPass<kVector>;  // wire vectors a lane holds
    constexpr int kRowItems = kWireItems / kRows;                          // of one row
    constexpr int kOutPerWire = kFp8 ? 2 : 1;                              // a code vector fills two BF16 vectors
    // FP8 rows are decoded as a whole, in place, and then stored destination by destination; ragged ones vector by
    // vector as they are stored, to all destinations, in half the registers (row_load_pass says what those are for).
    constexpr bool kDecodeInPlace = kFp8 && kVector, kDecodeAtStore = kFp8 && !kVector;
    constexpr int kWirePass = kRowItems * kWave;
    const int wire_vectors = kFp8 ? hidden / 16 : hidden / 8;
    const int rest = kVector ? 0 : (kFp8 ? hidden % 16 : hidden % 8) * 2;
    const int wire_total = wire_vectors + (rest ? 1 : 0);
    // Several rows are rows of one pass (receive_batch).
    static_assert(kRows == 1 || (kFp8 ? kBatchedFp8Columns : kBatchedBf16SlotBytes) <= kWirePass * 16, "a batched row must fit its share of the registers");
    // Metadata first (it arrives first), payload right behind it; lanes behind a row read 0.  A ragged row's last wire
    // vector is read whole: the slot's payload is padded to 16 bytes, the padding is not used.
    u32x4 meta_vector[kRows];
    RowItems<kDecodeInPlace ? 2 * kWireItems : kWireItems> row;
#pragma unroll
    for (int r = 0; r < kRows; ++r)
        meta_vector[r] = host_load_b128(host_resource(slot_base[r] + z.meta_offset, r < count ? uint32_t(z.meta_bytes) : 0u), uint32_t(lane) * 16u);
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const __amdgpu_buffer_rsrc_t payload = host_resource(slot_base[r], r < count ? uint32_t(z.meta_offset) : 0u);
        // First (usually only) pass of the row.
#pragma unroll
        for (int j = 0; j < kRowItems; ++j) {
            if (kRows == 1 && j >= kReadWindow && j * kWave < wire_total) asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kReadWindow - 1) : "memory");
            row.v[r * kRowItems + j] = host_load_b128(payload, uint32_t(j * kWave + lane) * 16u);
        }
    }
    PCIE_EP_PROFILE(profile.first(kProfileFirstRequestNs);)
    const int meta_dwords = z.meta_bytes / 4;  // a multiple of four; kRows records fit the scratch (receive_batch)
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        if (r < count && lane < meta_dwords / 4) {
            uint32_t* record = scratch + r * meta_dwords + lane * 4;
            record[0] = meta_vector[r][0];
            record[1] = meta_vector[r][1];
            record[2] = meta_vector[r][2];
            record[3] = meta_vector[r][3];
        }
    }
    fence_lds();
    PCIE_EP_PROFILE(profile.first(kProfileFirstDataNs);)
    bool stranger = false;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        const int token = int(scratch[r < count ? r * meta_dwords : 0]);
        stranger |= r < count && (token != ticket_token[r] || payload_sequence[r] != sequence(epoch, token));
    }
    if (__any(stranger)) {
        // Terminal: never forge an ACK for a slot whose identity is unknown
        // (advanced_dispatch.cuh:607-610).
        if (lane == 0) {
            record_error(state, kErrPayloadSequence);
            raise_abort(q);
        }
        return false;
    }

    // The rows have been requested; where they go depends on the receive prefixes,
    // which may still be on their way in the first microseconds of the kernel.
    PCIE_EP_PROFILE(const uint64_t prefix_begin = sampled ? profile.now() : 0;)
    while (!prefixes_known) {
        const int verdict = receive_prefix_verdict(state, epoch, lane);
        if (verdict < 0 || broadcast_first(aborted(q) ? 1 : 0)) return false;
        if (verdict > 0) prefixes_known = true;
        // The row itself is microseconds away: a slow poll costs nothing, and a couple of hundred
        // wavefronts polling fast would slow down the very stores of the prefixes they wait for.
        else __builtin_amdgcn_s_sleep(48);
    }

    PCIE_EP_PROFILE(if (sampled) profile.add(kProfileRxPrefixWaitSum, profile.now() - prefix_begin);)
    // Destination rows, one lane per branch.  Everything the row numbers are
    // made of comes from the peer: the token must be addressed to this rank and
    // its ordinals must lie inside the counts that peer announced, or a store
    // would land in another expert's rows or before the pool.  Same verdict as a
    // wrong identity: terminal, and the slot is not ACKed.
    // The prefixes of all rows are requested before the first is used.
    int my_expert[kRows], before[kRows], through[kRows], offset[kRows], first[kRows], end[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        my_expert[r] = -1;
        before[r] = through[r] = offset[r] = first[r] = end[r] = 0;
        if (r >= count) continue;
        if (lane < topk) {
            const int global_expert = int(scratch[r * meta_dwords + kMetaBranchOffset / 4 + lane]);
            const int expert = global_expert - me * local;
            if (global_expert >= 0 && expert >= 0 && expert < local) {
                my_expert[r] = expert;
                before[r] = device_load(state.source_expert_prefix + source[r] * local + expert);
                through[r] = source[r] + 1 < z.dims.num_ranks ? device_load(state.source_expert_prefix + (source[r] + 1) * local + expert)
                                                              : device_load(state.expert_counts + expert);
                if (scatter) offset[r] = device_load(state.expert_offsets + expert);
            }
        }
        if (lane == 0) {
            first[r] = device_load(state.source_offsets + source[r]);
            end[r] = device_load(state.source_offsets + source[r] + 1);
        }
    }
    int64_t my_row[kRows];
    const int64_t capacity = scatter ? state.expanded_capacity : unique_capacity(z.dims);
    bool out_of_range = false, beyond = false;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        my_row[r] = -1;
        if (r >= count) continue;
        const uint32_t* record = scratch + r * meta_dwords;
        out_of_range |= lane == 0 && !((record[1] >> me) & 1u);
        if (my_expert[r] >= 0) {
            const int ordinal = int(record[kMetaBranchOffset / 4 + topk + lane]);
            out_of_range |= ordinal < 0 || ordinal >= through[r] - before[r];
            if (scatter) my_row[r] = int64_t(offset[r]) + before[r] + ordinal;
        }
        if (lane == 0) {
            const int ordinal = int(record[kMetaRankOrdinalsOffset / 4 + me]);
            out_of_range |= ordinal < 0 || ordinal >= end[r] - first[r];
            if (!scatter) my_row[r] = int64_t(first[r]) + ordinal;
        }
        beyond |= my_row[r] >= capacity;
    }
    if (__any(out_of_range)) {
        if (lane == 0) {
            record_error(state, kErrPayloadSequence);
            raise_abort(q);
        }
        return false;
    }
    if (__any(beyond)) {
        if (lane == 0) {
            record_error(state, kErrExpandedCapacity);
            raise_abort(q);
        }
        return false;
    }
    uint16_t* output_base = scatter ? state.expanded_payload : state.unique_payload;
    if (lane == kWave - 1) test_delay(state.scatter_delay);

    for (int first_wire = 0; first_wire < wire_total; first_wire += kWirePass) {  // one pass with several rows
        if (kRows == 1 && first_wire > 0) {
            const __amdgpu_buffer_rsrc_t payload = host_resource(slot_base[0], uint32_t(z.meta_offset));
#pragma unroll
            for (int j = 0; j < kRowItems; ++j) row.v[j] = host_load_b128(payload, uint32_t(first_wire + j * kWave + lane) * 16u);
        }
        const bool last_pass = kRows > 1 || first_wire + kWirePass >= wire_total;
        if (last_pass) {
            // All loads of the staged rows have returned: the host slots may be released.
            wait_memory_ops();
            owed.acks = count;
            if (owed.prompt) settle_acks(state, owed, lane);
            PCIE_EP_PROFILE(if (sampled) profile.add(kProfileRxRequestSum, profile.now() - request_begin);)
        }
        if constexpr (kDecodeInPlace) {
            // 16 codes -> 16 BF16 (two 16-byte vectors); expanded in place from the top.
#pragma unroll
            for (int j = kWireItems - 1; j >= 0; --j) {
                u32x4 lo, hi;
                dequantize_vector(row.v[j], bits_float(scratch[(j / kRowItems < count ? j / kRowItems : 0) * meta_dwords + 2]), lo, hi);
                row.v[2 * j] = lo;
                row.v[2 * j + 1] = hi;
            }
        }
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
            if (r >= count) break;
            const uint64_t destinations = __ballot(my_row[r] >= 0);
            constexpr int kAtATime = kDecodeAtStore ? 1 : kRowItems;  // items that go to one destination before the next
#pragma unroll
            for (int item = 0; item < kRowItems; item += kAtATime) {
                u32x4 decoded[2];
                if constexpr (kDecodeAtStore) dequantize_vector(row.v[r * kRowItems + item], bits_float(scratch[r * meta_dwords + 2]), decoded[0], decoded[1]);
                uint64_t remaining = destinations;
                while (remaining) {
                    const int branch = __builtin_ctzll(remaining);
                    remaining &= remaining - 1;
                    uint16_t* output = output_base + size_t(__shfl(my_row[r], branch)) * hidden;
#pragma unroll
                    for (int j = item; j < item + kAtATime; ++j) {
                        // Wire vector i of an FP8 row holds elements [16 i, 16 i + 16): output vectors 2 i and 2 i + 1.
                        const int index = first_wire + j * kWave + lane;
                        const int held = (r * kRowItems + j) * kOutPerWire;
                        if (index < wire_vectors) {
#pragma unroll
                            for (int half = 0; half < kOutPerWire; ++half)
                                row_store_vector<kVector>(output, index * kOutPerWire + half, kDecodeAtStore ? decoded[half] : row.v[held + half]);
                        }
                        if constexpr (!kVector) {
                            // The ragged row's last wire vector.
                            if (rest && index == wire_vectors) {
                                char* tail = reinterpret_cast<char*>(output) + size_t(wire_vectors) * (kOutPerWire * 16);
                                const u32x4 value = kDecodeAtStore ? decoded[0] : row.v[held];
                                if (kFp8 && rest >= 16) {
                                    row_store_vector<false>(tail, 0, value);
                                    store_rest(tail + 16, rest - 16, decoded[1]);
                                } else {
                                    store_rest(tail, rest, value);
                                }
                            }
                        }
                    }
                }
            }
        }
    }

    // Row metadata (advanced_layout.cuh:207-215; layout.cuh:31-48).
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
        if (r >= count) break;
        const uint32_t* record = scratch + r * meta_dwords;
        if (scatter) {
            if (my_row[r] >= 0) {
                state.expanded_expert_idx[my_row[r]] = my_expert[r];
                state.expanded_weights[my_row[r]] = bits_float(record[kMetaBranchOffset / 4 + 2 * topk + lane]);
                state.expanded_source_meta[my_row[r] * 3] = source[r];
                state.expanded_source_meta[my_row[r] * 3 + 1] = ticket_token[r];
                state.expanded_source_meta[my_row[r] * 3 + 2] = lane;
            }
        } else {
            const int64_t out_row = __shfl(my_row[r], 0);
            if (lane < topk) {
                const int expert = int(record[kMetaBranchOffset / 4 + lane]);
                const bool is_local = expert >= me * local && expert < (me + 1) * local;
                state.unique_topk_idx[out_row * topk + lane] = is_local ? expert - me * local : -1;
                state.unique_topk_weights[out_row * topk + lane] = is_local ? bits_float(record[kMetaBranchOffset / 4 + 2 * topk + lane]) : 0.0f;
                state.unique_expert_ordinals[out_row * topk + lane] = int(record[kMetaBranchOffset / 4 + topk + lane]);
            }
            if (lane == 0) {
                state.unique_source_meta[out_row * 3] = source[r];
                state.unique_source_meta[out_row * 3 + 1] = ticket_token[r];
                state.unique_source_meta[out_row * 3 + 2] = -1;
            }
        }
    }
    count_rows(owed.record, kCountReads, count, lane);
    PCIE_EP_PROFILE(if (sampled) profile.add(kProfileRxScatterSum, profile.now() - request_begin);)
    fence_lds();  // scratch is reused by the next tickets
    if (lane < count) {
        int my_channel = channel[0];
#pragma unroll
        for (int r = 1; r < kRows; ++r)
            if (lane == r) my_channel = channel[r];
        device_add(&q.rx_retired[my_channel].value, 1u);
    }
    return true;
}

// ---------------------------------------------------------------------------------------
// Payload wavefront: moves rows of either direction
// ---------------------------------------------------------------------------------------
// A payload wavefront serves whichever direction needs it.  The two directions
// share the host link: row reads return on the downstream half, but their
// requests travel upstream beside the row writes, so a transmit side that runs
// flat out (about 24 GB/s next to saturated reads) takes request slots from the
// receive side (55 instead of 57 GB/s) and is then idle for the rest of the
// dispatch.  The wavefronts therefore split in proportion to the work that is
// LEFT in each direction: with rem_tx and rem_rx rows still unclaimed,
//     transmitting wavefronts : receiving wavefronts = kTxWeight * rem_tx : kRxWeight * (rem_rx - lead)
// (one wavefront's share of the link's write rate is about 4/9 of its share of
// the read rate; on the FP8 wire, where a transmitted row is half the bytes, read from
// HBM once, it is about the same), re-evaluated before every claim, so the writes are spread
// thinly over the whole dispatch whatever the routing's send/receive ratio is.
// `lead` makes the transmit side end a little earlier than the receive side (by
// the time the link needs for kTxLeadBytes, at most a quarter of the rows to
// receive): a transmitted row is only finished
// when its receivers have acknowledged it, and that round trip then hides
// behind the last received rows instead of following them.  The rule corrects
// itself: a direction that falls behind has more left and gets more wavefronts;
// at most transmit_wavefronts() of them transmit and, while anything is left to send, at
// least kMinTxWaves of those.  Until both totals are known (the receive total comes with
// the receive prefixes) those kMinTxWaves transmit and everybody else waits for
// the first descriptors.  A wavefront whose direction has nothing to
// claim takes a ticket of the other direction instead - at once when its own
// direction is finished, after kIdleCrossoverUs otherwise (at the start of a
// dispatch the first descriptors are a few microseconds away and a receive
// wavefront must not bind itself to a transmit row for them) - but only a
// ticket its producer has already reserved (head < tail), so it never commits
// itself to a row that does not exist yet.
// FP8 rows of 7168 columns, 8 ranks, us per dispatch with 9 : 4 (the writes crowd the beginning) and with 4 : 4: 2048
// tokens top-8 1275 / 1257, 8192 tokens 5070 / 5030, 2000 tokens hotspot top-4 872 / 848, 64-token graph replay 79 / 79;
// 4 ranks top-2, mostly transmitting, 427 / 427.  BF16, 2048 tokens: 2436 / 2441.
template <bool kFp8>
constexpr int64_t kTxWeight = kFp8 ? 4 : 9;
constexpr int64_t kRxWeight = 4;
constexpr int64_t kTxLeadBytes = 24 << 20;
constexpr int kMinTxWaves = 16;
constexpr uint64_t kIdleCrossoverUs = 30;
constexpr int kPreGateRows = 32;

template <bool kFp8, bool kVector, int kRows>
__device__ __forceinline__ void payload_worker(const DeviceState& state, TransportQueues& q, uint32_t* scratch, uint32_t* owed_record, int lane, int order, int waves, bool direct) {
    const uint64_t epoch = dispatch_epoch(state);
    Deadline deadline(now_ticks());
    if (lane < kWorkerCounts) owed_record[kOwedCounts + lane] = 0;
    Owed owed{owed_record};
    PCIE_EP_PROFILE(RoleProfile profile(state.clock_khz); uint64_t idle_begin = 0; int moves = 0;)
    bool prefixes_known = false, gate_open = false, plan_known = state.fused == 0;
    const int lead = int(kTxLeadBytes / int64_t(state.z.meta_offset + state.z.meta_bytes));
    const int transmitters = transmit_wavefronts(waves, kRows);
    // A wavefront that may be wanted for transmitting binds itself to one batch at a time.
    const int most_claims = 2 * order < waves || kRows == 1 ? kRows : kReceiveClaims;
    uint64_t idle_since = 0;  // 0: the last look found work
    fence_lds();
    bool go_on = true;
    direct = broadcast_first(direct ? 1 : 0) != 0;  // uniform, for the compiler too
    while (go_on) {
        // 0: nothing to do now, 1: transmit, 2: receive, -1: both directions are finished or the kernel aborts.
        // A direct row comes first and needs neither a look nor a ticket.
        int choice = direct ? 1 : 0, claims = 1, prompt = 1;
        PCIE_EP_PROFILE(const uint64_t look_begin = profile.now();)
        int gate_seen = gate_open ? 1 : 0;
        if (lane == 0 && !direct) {
            if (aborted(q)) choice = -1;
            else {
                const int tx_head = int(device_load(&q.tx_head.value)), rx_head = int(device_load(&q.rx_head.value));
                const bool tx_backlog = tx_head < int(device_load(&q.tx_tail.value));
                const int rx_tail = int(device_load(&q.rx_tail.value));
                bool rx_backlog = rx_head < rx_tail;
                // Receive tickets are there long before the first row may be requested (rx_rows
                // holds the gate).  Only the first kPreGateRows of them are claimed ahead of
                // it, by wavefronts that then wait with their addresses ready: if every
                // wavefront did, they would all fire at once and each would have its first
                // row after the time the link needs for all of them, with nobody left to transmit.
                if (rx_backlog && !gate_seen && rx_head >= kPreGateRows) {
                    gate_seen = (device_load(state.receive_prefix_state) & kPrefixRequested) != 0;
                    rx_backlog = gate_seen != 0;
                }
                // Tickets of the dispatch: its rows but for the direct ones.
                int tx_total = device_load(&q.tx_head.total);
                const int rx_total = device_load(&q.rx_head.total), tx_direct = device_load(&q.tx_head.direct);
                if (tx_total >= 0) tx_total -= tx_direct;
                const bool tx_done = tx_total >= 0 && tx_head >= tx_total, rx_done = rx_total >= 0 && rx_head >= rx_total;
                // Totals unknown: a handful of wavefronts start to transmit, the others
                // wait for the first descriptors.
                bool prefer_tx = order < kMinTxWaves && order < transmitters;
                if (tx_total >= 0 && rx_total >= 0) {
                    const int rx_rows = rx_total - rx_head - (lead < rx_total / 4 ? lead : rx_total / 4);
                    const int64_t tx_left = tx_done ? 0 : kTxWeight<kFp8> * (tx_total - tx_head), rx_left = rx_rows > 0 ? kRxWeight * rx_rows : 0;
                    prefer_tx = rx_done || (tx_left > 0 && order < transmitters &&
                                            (order < kMinTxWaves || int64_t(order) * (tx_left + rx_left) < int64_t(waves) * tx_left));
                }
                const bool own_backlog = prefer_tx ? tx_backlog : rx_backlog, other_backlog = prefer_tx ? rx_backlog : tx_backlog;
                const bool own_done = prefer_tx ? tx_done : rx_done;
                if (own_backlog) choice = prefer_tx ? 1 : 2;
                else if (other_backlog) {
                    const uint64_t now = now_ticks();
                    if (!idle_since) idle_since = now;
                    // Towards the receive side after a while; towards the transmit side only once
                    // everything has been received.  A transmit row waits for its receivers (slot ACK,
                    // descriptor credit); if every wavefront of a rank could end up in such a wait, two
                    // ranks whose receivers are each other's kernels could wait for each other for ever.
                    // The wavefronts that do not transmit by the rule above (transmit_wavefronts())
                    // therefore never do while a row may still come in.
                    if (own_done || (prefer_tx && now - idle_since > kIdleCrossoverUs * state.clock_khz / 1000)) choice = prefer_tx ? 2 : 1;
                }
                const int total = choice == 1 ? tx_total : rx_total;
                prompt = total < 0 || total - (choice == 1 ? tx_head : rx_head) <= waves;
                // A receiving wavefront takes its share of the tickets that are there, at most most_claims.
                if (choice == 2) {
                    const int share = (rx_tail - rx_head) / waves;
                    claims = share < 1 ? 1 : (share < most_claims ? share : most_claims);
                    if (kRows > 1 && !gate_seen && claims > kPreGateRows - rx_head) claims = kPreGateRows - rx_head;  // at least one is left: see rx_backlog
                }
                if (choice) idle_since = 0;
                else {
                    if (tx_done && rx_done) choice = -1;
                    else if (deadline.expired(state)) {
                        record_error(state, kErrRingProgressWait);
                        raise_abort(q);
                        choice = -1;
                    }
                }
            }
        }
        choice = broadcast_first(choice);
        gate_open = broadcast_first(gate_seen) != 0;
        if (choice < 0) break;
        if (choice == 0) {
            wait_memory_ops();
            settle(state, q, owed, lane);
            PCIE_EP_PROFILE(if (!idle_begin) idle_begin = profile.now();)
            // Every look is seven loads of the queue counters; a couple of hundred idle wavefronts
            // looking four times a microsecond would keep the producers' own updates of those
            // counters waiting.  About a microsecond between looks.
            __builtin_amdgcn_s_sleep(32);
            continue;
        }
        PCIE_EP_PROFILE(if (idle_begin) { profile.add(kProfileIdleSum, profile.now() - idle_begin); idle_begin = 0; })
        const bool transmit = choice == 1;
        QueueCounter& head = transmit ? q.tx_head : q.rx_head;
        PCIE_EP_PROFILE(profile.first(kProfileFirstClaimNs); const uint64_t claim_begin = profile.now(); if (!profile.values[kProfileFirstLookNs]) profile.values[kProfileFirstLookNs] = look_begin;)
        claims = broadcast_first(claims);
        owed.prompt = broadcast_first(prompt) != 0;
        int ticket_index = direct ? 0 : claim_tickets(head, claims, lane);
        const int end = ticket_index + claims;
        // Several wavefronts may have seen the same backlog: a claim beyond the last
        // ticket of the dispatch is simply dropped, an earlier one waits for its tag.
        // Rows whose tickets are ready never wait for a later ticket of the same claim: a
        // source may publish that one only when it has seen these rows acknowledged.
        while (go_on && ticket_index < end) {
            if (!direct && wait_ticket(state, q, transmit ? q.tx_ready : q.rx_ready, head, ticket_index, epoch, lane, deadline, [&] {
                    wait_memory_ops();
                    settle(state, q, owed, lane);
                }) < 0) {
                if (broadcast_first(aborted(q) ? 1 : 0)) go_on = false;
                break;
            }
            PCIE_EP_PROFILE(profile.first(kProfileFirstTaggedNs); profile.add(kProfileTicketWaitSum, profile.now() - claim_begin); const bool sampled = !direct && moves++ % kProfileSampleStride == 0;
                            if (sampled) profile.add(transmit ? kProfileSampledTxRows : kProfileSampledRxRows);)
            int count = 1;
            if (transmit) {
                go_on = tx_row<kFp8, kVector, kRows>(state, q, scratch, lane, ticket_index, direct, deadline, owed, plan_known PCIE_EP_PROFILE(, profile, sampled));
            } else {
                if constexpr (kRows > 1) {
                    const bool ready = lane < kRows && lane < end - ticket_index &&
                                       (lane == 0 || device_load(q.rx_ready + (ticket_index + lane) % kRing) == sequence(epoch, ticket_index + lane));
                    count = __builtin_ctzll(~__ballot(ready));
                }
                go_on = rx_rows<kFp8, kVector, kRows>(state, q, scratch, lane, ticket_index, count, owed, deadline, gate_open, prefixes_known PCIE_EP_PROFILE(, profile, sampled));
            }
            direct = false;
            ticket_index += count;
            PCIE_EP_PROFILE(profile.add(transmit ? kProfileTxRows : kProfileRxRows, uint64_t(count)); profile.last(kProfileLastRowNs);)
        }
    }
    wait_memory_ops();
    settle(state, q, owed, lane);
    // Workers serve every channel; their counts go to channel 0's row of the
    // per-channel statistics, whose column sums are what callers read.
    if (lane == 0) {
        auto* stats = reinterpret_cast<unsigned long long*>(state.channel_stats);
        const uint32_t* counts = owed_record + kOwedCounts;
        if (counts[kCountWrites] || counts[kCountCreditMiss]) {
            atomicAdd(stats + kStatHostWrites, static_cast<unsigned long long>(counts[kCountWrites]));
            atomicAdd(stats + kStatDeliveries, static_cast<unsigned long long>(counts[kCountDeliveries]));
            atomicAdd(stats + kStatDescriptors, static_cast<unsigned long long>(counts[kCountPublished]));
            atomicAdd(stats + kStatTxCreditMiss, static_cast<unsigned long long>(counts[kCountCreditMiss]));
        }
        if (counts[kCountReads]) atomicAdd(stats + kStatHostReads, static_cast<unsigned long long>(counts[kCountReads]));
    }
    PCIE_EP_PROFILE(profile.values[kProfileItems] = uint64_t(moves); profile.save(state.profiling, 2 * state.z.dims.channels + order, lane);)
}

// Workgroup b < C is the control workgroup of channel b (wavefront 0 TX control,
// wavefront 1 RX control); workgroups b >= C hold payload wavefronts only.  With
// no payload workgroups configured the control workgroups carry the payload
// wavefronts themselves.
template <bool kFp8, bool kVector, int kRows>
__global__ void __launch_bounds__(kTransportMaxThreads, kVector ? 3 : 4) transport_kernel(DeviceState launch_state) {
    // The launch argument is read where it lies, in the kernel-argument segment:
    // every field is then a scalar load from constant memory and every pointer in
    // it a global pointer.  A by-value copy would be a private object of 1 KB that
    // each role reads back through scratch loads, with generic pointers in it.
#if defined(__HIP_DEVICE_COMPILE__)
    const DeviceState& state = *reinterpret_cast<const DeviceState*>(__builtin_amdgcn_kernarg_segment_ptr());
#else
    const DeviceState& state = launch_state;  // the host pass only parses the kernel
#endif
    // The tables of a workgroup of the prologue, or one WaveScratch per wavefront of any other.
    extern __shared__ __align__(16) unsigned char dynamic_lds[];
    __shared__ int epoch_begun;
    const int channels = state.z.dims.channels;
    int block = transport_block(transport_grid(state), int(blockIdx.x));
    if (block < 0) return;  // a filler id
    int wave = threadIdx.x / kWave;
    const int lane = threadIdx.x % kWave;
    WaveScratch& own_scratch = reinterpret_cast<WaveScratch*>(dynamic_lds)[wave];
    uint32_t *scratch = own_scratch.words, *owed_record = own_scratch.owed;
    TransportQueues& q = *state.queues;
    const int payload_waves = state.tx_waves + state.rx_waves;
    const int payload_groups = state.worker_groups > 0 ? state.worker_groups : 0;
    const int waves_per_group = int(blockDim.x) / kWave;
    const int prologue_groups = fused_prologue_groups(state);
    // Role wavefronts of the launch: controls, payload and local-bypass wavefronts, the producer of the receive
    // prefixes where it is a wavefront of its own, one per prologue workgroup and a second one for the epoch begin.
    const uint32_t roles = uint32_t(2 * channels + (payload_groups ? payload_groups : channels) * payload_waves + state.local_groups * waves_per_group +
                                    (dedicated_prefix_producer(state) ? 1 : 0) + prologue_groups + (prologue_groups ? 1 : 0));
    bool begun = true;
    if (state.fused) {
        // The prologue's workgroups carry the lowest indices: they are started first.
        // Workgroup 0 begins the epoch, the ones after it lay out one chunk of tokens each.
        if (block < prologue_groups) {
            if (block == 0) {
                // The helpers' findings: zeroed before any wavefront of the workgroup goes its own way.
                __shared__ int findings[kTransportMaxThreads / kWave];
                if (threadIdx.x < kTransportMaxThreads / kWave) findings[threadIdx.x] = 0;
                __syncthreads();
                epoch_begin_role(state, wave, lane, waves_per_group, findings);
                if (wave >= 2) return;
                return finish_role(state, q, lane, roles);
            }
            prologue_chunk<8, true>(state, dynamic_lds, waves_per_group, state.prologue_chunks, block - 1);
            if (wave == 0) finish_role(state, q, lane, roles);
            return;
        }
        block -= prologue_groups;
    }
    const int channel_groups = control_groups(state);
    // Which control this wavefront is, if any - known before the role may start.  The two roles whose first
    // action is a read over the host link issue it now: a receive control its first look at the descriptor
    // queues, the producer of the prefixes its first look at the sources' counts_ready.  The wait for the epoch
    // begin (the queues are being reset; 3 us into the launch) then runs inside that round trip (4.4 us).
    const bool control_of_pair = payload_groups && block < channel_groups;
    const bool transmit_group = control_of_pair && (block + prologue_groups) % kControlXcds == 0;
    const bool prefix_producer = transmit_group && block / 2 == 0 && wave == 2 && dedicated_prefix_producer(state);
    int receive_channel = -1;
    if (control_of_pair && !transmit_group && wave < 2 && 2 * (block / 2) + wave < channels) receive_channel = 2 * (block / 2) + wave;
    if (!payload_groups && block < channel_groups && wave == 1) receive_channel = block;
    RxFirstPoll first_poll{{0u, 0u, 0u, 0u}, false};
    if (receive_channel >= 0) first_poll = rx_first_poll(state, receive_channel, lane);
    // Position of a payload wavefront among all of them, wavefront-major: a
    // direction's share is spread over the workgroups before it doubles up in one.
    bool direct = false;
    if (payload_groups && block >= channel_groups && block < channel_groups + payload_groups && wave < payload_waves)
        direct = direct_row<kFp8, kVector, kRows>(state, owed_record + kDirectTicket, wave * payload_groups + block - channel_groups, lane);
    PrefixFirstLook first_look{0, false};
    if (prefix_producer) first_look = prefix_first_look(state, lane);
    if (state.fused) {
        // (LDS only: the reads and stores issued above stay in flight.)
        if (threadIdx.x == blockDim.x - kWave) epoch_begun = int(wait_for_begin(state, q));
        lds_barrier();
        begun = epoch_begun != 0;
    } else if (__syncthreads_or(threadIdx.x == 0 ? int(load_error_code(state) != 0) : 0)) {
        return;  // the prologue kernel in front of this one failed
    }
    if (block >= channel_groups + payload_groups) {
        if (begun) local_rows<kVector>(state, q, lane, (block - channel_groups - payload_groups) * waves_per_group + wave, state.local_groups * waves_per_group);
        return finish_role(state, q, lane, roles);
    }
    if (block < channel_groups) {
        if (payload_groups) {
            // Control workgroups of their own: the two control XCDs alternate over their
            // ids, and a workgroup holds the controls of ONE direction for a pair of
            // channels (wavefront w: channel 2 * pair + w), transmit on one XCD, receive
            // on the other.  A receive control polls descriptors in host memory all the
            // time, and each of those reads stays in its XCD's memory queues for as long
            // as the row reads in front of it on the link take; the transmit controls,
            // the producer of the prefixes and the prologue only touch device memory
            // while rows flow and must not wait behind them.
            const bool transmit = (block + prologue_groups) % kControlXcds == 0;
            const int pair = block / 2, channel = 2 * pair + wave;
            if (wave < 2) {
                if (channel >= channels) return;
                if (begun) {
                    if (transmit) tx_control(state, q, channel, lane);
                    else rx_control(state, q, channel, lane, first_poll);
                }
                return finish_role(state, q, lane, roles);
            }
            // The producer of the receive prefixes: third wavefront of the first transmit control workgroup.
            if (!prefix_producer) return;
            if (begun) receive_prefix_role(state, lane, first_look);
            return finish_role(state, q, lane, roles);
        }
        if (wave < 2) {
            if (begun) {
                if (wave == 0) tx_control(state, q, block, lane);
                else rx_control(state, q, block, lane, first_poll);
            }
            return finish_role(state, q, lane, roles);
        }
        wave -= 2;
    }
    if (wave >= payload_waves) return;
    const int groups = payload_groups ? payload_groups : channels;
    const int group = payload_groups ? block - channel_groups : block;
    if (begun) payload_worker<kFp8, kVector, kRows>(state, q, scratch, owed_record, lane, wave * groups + group, groups * payload_waves, direct);
    finish_role(state, q, lane, roles);
    // Every role loop has an explicit completion, abort or timeout exit and no
    // workgroup barrier follows the entry verdict.
}

}  // namespace

int transport_threads(const DeviceState& state) {
    const int payload = state.tx_waves + state.rx_waves;
    const int control = state.worker_groups > 0 ? 2 : 2 + payload;
    return (control > payload ? control : payload) * kWave;
}

// The instantiation that `state` selects.  Rows of whole 16-byte vectors on both sides (FP8: of whole 16-code
// vectors on the wire) lie on 16-byte boundaries and have nothing behind their vectors; all others take the
// ragged form of the row code.
static auto transport_instance(const DeviceState& state) {
    const bool fp8 = state.z.dims.wire_fp8 != 0;
    const bool vector = fp8 ? state.z.dims.hidden % 16 == 0 : state.z.dims.hidden % 8 == 0;
    if (receive_batch(state.z) > 1) {
        if (fp8) return vector ? transport_kernel<true, true, kMaxReceiveBatch> : transport_kernel<true, false, kMaxReceiveBatch>;
        return vector ? transport_kernel<false, true, kMaxReceiveBatch> : transport_kernel<false, false, kMaxReceiveBatch>;
    }
    if (fp8) return vector ? transport_kernel<true, true, 1> : transport_kernel<true, false, 1>;
    return vector ? transport_kernel<false, true, 1> : transport_kernel<false, false, 1>;
}

// LDS that a launch asks for beyond what the kernel declares.
static size_t transport_lds_bytes(const DeviceState& state, int threads) {
    const size_t scratch = size_t(threads / kWave) * sizeof(WaveScratch);
    const size_t tables = state.fused ? prologue_lds_bytes(state.z, threads / kWave) : 0;
    return scratch > tables ? scratch : tables;
}

// How many transport workgroups one compute unit holds at once (registers, LDS and
// wavefront slots of the instantiation that `state` selects).
hipError_t transport_workgroups_per_unit(const DeviceState& state, int* per_unit) {
    const int threads = transport_threads(state);
    if (threads > kTransportMaxThreads) return hipErrorInvalidValue;
    return hipOccupancyMaxActiveBlocksPerMultiprocessor(per_unit, transport_instance(state), threads, transport_lds_bytes(state, threads));
}

hipError_t launch_transport(const DeviceState& state, hipStream_t stream) {
    const dim3 grid(transport_grid(state).blocks), block(transport_threads(state));
    if (int(block.x) > kTransportMaxThreads) return hipErrorInvalidValue;
    // The prologue's chunks are the workgroup's own wavefronts; the conditions are those of fused_prologue_fits().
    if (state.fused && !fused_prologue_fits(state.z, int(block.x), state.z.dims.max_tokens)) return hipErrorInvalidValue;
    hipLaunchKernelGGL(transport_instance(state), grid, block, transport_lds_bytes(state, int(block.x)), stream, state);
    return hipGetLastError();
}

}  // namespace pcie_ep
