// Whole-row helpers executed by one 64-lane wavefront: plain copy, FP8 wire
// quantisation (per-token amax -> scale -> E4M3FN codes) and de-quantisation.
// The quantiser restates quantize_transport_payload of the reference
// (csrc/kernels/host_staged/quantization.cuh:34-71) for one wavefront per token.
#pragma once

#include "device_common.h"

namespace pcie_ep {

__device__ __forceinline__ float wave_max(float value) {
    for (int offset = 32; offset > 0; offset >>= 1) value = fmaxf(value, __shfl_xor(value, offset));
    return value;
}

// A row helper's kVector says that the row is whole 16-byte vectors on 16-byte
// boundaries (hidden % 8 == 0; of 16-code vectors too where it goes over the FP8 wire:
// hidden % 16 == 0).  Any other row takes the ragged form of the same code.

// BF16 row copy within device memory.
template <bool kVector>
__device__ __forceinline__ void copy_row(const uint16_t* input, uint16_t* output, int hidden, int lane) {
    const int vectors = hidden / 8, rest = row_rest<kVector>(hidden);
    for (int first = 0; first < vectors; first += kRowPass<kVector> * kWave) {
        RowItems<kRowPass<kVector>> row;
        row_load_pass<kVector>(row, input, first, vectors, lane);
        row_store_pass<kVector>(row, output, first, vectors, lane);
    }
    if (rest && lane == 0)
        store_rest(reinterpret_cast<char*>(output + vectors * 8), rest, load_rest(reinterpret_cast<const char*>(input + vectors * 8), rest));
}

// BF16 row from device memory into a host slot.  A ragged row's last vector is stored
// whole, zeros behind the row: the slot's payload is padded to 16 bytes.
template <bool kVector, typename BeforeStores>
__device__ __forceinline__ void copy_row_to_host(const uint16_t* input, __amdgpu_buffer_rsrc_t slot, int hidden, int lane, BeforeStores before_stores) {
    const int vectors = hidden / 8, rest = row_rest<kVector>(hidden);
    u32x4 last = {0u, 0u, 0u, 0u};
    if (rest && lane == 0) last = load_rest(reinterpret_cast<const char*>(input + vectors * 8), rest);
    for (int first = 0; first < vectors; first += kRowPass<kVector> * kWave) {
        RowItems<kRowPass<kVector>> row;
        row_load_pass<kVector>(row, input, first, vectors, lane);
        if (first == 0) before_stores();
#pragma unroll
        for (int j = 0; j < kRowPass<kVector>; ++j) {
            const int index = first + j * kWave + lane;
            if (index < vectors) host_store_b128(slot, uint32_t(index) * 16u, row.v[j]);
        }
    }
    if (vectors == 0) before_stores();
    if (rest && lane == 0) host_store_b128(slot, uint32_t(vectors) * 16u, last);
}

__device__ __forceinline__ float vector_amax(float amax, const u32x4& v) {
#pragma unroll
    for (int word = 0; word < 4; ++word) {
        amax = fmaxf(amax, fabsf(bits_float(v[word] << 16)));
        amax = fmaxf(amax, fabsf(bits_float(v[word] & 0xFFFF0000u)));
    }
    return amax;
}
// 16 BF16 (two vectors, elements in order) -> 16 codes.
__device__ __forceinline__ u32x4 quantize_vector(const u32x4& lo, const u32x4& hi, float inverse) {
    return u32x4{fp8_quantize_word(lo[0], lo[1], inverse), fp8_quantize_word(lo[2], lo[3], inverse), fp8_quantize_word(hi[0], hi[1], inverse),
                 fp8_quantize_word(hi[2], hi[3], inverse)};
}

// BF16 row from device memory as FP8 codes into a host slot; returns the row scale.  Every
// lane takes 16 elements (two 16-byte loads) at a time to 16 codes (one 16-byte store).
// A row of whole vectors and of up to kGroups * 1024 elements is read once and waits in registers for its maximum; a ragged
// one is read again (from the L2; 1536 tokens of 1000 columns 232 us per dispatch, 236 with the row held), which
// leaves its kernel the registers for a fourth workgroup on a compute unit.  A ragged row's last codes are stored as
// a whole vector, zeros behind the row.
template <bool kVector, int kGroups, typename BeforeStores>  // kGroups: 16-element groups a lane holds
__device__ __forceinline__ float quantize_row_to_host(const uint16_t* input, __amdgpu_buffer_rsrc_t slot, int hidden, int lane, BeforeStores before_stores) {
    const int groups = hidden / 16, rest = kVector ? 0 : hidden % 16 * 2;
    float amax = 0.0f;
    u32x4 last_lo = {0u, 0u, 0u, 0u}, last_hi = {0u, 0u, 0u, 0u};
    if (rest && lane == 0) {
        const char* from = reinterpret_cast<const char*>(input + groups * 16);
        last_lo = rest < 16 ? load_rest(from, rest) : *reinterpret_cast<const u32x4_any*>(from);
        if (rest > 16) last_hi = load_rest(from + 16, rest - 16);
        amax = vector_amax(vector_amax(amax, last_lo), last_hi);
    }
    RowItems<2 * kGroups> row;
    const bool resident = kVector && groups <= kGroups * kWave;
    if (resident) {
#pragma unroll
        for (int j = 0; j < kGroups; ++j) {
            const int group = j * kWave + lane;
            row.v[2 * j] = row.v[2 * j + 1] = u32x4{0u, 0u, 0u, 0u};
            if (group < groups) {
                row.v[2 * j] = row_load_vector<kVector>(input, 2 * group);
                row.v[2 * j + 1] = row_load_vector<kVector>(input, 2 * group + 1);
            }
        }
#pragma unroll
        for (int j = 0; j < 2 * kGroups; ++j) amax = vector_amax(amax, row.v[j]);
    } else {
        for (int index = lane; index < groups * 2; index += kWave) amax = vector_amax(amax, row_load_vector<false>(input, index));
    }
    amax = wave_max(amax);
    const float scale = fp8_scale_from_amax(amax);
    // Multiply by the correctly rounded FP32 reciprocal, as the reference does
    // (quantization.cuh:66; pcie_ep/quantization.py:27-29), not a division per element.
    const float inverse = 1.0f / scale;
    before_stores();
    if (resident) {
#pragma unroll
        for (int j = 0; j < kGroups; ++j) {
            const int group = j * kWave + lane;
            if (group < groups) host_store_b128(slot, uint32_t(group) * 16u, quantize_vector(row.v[2 * j], row.v[2 * j + 1], inverse));
        }
    } else {
        for (int group = lane; group < groups; group += kWave) {
            const u32x4 lo = row_load_vector<false>(input, 2 * group), hi = row_load_vector<false>(input, 2 * group + 1);
            host_store_b128(slot, uint32_t(group) * 16u, quantize_vector(lo, hi, inverse));
        }
    }
    if (rest && lane == 0) host_store_b128(slot, uint32_t(groups) * 16u, quantize_vector(last_lo, last_hi, inverse));
    return scale;
}

// 16 codes -> two 16-byte vectors of BF16 (elements in order).
__device__ __forceinline__ void dequantize_vector(const u32x4& codes, float scale, u32x4& lo, u32x4& hi) {
#pragma unroll
    for (int word = 0; word < 4; ++word) {
        const uint32_t c = codes[word];
        uint32_t a, b;
        fp8_dequantize_word(c, scale, a, b);
        if (word < 2) {
            lo[word * 2] = a;
            lo[word * 2 + 1] = b;
        } else {
            hi[(word - 2) * 2] = a;
            hi[(word - 2) * 2 + 1] = b;
        }
    }
}

// Store one BF16 row (read once, into registers, pass by pass) to every
// destination row named by the lanes whose `my_row >= 0`.
template <bool kVector>
__device__ __forceinline__ void scatter_row(const uint16_t* input, uint16_t* output_base, int hidden, int64_t my_row, int lane) {
    const uint64_t destinations = __ballot(my_row >= 0);
    if (!destinations) return;
    const int vectors = hidden / 8, rest = row_rest<kVector>(hidden);
    u32x4 last = {0u, 0u, 0u, 0u};
    if (rest && lane == 0) last = load_rest(reinterpret_cast<const char*>(input + vectors * 8), rest);
    // Also a row shorter than one vector takes one pass, for its rest.
    for (int first = 0; first == 0 || first < vectors; first += kRowPass<kVector> * kWave) {
        RowItems<kRowPass<kVector>> row;
        row_load_pass<kVector>(row, input, first, vectors, lane);
        uint64_t remaining = destinations;
        while (remaining) {
            const int owner = __builtin_ctzll(remaining);
            remaining &= remaining - 1;
            uint16_t* output = output_base + size_t(__shfl(my_row, owner)) * hidden;
            row_store_pass<kVector>(row, output, first, vectors, lane);
            if (rest && first == 0 && lane == 0) store_rest(reinterpret_cast<char*>(output + vectors * 8), rest, last);
        }
    }
}

template <bool kVector>
__device__ __forceinline__ void zero_row(uint16_t* output, int hidden, int lane) {
    const int vectors = hidden / 8, rest = row_rest<kVector>(hidden);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int index = lane; index < vectors; index += kWave) row_store_vector<kVector>(output, index, zero);
    if (rest && lane == 0) store_rest(reinterpret_cast<char*>(output + vectors * 8), rest, zero);
}

// Alignment gaps of the local experts, rows [offset + count, next offset) of each:
// payload 0, expert -1, weight 0, metadata -1 (advanced_layout.cuh:250-265).  The gap
// rows of all experts are counted through, and wavefront `wave` of `waves` takes rows
// wave, wave + waves, ...: a small batch under a wide alignment is nothing but gap rows
// (16 tokens in 128-row tiles: 150 rows in use, 3 800 to zero), and with one wavefront
// per expert its 124 rows one after the other were the longest path of the dispatch
// (transport kernel at 7168 columns, 128-row alignment: T=16 535 us, 59 with the rows
// dealt over the local-bypass workgroups; T=96 185 us, 146, which is what it takes
// without any gap).  A wavefront finds its
// rows without memory traffic of its own: lane l holds expert l's gap, and a wave-wide
// scan of the gaps locates every row.
// The prefixes are read with device-scope loads: inside the transport kernel
// they were written by another wavefront of the same launch.
template <bool kVector>
__device__ __forceinline__ void zero_padding_rows(const DeviceState& state, int wave, int waves, int lane) {
    const int hidden = state.z.dims.hidden, local = state.z.local_experts;
    int before = 0;  // gap rows of the experts in front of this group of 64
    for (int begin = 0; begin < local; begin += kWave) {
        const int expert = begin + lane;
        int first = 0, gap = 0;
        if (expert < local) {
            first = device_load(state.expert_prefix + expert);
            const int64_t next = device_load(state.expert_offsets + expert + 1);
            const int64_t end = next < state.expanded_capacity ? next : state.expanded_capacity;
            gap = end > first ? int(end - first) : 0;
        }
        int through = gap;
        for (int offset = 1; offset < kWave; offset <<= 1) {
            const int other = __shfl_up(through, offset);
            if (lane >= offset) through += other;
        }
        const int total = __shfl(through, kWave - 1);
        for (int index = (wave + waves - before % waves) % waves; index < total; index += waves) {
            const int owner = __builtin_ctzll(__ballot(through > index));
            const int64_t row = __shfl(first, owner) + (index - (__shfl(through, owner) - __shfl(gap, owner)));
            zero_row<kVector>(state.expanded_payload + size_t(row) * hidden, hidden, lane);
            if (lane == 0) {
                state.expanded_expert_idx[row] = -1;
                state.expanded_weights[row] = 0.0f;
                state.expanded_source_meta[row * 3] = state.expanded_source_meta[row * 3 + 1] = state.expanded_source_meta[row * 3 + 2] = -1;
            }
        }
        before += total;
    }
}

// Local bypass of one own token: it never touches the host ring and keeps the
// original BF16 even on an FP8 wire (advanced_layout.cuh:217-248).  Returns
// false when a destination row lies beyond the expanded capacity.
template <bool kVector>
__device__ __forceinline__ bool local_token_rows(const DeviceState& state, int token, int lane) {
    const SegmentLayout& z = state.z;
    const int ranks = z.dims.num_ranks, topk = z.dims.topk, me = state.local_rank, local = z.local_experts;
    const int hidden = z.dims.hidden;
    if (!((state.plan_mask[token] >> me) & 1u)) return true;
    const uint16_t* input = state.x + size_t(token) * hidden;
    float weight = 1.0f;
    int expert_global = -1, ordinal = -1;
    if (lane < topk) {
        expert_global = state.plan_exp_idx[size_t(token) * topk + lane];
        ordinal = state.plan_exp_ord[size_t(token) * topk + lane];
        if (state.topk_weights) weight = state.topk_weights[size_t(token) * topk + lane];
    }
    const int expert = expert_global - me * local;
    const bool is_local = expert_global >= 0 && expert >= 0 && expert < local;
    if (state.expand && state.fuse_expand) {
        int64_t my_row = -1;
        if (is_local)
            my_row = int64_t(device_load(state.expert_offsets + expert)) + device_load(state.source_expert_prefix + me * local + expert) + ordinal;
        if (__any(my_row >= state.expanded_capacity)) return false;
        scatter_row<kVector>(input, state.expanded_payload, hidden, my_row, lane);
        if (my_row >= 0) {
            state.expanded_expert_idx[my_row] = expert;
            state.expanded_weights[my_row] = weight;
            state.expanded_source_meta[my_row * 3] = me;
            state.expanded_source_meta[my_row * 3 + 1] = token;
            state.expanded_source_meta[my_row * 3 + 2] = lane;
        }
    } else {
        const int64_t row = int64_t(device_load(state.source_offsets + me)) + state.plan_rank_ord[size_t(token) * ranks + me];
        copy_row<kVector>(input, state.unique_payload + size_t(row) * hidden, hidden, lane);
        if (lane < topk) {
            state.unique_topk_idx[row * topk + lane] = is_local ? expert : -1;
            state.unique_topk_weights[row * topk + lane] = is_local ? weight : 0.0f;
            state.unique_expert_ordinals[row * topk + lane] = ordinal;
        }
        if (lane == 0) {
            state.unique_source_meta[row * 3] = me;
            state.unique_source_meta[row * 3 + 1] = token;
            state.unique_source_meta[row * 3 + 2] = -1;
        }
    }
    return true;
}

}  // namespace pcie_ep
