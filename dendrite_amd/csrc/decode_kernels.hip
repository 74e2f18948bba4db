// Kernels of decode and prefill plans, of the merges and of the pool's small
// copies, and their launchers.  The items they run are in attend_device.hpp.
#include "attend_device.hpp"

namespace dh {
namespace {

// ---------------------------------------------------------------- attend16
// q in bf16 (KV bf16 / FP8 E4M3 / MXFP8) or f16 (KV f16); bf16/f16 MFMA.
// Partial-row layout seen by the merge: a lane loads 16 bytes of a state row.
template <int D, uint32_t OUT>
struct MergeShape {
    static constexpr int ES = OUT == 2 ? 4 : 2;      // bytes per partial element (f32 or scaled f16)
    static constexpr int EPL = 16 / ES;              // elements per lane per load
    static constexpr int LPS = D / EPL;              // lanes per state row
    static constexpr int SPI = 64 / LPS;             // states per load instruction
    static constexpr int MAX_NV = 64 / SPI < 16 ? 64 / SPI : 16;
    static_assert(LPS >= 1 && LPS <= 64 && 64 % LPS == 0, "head_dim");
    // loads per pass for rows of at most `states` states (a power of two)
    static constexpr int nv_for(int states) {
        int need = (states + SPI - 1) / SPI, nv = 1;
        while (nv < need && nv < MAX_NV) nv *= 2;
        return nv;
    }
};

template <int D, uint32_t OUT, int NV>
__device__ __forceinline__ void merge_row(const void* ws_o, const PartialLse* ws_lse, void* out, uint32_t hq,
                                          uint32_t b, uint32_t qh, uint32_t s0, uint32_t n, int lane);

// Direct decode plans: after its waves wrote their partial states, the
// workgroup merges its rows (one (sequence, KV head, row block): the rows of
// its first item) over the sequence's slots and writes out.  The states are
// read back through the cache right after they were written: a workgroup
// fence and barrier order the writes of every wave before the reads.
template <int D, uint32_t OUT>
__device__ __forceinline__ void wave_task_merge(const AttendArgs& a, int wave, int lane) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
    __syncthreads();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
    const Item it = uniform_item(a.items[a.n_group_items + (blockIdx.x - a.n_group_items) * kWaves]);
    for (uint32_t row = uint32_t(wave); row < it.nrows; row += kWaves) {
        uint32_t seq, slot, qh;
        row_target(a, it, row, seq, slot, qh);
        seq = __builtin_amdgcn_readfirstlane(seq);
        qh = __builtin_amdgcn_readfirstlane(qh);
        const uint32_t s0 = __builtin_amdgcn_readfirstlane(a.slot_ptr[seq]);
        const uint32_t n = __builtin_amdgcn_readfirstlane(a.slot_ptr[seq + 1]) - s0;
        // at most kWaves states per row
        merge_row<D, OUT, MergeShape<D, OUT>::nv_for(kWaves)>(a.ws_o, a.ws_lse, a.out, a.hq, seq, qh, s0, n, lane);
    }
}

template <int D, uint32_t KVF, bool F16>
__global__ __launch_bounds__(256, D >= 256 ? 1 : 2) void attend16_kernel(AttendArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    // Wave index as a wave-uniform (scalar) value: page-list reads then go
    // through the scalar cache and never wait on the vector loads in flight.
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t ng = group_item_count<false>(a);
    if (blockIdx.x < ng) {
        const Item it = a.items[blockIdx.x];
        if constexpr ((KVF == KVF_FP8 || KVF == KVF_MX) && D == 64) group_item<D, KVF, F16>(a, it, tid, wave, g, c);
        else if constexpr (KVF == KVF_FP8 || KVF == KVF_MX) group_item_dma8<D, KVF, F16, false>(a, it, tid, wave, g, c);
        else group_item_dma<D, F16, false>(a, it, tid, wave, g, c);
    } else {
        const uint32_t idx = wave_item_index<false>(a, blockIdx.x, wave, ng);
        if (idx < wave_item_end<false>(a)) {
            const Item it = a.csr_hdr ? csr_wave_item(a, idx, ng) : a.items[idx];
            if (it.npages) wave_item<D, KVF, F16>(a, it, g, c);   // direct tasks pad with empty items
        }
        if (a.wave_direct) wave_task_merge<D, F16 ? 0u : 1u>(a, wave, tid & 63);
    }
}

// Prefill plans: causal group items only (every workgroup one item); the
// 16-bit and FP8 / MXFP8 direct-load paths at head_dim 128 and 256 and the
// 16-bit one at 64.  A kernel of its own, so the per-row token masks do not
// add to the decode kernel's registers.
template <int D, uint32_t KVF, bool F16>
__global__ __launch_bounds__(256, D >= 256 ? 1 : 2) void prefill16_kernel(AttendArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (blockIdx.x >= a.n_group_items) return;
    const Item it = a.items[blockIdx.x];
    if constexpr (KVF == KVF_FP8 || KVF == KVF_MX) group_item_dma8<D, KVF, F16, true>(a, it, tid, wave, g, c);
    else group_item_dma<D, F16, true>(a, it, tid, wave, g, c);
}

// ---------------------------------------------------------------- attend32
template <int D>
__global__ __launch_bounds__(256) void attend32_kernel(AttendArgs a) {
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t idx = wave_item_index<false>(a, blockIdx.x, wave, group_item_count<false>(a));   // f32: no group items
    if (idx < wave_item_end<false>(a)) {
        const Item it = a.csr_hdr ? csr_wave_item(a, idx, 0) : a.items[idx];
        if (it.npages) attend32_item<D>(a, it, lane, g, c);   // direct tasks pad with empty items
    }
    if (a.wave_direct) wave_task_merge<D, 2u>(a, wave, lane);
}

// ------------------------------------------------------------------ merge
// One wave per (sequence, query head): log-sum-exp over the sequence's
// partial states; no partial state -> zeros (backend.rs:218-222).
// Lane l reads the log-sum-exp of slots l, l+64, ...; the wave reduces their
// max and weights with cross-lane operations, then accumulates the slots'
// O rows sixteen at a time so sixteen loads are in flight per lane instead of
// one dependent load per slot.
__device__ __forceinline__ float wave_max(float x) {
    #pragma unroll
    for (int o = 32; o >= 1; o >>= 1) x = fmaxf(x, __shfl_xor(x, o, 64));
    return x;
}

__device__ __forceinline__ float wave_sum(float x) {
    #pragma unroll
    for (int o = 32; o >= 1; o >>= 1) x += __shfl_xor(x, o, 64);
    return x;
}

// PL consecutive partial-O elements starting at element e of the partial
// rows: fp32 when the output is f32 (OUT == 2), else scaled f16.
template <int OUT, int PL>
__device__ __forceinline__ void load_partial(const void* ws, uint64_t e, float (&v)[PL]) {
    if constexpr (OUT == 2) {
        const float* o = static_cast<const float*>(ws) + e;
        #pragma unroll
        for (int q = 0; q < PL; ++q) v[q] = o[q];
    } else if constexpr (PL == 1) {
        v[0] = float(static_cast<const _Float16*>(ws)[e]);
    } else {
        const uint32_t* o = reinterpret_cast<const uint32_t*>(static_cast<const uint16_t*>(ws) + e);
        uint32_t w[PL / 2];
        #pragma unroll
        for (int q = 0; q < PL / 2; ++q) w[q] = o[q];
        #pragma unroll
        for (int q = 0; q < PL / 2; ++q) {
            v[2 * q] = unpack_lo(w[q], true);
            v[2 * q + 1] = unpack_hi(w[q], true);
        }
    }
}

// merge_row for at most 64 states: a lane loads 16 bytes of one state row
// (LPS lanes cover a row, so one load instruction reads SPI = 64 / LPS
// states), all of a pass's loads are issued together with the
// log-sum-exps, and the SPI lane groups' weighted sums are added across
// lanes at the end.  One pass covers NV * SPI states (NV chosen for the
// plan's most states per row), so such a row costs one memory round trip
// after its slot range.
template <int D, uint32_t OUT, int NV>
__device__ __forceinline__ void merge_row_v(const void* ws_o, const PartialLse* ws_lse, void* out, uint32_t hq,
                                            uint32_t b, uint32_t qh, uint32_t s0, uint32_t n, int lane) {
    using MS = MergeShape<D, OUT>;
    constexpr int ES = MS::ES, EPL = MS::EPL, LPS = MS::LPS, SPI = MS::SPI;
    static_assert(NV >= 1 && NV <= MS::MAX_NV, "loads per pass");
    const int grp = lane / LPS, e = lane % LPS;
    float acc[EPL];
    #pragma unroll
    for (int i = 0; i < EPL; ++i) acc[i] = 0.f;
    float W = 0.f;
    if (n != 0) {
        const PartialLse pk = uint32_t(lane) < n ? ws_lse[uint64_t(s0 + lane) * hq + qh]
                                                 : PartialLse{kNegInf, 0.f};
        const uint8_t* base = static_cast<const uint8_t*>(ws_o) + (uint64_t(s0) * hq + qh) * (D * ES) + 16 * e;
        const uint64_t sstride = uint64_t(hq) * (D * ES);
        u32x4 v[NV];
        auto load = [&](uint32_t j0) {
            #pragma unroll
            for (int u = 0; u < NV; ++u) {
                const uint32_t st = min(j0 + uint32_t(u * SPI + grp), n - 1);
                v[u] = *reinterpret_cast<const u32x4*>(base + st * sstride);
            }
        };
        load(0);
        const float M = wave_max(pk.lse);
        if (M != kNegInf) {
            const float wk = pk.lse == kNegInf ? 0.f : fast_exp2(pk.lse - M);
            W = wk;
            const float wo = __builtin_amdgcn_ldexpf(wk, int(pk.k));   // weight of the stored (scaled) O
            for (uint32_t j0 = 0; j0 < n; j0 += NV * SPI) {
                if (j0) load(j0);
                #pragma unroll
                for (int u = 0; u < NV; ++u) {
                    const uint32_t st = j0 + uint32_t(u * SPI + grp);
                    const float w = __shfl(wo, int(st & 63u), 64);
                    const float wu = st < n ? w : 0.f;
                    if constexpr (OUT == 2) {
                        #pragma unroll
                        for (int i = 0; i < 4; ++i) acc[i] += wu * __uint_as_float(v[u][i]);
                    } else {
                        #pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            acc[2 * i] += wu * unpack_lo(v[u][i], true);
                            acc[2 * i + 1] += wu * unpack_hi(v[u][i], true);
                        }
                    }
                }
            }
        }
    }
    #pragma unroll
    for (int o = LPS; o < 64; o <<= 1)
        #pragma unroll
        for (int i = 0; i < EPL; ++i) acc[i] += __shfl_xor(acc[i], o, 64);
    W = wave_sum(W);
    const float inv = W > 0.f ? 1.f / W : 0.f;
    if (lane < LPS) {
        uint8_t* o = static_cast<uint8_t*>(out) + ((uint64_t(b) * hq + qh) * D + e * EPL) * (OUT == 2 ? 4 : 2);
        if constexpr (OUT == 2) {
            *reinterpret_cast<f4*>(o) = f4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
        } else {
            u32x4 w;
            #pragma unroll
            for (int i = 0; i < 4; ++i) w[i] = pack2(acc[2 * i] * inv, acc[2 * i + 1] * inv, OUT == 0);
            *reinterpret_cast<u32x4*>(o) = w;
        }
    }
}

// One wave merges output row (b, qh) over partial slots s0 .. s0 + n - 1
// (no slot: zeros).  NV > 0: rows of up to 64 states take merge_row_v.
// Otherwise (NV = 0, and rows of more than 64 states) a lane loads 4-8 bytes
// of every state row, U partial rows per pass (32 for NV = 0, else 16): a
// row of at most U states costs one round trip after its slot range.  On
// MI355X the vector form is faster for 36 states at head_dim 64 (C2, one
// pass instead of two: 10.5 -> 9.6 us a step), the same for 2-9 (C1, C4,
// C5), and slower for 19 at head_dim 128 (C3: 28.0 against 27.6), which
// keeps the scalar form.
template <int D, uint32_t OUT, int NV>
__device__ __forceinline__ void merge_row(const void* ws_o, const PartialLse* ws_lse, void* out, uint32_t hq,
                                          uint32_t b, uint32_t qh, uint32_t s0, uint32_t n, int lane) {
    if constexpr (NV > 0) {
        if (n <= 64) {
            merge_row_v<D, OUT, NV>(ws_o, ws_lse, out, hq, b, qh, s0, n, lane);
            return;
        }
    }
    if constexpr (NV < 0) {   // loads per pass from the row's own state count (wave-uniform)
        using MS = MergeShape<D, OUT>;
        constexpr int S = MS::SPI, MX = MS::MAX_NV;
        if (n <= uint32_t(S)) {
            merge_row_v<D, OUT, 1>(ws_o, ws_lse, out, hq, b, qh, s0, n, lane);
            return;
        }
        if (n <= uint32_t(4 * S)) {
            merge_row_v<D, OUT, (MX < 4 ? MX : 4)>(ws_o, ws_lse, out, hq, b, qh, s0, n, lane);
            return;
        }
        if (n <= 64) {
            merge_row_v<D, OUT, MX>(ws_o, ws_lse, out, hq, b, qh, s0, n, lane);
            return;
        }
    }
    constexpr int U = NV == 0 ? 32 : 16;
    constexpr int PL = D / 64;
    float acc[PL];
    #pragma unroll
    for (int k = 0; k < PL; ++k) acc[k] = 0.f;
    float W = 0.f;
    if (n != 0 && n <= 64) {
        // One pass: the log-sum-exps and the first U partial rows are loaded
        // together (neither depends on the other), so a row with up to U
        // partial states costs one memory round trip after slot_ptr.
        const PartialLse pk = uint32_t(lane) < n ? ws_lse[uint64_t(s0 + lane) * hq + qh]
                                                 : PartialLse{kNegInf, 0.f};
        float v[U][PL];
        #pragma unroll
        for (int u = 0; u < U; ++u)
            load_partial<OUT, PL>(ws_o, (uint64_t(s0 + min(uint32_t(u), n - 1)) * hq + qh) * D + lane * PL, v[u]);
        const float M = wave_max(pk.lse);
        if (M != kNegInf) {
            const float wk = pk.lse == kNegInf ? 0.f : fast_exp2(pk.lse - M);
            W = wk;
            const float wo = __builtin_amdgcn_ldexpf(wk, int(pk.k));   // weight of the stored (scaled) O
            for (uint32_t j0 = 0; j0 < n; j0 += U) {
                if (j0) {
                    #pragma unroll
                    for (int u = 0; u < U; ++u)
                        load_partial<OUT, PL>(ws_o, (uint64_t(s0 + min(j0 + u, n - 1)) * hq + qh) * D + lane * PL,
                                              v[u]);
                }
                #pragma unroll
                for (int u = 0; u < U; ++u) {
                    const float w = (j0 + u < n) ? __shfl(wo, int(j0 + u), 64) : 0.f;
                    #pragma unroll
                    for (int q = 0; q < PL; ++q) acc[q] += w * v[u][q];
                }
            }
        }
    } else if (n > 64) {
        float M = kNegInf;
        for (uint32_t k = lane; k < n; k += 64) M = fmaxf(M, ws_lse[uint64_t(s0 + k) * hq + qh].lse);
        M = wave_max(M);
        if (M != kNegInf) {
            for (uint32_t base = 0; base < n; base += 64) {
                // Weight of slot base + lane, then the slots' O rows in groups of U.
                const uint32_t k = base + lane;
                const PartialLse pk = k < n ? ws_lse[uint64_t(s0 + k) * hq + qh] : PartialLse{kNegInf, 0.f};
                const float wk = pk.lse == kNegInf ? 0.f : fast_exp2(pk.lse - M);
                W += wk;
                const float wo = __builtin_amdgcn_ldexpf(wk, int(pk.k));   // weight of the stored (scaled) O
                const uint32_t cnt = min(64u, n - base);
                for (uint32_t j0 = 0; j0 < cnt; j0 += U) {
                    float v[U][PL];
                    #pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const uint32_t j = min(j0 + u, cnt - 1);
                        load_partial<OUT, PL>(ws_o, (uint64_t(s0 + base + j) * hq + qh) * D + lane * PL, v[u]);
                    }
                    #pragma unroll
                    for (int u = 0; u < U; ++u) {
                        const float w = (j0 + u < cnt) ? __shfl(wo, int(j0 + u), 64) : 0.f;
                        #pragma unroll
                        for (int q = 0; q < PL; ++q) acc[q] += w * v[u][q];
                    }
                }
            }
        }
    }
    W = wave_sum(W);
    const float inv = W > 0.f ? 1.f / W : 0.f;
    const uint64_t ob = (uint64_t(b) * hq + qh) * D + lane * PL;
    #pragma unroll
    for (int k = 0; k < PL; ++k) {
        const float v = acc[k] * inv;
        if constexpr (OUT == 2) reinterpret_cast<float*>(out)[ob + k] = v;
        else if constexpr (OUT == 1) reinterpret_cast<__bf16*>(out)[ob + k] = (__bf16)v;
        else reinterpret_cast<_Float16*>(out)[ob + k] = (_Float16)v;
    }
}

template <int D, uint32_t OUT, int NV>
__global__ __launch_bounds__(256) void merge_kernel(MergeArgs a) {
    const int lane = threadIdx.x & 63;
    const uint32_t row = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (a.status && blockIdx.x == 0 && threadIdx.x < 64) {   // the CSR call's status
        uint32_t bad = 0;
        for (uint32_t b = lane; b < a.batch; b += 64) bad |= a.seq_bad[b];
        const bool any = __ballot(bad != 0) != 0;
        if (lane == 0) *a.status = a.csr_hdr->overflow ? 2 : (any ? 1 : 0);   // DH_ENOMEM / DH_EINVAL / DH_OK
    }
    if (row >= a.batch * a.hq) return;
    const uint32_t b = row / a.hq, qh = row - b * a.hq;
    // Plans whose sequences all have n slots: the slot range is b*n .. +n,
    // one dependent load fewer before the partial states.
    const uint32_t s0 = a.uniform_slots ? b * a.uniform_slots : a.slot_ptr[b];
    const uint32_t n = a.uniform_slots ? a.uniform_slots
                                       : ((a.seq_bad && a.seq_bad[b]) ? 0u : a.slot_ptr[b + 1] - s0);
    merge_row<D, OUT, NV>(a.ws_o, a.ws_lse, a.out, a.hq, b, qh, s0, n, lane);
}

// Rows of a prefill plan's split blocks: one wave per (row, query head).
// Launch-bound (a few hundred rows of 2-12 states); the states are read one
// after another, their loads independent of the running sums, so several
// are in flight.  f32 states, so a split row holds no less than a whole one
// (error against 64 bits 0.0034 either way on the case at prefill_tail).
template <int D, bool F16>
__global__ __launch_bounds__(256) void prefill_merge_kernel(MergeArgs a, const uint32_t* rows, uint32_t n) {
    constexpr int PL = D / 64;
    const int lane = threadIdx.x & 63;
    const uint32_t w = blockIdx.x * kWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (w >= n * a.hq) return;
    const uint32_t i = w / a.hq, qh = w - i * a.hq;
    const uint32_t v = __builtin_amdgcn_readfirstlane(rows[i]);
    const uint32_t s0 = __builtin_amdgcn_readfirstlane(a.slot_ptr[v]);
    const uint32_t s1 = __builtin_amdgcn_readfirstlane(a.slot_ptr[v + 1]);
    float M = kNegInf;
    for (uint32_t s = s0; s < s1; ++s) M = fmaxf(M, a.ws_lse[uint64_t(s) * a.hq + qh].lse);
    float acc[PL], W = 0.f;
    #pragma unroll
    for (int k = 0; k < PL; ++k) acc[k] = 0.f;
    if (M != kNegInf) {
        #pragma unroll 4
        for (uint32_t s = s0; s < s1; ++s) {
            const uint64_t row = uint64_t(s) * a.hq + qh;
            const float l = a.ws_lse[row].lse;
            const float wk = l == kNegInf ? 0.f : fast_exp2(l - M);
            const float* o = static_cast<const float*>(a.ws_o) + row * D + lane * PL;
            W += wk;
            #pragma unroll
            for (int k = 0; k < PL; ++k) acc[k] += wk * o[k];
        }
    }
    const float inv = W > 0.f ? 1.f / W : 0.f;
    const uint64_t ob = (uint64_t(v) * a.hq + qh) * D + lane * PL;
    #pragma unroll
    for (int k = 0; k < PL; ++k) {
        if constexpr (F16) static_cast<_Float16*>(a.out)[ob + k] = (_Float16)(acc[k] * inv);
        else static_cast<__bf16*>(a.out)[ob + k] = (__bf16)(acc[k] * inv);
    }
}

// Element-wise two-state merge with natural-log LSE (cascade.rs:116-124).
__global__ __launch_bounds__(256) void merge_states_kernel(const float* o_a, const float* lse_a,
                                                           const float* o_b, const float* lse_b,
                                                           float* o_out, float* lse_out,
                                                           uint32_t n_rows, uint32_t d) {
    const uint64_t idx = uint64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    const bool valid = idx < uint64_t(n_rows) * d;
    const uint32_t row = valid ? uint32_t(idx / d) : 0u;
    const uint32_t col = valid ? uint32_t(idx - uint64_t(row) * d) : 1u;
    float res = 0.f, lse = kNegInf;
    if (valid) {
        const float la = lse_a[row], lb = lse_b[row];
        const float mx = fmaxf(la, lb);
        if (mx != kNegInf) {
            const float ea = expf(la - mx), eb = expf(lb - mx);
            const float sum = ea + eb;
            res = (o_a[idx] * ea + o_b[idx] * eb) / sum;
            lse = mx + logf(sum);
        }
    }
    __syncthreads();  // every read of this block's rows precedes the writes (outputs may alias inputs)
    if (valid) {
        o_out[idx] = res;
        if (col == 0) lse_out[row] = lse;
    }
}

// Copies the K and V planes of one KV head for a list of pages.
__global__ __launch_bounds__(256) void gather_kernel(const uint8_t* kv, const uint32_t* pages,
                                                     uint32_t n_pages, uint32_t kv_head, uint32_t hkv,
                                                     uint32_t head_dim, uint32_t eb, uint8_t* out) {
    const uint32_t plane = blockIdx.y;                 // 0 = K, 1 = V
    const uint32_t pi = blockIdx.x;
    const uint64_t bytes = uint64_t(kPageSize) * head_dim * eb;
    const uint8_t* src = kv + plane_offset(pages[pi], plane, kv_head, hkv, head_dim, eb);
    uint8_t* dst = out + (uint64_t(plane) * n_pages + pi) * bytes;
    for (uint64_t i = threadIdx.x * 4; i < bytes; i += blockDim.x * 4)
        *reinterpret_cast<uint32_t*>(dst + i) = *reinterpret_cast<const uint32_t*>(src + i);
}

// The decode kernels' E4M3 -> bf16 conversion, exposed for an exhaustive
// test: codes[4i..4i+3] are scaled by the E8M0 byte e8m0[i].
__global__ __launch_bounds__(256) void e4m3_debug_kernel(const uint32_t* codes, const uint8_t* e8m0,
                                                         uint32_t n4, uint32_t* out) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n4) return;
    uint32_t lo, hi;
    e4m3x4_to_bf16(codes[i], e8m0_to_float(e8m0[i]), lo, hi);
    out[2 * i] = lo;
    out[2 * i + 1] = hi;
}

// Scatters n records of rec bytes from a packed staging buffer to dst[ids[i]].
__global__ __launch_bounds__(256) void scatter_kernel(uint8_t* dst, const uint8_t* src,
                                                      const uint32_t* ids, uint64_t rec) {
    const uint8_t* s = src + uint64_t(blockIdx.x) * rec;
    uint8_t* d = dst + uint64_t(ids[blockIdx.x]) * rec;
    if ((rec & 15) == 0) {
        for (uint64_t o = uint64_t(threadIdx.x) * 16; o < rec; o += uint64_t(blockDim.x) * 16)
            *reinterpret_cast<u32x4*>(d + o) = *reinterpret_cast<const u32x4*>(s + o);
    } else {
        for (uint64_t o = uint64_t(threadIdx.x) * 4; o < rec; o += uint64_t(blockDim.x) * 4)
            *reinterpret_cast<uint32_t*>(d + o) = *reinterpret_cast<const uint32_t*>(s + o);
    }
}

template <int D>
hipError_t launch_prefill_d(const AttendArgs& a, uint32_t n, uint32_t q_dtype, uint32_t kvf, hipStream_t s) {
    dim3 grid(n), block(kWaves * 64);
    if (q_dtype == 1 && kvf == KVF_BF16) {
        hipLaunchKernelGGL((prefill16_kernel<D, KVF_BF16, false>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_F16) {
        hipLaunchKernelGGL((prefill16_kernel<D, KVF_F16, true>), grid, block, 0, s, a);
    } else if constexpr (D >= 128) {
        if (q_dtype == 1 && kvf == KVF_FP8) hipLaunchKernelGGL((prefill16_kernel<D, KVF_FP8, false>), grid, block, 0, s, a);
        else if (q_dtype == 1 && kvf == KVF_MX) hipLaunchKernelGGL((prefill16_kernel<D, KVF_MX, false>), grid, block, 0, s, a);
        else if (q_dtype == 0 && kvf == KVF_FP8) hipLaunchKernelGGL((prefill16_kernel<D, KVF_FP8, true>), grid, block, 0, s, a);
        else if (q_dtype == 0 && kvf == KVF_MX) hipLaunchKernelGGL((prefill16_kernel<D, KVF_MX, true>), grid, block, 0, s, a);
        else return hipErrorInvalidValue;
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int D>
hipError_t launch_attend_d(const AttendArgs& a, uint32_t n, uint32_t q_dtype, uint32_t kvf,
                           hipStream_t s) {
    dim3 grid(n), block(kWaves * 64);
    if (q_dtype == 2 && kvf == KVF_F32) {
        hipLaunchKernelGGL(attend32_kernel<D>, grid, block, 0, s, a);
    } else if (q_dtype == 1 && kvf == KVF_BF16) {
        hipLaunchKernelGGL((attend16_kernel<D, KVF_BF16, false>), grid, block, 0, s, a);
    } else if (q_dtype == 1 && kvf == KVF_FP8) {
        hipLaunchKernelGGL((attend16_kernel<D, KVF_FP8, false>), grid, block, 0, s, a);
    } else if (q_dtype == 1 && kvf == KVF_MX) {
        hipLaunchKernelGGL((attend16_kernel<D, KVF_MX, false>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_FP8) {   // f16 queries: codes into f16, f16 MFMAs
        hipLaunchKernelGGL((attend16_kernel<D, KVF_FP8, true>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_MX) {
        hipLaunchKernelGGL((attend16_kernel<D, KVF_MX, true>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_F16) {
        hipLaunchKernelGGL((attend16_kernel<D, KVF_F16, true>), grid, block, 0, s, a);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

template <int D>
hipError_t launch_merge_d(const MergeArgs& a, uint32_t q_dtype, hipStream_t s) {
    const uint32_t rows = a.batch * a.hq;
    if (rows == 0) return hipSuccess;
    dim3 grid((rows + 3) / 4), block(256);
    // Rows of 17-32 states: the scalar form, one pass of 32, below head_dim
    // 256.  There its 32 rows of 8 bytes a lane take 286 registers, one wave
    // a SIMD, and the vector form's one pass is faster (8 trees of 8 leaves,
    // 17-32 states, 16 / 2 heads, bf16: a step 32.4 -> 30.9 us; f32 states
    // keep the scalar form's 193 registers).  Otherwise the vector form with
    // loads per pass for the plan's most states per row, so a row loads no
    // state twice; not known on the host (0, the CSR path): chosen per row
    // from its own count.
    const int states = a.max_states > 64 ? 64 : int(a.max_states);
    auto go = [&](auto out_tag) {
        constexpr uint32_t OUT = decltype(out_tag)::value;
        using MS = MergeShape<D, OUT>;
        const int need = (states + MS::SPI - 1) / MS::SPI;
        if constexpr (D < 256 || OUT == 2) {
            if (states > 16 && states <= 32) {
                hipLaunchKernelGGL((merge_kernel<D, OUT, 0>), grid, block, 0, s, a);
                return;
            }
        }
        if (states == 0) hipLaunchKernelGGL((merge_kernel<D, OUT, -1>), grid, block, 0, s, a);
        else if (need <= 1) hipLaunchKernelGGL((merge_kernel<D, OUT, 1>), grid, block, 0, s, a);
        else if (need <= 2 && MS::MAX_NV >= 2) hipLaunchKernelGGL((merge_kernel<D, OUT, (MS::MAX_NV >= 2 ? 2 : 1)>), grid, block, 0, s, a);
        else if (need <= 4 && MS::MAX_NV >= 4) hipLaunchKernelGGL((merge_kernel<D, OUT, (MS::MAX_NV >= 4 ? 4 : 1)>), grid, block, 0, s, a);
        else if (need <= 8 && MS::MAX_NV >= 8) hipLaunchKernelGGL((merge_kernel<D, OUT, (MS::MAX_NV >= 8 ? 8 : 1)>), grid, block, 0, s, a);
        else hipLaunchKernelGGL((merge_kernel<D, OUT, MS::MAX_NV>), grid, block, 0, s, a);
    };
    if (q_dtype == 2) go(std::integral_constant<uint32_t, 2>{});
    else if (q_dtype == 1) go(std::integral_constant<uint32_t, 1>{});
    else go(std::integral_constant<uint32_t, 0>{});
    return hipGetLastError();
}

// Partial-state memory of dh_decode_batch_static: DH_STATIC_WORKSPACE_BYTES
// per GPU, held from the library's load to the end of the process.  Host
// code never uses this name as an address (on the host it is a stand-in,
// not device memory); it asks for the array's device address once per GPU
// (static_scratch_address, from dh_create) and passes that pointer.
static __device__ __align__(256) uint8_t scratch[DH_STATIC_WORKSPACE_BYTES];

}  // namespace

int static_scratch_address(void** out) { return int(hipGetSymbolAddress(out, HIP_SYMBOL(scratch))); }

bool attend_supported(uint32_t q_dtype, uint32_t kvf, uint32_t d) {
    if (d != 64 && d != 128 && d != 256) return false;
    return (q_dtype == 2 && kvf == KVF_F32) || (q_dtype == 1 && kvf == KVF_BF16) ||
           (q_dtype <= 1 && kvf == KVF_FP8) || (q_dtype <= 1 && kvf == KVF_MX) ||
           (q_dtype == 0 && kvf == KVF_F16);
}

int launch_attend(const AttendArgs& a, uint32_t n_items, uint32_t q_dtype, uint32_t kvf,
                  uint32_t d, bool prefill, void* stream) {
    if (n_items == 0) return hipSuccess;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    if (prefill) {
        switch (d) {
            case 64: return launch_prefill_d<64>(a, n_items, q_dtype, kvf, s);
            case 128: return launch_prefill_d<128>(a, n_items, q_dtype, kvf, s);
            case 256: return launch_prefill_d<256>(a, n_items, q_dtype, kvf, s);
            default: return hipErrorInvalidValue;
        }
    }
    switch (d) {
        case 64: return launch_attend_d<64>(a, n_items, q_dtype, kvf, s);
        case 128: return launch_attend_d<128>(a, n_items, q_dtype, kvf, s);
        case 256: return launch_attend_d<256>(a, n_items, q_dtype, kvf, s);
        default: return hipErrorInvalidValue;
    }
}

int launch_merge(const MergeArgs& a, uint32_t q_dtype, uint32_t d, void* stream) {
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (d) {
        case 64: return launch_merge_d<64>(a, q_dtype, s);
        case 128: return launch_merge_d<128>(a, q_dtype, s);
        case 256: return launch_merge_d<256>(a, q_dtype, s);
        default: return hipErrorInvalidValue;
    }
}

int launch_prefill_merge(const MergeArgs& a, const uint32_t* rows, uint32_t n_rows, uint32_t q_dtype, uint32_t d,
                         void* stream) {
    if (n_rows == 0) return hipSuccess;
    if (q_dtype > 1) return hipErrorInvalidValue;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    const dim3 grid(uint32_t((uint64_t(n_rows) * a.hq + kWaves - 1) / kWaves)), block(kWaves * 64);
    auto go = [&](auto f16) {
        constexpr bool F = decltype(f16)::value;
        switch (d) {
            case 64: hipLaunchKernelGGL((prefill_merge_kernel<64, F>), grid, block, 0, s, a, rows, n_rows); break;
            case 128: hipLaunchKernelGGL((prefill_merge_kernel<128, F>), grid, block, 0, s, a, rows, n_rows); break;
            case 256: hipLaunchKernelGGL((prefill_merge_kernel<256, F>), grid, block, 0, s, a, rows, n_rows); break;
            default: return hipErrorInvalidValue;
        }
        return hipGetLastError();
    };
    return q_dtype == 0 ? go(std::true_type{}) : go(std::false_type{});
}

int launch_merge_states(const float* o_a, const float* lse_a, const float* o_b, const float* lse_b,
                        float* o_out, float* lse_out, uint32_t n_rows, uint32_t d, void* stream) {
    const uint64_t n = uint64_t(n_rows) * d;
    if (n == 0) return hipSuccess;
    // One block covers whole rows only, so the in-block barrier orders every
    // read of a row before its writes.
    const uint32_t rows_per_block = d >= 256 ? 1u : 256u / d;
    dim3 block(rows_per_block * d);
    dim3 grid((n_rows + rows_per_block - 1) / rows_per_block);
    hipLaunchKernelGGL(merge_states_kernel, grid, block, 0, reinterpret_cast<hipStream_t>(stream),
                       o_a, lse_a, o_b, lse_b, o_out, lse_out, n_rows, d);
    return hipGetLastError();
}

int launch_e4m3_debug(const uint32_t* codes, const uint8_t* e8m0, uint32_t n4, uint32_t* out,
                      void* stream) {
    if (n4 == 0) return hipSuccess;
    hipLaunchKernelGGL(e4m3_debug_kernel, dim3((n4 + 255) / 256), dim3(256), 0,
                       reinterpret_cast<hipStream_t>(stream), codes, e8m0, n4, out);
    return hipGetLastError();
}

int launch_scatter(uint8_t* dst, const uint8_t* src, const uint32_t* ids, uint32_t n,
                   uint64_t rec_bytes, void* stream) {
    if (n == 0) return hipSuccess;
    if (rec_bytes & 3) return hipErrorInvalidValue;
    hipLaunchKernelGGL(scatter_kernel, dim3(n), dim3(256), 0, reinterpret_cast<hipStream_t>(stream),
                       dst, src, ids, rec_bytes);
    return hipGetLastError();
}

int launch_gather(const uint8_t* kv, const uint32_t* pages, uint32_t n_pages, uint32_t kv_head,
                  uint32_t hkv, uint32_t d, uint32_t eb, uint8_t* out, void* stream) {
    if (n_pages == 0) return hipSuccess;
    dim3 grid(n_pages, 2), block(256);
    hipLaunchKernelGGL(gather_kernel, grid, block, 0, reinterpret_cast<hipStream_t>(stream), kv,
                       pages, n_pages, kv_head, hkv, d, eb, out);
    return hipGetLastError();
}

}  // namespace dh
