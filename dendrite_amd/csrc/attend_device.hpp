// Attention items of the gfx950 (CDNA4) kernels: what one wave or workgroup
// does with an item, shared by the plan path's kernels (decode_kernels.hip)
// and the device-table ones (csr_kernels.hip).
//
// attend16 / attend32: a workgroup of four wave64s runs one task, either
//   - up to four wave items: each wave alone attends its item (<= 16 query
//     rows, i.e. one sequence's GQA group of a private tail, or a few
//     sequences of a small shared segment) over the item's pages, with the
//     next page pair's loads in flight behind the current pair's math; or
//   - one group item (<= 128 rows, a tree-shared prefix; 64 at head_dim 256
//     and with FP8 KV): every wave owns up to 32 rows and all four consume
//     the same page pairs, which the workgroup stages once into LDS (16-bit
//     KV: direct global->LDS loads into a ring of page pairs; FP8 / MXFP8:
//     through registers, double-buffered), so a shared page is fetched once
//     per 128 rows instead of once per wave.
// Each wave keeps an online softmax for its rows and writes one partial
// state per row.  ReferenceBackend::decode (crates/dendrite-core/src/
// attention/backend.rs:206-265) computes softmax(q K^T * scale) V over the
// concatenated pages; this is the same quantity, split over pages and merged
// exactly by log-sum-exp.
//
// Matrix-core mapping (lane l = 16*g + c, g = l / 16, c = l % 16):
//   S^T = K . Q^T with v_mfma_f32_16x16x32_{bf16,f16}: A = 16 tokens x 32 dims
//   of one page (lane holds token c, 8 consecutive dims), B = 32 dims x 16 query
//   rows (lane holds row c, the same 8 dims).  The accumulator gives lane
//   (g, c) the scores of row c for tokens 4g..4g+3.
//   O^T += V^T . P^T with the same instruction over two pages (32 tokens): the
//   B operand (P^T) is exactly the two pages' score accumulators of the lane
//   after exp2, so the probabilities never leave registers.  The A operand
//   (V^T) holds, for d-block e, V[token][c*EPL + e] for the lane's 8 tokens,
//   built by byte permutes from 16-byte row loads (EPL = head_dim / 16).
//   Lane (g, c) ends up holding O[row c][4g*EPL .. 4g*EPL + 4*EPL).
//   (The LDS path of group items builds V^T with transposing LDS reads
//   instead, and its lanes hold O[row c][16e + 4g + i]; see there.)
// FP8 E4M3 pages are converted to bf16 in registers (exact: E4M3 is a subset
// of bf16); the per-(page, head) fp32 scale multiplies the scores (K) and the
// probabilities (V), which equals dequantising every element.  MXFP8 pages
// are converted with their E8M0 group scale by v_cvt_scalef32_pk_bf16_fp8
// (exact: power-of-two scaling).
#pragma once
#include <hip/hip_runtime.h>
#include <math.h>
#include <type_traits>
#include "dh_device.hpp"
#include "dendrite_hip.h"

namespace dh {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f2 __attribute__((ext_vector_type(2)));

constexpr uint32_t KVF_F16 = 0, KVF_BF16 = 1, KVF_F32 = 2, KVF_FP8 = 3, KVF_MX = 4;
constexpr float kNegInf = -__builtin_inff();

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// Max over the four lanes l, l^16, l^32, l^48 (the four 16-lane rows of the
// wave) with the gfx950 permlane swaps: after swap(x, x) the two results hold
// x of the lane and of its partner row, so the max of the pair is the
// xor-16 / xor-32 reduction without a trip through the LDS crossbar.
__device__ __forceinline__ float rowgroup_max(float x) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

__device__ __forceinline__ float rowgroup_sum(float x) {
    auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Load n dwords (n in {1, 2, 4, 8}) from a naturally aligned address.
template <int N>
__device__ __forceinline__ void load_dwords(uint32_t* dst, const void* src) {
    if constexpr (N == 1) {
        dst[0] = *reinterpret_cast<const uint32_t*>(src);
    } else if constexpr (N == 2) {
        u32x2 v = *reinterpret_cast<const u32x2*>(src);
        dst[0] = v.x; dst[1] = v.y;
    } else {
        #pragma unroll
        for (int i = 0; i < N / 4; ++i) {
            u32x4 v = reinterpret_cast<const u32x4*>(src)[i];
            dst[4 * i + 0] = v.x; dst[4 * i + 1] = v.y;
            dst[4 * i + 2] = v.z; dst[4 * i + 3] = v.w;
        }
    }
}

// E8M0 scale byte -> float 2^(e-127); 255 -> NaN (OCP MX v1.0).
__device__ __forceinline__ float e8m0_to_float(uint32_t e) {
    uint32_t bits = e == 0 ? 0x00400000u : (e == 255 ? 0x7FC00000u : (e << 23));
    return __uint_as_float(bits);
}

// Four E4M3 bytes -> four bf16 (two dwords), multiplied by sc (a power of two).
__device__ __forceinline__ void e4m3x4_to_bf16(uint32_t x, float sc, uint32_t& lo, uint32_t& hi) {
    bf16x2 a = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, sc, false);
    bf16x2 b = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(x, sc, true);
    lo = __builtin_bit_cast(uint32_t, a);
    hi = __builtin_bit_cast(uint32_t, b);
}

// The same into f16 (H) or bf16: 8-bit pools under f16 queries compute in
// f16 (every E4M3 code is exact in f16; code x scale rounds once).
template <bool H>
__device__ __forceinline__ void e4m3x4_cvt(uint32_t x, float sc, uint32_t& lo, uint32_t& hi) {
    if constexpr (H) {
        f16x2 a = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(x, sc, false);
        f16x2 b = __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(x, sc, true);
        lo = __builtin_bit_cast(uint32_t, a);
        hi = __builtin_bit_cast(uint32_t, b);
    } else {
        e4m3x4_to_bf16(x, sc, lo, hi);
    }
}

__device__ __forceinline__ uint32_t pack2(float a, float b, bool f16) {
    if (f16) {
        f16x2 t = {(_Float16)a, (_Float16)b};
        return __builtin_bit_cast(uint32_t, t);
    }
    bf16x2 t = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, t);
}

__device__ __forceinline__ float unpack_lo(uint32_t v, bool f16) {
    if (f16) return float(__builtin_bit_cast(f16x2, v)[0]);
    return __uint_as_float(v << 16);
}

__device__ __forceinline__ float unpack_hi(uint32_t v, bool f16) {
    if (f16) return float(__builtin_bit_cast(f16x2, v)[1]);
    return __uint_as_float(v & 0xFFFF0000u);
}

template <bool F16>
__device__ __forceinline__ f4 mma16(const uint32_t* a, const uint32_t* b, f4 c) {
    u32x4 av = {a[0], a[1], a[2], a[3]};
    u32x4 bv = {b[0], b[1], b[2], b[3]};
    if constexpr (F16) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, av),
                                                      __builtin_bit_cast(f16x8, bv), c, 0, 0, 0);
    } else {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av),
                                                       __builtin_bit_cast(bf16x8, bv), c, 0, 0, 0);
    }
}

// acc *= alpha in place.  The rescale runs on a rarely taken branch; done
// through "+v" operands the accumulator keeps its registers on both paths,
// so the compiler needs no copies of the accumulators to merge the paths.
__device__ __forceinline__ void scale_inplace(f4& acc, float alpha) {
    float x = acc[0], y = acc[1], z = acc[2], w = acc[3];
    asm volatile("v_mul_f32 %0, %0, %4\n\tv_mul_f32 %1, %1, %4\n\tv_mul_f32 %2, %2, %4\n\tv_mul_f32 %3, %3, %4"
                 : "+v"(x), "+v"(y), "+v"(z), "+v"(w)
                 : "v"(alpha));
    acc = f4{x, y, z, w};
}

// Query head served by row rho of an item (GQA mapping per dh_gqa_mapping).
__device__ __forceinline__ void row_target(const AttendArgs& a, const Item& it, uint32_t row,
                                           uint32_t& seq, uint32_t& slot, uint32_t& qh) {
    uint32_t rho = it.row_begin + row;
    uint32_t sl = rho / a.r;
    uint32_t j = rho - sl * a.r;
    SeqSlot ss = a.seqslots[it.seq_off + sl];
    seq = ss.seq;
    slot = ss.slot;
    qh = a.gqa_tiled ? it.kv_head + j * a.hkv : it.kv_head * a.r + j;
}

// Group items of the launch: the plan's count, or on the CSR path what the
// CSR planning kernel of this call wrote (its group items come first).
// Without CSR (the plan path's kernels) csr_hdr is null.  The tests of it in
// this and the next two functions, and the item choice by it in the plan
// path's kernels, stay for the machine code they give those: a 64-leaf bf16
// tree took 24.3-24.4 us a step with them and 24.4-24.6 without, in six
// builds.
template <bool CSR>
__device__ __forceinline__ uint32_t group_item_count(const AttendArgs& a) {
    return CSR || a.csr_hdr ? __builtin_amdgcn_readfirstlane(a.csr_hdr[4]) : a.n_group_items;
}

// Item of wave `wave` in unit `unit` (a workgroup's) past the ng group items:
// on the plan path an index into the items (group items first), on the CSR
// path the wave item's own number (csr_item).
template <bool CSR>
__device__ __forceinline__ uint32_t wave_item_index(const AttendArgs& a, uint32_t unit, int wave, uint32_t ng) {
    return (CSR || a.csr_hdr ? 0u : ng) + (unit - ng) * kWaves + uint32_t(wave);
}

// Wave items on the plan path: the plan's count; on the CSR path: what the
// CSR planning kernel of this call wrote (its nodes' wave items, then one
// per chunk of each sequence's own pages).
template <bool CSR>
__device__ __forceinline__ uint32_t wave_item_end(const AttendArgs& a) {
    return CSR || a.csr_hdr ? __builtin_amdgcn_readfirstlane(a.csr_hdr[1]) + __builtin_amdgcn_readfirstlane(a.csr_hdr[6])
                     : a.n_group_items + a.n_wave_items;
}

// Wave item idx of a CSR call: the cascade's node wave items (stored after
// its ng group items in a.items), then the items derived from the tables.
__device__ __forceinline__ Item csr_wave_item(const AttendArgs& a, uint32_t idx, uint32_t ng);

// Wave item idx of a CSR call, derived from the tables: idx = (j * hkv +
// kv_head) * nrb + row block; seqslots[j] names the j-th chunk in dispatch
// order, chunk k of sequence b in slot slot_ptr[b] + G + k, pages
// indptr[b] + L + k * chunk .. (the last chunk ends at b's last page), where
// b's first L pages are read by group items into its first G slots (csr_skip;
// L = G = 0 without a cascade).  seq_off = j: the row's slot is read back from
// seqslots[j] (row_target).
__device__ __forceinline__ Item csr_item(const AttendArgs& a, uint32_t idx) {
    const uint32_t nrb = a.csr_nrb, per = a.hkv * nrb;
    const uint32_t j = idx / per, rem = idx - j * per;
    const uint32_t h = rem / nrb, rb = rem - h * nrb;
    const uint32_t b = __builtin_amdgcn_readfirstlane(a.seqslots[j].seq);
    const uint32_t slot = __builtin_amdgcn_readfirstlane(a.seqslots[j].slot);
    const uint32_t chunk = __builtin_amdgcn_readfirstlane(a.csr_hdr[0]);
    const uint32_t skip = a.csr_skip ? __builtin_amdgcn_readfirstlane(a.csr_skip[b]) : 0u;
    const uint32_t k = slot - __builtin_amdgcn_readfirstlane(a.csr_slot_ptr[b]) - (skip >> 16);
    const uint32_t p0 = uint32_t(__builtin_amdgcn_readfirstlane(a.csr_indptr[b])) + (skip & 0xFFFFu);
    const uint32_t n = uint32_t(__builtin_amdgcn_readfirstlane(a.csr_indptr[b + 1])) - p0;
    Item it;
    it.page_off = p0 + k * chunk;
    it.npages = min(chunk, n - k * chunk);
    it.seq_off = j;
    it.row_begin = rb * kWaveRows;
    it.nrows = min(uint32_t(kWaveRows), a.r - rb * kWaveRows);
    it.kv_head = h;
    it.flags = (k + 1) * chunk >= n ? kItemTail : 0u;
    it.tail_seq = b;
    return it;
}

__device__ __forceinline__ Item csr_wave_item(const AttendArgs& a, uint32_t idx, uint32_t ng) {
    const uint32_t nw = __builtin_amdgcn_readfirstlane(a.csr_hdr[6]);
    return idx < nw ? a.items[ng + idx] : csr_item(a, idx - nw);
}

// Valid tokens of page index i of an item.
__device__ __forceinline__ int page_tokens(const Item& it, uint32_t i, int last_len) {
    if (i >= it.npages) return 0;
    return ((it.flags & kItemTail) && i + 1 == it.npages) ? last_len : kPageSize;
}

// Tokens in the item's last page.  Read through readfirstlane: the value is
// wave-uniform, and telling the compiler so keeps every branch on the page
// fill (full pair / partial pair) a scalar branch instead of a masked
// execution of both sides.
__device__ __forceinline__ int item_last_len(const AttendArgs& a, const Item& it) {
    if (!(it.flags & kItemTail)) return kPageSize;
    int L;
    if (a.last_page_len)
        L = __builtin_amdgcn_readfirstlane(a.last_page_len[it.tail_seq]);
    else if (a.lpl_inline)   // 4 bits a sequence in the kernel arguments, 0 for 16
        L = int((__builtin_amdgcn_readfirstlane(a.lpl_nib[it.tail_seq >> 3]) >> (4 * (it.tail_seq & 7))) & 15u);
    else
        return kPageSize;
    return (L <= 0 || L > kPageSize) ? kPageSize : L;
}

// Partial states: fp32 for f32 queries; otherwise f16, each row scaled by a
// power of two 2^-k chosen from the row's largest magnitude (below 2^15
// after scaling), so f16's range never clips and its 11-bit significand
// holds every row at the same relative precision whatever the magnitude of
// V.  k goes with the row's log2-sum-exp (PartialLse); the merge folds 2^k
// into the row's weight, which is exact.
__device__ __forceinline__ int partial_exp(float row_max_abs) {
    if (!(row_max_abs > 0.f) || !(row_max_abs < 3.0e38f)) return 0;
    return max(__builtin_amdgcn_frexp_expf(row_max_abs) - 15, -100);   // row_max_abs < 2^(k + 15)
}

template <int N>
__device__ __forceinline__ void store_u32s(uint16_t* p, const uint32_t (&v)[N]) {
    if constexpr (N % 4 == 0) {
        #pragma unroll
        for (int k = 0; k < N; k += 4)
            *reinterpret_cast<u32x4*>(p + 2 * k) = u32x4{v[k], v[k + 1], v[k + 2], v[k + 3]};
    } else if constexpr (N == 2) {
        *reinterpret_cast<u32x2*>(p) = u32x2{v[0], v[1]};
    } else {
        static_assert(N == 1, "store width");
        *reinterpret_cast<uint32_t*>(p) = v[0];
    }
}

// Writes the partial states of one wave's rows: tiles rt < nrt, row
// row0 + 16*rt + c of the item, to partial rows dst[rt].  O[rt][e][i] is
// element d = (4g+i)*EPL + e.  lrow[rt]: the row's total weight when
// ROW_SUMMED, else this lane's share (summed over the row's four lanes here).
template <int D, int RT, bool ROW_SUMMED, bool F32>
__device__ __forceinline__ void write_wave_partial(const AttendArgs& a, const Item& it, uint32_t row0,
                                                   int nrt, const uint32_t (&dst)[RT], const float (&m)[RT],
                                                   const float (&lrow)[RT], const f4 (&O)[RT][D / 16], int g,
                                                   int c) {
    constexpr int EPL = D / 16;
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (rt >= nrt) break;
        const float lt = ROW_SUMMED ? lrow[rt] : rowgroup_sum(lrow[rt]);
        const uint32_t row = row0 + rt * kTileRows + c;
        const float inv = lt > 0.f ? 1.f / lt : 0.f;
        int k = 0;
        if constexpr (!F32) {
            float mx = 0.f;
            #pragma unroll
            for (int e = 0; e < EPL; ++e)
                #pragma unroll
                for (int i = 0; i < 4; ++i) mx = fmaxf(mx, fabsf(O[rt][e][i]));
            k = partial_exp(rowgroup_max(mx) * inv);
        }
        if (row < it.nrows) {
            if constexpr (F32) {
                float* o = static_cast<float*>(a.ws_o) + uint64_t(dst[rt]) * D;
                #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    #pragma unroll
                    for (int e = 0; e < EPL; e += 4) {
                        f4 v = {O[rt][e][i] * inv, O[rt][e + 1][i] * inv, O[rt][e + 2][i] * inv,
                                O[rt][e + 3][i] * inv};
                        *reinterpret_cast<f4*>(o + (4 * g + i) * EPL + e) = v;
                    }
                }
            } else {
                const float sc = __builtin_amdgcn_ldexpf(inv, -k);
                uint16_t* o = static_cast<uint16_t*>(a.ws_o) + uint64_t(dst[rt]) * D;
                #pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint32_t v[EPL / 2];
                    #pragma unroll
                    for (int e = 0; e < EPL; e += 2) v[e / 2] = pack2(O[rt][e][i] * sc, O[rt][e + 1][i] * sc, true);
                    store_u32s<EPL / 2>(o + (4 * g + i) * EPL, v);
                }
            }
            if (g == 0) a.ws_lse[dst[rt]] = PartialLse{lt > 0.f ? m[rt] + log2f(lt) : kNegInf, float(k)};
        }
    }
}

// Query rows of NRT tiles as B operands: lane (g, c) holds row row0+16*rt+c,
// dims kb*32 + 8g .. +8 (zero for rows outside the item).  K16: the order
// of 8-bit K rows loaded in 16-byte pieces (load_page_k): k-block kb = 2j + h
// holds dims 64j + 16g + 8h .. +8.  A dot product does not depend on the
// order of its terms, so K and q only have to agree on it.
template <int D, int RT, bool K16 = false>
__device__ __forceinline__ void load_q16(const AttendArgs& a, const Item& it, uint32_t row0, int nrt,
                                         uint32_t (&qB)[RT][D / 32][4], uint32_t (&dst)[RT], int g, int c) {
    constexpr int KB = D / 32;
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const uint32_t row = row0 + rt * kTileRows + c;
        dst[rt] = 0u;
        if (rt < nrt && row < it.nrows) {
            uint32_t seq, slot, qh;
            row_target(a, it, row, seq, slot, qh);
            dst[rt] = slot * a.hq + qh;
            const uint16_t* qp = reinterpret_cast<const uint16_t*>(a.q) + (uint64_t(seq) * a.hq + qh) * D;
            #pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                load_dwords<4>(qB[rt][kb], qp + (K16 ? 64 * (kb >> 1) + 16 * g + 8 * (kb & 1) : kb * 32 + 8 * g));
                #pragma unroll
                for (int i = 0; i < 4; ++i) qB[rt][kb][i] ^= a.q_sign;
            }
        } else {
            #pragma unroll
            for (int kb = 0; kb < KB; ++kb) qB[rt][kb][0] = qB[rt][kb][1] = qB[rt][kb][2] = qB[rt][kb][3] = 0u;
        }
    }
}

// ---------------------------------------------------------------- pair math
// Scores of a page pair for NRT row tiles: s[rt][p] = S^T tile of page p
// (k0 / k1: the two pages' K operands).
template <int D, bool F16, int NRT, int RT>
__device__ __forceinline__ void pair_scores(const uint32_t (&k0)[D / 32][4], const uint32_t (&k1)[D / 32][4],
                                            const uint32_t (&qB)[RT][D / 32][4], f4 (&s)[RT][2]) {
    constexpr int KB = D / 32;
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        s[rt][0] = f4{0.f, 0.f, 0.f, 0.f};
        s[rt][1] = f4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            s[rt][0] = mma16<F16>(k0[kb], qB[rt][kb], s[rt][0]);
            s[rt][1] = mma16<F16>(k1[kb], qB[rt][kb], s[rt][1]);
        }
    }
}

// Online softmax of a pair's scores and O^T += V^T P^T.  f0/f1: scale_log2
// times the pages' K scales; v0s/v1s: the pages' V scales (1 unless FP8
// block-scaled); n0/n1: valid tokens of the two pages (n1 = 0: no page).
// v0 / v1 hold, per page, the V rows of tokens 4g+j (bf16/f16 dwords, zero
// for invalid tokens).
//
// Running max: a row's reference max m only moves when some score exceeds it
// by more than kLazy (so every exp2 stays <= 2^kLazy).  Whether that happens
// is decided from each lane's own scores and a ballot; the cross-lane max and
// the O rescale run only then, which after the first pairs is rare.
// Row sum: one more MFMA per tile multiplies the rounded probabilities by an
// all-ones A operand, so L holds, in every lane of row c, the sum of exactly
// the weights the PV MFMAs used (O / L is then a convex combination of V rows
// whatever the rounding of P).
template <int D, bool F16, int NRT, int RT, bool BLOCK_SCALE>
__device__ __forceinline__ void pair_softmax(const f4 (&s)[RT][2], int n0, int n1, float f0, float f1,
                                             float v0s, float v1s, float (&m)[RT], f4 (&L)[RT],
                                             f4 (&O)[RT][D / 16], int g, uint32_t (&pB)[RT][4]) {
    constexpr int EPL = D / 16;
    constexpr float kLazy = 8.f;                  // running-max slack (log2 units)
    const uint32_t one2 = F16 ? 0x3C003C00u : 0x3F803F80u;
    const uint32_t ones[4] = {one2, one2, one2, one2};
    const bool full = (n0 == kPageSize) && (n1 == kPageSize);
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        float x0[4], x1[4];
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            x0[i] = s[rt][0][i];
            x1[i] = s[rt][1][i];
        }
        if (!full) {
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                if (4 * g + i >= n0) x0[i] = kNegInf;
                if (4 * g + i >= n1) x1[i] = kNegInf;
            }
        }
        // Lane-local max over raw scores: the scale factors are positive
        // (scale_log2 > 0; FP8 block scales are checked on write).
        const float r0 = fmaxf(fmaxf(x0[0], x0[1]), fmaxf(x0[2], x0[3]));
        const float r1 = fmaxf(fmaxf(x1[0], x1[1]), fmaxf(x1[2], x1[3]));
        const float lm = fmaxf(r0 * f0, r1 * f1);          // -inf * f stays -inf
        if (__ballot(lm > m[rt] + kLazy)) {
            const float mx = rowgroup_max(lm);
            const float mnew = mx > m[rt] + kLazy ? mx : m[rt];
            const float alpha = (m[rt] == kNegInf) ? 0.f : fast_exp2(m[rt] - mnew);
            m[rt] = mnew;
            scale_inplace(L[rt], alpha);
            #pragma unroll
            for (int e = 0; e < EPL; ++e) scale_inplace(O[rt][e], alpha);
        }
        const float nm = (m[rt] == kNegInf) ? 0.f : -m[rt];
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            x0[i] = fast_exp2(__builtin_fmaf(x0[i], f0, nm));
            x1[i] = fast_exp2(__builtin_fmaf(x1[i], f1, nm));
        }
        uint32_t pk[4];
        pk[0] = pack2(x0[0], x0[1], F16);
        pk[1] = pack2(x0[2], x0[3], F16);
        pk[2] = pack2(x1[0], x1[1], F16);
        pk[3] = pack2(x1[2], x1[3], F16);
        L[rt] = mma16<F16>(ones, pk, L[rt]);
        if constexpr (BLOCK_SCALE) {
            pB[rt][0] = pack2(unpack_lo(pk[0], F16) * v0s, unpack_hi(pk[0], F16) * v0s, F16);
            pB[rt][1] = pack2(unpack_lo(pk[1], F16) * v0s, unpack_hi(pk[1], F16) * v0s, F16);
            pB[rt][2] = pack2(unpack_lo(pk[2], F16) * v1s, unpack_hi(pk[2], F16) * v1s, F16);
            pB[rt][3] = pack2(unpack_lo(pk[3], F16) * v1s, unpack_hi(pk[3], F16) * v1s, F16);
        } else {
            #pragma unroll
            for (int k = 0; k < 4; ++k) pB[rt][k] = pk[k];
        }
    }
}

template <int D, bool F16, int NRT, int RT, bool BLOCK_SCALE>
__device__ __forceinline__ void pair_softmax_pv(const f4 (&s)[RT][2], const uint32_t (&v0)[4][D / 32],
                                                const uint32_t (&v1)[4][D / 32],
                                                int n0, int n1, float f0, float f1, float v0s, float v1s,
                                                float (&m)[RT], f4 (&L)[RT], f4 (&O)[RT][D / 16], int g) {
    constexpr int EPL = D / 16;
    uint32_t pB[RT][4];
    pair_softmax<D, F16, NRT, RT, BLOCK_SCALE>(s, n0, n1, f0, f1, v0s, v1s, m, L, O, g, pB);
    // The V operand of a d-block (element e of the lane's 8 tokens) is
    // shared by all row tiles.
    #pragma unroll
    for (int e = 0; e < EPL; ++e) {
        const int w = e >> 1;
        const uint32_t sel = (e & 1) ? 0x07060302u : 0x05040100u;
        uint32_t vA[4];
        vA[0] = __builtin_amdgcn_perm(v0[1][w], v0[0][w], sel);
        vA[1] = __builtin_amdgcn_perm(v0[3][w], v0[2][w], sel);
        vA[2] = __builtin_amdgcn_perm(v1[1][w], v1[0][w], sel);
        vA[3] = __builtin_amdgcn_perm(v1[3][w], v1[2][w], sel);
        #pragma unroll
        for (int rt = 0; rt < NRT; ++rt) O[rt][e] = mma16<F16>(vA, pB[rt], O[rt][e]);
    }
}

// Zeroes, in a lane's 16-bit V rows (tokens 4g+j), the tokens at or past
// nt (their probabilities are zero; garbage there must not reach O).
template <int D>
__device__ __forceinline__ void mask_v_rows(uint32_t (&v)[4][D / 32], int g, int nt) {
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
        const bool ok = 4 * g + j < nt;
        #pragma unroll
        for (int w = 0; w < D / 32; ++w) v[j][w] = ok ? v[j][w] : 0u;
    }
}

// ------------------------------------------------------------- wave items
// Raw pool bytes of one page for this lane (K rows of token c, V rows of
// tokens 4g..4g+3), plus the MX scale bytes that go with them.
template <int D, uint32_t KVF>
struct PageRaw {
    static constexpr bool FP8 = (KVF == KVF_FP8 || KVF == KVF_MX);
    static constexpr int KB = D / 32;
    static constexpr int EPL = D / 16;
    static constexpr int KW = FP8 ? 2 : 4;           // dwords per k-chunk
    static constexpr int VW = FP8 ? EPL / 4 : EPL / 2;
    static constexpr int G = D / 32;                 // MX groups per token
    uint32_t k[KB][KW];
    uint32_t v[4][VW];
    uint32_t ksc[KVF == KVF_MX ? G : 1];            // MX: K scale byte per k-chunk
    uint32_t vsc[KVF == KVF_MX ? 4 : 1];            // MX: V scale byte per token j
};

template <int D, uint32_t KVF>
__device__ __forceinline__ void load_page_k(PageRaw<D, KVF>& r, const AttendArgs& a, uint32_t page,
                                            uint32_t head, int g, int c) {
    using R = PageRaw<D, KVF>;
    constexpr int EB = R::FP8 ? 1 : 2;
    const uint8_t* kp = a.kv + plane_offset(page, 0, head, a.hkv, D, EB);
    if constexpr (R::FP8) {
        // 16 codes (16 bytes) per lane: dims 64j + 16g .. +16 of token c
        // feed k-blocks 2j and 2j + 1 (the query is loaded in the same
        // order), so a load instruction reads 64-byte runs of 16 rows
        // instead of 32-byte ones.
        #pragma unroll
        for (int j = 0; j < R::KB / 2; ++j) {
            uint32_t t[4];
            load_dwords<4>(t, kp + c * D + 64 * j + 16 * g);
            r.k[2 * j][0] = t[0];
            r.k[2 * j][1] = t[1];
            r.k[2 * j + 1][0] = t[2];
            r.k[2 * j + 1][1] = t[3];
        }
    } else {
        #pragma unroll
        for (int kb = 0; kb < R::KB; ++kb)
            load_dwords<R::KW>(r.k[kb], kp + (c * D + kb * 32 + 8 * g) * EB);
    }
    if constexpr (KVF == KVF_MX) {
        // the MX group (32 dims) of k-block 2j + h's codes is 2j + g / 2
        const uint8_t* s = reinterpret_cast<const uint8_t*>(a.scales) +
                           ((uint64_t(page) * 2 + 0) * a.hkv + head) * uint64_t(kPageSize) * R::G;
        #pragma unroll
        for (int kb = 0; kb < R::G; ++kb) r.ksc[kb] = s[c * R::G + 2 * (kb >> 1) + (g >> 1)];
    }
}

template <int D, uint32_t KVF>
__device__ __forceinline__ void load_page_v(PageRaw<D, KVF>& r, const AttendArgs& a, uint32_t page,
                                            uint32_t head, int g, int c) {
    using R = PageRaw<D, KVF>;
    constexpr int EB = R::FP8 ? 1 : 2;
    const uint8_t* vp = a.kv + plane_offset(page, 1, head, a.hkv, D, EB);
    #pragma unroll
    for (int j = 0; j < 4; ++j)
        load_dwords<R::VW>(r.v[j], vp + ((4 * g + j) * D + c * R::EPL) * EB);
    if constexpr (KVF == KVF_MX) {
        const uint8_t* s = reinterpret_cast<const uint8_t*>(a.scales) +
                           ((uint64_t(page) * 2 + 1) * a.hkv + head) * uint64_t(kPageSize) * R::G;
        #pragma unroll
        for (int j = 0; j < 4; ++j) r.vsc[j] = s[(4 * g + j) * R::G + (c * R::EPL) / 32];
    }
}

// K rows of a page as MFMA A operands (bf16/f16 dwords; 8-bit codes into
// f16 when H).
template <int D, uint32_t KVF, bool H>
__device__ __forceinline__ void k_operand(const PageRaw<D, KVF>& r, uint32_t (&op)[D / 32][4]) {
    using R = PageRaw<D, KVF>;
    #pragma unroll
    for (int kb = 0; kb < R::KB; ++kb) {
        if constexpr (!R::FP8) {
            #pragma unroll
            for (int w = 0; w < 4; ++w) op[kb][w] = r.k[kb][w];
        } else {
            const float sc = KVF == KVF_MX ? e8m0_to_float(r.ksc[kb]) : 1.f;
            e4m3x4_cvt<H>(r.k[kb][0], sc, op[kb][0], op[kb][1]);
            e4m3x4_cvt<H>(r.k[kb][1], sc, op[kb][2], op[kb][3]);
        }
    }
}

// V rows of a page (tokens 4g+j, dims c*EPL..) as bf16/f16 dwords; rows of
// tokens at or beyond nt are zero so that garbage past the valid tokens can
// never reach the accumulator (their probabilities are zero).
template <int D, uint32_t KVF, bool H>
__device__ __forceinline__ void v_operand(const PageRaw<D, KVF>& r, int g, int nt,
                                          uint32_t (&op)[4][D / 32]) {
    using R = PageRaw<D, KVF>;
    #pragma unroll
    for (int j = 0; j < 4; ++j) {
        const bool ok = 4 * g + j < nt;
        if constexpr (!R::FP8) {
            #pragma unroll
            for (int w = 0; w < R::VW; ++w) op[j][w] = ok ? r.v[j][w] : 0u;
        } else {
            const float sc = KVF == KVF_MX ? e8m0_to_float(r.vsc[j]) : 1.f;
            #pragma unroll
            for (int w = 0; w < R::VW; ++w)
                e4m3x4_cvt<H>(ok ? r.v[j][w] : 0u, sc, op[j][2 * w], op[j][2 * w + 1]);
        }
    }
}

// One wave attends a wave item (one tile of <= 16 rows) over all its pages.
// The next pair's K is requested as soon as the score MFMAs have consumed K,
// its V as soon as the PV MFMAs have consumed V, so the loads of pair i+1 are
// in flight behind the math of pair i without a second register buffer.
// Past the end the loads repeat the last page: issuing them unconditionally
// keeps one load order on every path, so the wait before a pair's scores
// covers K only.
template <int D, uint32_t KVF, bool F16>
__device__ __forceinline__ void wave_item(const AttendArgs& a, const Item& it, int g, int c) {
    constexpr int EPL = D / 16;
    constexpr int KB = D / 32;
    constexpr bool BLOCK_SCALE = (KVF == KVF_FP8);
    uint32_t qB[1][KB][4];
    uint32_t dst[1];
    load_q16<D, 1, PageRaw<D, KVF>::FP8>(a, it, 0, 1, qB, dst, g, c);
    float m[1] = {kNegInf};
    f4 L[1] = {f4{0.f, 0.f, 0.f, 0.f}};
    f4 O[1][EPL];
    #pragma unroll
    for (int e = 0; e < EPL; ++e) O[0][e] = f4{0.f, 0.f, 0.f, 0.f};

    const int last_len = item_last_len(a, it);
    const uint32_t head = it.kv_head;
    const uint32_t np = it.npages;
    const float* bsc = reinterpret_cast<const float*>(a.scales);
    // The item's page ids in registers (lane l holds ids l, l + 64, ...), so
    // a refill needs no memory round trip of its own: a load issued just
    // before a refill would be the newest outstanding one, and waiting for it
    // would also drain the page loads in flight.
    const int lane = 16 * g + c;
    uint32_t idv[kWaveIdRegs];
    bool bad = false;
    #pragma unroll
    for (int k = 0; k < kWaveIdRegs; ++k) {
        const uint32_t i = uint32_t(lane + 64 * k);
        idv[k] = i < np ? a.pages[it.page_off + i] : 0u;
        bad |= idv[k] >= a.page_limit;
        idv[k] = idv[k] < a.page_limit ? idv[k] : 0u;
    }
    if (__ballot(bad) && a.seq_bad && lane == 0) a.seq_bad[it.tail_seq] = 1u;
    auto page_id = [&](uint32_t i) -> uint32_t {
        i = i < np ? i : np - 1;
        uint32_t r = 0;
        #pragma unroll
        for (int k = 0; k < kWaveIdRegs; ++k)
            if ((i >> 6) == uint32_t(k)) r = __builtin_amdgcn_readlane(idv[k], int(i & 63));
        return r;
    };

    // DEPTH page pairs in flight: buffer p % DEPTH holds pair p; once pair
    // p's K (then V) has been consumed, its K (V) registers take pair
    // p + DEPTH's.  Two for E4M3 pages at head_dim <= 128 (a pair is 32
    // registers).  16-bit pages keep one: two fit in registers at head_dim
    // 128, but on C3 the extra traffic of the tails slowed the shared-prefix
    // items beside them more than it sped the tails (30.4 against 29.2 µs).
    constexpr int DEPTH = (KVF == KVF_FP8 && D <= 128) ? 2 : 1;
    PageRaw<D, KVF> pr[DEPTH][2];
    float ks[DEPTH][2], vs[DEPTH][2];
    #pragma unroll
    for (int d = 0; d < DEPTH; ++d) ks[d][0] = ks[d][1] = vs[d][0] = vs[d][1] = 1.f;
    auto load_pair = [&](int buf, uint32_t pair, bool kpart) {
        #pragma unroll
        for (int p = 0; p < 2; ++p) {
            const uint32_t pg = page_id(2 * pair + p);
            if (kpart) {
                load_page_k<D, KVF>(pr[buf][p], a, pg, head, g, c);
                if constexpr (BLOCK_SCALE) ks[buf][p] = bsc[(uint64_t(pg) * 2 + 0) * a.hkv + head];
            } else {
                load_page_v<D, KVF>(pr[buf][p], a, pg, head, g, c);
                if constexpr (BLOCK_SCALE) vs[buf][p] = bsc[(uint64_t(pg) * 2 + 1) * a.hkv + head];
            }
        }
    };
    const uint32_t npairs = (np + 1) >> 1;
    #pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
        if (uint32_t(d) < npairs) {
            load_pair(d, d, true);
            load_pair(d, d, false);
        }
    }
    auto step = [&](int buf, uint32_t pi) {
        const uint32_t i0 = 2 * pi;
        const int n0 = page_tokens(it, i0, last_len);
        const int n1 = page_tokens(it, i0 + 1, last_len);
        f4 sc[1][2];
        const float f0 = a.scale_log2 * ks[buf][0], f1 = a.scale_log2 * ks[buf][1];
        const float v0s = vs[buf][0], v1s = vs[buf][1];
        const bool refill = pi + DEPTH < npairs;
        const bool full = (n0 == kPageSize) && (n1 == kPageSize);
        if constexpr (!PageRaw<D, KVF>::FP8) {
            // 16-bit pages are their own MFMA operands (no copies).  V past
            // a page's valid tokens is zeroed in place (the registers are
            // refilled after the PV products).
            pair_scores<D, F16, 1, 1>(pr[buf][0].k, pr[buf][1].k, qB, sc);
            if (refill) load_pair(buf, pi + DEPTH, true);
            if (!full) {
                mask_v_rows<D>(pr[buf][0].v, g, n0);
                mask_v_rows<D>(pr[buf][1].v, g, n1);
            }
            pair_softmax_pv<D, F16, 1, 1, BLOCK_SCALE>(sc, pr[buf][0].v, pr[buf][1].v, n0, n1, f0, f1, v0s, v1s,
                                                       m, L, O, g);
        } else {
            uint32_t kop[2][KB][4];
            k_operand<D, KVF, F16>(pr[buf][0], kop[0]);
            k_operand<D, KVF, F16>(pr[buf][1], kop[1]);
            pair_scores<D, F16, 1, 1>(kop[0], kop[1], qB, sc);
            if (refill) load_pair(buf, pi + DEPTH, true);
            uint32_t vop[2][4][D / 32];
            if (full) {
                v_operand<D, KVF, F16>(pr[buf][0], g, kPageSize, vop[0]);
                v_operand<D, KVF, F16>(pr[buf][1], g, kPageSize, vop[1]);
            } else {
                v_operand<D, KVF, F16>(pr[buf][0], g, n0, vop[0]);
                v_operand<D, KVF, F16>(pr[buf][1], g, n1, vop[1]);
            }
            pair_softmax_pv<D, F16, 1, 1, BLOCK_SCALE>(sc, vop[0], vop[1], n0, n1, f0, f1, v0s, v1s, m, L, O, g);
        }
        if (refill) load_pair(buf, pi + DEPTH, false);
    };
    for (uint32_t pi = 0; pi < npairs; pi += DEPTH) {
        step(0, pi);
        if (DEPTH == 2 && pi + 1 < npairs) step(DEPTH - 1, pi + 1);
    }
    const float lr[1] = {L[0][0]};
    write_wave_partial<D, 1, true, false>(a, it, 0, 1, dst, m, lr, O, g, c);
}

// ------------------------------------------------------------ group items
// LDS stage of one page pair: planes K(page 0), K(page 1), V(page 0),
// V(page 1), each 16 rows with a 16-byte pad per row (bank spread), then the
// four MX scale records.
template <int D, uint32_t KVF>
struct GroupLayout {
    static constexpr bool FP8 = (KVF == KVF_FP8 || KVF == KVF_MX);
    static constexpr int EB = FP8 ? 1 : 2;
    static constexpr int RB = D * EB;               // row bytes
    static constexpr int RS = RB + 16;              // LDS row stride
    static constexpr int PLANE = kPageSize * RS;
    static constexpr int G = D / 32;
    static constexpr int SREC = kPageSize * G;      // MX scale record bytes
    static constexpr int STAGE = 4 * PLANE + (KVF == KVF_MX ? 4 * SREC : 0);
    static constexpr int CPP = kPageSize * RB / 16; // 16-byte chunks per plane
    static constexpr int NCH = 4 * CPP / (kWaves * 64);   // chunks per thread per pair
    static constexpr int NSC = (KVF == KVF_MX) ? 4 * SREC / 4 : 0;   // scale dwords per pair
    static_assert(NCH >= 1 && (4 * CPP) % (kWaves * 64) == 0, "pair must split evenly");
    static_assert(NSC <= kWaves * 64, "scale records must fit one dword per thread");
};

template <int D, uint32_t KVF>
struct Staged {
    uint32_t d[GroupLayout<D, KVF>::NCH][4];
    uint32_t sc;
};

// Issues the global loads of page pair `pair` of the item into registers.
template <int D, uint32_t KVF>
__device__ __forceinline__ void group_issue(const AttendArgs& a, const Item& it, const uint32_t* ids,
                                            uint32_t pair, Staged<D, KVF>& st, int tid) {
    using L = GroupLayout<D, KVF>;
    const uint32_t np = it.npages;
    const uint32_t i0 = 2 * pair;
    const uint32_t p0 = ids[i0 < np ? i0 : np - 1];
    const uint32_t p1 = ids[i0 + 1 < np ? i0 + 1 : np - 1];
    #pragma unroll
    for (int u = 0; u < L::NCH; ++u) {
        const int q = tid + u * kWaves * 64;
        const int plane = q / L::CPP, within = q - plane * L::CPP;
        const uint32_t page = (plane & 1) ? p1 : p0;
        const uint8_t* src = a.kv + plane_offset(page, plane >> 1, it.kv_head, a.hkv, D, L::EB) + within * 16;
        load_dwords<4>(st.d[u], src);
    }
    if constexpr (KVF == KVF_MX) {
        if (tid < L::NSC) {
            const int rec = tid / (L::SREC / 4), w = tid - rec * (L::SREC / 4);
            const uint32_t page = (rec & 1) ? p1 : p0;
            const uint8_t* src = reinterpret_cast<const uint8_t*>(a.scales) +
                                 ((uint64_t(page) * 2 + (rec >> 1)) * a.hkv + it.kv_head) * L::SREC + 4 * w;
            st.sc = *reinterpret_cast<const uint32_t*>(src);
        }
    }
}

template <int D, uint32_t KVF>
__device__ __forceinline__ void group_commit(uint8_t* stage, const Staged<D, KVF>& st, int tid) {
    using L = GroupLayout<D, KVF>;
    #pragma unroll
    for (int u = 0; u < L::NCH; ++u) {
        const int q = tid + u * kWaves * 64;
        const int plane = q / L::CPP, within = q - plane * L::CPP;
        const int row = within / (L::RB / 16), col = within - row * (L::RB / 16);
        u32x4 v = {st.d[u][0], st.d[u][1], st.d[u][2], st.d[u][3]};
        *reinterpret_cast<u32x4*>(stage + plane * L::PLANE + row * L::RS + col * 16) = v;
    }
    if constexpr (KVF == KVF_MX) {
        if (tid < L::NSC) *reinterpret_cast<uint32_t*>(stage + 4 * L::PLANE + 4 * tid) = st.sc;
    }
}

// Reads one wave's K / V operands of a staged pair from LDS (8-bit codes
// into f16 when H, else bf16).
template <int D, uint32_t KVF, bool H>
__device__ __forceinline__ void group_operands(const uint8_t* stage, int g, int c, int n0, int n1,
                                               uint32_t (&kop)[2][D / 32][4],
                                               uint32_t (&vop)[2][4][D / 32]) {
    using L = GroupLayout<D, KVF>;
    constexpr int KB = D / 32, EPL = D / 16;
    #pragma unroll
    for (int p = 0; p < 2; ++p) {
        const uint8_t* kp = stage + p * L::PLANE + c * L::RS;
        #pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
            if constexpr (!L::FP8) {
                load_dwords<4>(kop[p][kb], kp + (kb * 32 + 8 * g) * 2);
            } else {
                uint32_t raw[2];
                load_dwords<2>(raw, kp + kb * 32 + 8 * g);
                float sc = 1.f;
                if constexpr (KVF == KVF_MX) sc = e8m0_to_float(stage[4 * L::PLANE + p * L::SREC + c * L::G + kb]);
                e4m3x4_cvt<H>(raw[0], sc, kop[p][kb][0], kop[p][kb][1]);
                e4m3x4_cvt<H>(raw[1], sc, kop[p][kb][2], kop[p][kb][3]);
            }
        }
    }
    #pragma unroll
    for (int p = 0; p < 2; ++p) {
        const int nt = p ? n1 : n0;
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int tok = 4 * g + j;
            const uint8_t* vp = stage + (2 + p) * L::PLANE + tok * L::RS + c * EPL * L::EB;
            const bool ok = tok < nt;
            if constexpr (!L::FP8) {
                uint32_t raw[EPL / 2];
                load_dwords<EPL / 2>(raw, vp);
                #pragma unroll
                for (int w = 0; w < EPL / 2; ++w) vop[p][j][w] = ok ? raw[w] : 0u;
            } else {
                uint32_t raw[EPL / 4];
                load_dwords<EPL / 4>(raw, vp);
                float sc = 1.f;
                if constexpr (KVF == KVF_MX)
                    sc = e8m0_to_float(stage[4 * L::PLANE + (2 + p) * L::SREC + tok * L::G + (c * EPL) / 32]);
                #pragma unroll
                for (int w = 0; w < EPL / 4; ++w)
                    e4m3x4_cvt<H>(ok ? raw[w] : 0u, sc, vop[p][j][2 * w], vop[p][j][2 * w + 1]);
            }
        }
    }
}

// The group item's pair loop for a wave owning NRT tiles (NRT = 0: the
// wave's rows are all outside the item; it still stages pages and joins
// every barrier).  Two LDS stages; global loads run two pairs ahead in two
// register sets A and B (loop unrolled by two so the sets never move).
template <int D, uint32_t KVF, bool F16, int NRT, int RT>
__device__ __forceinline__ void group_loop(const AttendArgs& a, const Item& it, uint8_t* lds,
                                           const uint32_t* ids, const float* bscale, int tid,
                                           int g, int c, const uint32_t (&qB)[RT][D / 32][4],
                                           float (&m)[RT], f4 (&Lsum)[RT], f4 (&O)[RT][D / 16]) {
    using L = GroupLayout<D, KVF>;
    constexpr bool BLOCK_SCALE = (KVF == KVF_FP8);
    const int last_len = item_last_len(a, it);
    const uint32_t np = it.npages;
    const uint32_t npairs = (np + 1) >> 1;
    uint8_t* stage0 = lds;
    uint8_t* stage1 = lds + L::STAGE;

    auto compute = [&](const uint8_t* stage, uint32_t pair) {
        if constexpr (NRT > 0) {
            const uint32_t i0 = 2 * pair;
            const int n0 = page_tokens(it, i0, last_len);
            const int n1 = page_tokens(it, i0 + 1, last_len);
            float f0 = a.scale_log2, f1 = a.scale_log2, v0s = 1.f, v1s = 1.f;
            if constexpr (BLOCK_SCALE) {
                const uint32_t i1 = i0 + 1 < np ? i0 + 1 : i0;
                f0 *= bscale[2 * i0];
                f1 *= bscale[2 * i1];
                v0s = bscale[2 * i0 + 1];
                v1s = bscale[2 * i1 + 1];
            }
            uint32_t kop[2][D / 32][4];
            uint32_t vop[2][4][D / 32];
            group_operands<D, KVF, F16>(stage, g, c, n0, n1, kop, vop);
            f4 s[RT][2];
            pair_scores<D, F16, NRT, RT>(kop[0], kop[1], qB, s);
            pair_softmax_pv<D, F16, NRT, RT, BLOCK_SCALE>(s, vop[0], vop[1], n0, n1, f0, f1, v0s, v1s, m, Lsum,
                                                          O, g);
        }
    };

    Staged<D, KVF> A, B;
    group_issue<D, KVF>(a, it, ids, 0, A, tid);
    group_issue<D, KVF>(a, it, ids, 1, B, tid);
    group_commit<D, KVF>(stage0, A, tid);
    group_issue<D, KVF>(a, it, ids, 2, A, tid);
    __syncthreads();
    for (uint32_t pi = 0; pi < npairs; pi += 2) {
        compute(stage0, pi);
        group_commit<D, KVF>(stage1, B, tid);      // pair pi+1
        group_issue<D, KVF>(a, it, ids, pi + 3, B, tid);
        __syncthreads();
        if (pi + 1 >= npairs) break;
        compute(stage1, pi + 1);
        group_commit<D, KVF>(stage0, A, tid);      // pair pi+2
        group_issue<D, KVF>(a, it, ids, pi + 4, A, tid);
        __syncthreads();
    }
}

template <int D, uint32_t KVF, bool F16>
__device__ __forceinline__ void group_item(const AttendArgs& a, const Item& it, int tid, int wave, int g,
                                           int c) {
    __shared__ __attribute__((aligned(16))) uint8_t lds[2 * GroupLayout<D, KVF>::STAGE +
                                                        kGroupMaxPages * 4 * (KVF == KVF_FP8 ? 3 : 1)];
    constexpr int RT = kGroupTiles8;
    constexpr int EPL = D / 16;
    constexpr int KB = D / 32;
    // The item's page ids (and FP8 block scales) go to LDS once, so the pair
    // loop reads them without a vector load, whose wait would also drain the
    // page loads running ahead.
    uint32_t* ids = reinterpret_cast<uint32_t*>(lds + 2 * GroupLayout<D, KVF>::STAGE);
    float* bscale = reinterpret_cast<float*>(ids + kGroupMaxPages);
    for (uint32_t i = tid; i < it.npages; i += kWaves * 64) {
        uint32_t pg = a.pages[it.page_off + i];
        pg = pg < a.page_limit ? pg : 0u;
        ids[i] = pg;
        if constexpr (KVF == KVF_FP8) {
            const float* bsc = reinterpret_cast<const float*>(a.scales);
            bscale[2 * i] = bsc[(uint64_t(pg) * 2 + 0) * a.hkv + it.kv_head];
            bscale[2 * i + 1] = bsc[(uint64_t(pg) * 2 + 1) * a.hkv + it.kv_head];
        }
    }
    __syncthreads();
    const uint32_t row0 = uint32_t(wave) * RT * kTileRows;
    const int nrt = it.nrows > row0 ? min(RT, int((it.nrows - row0 + kTileRows - 1) / kTileRows)) : 0;
    uint32_t qB[RT][KB][4];
    uint32_t dst[RT];
    load_q16<D, RT>(a, it, row0, nrt, qB, dst, g, c);
    float m[RT];
    f4 L[RT];
    f4 O[RT][EPL];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m[rt] = kNegInf;
        L[rt] = f4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int e = 0; e < EPL; ++e) O[rt][e] = f4{0.f, 0.f, 0.f, 0.f};
    }
    if (nrt == RT) group_loop<D, KVF, F16, RT, RT>(a, it, lds, ids, bscale, tid, g, c, qB, m, L, O);
    else if (nrt == 1) group_loop<D, KVF, F16, 1, RT>(a, it, lds, ids, bscale, tid, g, c, qB, m, L, O);
    else group_loop<D, KVF, F16, 0, RT>(a, it, lds, ids, bscale, tid, g, c, qB, m, L, O);
    float lr[RT];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) lr[rt] = L[rt][0];
    write_wave_partial<D, RT, true, false>(a, it, row0, nrt, dst, m, lr, O, g, c);
}

// ------------------------------------------------- group items, 16-bit KV
// Pages reach LDS by direct global->LDS loads (global_load_lds_dwordx4, one
// 1 KiB wave load per 64 lanes x 16 bytes): no staging registers and no
// VALU work.  The LDS ring holds NP page pairs; pair p goes to slot p % NP.
// The loads are issued from inline assembly, so the compiler tracks none of
// them and inserts no wait of its own on the ring: before pair p is read
// each wave waits (vmcnt) until its own loads of pair p have landed, and the
// barrier that follows makes every wave's share of the pair visible.  After
// that barrier the slot of pair p - 1 is free and takes pair p + NP - 1.
//
// The item's query rows take the same route: at the start each wave loads
// its rows into the last QSLOTS slots (lane l of a wave load receives bytes
// 16 l.., so each lane reads its own MFMA operand back), then reads them to
// registers; a barrier frees those slots for pages.  The page ids, the row
// targets and the query rows thus cost one dependent memory round trip each
// at the start of an item instead of a chain of them.
//
// A slot holds one page: the K plane (16 rows) then the V plane.  The
// 16-byte chunks of row r are XOR-swizzled (chunk j at position j ^ swz(r)),
// which keeps both read patterns free of bank conflicts:
//   K (A operand of the scores): lane (g, c) reads row c, chunk 4kb + g;
//   V (A operand of O^T, by ds_read_b64_tr_b16): lane (g, c) reads 8 bytes of
//   row 4g + c/4 at dims 16e + 4(c%4); within each 16-lane group the
//   transpose hands lane c the values V[4g + j][16e + c], j = 0..3 — the
//   MFMA's k = 4g + j slots — so the accumulators hold O[row][16e + 4g + i].
// Each wave owns row tiles w, w+4 (RT = 2; one tile for D = 256) of the item.
template <int D>
struct DmaCfg {
    static constexpr int RB = 2 * D;                  // bytes per row
    static constexpr int PLANE = kPageSize * RB;
    static constexpr int PAGE = 2 * PLANE;            // 4, 8 or 16 KiB
    // Four page pairs.  At D = 64 eight pairs (64 KiB) are slower: prefill
    // of 12 prompts of 37-1 500 tokens, 32 / 4 heads, f16, 76.2 us against
    // 73.2.  Registers hold that kernel at two workgroups a CU either way, but
    // its code, unrolled over the ring's slots, was as long as the 64 KiB
    // instruction cache two CUs share, and is 37 KiB.  The decode kernel, of
    // fewer registers, goes from two workgroups a CU to three (a forked batch
    // of 32-page items: the same time).
    static constexpr int RING = D * 512;              // LDS bytes of the ring
    static constexpr int NP = RING / (2 * PAGE);      // page pairs in the ring
    static constexpr int DPP = PAGE / (kWaves * 64 * 16);   // wave loads per thread per page
    static constexpr int PER_PAIR = 2 * DPP;          // loads per thread per pair
    static constexpr int RT = group_tiles16(D);       // row tiles per wave
    static constexpr int QBYTES = kWaves * RT * (D / 32) * 1024;   // the item's query rows
    static constexpr int QSLOTS = (QBYTES + 2 * PAGE - 1) / (2 * PAGE);
    static_assert(NP - QSLOTS >= 2, "query rows leave two pair slots");
    static_assert(DPP >= 1 && PLANE % 1024 == 0, "a page must split into 1 KiB wave loads");
    static_assert(NP >= 3 && (NP - 2) * PER_PAIR <= 48, "vmcnt cases");
    static_assert(DPP <= 4, "DmaSrc holds four offsets");
};

// Row swizzle of the 16-byte chunks.  Both read patterns were measured on
// gfx950 (SQ_LDS_BANK_CONFLICT, one probe kernel per pattern): these values
// leave the K reads (ds_read_b128) and the transposed V reads
// (ds_read_b64_tr_b16) without bank conflicts at head_dim 64, 128 and 256.
// Setting bit 0 from row >> 3 as well makes the K reads two-way conflicted.
template <int D>
__device__ __forceinline__ int chunk_swz(int row) {
    if constexpr (D == 64) return ((row >> 1) & 3) << 1;
    else return (row & 7) << 1;
}

typedef short s16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
typedef __attribute__((address_space(3))) void lds_void;

template <bool F16>
__device__ __forceinline__ f4 mma16v(u32x4 a, u32x4 b, f4 c) {
    if constexpr (F16)
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b),
                                                      c, 0, 0, 0);
    else
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a),
                                                       __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

__device__ __forceinline__ void compiler_fence() { asm volatile("" ::: "memory"); }

// s_waitcnt vmcnt(n) for even n <= 48 (s_waitcnt takes an immediate).
__device__ __forceinline__ void wait_vmcnt(uint32_t n) {
    switch (n) {
        case 0: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
        case 2: asm volatile("s_waitcnt vmcnt(2)" ::: "memory"); break;
        case 4: asm volatile("s_waitcnt vmcnt(4)" ::: "memory"); break;
        case 6: asm volatile("s_waitcnt vmcnt(6)" ::: "memory"); break;
        case 8: asm volatile("s_waitcnt vmcnt(8)" ::: "memory"); break;
        case 10: asm volatile("s_waitcnt vmcnt(10)" ::: "memory"); break;
        case 12: asm volatile("s_waitcnt vmcnt(12)" ::: "memory"); break;
        case 14: asm volatile("s_waitcnt vmcnt(14)" ::: "memory"); break;
        case 16: asm volatile("s_waitcnt vmcnt(16)" ::: "memory"); break;
        case 18: asm volatile("s_waitcnt vmcnt(18)" ::: "memory"); break;
        case 20: asm volatile("s_waitcnt vmcnt(20)" ::: "memory"); break;
        case 22: asm volatile("s_waitcnt vmcnt(22)" ::: "memory"); break;
        case 24: asm volatile("s_waitcnt vmcnt(24)" ::: "memory"); break;
        case 26: asm volatile("s_waitcnt vmcnt(26)" ::: "memory"); break;
        case 28: asm volatile("s_waitcnt vmcnt(28)" ::: "memory"); break;
        case 30: asm volatile("s_waitcnt vmcnt(30)" ::: "memory"); break;
        case 32: asm volatile("s_waitcnt vmcnt(32)" ::: "memory"); break;
        case 34: asm volatile("s_waitcnt vmcnt(34)" ::: "memory"); break;
        case 36: asm volatile("s_waitcnt vmcnt(36)" ::: "memory"); break;
        case 38: asm volatile("s_waitcnt vmcnt(38)" ::: "memory"); break;
        case 40: asm volatile("s_waitcnt vmcnt(40)" ::: "memory"); break;
        case 42: asm volatile("s_waitcnt vmcnt(42)" ::: "memory"); break;
        case 44: asm volatile("s_waitcnt vmcnt(44)" ::: "memory"); break;
        case 46: asm volatile("s_waitcnt vmcnt(46)" ::: "memory"); break;
        case 48: asm volatile("s_waitcnt vmcnt(48)" ::: "memory"); break;
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    }
}

template <int N>
__device__ __forceinline__ void wait_vmcnt_const() {
    static_assert(N >= 0 && N <= 63, "vmcnt range");
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Barrier after this wave's LDS reads have returned (lgkmcnt(0)), so no
// read of a slot can still be in flight when another wave refills it.
__device__ __forceinline__ void block_barrier() {
    __builtin_amdgcn_s_waitcnt(0xC07F);
    compiler_fence();
    __builtin_amdgcn_s_barrier();
    compiler_fence();
}

// Lane byte offsets inside a slot of the K operand read of k-block 0 and
// the transposed V read of d-block 0.  The swizzle is an XOR on the chunk
// index (bits 4..7 of the offset): chunk 4kb + g -> (4kb + g) ^ swz =
// 4 (kb ^ (swz >> 2)) + (g ^ (swz & 3)), so k-block kb is at k ^ (kb << 6)
// and d-block e at v ^ (e << 5) (chunk 2e + h likewise).
struct LdsOffsets {
    uint32_t k;
    uint32_t v;
};

template <int D>
__device__ __forceinline__ LdsOffsets lds_offsets(int g, int c) {
    using C = DmaCfg<D>;
    LdsOffsets o;
    o.k = c * C::RB + ((g ^ chunk_swz<D>(c)) << 4);
    const int row = 4 * g + (c >> 2);
    o.v = C::PLANE + row * C::RB + ((((c & 3) >> 1) ^ chunk_swz<D>(row)) << 4) + ((c & 1) << 3);
    return o;
}

typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

// A lane's LDS read addresses for every k-block and d-block of a pair slot
// at byte offset 0 from `base`.  Bases and slots are multiples of 1 KiB, so
// the swizzle XOR (bits 4..7) and the slot offset commute: the block of a
// slot at offset s is at k[kb] + s, and with s known at compile time the
// read takes it as its immediate offset (no address arithmetic per pair).
template <int D>
struct LdsBases {
    uint32_t k[D / 32];
    uint32_t v[D / 16];
};

template <int D>
__device__ __forceinline__ LdsBases<D> lds_bases(uint32_t base, int g, int c) {
    const LdsOffsets o = lds_offsets<D>(g, c);
    LdsBases<D> b;
    #pragma unroll
    for (int kb = 0; kb < D / 32; ++kb) b.k[kb] = base + (o.k ^ uint32_t(kb << 6));
    #pragma unroll
    for (int e = 0; e < D / 16; ++e) b.v[e] = base + (o.v ^ uint32_t(e << 5));
    return b;
}

// Zeroes the V values of tokens 4g + j >= n (j = 0..3) in one page's half
// (dwords w0, w0+1) of a transposed V operand.
__device__ __forceinline__ void mask_v_tr(u32x4& v, int w0, int g, int n) {
    #pragma unroll
    for (int w = 0; w < 2; ++w) {
        const int t = 4 * g + 2 * w;
        const uint32_t keep = (t < n ? 0x0000FFFFu : 0u) | (t + 1 < n ? 0xFFFF0000u : 0u);
        v[w0 + w] &= keep;
    }
}

// Softmax pieces of the DMA path.  Scores are in log2 units once multiplied
// by f = scale_log2 > 0 (a negative scale is folded into the query's sign).
// A row's reference max m moves only when a score passes it by kLazyDma
// (kLazyDma16 when the probabilities are packed as f16); in between,
// exp2(x - m) stays below 2^32 (bf16 range) or 2^14 (f16, whose range ends
// at 2^16), so the accumulators are not rescaled on the common path.  The check compares the lane's raw score max with
// thr = (m + kLazyDma) / f, kept per row, so the common path spends no
// multiply on it.  The move (always on the item's first pair, where m and
// thr start at -inf) runs on a slow path.
constexpr float kLazyDma = 32.f;
constexpr float kLazyDma16 = 14.f;

template <int RT>
struct RowMax {
    float m[RT];     // reference max, log2 units
    float thr[RT];   // raw score above which m must move
};

// Masks invalid tokens (PARTIAL) and returns the lane's raw score max over
// the pair.
template <int RT, bool PARTIAL>
__device__ __forceinline__ float dma_lane_max(f4 (&s)[RT][2], int rt, int n0, int n1, int g) {
    f4& x0 = s[rt][0];
    f4& x1 = s[rt][1];
    if constexpr (PARTIAL) {
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (4 * g + i >= n0) x0[i] = kNegInf;
            if (4 * g + i >= n1) x1[i] = kNegInf;
        }
    }
    const float a = fmaxf(fmaxf(x0[0], x0[1]), x0[2]);
    const float b = fmaxf(fmaxf(a, x0[3]), x1[0]);
    const float c = fmaxf(fmaxf(b, x1[1]), x1[2]);
    return fmaxf(c, x1[3]);
}

// dma_lane_max for pages whose K scales (ks0, ks1 > 0) are applied to the
// scores rather than to K: the max of raw * ks.
template <int RT, bool PARTIAL>
__device__ __forceinline__ float dma_lane_max_ks(f4 (&s)[RT][2], int rt, int n0, int n1, int g, float ks0,
                                                 float ks1) {
    f4& x0 = s[rt][0];
    f4& x1 = s[rt][1];
    if constexpr (PARTIAL) {
        #pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (4 * g + i >= n0) x0[i] = kNegInf;
            if (4 * g + i >= n1) x1[i] = kNegInf;
        }
    }
    const float r0 = fmaxf(fmaxf(fmaxf(x0[0], x0[1]), x0[2]), x0[3]);
    const float r1 = fmaxf(fmaxf(fmaxf(x1[0], x1[1]), x1[2]), x1[3]);
    return fmaxf(r0 * ks0, r1 * ks1);
}

// The slow path: moves m of every row whose scores passed thr and rescales
// its accumulators.  Rows that did not move get alpha = 1.
template <int D, int NRT, bool F16>
__device__ __forceinline__ void dma_rescale(const float (&lm)[DmaCfg<D>::RT], RowMax<DmaCfg<D>::RT>& rm,
                                         f4 (&Lsum)[DmaCfg<D>::RT], f4 (&O)[DmaCfg<D>::RT][D / 16], float f,
                                         float finv) {
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        const float mx = rowgroup_max(lm[rt]);
        if (mx > rm.thr[rt]) {
            const float mnew = mx * f;
            const float alpha = rm.m[rt] == kNegInf ? 0.f : fast_exp2(rm.m[rt] - mnew);
            rm.m[rt] = mnew;
            rm.thr[rt] = (mnew + (F16 ? kLazyDma16 : kLazyDma)) * finv;
            Lsum[rt] *= alpha;
            #pragma unroll
            for (int e = 0; e < D / 16; ++e) O[rt][e] *= alpha;
        }
    }
}

// Probabilities of one tile with reference max m (finite: the item's first
// pair always sets it), packed for the PV MFMA, and the row sums they add
// (MFMA against an all-ones operand).
// f0, f1: the two pages' score factors (f times their K scales when those
// are applied to the scores).
template <bool F16>
__device__ __forceinline__ u32x4 dma_probs(const f4 (&x)[2], float f0, float f1, float m, f4& L) {
    const uint32_t one2 = F16 ? 0x3C003C00u : 0x3F803F80u;
    const u32x4 ones = {one2, one2, one2, one2};
    const float nm = -m;
    float p0[4], p1[4];
    #pragma unroll
    for (int i = 0; i < 4; ++i) {
        p0[i] = fast_exp2(__builtin_fmaf(x[0][i], f0, nm));
        p1[i] = fast_exp2(__builtin_fmaf(x[1][i], f1, nm));
    }
    const u32x4 pb = {pack2(p0[0], p0[1], F16), pack2(p0[2], p0[3], F16), pack2(p1[0], p1[1], F16),
                      pack2(p1[2], p1[3], F16)};
    L = mma16v<F16>(ones, pb, L);
    return pb;
}

struct DmaSrc {
    uint32_t loff[4];                 // this lane's source offsets inside a page (DPP <= 4)
    uint64_t page_stride;
};

// One wave load of 64 x 16 bytes from gbase + voff (per lane) to the LDS
// address lds (wave-uniform) + 16 * lane.  Issued from inline assembly: the
// compiler does not track it, so it adds no drain of its own before the LDS
// reads; the pair loop waits for it with explicit vmcnt counts.
__device__ __forceinline__ void dma_x4(uint32_t lds, const void* gbase, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(gbase)
                 : "memory", "m0");
}

// Issues this wave's share of the loads of pages pg0, pg1 into pair slot `ps`.
template <int D>
__device__ __forceinline__ void dma_pair_pages(const AttendArgs& a, uint32_t pg0, uint32_t pg1, const DmaSrc& src,
                                               uint32_t ring, uint32_t ps, int wave) {
    using C = DmaCfg<D>;
    #pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint8_t* base = a.kv + uint64_t(q == 0 ? pg0 : pg1) * src.page_stride;
        const uint32_t slot = ring + (2 * ps + q) * C::PAGE + wave * C::DPP * 1024;
        #pragma unroll
        for (int u = 0; u < C::DPP; ++u) dma_x4(slot + u * 1024, base, src.loff[u]);
    }
}

// Issues this wave's share of the loads of pair `pair` into pair slot `ps`.
template <int D>
__device__ __forceinline__ void dma_pair(const AttendArgs& a, const Item& it, const uint32_t* ids,
                                         const DmaSrc& src, uint32_t ring, uint32_t pair, uint32_t ps, int wave) {
    using C = DmaCfg<D>;
    const uint32_t np = it.npages;
    #pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t i = 2 * pair + q < np ? 2 * pair + q : np - 1;
        const uint32_t pg = __builtin_amdgcn_readfirstlane(ids[i]);
        const uint8_t* base = a.kv + uint64_t(pg) * src.page_stride;
        const uint32_t slot = ring + (2 * ps + q) * C::PAGE + wave * C::DPP * 1024;
        #pragma unroll
        for (int u = 0; u < C::DPP; ++u) dma_x4(slot + u * 1024, base, src.loff[u]);
    }
}

// K operands of the page pair in the slot at byte offset s (pages at s and
// s + PAGE from the bases' origin).
template <int D>
__device__ __forceinline__ void dma_k_operands(uint32_t s, const LdsBases<D>& lb, u32x4 (&kop)[2][D / 32]) {
    using C = DmaCfg<D>;
    #pragma unroll
    for (int kb = 0; kb < D / 32; ++kb) {
        kop[0][kb] = *reinterpret_cast<const lds_u32x4*>(uintptr_t(lb.k[kb] + s));
        kop[1][kb] = *reinterpret_cast<const lds_u32x4*>(uintptr_t(lb.k[kb] + s + C::PAGE));
    }
}

// Scores of a page pair for the wave's NRT tiles from its K operands.
template <int D, bool F16, int NRT>
__device__ __forceinline__ void dma_score_mma(const u32x4 (&kop)[2][D / 32],
                                              const u32x4 (&qB)[DmaCfg<D>::RT][D / 32],
                                              f4 (&sc)[DmaCfg<D>::RT][2]) {
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        sc[rt][0] = f4{0.f, 0.f, 0.f, 0.f};
        sc[rt][1] = f4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int kb = 0; kb < D / 32; ++kb) {
            sc[rt][0] = mma16v<F16>(kop[0][kb], qB[rt][kb], sc[rt][0]);
            sc[rt][1] = mma16v<F16>(kop[1][kb], qB[rt][kb], sc[rt][1]);
        }
    }
}

// Scores of the page pair in the slot at offset s for the wave's NRT tiles.
template <int D, bool F16, int NRT>
__device__ __forceinline__ void dma_scores(uint32_t s, const LdsBases<D>& lb,
                                           const u32x4 (&qB)[DmaCfg<D>::RT][D / 32],
                                           f4 (&sc)[DmaCfg<D>::RT][2]) {
    u32x4 kop[2][D / 32];
    dma_k_operands<D>(s, lb, kop);
    dma_score_mma<D, F16, NRT>(kop, qB, sc);
}

// The transposed V operands of the page pair in the slot at offset s, all
// d-blocks at once (read before the scores so they land behind the MFMAs).
template <int D>
__device__ __forceinline__ void dma_v_operands(uint32_t s, const LdsBases<D>& lb, u32x4 (&vop)[D / 16]) {
    using C = DmaCfg<D>;
    #pragma unroll
    for (int e = 0; e < D / 16; ++e) {
        const uint32_t ad = lb.v[e] + s;
        const s16x4 v0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)uintptr_t(ad));
        const s16x4 v1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4*)uintptr_t(ad + C::PAGE));
        vop[e] = __builtin_shufflevector(__builtin_bit_cast(u32x2, v0), __builtin_bit_cast(u32x2, v1), 0, 1, 2, 3);
    }
}

// Token masks of a page pair: s0[rt] / s1[rt] tokens of the two pages are
// visible to the lane's row of tile rt (scores of the others are masked),
// v0 / v1 tokens hold data (V past them is zeroed, so garbage past a
// sequence's last token cannot reach O through a zero weight).
template <int RT>
struct PairMask {
    int s0[RT], s1[RT];
    int v0, v1;
};

template <int RT>
__device__ __forceinline__ PairMask<RT> uniform_mask(int n0, int n1) {
    PairMask<RT> m;
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        m.s0[rt] = n0;
        m.s1[rt] = n1;
    }
    m.v0 = n0;
    m.v1 = n1;
    return m;
}

// Masks of the pair starting at token t of a causal item: row tile rt sees
// lenr[rt] tokens of the sequence, of which the item holds those below lmax
// (rows of a chunk before the last see past its end: the cap keeps a
// missing second page of the item's last pair masked).
template <int RT>
__device__ __forceinline__ PairMask<RT> causal_mask(int t, const uint32_t (&lenr)[RT], int lmax) {
    auto cl = [](int x) { return min(max(x, 0), kPageSize); };
    PairMask<RT> m;
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        const int len = min(int(lenr[rt]), lmax);
        m.s0[rt] = cl(len - t);
        m.s1[rt] = cl(len - t - kPageSize);
    }
    m.v0 = cl(lmax - t);
    m.v1 = cl(lmax - t - kPageSize);
    return m;
}

// One step of the pair loop after its barrier: the lazy-max check of pair
// p (scores already in sc) and its rare rescale, then the LDS reads (V of
// pair p from the slot at offset vs and, when NEXT, K of pair p + 1 from the
// slot at ks), the score MFMAs of pair p + 1 interleaved with the softmax of
// pair p, and the PV MFMAs.  PART masks tokens past n0 / n1 (the item's
// last pair only); the last pair has no next pair (NEXT false).  KS: the
// pages' K scales ks0, ks1 multiply the scores (K was staged unscaled).
template <int D, bool F16, int NRT, bool PART, bool NEXT, bool KS = false, bool PF16 = F16>
__device__ __forceinline__ void dma_step(uint32_t vs, uint32_t ks, const PairMask<DmaCfg<D>::RT>& pm,
                                         const LdsBases<D>& lb,
                                         const u32x4 (&qB)[DmaCfg<D>::RT][D / 32], f4 (&sc)[DmaCfg<D>::RT][2],
                                         u32x4 (&vop)[D / 16], RowMax<DmaCfg<D>::RT>& rm,
                                         f4 (&Lsum)[DmaCfg<D>::RT], f4 (&O)[DmaCfg<D>::RT][D / 16], int g,
                                         float f, float finv, float ks0 = 1.f, float ks1 = 1.f) {
    constexpr int RT = DmaCfg<D>::RT, KB = D / 32;
    bool need = false;
    float lm[RT];
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        if constexpr (KS) lm[rt] = dma_lane_max_ks<RT, PART>(sc, rt, pm.s0[rt], pm.s1[rt], g, ks0, ks1);
        else lm[rt] = dma_lane_max<RT, PART>(sc, rt, pm.s0[rt], pm.s1[rt], g);
        need |= lm[rt] > rm.thr[rt];
    }
    if (__ballot(need)) dma_rescale<D, NRT, PF16>(lm, rm, Lsum, O, f, finv);
    // Branch-free from here, so the scheduler sees one region, in this
    // order (pinned: a wave issues in order, and at most 15 LDS reads may
    // be outstanding before issue stalls): the K reads of pair p + 1; the
    // softmax of pair p (VALU), which needs no LDS, while they are in
    // flight; the score MFMAs of pair p + 1 with the V reads of pair p
    // issued one between each two; then the PV MFMAs of pair p.
    __builtin_amdgcn_sched_barrier(0);
    u32x4 kop[2][KB];
    if constexpr (NEXT) dma_k_operands<D>(ks, lb, kop);
    __builtin_amdgcn_sched_barrier(0);
    u32x4 pB[RT];
    const float f0 = KS ? f * ks0 : f, f1 = KS ? f * ks1 : f;
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) pB[rt] = dma_probs<PF16>(sc[rt], f0, f1, rm.m[rt], Lsum[rt]);
    __builtin_amdgcn_sched_barrier(0);
    dma_v_operands<D>(vs, lb, vop);
    if constexpr (NEXT) {
        dma_score_mma<D, F16, NRT>(kop, qB, sc);
        constexpr int NM = NRT * 2 * KB, NV = D / 8;   // score MFMAs, V reads
        #pragma unroll
        for (int k = 0; k < (NM > NV ? NM : NV); ++k) {
            if (k < NV) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);   // one LDS read
            if (k < NM) __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);   // one MFMA
        }
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (PART) {
        #pragma unroll
        for (int e = 0; e < D / 16; ++e) {
            mask_v_tr(vop[e], 0, g, pm.v0);
            mask_v_tr(vop[e], 2, g, pm.v1);
        }
    }
    #pragma unroll
    for (int e = 0; e < D / 16; ++e) {
        #pragma unroll
        for (int rt = 0; rt < NRT; ++rt) O[rt][e] = mma16v<PF16>(vop[e], pB[rt], O[rt][e]);
    }
}

// Compile-time loop index.
template <int J>
struct Idx {
    static constexpr int value = J;
};

template <int J, int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
    if constexpr (J < N) {
        f(Idx<J>{});
        static_for<J + 1, N>(f);
    }
}

// Where the rows of a wave's tiles come from and go to: the byte offset of
// the query row in q and the partial-state row, read once per item.  Rows
// past the item's last are given its last row (their query is zeroed and
// nothing is written for them).
template <int RT>
struct RowTargets {
    uint32_t qoff[RT];
    uint32_t dst[RT];
    uint32_t len[RT];    // tokens the row sees (causal items only)
};

template <int D, int RT>
__device__ __forceinline__ void dma_row_targets(const AttendArgs& a, const Item& it, int wave, int c,
                                                RowTargets<RT>& rtg) {
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        uint32_t row = uint32_t(rt * kWaves + wave) * kTileRows + c;
        row = row < it.nrows ? row : it.nrows - 1;
        uint32_t seq, slot, qh;
        row_target(a, it, row, seq, slot, qh);
        rtg.qoff[rt] = (seq * a.hq + qh) * uint32_t(D * 2);
        rtg.dst[rt] = slot * a.hq + qh;
        rtg.len[rt] = (it.flags & kItemCausal) ? a.row_len[seq] : 0u;
    }
}

template <int D, bool F16, int NRT, bool TAIL, bool CAUSAL>
__device__ __forceinline__ void dma_group_loop(const AttendArgs& a, const Item& it, const uint32_t* ids,
                                               uint8_t* ring, int tid, int wave, int g, int c,
                                               const RowTargets<DmaCfg<D>::RT>& rtg, int last_len,
                                               const ItemLim& lim,
                                               u32x4 (&qB)[DmaCfg<D>::RT][D / 32],
                                               RowMax<DmaCfg<D>::RT>& rm, f4 (&Lsum)[DmaCfg<D>::RT],
                                               f4 (&O)[DmaCfg<D>::RT][D / 16]) {
    using C = DmaCfg<D>;
    constexpr uint32_t P = C::NP, QS = C::QSLOTS;
    constexpr int KB = D / 32;
    const uint32_t np = it.npages;
    const uint32_t npairs = (np + 1) >> 1;
    DmaSrc src;
    src.page_stride = uint64_t(2) * a.hkv * C::PLANE;
    #pragma unroll
    for (int u = 0; u < C::DPP; ++u) {
        const int b = (wave * C::DPP + u) * 1024 + 16 * (tid & 63);
        const int plane = b / C::PLANE, rem = b - plane * C::PLANE;
        const int row = rem / C::RB, pos = (rem - row * C::RB) >> 4;
        const int j = pos ^ chunk_swz<D>(row);
        src.loff[u] = uint32_t((plane * a.hkv + it.kv_head) * C::PLANE + row * C::RB + j * 16);
    }
    const uint32_t ring_lds = __builtin_amdgcn_readfirstlane(uint32_t(reinterpret_cast<uintptr_t>(ring)));
    const LdsBases<D> lb = lds_bases<D>(ring_lds, g, c);
    const float f = a.scale_log2;   // > 0 (a negative scale is in q_sign)
    const float finv = 1.f / f;
    const uint32_t qsign = a.q_sign;
    // Every load the compiler issued (row targets, page ids) has landed
    // before the ring loads start, so no compiler-inserted wait can drain
    // the ring.
    __builtin_amdgcn_s_waitcnt(0x0070);
    compiler_fence();
    // Query rows into the last QS slots, the first pairs into the others.
    const uint32_t q_lds = ring_lds + (P - QS) * 2 * C::PAGE + wave * (C::RT * KB * 1024);
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        #pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            dma_x4(q_lds + (rt * KB + kb) * 1024, static_cast<const uint8_t*>(a.q), rtg.qoff[rt] + kb * 64 + 16 * g);
    }
    const uint32_t pro = min(P - QS, npairs);
    #pragma unroll 1
    for (uint32_t q = 0; q < pro; ++q) dma_pair<D>(a, it, ids, src, ring_lds, q, q, wave);
    wait_vmcnt(pro * C::PER_PAIR);   // loads land in issue order: the query rows are in
    if constexpr (NRT > 0) {
        const uint8_t* qw = ring + (P - QS) * 2 * C::PAGE + wave * (C::RT * KB * 1024) + 16 * (tid & 63);
        #pragma unroll
        for (int rt = 0; rt < NRT; ++rt) {
            const bool valid = uint32_t(rt * kWaves + wave) * kTileRows + c < it.nrows;
            #pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(qw + (rt * KB + kb) * 1024) ^ qsign;
                qB[rt][kb] = valid ? v : u32x4{0u, 0u, 0u, 0u};
            }
        }
    }
    block_barrier();   // every wave holds its query rows: their slots take pages
    #pragma unroll 1
    for (uint32_t q = pro; q < min(P - 1, npairs); ++q) dma_pair<D>(a, it, ids, src, ring_lds, q, q, wave);
    // Software pipeline: step pi computes the scores of pair pi + 1 while
    // it finishes pair pi.  It reads K of pair pi + 1 and V of pair pi;
    // after its barrier the slot of pair pi - 1 is free and takes pair
    // pi + P - 1.  Pair p sits in slot p % P, so the steps are unrolled
    // over the P slots and every LDS read takes its slot as an immediate
    // offset.  Issued before step pi: pairs < min(pi + P - 1, npairs).
    // Order inside a step (pinned with scheduling barriers, since a wave
    // issues in order): the row-max check of pair pi (its scores are
    // already in registers) and the rare rescale; then all LDS reads; then
    // the probabilities of pair pi (VALU) interleaved with the score MFMAs
    // of pair pi + 1; then the PV MFMAs of pair pi.  The last pair runs
    // apart: it may hold partial pages and has no next pair to score.
    constexpr int RT = C::RT;
    constexpr uint32_t SLOT = 2 * C::PAGE;
    f4 sc[RT][2];
    u32x4 vop[D / 16];
    wait_vmcnt((min(P - 1, npairs) - 1) * C::PER_PAIR);   // pair 0 has landed
    block_barrier();
    if constexpr (NRT > 0) dma_scores<D, F16, NRT>(0, lb, qB, sc);
    // Page ids of the pair the next refill loads (pair pi + P - 1), read from
    // LDS a step ahead so the refill does not wait on them.
    uint32_t nid0 = ids[min(2 * (P - 1), np - 1)];
    uint32_t nid1 = ids[min(2 * (P - 1) + 1, np - 1)];
    const uint32_t nmain = npairs - 1;
    #pragma unroll 1
    for (uint32_t p0 = 0; p0 < nmain; p0 += P) {
        static_for<0, int(P)>([&](auto J) {
            constexpr uint32_t j = decltype(J)::value;
            const uint32_t pi = p0 + j;
            if (pi >= nmain) return;
            // Most instructions of a step are eight bytes long; where they
            // straddle eight-byte words the prefill loop is slower (head_dim
            // 256, 16-bit, 1 148 items over 4 000 tokens: 179.4 us aligned,
            // 181.4 four bytes off; at 128 and 64 the same time).
            if constexpr (CAUSAL) asm volatile(".p2align 3");
            if (pi + P - 1 <= npairs) wait_vmcnt_const<(P - 3) * C::PER_PAIR>();   // pair pi + 1 has landed
            else wait_vmcnt((npairs - pi - 2) * C::PER_PAIR);
            block_barrier();
            if (pi + P - 1 < npairs)
                dma_pair_pages<D>(a, __builtin_amdgcn_readfirstlane(nid0), __builtin_amdgcn_readfirstlane(nid1),
                                  src, ring_lds, (j + P - 1) % P, wave);
            nid0 = ids[min(2 * (pi + P), np - 1)];
            nid1 = ids[min(2 * (pi + P) + 1, np - 1)];
            if constexpr (NRT > 0) {
                // A causal item's pairs below every row's last token need no
                // mask; the ones crossing the diagonal mask per row.
                const int t = CAUSAL ? int(lim.tok0 + 2 * kPageSize * pi) : 0;
                if (CAUSAL && t + 2 * kPageSize > int(lim.lmin))
                    dma_step<D, F16, NRT, true, true>(j * SLOT, ((j + 1) % P) * SLOT,
                                                      causal_mask<RT>(t, rtg.len, int(lim.lmax)), lb, qB, sc,
                                                      vop, rm, Lsum, O, g, f, finv);
                else
                    dma_step<D, F16, NRT, false, true>(j * SLOT, ((j + 1) % P) * SLOT,
                                                       uniform_mask<RT>(kPageSize, kPageSize), lb, qB, sc, vop,
                                                       rm, Lsum, O, g, f, finv);
            }
        });
    }
    // The last pair: its loads were waited for (vmcnt(0)) and made visible
    // by the previous step's barrier (or the prologue's); it refills nothing
    // and reads no K, so it needs no barrier of its own.
    if constexpr (NRT > 0) {
        const uint32_t pl = nmain;
        PairMask<RT> pm;
        if constexpr (CAUSAL) {
            pm = causal_mask<RT>(int(lim.tok0 + 2 * kPageSize * pl), rtg.len, int(lim.lmax));
        } else {
            const int n0 = TAIL && 2 * pl + 1 == np ? last_len : kPageSize;
            const int n1 = 2 * pl + 1 >= np ? 0 : (TAIL && 2 * pl + 2 == np ? last_len : kPageSize);
            pm = uniform_mask<RT>(n0, n1);
        }
        dma_step<D, F16, NRT, true, false>((pl % P) * SLOT, 0, pm, lb, qB, sc, vop, rm, Lsum, O, g, f, finv);
    }
}

// Query rows of a wave's tiles in a DMA group item: tile rt of wave w covers
// rows (rt * kWaves + w) * 16 .. +16.
template <int D, int RT, bool PF>
__device__ __forceinline__ void write_partial_dma(const AttendArgs& a, const Item& it, int wave, int nrt,
                                                  const RowTargets<RT>& rtg, const float (&m)[RT],
                                                  const f4 (&L)[RT], const f4 (&O)[RT][D / 16], int g, int c,
                                                  bool f16) {
    constexpr int EPL = D / 16;
    const uint32_t (&dst)[RT] = rtg.dst;
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        if (rt >= nrt) break;
        const uint32_t row = uint32_t(rt * kWaves + wave) * kTileRows + c;
        const float lt = L[rt][0];
        const float inv = lt > 0.f ? 1.f / lt : 0.f;
        if (PF && a.out_direct && (it.flags & kItemSplit)) {   // one of the row's chunks, in f32
            if (row < it.nrows) {
                float* o = static_cast<float*>(a.ws_o) + uint64_t(dst[rt]) * D;
                #pragma unroll
                for (int e = 0; e < EPL; ++e) *reinterpret_cast<f4*>(o + 16 * e + 4 * g) = O[rt][e] * inv;
                if (g == 0) a.ws_lse[dst[rt]] = PartialLse{lt > 0.f ? m[rt] + log2f(lt) : kNegInf, 0.f};
            }
            continue;
        }
        if (PF && a.out_direct) {   // the row's only partial state is its output
            if (row < it.nrows) {
                uint8_t* o = static_cast<uint8_t*>(a.out_direct) + rtg.qoff[rt];
                #pragma unroll
                for (int e = 0; e < EPL; ++e) {
                    const f4 v = O[rt][e] * inv;
                    *reinterpret_cast<u32x2*>(o + 2 * (16 * e + 4 * g)) =
                        u32x2{pack2(v[0], v[1], f16), pack2(v[2], v[3], f16)};
                }
            }
            continue;
        }
        float mx = 0.f;
        #pragma unroll
        for (int e = 0; e < EPL; ++e)
            #pragma unroll
            for (int i = 0; i < 4; ++i) mx = fmaxf(mx, fabsf(O[rt][e][i]));
        const int k = partial_exp(rowgroup_max(mx) * inv);
        const float sc = __builtin_amdgcn_ldexpf(inv, -k);
        if (row < it.nrows) {
            uint16_t* o = static_cast<uint16_t*>(a.ws_o) + uint64_t(dst[rt]) * D;
            #pragma unroll
            for (int e = 0; e < EPL; ++e) {
                const f4 v = O[rt][e] * sc;
                *reinterpret_cast<u32x2*>(o + 16 * e + 4 * g) = u32x2{pack2(v[0], v[1], true), pack2(v[2], v[3], true)};
            }
            if (g == 0) a.ws_lse[dst[rt]] = PartialLse{lt > 0.f ? m[rt] + log2f(lt) : kNegInf, float(k)};
        }
    }
}

template <int D, bool F16, int NRT, bool PF>
__device__ __forceinline__ void dma_group_run(const AttendArgs& a, const Item& it, const uint32_t* ids,
                                              uint8_t* ring, int tid, int wave, int g, int c,
                                              const RowTargets<DmaCfg<D>::RT>& rtg, int last_len) {
    using C = DmaCfg<D>;
    constexpr int RT = C::RT, EPL = D / 16, KB = D / 32;
    u32x4 qB[RT][KB];
    RowMax<RT> rm;
    f4 L[RT];
    f4 O[RT][EPL];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        rm.m[rt] = kNegInf;
        rm.thr[rt] = kNegInf;
        L[rt] = f4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int e = 0; e < EPL; ++e) O[rt][e] = f4{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (PF) {   // prefill plans: every item is causal
        const ItemLim lim = a.item_lim[blockIdx.x];
        dma_group_loop<D, F16, NRT, false, true>(a, it, ids, ring, tid, wave, g, c, rtg, last_len, lim, qB, rm, L,
                                                 O);
    } else if (it.flags & kItemTail) {
        dma_group_loop<D, F16, NRT, true, false>(a, it, ids, ring, tid, wave, g, c, rtg, last_len, ItemLim{},
                                                 qB, rm, L, O);
    } else {
        dma_group_loop<D, F16, NRT, false, false>(a, it, ids, ring, tid, wave, g, c, rtg, last_len, ItemLim{},
                                                  qB, rm, L, O);
    }
    write_partial_dma<D, RT, PF>(a, it, wave, NRT, rtg, rm.m, L, O, g, c, F16);
}

// Item fields as wave-uniform values (they are: the item is the workgroup's),
// so loop bounds and page addressing stay in scalar registers.
__device__ __forceinline__ Item uniform_item(const Item& it) {
    Item u;
    u.page_off = __builtin_amdgcn_readfirstlane(it.page_off);
    u.npages = __builtin_amdgcn_readfirstlane(it.npages);
    u.seq_off = __builtin_amdgcn_readfirstlane(it.seq_off);
    u.row_begin = __builtin_amdgcn_readfirstlane(it.row_begin);
    u.nrows = __builtin_amdgcn_readfirstlane(it.nrows);
    u.kv_head = __builtin_amdgcn_readfirstlane(it.kv_head);
    u.flags = __builtin_amdgcn_readfirstlane(it.flags);
    u.tail_seq = __builtin_amdgcn_readfirstlane(it.tail_seq);
    return u;
}

template <int D, bool F16, bool PF>
__device__ __forceinline__ void group_item_dma(const AttendArgs& a, const Item& item, int tid, int wave, int g,
                                               int c) {
    using C = DmaCfg<D>;
    __shared__ __attribute__((aligned(1024))) uint8_t ring[C::RING];
    __shared__ uint32_t ids[PF ? kPrefillMaxPages : kGroupMaxPages];
    const Item it = uniform_item(item);
    // Row targets, the last page's length and the page ids load together.
    RowTargets<C::RT> rtg;
    dma_row_targets<D, C::RT>(a, it, wave, c, rtg);
    const int last_len = item_last_len(a, it);
    for (uint32_t i = tid; i < it.npages; i += kWaves * 64) {
        const uint32_t pg = a.pages[it.page_off + i];
        ids[i] = pg < a.page_limit ? pg : 0u;
    }
    __syncthreads();
    // Tiles of this wave that hold rows: tiles w, w+4, ... below ceil(nrows/16).
    const int ntiles = int((it.nrows + kTileRows - 1) / kTileRows);
    const int nrt = ntiles > wave ? min(C::RT, (ntiles - wave + kWaves - 1) / kWaves) : 0;
    if (nrt >= 3) dma_group_run<D, F16, C::RT, PF>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
    else if (nrt == 2) dma_group_run<D, F16, 2, PF>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
    else if (nrt == 1) dma_group_run<D, F16, 1, PF>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
    else dma_group_run<D, F16, 0, PF>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
}

// ------------------------------------------- group items, FP8 / MXFP8 KV
// Raw E4M3 pages and their scales reach LDS by direct loads into a ring of
// NPR raw pairs.  Each raw pair is then converted by the whole workgroup
// into a bf16 pair slot laid out as the 16-bit path's (swizzled rows), and
// the 16-bit pair loop's compute (dma_step) runs on those slots.  MXFP8
// elements take their E8M0 group scale in the exact power-of-two conversion;
// with an E4M3 block scale, K codes are converted exactly (the scale then
// multiplies the scores, so a large attention scale cannot amplify a
// rounding of code * scale) and V is converted exactly to f32, multiplied
// by its scale and rounded once to bf16.  Per iteration pi: wait for raw pair
// pi + 1, barrier, refill the raw slot of pair pi - 1 (converted two
// iterations ago), convert raw pair pi + 1 into bf16 slot (pi + 1) & 1,
// barrier, compute.  Head_dim 128 and 256 (64 keeps the register path).
template <int D>
struct Dma8Cfg {
    using C16 = DmaCfg<D>;
    static constexpr int RAW_PLANE = kPageSize * D;              // E4M3 bytes of one plane
    static constexpr int RAW_PAGE = 2 * RAW_PLANE;
    static constexpr int RAW_PAIR = 2 * RAW_PAGE;
    static constexpr int NPR = 4;                                // raw ring pairs
    static constexpr int RDPP = RAW_PAGE / (kWaves * 1024);      // wave loads per thread per raw page
    static constexpr int PER_PAIR = 2 * RDPP + 1;                // + the pair's scale load
    static constexpr int SCALES = 1024;                          // LDS bytes of one raw pair's scales
    static constexpr int SREC = kPageSize * (D / 32);            // MXFP8 scale bytes of one plane
    static constexpr int NCH = 4 * SREC / 16;                    // 16-byte chunks of a pair's MX scales
    static constexpr int BF_PAIR = 2 * C16::PAGE;                // bf16 pair slot
    static constexpr int RAW_BYTES = NPR * (RAW_PAIR + SCALES);
    static constexpr int LDS = RAW_BYTES + 2 * BF_PAIR;
    static constexpr int CONV = RAW_PAIR / (kWaves * 64 * 32);   // 32-element runs per thread per pair
    static_assert(RDPP >= 1 && RDPP <= 4 && CONV >= 1, "head_dim 128 or 256");
    static_assert(C16::QBYTES <= 2 * BF_PAIR, "query rows fit the bf16 slots");
    static_assert(4 * SREC <= SCALES && NCH <= 64, "scale slot");
    static_assert(NPR * PER_PAIR <= 63, "vmcnt range");
};

// One wave load of 64 x 4 bytes from gbase + voff (per lane) to lds + 4 * lane.
__device__ __forceinline__ void dma_x1(uint32_t lds, const void* gbase, uint32_t voff) {
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dword %1, %2"
                 :
                 : "s"(lds), "v"(voff), "s"(gbase)
                 : "memory", "m0");
}

// s_waitcnt vmcnt(n), n <= 63, from a run-time value.
__device__ __forceinline__ void wait_vmcnt_any(uint32_t n) {
#define DH_VMCNT_CASE(k) case k: asm volatile("s_waitcnt vmcnt(" #k ")" ::: "memory"); break;
    switch (n) {
        DH_VMCNT_CASE(0) DH_VMCNT_CASE(1) DH_VMCNT_CASE(2) DH_VMCNT_CASE(3) DH_VMCNT_CASE(4)
        DH_VMCNT_CASE(5) DH_VMCNT_CASE(6) DH_VMCNT_CASE(7) DH_VMCNT_CASE(8) DH_VMCNT_CASE(9)
        DH_VMCNT_CASE(10) DH_VMCNT_CASE(11) DH_VMCNT_CASE(12) DH_VMCNT_CASE(13) DH_VMCNT_CASE(14)
        DH_VMCNT_CASE(15) DH_VMCNT_CASE(16) DH_VMCNT_CASE(17) DH_VMCNT_CASE(18) DH_VMCNT_CASE(19)
        DH_VMCNT_CASE(20) DH_VMCNT_CASE(21) DH_VMCNT_CASE(22) DH_VMCNT_CASE(23) DH_VMCNT_CASE(24)
        DH_VMCNT_CASE(25) DH_VMCNT_CASE(26) DH_VMCNT_CASE(27) DH_VMCNT_CASE(28) DH_VMCNT_CASE(29)
        DH_VMCNT_CASE(30) DH_VMCNT_CASE(31) DH_VMCNT_CASE(32) DH_VMCNT_CASE(33) DH_VMCNT_CASE(34)
        DH_VMCNT_CASE(35) DH_VMCNT_CASE(36) DH_VMCNT_CASE(37) DH_VMCNT_CASE(38) DH_VMCNT_CASE(39)
        DH_VMCNT_CASE(40) DH_VMCNT_CASE(41) DH_VMCNT_CASE(42) DH_VMCNT_CASE(43) DH_VMCNT_CASE(44)
        DH_VMCNT_CASE(45) DH_VMCNT_CASE(46) DH_VMCNT_CASE(47) DH_VMCNT_CASE(48)
        default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); break;
    }
#undef DH_VMCNT_CASE
}

// Source offsets (per lane) of one raw pair's loads.
template <int D>
struct Dma8Src {
    uint32_t loff[Dma8Cfg<D>::RDPP];    // inside a raw page, this wave's share
    uint64_t page_stride;
    uint32_t s_rel;                     // scale load: offset inside the (page, plane) record
    uint32_t s_plane;                   // scale load: plane of this lane's chunk
    bool s_page1;                       // scale load: this lane's chunk belongs to the pair's second page
};

template <int D, uint32_t KVF>
__device__ __forceinline__ Dma8Src<D> dma8_src(const AttendArgs& a, const Item& it, int wave, int lane) {
    using C8 = Dma8Cfg<D>;
    Dma8Src<D> s;
    s.page_stride = uint64_t(2) * a.hkv * C8::RAW_PLANE;
    #pragma unroll
    for (int u = 0; u < C8::RDPP; ++u) {
        const int b = (wave * C8::RDPP + u) * 1024 + 16 * lane;
        const int plane = b / C8::RAW_PLANE, rem = b - plane * C8::RAW_PLANE;
        s.loff[u] = uint32_t((plane * a.hkv + it.kv_head) * C8::RAW_PLANE + rem);
    }
    if constexpr (KVF == KVF_MX) {
        const int k = lane % C8::NCH, pp = k / (C8::SREC / 16);
        s.s_page1 = (pp >> 1) != 0;
        s.s_plane = uint32_t(pp & 1);
        s.s_rel = uint32_t((k % (C8::SREC / 16)) * 16);
    } else {
        const int e = lane & 3;
        s.s_page1 = (e >> 1) != 0;
        s.s_plane = uint32_t(e & 1);
        s.s_rel = 0;
    }
    return s;
}

// Issues this wave's loads of pages pg0, pg1 (and their scales) into raw slot rs.
template <int D, uint32_t KVF>
__device__ __forceinline__ void dma8_pair(const AttendArgs& a, const Item& it, uint32_t pg0, uint32_t pg1,
                                          const Dma8Src<D>& src, uint32_t raw_lds, uint32_t rs, int wave) {
    using C8 = Dma8Cfg<D>;
    const uint32_t slot = raw_lds + rs * (C8::RAW_PAIR + C8::SCALES);
    #pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint8_t* base = a.kv + uint64_t(q == 0 ? pg0 : pg1) * src.page_stride;
        const uint32_t dst = slot + q * C8::RAW_PAGE + wave * C8::RDPP * 1024;
        #pragma unroll
        for (int u = 0; u < C8::RDPP; ++u) dma_x4(dst + u * 1024, base, src.loff[u]);
    }
    const uint32_t pg = src.s_page1 ? pg1 : pg0;
    const uint32_t rec = (pg * 2 + src.s_plane) * a.hkv + it.kv_head;
    if constexpr (KVF == KVF_MX)
        dma_x4(slot + C8::RAW_PAIR, a.scales, rec * uint32_t(C8::SREC) + src.s_rel);
    else
        dma_x1(slot + C8::RAW_PAIR, a.scales, rec * 4u);
}

// Converts raw slot rs into bf16 slot bs (the whole workgroup; tid < 256).
template <int D, uint32_t KVF, bool HK, bool HV>
__device__ __forceinline__ void dma8_convert(uint8_t* ring, uint32_t rs, uint32_t bs, int tid) {
    using C8 = Dma8Cfg<D>;
    using C = DmaCfg<D>;
    const uint8_t* raw = ring + rs * (C8::RAW_PAIR + C8::SCALES);
    const uint8_t* scl = raw + C8::RAW_PAIR;
    uint8_t* bf = ring + C8::RAW_BYTES + bs * C8::BF_PAIR;
    #pragma unroll
    for (int k = 0; k < C8::CONV; ++k) {
        const int o = 32 * (tid + kWaves * 64 * k);
        const int page = o / C8::RAW_PAGE, po = o - page * C8::RAW_PAGE;
        const int plane = po / C8::RAW_PLANE, pr = po - plane * C8::RAW_PLANE;
        const int row = pr / D, col0 = pr - row * D;
        const u32x4 w0 = *reinterpret_cast<const u32x4*>(raw + o);
        const u32x4 w1 = *reinterpret_cast<const u32x4*>(raw + o + 16);
        const uint32_t wd[8] = {w0[0], w0[1], w0[2], w0[3], w1[0], w1[1], w1[2], w1[3]};
        uint32_t out[16];
        if constexpr (KVF == KVF_MX) {
            const float sc = e8m0_to_float(scl[(page * 2 + plane) * C8::SREC + row * (D / 32) + col0 / 32]);
            if (plane == 0) {
                #pragma unroll
                for (int w = 0; w < 8; ++w) e4m3x4_cvt<HK>(wd[w], sc, out[2 * w], out[2 * w + 1]);
            } else {
                #pragma unroll
                for (int w = 0; w < 8; ++w) e4m3x4_cvt<HV>(wd[w], sc, out[2 * w], out[2 * w + 1]);
            }
        } else if (plane == 0) {
            // K: the codes alone (exact in bf16); the block scale multiplies
            // the scores, so the attention scale does not amplify a rounding
            // of code * scale.  (plane is wave-uniform: a wave converts 2048
            // consecutive bytes, whole planes at head_dim 128 and 256.)
            #pragma unroll
            for (int w = 0; w < 8; ++w) e4m3x4_cvt<HK>(wd[w], 1.f, out[2 * w], out[2 * w + 1]);
        } else {
            // V: code * scale in f32, rounded once to bf16 or f16 (RNE).
            const float sc = *reinterpret_cast<const float*>(scl + 4 * (page * 2 + plane));
            #pragma unroll
            for (int w = 0; w < 8; ++w) {
                const f2 lo = __builtin_amdgcn_cvt_pk_f32_fp8(wd[w], false);
                const f2 hi = __builtin_amdgcn_cvt_pk_f32_fp8(wd[w], true);
                out[2 * w] = pack2(lo[0] * sc, lo[1] * sc, HV);
                out[2 * w + 1] = pack2(hi[0] * sc, hi[1] * sc, HV);
            }
        }
        uint8_t* rowp = bf + page * C::PAGE + plane * C::PLANE + row * C::RB;
        #pragma unroll
        for (int j = 0; j < 4; ++j) {
            const int pos = (col0 / 8 + j) ^ chunk_swz<D>(row);
            *reinterpret_cast<u32x4*>(rowp + pos * 16) = u32x4{out[4 * j], out[4 * j + 1], out[4 * j + 2], out[4 * j + 3]};
        }
    }
}

template <int D, uint32_t KVF, bool F16, int NRT, bool TAIL, bool CAUSAL, bool PF16 = F16>
__device__ __forceinline__ void dma8_group_loop(const AttendArgs& a, const Item& it, const uint32_t* ids,
                                                uint8_t* ring, int tid, int wave, int g, int c,
                                                const RowTargets<DmaCfg<D>::RT>& rtg, int last_len,
                                                const ItemLim& lim,
                                                u32x4 (&qB)[DmaCfg<D>::RT][D / 32],
                                                RowMax<DmaCfg<D>::RT>& rm, f4 (&Lsum)[DmaCfg<D>::RT],
                                                f4 (&O)[DmaCfg<D>::RT][D / 16]) {
    using C = DmaCfg<D>;
    using C8 = Dma8Cfg<D>;
    constexpr uint32_t P = C8::NPR;
    constexpr int RT = C::RT, KB = D / 32;
    const uint32_t np = it.npages;
    const uint32_t npairs = (np + 1) >> 1;
    const int lane = tid & 63;
    const Dma8Src<D> src = dma8_src<D, KVF>(a, it, wave, lane);
    const uint32_t raw_lds = __builtin_amdgcn_readfirstlane(uint32_t(reinterpret_cast<uintptr_t>(ring)));
    const uint32_t bf_lds = raw_lds + C8::RAW_BYTES;
    const LdsBases<D> lb = lds_bases<D>(bf_lds, g, c);
    const float f = a.scale_log2;   // > 0 (a negative scale is in q_sign)
    const float finv = 1.f / f;
    const uint32_t qsign = a.q_sign;
    // FP8 block scale: K is staged unscaled and the pages' K scales (in the
    // raw slot of the pair being finished, records [page][K|V]) multiply
    // the scores.
    constexpr bool KS = KVF == KVF_FP8;
    auto k_scales = [&](uint32_t rs, float& k0, float& k1) {
        const float* sk = reinterpret_cast<const float*>(ring + rs * (C8::RAW_PAIR + C8::SCALES) + C8::RAW_PAIR);
        k0 = sk[0];
        k1 = sk[2];
    };
    auto page_id = [&](uint32_t i) { return __builtin_amdgcn_readfirstlane(ids[i < np ? i : np - 1]); };
    // Every compiler-issued load (row targets, page ids) has landed before
    // the ring loads start, so no compiler-inserted wait drains the ring.
    __builtin_amdgcn_s_waitcnt(0x0070);
    compiler_fence();
    const uint32_t q_lds = bf_lds + wave * (RT * KB * 1024);
    #pragma unroll
    for (int rt = 0; rt < NRT; ++rt) {
        #pragma unroll
        for (int kb = 0; kb < KB; ++kb)
            dma_x4(q_lds + (rt * KB + kb) * 1024, static_cast<const uint8_t*>(a.q), rtg.qoff[rt] + kb * 64 + 16 * g);
    }
    const uint32_t pro = min(P - 1, npairs);
    #pragma unroll 1
    for (uint32_t q = 0; q < pro; ++q) dma8_pair<D, KVF>(a, it, page_id(2 * q), page_id(2 * q + 1), src, raw_lds, q, wave);
    wait_vmcnt_any(pro * C8::PER_PAIR);   // loads land in issue order: the query rows are in
    if constexpr (NRT > 0) {
        const uint8_t* qw = ring + C8::RAW_BYTES + wave * (RT * KB * 1024) + 16 * lane;
        #pragma unroll
        for (int rt = 0; rt < NRT; ++rt) {
            const bool valid = uint32_t(rt * kWaves + wave) * kTileRows + c < it.nrows;
            #pragma unroll
            for (int kb = 0; kb < KB; ++kb) {
                const u32x4 v = *reinterpret_cast<const u32x4*>(qw + (rt * KB + kb) * 1024) ^ qsign;
                qB[rt][kb] = valid ? v : u32x4{0u, 0u, 0u, 0u};
            }
        }
    }
    wait_vmcnt_any((pro - 1) * C8::PER_PAIR);   // raw pair 0 has landed
    block_barrier();                             // query rows read; raw pair 0 visible
    dma8_convert<D, KVF, F16, PF16>(ring, 0, 0, tid);
    block_barrier();
    f4 sc[RT][2];
    u32x4 vop[D / 16];
    if constexpr (NRT > 0) dma_scores<D, F16, NRT>(0, lb, qB, sc);
    uint32_t ps = 0, psn = 1;   // raw slots of pairs pi, pi + 1
    uint32_t nid0 = page_id(2 * (P - 1)), nid1 = page_id(2 * (P - 1) + 1);
    // Step pi: raw pair pi + 1 is converted into bf16 slot (pi + 1) & 1 while
    // pair pi is finished from slot pi & 1; steps are unrolled by two so the
    // bf16 slots are immediate offsets.  The last pair runs apart (partial
    // pages, nothing to score next, nothing to convert).
    const uint32_t nmain = npairs - 1;
    #pragma unroll 1
    for (uint32_t p0 = 0; p0 < nmain; p0 += 2) {
        static_for<0, 2>([&](auto J) {
            constexpr uint32_t j = decltype(J)::value;
            const uint32_t pi = p0 + j;
            if (pi >= nmain) return;
            // raw pair pi + 1 has landed: an immediate count while pairs
            // are still being issued (a runtime count is a tree of branches)
            if (pi + P - 1 <= npairs) wait_vmcnt_const<(P - 3) * C8::PER_PAIR>();
            else wait_vmcnt_any((npairs - pi - 2) * C8::PER_PAIR);
            block_barrier();
            if (pi + P - 1 < npairs) dma8_pair<D, KVF>(a, it, nid0, nid1, src, raw_lds, ps == 0 ? P - 1 : ps - 1, wave);
            nid0 = page_id(2 * (pi + P));
            nid1 = page_id(2 * (pi + P) + 1);
            dma8_convert<D, KVF, F16, PF16>(ring, psn, (j + 1) & 1, tid);
            block_barrier();
            if constexpr (NRT > 0) {
                float ks0 = 1.f, ks1 = 1.f;
                if constexpr (KS) k_scales(ps, ks0, ks1);
                const int t = CAUSAL ? int(lim.tok0 + 2 * kPageSize * pi) : 0;
                if (CAUSAL && t + 2 * kPageSize > int(lim.lmin))
                    dma_step<D, F16, NRT, true, true, KS, PF16>(j * C8::BF_PAIR, ((j + 1) & 1) * C8::BF_PAIR,
                                                                  causal_mask<RT>(t, rtg.len, int(lim.lmax)), lb, qB,
                                                                  sc, vop, rm, Lsum, O, g, f, finv, ks0, ks1);
                else
                    dma_step<D, F16, NRT, false, true, KS, PF16>(j * C8::BF_PAIR, ((j + 1) & 1) * C8::BF_PAIR,
                                                                   uniform_mask<RT>(kPageSize, kPageSize), lb, qB,
                                                                   sc, vop, rm, Lsum, O, g, f, finv, ks0, ks1);
            }
            ps = psn;
            psn = psn + 1 == P ? 0 : psn + 1;
        });
    }
    // The last pair was converted and made visible by the previous step (or
    // the prologue); every raw load has landed (the last wait was vmcnt(0)).
    if constexpr (NRT > 0) {
        const uint32_t pl = nmain;
        PairMask<RT> pm;
        if constexpr (CAUSAL) {
            pm = causal_mask<RT>(int(lim.tok0 + 2 * kPageSize * pl), rtg.len, int(lim.lmax));
        } else {
            const int n0 = TAIL && 2 * pl + 1 == np ? last_len : kPageSize;
            const int n1 = 2 * pl + 1 >= np ? 0 : (TAIL && 2 * pl + 2 == np ? last_len : kPageSize);
            pm = uniform_mask<RT>(n0, n1);
        }
        float ks0 = 1.f, ks1 = 1.f;
        if constexpr (KS) k_scales(ps, ks0, ks1);
        dma_step<D, F16, NRT, true, false, KS, PF16>((pl & 1) * C8::BF_PAIR, 0, pm, lb, qB, sc, vop, rm, Lsum, O,
                                                      g, f, finv, ks0, ks1);
    }
}

template <int D, uint32_t KVF, bool F16, int NRT, bool PF, bool PF16 = F16>
__device__ __forceinline__ void dma8_group_run(const AttendArgs& a, const Item& it, const uint32_t* ids,
                                               uint8_t* ring, int tid, int wave, int g, int c,
                                               const RowTargets<DmaCfg<D>::RT>& rtg, int last_len) {
    using C = DmaCfg<D>;
    constexpr int RT = C::RT, EPL = D / 16, KB = D / 32;
    u32x4 qB[RT][KB];
    RowMax<RT> rm;
    f4 L[RT];
    f4 O[RT][EPL];
    #pragma unroll
    for (int rt = 0; rt < RT; ++rt) {
        rm.m[rt] = kNegInf;
        rm.thr[rt] = kNegInf;
        L[rt] = f4{0.f, 0.f, 0.f, 0.f};
        #pragma unroll
        for (int e = 0; e < EPL; ++e) O[rt][e] = f4{0.f, 0.f, 0.f, 0.f};
    }
    if constexpr (PF) {   // prefill plans: every item is causal
        const ItemLim lim = a.item_lim[blockIdx.x];
        dma8_group_loop<D, KVF, F16, NRT, false, true, PF16>(a, it, ids, ring, tid, wave, g, c, rtg, last_len, lim, qB, rm,
                                                  L, O);
    } else if (it.flags & kItemTail) {
        dma8_group_loop<D, KVF, F16, NRT, true, false, PF16>(a, it, ids, ring, tid, wave, g, c, rtg, last_len, ItemLim{},
                                                  qB, rm, L, O);
    } else {
        dma8_group_loop<D, KVF, F16, NRT, false, false, PF16>(a, it, ids, ring, tid, wave, g, c, rtg, last_len, ItemLim{},
                                                   qB, rm, L, O);
    }
    write_partial_dma<D, RT, PF>(a, it, wave, NRT, rtg, rm.m, L, O, g, c, F16);
}

// Whether the V values of KV head h in page `page` fit f16: FP8's
// per-(page, head) scale at most 146 (448 x 146 < 65504), MXFP8's E8M0
// exponents of the page's 16 tokens x D/32 groups at most 134 (448 x 2^7).
// Smaller values only lose bits below f16's least subnormal, far under the
// output tolerance.
template <int D, uint32_t KVF>
__device__ __forceinline__ bool v_fits_f16(const AttendArgs& a, uint32_t page, uint32_t h) {
    const uint8_t* sc = static_cast<const uint8_t*>(a.scales);
    if constexpr (KVF == KVF_FP8) {
        const uint64_t rec = uint64_t(2) * a.hkv * 4;
        const float s = *reinterpret_cast<const float*>(sc + page * rec + (a.hkv + h) * 4);
        return s <= 146.f;   // NaN: false
    } else {
        constexpr int G = D / 32;
        const uint64_t rec = uint64_t(2) * a.hkv * kPageSize * G;
        const u32x4* p = reinterpret_cast<const u32x4*>(sc + page * rec + uint64_t(a.hkv + h) * kPageSize * G);
        uint32_t big = 0;
        #pragma unroll
        for (int j = 0; j < G; ++j) {
            const u32x4 w = p[j];
            #pragma unroll
            for (int i = 0; i < 4; ++i)
                #pragma unroll
                for (int b = 0; b < 32; b += 8) big |= ((w[i] >> b) & 0xFFu) > 134u ? 1u : 0u;
        }
        return big == 0;
    }
}

// 8-bit group item.  With bf16 queries the probabilities and V go into
// the PV products as f16 when every V value of the item's pages fits f16
// (checked on the scales with the page ids): bf16's 8-bit significand on
// the probabilities was the largest error term at C5's shape (1.2e-2 beyond
// the output rounding in an emulation of this arithmetic, 4e-3 with f16
// probabilities in the shared-prefix items).  The scores stay bf16 x bf16.
template <int D, uint32_t KVF, bool F16, bool PF>
__device__ __forceinline__ void group_item_dma8(const AttendArgs& a, const Item& item, int tid, int wave, int g,
                                                int c) {
    using C = DmaCfg<D>;
    using C8 = Dma8Cfg<D>;
    __shared__ __attribute__((aligned(1024))) uint8_t ring[C8::LDS];
    __shared__ uint32_t ids[PF ? kPrefillMaxPages : kGroupMaxPages];
    constexpr bool V16 = !F16 && !PF;   // probabilities may go f16
    const Item it = uniform_item(item);
    RowTargets<C::RT> rtg;
    dma_row_targets<D, C::RT>(a, it, wave, c, rtg);
    const int last_len = item_last_len(a, it);
    int big = 0;
    for (uint32_t i = tid; i < it.npages; i += kWaves * 64) {
        const uint32_t pg = a.pages[it.page_off + i];
        const uint32_t id = pg < a.page_limit ? pg : 0u;
        ids[i] = id;
        if constexpr (V16) big |= v_fits_f16<D, KVF>(a, id, it.kv_head) ? 0 : 1;
    }
    bool pf16 = false;
    if constexpr (V16) pf16 = __syncthreads_or(big) == 0;
    else __syncthreads();
    const int ntiles = int((it.nrows + kTileRows - 1) / kTileRows);
    const int nrt = ntiles > wave ? min(C::RT, (ntiles - wave + kWaves - 1) / kWaves) : 0;
    auto run = [&](auto pfI) {
        constexpr bool P16 = decltype(pfI)::value != 0;
        if (nrt >= 2) dma8_group_run<D, KVF, F16, C::RT, PF, P16>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
        else if (nrt == 1) dma8_group_run<D, KVF, F16, 1, PF, P16>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
        else dma8_group_run<D, KVF, F16, 0, PF, P16>(a, it, ids, ring, tid, wave, g, c, rtg, last_len);
    };
    if constexpr (V16) {
        if (pf16) run(Idx<1>{});
        else run(Idx<0>{});
    } else {
        run(Idx<F16 ? 1 : 0>{});
    }
}

// ---------------------------------------------------------------- attend32
// f32 q and f32 KV (wave items only): v_mfma_f32_16x16x4_f32, one page per
// step, 16 rows per wave.
//   S^T: A = K[token c][g*D/4 + kb], B = Q[row c][g*D/4 + kb], kb < D/4.
//   O^T: for token group i: A = V[4g+i][c*EPL + e], B = P[row c][4g+i].
// One wave item of attend32_kernel.
template <int D>
__device__ __forceinline__ void attend32_item(const AttendArgs& a, const Item& it, int lane, int g, int c) {
    constexpr int KQ = D / 4;
    constexpr int EPL = D / 16;

    float qv[KQ];
    uint32_t dst[1] = {0u};
    if (uint32_t(c) < it.nrows) {
        uint32_t seq, slot, qh;
        row_target(a, it, c, seq, slot, qh);
        dst[0] = slot * a.hq + qh;
        const float* qp = reinterpret_cast<const float*>(a.q) + (uint64_t(seq) * a.hq + qh) * D + g * KQ;
        load_dwords<KQ>(reinterpret_cast<uint32_t*>(qv), qp);
        #pragma unroll
        for (int k = 0; k < KQ; ++k) qv[k] = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, qv[k]) ^ a.q_sign);
    } else {
        #pragma unroll
        for (int k = 0; k < KQ; ++k) qv[k] = 0.f;
    }

    float m[1] = {kNegInf}, l[1] = {0.f};
    f4 O[1][EPL];
    #pragma unroll
    for (int e = 0; e < EPL; ++e) O[0][e] = f4{0.f, 0.f, 0.f, 0.f};

    const int last_len = item_last_len(a, it);
    const uint32_t* pages = a.pages + it.page_off;
    const uint32_t np = it.npages;
    const uint64_t plane_bytes = uint64_t(kPageSize) * D * 4;

    // DEPTH pages in flight: buffer p % DEPTH holds page p; once page p is
    // consumed its registers take page p + DEPTH.  Two at head_dim 64 (32
    // registers a page); one above (64 or 128), where a second page would
    // cost occupancy.
    constexpr int DEPTH = D <= 64 ? 2 : 1;
    float kb[DEPTH][KQ];
    float vb[DEPTH][4][EPL];
    bool bad = false;
    auto load = [&](int buf, uint32_t pi) {
        const uint32_t pg = pages[pi];
        bad |= pg >= a.page_limit;
        const uint8_t* kp = a.kv + plane_offset(pg < a.page_limit ? pg : 0u, 0, it.kv_head, a.hkv, D, 4);
        const uint8_t* vp = kp + uint64_t(a.hkv) * plane_bytes;
        load_dwords<KQ>(reinterpret_cast<uint32_t*>(kb[buf]), kp + (c * D + g * KQ) * 4);
        #pragma unroll
        for (int i = 0; i < 4; ++i)
            load_dwords<EPL>(reinterpret_cast<uint32_t*>(vb[buf][i]), vp + ((4 * g + i) * D + c * EPL) * 4);
    };
    #pragma unroll
    for (int d = 0; d < DEPTH; ++d)
        if (uint32_t(d) < np) load(d, d);
    #pragma unroll 1
    for (uint32_t p0 = 0; p0 < np; p0 += DEPTH) {
        static_for<0, DEPTH>([&](auto J) {
            constexpr int j = decltype(J)::value;
            const uint32_t pi = p0 + j;
            if (pi >= np) return;
            const int n0 = page_tokens(it, pi, last_len);
            f4 s = {0.f, 0.f, 0.f, 0.f};
            #pragma unroll
            for (int k = 0; k < KQ; ++k) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kb[j][k], qv[k], s, 0, 0, 0);
            float x[4];
            float mx = kNegInf;
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = (4 * g + i < n0) ? s[i] * a.scale_log2 : kNegInf;
                mx = fmaxf(mx, x[i]);
            }
            mx = rowgroup_max(mx);
            const float mnew = fmaxf(m[0], mx);
            const float muse = (mnew == kNegInf) ? 0.f : mnew;
            const float alpha = fast_exp2(m[0] - muse);
            m[0] = mnew;
            float ps = 0.f;
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                x[i] = fast_exp2(x[i] - muse);
                ps += x[i];
            }
            l[0] = l[0] * alpha + ps;
            #pragma unroll
            for (int e = 0; e < EPL; ++e) O[0][e] *= alpha;
            #pragma unroll
            for (int i = 0; i < 4; ++i) {
                // V past the page's valid tokens: zero (its weight is zero,
                // garbage there must not reach O).
                const bool ok = 4 * g + i < n0;
                #pragma unroll
                for (int e = 0; e < EPL; ++e)
                    O[0][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(ok ? vb[j][i][e] : 0.f, x[i], O[0][e], 0, 0, 0);
            }
            if (pi + DEPTH < np) load(j, pi + DEPTH);
        });
    }
    if (__ballot(bad) && a.seq_bad && lane == 0) a.seq_bad[it.tail_seq] = 1u;
    write_wave_partial<D, 1, false, true>(a, it, 0, 1, dst, m, l, O, g, c);
}

}  // namespace
}  // namespace dh
