// Kernels of dh_decode_csr, decode from page tables in device memory: the
// common prefixes, the planning and the attention, and their launchers.  The
// items the attention runs are in attend_device.hpp.
// A file, and so a code object, of their own: beside the plan path's kernels
// they moved those in memory, and with the same machine code a 64-leaf bf16
// tree took 24.2 us a step for 24.0, 8 trees of 8 leaves at head_dim 256 31.15
// for 30.9.
#include "attend_device.hpp"

namespace dh {
namespace {

// The kernel's arguments (the first and only parameter), read anew from the
// kernel argument segment through a pointer the compiler cannot see through:
// neither they nor anything derived from them is held in registers up to the
// call.
__device__ __forceinline__ const AttendArgs& fresh_args() {
    auto p = __builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const AttendArgs*)p;
}

// One unit of a CSR call: a group item, or past those ng four wave items.
template <int D, uint32_t KVF, bool F16>
__device__ __forceinline__ void csr_unit16(const AttendArgs& a, uint32_t unit, uint32_t ng, int tid) {
    const int lane = tid & 63, g = lane >> 4, c = lane & 15;
    // Wave index as a wave-uniform (scalar) value: page-list reads then go
    // through the scalar cache and never wait on the vector loads in flight.
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (unit < ng) {
        const Item it = a.items[unit];
        if constexpr ((KVF == KVF_FP8 || KVF == KVF_MX) && D == 64) group_item<D, KVF, F16>(a, it, tid, wave, g, c);
        else if constexpr (KVF == KVF_FP8 || KVF == KVF_MX) group_item_dma8<D, KVF, F16, false>(a, it, tid, wave, g, c);
        else group_item_dma<D, F16, false>(a, it, tid, wave, g, c);
    } else {
        const uint32_t idx = wave_item_index<true>(a, unit, wave, ng);
        if (idx < wave_item_end<true>(a)) {
            const Item it = csr_wave_item(a, idx, ng);
            if (it.npages) wave_item<D, KVF, F16>(a, it, g, c);
        }
    }
}

// The attention kernel of dh_decode_csr, whose unit count only the device
// knows.  Workgroup b of csr_grid takes unit b and then, where the call has
// more units than that, every csr_grid-th one.  One workgroup per unit the
// workspace could hold launched 10 000 mostly empty ones for a 64-leaf f16
// tree over 8 192 tokens, each waiting for 66 KiB of LDS to find that it had
// nothing to do: 47.8 us a call, 43.2 with the bounded grid.
// The first unit stands before the loop, in code of its own: a single loop
// body, its arguments held across the rounds, spilled 25-63 scalar registers
// into VGPR lanes and slowed most calls (48 ragged bf16 sequences: 246.7 ->
// 248.9 us; 96 f32 ones: 239.7 -> 244.4).  The loop reads its arguments and
// the thread index anew in each round (fresh_args) for the same reason.  Only
// group items use LDS, and they come first: no barrier stands between others.
template <int D, uint32_t KVF, bool F16>
__global__ __launch_bounds__(256, D >= 256 ? 1 : 2) void csr_attend16_kernel(AttendArgs a) {
    const int tid0 = threadIdx.x;
    const uint32_t first = blockIdx.x, next = first + a.csr_grid;
    const uint32_t ng = group_item_count<true>(a);
    const uint32_t end = ng + (wave_item_end<true>(a) + kWaves - 1) / kWaves;
    csr_unit16<D, KVF, F16>(a, first, ng, tid0);
    #pragma unroll 1
    for (uint32_t unit = next; unit < end; unit += fresh_args().csr_grid) {
        if (unit < ng) __syncthreads();   // every wave is done with the last group item's LDS
        int tid = tid0;
        asm volatile("" : "+v"(tid));
        csr_unit16<D, KVF, F16>(fresh_args(), unit, ng, tid);
    }
}

// As csr_unit16 and csr_attend16_kernel (f32: wave items only, no LDS).
template <int D>
__device__ __forceinline__ void csr_unit32(const AttendArgs& a, uint32_t unit, int tid) {
    const int lane = tid & 63, g = lane >> 4, c = lane & 15;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t idx = wave_item_index<true>(a, unit, wave, group_item_count<true>(a));
    if (idx < wave_item_end<true>(a)) {
        const Item it = csr_wave_item(a, idx, 0);
        if (it.npages) attend32_item<D>(a, it, lane, g, c);
    }
}

template <int D>
__global__ __launch_bounds__(256) void csr_attend32_kernel(AttendArgs a) {
    const int tid0 = threadIdx.x;
    const uint32_t first = blockIdx.x, next = first + a.csr_grid;
    const uint32_t end = (wave_item_end<true>(a) + kWaves - 1) / kWaves;
    csr_unit32<D>(a, first, tid0);
    #pragma unroll 1
    for (uint32_t unit = next; unit < end; unit += fresh_args().csr_grid) {
        int tid = tid0;
        asm volatile("" : "+v"(tid));
        csr_unit32<D>(fresh_args(), unit, tid);
    }
}

// ------------------------------------------------- decode from device CSR
// The CSR planning kernel runs as one workgroup of NT threads: one wave for
// batches of at most 64 sequences (one sequence a lane, no barriers between
// its passes), one wave per SIMD (256 threads) beyond.  Each thread keeps
// the page counts of its first csr_reg_seqs(NT) sequences in registers
// across the passes (the small variant's code stays short: it runs on a CU
// whose instruction cache has not seen it).
constexpr uint32_t kCsrSmallThreads = 64, kCsrThreads = 256;
constexpr uint32_t csr_reg_seqs(uint32_t nt) { return nt == kCsrSmallThreads ? 1u : 2u; }

// Inclusive scan over the wave (lane i: the sum, or minimum, of lanes
// 0..i): row shifts by 1, 2, 4, 8 within each 16-lane row, then the last
// lane of row 0 / 2 into rows 1 / 3 (row_bcast:15) and of row 1 into rows
// 2 and 3 (row_bcast:31).  A lane whose source is outside its row, or whose
// row is masked off, takes the identity.  Every lane must be active.
template <bool MIN>
__device__ __forceinline__ uint32_t wave_scan_dpp(uint32_t x) {
    const int id = MIN ? -1 : 0;
    auto op = [](uint32_t u, int v) { return MIN ? min(u, uint32_t(v)) : u + uint32_t(v); };
    x = op(x, __builtin_amdgcn_update_dpp(id, int(x), 0x111, 0xf, 0xf, false));   // row_shr:1
    x = op(x, __builtin_amdgcn_update_dpp(id, int(x), 0x112, 0xf, 0xf, false));   // row_shr:2
    x = op(x, __builtin_amdgcn_update_dpp(id, int(x), 0x114, 0xf, 0xf, false));   // row_shr:4
    x = op(x, __builtin_amdgcn_update_dpp(id, int(x), 0x118, 0xf, 0xf, false));   // row_shr:8
    x = op(x, __builtin_amdgcn_update_dpp(id, int(x), 0x142, 0xa, 0xf, false));   // row_bcast:15
    x = op(x, __builtin_amdgcn_update_dpp(id, int(x), 0x143, 0xc, 0xf, false));   // row_bcast:31
    return x;
}

// Inclusive prefix sums of x and y over the workgroup; tx / ty receive the
// totals.  lds: 2 * NT / 64 words.
template <uint32_t NT>
__device__ __forceinline__ void block_incl_scan2(uint32_t& x, uint32_t& y, uint32_t* lds, uint32_t& tx,
                                                 uint32_t& ty) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    x = wave_scan_dpp<false>(x);
    y = wave_scan_dpp<false>(y);
    if constexpr (NT == 64) {
        tx = __builtin_amdgcn_readlane(x, 63);
        ty = __builtin_amdgcn_readlane(y, 63);
    } else {
        constexpr int NW = NT / 64;
        if (lane == 63) {
            lds[wave] = x;
            lds[NW + wave] = y;
        }
        __syncthreads();
        uint32_t bx = 0, by = 0;
        #pragma unroll
        for (int w = 0; w < NW; ++w) {
            const uint32_t a = lds[w], b = lds[NW + w];
            bx += w < wave ? a : 0u;
            by += w < wave ? b : 0u;
            tx = w == 0 ? a : tx + a;
            ty = w == 0 ? b : ty + b;
        }
        x += bx;
        y += by;
        __syncthreads();
    }
}

// Workgroup reduction of K values per thread (MIN: minima, else sums);
// every thread receives the results.  lds: NT / 64 * K words.
// Only the values whose bit is set in `active` (uniform) are reduced.
template <uint32_t NT, bool MIN, uint32_t K>
__device__ __forceinline__ void block_reduce(uint32_t (&v)[K], uint32_t* lds, uint64_t active = ~uint64_t(0)) {
    #pragma unroll
    for (uint32_t i = 0; i < K; ++i)
        if ((active >> i) & 1u) v[i] = __builtin_amdgcn_readlane(wave_scan_dpp<MIN>(v[i]), 63);
    if constexpr (NT > 64) {
        constexpr uint32_t NW = NT / 64;
        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        if (lane == 0) {
            #pragma unroll
            for (uint32_t i = 0; i < K; ++i)
                if ((active >> i) & 1u) lds[wave * K + i] = v[i];
        }
        __syncthreads();
        #pragma unroll
        for (uint32_t i = 0; i < K; ++i) {
            if (!((active >> i) & 1u)) continue;
            uint32_t s = lds[i];
            #pragma unroll
            for (uint32_t w = 1; w < NW; ++w) s = MIN ? min(s, lds[w * K + i]) : s + lds[w * K + i];
            v[i] = s;
        }
        __syncthreads();
    }
}

// Chunk sizes (pages) a CSR call weighs: thirteen fixed ones and the size
// that gives one wave per wave slot.  An item costs kCsrStartPairs plus its
// page pairs (the planner's cost model for wave items).
constexpr uint32_t kCsrFixedCandidates = 13, kCsrStartPairs = 3, kCsrMaxStates = 64;

__device__ __forceinline__ uint32_t csr_candidate(uint32_t i) {
    switch (i) {
    case 0: return 1u;
    case 1: return 2u;
    case 2: return 4u;
    case 3: return 8u;
    case 4: return 16u;
    case 5: return 32u;
    case 6: return 48u;
    case 7: return 64u;
    case 8: return 96u;
    case 9: return 128u;
    case 10: return 160u;
    case 11: return 192u;
    default: return 256u;
    }
}

__device__ __forceinline__ uint32_t csr_cost(uint32_t pages) { return kCsrStartPairs + (pages + 1) / 2; }

// Common prefix of adjacent sequences (CSR cascade): one wave per (boundary
// b, slice s), b = 1 .. batch - 1, grid-strided.  The boundary's cap is one
// page short of the shorter sequence (each sequence keeps its last page,
// which alone may be partial); slice s covers positions s * kCsrLcpSlice ..
// of it, read 64 ids a load, every load of the slice issued before the
// first compare.  A sequence whose indptr entries are negative or decreasing
// shares nothing.
__global__ __launch_bounds__(256) void csr_lcp_kernel(const int32_t* indptr, const int32_t* indices,
                                                      uint32_t batch, uint32_t page_limit, uint32_t* lcp) {
    constexpr uint32_t U = kCsrLcpSlice / 64;
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t nw = gridDim.x * kWaves, total = (batch - 1) * kCsrLcpSlices;
    for (uint32_t w = blockIdx.x * kWaves + (threadIdx.x >> 6); w < total; w += nw) {
        const uint32_t b = 1 + w / kCsrLcpSlices, s = w % kCsrLcpSlices;
        const int32_t a0 = __builtin_amdgcn_readfirstlane(indptr[b - 1]);
        const int32_t a1 = __builtin_amdgcn_readfirstlane(indptr[b]);
        const int32_t b1 = __builtin_amdgcn_readfirstlane(indptr[b + 1]);
        uint32_t cap = 0;
        if (a0 >= 0 && a1 >= a0 && b1 >= a1) {
            const uint32_t m = min(uint32_t(a1 - a0), uint32_t(b1 - a1));
            cap = m ? min(m - 1, DH_MAX_SEQ_LEN / kPageSize - 1) : 0u;
        }
        const uint32_t lo = s * kCsrLcpSlice, hi = min(lo + kCsrLcpSlice, cap);
        uint32_t first = cap, bad = 0xFFFFu;
        if (lo < hi) {
            int32_t x[U], y[U];
            #pragma unroll
            for (uint32_t j = 0; j < U; ++j) {
                const uint32_t pos = lo + 64 * j + lane;
                x[j] = pos < hi ? indices[uint32_t(a0) + pos] : 0;
                y[j] = pos < hi ? indices[uint32_t(a1) + pos] : 0;
            }
            #pragma unroll
            for (int j = int(U) - 1; j >= 0; --j) {   // the lowest sub-block's positions win
                const uint32_t pos = lo + 64 * uint32_t(j) + lane;
                const uint64_t ne = __ballot(pos < hi && x[j] != y[j]);
                const uint64_t bd = __ballot(pos < hi && x[j] == y[j] && uint32_t(x[j]) >= page_limit);
                if (ne) first = lo + 64 * uint32_t(j) + uint32_t(__builtin_ctzll(ne));
                if (bd) bad = lo + 64 * uint32_t(j) + uint32_t(__builtin_ctzll(bd));
            }
            if (bad >= first) bad = 0xFFFFu;
        }
        if (lane == 0) lcp[b * kCsrLcpSlices + s] = first | (bad << 16);
    }
}

// Inclusive max-scan of x over the workgroup in thread order; *tot receives
// the maximum of all.  lds: NT / 64 words.
template <uint32_t NT>
__device__ __forceinline__ uint32_t block_max_scan(uint32_t x, uint32_t* lds, uint32_t& tot) {
    x = ~wave_scan_dpp<true>(~x);
    if constexpr (NT == 64) {
        tot = __builtin_amdgcn_readlane(x, 63);
        return x;
    } else {
        constexpr uint32_t NW = NT / 64;
        const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
        if (lane == 63) lds[wave] = x;
        __syncthreads();
        uint32_t before = 0;
        tot = 0;
        #pragma unroll
        for (uint32_t w = 0; w < NW; ++w) {
            const uint32_t v = lds[w];
            before = w < wave ? max(before, v) : before;
            tot = max(tot, v);
        }
        __syncthreads();
        return max(x, before);
    }
}

// The cascade of a CSR call (LDS): per sequence b (and boundary b, between
// sequences b - 1 and b) and per node.  A node is a run of consecutive
// sequences b0 .. b0 + cnt - 1 and the pages [pd, len) they share: their
// common prefix is at least len pages and their parent node's is pd.  Nodes
// nest as the shared prefixes of a fork tree do (the parent's run holds the
// child's).  Node kinds: group items (kind 1, rows over 64, or over 16 with
// more than 16 pages) or wave items of 16 rows (kind 0, chunks of
// kCsrWaveChunk pages), as the host planner treats shared segments.
constexpr uint32_t kCsrMaxLevels = 4, kCsrMaxNodes = 512, kCsrWaveChunk = 32, kCsrNoDepth = 0xFFFFFFFFu;
struct CsrCascade {
    uint32_t lcp[kCsrCascadeMaxBatch];     // common prefix of b - 1 and b (pages)
    uint32_t bad[kCsrCascadeMaxBatch];     // first shared id outside the pool there (0xFFFF: none)
    uint32_t pd[kCsrCascadeMaxBatch];      // depth of the deepest node holding b - 1 and b (kCsrNoDepth: none)
    uint32_t head[kCsrCascadeMaxBatch];    // run head of b at the current level
    uint32_t tmp[kCsrCascadeMaxBatch];     // scan scratch, later b's first slot
    uint32_t acc[kCsrCascadeMaxBatch];     // at a head: members | 1 << 31 if poisoned
    uint32_t mn[kCsrCascadeMaxBatch];      // at a head: shortest common prefix of its run
    uint32_t skip[kCsrCascadeMaxBatch];    // skip word of b (AttendArgs::csr_skip)
    uint32_t ip[kCsrCascadeMaxBatch];      // indptr[b]
    uint32_t ip_end;                       // indptr[batch]
    uint32_t lv[kCsrMaxLevels][kCsrCascadeMaxBatch];   // node id + 1 of b at a level | slot offset << 16
    uint32_t b0[kCsrMaxNodes], cnt[kCsrMaxNodes], npd[kCsrMaxNodes], len[kCsrMaxNodes];
    uint32_t gc[kCsrMaxNodes], kind[kCsrMaxNodes], item0[kCsrMaxNodes], ss0[kCsrMaxNodes];
    uint32_t nn;
};

// The cascade pass of the CSR planning kernel: nodes level by level from the
// adjacent common prefixes.  At each level a boundary is internal when its
// common prefix reaches kCsrMinShared pages past the depth of the deepest
// node holding both its sequences; maximal runs of internal boundaries are
// the level's nodes, each sharing down to the shortest prefix of its run.
// Group items take chunks of `gchunk` pages: the smallest power of two from
// 8 to 256 whose group items number at most 256 (one per CU), else 256.  A
// node whose shared pages hold a page id outside the pool poisons its
// members (s_bad[b] = 1).  When the items exceed gcap, or the slots leave
// fewer than one per sequence for the rest, nothing is grouped.  Writes the
// skip words (c.skip, p.skip), c.lv and the node records; returns the group
// items, *n_wave the nodes' wave items, *gslots the slots of node chunks.
// The nodes' share of the chip for the chunk choice of the sequences' own
// pages: wave slots they hold, their cost (page pairs plus kCsrStartPairs
// per item, times the waves of an item) and their largest item's cost.
struct CsrNodeLoad {
    uint32_t waves, cost, max_item;
};

template <uint32_t NT>
__device__ uint32_t csr_cascade(const CsrPlanArgs& p, CsrCascade& c, uint32_t* s_bad, uint32_t* red,
                                uint32_t& n_wave, uint32_t& gslots, uint32_t& gchunk, CsrNodeLoad& load) {
    const uint32_t B = p.batch, tid = threadIdx.x;
    // Every slice of a boundary loads at once (one memory round trip), and
    // indptr[b] goes to LDS for the items' page offsets.
    for (uint32_t b = tid; b < B; b += NT) {
        uint32_t mn = 0, bd = 0xFFFFu, v[kCsrLcpSlices];
        c.ip[b] = uint32_t(p.indptr[b]);
        #pragma unroll
        for (uint32_t s = 0; s < kCsrLcpSlices; ++s) v[s] = b > 0 ? p.lcp[b * kCsrLcpSlices + s] : 0u;
        if (b > 0) {
            mn = 0xFFFFu;
            #pragma unroll
            for (uint32_t s = 0; s < kCsrLcpSlices; ++s) {
                mn = min(mn, v[s] & 0xFFFFu);
                bd = min(bd, v[s] >> 16);
            }
        }
        c.lcp[b] = mn;
        c.bad[b] = bd;
        c.pd[b] = b > 0 ? 0u : kCsrNoDepth;
        c.skip[b] = 0u;
        #pragma unroll
        for (uint32_t l = 0; l < kCsrMaxLevels; ++l) c.lv[l][b] = 0u;
    }
    if (tid == 0) {
        c.nn = 0;
        c.ip_end = uint32_t(p.indptr[B]);
    }
    __syncthreads();
    auto internal = [&](uint32_t b) {
        return b > 0 && c.pd[b] != kCsrNoDepth && c.lcp[b] >= c.pd[b] + kCsrMinShared;
    };
    // Each level in one pass over the sequences (in rounds of NT), by
    // scans in thread order: b's run head is the max-scan of the non-internal
    // indices; the run's shortest prefix and first bad id so far are the
    // max-scans of (head << 16 | 0xFFFF - value), whose high half makes the
    // maximum stay inside the run.  A run's last member holds its totals and
    // records the node; its members read the node back from the head.
    uint32_t levels = 0;
    for (uint32_t lev = 0; lev < kCsrMaxLevels; ++lev) {
        for (uint32_t b = tid; b < B; b += NT) c.acc[b] = 0u;
        __syncthreads();
        const uint32_t nn0 = c.nn;
        uint32_t ch = 0, cm = 0, cb = 0, cn = 0;
        for (uint32_t base = 0; base < B; base += NT) {
            const uint32_t b = base + tid;
            const bool valid = b < B, in = valid && internal(b);
            uint32_t th, tm, tb;
            const uint32_t h = max(block_max_scan<NT>(valid && !in ? b : 0u, red, th), ch);
            const uint32_t mv = max(block_max_scan<NT>((h << 16) | (0xFFFFu - (in ? c.lcp[b] : 0xFFFFu)), red, tm), cm);
            const uint32_t bv = max(block_max_scan<NT>((h << 16) | (0xFFFFu - (in ? c.bad[b] : 0xFFFFu)), red, tb), cb);
            const bool last = valid && !(b + 1 < B && internal(b + 1));
            const uint32_t cntb = b - h + 1;
            // A run of fewer than 16 query rows is not worth a node: its
            // sequences read the shared pages themselves (the second read
            // mostly hits the caches), with fewer items and partial states.
            const bool node = last && cntb >= 2u && cntb * p.r >= uint32_t(kWaveRows);
            uint32_t x = node ? 1u : 0u, y = 0, tx, ty;
            block_incl_scan2<NT>(x, y, red, tx, ty);
            const uint32_t k = nn0 + cn + x - 1;
            if (valid) c.head[b] = h;
            if (node && k < kCsrMaxNodes) {
                const uint32_t len = 0xFFFFu - (mv & 0xFFFFu), fb = 0xFFFFu - (bv & 0xFFFFu);
                c.b0[k] = h;
                c.cnt[k] = cntb;
                c.npd[k] = c.pd[h + 1];            // h + 1 is internal: its pd is the run's
                c.len[k] = len;
                c.kind[k] = (lev << 1) | (fb < len ? 1u << 3 : 0u);   // level, poison; kind later
                c.acc[h] = k + 1;
                c.mn[h] = len;
            }
            ch = max(ch, th);
            cm = max(cm, tm);
            cb = max(cb, tb);
            cn += tx;
        }
        __syncthreads();
        if (cn == 0 || nn0 + cn > kCsrMaxNodes) break;   // no node, or too many: stop here
        // Members take the node of their run; boundaries inside a node go one
        // level deeper (their pd becomes the node's shared length).
        for (uint32_t b = tid; b < B; b += NT) {
            const uint32_t h = c.head[b], k1 = c.acc[h];
            c.lv[lev][b] = k1;
            c.tmp[b] = (k1 && internal(b)) ? c.mn[h] : kCsrNoDepth;
        }
        __syncthreads();
        uint32_t deeper[1] = {0u};
        for (uint32_t b = tid; b < B; b += NT) {
            c.pd[b] = c.tmp[b];
            deeper[0] |= (c.tmp[b] != kCsrNoDepth && c.lcp[b] >= c.tmp[b] + kCsrMinShared) ? 1u : 0u;
        }
        block_reduce<NT, false>(deeper, red);
        if (tid == 0) c.nn = nn0 + cn;
        __syncthreads();
        levels = lev + 1;
        if (!deeper[0]) break;   // no boundary reaches a deeper node
    }
    const uint32_t nn = c.nn;
    // Kinds, and the items and slots of each chunk-size candidate.
    constexpr uint32_t NC = 6;
    uint32_t sums[2 * NC + 2] = {};
    const uint32_t GR = p.group_rows;
    for (uint32_t k = tid; k < nn; k += NT) {
        const uint32_t rows = c.cnt[k] * p.r, pages = c.len[k] - c.npd[k];
        const bool grp = rows > 64u || (rows > 16u && pages > 16u);
        c.kind[k] |= grp ? 1u : 0u;
        if (grp) {
            const uint32_t rbk = (rows + GR - 1) / GR;
            #pragma unroll
            for (uint32_t i = 0; i < NC; ++i) {
                const uint32_t g = (pages + (8u << i) - 1) >> (3 + i);
                sums[i] += g * p.hkv * rbk;
                sums[NC + i] += g * c.cnt[k];
            }
        } else {
            const uint32_t g = (pages + kCsrWaveChunk - 1) / kCsrWaveChunk;
            sums[2 * NC] += g * p.hkv * ((rows + kWaveRows - 1) / kWaveRows);
            sums[2 * NC + 1] += g * c.cnt[k];
        }
    }
    block_reduce<NT, false>(sums, red);
    uint32_t pick = NC - 1, items_pick = sums[NC - 1], slots_pick = sums[2 * NC - 1];
    #pragma unroll
    for (int i = int(NC) - 1; i >= 0; --i) {
        if (sums[i] <= 256u) {
            pick = uint32_t(i);
            items_pick = sums[i];
            slots_pick = sums[NC + i];
        }
    }
    const uint64_t need_slots = uint64_t(slots_pick) + sums[2 * NC + 1];
    const bool on = nn > 0 && uint64_t(items_pick) + sums[2 * NC] <= p.gcap && need_slots + B <= p.slot_cap;
    gchunk = on ? 8u << pick : 0u;
    // Per node: chunks, first item (within its kind) and first seqslot; and
    // the load its items put on the chip.
    uint32_t ci = 0, cw = 0, cs = 0;
    uint32_t ld[1] = {0u}, mx[1] = {~0u};
    for (uint32_t base = 0; base < nn; base += NT) {
        const uint32_t k = base + tid;
        uint32_t gi = 0, wi = 0, ss = 0;
        if (on && k < nn) {
            const uint32_t rows = c.cnt[k] * p.r, pages = c.len[k] - c.npd[k];
            const bool grp = c.kind[k] & 1u;
            const uint32_t ch = grp ? gchunk : kCsrWaveChunk;
            const uint32_t g = (pages + ch - 1) / ch, per = p.hkv * (grp ? (rows + GR - 1) / GR
                                                                          : (rows + kWaveRows - 1) / kWaveRows);
            c.gc[k] = g;
            (grp ? gi : wi) = g * per;
            ss = g * c.cnt[k];
            const uint32_t w = grp ? uint32_t(kWaves) : 1u;
            ld[0] += ((g - 1) * csr_cost(ch) + csr_cost(pages - (g - 1) * ch)) * per * w;
            mx[0] = min(mx[0], ~csr_cost(min(ch, pages)));
        }
        uint32_t x = gi, y = wi, tx, ty;
        block_incl_scan2<NT>(x, y, red, tx, ty);
        uint32_t z = ss, zz = 0, tz, tzz;
        block_incl_scan2<NT>(z, zz, red, tz, tzz);
        if (on && k < nn) {
            c.item0[k] = (c.kind[k] & 1u) ? ci + x - gi : cw + y - wi;
            c.ss0[k] = cs + z - ss;
        }
        ci += tx;
        cw += ty;
        cs += tz;
    }
    block_reduce<NT, false>(ld, red);
    block_reduce<NT, true>(mx, red);
    load.waves = on ? ci * kWaves + cw : 0u;
    load.cost = on ? ld[0] : 0u;
    load.max_item = on && mx[0] != ~0u ? ~mx[0] : 0u;
    __syncthreads();
    // Per sequence: shared pages (its deepest node's), node chunks and the
    // slot offset of each level's chunks; poisoned if any node of it is.
    for (uint32_t b = tid; b < B; b += NT) {
        uint32_t depth = 0, chunks = 0;
        bool poison = false;
        for (uint32_t l = 0; l < levels; ++l) {
            const uint32_t k1 = c.lv[l][b] & 0xFFFFu;
            if (!on || !k1) continue;
            const uint32_t k = k1 - 1;
            c.lv[l][b] = k1 | (chunks << 16);
            chunks += c.gc[k];
            depth = c.len[k];
            poison |= (c.kind[k] >> 3) & 1u;
        }
        const uint32_t w = depth ? depth | (chunks << 16) : 0u;
        c.skip[b] = w;
        p.skip[b] = w;
        s_bad[b] = poison ? 1u : 0u;
    }
    __syncthreads();
    n_wave = on ? cw : 0u;
    gslots = on ? cs : 0u;
    if (!on && tid == 0) c.nn = 0;
    __syncthreads();
    return on ? ci : 0u;
}

// Items and seqslot entries of the cascade's nodes (first slots of the
// sequences in c.tmp; seqslot entries from n_chunks on, after the wave
// items' chunks).  Group items of a node cover unit u = chunk * hkv + KV
// head and row block rb; units are taken eight at a time, each with all its
// row blocks eight items apart, so the items reading the same pages run on
// the same XCD (workgroup i runs on XCD i mod 8) and share its L2.  A node's
// wave items (16 rows each) go unit by unit, row blocks within; they follow
// the group items in p.gitems.  red_scratch: the planning kernel's
// reduction space.
template <uint32_t NT>
__device__ void csr_cascade_emit(const CsrPlanArgs& p, const CsrCascade& c, uint32_t n_chunks, uint32_t n_group,
                                 uint32_t gchunk, uint32_t* red_scratch) {
    const uint32_t tid = threadIdx.x, GR = p.group_rows;
    // Seqslots, one thread per sequence: for each node of it (one a level),
    // its slot of every chunk (its first slot, the chunks of its shallower
    // nodes, then the chunk's index) at entry ss0 + chunk * cnt + member.
    for (uint32_t b = tid; b < p.batch; b += NT) {
        #pragma unroll
        for (uint32_t l = 0; l < kCsrMaxLevels; ++l) {
            const uint32_t w = c.lv[l][b], k1 = w & 0xFFFFu;
            if (!k1) continue;
            const uint32_t k = k1 - 1, cnt = c.cnt[k], g = c.gc[k];
            const uint32_t s0 = c.tmp[b] + (w >> 16);
            SeqSlot* dst = p.seqslots + n_chunks + c.ss0[k] + (b - c.b0[k]);
            for (uint32_t chk = 0; chk < g; ++chk) dst[chk * cnt] = SeqSlot{b, s0 + chk};
        }
    }
    // Items: the nodes' items as one range in node order (node k's at
    // s_ws[k] ..), cut into equal contiguous blocks, one a thread.  A thread
    // finds its block's first node by bisection, then walks the nodes'
    // item orders (csr_node_item's) with counters: one division each to
    // start a node, none per item.
    __shared__ uint32_t s_ws[kCsrMaxNodes + 1];
    auto n_items = [&](uint32_t k) {
        const uint32_t rows = c.cnt[k] * p.r;
        return c.gc[k] * p.hkv * ((c.kind[k] & 1u) ? (rows + GR - 1) / GR : (rows + kWaveRows - 1) / kWaveRows);
    };
    uint32_t carry = 0;
    for (uint32_t k0 = 0; k0 < c.nn; k0 += NT) {
        const uint32_t k = k0 + tid;
        const uint32_t v = k < c.nn ? n_items(k) : 0u;
        uint32_t x = v, y = 0u, tx, ty;
        block_incl_scan2<NT>(x, y, red_scratch, tx, ty);
        if (k < c.nn) s_ws[k] = carry + x - v;
        carry += tx;
    }
    if (tid == 0) s_ws[c.nn] = carry;
    __syncthreads();
    const uint32_t total = carry, per = (total + NT - 1) / NT;
    uint32_t f = min(total, tid * per);
    const uint32_t fend = min(total, f + per);
    if (f < fend) {
        uint32_t lo = 0, hi = c.nn;   // the last node starting at or before f
        while (hi - lo > 1) {
            const uint32_t mid = (lo + hi) >> 1;
            if (s_ws[mid] <= f) lo = mid;
            else hi = mid;
        }
        for (uint32_t k = lo; f < fend; ++k) {
            const uint32_t nk0 = s_ws[k], nk1 = s_ws[k + 1];
            if (nk1 <= f) continue;   // an empty node
            const uint32_t b0 = c.b0[k], cnt = c.cnt[k], pd = c.npd[k], len = c.len[k], g = c.gc[k];
            const uint32_t grp = c.kind[k] & 1u, item0 = c.item0[k], ss0 = c.ss0[k], p0 = c.ip[b0];
            const uint32_t rows = cnt * p.r;
            const uint32_t rbk = grp ? (rows + GR - 1) / GR : (rows + kWaveRows - 1) / kWaveRows;
            const uint32_t RR = grp ? GR : uint32_t(kWaveRows), ch = grp ? gchunk : kCsrWaveChunk;
            const uint32_t units = g * p.hkv;
            uint32_t i = f - nk0;
            const uint32_t iend = min(fend, nk1) - nk0;
            // Position of item i: group items take units eight at a time
            // (blk), all row blocks of the eight (rb), then the unit within
            // (uu of m); wave items a unit (blk) and its row blocks.
            uint32_t blk, rb, uu, m;
            if (grp) {
                blk = i / (8 * rbk);
                const uint32_t w = i - blk * 8 * rbk;
                m = min(8u, units - blk * 8);
                rb = w / m;
                uu = w - rb * m;
            } else {
                blk = i / rbk;
                rb = i - blk * rbk;
                uu = 0;
                m = 1;
            }
            const uint32_t u0 = grp ? blk * 8 : blk, u = u0 + uu;
            uint32_t chk0 = u0 / p.hkv, h0 = u0 - chk0 * p.hkv;     // unit blk * 8 (group items)
            uint32_t chk = u / p.hkv, h = u - chk * p.hkv;          // the item's unit
            auto next_unit = [&](uint32_t& ck, uint32_t& hh) {
                if (++hh == p.hkv) {
                    hh = 0;
                    ++ck;
                }
            };
            Item* out = p.gitems + (grp ? 0u : n_group) + item0;
            for (; i < iend; ++i) {
                Item it;
                it.page_off = p0 + pd + chk * ch;
                it.npages = min(ch, len - pd - chk * ch);
                it.seq_off = n_chunks + ss0 + chk * cnt;
                it.row_begin = rb * RR;
                it.nrows = min(RR, rows - rb * RR);
                it.kv_head = h;
                it.flags = 0u;
                it.tail_seq = b0;
                out[i] = it;
                // the next item's position
                if (grp) {
                    next_unit(chk, h);
                    if (++uu == m) {
                        uu = 0;
                        chk = chk0;
                        h = h0;
                        if (++rb == rbk) {
                            rb = 0;
                            for (uint32_t t = 0; t < m; ++t) next_unit(chk0, h0);
                            chk = chk0;
                            h = h0;
                            ++blk;
                            m = min(8u, units - min(units, blk * 8));
                        }
                    }
                } else if (++rb == rbk) {
                    rb = 0;
                    next_unit(chk, h);
                }
            }
            f = min(fend, nk1);
        }
    }
}

// Work decomposition of one dh_decode_csr call, on the device: sequence b's
// pages indptr[b] .. indptr[b+1] split into chunks of `chunk` pages (the last
// one shorter), chunk k of b in partial-state slot slot_ptr[b] + k.
//
// chunk: of the candidates whose chunks fit the workspace's slots, the one
// whose heaviest-first list schedule over kCsrWaveSlots wave slots is
// estimated to end first (ties: the larger chunk, fewer partial states).  The
// estimate is the largest item when the waves fit the slots at once, else
// the mean load plus the smallest item (the last ones placed), at least the
// largest item.  On 35 batches of 1-600 sequences it picks a chunk whose
// exact heaviest-first schedule ends 3 % after the best candidate's on
// average.  Chunks that give a sequence more than kCsrMaxStates partial
// states come last (C2, six 272-page sequences: 4-page chunks, 68 states a
// row, took the merge from the vector to the scalar path).  No candidate
// fitting (more chunks of kCsrMaxChunk pages than the workspace holds):
// overflow, no items, zeros out.
//
// Dispatch order (seqslots[j] = {sequence, slot} of the j-th chunk, j the
// wave item's index / per_chunk): the full chunks first, then the shorter
// last chunks by size, longest first, so the hardware's in-order dispatch
// to free slots is a heaviest-first list schedule.  Order does not change
// results: each chunk's partial state has its slot, merged in slot order.
//
// A sequence whose indptr entries are negative or decreasing, or that has
// more than DH_MAX_SEQ_LEN / 16 pages, gets no chunk and is marked bad
// (zeros out, status DH_EINVAL).
template <uint32_t NT>
__global__ __launch_bounds__(NT) void csr_plan_kernel(CsrPlanArgs p) {
    constexpr uint32_t KC = kCsrFixedCandidates, KM = KC + 1;
    __shared__ uint32_t red[(NT / 64) * 2 * KM];
    __shared__ uint32_t s_tail[kCsrMaxChunk];    // last chunks of each size, then their next position
    // Cascade: its nodes and per-sequence state; members of poisoned nodes.
    __shared__ CsrCascade cc;
    __shared__ uint32_t s_bad[kCsrCascadeMaxBatch];
    const uint32_t tid = threadIdx.x;
    constexpr uint32_t kMaxSeqPages = DH_MAX_SEQ_LEN / kPageSize;
    const uint32_t iters = (p.batch + NT - 1) / NT;
    // Shared prefixes of consecutive sequences first (nodes read by group or
    // multi-sequence wave items): each sequence's own wave items then cover
    // only the pages past its deepest node's.
    const bool casc = p.lcp != nullptr && p.batch >= 2 && p.batch <= kCsrCascadeMaxBatch;
    uint32_t n_gitems = 0, n_nwave = 0, gslots = 0, gchunk = 0;
    CsrNodeLoad nload{0u, 0u, 0u};
    if (casc) n_gitems = csr_cascade<NT>(p, cc, s_bad, red, n_nwave, gslots, gchunk, nload);
    const bool grouped = gslots > 0;
    auto load = [&](uint32_t b, bool& ok) -> uint32_t {
        ok = false;
        if (b >= p.batch) return 0u;
        // With a cascade indptr is in LDS already (no second round trip).
        const int32_t p0 = casc ? int32_t(cc.ip[b]) : p.indptr[b];
        const int32_t p1 = casc ? int32_t(b + 1 < p.batch ? cc.ip[b + 1] : cc.ip_end) : p.indptr[b + 1];
        ok = p0 >= 0 && p1 >= p0 && uint32_t(p1 - p0) <= kMaxSeqPages;
        if (!ok) return 0u;
        return uint32_t(p1 - p0) - (grouped ? (cc.skip[b] & 0xFFFFu) : 0u);
    };
    // Slots the wave items' chunks may take.
    const uint32_t cap_s = p.slot_cap - gslots;
    constexpr uint32_t R = csr_reg_seqs(NT);
    uint32_t nr[R], okr = 0;
    #pragma unroll
    for (uint32_t r = 0; r < R; ++r) {
        bool ok = false;
        nr[r] = load(r * NT + tid, ok);
        okr |= ok ? 1u << r : 0u;
    }
    // f(b, n, ok) over this thread's sequences in order, with a trip count
    // uniform over the workgroup (f may hold barriers); b >= batch: n = 0.
    auto each = [&](auto&& f) {
        #pragma unroll
        for (uint32_t r = 0; r < R; ++r)
            if (r < iters) f(r * NT + tid, nr[r], ((okr >> r) & 1u) != 0u);
        if constexpr (NT > kCsrSmallThreads) {
            for (uint32_t it = R; it < iters; ++it) {
                bool ok = false;
                const uint32_t b = it * NT + tid;
                const uint32_t n = load(b, ok);
                f(b, n, ok);
            }
        }
    };
    for (uint32_t i = tid; i < kCsrMaxChunk; i += NT) s_tail[i] = 0u;

    // Pass 1: pages in all (<= 2^16 * 2^13; the costs below, at most 4 a
    // page, fit 32 bits) and the longest sequence.
    uint32_t tot[1] = {0u}, nmax[1] = {~0u};
    each([&](uint32_t, uint32_t n, bool) {
        tot[0] += n;
        nmax[0] = min(nmax[0], ~n);
    });
    block_reduce<NT, false>(tot, red);
    block_reduce<NT, true>(nmax, red);
    const uint32_t total = tot[0], maxn = ~nmax[0];
    const uint32_t want = uint32_t(min(uint64_t(kCsrMaxChunk),
                                       max(uint64_t(1), (uint64_t(total) * p.per_chunk + kCsrWaveSlots - 1) /
                                                            kCsrWaveSlots)));
    // Candidates weighed (bit i: fixed candidate i; bit KC: want): the fixed
    // sizes from want / 8 up to want (a larger chunk costs more per item and
    // balances no better than want's; below want / 8 an item start costs
    // more than its pages), the smallest fixed size that leaves a sequence
    // at most kCsrMaxStates states, kCsrMaxChunk (the fallback) and want.
    // Sizes below that smallest one are not weighed: they rank after it
    // (more states a row) and need more slots, and it is at most
    // DH_MAX_SEQ_LEN / 16 / kCsrMaxStates = 128 pages, a fixed candidate.
    const uint32_t need = (maxn + kCsrMaxStates - 1) / kCsrMaxStates;
    uint32_t active = (1u << (KC - 1)) | (want >= need ? 1u << KC : 0u);
    bool need_met = false;
    #pragma unroll
    for (uint32_t i = 0; i < KC; ++i) {
        const uint32_t c = csr_candidate(i);
        if (8 * c >= want && c <= want && c >= need) active |= 1u << i;
        if (!need_met && c >= need) {
            active |= 1u << i;
            need_met = true;
        }
    }
    // Pass 2: per candidate, its chunks, their cost and the cheapest chunk.
    uint32_t sums[2 * KM] = {}, mins[KM];
    #pragma unroll
    for (uint32_t i = 0; i < KM; ++i) mins[i] = ~0u;
    each([&](uint32_t, uint32_t n, bool) {
        if (n == 0) return;
        #pragma unroll
        for (uint32_t i = 0; i < KM; ++i) {
            if (!((active >> i) & 1u)) continue;
            const uint32_t c = i < KC ? csr_candidate(i) : want, full = n / c, t = n - full * c;
            sums[i] += full + (t ? 1u : 0u);
            sums[KM + i] += full * csr_cost(c) + (t ? csr_cost(t) : 0u);
            mins[i] = min(mins[i], csr_cost(t ? t : c));
        }
    });
    block_reduce<NT, false>(sums, red, uint64_t(active) | (uint64_t(active) << KM));
    block_reduce<NT, true>(mins, red, active);

    // Chunks that leave a row more than kCsrMaxStates partial states (the
    // merge kernel's vector path) rank after every other fitting one.  The
    // cascade's node items (nload) hold wave slots and add their cost.
    auto end_of = [&](uint32_t c, uint32_t cnt, uint32_t cost, uint32_t mn) -> uint64_t {
        if (cnt > cap_s) return ~uint64_t(0);
        const uint64_t S = kCsrWaveSlots, mx = max(csr_cost(min(c, maxn)), nload.max_item);
        const uint64_t e = uint64_t(cnt) * p.per_chunk + nload.waves <= S
                               ? mx * S
                               : max(mx * S, uint64_t(cost) * p.per_chunk + nload.cost + uint64_t(mn) * S);
        return c < need ? e | (uint64_t(1) << 62) : e;     // more than kCsrMaxStates chunks of maxn pages
    };
    uint32_t chunk = kCsrMaxChunk, n_chunks = sums[KC - 1];
    uint64_t best = ~uint64_t(0);
    #pragma unroll
    for (uint32_t i = 0; i < KM; ++i) {
        if (!((active >> i) & 1u)) continue;
        const uint32_t c = i < KC ? csr_candidate(i) : want;
        const uint64_t e = end_of(c, sums[i], sums[KM + i], mins[i]);
        if (e < best || (e == best && e != ~uint64_t(0) && c > chunk)) {
            best = e;
            chunk = c;
            n_chunks = sums[i];
        }
    }
    const bool overflow = n_chunks > cap_s;

    // Pass 3: last chunks of each size; those of size t take the positions
    // n_chunks - (last chunks of size <= t) onwards, so the longest follow
    // the full chunks and the shortest end the order.
    each([&](uint32_t, uint32_t n, bool) {
        const uint32_t t = n - (n / chunk) * chunk;
        if (t) atomicAdd(&s_tail[t], 1u);
    });
    __syncthreads();
    {
        uint32_t carry = 0;
        for (uint32_t base = 1; base < chunk; base += NT) {
            const uint32_t t = base + tid;
            uint32_t v = t < chunk ? s_tail[t] : 0u, z = 0u, tv, tz;
            block_incl_scan2<NT>(v, z, red, tv, tz);
            if (t < chunk) s_tail[t] = n_chunks - (carry + v);
            carry += tv;
        }
        __syncthreads();
    }

    // Pass 4: each sequence's first slot (prefix sum of the chunk counts)
    // and its chunks' positions: full chunks after the full chunks of the
    // sequences before it, its last chunk from its size's range.
    // With a cascade, a sequence's slots are its group chunks' (one per
    // chunk of its group's shared pages) and then its wave items' chunks.
    uint32_t carry = 0, carry_t = 0, carry_g = 0;
    each([&](uint32_t b, uint32_t n, bool ok) {
        const uint32_t full = n / chunk, t = n - full * chunk, has_t = t ? 1u : 0u, cnt = full + has_t;
        const uint32_t gcb = (grouped && b < p.batch) ? cc.skip[b] >> 16 : 0u;
        uint32_t x = cnt + gcb, y = has_t, tx, ty;
        block_incl_scan2<NT>(x, y, red, tx, ty);
        uint32_t xg = gcb, yg = 0, txg = 0, tyg;
        if (grouped) block_incl_scan2<NT>(xg, yg, red, txg, tyg);
        const uint32_t first = carry + x - cnt - gcb;
        const uint32_t fpos = first - (carry_g + xg - gcb) - (carry_t + y - has_t);
        if (b < p.batch) {
            p.slot_ptr[b] = first;
            p.seq_bad[b] = (ok && !overflow && !(grouped && s_bad[b])) ? 0u : 1u;
            if (grouped) cc.tmp[b] = first;
            if (!overflow && t) {
                const uint32_t pos = atomicAdd(&s_tail[t], 1u);
                if (pos < p.slot_cap) p.seqslots[pos] = SeqSlot{b, first + gcb + full};
            }
        }
        // Full chunks: each lane its own sequence's, or, in the one-wave
        // variant when a sequence has more of them than there are
        // sequences, the whole wave one sequence's after another.
        bool by_wave = false;
        if constexpr (NT == kCsrSmallThreads)
            by_wave = ~uint32_t(__builtin_amdgcn_readlane(wave_scan_dpp<true>(~full), 63)) > p.batch;
        if (!overflow && by_wave) {
            for (uint32_t sq = 0; sq < p.batch; ++sq) {
                const uint32_t fs = __builtin_amdgcn_readlane(full, sq), ps = __builtin_amdgcn_readlane(fpos, sq);
                const uint32_t ss = __builtin_amdgcn_readlane(first + gcb, sq);
                for (uint32_t k = tid; k < fs && ps + k < p.slot_cap; k += kCsrSmallThreads)
                    p.seqslots[ps + k] = SeqSlot{sq, ss + k};
            }
        } else if (!overflow && b < p.batch) {
            for (uint32_t k = 0; k < full && fpos + k < p.slot_cap; ++k)
                p.seqslots[fpos + k] = SeqSlot{b, first + gcb + k};
        }
        carry += tx;
        carry_t += ty;
        carry_g += txg;
    });
    // The nodes' items and seqslots (entries n_chunks .. n_chunks + gslots,
    // after the wave items' chunks in dispatch order).
    const bool emit = grouped && !overflow;
    if (emit) {
        __syncthreads();   // first slots (cc.tmp) of every sequence
        csr_cascade_emit<NT>(p, cc, n_chunks, n_gitems, gchunk, red);
    }
    if (tid == 0) {
        const uint32_t slots = n_chunks + gslots;
        p.slot_ptr[p.batch] = overflow ? 0u : slots;
        p.hdr->chunk = chunk;
        p.hdr->n_items = overflow ? 0u : n_chunks * p.per_chunk;
        p.hdr->overflow = overflow ? 1u : 0u;
        p.hdr->n_chunks = slots;
        p.hdr->n_group = emit ? n_gitems : 0u;
        p.hdr->group_chunk = gchunk;
        p.hdr->n_node_waves = emit ? n_nwave : 0u;
    }
}

template <int D>
hipError_t launch_csr_attend_d(const AttendArgs& a, uint32_t q_dtype, uint32_t kvf, hipStream_t s) {
    dim3 grid(a.csr_grid), block(kWaves * 64);
    if (q_dtype == 2 && kvf == KVF_F32) {
        hipLaunchKernelGGL(csr_attend32_kernel<D>, grid, block, 0, s, a);
    } else if (q_dtype == 1 && kvf == KVF_BF16) {
        hipLaunchKernelGGL((csr_attend16_kernel<D, KVF_BF16, false>), grid, block, 0, s, a);
    } else if (q_dtype == 1 && kvf == KVF_FP8) {
        hipLaunchKernelGGL((csr_attend16_kernel<D, KVF_FP8, false>), grid, block, 0, s, a);
    } else if (q_dtype == 1 && kvf == KVF_MX) {
        hipLaunchKernelGGL((csr_attend16_kernel<D, KVF_MX, false>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_FP8) {
        hipLaunchKernelGGL((csr_attend16_kernel<D, KVF_FP8, true>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_MX) {
        hipLaunchKernelGGL((csr_attend16_kernel<D, KVF_MX, true>), grid, block, 0, s, a);
    } else if (q_dtype == 0 && kvf == KVF_F16) {
        hipLaunchKernelGGL((csr_attend16_kernel<D, KVF_F16, true>), grid, block, 0, s, a);
    } else {
        return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace

int launch_csr_attend(const AttendArgs& a, uint32_t q_dtype, uint32_t kvf, uint32_t d, void* stream) {
    if (a.csr_grid == 0) return hipSuccess;
    hipStream_t s = reinterpret_cast<hipStream_t>(stream);
    switch (d) {
        case 64: return launch_csr_attend_d<64>(a, q_dtype, kvf, s);
        case 128: return launch_csr_attend_d<128>(a, q_dtype, kvf, s);
        case 256: return launch_csr_attend_d<256>(a, q_dtype, kvf, s);
        default: return hipErrorInvalidValue;
    }
}

int launch_csr_lcp(const int32_t* indptr, const int32_t* indices, uint32_t batch, uint32_t page_limit,
                   uint32_t* lcp, void* stream) {
    if (batch < 2) return hipSuccess;
    const uint64_t waves = uint64_t(batch - 1) * kCsrLcpSlices;
    const uint64_t want = (waves + kWaves - 1) / kWaves;
    const uint32_t blocks = uint32_t(want < 1024 ? want : 1024);
    hipLaunchKernelGGL(csr_lcp_kernel, dim3(blocks), dim3(kWaves * 64), 0, reinterpret_cast<hipStream_t>(stream),
                       indptr, indices, batch, page_limit, lcp);
    return hipGetLastError();
}

int launch_csr_plan(const CsrPlanArgs& p, void* stream) {
    if (p.batch == 0 || p.slot_cap <= p.batch) return hipErrorInvalidValue;
    const auto s = reinterpret_cast<hipStream_t>(stream);
    if (p.batch <= kCsrSmallThreads)
        hipLaunchKernelGGL(csr_plan_kernel<kCsrSmallThreads>, dim3(1), dim3(kCsrSmallThreads), 0, s, p);
    else
        hipLaunchKernelGGL(csr_plan_kernel<kCsrThreads>, dim3(1), dim3(kCsrThreads), 0, s, p);
    return hipGetLastError();
}

}  // namespace dh
