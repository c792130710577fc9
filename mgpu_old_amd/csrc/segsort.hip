// Segmented LSD radix sort for gfx950: thousands of independent arrays of
// uneven sizes sorted in one persistent launch.  Each segment's result is
// exactly what sortArray would produce on it alone (stable by the bit field,
// values following), left on side `result_side` of its ping-pong buffers.
//
// No reference counterpart: the reference sorts one array per sortArray call
// (sort/src/mgpusort/mgpusort.cpp:607-616); its per-block ranking and scatter
// steps (sort/src/kernels/sort.cu:54-479) appear here inside one workgroup.
//
// Work is split by size on the host:
//   small  (n <= 64*IPT)     one wave sorts the segment in LDS, all passes;
//   block  (n <= BLOCK*IPT)  one workgroup sorts it in LDS, all passes;
//   global (larger)          one workgroup runs every pass through global
//                            memory, tile by tile, with running digit offsets
//                            (no cross-workgroup lookback needed).
// Workgroups first drain the block/global list (largest first, from a cursor
// per group of workgroups), then their waves take the small list round-robin,
// one segment per wave at a time.  The last workgroup of a group to finish
// puts its cursor back to zero, so a captured graph of this launch can be
// replayed as is.
//
// In-LDS routines carry (key, payload) through the passes, one 64-bit LDS
// word per slot: the payload is the value with one value array, else the
// source index (the value in index mode; several arrays are gathered through
// it once at the end).  The global routine carries the values through each
// pass.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "kernel_args.h"
#include "localsort.h"
#include "radix_device.h"

MGPU_EXPORT_ARGS_LAYOUT

namespace {

using mgpu::block_exclusive_scan;
using mgpu::st_agent;
using mgpu::wave_inclusive_scan;
using mgpu::wave_rank;


// Orders this wave's LDS accesses before and after the call.
__device__ __forceinline__ void wave_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Stable rank of this lane's digit d among the active lanes of the wave
// with the same digit, counted from count[d], which it advances.  rank1: one
// LDS atomic add per lane (served in ascending lane order, as the engine
// checked at creation), or a single add when every active lane holds the
// same digit (sorted or constant keys would serialize 64 adds on one word);
// else by match masks (wave_rank).
__device__ __forceinline__ uint32_t seg_rank(uint32_t d, uint32_t lane, uint32_t* count,
                                             uint64_t* match, bool rank1) {
    if (!rank1) return wave_rank(d, lane, count, match);
    const uint32_t f = __builtin_amdgcn_readfirstlane(d);
    const uint64_t exec = __builtin_amdgcn_read_exec();
    if (__builtin_amdgcn_ballot_w64(d == f) == exec) {
        const uint32_t below = mgpu::lanes_below(exec);
        uint32_t b = 0;
        if (below == 0)
            b = __hip_atomic_fetch_add(&count[f], (uint32_t)__builtin_popcountll(exec),
                                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        return __builtin_amdgcn_readfirstlane(b) + below;
    }
    return __hip_atomic_fetch_add(&count[d], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}

// Bit field of pass p: shift and mask (the split of mgpuSegArgs).
__device__ __forceinline__ void pass_field(const mgpuSegArgs& a, uint32_t p, uint32_t& shift,
                                           uint32_t& mask) {
    const uint32_t np = a.num_passes, base = a.num_bits / np, extra = a.num_bits % np;
    const uint32_t wide_from = np - extra;  // passes from here take base + 1 bits
    shift = a.first_bit + p * base + (p > wide_from ? p - wide_from : 0u);
    mask = (1u << (base + (p >= wide_from ? 1u : 0u))) - 1u;
}

// Shared memory of one workgroup of BLOCK threads (W waves).  The in-LDS
// routines stage a slot's key and payload together, one 64-bit word; the
// global routine uses the stage's first TILE 32-bit words.  Wave w's slice
// (64 * IPT words from w * 64 * IPT) also holds, in its first RADIX words,
// the wave's match-mask table of the match-mask ranking (match_table), which
// the staging overwrites: that ranking clears it first (clear_match).
template <int RB, int IPT, int BLOCK>
struct SegShared {
    static constexpr int W = BLOCK / 64;
    static constexpr int RADIX = 1 << RB;
    static constexpr int TILE = BLOCK * IPT;
    static constexpr int MAXP = (32 + RB - 1) / RB;
    static_assert(64 * IPT >= RADIX, "a wave's stage slice holds its match-mask table");
    uint64_t stage[TILE];
    uint32_t count[W][RADIX + 4] __attribute__((aligned(16)));
    uint32_t base[MAXP][RADIX];  // global routine: per-pass digit starts
    uint32_t run[RADIX];         // global routine: running digit offsets
    uint32_t dst[RADIX];         // global routine: output base per digit for a tile
    uint32_t tmp[W];
    uint32_t item;
};

template <int RB, int IPT, int BLOCK>
__device__ __forceinline__ uint64_t* match_table(SegShared<RB, IPT, BLOCK>& sh, uint32_t wave) {
    return sh.stage + wave * 64 * IPT;
}

// Zeroes the wave's match-mask table before a ranking by match masks (the
// atomic-add ranking does not use it).  Orders the wave's LDS accesses.
template <int RB, int IPT, int BLOCK>
__device__ __forceinline__ void clear_match(const mgpuSegArgs& a, SegShared<RB, IPT, BLOCK>& sh,
                                            uint32_t lane, uint32_t wave) {
    if (a.rank1) return;
    uint64_t* m = match_table(sh, wave);
    for (uint32_t i = lane; i < (uint32_t)SegShared<RB, IPT, BLOCK>::RADIX; i += 64) m[i] = 0;
    wave_sync();
}

// The payload a slot carries through the in-LDS passes: its value when the
// sort has exactly one value array (read once, in order, at the start, and
// written at the end with no gather), else its source index (the value
// itself in index mode; the gather index of every array otherwise).
__device__ __forceinline__ bool carries_value(const mgpuSegArgs& a) {
    return !a.index_mode && a.num_values == 1;
}

// Writes the sorted keys and the values: the carried payload when it is the
// value (one array, or indices), else every value array gathered through the
// source indices, out[pos] = in[src[pos]].  `sync` orders the gathers of the
// whole group before any store (the result side may be the input side).
template <int IPT, typename Sync>
__device__ __forceinline__ void emit(const mgpuSegArgs& a, const mgpuSegDesc& s, uint32_t n,
                                     const uint32_t* key, const uint32_t* pay, const uint32_t* idx,
                                     Sync sync) {
    const uint32_t side = a.result_side;
    const auto ko = mgpu::to_global(s.keys[side]);
#pragma unroll
    for (int j = 0; j < IPT; ++j)
        if (idx[j] < n) ko[idx[j]] = key[j];
    if (a.index_mode || carries_value(a)) {
        const auto vo = mgpu::to_global(s.vals[0][side]);
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) vo[idx[j]] = pay[j];
        return;
    }
    for (uint32_t v = 0; v < a.num_values; ++v) {
        const auto vi = mgpu::to_global(s.vals[v][0]);
        const auto vo = mgpu::to_global(s.vals[v][side]);
        uint32_t val[IPT];
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) val[j] = vi[pay[j]];
        sync();
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) vo[idx[j]] = val[j];
        sync();
    }
}

// Initial registers of an in-LDS sort: slot j's key and payload.
template <int IPT>
__device__ __forceinline__ void load_slots(const mgpuSegArgs& a, const mgpuSegDesc& s, uint32_t n,
                                           const uint32_t* idx, uint32_t* key, uint32_t* pay) {
    const auto ki = mgpu::to_global(s.keys[0]);
    const bool value = carries_value(a);
    const auto vi = mgpu::to_global(s.vals[0][0]);
#pragma unroll
    for (int j = 0; j < IPT; ++j) {
        key[j] = idx[j] < n ? ki[idx[j]] : 0u;
        pay[j] = idx[j] < n && value ? vi[idx[j]] : idx[j];
    }
}

// ---- one wave, whole segment in registers + this wave's LDS slice ---------
template <int RB, int IPT, int BLOCK>
__device__ __forceinline__ void wave_sort(const mgpuSegArgs& a, const mgpuSegDesc& s, SegShared<RB, IPT, BLOCK>& sh,
                          uint32_t lane, uint32_t wave) {
    constexpr int RADIX = SegShared<RB, IPT, BLOCK>::RADIX;
    constexpr int DPL = RADIX >= 64 ? RADIX / 64 : 1;  // digits per lane in the scan
    const uint32_t n = s.n;
    uint64_t* stage = sh.stage + wave * 64 * IPT;
    uint32_t* count = sh.count[wave];
    uint64_t* match = match_table(sh, wave);

    uint32_t key[IPT], pay[IPT], idx[IPT], pos[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) idx[j] = j * 64 + lane;
    load_slots<IPT>(a, s, n, idx, key, pay);
    for (uint32_t p = 0; p < a.num_passes; ++p) {
        uint32_t shift, mask;
        pass_field(a, p, shift, mask);
#pragma unroll
        for (int i = 0; i < DPL; ++i)
            if (lane * DPL + i < (uint32_t)RADIX) count[lane * DPL + i] = 0;
        wave_sync();
        clear_match(a, sh, lane, wave);
        uint32_t rank[IPT];
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n)
                rank[j] = seg_rank((key[j] >> shift) & mask, lane, count, match, a.rank1 != 0);
        wave_sync();
        // Exclusive scan of the digit counts across the wave.
        uint32_t c[DPL], sum = 0;
#pragma unroll
        for (int i = 0; i < DPL; ++i) {
            c[i] = lane * DPL + i < (uint32_t)RADIX ? count[lane * DPL + i] : 0u;
            sum += c[i];
        }
        uint32_t run = wave_inclusive_scan(sum, lane) - sum;
#pragma unroll
        for (int i = 0; i < DPL; ++i)
            if (lane * DPL + i < (uint32_t)RADIX) {
                count[lane * DPL + i] = run;
                run += c[i];
            }
        wave_sync();
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) {
                pos[j] = count[(key[j] >> shift) & mask] + rank[j];
                stage[pos[j]] = (uint64_t)pay[j] << 32 | key[j];
            }
        wave_sync();
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) {
                const uint64_t t = stage[idx[j]];
                key[j] = (uint32_t)t;
                pay[j] = (uint32_t)(t >> 32);
            }
        wave_sync();
    }
    emit<IPT>(a, s, n, key, pay, idx, [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        wave_sync();
    });
}

// ---- one wave, at most 64 keys: a bitonic network in registers -------------
// Lane i holds key i.  The network orders 64-bit compare keys (the sort's bit
// field above the lane index, all ones past n), so equal fields keep their
// input order and the result is the stable sort by the field, as the passes
// would leave it; each lane then takes its key and payload from the lane its
// compare key came from.  No LDS and no atomics: two shuffles per step, 21
// steps.
__device__ __forceinline__ void wave_bitonic64(const mgpuSegArgs& a, const mgpuSegDesc& s, uint32_t lane) {
    const uint32_t n = s.n;
    uint32_t idx[1] = {lane}, key[1], pay[1];
    load_slots<1>(a, s, n, idx, key, pay);
    const uint32_t field = a.num_bits >= 32 ? key[0] >> a.first_bit
                                            : (key[0] >> a.first_bit) & ((1u << a.num_bits) - 1u);
    uint64_t ck = lane < n ? ((uint64_t)field << 6) | lane : ~0ull;
#pragma unroll
    for (uint32_t k = 2; k <= 64; k <<= 1) {
#pragma unroll
        for (uint32_t j = k >> 1; j > 0; j >>= 1) {
            const uint32_t olo = (uint32_t)__shfl_xor((int)(uint32_t)ck, (int)j, 64);
            const uint32_t ohi = (uint32_t)__shfl_xor((int)(uint32_t)(ck >> 32), (int)j, 64);
            const uint64_t other = ((uint64_t)ohi << 32) | olo;
            // Ascending blocks of k (all of them at k = 64); the lower lane
            // of a pair keeps the smaller key in an ascending block.
            const bool keep_min = ((lane & j) == 0) == ((lane & k) == 0);
            if (keep_min ? other < ck : other > ck) ck = other;
        }
    }
    const int src = (int)((uint32_t)ck & 63u);
    uint32_t k2[1] = {(uint32_t)__shfl((int)key[0], src, 64)};
    uint32_t p2[1] = {(uint32_t)__shfl((int)pay[0], src, 64)};
    emit<1>(a, s, n, k2, p2, idx, [] {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
        wave_sync();
    });
}

// ---- one workgroup, whole segment in registers + LDS ----------------------
template <int RB, int IPT, int BLOCK>
__device__ __forceinline__ void block_sort(const mgpuSegArgs& a, const mgpuSegDesc& s, SegShared<RB, IPT, BLOCK>& sh,
                           uint32_t tid, uint32_t lane, uint32_t wave) {
    constexpr int RADIX = SegShared<RB, IPT, BLOCK>::RADIX;
    constexpr int W = BLOCK / 64;
    const uint32_t n = s.n;
    uint32_t key[IPT], pay[IPT], idx[IPT], pos[IPT];
#pragma unroll
    for (int j = 0; j < IPT; ++j) idx[j] = wave * 64 * IPT + j * 64 + lane;
    load_slots<IPT>(a, s, n, idx, key, pay);
    for (uint32_t p = 0; p < a.num_passes; ++p) {
        uint32_t shift, mask;
        pass_field(a, p, shift, mask);
        // (The previous pass's reads of the stage end before this barrier,
        // and its writes of the next pass come after two more.)
        for (uint32_t i = tid; i < (uint32_t)(W * (RADIX + 4)); i += BLOCK) (&sh.count[0][0])[i] = 0;
        __syncthreads();
        clear_match(a, sh, lane, wave);
        uint32_t rank[IPT];
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n)
                rank[j] = seg_rank((key[j] >> shift) & mask, lane, sh.count[wave],
                                   match_table(sh, wave), a.rank1 != 0);
        __syncthreads();
        uint32_t total = 0;
        if (tid < (uint32_t)RADIX) {
#pragma unroll
            for (int w = 0; w < W; ++w) {
                uint32_t c = sh.count[w][tid];
                sh.count[w][tid] = total;
                total += c;
            }
        }
        const uint32_t start = block_exclusive_scan<BLOCK>(total, sh.tmp, lane, wave);
        if (tid < (uint32_t)RADIX) {
#pragma unroll
            for (int w = 0; w < W; ++w) sh.count[w][tid] += start;
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) {
                pos[j] = sh.count[wave][(key[j] >> shift) & mask] + rank[j];
                sh.stage[pos[j]] = (uint64_t)pay[j] << 32 | key[j];
            }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IPT; ++j)
            if (idx[j] < n) {
                const uint64_t t = sh.stage[idx[j]];
                key[j] = (uint32_t)t;
                pay[j] = (uint32_t)(t >> 32);
            }
    }
    emit<IPT>(a, s, n, key, pay, idx, [] { __syncthreads(); });
}

// ---- one workgroup, passes through global memory ---------------------------
template <int RB, int IPT, int BLOCK>
__device__ __forceinline__ void global_sort(const mgpuSegArgs& a, const mgpuSegDesc& s, SegShared<RB, IPT, BLOCK>& sh,
                            uint32_t tid, uint32_t lane, uint32_t wave) {
    constexpr int RADIX = SegShared<RB, IPT, BLOCK>::RADIX;
    uint32_t* const st = reinterpret_cast<uint32_t*>(sh.stage);  // TILE words of it
    constexpr int W = BLOCK / 64;
    constexpr uint32_t TILE = SegShared<RB, IPT, BLOCK>::TILE;
    const uint32_t n = s.n;
    const uint32_t np = a.num_passes;

    // Digit histograms of every pass in one read, then their exclusive scans.
    for (uint32_t i = tid; i < np * RADIX; i += BLOCK) (&sh.base[0][0])[i] = 0;
    __syncthreads();
    for (uint32_t i = tid; i < n; i += BLOCK) {
        const uint32_t k = mgpu::to_global(s.keys[0])[i];
        for (uint32_t p = 0; p < np; ++p) {
            uint32_t shift, mask;
            pass_field(a, p, shift, mask);
            __hip_atomic_fetch_add(&sh.base[p][(k >> shift) & mask], 1u, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_WORKGROUP);
        }
    }
    __syncthreads();
    for (uint32_t p = 0; p < np; ++p) {
        uint32_t c = tid < (uint32_t)RADIX ? sh.base[p][tid] : 0u;
        uint32_t e = block_exclusive_scan<BLOCK>(c, sh.tmp, lane, wave);
        if (tid < (uint32_t)RADIX) sh.base[p][tid] = e;
    }

    const uint32_t nv = a.num_values;
    for (uint32_t p = 0; p < np; ++p) {
        const uint32_t in = p & 1, out = in ^ 1;
        uint32_t shift, mask;
        pass_field(a, p, shift, mask);
        const auto ki = mgpu::to_global(s.keys[in]);
        const auto ko = mgpu::to_global(s.keys[out]);
        if (tid < (uint32_t)RADIX) sh.run[tid] = sh.base[p][tid];
        for (uint32_t tb = 0; tb < n; tb += TILE) {
            for (uint32_t i = tid; i < (uint32_t)(W * (RADIX + 4)); i += BLOCK) (&sh.count[0][0])[i] = 0;
            __syncthreads();
            clear_match(a, sh, lane, wave);
            uint32_t key[IPT], rank[IPT], pos[IPT], dest[IPT];
            const uint32_t wb = tb + wave * 64 * IPT;
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                const uint32_t i = wb + j * 64 + lane;
                if (i < n) {
                    key[j] = ki[i];
                    rank[j] = seg_rank((key[j] >> shift) & mask, lane, sh.count[wave],
                                       match_table(sh, wave), a.rank1 != 0);
                }
            }
            __syncthreads();
            uint32_t total = 0;
            if (tid < (uint32_t)RADIX) {
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    uint32_t c = sh.count[w][tid];
                    sh.count[w][tid] = total;
                    total += c;
                }
            }
            const uint32_t start = block_exclusive_scan<BLOCK>(total, sh.tmp, lane, wave);
            if (tid < (uint32_t)RADIX) {
#pragma unroll
                for (int w = 0; w < W; ++w) sh.count[w][tid] += start;
                sh.dst[tid] = sh.run[tid] - start;
                sh.run[tid] += total;
            }
            __syncthreads();
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                const uint32_t i = wb + j * 64 + lane;
                if (i < n) {
                    pos[j] = sh.count[wave][(key[j] >> shift) & mask] + rank[j];
                    st[pos[j]] = key[j];
                }
            }
            __syncthreads();
            const uint32_t valid = min(TILE, n - tb);
#pragma unroll
            for (int j = 0; j < IPT; ++j) {
                const uint32_t q = j * BLOCK + tid;
                dest[j] = n;
                if (q < valid) {
                    const uint32_t k = st[q];
                    dest[j] = sh.dst[(k >> shift) & mask] + q;
                    if (dest[j] < n) ko[dest[j]] = k;
                    else mgpu::set_error(a.error_flag, 4u);
                }
            }
            for (uint32_t v = 0; v < nv; ++v) {
                const bool gen = a.index_mode && p == 0;
                const auto vi = mgpu::to_global(s.vals[v][in]);
                uint32_t val[IPT];
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const uint32_t i = wb + j * 64 + lane;
                    if (i < n) val[j] = gen ? i : vi[i];
                }
                __syncthreads();
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const uint32_t i = wb + j * 64 + lane;
                    if (i < n) st[pos[j]] = val[j];
                }
                __syncthreads();
                const auto vo = mgpu::to_global(s.vals[v][out]);
#pragma unroll
                for (int j = 0; j < IPT; ++j) {
                    const uint32_t q = j * BLOCK + tid;
                    if (q < valid && dest[j] < n) vo[dest[j]] = st[q];
                }
            }
            __syncthreads();
        }
        // This pass's stores must be seen by the next pass's loads of the
        // same workgroup (the L1 may hold lines read two passes ago).
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "agent");
        __syncthreads();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "agent");
    }

    // The result is on side (np & 1); move it when the launch wants the other.
    if ((np & 1) != a.result_side) {
        const uint32_t from = np & 1, to = a.result_side;
        const auto kt = mgpu::to_global(s.keys[to]);
        const auto kf = mgpu::to_global(s.keys[from]);
        for (uint32_t i = tid; i < n; i += BLOCK) kt[i] = kf[i];
        for (uint32_t v = 0; v < nv; ++v)
            for (uint32_t i = tid; i < n; i += BLOCK)
                mgpu::to_global(s.vals[v][to])[i] = mgpu::to_global(s.vals[v][from])[i];
    }
}

// ---- 8-bit digits ranked by ordered LDS adds --------------------------------
// (What the shipped table's kernels run; the routines above serve the other
// digit widths and the match-mask ranking.)
//
// Bound by LDS round trips and, in the small list, by the chain of reads from
// a list entry to its keys: a batch's bytes pass in a few microseconds.  So
// the ranks of all slots are requested before the first is used, keys and
// payloads lie in 32-bit words of their own, a segment takes no more slots per
// thread than it fills, and the small list's reads run ahead of the sorts.
// Plan replays, the routines above -> these (with one cursor for all
// workgroups), keys only / key + value / two values, us: 60000 segments log-uniform in [1, 512] 109 -> 75 / 123 -> 85 /
// 135 -> 95; 130000 in [1, 64] 143 -> 85 / 162 -> 98 / 186 -> 112; 20000 in
// [64, 4096] 297 -> 186 / 357 -> 214 / 411 -> 261; 5000 of 512 105 -> 72 /
// 125 -> 79 / 134 -> 85.

using mgpu::ConstDesc;
using mgpu::ConstWords;

// A segment's arrays, read through the constant address space.
struct SegArrays {
    const uint32_t *ki, *vi;  // keys and the first values, input side
    uint32_t *ko, *vo;        // result side
    uint32_t seg, n;
};

__device__ __forceinline__ SegArrays seg_arrays(const mgpuSegArgs& a, uint32_t seg) {
    const ConstDesc d = (ConstDesc)(a.segs + seg);
    SegArrays s;
    s.ki = d->keys[0];
    s.ko = a.result_side ? d->keys[1] : d->keys[0];
    s.vi = d->vals[0][0];
    s.vo = a.result_side ? d->vals[0][1] : d->vals[0][0];
    s.seg = seg;
    s.n = d->n;
    return s;
}
__device__ __forceinline__ const uint32_t* seg_vals_in(const mgpuSegArgs& a, const SegArrays& s, uint32_t v) {
    return ((ConstDesc)(a.segs + s.seg))->vals[v][0];
}
__device__ __forceinline__ uint32_t* seg_vals_out(const mgpuSegArgs& a, const SegArrays& s, uint32_t v) {
    return ((ConstDesc)(a.segs + s.seg))->vals[v][a.result_side];
}

// The same for local_sort_items.
struct SegIO {
    const mgpuSegArgs& a;
    const SegArrays& s;
    __device__ __forceinline__ const uint32_t* keys_in() const { return s.ki; }
    __device__ __forceinline__ uint32_t* keys_out() const { return s.ko; }
    __device__ __forceinline__ const uint32_t* vals_in(uint32_t v) const { return seg_vals_in(a, s, v); }
    __device__ __forceinline__ uint32_t* vals_out(uint32_t v) const { return seg_vals_out(a, s, v); }
    __device__ __forceinline__ uint32_t mode() const {
        return a.index_mode          ? MGPU_VALUES_INDEX
               : a.num_values == 1   ? MGPU_VALUES_SINGLE
                                     : MGPU_VALUES_MULTI;
    }
    __device__ __forceinline__ uint32_t num_values() const { return a.num_values; }
    __device__ __forceinline__ uint32_t read(uint32_t k) const { return k; }
    __device__ __forceinline__ uint32_t write(uint32_t k) const { return k; }
};

// One wave, at most 64 keys, one per lane: a key's place is the number of keys
// before it in the stable order, counted against each key in turn (a scalar
// broadcast, two compares and an add with carry).  No LDS, no dependence on
// the sort's width, and the work is n steps where a bitonic network takes 21
// of two LDS shuffles whatever n.  Every store goes straight to its place.
__device__ __forceinline__ void wave_place64(const mgpuSegArgs& a, const SegArrays& s, uint32_t lane,
                                             uint32_t key, uint32_t pay) {
    const uint32_t n = s.n;
    const uint32_t f = lane < n ? (a.num_bits >= 32 ? key : __builtin_amdgcn_ubfe(key, a.first_bit, a.num_bits))
                                : 0xFFFFFFFFu;
    uint32_t place = 0;
    for (uint32_t j = 0; j < n; j += 4) {
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) {
            // (Lanes past n hold all ones and lie after every key: counting
            // against them changes nothing.)
            const uint32_t o = (uint32_t)__builtin_amdgcn_readlane((int)f, (int)((j + i) & 63u));
            place += (o < f || (o == f && lane > j + i)) ? 1u : 0u;
        }
    }
    const uint32_t off = lane < n ? place * 4u : n * 4u;  // past the range: dropped
    __builtin_amdgcn_raw_buffer_store_b32(key, mgpu::words_rsrc(s.ko, n), (int)off, 0, 0);
    if (a.num_values == 0) return;
    if (a.index_mode || a.num_values == 1) {
        __builtin_amdgcn_raw_buffer_store_b32(a.index_mode ? lane : pay, mgpu::words_rsrc(s.vo, n),
                                              (int)off, 0, 0);
        return;
    }
    for (uint32_t v = 0; v < a.num_values; ++v) {
        const uint32_t val = __builtin_amdgcn_raw_buffer_load_b32(mgpu::words_rsrc(seg_vals_in(a, s, v), n),
                                                                  (int)(lane * 4u), 0, 0);
        __builtin_amdgcn_raw_buffer_store_b32(val, mgpu::words_rsrc(seg_vals_out(a, s, v), n), (int)off, 0, 0);
    }
}

// One wave, at most 64 * IT keys, in the wave's rows of the counts and the
// stage: no barriers.  Slots past n hold all ones, so they stay behind every
// key.  taken() is called once kin and pin have been read.
template <int IT, bool PAY, typename Taken>
__device__ __forceinline__ void wave_sort8(const mgpuSegArgs& a, const SegArrays& s, uint32_t* row,
                                           uint32_t* skey, uint32_t* spay, uint32_t lane,
                                           const uint32_t* kin, const uint32_t* pin, Taken taken) {
    const uint32_t n = s.n;
    uint32_t key[IT], pay[PAY ? IT : 1];
    // The slots that the caller has not read.
    uint32_t more_k[8] = {}, more_v[8] = {};
    if constexpr (IT > 8) {
        const __amdgpu_buffer_rsrc_t rk = mgpu::words_rsrc(s.ki, n);
#pragma unroll
        for (int j = 8; j < IT; ++j)
            more_k[j - 8] =
                __builtin_amdgcn_raw_buffer_load_b32(rk, (int)((j * 64 + lane) * 4u), 0, 0);
        if (PAY && !a.index_mode && a.num_values == 1) {
            const __amdgpu_buffer_rsrc_t rv = mgpu::words_rsrc(s.vi, n);
#pragma unroll
            for (int j = 8; j < IT; ++j)
                more_v[j - 8] =
                    __builtin_amdgcn_raw_buffer_load_b32(rv, (int)((j * 64 + lane) * 4u), 0, 0);
        }
    }
#pragma unroll
    for (int j = 0; j < IT; ++j) {
        key[j] = j * 64 + lane < n ? (j < 8 ? kin[j & 7] : more_k[j & 7]) : 0xFFFFFFFFu;
        if constexpr (PAY)
            pay[j] = a.index_mode || a.num_values > 1 ? j * 64 + lane
                     : j < 8                          ? pin[j & 7]
                                                      : more_v[j & 7];
    }
    taken();
    uint32_t shift = a.first_bit, left = a.num_bits;
    for (uint32_t p = 0; p < a.num_passes; ++p) {
        const uint32_t width = left / (a.num_passes - p);
        reinterpret_cast<uint4*>(row)[lane] = make_uint4(0u, 0u, 0u, 0u);
        uint32_t d[IT], pos[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) d[j] = __builtin_amdgcn_ubfe(key[j], shift, width);
        mgpu::rank_slots<IT>(d, row, lane, pos);
        wave_sync();
        const uint4 c = reinterpret_cast<const uint4*>(row)[lane];
        const uint32_t sum = c.x + c.y + c.z + c.w;
        const uint32_t at = mgpu::wave_inclusive_scan_dpp(sum) - sum;
        reinterpret_cast<uint4*>(row)[lane] =
            make_uint4(at, at + c.x, at + c.x + c.y, at + c.x + c.y + c.z);
        wave_sync();
#pragma unroll
        for (int j = 0; j < IT; ++j) pos[j] += row[d[j]];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            skey[pos[j]] = key[j];
            if constexpr (PAY) spay[pos[j]] = pay[j];
        }
        wave_sync();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            key[j] = skey[j * 64 + lane];
            if constexpr (PAY) pay[j] = spay[j * 64 + lane];
        }
        wave_sync();
        shift += width;
        left -= width;
    }
    const __amdgpu_buffer_rsrc_t rk = mgpu::words_rsrc(s.ko, n);
#pragma unroll
    for (int j = 0; j < IT; ++j)
        __builtin_amdgcn_raw_buffer_store_b32(key[j], rk, (int)((j * 64 + lane) * 4u), 0, 0);
    if constexpr (PAY) {
        if (a.index_mode || a.num_values == 1) {
            const __amdgpu_buffer_rsrc_t rv = mgpu::words_rsrc(s.vo, n);
#pragma unroll
            for (int j = 0; j < IT; ++j)
                __builtin_amdgcn_raw_buffer_store_b32(pay[j], rv, (int)((j * 64 + lane) * 4u), 0, 0);
            return;
        }
        for (uint32_t v = 0; v < a.num_values; ++v) {
            const __amdgpu_buffer_rsrc_t ri = mgpu::words_rsrc(seg_vals_in(a, s, v), n);
            const __amdgpu_buffer_rsrc_t ro = mgpu::words_rsrc(seg_vals_out(a, s, v), n);
            uint32_t val[IT];
#pragma unroll
            for (int j = 0; j < IT; ++j)
                val[j] = __builtin_amdgcn_raw_buffer_load_b32(ri, (int)(pay[j] * 4u), 0, 0);
            // Every gather has its data before the first store (the result
            // side may be the input side).
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll
            for (int j = 0; j < IT; ++j)
                __builtin_amdgcn_raw_buffer_store_b32(val[j], ro, (int)((j * 64 + lane) * 4u), 0, 0);
        }
    }
}

// One workgroup, with the least keys per thread that hold the segment.
template <int IPT, int BLOCK, bool PAY>
__device__ __forceinline__ void block_sort8(const mgpuSegArgs& a, const SegArrays& s,
                                            const mgpu::LocalMem& mem) {
    const SegIO io{a, s};
    const uint32_t n = s.n;
    if (n <= 2 * BLOCK) mgpu::local_sort_items<BLOCK, 2, PAY>(io, mem, n, 0u, a.first_bit, a.num_bits);
    else if (n <= 4 * BLOCK) mgpu::local_sort_items<BLOCK, 4, PAY>(io, mem, n, 0u, a.first_bit, a.num_bits);
    else if (n <= 6 * BLOCK) mgpu::local_sort_items<BLOCK, 6, PAY>(io, mem, n, 0u, a.first_bit, a.num_bits);
    else if (n <= 8 * BLOCK) mgpu::local_sort_items<BLOCK, 8, PAY>(io, mem, n, 0u, a.first_bit, a.num_bits);
    else if constexpr (IPT > 8) {
        if (n <= 12 * BLOCK) mgpu::local_sort_items<BLOCK, 12, PAY>(io, mem, n, 0u, a.first_bit, a.num_bits);
        else mgpu::local_sort_items<BLOCK, 16, PAY>(io, mem, n, 0u, a.first_bit, a.num_bits);
    }
}

// The small list, one segment per wave at a time, dealt round-robin over the
// grid's waves.  A wave's segments are a chain of dependent reads (list,
// descriptor, keys) and little else, so while one is sorted the next one's
// descriptor and keys are read, and the list entry of the one after.
template <int IPT, int BLOCK, bool PAY>
__device__ __forceinline__ void wave_phase8(const mgpuSegArgs& a, uint32_t* row, uint32_t* skey, uint32_t* spay,
                            uint32_t lane, uint32_t wave) {
    const uint32_t stride = gridDim.x * (BLOCK / 64);
    const ConstWords list = (ConstWords)a.small_list;
    uint32_t item = blockIdx.x * (BLOCK / 64) + wave;
    if (item >= a.num_small) return;
    const uint32_t last = a.num_small - 1;
    const bool value = PAY && !a.index_mode && a.num_values == 1;
    // (Of a segment of more than 512 keys the first 512: with all 16 slots the
    // kernel took 201 registers, one workgroup of 512 threads to a CU.)
    constexpr int AHEAD = 8;
    uint32_t key[AHEAD], pay[PAY ? AHEAD : 1];
    auto load = [&](const SegArrays& s) {
        const __amdgpu_buffer_rsrc_t rk = mgpu::words_rsrc(s.ki, s.n);
#pragma unroll
        for (int j = 0; j < AHEAD; ++j)
            if (j == 0 || s.n > j * 64u)
                key[j] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)((j * 64 + lane) * 4u), 0, 0);
        if constexpr (PAY) {
            if (value) {
                const __amdgpu_buffer_rsrc_t rv = mgpu::words_rsrc(s.vi, s.n);
#pragma unroll
                for (int j = 0; j < AHEAD; ++j)
                    if (j == 0 || s.n > j * 64u)
                        pay[j] = __builtin_amdgcn_raw_buffer_load_b32(
                            rv, (int)((j * 64 + lane) * 4u), 0, 0);
            }
        }
    };
    // (Past the end the last segment is read again and not used.)
    SegArrays cur = seg_arrays(a, list[item]);
    uint32_t ahead = list[min(item + stride, last)];
    load(cur);
    while (true) {
        const SegArrays next = seg_arrays(a, ahead);
        ahead = list[min(item + 2 * stride, last)];
        const bool more = item + stride < a.num_small;
        auto taken = [&] {
            if (more) load(next);
        };
        if (cur.n <= 64) {
            const uint32_t k = key[0], v = PAY ? pay[0] : 0u;
            taken();
            wave_place64(a, cur, lane, k, v);
        } else if (cur.n <= 128) {
            wave_sort8<2, PAY>(a, cur, row, skey, spay, lane, key, pay, taken);
        } else if (cur.n <= 256) {
            wave_sort8<4, PAY>(a, cur, row, skey, spay, lane, key, pay, taken);
        } else if (IPT == 8 || cur.n <= 512) {
            wave_sort8<8, PAY>(a, cur, row, skey, spay, lane, key, pay, taken);
        } else {
            wave_sort8<IPT, PAY>(a, cur, row, skey, spay, lane, key, pay, taken);
        }
        if (!more) break;
        item += stride;
        cur = next;
    }
}

// GLOBAL: the kernel carries the one-workgroup routine for segments larger
// than a workgroup's LDS tile.  That routine sets the kernel's register
// count (r8, 8 keys per thread, 512 threads: 149 VGPRs with it, 96 without), so
// launches whose block-list segments all fit the tile take the kernel
// without it, which fits more waves per SIMD.
template <int RB, int IPT, int BLOCK, bool GLOBAL>
__device__ __forceinline__ void segsort_body(const mgpuSegArgs& a) {
    static_assert(BLOCK >= (1 << RB), "a thread per digit in the block scans");
    constexpr int W = BLOCK / 64;
    __shared__ SegShared<RB, IPT, BLOCK> sh;
    const uint32_t tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;

    // 8-bit digits and the ordered adds: the routines written for them.
    const bool fast = RB == 8 && a.rank1 != 0;
    uint32_t* const words = reinterpret_cast<uint32_t*>(sh.stage);
    const mgpu::LocalMem mem{&sh.count[0][0], sh.tmp, words, words + SegShared<RB, IPT, BLOCK>::TILE};

    // Workgroup phase: block and global segments, largest first.  The first
    // of a workgroup is its own number; the others it draws from a counter of
    // its group (workgroups of the same number modulo the groups: with 8, of
    // one XCD), asked for before the segment at hand is sorted.  One counter
    // for all served a draw in ~25 ns, so 3000 segments of 4096 keys took the
    // 75 us of that queue and more, and every launch paid for counting its
    // workgroups out: plan replays, one counter -> these, keys only / key +
    // value, us: 3000 of 4096 125 -> 88 / 143 -> 106; 16000 in [1, 8192] 156 ->
    // 120 / 183 -> 138; 5000 of 512 (nothing drawn) 72 -> 46 / 79 -> 52; 60000
    // in [1, 512] 76 -> 63 / 85 -> 69.
    // (Dealt round-robin like the small ones below, they measured slower where
    // they are many: 20000 segments log-uniform in [2^6, 2^12] 0.44 -> 0.68
    // ms, since a workgroup that starts late still holds a full share.)
    const uint32_t groups = gridDim.x % MGPU_SEG_CURSORS == 0 ? MGPU_SEG_CURSORS : 1u;
    const uint32_t group = blockIdx.x % groups;
    uint32_t* const cursor = a.counters + group * MGPU_SEG_CURSOR_WORDS;
    const bool draws = a.num_big > gridDim.x;
    for (uint32_t item = blockIdx.x; item < a.num_big;) {
        uint32_t drawn = 0;
        if (draws && tid == 0)
            drawn = __hip_atomic_fetch_add(&cursor[0], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const mgpuSegDesc& s = a.segs[a.big_list[item]];
        if (fast && s.n <= (uint32_t)SegShared<RB, IPT, BLOCK>::TILE) {
            if constexpr (RB == 8) {
                const SegArrays io = seg_arrays(a, (uint32_t)__builtin_amdgcn_readfirstlane((int)a.big_list[item]));
                if (a.num_values == 0) block_sort8<IPT, BLOCK, false>(a, io, mem);
                else block_sort8<IPT, BLOCK, true>(a, io, mem);
            }
        } else if (s.n <= (uint32_t)SegShared<RB, IPT, BLOCK>::TILE) {
            block_sort<RB, IPT, BLOCK>(a, s, sh, tid, lane, wave);
        } else if constexpr (GLOBAL) {
            global_sort<RB, IPT, BLOCK>(a, s, sh, tid, lane, wave);
        } else if (tid == 0) {
            mgpu::set_error(a.error_flag, 7u);  // the host never sends one here
        }
        if (!draws) {
            __syncthreads();
            break;
        }
        if (tid == 0) sh.item = gridDim.x + drawn * groups + group;
        __syncthreads();
        item = (uint32_t)__builtin_amdgcn_readfirstlane((int)sh.item);
        __syncthreads();
    }

    if constexpr (RB == 8) {
        if (fast) {
            const uint32_t w = (uint32_t)__builtin_amdgcn_readfirstlane((int)wave);
            uint32_t* const slice = words + w * (2 * 64 * IPT);  // keys, then payloads
            if (a.num_values == 0)
                wave_phase8<IPT, BLOCK, false>(a, sh.count[w], slice, slice + 64 * IPT, lane, w);
            else
                wave_phase8<IPT, BLOCK, true>(a, sh.count[w], slice, slice + 64 * IPT, lane, w);
        }
    }
    // Wave phase: one small segment per wave at a time, dealt round-robin
    // over the grid's waves.  (A shared cursor costs a device-wide atomic on
    // one word per segment: ~25 ns each, serialized, which bounded a batch
    // of 130K segments of up to 64 keys at 3.3 ms whatever the kernel.)
    for (uint32_t item = fast ? a.num_small : blockIdx.x * W + wave; item < a.num_small;
         item += gridDim.x * W) {
        const mgpuSegDesc& s = a.segs[a.small_list[item]];
        if (s.n <= 64) wave_bitonic64(a, s, lane);
        else wave_sort<RB, IPT, BLOCK>(a, s, sh, lane, wave);
    }

    // The last of the group to be done drawing puts its cursor back.
    if (draws && tid == 0) {
        const uint32_t done =
            __hip_atomic_fetch_add(&cursor[1], 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (done == gridDim.x / groups - 1) {
            st_agent(&cursor[0], 0u);
            st_agent(&cursor[1], 0u);
        }
    }
}

}  // namespace

#define MGPU_SEG_SLOTS(B, TILE)                                                                \
    extern "C" __global__ void __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(4)))    \
        mgpu_seg_slots_b##B##_k(mgpuSegSlotArgs a) {                                            \
        __shared__ mgpu::LocalShared<B, TILE, false> sh;                                        \
        mgpu::sort_slot<B, TILE, false>(a, mgpu::local_mem(sh), blockIdx.x);                    \
    }                                                                                          \
    extern "C" __global__ void __launch_bounds__(B) __attribute__((amdgpu_waves_per_eu(4)))    \
        mgpu_seg_slots_b##B##_kv(mgpuSegSlotArgs a) {                                           \
        __shared__ mgpu::LocalShared<B, TILE, true> sh;                                         \
        mgpu::sort_slot<B, TILE, true>(a, mgpu::local_mem(sh), blockIdx.x);                     \
    }
MGPU_SEG_SLOTS(512, 8192)
MGPU_SEG_SLOTS(1024, 16384)

// Kernel variants: digit width RB (4..8 bits) x keys per thread IPT (8, 16)
// x workgroup size BLOCK (128 for digits up to 7 bits, 256, 512), each with
// the one-workgroup global-memory routine and without it (_ng).
// 512 threads: at most 96 registers with 8 keys per thread, so that two
// workgroups of a device-wide pass (80 registers, 42 KB) run beside one of
// this kernel on a CU instead of one; at most 128 with 16, so that two fit a
// CU (the LDS allows both).
#define MGPU_SEG_WAVES(IPT, B) \
    __attribute__((amdgpu_waves_per_eu(B < 512 ? 1 : IPT == 8 ? 5 : 4)))
#define MGPU_SEGSORT(RB, IPT, B)                                                                \
    extern "C" __global__ void __launch_bounds__(B)                                            \
        mgpu_segsort_r##RB##_i##IPT##_b##B(mgpuSegArgs a) {                                    \
        segsort_body<RB, IPT, B, true>(a);                                                     \
    }                                                                                          \
    extern "C" __global__ void __launch_bounds__(B) MGPU_SEG_WAVES(IPT, B)                        \
        mgpu_segsort_r##RB##_i##IPT##_b##B##_ng(mgpuSegArgs a) {                               \
        segsort_body<RB, IPT, B, false>(a);                                                    \
    }
#define MGPU_SEGSORT_BLOCKS(RB, IPT)                                                           \
    MGPU_SEGSORT(RB, IPT, 256)                                                                 \
    MGPU_SEGSORT(RB, IPT, 512)

MGPU_SEGSORT(4, 8, 128)
MGPU_SEGSORT(4, 16, 128)
MGPU_SEGSORT(5, 8, 128)
MGPU_SEGSORT(5, 16, 128)
MGPU_SEGSORT(6, 8, 128)
MGPU_SEGSORT(6, 16, 128)
MGPU_SEGSORT(7, 8, 128)
MGPU_SEGSORT(7, 16, 128)
MGPU_SEGSORT_BLOCKS(4, 8)
MGPU_SEGSORT_BLOCKS(4, 16)
MGPU_SEGSORT_BLOCKS(5, 8)
MGPU_SEGSORT_BLOCKS(5, 16)
MGPU_SEGSORT_BLOCKS(6, 8)
MGPU_SEGSORT_BLOCKS(6, 16)
MGPU_SEGSORT_BLOCKS(7, 8)
MGPU_SEGSORT_BLOCKS(7, 16)
MGPU_SEGSORT_BLOCKS(8, 8)
MGPU_SEGSORT_BLOCKS(8, 16)
