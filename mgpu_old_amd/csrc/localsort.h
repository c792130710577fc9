// Stable LSD sort of up to 16384 keys by one workgroup, all digit passes in
// registers and LDS: one launch and one read and write of the data, where the
// device-wide passes take a launch per pass.
//
// Bound: a pass is a chain of LDS round trips and four barriers, not
// bandwidth (16384 pairs are 256 KB): key + value, with the fill of the input,
// 1000 keys 34.6 -> 8.9 us a sort, 4096 36.3 -> 10.7, 16384 44.7 -> 23.7
// against the device-wide passes (a launch each, ~6 us whatever the size);
// keys only 32.5 -> 8.8, 33.4 -> 9.1, 39.0 -> 19.0.  So every slot's rank is
// requested before the first one is used, and the digit scan runs over all
// threads at once: thread (digit, group) adds the counts of four waves, and one
// scan over the threads in that order gives each wave's start of each digit
// directly.
#pragma once
#include "kernel_args.h"
#include "radix_device.h"

namespace mgpu {

constexpr int kLocalBlock = MGPU_LOCAL_THREADS;
constexpr uint32_t kLocalTile = MGPU_LOCAL_MAX_KEYS;
// Words from one wave's digit counts to the next: a multiple of 4 for 16-byte
// clearing, and not of 64, so that the scan's threads (digit, group of four
// waves) read different banks.
constexpr uint32_t kLocalRow = MGPU_RADIX + 4;

template <int BLOCK, uint32_t TILE, bool PAY>
struct LocalShared {
    uint32_t count[BLOCK / 64 * kLocalRow] __attribute__((aligned(16)));
    uint32_t tmp[BLOCK / 64];
    uint32_t key[TILE];
    uint32_t pay[PAY ? TILE : 1];
};

// The words of it a sort uses.
struct LocalMem {
    uint32_t *count, *tmp, *key, *pay;
};
template <int BLOCK, uint32_t TILE, bool PAY>
__device__ __forceinline__ LocalMem local_mem(LocalShared<BLOCK, TILE, PAY>& sh) {
    return {sh.count, sh.tmp, sh.key, sh.pay};
}

// Buffer resource over words [0, n) at p: loads past n return 0, stores there
// are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t words_rsrc(const uint32_t* p, uint32_t n) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint32_t*>(p), 0, (int)(n * 4u),
                                             0x00020000);
}

// Where a sort of a whole array or a bucket reads and writes (elements from
// `begin` of the arrays of `a`); the sorts below take any type with these
// members.
struct LocalArrays {
    const mgpuLocalArgs& a;
    uint32_t begin;
    __device__ __forceinline__ const uint32_t* keys_in() const { return a.keys_in + begin; }
    __device__ __forceinline__ uint32_t* keys_out() const { return a.keys_out + begin; }
    __device__ __forceinline__ const uint32_t* vals_in(uint32_t v) const { return a.vals_in[v] + begin; }
    __device__ __forceinline__ uint32_t* vals_out(uint32_t v) const { return a.vals_out[v] + begin; }
    __device__ __forceinline__ uint32_t mode() const { return a.vals_mode; }
    __device__ __forceinline__ uint32_t num_values() const { return a.num_values; }
    __device__ __forceinline__ uint32_t read(uint32_t k) const { return mgpu_key_map(k, a.in_lo, a.in_hi); }
    __device__ __forceinline__ uint32_t write(uint32_t k) const { return mgpu_key_map(k, a.out_lo, a.out_hi); }
};

// Sorts the n elements of `io`, 0 < n <= IT * BLOCK, by bits [shift0, shift0 +
// bits) of (key - base).  IT keys per thread: wave w holds keys w * 64 * IT +
// j * 64 + lane.  Slots past n hold all ones in every digit, so they stay
// behind every key.  MANY: whether io carries two or more values (-1: io.mode()
// says so).
template <int BLOCK, int IT, bool PAY, int MANY = -1, typename IO>
__device__ __forceinline__ void local_sort_items(const IO& io, const LocalMem& sh, uint32_t n, uint32_t base,
                                 uint32_t shift0, uint32_t bits) {
    constexpr uint32_t G = BLOCK / MGPU_RADIX;  // threads per digit in the scan
    static_assert(BLOCK % MGPU_RADIX == 0 && BLOCK / 64 == 4 * G,
                  "the scan gives a thread one digit of four waves");
    const uint32_t tid = threadIdx.x, lane = tid & 63;
    const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(tid >> 6));
    const uint32_t first = wave * 64 * IT + lane;  // this lane's key of slot 0
    const uint32_t off = first * 4u;
    const uint32_t fill = io.mode();
    uint32_t key[IT], pay[PAY ? IT : 1];
    {
        const __amdgpu_buffer_rsrc_t rk = words_rsrc(io.keys_in(), n);
#pragma unroll
        for (int j = 0; j < IT; ++j)
            key[j] = __builtin_amdgcn_raw_buffer_load_b32(rk, (int)(off + j * 256u), 0, 0);
        if constexpr (PAY) {
            if (MANY != 1 && fill == MGPU_VALUES_SINGLE) {
                const __amdgpu_buffer_rsrc_t rv = words_rsrc(io.vals_in(0), n);
#pragma unroll
                for (int j = 0; j < IT; ++j)
                    pay[j] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)(off + j * 256u), 0, 0);
            } else {
#pragma unroll
                for (int j = 0; j < IT; ++j) pay[j] = first + j * 64u;
            }
        }
    }
#pragma unroll
    for (int j = 0; j < IT; ++j)
        key[j] = first + j * 64u < n ? io.read(key[j]) - base : 0xFFFFFFFFu;

    uint32_t* const row = sh.count + wave * kLocalRow;
    const uint32_t dq = tid / G, g = tid % G;  // the scan's digit and group of waves
    uint32_t* const col = sh.count + g * 4 * kLocalRow + dq;
    const uint32_t passes = (bits + MGPU_RADIX_BITS - 1) / MGPU_RADIX_BITS;
    uint32_t shift = shift0, left = bits;
    for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t width = left / (passes - p);  // the narrower digits first
        // The wave's counts are its own between the scans: no barrier.
        reinterpret_cast<uint4*>(row)[lane] = make_uint4(0u, 0u, 0u, 0u);
        uint32_t d[IT], pos[IT];
#pragma unroll
        for (int j = 0; j < IT; ++j) d[j] = __builtin_amdgcn_ubfe(key[j], shift, width);
        rank_slots<IT>(d, row, lane, pos);
        __syncthreads();
        const uint32_t c0 = col[0], c1 = col[kLocalRow], c2 = col[2 * kLocalRow],
                       c3 = col[3 * kLocalRow];
        const uint32_t start =
            block_exclusive_scan_dpp<BLOCK>(c0 + c1 + c2 + c3, sh.tmp, lane, wave);
        col[0] = start;
        col[kLocalRow] = start + c0;
        col[2 * kLocalRow] = start + c0 + c1;
        col[3 * kLocalRow] = start + c0 + c1 + c2;
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) pos[j] += row[d[j]];
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            sh.key[pos[j]] = key[j];
            if constexpr (PAY) sh.pay[pos[j]] = pay[j];
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < IT; ++j) {
            key[j] = sh.key[first + j * 64];
            if constexpr (PAY) pay[j] = sh.pay[first + j * 64];
        }
        shift += width;
        left -= width;
    }
    // (No pass, as for a bucket of one value: the loads above still come
    // before every store.)
    if (passes == 0) {
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
    }

    // Every key and carried value was loaded before a barrier above, so the
    // output may be the input's buffers.
    {
        const __amdgpu_buffer_rsrc_t rk = words_rsrc(io.keys_out(), n);
#pragma unroll
        for (int j = 0; j < IT; ++j)
            __builtin_amdgcn_raw_buffer_store_b32(io.write(key[j] + base), rk,
                                                  (int)(off + j * 256u), 0, 0);
    }
    if constexpr (PAY) {
        if (MANY == 0 || (MANY < 0 && fill != MGPU_VALUES_MULTI)) {
            const __amdgpu_buffer_rsrc_t rv = words_rsrc(io.vals_out(0), n);
#pragma unroll
            for (int j = 0; j < IT; ++j)
                __builtin_amdgcn_raw_buffer_store_b32(pay[j], rv, (int)(off + j * 256u), 0, 0);
        } else if constexpr (MANY != 0) {
            // Two or more arrays, each through a stage in LDS: read in order,
            // taken in the keys' order, written in order, so that every global
            // access is whole lines.  Against a gather from global memory through
            // the source index, 16384 keys with six arrays: by 8 bits 50.9 -> 20.5
            // us (device-wide pass 23.0), by 32 bits 63.7 -> 33.4; 3 * 2^20 keys
            // with six in buckets 143.6 -> 120.3.  The two stages alternate:
            // one barrier an array, as a wave that writes a stage again has
            // passed the barrier that follows all reads of it.
            uint32_t val[IT];
            auto load = [&](uint32_t v) {
                const __amdgpu_buffer_rsrc_t rv = words_rsrc(io.vals_in(v), n);
#pragma unroll
                for (int j = 0; j < IT; ++j)
                    val[j] = __builtin_amdgcn_raw_buffer_load_b32(rv, (int)(off + j * 256u), 0, 0);
            };
            load(0);
            __syncthreads();  // the last pass's reads of the stages
            for (uint32_t v = 0; v < io.num_values(); ++v) {
                uint32_t* const stage = v & 1 ? sh.pay : sh.key;
#pragma unroll
                for (int j = 0; j < IT; ++j) stage[first + j * 64] = val[j];
                if (v + 1 < io.num_values()) load(v + 1);
                // Every wave has read this array before any writes it (the two
                // sides may be one buffer).
                __syncthreads();
                const __amdgpu_buffer_rsrc_t ro = words_rsrc(io.vals_out(v), n);
                uint32_t out[IT];
#pragma unroll
                for (int j = 0; j < IT; ++j) out[j] = stage[pay[j]];
#pragma unroll
                for (int j = 0; j < IT; ++j)
                    __builtin_amdgcn_raw_buffer_store_b32(out[j], ro, (int)(off + j * 256u), 0, 0);
            }
        }
    }
}

// The same with the least IT that holds n <= 16 * B elements.
template <bool PAY, int B = kLocalBlock, int MANY = -1, typename IO>
__device__ __forceinline__ void local_sort(const IO& io, const LocalMem& sh, uint32_t n,
                                           uint32_t base, uint32_t shift, uint32_t bits) {
    if (n <= 1 * B) local_sort_items<B, 1, PAY, MANY>(io, sh, n, base, shift, bits);
    else if (n <= 2 * B) local_sort_items<B, 2, PAY, MANY>(io, sh, n, base, shift, bits);
    else if (n <= 4 * B) local_sort_items<B, 4, PAY, MANY>(io, sh, n, base, shift, bits);
    else if (n <= 8 * B) local_sort_items<B, 8, PAY, MANY>(io, sh, n, base, shift, bits);
    else if (n <= 12 * B) local_sort_items<B, 12, PAY, MANY>(io, sh, n, base, shift, bits);
    else local_sort_items<B, 16, PAY, MANY>(io, sh, n, base, shift, bits);
}

// A segment's descriptor does not change while a kernel that sorts it runs, so
// it is read through the constant address space: scalar loads, once a wave.
typedef const __attribute__((address_space(4))) mgpuSegDesc* ConstDesc;
typedef const __attribute__((address_space(4))) uint32_t* ConstWords;

// A slot's elements for local_sort_items.
struct SlotIO {
    ConstDesc d;
    uint32_t begin, in, out, fill, values;
    __device__ __forceinline__ const uint32_t* keys_in() const { return d->keys[in] + begin; }
    __device__ __forceinline__ uint32_t* keys_out() const { return d->keys[out] + begin; }
    __device__ __forceinline__ const uint32_t* vals_in(uint32_t v) const { return d->vals[v][in] + begin; }
    __device__ __forceinline__ uint32_t* vals_out(uint32_t v) const { return d->vals[v][out] + begin; }
    __device__ __forceinline__ uint32_t mode() const { return fill; }
    __device__ __forceinline__ uint32_t num_values() const { return values; }
    __device__ __forceinline__ uint32_t read(uint32_t k) const { return k; }
    __device__ __forceinline__ uint32_t write(uint32_t k) const { return k; }
};

// A workgroup per bucket (read from side
// 1, where the one scatter left it) or whole segment.  Bound by LDS round trips
// and barriers as local_sort_items is (4096 segments log-uniform in [1, 2^16]:
// 23 M pairs at ~150 keys a nanosecond, 2.4 TB/s), so buckets are of a size
// that fits two workgroups on a CU: with 1024 threads and 11520 keys, one on a
// CU, that batch took 371 us in all instead of 329, keys only 298 instead of
// 239.
template <int BLOCK, uint32_t TILE, bool PAY>
__device__ __forceinline__ void sort_slot(const mgpuSegSlotArgs& a, const LocalMem& mem, uint32_t slot) {
    const uint32_t seg = a.slots[2 * slot], bucket = a.slots[2 * slot + 1];
    // (Known without a look at the segment: 512 segments in [2^15, 2^17] of
    // low-entropy pairs 830 -> 822 us, keys with two thirds in one digit 548 -> 538.)
    if (a.lsd_segments != nullptr && slot >= a.num_whole && *a.lsd_segments == a.num_wide) return;
    const uint32_t moved = a.num_values > 1 ? MGPU_VALUES_MULTI : MGPU_VALUES_SINGLE;
    SlotIO io{(ConstDesc)(a.segs + seg), 0u, 0u, a.result_side,
              a.index_mode ? MGPU_VALUES_INDEX : moved, a.num_values};
    uint32_t n, base = 0, bits = a.num_bits;
    if (bucket == MGPU_SLOT_WHOLE) {
        n = io.d->n;
    } else {
        io.d = (ConstDesc)(a.wide + seg);
        if (io.d->route == 0) return;
        const ConstWords at = (ConstWords)(a.digit_start + (size_t)seg * (MGPU_MAX_PASSES * MGPU_RADIX) +
                                           MGPU_RADIX + 4 * bucket);
        io.begin = at[0];
        io.in = 1;
        io.fill = moved;
        n = at[1];
        bits = at[2];
        base = at[3];
        if (n == 0) return;
    }
    if (n > TILE || io.begin > io.d->n || n > io.d->n - io.begin) {  // only from a broken plan
        if (threadIdx.x == 0) set_error(a.error_flag, 8u);
        return;
    }
    local_sort<PAY, BLOCK>(io, mem, n, base, a.first_bit, bits);
}

}  // namespace mgpu
