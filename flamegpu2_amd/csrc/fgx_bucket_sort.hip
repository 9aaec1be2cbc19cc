// Stable sort of a list's elements by bin, through LDS, for gfx950 (wave64).
//
//   count   per tile of the list: how many elements fall into each bucket of bins
//   prefix  per bucket: the elements of the tiles before
//   split   per tile: (bin within the bucket, element index) to the bucket, stably
//   sort    per bucket: stable order by bin in LDS, the bin starts, and every variable
//
// A list whose keys never fall from one element to the next (agents that stay in their bins) is
// copied by the split, and the sort has only the bins that no element begins left to write.
//
// Ranks are taken in list order (per-wave counters, and the lanes of a wave that share a
// key), so no pass depends on the order in which atomics land and none has to restore it.
// Lists of one tile are sorted by one block in one launch.
//
// What bounds it: from some 100,000 elements on, the gathers and stores of the last pass;
// below, the launches, of which there are four (the sort through global atomics takes
// seven).  1,048,576 messages of 28 bytes over 64^3 bins, in the order of the step before:
// 69.3 us with atomics, 52.6 us this way; 8,388,593 of 20 bytes in no order: 2,069 and 530 us;
// sort of 250,007 agents: 36.4 and 31.8 us.  Lists in order, 28 bytes, with atomics (which find
// them in order too), as any other list this way, and copied: 250,007 messages 24.7, 30.7 and
// 22.0 us, 1 M 38.6, 49.9 and 34.6, 4 M over 80,000 bins 72.8, 155 and 67; the two passes that find
// the order cost other lists up to 0.5 us.
#include "fgx_bucket_sort.h"

#include <algorithm>

namespace fgx {

constexpr uint32_t kMaxBuckets = 2048;     // per-wave 16-bit counters of a split: 64 KB for 16 waves

// How the last pass gets at a bucket's variables: from the whole list; from the bucket's place in
// the output arrays, where the split has moved them (see k_bucket_split); or, of a list whose
// keys never fall from one element to the next, from that same place in the list.
constexpr uint32_t kGather = 0u, kStage = 1u, kCopy = 2u;
constexpr uint32_t kDisorder = 1u << 31;   // of a tile: some element has a smaller key than the one before

struct BucketArgs {
    KeyArgs ka;
    const uint32_t* d_n;
    uint32_t n_cap;
    uint32_t shift, buckets, tiles, tile, bins;   // tile: elements a tile
    uint32_t piece_log;   // elements of a piece of an oversize bucket: 1 << piece_log, no fewer than a block sorts
    const float* x;
    const float* y;
    const float* z;
    uint32_t* rows;       // [pieces of oversize buckets][1 << shift] elements of each bin, or NULL: none of more than one piece
    uint32_t* counts;     // [tiles][buckets] elements; after the prefix pass those of the tiles before
    uint32_t* totals;     // [buckets] elements
    uint32_t* starts;     // [buckets + 1] first element
    uint32_t* met;        // [tiles] buckets that occur in the tile, and kDisorder
    uint32_t* edges;      // [tiles][2] first and last key; in the words of idx, which the split writes
    uint32_t* mode;       // how the list moves (kGather, kStage, kCopy); its elements; whether rows are counted
    uint32_t stage_above; // sum of `met` above which the split moves the variables; 0: never
    uint16_t* fine;       // bin within the bucket, in bucket order
    uint32_t* idx;        // element index, in bucket order
    uint32_t* start_out;  // bin starts, or NULL
};

__device__ __forceinline__ uint32_t key_of(const BucketArgs& a, uint32_t i) {
    return bin_key(a.ka, a.x[i], a.y[i], a.ka.dims == 3 ? a.z[i] : 0.0f);
}

// Exclusive sum over the block's threads (W waves); *total receives the block's sum.
template <uint32_t W>
__device__ __forceinline__ uint32_t block_prefix(uint32_t v, uint32_t* s_red, uint32_t* total) {
    const uint32_t w = threadIdx.x >> 6;
    // the opaque lane keeps the lanes' shuffle addresses from being shared between calls: held
    // over a whole kernel they are spilled
    uint32_t lane = lane_id(), incl = v;
    asm volatile("" : "+v"(lane));
#pragma unroll
    for (uint32_t o = 1; o < 64; o <<= 1) {
        const uint32_t b = (uint32_t)__builtin_amdgcn_ds_bpermute((int)((lane - o) << 2), (int)incl);
        incl += lane >= o ? b : 0u;
    }
    __syncthreads();   // s_red may still be read by the call before
    if (lane_id() == 63) s_red[w] = incl;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (uint32_t k = 0; k < W; ++k) {
        off += k < w ? s_red[k] : 0u;
        tot += s_red[k];
    }
    *total = tot;
    return off + incl - v;
}

// ---------------------------------------------------------------- stable split in LDS
// Elements are numbered (wave, chunk, lane); rows[w * keys + k] counts wave w's elements of
// key k in 16 bits (a wave holds at most 1,024).
__device__ __forceinline__ void split_count(uint16_t* rows, uint32_t row, uint32_t k) {
    const uint32_t at = row + k;
    atomicAdd(reinterpret_cast<uint32_t*>(rows) + (at >> 1), 1u << ((at & 1u) * 16u));
}

// After the counts: rows become each wave's first place within its key, s_start the keys'
// first places.  Thread t owns keys [t * q, t * q + q).
template <uint32_t W>
__device__ __forceinline__ void split_scan(uint16_t* rows, uint32_t stride, uint32_t keys, uint32_t* s_start,
                                           uint32_t* s_red) {
    const uint32_t q = (keys + W * 64u - 1u) / (W * 64u);
    const uint32_t k0 = threadIdx.x * q;
    uint32_t sum = 0;
    for (uint32_t j = 0; j < q && k0 + j < keys; ++j) {
        uint32_t c[W];
#pragma unroll
        for (uint32_t w = 0; w < W; ++w) c[w] = rows[w * stride + k0 + j];
        uint32_t run = 0;
#pragma unroll
        for (uint32_t w = 0; w < W; ++w) {
            rows[w * stride + k0 + j] = (uint16_t)run;
            run += c[w];
        }
        s_start[k0 + j] = run;
        sum += run;
    }
    uint32_t total;
    uint32_t base = block_prefix<W>(sum, s_red, &total);
    for (uint32_t j = 0; j < q && k0 + j < keys; ++j) {
        const uint32_t c = s_start[k0 + j];
        s_start[k0 + j] = base;
        base += c;
    }
    __syncthreads();
}

// The place of one element of the wave's next chunk.  Lanes with the same key take places in
// lane order; the last of them moves the wave's counter on (LDS runs a wave's accesses in
// program order, which `volatile` keeps).
__device__ __forceinline__ uint32_t split_place(uint16_t* s_rows, const uint32_t* s_start, uint32_t row, uint32_t k,
                                                bool valid, uint32_t bits) {
    volatile __attribute__((address_space(3))) uint16_t* rows = (__attribute__((address_space(3))) uint16_t*)s_rows;
    uint64_t same = __ballot(valid);
    for (uint32_t b = 0; b < bits; ++b) {
        const bool on = (k >> b) & 1u;
        const uint64_t m = __ballot(on);
        same &= on ? m : ~m;
    }
    if (!valid) return 0u;
    const uint32_t lane = lane_id();
    const uint32_t before = rows[row + k];
    const uint32_t place = s_start[k] + before + (uint32_t)__builtin_popcountll(same & ((1ull << lane) - 1ull));
    if (lane == 63u - (uint32_t)__builtin_clzll(same)) rows[row + k] = (uint16_t)(before + (uint32_t)__builtin_popcountll(same));
    return place;
}

__device__ __forceinline__ uint32_t key_bits(uint32_t keys) { return keys > 1u ? 32u - (uint32_t)__builtin_clz(keys - 1u) : 0u; }

template <uint32_t BT>
__device__ __forceinline__ void zero_rows(uint16_t* rows, uint32_t n) {
    for (uint32_t k = threadIdx.x; k < (n + 1u) / 2u; k += BT) reinterpret_cast<uint32_t*>(rows)[k] = 0u;
}

// The tiles of `size` elements that hold elements (at least one): only these are counted, summed
// and split, on all XCDs, whatever the capacity the launches are sized for (predator-prey, 1 M
// prey in lists about 40 % full, a launch on average: count 11.3 -> 7.4 us, prefix 7.8 -> 5.8,
// split 27.4 -> 15.6).
__device__ __forceinline__ uint32_t filled_tiles(uint32_t n, uint32_t size) {
    const uint32_t f = (__builtin_amdgcn_readfirstlane(n) + size - 1u) / size;
    return f ? f : 1u;
}

// A bucket of more than one piece of P = 1 << log elements (sort_piece) has a row of bin counts
// for each piece: that of the piece with the bucket's element e.  A bucket of m > P elements
// owns rows floor(2 first / P) on, ceil(m / P) <= floor(2 m / P) of them, so those of different
// buckets are apart and n elements need at most floor(2 n / P) rows.
__device__ __forceinline__ uint32_t piece_row(uint32_t first, uint32_t e, uint32_t log) { return (2u * first >> log) + (e >> log); }

// Adds 1 to rows[word] for each lane that is `on`: lanes with the same word as the first one
// left add together, four times over (few bins that hold much); the rest one by one.
__device__ __forceinline__ void count_in_row(uint32_t* rows, uint32_t word, bool on) {
    uint64_t left = __ballot(on);
    for (uint32_t r = 0; r < 4 && left; ++r) {
        const uint32_t lane = (uint32_t)__builtin_ctzll(left);
        const uint64_t same = __ballot(on && word == (uint32_t)__builtin_amdgcn_readlane((int)word, (int)lane));
        if (lane_id() == lane) atomicAdd(rows + word, (uint32_t)__builtin_popcountll(same));
        left &= ~same;
    }
    if ((left >> lane_id()) & 1ull) atomicAdd(rows + word, 1u);
}

// ---------------------------------------------------------------- count
template <uint32_t BT, uint32_t ITEMS>
__global__ void __launch_bounds__(BT) k_bucket_count(BucketArgs a) {
    constexpr uint32_t W = BT / 64u;
    __shared__ uint32_t s_hist[kMaxBuckets];
    __shared__ uint32_t s_met;
    __shared__ uint32_t s_first[W], s_last[W];   // first and last key of each wave
    const uint32_t t = threadIdx.x, w = t >> 6, lane = lane_id();
    const uint32_t n = load_count(a.d_n, a.n_cap);
    const uint32_t tile = xcd_filled_block(filled_tiles(n, BT * ITEMS));
    if (tile == kNoBlock) return;
    for (uint32_t b = t; b < a.buckets; b += BT) s_hist[b] = 0u;
    if (t == 0) s_met = 0u;
    if (t == 0 && tile == 0) a.mode[2] = 0u;
    __syncthreads();
    const uint32_t base = tile * BT * ITEMS;
    if (a.rows) {
        // this tile's share of the rows that n elements can need, for the split to count in
        const uint32_t words = (2u * n >> a.piece_log) << a.shift;
        const uint64_t share = (uint64_t)(2u * BT * ITEMS) << a.shift;
        const uint32_t w0 = (uint32_t)(tile * share >> a.piece_log), w1 = (uint32_t)((tile + 1u) * share >> a.piece_log);
        for (uint32_t k = w0 + t; k < w1 && k < words; k += BT) a.rows[k] = 0u;
    }
    // elements are numbered (wave, item, lane), so that nearly each one's predecessor is in its wave
    if (base < n) {
        const uint32_t e0 = base + w * ITEMS * 64u + lane;
        uint32_t k[ITEMS];
#pragma unroll
        for (uint32_t j = 0; j < ITEMS; ++j) k[j] = key_of(a, e0 + j * 64u < n ? e0 + j * 64u : base);
        uint32_t before = 0u;
        bool fell = false;
#pragma unroll
        for (uint32_t j = 0; j < ITEMS; ++j) {
            const bool on = e0 + j * 64u < n;
            // the key of the lane before (wave_shr:1); lane 0 keeps the item before's last
            const uint32_t p = (uint32_t)__builtin_amdgcn_update_dpp((int)before, (int)k[j], 0x138, 0xF, 0xF, false);
            const uint32_t b = k[j] >> a.shift;
            fell = fell || (on && k[j] < p);
            before = (uint32_t)__builtin_amdgcn_readlane((int)k[j], 63);
            // lanes with the first one's bucket add together: most do in a list nearly in order
            const bool with_first = b == __builtin_amdgcn_readfirstlane(b);
            const uint64_t same = __ballot(on && with_first);
            if (on && !with_first) atomicAdd(&s_hist[b], 1u);
            if (lane == 0 && same) atomicAdd(&s_hist[b], (uint32_t)__builtin_popcountll(same));
        }
        if (lane == 0) s_first[w] = k[0];
        if (lane == 0) s_last[w] = before;
        if (__ballot(fell) && lane == 0) atomicOr(&s_met, kDisorder);
    }
    __syncthreads();
    uint32_t met = 0;
    for (uint32_t b = t; b < a.buckets; b += BT) {
        const uint32_t c = s_hist[b];
        a.counts[(size_t)tile * a.buckets + b] = c;
        met += c ? 1u : 0u;
    }
    if (a.stage_above) {
        met = wave_sum_u32(met);
        if (lane == 0) atomicAdd(&s_met, met);
        __syncthreads();
    }
    if (t < 64u) {
        const bool fell = t && t < W && base + t * ITEMS * 64u < n && s_first[t] < s_last[t - 1u];
        const uint32_t any = __ballot(fell) ? kDisorder : 0u;
        if (t == 0) {
            a.met[tile] = s_met | any;
            a.edges[2u * tile] = s_first[0];
            a.edges[2u * tile + 1u] = s_last[W - 1u];
        }
    }
}

// ---------------------------------------------------------------- prefix
// Block g: buckets [64 g, 64 g + 64), one per lane; each of the 16 waves takes a run of the
// tiles, 8 loads in flight.  One block more finds out how the list moves.
__global__ void __launch_bounds__(1024) k_bucket_prefix(BucketArgs a) {
    __shared__ uint32_t s_sum[16][64];
    __shared__ uint32_t s_red[16];
    __shared__ uint32_t s_fell;
    const uint32_t lane = lane_id(), w = threadIdx.x >> 6;
    const uint32_t b = blockIdx.x * 64u + lane;
    const uint32_t n = load_count(a.d_n, a.n_cap), tiles = filled_tiles(n, a.tile);
    if (blockIdx.x * 64u >= a.buckets) {
        uint32_t met = 0, fell = 0, all = 0;
        if (threadIdx.x == 0) s_fell = 0u;
        for (uint32_t t = threadIdx.x; t < tiles; t += 1024u) {
            const uint32_t m = a.met[t];
            met += m & ~kDisorder;
            fell |= t && a.edges[2u * t] < a.edges[2u * t - 1u] ? kDisorder : m;
        }
        __syncthreads();
        if (fell & kDisorder) s_fell = 1u;
        block_prefix<16>(met, s_red, &all);
        if (threadIdx.x == 0) {
            a.mode[0] = !s_fell ? kCopy : (a.stage_above && all > a.stage_above ? kStage : kGather);
            a.mode[1] = n;
        }
        return;
    }
    const uint32_t per = (tiles + 15u) / 16u;
    const uint32_t t0 = w * per < tiles ? w * per : tiles, t1 = t0 + per < tiles ? t0 + per : tiles;
    const bool on = b < a.buckets;
    uint32_t sum = 0;
    for (uint32_t t = t0; t < t1; t += 8u) {
        uint32_t c[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) c[j] = on && t + j < t1 ? a.counts[(size_t)(t + j) * a.buckets + b] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) sum += c[j];
    }
    s_sum[w][lane] = sum;
    __syncthreads();
    uint32_t run = 0, total = 0;
#pragma unroll
    for (uint32_t k = 0; k < 16; ++k) {
        run += k < w ? s_sum[k][lane] : 0u;
        total += s_sum[k][lane];
    }
    for (uint32_t t = t0; t < t1; t += 8u) {
        uint32_t c[8];
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) c[j] = on && t + j < t1 ? a.counts[(size_t)(t + j) * a.buckets + b] : 0u;
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            if (on && t + j < t1) a.counts[(size_t)(t + j) * a.buckets + b] = run;
            run += c[j];
        }
    }
    if (w == 0 && on) {
        a.totals[b] = total;
        if (a.rows && total > 1u << a.piece_log) a.mode[2] = 1u;
    }
}

// ---------------------------------------------------------------- lists in order
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// Elements [lo, hi) of every variable to the same places: 16 bytes a load, four variables in
// flight.  lo is a multiple of 16, so the ranges start on 16 bytes where the arrays do.
template <uint32_t BT>
__device__ __forceinline__ void copy_range(const VarTable& vt, uint32_t lo, uint32_t hi) {
    constexpr uint32_t V = 4;
    const uint32_t t = threadIdx.x, even = lo + ((hi - lo) & ~15u);
    for (uint32_t v0 = 0; v0 < vt.n; v0 += V) {
        const u32x4* in[V];
        u32x4* out[V];
        uint32_t len[V], most = 0;
#pragma unroll
        for (uint32_t k = 0; k < V; ++k) {
            const uint32_t v = v0 + k < vt.n ? v0 + k : v0, b = vt.bytes[v];
            const char* i = vt.in[v] + (size_t)lo * b;
            char* o = vt.out[v] + (size_t)lo * b;
            const bool aligned = (((uintptr_t)i | (uintptr_t)o) & 15u) == 0u;
            in[k] = reinterpret_cast<const u32x4*>(i);
            out[k] = reinterpret_cast<u32x4*>(o);
            len[k] = aligned && v0 + k < vt.n ? (even - lo) / 16u * b : 0u;
            most = len[k] > most ? len[k] : most;
            if (!aligned && v0 + k < vt.n)
                for (uint32_t e = lo + t; e < even; e += BT) copy_var(vt, v, e, e);
        }
        for (uint32_t c = t; c < most; c += BT) {
            u32x4 x[V];
#pragma unroll
            for (uint32_t k = 0; k < V; ++k)
                if (c < len[k]) x[k] = in[k][c];
#pragma unroll
            for (uint32_t k = 0; k < V; ++k)
                if (c < len[k]) out[k][c] = x[k];
        }
    }
    if (even + t < hi) copy_element(vt, even + t, even + t);   // the list's last few
    for (uint32_t e = lo + t; e < hi; e += BT) write_record(vt, e, e);
}

// Elements [lo, hi) of a list in order, lo a multiple of 16: the copy, and the starts of the bins
// of which they are the first, or of the empty bins before, as far as the element's bucket
// goes (end_bucket writes the others).
template <uint32_t BT>
__device__ __forceinline__ void copy_in_order(const BucketArgs& a, const VarTable& vt, uint32_t lo, uint32_t hi) {
    if (a.start_out) {
        for (uint32_t e = lo + threadIdx.x; e < hi; e += BT) {
            const uint32_t k = key_of(a, e), low = k >> a.shift << a.shift;
            uint32_t p = __shfl_up(k, 1, 64);
            if (lane_id() == 0 && e) p = key_of(a, e - 1u);
            for (uint32_t j = e && p >= low ? p + 1u : low; j <= k; ++j) a.start_out[j] = e;
        }
    }
    copy_range<BT>(vt, lo, hi);
}

// ---------------------------------------------------------------- split
// A tile's elements in bucket order are laid out in LDS first, so that the stores to each
// bucket are runs.  When the list is in no order (a tile meets so many buckets that its
// elements of one are fewer than a cache line's worth), the variables move with the split,
// to the bucket's place in the output arrays: the last pass then permutes each bucket in
// place, where it would otherwise gather every element's line of every variable from the
// whole list.
template <uint32_t BT, uint32_t ITEMS, uint32_t MAXB>
__global__ void __launch_bounds__(BT) k_bucket_split(BucketArgs a, VarTable vt) {
    constexpr uint32_t W = BT / 64u, T = BT * ITEMS;
    __shared__ alignas(16) uint16_t s_rows[W * MAXB];
    __shared__ uint32_t s_start[MAXB];
    __shared__ uint32_t s_delta[MAXB];
    __shared__ uint32_t s_big[MAXB];   // if any: first element of a bucket of more than one piece, or kNoBlock
    __shared__ uint32_t s_key[T];
    __shared__ uint16_t s_loc[T];
    __shared__ uint32_t s_red[W];
    const uint32_t t = threadIdx.x, w = t >> 6, lane = lane_id();
    const uint32_t mode = a.mode[0], n = a.mode[1], any = a.mode[2], nb = a.buckets;
    const uint32_t tile = xcd_filled_block(filled_tiles(n, T));
    if (tile == kNoBlock) return;
    const uint32_t base = tile * T;
    const uint32_t cnt = base < n ? (n - base < T ? n - base : T) : 0u;
    // this thread's buckets: their totals and the tile's offsets are loaded beside the positions
    constexpr uint32_t Q = MAXB / BT;
    const uint32_t q = (nb + BT - 1u) / BT, b0 = t * q;
    if (mode == kCopy) {
        copy_in_order<BT>(a, vt, base, base + cnt);
        if (tile) return;
        uint32_t sum = 0, total;
        for (uint32_t j = 0; j < q && b0 + j < nb; ++j) sum += a.totals[b0 + j];
        uint32_t run = block_prefix<W>(sum, s_red, &total);
        for (uint32_t j = 0; j < q && b0 + j < nb; ++j) {
            a.starts[b0 + j] = run;
            run += a.totals[b0 + j];
        }
        if (t == 0) a.starts[nb] = total;
        return;
    }
    uint32_t total_of[Q], offset_of[Q];
#pragma unroll
    for (uint32_t j = 0; j < Q; ++j) {
        const bool on = j < q && b0 + j < nb;
        total_of[j] = on ? a.totals[b0 + j] : 0u;
        offset_of[j] = on ? a.counts[(size_t)tile * nb + b0 + j] : 0u;
    }
    uint32_t key[ITEMS];
#pragma unroll
    for (uint32_t c = 0; c < ITEMS; ++c) {
        const uint32_t e = (w * ITEMS + c) * 64u + lane;
        key[c] = cnt ? key_of(a, base + (e < cnt ? e : 0u)) : 0u;
    }
    zero_rows<BT>(s_rows, W * nb);
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < ITEMS; ++c)
        if ((w * ITEMS + c) * 64u + lane < cnt) split_count(s_rows, w * nb, key[c] >> a.shift);
    __syncthreads();
    split_scan<W>(s_rows, nb, nb, s_start, s_red);
    // where the tile's elements of each bucket go: the bucket's start + those of the tiles before
    {
        uint32_t sum = 0, total;
#pragma unroll
        for (uint32_t j = 0; j < Q; ++j) sum += total_of[j];
        uint32_t run = block_prefix<W>(sum, s_red, &total);
#pragma unroll
        for (uint32_t j = 0; j < Q; ++j) {
            if (j >= q || b0 + j >= nb) continue;
            s_delta[b0 + j] = run + offset_of[j] - s_start[b0 + j];
            if (tile == 0) a.starts[b0 + j] = run;
            run += total_of[j];
        }
        if (tile == 0 && t == 0) a.starts[nb] = total;
    }
    const uint32_t bits = key_bits(nb);
#pragma unroll
    for (uint32_t c = 0; c < ITEMS; ++c) {
        const uint32_t e = (w * ITEMS + c) * 64u + lane;
        const bool valid = e < cnt;
        const uint32_t p = split_place(s_rows, s_start, w * nb, key[c] >> a.shift, valid, bits);
        if (valid) {
            s_key[p] = key[c];
            s_loc[p] = (uint16_t)e;
        }
    }
    __syncthreads();
    const uint32_t mask = (1u << a.shift) - 1u;
    if (any) {
#pragma unroll
        for (uint32_t j = 0; j < Q; ++j) {
            if (j >= q || b0 + j >= nb) continue;
            const uint32_t first = s_delta[b0 + j] + s_start[b0 + j] - offset_of[j];
            s_big[b0 + j] = total_of[j] > 1u << a.piece_log ? first : kNoBlock;
        }
        __syncthreads();
    }
    uint32_t src[ITEMS], dst[ITEMS];
#pragma unroll
    for (uint32_t j = 0; j < ITEMS; ++j) {
        const uint32_t p = j * BT + t;
        src[j] = dst[j] = 0u;
        if (p < cnt) {
            const uint32_t k = s_key[p];
            dst[j] = s_delta[k >> a.shift] + p;
            src[j] = base + s_loc[p];
            a.fine[dst[j]] = (uint16_t)(k & mask);
            a.idx[dst[j]] = src[j];
            if (any) {
                const uint32_t first = s_big[k >> a.shift];
                count_in_row(a.rows, (piece_row(first, dst[j] - first, a.piece_log) << a.shift) + (k & mask), first != kNoBlock);
            }
        }
    }
    if (mode != kStage) return;
    for (uint32_t v = 0; v < vt.n; ++v) {
        if (vt.bytes[v] == 4) {
            const uint32_t* in = reinterpret_cast<const uint32_t*>(vt.in[v]);
            uint32_t* out = reinterpret_cast<uint32_t*>(vt.out[v]);
            uint32_t x[ITEMS];
#pragma unroll
            for (uint32_t j = 0; j < ITEMS; ++j)
                if (j * BT + t < cnt) x[j] = in[src[j]];
#pragma unroll
            for (uint32_t j = 0; j < ITEMS; ++j)
                if (j * BT + t < cnt) out[dst[j]] = x[j];
        } else {
            for (uint32_t j = 0; j < ITEMS; ++j)
                if (j * BT + t < cnt) copy_var(vt, v, src[j], dst[j]);
        }
    }
}

// ---------------------------------------------------------------- sort within a bucket
// Copies m elements, the p-th from input element place.src(p) to output element place.dst(p).
// Two of them and up to eight 4-byte variables per thread are loaded before the first store.
template <uint32_t BT, uint32_t V, typename Place>
__device__ __forceinline__ void write_elements(const VarTable& vt, uint32_t m, Place place) {
    constexpr uint32_t P = 2;
    for (uint32_t p0 = threadIdx.x; p0 < m; p0 += P * BT) {
        uint32_t e[P];
        bool on[P];
#pragma unroll
        for (uint32_t j = 0; j < P; ++j) {
            const uint32_t p = p0 + j * BT;
            on[j] = p < m;
            e[j] = on[j] ? place.src(p) : 0u;
        }
        uint32_t r[4][P] = {};
        for (uint32_t v0 = 0; v0 < vt.n; v0 += V) {
            uint32_t x[V][P];
#pragma unroll
            for (uint32_t k = 0; k < V; ++k) {
                if (v0 + k >= vt.n || vt.bytes[v0 + k] != 4) continue;
                const uint32_t* src = reinterpret_cast<const uint32_t*>(vt.in[v0 + k]);
#pragma unroll
                for (uint32_t j = 0; j < P; ++j)
                    if (on[j]) x[k][j] = src[e[j]];
            }
#pragma unroll
            for (uint32_t k = 0; k < V; ++k) {
                if (v0 + k >= vt.n) continue;
                if (vt.bytes[v0 + k] == 4) {
                    uint32_t* out = reinterpret_cast<uint32_t*>(vt.out[v0 + k]);
#pragma unroll
                    for (uint32_t j = 0; j < P; ++j)
                        if (on[j]) out[place.dst(p0 + j * BT)] = x[k][j];
                    // the record's words are variables just loaded (a second gather of four words
                    // cost as much as four variables: 29.1 against 23.5 us for 1 M messages)
#pragma unroll
                    for (uint32_t c = 0; c < 4; ++c) {
                        if (vt.rec_var[c] != (int32_t)(v0 + k)) continue;
#pragma unroll
                        for (uint32_t j = 0; j < P; ++j) r[c][j] = x[k][j];
                    }
                } else {
                    for (uint32_t j = 0; j < P; ++j)
                        if (on[j]) copy_var(vt, v0 + k, e[j], place.dst(p0 + j * BT));
                }
            }
        }
        if (vt.rec) {
#pragma unroll
            for (uint32_t j = 0; j < P; ++j)
                if (on[j]) reinterpret_cast<uint4*>(vt.rec)[place.dst(p0 + j * BT)] = make_uint4(r[0][j], r[1][j], r[2][j], r[3][j]);
        }
    }
}

// Output elements first + [0, m): place p takes input element s_src[p] (or in[first + p] when
// s_src is NULL).
struct SortedPlace {
    const uint32_t* s_src;
    const uint32_t* in;
    uint32_t first;
    __device__ __forceinline__ uint32_t src(uint32_t p) const { return s_src ? s_src[p] : in[first + p]; }
    __device__ __forceinline__ uint32_t dst(uint32_t p) const { return first + p; }
};
template <uint32_t BT>
__device__ __forceinline__ void write_sorted(const VarTable& vt, const uint32_t* s_src, const uint32_t* in, uint32_t first,
                                             uint32_t m) {
    write_elements<BT, 8>(vt, m, SortedPlace{s_src, in, first});
}

// The same for a bucket whose variables the split has moved to the output arrays already: place
// p takes element first + s_src[p] of the output arrays, so all of a variable's m <= S * BT
// elements are read before the first of them is written.
template <uint32_t BT, uint32_t S>
__device__ __forceinline__ void permute_sorted(const VarTable& vt, const uint32_t* s_src, uint32_t first, uint32_t m) {
    const uint32_t t = threadIdx.x;
    uint32_t e[S];
#pragma unroll
    for (uint32_t j = 0; j < S; ++j) e[j] = first + (j * BT + t < m ? s_src[j * BT + t] : 0u);
    if (vt.rec) {
#pragma unroll
        for (uint32_t j0 = 0; j0 < S; j0 += 2) {
            uint32_t r[4][2];
#pragma unroll
            for (uint32_t k = 0; k < 4; ++k) {
                const int32_t v = vt.rec_var[k];
#pragma unroll
                for (uint32_t j = 0; j < 2; ++j)
                    r[k][j] = v >= 0 && (j0 + j) * BT + t < m
                                  ? reinterpret_cast<const uint32_t*>(vt.out[v < 0 ? 0 : v])[e[j0 + j]] : 0u;
            }
#pragma unroll
            for (uint32_t j = 0; j < 2; ++j)
                if ((j0 + j) * BT + t < m)
                    reinterpret_cast<uint4*>(vt.rec)[first + (j0 + j) * BT + t] = make_uint4(r[0][j], r[1][j], r[2][j], r[3][j]);
        }
        __syncthreads();   // the records are read from arrays that are permuted next
    }
    for (uint32_t v = 0; v < vt.n; ++v) {
        // elements of any size move as words, or as bytes: piece by piece, each of them read by
        // every thread before any is written
        const uint32_t b = vt.bytes[v], step = (b & 3u) ? 1u : 4u;
        for (uint32_t at = 0; at < b; at += step) {
            uint32_t x[S];
#pragma unroll
            for (uint32_t j = 0; j < S; ++j) {
                x[j] = 0u;
                if (j * BT + t >= m) continue;
                const char* s = vt.out[v] + (size_t)e[j] * b + at;
                x[j] = step == 4 ? *reinterpret_cast<const uint32_t*>(s) : (uint32_t)*reinterpret_cast<const uint8_t*>(s);
            }
            // every load is back before any thread stores: the loaded values are used here
#pragma unroll
            for (uint32_t j = 0; j < S; ++j) asm volatile("" ::"v"(x[j]));
            __syncthreads();
#pragma unroll
            for (uint32_t j = 0; j < S; ++j) {
                if (j * BT + t >= m) continue;
                char* d = vt.out[v] + (size_t)(first + j * BT + t) * b + at;
                if (step == 4) *reinterpret_cast<uint32_t*>(d) = x[j];
                else *reinterpret_cast<uint8_t*>(d) = (uint8_t)x[j];
            }
        }
    }
}

// LDS of one sorting block: the split's counters (in a piece of an oversize bucket, after them,
// the output element of each place), the bins' first places, the source of each place.
template <uint32_t BT, uint32_t MAXF, uint32_t S>
struct SortLds {
    static constexpr uint32_t kCap = BT * S;   // S elements per thread
    static constexpr uint32_t kRowWords = (BT / 64u) * MAXF / 2u;
    uint32_t rows[kRowWords > kCap ? kRowWords : kCap];
    uint32_t start[MAXF];
    uint32_t dest[MAXF];   // oversize buckets: where a piece's elements of each bin go
    uint32_t src[kCap];
    uint32_t red[BT / 64u];
    uint32_t lo, hi;
};

// Elements (f[c], id[c]) of chunk c < cw of each wave, m in all, numbered (wave, chunk, lane):
// s.src[place] = id in stable order by f, s.start[f] = first place.
template <uint32_t BT, uint32_t MAXF, uint32_t S, uint32_t C>
__device__ __forceinline__ void sort_in_lds(SortLds<BT, MAXF, S>& s, uint32_t keys, const uint32_t (&f)[C],
                                            const uint32_t (&id)[C], uint32_t cw, uint32_t m) {
    constexpr uint32_t W = BT / 64u;
    const uint32_t w = threadIdx.x >> 6, lane = lane_id();
    uint16_t* rows = reinterpret_cast<uint16_t*>(s.rows);
    const uint32_t stride = (keys + 1u) & ~1u;
    zero_rows<BT>(rows, W * stride);
    __syncthreads();
#pragma unroll
    for (uint32_t c = 0; c < C; ++c)
        if (c < cw && (w * cw + c) * 64u + lane < m) split_count(rows, w * stride, f[c]);
    __syncthreads();
    split_scan<W>(rows, stride, keys, s.start, s.red);
    const uint32_t bits = key_bits(keys);
#pragma unroll
    for (uint32_t c = 0; c < C; ++c) {
        if (c >= cw) continue;
        const bool valid = (w * cw + c) * 64u + lane < m;
        const uint32_t p = split_place(rows, s.start, w * stride, f[c], valid, bits);
        if (valid) s.src[p] = id[c];
    }
    __syncthreads();
}

struct PiecePlace {
    const uint32_t* s_src;
    const uint32_t* s_dst;
    __device__ __forceinline__ uint32_t src(uint32_t p) const { return s_src[p]; }
    __device__ __forceinline__ uint32_t dst(uint32_t p) const { return s_dst[p]; }
};

// An oversize bucket of m elements is shared by blocks of one piece each: block `piece` places
// elements [piece * P, ...) of the bucket's order, in rounds of a quarter of what its LDS holds (fewer
// registers: a block's worth at once spilled 45, also where no bucket is oversize).
// The split has counted the bins of every piece (a.rows), so a block knows from the rows of
// the pieces before where its elements of each bin go, and reads no elements but its own: the
// cost stays near linear however the bins are filled.  1,048,576 messages of 28 bytes in no order
// 142 us, with half of them in one bin 138, all of them 82; 250,007 of them 42, 52 and 50.
// (Counting the bucket and selecting from it in every piece cost m^2 / 4,096 reads: 3,466 and
// 6,462 us of 1 M, 2,024 and 3,826 of 250,007.)
template <uint32_t BT, uint32_t MAXF, uint32_t S>
__device__ __forceinline__ void sort_piece(const BucketArgs& a, const VarTable& vt, SortLds<BT, MAXF, S>& s, uint32_t bucket,
                                           uint32_t first, uint32_t m, uint32_t piece) {
    constexpr uint32_t W = BT / 64u, C = S / 4u, kRound = BT * C;
    const uint32_t t = threadIdx.x, w = t >> 6, lane = lane_id();
    const uint32_t keys = 1u << a.shift, P = 1u << a.piece_log, pieces = (m + P - 1u) >> a.piece_log;
    // s.start: the bucket's elements of each bin; s.dest: those of the pieces before
    for (uint32_t k = t; k < keys; k += BT) s.start[k] = s.dest[k] = 0u;
    if (pieces == 1u) {
        __syncthreads();
        for (uint32_t e = t; e < m; e += BT) atomicAdd(&s.start[a.fine[first + e]], 1u);
        __syncthreads();
    } else {
        const uint32_t* rows = a.rows + ((size_t)piece_row(first, 0u, a.piece_log) << a.shift);
        for (uint32_t k = t; k < keys; k += BT) {
            uint32_t all = 0, before = 0;
            for (uint32_t r0 = 0; r0 < pieces; r0 += 8u) {
                uint32_t c[8];
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) c[j] = r0 + j < pieces ? rows[(size_t)(r0 + j) * keys + k] : 0u;
#pragma unroll
                for (uint32_t j = 0; j < 8; ++j) {
                    all += c[j];
                    before += r0 + j < piece ? c[j] : 0u;
                }
            }
            s.start[k] = all;
            s.dest[k] = before;
        }
        __syncthreads();
    }
    // s.dest: where this piece's elements of each bin go
    {
        const uint32_t q = (keys + BT - 1u) / BT, k0 = t * q;
        uint32_t sum = 0, total;
        for (uint32_t j = 0; j < q && k0 + j < keys; ++j) sum += s.start[k0 + j];
        uint32_t run = first + block_prefix<W>(sum, s.red, &total);
        for (uint32_t j = 0; j < q && k0 + j < keys; ++j) {
            const uint32_t bin = (bucket << a.shift) + k0 + j;
            if (a.start_out && piece == 0 && bin < a.bins) a.start_out[bin] = run;
            s.dest[k0 + j] += run;
            run += s.start[k0 + j];
        }
    }
    const uint32_t end = (piece + 1u) * P < m ? (piece + 1u) * P : m;
    for (uint32_t e0 = piece * P; e0 < end; e0 += kRound) {
        const uint32_t len = end - e0 < kRound ? end - e0 : kRound;
        const uint32_t cw = ((len + 63u) / 64u + W - 1u) / W;
        __syncthreads();   // the round before reads s.start, and moves s.dest on
        uint32_t f[C], id[C];
#pragma unroll
        for (uint32_t c = 0; c < C; ++c) {
            const uint32_t e = (w * cw + c) * 64u + lane;
            f[c] = c < cw && e < len ? a.fine[first + e0 + e] : 0u;
            id[c] = f[c] << 16 | e;   // a round is at most 2^16
        }
        sort_in_lds(s, keys, f, id, cw, len);
        // the split's counters are done with: the words hold each place's output element now
        for (uint32_t p = t; p < len; p += BT) {
            const uint32_t v = s.src[p], k = v >> 16;
            s.rows[p] = s.dest[k] + (p - s.start[k]);
            s.src[p] = a.idx[first + e0 + (v & 0xFFFFu)];
        }
        write_elements<BT, 4>(vt, len, PiecePlace{s.src, s.rows});   // a thread takes the places it has just written
        __syncthreads();
        for (uint32_t k = t; k < keys; k += BT) s.dest[k] += (k + 1u < keys ? s.start[k + 1u] : len) - s.start[k];
    }
}

// The bins after the last element of this block's bucket, of a list that is in order.
template <uint32_t BT>
__device__ __forceinline__ void end_bucket(const BucketArgs& a) {
    const uint32_t b = blockIdx.x;
    if (!a.start_out || b >= a.buckets) return;
    const uint32_t first = a.starts[b], next = a.starts[b + 1u], b0 = b << a.shift;
    const uint32_t end = a.bins - b0 < 1u << a.shift ? a.bins : b0 + (1u << a.shift);
    for (uint32_t k = (next > first ? key_of(a, next - 1u) + 1u : b0) + threadIdx.x; k < end; k += BT) a.start_out[k] = next;
    if (b == a.buckets - 1u && threadIdx.x == 0) a.start_out[a.bins] = next;
}

// Two blocks of 1,024 threads share a CU where S is 8 (at most 64 VGPRs): one loads while the
// other ranks.
template <uint32_t BT, uint32_t MAXF, uint32_t S>
__global__ void __launch_bounds__(BT, S == 8 ? 8 : 4) k_bucket_sort(BucketArgs a, VarTable vt) {
    constexpr uint32_t W = BT / 64u, kCap = SortLds<BT, MAXF, S>::kCap, kWindow = kCap / 2u;
    __shared__ SortLds<BT, MAXF, S> s;
    const uint32_t t = threadIdx.x, w = t >> 6, lane = lane_id(), nb = a.buckets;
    // one block per bucket, neighbouring buckets on one XCD
    uint32_t b = blockIdx.x < nb ? xcd_filled_block(nb) : 0u, piece = 0;
    uint32_t first = a.starts[b], next = a.starts[b + 1u];
    const uint32_t mode = *a.mode;
    if (mode == kCopy) {
        end_bucket<BT>(a);
        return;
    }
    if (blockIdx.x >= nb) {
        // further blocks: the pieces after the first of buckets that one block does not hold
        const uint32_t q = (nb + BT - 1u) / BT, b0 = t * q, want = blockIdx.x - nb;
        const uint32_t size = a.shift ? 1u << a.piece_log : kWindow;
        if (t == 0) s.lo = 0xFFFFFFFFu;
        uint32_t sum = 0, total;
        for (uint32_t j = 0; j < q && b0 + j < nb; ++j) {
            const uint32_t m = a.starts[b0 + j + 1u] - a.starts[b0 + j];
            sum += m > kCap ? (m - 1u) / size : 0u;
        }
        uint32_t run = block_prefix<W>(sum, s.red, &total);
        if (want >= total) return;
        for (uint32_t j = 0; j < q && b0 + j < nb; ++j) {
            const uint32_t m = a.starts[b0 + j + 1u] - a.starts[b0 + j];
            const uint32_t more = m > kCap ? (m - 1u) / size : 0u;
            if (want >= run && want < run + more) {
                s.lo = b0 + j;
                s.hi = want - run + 1u;
            }
            run += more;
        }
        __syncthreads();
        b = s.lo;
        piece = s.hi;
        __syncthreads();
        first = a.starts[b];
        next = a.starts[b + 1u];
    }
    const uint32_t m = next - first;
    if (a.start_out && b == nb - 1u && piece == 0 && t == 0) a.start_out[a.bins] = first + m;
    if (a.shift == 0) {
        // a bucket is one bin and already in order: pieces of kWindow elements
        if (a.start_out && piece == 0 && t == 0) a.start_out[b] = first;
        const uint32_t p = m > kCap ? piece * kWindow : 0u;
        const uint32_t len = m > kCap ? (m - p < kWindow ? m - p : kWindow) : m;
        write_sorted<BT>(vt, nullptr, a.idx, first + p, len);
        return;
    }
    if (m == 0) {
        if (a.start_out)
            for (uint32_t k = t; k < 1u << a.shift; k += BT)
                if ((b << a.shift) + k < a.bins) a.start_out[(b << a.shift) + k] = first;
        return;
    }
    if (m > kCap) {
        sort_piece<BT, MAXF, S>(a, vt, s, b, first, m, piece);
        return;
    }
    const bool staged = mode == kStage;
    const uint32_t cw = ((m + 63u) / 64u + W - 1u) / W;
    uint32_t f[S], id[S];
#pragma unroll
    for (uint32_t c = 0; c < S; ++c) {
        const uint32_t e = (w * cw + c) * 64u + lane;
        const bool valid = c < cw && e < m;
        f[c] = valid ? a.fine[first + e] : 0u;
        id[c] = staged ? e : (valid ? a.idx[first + e] : 0u);
    }
    const uint32_t keys = 1u << a.shift;
    sort_in_lds(s, keys, f, id, cw, m);
    if (a.start_out)
        for (uint32_t k = t; k < keys; k += BT)
            if ((b << a.shift) + k < a.bins) a.start_out[(b << a.shift) + k] = first + s.start[k];
    if (staged) permute_sorted<BT, S>(vt, s.src, first, m);
    else write_sorted<BT>(vt, s.src, nullptr, first, m);
}

// The whole list by one block: keys from the positions, sorted in LDS.
template <uint32_t BT, uint32_t MAXF, uint32_t S>
__global__ void __launch_bounds__(BT) k_sort_one_block(BucketArgs a, VarTable vt) {
    constexpr uint32_t W = BT / 64u;
    __shared__ SortLds<BT, MAXF, S> s;
    const uint32_t t = threadIdx.x, w = t >> 6, lane = lane_id();
    const uint32_t n = load_count(a.d_n, a.n_cap);
    const uint32_t cw = ((n + 63u) / 64u + W - 1u) / W;
    uint32_t f[S], id[S];
#pragma unroll
    for (uint32_t c = 0; c < S; ++c) {
        const uint32_t e = (w * cw + c) * 64u + lane;
        const bool valid = c < cw && e < n;
        f[c] = valid ? key_of(a, e) : 0u;
        id[c] = e;
    }
    sort_in_lds(s, a.bins, f, id, cw, n);
    if (a.start_out) {
        for (uint32_t k = t; k < a.bins; k += BT) a.start_out[k] = s.start[k];
        if (t == 0) a.start_out[a.bins] = n;
    }
    write_sorted<BT>(vt, s.src, nullptr, 0u, n);
}

// ---------------------------------------------------------------- host
constexpr uint32_t kOneBlockMax = 4096u;
constexpr uint32_t kMaxBins = 1024u;       // bins of a bucket: a sorting block's counters

bool bucket_plan(uint32_t n_cap, uint32_t bins, uint64_t used, BucketPlan* p) {
    // 12.58 M elements are where measuring stopped: 2,048 buckets of 16,384 places would hold an
    // evenly filled list of twice that
    if (!n_cap || !bins || n_cap > (3u << 22)) return false;
    *p = BucketPlan{};
    // one block sorts a list of 1,024 elements in 7 us; the four passes take 23 us on one of
    // 16,384, launches and all
    if (n_cap <= kOneBlockMax && bins <= kMaxBins) {
        p->one_block = 1;
        p->threads = 1024;
        return true;
    }
    // Elements per bucket, at most (the bins that occur evenly filled): a half or less of what
    // a sorting block holds, so that denser regions still fit.  Lists below 262,144 elements
    // take blocks of 256 threads (2,048 elements), and smaller buckets below 65,536, so that
    // there are enough blocks; larger ones 1,024 threads (8,192 elements); from 3 M on the
    // buckets a tile can count are too few for that (16,384 elements, tiles of 8,192).
    uint32_t per, most;
    if (n_cap < (1u << 18)) {
        p->threads = 256;
        p->items = 4;
        per = n_cap < (1u << 16) ? 256 : 1024;
        most = 1024;
    } else if (n_cap < (3u << 20)) {
        p->threads = 1024;
        p->items = 4;
        per = 2048;
        most = kMaxBuckets;
    } else {
        p->threads = 1024;
        p->items = 8;
        per = 4096;
        most = kMaxBuckets;
    }
    const uint64_t want = std::max<uint64_t>(1, n_cap / per);
    used = std::max<uint64_t>(1, std::min<uint64_t>(used, bins));
    while ((used >> (p->shift + 1)) >= want && (2u << p->shift) <= kMaxBins) ++p->shift;
    auto buckets = [&] { return ((uint64_t)bins + (1ull << p->shift) - 1) >> p->shift; };
    while (buckets() > most && (2u << p->shift) <= kMaxBins) ++p->shift;
    const uint64_t nb = buckets();
    if (nb > most) return false;
    p->buckets = (uint32_t)nb;
    p->tiles = ceil_div(n_cap, p->threads * p->items);
    // the tables fit the scratch that every bin sort of this size has
    if ((uint64_t)p->tiles * p->buckets > n_cap) return false;
    const uint64_t tables = (uint64_t)p->tiles + 2ull * p->buckets + 8ull;
    // Pieces of oversize buckets hold what a block does (2,048, 8,192 or 16,384 elements); blocks
    // of 256 threads take up to 8,192, round by round, where the rows of bin counts would not fit.
    const uint32_t cap = p->threads * (p->items == 8 ? 16u : 8u);
    for (p->piece_log = cap == 2048u ? 11u : (cap == 8192u ? 13u : 14u); ; ++p->piece_log) {
        p->rows = p->shift && n_cap > 1u << p->piece_log ? (2u * n_cap >> p->piece_log) << p->shift : 0u;
        if (tables + p->rows <= n_cap / 2) return true;
        if (p->piece_log >= 13u) return false;
    }
}

template <uint32_t BT, uint32_t ITEMS, uint32_t MAXB, uint32_t S>
static int launch_passes(const BucketArgs& a, const VarTable& vt, hipStream_t st) {
    constexpr uint32_t kWindow = BT * S / 2u;
    hipLaunchKernelGGL((k_bucket_count<BT, ITEMS>), dim3(a.tiles), dim3(BT), 0, st, a);
    FGX_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_bucket_prefix, dim3(ceil_div(a.buckets, 64) + 1u), dim3(1024), 0, st, a);
    FGX_HIP(hipGetLastError());
    hipLaunchKernelGGL((k_bucket_split<BT, ITEMS, MAXB>), dim3(a.tiles), dim3(BT), 0, st, a, vt);
    FGX_HIP(hipGetLastError());
    // a bucket of m elements has (m - 1) / size pieces after its first
    const uint32_t size = a.shift ? 1u << a.piece_log : kWindow;
    hipLaunchKernelGGL((k_bucket_sort<BT, kMaxBins, S>), dim3(a.buckets + a.n_cap / size), dim3(BT), 0, st, a, vt);
    FGX_HIP(hipGetLastError());
    return FGX_OK;
}

int bucket_sort(const BucketPlan& p, const KeyArgs& ka, uint32_t bins, const uint32_t* d_n, uint32_t n_cap, const float* x,
                const float* y, const float* z, const VarTable& vt, uint32_t* start_out, uint32_t* words_a,
                uint32_t* words_b, uint32_t* words_c, hipStream_t st) {
    BucketArgs a{};
    a.ka = ka;
    a.d_n = d_n;
    a.n_cap = n_cap;
    a.shift = p.shift;
    a.buckets = p.buckets;
    a.tiles = p.tiles;
    a.tile = p.threads * p.items;
    a.bins = bins;
    a.piece_log = p.piece_log;
    a.x = x;
    a.y = y;
    a.z = z;
    a.start_out = start_out;
    if (p.one_block) {
        hipLaunchKernelGGL((k_sort_one_block<1024, kMaxBins, kOneBlockMax / 1024u>), dim3(1), dim3(1024), 0, st, a, vt);
        FGX_HIP(hipGetLastError());
        return FGX_OK;
    }
    // words_a: n_cap 16-bit bins, then the small tables; words_b: indices; words_c: the counts
    a.fine = reinterpret_cast<uint16_t*>(words_a);
    uint32_t* tables = words_a + (n_cap + 1u) / 2u;
    a.mode = tables;
    a.totals = tables + 4;
    a.starts = a.totals + p.buckets;
    a.met = a.starts + p.buckets + 1;
    if (p.rows) a.rows = a.met + p.tiles;
    a.idx = a.edges = words_b;
    a.counts = words_c;
    // Elements of a tile that share a bucket lie next to each other in it; below 16 of them
    // (a half cache line of a 4-byte variable) gathering from the whole list costs more than
    // moving the variables twice, once the list is larger than the L2s hold.
    if (p.items == 8 && p.shift) a.stage_above = ceil_div(n_cap, 16u);
    if (p.threads == 256) return launch_passes<256, 4, 1024, 8>(a, vt, st);
    if (p.items == 4) return launch_passes<1024, 4, kMaxBuckets, 8>(a, vt, st);
    return launch_passes<1024, 8, kMaxBuckets, 16>(a, vt, st);
}

}  // namespace fgx
