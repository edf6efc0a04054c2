// k_sort.hip -- stable LSD radix sort of (64-bit key, 32-bit index) pairs.
//
// Replaces TreeNS::prepareSorting + HelperNS::sortArray = cub::DeviceRadixSort::SortPairs
// (tree.cu:1404-1413, helper.cu:150-167): same result, a stable sort by key in which
// ties keep ascending index order.  Eight passes of 8-bit digits.  Per pass:
//   count   -- digit histogram of each tile (LDS atomics);
//   scan    -- one workgroup per digit scans the tile histograms (digit-major) and writes the
//              digit's total;
//   scatter -- each wave ranks its slots of 64 keys with a ballot multisplit (peers
//              = lanes holding the same digit), the block stages the tile in LDS in
//              digit order and writes each digit run contiguously, behind the keys of smaller
//              digits (a scan of the 256 totals in every block: a separate pass over all keys for
//              the digit totals took 13 us at 1M keys and 122 us at 16.7M).
// Tiles of 2048 keys, of 1024 while these are at most SORT_SMALL_TILES: a tile's chain of ranking
// steps is then the pass's time (sorts of 300,007 keys 107 us, 500,009 keys 121 us; 1,000,003 keys take
// 172 us with the small tiles, 151 us with the large ones, 186 us before these two changes).
// HBM bytes per pass: count reads 8 B/key, scatter reads 12 and writes 12.
//
// Small sets are sorted by rank instead (k_sort_rank, k_sort_merge): a key's place is the number
// of keys before it, counted directly, which is one or two launches and no host wait.
#include <algorithm>
#include <mutex>

#include "mhpc_internal.h"

#define SORT_BLOCK 256
#define SORT_WAVES (SORT_BLOCK / 64)
#define SORT_ITEMS_LARGE (MHPC_SORT_TILE / SORT_BLOCK)   // 8
#define SORT_ITEMS_SMALL 4
#define SORT_SMALL_TILES 512

// check_flag (may be null): cleared for k_sort_check
template <int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_sort_count(const uint64_t *__restrict__ keys,
                                                           int64_t n, int shift,
                                                           uint32_t *__restrict__ tile_hist,
                                                           int64_t ntiles, uint32_t *check_flag) {
    __shared__ uint32_t h[MHPC_SORT_BUCKETS];
    h[threadIdx.x] = 0;
    if (check_flag && blockIdx.x == 0 && threadIdx.x == 0) *check_flag = 0u;
    __syncthreads();
    const int64_t base = (int64_t)blockIdx.x * (SORT_BLOCK * ITEMS);
    uint64_t k[ITEMS];
#pragma unroll
    for (int s = 0; s < ITEMS; s++) {
        const int64_t idx = base + s * SORT_BLOCK + threadIdx.x;
        k[s] = idx < n ? keys[idx] : 0ull;
    }
#pragma unroll
    for (int s = 0; s < ITEMS; s++) {
        const bool valid = base + s * SORT_BLOCK + threadIdx.x < n;
        const uint32_t d = (uint32_t)((k[s] >> shift) & 255u);
        // a wave whose keys share the digit (the high digits of sorted or clustered keys) adds
        // once: 64 LDS atomics on one word would serialise
        const uint64_t m = wave_ballot(valid);
        if (m == 0) continue;
        const uint32_t d0 = __builtin_amdgcn_readfirstlane(d);
        if (wave_ballot(valid && d != d0) == 0 && (m & 1ull)) {
            if (wave_lane() == 0) atomicAdd(&h[d0], (uint32_t)popc64(m));
        } else if (valid) {
            atomicAdd(&h[d], 1u);
        }
    }
    __syncthreads();
    tile_hist[(int64_t)threadIdx.x * ntiles + blockIdx.x] = h[threadIdx.x];
}

__global__ __launch_bounds__(SORT_BLOCK) void k_sort_scan(const uint32_t *__restrict__ tile_hist,
                                                          uint32_t *__restrict__ tile_off,
                                                          int64_t ntiles, uint32_t *__restrict__ digit_total) {
    __shared__ uint32_t lds4[SORT_WAVES];
    const int d = blockIdx.x;
    const uint32_t tot = block_scan_row(tile_hist + (int64_t)d * ntiles, tile_off + (int64_t)d * ntiles, ntiles, 0u,
                                        lds4);
    if (threadIdx.x == 0) digit_total[d] = tot;
}

template <int ITEMS>
__global__ __launch_bounds__(SORT_BLOCK) void k_sort_scatter(const uint64_t *__restrict__ kin,
                                                             const int32_t *__restrict__ vin,
                                                             uint64_t *__restrict__ kout,
                                                             int32_t *__restrict__ vout, int64_t n,
                                                             int shift,
                                                             const uint32_t *__restrict__ tile_off,
                                                             int64_t ntiles,
                                                             const uint32_t *__restrict__ digit_total) {
    constexpr int TILE = SORT_BLOCK * ITEMS;
    __shared__ uint64_t skeys[TILE];
    __shared__ int32_t svals[TILE];
    __shared__ uint32_t wcnt[SORT_WAVES][MHPC_SORT_BUCKETS];
    __shared__ uint32_t dstart[MHPC_SORT_BUCKETS];
    __shared__ uint32_t goff[MHPC_SORT_BUCKETS];
    __shared__ uint32_t lds4[SORT_WAVES];

    const int tid = threadIdx.x, w = tid / 64, lane = wave_lane();
    const int64_t base = (int64_t)blockIdx.x * TILE;
    // the tile's keys and values are requested before the digit offsets' scan
    uint64_t kr[ITEMS];
    int32_t vr[ITEMS];
    uint32_t rank[ITEMS];
#pragma unroll
    for (int s = 0; s < ITEMS; s++) {
        const int64_t idx = base + (int64_t)w * (64 * ITEMS) + s * 64 + lane;
        kr[s] = idx < n ? kin[idx] : 0ull;
        vr[s] = idx < n ? (vin ? vin[idx] : (int32_t)idx) : 0;
    }
#pragma unroll
    for (int k = 0; k < SORT_WAVES; k++) wcnt[k][tid] = 0;
    {
        const uint32_t off = tile_off[(int64_t)tid * ntiles + blockIdx.x];
        uint32_t smaller;   // keys with a smaller digit
        block_excl_scan256(digit_total[tid], &smaller, lds4);
        goff[tid] = smaller + off;
    }
    __syncthreads();

    const uint64_t lt = lanemask_lt();
#pragma unroll
    for (int s = 0; s < ITEMS; s++) {
        const int64_t idx = base + (int64_t)w * (64 * ITEMS) + s * 64 + lane;
        const bool valid = idx < n;
        const uint64_t key = kr[s];
        const uint32_t d = (uint32_t)((key >> shift) & 255u);
        uint64_t peers = wave_ballot(valid);
#pragma unroll
        for (int b = 0; b < MHPC_SORT_BITS; b++) {
            const bool bit = (d >> b) & 1u;
            const uint64_t m = wave_ballot(bit);
            peers &= bit ? m : ~m;
        }
        const uint32_t r = (uint32_t)popc64(peers & lt);
        uint32_t prior = 0;
        if (valid) prior = wcnt[w][d];
        wave_sync();
        if (valid && r == 0) wcnt[w][d] = prior + (uint32_t)popc64(peers);
        wave_sync();
        rank[s] = prior + r;
    }
    __syncthreads();
    {
        const uint32_t c0 = wcnt[0][tid], c1 = wcnt[1][tid], c2 = wcnt[2][tid], c3 = wcnt[3][tid];
        const uint32_t tot = c0 + c1 + c2 + c3;
        __syncthreads();
        wcnt[0][tid] = 0;
        wcnt[1][tid] = c0;
        wcnt[2][tid] = c0 + c1;
        wcnt[3][tid] = c0 + c1 + c2;
        uint32_t excl;
        block_excl_scan256(tot, &excl, lds4);
        dstart[tid] = excl;
    }
    __syncthreads();
#pragma unroll
    for (int s = 0; s < ITEMS; s++) {
        const int64_t idx = base + (int64_t)w * (64 * ITEMS) + s * 64 + lane;
        if (idx < n) {
            const uint32_t d = (uint32_t)((kr[s] >> shift) & 255u);
            const uint32_t pos = dstart[d] + wcnt[w][d] + rank[s];
            skeys[pos] = kr[s];
            svals[pos] = vr[s];
        }
    }
    __syncthreads();
    const int64_t rem = n - base;
    const int cnt = rem < TILE ? (int)rem : TILE;
    for (int t = tid; t < cnt; t += SORT_BLOCK) {
        const uint64_t key = skeys[t];
        const uint32_t d = (uint32_t)((key >> shift) & 255u);
        const uint32_t o = goff[d] + ((uint32_t)t - dstart[d]);
        if (o < (uint64_t)n) {
            kout[o] = key;
            vout[o] = svals[t];
        }
    }
}

// ------------------------------------------------------------------------------------
// Sort by rank.  A workgroup takes 64 keys of a tile of T keys (each lane one, the same in every
// wavefront); its 16 wavefronts count, each over a sixteenth of the tile, the keys that come
// before the lane's: smaller ones, and equal ones at smaller positions (a stable sort).  The
// tile's keys are wave-uniform, so they come through scalar loads, and a comparison is two or
// three instructions.  Writes each tile in sorted order.
//
// One tile (n <= SORT_RANK_MAX): the whole sort, one launch instead of 14 to 26 and the host's
// check of a partial sort (2048 keys: 9 us, the radix passes 85 us with their launches).
// Several tiles (n <= SORT_MERGE_MAX): k_sort_merge follows.  65,536 keys: 20 + 18 us against 121 us
// of radix passes; at 103,823 keys 33 + 44 us against 75 us of partial passes, so the line lies there.
#define SORT_RANK_WAVES 16
#define SORT_RANK_MAX 8192
#define SORT_RANK_TILE 2048
#define SORT_MERGE_MAX 98304

__global__ __launch_bounds__(64 * SORT_RANK_WAVES) void k_sort_rank(const uint64_t *__restrict__ keys, int n, int T,
                                                                   uint64_t *__restrict__ kout,
                                                                   int32_t *__restrict__ vout) {
    __shared__ int part[SORT_RANK_WAVES][64];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = wave_lane();
    const int base = blockIdx.x * 64;              // T is a multiple of 64: one tile per workgroup
    const int t0 = base / T * T, t1 = min(t0 + T, n);
    const int i = base + lane;
    const uint64_t key = i < n ? keys[i] : 0ull;
    const int share = (t1 - t0 + SORT_RANK_WAVES - 1) / SORT_RANK_WAVES;
    const int j0 = min(t0 + w * share, t1), j1 = min(j0 + share, t1);
    int cnt = 0;
    const int before = min(max(base, j0), j1);     // [j0, before): positions before the 64
#pragma unroll 8
    for (int j = j0; j < before; j++) cnt += keys[j] <= key ? 1 : 0;
    const int own = min(max(base + 64, j0), j1);   // [before, own): among the 64
    for (int j = before; j < own; j++) cnt += (keys[j] < key || (keys[j] == key && j < i)) ? 1 : 0;
#pragma unroll 8
    for (int j = own; j < j1; j++) cnt += keys[j] < key ? 1 : 0;
    part[w][lane] = cnt;
    __syncthreads();
    if (w != 0 || i >= n) return;
    int rank = t0;
#pragma unroll
    for (int v = 0; v < SORT_RANK_WAVES; v++) rank += part[v][lane];
    kout[rank] = key;
    vout[rank] = i;
}

// The tiles of k_sort_rank merged by rank: a key's place is its position in its own tile plus, by
// binary search, the keys of every other tile that come before it (equal ones of earlier tiles).
// A workgroup takes 64 keys, consecutive in their tile, so their searches share cache lines; its
// 16 wavefronts share the other tiles, up to four each, whose searches are independent chains of
// loads (one wavefront searching every tile was a chain of 96 load latencies, 64 us for 65,536
// keys; 18 us).
static_assert(SORT_MERGE_MAX <= 4 * SORT_RANK_WAVES * SORT_RANK_TILE, "four tiles per wavefront");
__global__ __launch_bounds__(64 * SORT_RANK_WAVES) void k_sort_merge(const uint64_t *__restrict__ kin,
                                                                    const int32_t *__restrict__ vin, int n,
                                                                    uint64_t *__restrict__ kout,
                                                                    int32_t *__restrict__ vout) {
    __shared__ int part[SORT_RANK_WAVES][64];
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = wave_lane();
    const int e = blockIdx.x * 64 + lane;
    const uint64_t key = e < n ? kin[e] : 0ull;
    const int own = blockIdx.x / (SORT_RANK_TILE / 64);
    int cnt = 0;
    int pos[4] = {0, 0, 0, 0};
    // does the key at place `at` of this wavefront's tile u come before this one?
    auto before = [&](int u, int at) {
        const int t = w + u * SORT_RANK_WAVES, j = t * SORT_RANK_TILE + at;
        if (t == own || at >= SORT_RANK_TILE || j >= n) return false;
        const uint64_t k = kin[j];
        return t < own ? k <= key : k < key;
    };
#pragma unroll
    for (int step = SORT_RANK_TILE / 2; step >= 1; step >>= 1)
#pragma unroll
        for (int u = 0; u < 4; u++) pos[u] += before(u, pos[u] + step - 1) ? step : 0;
    // the steps sum to T - 1: one last key decides whether the whole tile comes before
#pragma unroll
    for (int u = 0; u < 4; u++) cnt += pos[u] + (before(u, pos[u]) ? 1 : 0);
    part[w][lane] = cnt;
    __syncthreads();
    if (w != 0 || e >= n) return;
    int rank = e - own * SORT_RANK_TILE;
#pragma unroll
    for (int v = 0; v < SORT_RANK_WAVES; v++) rank += part[v][lane];
    kout[rank] = key;
    vout[rank] = vin[e];
}

// stable sort of n <= SORT_MERGE_MAX keys; keyB / valB: scratch of n elements.  in_place: the
// outputs may overlap the keys, which the one-launch form would overwrite while they are read.
static void sort_by_rank(hipStream_t stream, const uint64_t *keys, int64_t n, uint64_t *keyB, int32_t *valB,
                         uint64_t *kout, int32_t *vout, bool in_place) {
    const unsigned g = (unsigned)ceil_div(n, 64);
    if (n <= SORT_RANK_MAX && !in_place) {
        hipLaunchKernelGGL(k_sort_rank, dim3(g), dim3(64 * SORT_RANK_WAVES), 0, stream, keys, (int)n,
                           (int)(ceil_div(n, 64) * 64), kout, vout);
        return;
    }
    hipLaunchKernelGGL(k_sort_rank, dim3(g), dim3(64 * SORT_RANK_WAVES), 0, stream, keys, (int)n, SORT_RANK_TILE, keyB,
                       valB);
    hipLaunchKernelGGL(k_sort_merge, dim3(g), dim3(64 * SORT_RANK_WAVES), 0, stream, keyB, valB, (int)n, kout,
                       vout);
}

// the buffers of the LSD passes: input keys (values = positions), the even passes' outputs,
// the odd passes' outputs (the last pass's, so the result) and the per-pass tables
struct SortBufs {
    const uint64_t *kin;
    uint64_t *keyB;
    int32_t *valB;
    uint64_t *kout;
    int32_t *vout;
    uint32_t *tile_hist, *tile_off, *digit_total;
};
static void sort_passes(hipStream_t stream, int64_t n, int first, const SortBufs &b, uint32_t *check_flag);
static SortBufs ctx_bufs(mhpc_ctx *c) {
    return SortBufs{c->key, c->keyB, c->valB, c->skey, c->perm, c->tile_hist, c->tile_off, c->digit_hist};
}

static bool sort_small_tiles(int64_t n) { return ceil_div(n, SORT_BLOCK * SORT_ITEMS_SMALL) <= SORT_SMALL_TILES; }

// tiles of the largest sort up to cap keys
int64_t sort_tiles_cap(int64_t cap) {
    return std::max<int64_t>(ceil_div(cap, MHPC_SORT_TILE),
                             std::min<int64_t>(ceil_div(cap, SORT_BLOCK * SORT_ITEMS_SMALL), SORT_SMALL_TILES));
}

// Adjacent sorted keys equal in the bits the passes sorted (>= shift): their order in the low
// bits is not established.  Sets *flag.
__global__ __launch_bounds__(256) void k_sort_check(const uint64_t *__restrict__ skey, int64_t n, int shift,
                                                    uint32_t *__restrict__ flag) {
    const int64_t k = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
    if (k >= 1 && k < n && (skey[k] >> shift) == (skey[k - 1] >> shift)) *flag = 1u;
}

// The sort only needs the key levels at which particles are distinct.  The previous tree of
// this context had leaves no deeper than its deepest cell level + 1; with one level of margin
// the passes covering levels 1 .. depth + 2 usually suffice (4 of 8 on a 128^3 lattice).  Those
// passes run first; a check over the result finds any adjacent keys still equal in the sorted
// bits, the host reads it, and only then the full sort runs (from the untouched input keys).
// The result is the full sort's either way: distinct sorted prefixes fix the whole order.
void launch_sort(mhpc_ctx *c) {
    const int64_t n = c->n;
    if (n <= 0) return;
    if (n <= SORT_MERGE_MAX) {
        sort_by_rank(c->stream, c->key, n, c->keyB, c->valB, c->skey, c->perm, false);
        return;
    }
    const int levels = c->com_depth_hint + 2;
    const int first = levels < MHPC_LEVELS ? 3 * (MHPC_LEVELS - levels) / MHPC_SORT_BITS : 0;
    if (first > 0) {
        sort_passes(c->stream, n, first, ctx_bufs(c), c->sort_check);
        hipLaunchKernelGGL(k_sort_check, dim3((unsigned)ceil_div(n, 256)), dim3(256), 0, c->stream, c->skey, n,
                           MHPC_SORT_BITS * first, c->sort_check);
        if (ctx_fetch_status(c) == hipSuccess && c->h_status->sort_check == 0u) return;
    }
    sort_passes(c->stream, n, 0, ctx_bufs(c), nullptr);
}

// LSD passes first .. MHPC_SORT_PASSES - 1 from the input keys; the last (odd) pass writes
// kout / vout
template <int ITEMS>
static void sort_passes_t(hipStream_t stream, int64_t n, int first, const SortBufs &b, uint32_t *check_flag) {
    const unsigned ntiles = (unsigned)ceil_div(n, SORT_BLOCK * ITEMS);
    const uint64_t *kin = b.kin;
    const int32_t *vin = nullptr;
    for (int pass = first; pass < MHPC_SORT_PASSES; pass++) {
        uint64_t *kout = (pass & 1) ? b.kout : b.keyB;
        int32_t *vout = (pass & 1) ? b.vout : b.valB;
        const int shift = MHPC_SORT_BITS * pass;
        hipLaunchKernelGGL(k_sort_count<ITEMS>, dim3(ntiles), dim3(SORT_BLOCK), 0, stream, kin, n, shift, b.tile_hist,
                           (int64_t)ntiles, pass == first ? check_flag : nullptr);
        hipLaunchKernelGGL(k_sort_scan, dim3(MHPC_SORT_BUCKETS), dim3(SORT_BLOCK), 0, stream, b.tile_hist,
                           b.tile_off, (int64_t)ntiles, b.digit_total);
        hipLaunchKernelGGL(k_sort_scatter<ITEMS>, dim3(ntiles), dim3(SORT_BLOCK), 0, stream, kin, vin, kout, vout, n,
                           shift, b.tile_off, (int64_t)ntiles, b.digit_total);
        kin = kout;
        vin = vout;
    }
}

static void sort_passes(hipStream_t stream, int64_t n, int first, const SortBufs &b, uint32_t *check_flag) {
    if (sort_small_tiles(n)) sort_passes_t<SORT_ITEMS_SMALL>(stream, n, first, b, check_flag);
    else sort_passes_t<SORT_ITEMS_LARGE>(stream, n, first, b, check_flag);
}

// ------------------------------------------------------------------------------------
// The key sort without allocation (mhpc_sort_keys_noalloc): the same passes on caller-owned
// device arrays, with every buffer beyond the inputs and outputs carved from `scratch`, one
// static array per GPU that lives until the process ends.  Layout (byte offsets, each
// 256-aligned): even passes' keys and values, per-tile histograms and offsets, the digit totals.
#define NA_TILES (MHPC_NOALLOC_SORT_MAX / MHPC_SORT_TILE)
#define NA_KEYB 0
#define NA_VALB (NA_KEYB + 8 * (size_t)MHPC_NOALLOC_SORT_MAX)
#define NA_THIST (NA_VALB + 4 * (size_t)MHPC_NOALLOC_SORT_MAX)
#define NA_TOFF (NA_THIST + 4 * (size_t)MHPC_SORT_BUCKETS * NA_TILES)
#define NA_DHIST (NA_TOFF + 4 * (size_t)MHPC_SORT_BUCKETS * NA_TILES)
#define NA_BYTES (NA_DHIST + 4 * (size_t)MHPC_SORT_BUCKETS)
static_assert(MHPC_NOALLOC_SORT_MAX % MHPC_SORT_TILE == 0, "whole tiles");
static_assert(NA_VALB % 256 == 0 && NA_THIST % 256 == 0 && NA_TOFF % 256 == 0 && NA_DHIST % 256 == 0 &&
                  NA_BYTES % 256 == 0, "256-aligned parts");
static_assert(NA_TILES >= SORT_SMALL_TILES, "the tables hold the small tiles too");

static __device__ __align__(256) unsigned char scratch[NA_BYTES];

#define NA_MAX_DEVICES 64
static std::mutex na_mutex;
static unsigned char *na_ptr[NA_MAX_DEVICES];   // device address of `scratch` on each GPU

// `scratch`'s address on the current device, looked up once per device (the host-side name is
// not a device address)
static int na_scratch(unsigned char **out) {
    int dev = 0;
    if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= NA_MAX_DEVICES) return MHPC_E_HIP;
    std::lock_guard<std::mutex> lock(na_mutex);
    if (!na_ptr[dev]) {
        void *p = nullptr;
        if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return MHPC_E_HIP;
        na_ptr[dev] = static_cast<unsigned char *>(p);
    }
    *out = na_ptr[dev];
    return MHPC_OK;
}

extern "C" int mhpc_sort_keys_noalloc(const uint64_t *keys, int64_t n, uint64_t *sorted_keys, int32_t *sorted,
                                      void *stream) {
    if (n < 0 || (n > 0 && (!keys || !sorted_keys || !sorted))) return MHPC_E_ARG;
    if (n > MHPC_NOALLOC_SORT_MAX) return MHPC_E_SCRATCH;
    if (n == 0) return MHPC_OK;
    unsigned char *ptr = nullptr;
    const int st = na_scratch(&ptr);
    if (st != MHPC_OK) return st;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (n <= SORT_MERGE_MAX) {
        const uintptr_t k0 = reinterpret_cast<uintptr_t>(keys), k1 = k0 + sizeof(uint64_t) * (size_t)n;
        auto overlaps = [&](const void *p, size_t bytes) {
            const uintptr_t a = reinterpret_cast<uintptr_t>(p);
            return a < k1 && a + bytes > k0;
        };
        sort_by_rank(s, keys, n, reinterpret_cast<uint64_t *>(ptr + NA_KEYB),
                     reinterpret_cast<int32_t *>(ptr + NA_VALB), sorted_keys, sorted,
                     overlaps(sorted_keys, sizeof(uint64_t) * (size_t)n) || overlaps(sorted, sizeof(int32_t) * (size_t)n));
        return hipGetLastError() == hipSuccess ? MHPC_OK : MHPC_E_HIP;
    }
    const SortBufs b{keys,
                     reinterpret_cast<uint64_t *>(ptr + NA_KEYB),
                     reinterpret_cast<int32_t *>(ptr + NA_VALB),
                     sorted_keys,
                     sorted,
                     reinterpret_cast<uint32_t *>(ptr + NA_THIST),
                     reinterpret_cast<uint32_t *>(ptr + NA_TOFF),
                     reinterpret_cast<uint32_t *>(ptr + NA_DHIST)};
    sort_passes(s, n, 0, b, nullptr);
    return hipGetLastError() == hipSuccess ? MHPC_OK : MHPC_E_HIP;
}
