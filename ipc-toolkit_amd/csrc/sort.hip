// Device-wide scan, stable LSD radix sort and run-length encoding.
//
// Scans, run lengths and sort passes read their input once and run in one
// launch each: a tile publishes its own sum, then adds up the sums of the
// tiles before it until it meets one that already knows its prefix
// (decoupled look-back, Merrill & Garland 2016).  Tiles take their index
// from an atomic ticket, so a tile only ever waits for tiles that are already
// running and publish without waiting for anything.  A published word holds
// the launch's epoch, its state and the value together: one relaxed 64-bit
// atomic, no fences (on gfx950 a device-scope fence writes back and
// invalidates an L2), and no clearing between launches.
//
// Radix sort (8-bit digits): jobs (independent arrays) share every launch.
// Arrays of up to SB_MAX keys are sorted by one workgroup in LDS, all
// digits in one launch.  Larger ones take one histogram launch for all
// digits and one launch per digit over tiles of keys: each wave owns
// consecutive keys, ranks a 64-key chunk at a time by matching digits with 8
// ballots and keeps a running per-digit count in LDS; wave counts are
// prefix-summed across the workgroup, the look-back (a thread per digit) gives
// the tile's first slot of every digit, and the keys leave in digit order
// through LDS.  Tiles hold 2048 keys (short arrays: more workgroups) or,
// past BIG_TILES of those, 4096 64-bit or 8192 32-bit keys: a ticket takes
// about 12 ns whatever the width of the launch (75 M 32-bit keys: 0.49 ms
// a pass, 0.82 ms with 2048-key tiles, 0.76 ms in the three launches before).
//
// The form before took three to five launches per digit and array.  Three
// Morton arrays (8 K, 24 K and 16 K keys): 0.42 ms in 88 launches before,
// 0.15 ms in 10 now; 6.3 M, 4.2 M and 2.1 M keys: 1.30 ms before, 1.17 ms now.
#include "shard.hpp"
#include "sort.hpp"

#include <cstring>

namespace ipcg {

namespace {

constexpr int SCAN_BLOCK = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_BLOCK * SCAN_ITEMS;

template <class T> __device__ T block_exclusive_scan(T v, T& total)
{
    __shared__ T wsum[SCAN_BLOCK / WAVE];
    const int l = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    T x = v;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const T y = __shfl_up(x, o, WAVE);
        if (l >= o) x += y;
    }
    if (l == WAVE - 1) wsum[w] = x;
    __syncthreads();
    T off = 0, tot = 0;
#pragma unroll
    for (int i = 0; i < SCAN_BLOCK / WAVE; i++) {
        const T s = wsum[i];
        if (i < w) off += s;
        tot += s;
    }
    __syncthreads();
    total = tot;
    return off + x - v;
}

template <class T>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_partials(const T* in, int64_t n, T* partial)
{
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
    T s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        const int64_t i = base + (int64_t)j * SCAN_BLOCK + threadIdx.x;
        if (i < n) s += in[i];
    }
    T tot;
    block_exclusive_scan<T>(s, tot);
    if (threadIdx.x == 0) partial[blockIdx.x] = tot;
}

// single block scans the partials in place (any count, looping)
template <class T>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_single(T* partial, int64_t m, T* total)
{
    T carry = 0;
    for (int64_t base = 0; base < m; base += SCAN_TILE) {
        T v[SCAN_ITEMS];
        T s = 0;
#pragma unroll
        for (int j = 0; j < SCAN_ITEMS; j++) {
            const int64_t i = base + (int64_t)threadIdx.x * SCAN_ITEMS + j;
            v[j] = i < m ? partial[i] : 0;
            s += v[j];
        }
        T tot;
        T off = block_exclusive_scan<T>(s, tot) + carry;
#pragma unroll
        for (int j = 0; j < SCAN_ITEMS; j++) {
            const int64_t i = base + (int64_t)threadIdx.x * SCAN_ITEMS + j;
            if (i < m) partial[i] = off;
            off += v[j];
        }
        carry += tot;
    }
    if (threadIdx.x == 0 && total) *total = carry;
}

template <class T>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_final(const T* in, T* out, int64_t n,
                                                           const T* partial)
{
    const int64_t base = (int64_t)blockIdx.x * SCAN_TILE;
    T v[SCAN_ITEMS];
    T s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        const int64_t i = base + (int64_t)threadIdx.x * SCAN_ITEMS + j;
        v[j] = i < n ? in[i] : 0;
        s += v[j];
    }
    T tot;
    T off = block_exclusive_scan<T>(s, tot) + partial[blockIdx.x];
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        const int64_t i = base + (int64_t)threadIdx.x * SCAN_ITEMS + j;
        if (i < n) out[i] = off;
        off += v[j];
    }
}

// n <= SCAN_TILE: the whole scan in one workgroup (one launch instead of
// three)
template <class T>
__global__ __launch_bounds__(SCAN_BLOCK) void k_scan_one(const T* in, T* out, int64_t n,
                                                         T* total)
{
    T v[SCAN_ITEMS];
    T s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        const int64_t i = (int64_t)threadIdx.x * SCAN_ITEMS + j;
        v[j] = i < n ? in[i] : 0;
        s += v[j];
    }
    T tot;
    T off = block_exclusive_scan<T>(s, tot);
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        const int64_t i = (int64_t)threadIdx.x * SCAN_ITEMS + j;
        if (i < n) out[i] = off;
        off += v[j];
    }
    if (threadIdx.x == 0 && total) *total = tot;
}

// u64 sums (two packed counts) do not fit a look-back word: three launches
void scan_three(const uint64_t* in, uint64_t* out, int64_t n, uint64_t* total, void* tmp,
                hipStream_t s)
{
    using T = uint64_t;
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    T* partial = static_cast<T*>(tmp);
    if (n <= 0) {
        if (total) IPCG_HIP(hipMemsetAsync(total, 0, sizeof(T), s));
        return;
    }
    if (nb == 1) {
        hipLaunchKernelGGL(k_scan_one<T>, dim3(1), dim3(SCAN_BLOCK), 0, s, in, out, n, total);
        IPCG_CHECK_LAUNCH();
        return;
    }
    hipLaunchKernelGGL(k_scan_partials<T>, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, n,
                       partial);
    hipLaunchKernelGGL(k_scan_single<T>, dim3(1), dim3(SCAN_BLOCK), 0, s, partial, nb, total);
    hipLaunchKernelGGL(k_scan_final<T>, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, out, n,
                       partial);
    IPCG_CHECK_LAUNCH();
}

// ---- look-back ---------------------------------------------------------------
// word: epoch (30 bits) | state (2 bits) | value (32 bits)
constexpr unsigned LB_SUM = 1, LB_PREFIX = 2;

__device__ __forceinline__ void lb_publish(unsigned long long* w, unsigned epoch, unsigned state,
                                           uint32_t value)
{
    __hip_atomic_store(w, ((unsigned long long)(epoch << 2 | state) << 32) | value,
                       __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Sum of the values of tiles 0 .. tile - 1, word k at w[k * stride].  All
// tiles in flight publish their sums at about the same time, so a tile walks
// back over many of them: LB_WINDOW words are read at once (one memory round
// trip) and used as far as they are there.
constexpr int LB_WINDOW = 8;

__device__ __forceinline__ uint32_t lb_before(const unsigned long long* w, int64_t stride,
                                              int64_t tile, unsigned epoch)
{
    uint32_t sum = 0;
    bool done = tile == 0;
    for (int64_t k = tile - 1; !done;) {
        unsigned long long x[LB_WINDOW];
#pragma unroll
        for (int j = 0; j < LB_WINDOW; j++) {
            const int64_t at = k - j > 0 ? k - j : 0;
            x[j] = __hip_atomic_load(w + at * stride, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        bool there = true;
        int used = 0;
#pragma unroll
        for (int j = 0; j < LB_WINDOW; j++) {
            const unsigned tag = (unsigned)(x[j] >> 32);
            there = there && !done && tag >> 2 == epoch;
            if (there) {
                sum += (uint32_t)x[j];
                used++;
                done = (tag & 3u) == LB_PREFIX; // tile 0 publishes its prefix
            }
        }
        if (used == 0) __builtin_amdgcn_s_sleep(1); // the next word is not there yet
        k -= used;
    }
    return sum;
}

// The same for one value per tile, read by a whole wave: 64 words at once.
__device__ __forceinline__ uint32_t lb_before_wave(const unsigned long long* w, int64_t tile,
                                                   unsigned epoch)
{
    uint32_t sum = 0;
    for (int64_t k = tile - 1; k >= 0;) {
        const int64_t at = k - lane_id();
        const unsigned long long x = at >= 0
            ? __hip_atomic_load(w + at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)
            : 0ull;
        const unsigned tag = (unsigned)(x >> 32);
        const unsigned long long there = __ballot(at >= 0 && tag >> 2 == epoch);
        const unsigned long long prefix =
            __ballot(at >= 0 && tag >> 2 == epoch && (tag & 3u) == LB_PREFIX);
        // words up to the first one missing, or up to the first prefix
        int m = __builtin_ctzll(~there | (1ull << 63));
        if (there == ~0ull) m = WAVE;
        const int p = prefix ? __ffsll((long long)prefix) - 1 : WAVE;
        const bool done = p < m;
        const int use = done ? p + 1 : m;
        uint32_t v = lane_id() < use ? (uint32_t)x : 0u;
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
        sum += v;
        if (done) break;
        if (use == 0) __builtin_amdgcn_s_sleep(1);
        k -= use;
    }
    return sum;
}

// This workgroup's tile; the last ticket of a launch winds the counter back
// for the next.  Every thread must call it.
__device__ __forceinline__ int64_t lb_ticket(unsigned* ticket, unsigned tiles)
{
    __shared__ unsigned t;
    if (threadIdx.x == 0) {
        t = atomicAdd(ticket, 1u);
        if (t == tiles - 1)
            __hip_atomic_store(ticket, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    __syncthreads();
    return t;
}

// exclusive prefix of this tile's total over the tiles before it, the same in
// every thread
__device__ __forceinline__ uint32_t lb_scan(unsigned long long* w, int64_t tile, uint32_t total,
                                            unsigned epoch)
{
    __shared__ uint32_t before;
    if (threadIdx.x < WAVE) {
        if (threadIdx.x == 0) lb_publish(w + tile, epoch, tile ? LB_SUM : LB_PREFIX, total);
        const uint32_t b = lb_before_wave(w, tile, epoch);
        if (threadIdx.x == 0) {
            if (tile) lb_publish(w + tile, epoch, LB_PREFIX, b + total);
            before = b;
        }
    }
    __syncthreads();
    return before;
}

__global__ __launch_bounds__(SCAN_BLOCK) void k_scan(const uint32_t* in, uint32_t* out, int64_t n,
                                                     uint32_t* total, unsigned long long* w,
                                                     unsigned* ticket, unsigned epoch)
{
    const int64_t tile = lb_ticket(ticket, gridDim.x);
    const int64_t base = tile * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    uint32_t v[SCAN_ITEMS];
    uint32_t s = 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        v[j] = base + j < n ? in[base + j] : 0;
        s += v[j];
    }
    uint32_t tot;
    uint32_t off = block_exclusive_scan<uint32_t>(s, tot);
    const uint32_t before = lb_scan(w, tile, tot, epoch);
    off += before;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        if (base + j < n) out[base + j] = off;
        off += v[j];
    }
    if (threadIdx.x == 0 && total && tile == (int64_t)gridDim.x - 1) *total = before + tot;
}

// Sorted keys -> unique keys, first position of each run (start[number of
// runs] = n) and the number of runs.
__global__ __launch_bounds__(SCAN_BLOCK) void k_rle(const uint64_t* keys, int64_t n,
                                                    uint64_t* ukeys, uint32_t* start, uint32_t* nu,
                                                    unsigned long long* w, unsigned* ticket,
                                                    unsigned epoch)
{
    const int64_t tile = lb_ticket(ticket, gridDim.x);
    const int64_t base = tile * SCAN_TILE + (int64_t)threadIdx.x * SCAN_ITEMS;
    uint64_t k[SCAN_ITEMS];
    bool head[SCAN_ITEMS];
    uint32_t s = 0;
    uint64_t prev = base > 0 && base < n ? keys[base - 1] : 0;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++) {
        const int64_t i = base + j;
        k[j] = i < n ? keys[i] : 0;
        head[j] = i < n && (i == 0 || k[j] != prev);
        prev = k[j];
        s += head[j];
    }
    uint32_t tot;
    uint32_t off = block_exclusive_scan<uint32_t>(s, tot);
    const uint32_t before = lb_scan(w, tile, tot, epoch);
    off += before;
#pragma unroll
    for (int j = 0; j < SCAN_ITEMS; j++)
        if (head[j]) {
            ukeys[off] = k[j];
            start[off] = (uint32_t)(base + j);
            off++;
        }
    if (threadIdx.x == 0 && tile == (int64_t)gridDim.x - 1) {
        *nu = before + tot;
        start[before + tot] = (uint32_t)n;
    }
}

// ---------------------------------------------------------------------------
constexpr int RS_BLOCK = 256;
constexpr int RS_CHUNKS = 8; // 64-key chunks per wave
constexpr int RS_TILE = RS_BLOCK * RS_CHUNKS;
constexpr int BIG_BLOCK = 512;
constexpr int64_t BIG_TILES = 2048;
template <class K> constexpr int big_chunks() { return sizeof(K) == 8 ? 8 : 16; }

constexpr int MAX_DIGITS = 8;

// one array of a sort as the kernels see it
struct KeyJob {
    const void* keys;
    const uint32_t* vals; // null: the positions
    void* okeys;
    uint32_t* ovals;
    int64_t n;
    unsigned long long mask;       // bits that may vary
    int64_t tile0, ntiles;         // its tiles of the launch
    int shift;                     // this launch's digit, -1: none
    const uint32_t* hist;          // counts of that digit
    unsigned long long* status;    // look-back words, 256 per tile
};
struct KeyJobs {
    KeyJob j[SORT_JOBS];
    int n;
};

// Ranks 64 keys by digit among the wave's keys so far: lanes of one digit
// count up from wcnt[d] (the wave's running counts).
__device__ __forceinline__ uint32_t wave_rank(uint32_t d, bool valid, uint32_t* wcnt,
                                              unsigned long long lt)
{
    unsigned long long peers = __ballot(valid);
#pragma unroll
    for (int b = 0; b < 8; b++) {
        const unsigned long long m = __ballot((d >> b) & 1);
        peers &= ((d >> b) & 1) ? m : ~m;
    }
    const uint32_t r = (uint32_t)__popcll(peers & lt);
    const uint32_t before = valid ? wcnt[d] : 0;
    __builtin_amdgcn_wave_barrier();
    if (valid && r == 0) wcnt[d] = before + (uint32_t)__popcll(peers);
    __builtin_amdgcn_wave_barrier();
    return before + r;
}

// Per digit d (threads 0 .. 255): wave counts -> offsets within the digit;
// dstart[d] = first slot of the digit in the tile.  Returns the digit's
// total.  Every thread of the workgroup must call it.
template <int WAVES>
__device__ __forceinline__ uint32_t digit_starts(uint32_t (*wcnt)[256], uint32_t* dstart,
                                                 uint32_t* wtot)
{
    const int d = threadIdx.x, lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    uint32_t total = 0, x = 0;
    if (d < 256) {
        uint32_t c[WAVES]; // every read before the writes
#pragma unroll
        for (int ww = 0; ww < WAVES; ww++) c[ww] = wcnt[ww][d];
#pragma unroll
        for (int ww = 0; ww < WAVES; ww++) {
            wcnt[ww][d] = total;
            total += c[ww];
        }
        x = total;
#pragma unroll
        for (int o = 1; o < WAVE; o <<= 1) {
            const uint32_t y = __shfl_up(x, o, WAVE);
            if (lane >= o) x += y;
        }
        if (lane == WAVE - 1) wtot[w] = x;
    }
    __syncthreads();
    if (d < 256) {
        uint32_t wpre = 0;
#pragma unroll
        for (int ww = 0; ww < 256 / WAVE; ww++)
            if (ww < w) wpre += wtot[ww];
        dstart[d] = wpre + x - total;
    }
    __syncthreads();
    return total;
}

// All digits of an array of at most SB_MAX keys in one workgroup: keys and
// values stay in registers and cross LDS once per digit (112 KB).
constexpr int SB_BLOCK = 1024;
constexpr int SB_WAVES = SB_BLOCK / WAVE;
constexpr int SB_CHUNKS = 8;
constexpr int64_t SB_MAX = (int64_t)SB_BLOCK * SB_CHUNKS;

template <class K> __global__ __launch_bounds__(SB_BLOCK) void k_sort_block(KeyJobs J)
{
    __shared__ K sk[SB_MAX];
    __shared__ uint32_t sv[SB_MAX];
    __shared__ uint32_t wcnt[SB_WAVES][256];
    __shared__ uint32_t dstart[256], wtot[256 / WAVE];
    const KeyJob j = J.j[blockIdx.x];
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const unsigned long long lt = (1ull << lane) - 1ull;
    // waves share the keys evenly, in chunks of 64
    const int n = (int)j.n, chunks = (n + SB_BLOCK - 1) / SB_BLOCK;
    const int base = w * chunks * WAVE + lane;
    K k[SB_CHUNKS];
    uint32_t v[SB_CHUNKS], rank[SB_CHUNKS];
#pragma unroll
    for (int c = 0; c < SB_CHUNKS; c++) {
        const int i = base + c * WAVE;
        const bool in = c < chunks && i < n;
        k[c] = in ? static_cast<const K*>(j.keys)[i] : 0;
        v[c] = in ? (j.vals ? j.vals[i] : (uint32_t)i) : 0;
    }
    for (int shift = 0; shift < 8 * (int)sizeof(K); shift += 8) {
        if (((j.mask >> shift) & 0xFFull) == 0) continue;
        for (int i = threadIdx.x; i < SB_WAVES * 256; i += SB_BLOCK) (&wcnt[0][0])[i] = 0;
        __syncthreads();
#pragma unroll
        for (int c = 0; c < SB_CHUNKS; c++)
            if (c < chunks)
                rank[c] = wave_rank((uint32_t)(k[c] >> shift) & 0xFF, base + c * WAVE < n,
                                    wcnt[w], lt);
        __syncthreads();
        digit_starts<SB_WAVES>(wcnt, dstart, wtot);
#pragma unroll
        for (int c = 0; c < SB_CHUNKS; c++)
            if (c < chunks && base + c * WAVE < n) {
                const uint32_t d = (uint32_t)(k[c] >> shift) & 0xFF;
                const uint32_t at = dstart[d] + wcnt[w][d] + rank[c];
                sk[at] = k[c];
                sv[at] = v[c];
            }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < SB_CHUNKS; c++)
            if (c < chunks && base + c * WAVE < n) {
                k[c] = sk[base + c * WAVE];
                v[c] = sv[base + c * WAVE];
            }
    }
#pragma unroll
    for (int c = 0; c < SB_CHUNKS; c++) {
        const int i = base + c * WAVE;
        if (c < chunks && i < n) {
            static_cast<K*>(j.okeys)[i] = k[c];
            j.ovals[i] = v[c];
        }
    }
}

// Digit counts of every job and digit (hist: SORT_JOBS x MAX_DIGITS x 256,
// zero on entry).
template <class K>
__global__ __launch_bounds__(RS_BLOCK) void k_sort_hist(KeyJobs J, uint32_t* hist)
{
    __shared__ uint32_t h[MAX_DIGITS][256];
    int q = 0;
    while (q + 1 < J.n && (int64_t)blockIdx.x >= J.j[q + 1].tile0) q++;
    const K* const keys = static_cast<const K*>(J.j[q].keys);
    const int64_t n = J.j[q].n, stride = J.j[q].ntiles * RS_TILE;
    const unsigned long long mask = J.j[q].mask;
#pragma unroll
    for (int p = 0; p < MAX_DIGITS; p++) h[p][threadIdx.x] = 0;
    __syncthreads();
    for (int64_t base = ((int64_t)blockIdx.x - J.j[q].tile0) * RS_TILE; base < n; base += stride)
#pragma unroll
        for (int c = 0; c < RS_CHUNKS; c++) {
            const int64_t i = base + c * RS_BLOCK + threadIdx.x;
            if (i < n) {
                const K k = keys[i];
#pragma unroll
                for (int p = 0; p < (int)sizeof(K); p++)
                    if ((mask >> (8 * p)) & 0xFFull) atomicAdd(&h[p][(k >> (8 * p)) & 0xFF], 1u);
            }
        }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < MAX_DIGITS; p++) {
        const uint32_t c = h[p][threadIdx.x];
        if (c) atomicAdd(hist + (q * MAX_DIGITS + p) * 256 + threadIdx.x, c);
    }
}

// One stable digit pass of every job that has this digit.  `clear`: the
// other histogram buffer, zeroed for the next sort.
template <class K, int BLOCK, int CHUNKS>
__global__ __launch_bounds__(BLOCK, 4) void k_sort_pass(KeyJobs J, unsigned tiles,
                                                        unsigned* ticket, unsigned epoch,
                                                        uint32_t* clear)
{
    constexpr int WAVES = BLOCK / WAVE, TILE = BLOCK * CHUNKS;
    __shared__ uint32_t wcnt[WAVES][256];
    __shared__ uint32_t tile_off[256];
    __shared__ uint32_t dstart[256]; // first slot of each digit in the tile
    __shared__ uint32_t wtot[256 / WAVE], gtot[256 / WAVE];
    __shared__ K sk[TILE];
    __shared__ uint32_t sv[TILE];
    const int lane = threadIdx.x % WAVE, w = threadIdx.x / WAVE;
    const int64_t t = lb_ticket(ticket, tiles);
    if (clear && t == 0)
        for (int i = threadIdx.x; i < SORT_JOBS * MAX_DIGITS * 256; i += BLOCK) clear[i] = 0;
    int q = 0;
    while (q + 1 < J.n && t >= J.j[q + 1].tile0) q++;
    const KeyJob& j = J.j[q];
    const K* const keys = static_cast<const K*>(j.keys);
    const int64_t n = j.n, tile = t - j.tile0;
    const int shift = j.shift;
    for (int i = threadIdx.x; i < WAVES * 256; i += BLOCK) (&wcnt[0][0])[i] = 0;
    // first slot of every digit in the output
    const bool digit = threadIdx.x < 256; // a thread per digit
    const uint32_t gh = digit ? j.hist[threadIdx.x] : 0;
    uint32_t gx = gh;
#pragma unroll
    for (int o = 1; o < WAVE; o <<= 1) {
        const uint32_t y = __shfl_up(gx, o, WAVE);
        if (lane >= o) gx += y;
    }
    if (digit && lane == WAVE - 1) gtot[w] = gx;
    __syncthreads();
    uint32_t first = gx - gh;
#pragma unroll
    for (int ww = 0; ww < 256 / WAVE; ww++)
        if (ww < w) first += gtot[ww];
    const int64_t at0 = tile * TILE;
    const int64_t base = at0 + (int64_t)w * (CHUNKS * WAVE) + lane;
    const unsigned long long lt = (1ull << lane) - 1ull;
    K k[CHUNKS];
    uint32_t v[CHUNKS];
    uint32_t rank[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; c++) {
        const int64_t i = base + c * WAVE;
        k[c] = i < n ? keys[i] : 0;
        v[c] = i < n ? (j.vals ? j.vals[i] : (uint32_t)i) : 0;
    }
#pragma unroll
    for (int c = 0; c < CHUNKS; c++)
        rank[c] = wave_rank((uint32_t)(k[c] >> shift) & 0xFF, base + c * WAVE < n, wcnt[w], lt);
    __syncthreads();
    const uint32_t total = digit_starts<WAVES>(wcnt, dstart, wtot);
    if (digit) {
        unsigned long long* const word = j.status + threadIdx.x;
        lb_publish(word + 256 * tile, epoch, tile ? LB_SUM : LB_PREFIX, total);
        const uint32_t before = lb_before(word, 256, tile, epoch);
        if (tile) lb_publish(word + 256 * tile, epoch, LB_PREFIX, before + total);
        tile_off[threadIdx.x] = first + before;
    }
    // keys in digit order in LDS, then each digit's run to its place, so
    // that neighbouring lanes write neighbouring addresses
#pragma unroll
    for (int c = 0; c < CHUNKS; c++)
        if (base + c * WAVE < n) {
            const uint32_t d = (uint32_t)(k[c] >> shift) & 0xFF;
            const uint32_t lp = dstart[d] + wcnt[w][d] + rank[c];
            sk[lp] = k[c];
            sv[lp] = v[c];
        }
    __syncthreads();
    const int tn = (int)(n - at0 < TILE ? n - at0 : TILE);
    for (int i = threadIdx.x; i < tn; i += BLOCK) {
        const K key = sk[i];
        const uint32_t d = (uint32_t)(key >> shift) & 0xFF;
        const int64_t pos = (int64_t)tile_off[d] + (i - (int)dstart[d]);
        static_cast<K*>(j.okeys)[pos] = key;
        j.ovals[pos] = sv[i];
    }
}

} // namespace

size_t scan_tmp_bytes(int64_t n)
{
    return sizeof(uint64_t) * (size_t)((n + SCAN_TILE - 1) / SCAN_TILE + 1) + 256;
}

// Makes room for `words` look-back words and returns the launch's epoch.
// Old words never match a new epoch; new memory is cleared once.
static unsigned lb_begin(SortSpace& ws, int64_t words, hipStream_t s)
{
    constexpr unsigned EPOCHS = 1u << 30;
    const size_t bytes = sizeof(unsigned long long) * (size_t)words;
    bool clear = bytes > ws.status.bytes;
    ws.status.reserve(bytes);
    if (++ws.epoch == EPOCHS) {
        ws.epoch = 1;
        clear = true;
    }
    if (clear) IPCG_HIP(hipMemsetAsync(ws.status.p, 0, ws.status.bytes, s));
    if (!ws.ticket.p) {
        ws.ticket.reserve(256);
        IPCG_HIP(hipMemsetAsync(ws.ticket.p, 0, ws.ticket.bytes, s));
    }
    return ws.epoch;
}

void exclusive_scan_u32(SortSpace& ws, const uint32_t* in, uint32_t* out, int64_t n,
                        uint32_t* total_dev, hipStream_t s)
{
    if (n <= 0) {
        if (total_dev) IPCG_HIP(hipMemsetAsync(total_dev, 0, sizeof(uint32_t), s));
        return;
    }
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    if (nb == 1) {
        hipLaunchKernelGGL(k_scan_one<uint32_t>, dim3(1), dim3(SCAN_BLOCK), 0, s, in, out, n,
                           total_dev);
        IPCG_CHECK_LAUNCH();
        return;
    }
    const unsigned epoch = lb_begin(ws, nb, s);
    hipLaunchKernelGGL(k_scan, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, in, out, n, total_dev,
                       ws.status.as<unsigned long long>(), ws.ticket.as<unsigned>(), epoch);
    IPCG_CHECK_LAUNCH();
}

void exclusive_scan_u64(const uint64_t* in, uint64_t* out, int64_t n, uint64_t* total_dev,
                        void* tmp, hipStream_t s)
{
    scan_three(in, out, n, total_dev, tmp, s);
}

void run_length_encode(SortSpace& ws, const uint64_t* keys, int64_t n, uint64_t* unique_keys,
                       uint32_t* run_start, uint32_t* n_unique_dev, hipStream_t s)
{
    if (n <= 0) {
        IPCG_HIP(hipMemsetAsync(n_unique_dev, 0, sizeof(uint32_t), s));
        IPCG_HIP(hipMemsetAsync(run_start, 0, sizeof(uint32_t), s));
        return;
    }
    const int64_t nb = (n + SCAN_TILE - 1) / SCAN_TILE;
    const unsigned epoch = lb_begin(ws, nb, s);
    hipLaunchKernelGGL(k_rle, dim3((unsigned)nb), dim3(SCAN_BLOCK), 0, s, keys, n, unique_keys,
                       run_start, n_unique_dev, ws.status.as<unsigned long long>(),
                       ws.ticket.as<unsigned>(), epoch);
    IPCG_CHECK_LAUNCH();
}

template <class K> static void sort_jobs(SortSpace& ws, SortJob* jobs, int njobs, hipStream_t s)
{
    if (njobs > SORT_JOBS) throw Error(IPCG_ERR_ARG, "too many arrays in one sort");
    KeyJobs small {}, large {};
    SortJob* of_large[SORT_JOBS];
    int64_t tiles = 0;
    for (int q = 0; q < njobs; q++) {
        SortJob& j = jobs[q];
        if (sizeof(K) < 8) j.mask &= (1ull << (8 * sizeof(K) % 64)) - 1ull;
        j.in_alt = false;
        if (j.n >= (1ll << 32)) throw Error(IPCG_ERR_ARG, "too many keys for one sort");
        if (j.n <= 0) continue;
        KeyJob k {};
        k.keys = j.keys;
        k.vals = j.iota ? nullptr : j.vals;
        k.okeys = j.keys;
        k.ovals = j.vals;
        k.n = j.n;
        k.mask = j.mask;
        if (j.n <= SB_MAX) {
            small.j[small.n++] = k;
            continue;
        }
        if (j.mask == 0) throw Error(IPCG_ERR_ARG, "a sort needs key bits");
        k.ntiles = (j.n + RS_TILE - 1) / RS_TILE; // (short tiles)
        tiles += k.ntiles;
        of_large[large.n] = &j;
        large.j[large.n++] = k;
    }
    if (small.n) {
        hipLaunchKernelGGL(k_sort_block<K>, dim3(small.n), dim3(SB_BLOCK), 0, s, small);
        IPCG_CHECK_LAUNCH();
    }
    if (!large.n) return;
    constexpr size_t HIST = SORT_JOBS * MAX_DIGITS * 256; // one buffer
    const bool fresh = !ws.hist.p || ws.torn;
    ws.hist.reserve(sizeof(uint32_t) * 2 * HIST);
    if (fresh) IPCG_HIP(hipMemsetAsync(ws.hist.p, 0, sizeof(uint32_t) * 2 * HIST, s));
    ws.torn = true; // until every launch below is in the stream
    uint32_t* const hist = ws.hist.as<uint32_t>() + (ws.flip ? HIST : 0);
    uint32_t* const other = ws.hist.as<uint32_t>() + (ws.flip ? 0 : HIST);
    ws.flip = !ws.flip;
    { // at most HIST_GROUPS workgroups per array (each adds up to 2048 counts)
        constexpr int64_t HIST_GROUPS = 512;
        KeyJobs h = large;
        int64_t at = 0;
        for (int q = 0; q < h.n; q++) {
            h.j[q].tile0 = at;
            h.j[q].ntiles = h.j[q].ntiles < HIST_GROUPS ? h.j[q].ntiles : HIST_GROUPS;
            at += h.j[q].ntiles;
        }
        hipLaunchKernelGGL(k_sort_hist<K>, dim3((unsigned)at), dim3(RS_BLOCK), 0, s, h, hist);
        IPCG_CHECK_LAUNCH();
    }
    const bool big = tiles > BIG_TILES;
    const int tile = big ? BIG_BLOCK * big_chunks<K>() : RS_TILE;
    for (int q = 0; q < large.n; q++) large.j[q].ntiles = (large.j[q].n + tile - 1) / tile;
    bool first = true;
    for (int p = 0; p < (int)sizeof(K); p++) {
        KeyJobs pass {};
        int64_t at = 0;
        for (int q = 0; q < large.n; q++) {
            KeyJob& k = large.j[q];
            SortJob& j = *of_large[q];
            if (((k.mask >> (8 * p)) & 0xFFull) == 0) continue;
            K* const a = static_cast<K*>(j.keys);
            K* const b = static_cast<K*>(j.keys_alt);
            k.keys = j.in_alt ? b : a;
            k.vals = j.iota ? nullptr : (j.in_alt ? j.vals_alt : j.vals);
            k.okeys = j.in_alt ? a : b;
            k.ovals = j.in_alt ? j.vals : j.vals_alt;
            k.shift = 8 * p;
            k.hist = hist + (q * MAX_DIGITS + p) * 256;
            KeyJob out = k;
            out.tile0 = at;
            at += k.ntiles;
            pass.j[pass.n++] = out;
            j.in_alt = !j.in_alt;
            j.iota = false; // the values exist from here on
        }
        if (!pass.n) continue;
        const unsigned epoch = lb_begin(ws, 256 * at, s);
        for (int q = 0; q < pass.n; q++)
            pass.j[q].status = ws.status.as<unsigned long long>() + 256 * pass.j[q].tile0;
        if (big)
            hipLaunchKernelGGL((k_sort_pass<K, BIG_BLOCK, big_chunks<K>()>), dim3((unsigned)at),
                               dim3(BIG_BLOCK), 0, s, pass, (unsigned)at,
                               ws.ticket.as<unsigned>(), epoch, first ? other : nullptr);
        else
            hipLaunchKernelGGL((k_sort_pass<K, RS_BLOCK, RS_CHUNKS>), dim3((unsigned)at),
                               dim3(RS_BLOCK), 0, s, pass, (unsigned)at,
                               ws.ticket.as<unsigned>(), epoch, first ? other : nullptr);
        IPCG_CHECK_LAUNCH();
        first = false;
    }
    ws.torn = false;
}

void radix_sort_jobs(SortSpace& ws, SortJob* jobs, int njobs, hipStream_t s)
{
    sort_jobs<uint64_t>(ws, jobs, njobs, s);
}

bool radix_sort_pairs(SortSpace& ws, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                      uint32_t* vals_alt, int64_t n, unsigned long long bit_mask, bool iota,
                      hipStream_t s)
{
    SortJob j { keys, keys_alt, vals, vals_alt, n, bit_mask, iota, false };
    sort_jobs<uint64_t>(ws, &j, 1, s);
    return j.in_alt;
}

bool radix_sort_pairs(SortSpace& ws, uint32_t* keys, uint32_t* vals, uint32_t* keys_alt,
                      uint32_t* vals_alt, int64_t n, unsigned long long bit_mask, bool iota,
                      hipStream_t s)
{
    SortJob j { keys, keys_alt, vals, vals_alt, n, bit_mask, iota, false };
    sort_jobs<uint32_t>(ws, &j, 1, s);
    return j.in_alt;
}

// one workgroup per counter set: the offsets of its shards, its total and its
// largest shard count
__global__ __launch_bounds__(SHARDS) void k_shard_summary(const unsigned long long* cnt,
                                                          const unsigned long long* extra,
                                                          int64_t* off,
                                                          unsigned long long* out)
{
    static_assert(SHARDS == SCAN_BLOCK, "block_exclusive_scan");
    __shared__ unsigned long long wmax[SHARDS / WAVE];
    const unsigned long long v =
        cnt[(int64_t)blockIdx.x * SHARDS * SHARD_PAD + (int64_t)threadIdx.x * SHARD_PAD];
    unsigned long long mx = v, total;
    for (int o = WAVE / 2; o > 0; o >>= 1) {
        const unsigned long long y = __shfl_xor(mx, o, WAVE);
        mx = y > mx ? y : mx;
    }
    if (threadIdx.x % WAVE == 0) wmax[threadIdx.x / WAVE] = mx;
    int64_t* const so = off + (int64_t)blockIdx.x * (SHARDS + 1);
    so[threadIdx.x] = (int64_t)block_exclusive_scan<unsigned long long>(v, total);
    if (threadIdx.x == 0) {
        so[SHARDS] = (int64_t)total;
        unsigned long long m = 0;
        for (int w = 0; w < SHARDS / WAVE; w++) m = wmax[w] > m ? wmax[w] : m;
        out[2 * blockIdx.x] = total;
        out[2 * blockIdx.x + 1] = m;
        if (blockIdx.x == 0) out[2 * gridDim.x] = extra ? *extra : 0ull;
    }
}

void shard_counts_n(const unsigned long long* cnt_dev, int nsets, unsigned long long* sum_dev,
                    int64_t* off_dev, void* pinned, hipStream_t s, ShardCounts* out,
                    const void* extra_dev, void* extra)
{
    hipLaunchKernelGGL(k_shard_summary, dim3(nsets), dim3(SHARDS), 0, s, cnt_dev,
                       static_cast<const unsigned long long*>(extra_dev), off_dev, sum_dev);
    IPCG_CHECK_LAUNCH();
    unsigned long long* h = static_cast<unsigned long long*>(pinned);
    IPCG_HIP(hipMemcpyAsync(h, sum_dev, sizeof(unsigned long long) * (2 * nsets + 1),
                            hipMemcpyDeviceToHost, s));
    IPCG_HIP(hipStreamSynchronize(s));
    for (int k = 0; k < nsets; k++) {
        out[k].total = (int64_t)h[2 * k];
        out[k].max = (int64_t)h[2 * k + 1];
    }
    if (extra) std::memcpy(extra, h + 2 * nsets, sizeof(*h));
}

ShardCounts shard_counts(const unsigned long long* cnt_dev, unsigned long long* sum_dev,
                         int64_t* off_dev, void* pinned, hipStream_t s)
{
    ShardCounts r;
    shard_counts_n(cnt_dev, 1, sum_dev, off_dev, pinned, s, &r);
    return r;
}

} // namespace ipcg
