// Hand-written device-wide primitives for gfx950: exclusive scan, stable
// LSD radix sort of (uint64 or uint32 key, uint32 value) pairs with 8-bit digits,
// run-length encoding of sorted keys.  Declarations; kernels in sort.hip.
#pragma once

#include "common.hpp"

namespace ipcg {

// Scratch of the primitives below, one per context (a context's calls do not
// overlap): look-back words tagged with the launch's epoch, the ticket
// counter and two digit histogram buffers, each cleared while the other is in
// use (`torn`: a sort was cut short, clear both).
struct SortSpace {
    DevBuf status, ticket, hist;
    unsigned epoch = 0;
    bool flip = false, torn = false;
};

// out[i] = sum(in[0..i)), returns nothing; total written to *total_dev if
// non-null (device pointer).  The u64 form's tmp must hold scan_tmp_bytes(n).
size_t scan_tmp_bytes(int64_t n);
void exclusive_scan_u32(SortSpace& ws, const uint32_t* in, uint32_t* out, int64_t n,
                        uint32_t* total_dev, hipStream_t s);
void exclusive_scan_u64(const uint64_t* in, uint64_t* out, int64_t n, uint64_t* total_dev,
                        void* tmp, hipStream_t s);

// Stable sort of n (key, value) pairs by the 8-bit digits of key that hold a
// bit of mask (the others are known to be constant), with no host round
// trip.  iota: the values are the positions 0 .. n - 1 (vals is written, not
// read).  in_alt: the sorted pairs ended in keys_alt / vals_alt.
struct SortJob {
    void* keys;
    void* keys_alt;
    uint32_t* vals;
    uint32_t* vals_alt;
    int64_t n;
    unsigned long long mask;
    bool iota;
    bool in_alt;
};
constexpr int SORT_JOBS = 5;
// uint64 keys of several arrays in the same launches
void radix_sort_jobs(SortSpace& ws, SortJob* jobs, int njobs, hipStream_t s);
// one array; returns in_alt
bool radix_sort_pairs(SortSpace& ws, uint64_t* keys, uint32_t* vals, uint64_t* keys_alt,
                      uint32_t* vals_alt, int64_t n, unsigned long long bit_mask, bool iota,
                      hipStream_t s);
bool radix_sort_pairs(SortSpace& ws, uint32_t* keys, uint32_t* vals, uint32_t* keys_alt,
                      uint32_t* vals_alt, int64_t n, unsigned long long bit_mask, bool iota,
                      hipStream_t s);

// Sorted keys -> unique keys, run starts (n_unique + 1 entries, last = n)
// and the number of unique keys (device scalar).
void run_length_encode(SortSpace& ws, const uint64_t* keys, int64_t n, uint64_t* unique_keys,
                       uint32_t* run_start, uint32_t* n_unique_dev, hipStream_t s);

// every bit below `bits`
inline unsigned long long low_bits(int bits)
{
    return bits >= 64 ? ~0ull : (1ull << bits) - 1ull;
}

} // namespace ipcg
