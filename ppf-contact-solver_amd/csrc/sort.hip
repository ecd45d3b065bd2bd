// sort.hip -- stable LSD radix sort of (uint32 key, uint32 value) pairs.
//
// 8-bit digits, one histogram + one scatter kernel per digit. Stability comes
// from ranking inside a tile in input order: each 64-pair round of a wave is
// ranked with ballots (8 ballots give every lane the mask of lanes holding the
// same digit), and per-wave digit places in LDS carry the order across rounds
// and waves. Replaces the reference's 4-bit,
// 8-pass sort (kernels/radix_sort.cu:22-178): 30-bit Morton keys need 4 passes.
#include "scan.hpp"
#include "sort.hpp"

namespace ppf {

namespace {

constexpr int kThreads = 256;
constexpr int kWaves = kThreads / kWave;
constexpr int kTile = 4 * kThreads; // the small tile
// Tiles of 16 rounds once they fill the chip (1,048,576 pairs: 256 of them): a
// digit's run in a tile is then 16 pairs, two cache lines of keys and values,
// and the scans read a quarter of the counts. Below, tiles of 4 rounds.
constexpr int kBigRounds = 16;
constexpr size_t kBigSort = 256 * (size_t)kBigRounds * kThreads;

// A wave's count of digit d into h: one addition when all its pairs share a
// digit (the upper digits of sorted pairs), where 64 would wait for each other.
__device__ inline void count_digit(uint32_t *h, uint32_t d, bool valid) {
    const uint64_t all = __ballot(valid);
    if (all == 0) {
        return;
    }
    const uint32_t d0 = __shfl(d, __builtin_ctzll(all));
    if (__ballot(valid && d == d0) == all) {
        if ((threadIdx.x & (kWave - 1)) == 0) {
            atomicAdd(h + d0, (uint32_t)__popcll(all));
        }
    } else if (valid) {
        atomicAdd(h + d, 1u);
    }
}

template <int ROUNDS>
__global__ __launch_bounds__(kThreads) void k_digit_hist(const uint32_t *__restrict__ keys,
                                                         size_t n, uint32_t shift, uint32_t ntiles,
                                                         uint32_t *__restrict__ hist) {
    __shared__ uint32_t h[kWaves][256];
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
        h[q][threadIdx.x] = 0;
    }
    __syncthreads();
    const size_t base = (size_t)blockIdx.x * ROUNDS * kThreads + threadIdx.x;
    uint32_t k[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const size_t i = base + (size_t)r * kThreads;
        k[r] = i < n ? keys[i] : 0u;
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        count_digit(h[threadIdx.x / kWave], (k[r] >> shift) & 0xffu,
                    base + (size_t)r * kThreads < n);
    }
    __syncthreads();
    uint32_t sum = 0;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
        sum += h[q][threadIdx.x];
    }
    hist[(size_t)threadIdx.x * ntiles + blockIdx.x] = sum;
}

// A tile's pairs, ranked as in k_sort_one (a wave owns a contiguous segment),
// are put in digit order in LDS and leave from there, so that a digit's pairs
// are written as one run: 3M pairs 56 -> 20 us a pass (2.4 TB/s), 0.1M 11 -> 9.
template <int ROUNDS>
__global__ __launch_bounds__(kThreads) void k_digit_scatter(
    const uint32_t *__restrict__ keys, const uint32_t *__restrict__ vals, size_t n, uint32_t shift,
    uint32_t ntiles, const uint32_t *__restrict__ hist_scan, uint32_t *__restrict__ okeys,
    uint32_t *__restrict__ ovals) {
    __shared__ uint32_t lk[ROUNDS * kThreads], lv[ROUNDS * kThreads];
    __shared__ uint32_t cnt[kWaves][256]; // per wave and digit: counts, then places
    __shared__ uint32_t to[256];          // output place of LDS place 0, per digit
    __shared__ uint32_t wsum[kWaves];
    const uint32_t lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
    const size_t tile = (size_t)blockIdx.x * ROUNDS * kThreads;
    const size_t base = tile + w * ROUNDS * kWave + lane;
    uint32_t k[ROUNDS], v[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const size_t i = base + r * kWave;
        k[r] = i < n ? keys[i] : 0u;
        v[r] = i < n ? vals[i] : 0u;
    }
    const uint32_t first = hist_scan[(size_t)threadIdx.x * ntiles + blockIdx.x];
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
        cnt[q][threadIdx.x] = 0;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        count_digit(cnt[w], (k[r] >> shift) & 0xffu, base + r * kWave < n);
    }
    __syncthreads();
    uint32_t total = 0;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
        total += cnt[q][threadIdx.x];
    }
    uint32_t incl = total;
#pragma unroll
    for (int off = 1; off < kWave; off <<= 1) {
        const uint32_t t = __shfl_up(incl, off, kWave);
        if (lane >= (uint32_t)off) {
            incl += t;
        }
    }
    if (lane == kWave - 1) {
        wsum[w] = incl;
    }
    __syncthreads();
    uint32_t run = incl - total;
    for (uint32_t q = 0; q < w; ++q) {
        run += wsum[q];
    }
    to[threadIdx.x] = first - run;
#pragma unroll
    for (int q = 0; q < kWaves; ++q) {
        const uint32_t c = cnt[q][threadIdx.x];
        cnt[q][threadIdx.x] = run;
        run += c;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const bool valid = base + r * kWave < n;
        const uint32_t d = (k[r] >> shift) & 0xffu;
        uint64_t peers = __ballot(valid);
#pragma unroll
        for (int b = 0; b < 8; ++b) {
            const uint64_t m = __ballot(valid && ((d >> b) & 1u));
            peers &= ((d >> b) & 1u) ? m : ~m;
        }
        if (valid) {
            const uint32_t at = cnt[w][d] + __popcll(peers & below);
            lk[at] = k[r];
            lv[at] = v[r];
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (valid && (peers & below) == 0) {
            cnt[w][d] += (uint32_t)__popcll(peers);
        }
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const uint32_t j = r * kThreads + threadIdx.x;
        if (tile + j < n) {
            const uint32_t key = lk[j], pos = to[(key >> shift) & 0xffu] + j;
            okeys[pos] = key;
            ovals[pos] = lv[j];
        }
    }
}

// The whole sort of up to 8,192 pairs in one workgroup. Every wave owns a
// contiguous segment, 64 pairs a round in registers; a pass counts digits per
// wave, scans the counts by (digit, wave), and ranks each wave's pairs in
// order with ballots, so the order is the stable one of the passes above.
// Bound by latency, LDS and ballots of one CU: a pass over 8,192 pairs is 13 us,
// over 4,096 pairs 7, against four launches of 2 to 8 us with their gaps, 20 us.
// 16 rounds (16,384 pairs) took 24 us a pass and leave the line at 8,192.
constexpr int kOneThreads = 1024;
constexpr int kOneWaves = kOneThreads / kWave;
constexpr size_t kOneMax = 8 * kOneThreads;

template <int ROUNDS>
__global__ __launch_bounds__(kOneThreads) void k_sort_one(uint32_t *__restrict__ keys,
                                                          uint32_t *__restrict__ vals, uint32_t n,
                                                          uint32_t key_bits) {
    __shared__ uint32_t lk[ROUNDS * kOneThreads], lv[ROUNDS * kOneThreads];
    __shared__ uint32_t cnt[kOneWaves][256]; // per wave and digit: counts, then places
    __shared__ uint32_t wsum[4];
    const uint32_t lane = threadIdx.x & (kWave - 1), w = threadIdx.x / kWave;
    const uint64_t below = lane == 0 ? 0ull : (~0ull >> (kWave - lane));
    const uint32_t base = w * ROUNDS * kWave + lane;
    uint32_t k[ROUNDS], v[ROUNDS];
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const uint32_t i = base + r * kWave;
        k[r] = i < n ? keys[i] : 0u;
        v[r] = i < n ? vals[i] : 0u;
    }
    for (uint32_t shift = 0; shift < key_bits; shift += 8) {
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            cnt[w][lane + q * kWave] = 0;
        }
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            if (base + r * kWave < n) {
                atomicAdd(&cnt[w][(k[r] >> shift) & 0xffu], 1u);
            }
        }
        __syncthreads();
        // digit d's threads (the first four waves): total over the waves, scan
        uint32_t total = 0, incl = 0;
        if (threadIdx.x < 256) {
#pragma unroll
            for (int q = 0; q < kOneWaves; ++q) {
                total += cnt[q][threadIdx.x];
            }
            incl = total;
#pragma unroll
            for (int off = 1; off < kWave; off <<= 1) {
                const uint32_t t = __shfl_up(incl, off, kWave);
                if (lane >= (uint32_t)off) {
                    incl += t;
                }
            }
            if (lane == kWave - 1) {
                wsum[w] = incl;
            }
        }
        __syncthreads();
        if (threadIdx.x < 256) {
            uint32_t run = incl - total;
            for (uint32_t q = 0; q < w; ++q) {
                run += wsum[q];
            }
#pragma unroll
            for (int q = 0; q < kOneWaves; ++q) {
                const uint32_t c = cnt[q][threadIdx.x];
                cnt[q][threadIdx.x] = run;
                run += c;
            }
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const bool valid = base + r * kWave < n;
            const uint32_t d = (k[r] >> shift) & 0xffu;
            uint64_t peers = __ballot(valid);
#pragma unroll
            for (int b = 0; b < 8; ++b) {
                const uint64_t m = __ballot(valid && ((d >> b) & 1u));
                peers &= ((d >> b) & 1u) ? m : ~m;
            }
            if (valid) {
                const uint32_t at = cnt[w][d] + __popcll(peers & below);
                lk[at] = k[r];
                lv[at] = v[r];
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            if (valid && (peers & below) == 0) {
                cnt[w][d] += (uint32_t)__popcll(peers);
            }
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        }
        __syncthreads();
#pragma unroll
        for (int r = 0; r < ROUNDS; ++r) {
            const uint32_t i = base + r * kWave;
            if (i < n) {
                k[r] = lk[i];
                v[r] = lv[i];
            }
        }
        __syncthreads(); // the places and pairs are read before the next pass
    }
#pragma unroll
    for (int r = 0; r < ROUNDS; ++r) {
        const uint32_t i = base + r * kWave;
        if (i < n) {
            keys[i] = k[r];
            vals[i] = v[r];
        }
    }
}

size_t tiles(size_t n) { return (n + kTile - 1) / kTile; }

} // namespace

size_t radix_sort_scratch_words(size_t n) {
    const size_t h = 256 * tiles(n);
    return 2 * n + 2 * h + scan_scratch_words(h);
}

hipError_t radix_sort_pairs(uint32_t *keys, uint32_t *vals, size_t n,
                            uint32_t key_bits, uint32_t *scratch,
                            hipStream_t s) {
    if (n <= 1) {
        return hipSuccess;
    }
    if (n <= kOneMax && key_bits > 0) {
        if (n <= 4 * kOneThreads) {
            k_sort_one<4><<<1, kOneThreads, 0, s>>>(keys, vals, (uint32_t)n, key_bits);
        } else {
            k_sort_one<8><<<1, kOneThreads, 0, s>>>(keys, vals, (uint32_t)n, key_bits);
        }
        return hipGetLastError();
    }
    const bool big = n >= kBigSort;
    const uint32_t nt = (uint32_t)(big ? (n + kBigRounds * kThreads - 1) / (kBigRounds * kThreads)
                                       : tiles(n));
    const size_t h = 256 * (size_t)nt;
    uint32_t *k2 = scratch, *v2 = scratch + n;
    uint32_t *hist = scratch + 2 * n, *hscan = hist + h, *sscr = hscan + h;
    uint32_t *ka = keys, *va = vals, *kb = k2, *vb = v2;
    const uint32_t passes = (key_bits + 7) / 8;
    for (uint32_t p = 0; p < passes; ++p) {
        const uint32_t shift = 8 * p;
        if (big) {
            k_digit_hist<kBigRounds><<<nt, kThreads, 0, s>>>(ka, n, shift, nt, hist);
        } else {
            k_digit_hist<4><<<nt, kThreads, 0, s>>>(ka, n, shift, nt, hist);
        }
        hipError_t e = hipGetLastError();
        if (e != hipSuccess) {
            return e;
        }
        e = exclusive_scan_u32(hist, hscan, h, sscr, s);
        if (e != hipSuccess) {
            return e;
        }
        if (big) {
            k_digit_scatter<kBigRounds>
                <<<nt, kThreads, 0, s>>>(ka, va, n, shift, nt, hscan, kb, vb);
        } else {
            k_digit_scatter<4><<<nt, kThreads, 0, s>>>(ka, va, n, shift, nt, hscan, kb, vb);
        }
        e = hipGetLastError();
        if (e != hipSuccess) {
            return e;
        }
        std::swap(ka, kb);
        std::swap(va, vb);
    }
    if (ka != keys) {
        hipError_t e = hipMemcpyAsync(keys, ka, n * sizeof(uint32_t),
                                      hipMemcpyDeviceToDevice, s);
        if (e != hipSuccess) {
            return e;
        }
        return hipMemcpyAsync(vals, va, n * sizeof(uint32_t),
                              hipMemcpyDeviceToDevice, s);
    }
    return hipSuccess;
}

} // namespace ppf
