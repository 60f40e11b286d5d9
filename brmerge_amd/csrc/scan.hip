// Device-wide exclusive prefix sums (int64 output), reduce-then-scan.
//
// Replaces opt_prefix_sum / para_prefix_sum (BRMerge-SpGEMM/inc/spgemm.h:147-187)
// and fuses the per-A-entry product count of compute_flop (spgemm.h:39-41):
// scan_alen() turns each A entry j into alen[j] = |B row acol[j]| on the fly,
// so out[j] is the global index of entry j's first intermediate product and
// out[arpt[i+1]] - out[arpt[i]] is row i's product count.
//
// Each block owns a tile of consecutive elements, a quarter to each wavefront.
// A thread's elements are loaded before the first is used (the product counts
// are dependent pairs of loads), each wavefront scans 64 at a time with DPP
// adds, and the block meets twice per tile, not twice per 256 elements.  Block
// totals are scanned by every block for itself, or by a single block.
//
// The product counts of the first pass are kept, as 32-bit values in the first
// half of the tile's place in out[], and read from there by the second: they
// cost a random access of B's row pointer each, which bounds the first pass.
// 18 M entries over 1.5 M rows: two passes of 124 and 159 us without, 138, 8
// (tile totals) and 48 us with it; 600,000 entries: 9 and 12 us, now 6 and 10.
#include "brm_device.h"
#include "brm_internal.h"

namespace brm {
namespace {

constexpr int SCAN_NT = 256;
constexpr int SCAN_NW = SCAN_NT / BRM_WAVE;
constexpr int SCAN_PNT = 1024;  // of the scan of the tile totals

// A column outside [0, K) counts 0 products (validation reports it), so no
// B row pointer outside the array is read.
struct AlenF {
    static constexpr bool STASH = true;  // the first pass leaves f in out[]
    const int* acol;
    const int* brpt;
    int K;
    // the elements j[0 .. N), each below n or skipped
    template <int N, typename T>
    __device__ void load(const int64_t (&j)[N], int64_t n, T (&x)[N]) const {
        int c[N];
#pragma unroll
        for (int i = 0; i < N; ++i) c[i] = acol[min(j[i], n - 1)];
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const bool ok = j[i] < n && (unsigned)c[i] < (unsigned)K;
            const int r = ok ? c[i] : 0;
            const int len = K > 0 ? brpt[r + 1] - brpt[r] : 0;
            x[i] = ok ? (T)len : (T)0;
        }
    }
};
// Array elements.
struct ArrayF {
    static constexpr bool STASH = false;
    const int64_t* p;
    template <int N, typename T>
    __device__ void load(const int64_t (&j)[N], int64_t n, T (&x)[N]) const {
#pragma unroll
        for (int i = 0; i < N; ++i) x[i] = j[i] < n ? p[j[i]] : 0;
    }
};
// Element i of this thread's share of the tile at base.
template <int ITEMS>
__device__ __forceinline__ void scan_elements(int64_t base, int64_t (&j)[ITEMS]) {
    const int64_t b = base + (int64_t)(threadIdx.x / BRM_WAVE) * (ITEMS * BRM_WAVE) + lane_id();
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) j[i] = b + i * BRM_WAVE;
}

template <typename F, int ITEMS>
__global__ __launch_bounds__(SCAN_NT) void k_scan_reduce(F f, int64_t n, int64_t* part, int64_t* out) {
    __shared__ int64_t sm[SCAN_NW + 1];
    const int64_t base = (int64_t)blockIdx.x * (SCAN_NT * ITEMS);
    int64_t j[ITEMS];
    scan_elements(base, j);
    int64_t acc = 0;
    if constexpr (F::STASH) {
        int x[ITEMS];
        f.load(j, n, x);
        int* st = reinterpret_cast<int*>(out + base);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) {
            acc += x[i];
            if (j[i] < n) st[j[i] - base] = x[i];
        }
    } else {
        int64_t x[ITEMS];
        f.load(j, n, x);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) acc += x[i];
    }
    const int64_t tot = block_sum<SCAN_NT>(acc, sm);
    if (threadIdx.x == 0) part[blockIdx.x] = tot;
}

// The tile's exclusive prefixes, from `carry` on.  Returns the tile's total.
template <int NT, typename F, int ITEMS>
__device__ __forceinline__ int64_t scan_tile(F f, int64_t n, int64_t base, int64_t carry, int64_t* out, int64_t* sm) {
    int64_t j[ITEMS], x[ITEMS];
    scan_elements(base, j);
    if constexpr (F::STASH) {
        const int* st = reinterpret_cast<const int*>(out + base);
#pragma unroll
        for (int i = 0; i < ITEMS; ++i) x[i] = j[i] < n ? st[j[i] - base] : 0;
    } else {
        f.load(j, n, x);
    }
    int64_t run = 0;  // of this wavefront, uniform
#pragma unroll
    for (int i = 0; i < ITEMS; ++i) {
        const int64_t inc = wave_incl_scan(x[i]);
        x[i] = run + inc - x[i];
        run += wave_last(inc);
    }
    const int w = threadIdx.x / BRM_WAVE;
    if (lane_id() == 0) sm[w] = run;
    __syncthreads();  // every element of the tile has been read, too
    int64_t before = carry, tot = 0;
#pragma unroll
    for (int i = 0; i < NT / BRM_WAVE; ++i) {
        before += i < w ? sm[i] : 0;
        tot += sm[i];
    }
#pragma unroll
    for (int i = 0; i < ITEMS; ++i)
        if (j[i] < n) out[j[i]] = before + x[i];
    return tot;
}

// Exclusive scan of part[0..nb) in place; part[nb] = total.  One block.
__global__ __launch_bounds__(SCAN_PNT) void k_scan_partials(int64_t* part, int64_t nb) {
    __shared__ int64_t sm[SCAN_PNT / BRM_WAVE + 1];
    constexpr int ITEMS = 8;
    int64_t carry = 0;
    for (int64_t base = 0; base < nb; base += SCAN_PNT * ITEMS) {
        carry += scan_tile<SCAN_PNT, ArrayF, ITEMS>(ArrayF{part}, nb, base, carry, part, sm);
        __syncthreads();  // sm is written again
    }
    if (threadIdx.x == 0) part[nb] = carry;
}

template <typename F, int ITEMS>
__global__ __launch_bounds__(SCAN_NT) void k_scan_down(F f, int64_t n, const int64_t* part, int64_t nb,
                                                       int64_t* out) {
    __shared__ int64_t sm[SCAN_NW + 1];
    scan_tile<SCAN_NT, F, ITEMS>(f, n, (int64_t)blockIdx.x * (SCAN_NT * ITEMS), part[blockIdx.x], out, sm);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = part[nb];
}

// Down pass that also forms its own block's carry: the sum of the tile
// totals part[0 .. blockIdx.x), reduced by the block (for up to
// SCAN_FUSE_TILES tiles, so that this costs a few loads per thread).  Saves
// the one-block scan of the tile totals and its launch.
constexpr int64_t SCAN_FUSE_TILES = 8192;
template <typename F, int ITEMS>
__global__ __launch_bounds__(SCAN_NT) void k_scan_down_fused(F f, int64_t n, const int64_t* part, int64_t* out) {
    __shared__ int64_t sm[SCAN_NW + 1], sm2[SCAN_NW + 1];
    int64_t pre = 0;
    for (int64_t b = threadIdx.x; b < blockIdx.x; b += SCAN_NT) pre += part[b];
    const int64_t carry = block_sum<SCAN_NT>(pre, sm);
    const int64_t tot = scan_tile<SCAN_NT, F, ITEMS>(f, n, (int64_t)blockIdx.x * (SCAN_NT * ITEMS), carry, out, sm2);
    if (blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) out[n] = carry + tot;
}

__global__ void k_zero1(int64_t* out) { out[0] = 0; }

template <typename F, int ITEMS>
hipError_t scan_impl(F f, int64_t n, int64_t* out, hipStream_t s) {
    constexpr int64_t TILE = SCAN_NT * ITEMS;
    const int64_t nb = (n + TILE - 1) / TILE;
    int64_t* part = (int64_t*)dev_alloc(sizeof(int64_t) * (size_t)(nb + 1));
    if (!part) return hipErrorOutOfMemory;
    {
        ProfScope ps_("k_scan_reduce", s);
        k_scan_reduce<F, ITEMS><<<(unsigned)nb, SCAN_NT, 0, s>>>(f, n, part, out);
    }
    if (nb <= SCAN_FUSE_TILES) {
        ProfScope ps_("k_scan_down", s);
        k_scan_down_fused<F, ITEMS><<<(unsigned)nb, SCAN_NT, 0, s>>>(f, n, part, out);
    } else {
        {
            ProfScope ps_("k_scan_partials", s);
            k_scan_partials<<<1, SCAN_PNT, 0, s>>>(part, nb);
        }
        ProfScope ps_("k_scan_down", s);
        k_scan_down<F, ITEMS><<<(unsigned)nb, SCAN_NT, 0, s>>>(f, n, part, nb, out);
    }
    hipError_t e = hipGetLastError();
    dev_defer_free(part);  // still referenced by the queued kernels
    return e;
}

// Tiles of 1,024 elements while those are at most two per CU, so that a short
// scan is spread over the chip (26 scans of a served batch's 20 requests: 846 us
// in tiles of 4,096, now 357 us), else of 2,048 (of 4,096 a thread's elements
// take 98 registers and a batch of 192 products 20 us more).  In the
// fixed-buffer arena 4,096 always: the tile totals take its room.
template <typename F>
hipError_t scan(F f, int64_t n, int64_t* out, hipStream_t s) {
    if (n <= 0) {
        ProfScope ps_("k_zero1", s);
        k_zero1<<<1, 1, 0, s>>>(out);
        return hipGetLastError();
    }
    if (arena_remaining() >= 0) return scan_impl<F, 16>(f, n, out, s);
    return n <= 512 * 4 * SCAN_NT ? scan_impl<F, 4>(f, n, out, s) : scan_impl<F, 8>(f, n, out, s);
}

}  // namespace

hipError_t scan_alen(const int* acol, const int* brpt, int K, int64_t n, int64_t* out, hipStream_t s) {
    return scan(AlenF{acol, brpt, K}, n, out, s);
}
hipError_t scan_i64(const int64_t* in, int64_t n, int64_t* out, hipStream_t s) {
    return scan(ArrayF{in}, n, out, s);
}

}  // namespace brm
