// CSR transpose on the device (the step before P^T * (A*P) in the AMG
// Galerkin product; the reference forms transposes on the host by sorting,
// Existing-SpGEMM/inc/convert.h:6-58).
//
// Entry e of row r becomes entry (col[e], r) of the transpose.  A stable
// radix sort of the entry indices by column (hipCUB) keeps the rows of every
// output row in increasing order, so the result is the canonical CSR of A^T;
// the output row pointer is searched in the sorted columns.  (For an
// aggregation of 884,736 rows of one entry, counting the columns by atomics, a
// wavefront per row, took 145 us and the scan of the counts with its launches
// 25; the entries' rows, lanes by the average row and long rows apart, and the
// search take 5 and 7.)
#include <hipcub/hipcub.hpp>

#include <algorithm>

#include "brm_device.h"
#include "pipeline.h"

namespace brm {
namespace {

constexpr int TP_NT = 256;

// Rows of more entries than this are written in pieces, by wavefronts of their
// own, so that no lane has more than this many to write (a row of 10^6 entries
// among 10^6 rows of one took 30 ms by the one lane that such rows get; the whole
// transpose now takes 0.22).
constexpr int TP_LONG = 512;
constexpr int64_t TP_ROW_BLOCKS = 1 << 22;  // a launch stays below 2^32 threads

// Row of entry x: the least r with rpt[r + 1] > x (64-way search by a wavefront).
__device__ __forceinline__ int tp_row_of(const int* __restrict__ rpt, int M, int x) {
    int lo = 0, hi = M;  // rpt[lo] <= x < rpt[hi]
    while (hi - lo > 1) {
        const int step = (int)(((int64_t)hi - lo + BRM_WAVE - 1) / BRM_WAVE);
        const int64_t p = lo + (int64_t)(lane_id() + 1) * step;
        const int f = __ffsll((long long)__ballot(p >= hi || rpt[p] > x)) - 1;
        hi = (int)min((int64_t)hi, lo + (int64_t)(f + 1) * step);
        lo += f * step;
    }
    return lo;
}

// Row and index of every entry.  The first workgroups: the entries of long
// rows, a wavefront each from entry c * TP_LONG on (a long row holds such an entry; the
// wavefront of the first also writes those before it).  The other workgroups:
// the other rows, L lanes each.
template <int L>
__global__ __launch_bounds__(TP_NT) void k_tp_entries(const int* __restrict__ rpt, int M, int nnz, int piece_blocks,
                                                      int* __restrict__ row_of, int* __restrict__ idx) {
    if ((int)blockIdx.x < piece_blocks) {
        const int64_t x = ((int64_t)blockIdx.x * (TP_NT / BRM_WAVE) + threadIdx.x / BRM_WAVE) * TP_LONG;
        if (x >= nnz) return;
        const int r = tp_row_of(rpt, M, (int)x);
        const int e0 = rpt[r], e1 = rpt[r + 1];
        if (e1 - e0 <= TP_LONG) return;
        const int64_t end = min((int64_t)e1, x + TP_LONG);
        for (int64_t e = (x - e0 < TP_LONG ? e0 : x) + lane_id(); e < end; e += BRM_WAVE) {
            row_of[e] = r;
            idx[e] = (int)e;
        }
        return;
    }
    const int64_t blocks = (int64_t)gridDim.x - piece_blocks;
    for (int64_t r = ((int64_t)blockIdx.x - piece_blocks) * (TP_NT / L) + threadIdx.x / L; r < M;
         r += blocks * (TP_NT / L)) {
        const int e0 = rpt[r], n = rpt[r + 1] - e0;
        if (n > TP_LONG) continue;
        for (int k = (int)(threadIdx.x % L); k < n; k += L) {
            row_of[e0 + k] = (int)r;
            idx[e0 + k] = e0 + k;
        }
    }
}

template <int L>
void launch_entries(const int* rpt, int M, int64_t nnz, int* row_of, int* idx, hipStream_t s) {
    constexpr int R = TP_NT / L, PIECE = TP_NT / BRM_WAVE * TP_LONG;
    const int64_t rows = std::min(((int64_t)M + R - 1) / R, TP_ROW_BLOCKS);
    const int pieces = nnz > TP_LONG ? (int)((nnz + PIECE - 1) / PIECE) : 0;
    k_tp_entries<L><<<(unsigned)(pieces + rows), TP_NT, 0, s>>>(rpt, M, (int)nnz, pieces, row_of, idx);
}

// Row pointer of the transpose: the first of the n sorted columns that is at
// least c, for every c up to N.
__global__ __launch_bounds__(TP_NT) void k_tp_rpt(const int* __restrict__ keys, int n, int N, int* __restrict__ trpt) {
    const int64_t c = (int64_t)blockIdx.x * TP_NT + threadIdx.x;
    if (c > N) return;
    int lo = 0, hi = n;
    while (lo < hi) {
        const int mid = lo + ((hi - lo) >> 1);
        if (keys[mid] < c) lo = mid + 1;
        else hi = mid;
    }
    trpt[c] = lo;
}

__global__ __launch_bounds__(TP_NT) void k_tp_gather(const int* __restrict__ perm, int64_t nnz,
                                                     const int* __restrict__ row_of, const double* __restrict__ val,
                                                     int* __restrict__ tcol, double* __restrict__ tval) {
    const int64_t k = (int64_t)blockIdx.x * TP_NT + threadIdx.x;
    if (k >= nnz) return;
    const int e = perm[k];
    tcol[k] = row_of[e];
    tval[k] = val[e];
}

unsigned tp_blocks(int64_t n) { return (unsigned)((n + TP_NT - 1) / TP_NT); }

int transpose_dev(const int* rpt, const int* col, const double* val, int64_t nnz, int M, int N, int* trpt,
                  int* tcol, double* tval, hipStream_t s) {
    Scratch sc;
    int *row_of, *perm_in, *perm_out, *keys_out, *derr;
    BRMC(sc.alloc(&derr, 1, "error flag"));
    BRMC(sc.alloc(&row_of, nnz, "row ids"));
    BRMC(sc.alloc(&perm_in, nnz, "entry ids"));
    BRMC(sc.alloc(&perm_out, nnz, "sorted entry ids"));
    BRMC(sc.alloc(&keys_out, nnz, "sorted columns"));
    HIPC(launch_fill_i32(derr, 1, 0, s));
    // the input must be well formed: row pointers and column range
    RowArgs a{};
    a.arpt = rpt;
    a.acol = col;
    a.M = M;
    a.K = N;
    HIPC(launch_validate(a, nnz, -1, derr, s));
    BRMC(check_dev_err(derr, s, "transpose input"));
    if (nnz > 0) {
        // lanes per row: a power of two of about its entries
        const int64_t avg = nnz / M;
        if (avg <= 2) launch_entries<1>(rpt, M, nnz, row_of, perm_in, s);
        else if (avg <= 8) launch_entries<4>(rpt, M, nnz, row_of, perm_in, s);
        else if (avg <= 32) launch_entries<16>(rpt, M, nnz, row_of, perm_in, s);
        else launch_entries<BRM_WAVE>(rpt, M, nnz, row_of, perm_in, s);
        HIPC(hipGetLastError());
        int end_bit = 1;
        while (end_bit < 31 && ((int64_t)1 << end_bit) < N) ++end_bit;
        size_t tmp_bytes = 0;
        HIPC(hipcub::DeviceRadixSort::SortPairs(nullptr, tmp_bytes, col, keys_out, perm_in, perm_out, (int)nnz, 0,
                                                end_bit, s));
        unsigned char* tmp;
        BRMC(sc.alloc(&tmp, (int64_t)tmp_bytes, "sort scratch"));
        HIPC(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, col, keys_out, perm_in, perm_out, (int)nnz, 0,
                                                end_bit, s));
        k_tp_gather<<<tp_blocks(nnz), TP_NT, 0, s>>>(perm_out, nnz, row_of, val, tcol, tval);
        HIPC(hipGetLastError());
    }
    k_tp_rpt<<<tp_blocks((int64_t)N + 1), TP_NT, 0, s>>>(keys_out, (int)nnz, N, trpt);
    HIPC(hipGetLastError());
    HIPC(hipStreamSynchronize(s));
    return BRM_OK;
}

}  // namespace
}  // namespace brm

using namespace brm;

extern "C" int brm_csr_transpose_dev(const int* rpt, const int* col, const double* val, int64_t nnz, int M, int N,
                                     int* trpt, int* tcol, double* tval, void* stream) {
    if (M < 0 || N < 0 || nnz < 0 || nnz > INT32_MAX || !trpt || (M > 0 && !rpt) ||
        (nnz > 0 && (!col || !val || !tcol || !tval))) {
        set_err("invalid argument");
        return BRM_E_INVALID;
    }
    BRMC(use_device());
    const int st = transpose_dev(rpt, col, val, nnz, M, N, trpt, tcol, tval, (hipStream_t)stream);
    dev_flush_deferred();
    return st;
}
