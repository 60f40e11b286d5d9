// LDS pieces shared by the kernels that rank columns with bitmaps and bucket
// contributions by output (rmed.hip, btile.hip).
#pragma once
#include "brm_device.h"

namespace brm {

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
}

// Bits of w below bit b (b taken mod 32).
__device__ __forceinline__ int popc_below(unsigned w, unsigned b) {
    return __popc(__builtin_amdgcn_ubfe(w, 0u, b & 31u));
}

// Eight list ids of an LDS bucket (ids below 64, one byte each), from any byte.
__device__ __forceinline__ uint64_t ids8(const unsigned char* p) {
    uint64_t w;
    __builtin_memcpy(&w, p, 8);
    return w;
}

// Orders a bucket by list id (ids below 64).
__device__ inline void bucket_order(unsigned char* lp, double* val, int m) {
    for (int t = 1; t < m; ++t) {
        const int l = lp[t];
        const double x = val[t];
        int u = t;
        for (; u > 0 && (int)lp[u - 1] > l; --u) {
            lp[u] = lp[u - 1];
            val[u] = val[u - 1];
        }
        lp[u] = (unsigned char)l;
        val[u] = x;
    }
}

// Sum of one bucket (m >= 3 contributions from distinct lists, ids below 64)
// as the aligned tree over list positions: one pass over the contributions in
// list order with the pending left subtrees on a stack.  The pending heights
// shrink towards the top of the stack, so one bit mask holds them; when the
// next list first differs from the last one at bit d, the pending subtrees
// below height d are complete on its left and are added (left + right), and
// the sum waits at height d.  The stack's top is in a register, the rest
// takes the place of contributions already read (LDS): a push is about a
// dozen instructions (with one register per height every push selects over
// all heights), and the only LDS read it may wait for is a second pop's.  Ids
// come eight at a time, the next value one push ahead.
// The caller's ids may be read up to 7 bytes past the bucket.
__device__ inline double rb_bucket_sum(unsigned char* lp, double* val, int m) {
    // contributions placed by one register step of a wavefront may be out of
    // list order: ids of a bucket in order ascend bytewise, which the guard
    // bits of one subtraction show for eight pairs at once
    bool ordered = true;
    for (int t = 0; t + 1 < m; t += 7) {
        const uint64_t w = ids8(lp + t);
        const uint64_t d = ((w >> 8) | 0x8080808080808080ull) - (w & 0x00ffffffffffffffull);
        const int n = min(m - 1 - t, 7);  // pairs (t, t + 1) .. of this step
        ordered = ordered && (~d & (0x8080808080808080ull >> (8 * (8 - n)))) == 0ull;
    }
    if (!ordered) bucket_order(lp, val, m);
    uint64_t w = ids8(lp);
    int prev = (int)(w & 0xffu), depth = 0;
    double cur = val[0], nxt = val[1], top = 0.0;
    unsigned pend = 0u;
    for (int t = 1; t < m; ++t) {
        w = (t & 7) ? w >> 8 : ids8(lp + t);
        const int l = (int)(w & 0xffu);
        const double x = nxt;
        nxt = val[min(t + 1, m - 1)];
        const unsigned bit = 1u << (31 - __clz(prev ^ l));
        unsigned low = pend & (bit - 1u);
        pend = (pend & ~(bit - 1u)) | bit;
        while (low) {
            cur = fadd(top, cur);
            low &= low - 1u;
            if (--depth > 0) top = val[depth - 1];
        }
        if (depth > 0) val[depth - 1] = top;
        top = cur;
        ++depth;
        cur = x;
        prev = l;
    }
    while (depth > 0) {
        cur = fadd(top, cur);
        if (--depth > 0) top = val[depth - 1];
    }
    return cur;
}

}  // namespace brm
