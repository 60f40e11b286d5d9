// Register merge of one short row (at most G products, one per lane of a
// group of G lanes), shared by the short tier (short.hip) and the fused
// small-product path (small.hip).
//
// Each lane holds one product (column, list position, value).  The products
// are first put in (column, position) order, equal columns adjacent and
// ordered by position:
//  - when the columns fit 32 - log2(G) bits, a bitonic sort of 32-bit keys
//    (column, lane) over the group's lanes -- lanes are in list order, so
//    within one column the lane order is the position order.  Every merge
//    begins with the mirrored exchange (lane i with lane K-1-i), so that all
//    exchanges ascend and one mask per lane bit selects the minimum or the
//    maximum by v_med3; the exchanges are DPP moves up to distance 15 and
//    ds_swizzle beyond.  Each sorted lane then fetches its value and position
//    from the lane its key names;
//  - otherwise a rank sort by 64-bit (column, position) keys (v_readlane
//    broadcasts, or shuffles inside a half-wavefront), and ds_permute moves
//    every lane's product to its rank.
// The merge tree of BRMerge (BRMerge-SpGEMM/inc/spgemm.h:639-707: lists
// paired (2j, 2j+1) level by level, odd list carried) is then evaluated
// column-wise.  Entry j of a column joins the entries before it at the level
// of the highest bit in which its position differs from that of entry j - 1
// (the node that holds both), so each entry's level is known from one
// neighbour; at level l the entries of that level add their value to the
// nearest live entry on their left, which keeps the sum.  Which lanes receive
// is found on the scalar unit, by the carries of one addition.  That is
// exactly the reference's value rule -- an aligned binary tree over list
// positions in which a node with one present child passes it through -- so
// the sums are bit-identical.
//
// Bound by vector instructions: the sort takes two per exchange (three to
// four as minimum, maximum and select) and a level a dozen (thirty when every
// lane looks up its next live lane's column and position).  A * P of a
// 27-point operator on 96^3 points with an aggregation, two rows of 27
// products per wavefront and pass: 365 vector instructions per pass before,
// 205 now.
#pragma once
#include "brm_device.h"
#include "bucket_sum.h"

#include <type_traits>

namespace brm {

__device__ __forceinline__ int permute_i32(int dst_lane, int x) {
    return __builtin_amdgcn_ds_permute(dst_lane << 2, x);
}
__device__ __forceinline__ double permute_f64(int dst_lane, double x) {
    int lo = __builtin_amdgcn_ds_permute(dst_lane << 2, __double2loint(x));
    int hi = __builtin_amdgcn_ds_permute(dst_lane << 2, __double2hiint(x));
    return __hiloint2double(hi, lo);
}

// x of lane (this lane ^ J), for the distances the sort uses.
template <int J>
__device__ __forceinline__ uint32_t xor_lanes(uint32_t x) {
    if constexpr (J == 1) {
        return (uint32_t)dpp_mov<0xB1, 0xF>((int)x, 0);  // quad_perm [1,0,3,2]
    } else if constexpr (J == 2) {
        return (uint32_t)dpp_mov<0x4E, 0xF>((int)x, 0);  // quad_perm [2,3,0,1]
    } else if constexpr (J == 3) {
        return (uint32_t)dpp_mov<0x1B, 0xF>((int)x, 0);  // quad_perm [3,2,1,0]
    } else if constexpr (J == 4) {
        return xor_lanes<3>(xor_lanes<7>(x));
    } else if constexpr (J == 7) {
        return (uint32_t)dpp_mov<0x141, 0xF>((int)x, 0);  // row_half_mirror
    } else if constexpr (J == 8) {
        return (uint32_t)dpp_mov<0x128, 0xF>((int)x, 0);  // row_ror:8
    } else if constexpr (J == 15) {
        return (uint32_t)dpp_mov<0x140, 0xF>((int)x, 0);  // row_mirror
    } else if constexpr (J < 32) {
        return (uint32_t)__builtin_amdgcn_ds_swizzle((int)x, 0x1F | (J << 10));  // bitmask mode, xor J
    } else {
        return (uint32_t)__builtin_amdgcn_ds_bpermute((lane_id() ^ J) << 2, (int)x);
    }
}

// One exchange at distance J: lanes with bit HALF of gl take the maximum.
template <int J, int HALF>
__device__ __forceinline__ uint32_t exchange(uint32_t key, int gl) {
    const uint32_t o = xor_lanes<J>(key);
    const uint32_t upper = (gl & HALF) ? 0xFFFFFFFFu : 0u;
    return max(min(key, o), min(max(key, o), upper));  // v_med3_u32
}

template <int J>
__device__ __forceinline__ void half_clean(uint32_t& key, int gl) {
    key = exchange<J, J>(key, gl);
    if constexpr (J > 1) half_clean<J / 2>(key, gl);
}

// Ascending sort of one key per lane over each group of G lanes.
template <int K, int G>
__device__ __forceinline__ void bitonic_sort(uint32_t& key, int gl) {
    key = exchange<K - 1, K / 2>(key, gl);
    if constexpr (K > 2) half_clean<K / 4>(key, gl);
    if constexpr (K < G) bitonic_sort<K * 2, G>(key, gl);
}

// Of two wavefront-uniform values the one of this lane's half (two vector
// instructions, where a select of two scalars takes three).
__device__ __forceinline__ uint32_t of_half(uint32_t lo, uint32_t hi, int gbase) {
    const uint32_t m = (uint32_t)-(gbase >> 5);
    return (lo & ~m) | (hi & m);
}

// The group's bits of a lane mask, and'ed with `with`: bit i is lane gbase + i.
template <int G>
__device__ __forceinline__ auto group_bits(uint64_t m, int gbase, std::conditional_t<G == BRM_WAVE, uint64_t, uint32_t> with) {
    if constexpr (G == BRM_WAVE) {
        return m & with;
    } else {
        const uint32_t h = (uint32_t)-(gbase >> 5);
        return ((uint32_t)m & (with & ~h)) | ((uint32_t)(m >> 32) & (with & h));
    }
}

// Lowest and highest set bit; any value when there is none.
__device__ __forceinline__ int low_bit(uint32_t x) {
    int r;
    asm("v_ffbl_b32 %0, %1" : "=v"(r) : "v"(x));
    return r;
}
__device__ __forceinline__ int high_bit(uint32_t x) {
    int r;
    asm("v_ffbh_u32 %0, %1" : "=v"(r) : "v"(x));
    return 31 - r;
}

// Number of set bits of m in the lanes below this one, of its group only.
template <int G>
__device__ __forceinline__ int group_rank(uint64_t m, int gbase) {
    const int r = (int)__builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0u));
    if constexpr (G == BRM_WAVE) return r;
    else return r - (int)of_half(0u, __popc((unsigned)m), gbase);
}

// Inclusive sum over the lanes of each group.
template <int G>
__device__ __forceinline__ int group_incl_scan(int x) {
    if constexpr (G == BRM_WAVE) return wave_incl_scan(x);
    x += dpp_take<0x111, 0xF>(x);  // row_shr:1
    x += dpp_take<0x112, 0xF>(x);  // row_shr:2
    x += dpp_take<0x114, 0xF>(x);  // row_shr:4
    x += dpp_take<0x118, 0xF>(x);  // row_shr:8
    return x + dpp_take<0x142, 0xA>(x);  // row_bcast15 into rows 1 and 3
}

// The list of each product lane: lists of one row (list q of the group in
// its lane q) are laid out one after the other over the group's lanes.
struct alignas(16) ListSlot {
    int q;       // list
    int rel;     // index in B of the product less its lane
    double av;   // A value
};
// ne: this lane's list is not empty and begins at product off < G.  ws: the
// wavefront's 64 slots in LDS.  Product lanes (below the row's products) get
// their list's slot; other lanes any slot.
template <int G>
__device__ __forceinline__ ListSlot list_of(ListSlot* ws, int gl, int gbase, bool ne, int off, int bst, double av) {
    ws[gbase + gl].q = -1;
    wave_lds_sync();
    if (ne) ws[gbase + off] = ListSlot{gl, bst - off, av};
    wave_lds_sync();
    const uint64_t begins = __ballot(ws[gbase + gl].q >= 0);
    // last list begin at or before this lane
    int s;
    if constexpr (G == BRM_WAVE) {
        const uint64_t b = begins & (~0ull >> (BRM_WAVE - 1 - gl));
        s = b ? 63 - __clzll((long long)b) : 0;
    } else {
        s = high_bit(group_bits<G>(begins, gbase, ~0u >> (31 - gl)));
    }
    const ListSlot r = ws[gbase + (s & (G - 1))];
    wave_lds_sync();
    return r;
}

// Whether columns below N fit the 32-bit sort keys of groups of G lanes
// (the all-ones key marks an empty lane).
template <int G>
__host__ __device__ constexpr bool short_keys_fit(int N) {
    return (int64_t)N < ((int64_t)1 << (32 - (G == 64 ? 6 : 5)));
}

// Result for the calling lane: its output entry (col, val) when alive, at
// position idx of the row; nout entries in all.  With NUMERIC false only
// nout is computed (the distinct columns).
struct ShortMerged {
    int col;
    double val;
    bool alive;
    int idx;
    int nout;
};

// Every lane of the wavefront calls this (groups of G lanes; G = 64 or 32).
// gl: lane within the group; gbase: the group's first lane; gmask: its
// lanes; act: the lane holds a product (gl < ip); ip: products of the group's
// row (uniform over the group; for G = 64, over the wavefront); narrow:
// short_keys_fit<G>(N) for the product's N (uniform over the wavefront).
template <bool NUMERIC, int G>
__device__ __forceinline__ ShortMerged short_merge(int col, int p, double val, bool act, int ip, int gl, int gbase,
                                                   uint64_t gmask, bool narrow) {
    const int lane = lane_id();
    constexpr int S = G == 64 ? 6 : 5;
    const bool alive = gl < ip;
    int pos;
    if (narrow) {
        uint32_t key = act ? (((uint32_t)col << S) | (uint32_t)gl) : 0xFFFFFFFFu;
        bitonic_sort<2, G>(key, gl);
        const int src = gbase + (int)(key & (G - 1));
        col = (int)(key >> S);
        if (!NUMERIC) {
            const int prv = __shfl(col, (lane + BRM_WAVE - 1) & (BRM_WAVE - 1), BRM_WAVE);
            ShortMerged r{};
            r.nout = __popcll(__ballot(alive && (gl == 0 || prv != col)) & gmask);
            return r;
        }
        pos = __builtin_amdgcn_ds_bpermute(src << 2, p);
        int lo = __builtin_amdgcn_ds_bpermute(src << 2, __double2loint(val));
        int hi = __builtin_amdgcn_ds_bpermute(src << 2, __double2hiint(val));
        val = __hiloint2double(hi, lo);
    } else {
        const uint64_t key = act ? (((uint64_t)(uint32_t)col << 32) | (uint32_t)p) : ~0ull;
        const uint32_t klo_me = (uint32_t)key, khi_me = (uint32_t)(key >> 32);
        int rank = 0;
        bool dup = false;
        if (G == BRM_WAVE) {
            const int n = __builtin_amdgcn_readfirstlane(ip);
            for (int k = 0; k < n; ++k) {
                const uint32_t klo = (uint32_t)__builtin_amdgcn_readlane((int)klo_me, k);
                const uint32_t khi = (uint32_t)__builtin_amdgcn_readlane((int)khi_me, k);
                const uint64_t kk = ((uint64_t)khi << 32) | klo;
                const bool lt = kk < key;
                rank += lt;
                dup |= lt && (khi == khi_me);
            }
        } else {
#pragma unroll 8
            for (int k = 0; k < G; ++k) {
                const uint32_t klo = (uint32_t)__shfl((int)klo_me, gbase + k, BRM_WAVE);
                const uint32_t khi = (uint32_t)__shfl((int)khi_me, gbase + k, BRM_WAVE);
                const uint64_t kk = ((uint64_t)khi << 32) | klo;
                const bool lt = kk < key;
                rank += lt;
                dup |= lt && (khi == khi_me);
            }
        }
        if (!NUMERIC) {
            ShortMerged r{};
            r.nout = __popcll(__ballot(act && !dup) & gmask);
            return r;
        }
        const int dst = act ? gbase + rank : lane;
        col = permute_i32(dst, col);
        pos = permute_i32(dst, p);
        val = permute_f64(dst, val);
    }

    // ---- the tree: lvl is the level at which this entry joins the one on its left
    const int pcol = dpp_mov<0x138, 0xF>(col, 0);  // wave_shr:1
    const int ppos = dpp_mov<0x138, 0xF>(pos, 0);
    const bool joins = alive && gl > 0 && pcol == col;
    // Positions of one column differ, unless a row of B has a column twice or
    // columns past N meet in the packed keys (the fused path merges beside the
    // check of B).  The 1 then gives level 0, so that every entry that joins has
    // a level from 0 to 31 and the loop below ends whatever the operands are; its
    // indexes are lanes of the group all the same, and the product is refused.
    // (A bound on the loop instead takes five scalar instructions a level; here
    // the compiler drops the minimum that __clz needs for 0.)
    int lvl = joins ? 31 - __clz((pos ^ ppos) | 1) : -1;
    asm volatile("" : "+v"(lvl));  // compared as it is, not by its parts
    uint64_t am = __ballot(alive), todo = __ballot(joins);
    for (int l = 0; todo != 0ull; ++l) {
        const uint64_t die = __ballot(lvl == l);
        if (die == 0ull) continue;
        todo &= ~die;
        // the live lane before each of `die`: in reversed order a carry from
        // each runs through the dead lanes and stops at the next live one
        // (two entries of one level never follow each other)
        const uint64_t rl = __brevll(am);
        const bool gets = __builtin_amdgcn_inverse_ballot_w64(__brevll((~rl + (__brevll(die) << 1)) & rl));
        int nxt;  // byte address of the next lane of `die` (a lane that gets is not in it)
        if constexpr (G == BRM_WAVE) {
            nxt = (__ffsll((long long)(die & (~0ull << gl))) - 1) << 2;
        } else {
            nxt = (low_bit(group_bits<G>(die, gbase, ~0u << gl)) << 2) + (gbase << 2);
        }
        const int nlo = __builtin_amdgcn_ds_bpermute(nxt, __double2loint(val));  // address modulo 256
        const int nhi = __builtin_amdgcn_ds_bpermute(nxt, __double2hiint(val));
        if (gets) val = fadd(val, __hiloint2double(nhi, nlo));
        am &= ~die;
    }
    ShortMerged r{};
    r.col = col;
    r.val = val;
    r.alive = __builtin_amdgcn_inverse_ballot_w64(am);
    r.idx = group_rank<G>(am, gbase);
    if constexpr (G == BRM_WAVE) r.nout = __popcll(am);
    else r.nout = (int)of_half(__popc((uint32_t)am), __popc((uint32_t)(am >> 32)), gbase);
    return r;
}

}  // namespace brm
