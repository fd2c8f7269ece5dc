// Attention of calls with few query blocks for gfx950: bf16 in, fp32 MFMA accumulation and softmax, bf16 out, over key
// tile images or (KR) key rows, and value rows. The same contract, tile layouts, MFMA steps and fixed-reference softmax
// as the streaming kernel (attn_stream.hip); what differs is how the work is cut.
//
// What bounds these calls is that one 256-query block a compute unit leaves most units idle (1,280 tokens x 24 heads are
// 120 blocks), and cutting a block's keys over workgroups costs a partial written to and merged from memory (~10 us).
// Here a workgroup is 128 queries of one head and its 8 waves are two groups of four: each wave owns 32 queries, group
// g takes the key tiles g, g + 2, g + 4, ... So twice as many workgroups have work, every SIMD still holds two waves
// (one's softmax under the other's MFMAs), a block's critical path is half its tiles, and the two groups' results are
// merged through LDS at the end: each wave sends its partner the 64 dims it does not write and merges the other 64.
//
//  * LDS, 160 KB: per group a ring of two key tiles and two value tiles (64 KB), and the block's queries as operand
//    fragments (32 KB, brought in once by the direct loads of both groups, so no wave loads a query twice). A step's
//    refills (the next key tile and this step's value tile) are issued over its first half and have landed at its end.
//  * Causal blocks differ in length: they are dispatched longest first, so that the last ones to run are the short ones.
#include "lr_common.h"
#include "lr_kernels.h"
#include "tile_image.h"

namespace lr {

namespace {

#include "attn_common.inc"

constexpr int RA = 3;             // fragments read ahead
constexpr int FR = 4;             // fragment ring entries
constexpr int KW = 2;             // key groups
constexpr int QW = 4;             // waves (of 32 queries) per group
constexpr int KBM = 32 * QW;      // queries per block
constexpr int GROUP_LDS = 4 * IMG_TILE_BYTES;            // a group's ring: two key tiles, two value tiles
constexpr int Q_LDS = KW * GROUP_LDS;                    // the queries: QW x 8 fragments of 1 KB
constexpr int KS_LDS = Q_LDS + QW * 8 * IMG_FRAG_BYTES;
// the merge, over the rings: 8 KB a wave (the 32 accumulators its partner writes), then (m, l) per lane, then one flag
// per 32 queries
constexpr int MG_ML = KW * QW * 8192, MG_FLAG = MG_ML + KW * QW * 512;
static_assert(MG_FLAG + 4 * QW <= Q_LDS && KS_LDS <= 160 * 1024, "LDS areas");

#include "attn_tiles.inc"

// One 1 KB direct load, global -> LDS: lane l's 16 bytes come from gaddr + voff and land at lds + 16 l.
__device__ __forceinline__ void dma1(uint64_t gaddr, uint32_t voff, uint32_t lds) {
    LR_ASM_M0_BEGIN
    asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(gaddr), "s"(lds)
                 : "memory", "m0");
    LR_ASM_M0_END
}
// Four query fragments gathered from rows: load i takes each lane's 16 bytes at addr + 32 i (the row's next 16 dims) to
// lds + 1024 i + 16 l (the instruction offset applies to both addresses, so M0 takes the other 992 i).
__device__ __forceinline__ void dma4_rows_far(uint64_t addr, uint32_t lds) {
    LR_ASM_M0_BEGIN
    asm volatile(
        "s_mov_b32 m0, %1\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off offset:0\n\t"
        "s_add_u32 m0, %1, 0x3e0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off offset:32\n\t"
        "s_add_u32 m0, %1, 0x7c0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off offset:64\n\t"
        "s_add_u32 m0, %1, 0xba0\n\t"
        "s_nop 0\n\t"
        "global_load_lds_dwordx4 %0, off offset:96" ::"v"(addr),
        "s"(lds)
        : "memory", "m0", "scc");
    LR_ASM_M0_END
}

// n / d for 0 <= n < 2^31, d >= 1, given rcp = floor(2^32 / d) (2^32 - 1 for d = 1): the high product is the quotient or
// one less. (Four scalar instructions; a division by a value the compiler does not know is ~40, in front of the first
// load.)
__device__ __forceinline__ int div_small(int n, int d, uint32_t rcp) {
    const uint32_t q = (uint32_t)(((uint64_t)(uint32_t)n * rcp) >> 32);
    return (int)(q + ((uint32_t)n - q * (uint32_t)d >= (uint32_t)d ? 1u : 0u));
}

template <bool KR>
__global__ __launch_bounds__(512, 1) __attribute__((amdgpu_waves_per_eu(2, 2))) void attn_keysplit_kernel(AttnArgs a) {
    __shared__ __attribute__((aligned(1024))) uint8_t lds[KS_LDS];

    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave / QW, wv = wave % QW;
    const int n = lane & 31, hf = lane >> 5;

    // ---- the block. Hardware workgroup b runs on XCD b % 8. Causal: longest blocks first, each XCD working on heads of
    // its own when they divide evenly; otherwise each XCD takes a contiguous range of blocks (query blocks of one head
    // share its keys in the XCD's L2).
    const int nwg = gridDim.x, b = blockIdx.x;
    const int nqb = (a.W + KBM - 1) / KBM;
    int head, qblk;
    if (a.causal) {
        const int h = b - div_small(b, a.H, a.rcp_h) * a.H;
        qblk = nqb - 1 - div_small(b, a.H, a.rcp_h);
        head = a.H % 8 == 0 ? (h & 7) * (a.H >> 3) + (h >> 3) : h;
    } else {
        const int per = nwg >> 3, rem8 = nwg & 7, xcd = b & 7, idx = b >> 3;
        const int logical = xcd < rem8 ? xcd * (per + 1) + idx : rem8 * (per + 1) + (xcd - rem8) * per + idx;
        head = div_small(logical, nqb, a.rcp_nqb);
        qblk = logical - head * nqb;
    }
    const int hk = div_small(head, a.G, a.rcp_g);
    const int row0 = qblk * KBM, wrow0 = row0 + 32 * wv;
    const int T = (a.nkeys + IMG_TILE_KEYS - 1) / IMG_TILE_KEYS;
    const int tb = a.causal ? min(T, (a.p0 + min(row0 + KBM, a.W) - 1) / IMG_TILE_KEYS + 1) : T;
    const int nsteps = (tb + KW - 1) / KW;   // steps of both groups: group g's step u is tile g + 2 u (tiles past the
                                             // block's last one are masked whole)

    // ---- direct loads
    const uint64_t khead = (uint64_t)(uintptr_t)a.k +
                           (uint64_t)hk * (KR ? (uint64_t)a.k_hs * 2 : (uint64_t)T * IMG_TILE_BYTES);
    const uint64_t vhead = (uint64_t)(uintptr_t)a.v + (uint64_t)hk * (uint64_t)a.v_hs * 2;
    const uint32_t rowb = (uint32_t)a.v_rs * 2u;                       // < 2^25: the launch checks the strides
    const uint32_t krowb = KR ? (uint32_t)a.k_rs * 2u : 0u;
    const uint32_t lds0 = lds_addr(lds), ring = lds0 + (uint32_t)(grp * GROUP_LDS), qlds = lds0 + Q_LDS;
    const uint32_t lane16 = (uint32_t)lane * 16u;
    const int vfull = a.nkeys >> 6;   // tiles t < vfull hold 64 rows
    // A tile is four 1 KB loads of each of the group's waves. Load i of a key tile: fragment 4 wv + i (key block wv >> 1,
    // k-step 4 (wv & 1) + i); KR: lane 32 hf + n takes row 32 (wv >> 1) + key_perm(n), its offset in the tile in ko.
    // Load i of a value tile: rows 16 wv + 4 i + vt_lane_row(lane) in the row-block layout (attn_tiles.inc), offset
    // vo[i]. In the head's last, partial tile rows past nkeys read the last row (finite: their scores are masked and
    // their P is 0).
    const uint32_t krow = (uint32_t)(32 * (wv >> 1) + img_key_perm(n)), kcol = (uint32_t)(128 * (wv & 1) + 16 * hf);
    const uint32_t vrow = (uint32_t)(16 * wv + vt_lane_row(lane)), vchunk = (uint32_t)(16 * vt_lane_chunk(lane));
    uint32_t ko = KR ? krow * krowb + kcol : lane16, vo[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) vo[i] = (vrow + 4 * i) * rowb + vchunk;
    auto tile_of = [&](int u) __attribute__((always_inline)) { return min(grp + KW * u, tb - 1); };
    auto k_src = [&](int t) __attribute__((always_inline)) {
        if (KR && t >= vfull)
            ko = min(krow, (uint32_t)(a.nkeys - 1 - IMG_TILE_KEYS * t)) * krowb + kcol;
        return khead + (KR ? (uint64_t)t * ((uint64_t)IMG_TILE_KEYS * krowb)
                           : (uint64_t)t * IMG_TILE_BYTES + (uint64_t)(wv * 4096));
    };
    auto v_src = [&](int t) __attribute__((always_inline)) {
        if (t >= vfull) {
            const uint32_t lim = (uint32_t)(a.nkeys - 1 - IMG_TILE_KEYS * t);
#pragma unroll
            for (int i = 0; i < 4; ++i) vo[i] = min(vrow + 4 * i, lim) * rowb + vchunk;
        }
        return vhead + (uint64_t)t * ((uint64_t)IMG_TILE_KEYS * rowb);
    };
    // (KR: the row's next 16 dims, a 32-byte step; the image: the next 1 KB)
    auto load_k1 = [&](uint64_t src, uint32_t dst, int i) __attribute__((always_inline)) {
        dma1(src + (uint64_t)(i * (KR ? 32 : 1024)), ko, dst + (uint32_t)(wv * 4096 + 1024 * i));
    };
    auto load_v1 = [&](uint64_t src, uint32_t dst, int i) __attribute__((always_inline)) {
        dma1(src, vo[i], dst + (uint32_t)(wv * 4096 + 1024 * i));
    };

    // ---- registers (as the streaming kernel's)
    bf16x8 qa[8];
    f32x16 o[4], s[2], negm;
    u32x4 p[2][2];
    float ls = 0.0f;
    bf16x8 fr[FR];
    const uint32_t vlane = (uint32_t)vt_lane(lane);
    auto vfrag_off = [](int x) __attribute__((always_inline)) { return 4096 * (x >> 2) + 256 * (x & 3); };

    // ---- prologue: the queries (each group half of the fragments) and the first key tile; the next key tile and the
    // first value tile follow in step 0. (A load of 64 rows' pieces holds the memory pipe ~30 cycles: all of the first
    // 16 loads of 8 waves issued here kept the first scores waiting for 3,500 cycles.)
    {
        // lane 32 hf + n: row n, dims 64 grp + 16 i + 8 hf .. +7 (k-steps 4 grp + i, i < 4)
        const uint16_t* src = a.q + (int64_t)min(wrow0 + n, a.W - 1) * a.q_rs + head * D + 64 * grp + 8 * hf;
        dma4_rows_far((uint64_t)(uintptr_t)src, qlds + (uint32_t)((8 * wv + 4 * grp) * IMG_FRAG_BYTES));
        const uint64_t ks = k_src(tile_of(0));
#pragma unroll
        for (int i = 0; i < 4; ++i) load_k1(ks, ring, i);
    }
    const uint32_t vring = ring + 2 * IMG_TILE_BYTES;

    // masks: keys past nkeys and, causal, past the query's position
    auto mask_half = [&](f32x16& sb, int j) __attribute__((always_inline)) {
        int lim = a.nkeys;
        if (a.causal) lim = min(lim, a.p0 + wrow0 + n + 1);
        lim -= 32 * j + 8 * hf;
#pragma unroll
        for (int r = 0; r < 16; ++r)
            if (!(16 * (r >> 3) + (r & 7) < lim)) sb[r] = -INFINITY;
    };
    int jm = a.nkeys >> 5;   // the first half-tile that needs a mask for this wave
    if (a.causal) jm = min(jm, (a.p0 + wrow0 + 1) >> 5);

    float e0 = 0.0f, e1 = 0.0f;
    const float c = a.c;
    auto stage_e = [&](const f32x16& sb, int w) __attribute__((always_inline)) {
        e0 = __builtin_amdgcn_exp2f(sb[8 * (w >> 2) + 2 * (w & 3)] * c);
        e1 = __builtin_amdgcn_exp2f(sb[8 * (w >> 2) + 2 * (w & 3) + 1] * c);
        asm volatile("" ::"v"(e0), "v"(e1));   // computed in this slot, not sunk towards the next use
    };
    // (the sum is that of the rounded probabilities, which are what multiplies the values: a row that one key dominates
    // then keeps that key's value to the output's rounding, as in the pipelined kernel. Relative error against 64 bits of
    // causal calls, 500 queries x 16 heads 2.30e-3 -> 2.12e-3, 4,000 x 24 2.29e-3 -> 2.18e-3; 1 to 3 % of the time: 13.6 ->
    // 13.9 us, 122.4 -> 124.2.)
    const bf16x2 ones2 = {(bf16)1.0f, (bf16)1.0f};
    auto stage_c = [&](u32x4 (&pb)[2], int w) __attribute__((always_inline)) {
        const uint32_t x = pack_bf16x2(e0, e1);
        pb[w >> 2][w & 3] = x;
        ls = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, x), ones2, ls, false);
        asm volatile("" ::"v"(x), "v"(ls));
    };
    // one half-step of 16 MFMA slots, as the streaming kernel's: the next half-tile's scores, the previous one's P V,
    // this one's P
    auto half_step = [&](f32x16& so, const u32x4 (&ppv)[2], const f32x16& si, u32x4 (&po)[2], auto pv_tag,
                         auto&& rd) __attribute__((always_inline)) {
        constexpr bool HAS_PV = decltype(pv_tag)::value;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int f = 0; f < 16; ++f) {
            if (f < 8) {
                if (f == 0) qk_init(so, fr[0], qa[0], negm);
                else qk_acc(so, fr[f % FR], qa[f]);
            } else {
                if constexpr (HAS_PV) pv(o[(f - 8) & 3], fr[f % FR], ppv[(f - 8) >> 2]);
            }
            if ((f & 1) == 0) stage_e(si, f >> 1);
            else stage_c(po, f >> 1);
            rd(f + RA);
            __builtin_amdgcn_sched_barrier(0);
        }
    };

    // a step's refills, one load every other slot of its first half (all at once would hold the wave's issue up behind
    // the memory pipe): V(u), then K(u + 1) (past the last tile a repeat of it, never read)
    auto refill = [&](int f, uint64_t vs, uint32_t vd, uint64_t ks, uint32_t kd) __attribute__((always_inline)) {
        if (f % 2 == 0) {
            if (f < 8) load_v1(vs, vd, f / 2);
            else load_k1(ks, kd, (f - 8) / 2);
        }
    };

    // ---- the queries and K(0) resident; S of the group's first half-tile and the fixed reference m = its maximum. A row with
    // no key in it (causal) keeps m = 0 and P = 0.
#pragma unroll
    for (int db = 0; db < 4; ++db) o[db] = f32x16{};
    LR_WAIT_VMCNT(0);
    block_barrier();
    {
        const uint64_t vs = v_src(tile_of(0));
#pragma unroll
        for (int i = 0; i < 4; ++i) load_v1(vs, vring, i);
    }
    float mref;
    {
        uint32_t kb0 = ring + lane16, qb0 = qlds + (uint32_t)(8 * wv * IMG_FRAG_BYTES) + lane16;
        asm volatile("" : "+v"(kb0), "+v"(qb0));
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) qa[ks] = frag_at(qb0 + (uint32_t)(ks * IMG_FRAG_BYTES));
        fence_q8(qa);
#pragma unroll
        for (int ks = 0; ks < 8; ++ks) {
            const bf16x8 kf = frag_at(kb0 + (uint32_t)(ks * IMG_FRAG_BYTES));
            if (ks == 0) qk_zero(s[0], kf, qa[0]);
            else qk_acc(s[0], kf, qa[ks]);
        }
        fence_s(s[0]);
        if (2 * grp >= jm) mask_half(s[0], 2 * grp);
        float mx = s[0][0];
#pragma unroll
        for (int q = 1; q < 16; ++q) mx = fmaxf(mx, s[0][q]);
        mx = wave_pair_max(mx);
        // (the maximum itself, not the next integer: where it is the row's, its probability is 1, with no rounding of its
        // own. Relative error against 64 bits of causal calls, 500 queries x 16 heads 2.12e-3 -> 2.00e-3, 4,000 x 24 2.18e-3 ->
        // 2.09e-3, as the pipelined kernel's; the same time)
        const float m0 = mx > -INFINITY ? mx : 0.0f;
        mref = m0 * c;
        negm = f32x16{} - m0;
        s[0] -= m0;
        asm volatile(LR_NOP48 : "+v"(negm));
    }
    // ---- step 0: S of half-tile 1 (K(0), fragments 8-15), P of half-tile 0
    {
        const uint64_t ks = k_src(tile_of(1));   // (one tile in all: a repeat of it, never read)
        uint32_t kb = ring + lane16;
        asm volatile("" : "+v"(kb));
        auto rd0 = [&](int f) __attribute__((always_inline)) {
            if (f < 8) fr[f % FR] = frag_at(kb + (8 + f) * IMG_FRAG_BYTES);
        };
#pragma unroll
        for (int f = 0; f < RA; ++f) rd0(f);
        half_step(s[1], p[1], s[0], p[0], BoolTag<false>{}, [&](int f) __attribute__((always_inline)) {
            if ((f - RA) % 2 == 0 && f - RA < 8) load_k1(ks, ring + IMG_TILE_BYTES, (f - RA) / 2);
            rd0(f);
        });
        LR_WAIT_VMCNT(0);
        block_barrier();
    }
    // ---- step u: key tile u (both halves), value tile u - 1. Its refills go to the slots of V(u - 2) and K(u - 1), both
    // read before the last barrier, and have landed at its end.
    for (int u = 1; u < nsteps; ++u) {
        const int j = 2 * (grp + KW * u);   // the tile's first half-tile; the one before it is 2 (grp + KW (u - 1)) + 1
        const uint32_t par = (uint32_t)((u & 1) * IMG_TILE_BYTES), par1 = par ^ IMG_TILE_BYTES;
        const uint64_t vs = v_src(tile_of(u)), ks = k_src(tile_of(u + 1));
        uint32_t kb = ring + par + lane16, vb = vring + par1 + vlane;
        asm volatile("" : "+v"(kb), "+v"(vb));
        auto rd_b = [&](int f) __attribute__((always_inline)) {
            if (f < 8) fr[f % FR] = frag_at(kb + f * IMG_FRAG_BYTES);
            else if (f < 16) fr[f % FR] = vfrag_at(vb + vfrag_off(f - 8));
            else fr[f % FR] = frag_at(kb + (f - 8) * IMG_FRAG_BYTES);
        };
        auto rd_a = [&](int f) __attribute__((always_inline)) {
            if (f < 8) fr[f % FR] = frag_at(kb + (8 + f) * IMG_FRAG_BYTES);
            else if (f < 16) fr[f % FR] = vfrag_at(vb + vfrag_off(f));
        };
#pragma unroll
        for (int f = 0; f < RA; ++f) rd_b(f);
        if (j - 2 * KW + 1 >= jm) mask_half(s[1], j - 2 * KW + 1);
        half_step(s[0], p[0], s[1], p[1], BoolTag<true>{}, [&](int f) __attribute__((always_inline)) {
            refill(f - RA, vs, vring + par, ks, ring + par1);
            rd_b(f);
        });
        if (j >= jm) mask_half(s[0], j);
        half_step(s[1], p[1], s[0], p[0], BoolTag<true>{}, rd_a);
        LR_WAIT_VMCNT(0);
        block_barrier();
    }
    // ---- the last half-tile's P and the last value tile's products, then the merge: group g writes dims 64 g .. 64 g + 63
    // of its 32 queries and sends the other 64 to its partner, the wave of the other group with the same queries. The
    // products of the dims to send come first, so that sending them runs beside the last products of the others. (Two
    // code paths, not selects: the accumulators stay where they are.)
    float* ml = reinterpret_cast<float*>(lds + MG_ML);
    int* flag = reinterpret_cast<int*>(lds + MG_FLAG);
    const int qrow = wrow0 + n;
    auto finish = [&](auto grp_tag) __attribute__((always_inline)) {
        constexpr int G = decltype(grp_tag)::value, SEND = 2 - 2 * G, KEEP = 2 * G;   // 32-dim blocks
        {
            const int u = nsteps - 1, j = 2 * (grp + KW * u) + 1;
            if (j >= jm) mask_half(s[1], j);
            uint32_t vb0 = vring + (uint32_t)((u & 1) * IMG_TILE_BYTES) + vlane;
            asm volatile("" : "+v"(vb0));
            // product x: 16-key step kk(x) of the tile, 32-dim block db(x): the first half-tile's (P of buffer 0), the
            // dims to send first, then the second half-tile's
            auto kk = [](int x) __attribute__((always_inline)) { return 2 * (x >> 3) + ((x >> 1) & 1); };
            auto db = [](int x) __attribute__((always_inline)) { return ((x >> 2) & 1 ? KEEP : SEND) + (x & 1); };
            auto off = [&](int x) __attribute__((always_inline)) { return (uint32_t)vfrag_off(4 * kk(x) + db(x)); };
            bf16x8 vf[4];
#pragma unroll
            for (int x = 0; x < 3; ++x) vf[x] = vfrag_at(vb0 + off(x));
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int x = 0; x < 16; ++x) {
                if (x + 3 < 16) vf[(x + 3) & 3] = vfrag_at(vb0 + off(x + 3));
                pv(o[db(x)], vf[x & 3], (x < 8 ? p[0] : p[1])[(x >> 1) & 1]);
                if (x < 8) {
                    stage_e(s[1], x);
                    stage_c(p[1], x);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        const float l = wave_pair_sum(ls);
        block_barrier();   // every wave is done with the rings
        float* mg = reinterpret_cast<float*>(lds + 8192 * wave) + 4 * lane;
        const float* mgp = reinterpret_cast<const float*>(lds + 8192 * (wave ^ QW)) + 4 * lane;
#pragma unroll
        for (int gi = 0; gi < 8; ++gi) {
            f32x4 x;
#pragma unroll
            for (int e = 0; e < 4; ++e) x[e] = o[SEND + (gi >> 2)][4 * (gi & 3) + e];
            *reinterpret_cast<f32x4*>(mg + 256 * gi) = x;
        }
        ml[128 * wave + 2 * lane] = mref;
        ml[128 * wave + 2 * lane + 1] = l;
        if (G == 0 && lane == 0) flag[wv] = 0;
        __syncthreads();
        // weights relative to M, the largest reference of a group that saw a key, times 1 / l: in group order, so that
        // both waves of a query compute the same. A sum past 2^100 (or not a number) means the fixed reference
        // overflowed: the row is recomputed.
        const float m0 = ml[128 * wv + 2 * lane], l0 = ml[128 * wv + 2 * lane + 1];
        const float m1 = ml[128 * (wv + QW) + 2 * lane], l1 = ml[128 * (wv + QW) + 2 * lane + 1];
        const float M = fmaxf(l0 > 0.0f ? m0 : -INFINITY, l1 > 0.0f ? m1 : -INFINITY);
        float w0 = l0 > 0.0f ? __builtin_amdgcn_exp2f(m0 - M) : 0.0f;
        float w1 = l1 > 0.0f ? __builtin_amdgcn_exp2f(m1 - M) : 0.0f;
        const float inv = 1.0f / fmaf(w1, l1, w0 * l0);   // (spelled out: every instantiation rounds alike)
        w0 *= inv;
        w1 *= inv;
        const float wm = G == 0 ? w0 : w1, wp = G == 0 ? w1 : w0;
        float nan = l0 <= 0x1p100f && l1 <= 0x1p100f ? 0.0f : __builtin_nanf("");   // NaN iff the row is not finite
        const bf16x2 zero2 = {(bf16)0.0f, (bf16)0.0f};
        u32x2 w[8];
#pragma unroll
        for (int gi = 0; gi < 8; ++gi) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(mgp + 256 * gi);
            float y[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = fmaf(wp, x[e], wm * o[KEEP + (gi >> 2)][4 * (gi & 3) + e]);
            w[gi][0] = pack_bf16x2(y[0], y[1]);
            w[gi][1] = pack_bf16x2(y[2], y[3]);
            nan = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, (uint32_t)w[gi][0]), zero2, nan, false);
            nan = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, (uint32_t)w[gi][1]), zero2, nan, false);
        }
        if (__builtin_amdgcn_ballot_w64(nan != 0.0f && qrow < a.W) && lane == 0) flag[wv] = 1;
        __syncthreads();
        if (__builtin_amdgcn_readfirstlane(flag[wv])) return true;
        // 8 dims a store: the lower lanes take both halves' words of the even 8-dim groups, the upper lanes of the odd
        // ones
        uint16_t* dst = a.out + (int64_t)qrow * a.o_rs + head * D + 64 * G + 8 * hf;
#pragma unroll
        for (int x = 0; x < 4; ++x) {
            const auto r0 = __builtin_amdgcn_permlane32_swap(w[2 * x][0], w[2 * x + 1][0], false, false);
            const auto r1 = __builtin_amdgcn_permlane32_swap(w[2 * x][1], w[2 * x + 1][1], false, false);
            if (qrow < a.W) *reinterpret_cast<u32x4*>(dst + 32 * (x >> 1) + 16 * (x & 1)) = u32x4{r0[0], r1[0], r0[1], r1[1]};
        }
        return false;
    };
    // a row of these 32 overflowed its fixed reference: all of them again with the exact maximum (the queries are still
    // there when they are the output rows: neither wave has written)
    if (grp == 0) {
        if (finish(IntTag<0>{})) redo_exact<KR>(a, head, hk, row0, tb, wv);
    } else {
        finish(IntTag<1>{});
    }
}

}  // namespace

hipError_t launch_keysplit(const AttnArgs& a, hipStream_t stream, bool key_rows) {
    if (a.W < 1 || a.H < 1) return hipErrorInvalidValue;
    if (a.v_rs < D || a.v_rs > STREAM_MAX_V_RS || a.v_rs % 8 || a.v_hs < 0 || a.v_hs % 8) return hipErrorInvalidValue;
    if (key_rows && (a.k_rs < D || a.k_rs > STREAM_MAX_V_RS || a.k_rs % 8 || a.k_hs < 0 || a.k_hs % 8))
        return hipErrorInvalidValue;
    const int64_t blocks = (int64_t)((a.W + KBM - 1) / KBM) * a.H;
    if (blocks > 0x7fffffff) return hipErrorInvalidValue;
    auto rcp = [](int64_t d) { return d > 1 ? (uint32_t)(((uint64_t)1 << 32) / (uint64_t)d) : 0xffffffffu; };
    AttnArgs b = a;
    b.rcp_nqb = rcp((a.W + KBM - 1) / KBM);
    b.rcp_h = rcp(a.H);
    b.rcp_g = rcp(a.G);
    if (key_rows) hipLaunchKernelGGL(attn_keysplit_kernel<true>, dim3((unsigned)blocks), dim3(512), 0, stream, b);
    else hipLaunchKernelGGL(attn_keysplit_kernel<false>, dim3((unsigned)blocks), dim3(512), 0, stream, b);
    return hipGetLastError();
}

}  // namespace lr
