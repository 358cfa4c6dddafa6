// Chunked prefill with 256 query rows per workgroup, for launches of several rounds of workgroups
// (pd_prefill.hip's kernel takes 192). Same interface and partials. The (token, head of one kv head) pairs of a
// sequence are its rows, token-major; a workgroup takes kFwRows consecutive rows (4 waves of 4
// blocks of 16) and streams every visible 32-key tile once:
//   HBM -> LDS   the waves copy a step of two tiles together (9 copies each) into a 6-tile ring,
//                two steps ahead; one barrier per step publishes it and frees its predecessor;
//   int8 -> fp16 each wave widens the operands that it reads in registers, exactly (no bias), between the
//                products of the operand before (score_products, value_products);
//   MFMA         S^T = K Q^T and O^T += V^T P'^T on fp16 MFMA with fp32 accumulation; Q in 128 vector
//                registers, O in all 256 accumulation registers.
// What bounds it: a tile's 32 blocks of 4 MFMAs and 8 conversions take 2,327 cycles and its softmax 884 (measured
// alone), but under that load the card runs at 1.5-2.0 GHz instead of 2.4; the whole tile takes 1.85 us (2.35
// GHz), where 192 rows take 1.62 us in pd_prefill.hip: 13 % less per row. It pays where its larger
// workgroups do not cost a round (launch_prefill): 2,048 tokens over 61,440 keys (24 q / 4 kv heads) 3.15 ms ->
// 2.92 in 4 splits. A widening through LDS once per workgroup (3.29 ms: the LDS latency shows) and two waves of
// 32 rows per SIMD (3.66 ms: each conversion then serves half the products) were slower. The exact widening
// leaves the default numerics' error at its fp16 weights: 2.1e-4 of the result at 63,488 keys, 7.9e-3 with the
// biased one.
// kExact (pth_fa_forward_exact) carries P' as fp16 hi + lo, which doubles the P.V products; the
// default rounds P' once to fp16.
#include <type_traits>

#include "pd_tile.hpp"
#include "pth_dec.h"

namespace pd {

constexpr int kFwWaves = 4;
constexpr int kFwRB = 4;                          // 16-row blocks per wave
static_assert(kFwRows == kFwWaves * kFwRB * 16, "rows of a workgroup");
constexpr int kFwStep = 2;                        // tiles per barrier
constexpr int kFwAhead = 2;                       // steps in flight
constexpr int kFwRing = kFwStep * (kFwAhead + 1);  // tile slots
// A slot: the K and V images of pd_tile.hpp (V from byte 260 of the row, so its 16 blocks hold whole
// dim blocks), then the tile's scales: k_scale [32], v_scale [32].
constexpr int kFwImgV = kImgV;
constexpr int kFwImgS = 16 * kBlk;
constexpr int kFwSlot = kFwImgS + 256;
constexpr int kFwCopies = 4 * kFwStep + 1;        // copies of a wave per step
constexpr int kFwBt = 6144;                       // 16-key blocks (or pages) of the LDS block table

// The products of one widened operand `cur` with the four row blocks of a wave, and between them the
// widening of the next operand from its bytes (w0, w1): a 16x16x32 MFMA keeps the matrix core busy
// for 16 cycles and leaves the issue slots of about three of these conversions. The order is
// written out because the compiler gathers the conversions before the products. (The trailing
// s_nop keeps the last conversion two slots from the next block's first product, which reads it.)
#define PD_CVT(d, w, half, byte, keep) \
    "v_cvt_f16_i16_sdwa " d ", sext(" w ") dst_sel:WORD_" half " dst_unused:UNUSED_" keep " src0_sel:BYTE_" byte "\n\t"
#define PD_PRODUCTS_AND_WIDEN(C0, C1, C2, C3)                                    \
    "v_mfma_f32_16x16x32_f16 %0, %8, %9, " C0 "\n\t"                              \
    PD_CVT("%4", "%13", "0", "0", "PAD") PD_CVT("%5", "%13", "0", "2", "PAD") PD_CVT("%6", "%14", "0", "0", "PAD") \
    "v_mfma_f32_16x16x32_f16 %1, %8, %10, " C1 "\n\t"                             \
    PD_CVT("%7", "%14", "0", "2", "PAD") PD_CVT("%4", "%13", "1", "1", "PRESERVE") PD_CVT("%5", "%13", "1", "3", "PRESERVE") \
    "v_mfma_f32_16x16x32_f16 %2, %8, %11, " C2 "\n\t"                             \
    PD_CVT("%6", "%14", "1", "1", "PRESERVE") PD_CVT("%7", "%14", "1", "3", "PRESERVE")    \
    "v_mfma_f32_16x16x32_f16 %3, %8, %12, " C3 "\n\ts_nop 0"
// scores: accumulators in vector registers (the softmax reads them)
template <bool kFirst>
__device__ __forceinline__ half8_t score_products(float4_t& s0, float4_t& s1, float4_t& s2, float4_t& s3, half8_t cur,
                                                  half8_t q0, half8_t q1, half8_t q2, half8_t q3, unsigned w0,
                                                  unsigned w1) {
    uint4_t n;
    if constexpr (kFirst)
        asm volatile(PD_PRODUCTS_AND_WIDEN("0", "0", "0", "0")
                     : "=&v"(s0), "=&v"(s1), "=&v"(s2), "=&v"(s3), "=&v"(n.x), "=&v"(n.y), "=&v"(n.z), "=&v"(n.w)
                     : "v"(cur), "v"(q0), "v"(q1), "v"(q2), "v"(q3), "v"(w0), "v"(w1));
    else
        asm volatile(PD_PRODUCTS_AND_WIDEN("%0", "%1", "%2", "%3")
                     : "+v"(s0), "+v"(s1), "+v"(s2), "+v"(s3), "=&v"(n.x), "=&v"(n.y), "=&v"(n.z), "=&v"(n.w)
                     : "v"(cur), "v"(q0), "v"(q1), "v"(q2), "v"(q3), "v"(w0), "v"(w1));
    return __builtin_bit_cast(half8_t, n);
}
// values: O stays in the accumulation registers
__device__ __forceinline__ half8_t value_products(float4_t& o0, float4_t& o1, float4_t& o2, float4_t& o3, half8_t cur,
                                                  half8_t p0, half8_t p1, half8_t p2, half8_t p3, unsigned w0,
                                                  unsigned w1) {
    uint4_t n;
    asm volatile(PD_PRODUCTS_AND_WIDEN("%0", "%1", "%2", "%3")
                 : "+a"(o0), "+a"(o1), "+a"(o2), "+a"(o3), "=&v"(n.x), "=&v"(n.y), "=&v"(n.z), "=&v"(n.w)
                 : "v"(cur), "v"(p0), "v"(p1), "v"(p2), "v"(p3), "v"(w0), "v"(w1));
    return __builtin_bit_cast(half8_t, n);
}
__device__ __forceinline__ void value_products_only(float4_t& o0, float4_t& o1, float4_t& o2, float4_t& o3, half8_t cur,
                                                    half8_t p0, half8_t p1, half8_t p2, half8_t p3) {
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %4, %5, %0\n\tv_mfma_f32_16x16x32_f16 %1, %4, %6, %1\n\t"
                 "v_mfma_f32_16x16x32_f16 %2, %4, %7, %2\n\tv_mfma_f32_16x16x32_f16 %3, %4, %8, %3"
                 : "+a"(o0), "+a"(o1), "+a"(o2), "+a"(o3)
                 : "v"(cur), "v"(p0), "v"(p1), "v"(p2), "v"(p3));
}
// Wait states between asm MFMAs and the first other instruction that touches their results (the
// operands keep the compiler from moving such an instruction before the wait).
__device__ __forceinline__ void settle_scores(float4_t (&s)[kFwRB][2]) {
    asm volatile("s_nop 15" : "+v"(s[0][0]), "+v"(s[0][1]), "+v"(s[1][0]), "+v"(s[1][1]), "+v"(s[2][0]), "+v"(s[2][1]),
                 "+v"(s[3][0]), "+v"(s[3][1]));
}
__device__ __forceinline__ void settle_values(float4_t (&o)[16]) {
    asm volatile("s_nop 15" : "+a"(o[0]), "+a"(o[1]), "+a"(o[2]), "+a"(o[3]), "+a"(o[4]), "+a"(o[5]), "+a"(o[6]), "+a"(o[7]));
    asm volatile("" : "+a"(o[8]), "+a"(o[9]), "+a"(o[10]), "+a"(o[11]), "+a"(o[12]), "+a"(o[13]), "+a"(o[14]), "+a"(o[15]));
}
// The wait before the products of P' (see settle_operand), once for all of its row blocks.
template <bool kExact>
__device__ __forceinline__ void settle_weights(half8_t (&p)[kFwRB], half8_t (&lo)[kFwRB]) {
    if constexpr (kExact)
        asm volatile("s_nop 1" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]), "+v"(lo[0]), "+v"(lo[1]), "+v"(lo[2]), "+v"(lo[3]));
    else
        asm volatile("s_nop 1" : "+v"(p[0]), "+v"(p[1]), "+v"(p[2]), "+v"(p[3]));
}

template <bool kFast, bool kExact, bool kSplit, class T>
__global__ void __launch_bounds__(kFwWaves * 64, 1) pd_prefill_wide_kernel(const FaParams a) {
    constexpr int kLdsBt = kFwRing * kFwSlot;
    constexpr int kLdsScr = kLdsBt + kFwBt * 4;  // 4 KiB per wave for the rescale of O
    constexpr int kLdsBytes = kLdsScr + kFwWaves * 4096;
    static_assert(kLdsBytes <= 160 * 1024, "gfx950 has 160 KiB of LDS per CU");
    __shared__ __attribute__((aligned(16))) unsigned char lds[kLdsBytes];

    // Workgroups are dispatched to the 8 XCDs round robin (linear id L to XCD L % 8), and each XCD
    // has its own L2. Every query tile of a (sequence, kv head) streams the same keys, so the
    // logical workgroup index (query tile fastest) is laid out XCD by XCD: XCD x takes a
    // contiguous range of it, and the query tiles sharing a kv head mostly share an L2.
    const unsigned nx = gridDim.x, ny = gridDim.y, nwg = nx * ny * gridDim.z;
    const unsigned lin = blockIdx.x + nx * (blockIdx.y + ny * blockIdx.z);
    const unsigned xcd = lin % 8u;
    const unsigned lidx = xcd * (nwg / 8u) + min(xcd, nwg % 8u) + lin / 8u;
    // x = split * (query tiles) + query tile: the query tiles of one split and kv head (which
    // stream the same keys) stay neighbours in the XCD order
    const int x = (int)(lidx % nx), g = (int)((lidx / nx) % ny), b = (int)(lidx / (nx * ny));
    const int nqt = kSplit ? (int)nx / a.nsplit : (int)nx;
    const int qt = kSplit ? x % nqt : x, split = kSplit ? x / nqt : 0;
    const int tid = threadIdx.x, l = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = a.G;
    // rows of this workgroup: [row0, row0 + nrow) of the sequence's Sq * G (token, head) rows
    const int64_t row0 = (int64_t)qt * kFwRows;
    const int nrow = (int)min((int64_t)kFwRows, (int64_t)a.Sq * G - row0);
    const int tok0 = (int)(row0 / G), tok_last = (int)((row0 + nrow - 1) / G);
    const int tok0_row = (int)(row0 - (int64_t)tok0 * G);  // rows of the first token that come before
    const int seq_len = a.seq_lens[b];
    const int qabs = a.q_abs ? a.q_abs[b] : seq_len - a.Sq;
    // keys any row can see: [0, min(seq_len, last row's position + 1))
    const int hi = min(seq_len, qabs + tok_last + 1);
    const int ntiles = hi > 0 ? (hi - 1) / kTile + 1 : 0;
    const int pmin = qabs + tok0;                      // smallest row position
    // this workgroup's run of key tiles [t0, t1): all of them unless the keys are split
    const int per = kSplit ? (ntiles + a.nsplit - 1) / a.nsplit : ntiles;
    const int t0 = kSplit ? min(ntiles, split * per) : 0, t1 = kSplit ? min(ntiles, t0 + per) : ntiles;

    // The lane number as a value of its own: what is computed from it stays where it is used instead
    // of being kept in registers across the tile loop.
    auto lane_here = [&]() __attribute__((always_inline)) {
        int x = l;
        asm volatile("" : "+v"(x));
        return x;
    };

    // ---- rows of this wave: row r = 64 w + 16 rb + li -> (token, head). Looked up again where
    //      needed (the tile loop has no registers to keep them) ----
    struct Row {
        bool valid;
        int tok, head;
    };
    auto row_of = [&](int rb) __attribute__((always_inline)) {
        int r = 64 * w + 16 * rb + (lane_here() & 15);
        Row x;
        x.valid = r < nrow;
        r = tok0_row + (x.valid ? r : 0);  // row of the workgroup's first token's rows
        x.tok = r / G;
        x.head = r - x.tok * G;
        x.tok += tok0;
        return x;
    };
    half8_t qop[kFwRB][8];
#pragma unroll
    for (int rb = 0; rb < kFwRB; ++rb) {
        const Row r = row_of(rb);
        const T* qrow = static_cast<const T*>(a.q) + (int64_t)b * a.q_sb + (int64_t)(g * G + r.head) * a.q_sh +
                        (int64_t)r.tok * a.q_st;
#pragma unroll
        for (int st = 0; st < 8; ++st) {
            const half8_t v = load_q8<T>(qrow + 64 * (st >> 1) + 16 * (l >> 4) + 8 * (st & 1));
            qop[rb][st] = r.valid ? v : (half8_t)(_Float16)0.0f;
        }
        // one row block's loads at a time: four do not fit the registers in fp32
        asm volatile("" : "+v"(qop[rb][0]), "+v"(qop[rb][1]), "+v"(qop[rb][2]), "+v"(qop[rb][3]), "+v"(qop[rb][4]),
                     "+v"(qop[rb][5]), "+v"(qop[rb][6]), "+v"(qop[rb][7]));
    }
    asm volatile("" ::: "memory");  // every Q load is issued before the block table is read

    lds_u8* L = (lds_u8*)lds;
    const unsigned lds_base = (unsigned)(uintptr_t)L;
    const int8_t* gbase = a.kc + (int64_t)g * a.k_sh;
    // ---- block table of the workgroup's keys into LDS: for bs % 16 == 0 the byte offset / 8 of
    //      every 16-key block's first row, else the page numbers ----
    PageTable pt;
    pt.glob = (const_int_ptr)(uintptr_t)(a.block_table + (int64_t)b * a.bt_stride);
    pt.lds = (const lds_int*)(L + kLdsBt);
    pt.rows16 = nullptr;
    pt.pfirst = 0;
    {
        const int* bt_glob = a.block_table + (int64_t)b * a.bt_stride;
        lds_int* dst = (lds_int*)(L + kLdsBt);
        if constexpr (kFast) {
            const int nblk = 2 * (t1 - t0);  // the workgroup's tiles t0 + i / 2
            pt.in_lds = a.bt32 && nblk <= kFwBt;
            if (pt.in_lds) {
                for (int i = tid; i < nblk; i += kFwWaves * 64) {
                    const int kb = (t0 + (i >> 1)) * kTile;
                    const int klast = min(kb + kTile - 1, hi - 1);
                    const int key0 = min(kb + 16 * (i & 1), klast) & ~15;
                    const int lb = a.bs_shift >= 0 ? key0 >> a.bs_shift : key0 / a.block_size;
                    const int64_t off = (int64_t)bt_glob[lb] * a.k_sb + (int64_t)(key0 - lb * a.block_size) * a.k_ss;
                    dst[i] = (int)(unsigned)((uint64_t)off >> 3);
                }
            }
        } else {
            const int npages = hi > 0 ? (hi - 1) / a.block_size + 1 : 0;
            pt.in_lds = npages <= kFwBt;
            if (pt.in_lds)
                for (int i = tid; i < npages; i += kFwWaves * 64) dst[i] = bt_glob[i];
        }
    }
    __syncthreads();  // the LDS block table is complete

    // Relative scores carry +kPLog2: p' = 2^(s - m + kPLog2) = 16 p, so P' = p' * v_scale spans the
    // same fp16 range as in the decode kernel; l accumulates p' and the final 1 / l removes it.
    constexpr float kPLog2 = 4.0f;
    float l_run[kFwRB];
    // per row: the score offset -m + kPLog2 (kPLog2 while the row has seen no key) and the
    // relative score above which the running max m must be raised (any finite score while fresh)
    float nm_run[kFwRB], thr_run[kFwRB];
    float4_t oacc[kFwRB][16];
#pragma unroll
    for (int rb = 0; rb < kFwRB; ++rb) {
        l_run[rb] = 0.f;
        nm_run[rb] = kPLog2;
        thr_run[rb] = kNegInf;
#pragma unroll
        for (int m = 0; m < 16; ++m) oacc[rb][m] = (float4_t)0.f;
    }

    // tiles [0, n_int) are visible to every row of the workgroup: keys below its first row's
    // position and below hi
    const int n_int = min(pmin + 1 >= 0 ? (pmin + 1) / kTile : 0, hi / kTile);

    // ---- this lane's positions in a slot ----
    // K operand (32-dim step pair c, 16-key block u): 16 source bytes of key row 16 u + li
    int kro[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) kro[c] = ((l & 15) >> 2) * kBlk + 256 * (l & 3) + 64 * (c ^ (l & 3)) + 16 * (l >> 4);
    // transposed V reads: 8 keys of one dim of block m (lanes 2 i, 2 i + 1 of a 16-lane group name tile
    // row tkey); odd row groups hold blocks 0..7 in their second half
    int vro_lo, vro_hi;
    {
        const int h = l >> 4, i = (l & 15) >> 1;
        const int tkey = i < 4 ? 4 * h + i : 12 + 4 * h + i;
        const int at = kFwImgV + ((tkey & 3) + 4 * (tkey >> 4)) * kBlk + 256 * h + 8 * (l & 1);
        vro_lo = at + ((h & 1) ? 128 : 0);
        vro_hi = at - ((h & 1) ? 128 : 0);
    }
    const int sro = kFwImgS + 16 * (l >> 4);  // scales of keys 16 u + 4 lg + j at + 64 u + 4 j

    uint4_t kr[3];       // K bytes of step i = 4 u + c: [i % 3]
    float4_t sc[4];      // k_scale of keys 4 lg .. (u = 0, 1), then v_scale
    auto kread = [&](const lds_u8* S, int i) __attribute__((always_inline)) {
        kr[i % 3] = *(const lds_uint4*)(S + kro[i & 3] + (i >> 2) * 4 * kBlk);
    };
    // the first reads of a tile: two K steps and the scales
    auto tile_start = [&](const lds_u8* S) __attribute__((always_inline)) {
        kread(S, 0);
        kread(S, 1);
#pragma unroll
        for (int j = 0; j < 4; ++j) sc[j] = *(const lds_float4*)(S + sro + 64 * j);
    };

    // ---- tile n from its slot S (its first reads are under way); mid() runs between the scores and the
    //      softmax, next() before the last products ----
    auto tile = [&](int n, const lds_u8* S, auto mid, auto next) __attribute__((always_inline)) {
        float4_t sacc[kFwRB][2];
        constexpr int kVAhead = 2;
        int2_t vr[16];
        auto vread = [&](int m) __attribute__((always_inline)) {
            vr[m] = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_int2*)(S + (m < 8 ? vro_lo : vro_hi) + 16 * m));
        };
        half8_t op = widen_i8x8_exact(kr[0].x, kr[0].y);
        settle_operand(op);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int u = i >> 2, c = i & 3;
            if (i < 6)
                kread(S, i + 2);
            else if (i == 6)
                vread(0);
            else {
#pragma unroll
                for (int m = 1; m < kVAhead; ++m) vread(m);
            }
            if (c == 0)
                op = score_products<true>(sacc[0][u], sacc[1][u], sacc[2][u], sacc[3][u], op, qop[0][2 * c], qop[1][2 * c],
                                          qop[2][2 * c], qop[3][2 * c], kr[i % 3].z, kr[i % 3].w);
            else
                op = score_products<false>(sacc[0][u], sacc[1][u], sacc[2][u], sacc[3][u], op, qop[0][2 * c], qop[1][2 * c],
                                           qop[2][2 * c], qop[3][2 * c], kr[i % 3].z, kr[i % 3].w);
            // the operand after the last is the first of V
            const unsigned w0 = i < 7 ? kr[(i + 1) % 3].x : (unsigned)vr[0].x, w1 = i < 7 ? kr[(i + 1) % 3].y : (unsigned)vr[0].y;
            op = score_products<false>(sacc[0][u], sacc[1][u], sacc[2][u], sacc[3][u], op, qop[0][2 * c + 1],
                                       qop[1][2 * c + 1], qop[2][2 * c + 1], qop[3][2 * c + 1], w0, w1);
        }
        float ks[8], vs[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            ks[e] = sc[e >> 2][e & 3] * a.scale_log2;
            vs[e] = sc[2 + (e >> 2)][e & 3];
        }
        mid();
        settle_scores(sacc);
        float sv[kFwRB][8];
#pragma unroll
        for (int rb = 0; rb < kFwRB; ++rb)
#pragma unroll
            for (int e = 0; e < 8; ++e) sv[rb][e] = __builtin_fmaf(sacc[rb][e >> 2][e & 3], ks[e], nm_run[rb]);
        if (n >= n_int) {  // the tile crosses the causal diagonal or seq_len
            const int key = n * kTile + 4 * (lane_here() >> 4);
            // keys past seq_len may hold garbage scales (even NaN): v_scale 0 makes their P' 0
#pragma unroll
            for (int e = 0; e < 8; ++e) vs[e] = key + 16 * (e >> 2) + (e & 3) < hi ? vs[e] : 0.f;
#pragma unroll
            for (int rb = 0; rb < kFwRB; ++rb) {
                const Row row = row_of(rb);
                const int last = row.valid ? min(hi - 1, qabs + row.tok) : -1;
#pragma unroll
                for (int e = 0; e < 8; ++e) sv[rb][e] = key + 16 * (e >> 2) + (e & 3) <= last ? sv[rb][e] : kNegInf;
            }
        }
        uint64_t need = 0;
#pragma unroll
        for (int rb = 0; rb < kFwRB; ++rb) {
            float mx = kNegInf;
#pragma unroll
            for (int e = 0; e < 8; ++e) mx = fmaxf(mx, sv[rb][e]);
            need |= __builtin_amdgcn_ballot_w64(mx > thr_run[rb]);
        }
        // rare: raise the running max of the rows that need it, shift their scores, rescale their
        // state (O is still zero while every row of a block is fresh: no rescale then)
        if (need != 0) {
#pragma unroll
            for (int rb = 0; rb < kFwRB; ++rb) {
                float mloc = kNegInf;
#pragma unroll
                for (int e = 0; e < 8; ++e) mloc = fmaxf(mloc, sv[rb][e]);
                const float mrow = xor_max(xor_max(mloc, 16), 32) - kPLog2;  // tile max relative to m
                const bool fresh = thr_run[rb] == kNegInf;
                const bool raise = fresh ? mrow > kNegInf : mrow > kLazy;
                const float shift = raise ? mrow : 0.f;
                const float alpha = fresh ? 0.f : __builtin_amdgcn_exp2f(-shift);
                nm_run[rb] -= shift;
                if (raise) thr_run[rb] = kLazy + kPLog2;
#pragma unroll
                for (int e = 0; e < 8; ++e) sv[rb][e] -= shift;
                l_run[rb] *= alpha;
                if (__builtin_amdgcn_ballot_w64(raise && !fresh) != 0) {
                    settle_values(oacc[rb]);
#pragma unroll
                    for (int m = 0; m < 16; m += 4)
                        agpr_scale4_via_lds(oacc[rb][m], oacc[rb][m + 1], oacc[rb][m + 2], oacc[rb][m + 3], alpha,
                                            lds_base + kLdsScr + 4096 * w + 16 * lane_here());
                }
            }
        }
        // p' = 2^sv, P' = p' * v_scale in fp16, O^T += V^T P'^T
        half8_t pop[kFwRB], plo[kFwRB];
#pragma unroll
        for (int rb = 0; rb < kFwRB; ++rb) {
            float psum = 0.f;
#pragma unroll
            for (int e = 0; e < 8; e += 2) {
                const float p0 = __builtin_amdgcn_exp2f(sv[rb][e]);
                const float p1 = __builtin_amdgcn_exp2f(sv[rb][e + 1]);
                psum = e == 0 ? p0 : psum + p0;
                psum += p1;
                if constexpr (kExact) {
                    half2_t ph, pl;
                    split_fp16x2(p0, vs[e], p1, vs[e + 1], ph, pl);
                    pop[rb][e] = ph.x;
                    pop[rb][e + 1] = ph.y;
                    plo[rb][e] = pl.x;
                    plo[rb][e + 1] = pl.y;
                } else {
                    const half2_t ph = __builtin_convertvector((float2_t){p0 * vs[e], p1 * vs[e + 1]}, half2_t);
                    pop[rb][e] = ph.x;
                    pop[rb][e + 1] = ph.y;
                }
            }
            l_run[rb] += psum;
        }
        settle_weights<kExact>(pop, plo);
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            if (m + kVAhead < 16) vread(m + kVAhead);
            if (m == 14) next();
            if constexpr (kExact) value_products_only(oacc[0][m], oacc[1][m], oacc[2][m], oacc[3][m], op, plo[0], plo[1], plo[2], plo[3]);
            if (m < 15)
                op = value_products(oacc[0][m], oacc[1][m], oacc[2][m], oacc[3][m], op, pop[0], pop[1], pop[2], pop[3],
                                    (unsigned)vr[m + 1].x, (unsigned)vr[m + 1].y);
            else
                value_products_only(oacc[0][m], oacc[1][m], oacc[2][m], oacc[3][m], op, pop[0], pop[1], pop[2], pop[3]);
        }
    };

    const int nsteps = (t1 - t0 + kFwStep - 1) / kFwStep;
    const bool busy = 64 * w < nrow;  // a wave without rows only copies

    auto tile_loop = [&](auto lds_flag) __attribute__((always_inline)) {
        constexpr bool kLds = decltype(lds_flag)::value;
        // Starts of the 16-key blocks that this wave's copies of a step read: block u of the step's two tiles and
        // both blocks of tile u (for the scales); with the table in LDS its entries are read together.
        struct Blocks {
            int e[3];  // block u of tile 1 - u, then blocks 0 and 1 of tile u
        };
        const int u = w >> 1;
        auto step_tile = [&](int s, int j) __attribute__((always_inline)) { return min(t0 + kFwStep * s + j, t1 - 1); };
        auto fetch = [&](int s, Blocks& x) __attribute__((always_inline)) {
            if constexpr (kFast && kLds) {
                const int other = step_tile(s, 1 - u) - t0, own = step_tile(s, u) - t0;
                x.e[0] = pt.lds[2 * other + u];
                x.e[1] = pt.lds[2 * own];
                x.e[2] = pt.lds[2 * own + 1];
            }
        };
        auto block_base = [&](int entry, int n, int u) __attribute__((always_inline)) -> const int8_t* {
            if constexpr (kLds) {
                return gbase + ((int64_t)(unsigned)__builtin_amdgcn_readfirstlane(entry) << 3);
            } else {
                const int kb = n * kTile, klast = min(kb + kTile - 1, hi - 1);
                const int key0 = min(kb + 16 * u, klast) & ~15;
                const int lb = a.bs_shift >= 0 ? key0 >> a.bs_shift : key0 / a.block_size;
                return gbase + (int64_t)pt.glob[lb] * a.k_sb + (int64_t)(key0 - lb * a.block_size) * a.k_ss;
            }
        };
        auto row_base = [&](int n, int row) __attribute__((always_inline)) -> const int8_t* {
            const int key = min(n * kTile + row, hi - 1);
            const int lb = a.bs_shift >= 0 ? key >> a.bs_shift : key / a.block_size;
            return gbase + pt.get<kLds>(lb) * a.k_sb + (int64_t)(key - lb * a.block_size) * a.k_ss;
        };
        // This wave's copies of step s: K and V blocks 2 w, 2 w + 1 of both tiles, and 32 scales of tile w >> 1
        // (k_scale for even w, v_scale for odd; lanes 32 (w & 1) .., the others copy nothing). The tile
        // past an odd end is the last one again, so that every step is kFwCopies copies.
        auto issue = [&](int s, int slot0, const Blocks& x) __attribute__((always_inline)) {
            const int k4 = 2 * (w & 1);
            // this lane's source bytes of a K and of a V copy (4 rows x 256 bytes each) and of a scale
            const int lh = lane_here(), qq = lh >> 4, c16 = lh & 15;
            const unsigned kvo = (unsigned)(kFast ? qq * a.k_ss : 0) + 16u * (unsigned)(c16 ^ (4 * qq));
            const unsigned vvo = (unsigned)(kFast ? 4 * qq * a.k_ss : 0) + 260u + 16u * (unsigned)(c16 ^ (8 * (qq & 1)));
            const unsigned first = lds_base + (unsigned)slot0;
            const int8_t *src, *b0, *b1;
            if constexpr (kFast) {
                b0 = block_base(x.e[1], step_tile(s, u), 0);
                b1 = block_base(x.e[2], step_tile(s, u), 1);
            }
#pragma unroll
            for (int j = 0; j < kFwStep; ++j) {
                const unsigned slot = first + (unsigned)(j * kFwSlot);
                if constexpr (kFast) {
                    const int8_t* base = j == u ? (u ? b1 : b0) : block_base(x.e[0], step_tile(s, 1 - u), u);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        dma16_s(base + (int64_t)(4 * (k4 + h)) * a.k_ss, kvo, slot + kImgK + (2 * w + h) * kBlk);
                        dma16_s(base + (int64_t)(k4 + h) * a.k_ss, vvo, slot + kFwImgV + (2 * w + h) * kBlk);
                    }
                } else {
                    const int n = step_tile(s, j);
#pragma unroll
                    for (int h = 0; h < 2; ++h) {
                        dma16_v<0>(row_base(n, 16 * u + 4 * (k4 + h) + qq) + kvo, slot + kImgK + (2 * w + h) * kBlk);
                        dma16_v<0>(row_base(n, 16 * u + (k4 + h) + 4 * qq) + vvo, slot + kFwImgV + (2 * w + h) * kBlk);
                    }
                }
            }
            if constexpr (kFast)
                src = ((lh >> 4) & 1 ? b1 : b0) + (unsigned)(c16 * a.k_ss);
            else
                src = row_base(step_tile(s, u), lh & 31);
            if ((lh >> 5) == (w & 1))
                dma4_v(reinterpret_cast<const int*>(src + (lh < 32 ? 256 : 516)), first + (unsigned)(u * kFwSlot + kFwImgS));
        };
        constexpr int kStepBytes = kFwStep * kFwSlot, kRingBytes = kFwRing * kFwSlot;
        Blocks blk;
        int slot_in = 0, slot_out = 0;  // ring positions (bytes) of the next step to copy and to compute
        auto issue_next = [&](int s) __attribute__((always_inline)) {
            fetch(s, blk);
            issue(s, slot_in, blk);
            slot_in = slot_in + kStepBytes == kRingBytes ? 0 : slot_in + kStepBytes;
        };
        for (int s = 0; s < min(nsteps, kFwAhead); ++s) issue_next(s);
        const int ntl = t1 - t0;
#pragma unroll 1
        for (int i = 0; i < ntl; ++i) {
            const int s = i / kFwStep;
            const bool first = i % kFwStep == 0;
            const lds_u8* S = L + slot_out;
            slot_out = slot_out + kFwSlot == kRingBytes ? 0 : slot_out + kFwSlot;
            if (first) {
                // this wave's copies of step s have landed; then every wave's, and step s - 1 is done
                if (s + 1 < nsteps)
                    wait_vm<kFwCopies>();
                else
                    wait_vm<0>();
                __syncthreads();
                tile_start(S);
            }
            const bool more = first && s + kFwAhead < nsteps;
            if (busy)
                tile(t0 + i, S, [&]() __attribute__((always_inline)) { if (more) issue_next(s + kFwAhead); },
                     // (after the last tile of a step these reads are thrown away)
                     [&]() __attribute__((always_inline)) { tile_start(L + slot_out); });
            else if (more)
                issue_next(s + kFwAhead);
        }
    };
    if (pt.in_lds)
        tile_loop(std::true_type{});
    else
        tile_loop(std::false_type{});

    // ---- normalise and store: out[b, tok, g G + hh, :]; with the keys split, the unnormalised
    //      partial O, the running max m and the sum l of the row instead ----
#pragma unroll
    for (int rb = 0; rb < kFwRB; ++rb) {
        const int lg = l >> 4;
        settle_values(oacc[rb]);
        const float l_row = xor_sum(xor_sum(l_run[rb], 16), 32);
        const Row row = row_of(rb);
        if (!row.valid) continue;
        const int tok = row.tok, head = g * G + row.head;
        if constexpr (kSplit) {
            const int64_t pr = (((int64_t)b * a.Sq + tok) * a.Hq + head) * a.nsplit + split;
            float* prow = a.part_o + pr * kDim + 4 * lg;
#pragma unroll
            for (int m = 0; m < 16; ++m) *reinterpret_cast<float4_t*>(prow + 16 * m) = oacc[rb][m];
            if (lg == 0) {
                a.part_m[pr] = thr_run[rb] == kNegInf ? kNegInf : kPLog2 - nm_run[rb];
                a.part_l[pr] = l_row;
            }
        } else {
            const float inv = l_row > 0.f ? 1.f / l_row : 0.f;
            T* orow = static_cast<T*>(a.out) + (int64_t)b * a.o_sb + (int64_t)tok * a.o_st + (int64_t)head * a.o_sh + 4 * lg;
#pragma unroll
            for (int m = 0; m < 16; ++m) store_out4<T>(orow + 16 * m, oacc[rb][m] * inv);
        }
    }
}

// ---------------------------------------------------------------------------------------
// host side

template <bool kSplit, class T>
static void launch_wide(const FaParams& p, dim3 grid, hipStream_t stream, bool fast, bool exact) {
    const dim3 block(kFwWaves * 64);
    if (fast && !exact)
        hipLaunchKernelGGL((pd_prefill_wide_kernel<true, false, kSplit, T>), grid, block, 0, stream, p);
    else if (!exact)
        hipLaunchKernelGGL((pd_prefill_wide_kernel<false, false, kSplit, T>), grid, block, 0, stream, p);
    else if (fast)
        hipLaunchKernelGGL((pd_prefill_wide_kernel<true, true, kSplit, T>), grid, block, 0, stream, p);
    else
        hipLaunchKernelGGL((pd_prefill_wide_kernel<false, true, kSplit, T>), grid, block, 0, stream, p);
}

hipError_t launch_prefill_wide(const FaParams& p, int batch, int heads_kv, int dtype, hipStream_t stream, bool exact) {
    const int64_t qtiles = ((int64_t)p.Sq * p.G + kFwRows - 1) / kFwRows;
    const dim3 grid((unsigned)(qtiles * p.nsplit), heads_kv, batch);
    const bool fast = fast_block_table(p.block_size, p.k_ss);
    if (dtype == PD_DTYPE_FP16) {
        if (p.nsplit == 1)
            launch_wide<false, _Float16>(p, grid, stream, fast, exact);
        else
            launch_wide<true, _Float16>(p, grid, stream, fast, exact);
    } else {
        if (p.nsplit == 1)
            launch_wide<false, float>(p, grid, stream, fast, exact);
        else
            launch_wide<true, float>(p, grid, stream, fast, exact);
    }
    return hipGetLastError();
}

}  // namespace pd
