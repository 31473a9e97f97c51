// zh_dmmv_mfma.hip -- batched decode DMMV: Q4_K and Q6_K mat-vecs over 2 to 16
// activation vectors (a skinny GEMM, recordBatchDispatchPush
// dmmv.zig:880-925 / dmmv_q4k_batch.comp, dmmv_q6k_batch.comp) on the int8
// MFMA units.
//
// An XQ activation is three int8 limbs per element (zh_device.h), a weight a
// 4- or 6-bit code, so the products of one 32-element block are exact int32
// matrix products: v_mfma_i32_16x16x32_i8 with 16 weight rows on one side
// and 4 vectors x 3 limbs (+ 1 unused) on the other. Lane l of the result
// holds row l % 16 of vector l / 16 with one limb per register, so the limb
// combination, the block scales and the f32 accumulation are lane-local and
// run in the one-vector tile kernels' order (zh_dmmv_lpb.hip): super-blocks
// (Q6_K: their halves) one by one, then summed pairwise in an aligned binary
// tree. Every output therefore equals its one-vector DMMV on those kernels bit
// for bit (and on k_dmmv_q6k_lpb at widths of no multiple of 2048).
#include "zh_device.h"
#include "zh_internal.h"

#include "zh_lpb_common.h"

typedef int i32x4 __attribute__((ext_vector_type(4)));

constexpr int BM_MAXV = ZH_DMMV_MAX_COLS;
constexpr uint32_t BM_SLAB = 16;  // super-blocks of a K slab
// Waves of a workgroup: 16, a super-block of the slab each, where 128
// registers hold the operands; else 8 with two.
constexpr uint32_t bm_waves(uint32_t qtype, uint32_t G) { return G >= (qtype == ZH_Q6_K ? 3 : 4) ? 8 : 16; }
// 16-byte chunks of a row of n super-blocks in LDS, from the 16-byte boundary
// at or below its start; odd, so that 16 rows at one offset hit every bank
// once.
constexpr uint32_t bm_pitch(uint32_t qtype, uint32_t n) {
    return (qtype == ZH_Q4_K ? 9 * n : (210 * n + 14 + 15) / 16) | 1;
}

// Bytes of one 64-element pair of a group of 4 vectors in the activation
// image: 4 vectors x 3 limbs x 4 lane groups x 16 bytes.
constexpr uint32_t BM_PAIR = 768;
constexpr uint32_t bm_image_bytes(uint32_t K, uint32_t G) { return K / 64 * G * BM_PAIR; }
// float4s of scales per 256 elements and vector: Q4_K one per 64 elements
// (xs, sum of x; twice), Q6_K one per 32 (xs, -32 x the two 16-element sums)
constexpr uint32_t bm_scales(uint32_t qtype) { return qtype == ZH_Q4_K ? 4u : 8u; }
constexpr uint32_t bm_scale_bytes(uint32_t qtype, uint32_t K, uint32_t G) { return K / 256 * bm_scales(qtype) * 4 * G * 16; }
// (the widest K and most groups of zhk_dmmv_mfma)
constexpr uint32_t BM_MAXK = 4 * BM_SLAB * 256;
static_assert(bm_image_bytes(BM_MAXK, 4) + bm_scale_bytes(ZH_Q4_K, BM_MAXK, 4) + 3 * BM_MAXV * 8 <= ZH_BMM_WS &&
                  bm_image_bytes(BM_MAXK, 3) + bm_scale_bytes(ZH_Q6_K, BM_MAXK, 3) + 3 * BM_MAXV * 8 <= ZH_BMM_WS,
              "the context's workspace");

struct BmStageP {
    const float *x[BM_MAXV];    // f32 vectors, or
    const uint8_t *xq[BM_MAXV]; // XQ vectors (x[0] == nullptr)
    const float *norm_w;
    float eps;
    uint32_t K, G, q6;
    uint8_t *img;  // [K / 64][G][lane group][vector % 4][limb][2][8] int8
    float4 *sc;    // [K / 64 or K / 32][4 G]
    float *y[3][BM_MAXV];
    float **ytab;  // [3][BM_MAXV]: the outputs, where k_bmm's lanes can index them
};

// The activations of one launch as MFMA operands: each vector RMS-normalised
// (optional), quantised exactly as the one-vector kernels' staging
// (zh_lpb_common.h stage_x_finish) and written in the order the lanes of
// k_bmm load it. Workgroup (v, y) takes 1024 elements of vector v
// (the whole vector's sum of squares first: 16 KB from the L2).
__global__ __launch_bounds__(256) void k_bmm_stage(BmStageP p) {
    __shared__ float red[4];
    const uint32_t v = blockIdx.x, tid = threadIdx.x, e0 = blockIdx.y * 1024u + tid * 4;
    const uint32_t c4 = v & 3, g = v >> 2;
    const float *x = p.x[v];
    if (blockIdx.y == 0 && tid == 0)
        for (uint32_t s = 0; s < 3; s++) p.ytab[s * BM_MAXV + v] = p.y[s][v];
    float rms_inv = 1.f;
    if (p.norm_w) {
        float sq = 0.f;
#pragma unroll 4
        for (uint32_t i = tid * 4; i < p.K; i += 1024) {
            const f32x4 a = *(const f32x4 *)(x + i);
            sq = fmaf(a.x, a.x, sq); sq = fmaf(a.y, a.y, sq); sq = fmaf(a.z, a.z, sq); sq = fmaf(a.w, a.w, sq);
        }
        sq = wave_sum(sq);
        if ((tid & 63) == 0) red[tid >> 6] = sq;
        __syncthreads();
        const float tot = red[0] + red[1] + red[2] + red[3];
        rms_inv = 1.0f / sqrtf(tot / (float)p.K + p.eps);
    }
    // 8 lanes per 32-element block, 4 consecutive elements per lane
    if (e0 < p.K) {
        const uint32_t blk = e0 / 32, sub = tid & 7;
        uint32_t w[3];
        float sc, z;  // z: the 16-element sum of the lane's half (valid in lanes sub 0 and 4)
        if (x) {
            f32x4 a = *(const f32x4 *)(x + e0);
            if (p.norm_w) {
                const f32x4 nw = *(const f32x4 *)(p.norm_w + e0);
                a.x = nw.x * (a.x * rms_inv); a.y = nw.y * (a.y * rms_inv);
                a.z = nw.z * (a.z * rms_inv); a.w = nw.w * (a.w * rms_inv);
            }
            const float amax = row8_max(fmaxf(fmaxf(fabsf(a.x), fabsf(a.y)), fmaxf(fabsf(a.z), fabsf(a.w))));
            float inv;
            xq_scales(amax, inv, sc);
            const int X[4] = {xq_quant(a.x, inv), xq_quant(a.y, inv), xq_quant(a.z, inv), xq_quant(a.w, inv)};
            int l0[4], l1[4], l2[4];
#pragma unroll
            for (int q = 0; q < 4; q++) xq_limbs(X[q], l0[q], l1[q], l2[q]);
            w[0] = pack4(l0[0], l0[1], l0[2], l0[3]);
            w[1] = pack4(l1[0], l1[1], l1[2], l1[3]);
            w[2] = pack4(l2[0], l2[1], l2[2], l2[3]);
            int sm = X[0] + X[1] + X[2] + X[3];
            sm += __builtin_amdgcn_update_dpp(0, sm, 0xB1, 0xF, 0xF, false);  // 16 elements = 4 lanes
            sm += __builtin_amdgcn_update_dpp(0, sm, 0x4E, 0xF, 0xF, false);
            z = (float)sm * sc;
        } else {
            const XQView q = xq_view((void *)p.xq[v], p.K / 32);
#pragma unroll
            for (int k = 0; k < 3; k++) w[k] = *(const uint32_t *)(q.limb + (size_t)blk * 96 + k * 32 + 4 * sub);
            sc = q.xs[blk];
            z = q.xsum[2 * blk + (sub >> 2)];
        }
        uint8_t *dst = p.img + (size_t)(blk / 2 * p.G + g) * BM_PAIR + (sub >> 1) * 192 + (blk & 1) * 8 + (sub & 1) * 4;
#pragma unroll
        for (int k = 0; k < 3; k++) *(uint32_t *)(dst + (c4 * 3 + k) * 16) = w[k];
        const float zh = dpp_f<0x141>(z);  // lane 7 - sub of the 8: the other half's sum
        if (sub == 0) {
            if (p.q6) p.sc[(size_t)blk * 4 * p.G + v] = float4{sc, -32.f * z, -32.f * zh, 0.f};
            else ((float2 *)(p.sc + (size_t)(blk / 2) * 4 * p.G + v))[blk & 1] = float2{sc, z + zh};
        }
    }
}

struct BmP {
    const uint8_t *W[3];  // stacked matrices sharing the vectors
    const uint8_t *W2;    // up matrix (gate/up)
    float *const *ytab;   // [3][BM_MAXV]
    uint32_t M[3], unit_end[3];  // rows; units of 16 NW / kw rows up to and with each matrix
    uint32_t nv, nb, row_bytes, acc;
    uint32_t kw;           // waves that split a slab's super-blocks (a power of two); NW / kw row tiles per unit
    uint32_t nslab, nloc;  // K slabs; units of one matrix per workgroup (at most)
    uint32_t nslot, nred;  // ring slots per wave; units per reduction
    const uint8_t *img;
    const float4 *sc;
};

// A lane's share of one super-block of its row, read from LDS: 8 of every 32
// elements' codes, and the block's scales.
struct BmQ4K {
    static constexpr uint32_t QT = ZH_Q4_K;
    static constexpr uint32_t BPB = 144;
    struct Raw { u32x4 hdr; uint2 q[4]; };
    ZH_DEVM static void load(const uint8_t *blk, uint32_t lg, Raw &r) {
        r.hdr = *(const u32x4 *)blk;
#pragma unroll
        for (int p = 0; p < 4; p++) r.q[p] = *(const uint2 *)(blk + 16 + 32 * p + 8 * lg);
    }
};
struct BmQ6K {
    static constexpr uint32_t QT = ZH_Q6_K;
    static constexpr uint32_t BPB = 210;  // 2-byte aligned: whole dwords, realigned
    struct Raw { uint32_t sc[4]; uint2 ql[4], qh[2]; uint32_t d; };
    ZH_DEVM static uint2 get8(const uint32_t *a, uint32_t sh) {
        const uint32_t x = a[0], y = a[1], z = a[2];
        return uint2{__builtin_amdgcn_alignbyte(y, x, sh), __builtin_amdgcn_alignbyte(z, y, sh)};
    }
    ZH_DEVM static void load(const uint8_t *blk, uint32_t lg, Raw &r) {
        const uint32_t sh = lds_addr(blk) & 3;
        const uint32_t *a = (const uint32_t *)(blk - sh) + 2 * lg;
#pragma unroll
        for (int i = 0; i < 4; i++) r.ql[i] = get8(a + 8 * i, sh);
#pragma unroll
        for (int i = 0; i < 2; i++) r.qh[i] = get8(a + 32 + 8 * i, sh);
        const uint32_t *s = (const uint32_t *)(blk - sh) + 48;
        uint32_t w[6];
#pragma unroll
        for (int i = 0; i < 6; i++) w[i] = s[i];  // (the last may lie past the row: its bytes go unused)
#pragma unroll
        for (int i = 0; i < 4; i++) r.sc[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], sh);
        r.d = __builtin_amdgcn_alignbyte(w[5], w[4], sh);
    }
};

// A choice among values: written on variables that lambdas capture, it
// becomes one load from a chosen address, which keeps them in scratch memory.
template <class T>
ZH_DEV T sel3(uint32_t i, T a, T b, T c) { return i == 0 ? a : i == 1 ? b : c; }

ZH_DEV i32x4 mfma_i8(uint32_t a0, uint32_t a1, uint32_t b0, uint32_t b1) {
    return __builtin_amdgcn_mfma_i32_16x16x32_i8((long)((uint64_t)a1 << 32 | a0), (long)((uint64_t)b1 << 32 | b0),
                                                 i32x4{0, 0, 0, 0}, 0, 0, 0);
}

// comb_i as two shift-adds (the compiler's own order takes three instructions)
ZH_DEV int bm_comb(i32x4 d) {
    int t = (d[2] << 8) + d[1];
    asm("" : "+v"(t));
    return (t << 8) + d[0];
}

// One super-block of 16 rows x 4 G vectors; sc(j, g): scale float4 j of the
// lane's vector of group g.
template <int G, class S>
ZH_DEV void bm_block(const BmQ4K::Raw &r, const u32x4 (&A)[4][G], const S &sc, float (&res)[G]) {
    uint32_t raw[4] = {r.hdr.x, r.hdr.y, r.hdr.z, r.hdr.w};
    LpbQ4K::Hdr h = LpbQ4K::header(raw);
    asm("" : "+v"(h.scA), "+v"(h.mA));  // (else each scale is a bit-field extract and a conversion)
    float accd[G], accm[G];
#pragma unroll
    for (int g = 0; g < G; g++) accd[g] = accm[g] = 0.f;
#pragma unroll
    for (int p = 0; p < 4; p++) {
        const uint32_t l0 = r.q[p].x & 0x0F0F0F0Fu, l1 = r.q[p].y & 0x0F0F0F0Fu;
        const uint32_t h0 = (r.q[p].x >> 4) & 0x0F0F0F0Fu, h1 = (r.q[p].y >> 4) & 0x0F0F0F0Fu;
        const uint32_t scw = p < 2 ? h.scA : h.scB, mw = p < 2 ? h.mA : h.mB;
        const float sc0 = ubyte_f(scw, (2 * p) & 3), sc1 = ubyte_f(scw, (2 * p + 1) & 3);
        const float m0 = ubyte_f(mw, (2 * p) & 3), m1 = ubyte_f(mw, (2 * p + 1) & 3);
#pragma unroll
        for (int g = 0; g < G; g++) {
            const i32x4 D0 = mfma_i8(A[p][g].x, A[p][g].y, l0, l1), D1 = mfma_i8(A[p][g].z, A[p][g].w, h0, h1);
            const float4 s = sc(p, g);
            accd[g] = fmaf(sc0 * s.x, (float)bm_comb(D0), accd[g]);
            accd[g] = fmaf(sc1 * s.z, (float)bm_comb(D1), accd[g]);
            accm[g] = fmaf(m0, s.y, accm[g]);
            accm[g] = fmaf(m1, s.w, accm[g]);
        }
        __builtin_amdgcn_sched_barrier(0);  // (the next pair's products wait: more in flight spill)
    }
#pragma unroll
    for (int g = 0; g < G; g++) res[g] = fmaf(h.d, accd[g], -h.dmin * accm[g]);
}

// Q6_K has a scale per 16 elements: two products per block, the codes of the
// other 16 elements (the lane groups 0-1 or 2-3) masked to zero.
template <int G, class S>
ZH_DEV void bm_block(const BmQ6K::Raw &r, const u32x4 (&A)[4][G], const S &sc, float (&res)[G]) {
    const uint32_t m0 = (threadIdx.x & 32) ? 0u : ~0u, m1 = ~m0;
    const float d = h2f(r.d);
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float acc[G];
#pragma unroll
        for (int g = 0; g < G; g++) acc[g] = 0.f;
#pragma unroll
        for (int s4 = 0; s4 < 4; s4++) {
            const uint2 ql = r.ql[2 * h + (s4 & 1)], qh = r.qh[h];
            const uint32_t q0 = ((ql.x >> (4 * (s4 >> 1))) & 0x0F0F0F0Fu) | (((qh.x >> (2 * s4)) << 4) & 0x30303030u);
            const uint32_t q1 = ((ql.y >> (4 * (s4 >> 1))) & 0x0F0F0F0Fu) | (((qh.y >> (2 * s4)) << 4) & 0x30303030u);
            const int i0 = 8 * h + 2 * s4, i1 = i0 + 1;
            const float s0 = (float)(int)(int8_t)((r.sc[i0 >> 2] >> (8 * (i0 & 3))) & 0xFF);
            const float s1 = (float)(int)(int8_t)((r.sc[i1 >> 2] >> (8 * (i1 & 3))) & 0xFF);
            const int j = 4 * h + s4;  // 32-element block of the super-block
#pragma unroll
            for (int g = 0; g < G; g++) {
                const uint32_t a0 = j & 1 ? A[j >> 1][g].z : A[j >> 1][g].x, a1 = j & 1 ? A[j >> 1][g].w : A[j >> 1][g].y;
                const i32x4 D0 = mfma_i8(a0, a1, q0 & m0, q1 & m0), D1 = mfma_i8(a0, a1, q0 & m1, q1 & m1);
                const float4 s = sc(j, g);
                acc[g] = fmaf(s0, fmaf(s.x, comb_f(D0[0], D0[1], D0[2]), s.y), acc[g]);
                acc[g] = fmaf(s1, fmaf(s.x, comb_f(D1[0], D1[1], D1[2]), s.z), acc[g]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
#pragma unroll
        for (int g = 0; g < G; g++) {  // (rounded before the halves are summed, as in the one-vector kernel's lanes)
            float t = d * acc[g];
            asm("" : "+v"(t));  // (else one multiply-add)
            res[g] = h ? res[g] + t : t;
        }
    }
}

// Bound by HBM up to about 8 vectors of Q4_K, by the per-block VALU work
// (limb combination, scales) past that. A wave keeps the operands of its
// super-blocks of every vector in registers for the whole slab, and 16 rows
// at a time of those super-blocks stream past it through its own ring of LDS
// slots, filled by its own copies: no wave waits for another until the
// partial rows of `nred` units are summed over the waves (one barrier; two
// buffers). Measured on the way, gate/up (2 x 12288 x 4096) of 6 vectors:
// rows loaded straight into registers in the operand's layout, where lanes 16
// apart share a row and do not coalesce, 29 us; whole rows copied by all
// waves with a barrier per unit 21 us. K beyond 16 super-blocks is walked in
// slabs, the partial rows kept in LDS.
template <class F, int G, int MODE>
__global__ __launch_bounds__(bm_waves(F::QT, G) * 64) void k_bmm(BmP p) {
    extern __shared__ __align__(16) uint8_t lds[];
    constexpr int NM = MODE == LPB_GATE_UP ? 2 : 1;
    constexpr int NS = F::BPB == 144 ? 4 : 8;  // scale float4s per super-block and vector
    constexpr uint32_t NW = bm_waves(F::QT, G), SPW = BM_SLAB / NW, T = NW * 64;  // SPW: super-blocks per wave
    constexpr uint32_t SLAB_BYTES = BM_SLAB * F::BPB, PITCH = bm_pitch(F::QT, SPW);  // chunks per row of a slot
    constexpr uint32_t ND = (16 * PITCH + 63) / 64, SLOT = 256 * PITCH;              // copies and bytes of a slot
    constexpr uint32_t RED = NW * G * 64;                                            // partial sums of a unit
    const uint32_t tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t lane = tid & 63, lj = lane & 15, lg = lane >> 4;
    const uint32_t nslot = p.nslot, nred = p.nred, nb = p.nb, nslab = p.nslab, row_bytes = p.row_bytes;
    uint8_t *const ring = lds + wave * nslot * SLOT;
    float **ytab = (float **)(lds + NW * nslot * SLOT);             // [3][BM_MAXV]
    float4 *scl = (float4 *)(ytab + 3 * BM_MAXV) + wave * (SPW * NS * 4 * G);  // this wave's [SPW NS][4 G] scales
    float *red = (float *)((float4 *)(ytab + 3 * BM_MAXV) + BM_SLAB * NS * 4 * G);  // [2][nred][NW][G][64]
    float *part = red + 2 * nred * RED;                             // [nloc][NM][G * 64] (x 2 for 4 slabs)
    const uint32_t kw = wave & (p.kw - 1), rw = wave / p.kw, RW = NW / p.kw, UR = 16 * RW;
    // (as values: indexed by a unit's matrix, the argument's arrays would be copied to scratch memory)
    const uint32_t ue0 = p.unit_end[0], ue1 = p.unit_end[1], nround = p.unit_end[2];
    const uint32_t M0 = p.M[0], M1 = p.M[1], M2 = p.M[2];
    const uint8_t *const W0 = p.W[0], *const W1 = p.W[1], *const W2 = p.W[2], *const Wu = p.W2;
    const uint32_t ring0 = lds_addr(ring);
    const uint32_t nloc = (nround - blockIdx.x + gridDim.x - 1) / gridDim.x;  // units of one matrix and slab here
    const uint32_t nu = nslab * nloc * NM;
    // Units run slab by slab, in a slab round by round, gate before up. A
    // unit's rows are [r0, r0 + UR) of its matrix, moved up to end with it
    // (rows below rlo are another unit's).
    struct Unit { uint32_t slab, loc, m, slot; };
    struct Rows { uint32_t r0, rlo, Ms, sg; };
    auto advance = [&](Unit &t) __attribute__((always_inline)) {
        t.slot = t.slot + 1 == nslot ? 0u : t.slot + 1;
        if (NM == 2 && (t.m ^= 1u)) return;
        if (++t.loc == nloc) t.loc = 0, t.slab++;
    };
    auto rows_of = [&](uint32_t loc) __attribute__((always_inline)) {
        Rows r;
        const uint32_t rd = blockIdx.x + loc * gridDim.x;
        r.sg = (rd >= ue0 ? 1u : 0u) + (rd >= ue1 ? 1u : 0u);
        r.Ms = sel3(r.sg, M0, M1, M2);
        r.rlo = UR * (rd - sel3(r.sg, 0u, ue0, ue1));
        r.r0 = r.Ms >= UR ? min(r.rlo, r.Ms - UR) : 0u;
        return r;
    };
    // 16 rows x SPW super-blocks of the wave's: row r's bytes from the
    // 16-byte boundary at or below their start. With rows of a multiple of 16
    // bytes the lane's offsets serve every unit of a whole slab.
    const uint32_t nbs = min(nb, BM_SLAB);
    auto place = [&](uint32_t i, uint32_t bytes, uint64_t base, uint32_t rmax) __attribute__((always_inline)) {
        const uint32_t pos = i * 64 + lane, r = pos / PITCH, ch = pos - r * PITCH;  // (r < 16: lanes past it copy nothing)
        const uint64_t a = base + (uint64_t)min(rw * 16 + r, rmax) * row_bytes + SPW * kw * F::BPB;
        const uint32_t sh = (uint32_t)a & 15;
        return a - sh + 16 * min(ch, (sh + bytes - 1) / 16);
    };
    const uint32_t rmax0 = min(UR, M0) - 1;
    const uint32_t wbytes = SPW * kw < nbs ? min(SPW, nbs - SPW * kw) * F::BPB : 0u;  // of a row, in a whole slab
    uint32_t off[ND];
#pragma unroll
    for (uint32_t i = 0; i < ND; i++) off[i] = (uint32_t)place(i, max(wbytes, 1u), 0, rmax0);
    const uint32_t sh0 = (min(rw * 16 + lj, rmax0) * row_bytes + SPW * kw * F::BPB) & 15;  // of the row this lane computes
    auto copy = [&](const Unit &t) __attribute__((always_inline)) {
        const Rows tr = rows_of(t.loc);
        const uint64_t base = (uint64_t)(uintptr_t)(t.m ? Wu : sel3(tr.sg, W0, W1, W2)) + (uint64_t)tr.r0 * row_bytes +
                              t.slab * SLAB_BYTES;
        const uint32_t dst = ring0 + t.slot * SLOT, b = t.slab * BM_SLAB + SPW * kw;
        if (b >= nb) return;
        const bool whole = row_bytes % 16 == 0 && nb - t.slab * BM_SLAB >= nbs;
        const uint32_t bytes = min(SPW, nb - b) * F::BPB;
#pragma unroll
        for (uint32_t i = 0; i < ND; i++)
            if (i * 64 + 64 <= 16 * PITCH || lane < 16 * PITCH - i * 64)
                dma16((const void *)(whole ? base + off[i] : place(i, bytes, base, tr.Ms - 1 - tr.r0)), dst + i * 1024);
    };
    u32x4 A[SPW][4][G];
    // the scales in registers where they leave room (their LDS reads cost as much as the weights')
    constexpr bool SREG = F::QT == ZH_Q4_K ? G <= 2 : G == 1;
    float4 S[SREG ? NS : 1][G];
    auto load_x = [&](uint32_t slab) __attribute__((always_inline)) {
        const uint32_t b = slab * BM_SLAB + SPW * kw;
        const uint32_t limb = lj & 3;
        const uint8_t *xi = p.img + (lg * 12 + (lj >> 2) * 3 + limb) * 16;
#pragma unroll
        for (int i = 0; i < 4 * (int)SPW; i++)
#pragma unroll
            for (int g = 0; g < G; g++) {
                A[i >> 2][i & 3][g] = u32x4{0, 0, 0, 0};
                if (limb < 3) A[i >> 2][i & 3][g] = *(const u32x4 *)(xi + (min(4 * b + i, 4 * nb - 1) * G + g) * BM_PAIR);
            }
        constexpr uint32_t NSC = SPW * NS * 4 * G;  // one load each, then broadcast from LDS
#pragma unroll
        for (uint32_t i = 0; i < (NSC + 63) / 64; i++) {
            const uint32_t e = i * 64 + lane;
            if (NSC % 64 == 0 || e < NSC) scl[e] = p.sc[min(NS * b * 4 * G + e, NS * nb * 4 * G - 1)];
        }
        if constexpr (SREG)
#pragma unroll
            for (int j = 0; j < NS; j++)
#pragma unroll
                for (int g = 0; g < G; g++) S[j][g] = scl[(j * G + g) * 4 + lg];
        // wait for them here: a wait at their first use would sit in the unit
        // loop and drain the copies in flight every time round
#pragma unroll
        for (int i = 0; i < 4 * (int)SPW; i++)
#pragma unroll
            for (int g = 0; g < G; g++) asm volatile("" : "+v"(A[i >> 2][i & 3][g]));
    };
    const uint32_t nvalid = SPW * kw < nb ? (nb - SPW * kw + BM_SLAB - 1) / BM_SLAB * nloc * NM : 0u;
    Unit cu = {0, 0, 0, 0}, nx = {0, 0, 0, 0};  // the unit computed, the next to copy
    copy(nx);
    advance(nx);
    float *yp0 = nullptr;
    if (tid < 3 * BM_MAXV) yp0 = p.ytab[tid];
    load_x(0);
    if (tid < 3 * BM_MAXV) ytab[tid] = yp0;
    uint32_t issued = 1;
    for (; issued < nslot && issued < nu; issued++) {
        copy(nx);
        advance(nx);
    }
    for (uint32_t u = 0, ug = 0, buf = 0; u < nu; u++, advance(cu)) {
        const Unit t = cu;
        if (u && t.loc == 0 && t.m == 0) load_x(t.slab);
        const uint32_t b = t.slab * BM_SLAB + SPW * kw;
        float res[G];
#pragma unroll
        for (int g = 0; g < G; g++) res[g] = 0.f;
        if (b < nb) {
            // this unit's copies: those of the units after it (of slabs the wave has a part of) may be in flight
            switch (min(issued, nvalid) - u - 1) {
            case 0: wait_vm<0>(); break;
            case 1: wait_vm<ND>(); break;
            default: wait_vm<2 * ND>(); break;  // (nslot <= 3)
            }
            uint32_t sh = sh0;
            if (F::BPB != 144 && row_bytes % 16) {
                const Rows tr = rows_of(t.loc);
                sh = ((uint32_t)(uintptr_t)(t.m ? Wu : sel3(tr.sg, W0, W1, W2)) + SPW * kw * F::BPB +
                      (tr.r0 + min(rw * 16 + lj, tr.Ms - 1 - tr.r0)) * row_bytes) & 15u;
            }
            const uint8_t *row = ring + t.slot * SLOT + lj * PITCH * 16 + sh;
            typename F::Raw raw[SPW];
#pragma unroll
            for (uint32_t i = 0; i < SPW; i++) F::load(row + i * F::BPB, lg, raw[i]);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            if (issued < nu) copy(nx);  // into the slot just read
            bm_block<G>(raw[0], A[0], [&](int j, int g) __attribute__((always_inline)) {
                if constexpr (SREG) return S[j][g];
                else return scl[(j * G + g) * 4 + lg];
            }, res);
            if (SPW == 2 && b + 1 < nb) {
                float r1[G];
                bm_block<G>(raw[SPW - 1], A[SPW - 1], [&](int j, int g) __attribute__((always_inline)) {
                    return scl[((NS + j) * G + g) * 4 + lg];
                }, r1);
#pragma unroll
                for (int g = 0; g < G; g++) res[g] += r1[g];
            }
        } else if (issued < nu) {
            copy(nx);
        }
        if (issued < nu) {
            issued++;
            advance(nx);
        }
        float *rb = red + buf * nred * RED + (ug * NW + wave) * (G * 64) + lane;
#pragma unroll
        for (int g = 0; g < G; g++) rb[g * 64] = res[g];
        if (++ug < nred && u + 1 < nu) continue;
        // ---- sum the waves' partial rows of the last ug units
        lds_bar();
        const float *rsum = red + buf * nred * RED;
        const uint32_t u0 = u + 1 - ug;
        // the sum of unit j's row tile irw, vector group g, this lane's vector and row
        auto total = [&](uint32_t j, uint32_t irw, uint32_t g) __attribute__((always_inline)) {
            const float *r = rsum + ((j * NW + irw * p.kw) * G + g) * 64 + lane;
            float v[NW];
#pragma unroll
            for (uint32_t k = 0; k < NW; k++) {
                v[k] = r[min(k, p.kw - 1) * (G * 64)];
                v[k] = k < p.kw ? v[k] : 0.f;
            }
#pragma unroll
            for (uint32_t w = NW / 2; w; w /= 2)
#pragma unroll
                for (uint32_t k = 0; k < w; k++) v[k] = v[2 * k] + v[2 * k + 1];
            return v[0];
        };
        auto store = [&](uint32_t loc, uint32_t irw, uint32_t g, float s) __attribute__((always_inline)) {
            const Rows tr = rows_of(loc);
            const uint32_t row = tr.r0 + irw * 16 + lj, v = 4 * g + lg;
            if (row < tr.rlo || row >= tr.Ms || v >= p.nv) return;
            typedef __attribute__((address_space(1))) float gfloat;  // (a flat access would wait for the ring too)
            gfloat *yp = (gfloat *)(uintptr_t)ytab[tr.sg * BM_MAXV + v] + row;
            if (p.acc) s += *yp;
            *yp = s;
        };
        if (nslab == 1) {  // (u0 and ug are even where a gate waits for its up)
#pragma nounroll
            for (uint32_t i = wave; i < ug / NM * RW * G; i += NW) {
                const uint32_t g = i % G, irw = i / G % RW, j = i / G / RW;
                const float s = total(NM * j, irw, g);
                if (NM == 2) store(u0 / 2 + j, irw, g, silu_mul(s, total(NM * j + 1, irw, g)));
                else store(u0 + j, irw, g, s);
            }
        } else if (wave < G) {  // one row tile per unit; its slabs' sums in order: (s0 + s1) + (s2 + s3)
            uint32_t rest = u0 / NM, slab = rest / nloc, loc = rest - slab * nloc, m = NM == 2 ? u0 & 1 : 0u;
            float gate = 0.f;
#pragma nounroll
            for (uint32_t j = 0; j < ug; j++) {
                float s = total(j, 0, wave);
                float *pt = part + (loc * NM + m) * (G * 64) + wave * 64 + lane, *pt2 = pt + p.nloc * NM * G * 64;
                const bool last = slab + 1 == nslab;
                if (slab == 1) s = *pt + s;
                if (slab == 2 && last) s = *pt + s;
                if (slab == 3) s = *pt + (*pt2 + s);
                if (!last) *(slab == 2 ? pt2 : pt) = s;
                else if (NM == 1) store(loc, 0, wave, s);
                else if (m == 0) gate = s;
                else store(loc, 0, wave, silu_mul(gate, s));
                if (NM == 2 && (m ^= 1u)) continue;
                if (++loc == nloc) loc = 0, slab++;
            }
        }
        ug = 0;
        buf ^= 1;
    }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
template <class F, int G, int MODE>
static int bm_launch(zh_ctx *c, BmP &p) {
    constexpr uint32_t NM = MODE == LPB_GATE_UP ? 2 : 1, NS = F::BPB == 144 ? 4 : 8, NW = bm_waves(F::QT, G);
    constexpr uint32_t LDS = 160 * 1024, SLOTS = NW * 256 * bm_pitch(F::QT, BM_SLAB / NW), RED = 2 * NW * G * 256;
    constexpr uint32_t fixed = 3 * BM_MAXV * 8 + BM_SLAB * NS * 4 * G * 16;
    static_assert(2 * SLOTS + fixed + NM * RED + 2 * NM * G * 256 <= LDS, "two ring slots and one unit's rows");
    const uint32_t nround = p.unit_end[2];
    const uint32_t slab = p.nslab > 1 ? NM * G * 256 * (p.nslab > 3 ? 2 : 1) : 0;  // per unit of a workgroup
    uint32_t wgs = (uint32_t)c->cu_count < nround ? (uint32_t)c->cu_count : nround;
    p.nloc = (nround + wgs - 1) / wgs;
    while (p.nloc > 1 && 2 * SLOTS + fixed + NM * RED + p.nloc * slab > LDS) {  // more workgroups, fewer units each
        p.nloc--;
        wgs = (nround + p.nloc - 1) / p.nloc;
    }
    // three slots if a reduction every two units fits beside them, then as many units per reduction as fit
    const uint32_t room = LDS - fixed - p.nloc * slab, nu = p.nslab * p.nloc * NM;
    p.nslot = 3 * SLOTS + 2 * RED <= room ? 3 : 2;
    p.nred = (room - p.nslot * SLOTS) / (RED * NM) * NM;
    if (p.nred > 4) p.nred = 4;
    if (p.nred > nu) p.nred = nu;
    const uint32_t lds = p.nslot * SLOTS + fixed + p.nred * RED + p.nloc * slab;
    hipLaunchKernelGGL((k_bmm<F, G, MODE>), dim3(wgs), dim3(NW * 64), lds, c->stream, p);
    ZH_LAUNCH_CHECK(c);
    return ZH_OK;
}
template <class F, int MODE>
static int bm_launch_g(zh_ctx *c, BmP &p, uint32_t G) {
    switch (G) {
    case 1: return bm_launch<F, 1, MODE>(c, p);
    case 2: return bm_launch<F, 2, MODE>(c, p);
    case 3: return bm_launch<F, 3, MODE>(c, p);
    default: break;
    }
    if constexpr (F::QT == ZH_Q4_K) return bm_launch<F, 4, MODE>(c, p);
    return zh_set_err(c, ZH_ERR_INVALID_ARGUMENT, "batched dmmv: %u vectors", p.nv);
}

bool zhk_dmmv_mfma_fits(uint32_t qtype, int mode, uint32_t nseg, const uint8_t *const *W, const uint8_t *W2,
                        const uint32_t *M, uint32_t K) {
    const uint32_t nb = K / 256, unit_rows = nb > 8 ? 16 : nb > 4 ? 32 : nb > 2 ? 64 : 128;
    bool fits = K % 256 == 0 && nb && K <= BM_MAXK && nseg >= 1 && nseg <= 3 &&
                (qtype == ZH_Q4_K || qtype == ZH_Q6_K) &&
                (mode == LPB_PLAIN || (qtype == ZH_Q4_K && nseg == 1 && ((uintptr_t)W2 & 15) == 0));
    // 16-byte aligned matrices; stacked ones at least a unit tall
    for (uint32_t s = 0; fits && s < nseg; s++)
        fits = M[s] && ((uintptr_t)W[s] & 15) == 0 && (nseg == 1 || M[s] >= unit_rows);
    return fits;
}

// y[s * y_stride + v] (= or +=) W[s] x_v for v < nv <= 16 on one pass over
// the weights (two for Q6_K past 12), x_v = x[v] (f32, with the optional
// fused RMSNorm) or xq[v] (XQ; x == nullptr), where zhk_dmmv_mfma_fits.
int zhk_dmmv_mfma(zh_ctx *c, uint32_t qtype, int mode, uint32_t nseg, const uint8_t *const *W, const uint8_t *W2,
                  const uint32_t *M, uint32_t K, uint32_t n_vec, const float *const *x, const void *const *xq,
                  float *const *y, uint32_t y_stride, const float *norm_w, float eps, uint32_t acc) {
    const uint32_t nb = K / 256;
    for (uint32_t v0 = 0; v0 < n_vec;) {
        // Q6_K: past 12 vectors the scales and partial rows leave the LDS no
        // second ring slot; 13 to 16 run as 8 and the rest
        const uint32_t left = n_vec - v0, most = qtype == ZH_Q6_K ? 12 : 16;
        const uint32_t nv = left <= most ? left : qtype == ZH_Q6_K ? 8u : 16u;
        // waves that split K: all from 9 super-blocks on
        const uint32_t G = (nv + 3) / 4, NW = bm_waves(qtype, G), unit_rows = nb > 8 ? 16 : nb > 4 ? 32 : nb > 2 ? 64 : 128;
        const uint32_t img = bm_image_bytes(K, G), scb = bm_scale_bytes(qtype, K, G);
        BmStageP sp = {};
        BmP p = {};
        for (uint32_t v = 0; v < nv; v++) {
            sp.x[v] = x ? x[v0 + v] : nullptr;
            sp.xq[v] = x ? nullptr : (const uint8_t *)xq[v0 + v];
            for (uint32_t s = 0; s < nseg; s++) sp.y[s][v] = y[s * y_stride + v0 + v];
        }
        sp.norm_w = x ? norm_w : nullptr; sp.eps = eps; sp.K = K; sp.G = G; sp.q6 = qtype == ZH_Q6_K;
        sp.img = (uint8_t *)c->bmm_ws;
        sp.sc = (float4 *)(sp.img + img);
        sp.ytab = (float **)(sp.img + img + scb);
        hipLaunchKernelGGL(k_bmm_stage, dim3(nv, (K + 1023) / 1024), dim3(256), 0, c->stream, sp);
        ZH_LAUNCH_CHECK(c);
        uint32_t end = 0;
        for (uint32_t s = 0; s < 3; s++) {
            if (s < nseg) {
                p.W[s] = W[s];
                p.M[s] = M[s];
                end += (M[s] + unit_rows - 1) / unit_rows;
            }
            p.unit_end[s] = end;
        }
        p.W2 = W2;
        p.nv = nv; p.nb = nb; p.row_bytes = (uint32_t)zh_tensor_bytes(qtype, 1, K); p.acc = acc;
        p.kw = 16 * NW / unit_rows;
        p.nslab = (nb + BM_SLAB - 1) / BM_SLAB;
        p.img = sp.img; p.sc = sp.sc; p.ytab = sp.ytab;
        const int rl = qtype == ZH_Q6_K      ? bm_launch_g<BmQ6K, LPB_PLAIN>(c, p, G)
                       : mode == LPB_GATE_UP ? bm_launch_g<BmQ4K, LPB_GATE_UP>(c, p, G)
                                             : bm_launch_g<BmQ4K, LPB_PLAIN>(c, p, G);
        if (rl) return rl;
        v0 += nv;
    }
    return ZH_OK;
}
