// gemm.hip -- batched projection for prefill on gfx950 matrix cores:
//   C[t][r] = sum_k f16(dequant(W)[r][k]) * X[t][k]     (f32 accumulate)
// for n tokens t at once (reference: the batched-prefill MMQ kernels
// qwen3_5/metal.odin:493-609 and gemm_harness/gemm_test.odin:97-135, 297-337,
// which stage both operands in half precision and accumulate in float).
// X is token-major f16 [n][K], C token-major f32 [n][M] (the transposes of the
// reference harness's B[K][N] and C[M][N]; same products).
//
// Work layout: a workgroup of 8 waves computes 128 rows x 16 TT tokens (TT = 8,
// 6, 4 or 2) over a slice of K, walked in chunks of 256 (one Q4_K / Q6_K
// super-block, eight Q8_0 blocks).  Per chunk the activations and the raw
// weight bytes are staged in LDS; wave (rg, kh) takes rows 32 rg .. +31 and
// half kh of the chunk's sixteen 16-wide K steps, in v_mfma_f32_32x32x16_f16
// accumulators (TT / 2 tiles of 32 tokens), so every weight is dequantized once
// per workgroup; the two K halves are added through LDS at the end.
//
// What bounds it: no unit, but how far two waves a SIMD with two barriers a chunk
// overlap them.  Per chunk at TT = 8 (counters, gate and up of the 8B shape at 512
// tokens), of 4800 clocks: the products 2050 a SIMD, the vector instructions 2090 with
// the products' issue, the LDS 2170 and 170 of conflicts; 1.57 us a chunk alone and
// 2.1 - 2.3 with every CU busy on random data, where the card lowers its clock (a plain
// 8192^3 f16 product: 1795 TFLOP/s on zeros, 1315 on random data).  Measured on the way:
//   - The weights go through LDS because of the loads: straight into the operand
//     layout (16 rows x 64 bytes per instruction, the row in the fast lanes) a
//     16-byte-per-lane load takes 65 clocks of the CU's address unit, with the
//     four lanes of a row side by side 19-25 (L2-resident), and that alone took
//     1560 clocks a chunk.
//   - Two 16x16x32 products in place of one 32x32x16 hold up twice as many issue
//     slots of the vector instructions beside them: 1.69 against 1.57 us a chunk;
//     codes converted by v_cvt_f32_ubyte* instead of codes8: 1.84.
//   - 128 tokens per workgroup halve the dequantization per product against 64.
// 512 tokens, Q4_K, against 128 rows x 64 tokens with the weights loaded into the
// operand layout: 4096 x 12288 86 -> 62 us, gate and up 2 x 12288 x 4096 with the
// SwiGLU 159 -> 132 us; Q6_K 4096 x 12288 at 333 tokens 91.5 -> 63 us.
//
// Dequantization follows ggml/quant.odin exactly (separately rounded products,
// (d*sc)*q for Q6_K), then rounds to f16 (RNE), as the reference's staging.
// The K order inside a chunk is a permutation chosen so that each lane's bytes
// are contiguous; the activation octets are read by the same permutation
// (octet), so every product pairs the right weight with the right activation.
//
// The FFN's gate and up projections can run as one pass (gemm_q_kernel<G, 2>,
// launch_gemm_swiglu) that writes the f16 SwiGLU of the pair instead of two
// f32 products.
//
// Operand layout of v_mfma_f32_32x32x16_f16 (per lane l, 8 halves each):
//   A[i][k]: i = l % 32, k = 8 (l / 32) + e;  B[k][j]: j = l % 32, k = 8 (l / 32) + e
//   D[i][j] (16 floats): j = l % 32, i = 8 (v / 4) + 4 (l / 32) + v % 4.

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include "device_common.h"

namespace oi {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f32x4v __attribute__((ext_vector_type(4)));
typedef float f32x16v __attribute__((ext_vector_type(16)));
typedef float f32x2v __attribute__((ext_vector_type(2)));

typedef __amdgpu_buffer_rsrc_t rsrc_t;
// raw buffer descriptors (data format 32, the gfx9 value for untyped access):
// 32-bit per-lane offsets and a uniform per-chunk offset, so the loads need no
// 64-bit address arithmetic; reads past `bytes` return zero
static __device__ __forceinline__ rsrc_t make_rsrc(const void *p, size_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(p), (short)0, (int)(uint32_t)bytes, 0x00020000);
}
static __device__ __forceinline__ u32x4 bld16(rsrc_t r, uint32_t voff, uint32_t soff) {
    return __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0);
}

constexpr int GM_THREADS = 512;
constexpr int GM_ROWS = 128;  // rows per workgroup (64 of each matrix when two share it)
constexpr int GM_KC = 256;    // K per chunk

// one projection of a launch: its matrix, partial products ([split][n][rows]),
// K chunks per slice, row tiles, and its first block
struct GemmSeg {
    DMat m;
    float *c;
    int32_t cps, nx, first;
};
constexpr int GM_MAX_SEG = 4;
// projections of the same x (same type and K) in one launch: a flat grid whose
// block b belongs to the last segment with first <= b
struct GemmArgs {
    const uint16_t *x;  // [n][K] f16
    int32_t n, nseg;
    GemmSeg seg[GM_MAX_SEG];
    DMat m2;            // two matrices: the up matrix (seg[0].m is gate), same type and shape
    uint16_t *h;        // two matrices: [n][M] f16 silu(gate x) * (up x)
};

// f32 -> f16 (RNE) of values already rounded to f32 (the empty asm keeps the
// conversion apart from the fma that produced the value, see f2h; two values
// convert with one v_cvt_pk_f16_f32)
static __device__ __forceinline__ h8 cvt8(float (&v)[8]) {
    u32x4 r;
#pragma unroll
    for (int e = 0; e < 4; e++) {
        asm("" : "+v"(v[2 * e]));
        asm("" : "+v"(v[2 * e + 1]));
        r[e] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2v{v[2 * e], v[2 * e + 1]}), h2v));
    }
    return __builtin_bit_cast(h8, r);
}
static __device__ __forceinline__ uint32_t byte_of(uint32_t lo, uint32_t hi, int e) {
    return ((e < 4 ? lo : hi) >> (8 * (e & 3))) & 0xFFu;
}
// scale q + off, rounded once to f32, of the eight codes q in the bytes of
// (lo, hi) under mask (a code below 2^10 in each half word).  A code is
// not converted: as f16 bits it is the denormal q 2^-24, which v_fma_mix_f32
// takes as it is, and the scale carries the 2^24 (exactly) -- 3 instructions per
// 4 codes where v_cvt_f32_ubyte* takes one for each after the extraction
// (2.25 instead of 2.9 instructions per Q4_K weight in all).
constexpr float GM_DEN = 16777216.f;  // 2^24
static __device__ __forceinline__ void codes8(uint32_t lo, uint32_t hi, uint32_t mask, float scale, float off,
                                              float (&v)[8]) {
#pragma unroll
    for (int w = 0; w < 2; w++) {
        const uint32_t x = w ? hi : lo;
        const h2v a = __builtin_bit_cast(h2v, x & mask), b = __builtin_bit_cast(h2v, (x >> 8) & mask);
        v[4 * w] = __builtin_fmaf((float)a[0], scale, off);
        v[4 * w + 1] = __builtin_fmaf((float)b[0], scale, off);
        v[4 * w + 2] = __builtin_fmaf((float)a[1], scale, off);
        v[4 * w + 3] = __builtin_fmaf((float)b[1], scale, off);
    }
}

// ---- per-type staging and step dequantization ---------------------------------
// A chunk of one row is PL planes of four 16-byte pieces (one per 64-weight unit)
// and a 16-byte tail (scales; tail_of() the row's, one per chunk), plus for Q6_K an f16 d.
// A lane of operand half hf owns its row's units 2 hf and 2 hf + 1: raw() takes
// their bytes and scales for K half kh from LDS, deq(uu, i) makes the 8 weights of
// unit 2 hf + uu, step 4 kh + i the A operand; octet(u, st): the activation octet
// (8 consecutive K) that the weights of unit u, step st multiply.

// one workgroup's staged weights: piece (row, q) of a plane at slot 4 row + (q ^
// (row / 2) % 4), so 8 rows' pieces of one q fall into 8 different bank groups
struct GmW {
    u32x4 *pl;    // [PL][GM_THREADS]
    u32x4 *tail;  // [GM_ROWS]
    uint32_t *d;  // [GM_ROWS] (Q6_K)
};
static __device__ __forceinline__ int gm_slot(int row, int q) { return 4 * row + (q ^ ((row >> 1) & 3)); }

// Q4_K, chunk = super-block c; unit u of it: bytes 0-15 in plane 0, 16-31 in plane
// 1.  Step st = 4h + 2p + b: nibble h (group 2u + h), plane p, bytes 8b .. 8b+7 of
// that plane; weight = 64u + 32h + 16p + 8b + e, so the octet is 8u + st; K half
// kh: nibble kh.  ggml/quant.odin:178-209.
struct GQ4K {
    static constexpr int PL = 2, TMAX = 8;
    static constexpr bool D = false;
    static __device__ __forceinline__ const u32x4 *tail_of(const DMat &m, int row) {
        return (const u32x4 *)m.s + (size_t)row * (m.cols >> 8);
    }
    struct Raw {
        u32x4 p[2][2];  // [unit][plane]
        float d1[2], mm[2];
    };
    static __device__ __forceinline__ void raw(const GmW &w, int row, int hf, int kh, Raw &r) {
        const u32x4 h = w.tail[row];
        const float d = h2f(h.x & 0xFFFFu) * (kh ? GM_DEN / 16.f : GM_DEN), dmin = -h2f(h.x >> 16);
#pragma unroll
        for (int uu = 0; uu < 2; uu++) {
            const int s = gm_slot(row, 2 * hf + uu);
            r.p[uu][0] = w.pl[s];
            r.p[uu][1] = w.pl[GM_THREADS + s];
            // the unit's 24-bit field: sc(2u) | m(2u) << 6 | sc(2u+1) << 12 | m(2u+1) << 18
            const uint32_t f = __builtin_amdgcn_alignbit(hf ? (uu ? 0u : h.w) : h.z, hf ? (uu ? h.w : h.z) : h.y,
                                                         hf ? (uu ? 8 : 16) : (uu ? 24 : 0)) >> (12 * kh);
            r.d1[uu] = d * (float)(f & 63u);
            r.mm[uu] = dmin * (float)((f >> 6) & 63u);
        }
    }
    // d1 * nib is exact in f32 (at most 11 + 6 + 4 significant bits), so the
    // fused d1 * nib - mm rounds exactly as the separate product and difference;
    // the high nibbles stay where they are, 16 times their value
    static __device__ __forceinline__ h8 deq(const Raw &r, int uu, int i, int kh) {
        const u32x4 &w = r.p[uu][i >> 1];
        float v[8];
        codes8((i & 1) ? w.z : w.x, (i & 1) ? w.w : w.y, kh ? 0x00F000F0u : 0x000F000Fu, r.d1[uu], r.mm[uu], v);
        return cvt8(v);
    }
    static __device__ __forceinline__ int octet(int u, int st) { return 8 * u + st; }
};

// Q6_K, chunk = super-block c; unit u of it is unit u' = u % 2 of half h = u / 2,
// bytes 0-15 of its ql-low, ql-high and qh planes.  Step
// st = 2s + b: run s (ql-low/high nibble and qh bits 2s, scale 8h + u' + 2s),
// bytes 8b .. 8b+7; weight = 128h + 32s + 16u' + 8b + e, octet
// 16h + 4s + 2u' + b.  K half kh: runs 2 kh and 2 kh + 1.  ggml/quant.odin:212-247.
struct GQ6K {
    static constexpr int PL = 3, TMAX = 8;
    static constexpr bool D = true;
    static __device__ __forceinline__ const u32x4 *tail_of(const DMat &m, int row) {
        return (const u32x4 *)m.s + (size_t)row * (m.cols >> 8);
    }
    struct Raw {
        u32x4 l[2][2], h[2];  // [unit][ql-low, ql-high]; qh
        float ds[2][2], off[2][2];  // [unit][run - 2 kh]
    };
    static __device__ __forceinline__ void raw(const GmW &w, int row, int hf, int kh, Raw &r) {
        // unit 2 hf + u' is unit u' of half hf; scales 8 hf + u' + 2s of runs s = 2 kh,
        // 2 kh + 1: bytes u' and u' + 2 of one word
        const uint32_t sw = ((const uint32_t *)(w.tail + row))[2 * hf + kh];
        const float d = h2f(w.d[row]);
#pragma unroll
        for (int uu = 0; uu < 2; uu++) {
            const int s = gm_slot(row, 2 * hf + uu);
            r.l[uu][0] = w.pl[s];
            r.l[uu][1] = w.pl[GM_THREADS + s];
            r.h[uu] = w.pl[2 * GM_THREADS + s];
#pragma unroll
            for (int j = 0; j < 2; j++) {
                const float ds = d * (float)(int8_t)((sw >> (8 * uu + 16 * j)) & 0xFFu);
                r.ds[uu][j] = ds * GM_DEN;
                r.off[uu][j] = -32.f * ds;
            }
        }
    }
    // ds * (code - 32) as one fused ds * code - 32 ds: the exact value is the
    // same and the fma rounds it once, as the reference's single product
    static __device__ __forceinline__ h8 deq(const Raw &r, int uu, int i, int kh) {
        const int j = i >> 1, b = i & 1;
        const u32x4 &l = r.l[uu][j], &h = r.h[uu];
        const uint32_t llo = ((b ? l.z : l.x) >> (4 * kh)) & 0x0F0F0F0Fu;
        const uint32_t lhi = ((b ? l.w : l.y) >> (4 * kh)) & 0x0F0F0F0Fu;
        const uint32_t hlo = (((b ? h.z : h.x) >> (4 * kh + 2 * j)) & 0x03030303u) << 4;
        const uint32_t hhi = (((b ? h.w : h.y) >> (4 * kh + 2 * j)) & 0x03030303u) << 4;
        float v[8];
        codes8(llo | hlo, lhi | hhi, 0x00FF00FFu, r.ds[uu][j], r.off[uu][j], v);  // 6-bit codes, one per byte
        return cvt8(v);
    }
    static __device__ __forceinline__ int octet(int u, int st) {
        return 16 * (u >> 1) + 4 * (st >> 1) + 2 * (u & 1) + (st & 1);
    }
};

// Q8_0, chunk = blocks 8c .. 8c+7; unit u of it: blocks 8c + 2u and 8c + 2u + 1;
// plane 2 blk + half holds bytes 16 half .. +15 of block blk.  Step st = 4 blk + 2
// half + b: weight 64u + 8st + e, octet 8u + st; K half kh: block kh of the unit.  (Four planes
// and the scales beside 128 tokens would be 2 KB more than the LDS: TMAX 6, 96
// tokens.)  ggml/quant.odin:87-96.
struct GQ80 {
    static constexpr int PL = 4, TMAX = 6;
    static constexpr bool D = false;
    static __device__ __forceinline__ const u32x4 *tail_of(const DMat &m, int row) {  // eight block scales per chunk
        return (const u32x4 *)m.d + (size_t)row * (m.cols >> 8);
    }
    struct Raw {
        u32x4 p[2][2];  // [unit][half of block kh]
        float d[2];
    };
    static __device__ __forceinline__ void raw(const GmW &w, int row, int hf, int kh, Raw &r) {
#pragma unroll
        for (int uu = 0; uu < 2; uu++) {
            const int s = gm_slot(row, 2 * hf + uu);
            r.p[uu][0] = w.pl[2 * kh * GM_THREADS + s];
            r.p[uu][1] = w.pl[(2 * kh + 1) * GM_THREADS + s];
            r.d[uu] = h2f((((const uint32_t *)(w.tail + row))[2 * hf + uu] >> (16 * kh)) & 0xFFFFu);
        }
    }
    static __device__ __forceinline__ h8 deq(const Raw &r, int uu, int i, int) {
#pragma clang fp contract(off)
        const u32x4 &w = r.p[uu][i >> 1];
        const uint32_t lo = (i & 1) ? w.z : w.x, hi = (i & 1) ? w.w : w.y;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = r.d[uu] * (float)(int8_t)byte_of(lo, hi, e);
        return cvt8(v);
    }
    static __device__ __forceinline__ int octet(int u, int st) { return 8 * u + st; }
};

template <class G>
static constexpr size_t gm_lds(int tt) {
    return (size_t)2 * 16 * tt * (GM_KC / 8) * 16 + (size_t)G::PL * GM_THREADS * 16 + GM_ROWS * 16 + (G::D ? GM_ROWS * 4 : 0);
}

// One workgroup: 128 rows (NP == 2: 64 rows of each matrix), 16 TT tokens, a
// slice of cps chunks of K.  Chunk c + 1 is loaded into registers while chunk c
// is computed and stored to LDS when chunk c's weights have been taken out of
// it: activations double-buffered (piece (token j, octet o) at slot TOK o + (j ^
// (o % 8)): conflict-free stores of 8 consecutive octets and conflict-free
// 16-lane operand reads), weights in one buffer that every wave copies its
// operand bytes from first.  With more than one K slice (split > 1) slice z
// writes its partial products to c + z n M; the consumer sums them in slice
// order.
//
// NP == 2 (gate and up of the FFN, one K slice): the operand's rows 0-15 are the
// gate matrix's, 16-31 the up matrix's same rows, and the epilogue writes the f16
// SwiGLU of the pair (infer/forward.odin:128-132: v *= 1/(1+exp(-v)); v *= up;
// then the half staging of the next projection's input).
//
// Consecutive blocks go to different XCDs; the block index is turned so that
// each XCD takes a contiguous range of (slice, row tile, token tile), the token
// tiles of one row tile together: its L2 reads those weights once.
template <class G, int NP, int TT>
__global__ __launch_bounds__(GM_THREADS) void gemm_q_kernel(GemmArgs a) {
    constexpr int TOK = 16 * TT, TH = TT / 2, XV = TOK * GM_KC / 8, XPT = XV / GM_THREADS, PL = G::PL;
    extern __shared__ __attribute__((aligned(16))) u32x4 gm_smem[];
    u32x4 *xs = gm_smem;  // [2][XV]
    GmW ws;
    ws.pl = gm_smem + 2 * XV;
    ws.tail = ws.pl + PL * GM_THREADS;
    ws.d = (uint32_t *)(ws.tail + GM_ROWS);
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), hf = lane >> 5, li = lane & 31;
    const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE), rg = wave >> 1, kh = wave & 1;
    // the block's projection, row tile, token tile and K slice
    int b = (int)blockIdx.x;
    {
        const int nb = (int)gridDim.x, per = nb >> 3, rem = nb & 7, xcd = b & 7;
        b = xcd * per + min(xcd, rem) + (b >> 3);
    }
    int sg = 0;
#pragma unroll
    for (int i = 1; i < GM_MAX_SEG; i++)
        if (i < a.nseg && b >= a.seg[i].first) sg = i;
    const GemmSeg &g = a.seg[sg];
    const DMat &mat = g.m;
    const int ny = (a.n + TOK - 1) / TOK, loc = b - g.first, bz = loc / (g.nx * ny);
    const int bx = (loc - bz * g.nx * ny) / ny, t0 = (loc - (bz * g.nx + bx) * ny) * TOK;
    const int M = mat.rows, K = mat.cols, nchunk = K / GM_KC;
    const int c0 = bz * g.cps, c1 = min(nchunk, c0 + g.cps);

    // local row lr = 32 rg + i: matrix row (rows past M: read, not stored)
    auto row_of = [&](int lr) {
        return min(NP == 2 ? bx * (GM_ROWS / 2) + (lr >> 5) * 16 + (lr & 15) : bx * GM_ROWS + lr, M - 1);
    };
    // staging loads: piece tid % 4 of local row tid / 4 per plane, the tail of row tid
    const size_t pbytes = (size_t)PL * mat.plane;
    // (two matrices: the wave's pieces are of one of them)
    const bool tsecond = NP == 2 && (tid & 16);
    const uint32_t woff = (uint32_t)((row_of(tid >> 2) * (K >> 6) + (tid & 3)) * 16);
    const int trow = row_of(tid & (GM_ROWS - 1));
    const rsrc_t wsrc = make_rsrc(NP == 2 && (wave & 1) ? a.m2.q : mat.q, pbytes);
    const u32x4 *tsrc = G::tail_of(tsecond ? a.m2 : mat, trow);
    const uint16_t *dsrc = (tsecond ? a.m2.d : mat.d) + (size_t)trow * (K >> 8);
    const rsrc_t xsrc = make_rsrc(a.x, (size_t)a.n * K * 2);
    uint32_t xoff[XPT];
#pragma unroll
    for (int i = 0; i < XPT; i++) {
        const int p = tid + i * GM_THREADS;
        xoff[i] = (uint32_t)(min(t0 + (p >> 5), a.n - 1) * K * 2 + 16 * (p & 31));
    }
    // a chunk on its way from memory to LDS, in registers
    struct Stage {
        u32x4 x[XPT], w[PL], t;
        uint32_t d;
    };
    auto wfetch = [&](int c, Stage &r) {
#pragma unroll
        for (int k = 0; k < PL; k++) r.w[k] = bld16(wsrc, woff + (uint32_t)(k * mat.plane), 64 * c);
        if (tid < GM_ROWS) {
            r.t = tsrc[c];
            if constexpr (G::D) r.d = dsrc[c];
        }
    };
    auto wstore = [&](const Stage &r) {
#pragma unroll
        for (int k = 0; k < PL; k++) ws.pl[k * GM_THREADS + gm_slot(tid >> 2, tid & 3)] = r.w[k];
        if (tid < GM_ROWS) {
            ws.tail[tid] = r.t;
            if constexpr (G::D) ws.d[tid] = r.d;
        }
    };
    auto xfetch = [&](int c, int i, Stage &r) { r.x[i] = bld16(xsrc, xoff[i], c * GM_KC * 2); };
    u32x4 *const xput = xs + (tid & 31) * TOK + ((tid >> 5) ^ (tid & 7));  // piece tid's slot; piece tid + 512 i's: 16 i on
    auto xstore = [&](int buf, int i, const Stage &r) { xput[buf * XV + 16 * i] = r.x[i]; };
    Stage next;

    f32x16v acc[TH];
#pragma unroll
    for (int t = 0; t < TH; t++)
#pragma unroll
        for (int e = 0; e < 16; e++) acc[t][e] = 0.f;
    // Software pipeline over the K half's eight 16-wide K steps: a step's products
    // run beside the next step's operand reads and dequantization and a part of the
    // next chunk's staging (issued together ahead of the products, the staging
    // alone held the waves up for longer than the products take).  Barrier Q (step
    // 2): every wave has taken chunk c's weights out of LDS and is done with chunk
    // c - 1's activations, so chunk c + 1 may be stored over them.  Barrier P
    // (step 6): chunk c + 1 is staged; steps 6 and 7 read ahead into it.
    constexpr int XQ = (XPT + 3) / 4;  // X pieces staged in each of steps 2 - 5
    typename G::Raw raw;
    h8 A[2], B[2][TH];
    auto readx = [&](int buf, int s, h8 (&d)[TH]) {
        const int o = G::octet(2 * hf + (s >> 2), 4 * kh + (s & 3));
        const u32x4 *xp = xs + buf * XV + o * TOK + (li ^ (o & 7));
#pragma unroll
        for (int t = 0; t < TH; t++) d[t] = __builtin_bit_cast(h8, xp[32 * t]);
    };
    if (c0 < c1) {
        // the first two chunks are requested together (the second after the first
        // had arrived, every workgroup waited for memory twice)
        Stage first;
        const int cs = min(c0 + 1, c1 - 1);
        wfetch(c0, first);
#pragma unroll
        for (int i = 0; i < XPT; i++) xfetch(c0, i, first);
        wfetch(cs, next);
#pragma unroll
        for (int i = 0; i < XPT; i++) xfetch(cs, i, next);
        wstore(first);
#pragma unroll
        for (int i = 0; i < XPT; i++) xstore(0, i, first);
        __syncthreads();
        G::raw(ws, 32 * rg + li, hf, kh, raw);
        readx(0, 0, B[0]);
        A[0] = G::deq(raw, 0, 0, kh);
    }
    for (int c = c0; c < c1; c++) {
        const int buf = (c - c0) & 1, cn = min(c + 2, c1 - 1);
#pragma unroll
        for (int s = 0; s < 8; s++) {
            const int cur = s & 1, nxt = cur ^ 1, sn = (s + 1) & 7;
            if (s == 2) {
                __syncthreads();  // Q
                wstore(next);
                wfetch(cn, next);
            }
            if (s == 6) __syncthreads();  // P
            if (s == 7) G::raw(ws, 32 * rg + li, hf, kh, raw);  // (past the last chunk: that chunk again, unused)
            readx(s == 7 ? buf ^ 1 : buf, sn, B[nxt]);
            if (s >= 2 && s < 6) {
#pragma unroll
                for (int j = XQ * (s - 2); j < XQ * (s - 1) && j < XPT; j++) {
                    xstore(buf ^ 1, j, next);
                    xfetch(cn, j, next);
                }
            }
            A[nxt] = G::deq(raw, sn >> 2, sn & 3, kh);
#pragma unroll
            for (int t = 0; t < TH; t++)
                acc[t] = __builtin_amdgcn_mfma_f32_32x32x16_f16(A[cur], B[cur][t], acc[t], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // the two K halves through LDS ([kh][token][row], the row's 16-byte pieces
    // turned by the token against bank conflicts), then coalesced stores of
    // their sums: lane (j, h) of tile t holds rows 8 g + 4 h .. +3 of token j in
    // floats 4 g .. 4 g + 3
    __syncthreads();
    f32x4v *yo = (f32x4v *)gm_smem;  // [2][TOK][32]
#pragma unroll
    for (int t = 0; t < TH; t++)
#pragma unroll
        for (int g = 0; g < 4; g++) {
            const int tk = 32 * t + li;
            yo[(kh * TOK + tk) * 32 + ((8 * rg + 2 * g + hf) ^ (tk & 7))] =
                f32x4v{acc[t][4 * g], acc[t][4 * g + 1], acc[t][4 * g + 2], acc[t][4 * g + 3]};
        }
    __syncthreads();
    auto sum = [&](int tk, int col) {
        const int i = tk * 32 + (col ^ (tk & 7));
        return yo[i] + yo[TOK * 32 + i];
    };
    if constexpr (NP == 2) {
#pragma unroll
        for (int i = 0; i < TOK * 16 / GM_THREADS; i++) {
            const int p = tid + i * GM_THREADS, tk = p >> 4, cc = p & 15;  // row piece 4 cc of the 64 rows
            if (t0 + tk >= a.n) continue;
            const f32x4v gv = sum(tk, 8 * (cc >> 2) + (cc & 3)), uv = sum(tk, 8 * (cc >> 2) + 4 + (cc & 3));
            uint16_t hv[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
#pragma clang fp contract(off)
                float v = gv[e];
                v *= 1.0f / (1.0f + expf(-v));
                v *= uv[e];
                hv[e] = f2h(v);
            }
            const int r0 = bx * (GM_ROWS / 2) + 4 * cc;
            uint16_t *dst = a.h + (size_t)(t0 + tk) * M + r0;
            if (r0 + 3 < M && (M & 3) == 0) {
                *(u32x2 *)dst = u32x2{(uint32_t)hv[0] | ((uint32_t)hv[1] << 16), (uint32_t)hv[2] | ((uint32_t)hv[3] << 16)};
                continue;
            }
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (r0 + e < M) dst[e] = hv[e];
        }
    } else {
        float *out = g.c + (size_t)bz * a.n * M;
        if (M & 3) {  // rows of C not 16-byte aligned: one float per lane, side by side
            const float *yf = (const float *)yo;
            const int row = tid & (GM_ROWS - 1), r0 = bx * GM_ROWS + row;
#pragma unroll 8
            for (int tk = tid / GM_ROWS; tk < TOK; tk += GM_THREADS / GM_ROWS) {
                const int k = 4 * (tk * 32 + ((row >> 2) ^ (tk & 7))) + (row & 3);
                if (t0 + tk < a.n && r0 < M) out[(size_t)(t0 + tk) * M + r0] = yf[k] + yf[4 * TOK * 32 + k];
            }
            return;
        }
#pragma unroll
        for (int i = 0; i < XPT; i++) {
            const int p = tid + i * GM_THREADS, tk = p >> 5, cc = p & 31;
            if (t0 + tk >= a.n) continue;
            const int r0 = bx * GM_ROWS + 4 * cc;
            if (r0 < M) *(f32x4v *)(out + (size_t)(t0 + tk) * M + r0) = sum(tk, cc);
        }
    }
}

// ---- 16-row waves ---------------------------------------------------------------
// gemm_r_kernel: 128 rows x 64 tokens, wave w rows 16w .. 16w+15 of every chunk in
// four v_mfma_f32_16x16x32_f16 accumulators (A[i][k]: i = l % 16, k = 8 (l / 16) + e;
// D[i][j]: j = l % 16, i = 4 (l / 16) + e).  The weights go from memory straight into
// the operand layout, one chunk ahead in registers: lane quarter q holds unit 4c + q
// of its row, and the chunk's eight 32-wide K steps take 8 of its weights each.  Only
// the activations are staged, so the first product waits for less, nothing is summed
// at the end, and two workgroups fit a CU; against that every chunk takes longer
// (the loads' address work, twice the matrix instructions).  The codes are converted
// by v_cvt_f32_ubyte{0..3} here: codes8 measured 3 - 5% slower (4069 x 2816 Q6_K, 79
// tokens: 14.3 us against 13.8).
// keeps a masked word opaque, so that its bytes convert with v_cvt_f32_ubyte{0..3}
// instead of being re-extracted one by one from the unmasked word
static __device__ __forceinline__ uint32_t opaque(uint32_t v) {
    asm volatile("" : "+v"(v));
    return v;
}
struct RQ4K {  // step st = 4h + 2p + b: nibble h, plane p, bytes 8b .. 8b+7; octet 8q + st
    struct Src {
        rsrc_t q, s;
        uint32_t plane, qo, so;
    };
    struct Raw {
        u32x4 p[2], hdr;
    };
    struct Pre {
        float d1[2], mm[2];
    };
    static __device__ __forceinline__ Src src(const DMat &m, int row, int q) {
        return Src{make_rsrc(m.q, 2 * m.plane), make_rsrc(m.s, (size_t)m.rows * (m.cols >> 8) * 16), (uint32_t)m.plane,
                   (uint32_t)((row * (m.cols >> 6) + q) * 16), (uint32_t)(row * (m.cols >> 8) * 16)};
    }
    static __device__ __forceinline__ void raw(const Src &g, int c, Raw &r) {
        r.p[0] = bld16(g.q, g.qo, 64 * c);
        r.p[1] = bld16(g.q, g.qo + g.plane, 64 * c);
        r.hdr = bld16(g.s, g.so, 16 * c);
    }
    static __device__ __forceinline__ Pre pre(const Raw &r, int q) {
        const float d = h2f(r.hdr.x & 0xFFFFu), dmin = h2f(r.hdr.x >> 16);
        uint32_t sc0, m0, sc1, m1;
        q4k_scales(q, r.hdr.y, r.hdr.z, r.hdr.w, sc0, m0, sc1, m1);
        return Pre{{d * (float)sc0, d * (float)sc1}, {dmin * (float)m0, dmin * (float)m1}};
    }
    static __device__ __forceinline__ h8 deq(const Raw &r, const Pre &p, int st) {
        const int h = st >> 2, b = st & 1;
        const u32x4 &w = r.p[(st >> 1) & 1];
        const uint32_t lo = opaque(((b ? w.z : w.x) >> (4 * h)) & 0x0F0F0F0Fu);
        const uint32_t hi = opaque(((b ? w.w : w.y) >> (4 * h)) & 0x0F0F0F0Fu);
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = __builtin_fmaf(p.d1[h], (float)byte_of(lo, hi, e), -p.mm[h]);
        return cvt8(v);
    }
};
struct RQ6K {  // step st = 2s + b: run s, bytes 8b .. 8b+7; octet 16 (q / 2) + 4s + 2 (q % 2) + b
    struct Src {
        rsrc_t q, s, d;
        uint32_t plane, qo, so, dof;
    };
    struct Raw {
        u32x4 l[2], h;
        u32x2 sc;
        uint32_t d;
    };
    struct Pre {
        float ds[4], off[4];
    };
    static __device__ __forceinline__ Src src(const DMat &m, int row, int q) {
        const int nsb = m.cols >> 8;
        return Src{make_rsrc(m.q, 3 * m.plane), make_rsrc(m.s, (size_t)m.rows * nsb * 16),
                   make_rsrc(m.d, (size_t)m.rows * nsb * 2), (uint32_t)m.plane, (uint32_t)((row * (m.cols >> 6) + q) * 16),
                   (uint32_t)(row * nsb * 16 + 8 * (q >> 1)), (uint32_t)(row * nsb * 2)};
    }
    static __device__ __forceinline__ void raw(const Src &g, int c, Raw &r) {
        r.l[0] = bld16(g.q, g.qo, 64 * c);
        r.l[1] = bld16(g.q, g.qo + g.plane, 64 * c);
        r.h = bld16(g.q, g.qo + 2 * g.plane, 64 * c);
        r.sc = __builtin_bit_cast(u32x2, __builtin_amdgcn_raw_buffer_load_b64(g.s, g.so, 16 * c, 0));
        r.d = __builtin_amdgcn_raw_buffer_load_b16(g.d, g.dof, 2 * c, 0);
    }
    static __device__ __forceinline__ Pre pre(const Raw &r, int q) {
        Pre p;
        const float d = h2f(r.d);
#pragma unroll
        for (int s = 0; s < 4; s++) {
            p.ds[s] = d * (float)(int8_t)byte_of(r.sc.x, r.sc.y, (q & 1) + 2 * s);
            p.off[s] = -32.f * p.ds[s];
        }
        return p;
    }
    static __device__ __forceinline__ h8 deq(const Raw &r, const Pre &p, int st) {
        const int s = st >> 1, b = st & 1;
        const u32x4 &l = r.l[s & 1];
        const uint32_t llo = ((b ? l.z : l.x) >> (4 * (s >> 1))) & 0x0F0F0F0Fu;
        const uint32_t lhi = ((b ? l.w : l.y) >> (4 * (s >> 1))) & 0x0F0F0F0Fu;
        const uint32_t hlo = (((b ? r.h.z : r.h.x) >> (2 * s)) & 0x03030303u) << 4;
        const uint32_t hhi = (((b ? r.h.w : r.h.y) >> (2 * s)) & 0x03030303u) << 4;
        const uint32_t wlo = opaque(llo | hlo), whi = opaque(lhi | hhi);  // 6-bit codes, one per byte
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = __builtin_fmaf(p.ds[s], (float)byte_of(wlo, whi, e), p.off[s]);
        return cvt8(v);
    }
};
struct RQ80 {  // step st = 4 blk + 2 half + b: octet 8q + st
    struct Src {
        rsrc_t q, d;
        uint32_t plane, qo, dof;
    };
    struct Raw {
        u32x4 p[4];
        uint32_t d;
    };
    struct Pre {
        float d[2];
    };
    static __device__ __forceinline__ Src src(const DMat &m, int row, int q) {
        return Src{make_rsrc(m.q, 4 * m.plane), make_rsrc(m.d, (size_t)m.rows * (m.cols >> 5) * 2), (uint32_t)m.plane,
                   (uint32_t)((row * (m.cols >> 6) + q) * 16), (uint32_t)((row * (m.cols >> 5) + 2 * q) * 2)};
    }
    static __device__ __forceinline__ void raw(const Src &g, int c, Raw &r) {
#pragma unroll
        for (int k = 0; k < 4; k++) r.p[k] = bld16(g.q, g.qo + k * g.plane, 64 * c);
        r.d = __builtin_amdgcn_raw_buffer_load_b32(g.d, g.dof, 16 * c, 0);
    }
    static __device__ __forceinline__ Pre pre(const Raw &r, int) { return Pre{{h2f(r.d & 0xFFFFu), h2f(r.d >> 16)}}; }
    static __device__ __forceinline__ h8 deq(const Raw &r, const Pre &p, int st) {
#pragma clang fp contract(off)
        const u32x4 &w = r.p[st >> 1];
        const uint32_t lo = (st & 1) ? w.z : w.x, hi = (st & 1) ? w.w : w.y;
        float v[8];
#pragma unroll
        for (int e = 0; e < 8; e++) v[e] = p.d[st >> 2] * (float)(int8_t)byte_of(lo, hi, e);
        return cvt8(v);
    }
};

template <class G, class R>
__global__ __launch_bounds__(GM_THREADS) void gemm_r_kernel(GemmArgs a) {
    constexpr int TOK = 64, XV = TOK * GM_KC / 8, XPT = XV / GM_THREADS;
    __shared__ __attribute__((aligned(16))) u32x4 xs[2][XV];  // as gemm_q_kernel's
    const int tid = threadIdx.x, lane = tid & (WAVE - 1), wave = tid / WAVE, q = lane >> 4, li = lane & 15;
    // one projection: grid (row tiles, token tiles, K slices), else flat
    int sg = 0, bx = (int)blockIdx.x, by = (int)blockIdx.y, bz = (int)blockIdx.z;
    if (a.nseg > 1) {
#pragma unroll
        for (int i = 1; i < GM_MAX_SEG; i++)
            if (i < a.nseg && bx >= a.seg[i].first) sg = i;
        const int nx = a.seg[sg].nx, ny = (a.n + TOK - 1) / TOK, loc = bx - a.seg[sg].first;
        bz = loc / (nx * ny);
        by = (loc - bz * nx * ny) / nx;
        bx = loc - (bz * ny + by) * nx;
    }
    const GemmSeg &g = a.seg[sg];
    const DMat &mat = g.m;
    const int t0 = by * TOK;
    const int M = mat.rows, K = mat.cols, c0 = bz * g.cps, c1 = min(K / GM_KC, c0 + g.cps);
    const typename R::Src src = R::src(mat, min(bx * GM_ROWS + 16 * wave + li, M - 1), q);  // rows past M: not stored

    const rsrc_t xsrc = make_rsrc(a.x, (size_t)a.n * K * 2);
    uint32_t xoff[XPT];
#pragma unroll
    for (int i = 0; i < XPT; i++) {
        const int p = tid + i * GM_THREADS;
        xoff[i] = (uint32_t)(min(t0 + (p >> 5), a.n - 1) * K * 2 + 16 * (p & 31));
    }
    u32x4 xr[XPT];
    auto xfetch = [&](int c) {
#pragma unroll
        for (int i = 0; i < XPT; i++) xr[i] = bld16(xsrc, xoff[i], c * GM_KC * 2);
    };
    f32x4v acc[4];
#pragma unroll
    for (int t = 0; t < 4; t++) acc[t] = f32x4v{0.f, 0.f, 0.f, 0.f};
    typename R::Raw ring[2];
    if (c0 < c1) {
        R::raw(src, c0, ring[0]);
        xfetch(c0);
    }
    for (int cb = c0; cb < c1; cb += 2) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const int c = cb + r;
            if (c >= c1) break;
            R::raw(src, c + 1 < c1 ? c + 1 : c0, ring[r ^ 1]);  // (past the slice: its first chunk, unused)
#pragma unroll
            for (int i = 0; i < XPT; i++) {
                const int p = tid + i * GM_THREADS, j = p >> 5, o = p & 31;
                xs[r][o * TOK + (j ^ (o & 7))] = xr[i];
            }
            if (c + 1 < c1) xfetch(c + 1);
            __syncthreads();  // chunk c staged; every wave is done with chunk c - 2's buffer
            const typename R::Pre pre = R::pre(ring[r], q);
#pragma unroll
            for (int st = 0; st < 8; st++) {
                const int o = G::octet(q, st);
                h8 B[4];
#pragma unroll
                for (int t = 0; t < 4; t++) B[t] = __builtin_bit_cast(h8, xs[r][o * TOK + ((16 * t + li) ^ (o & 7))]);
                const h8 A = R::deq(ring[r], pre, st);
#pragma unroll
                for (int t = 0; t < 4; t++) acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_f16(A, B[t], acc[t], 0, 0, 0);
            }
        }
    }
    // lane (j, q) of tile t holds rows 4q .. 4q+3 of token 16t + j
    const int r0 = bx * GM_ROWS + 16 * wave + 4 * q;
#pragma unroll
    for (int t = 0; t < 4; t++) {
        const int tk = t0 + 16 * t + li;
        if (tk >= a.n) continue;
        float *dst = g.c + ((size_t)bz * a.n + tk) * M + r0;
        if (r0 + 3 < M && (M & 3) == 0) {
            *(f32x4v *)dst = acc[t];
            continue;
        }
#pragma unroll
        for (int e = 0; e < 4; e++)
            if (r0 + e < M) dst[e] = acc[t][e];
    }
}

// c[i] = sum over slices z (in order) of part[z][i]; NB slices' loads are in
// flight together (a loop of load and add waits for each in turn)
template <int NB>
__global__ __launch_bounds__(WG) void gemm_reduce(const float *part, float *c, int64_t total, int split) {
    const int64_t i = (int64_t)blockIdx.x * WG + threadIdx.x;
    if (4 * i + 3 < total) {
        f32x4v s = {0.f, 0.f, 0.f, 0.f};
        for (int z0 = 0; z0 < split; z0 += NB) {
            f32x4v v[NB];
#pragma unroll
            for (int k = 0; k < NB; k++) v[k] = *(const f32x4v *)(part + min(z0 + k, split - 1) * total + 4 * i);
#pragma unroll
            for (int k = 0; k < NB; k++)
                if (z0 + k < split) s = z0 + k ? s + v[k] : v[k];
        }
        *(f32x4v *)(c + 4 * i) = s;
    } else {
        for (int64_t k = 4 * i; k < total; k++) {
            float s = part[k];
            for (int z = 1; z < split; z++) s += part[z * total + k];
            c[k] = s;
        }
    }
}

bool gemm_supported(const DMat &m) {
    return (m.type == T_Q4_K || m.type == T_Q6_K || m.type == T_Q8_0) && m.cols % GM_KC == 0;
}

// Kernel, token tiles (of 16) per workgroup and K split of a launch of `rt` row tiles:
// those of least estimated time with at most `cap` slices.  The estimate (us) has a
// CU's workgroups one after another (two of 32 tokens fit a CU, and take twice as
// long; a second one of gemm_r_kernel's adds 0.8 of the first): a chunk and a fixed
// time per workgroup, every slice written and read back, and the reduction's launch
// if the caller has one.  Its constants are fitted to 210 shapes (500 - 12288 rows,
// 1024 - 12288 columns, 8 - 512 tokens, the three types) run with every kernel and
// tile at two or three splits, on three sets of inputs in turn: the choice takes 1.8%
// (Q4_K), 1.4% (Q6_K) and 1.7% (Q8_0) longer than the fastest one on average.
// gemm_r_kernel wins where up to 64 tokens fill 150 workgroups or more (the weights'
// stream bounds it: 4096 x 4096 Q4_K, 64 tokens: 11.8 us against 12.5), and where whole
// tiles of 64 tokens fill every CU once with few chunks, or once and a half with many.
// Without it 37 of the shapes took over 2% longer than with it alone (up to 15%, for
// 8% less on average); now 5 do, up to 6% in all but one.  With the tile taken from n
// alone (32 tokens up to 32, 64 or 128 above) it was up to 41%: few rows or columns
// want more and smaller tiles at any n (3095 x 1024 Q4_K, 157 tokens: 9.1 us at 32
// tokens a tile, 10.6 at 64).  Tiles of 96 tokens are worth 3.5% on average for Q8_0,
// which has no larger one, and 0.7% for the others.
struct GemmPlan {
    int tt, split;
    bool r16;  // gemm_r_kernel (tt 4)
};
static GemmPlan gemm_plan(int type, int rt, int nchunk, int32_t n, double out, int cap, bool reduce, bool pair = false) {
    const char *only = std::getenv("OI_GEMM_TILE");  // 32, 64, 96, 128 tokens or "r16": that kernel alone (tests)
    const double unit = type == T_Q4_K ? 0.9 : 1.0;  // (the fewest instructions per weight)
    struct Tile {
        int tt, tiles;
        bool r16;
        double chunk, fixed;
    } tile[5];
    int nt = 0;
    auto add = [&](int tt, bool r16, double chunk, double fixed) {
        if (only && ((std::strcmp(only, "r16") == 0) != r16 || (!r16 && std::atoi(only) != 16 * tt))) return;
        tile[nt++] = Tile{tt, rt * ((n + 16 * tt - 1) / (16 * tt)), r16, unit * chunk, fixed};
    };
    add(2, false, 1.35, 2.2);
    add(4, false, 1.65, 2.9);
    add(6, false, 1.78, 4.5);
    if (type != T_Q8_0) add(8, false, 1.9, 6.3);
    if (!pair) add(4, true, n <= 64 ? 1.6 : 1.7, n <= 64 ? 1.2 : 2.7);  // (gemm_r_kernel takes one matrix)
    GemmPlan best{2, 1, false};
    double bt = 1e30;
    const int smax = std::max(1, std::min(nchunk / 2, cap));
    for (int cps = (nchunk + smax - 1) / smax; cps <= nchunk; cps++) {  // chunks per slice
        const int s = (nchunk + cps - 1) / cps;
        if ((nchunk + s - 1) / s != cps) continue;  // as many slices of fewer chunks
        const double tail = s > 1 ? s * out * 1.4e-6 + (reduce ? 3.3 : 0.0) : 0.0;
        for (int i = 0; i < nt; i++) {
            const int wgs = tile[i].tiles * s, rest = wgs % 512;
            const double per = tile[i].r16 ? wgs / 512 * 1.8 + (rest > 256 ? 1.8 : rest ? 1.0 : 0.0) : (wgs + 255) / 256;
            const double t = per * (cps * tile[i].chunk + tile[i].fixed) + tail;
            if (t < bt) {
                bt = t;
                best = GemmPlan{tile[i].tt, s, tile[i].r16};
            }
        }
    }
    return best;
}
static int gemm_rt(const DMat &m, int rows = GM_ROWS) { return (m.rows + rows - 1) / rows; }
static int gemm_cap(const DMat &m, int32_t n, size_t part_bytes) {
    return (int)std::max<size_t>(1, std::min<size_t>(64, part_bytes / ((size_t)n * m.rows * 4)));
}
static GemmPlan gemm_plan(const DMat &m, int32_t n, size_t part_bytes) {
    return gemm_plan(m.type, gemm_rt(m), m.cols / GM_KC, n, (double)n * m.rows, gemm_cap(m, n, part_bytes), true);
}

int gemm_split(const DMat &m, int32_t n, size_t part_bytes) { return gemm_plan(m, n, part_bytes).split; }

template <class G, class R, int NP>
static hipError_t gemm_launch_t(const GemmArgs &a, int blocks, const GemmPlan &p, hipStream_t st) {
    const dim3 grid((unsigned)blocks), block(GM_THREADS);
    if constexpr (NP == 1) {
        if (p.r16) {
            const dim3 one((unsigned)a.seg[0].nx, (unsigned)((a.n + 63) / 64), (unsigned)p.split);
            hipLaunchKernelGGL((gemm_r_kernel<G, R>), a.nseg > 1 ? grid : one, block, 0, st, a);
            return hipGetLastError();
        }
    }
    switch (p.tt) {
    case 2: hipLaunchKernelGGL((gemm_q_kernel<G, NP, 2>), grid, block, gm_lds<G>(2), st, a); break;
    case 4: hipLaunchKernelGGL((gemm_q_kernel<G, NP, 4>), grid, block, gm_lds<G>(4), st, a); break;
    case 6: hipLaunchKernelGGL((gemm_q_kernel<G, NP, 6>), grid, block, gm_lds<G>(6), st, a); break;
    default:
        if constexpr (G::TMAX >= 8) hipLaunchKernelGGL((gemm_q_kernel<G, NP, 8>), grid, block, gm_lds<G>(8), st, a);
        else return hipErrorInvalidValue;
        break;
    }
    return hipGetLastError();
}
template <int NP>
static hipError_t gemm_launch(const GemmArgs &a, int blocks, const GemmPlan &p, hipStream_t st) {
    switch (a.seg[0].m.type) {
    case T_Q4_K: return gemm_launch_t<GQ4K, RQ4K, NP>(a, blocks, p, st);
    case T_Q6_K: return gemm_launch_t<GQ6K, RQ6K, NP>(a, blocks, p, st);
    default: return gemm_launch_t<GQ80, RQ80, NP>(a, blocks, p, st);
    }
}
// appends one projection's blocks to the launch
static void gemm_seg(GemmArgs &a, const DMat &m, float *c, const GemmPlan &p, int rows_per_tile, int &blocks) {
    const int nchunk = m.cols / GM_KC, nx = gemm_rt(m, rows_per_tile);
    a.seg[a.nseg++] = GemmSeg{m, c, (nchunk + p.split - 1) / p.split, nx, blocks};
    blocks += nx * ((a.n + 16 * p.tt - 1) / (16 * p.tt)) * p.split;
}

// With split > 1 the slices' partial products go to `part` (split * n * rows
// floats) and gemm_reduce sums them into c.
hipError_t launch_gemm(const DMat &m, const uint16_t *x, int32_t n, float *c, float *part, size_t part_bytes,
                       hipStream_t st) {
    if (!gemm_supported(m) || n <= 0) return hipErrorInvalidValue;
    const GemmPlan p = gemm_plan(m, n, part ? part_bytes : 0);
    const int split = p.split;
    GemmArgs a{};
    a.x = x;
    a.n = n;
    int blocks = 0;
    gemm_seg(a, m, split > 1 ? part : c, p, GM_ROWS, blocks);
    const hipError_t r = gemm_launch<1>(a, blocks, p, st);
    if (r != hipSuccess) return r;
    if (split > 1) {
        const int64_t total = (int64_t)n * m.rows;
        const int64_t nb = ((total + 3) / 4 + WG - 1) / WG;
        // (the last group loads its last slice again: no more of them than the slices need)
        if (split <= 2) hipLaunchKernelGGL(gemm_reduce<2>, dim3((unsigned)nb), dim3(WG), 0, st, part, c, total, split);
        else if (split <= 4) hipLaunchKernelGGL(gemm_reduce<4>, dim3((unsigned)nb), dim3(WG), 0, st, part, c, total, split);
        else hipLaunchKernelGGL(gemm_reduce<8>, dim3((unsigned)nb), dim3(WG), 0, st, part, c, total, split);
    }
    return hipGetLastError();
}

// h[t][r] = f16(silu(gate x)[t][r] * (up x)[t][r]) in one pass over K: worth it
// where its tiles, which cannot split K, fill half of the CUs
bool gemm_swiglu_supported(const DMat &gate, const DMat &up, int32_t n) {
    if (!gemm_supported(gate) || up.type != gate.type || up.rows != gate.rows || up.cols != gate.cols || n <= 0) return false;
    const int rt = gemm_rt(gate, GM_ROWS / 2);
    return rt * ((n + 127) / 128) >= 128;
}

hipError_t launch_gemm_swiglu(const DMat &gate, const DMat &up, const uint16_t *x, int32_t n, uint16_t *h,
                              hipStream_t st) {
    if (!gemm_swiglu_supported(gate, up, n) || !h) return hipErrorInvalidValue;
    GemmArgs a{};
    a.x = x;
    a.n = n;
    a.m2 = up;
    a.h = h;
    const GemmPlan p = gemm_plan(gate.type, gemm_rt(gate, GM_ROWS / 2), gate.cols / GM_KC, n, 0.0, 1, false, true);
    int blocks = 0;
    gemm_seg(a, gate, nullptr, p, GM_ROWS / 2, blocks);
    return gemm_launch<2>(a, blocks, p, st);
}

hipError_t launch_gemm_parts(const DMat &m, const uint16_t *x, int32_t n, float *part, size_t part_bytes, int *split,
                             hipStream_t st) {
    const DMat *ms[1] = {&m};
    return launch_gemm_parts_multi(ms, &part, &part_bytes, 1, x, n, split, st);
}

// up to GM_MAX_SEG projections of the same x in one launch (same type and K):
// one launch's fixed cost instead of nseg (the DeltaNet layer's four input
// projections at 64 tokens: 28.7 us in four launches), and one plan for all of
// them, chosen for the launch's blocks together
hipError_t launch_gemm_parts_multi(const DMat *const *m, float *const *part, const size_t *part_bytes, int nseg,
                                   const uint16_t *x, int32_t n, int *split, hipStream_t st) {
    if (nseg < 1 || nseg > GM_MAX_SEG || n <= 0) return hipErrorInvalidValue;
    int rt = 0, cap = 64;
    double out = 0;
    for (int i = 0; i < nseg; i++) {
        if (!gemm_supported(*m[i]) || m[i]->type != m[0]->type || m[i]->cols != m[0]->cols || !part[i] ||
            part_bytes[i] < (size_t)n * m[i]->rows * 4)
            return hipErrorInvalidValue;
        rt += gemm_rt(*m[i]);
        out += (double)n * m[i]->rows;
        cap = std::min(cap, gemm_cap(*m[i], n, part_bytes[i]));
    }
    const GemmPlan p = gemm_plan(m[0]->type, rt, m[0]->cols / GM_KC, n, out, cap, false);
    GemmArgs a{};
    a.x = x;
    a.n = n;
    int blocks = 0;
    for (int i = 0; i < nseg; i++) {
        split[i] = p.split;
        gemm_seg(a, *m[i], part[i], p, GM_ROWS, blocks);
    }
    return gemm_launch<1>(a, blocks, p, st);
}

}  // namespace oi
