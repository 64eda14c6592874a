// bulk.hip -- prompt panels (mi_prefill, mi_teacher): up to kBulkM tokens per pass over the
// weights, one launch per phase (the reference runs its prompt in chunks of up to 8 tokens
// through forward_batch, cuda_infer.cu:990-1026, 1133-1144; mega.cu:622, 819-820).
//
// A prompt in 8-token steps reads the weights once per 8 tokens and pays ~291 grid barriers
// per step: 1.4 ms a step on the 1.5B shape, 84.1 ms for 512 tokens, 530 ms for 3001. Panels
// read them once per 2048 tokens: 4.5 and 29.9 ms.
//
// Every value equals the single-token step's bit for bit (the reduction plan at the top of
// kernels.hip):
//   q4_0 x int8   the integer block dots on int8 MFMA (exact); dw*dx of a block is an outer
//                 product of fp16 values, taken by an f16 MFMA (exact: 11 x 11 bits); the fp32
//                 chain acc = fma(dw*dx, float(dot), acc) stays on the VALU. Chunk sums and
//                 segments are added left to right as everywhere.
//   attention     an f32 MFMA is a chain of fused multiply-adds in k order (one rounding per
//                 term), which is what the canonical q.k and p.v chains are.
#include "bulk.hpp"
#include "device.hpp"

#include <algorithm>
#include <type_traits>

namespace mi {

#define LAUNCH(kern, grid, block, stream, ...) hipLaunchKernelGGL(kern, dim3(grid), dim3(block), 0, stream, __VA_ARGS__)

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef int i32x16 __attribute__((ext_vector_type(16)));

constexpr int kBMaxE = kMaxE;
constexpr int kBThreads = 256;
constexpr int kBulkWgs = 288;      // 9/8 of the 256 CUs
constexpr int kKW = 8, kGThreads = 64 * kKW;   // waves of a GEMM workgroup: the chunks it runs at once

static size_t rec_floats(int NH, int HD, int nsp) { return (size_t)NH * nsp * (HD + 4); }   // of one token

static size_t pad256(size_t n) { return (n + 255) & ~size_t(255); }

BulkSizes bulk_sizes(int E, int FF, int NH, int HD, int QKV, int V, int maxseq, int ks_d, size_t kv) {
    const size_t M = std::min(kBulkM, (maxseq + 63) / 64 * 64);
    const int nsp = (maxseq + kAttnChunk * kAttnSplit - 1) / (kAttnChunk * kAttnSplit);
    const size_t tok = nsp > 1 ? rec_floats(NH, HD, nsp) : 0;
    BulkSizes s;
    s.h = M * E;
    s.xq = M * E;
    s.xd = M * (E / 32);
    s.qkv = M * QKV;
    s.aq = M * FF;
    s.ad = M * (FF / 32);
    s.dpart = (size_t)ks_d * std::min<size_t>(kBulkSplitM, M) * E;
    s.cand = M * (V / 64);
    const size_t idle = pad256(s.aq) + pad256(4 * s.ad) + pad256(4 * s.dpart) + pad256(16 * s.cand);
    s.rec = std::max(idle / 4, std::min(M * tok, std::max(std::max(kBulkRecFloats, kv / 4), 32 * tok)));
    return s;
}

size_t bulk_bind(const BulkSizes& s, void* base, BulkBuf* B) {
    size_t off = 0;
    auto take = [&](size_t bytes) {
        void* p = base ? static_cast<uint8_t*>(base) + off : nullptr;
        off += pad256(bytes);
        return p;
    };
    BulkBuf b;
    b.h = static_cast<float*>(take(4 * s.h));
    b.xq = static_cast<int8_t*>(take(s.xq));
    b.xd = static_cast<uint32_t*>(take(4 * s.xd));
    b.qkv = static_cast<float*>(take(4 * s.qkv));
    const size_t rec = off;
    b.aq = static_cast<int8_t*>(take(s.aq));
    b.ad = static_cast<uint32_t*>(take(4 * s.ad));
    b.dpart = static_cast<float*>(take(4 * s.dpart));
    b.cand = static_cast<float4*>(take(16 * s.cand));
    b.rec = reinterpret_cast<float*>(b.aq);
    b.rec_floats = s.rec;
    if (base) *B = b;
    return std::max(off, rec + pad256(4 * s.rec));
}

int bulk_attn_tokens(size_t room, int NH, int HD, int nsp, int m) {
    const int fit = std::max<int>(32, (int)std::min<size_t>(kBulkM, room / rec_floats(NH, HD, nsp)) / 32 * 32);
    if (m <= fit) return m;
    const int n = (m + fit - 1) / fit;                       // even launches
    return ((m + n - 1) / n + 31) / 32 * 32;
}

__device__ __forceinline__ uint16_t f2h_bits(float v) { return __half_as_ushort(__float2half(v)); }

// ------------------------------------------------------------------ GEMM
// D layout of a 32x32 MFMA tile: lane l holds column l % 32, rows 8(j/4) + 4(l/32) + j%4.
__device__ __forceinline__ int drow(int j, int half) { return 8 * (j >> 2) + 4 * half + (j & 3); }

// 16 nibbles of one half block as int8 16*(n - 8): the low nibbles (elements 0..15) on
// lanes 0..31, the high ones (16..31) on lanes 32..63. In the byte's upper half and with
// its top bit flipped a nibble is the signed byte 16(n - 8); the factor 16 comes off
// the finished sums (a power of two, so exactly).
template <class V>
__device__ __forceinline__ i32x4 unpack16(V w, int sh) {
    const uint32_t m = 0xF0F0F0F0u, x = 0x80808080u;
    return i32x4{(int)((((uint32_t)w.x << sh) & m) ^ x), (int)((((uint32_t)w.y << sh) & m) ^ x),
                 (int)((((uint32_t)w.z << sh) & m) ^ x), (int)((((uint32_t)w.w << sh) & m) ^ x)};
}

enum BEpi { BE_PART, BE_RES, BE_GU, BE_LM };

// One 32 x 32 tile, two blocks: acc += their terms of the chain. a0, a1: the blocks' weight
// codes (unpack16); b0, b1: the tokens' codes; dw, dx: fp16 bits of the row and token scales,
// the first block's on lanes 0..31, the second's on 32..63.
// The asm statements keep one tile's products at a time in registers, and its conversions
// together ahead of the chain (back to back they would wait on each other). 109 ns per SIMD
// with two waves on it, of which the 64 vector instructions are 97; with the outer product
// on the f32 MFMA 136, on the vector unit 113, with f16 dots (no conversion) 109-115.
__device__ __forceinline__ void tile_pair(float (&acc)[16], i32x4 a0, i32x4 a1, i32x4 b0, i32x4 b1, uint32_t dw, uint32_t dx) {
    uint2 dw2 = make_uint2(dw, 0u), dx2 = make_uint2(dx, 0u);
    asm volatile("" : "+v"(dx2.x), "+v"(b0), "+v"(b1));
    // dw * dx of both blocks: k = 0 of a two-block f16 outer product (exact in fp32)
    f32x32 pr = {};
    pr = __builtin_amdgcn_mfma_f32_32x32x4f16(__builtin_bit_cast(f16x4, dw2), __builtin_bit_cast(f16x4, dx2), pr, 0, 0, 0);
    i32x16 d0 = {}, d1 = {};
    d0 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a0, b0, d0, 0, 0, 0);
    d1 = __builtin_amdgcn_mfma_i32_32x32x32_i8(a1, b1, d1, 0, 0, 0);
    asm volatile("" : "+v"(d0), "+v"(d1), "+v"(pr));
    f32x16 t0, t1;
#pragma unroll
    for (int j = 0; j < 16; j++) t0[j] = __int2float_rn(d0[j]);
#pragma unroll
    for (int j = 0; j < 16; j++) t1[j] = __int2float_rn(d1[j]);
    asm volatile("" : "+v"(t0), "+v"(t1));
#pragma unroll
    for (int j = 0; j < 16; j++) acc[j] = __fmaf_rn(pr[j], t0[j], acc[j]);
#pragma unroll
    for (int j = 0; j < 16; j++) acc[j] = __fmaf_rn(pr[16 + j], t1[j], acc[j]);
    // element by element: a 16-register tuple here turns half of the v_fmac into v_fma with
    // all operands in one register bank (2.75 against 1.35 ns)
#pragma unroll
    for (int j = 0; j < 16; j += 4) asm volatile("" : "+v"(acc[j]), "+v"(acc[j + 1]), "+v"(acc[j + 2]), "+v"(acc[j + 3]));
}

// gate and up sums of the same 16 rows (D layout) and token: silu(g)*u, then the token's int8
// block, codes packed per 4 rows; returns the block scale
__device__ __forceinline__ float silu_quant(const float (&gt)[16], const float (&up)[16], uint32_t (&w)[4]) {
    float a[16], mx = 0.f;
#pragma unroll
    for (int i = 0; i < 16; i++) {
        const float e = mi_expf(-gt[i]);
        a[i] = __fmul_rn(__fdiv_rn(gt[i], __fadd_rn(1.0f, e)), up[i]);
        mx = fmaxf(mx, fabsf(a[i]));
    }
    float x, y;
    pair32(mx, x, y);
    mx = fmaxf(x, y);
    const float inv = mx > 0.f ? __fdiv_rn(127.f, mx) : 0.f;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        w[j] = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) w[j] |= (uint32_t)(__float2int_rn(__fmul_rn(a[4 * j + i], inv)) & 0xFF) << (8 * i);
    }
    return __fdiv_rn(mx, 127.f);
}

struct BStage {                    // one pair of blocks: 64 weight rows, 64 tokens
    uint4 a[2][2];                 // [32-row tile][block]
    i32x4 b[2][2];                 // [32-token tile][block]
    uint32_t dx[2];                // token scales (fp16 bits): block 2p on lanes 0..31, 2p + 1 on 32..63
    uint32_t sw[2];                // row scales of both blocks (fp16 x 2), [32-row tile]
};

// One workgroup: 64 rows x 64 tokens, eight waves. Wave w takes chunks w, w + 8, ... of the K
// range: per chunk the 2 x 2 tiles of 32 x 32 outputs run their block chains; then the
// waves' chunk sums meet in LDS and are added in chunk order, each wave for an eighth of the
// outputs (both row tiles, token tile w % 2, rows 8(w/2) + 4(l/32) .. + 3). Weights and
// activations go straight to registers (each wave reads its own K range, so there is nothing
// to share inside the workgroup), one block pair ahead.
// W: rows of the GEMM; xq/xd: the first token tile; out[..]: token 0 of the first tile.
// Grid (1-D): XCD x = id % 8 holds row groups g % 8 == x and walks their token tiles next
// to each other, so a group's weights come from HBM once and are then in that XCD's L2.
template <int CB, int EPI>
__global__ __launch_bounds__(kGThreads, 2) void k_bgemm(PMat W, const int8_t* xq, const uint32_t* xd, int ntt, int nseg,
                                                        float* out, int ostride, int8_t* oq, uint32_t* od) {
    __shared__ float4 red[kKW][4][4][64];                    // [chunk of the window][tile][j][lane]
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, half = lane >> 5,
              col = lane & 31;
    const int ng = W.rows >> 6, per = ntt * nseg, id = blockIdx.x;
    const int k0 = id >> 3, gi = k0 / per, rest = k0 - gi * per, g = gi * 8 + (id & 7);
    if (g >= ng) return;
    const int sidx = rest / ntt, tt = rest - sidx * ntt;
    // K segments [s0, s1) of the plan: all of them, or one per workgroup
    const int s0 = nseg > 1 ? sidx : 0, s1 = nseg > 1 ? sidx + 1 : W.ks;
    const int cbeg = s0 * W.nc / W.ks, cend = s1 * W.nc / W.ks;
    const uint8_t* wbase = W.base + (size_t)g * W.nc * (CB * 1152);
    const int8_t* xt = xq + (size_t)(2 * tt) * W.nb * 1024;
    const uint32_t* dt = xd + (size_t)(2 * tt) * W.nb * 32;
    const size_t xstep = (size_t)W.nb * 1024, dstep = (size_t)W.nb * 32;
    const int sh = half ? 0 : 4;

    // uniform base (the wave's chunk) + lane offset
    const int woff = col * 16, xoff = lane * 16, soff = CB * 1024 + col * (CB * 2);
    auto load_pair = [&](BStage& s, int c, int p) {
        const uint8_t* t = wbase + (size_t)c * (CB * 1152);
        const int b = c * CB + 2 * p;
        const int8_t* x0 = xt + (size_t)b * 1024;
        const uint32_t* f0 = dt + (size_t)b * 32;
#pragma unroll
        for (int k = 0; k < 2; k++) {
            s.a[0][k] = *reinterpret_cast<const uint4*>(t + (2 * p + k) * 1024 + woff);
            s.a[1][k] = *reinterpret_cast<const uint4*>(t + (2 * p + k) * 1024 + 512 + woff);
            s.b[0][k] = *reinterpret_cast<const i32x4*>(x0 + k * 1024 + xoff);
            s.b[1][k] = *reinterpret_cast<const i32x4*>(x0 + xstep + k * 1024 + xoff);
        }
        s.dx[0] = f0[lane];
        s.dx[1] = (f0 + dstep)[lane];
        s.sw[0] = *reinterpret_cast<const uint32_t*>(t + 4 * p + soff);
        s.sw[1] = *reinterpret_cast<const uint32_t*>(t + 4 * p + 32 * CB * 2 + soff);
        asm volatile("" ::: "memory");                       // issued here, not where they are used
    };
    float acc[2][2][16];
    auto pair = [&](const BStage& s) {
#pragma unroll
        for (int r = 0; r < 2; r++) {
            const i32x4 a0 = unpack16(s.a[r][0], sh), a1 = unpack16(s.a[r][1], sh);
            const uint32_t dw = (s.sw[r] >> (half * 16)) & 0xFFFFu;
#pragma unroll
            for (int t = 0; t < 2; t++) tile_pair(acc[r][t], a0, a1, s.b[t][0], s.b[t][1], dw, s.dx[t]);
        }
    };

    BStage st[2];
    const int ot = wave & 1, oj = wave >> 1;                 // this wave's share of the outputs
    float sg[8], tot[8];
#pragma unroll
    for (int i = 0; i < 8; i++) sg[i] = tot[i] = 0.f;
    int s = s0, sb = cbeg, se = (s0 + 1) * W.nc / W.ks;      // the segment the sums are in
    if (cbeg + wave < cend) load_pair(st[0], cbeg + wave, 0);
    for (int c0 = cbeg; c0 < cend; c0 += kKW) {
        const int c = c0 + wave;
        if (c < cend) {
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int j = 0; j < 16; j++) acc[r][t][j] = 0.f;
#pragma unroll
            for (int p = 0; p < CB / 2; p++) {
                if (p + 1 < CB / 2) {
                    load_pair(st[(p + 1) & 1], c, p + 1);
                } else if (c + kKW < cend) {
                    load_pair(st[(p + 1) & 1], c + kKW, 0);
                }
                pair(st[p & 1]);
            }
#pragma unroll
            for (int r = 0; r < 2; r++)
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        red[wave][2 * r + t][j][lane] =
                            make_float4(acc[r][t][4 * j], acc[r][t][4 * j + 1], acc[r][t][4 * j + 2], acc[r][t][4 * j + 3]);
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < kKW; i++) {
            const int ci = c0 + i;
            if (ci < cend) {
                const bool first = ci == sb;
#pragma unroll
                for (int r = 0; r < 2; r++) {
                    const float4 v = red[i][2 * r + ot][oj][lane];
                    sg[4 * r] = first ? v.x : __fadd_rn(sg[4 * r], v.x);
                    sg[4 * r + 1] = first ? v.y : __fadd_rn(sg[4 * r + 1], v.y);
                    sg[4 * r + 2] = first ? v.z : __fadd_rn(sg[4 * r + 2], v.z);
                    sg[4 * r + 3] = first ? v.w : __fadd_rn(sg[4 * r + 3], v.w);
                }
                if (ci + 1 == se) {                          // segment done: segments left to right
#pragma unroll
                    for (int j = 0; j < 8; j++) tot[j] = s == s0 ? sg[j] : __fadd_rn(tot[j], sg[j]);
                    s++;
                    sb = se;
                    se = (s + 1) * W.nc / W.ks;
                }
            }
        }
        __syncthreads();
    }

    // the weight codes were 16(n - 8): 1/16 here is exact, and so is every step before (all
    // terms are multiples of 2^-48, so the chains never meet a denormal)
#pragma unroll
    for (int i = 0; i < 8; i++) tot[i] = __fmul_rn(tot[i], 0.0625f);
    // tot[4r + i]: row 32r + 8 oj + 4 half + i of the group, token tok
    const int tok = (2 * tt + ot) * 32 + col;
    if constexpr (EPI != BE_GU) {
        float* o = out + (size_t)sidx * ostride + (size_t)tok * W.rows + g * 64 + 8 * oj + 4 * half;
#pragma unroll
        for (int r = 0; r < 2; r++) {
            float4 v = make_float4(tot[4 * r], tot[4 * r + 1], tot[4 * r + 2], tot[4 * r + 3]);
            float4* q = reinterpret_cast<float4*>(o + 32 * r);
            if constexpr (EPI == BE_RES) {
                const float4 h = *q;
                v = make_float4(__fadd_rn(h.x, v.x), __fadd_rn(h.y, v.y), __fadd_rn(h.z, v.z), __fadd_rn(h.w, v.w));
            }
            *q = v;
        }
    } else {
        // rows 0..31 of a group are gate rows, 32..63 their up rows: silu(g)*u, then one int8
        // block per token, its max over the four waves of the token tile
        float a[4], mx = 0.f;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float e = mi_expf(-tot[i]);
            a[i] = __fmul_rn(__fdiv_rn(tot[i], __fadd_rn(1.0f, e)), tot[4 + i]);
            mx = fmaxf(mx, fabsf(a[i]));
        }
        float x, y;
        pair32(mx, x, y);
        float* ml = reinterpret_cast<float*>(red);           // [4 waves][2 tiles][32 tokens]
        if (half == 0) ml[(oj * 2 + ot) * 32 + col] = fmaxf(x, y);
        __syncthreads();
        mx = 0.f;
#pragma unroll
        for (int j = 0; j < 4; j++) mx = fmaxf(mx, ml[(j * 2 + ot) * 32 + col]);
        const float inv = mx > 0.f ? __fdiv_rn(127.f, mx) : 0.f;
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) w |= (uint32_t)(__float2int_rn(__fmul_rn(a[i], inv)) & 0xFF) << (8 * i);
        *reinterpret_cast<uint32_t*>(oq + bx_at(ng, tok, g, 8 * oj + 4 * half)) = w;
        if (oj == 0 && half == 0) od[bd_at(ng, tok, g)] = f2h_bits(__fdiv_rn(mx, 127.f));
    }
}

// The same product for gate/up and lm_head, whose row groups alone fill the chip: no K split
// (their plan has one segment), so no exchange of chunk sums; each wave runs 32 rows x 64
// tokens through all of K and keeps the running sums in registers. A workgroup is 64 rows x
// 128 tokens, two workgroups per CU. Weights and activations are loaded four block pairs
// ahead: a wave's loads return in order, so the activations (L2) wait for the weights (HBM)
// issued before them.
// GU: the group's gate rows 0..31 and up rows 32..63 meet in LDS, silu(g)*u -> oq / od.
// LM: the group's argmax candidate per token -> cand.
template <int CB, int EPI>
__global__ __launch_bounds__(kBThreads, 2) void k_bgemm_w(PMat W, const int8_t* xq, const uint32_t* xd, int ntt, int8_t* oq,
                                                          uint32_t* od, float4* cand) {
    __shared__ float4 ex[4][2][4][64];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, half = lane >> 5,
              col = lane & 31;
    const int ng = W.rows >> 6, per = (ntt + 1) >> 1, id = blockIdx.x;
    const int k0 = id >> 3, gi = k0 / per, g = gi * 8 + (id & 7);
    if (g >= ng) return;
    const int rt = wave & 1, tt = 2 * (k0 - gi * per) + (wave >> 1);
    const bool active = tt < ntt;                            // an odd number of token tiles
    constexpr int PC = CB / 2;                               // block pairs per chunk
    const int np = W.nb / 2, sh = half ? 0 : 4;
    const uint8_t* wb = W.base + (size_t)g * W.nc * (CB * 1152) + rt * 512;
    const uint8_t* wsc = W.base + (size_t)g * W.nc * (CB * 1152) + CB * 1024 + rt * 32 * CB * 2;
    const int8_t* x0 = xq + (size_t)(2 * tt) * W.nb * 1024;
    const uint32_t* f0 = xd + (size_t)(2 * tt) * W.nb * 32;
    const size_t xstep = (size_t)W.nb * 1024, dstep = (size_t)W.nb * 32;
    const int woff = col * 16, xoff = lane * 16, soff = col * (CB * 2);

    struct Slot { i32x4 a[2], b[2][2]; uint32_t sw, dx[2]; };
    auto load = [&](Slot& s, int q) {
        const int c = q / PC, p = q - c * PC;
        const uint8_t* t = wb + (size_t)c * (CB * 1152) + 2 * p * 1024;
        const int8_t* x = x0 + (size_t)q * 2048;
        const uint32_t* f = f0 + (size_t)q * 64;
        s.sw = *reinterpret_cast<const uint32_t*>(wsc + (size_t)c * (CB * 1152) + 4 * p + soff);
        s.dx[0] = f[lane];
        s.dx[1] = (f + dstep)[lane];
#pragma unroll
        for (int k = 0; k < 2; k++) {
            s.a[k] = *reinterpret_cast<const i32x4*>(t + k * 1024 + woff);
            s.b[0][k] = *reinterpret_cast<const i32x4*>(x + k * 1024 + xoff);
            s.b[1][k] = *reinterpret_cast<const i32x4*>(x + xstep + k * 1024 + xoff);
        }
        asm volatile("" ::: "memory");                       // issued here, not where they are used
    };
    constexpr int NS = 4;
    Slot sl[NS];
    float acc[2][16];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < 16; j++) acc[t][j] = 0.f;
    // the running sums, each lane's own words in LDS (in registers they would make the loop
    // spill, and a reload waits for every load in flight); -0 + x = x
    float4 (&sum)[2][4][64] = ex[wave];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) sum[t][j][lane] = make_float4(-0.f, -0.f, -0.f, -0.f);
    if (active) {
        // past the end the last pair is loaded again (a branch around the load keeps the old
        // slot alive and costs copies)
#pragma unroll
        for (int u = 0; u < NS; u++) load(sl[u], min(u, np - 1));
        auto step = [&](Slot& s, int q, bool chunk_end) {
            // nothing of this pair is computed (and so waited for) before the last one is done
            asm volatile("" : "+v"(s.sw), "+v"(s.a[0]), "+v"(s.a[1]));
            const i32x4 a0 = unpack16(s.a[0], sh), a1 = unpack16(s.a[1], sh);
            const uint32_t dw = (s.sw >> (half * 16)) & 0xFFFFu;
#pragma unroll
            for (int t = 0; t < 2; t++) tile_pair(acc[t], a0, a1, s.b[t][0], s.b[t][1], dw, s.dx[t]);
            load(s, min(q + NS, np - 1));
            if (chunk_end) {                                 // compile time: a chunk is 2 or 4 pairs
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int j = 0; j < 4; j++) {
                        const float4 v = sum[t][j][lane];
                        sum[t][j][lane] = make_float4(__fadd_rn(v.x, acc[t][4 * j]), __fadd_rn(v.y, acc[t][4 * j + 1]),
                                                      __fadd_rn(v.z, acc[t][4 * j + 2]), __fadd_rn(v.w, acc[t][4 * j + 3]));
                        acc[t][4 * j] = acc[t][4 * j + 1] = acc[t][4 * j + 2] = acc[t][4 * j + 3] = 0.f;
                    }
            }
        };
        // no branch inside the four steps: the compiler then counts the loads in flight exactly
        int q = 0;
        for (; q + NS <= np; q += NS)
#pragma unroll
            for (int u = 0; u < NS; u++) step(sl[u], q + u, (u + 1) % PC == 0);
        if constexpr (CB == 4)
            if (q < np) {                                    // an odd number of chunks of two pairs
                step(sl[0], q, false);
                step(sl[1], q + 1, true);
            }
    }
    // 1/16: the weight codes were 16(n - 8)
    float sg[2][16];
#pragma unroll
    for (int t = 0; t < 2; t++)
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float4 v = sum[t][j][lane];
            sg[t][4 * j] = __fmul_rn(v.x, 0.0625f); sg[t][4 * j + 1] = __fmul_rn(v.y, 0.0625f);
            sg[t][4 * j + 2] = __fmul_rn(v.z, 0.0625f); sg[t][4 * j + 3] = __fmul_rn(v.w, 0.0625f);
        }
    if constexpr (EPI == BE_GU) {
        // wave rt finishes token tile rt of its pair: it hands the other one over
#pragma unroll
        for (int j = 0; j < 4; j++)
            ex[wave][0][j][lane] = rt ? make_float4(sg[0][4 * j], sg[0][4 * j + 1], sg[0][4 * j + 2], sg[0][4 * j + 3])
                                   : make_float4(sg[1][4 * j], sg[1][4 * j + 1], sg[1][4 * j + 2], sg[1][4 * j + 3]);
        __syncthreads();
        if (!active) return;
        float gt[16], up[16];
#pragma unroll
        for (int j = 0; j < 4; j++) {
            const float4 o = ex[wave ^ 1][0][j][lane];
            const float ov[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                gt[4 * j + i] = rt ? ov[i] : sg[0][4 * j + i];
                up[4 * j + i] = rt ? sg[1][4 * j + i] : ov[i];
            }
        }
        const int tok = (2 * tt + rt) * 32 + col;
        uint32_t w[4];
        const float d = silu_quant(gt, up, w);
#pragma unroll
        for (int j = 0; j < 4; j++) *reinterpret_cast<uint32_t*>(oq + bx_at(ng, tok, g, 8 * j + 4 * half)) = w[j];
        if (half == 0) od[bd_at(ng, tok, g)] = f2h_bits(d);
    } else {
        Top2 tp[2];
#pragma unroll
        for (int t = 0; t < 2; t++) {
            tp[t] = Top2{-__builtin_inff(), INT_MAX, -__builtin_inff()};
#pragma unroll
            for (int j = 0; j < 16; j++) top2_push(tp[t], sg[t][j], g * 64 + rt * 32 + drow(j, half));
            ex[wave][0][t][lane] = make_float4(tp[t].best, __int_as_float(tp[t].idx), tp[t].second, 0.f);
        }
        __syncthreads();
        if (!active || half) return;
        // wave rt: token tile rt; the four parts are its two halves and the other wave's
        Top2 a{-__builtin_inff(), INT_MAX, -__builtin_inff()};
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float4 o = ex[(wave & 2) + (k >> 1)][0][rt][32 * (k & 1) + col];
            top2_merge(a, o.x, __float_as_int(o.y), o.z);
        }
        cand[(size_t)((2 * tt + rt) * 32 + col) * ng + g] = make_float4(a.best, __int_as_float(a.idx), a.second, 0.f);
    }
}

// argmax and margin of one token: the candidates of its V/64 row groups (candidate row
// blockIdx, position p0 + blockIdx); top-2 merging is associative and commutative
__global__ __launch_bounds__(kBThreads) void k_bargmax(const float4* cand, int ng, int V, int p0, int32_t* out_tok,
                                                       float* out_margin) {
    __shared__ float4 wl[kBThreads / 64];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    Top2 a{-__builtin_inff(), INT_MAX, -__builtin_inff()};
    for (int i = tid; i < ng; i += kBThreads) {
        const float4 c = cand[(size_t)t * ng + i];
        top2_merge(a, c.x, __float_as_int(c.y), c.z);
    }
    top2_wave(a);
    if (lane == 0) wl[tid >> 6] = make_float4(a.best, __int_as_float(a.idx), a.second, 0.f);
    __syncthreads();
    if (tid) return;
    for (int w = 1; w < kBThreads / 64; w++) top2_merge(a, wl[w].x, __float_as_int(wl[w].y), wl[w].z);
    out_tok[p0 + t] = top2_token(a, V);
    out_margin[p0 + t] = __fsub_rn(a.best, a.second);
}

// ------------------------------------------------------------------ residual, norm, quant
// One workgroup per token: h (layer 0: the embedding row) + the down partials in order,
// written back; RMSNorm and int8 quantisation into the GEMM operand. prows: rows of one partial. Thread i holds elements
// 4i .. + 3 (and those 1024 further on); the row meets in LDS, where every wave takes the
// canonical sum of squares (lane l: elements 256j + 4l + i over j, then i). A wave per token
// was a chain of its partials' loads on 16 CUs at 64 tokens: 20.4 us with the 10 partials of
// the 1.5B shape.
__global__ __launch_bounds__(kBThreads) void k_bnorm(int n, float eps, const float* w, float* h, const float* emb,
                                                     const int32_t* tok, const float* part, int ks, int prows,
                                                     int8_t* xq, uint32_t* xd) {
    constexpr int NI = kBMaxE / (4 * kBThreads);
    __shared__ __align__(16) float row[kBMaxE];
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid & 63;
    const float* src = emb ? emb + (size_t)tok[t] * n : h + (size_t)t * n;
    float4 x[NI], wv[NI];
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int e = 4 * (tid + i * kBThreads);
        x[i] = wv[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (e < n) {
            x[i] = *reinterpret_cast<const float4*>(src + e);
            wv[i] = *reinterpret_cast<const float4*>(w + e);
            if (ks > 0) {
                const float* pt = part + (size_t)t * n + e;
                const size_t step = (size_t)prows * n;
                float4 s = *reinterpret_cast<const float4*>(pt);
                auto add = [&](float4 p) {
                    s = make_float4(__fadd_rn(s.x, p.x), __fadd_rn(s.y, p.y), __fadd_rn(s.z, p.z), __fadd_rn(s.w, p.w));
                };
                int k = 1;
                for (; k + 3 <= ks; k += 3) {                // three loads ahead of their adds
                    const float4 a = *reinterpret_cast<const float4*>(pt + k * step);
                    const float4 b = *reinterpret_cast<const float4*>(pt + (k + 1) * step);
                    const float4 c = *reinterpret_cast<const float4*>(pt + (k + 2) * step);
                    add(a);
                    add(b);
                    add(c);
                }
                for (; k < ks; k++) add(*reinterpret_cast<const float4*>(pt + k * step));
                x[i] = make_float4(__fadd_rn(x[i].x, s.x), __fadd_rn(x[i].y, s.y), __fadd_rn(x[i].z, s.z), __fadd_rn(x[i].w, s.w));
            }
            if (emb || ks > 0) *reinterpret_cast<float4*>(h + (size_t)t * n + e) = x[i];
        }
        *reinterpret_cast<float4*>(row + e) = x[i];          // zeros past n: fma(0, 0, a) = a
    }
    __syncthreads();
    float a = 0.f;
    for (int j = 0; 256 * j < n; j++) {
        const float4 u = *reinterpret_cast<const float4*>(row + 256 * j + 4 * lane);
        a = __fmaf_rn(u.x, u.x, a); a = __fmaf_rn(u.y, u.y, a);
        a = __fmaf_rn(u.z, u.z, a); a = __fmaf_rn(u.w, u.w, a);
    }
    a = bfly_sum64(a);
    const float sc = __fdiv_rn(1.0f, __builtin_sqrtf(__fadd_rn(__fdiv_rn(a, (float)n), eps)));
    const int nb = n / 32;
#pragma unroll
    for (int i = 0; i < NI; i++) {
        const int e = 4 * (tid + i * kBThreads);             // a block is 8 lanes: all in or all past n
        float4 y = make_float4(__fmul_rn(__fmul_rn(x[i].x, sc), wv[i].x), __fmul_rn(__fmul_rn(x[i].y, sc), wv[i].y),
                               __fmul_rn(__fmul_rn(x[i].z, sc), wv[i].z), __fmul_rn(__fmul_rn(x[i].w, sc), wv[i].w));
        const float mx = max8(fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w))));
        const float inv = mx > 0.f ? __fdiv_rn(127.f, mx) : 0.f;
        const int q0 = __float2int_rn(__fmul_rn(y.x, inv)), q1 = __float2int_rn(__fmul_rn(y.y, inv));
        const int q2 = __float2int_rn(__fmul_rn(y.z, inv)), q3 = __float2int_rn(__fmul_rn(y.w, inv));
        if (e < n) {
            *reinterpret_cast<uint32_t*>(xq + bx_at(nb, t, e >> 5, e & 31)) =
                (uint32_t)(q0 & 0xFF) | ((uint32_t)(q1 & 0xFF) << 8) | ((uint32_t)(q2 & 0xFF) << 16) | ((uint32_t)q3 << 24);
            if ((lane & 7) == 0) xd[bd_at(nb, t, e >> 5)] = f2h_bits(__fdiv_rn(mx, 127.f));
        }
    }
}

// ------------------------------------------------------------------ bias, RoPE, K/V append
// One thread per (token, head of q|k|v, pair i, i + HD/2): the QKV row + bias, rotated for q
// (in place) and k; k and v rounded to fp16 into the cache (cpu_infer.cpp:49-61, 114-120).
template <int HD>
__global__ __launch_bounds__(kBThreads) void k_brope(float* qkv, const float* bias, const float2* rope, int NH, int NKV,
                                                     int QKV, int m, int p0, int maxseq, __half* kc, __half* vc) {
    constexpr int half = HD / 2;
    const int nh = NH + 2 * NKV;
    const size_t id = (size_t)blockIdx.x * kBThreads + threadIdx.x;
    const int i = (int)(id % half), h = (int)((id / half) % nh), t = (int)(id / half / nh);
    if (t >= m) return;
    float* r = qkv + (size_t)t * QKV + h * HD;
    const float x0 = __fadd_rn(r[i], bias[h * HD + i]), x1 = __fadd_rn(r[i + half], bias[h * HD + i + half]);
    if (h >= NH + NKV) {
        __half* d = vc + ((size_t)(h - NH - NKV) * maxseq + p0 + t) * HD;
        d[i] = __float2half(x0);
        d[i + half] = __float2half(x1);
        return;
    }
    const float2 cz = rope[(size_t)(p0 + t) * half + i];
    const float y0 = __fsub_rn(__fmul_rn(x0, cz.x), __fmul_rn(x1, cz.y));
    const float y1 = __fadd_rn(__fmul_rn(x0, cz.y), __fmul_rn(x1, cz.x));
    if (h < NH) {
        r[i] = y0;
        r[i + half] = y1;
    } else {
        __half* d = kc + ((size_t)(h - NH) * maxseq + p0 + t) * HD;
        d[i] = __float2half(y0);
        d[i + half] = __float2half(y1);
    }
}

// ------------------------------------------------------------------ attention
// mi_expf without its branches (the same value for every input)
__device__ __forceinline__ float mi_expf_sel(float x) {
    const float n = __builtin_rintf(__fmul_rn(x, 0x1.715476p+0f));
    float r = __fmaf_rn(n, -0x1.62e4p-1f, x);
    r = __fmaf_rn(n, -0x1.7f7d1cp-20f, r);
    float p = 0x1.a01a02p-13f;
    p = __fmaf_rn(p, r, 0x1.6c16c2p-10f);
    p = __fmaf_rn(p, r, 0x1.111112p-7f);
    p = __fmaf_rn(p, r, 0x1.555556p-5f);
    p = __fmaf_rn(p, r, 0x1.555556p-3f);
    p = __fmaf_rn(p, r, 0x1p-1f);
    p = __fmaf_rn(p, r, 1.0f);
    p = __fmaf_rn(p, r, 1.0f);
    p = __builtin_ldexpf(p, (int)n);
    p = x < -87.0f ? 0.f : p;
    p = x > 88.72283f ? __builtin_inff() : p;
    return x != x ? x : p;
}

// One workgroup, four waves: 16 tokens of one query head against one split (16 chunks of 64
// positions); two workgroups per CU. An f32 MFMA is a chain of fused multiply-adds in k order,
// so both canonical contractions run on it:
//   scores   unit = 32 positions x 16 tokens, units round-robin over the waves: 16x16x4 MFMAs,
//            one accumulator per chain d mod 4 (k = 0..3 are d, d + 4, d + 8, d + 12 of a chain)
//   softmax  four lanes per (chunk, token), 16 positions each (position mod 4): the chunk max,
//            exp and the canonical butterfly sum (in the lane over xor 32, 16, 8, 4, then over
//            the quad for xor 2, 1)
//   p.v      wave: HD/4 dims x 16 tokens through all chunks in order by 16x16x4 MFMAs, each
//            chunk's output merged as it is done (the split's max is known by then), so no
//            outputs are exchanged
// Scores and probabilities stay in LDS, 4 KB per chunk: word (position, token) at
// ((chunk * 4 + position % 4) * 16 + token) * 16 + position / 4, the four-word groups swizzled
// (ps_at).
// K and V rows are read without a clamp: rows past the panel are masked (scores) or meet
// p = 0 (see below), and the cache is allocated a chunk longer than its last row.
// nsp == 1: o / den goes straight into the O GEMM's int8 operand; otherwise the record of
// (token, head, split): o[HD], M, den.
// Bound by the MFMAs and the vector unit, which f32 MFMAs hold up. Per layer of the 1.5B shape
// with 512-token panels: 64 tokens 8.5 us, 512 tokens 30, tokens 1024..1535 71, 2048..2559
// 112; 32-token workgroups (one per CU) 9.9, 34, 116, 132; the waves on whole chunks, their
// outputs exchanged, everything unrolled (an 8k-line loop body) 23, 41, 105, 178.
constexpr int kAT = 16, kAWaves = 4, kAThreads = 64 * kAWaves;
__device__ __forceinline__ int ps_at(int c, int pos, int tok) {
    const int k = pos & 3, i = pos >> 2;
    return ((c * 4 + k) * kAT + tok) * 16 + ((((i >> 2) ^ (tok >> 2) ^ k) & 3) << 2) + (i & 3);
}
template <int HD>
__global__ __launch_bounds__(kAThreads, 2) void k_battn(const float* qkv, int QKV, const __half* kc, const __half* vc,
                                                        int NH, int G, int m, int p0, int maxseq, int nsp, float scale,
                                                        float* rec, int nb, int8_t* xq, uint32_t* xd) {
    constexpr int NJ = HD / 16, NU = HD / 64;
    __shared__ __align__(16) float ps[kAttnSplit * 4 * kAT * 16];
    __shared__ float mt[kAttnSplit][kAT], lt[kAttnSplit][kAT], wt[kAttnSplit][kAT], amx[4][kAT];
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
    const int ntile = (m + kAT - 1) / kAT;
    // whole splits before the ragged last one, late (long) tiles first
    const int h = blockIdx.x % NH, rest = blockIdx.x / NH, sp = rest / ntile, tile = ntile - 1 - (rest - sp * ntile);
    const int tbase = tile * kAT, tlast = min(tbase + kAT - 1, m - 1), c0 = sp * kAttnSplit;
    const int nch = (p0 + tlast) / kAttnChunk + 1 - c0;      // chunks of this split, if positive
    if (nch <= 0) return;
    const int nc = min(nch, kAttnSplit), kvh = h / G;
    const __half* kb = kc + ((size_t)kvh * maxseq + c0 * kAttnChunk) * HD;
    const __half* vb = vc + ((size_t)kvh * maxseq + c0 * kAttnChunk) * HD;
    const int kk = lane >> 4, tk = lane & 15, tok = min(tbase + tk, tlast), pos = p0 + tok;
    const int nct = min(pos / kAttnChunk + 1 - c0, kAttnSplit);   // this token's chunks of the split, may be <= 0

    // p.v: wave's dims d0 .., dim d0 + NU r + u on row r of D tile u; a lane's V rows are 4i + kk
    const int d0 = wave * 16 * NU;
    typedef typename std::conditional<NU == 2, uint32_t, uint16_t>::type VT;
    typedef uint32_t VR;                                     // in a whole register
    const int voff = kk * HD + NU * tk;
    auto vld = [&](int c, int i) {
        return (VR)*reinterpret_cast<const VT*>(vb + ((size_t)c * kAttnChunk + 4 * i) * HD + d0 + voff);
    };
    auto vf = [](VR w, int u) { return u ? h2f_hi(w) : h2f_lo(w); };
    VR vr[16];
#pragma unroll
    for (int i = 0; i < 16; i++) vr[i] = vld(0, i);          // the first chunk's, while the scores run
    asm volatile("" ::: "memory");

    {   // scores
        float q[NJ][4];                                      // q[token][16j + 4 kk + i]
#pragma unroll
        for (int j = 0; j < NJ; j++) {
            const float4 v = *reinterpret_cast<const float4*>(qkv + (size_t)tok * QKV + h * HD + 16 * j + 4 * kk);
            q[j][0] = v.x; q[j][1] = v.y; q[j][2] = v.z; q[j][3] = v.w;
        }
        // a unit's K rows, all at once (a line's pieces find it in the L1), a unit ahead
        uint2 kr[2][NJ], kn[2][NJ];
        const int koff = tk * HD + 4 * kk;
        auto kload = [&](uint2 (&k)[2][NJ], int unit) {
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < NJ; j++)
                    k[t][j] = *reinterpret_cast<const uint2*>(kb + (size_t)(unit * 32 + 16 * t) * HD + 16 * j + koff);
            asm volatile("" ::: "memory");
        };
        if (wave < 2 * nc) kload(kr, wave);
        for (int unit = wave; unit < 2 * nc; unit += kAWaves) {
            kload(kn, min(unit + kAWaves, 2 * nc - 1));
            f32x4 s[2][4];
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int i = 0; i < 4; i++) s[t][i] = f32x4{};
#pragma unroll
            for (int j = 0; j < NJ; j++)
#pragma unroll
                for (int t = 0; t < 2; t++) {
                    uint2 w = kr[t][j];
                    asm volatile("" : "+v"(w.x), "+v"(w.y));     // its wait stays here
                    const float kv[4] = {h2f_lo(w.x), h2f_hi(w.x), h2f_lo(w.y), h2f_hi(w.y)};
#pragma unroll
                    for (int i = 0; i < 4; i++) s[t][i] = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i], q[j][i], s[t][i], 0, 0, 0);
                }
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int j = 0; j < NJ; j++) kr[t][j] = kn[t][j];
            // the lane holds positions 16t + 4 kk + r of the unit, token tk
            const int c = unit >> 1, o = 32 * (unit & 1) + 4 * kk, t0 = (c0 + c) * kAttnChunk;
#pragma unroll
            for (int t = 0; t < 2; t++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float v = __fmul_rn(__fadd_rn(__fadd_rn(s[t][0][r], s[t][1][r]), __fadd_rn(s[t][2][r], s[t][3][r])), scale);
                    ps[ps_at(c, o + 16 * t + r, tk)] = t0 + o + 16 * t + r <= pos ? v : -__builtin_inff();
                }
        }
    }
    __syncthreads();
    for (int it = tid; it < nc * 4 * kAT; it += kAThreads) { // softmax
        const int k = it & 3, t2 = (it >> 2) & (kAT - 1), c = it / (4 * kAT);
        const int last = p0 + min(tbase + t2, tlast) - (c0 + c) * kAttnChunk;     // the token's own offset in the chunk
        float v[16];
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const float4 f = *reinterpret_cast<const float4*>(ps + ps_at(c, 16 * i + k, t2));
            v[4 * i] = f.x; v[4 * i + 1] = f.y; v[4 * i + 2] = f.z; v[4 * i + 3] = f.w;
        }
        float mx = v[0];
#pragma unroll
        for (int i = 1; i < 16; i++) mx = fmaxf(mx, v[i]);
        mx = fmaxf(mx, dppf<kDppXor2>(mx));
        mx = fmaxf(mx, dppf<kDppXor1>(mx));
#pragma unroll
        for (int i = 0; i < 16; i++) {
            float e = mi_expf_sel(__fsub_rn(v[i], mx));
            asm("" : "+v"(e));                               // a select, not a branch around the exp
            v[i] = 4 * i + k <= last ? e : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 4; i++)
            *reinterpret_cast<float4*>(ps + ps_at(c, 16 * i + k, t2)) = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
#pragma unroll
        for (int d = 8; d >= 1; d >>= 1)                     // xor 32, 16, 8, 4 over positions
#pragma unroll
            for (int i = 0; i < d; i++) v[i] = __fadd_rn(v[i], v[i + d]);
        float l = __fadd_rn(v[0], dppf<kDppXor2>(v[0]));
        l = __fadd_rn(l, dppf<kDppXor1>(l));
        if (k == 0) {
            mt[c][t2] = mx;
            lt[c][t2] = l;
        }
    }
    __syncthreads();
    {   // chunk weights exp(m_c - M) of the split: a thread per (chunk, token)
        const int c = tid / kAT, t2 = tid & (kAT - 1);
        const int n2 = min((p0 + min(tbase + t2, tlast)) / kAttnChunk + 1 - c0, kAttnSplit);
        float M = mt[0][t2];
        for (int i = 1; i < n2; i++) M = fmaxf(M, mt[i][t2]);
        if (c < n2) wt[c][t2] = mi_expf_sel(__fsub_rn(mt[c][t2], M));
        if (c == 0) amx[0][t2] = M;
    }
    __syncthreads();
    const float Ms = amx[0][tk];

    float den = 0.f;
    f32x4 as[NU];
#pragma unroll
    for (int u = 0; u < NU; u++) as[u] = f32x4{};
    for (int c = 0; c < nc; c++) {
        f32x4 o[NU];
#pragma unroll
        for (int u = 0; u < NU; u++) o[u] = f32x4{};
        const int cn = min(c + 1, nc - 1);
        float4 pv[4];
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++) pv[i4] = *reinterpret_cast<const float4*>(ps + ps_at(c, 16 * i4 + kk, tk));
#pragma unroll
        for (int i4 = 0; i4 < 4; i4++) {
            const float pb[4] = {pv[i4].x, pv[i4].y, pv[i4].z, pv[i4].w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                VR w = vr[4 * i4 + i];
                asm volatile("" : "+v"(w));
                vr[4 * i4 + i] = vld(cn, 4 * i4 + i);        // the next chunk's, a chunk ahead
                asm volatile("" ::: "memory");
#pragma unroll
                for (int u = 0; u < NU; u++) o[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf(w, u), pb[i], o[u], 0, 0, 0);
            }
        }
        // A position past a token's own has p = 0, which adds exactly nothing unless its V
        // holds an infinity or NaN (0 * inf): the canonical chain stops before it. So where
        // the chunk reaches past the tile's first token and a result is NaN, the chain runs
        // again one position at a time, each result kept only for the tokens that see it.
        if ((c0 + c + 1) * kAttnChunk - 1 > p0 + tbase) {
            bool nan = false;
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int j = 0; j < 4; j++) nan |= o[u][j] != o[u][j];
            if (__builtin_amdgcn_ballot_w64(nan)) {
#pragma unroll
                for (int u = 0; u < NU; u++) o[u] = f32x4{};
#pragma unroll 1
                for (int k = 0; k < kAttnChunk; k++) {
                    const bool on = (k & 3) == kk, sees = (c0 + c) * kAttnChunk + k <= pos;
                    const float pk = on ? ps[ps_at(c, k, tk)] : 0.f;
                    const VR w = vld(c, k >> 2);
#pragma unroll
                    for (int u = 0; u < NU; u++) {
                        const f32x4 z = __builtin_amdgcn_mfma_f32_16x16x4f32(on ? vf(w, u) : 0.f, pk, o[u], 0, 0, 0);
#pragma unroll
                        for (int j = 0; j < 4; j++) o[u][j] = sees ? z[j] : o[u][j];
                    }
                }
            }
        }
        if (c < nct) {
            const float w = wt[c][tk];
            den = __fmaf_rn(lt[c][tk], w, den);
#pragma unroll
            for (int u = 0; u < NU; u++)
#pragma unroll
                for (int j = 0; j < 4; j++) as[u][j] = __fmaf_rn(o[u][j], w, as[u][j]);
        }
    }
    // the lane's 4 NU consecutive dims, from d0 + 4 NU kk
    float out[4 * NU];
#pragma unroll
    for (int j = 0; j < 4; j++)
#pragma unroll
        for (int u = 0; u < NU; u++) out[NU * j + u] = as[u][j];
    const bool mine = tbase + tk <= tlast && nct > 0;
    if (nsp > 1) {
        if (!mine) return;
        float* rp = rec + (((size_t)tok * NH + h) * nsp + sp) * (HD + 4);
#pragma unroll
        for (int u = 0; u < NU; u++)
            *reinterpret_cast<float4*>(rp + d0 + 4 * NU * kk + 4 * u) = make_float4(out[4 * u], out[4 * u + 1], out[4 * u + 2], out[4 * u + 3]);
        if (wave == 0 && kk == 0) {
            rp[HD] = Ms;
            rp[HD + 1] = den;
        }
        return;
    }
    float mx = 0.f;
#pragma unroll
    for (int e = 0; e < 4 * NU; e++) {
        out[e] = __fdiv_rn(out[e], den);
        mx = fmaxf(mx, fabsf(out[e]));
    }
    float x, y;
    pair32(mx, x, y);
    mx = fmaxf(x, y);
    pair16(mx, x, y);
    mx = fmaxf(x, y);
    if constexpr (NU == 1) {                                 // a block's 32 dims lie on two waves
        __syncthreads();
        amx[wave][tk] = mx;
        __syncthreads();
        mx = fmaxf(mx, amx[wave ^ 1][tk]);
    }
    if (!mine) return;
    const float inv = mx > 0.f ? __fdiv_rn(127.f, mx) : 0.f;
    const int e0 = h * HD + d0 + 4 * NU * kk;
#pragma unroll
    for (int u = 0; u < NU; u++) {
        uint32_t w = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) w |= (uint32_t)(__float2int_rn(__fmul_rn(out[4 * u + i], inv)) & 0xFF) << (8 * i);
        *reinterpret_cast<uint32_t*>(xq + bx_at(nb, tok, e0 >> 5, (e0 & 31) + 4 * u)) = w;
    }
    if ((e0 & 31) == 0) xd[bd_at(nb, tok, e0 >> 5)] = f2h_bits(__fdiv_rn(mx, 127.f));
}

// split merge of (token, head) by one wave (lane = dims 64e + lane), then int8 blocks into
// the O GEMM's operand
template <int HD>
__global__ __launch_bounds__(kBThreads) void k_bcomb(const float* rec, int NH, int m, int p0, int nsp, int nb, int8_t* xq,
                                                     uint32_t* xd) {
    constexpr int DPL = HD / 64;
    const int item = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (item >= m * NH) return;
    const int t = item / NH, h = item - t * NH;
    const int ns = (p0 + t) / (kAttnChunk * kAttnSplit) + 1;
    const float* r = rec + (size_t)item * nsp * (HD + 4);
    float den, o[DPL];
    if (ns == 1) {
        den = r[HD + 1];
#pragma unroll
        for (int e = 0; e < DPL; e++) o[e] = r[64 * e + lane];
    } else {
        float Mx = -__builtin_inff();
        for (int s = lane; s < ns; s += 64) Mx = fmaxf(Mx, r[(size_t)s * (HD + 4) + HD]);
        Mx = wave_max(Mx);
        den = 0.f;
#pragma unroll
        for (int e = 0; e < DPL; e++) o[e] = 0.f;
        for (int s = 0; s < ns; s++) {
            const float* q = r + (size_t)s * (HD + 4);
            const float w = mi_expf(__fsub_rn(q[HD], Mx));
            den = __fmaf_rn(q[HD + 1], w, den);
#pragma unroll
            for (int e = 0; e < DPL; e++) o[e] = __fmaf_rn(q[64 * e + lane], w, o[e]);
        }
    }
#pragma unroll
    for (int e = 0; e < DPL; e++) {
        int q, s8;
        float d;
        quant32_vals(__fdiv_rn(o[e], den), q, d, s8);
        const int el = h * HD + 64 * e + lane;
        const uint32_t b = (uint32_t)(q & 0xFF);
        const uint32_t wd = b | (__shfl_down(b, 1) << 8) | (__shfl_down(b, 2) << 16) | (__shfl_down(b, 3) << 24);
        if ((lane & 3) == 0) *reinterpret_cast<uint32_t*>(xq + bx_at(nb, t, el >> 5, el & 31)) = wd;
        if ((lane & 31) == 0) xd[bd_at(nb, t, el >> 5)] = f2h_bits(d);
    }
}

// ------------------------------------------------------------------ host side
template <int EPI>
static void gemm(const PMat& W, const int8_t* xq, const uint32_t* xd, int ntt, int nseg, float* out, int ostride, int8_t* oq,
                 uint32_t* od, hipStream_t s) {
    const int grid = 8 * (((W.rows >> 6) + 7) / 8) * ntt * nseg;
    if (W.cb == 8) LAUNCH((k_bgemm<8, EPI>), grid, kGThreads, s, W, xq, xd, ntt, nseg, out, ostride, oq, od);
    else LAUNCH((k_bgemm<4, EPI>), grid, kGThreads, s, W, xq, xd, ntt, nseg, out, ostride, oq, od);
}
template <int EPI>
static void gemm_w(const PMat& W, const int8_t* xq, const uint32_t* xd, int ntt, int8_t* oq, uint32_t* od, float4* cand,
                   hipStream_t s) {
    const int grid = 8 * (((W.rows >> 6) + 7) / 8) * ((ntt + 1) / 2);
    if (W.cb == 8) LAUNCH((k_bgemm_w<8, EPI>), grid, kBThreads, s, W, xq, xd, ntt, oq, od, cand);
    else LAUNCH((k_bgemm_w<4, EPI>), grid, kBThreads, s, W, xq, xd, ntt, oq, od, cand);
}

void launch_bulk(const DModel& M, const DLayer* layers, const BulkBuf& B, int p0, int m, bool all, bool last,
                 hipStream_t s) {
    const int E = M.E, ntt = (m + 63) / 64, nbE = E / 32;
    const int nsp = (p0 + m - 1) / (kAttnChunk * kAttnSplit) + 1;
    auto norm = [&](const float* w, const float* emb, int ks) {
        LAUNCH(k_bnorm, m, kBThreads, s, E, M.eps, w, B.h, emb, M.tokbuf + p0, B.dpart, ks, ntt * 64, B.xq, B.xd);
    };
    int ks = 0;                                              // down partials the next norm adds
    for (int l = 0; l < M.NL; l++) {
        const DLayer& L = layers[l];
        norm(L.an, l == 0 ? M.emb : nullptr, ks);
        gemm<BE_PART>(L.qkv, B.xq, B.xd, ntt, 1, B.qkv, 0, nullptr, nullptr, s);
        const size_t kv = (size_t)l * M.NKV * M.maxseq * M.HD;
        auto attn = [&](auto hd) {
            constexpr int HD = decltype(hd)::value;
            const size_t threads = (size_t)m * (M.NH + 2 * M.NKV) * (HD / 2);
            LAUNCH((k_brope<HD>), (unsigned)((threads + kBThreads - 1) / kBThreads), kBThreads, s, B.qkv, L.bqkv, M.rope, M.NH,
                   M.NKV, M.QKV, m, p0, M.maxseq, M.kc + kv, M.vc + kv);
            // all tokens at once, or as many as the split records have room for: q, K/V and the
            // operand are addressed from the launch's first token
            const int per = nsp > 1 ? bulk_attn_tokens(B.rec_floats, M.NH, HD, nsp, m) : m;
            for (int t = 0; t < m; t += per) {
                const int mt = std::min(per, m - t), ns = (p0 + t + mt - 1) / (kAttnChunk * kAttnSplit) + 1;
                int8_t* xq = B.xq + bx_at(nbE, t, 0, 0);
                uint32_t* xd = B.xd + bd_at(nbE, t, 0);
                LAUNCH((k_battn<HD>), (unsigned)(M.NH * ns * ((mt + kAT - 1) / kAT)), kAThreads, s, B.qkv + (size_t)t * M.QKV,
                       M.QKV, M.kc + kv, M.vc + kv, M.NH, M.G, mt, p0 + t, M.maxseq, ns, M.scale, B.rec, nbE, xq, xd);
                if (ns > 1)
                    LAUNCH((k_bcomb<HD>), (mt * M.NH + 3) / 4, kBThreads, s, B.rec, M.NH, mt, p0 + t, ns, nbE, xq, xd);
            }
        };
        if (M.HD == 64) attn(std::integral_constant<int, 64>());
        else attn(std::integral_constant<int, 128>());
        gemm<BE_RES>(L.o, B.xq, B.xd, ntt, 1, B.h, 0, nullptr, nullptr, s);
        norm(L.fn, nullptr, 0);
        // K split while the 64 x 64 tiles are about one per CU (us, split / whole K, at 152 and 280
        // row groups: 64 tokens 7.4 / 12.0 and 18.1 / 21.1; 128 tokens 13.9 / 13.0 and 28.6 / 24.3;
        // 512 tokens 32.5 / 26.9 and 73.5 / 56.5); not measured at the 344 of the 3B shape
        if ((L.gu.rows >> 6) * ntt <= kBulkWgs) gemm<BE_GU>(L.gu, B.xq, B.xd, ntt, 1, nullptr, 0, B.aq, B.ad, s);
        else gemm_w<BE_GU>(L.gu, B.xq, B.xd, ntt, B.aq, B.ad, nullptr, s);
        ks = ntt * 64 <= kBulkSplitM ? L.d.ks : 0;
        if (ks) gemm<BE_PART>(L.d, B.aq, B.ad, ntt, ks, B.dpart, ntt * 64 * E, nullptr, nullptr, s);
        else gemm<BE_RES>(L.d, B.aq, B.ad, ntt, 1, B.h, 0, nullptr, nullptr, s);
    }
    if (!all && !last) return;
    norm(M.out_norm, nullptr, ks);
    // predictions of every token, or of the last one
    if (all)
        gemm_w<BE_LM>(M.lm, B.xq, B.xd, ntt, nullptr, nullptr, B.cand, s);
    else
        launch_lm_token(M.lm, B.xq, B.xd, m - 1, B.cand, s);
    LAUNCH(k_bargmax, all ? m : 1, kBThreads, s, B.cand, M.V / 64, M.V, p0 + (all ? 0 : m - 1), M.out_tok, M.out_margin);
}

}  // namespace mi
