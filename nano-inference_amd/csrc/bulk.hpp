// bulk.hpp -- prompt panels: up to kBulkM consecutive tokens through every layer at once
// (bulk.hip). Used by mi_prefill and mi_teacher; results equal one step per token bit for
// bit.
#pragma once
#include "kernels.hpp"

#include <cstddef>

namespace mi {

constexpr int kBulkM = 2048;       // tokens of one panel, a multiple of 64. 1025 tokens in panels of 512 / 1024 /
                                   // 2048: 12.9 / 10.3 / 8.7 ms, 3001: 35.7 / 30.8 / 29.9 (1.5B shape): whole rounds
                                   // of workgroups and fewer launches
// Up to 8 tokens one multi-token step is faster: 1.41 ms on the 1.5B shape and 0.98 on the 0.5B
// one against 1.95 and 1.20 for a panel; 9 tokens take a second step: 2.3 and 1.5.
constexpr int kBulkMin = 9;
// Up to this many tokens the down GEMM runs one workgroup per K segment: its 64 x 64 tiles alone
// are too few for the CUs. Whole prefill, split / not, ms: 1.5B shape 129 tokens 2.85 / 3.24,
// 256 3.16 / 3.37, 257 3.56 / 3.62, 321 3.85 / 3.73, 512 4.85 / 4.36; 0.5B shape 1.69 / 1.74,
// 1.76 / 1.80, 1.94 / 1.85, 2.13 / 1.93, 2.62 / 2.28.
constexpr int kBulkSplitM = 256;
// Attention split records of one launch: they grow with the context (2048 tokens over a 32768-token
// context of the 1.5B shape: 415 MB). They live in the memory of the buffers that are idle
// during attention and, past that, in no more than this or a quarter of the K/V cache; where
// that holds fewer tokens than the panel has, its attention goes out in several launches
// (bulk_attn_tokens). 1.5B shape, ms per prompt of 8192 / 20000 / 32000 tokens: all at once
// 120.2 / 548.5 / 1287.7, as here 120.2 / 548.0 / 1292.2, in 78 MB 121.3 / 558.2 / 1322.5 (each launch
// ends in a round of workgroups that empties the chip).
constexpr size_t kBulkRecFloats = size_t(16) << 20;

// Work buffers of a panel (device memory, one block kept by the engine). Int8 activations of an
// nb-block vector per token are stored as the GEMM's MFMA operand: 32-token tiles, per tile
// and block 64 lanes x 16 codes (lane l: token l % 32, elements 16 (l / 32) .. + 15), with
// the block scales (fp16 bits, a word each) [tile][nb][32] beside them.
struct BulkBuf {                   // M: the longest panel, kBulkM or the whole context if that is shorter
    float* h;                      // [M][E] residual
    int8_t* xq;                    // [M/32][E/32][64][16]
    uint32_t* xd;                  // [M/32][E/32][32]
    float* qkv;                    // [M][QKV] projections, then q rotated in place
    int8_t* aq;                    // [M/32][FF/32][64][16] gate/up output
    uint32_t* ad;                  // [M/32][FF/32][32]
    float* dpart;                  // [ks of down][the panel's tokens, whole tiles][E]
    float4* cand;                  // [M][V/64] argmax candidates
    float* rec;                    // [tokens of one launch][NH][splits][HD + 4] attention split records, over aq,
    size_t rec_floats;             // ad, dpart and cand: nothing in them outlives a layer's start
};
// element offset of (token t, block b, element e of the block) in an operand buffer
__host__ __device__ __forceinline__ size_t bx_at(int nb, int t, int b, int e) {
    return ((((size_t)(t >> 5) * nb + b) * 64 + (e >> 4) * 32 + (t & 31)) << 4) + (e & 15);
}
__host__ __device__ __forceinline__ size_t bd_at(int nb, int t, int b) { return ((size_t)(t >> 5) * nb + b) * 32 + (t & 31); }

// lm_head of token t of a panel (kernels.hip): V/64 argmax candidates
void launch_lm_token(const PMat& W, const int8_t* xq, const uint32_t* xd, int t, float4* cand, hipStream_t s);

struct BulkSizes { size_t h, xq, xd, qkv, aq, ad, dpart, cand, rec; };   // in elements
// kv: elements of the K (or V) cache
BulkSizes bulk_sizes(int E, int FF, int NH, int HD, int QKV, int V, int maxseq, int ks_d, size_t kv);
// bytes of the block; base != nullptr: B's pointers into it
size_t bulk_bind(const BulkSizes& s, void* base, BulkBuf* B);
// tokens per panel of an n-token prompt: even panels, whole tiles
inline int bulk_panel_tokens(int n) {
    const int np = (n + kBulkM - 1) / kBulkM;
    return ((n + np - 1) / np + 63) / 64 * 64;
}
// tokens per attention launch of an m-token panel over nsp > 1 splits: whole 32-token tiles
// whose records fit rec_floats
int bulk_attn_tokens(size_t rec_floats, int NH, int HD, int nsp, int m);

// tokens tokbuf[p0 .. p0+m-1] (m <= kBulkM) at positions p0..: K/V appended to the cache.
// all: every position's prediction goes to out_tok / out_margin; otherwise, when last is
// set, only the last position's. layers: the host copy of M.layers.
void launch_bulk(const DModel& M, const DLayer* layers, const BulkBuf& B, int p0, int m, bool all, bool last,
                 hipStream_t s);

}  // namespace mi
