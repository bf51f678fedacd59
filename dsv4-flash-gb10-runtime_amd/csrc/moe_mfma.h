// moe_mfma.h — the routed layer's matrix-core kernels as the decode entries
// (mxfp4_grouped_gemv.hip) call them; defined in mxfp4_moe_prefill.hip. Not
// part of the C ABI.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace dsv4 {

// The expert-grouped pairs of a decode batch, as moe_route_kernel leaves them:
// slot u < *n_unique is expert uexp[u] with pairs off[u] .. off[u + 1] - 1, and
// pair p is token pair_tok[p] with weight pair_w[p].
struct SlotTables {
    const int32_t* n_unique;
    const int32_t* uexp;
    const int32_t* off;
    const int32_t* pair_tok;
    const float* pair_w;
    int n_slots;                 // capacity of the slot tables
    int n_pairs;                 // capacity of the pair tables (tokens * topk)
    int n_experts;
};

// Shapes and alignments that each stage takes (tokens <= 64).
bool mfma_swiglu_ok(int K, int hidden, const void* x, const void* w1, const void* w3, const void* s1,
                    const void* s3);
bool mfma_down_ok(int hidden, int out_dim, const void* M, const void* w2, const void* s2);

// M[p, :] = bf16(silu(W1_e x_t) * (W3_e x_t)) for every pair p.
hipError_t mfma_swiglu(const uint16_t* x, const uint8_t* w1, const uint8_t* w3, const uint8_t* s1,
                       const uint8_t* s3, int T, int K, int hidden, const SlotTables& st, uint16_t* M,
                       hipStream_t stream);

// out[t, :] = bf16(sum over the pairs p of t of w_p * (W2_e M_p)).
hipError_t mfma_down(const uint16_t* M, const uint8_t* w2, const uint8_t* s2, int T, int hidden, int out_dim,
                     const SlotTables& st, uint16_t* out, hipStream_t stream);

}  // namespace dsv4

// Which stages of a decode batch with 16-byte aligned operands run on the
// matrix cores: bit 0 stage A, bit 1 stage B (so that the tests can name the
// path that a case takes; needs no GPU).
extern "C" int mxfp4_moe_decode_stages(int T, int topk, int n_experts, int K_in, int hidden, int out_dim);

// Whether a prefill chunk with 16-byte aligned scales takes the wide tiles
// (likewise).
extern "C" int mxfp4_moe_prefill_wide(int T, int topk, int n_experts, int K_in, int hidden, int out_dim);
