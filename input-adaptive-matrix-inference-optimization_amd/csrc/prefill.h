// Launchers of the batched prefill: the layer kernels over a chunk of prompt
// tokens (no argument checks: the model calls them on its own buffers).
#pragma once

#include "internal.h"

namespace iam {

constexpr int kPfGroup = 16;        // tokens per group: one wave's accumulators
constexpr int kPfMaxTokens = 512;   // tokens per chunk at most

inline int pf_groups(int tokens) { return (tokens + kPfGroup - 1) / kPfGroup; }

// Per-input selections of a product's tokens, in groups of kPfGroup:
// count[(group*in + i)*16 + token] = the ranks selected, when they are the
// first ones (0x80 added to token 0's when some token's are not), and the
// ranks themselves as 16-bit masks.
struct PfSelection {
    uint8_t* count;
    uint16_t* mask;
};

// The cutoffs of n matrices for each token: x is [tokens][ld], cut
// [n][kPfMaxTokens]; hints[j] (or null) takes the last token's.
int pf_cutoffs(Ctx* c, int n, const uint16_t* const* probes, const float* x, int ld, int tokens, int quantile, float* cut,
               float* const* hints);

// The selections of n matrices of the same inputs, and the inputs as fp64,
// xd[(group*in + i)*16 + token] (0 past the last token).  label: the
// matrices' counter block.
int pf_select(Ctx* c, int n, const iam_bucket_matrix* mats, const float* x, int ld, int tokens, int in_dim,
              const float* cut, int sel_block, int label, const PfSelection* sel, double* xd);

// The products: part[split][token][16 * the matrices' columns, one after the
// other] (16 * pf_groups(tokens) token rows), splits chosen by pf_splits.
int pf_splits(int n, const iam_bucket_matrix* mats, int tokens, int in_dim);
int pf_products(Ctx* c, int n, const iam_bucket_matrix* mats, int tokens, int in_dim, int splits, const PfSelection* sel,
                const double* xd, double* part);

// partial sums [splits][rows][width]
struct PfPart {
    const double* p = nullptr;
    int splits = 0;
    int rows = 0;
    int width = 0;
};
// h = the embedding rows of tokens (times scale, when set), or h + the sums;
// then x = rmsnorm(h) * gain
int pf_embed_norm(Ctx* c, const uint16_t* embed, const int* tokens, int vocab, const float* scale, float* h,
                  const uint16_t* gain, int dim, float eps, int n_tokens, float* x);
int pf_res_norm(Ctx* c, const PfPart& part, float* h, const uint16_t* gain, int dim, float eps, int n_tokens, float* x);
// RoPE of q (to q_rot [tokens][dim]) and k, and the KV append at positions pos0 ..
int pf_rope_append(Ctx* c, const PfPart& qkv, const float* rope, int pos0, int n_heads, int n_kv, int n_tokens,
                   float* q_rot, uint16_t* kc, uint16_t* vc);
// s[token][ffn] = up * gate / (1 + exp(-gate)) of the sums gate | up
int pf_silu(Ctx* c, const PfPart& gu, int ffn, int n_tokens, float* s);
// hist[pos0 + t + 1] = the first maximum of token t's sums (logits)
int pf_pick(Ctx* c, const PfPart& logits, int pos0, int n_tokens, int* hist, int hist_len);

}  // namespace iam
