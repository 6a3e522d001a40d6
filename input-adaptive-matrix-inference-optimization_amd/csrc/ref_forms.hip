// The reference's own fp32 forms, for callers that need its numbers rather
// than the decode step's faster ones:
//   - its KV cache layout (K and V repeated to every query head, fp32
//     [max_ctx][n_heads][head_dim] per layer, model.hpp:97-98) with the
//     RoPE + append of attention.hpp:172-189 / :281-309 and its fp32
//     attention (dotSetScore2, sum_of_exps32_mx, softmax_add32_mx,
//     sumScores32: aux.cl:204-225, :370-384, :497-540);
//   - its dense fp16 LM head, matmul16x32 (aux.cl:454-490, model.hpp:207-227).
// Every fp32 operation is a single IEEE-rounded one (no contraction), in the
// reference's order where that order is fixed; where the reference's order
// depends on scheduling (the float atomics of sum_of_exps32_mx) a fixed one
// is used.  The results then equal the oracle's restatement of the same
// order (exp excepted: the device's expf may differ from the C library's by
// an ulp).
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "internal.h"
#include "layer_ops.h"

namespace iam {

namespace {

__device__ __forceinline__ float f16(uint32_t bits) { return __half2float(__ushort_as_half((unsigned short)(bits & 0xffffu))); }

constexpr int kSplit = 64;        // positions per split of the fp32 attention
constexpr int kHD = 128;          // head dimension
constexpr int kDenseWG = 256;     // work-items per row of matmul16x32 (model.hpp:223-224)

}  // namespace

// ---------------------------------------------------------------- append ---
// RoPE of q (n_heads heads) and of k (n_kv heads), then the K row after RoPE
// and the V row of KV head h / rep stored for every query head h at the
// position (repeat4x32 + rope_mx + the cache copies).
__global__ void k_rope_kv_rep32(const float* __restrict__ q, const float* __restrict__ k,
                                const float* __restrict__ v, const float* __restrict__ table,
                                const int* __restrict__ pos_p, int n_heads, int n_kv, int max_ctx,
                                float* __restrict__ q_out, float* __restrict__ kc, float* __restrict__ vc)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    const int pos = *pos_p;
    if (pos < 0 || pos >= max_ctx) return;
    const int nq = n_heads * kHD;
    const int rep = n_heads / n_kv;
    const float* row = table + (size_t)pos * kHD;
    if (i < nq) {
        const int h = i / kHD, d = i - h * kHD;
        q_out[i] = rope_one(q + h * kHD, row, d, kHD / 2);
    } else if (i < 2 * nq) {
        const int j = i - nq;
        const int h = j / kHD, d = j - h * kHD;
        kc[(size_t)pos * nq + j] = rope_one(k + (h / rep) * kHD, row, d, kHD / 2);
    } else if (i < 3 * nq) {
        const int j = i - 2 * nq;
        const int h = j / kHD, d = j - h * kHD;
        vc[(size_t)pos * nq + j] = v[(h / rep) * kHD + d];
    }
}

// ------------------------------------------------------------- attention ---
// Pass 1, workgroup (head h, split j) of 4 waves: the score of each position
// t of the split (wave w takes positions t0 + w, t0 + w + 4, ...) as
// dotSetScore2 forms it -- lane l multiplies dimensions l and l + 64, adds
// the two (the tree's stride 64), and the strides 32 .. 1 follow as
// shuffles, so the sum is the reference's work-group tree -- divided by
// sqrt(128); e_t = exp(s_t) (no maximum subtracted) goes to e[h][t].  The
// split's sum of e in position order goes to ssum[h][j].  A wave holds its 16
// K rows at once and runs their trees side by side: with a row loaded, summed
// and finished before the next, the latencies added up (32 heads, 2047
// positions: 13.8 -> 10.3 us, 33.5 MB).
__global__ __launch_bounds__(256) void k_att32_score(const float* __restrict__ q, const float* __restrict__ kc,
                                                     const int* __restrict__ pos_p, int n_heads, int max_ctx,
                                                     float* __restrict__ e, float* __restrict__ ssum)
{
#pragma clang fp contract(off)
    __shared__ __align__(16) float se[kSplit];
    const int h = blockIdx.x, j = blockIdx.y;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int n_tok = min(*pos_p + 1, max_ctx);
    const int t0 = j * kSplit;
    const int nt = min(kSplit, n_tok - t0);
    if (nt <= 0) return;
    const float root = __fsqrt_rn((float)kHD);
    const float q0 = q[h * kHD + lane], q1 = q[h * kHD + 64 + lane];
    // the wave's positions' K rows all loaded before the first is used (past
    // the split: its last row again)
    constexpr int PW = kSplit / 4;
    float k0[PW], k1[PW];
#pragma unroll
    for (int u = 0; u < PW; u++) {
        const float* kr = kc + ((size_t)(t0 + min(w + 4 * u, nt - 1)) * n_heads + h) * kHD;
        k0[u] = kr[lane];
        k1[u] = kr[64 + lane];
    }
    // the trees of all positions side by side; lane u then holds position u's
    float a[PW], mine = 0.0f;
#pragma unroll
    for (int u = 0; u < PW; u++) a[u] = __fadd_rn(__fmul_rn(q0, k0[u]), __fmul_rn(q1, k1[u]));
#pragma unroll
    for (int st = 32; st > 0; st >>= 1)
#pragma unroll
        for (int u = 0; u < PW; u++) a[u] = __fadd_rn(a[u], __shfl_down(a[u], st, 64));
#pragma unroll
    for (int u = 0; u < PW; u++) {
        const float v = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(a[u])));
        if (lane == u) mine = v;
    }
    const int i = w + 4 * lane;
    if (lane < PW) {
        const float ev = i < nt ? expf(__fdiv_rn(mine, root)) : 0.0f;
        se[i] = ev;
        if (i < nt) e[(size_t)h * max_ctx + t0 + i] = ev;
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        float4 v[kSplit / 4];
#pragma unroll
        for (int u = 0; u < kSplit / 4; u++) v[u] = *reinterpret_cast<const float4*>(se + 4 * u);
        float s = 0.0f;   // past the split: + 0, which changes no sum of exponentials
#pragma unroll
        for (int u = 0; u < kSplit / 4; u++)
            s = __fadd_rn(__fadd_rn(__fadd_rn(__fadd_rn(s, v[u].x), v[u].y), v[u].z), v[u].w);
        ssum[(size_t)h * gridDim.y + j] = s;
    }
}

// 0 + p[0] + p[step] + ..., in order, 16 loads in flight
__device__ __forceinline__ float sum_in_order(const float* __restrict__ p, int step, int n)
{
    float s = 0.0f;
    for (int i = 0; i < n; i += 16) {
        float v[16];
#pragma unroll
        for (int u = 0; u < 16; u++) v[u] = p[(size_t)min(i + u, n - 1) * step];
#pragma unroll
        for (int u = 0; u < 16; u++)
            if (i + u < n) s = __fadd_rn(s, v[u]);
    }
    return s;
}

// Pass 2, workgroup (head h, split j), thread d: the total of the splits'
// sums in split order, p_t = e_t / total (softmax_add32_mx), and the split's
// sum of p_t * v_t[d] in position order (sumScores32's products) into
// part[h][j][d].  16 rows in flight, the first of them during the splits'
// sums (10.9 -> 9.2 us).
__global__ __launch_bounds__(kHD) void k_att32_pv(const float* __restrict__ vc, const int* __restrict__ pos_p,
                                                  int n_heads, int max_ctx, const float* __restrict__ e,
                                                  const float* __restrict__ ssum, float* __restrict__ part)
{
#pragma clang fp contract(off)
    __shared__ float sp[kSplit];
    const int h = blockIdx.x, j = blockIdx.y, d = threadIdx.x;
    const int n_tok = min(*pos_p + 1, max_ctx);
    const int t0 = j * kSplit;
    const int nt = min(kSplit, n_tok - t0);
    if (nt <= 0) return;
    const int ns = (n_tok + kSplit - 1) / kSplit;
    // the split's first V rows go out before the sums they wait for
    const float* vr = vc + ((size_t)t0 * n_heads + h) * kHD + d;
    const size_t step = (size_t)n_heads * kHD;
    constexpr int B = 16;   // rows in flight
    float v[B];
#pragma unroll
    for (int u = 0; u < B; u++) v[u] = vr[min(u, nt - 1) * step];
    const float total = sum_in_order(ssum + (size_t)h * gridDim.y, 1, ns);
    if (d < nt) sp[d] = __fdiv_rn(e[(size_t)h * max_ctx + t0 + d], total);
    __syncthreads();
    float acc = 0.0f;
    for (int i = 0; i < nt; i += B) {
        float c[B];
#pragma unroll
        for (int u = 0; u < B; u++) {
            c[u] = v[u];
            v[u] = vr[min(i + B + u, nt - 1) * step];
        }
        if (i + B <= nt) {
#pragma unroll
            for (int u = 0; u < B; u++) acc = __fadd_rn(acc, __fmul_rn(sp[i + u], c[u]));
        } else {
#pragma unroll
            for (int u = 0; u < B; u++)
                if (i + u < nt) acc = __fadd_rn(acc, __fmul_rn(sp[i + u], c[u]));
        }
    }
    part[((size_t)h * gridDim.y + j) * kHD + d] = acc;
}

// Pass 3, workgroup h, thread d: out[h][d] = the splits' sums in split order
// (9.1 us with a load at a time for 32 splits, 3.4 with 16 in flight).
__global__ __launch_bounds__(kHD) void k_att32_sum(const int* __restrict__ pos_p, int max_ctx, int nsplit,
                                                   const float* __restrict__ part, float* __restrict__ out)
{
#pragma clang fp contract(off)
    const int h = blockIdx.x, d = threadIdx.x;
    const int n_tok = min(*pos_p + 1, max_ctx);
    const int ns = n_tok > 0 ? (n_tok + kSplit - 1) / kSplit : 0;
    out[(size_t)h * kHD + d] = sum_in_order(part + (size_t)h * nsplit * kHD + d, kHD, ns);
}

// ----------------------------------------------------------------- dense ---
// matmul16x32 with 256 work-items per row: work-item l of a row sums the
// products of columns l, l + 256, ... in order, then the 256 partial sums
// go through the tree p[l] += p[l + stride], stride 128 .. 1.  Here one
// wave holds a row's 256 work-items, lane i the four l = 4i .. 4i + 3 (one
// 8-byte load per 256 columns); the tree's strides 128 .. 4 are shuffles
// between lanes 32 .. 1 apart, strides 2 and 1 stay in lane 0.  x is staged
// in LDS; each wave walks rows wave, wave + waves, ... two at a time, eight
// loads of a row in flight (32000 x 4096: 64.8 us with the loads the compiler
// left between the adds, 42 with these, 6.2 TB/s), and of a shorter row or
// rest its 4, 2 and 1 blocks together, the partial one's first (32000 x 1024
// and 1000: 32 and 33 us with a loop over single blocks behind the eights, 21
// where that loop stood alone, 16 and 19 with these).  5 waves a SIMD: one
// more in flight than the compiler's choice (45 us for 32000 x 4096).
constexpr int kDenseThreads = 256;
constexpr int kDenseMaxCols = 16384;

template <bool VEC>
__global__ __launch_bounds__(kDenseThreads, 5) void k_matmul16x32(const uint16_t* __restrict__ W,
                                                               const float* __restrict__ x, int rows, int cols,
                                                               float* __restrict__ out)
{
#pragma clang fp contract(off)
    extern __shared__ __align__(16) float sx[];   // x, cols floats
    for (int i = threadIdx.x; i < cols; i += kDenseThreads) sx[i] = x[i];
    __syncthreads();
    const int lane = threadIdx.x & 63;
    const int waves = gridDim.x * (kDenseThreads / 64);
    const int wv = blockIdx.x * (kDenseThreads / 64) + (threadIdx.x >> 6);
    const int nk = (cols + kDenseWG - 1) / kDenseWG;
    auto row_sums = [&](int r, float (&s)[4]) {
        const uint16_t* w = W + (size_t)r * cols;
#pragma unroll
        for (int c = 0; c < 4; c++) s[c] = 0.0f;
        int k = 0;
        // Whole columns blocks: 8 loads in flight a row, added in order, then
        // the 4, 2 and 1 of what is left; a partial block's load goes out
        // ahead of them all.
        if constexpr (VEC) {
            typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
            auto load = [&](int b) { return __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(w + b)); };
            auto add = [&](const u32x2& p, int b) {
                const float4 xv = *reinterpret_cast<const float4*>(sx + b);
                s[0] = __fadd_rn(s[0], __fmul_rn(f16(p.x), xv.x));
                s[1] = __fadd_rn(s[1], __fmul_rn(f16(p.x >> 16), xv.y));
                s[2] = __fadd_rn(s[2], __fmul_rn(f16(p.y), xv.z));
                s[3] = __fadd_rn(s[3], __fmul_rn(f16(p.y >> 16), xv.w));
            };
            auto blocks = [&](auto n_tag) {
                constexpr int N = decltype(n_tag)::value;
                u32x2 p[N];
#pragma unroll
                for (int u = 0; u < N; u++) p[u] = load((k + u) * kDenseWG + 4 * lane);
#pragma unroll
                for (int u = 0; u < N; u++) add(p[u], (k + u) * kDenseWG + 4 * lane);
                k += N;
            };
            const int whole = cols / kDenseWG, last = whole * kDenseWG + 4 * lane;
            u32x2 part{};
            if (last < cols) part = load(last);
            while (k + 8 <= whole) blocks(std::integral_constant<int, 8>{});
            if (k + 4 <= whole) blocks(std::integral_constant<int, 4>{});
            if (k + 2 <= whole) blocks(std::integral_constant<int, 2>{});
            if (k < whole) blocks(std::integral_constant<int, 1>{});
            if (last < cols) add(part, last);
            return;
        }
        for (; k < nk; k++) {
            const int b = k * kDenseWG + 4 * lane;
            uint32_t v[4];
#pragma unroll
            for (int c = 0; c < 4; c++) v[c] = b + c < cols ? (uint32_t)w[b + c] : 0u;
#pragma unroll
            for (int c = 0; c < 4; c++)
                if (b + c < cols) s[c] = __fadd_rn(s[c], __fmul_rn(f16(v[c]), sx[b + c]));
        }
    };
    auto tree = [&](float (&s)[4]) -> float {
#pragma unroll
        for (int st = 32; st > 0; st >>= 1) {
#pragma unroll
            for (int c = 0; c < 4; c++) s[c] = __fadd_rn(s[c], __shfl_down(s[c], st, 64));
        }
        const float a0 = __fadd_rn(s[0], s[2]), a1 = __fadd_rn(s[1], s[3]);
        return __fadd_rn(a0, a1);
    };
    for (int r = wv; r < rows; r += 2 * waves) {
        float s0[4], s1[4];
        const int r1 = r + waves;
        row_sums(r, s0);
        if (r1 < rows) row_sums(r1, s1);
        const float y0 = tree(s0);
        if (lane == 0) out[r] = y0;
        if (r1 < rows) {
            const float y1 = tree(s1);
            if (lane == 0) out[r1] = y1;
        }
    }
}

}  // namespace iam

using namespace iam;

int iam::ensure_attn32_scratch(Ctx* c, size_t floats)
{
    if (floats <= c->attn32_cap && c->attn32) return IAM_OK;
    if (c->capturing) return fail(IAM_E_STATE, "fp32 attention scratch growth during graph capture");
    if (c->attn32) IAM_TRY(ctx_free(c, c->attn32));
    c->attn32 = nullptr;
    c->attn32_cap = 0;
    IAM_TRY(ctx_alloc(c, floats * sizeof(float), (void**)&c->attn32));
    c->attn32_cap = floats;
    c->scratch_gen++;
    return IAM_OK;
}

int iam::matmul_f16_dense(Ctx* c, const uint16_t* W, const float* x, int rows, int cols, float* out)
{
    const int waves_needed = (rows + 1) / 2;
    const int blocks = std::max(1, std::min(2048, (waves_needed + 3) / 4));
    const bool vec = (cols % 4) == 0 && ((uintptr_t)W & 7) == 0;
    const size_t lds = (size_t)cols * sizeof(float);
    if (vec)
        return launch(c, "matmul16x32", k_matmul16x32<true>, dim3(blocks), dim3(kDenseThreads), lds, W, x, rows,
                      cols, out);
    return launch(c, "matmul16x32", k_matmul16x32<false>, dim3(blocks), dim3(kDenseThreads), lds, W, x, rows, cols,
                  out);
}

extern "C" {

int iam_rope_kv_append_f32(iam_ctx* c, const float* q, const float* k, const float* v, const float* table,
                           const int* pos, int n_heads, int n_kv, int head_dim, int max_ctx, float* q_out,
                           float* kc, float* vc)
{
    if (!c || !q || !k || !v || !table || !pos || !q_out || !kc || !vc)
        return fail(IAM_E_INVALID, "rope_kv_append_f32: null argument");
    IAM_REQUIRE(head_dim == kHD, "rope_kv_append_f32: head_dim must be 128");
    IAM_REQUIRE(n_kv > 0 && n_heads >= n_kv && n_heads % n_kv == 0 && max_ctx > 0,
                "rope_kv_append_f32: n_heads must be a positive multiple of n_kv");
    const size_t nq = (size_t)n_heads * kHD, nk = (size_t)n_kv * kHD;
    IAM_TRY(check_dev_range(c, q, nq * 4, "rope_kv_f32 q"));
    IAM_TRY(check_dev_range(c, k, nk * 4, "rope_kv_f32 k"));
    IAM_TRY(check_dev_range(c, v, nk * 4, "rope_kv_f32 v"));
    IAM_TRY(check_dev_range(c, q_out, nq * 4, "rope_kv_f32 q_out"));
    IAM_TRY(check_dev_range(c, table, (size_t)max_ctx * kHD * 4, "rope_kv_f32 table"));
    IAM_TRY(check_dev_range(c, kc, (size_t)max_ctx * nq * 4, "rope_kv_f32 kcache"));
    IAM_TRY(check_dev_range(c, vc, (size_t)max_ctx * nq * 4, "rope_kv_f32 vcache"));
    IAM_TRY(check_dev_range(c, pos, 4, "rope_kv_f32 pos"));
    const int n = 3 * (int)nq;
    return launch(c, "rope_kv_append_f32", k_rope_kv_rep32, dim3((n + 255) / 256), dim3(256), 0, q, k, v, table,
                  pos, n_heads, n_kv, max_ctx, q_out, kc, vc);
}

int iam_attention_decode_f32(iam_ctx* c, const float* q, const float* kc, const float* vc, const int* pos,
                             int n_heads, int head_dim, int max_ctx, float* out)
{
    if (!c || !q || !kc || !vc || !pos || !out) return fail(IAM_E_INVALID, "attention_f32: null argument");
    IAM_REQUIRE(head_dim == kHD, "attention_f32: head_dim must be 128");
    IAM_REQUIRE(n_heads >= 1 && n_heads <= 1024, "attention_f32: n_heads must be in [1, 1024]");
    IAM_REQUIRE(max_ctx >= 1 && max_ctx <= (1 << 20), "attention_f32: max_ctx must be in [1, 2^20]");
    const size_t nq = (size_t)n_heads * kHD;
    IAM_TRY(check_dev_range(c, q, nq * 4, "attention_f32 q"));
    IAM_TRY(check_dev_range(c, kc, (size_t)max_ctx * nq * 4, "attention_f32 kcache"));
    IAM_TRY(check_dev_range(c, vc, (size_t)max_ctx * nq * 4, "attention_f32 vcache"));
    IAM_TRY(check_dev_range(c, out, nq * 4, "attention_f32 out"));
    IAM_TRY(check_dev_range(c, pos, 4, "attention_f32 pos"));
    const int nsplit = (max_ctx + kSplit - 1) / kSplit;
    // scratch: e [n_heads][max_ctx], split sums [n_heads][nsplit], split partials [n_heads][nsplit][128]
    const size_t ne = (size_t)n_heads * max_ctx, ns = (size_t)n_heads * nsplit, np = ns * kHD;
    IAM_TRY(ensure_attn32_scratch(c, ne + ns + np));
    float* e = c->attn32;
    float* ssum = e + ne;
    float* part = ssum + ns;
    IAM_TRY(launch(c, "attention_f32.score", k_att32_score, dim3(n_heads, nsplit), dim3(256), 0, q, kc, pos, n_heads,
                   max_ctx, e, ssum));
    IAM_TRY(launch(c, "attention_f32.pv", k_att32_pv, dim3(n_heads, nsplit), dim3(kHD), 0, vc, pos, n_heads, max_ctx,
                   (const float*)e, (const float*)ssum, part));
    return launch(c, "attention_f32.sum", k_att32_sum, dim3(n_heads), dim3(kHD), 0, pos, max_ctx, nsplit,
                  (const float*)part, out);
}

int iam_matmul_f16_dense(iam_ctx* c, const uint16_t* W, const float* x, int rows, int cols, float* out)
{
    if (!c || !W || !x || !out) return fail(IAM_E_INVALID, "matmul_f16_dense: null argument");
    IAM_REQUIRE(rows >= 1 && cols >= 1 && cols <= kDenseMaxCols, "matmul_f16_dense: rows >= 1, 1 <= cols <= 16384");
    IAM_TRY(check_dev_range(c, W, (size_t)rows * cols * 2, "matmul_f16_dense W"));
    IAM_TRY(check_dev_range(c, x, (size_t)cols * 4, "matmul_f16_dense x"));
    IAM_TRY(check_dev_range(c, out, (size_t)rows * 4, "matmul_f16_dense out"));
    return matmul_f16_dense(c, W, x, rows, cols, out);
}

}  // extern "C"
