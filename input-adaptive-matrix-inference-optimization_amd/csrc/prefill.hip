// Prefill of several prompt tokens at a time.
//
// The decode step walks each token's selected rows, one launch chain per
// token; a prompt's tokens are independent within a layer except for
// attention, so here a layer's kernels run over a whole chunk of tokens, the
// weights are read once for all of them, and every output is the same sum of
// exact fp64 products of the same selected rows (in another order, far below
// an fp32 ulp).  Per product of the layer:
//   cutoffs     one workgroup per (token, matrix)
//   selection   thread = input: the tokens' selected ranks
//   products    k_pf_products, partial sums over splits of the inputs
// and the consumer adds the splits' sums in order.
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <type_traits>

#include "layer_ops.h"
#include "prefill.h"
#include "wave.h"

namespace iam {

namespace {

__device__ __forceinline__ float h2f(uint32_t b) { return __half2float(__ushort_as_half((unsigned short)(b & 0xffffu))); }

// a kernel argument's memory as constant: uniform loads from it are scalar
template <typename T>
using const_ptr = const __attribute__((address_space(4))) T*;
template <typename T>
__device__ __forceinline__ const_ptr<T> as_const(const T* p)
{
    return (const_ptr<T>)(uintptr_t)p;
}

}  // namespace

// ------------------------------------------------------------- selection ---
// prepareDispatch's rule (bucketMul.cl:351-386) for 16 tokens: thread = input
// i of all of them, its 16 ranks' stats read once.  A rank is selected iff
// 1e5 * |x * stat| >= cutoff in fp32 (NaN never is); block mode as the walk's.
// The stats of a converted matrix fall with the rank, so the selected ranks
// are the first `count`; any others are flagged and taken from the masks.
struct PfSelectArgs {
    const uint16_t* stats[kMaxMulti];   // compact: one value per row
    uint8_t* count[kMaxMulti];
    uint16_t* mask[kMaxMulti];
    int cols[kMaxMulti];
    const float* x;
    double* xd;
    const float* cut;                   // [n][kPfMaxTokens]
    unsigned long long* counters;
    int ld, tokens, in_dim, blk;
};

__global__ __launch_bounds__(256) void k_pf_select(PfSelectArgs a)
{
#pragma clang fp contract(off)
    const int i = blockIdx.x * 256 + threadIdx.x, g = blockIdx.y, m = blockIdx.z;
    const bool ok = i < a.in_dim;
    const int ic = min(i, a.in_dim - 1);
    float st[16];
    {
        const uint4* s = reinterpret_cast<const uint4*>(a.stats[m]) + 2 * (size_t)ic;
        const uint4 lo = s[0], hi = s[1];
        const uint32_t w[8] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
#pragma unroll
        for (int k = 0; k < 16; k++) st[k] = h2f(w[k >> 1] >> (16 * (k & 1)));
    }
    uint32_t cnt[4] = {0u, 0u, 0u, 0u}, msk[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    double xv[16];
    bool irregular = false;
    int rows = 0;
#pragma unroll
    for (int t = 0; t < kPfGroup; t++) {
        const int tt = g * kPfGroup + t;
        uint32_t sel = 0;
        float xi = 0.0f;
        if (tt < a.tokens) {
            xi = a.x[(size_t)tt * a.ld + ic];
            const float cut = a.cut[m * kPfMaxTokens + tt];
#pragma unroll
            for (int k = 0; k < 16; k++) {
                const float imp = __fmul_rn(100000.0f, fabsf(__fmul_rn(xi, st[k])));   // bucketMul.cl:17, :380
                if (imp >= cut) sel |= 1u << k;
            }
            if (!ok) sel = 0u;
            for (int o = 1; o < a.blk; o <<= 1) sel |= (uint32_t)__shfl_xor((int)sel, o, 64);
            if (!ok) sel = 0u;
        }
        const int c = __popc(sel);
        irregular |= (sel & (sel + 1u)) != 0u;
        rows += c;
        cnt[t >> 2] |= (uint32_t)c << (8 * (t & 3));
        msk[t >> 1] |= sel << (16 * (t & 1));
        xv[t] = (double)xi;
    }
    if (irregular) cnt[0] |= 0x80u;
    if (ok) {
        const size_t at = (size_t)g * a.in_dim + i;
        reinterpret_cast<uint4*>(a.count[m])[at] = make_uint4(cnt[0], cnt[1], cnt[2], cnt[3]);
        uint4* mp = reinterpret_cast<uint4*>(a.mask[m]) + 2 * at;
        mp[0] = make_uint4(msk[0], msk[1], msk[2], msk[3]);
        mp[1] = make_uint4(msk[4], msk[5], msk[6], msk[7]);
        if (m == 0) {
            double2* xp = reinterpret_cast<double2*>(a.xd) + 8 * at;
#pragma unroll
            for (int t = 0; t < 8; t++) xp[t] = make_double2(xv[2 * t], xv[2 * t + 1]);
        }
    }
    if (a.counters) {   // as the walk counts: bytes, rows, matrices
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) rows += __shfl_xor(rows, o, 64);
        if ((threadIdx.x & 63) == 0) {
            unsigned long long* cr = a.counters + (blockIdx.x % kCounterLanes) * 4;
            atomicAdd(cr + 0, (unsigned long long)rows * (unsigned long long)a.cols[m] * 2ull);
            atomicAdd(cr + 1, (unsigned long long)rows);
            if (blockIdx.x == 0 && threadIdx.x == 0)
                atomicAdd(cr + 2, (unsigned long long)min(kPfGroup, a.tokens - g * kPfGroup));
        }
    }
}

int pf_select(Ctx* c, int n, const iam_bucket_matrix* mats, const float* x, int ld, int tokens, int in_dim,
              const float* cut, int sel_block, int label, const PfSelection* sel, double* xd)
{
    PfSelectArgs a{};
    for (int j = 0; j < n; j++) {
        a.stats[j] = mats[j].stats;
        a.count[j] = sel[j].count;
        a.mask[j] = sel[j].mask;
        a.cols[j] = mats[j].bucket_cols;
    }
    a.x = x;
    a.xd = xd;
    a.cut = cut;
    a.counters = c->counting ? c->counters + (size_t)label * kCounterLanes * 4 : nullptr;
    a.ld = ld;
    a.tokens = tokens;
    a.in_dim = in_dim;
    a.blk = sel_block;
    return launch(c, "prefill.select", k_pf_select, dim3((in_dim + 255) / 256, pf_groups(tokens), n), dim3(256), 0, a);
}

// -------------------------------------------------------------- products ---
// y[t][o] += x[t][i] * w for every input i and output o whose weight's rank is
// among the ranks token t selected for i.  Each of the 16 outputs of a bucket
// has one weight of every input, so a workgroup of 4 waves takes 16 columns
// (256 outputs), lays 16 inputs' weights out by output in LDS (the weight as
// fp32, exact, its rank in the free low bits), and each wave multiplies them
// for 16 tokens, accumulators in registers: lane = OPL consecutive outputs,
// the tokens' x and counts in scalar registers, one compare and one fp64 fma
// (exact product, one rounding) per weight and token, the fma under the
// compare's mask.  Waves: WT token groups x 4 / WT quarters of the outputs.
//
// 389 tokens through 8 layers (4096 wide, FFN 14336) and the LM head at effort
// 0.25: 212.4 ms by steps, 67.4 ms by this; at effort 1.0 four layers of 130
// tokens 65.6 -> 13.2 ms.  The time does not depend on the effort: the
// unselected weights' compare and masked fma are issued too.  Taking only the
// selected ones as the walk does, with LDS atomics (6 a clock and CU), would
// be 46 ms at effort 0.25 at the least, and four times that at effort 1.0.
// What bounds it: compare, fma and the write of exec take 11.1 clocks of a
// SIMD in a loop of nothing else (the fma alone 5-6), here 13-14 with the
// staging and the waits.  Two selections more tried: compares into scalar
// pairs and exec moved from those, 12.3 clocks; compare, select and fma, 15.3.
// The scalar loads set the pace with less ahead than one input: loaded where
// they are used 116 ms, half an input ahead 90, one input ahead 79 (all with
// the split of 25 token groups in 7 workgroup rows; 67 with 24 in 6).
//
// A bucket whose 16 position bits are not a permutation, and an input some
// token's selected ranks of which are not the first ones, are added row by
// row from the codes and the masks instead (slow_input).
struct PfGemmArgs {
    const uint16_t* W[kMaxMulti];
    const uint8_t* count[kMaxMulti];
    const uint16_t* mask[kMaxMulti];
    int cols[kMaxMulti];
    int ofs[kMaxMulti];        // the matrix's first output in a row of part
    int first[kMaxMulti];      // its first tile
    int n, tiles;
    const double* xd;
    double* part;
    int in_dim, groups, token_blocks, per;   // inputs per split (a multiple of 16)
    int width;
};

constexpr int kPfInputs = 16;                 // inputs staged at a time
constexpr int kPfTile = 256;                  // outputs per workgroup
// partial sums of a chunk: splits * token rows at most (8 splits always allowed)
constexpr int kPfMaxPartRows = 3072;

// acc += x * w in the lanes whose rank is below n; exec is full before and
// after (volatile: in order with the pins of the loads, below)
__device__ __forceinline__ void fma_below(double& acc, double w, uint32_t rank, double x, uint32_t n)
{
    asm volatile("v_cmpx_gt_u32_e32 vcc, %3, %4\n\tv_fma_f64 %0, %1, %2, %0\n\ts_mov_b64 exec, -1"
                 : "+v"(acc)
                 : "s"(x), "v"(w), "s"(n), "v"(rank)
                 : "vcc");
}

// A vector instruction's write of exec wants 4 wait states before a lane read
// or write (5 before a DPP operand).  The compiler sees no such write in the
// asm, and it spills scalars with lane writes.  This stands after a run of
// fma_below; within the run nothing but scalar arithmetic may fall between
// them, which the source cannot say: tests/test_prefill_asm.py reads the
// assembly for it.
__device__ __forceinline__ void exec_settled() { asm volatile("s_nop 3"); }

template <int WT>
__global__ __launch_bounds__(256, 3) void k_pf_products(PfGemmArgs a)
{
    constexpr int OPL = WT;   // outputs per lane
    static_assert(WT == 1 || WT == 2 || WT == 4, "token groups per workgroup");
    __shared__ __align__(16) uint32_t s_w[2][kPfInputs][kPfTile];
    __shared__ uint32_t s_bad[3];   // staged inputs with a bucket that is no permutation, by turns
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    // token blocks of one tile next to each other (they share its weights in
    // one XCD's L2), then the tiles, then the splits
    const int b = xcd_remap((int)blockIdx.x, (int)gridDim.x);
    const int tb = b % a.token_blocks;
    const int tile_all = (b / a.token_blocks) % a.tiles;
    const int split = b / (a.token_blocks * a.tiles);
    const int m = a.n > 2 && tile_all >= a.first[2] ? 2 : a.n > 1 && tile_all >= a.first[1] ? 1 : 0;
    const int tile = tile_all - a.first[m];
    const int C = a.cols[m];
    const uint16_t* W = a.W[m];
    const int k0 = split * a.per, k1 = min(a.in_dim, k0 + a.per);
    const int g = tb * WT + wave % WT;
    const int o_lane = (wave / WT) * (64 * OPL) + lane * OPL;   // first output in the tile
    const bool active = g < a.groups;
    const int gc = min(g, a.groups - 1);
    const const_ptr<double> xd = as_const(a.xd) + (size_t)gc * a.in_dim * kPfGroup;
    const const_ptr<uint32_t> cnt = as_const(reinterpret_cast<const uint32_t*>(a.count[m])) + (size_t)gc * a.in_dim * 4;
    const const_ptr<uint32_t> msk = as_const(reinterpret_cast<const uint32_t*>(a.mask[m])) + (size_t)gc * a.in_dim * 8;

    double acc[kPfGroup][OPL];
#pragma unroll
    for (int t = 0; t < kPfGroup; t++)
#pragma unroll
        for (int o = 0; o < OPL; o++) acc[t][o] = 0.0;

    // staging: thread (input, eight ranks, column pair), a 4-byte load (at any
    // 2-byte boundary) per rank; a pair past the last column starts one earlier
    const int si = tid >> 4, sr = (tid & 8) ? 8 : 0, sc = 2 * (tid & 7);
    const int scol = tile * 16 + sc;
    const int lcol = max(0, min(scol, C - 2));
    const uint16_t* sp = W + ((size_t)si * 16 + sr) * C + lcol;
    uint32_t code[8];
    auto fetch = [&](int k) {
        const uint16_t* p = sp + (size_t)min(k, k1 - kPfInputs) * 16 * C;
        typedef uint32_t u32u __attribute__((aligned(2)));
        if (C > 1) {
#pragma unroll
            for (int r = 0; r < 8; r++) code[r] = *reinterpret_cast<const u32u*>(p + (size_t)r * C);
        } else {
#pragma unroll
            for (int r = 0; r < 8; r++) code[r] = p[(size_t)r * C];
        }
    };
    const int shift = 16 * min(scol - lcol, 1);   // the pair's first code in an earlier start's word
    // the row-by-row form for one input: every code of the lane's column
    auto slow_input = [&](int i) {
        const int col = tile * 16 + (o_lane >> 4);
        const uint16_t* p = W + (size_t)i * 16 * C + min(col, C - 1);
#pragma unroll 1
        for (int r = 0; r < 16; r++) {
            const uint32_t cd = p[(size_t)r * C];
            const uint32_t at = (cd & 15u) - (uint32_t)(o_lane & 15);
            const double w = (double)h2f(cd);
#pragma unroll
            for (int t = 0; t < kPfGroup; t++) {
                const uint32_t ranks = msk[(size_t)i * 8 + (t >> 1)] >> (16 * (t & 1));
                const uint32_t out = (ranks >> r) & 1u ? at : 16u;   // the lane's output of this weight, if selected
#pragma unroll
                for (int o = 0; o < OPL; o++)
                    fma_below(acc[t][o], w, out == (uint32_t)o ? 0u : 1u, xd[(size_t)i * kPfGroup + t], 1u);
            }
            exec_settled();
        }
    };
    // An input's scalar loads (its tokens' x and counts), issued one input
    // ahead: each wave reads other ones, so they come from L2.  `pin` is their
    // first use: the wait stands there, before the next ones go out.
    auto load_input = [&](int i, double (&x)[kPfGroup], uint32_t (&n)[4]) {
#pragma unroll
        for (int t = 0; t < kPfGroup; t++) x[t] = xd[(size_t)i * kPfGroup + t];
#pragma unroll
        for (int q = 0; q < 4; q++) n[q] = cnt[(size_t)i * 4 + q];
    };
    if (tid < 3) s_bad[tid] = 0u;
    fetch(k0);
    double xa[kPfGroup], xb[kPfGroup];
    uint32_t na[4], nb[4], word[OPL], slow = 0;
    load_input(k0, xa, na);
    __syncthreads();
    // One barrier per staging: the waves are all past the products of the
    // staging before when it opens, so the next one may overwrite that one's
    // weights, and its flags may be cleared (the one after the next uses them).
    int buf = 0, turn = 0;
    // input k + ii: x and n in hand, the next input's go to xn and nn
    auto input = [&](int k, int ii, double (&x)[kPfGroup], uint32_t (&n)[4], double (&xn)[kPfGroup], uint32_t (&nn)[4]) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+s"(x[0]), "+s"(x[8]), "+s"(n[0]), "+v"(word[0]));
        __builtin_amdgcn_sched_barrier(0);
        load_input(min(k + ii + 1, k1 - 1), xn, nn);
        uint32_t rank[OPL];
        double w[OPL];
#pragma unroll
        for (int o = 0; o < OPL; o++) {
            rank[o] = word[o] & 15u;
            w[o] = (double)__uint_as_float(word[o] & ~15u);
        }
#pragma unroll
        for (int o = 0; o < OPL; o++) word[o] = s_w[buf][min(ii + 1, kPfInputs - 1)][o_lane + o];
        __builtin_amdgcn_sched_barrier(0);
        slow |= ((n[0] >> 7) & 1u) << ii;
        if ((slow >> ii) & 1u) n[0] = n[1] = n[2] = n[3] = 0u;   // nothing here
#pragma unroll
        for (int t = 0; t < kPfGroup; t++) {
            const uint32_t nt = (n[t >> 2] >> (8 * (t & 3))) & 0x1fu;
#pragma unroll
            for (int o = 0; o < OPL; o++) fma_below(acc[t][o], w[o], rank[o], x[t], nt);
        }
        exec_settled();
    };
    for (int k = k0; k < k1; k += kPfInputs, buf ^= 1, turn = turn == 2 ? 0 : turn + 1) {
        uint32_t perm0 = 0, perm1 = 0;
#pragma unroll
        for (int r = 0; r < 8; r++) {
            const uint32_t c0 = code[r] >> shift, c1 = code[r] >> 16;
            const uint32_t p0 = c0 & 15u, p1 = c1 & 15u;
            perm0 |= 1u << p0;
            perm1 |= 1u << p1;
            // an fp16's fp32 form has 13 zero bits
            s_w[buf][si][sc * 16 + p0] = __float_as_uint(h2f(c0)) | (uint32_t)(sr + r);
            s_w[buf][si][sc * 16 + 16 + p1] = __float_as_uint(h2f(c1)) | (uint32_t)(sr + r);
        }
        // each position once among the bucket's 16 codes (the other eight are 8 lanes away)
        perm0 |= (uint32_t)__shfl_xor((int)perm0, 8, 64);
        perm1 |= (uint32_t)__shfl_xor((int)perm1, 8, 64);
        if ((perm0 != 0xffffu && scol < C) || (perm1 != 0xffffu && scol + 1 < C)) atomicOr(&s_bad[turn], 1u << si);
        fetch(k + kPfInputs);
        __syncthreads();
        if (tid == 0) s_bad[turn == 0 ? 2 : turn - 1] = 0u;
        if (active) {
            slow = __builtin_amdgcn_readfirstlane(s_bad[turn]);
#pragma unroll
            for (int o = 0; o < OPL; o++) word[o] = s_w[buf][0][o_lane + o];
#pragma unroll 1
            for (int ii = 0; ii < kPfInputs; ii += 2) {
                input(k, ii, xa, na, xb, nb);
                input(k, ii + 1, xb, nb, xa, na);
            }
            for (; slow; slow &= slow - 1u) slow_input(k + __builtin_ctz(slow));
        }
    }
    if (!active || tile * kPfTile + o_lane >= C * 16) return;
    double* out = a.part + ((size_t)split * a.groups + g) * kPfGroup * a.width + a.ofs[m] + tile * kPfTile + o_lane;
#pragma unroll
    for (int t = 0; t < kPfGroup; t++)
#pragma unroll
        for (int o = 0; o < OPL; o++) out[(size_t)t * a.width + o] = acc[t][o];
}

static int pf_wt(int groups) { return groups >= 3 ? 4 : groups; }   // token groups per workgroup

static int pf_tiles(int n, const iam_bucket_matrix* mats)
{
    int t = 0;
    for (int j = 0; j < n; j++) t += (mats[j].bucket_cols + 15) / 16;
    return t;
}

// inputs of a split, when there are to be s of them
static int pf_per_split(int in_dim, int s) { return ((in_dim + s - 1) / s + kPfInputs - 1) / kPfInputs * kPfInputs; }

// Splits of the inputs: the launch runs in rounds of the workgroups the chip
// holds (three per CU), each round as long as a split; more splits leave less
// of the last round idle, at the cost of their partial sums (about 40 inputs'
// time each).
int pf_splits(int n, const iam_bucket_matrix* mats, int tokens, int in_dim)
{
    const int G = pf_groups(tokens), wt = pf_wt(G);
    const int blocks = pf_tiles(n, mats) * ((G + wt - 1) / wt);
    int best = 1;
    double best_cost = 1e30;
    const int most = std::min(32, std::max(8, kPfMaxPartRows / (G * kPfGroup)));
    for (int s = 1; s <= most && s * 64 <= in_dim; s++) {
        const int per = pf_per_split(in_dim, s), used = (in_dim + per - 1) / per;
        const double rounds = std::ceil(blocks * (double)used / 768.0);
        const double cost = rounds * (per + 40.0);
        if (cost < best_cost * 0.98) {
            best_cost = cost;
            best = used;
        }
    }
    return best;
}

int pf_products(Ctx* c, int n, const iam_bucket_matrix* mats, int tokens, int in_dim, int splits, const PfSelection* sel,
                const double* xd, double* part)
{
    PfGemmArgs a{};
    a.n = n;
    int tiles = 0, width = 0;
    for (int j = 0; j < n; j++) {
        a.W[j] = mats[j].buckets;
        a.count[j] = sel[j].count;
        a.mask[j] = sel[j].mask;
        a.cols[j] = mats[j].bucket_cols;
        a.ofs[j] = width;
        a.first[j] = tiles;
        tiles += (mats[j].bucket_cols + 15) / 16;
        width += mats[j].bucket_cols * 16;
    }
    a.tiles = tiles;
    a.width = width;
    a.xd = xd;
    a.part = part;
    a.in_dim = in_dim;
    a.groups = pf_groups(tokens);
    const int wt = pf_wt(a.groups);
    a.token_blocks = (a.groups + wt - 1) / wt;
    a.per = pf_per_split(in_dim, splits);
    IAM_REQUIRE((in_dim + a.per - 1) / a.per == splits && in_dim % kPfInputs == 0, "prefill: bad split");
    const dim3 grid((unsigned)(tiles * a.token_blocks * splits));
    if (wt == 4) return launch(c, "prefill.products", k_pf_products<4>, grid, dim3(256), 0, a);
    if (wt == 2) return launch(c, "prefill.products", k_pf_products<2>, grid, dim3(256), 0, a);
    return launch(c, "prefill.products", k_pf_products<1>, grid, dim3(256), 0, a);
}

// ------------------------------------------------- the layer's other steps ---

__device__ __forceinline__ float part_sum(const PfPart& P, int t, int o)
{
    const double* p = P.p + (size_t)t * P.width + o;
    const size_t step = (size_t)P.rows * P.width;
    double s = p[0];
    int k = 1;
    for (; k + 4 <= P.splits; k += 4) {   // four loads in flight, added in order
        const double a = p[k * step], b = p[(k + 1) * step], c = p[(k + 2) * step], d = p[(k + 3) * step];
        s += a;
        s += b;
        s += c;
        s += d;
    }
    for (; k < P.splits; k++) s += p[k * step];
    return (float)s;
}

// The residual stream and its norm, workgroup = token, in the walk's order:
// thread's n / 256 consecutive squares in order, then the 256-way tree.
__global__ __launch_bounds__(256) void k_pf_norm(PfPart part, const uint16_t* __restrict__ embed,
                                                 const int* __restrict__ tokens, int vocab,
                                                 const float* __restrict__ scale, float* h,
                                                 const uint16_t* __restrict__ gain, float eps, int n,
                                                 float* __restrict__ x)
{
#pragma clang fp contract(off)
    __shared__ float sum[256];
    const int tid = threadIdx.x, t = blockIdx.x;
    h += (size_t)t * n;
    x += (size_t)t * n;
    const int tok = part.p ? 0 : tokens[t];
    for (int i = tid; i < n; i += 256) {
        float v;
        if (part.p) {
            v = __fadd_rn(h[i], part_sum(part, t, i));
        } else {
            v = tok >= 0 && tok < vocab ? h2f(embed[(size_t)tok * n + i]) : 0.0f;
            if (scale) v = __fmul_rn(v, scale[i]);
        }
        h[i] = v;
    }
    __syncthreads();
    const int per = n / 256;
    float s = 0.0f;
    for (int k = 0; k < per; k++) {
        const float v = h[tid * per + k];
        s = __fadd_rn(s, __fmul_rn(v, v));
    }
    sum[tid] = s;
    __syncthreads();
    for (int st = 128; st > 0; st >>= 1) {
        if (tid < st) sum[tid] = __fadd_rn(sum[tid], sum[tid + st]);
        __syncthreads();
    }
    const float mean = __fdiv_rn(sum[0], (float)n);
    const float sc = (float)(1.0 / sqrt((double)__fadd_rn(mean, eps)));
    for (int i = tid; i < n; i += 256) x[i] = __fmul_rn(h2f(gain[i]), __fmul_rn(h[i], sc));
}

int pf_embed_norm(Ctx* c, const uint16_t* embed, const int* tokens, int vocab, const float* scale, float* h,
                  const uint16_t* gain, int dim, float eps, int n_tokens, float* x)
{
    return launch(c, "prefill.norm", k_pf_norm, dim3(n_tokens), dim3(256), 0, PfPart{}, embed, tokens, vocab,
                  scale, h, gain, eps, dim, x);
}

int pf_res_norm(Ctx* c, const PfPart& part, float* h, const uint16_t* gain, int dim, float eps, int n_tokens, float* x)
{
    return launch(c, "prefill.norm", k_pf_norm, dim3(n_tokens), dim3(256), 0, part, (const uint16_t*)nullptr,
                  (const int*)nullptr, 0, (const float*)nullptr, h, gain, eps, dim, x);
}

// RoPE and KV append: workgroup (token, four heads), wave = head of q, k or
// v, lane = the rotation pair (lane, 64 + lane)
__global__ __launch_bounds__(256) void k_pf_rope(PfPart qkv, const float* __restrict__ rope, int pos0, int n_heads, int n_kv,
                                                 float* __restrict__ q_rot, uint16_t* __restrict__ kc,
                                                 uint16_t* __restrict__ vc)
{
#pragma clang fp contract(off)
    const int t = blockIdx.y, lane = threadIdx.x & 63;
    const int hd = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (hd >= n_heads + 2 * n_kv) return;
    const int pos = pos0 + t;
    const float lo = part_sum(qkv, t, hd * 128 + lane), hi = part_sum(qkv, t, hd * 128 + 64 + lane);
    const float c = rope[(size_t)pos * 128 + 2 * lane], sn = rope[(size_t)pos * 128 + 2 * lane + 1];
    const float r0 = __fsub_rn(__fmul_rn(lo, c), __fmul_rn(hi, sn)), r1 = __fadd_rn(__fmul_rn(hi, c), __fmul_rn(lo, sn));
    if (hd < n_heads) {
        float* q = q_rot + ((size_t)t * n_heads + hd) * 128;
        q[lane] = r0;
        q[64 + lane] = r1;
        return;
    }
    const bool isk = hd < n_heads + n_kv;
    const int kv = hd - n_heads - (isk ? 0 : n_kv);
    uint16_t* o = (isk ? kc : vc) + ((size_t)pos * n_kv + kv) * 128;
    o[lane] = __half_as_ushort(__float2half_rn(isk ? r0 : lo));
    o[64 + lane] = __half_as_ushort(__float2half_rn(isk ? r1 : hi));
}

int pf_rope_append(Ctx* c, const PfPart& qkv, const float* rope, int pos0, int n_heads, int n_kv, int n_tokens,
                   float* q_rot, uint16_t* kc, uint16_t* vc)
{
    return launch(c, "prefill.rope", k_pf_rope, dim3((n_heads + 2 * n_kv + 3) / 4, n_tokens), dim3(256), 0, qkv, rope, pos0,
                  n_heads, n_kv, q_rot, kc, vc);
}

__global__ __launch_bounds__(256) void k_pf_silu(PfPart gu, int ffn, float* __restrict__ s)
{
    const int i = blockIdx.x * 256 + threadIdx.x, t = blockIdx.y;
    if (i >= ffn) return;
    const float gv = part_sum(gu, t, i), uv = part_sum(gu, t, ffn + i);
    const double x1 = (double)gv;
    s[(size_t)t * ffn + i] = (float)((double)uv * x1 / (1.0 + exp(-x1)));   // silu32, matrix.cl:27-32
}

int pf_silu(Ctx* c, const PfPart& gu, int ffn, int n_tokens, float* s)
{
    return launch(c, "prefill.silu", k_pf_silu, dim3((ffn + 255) / 256, n_tokens), dim3(256), 0, gu, ffn, s);
}

// greedy pick of each token's logits: first maximum (test_generation.cpp:235)
__global__ __launch_bounds__(1024) void k_pf_pick(PfPart lg, int pos0, int* __restrict__ hist, int hist_len)
{
    __shared__ float sv[16];
    __shared__ int si[16];
    const int tid = threadIdx.x, t = blockIdx.x;
    float bv = -INFINITY;
    int bi = 0x7fffffff;
    auto take = [&](float v, int i) {
        if (v > bv || (v == bv && i < bi)) {
            bv = v;
            bi = i;
        }
    };
    for (int i = tid; i < lg.width; i += 1024) take(part_sum(lg, t, i), i);
    for (int o = 32; o > 0; o >>= 1) {
        const float ov = __shfl_xor(bv, o, 64);
        const int oi = __shfl_xor(bi, o, 64);
        take(ov, oi);
    }
    if ((tid & 63) == 0) {
        sv[tid >> 6] = bv;
        si[tid >> 6] = bi;
    }
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; w++) take(sv[w], si[w]);
        const int at = pos0 + t + 1;
        if (at < hist_len) hist[at] = bi < lg.width ? bi : 0;
    }
}

int pf_pick(Ctx* c, const PfPart& logits, int pos0, int n_tokens, int* hist, int hist_len)
{
    return launch(c, "prefill.pick", k_pf_pick, dim3(n_tokens), dim3(1024), 0, logits, pos0, hist, hist_len);
}

}  // namespace iam
