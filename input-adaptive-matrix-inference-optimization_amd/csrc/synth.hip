// Synthetic weights and the bucket-layout producer on the GPU.
//
// Generator: element n of tensor `tid` = mean + sigma * N, with
// N = (sum of 12 uniform uint32 - 6*2^32) / 2^32 drawn from a counter-based
// splitmix64 stream keyed by (seed, tid).  Integer sums and power-of-two
// scaling are exact, the affine map uses explicitly rounded double ops and
// the result is rounded once (to fp16 or to float), so the bytes equal the
// CPU generator's on any machine.
//
// Bucketizer: bucketize_fp16_packed (preprocess_layer_fixed_gpu.py:110-242)
// with its exact numerics:
//   probes  fp16(float32 sum over j of |W[j,i]| in j order / out_dim) (:145, :154)
//   buckets rows i*16 + rank, |w| descending within each bucket of 16, ties in
//           original order (:163-188); code = (fp16 bits & 0xFFF0) | position (:192-200)
//   stats   fp16(numpy pairwise float32 sum of the row's |values| / nb),
//           replicated into 4 channels (:211-221)
#include <hip/hip_fp16.h>

#include "internal.h"
#include "layer_ops.h"
#include "wave.h"

namespace iam {

constexpr uint64_t kGolden = 0x9E3779B97F4A7C15ULL;

__host__ __device__ inline uint64_t mix64(uint64_t z)
{
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ULL;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBULL;
    return z ^ (z >> 31);
}

static uint64_t stream_key(uint64_t seed, uint64_t tid)
{
    return mix64(mix64(seed + kGolden) ^ (tid * 0xD1B54A32D192ED03ULL));
}

__device__ inline double gen_normal(uint64_t key, uint64_t n)
{
    uint64_t s = 0;
#pragma unroll
    for (int j = 0; j < 6; j++) {
        const uint64_t u = mix64(key + (n * 6 + (uint64_t)j + 1) * kGolden);
        s += (u & 0xffffffffULL) + (u >> 32);
    }
    const int64_t c = (int64_t)s - (int64_t)(6ULL << 32);
    return (double)c * (1.0 / 4294967296.0);
}

__global__ void k_gen_f16(uint64_t key, size_t count, double mean, double sigma, uint16_t* __restrict__ out)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) {
        const double v = __dadd_rn(mean, __dmul_rn(sigma, gen_normal(key, i)));
        const _Float16 h = static_cast<_Float16>(v);   // one rounding, double -> fp16
        out[i] = __builtin_bit_cast(uint16_t, h);
    }
}

__global__ void k_gen_f32(uint64_t key, size_t count, double mean, double sigma, float* __restrict__ out)
{
    size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t stride = (size_t)gridDim.x * blockDim.x;
    for (; i < count; i += stride) {
        const double v = __dadd_rn(mean, __dmul_rn(sigma, gen_normal(key, i)));
        out[i] = __double2float_rn(v);
    }
}

__device__ __forceinline__ float h2f(uint16_t b) { return __half2float(__ushort_as_half(b)); }

// ------------------------------------------------------------ bucketizer ---
// One pass over W.  Workgroup g owns the 16 inputs (columns of W) 16g ..
// 16g + 15 and walks the buckets in order, 64 at a time; 8 waves sort and
// emit, a ninth adds the probes.  Per chunk of 64 buckets:
//   sort    thread (column pair, bucket) holds 2 columns x 16 rows (its loads
//           for the next chunk go out before the barrier), sorts each
//           column's 16 keys by a network, and stores them by rank in LDS
//           (s_key) and, in row order, for the probes (s_raw)
//   emit    the rows' codes (lane = bucket: 128 consecutive bytes a wave
//           store), and the rows' sums for the stats: 8 lanes per row, one
//           per accumulator of numpy's 8-way unrolled block
//   probes  the ninth wave adds each column's |w| in row order, the first
//           half of the chunk during its emit, the second during the next
//           sort
// 14336 x 4096, with the compact stats: 1420 us a call for three passes (the
// probes with one load chain per column, a sort whose 2-byte stores lay 2 * nb
// bytes apart, then the sums re-reading W through the codes' positions), now
// 138 us; 2000 x 300: 32.9 -> 10.3 us.  W and the codes once at the part's
// copy rate are 47 us.  What bounds it now: the phases of the one workgroup a
// CU holds follow each other (sorting, emitting and adding are about 50 us of
// vector instructions, the waits between them as much again), and the probes'
// chain of dependent adds takes issue slots from one SIMD (without it: 106 of
// 142 us, measured before the emit's and the sums' LDS reads went out together).
// 8 columns per workgroup, two to a CU: 226 us.
constexpr int kBkInputs = 16;               // columns of W per workgroup
constexpr int kBkChunk = 64;                // buckets per chunk
constexpr int kBkWorkers = 512;             // sorting threads (8 column pairs x 64 buckets)
constexpr int kBkThreads = kBkWorkers + 64; // and the wave of the probes
constexpr int kBkKeyStride = kBkChunk + 4;  // words per (rank, column): 8 column pairs x 8 buckets on 64 banks
constexpr int kBkRawStride = kBkChunk * 16 + 8;   // halves per column: 16-byte reads on disjoint banks
constexpr int kBkDepth = 24;                // levels of the pairwise tree: blocks of at least 64, up to 2^27 buckets

// One element's sort key: |w| (15 bits), then the earlier position first,
// with the sign along: descending keys are the reference's order (|w|
// descending, ties in original order), and each key holds its code and its
// |w|.  A NaN sorts by its bits, above infinity.
__device__ __forceinline__ uint32_t bucket_key(uint32_t w, int p)
{
    return ((w & 0x7fffu) << 5) | ((uint32_t)(15 - p) << 1) | ((w >> 15) & 1u);
}
__device__ __forceinline__ uint16_t bucket_code(uint32_t key)
{
    return (uint16_t)(((key & 1u) << 15) | ((key >> 5) & 0x7ff0u) | (15u - ((key >> 1) & 15u)));
}

// Batcher's odd-even merge sort of 16 keys, descending (63 comparators)
__device__ __forceinline__ void sort16(uint32_t (&k)[16])
{
#pragma unroll
    for (int p = 1; p < 16; p *= 2)
#pragma unroll
        for (int q = p; q >= 1; q /= 2)
#pragma unroll
            for (int j = q % p; j <= 15 - q; j += 2 * q)
#pragma unroll
                for (int i = 0; i < q; i++)
                    if (i + j + q < 16 && (i + j) / (p * 2) == (i + j + q) / (p * 2)) {
                        const uint32_t a = k[i + j], b = k[i + j + q];
                        k[i + j] = max(a, b);
                        k[i + j + q] = min(a, b);
                    }
}

// acc + |h|, h in the low or high half of w: one fp32 rounding, as the add's
// (the product with 1 is exact)
template <int HI>
__device__ __forceinline__ float add_abs_half(float acc, uint32_t w)
{
    if constexpr (HI) asm("v_fma_mix_f32 %0, |%1|, 1.0, %0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(acc) : "v"(w));
    else asm("v_fma_mix_f32 %0, |%1|, 1.0, %0 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "+v"(acc) : "v"(w));
    return acc;
}

// The block of numpy's pairwise summation (split at n/2 rounded down to a
// multiple of 8 while n > 128) that holds element a of n: its end, and how
// many subtrees end with it (each adds its left half's sum).
__device__ __forceinline__ void pairwise_block(int n, int a, int& end, int& closes)
{
    int lo = 0;
    closes = 0;
    while (n > 128) {
        int n2 = n / 2;
        n2 -= n2 % 8;
        if (a < lo + n2) {
            n = n2;
            closes = 0;
        } else {
            lo += n2;
            n -= n2;
            closes++;
        }
    }
    end = lo + n;
}

struct BucketLds {
    uint32_t key[16 * kBkInputs * kBkKeyStride];            // [rank][column][bucket]
    __align__(16) uint16_t raw[2][kBkInputs * kBkRawStride];   // [column][row of the chunk], two chunks
    float tree[kBkDepth][16 * kBkInputs];                   // the pairwise sums waiting for their right halves
};

// The block's work; WHOLE: it has all 16 columns (the last workgroup of an
// in_dim that is no multiple of 16 re-reads its last one).
template <bool WHOLE>
__device__ __forceinline__ void bucketize_block(BucketLds& S, const uint16_t* __restrict__ W, int in_dim, int nb, int i0,
                                                int ni, uint16_t* __restrict__ buckets, uint16_t* __restrict__ stats,
                                                uint16_t* __restrict__ probes)
{
#pragma clang fp contract(off)
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const bool worker = tid < kBkWorkers;
    const int c2 = tid & 7, bl = tid >> 3;   // column pair and bucket of a sorting thread
    const int ca = min(2 * c2, ni - 1), cb = min(2 * c2 + 1, ni - 1);
    // columns 2*c2 and 2*c2 + 1 of a bucket's rows, as one 4-byte load at any
    // 2-byte boundary; threads past the last bucket re-read it, so that every
    // chunk has the same number of loads in flight
    auto load = [&](int b0, uint32_t (&v)[16]) {
        const uint16_t* p = W + (size_t)min(b0 + bl, nb - 1) * 16 * in_dim + i0;
#pragma unroll
        for (int r = 0; r < 16; r++) {
            typedef uint32_t u32u __attribute__((aligned(2)));
            if constexpr (WHOLE) v[r] = *reinterpret_cast<const u32u*>(p + (size_t)r * in_dim + 2 * c2);
            else v[r] = (uint32_t)p[(size_t)r * in_dim + ca] | ((uint32_t)p[(size_t)r * in_dim + cb] << 16);
        }
    };
    // the stats: wave w takes the rows (rank, column) 32w .. 32w + 31, eight
    // at a time, lane = 8 * row + accumulator
    constexpr int kRowSets = 16 * kBkInputs / (kBkWorkers / 8);
    float acc[kRowSets];
#pragma unroll
    for (int s = 0; s < kRowSets; s++) acc[s] = 0.0f;
    int depth = 0;      // pairwise sums on the stack (the same for every row)
    int blk_end = 0, closes = 0;
    // the ninth wave, lane = column: the column's sum over buckets g0 .. g1 - 1
    // of a chunk; the next bucket's rows are read during this one's adds
    float psum = 0.0f;
    auto add_probes = [&](int buf, int g0, int g1) {
        if (g0 >= g1) return;
        const uint4* p = reinterpret_cast<const uint4*>(S.raw[buf] + (lane & 15) * kBkRawStride);
        uint4 a = p[2 * g0], b = p[2 * g0 + 1];
        for (int g = g0; g < g1; g++) {
            const uint32_t w[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
            const int nx = min(g + 1, g1 - 1);
            a = p[2 * nx];
            b = p[2 * nx + 1];
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < 8; k++) {
                psum = add_abs_half<0>(psum, w[k]);
                psum = add_abs_half<1>(psum, w[k]);
            }
        }
    };
    int nc_prev = 0;
    auto chunk = [&](int b0, int buf, uint32_t (&v)[16]) {
        const int nc = min(kBkChunk, nb - b0);
        // ---- sort
        if (worker) {
            if (bl < nc) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int c = 2 * c2 + h;
                    uint32_t k[16], raw[8];
#pragma unroll
                    for (int r = 0; r < 16; r++) {
                        const uint32_t w = h ? v[r] >> 16 : v[r] & 0xffffu;
                        k[r] = bucket_key(w, r);
                        raw[r >> 1] = r & 1 ? raw[r >> 1] | (w << 16) : w;
                    }
                    uint4* rp = reinterpret_cast<uint4*>(S.raw[buf] + c * kBkRawStride + bl * 16);
                    rp[0] = make_uint4(raw[0], raw[1], raw[2], raw[3]);
                    rp[1] = make_uint4(raw[4], raw[5], raw[6], raw[7]);
                    sort16(k);
#pragma unroll
                    for (int r = 0; r < 16; r++) S.key[(r * kBkInputs + c) * kBkKeyStride + bl] = k[r];
                }
            }
        } else {
            add_probes(buf ^ 1, nc_prev / 2, nc_prev);
        }
        nc_prev = nc;
        __syncthreads();
        // ---- emit: lane = 4 buckets (8 bytes at any 2-byte boundary) of one
        // of 4 rows; then this buffer's next loads, behind the stores (the
        // wait for them then waits for no later store)
        if (worker) {
            // (a full chunk's eight LDS reads go out together)
            const int q = 4 * (lane & 15), rc0 = wave * 32 + (lane >> 4);
            typedef uint32_t u32x2u __attribute__((ext_vector_type(2), aligned(2)));
            auto codes = [](const uint4& k) -> u32x2u {
                return u32x2u{bucket_code(k.x) | ((uint32_t)bucket_code(k.y) << 16),
                              bucket_code(k.z) | ((uint32_t)bucket_code(k.w) << 16)};
            };
            auto row_out = [&](int rc) {
                return buckets + ((size_t)(i0 + rc % kBkInputs) * 16 + rc / kBkInputs) * nb + b0 + q;
            };
            if (WHOLE && nc == kBkChunk) {
                uint4 k[8];
#pragma unroll
                for (int s = 0; s < 8; s++) k[s] = *reinterpret_cast<const uint4*>(S.key + (rc0 + 4 * s) * kBkKeyStride + q);
#pragma unroll
                for (int s = 0; s < 8; s++) *reinterpret_cast<u32x2u*>(row_out(rc0 + 4 * s)) = codes(k[s]);
            } else {
                for (int s = 0; s < 8; s++) {
                    const int rc = rc0 + 4 * s;
                    if (q >= nc || rc % kBkInputs >= ni) continue;
                    const u32x2u c = codes(*reinterpret_cast<const uint4*>(S.key + rc * kBkKeyStride + q));
                    uint16_t* o = row_out(rc);
                    if (q + 4 <= nc) {
                        *reinterpret_cast<u32x2u*>(o) = c;
                    } else {
                        o[0] = (uint16_t)c.x;
                        if (q + 1 < nc) o[1] = (uint16_t)(c.x >> 16);
                        if (q + 2 < nc) o[2] = (uint16_t)c.y;
                    }
                }
            }
            load(b0 + 2 * kBkChunk, v);
            const int row = wave * 32 + (lane >> 3), j = lane & 7;
            for (int e = 0; e < nc;) {
                if (b0 + e >= blk_end) pairwise_block(nb, b0 + e, blk_end, closes);
                const int stop = min(nc, blk_end - b0);   // blocks start at multiples of 8
                for (; e + 32 <= stop; e += 32) {   // 16 LDS reads in flight
                    uint32_t k[4][kRowSets];
#pragma unroll
                    for (int u = 0; u < 4; u++)
#pragma unroll
                        for (int s = 0; s < kRowSets; s++) k[u][s] = S.key[(row + 8 * s) * kBkKeyStride + e + 8 * u + j];
#pragma unroll
                    for (int u = 0; u < 4; u++)
#pragma unroll
                        for (int s = 0; s < kRowSets; s++) acc[s] = __fadd_rn(acc[s], h2f((uint16_t)(k[u][s] >> 5)));
                }
                for (; e + 8 <= stop; e += 8) {
#pragma unroll
                    for (int s = 0; s < kRowSets; s++) {
                        const uint32_t k = S.key[(row + 8 * s) * kBkKeyStride + e + j];
                        acc[s] = __fadd_rn(acc[s], h2f((uint16_t)(k >> 5)));
                    }
                }
                if (b0 + stop < blk_end) break;   // the block goes on in the next chunk
                // the block's end: ((r0+r1) + (r2+r3)) + ((r4+r5) + (r6+r7)),
                // the elements past its last whole 8 in order, then the
                // subtrees it completes
#pragma unroll
                for (int s = 0; s < kRowSets; s++) {
                    float a = acc[s];
                    a = __fadd_rn(a, __shfl_down(a, 1, 8));
                    a = __fadd_rn(a, __shfl_down(a, 2, 8));
                    a = __fadd_rn(a, __shfl_down(a, 4, 8));
                    acc[s] = 0.0f;
                    if (j == 0) {
                        for (int x = e; x < stop; x++)
                            a = __fadd_rn(a, h2f((uint16_t)(S.key[(row + 8 * s) * kBkKeyStride + x] >> 5)));
                        int d = depth;
                        for (int x = 0; x < closes; x++) a = __fadd_rn(S.tree[--d][row + 8 * s], a);
                        S.tree[d][row + 8 * s] = a;
                    }
                }
                depth += 1 - closes;
                e = stop;
            }
        } else {
            add_probes(buf, 0, nc / 2);
        }
        __syncthreads();
    };
    uint32_t va[16], vb[16];
    if (worker) {
        load(0, va);
        load(kBkChunk, vb);
    } else {
        __builtin_amdgcn_s_setprio(3);   // the serial chain goes first
    }
    int last = 0;   // the last chunk's buffer
    for (int b0 = 0; b0 < nb; b0 += 2 * kBkChunk) {
        chunk(b0, 0, va);
        last = 0;
        if (b0 + kBkChunk >= nb) break;
        chunk(b0 + kBkChunk, 1, vb);
        last = 1;
    }
    if (!worker) {
        add_probes(last, nc_prev / 2, nc_prev);
        if (lane < ni) probes[i0 + lane] = __half_as_ushort(__float2half_rn(__fdiv_rn(psum, (float)(nb * 16))));
        return;
    }
    if (tid < 16 * kBkInputs) {   // row (rank, column) = tid: the tree's one remaining sum
        const int r = tid / kBkInputs, c = tid % kBkInputs;
        if (c < ni) {
            const uint16_t m = __half_as_ushort(__float2half_rn(__fdiv_rn(__fadd_rn(0.0f, S.tree[0][tid]), (float)nb)));
            const uint32_t m2 = (uint32_t)m | ((uint32_t)m << 16);
            reinterpret_cast<uint2*>(stats)[(size_t)(i0 + c) * 16 + r] = make_uint2(m2, m2);
        }
    }
}

__global__ __launch_bounds__(kBkThreads) void k_bucketize(const uint16_t* __restrict__ W, int in_dim, int nb,
                                                          uint16_t* __restrict__ buckets,
                                                          uint16_t* __restrict__ stats, uint16_t* __restrict__ probes)
{
    __shared__ BucketLds S;
    const int i0 = xcd_remap((int)blockIdx.x, (int)gridDim.x) * kBkInputs;   // neighbours share W's lines in one L2
    const int ni = min(kBkInputs, in_dim - i0);
    if (ni == kBkInputs) bucketize_block<true>(S, W, in_dim, nb, i0, ni, buckets, stats, probes);
    else bucketize_block<false>(S, W, in_dim, nb, i0, ni, buckets, stats, probes);
}

// Fewer than 8 buckets: thread = input, its codes, stats and probe in
// registers (numpy's pairwise sum of fewer than 8 values adds them in order,
// and an input's 16 rows lie together, so they leave in 16-byte stores at any
// 2-byte boundary).  k_bucketize would fill a CU's LDS for a seventh of a
// chunk at most, one workgroup a CU at a time: 16, 64 and 112 x 65536 with the
// compact stats 87, 91 and 103 us that way, 11.7, 18.6 and 23.4 by this one
// (18, 44 and 68 in three passes over W); up to 4096 inputs the two are alike.
template <int NB>
__global__ __launch_bounds__(64) void k_bucketize_few(const uint16_t* __restrict__ W, int in_dim,
                                                      uint16_t* __restrict__ buckets, uint16_t* __restrict__ stats,
                                                      uint16_t* __restrict__ probes)
{
#pragma clang fp contract(off)
    static_assert(NB >= 1 && NB < 8, "sums in order");
    const int i = blockIdx.x * 64 + threadIdx.x;
    if (i >= in_dim) return;
    float psum = 0.0f, sum[16];
    uint32_t out[8 * NB];   // the codes [rank][bucket], two a word
#pragma unroll
    for (int r = 0; r < 16; r++) sum[r] = 0.0f;
#pragma unroll
    for (int k = 0; k < 8 * NB; k++) out[k] = 0u;
#pragma unroll
    for (int b = 0; b < NB; b++) {
        uint32_t k[16];
#pragma unroll
        for (int r = 0; r < 16; r++) k[r] = W[(size_t)(b * 16 + r) * in_dim + i];
#pragma unroll
        for (int r = 0; r < 16; r++) {
            psum = __fadd_rn(psum, fabsf(h2f((uint16_t)k[r])));
            k[r] = bucket_key(k[r], r);
        }
        sort16(k);
#pragma unroll
        for (int r = 0; r < 16; r++) {
            sum[r] = __fadd_rn(sum[r], h2f((uint16_t)(k[r] >> 5)));
            out[(r * NB + b) >> 1] |= (uint32_t)bucket_code(k[r]) << (16 * ((r * NB + b) & 1));
        }
    }
    typedef uint32_t u32x4u __attribute__((ext_vector_type(4), aligned(2)));
    u32x4u* o = reinterpret_cast<u32x4u*>(buckets + (size_t)i * 16 * NB);
#pragma unroll
    for (int k = 0; k < 2 * NB; k++) o[k] = u32x4u{out[4 * k], out[4 * k + 1], out[4 * k + 2], out[4 * k + 3]};
#pragma unroll
    for (int r = 0; r < 16; r++) {
        const uint16_t m = __half_as_ushort(__float2half_rn(__fdiv_rn(sum[r], (float)NB)));
        const uint32_t m2 = (uint32_t)m | ((uint32_t)m << 16);
        reinterpret_cast<uint2*>(stats)[(size_t)i * 16 + r] = make_uint2(m2, m2);
    }
    probes[i] = __half_as_ushort(__float2half_rn(__fdiv_rn(psum, (float)(NB * 16))));
}

static unsigned grid_for(size_t n, unsigned block, unsigned cap = 65535u * 4)
{
    size_t g = (n + block - 1) / block;
    return (unsigned)(g < cap ? (g ? g : 1) : cap);
}

int gen_f16(Ctx* c, uint64_t seed, uint64_t tid, size_t count, double mean, double sigma, uint16_t* out)
{
    return launch(c, "gen_f16", k_gen_f16, dim3(grid_for(count, 256)), dim3(256), 0, stream_key(seed, tid), count,
                  mean, sigma, out);
}

int gen_f32(Ctx* c, uint64_t seed, uint64_t tid, size_t count, double mean, double sigma, float* out)
{
    return launch(c, "gen_f32", k_gen_f32, dim3(grid_for(count, 256)), dim3(256), 0, stream_key(seed, tid), count,
                  mean, sigma, out);
}

int bucketize(Ctx* c, const uint16_t* w, int out_dim, int in_dim, uint16_t* buckets, uint16_t* stats,
              uint16_t* probes)
{
    const dim3 few((unsigned)((in_dim + 63) / 64));
    switch (out_dim / 16) {
    case 1: return launch(c, "bucketize", k_bucketize_few<1>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    case 2: return launch(c, "bucketize", k_bucketize_few<2>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    case 3: return launch(c, "bucketize", k_bucketize_few<3>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    case 4: return launch(c, "bucketize", k_bucketize_few<4>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    case 5: return launch(c, "bucketize", k_bucketize_few<5>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    case 6: return launch(c, "bucketize", k_bucketize_few<6>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    case 7: return launch(c, "bucketize", k_bucketize_few<7>, few, dim3(64), 0, w, in_dim, buckets, stats, probes);
    default: break;
    }
    return launch(c, "bucketize", k_bucketize, dim3((unsigned)((in_dim + kBkInputs - 1) / kBkInputs)), dim3(kBkThreads),
                  0, w, in_dim, out_dim / 16, buckets, stats, probes);
}

}  // namespace iam

using namespace iam;

extern "C" {

int iam_gen_f16(iam_ctx* c, uint64_t seed, uint64_t tid, size_t count, double mean, double sigma, uint16_t* out)
{
    if (!c || !out) return fail(IAM_E_INVALID, "gen_f16: null argument");
    if (count == 0) return IAM_OK;
    IAM_TRY(check_dev_range(c, out, count * 2, "gen_f16 out"));
    return gen_f16(c, seed, tid, count, mean, sigma, out);
}

int iam_gen_f32(iam_ctx* c, uint64_t seed, uint64_t tid, size_t count, double mean, double sigma, float* out)
{
    if (!c || !out) return fail(IAM_E_INVALID, "gen_f32: null argument");
    if (count == 0) return IAM_OK;
    IAM_TRY(check_dev_range(c, out, count * 4, "gen_f32 out"));
    return gen_f32(c, seed, tid, count, mean, sigma, out);
}

int iam_bucketize(iam_ctx* c, const uint16_t* w, int out_dim, int in_dim, uint16_t* buckets, uint16_t* stats,
                  uint16_t* probes)
{
    if (!c || !w || !buckets || !stats || !probes) return fail(IAM_E_INVALID, "bucketize: null argument");
    IAM_REQUIRE(out_dim > 0 && in_dim > 0 && out_dim % 16 == 0,
                "bucketize: out_dim must be a positive multiple of 16");
    const size_t n = (size_t)out_dim * in_dim;
    IAM_TRY(check_dev_range(c, w, n * 2, "bucketize W"));
    IAM_TRY(check_dev_range(c, buckets, n * 2, "bucketize buckets"));
    IAM_TRY(check_dev_range(c, stats, (size_t)in_dim * 16 * 4 * 2, "bucketize stats"));
    IAM_TRY(check_dev_range(c, probes, (size_t)in_dim * 2, "bucketize probes"));
    IAM_REQUIRE((((uintptr_t)stats) & 7) == 0, "bucketize: stats must be 8-byte aligned");
    return bucketize(c, w, out_dim, in_dim, buckets, stats, probes);
}

}  // extern "C"
