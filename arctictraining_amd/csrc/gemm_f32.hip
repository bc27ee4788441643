// Ragged grouped GEMMs in float32.  The float32 matrix instruction runs at a sixteenth of the bfloat16 one, so each operand
// is split into three bfloat16 parts, x = h + m + l, which hold all 24 bits of it, and of the nine products of parts the six
// that can reach the last bits of a float32 sum are taken, on v_mfma_f32_16x16x32_bf16, into float32 accumulators: h h in
// one, the five small ones in another.
// Error against float64, 2-norm, normal inputs: 0.9 to 4e-7 where v_mfma_f32_32x32x2_f32, which adds two products at a time,
// had 3e-7 to 1.1e-6 (K 256 to 4096; weight gradients of 5 to 700 rows 0.3 to 1.5e-7, before 0.4 to 4.8e-7), whatever the
// operands' magnitude: what bfloat16's range does not hold of the parts is dealt with at split3 and redo_exact.
//
// What bounds it: vector instructions, 13 to split two values (of the 16 cycles of a matrix instruction 8 are free for those of either
// wavefront, two of them; there are four and a half to one, so that putting them between the MFMAs of the step before gained nothing) and
// LDS traffic (three planes of every stage), so that tiles are as wide as the number of them allows.  One MI355X, 39 experts
// x 709 rows, 768 x 1856 and 928 x 768: A B 800 and 407 -> 549 and 281 us, A B^T 416 and 782 -> 285 and 520, weight
// gradients 423 and 827 -> 275 and 503 (140-157 TFLOP/s; the float32 instruction's peak is 157).  8 experts x 512 rows,
// 512 x 2048 and 1024 x 512: 106 and 68 -> 77 and 44, 61 and 131 -> 46 and 81, 61 and 100 -> 43 and 61: there are about as
// many tiles as compute units, and the last round's few are worked off in parts (most_in_parts).  Dealing each XCD a contiguous eighth of the tiles changed none of these figures.
#include "amoe_common.h"
#include "gemm_launch.h"

#include <type_traits>

typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 mfma_bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float mfma_f32x4;
typedef __attribute__((__vector_size__(16 * sizeof(float)))) float mfma_f32x16;

int amoe_build_tile_map(const int32_t* offsets, int R, int E, int bm, void* workspace, size_t workspace_bytes,
                        const int4** tile_map, const int32_t** n_mtiles, int* max_mtiles, hipStream_t s, bool ready);

namespace {

constexpr int BK = 32, NT = 256;
constexpr int BM_ROWS = 128, BN_ROWS = 64;

struct GemmArgsF32 {
    const float* A;
    const float* B;
    float* C;
    const int32_t* a_row_map;
    const int32_t* b_row_map;  // weight gradient only
    const int32_t* offsets;
    const int4* tile_map;
    const int32_t* n_mtiles;
    int lda, ldb, ldc;
    long long strideB, strideC;
    int E, Kd, M, N, n_ntiles, n_mt;
    float* inter;              // gated products: [R, N / 2]
    const float* row_scale;    // null: 1
    int act;
    int max_mtiles;            // entries of tile_map
    int cus;                   // compute units; 0: every tile is whole
};

// Gated products: a vector of C is (gate, up) of two intermediate columns, which leave the epilogue as row_scale up act(gate).
// With a kernel of its own that read C again and wrote them / so, a forward pass, us: 2048 tokens x 2 of 8 experts of 512 x 1024
// 147 / 143, 4096 x 2 of 8 of 1024 x 2048 729 / 713, 650 x 6 of 20 of 384 x 160 and a shared one 80 / 75, one token 57 / 54; a
// training step of the first 388 / 383.  Few rows an expert, where a tile's epilogue counts most, with that kernel / with row scales read in
// the epilogue and dead blocks of 16 rows activated / as now: 167 x 3 of 242 of 288 x 352 166.5 / 173.9 / 165.6, 40 x 4 of 128 of 512 x
// 768 162.9 / 167.1 / 162.0, 300 x 4 of 64 of 1024 x 512 136.5 / 137.3 / 135.2.
__device__ __forceinline__ float activate(int act, float g)
{
    switch (act) {
        case AMOE_ACT_SILU: return act_fwd<AMOE_ACT_SILU>(g);
        case AMOE_ACT_GELU: return act_fwd<AMOE_ACT_GELU>(g);
        case AMOE_ACT_RELU: return act_fwd<AMOE_ACT_RELU>(g);
        default: return act_fwd<AMOE_ACT_GPT_OSS>(g);
    }
}
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ f32x2_t gated(const GemmArgsF32& p, float s, const f32x4_t& c)
{
    return f32x2_t{s * c[1] * activate(p.act, c[0]), s * c[3] * activate(p.act, c[2])};
}
__device__ __forceinline__ void store_gated(const GemmArgsF32& p, int row, int col, const f32x4_t& c)
{
    *reinterpret_cast<f32x2_t*>(p.inter + (long long)row * (p.N / 2) + col / 2) = gated(p, p.row_scale ? p.row_scale[row] : 1.0f, c);
}
// the same of `rows` x `cols` elements of C that this wavefront has written one by one (redo_exact)
__device__ __forceinline__ void store_gated_again(const GemmArgsF32& p, int m0, int mend, int n0, int rows, int cols)
{
    __threadfence();
    for (int v = threadIdx.x & 63; v < rows * cols / 4; v += 64) {
        const int row = m0 + v / (cols / 4), col = n0 + v % (cols / 4) * 4;
        if (row < mend && col < p.N) store_gated(p, row, col, *reinterpret_cast<const f32x4_t*>(p.C + (long long)row * p.ldc + col));
    }
}

// The parts are of 2^16 x: of x itself, those of a value below 2^-110 would reach below bfloat16's smallest, 2^-133, which is
// float32's smallest times 2^16.  A sum of products is 2^32 times what it stands for.  (Results of 2^96 and more overflow
// on the way, as operands of 2^112 and more do in their parts: see redo_exact.)  Without it a product of operands at 2^-118 is
// off by 9e-6, at 2^-126 by 2e-3; it costs two of the 13 instructions, 3 to 4 % of the time.  (The remainder by a dot product of
// two bfloat16, four instructions fewer, is slower: that one runs at half the rate.)
constexpr float PART_SCALE = 65536.0f, SUM_SCALE = 1.0f / (65536.0f * 65536.0f);

// 2^16 x = h + m + l in three bf16 (round to nearest: |m| <= 2^-8 |h|, |l| <= 2^-16 |h|, nothing is left)
__device__ __forceinline__ void split3(const f32x4_t& v, u32x2_t (&out)[3])
{
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        const float x0 = v[2 * i] * PART_SCALE, x1 = v[2 * i + 1] * PART_SCALE;
        const uint32_t h = pack_bf16x2(x0, x1);
        const float r0 = x0 - bf16_lo(h), r1 = x1 - bf16_hi(h);
        const uint32_t m = pack_bf16x2(r0, r1);
        out[0][i] = h;
        out[1][i] = m;
        out[2][i] = pack_bf16x2(r0 - bf16_lo(m), r1 - bf16_hi(m));
    }
}

// workgroup barrier for data exchanged through LDS; loads from global memory stay in flight (__syncthreads awaits them)
__device__ __forceinline__ void lds_sync() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// One operand's stage in LDS, ROWS rows (or columns) x 32 k, three planes of bf16.  A fragment's lane (lq, l16) holds
// k 4 lq .. + 3 and 16 + 4 lq .. + 3 of row l16 (any order will do that both operands share: with this one the loads of
// an operand that goes straight into registers read 64 bytes of a row together).
// K-contiguous: [row][32 k] in that order, a fragment is 16 bytes of a row, a wavefront's 16 rows of them 1 KB in a row.
// K-strided: [k][ROWS], read with the transposing LDS read; 16-byte chunk c of row k stands at c ^ key(k), so that the
// eight k rows that 32 lanes read together (two chunks each) lie in different banks.
template <bool KC, int ROWS>
struct Stage {
    static constexpr uint32_t plane = ROWS * BK * 2;
    static constexpr int NV = ROWS * BK / 4 / NT;        // 16-byte vectors a thread loads
    __device__ static __forceinline__ uint32_t key(int k) { return ROWS == 64 ? 2 * ((k >> 1) & 3) : 2 * (k & 7); }
    // row (K-contiguous) or k (K-strided) of vector v, and where in it the vector starts
    __device__ static __forceinline__ int line(int tid, int v) { return KC ? (tid >> 3) + NT / 8 * v : tid / (ROWS / 4) + NT * 4 / ROWS * v; }
    __device__ static __forceinline__ int start(int tid) { return KC ? (tid & 7) * 4 : (tid & (ROWS / 4 - 1)) * 4; }
    __device__ static __forceinline__ uint32_t write_at(int tid, int v)
    {
        const int r = line(tid, v), c = start(tid);
        return KC ? r * (BK * 2) + ((c >> 2) & 3) * 16 + (c >> 4) * 8 : r * (ROWS * 2) + ((uint32_t)(c >> 3) ^ key(r)) * 16u + (c & 4) * 2;
    }
    // fragment of rows (columns) r0 .. r0 + 15
    __device__ static __forceinline__ mfma_bf16x8 read(uint32_t base, int r0, int l16, int lq)
    {
        if (KC) return *(const __attribute__((address_space(3))) mfma_bf16x8*)(uintptr_t)(base + (uint32_t)((r0 + l16) * (BK * 2) + lq * 16));
        const int k = 4 * lq + (l16 >> 2), c = (r0 >> 3) + ((l16 & 3) >> 1);
        const uint32_t at = base + k * (ROWS * 2) + ((uint32_t)c ^ key(k)) * 16u + (l16 & 1) * 8;
        typedef short i16x4_t __attribute__((ext_vector_type(4)));
        typedef __attribute__((address_space(3))) i16x4_t* tr_ptr;
        const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)at));
        // (sixteen rows on: the key does not look at that bit of k)
        const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)(at + 16 * ROWS * 2)));
        return __builtin_bit_cast(mfma_bf16x8, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
    }
    __device__ static __forceinline__ void put(uint32_t at, int tid, int v, const f32x4_t& x)
    {
        u32x2_t s[3];
        split3(x, s);
#pragma unroll
        for (int q = 0; q < 3; ++q) *(__attribute__((address_space(3))) u32x2_t*)(uintptr_t)(at + write_at(tid, v) + q * plane) = s[q];
    }
};

__device__ __forceinline__ bool finite4(const f32x4_t& c)
{
    bool ok = true;
#pragma unroll
    for (int v = 0; v < 4; ++v) ok = ok && (__float_as_uint(c[v]) & 0x7f800000u) != 0x7f800000u;
    return ok;
}

// An infinity or a NaN in an operand has no three parts (inf - inf), and large values overflow (see split3): a
// wavefront that met either works its rows x columns out again with the float32 instruction, straight from memory.
// a_at(row, k), b_at(k, column): addresses of elements that exist
template <typename FA, typename FB, typename FC>
__device__ __forceinline__ void redo_exact(int rows, int cols, int k_len, FA a_at, FB b_at, FC store)
{
    const int lane = threadIdx.x & 63, lj = lane & 31, lg = lane >> 5;
#pragma unroll 1
    for (int i = 0; i < rows; i += 32)
#pragma unroll 1
        for (int j = 0; j < cols; j += 32) {
            mfma_f32x16 acc;
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[v] = 0.f;
#pragma unroll 1
            for (int k0 = 0; k0 < k_len; k0 += 2) {
                const int k = k0 + lg;
                const bool live = k < k_len;
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(live ? *a_at(i + lj, k) : 0.f, live ? *b_at(k, j + lj) : 0.f, acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 16; ++v) store(i + 8 * (v >> 2) + 4 * lg + (v & 3), j + lj, acc[v]);
        }
}

// A tile of 32 rows x 64 columns whose NW wavefronts take every NW-th step of 32 k: both operands go straight into registers, and
// the partial sums meet in LDS, in a fixed order.  (The two halves of 16 rows in turn, a row of red for each wavefront.)
template <bool B_KC, bool GATED, int NW>
__device__ __forceinline__ void deep_tile(const GemmArgsF32& p, const int4& tm, int m0, int n0, f32x4_t (*red)[4 * 64])
{
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int mend = tm.z, k_len = p.Kd;
    const float* const Bb = p.B + (long long)tm.x * p.strideB;

    // (copies past the ends as above)
    const float* a_ptr[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        int gr = min(m0 + i * 16 + l16, mend - 1);
        if (p.a_row_map) gr = p.a_row_map[gr];
        a_ptr[i] = p.A + (long long)gr * p.lda;
    }
    // Fragment j: K-contiguous, column j * 16 + l16, two vectors of four k; K-strided, column 4 l16 + j, of the eight k rows' vectors
    // of four columns each.
    const float* b_ptr[B_KC ? 4 : 1];
#pragma unroll
    for (int j = 0; j < (B_KC ? 4 : 1); ++j)
        b_ptr[j] = B_KC ? Bb + (long long)min(n0 + j * 16 + l16, p.N - 1) * p.ldb : Bb + min(n0 + 4 * l16, p.N - 4);

    f32x4_t xa[2][2], xb[8];
    auto fetch = [&](int k0) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int k = min(k0 + 16 * h + 4 * lq, k_len - 4);
#pragma unroll
            for (int i = 0; i < 2; ++i) xa[i][h] = *reinterpret_cast<const f32x4_t*>(a_ptr[i] + k);
#pragma unroll
            for (int j = 0; j < 4; ++j)
                xb[h * 4 + j] = *reinterpret_cast<const f32x4_t*>(B_KC ? b_ptr[B_KC ? j : 0] + k : b_ptr[0] + (long long)(k + j) * p.ldb);
        }
    };
    mfma_f32x4 hi[2][4], lo[2][4];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) hi[i][j] = lo[i][j] = mfma_f32x4{0.f, 0.f, 0.f, 0.f};
    const int stride = NW * BK;
    fetch(wave * BK);
    for (int k0 = wave * BK; k0 < k_len; k0 += stride) {
        if (k0 + BK > k_len) {
            const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (k0 + 16 * h + 4 * lq >= k_len) {   // (zeros in one operand would do but for infinities in the other's copies)
                    xa[0][h] = xa[1][h] = zero4;
#pragma unroll
                    for (int j = 0; j < 4; ++j) xb[h * 4 + j] = zero4;
                }
        }
        auto join = [&](const f32x4_t& x0, const f32x4_t& x1, mfma_bf16x8 (&f)[3]) {
            u32x2_t s0[3], s1[3];
            split3(x0, s0);
            split3(x1, s1);
#pragma unroll
            for (int q = 0; q < 3; ++q) f[q] = __builtin_bit_cast(mfma_bf16x8, u32x4_t{s0[q][0], s0[q][1], s1[q][0], s1[q][1]});
        };
        mfma_bf16x8 fa[2][3], fb[4][3];
#pragma unroll
        for (int i = 0; i < 2; ++i) join(xa[i][0], xa[i][1], fa[i]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if (B_KC) join(xb[j], xb[4 + j], fb[j]);
            else join(f32x4_t{xb[0][j], xb[1][j], xb[2][j], xb[3][j]}, f32x4_t{xb[4][j], xb[5][j], xb[6][j], xb[7][j]}, fb[j]);
        }
        fetch(k0 + stride);
        auto mma = [&](int qa, int qb, mfma_f32x4 (&c)[2][4]) {
#pragma unroll
            for (int j = 0; j < 4; ++j)
#pragma unroll
                for (int i = 0; i < 2; ++i) c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[j][qb], fa[i][qa], c[i][j], 0, 0, 0);
        };
        mma(0, 0, hi);
        mma(1, 0, lo);
        mma(2, 0, lo);
        mma(0, 1, lo);
        mma(1, 1, lo);
        mma(0, 2, lo);
    }

    // the wavefronts' sums, 16 rows at a time.  Lane (lq, l16) holds row l16 and, for j and v, column j * 16 + 4 lq + v (K-contiguous) or
    // 16 lq + 4 v + j (K-strided): four neighbouring columns are one vector.
    bool finite = true;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (i) __syncthreads();
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            f32x4_t c;
#pragma unroll
            for (int w = 0; w < 4; ++w) c[w] = B_KC ? hi[i][u][w] + lo[i][u][w] : hi[i][w][u] + lo[i][w][u];
            red[wave][u * 64 + lane] = c;
        }
        __syncthreads();
        if (tid < 256) {
            f32x4_t c = red[0][tid];
#pragma unroll
            for (int w = 1; w < NW; ++w) c += red[w][tid];
            c *= SUM_SCALE;
            finite = finite && finite4(c);
            const int l = tid & 63, u = tid >> 6;
            const int row = m0 + i * 16 + (l & 15), col = n0 + (B_KC ? u * 16 + 4 * (l >> 4) : 16 * (l >> 4) + 4 * u);
            if (row < mend && col < p.N) {
                *reinterpret_cast<f32x4_t*>(p.C + (long long)row * p.ldc + col) = c;
                if constexpr (GATED) store_gated(p, row, col, c);
            }
        }
    }
    if (!__syncthreads_or(!finite) || wave) return;
    redo_exact(32, 64, k_len,
               [&](int i, int k) {
                   const int gr = min(m0 + i, mend - 1);
                   return p.A + (long long)(p.a_row_map ? p.a_row_map[gr] : gr) * p.lda + k;
               },
               [&](int k, int j) { return B_KC ? Bb + (long long)min(n0 + j, p.N - 1) * p.ldb + k : Bb + (long long)k * p.ldb + min(n0 + j, p.N - 1); },
               [&](int i, int j, float c) {
                   if (m0 + i < mend && n0 + j < p.N) p.C[(long long)(m0 + i) * p.ldc + n0 + j] = c;
               });
    if constexpr (GATED) store_gated_again(p, m0, mend, n0, 32, 64);
}

// Up to how many tiles of the last round are worked off in parts, behind `full` others.  A part takes more than a quarter of a tile's time, with B^T, which it
// reads straight into registers in pieces of a row, more yet.  8 x 512, 8 x 480, 16 x 256 and 39 x 100 rows, K from 512 to 4096, times as fast in parts
// as whole, A B / A B^T / gated, by the tiles on a compute unit: 1.07 to 1.13 1.18-1.23 / 1.14-1.17 / 1.16-1.25; 1.22 to 1.25 0.98-1.17 / 1.00-1.11 / 1.12-1.17; 1.38
// 0.91-1.12 (up to K = 1024 0.91-0.98, in another run 1.04-1.10) / 0.87-1.00 / 1.03-1.10; 1.5 0.91-1.16 / 0.75-0.99 / 0.90-1.09; 2.1 1.22-1.29 / 1.18-1.25 / 1.23-1.31; 2.38 to 2.5
// 1.08-1.14 / 1.02-1.06 / 1.06-1.14; 2.6 1.01-1.06 / 0.91-0.95 / 1.00-1.06; 2.75 1.00-1.06 / 0.88-0.95 / 0.98-1.03; 3.2 1.07-1.17 / 1.03-1.09 / 1.05-1.12; 3.5
// 0.99-1.10 / 0.92-1.00 / 0.99-1.04; 3.6 0.97-1.03 / 0.88-0.94 / 0.96-1.00; 4.5 1.01-1.05 / 0.97-1.01 / 1.01-1.04; 5.2 1.03-1.08 / 1.00-1.06 / 1.01-1.08;
// 5.5 1.01-1.03 / 0.92-1.00 / 1.00-1.02; 5.75 0.97-1.00 / 0.93-0.95 / 0.95-1.00.  One line for A B and gated, whose sums are the same.  (us: down product of 8 x 512 rows, K = 1024, 288 tiles 55.4 / 46.1.)
__host__ __device__ __forceinline__ int most_in_parts(int cus, int full, bool b_kc)
{
    const int rounds = full / cus;
    const int sixteenths = b_kc ? (rounds == 1 ? 4 : rounds == 2 ? 8 : 5) : rounds == 1 ? 7 : rounds == 2 ? 10 : 8;
    return cus * sixteenths / 16;
}

// ------------------------------------------------------------------ row-grouped products
// Four wavefronts of 32 rows x 64 columns.  Each loads its rows of A straight into registers and splits them there; B is
// split once for all four and goes through LDS.
template <bool B_KC, int KG, bool GATED>
__global__ void __launch_bounds__(NT * KG, 2)
grouped_gemm_f32_kernel(GemmArgsF32 p)
{
    typedef Stage<B_KC, BN_ROWS> SB;
    constexpr int TN = BN_ROWS / 16;
    constexpr uint32_t stage_bytes = 3 * SB::plane;
    constexpr uint32_t sum_bytes = (KG - 1) * BM_ROWS * BN_ROWS * 4;
    __shared__ __attribute__((aligned(1024))) char smem[2 * KG * stage_bytes > sum_bytes ? 2 * KG * stage_bytes : sum_bytes];
    const int group = KG == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / NT);
    const uint32_t lds = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem + (uint32_t)group * 2 * stage_bytes;
    const int tid = KG == 1 ? threadIdx.x : threadIdx.x % NT, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int l16 = lane & 15, lq = lane >> 4;
    const int total = min(*p.n_mtiles, p.max_mtiles) * p.n_ntiles;
    int tile = blockIdx.x;
    if (KG == 1 && p.cus) {
        // The last round's tiles, if they are few, as four workgroups of 32 rows each: a round lasts as long as a tile.
        const int full = total - total % p.cus;
        if (full && total - full <= most_in_parts(p.cus, full, B_KC) && tile >= full) {
            const int sub = (tile - full) & 3;
            tile = full + ((tile - full) >> 2);
            if (tile >= total) return;
            const int pm = tile / p.n_ntiles;
            const int4 tm = p.tile_map[pm];
            if (tm.y + sub * 32 >= tm.z) return;
            deep_tile<B_KC, GATED, NT / 64>(p, tm, tm.y + sub * 32, (tile - pm * p.n_ntiles) * BN_ROWS, reinterpret_cast<f32x4_t(*)[4 * 64]>(smem));
            return;
        }
    }
    if (tile >= total) return;
    const int pm = tile / p.n_ntiles, nt = tile - pm * p.n_ntiles;
    const int4 tm = p.tile_map[pm];
    const int m0 = tm.y + wave * 32, mend = tm.z, n0 = nt * BN_ROWS, k_len = p.Kd;
    const bool live = m0 < mend;
    const float* const Bb = p.B + (long long)tm.x * p.strideB;

    // Rows, columns and k past the end are copies of the last ones: the products of the first two are not stored, the last
    // are set to zero before they are split.  (No load is behind a branch: its result would pass through a copy, and the
    // copy awaits it.)
    // (Row scales as well: behind the stores of an epilogue a load waits for them too.)
    const float* a_ptr[2];
    float scale[2] = {1.0f, 1.0f};
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        int gr = min(m0 + i * 16 + l16, mend - 1);
        if (GATED && p.row_scale) scale[i] = p.row_scale[gr];
        if (p.a_row_map) gr = p.a_row_map[gr];
        a_ptr[i] = p.A + (long long)gr * p.lda;
    }
    const float* b_ptr[SB::NV];
    const int b_k = SB::start(tid);
#pragma unroll
    for (int v = 0; v < SB::NV; ++v) b_ptr[v] = B_KC ? Bb + (long long)min(n0 + SB::line(tid, v), p.N - 1) * p.ldb : Bb + min(n0 + b_k, p.N - 4);

    struct Vectors {
        f32x4_t a[2][2], b[SB::NV];
    };
    auto fetch = [&](Vectors& x, int k0) {
#pragma unroll
        for (int v = 0; v < SB::NV; ++v)
            x.b[v] = *reinterpret_cast<const f32x4_t*>(b_ptr[v] + (B_KC ? (long long)min(k0 + b_k, k_len - 4) : (long long)min(k0 + SB::line(tid, v), k_len - 1) * p.ldb));
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < 2; ++i) x.a[i][h] = *reinterpret_cast<const f32x4_t*>(a_ptr[i] + min(k0 + 16 * h + 4 * lq, k_len - 4));
    };
    auto cut = [&](Vectors& x, int k0) {
        const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < SB::NV; ++v)
            if (k0 + (B_KC ? b_k : SB::line(tid, v)) >= k_len) x.b[v] = zero4;
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (k0 + 16 * h + 4 * lq >= k_len) x.a[0][h] = x.a[1][h] = zero4;
    };

    // hi: the products of the leading parts; lo: the five smaller ones, added at the end
    mfma_f32x4 hi[2][TN], lo[2][TN];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) hi[i][j] = lo[i][j] = mfma_f32x4{0.f, 0.f, 0.f, 0.f};

    // Splits x (the stage from k0 on), requests the one after the next into it, and multiplies.
    auto step = [&](Vectors& x, int k0, uint32_t at) {
        if (k0 + BK > k_len) cut(x, k0);
#pragma unroll
        for (int v = 0; v < SB::NV; ++v) SB::put(at, tid, v, x.b[v]);
        mfma_bf16x8 fa[3][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            u32x2_t s0[3], s1[3];
            split3(x.a[i][0], s0);
            split3(x.a[i][1], s1);
#pragma unroll
            for (int q = 0; q < 3; ++q) fa[q][i] = __builtin_bit_cast(mfma_bf16x8, u32x4_t{s0[q][0], s0[q][1], s1[q][0], s1[q][1]});
        }
        fetch(x, k0 + 2 * KG * BK);
        lds_sync();   // (of the two LDS stages the other is written next: whoever still reads it has not passed this barrier)
        if (live) {
            mfma_bf16x8 fb[3][TN];
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[q][j] = SB::read(at + q * SB::plane, j * 16, l16, lq);
            auto mma = [&](int qa, int qb, mfma_f32x4 (&c)[2][TN]) {
#pragma unroll
                for (int j = 0; j < TN; ++j)
#pragma unroll
                    for (int i = 0; i < 2; ++i) c[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[qb][j], fa[qa][i], c[i][j], 0, 0, 0);
            };
            mma(0, 0, hi);
            mma(1, 0, lo);
            mma(2, 0, lo);
            mma(0, 1, lo);
            mma(1, 1, lo);
            mma(0, 2, lo);
        }
    };
    Vectors x0, x1;
    fetch(x0, group * BK);
    fetch(x1, (KG + group) * BK);
    for (int k0 = 0; k0 < k_len; k0 += 2 * KG * BK) {   // (the same number of steps for every group: those past the end are of zeros)
        step(x0, k0 + group * BK, lds);
        if (k0 + KG * BK < k_len) step(x1, k0 + (KG + group) * BK, lds + stage_bytes);
    }

    if constexpr (KG > 1) {   // the other groups' sums, added in their order
        __syncthreads();
        f32x4_t* const sums = reinterpret_cast<f32x4_t*>(smem);
        if (group) {
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) sums[(((group - 1) * 2 + i) * TN + j) * NT + tid] = hi[i][j] + lo[i][j];
        }
        __syncthreads();
        if (group) return;
#pragma unroll
        for (int g = 0; g < KG - 1; ++g)
#pragma unroll
            for (int i = 0; i < 2; ++i)
#pragma unroll
                for (int j = 0; j < TN; ++j) hi[i][j] += sums[((g * 2 + i) * TN + j) * NT + tid];
    }

    // Lane (lq, l16) holds columns 4 lq .. + 3 of row l16 of each 16 x 16 tile.
    bool finite = true;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
        if (m0 + i * 16 >= mend) break;
        const int row = m0 + i * 16 + l16;
        f32x2_t h[TN];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const f32x4_t c = (hi[i][j] + lo[i][j]) * SUM_SCALE;
            finite = finite && finite4(c);
            const int col = n0 + j * 16 + 4 * lq;
            if (row < mend && col < p.N) *reinterpret_cast<f32x4_t*>(p.C + (long long)row * p.ldc + col) = c;
            if constexpr (GATED) h[j] = gated(p, scale[i], c);
        }
        if constexpr (GATED) {
            // of tiles j and j + 1 lane quarters 0 and 2 take j's columns, 1 and 3 the other's: 16 bytes a lane, 64 of a row together
#pragma unroll
            for (int j = 0; j < TN; j += 2) {
                f32x4_t x;
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    const auto t = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[j][v]), __float_as_uint(h[j + 1][v]), false, false);
                    x[v] = __uint_as_float(t[0]);
                    x[2 + v] = __uint_as_float(t[1]);
                }
                const int col = n0 / 2 + (j + (lq & 1)) * 8 + (lq >> 1) * 4;
                if (row < mend && 2 * col < p.N) *reinterpret_cast<f32x4_t*>(p.inter + (long long)row * (p.N / 2) + col) = x;
            }
        }
    }
    if (!live || !__any(!finite)) return;
    redo_exact(32, BN_ROWS, k_len,
               [&](int i, int k) {
                   const int gr = min(m0 + i, mend - 1);
                   return p.A + (long long)(p.a_row_map ? p.a_row_map[gr] : gr) * p.lda + k;
               },
               [&](int k, int j) { return B_KC ? Bb + (long long)min(n0 + j, p.N - 1) * p.ldb + k : Bb + (long long)k * p.ldb + min(n0 + j, p.N - 1); },
               [&](int i, int j, float c) {
                   if (m0 + i < mend && n0 + j < p.N) p.C[(long long)(m0 + i) * p.ldc + n0 + j] = c;
               });
    if constexpr (GATED) store_gated_again(p, m0, mend, n0, 32, BN_ROWS);
}

// The same products where 128 x 64 tiles do not give every compute unit two workgroups: a wavefront on its own issues a
// vector instruction in twice the time that two take in turn.  A workgroup is 32 rows (a part of a map's tile) x 64 columns.
constexpr int NW_DEEP = 8;

template <bool B_KC, bool GATED>
__global__ void __launch_bounds__(NW_DEEP * 64, 2)
grouped_gemm_f32_deep_kernel(GemmArgsF32 p)
{
    __shared__ f32x4_t red[NW_DEEP][4 * 64];
    const int sub = blockIdx.x / p.n_ntiles;
    const int n0 = (blockIdx.x - sub * p.n_ntiles) * 64;
    const int pm = sub / (BM_ROWS / 32);
    if (pm >= *p.n_mtiles) return;
    const int4 tm = p.tile_map[pm];
    const int m0 = tm.y + (sub % (BM_ROWS / 32)) * 32;
    if (m0 >= tm.z) return;
    deep_tile<B_KC, GATED, NW_DEEP>(p, tm, m0, n0, red);
}

// ------------------------------------------------------------------ weight gradients
// C[e] = A[rows_e,:]^T @ B[rows_e,:], both operands K-strided and through LDS; four wavefronts of BM / 2 x BN / 2.
// MAPS: 1 = the rows of A, 2 = the rows of B are gathered through a row map
template <int BM, int BN, int MAPS>
__global__ void __launch_bounds__(NT, 2)
grouped_gemm_f32_wgrad_kernel(GemmArgsF32 p)
{
    typedef Stage<false, BM> SA;
    typedef Stage<false, BN> SB;
    constexpr int TM = BM / 32, TN = BN / 32;
    __shared__ __attribute__((aligned(1024))) char smem[3 * (SA::plane + SB::plane)];
    const uint32_t lds_a = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) void*)smem, lds_b = lds_a + 3 * SA::plane;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1;
    const int l16 = lane & 15, lq = lane >> 4;
    const int pm = blockIdx.x / p.n_ntiles, nt = blockIdx.x - pm * p.n_ntiles;
    const int e = pm / p.n_mt;
    const int m0 = (pm - e * p.n_mt) * BM, n0 = nt * BN;
    const int r0 = p.offsets[e], k_len = p.offsets[e + 1] - r0;
    float* const Cb = p.C + (long long)e * p.strideC;

    // (rows and columns past the end as above)
    const float* const a_ptr = (MAPS == 1 ? p.A : p.A + (long long)r0 * p.lda) + min(m0 + SA::start(tid), p.M - 4);
    const float* const b_ptr = (MAPS == 2 ? p.B : p.B + (long long)r0 * p.ldb) + min(n0 + SB::start(tid), p.N - 4);
    struct Vectors {
        f32x4_t a[SA::NV], b[SB::NV];
    };
    typedef std::conditional_t<MAPS == 2, SB, SA> SG;
    int idx[SG::NV];                          // gathered rows of the stage that is fetched next
    auto fetch_idx = [&](int k0) {
        if constexpr (MAPS != 0) {
#pragma unroll
            for (int v = 0; v < SG::NV; ++v) idx[v] = (MAPS == 1 ? p.a_row_map : p.b_row_map)[r0 + min(k0 + SG::line(tid, v), k_len - 1)];
        }
    };
    auto fetch = [&](Vectors& x, int k0) {
        const float *pa[SA::NV], *pb[SB::NV];
#pragma unroll
        for (int v = 0; v < SA::NV; ++v) pa[v] = a_ptr + (long long)(MAPS == 1 ? idx[v] : min(k0 + SA::line(tid, v), k_len - 1)) * p.lda;
#pragma unroll
        for (int v = 0; v < SB::NV; ++v) pb[v] = b_ptr + (long long)(MAPS == 2 ? idx[v] : min(k0 + SB::line(tid, v), k_len - 1)) * p.ldb;
        fetch_idx(k0 + BK);                   // (ahead of the loads: they stay in flight when it is awaited)
#pragma unroll
        for (int v = 0; v < SA::NV; ++v) x.a[v] = *reinterpret_cast<const f32x4_t*>(pa[v]);
#pragma unroll
        for (int v = 0; v < SB::NV; ++v) x.b[v] = *reinterpret_cast<const f32x4_t*>(pb[v]);
    };
    auto cut = [&](Vectors& x, int k0) {
        const f32x4_t zero4 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int v = 0; v < SA::NV; ++v)
            if (k0 + SA::line(tid, v) >= k_len) x.a[v] = zero4;
#pragma unroll
        for (int v = 0; v < SB::NV; ++v)
            if (k0 + SB::line(tid, v) >= k_len) x.b[v] = zero4;
    };

    mfma_f32x4 hi[TM][TN], lo[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) hi[i][j] = lo[i][j] = mfma_f32x4{0.f, 0.f, 0.f, 0.f};
    if (k_len > 0) {   // (an expert without rows has a gradient of zeros)
        Vectors x;
        fetch_idx(0);
        fetch(x, 0);
        for (int k0 = 0; k0 < k_len; k0 += BK) {
            if (k0 + BK > k_len) cut(x, k0);
            lds_sync();   // (the stage is read before it is written again)
#pragma unroll
            for (int v = 0; v < SA::NV; ++v) SA::put(lds_a, tid, v, x.a[v]);
#pragma unroll
            for (int v = 0; v < SB::NV; ++v) SB::put(lds_b, tid, v, x.b[v]);
            lds_sync();
            fetch(x, k0 + BK);
            mfma_bf16x8 fb[3][TN];
#pragma unroll
            for (int q = 0; q < 3; ++q)
#pragma unroll
                for (int j = 0; j < TN; ++j) fb[q][j] = SB::read(lds_b + q * SB::plane, wn * (BN / 2) + j * 16, l16, lq);
#pragma unroll
            for (int qa = 0; qa < 3; ++qa) {
                mfma_bf16x8 fa[TM];
#pragma unroll
                for (int i = 0; i < TM; ++i) fa[i] = SA::read(lds_a + qa * SA::plane, wm * (BM / 2) + i * 16, l16, lq);
#pragma unroll
                for (int qb = 0; qb < 3 - qa; ++qb)
#pragma unroll
                    for (int j = 0; j < TN; ++j)
#pragma unroll
                        for (int i = 0; i < TM; ++i) {
                            mfma_f32x4& c = qa + qb ? lo[i][j] : hi[i][j];
                            c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[qb][j], fa[i], c, 0, 0, 0);
                        }
            }
        }
    }
    bool finite = true;
    const int mw = m0 + wm * (BM / 2), nw = n0 + wn * (BN / 2);
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const f32x4_t c = (hi[i][j] + lo[i][j]) * SUM_SCALE;
            finite = finite && finite4(c);
            const int row = mw + i * 16 + l16, col = nw + j * 16 + 4 * lq;
            if (row < p.M && col < p.N) *reinterpret_cast<f32x4_t*>(Cb + (long long)row * p.ldc + col) = c;
        }
    if (!__any(!finite)) return;
    redo_exact(BM / 2, BN / 2, k_len,
               [&](int i, int k) { return p.A + (long long)(MAPS == 1 ? p.a_row_map[r0 + k] : r0 + k) * p.lda + min(mw + i, p.M - 1); },
               [&](int k, int j) { return p.B + (long long)(MAPS == 2 ? p.b_row_map[r0 + k] : r0 + k) * p.ldb + min(nw + j, p.N - 1); },
               [&](int i, int j, float c) {
                   if (mw + i < p.M && nw + j < p.N) Cb[(long long)(mw + i) * p.ldc + nw + j] = c;
               });
}

template <int BM, int BN, int MAPS>
int launch_wgrad(GemmArgsF32 a, hipStream_t s)
{
    a.n_mt = (a.M + BM - 1) / BM;
    a.n_ntiles = (a.N + BN - 1) / BN;
    const long long grid = (long long)a.E * a.n_mt * a.n_ntiles;
    AMOE_REQUIRE(grid < (1ll << 31), AMOE_ERR_UNSUPPORTED, "grouped_gemm_wgrad(f32): grid too large");
    hipLaunchKernelGGL((grouped_gemm_f32_wgrad_kernel<BM, BN, MAPS>), dim3((int)grid), dim3(NT), 0, s, a);
    return amoe_check_launch("grouped_gemm_wgrad_f32");
}
template <int BM, int BN>
int launch_wgrad(const GemmArgsF32& a, hipStream_t s)
{
    if (a.a_row_map) return launch_wgrad<BM, BN, 1>(a, s);
    return a.b_row_map ? launch_wgrad<BM, BN, 2>(a, s) : launch_wgrad<BM, BN, 0>(a, s);
}

template <bool B_KC, bool GATED = false>
void launch_rows(const GemmArgsF32& a, int grid, int form, hipStream_t s)
{
    if (form == 2) hipLaunchKernelGGL((grouped_gemm_f32_deep_kernel<B_KC, GATED>), dim3(grid * (BM_ROWS / 32)), dim3(NW_DEEP * 64), 0, s, a);
    else if (form == 1) hipLaunchKernelGGL((grouped_gemm_f32_kernel<B_KC, 2, GATED>), dim3(grid), dim3(NT * 2), 0, s, a);
    else hipLaunchKernelGGL((grouped_gemm_f32_kernel<B_KC, 1, GATED>), dim3(grid), dim3(NT), 0, s, a);
}

}  // namespace

// rows mode: C[rows_e, :N] = A[rows_e, :Kred] @ op(B[e]);  b_kc selects B stored [N,Kred]; inter (B as it is only): the gated activation too
int amoe_f32_rows(const void* A, const int32_t* a_row_map, const void* B, const int32_t* offsets, void* C, int R, int E,
                  int Kred, int N, int ldb, long long strideB, bool b_kc, void* workspace, size_t workspace_bytes,
                  bool map_ready, hipStream_t s, float* inter, const float* row_scale, int act)
{
    GemmArgsF32 a = {};
    a.inter = inter;
    a.row_scale = row_scale;
    a.act = act;
    int max_mtiles = 0;
    // map_ready (AMOE_TILE_MAP_READY): the workspace already holds the map for these offsets, nothing is launched
    int rc = amoe_build_tile_map(offsets, R, E, BM_ROWS, workspace, workspace_bytes, &a.tile_map, &a.n_mtiles, &max_mtiles, s,
                                 map_ready);
    if (rc) return rc;
    a.A = (const float*)A;
    a.B = (const float*)B;
    a.C = (float*)C;
    a.a_row_map = a_row_map;
    a.offsets = offsets;
    a.lda = Kred;
    a.ldb = ldb;
    a.ldc = N;
    a.strideB = strideB;
    a.E = E;
    a.Kd = Kred;
    a.M = R;
    a.N = N;
    a.n_ntiles = (N + BN_ROWS - 1) / BN_ROWS;
    a.max_mtiles = max_mtiles;
    long long grid = (long long)max_mtiles * a.n_ntiles;
    AMOE_REQUIRE(grid * (BM_ROWS / 32) < (1ll << 31), AMOE_ERR_UNSUPPORTED, "grouped_gemm(f32): grid too large");
    // Few tiles, which the wavefronts of a compute unit then have to share.  One MI355X, us (with 11 instructions for two values), one group of wavefronts / two groups / the
    // eight-wave form:
    //   32 x 64 tiles (an expert's last one is not full) up to 400: 8 experts, 256 rows, K = 1024, N = 512 29.6 / 24.1 / 11.1; 38 experts,
    //   497 rows, K = 800, N = 288 24.1 / 20.8 / 18.0; past the line K = 288, N = 800 13.6 / 20.5 / 20.4.
    //   128 x 64 tiles (the last one half full) up to 256: 4 experts, 1000 rows, K = 2048, N = 1024 66 / 49 / 48, K = 4096 119 / 88 / 136;
    //   9 experts, 1380 rows, K = 1888, N = 736 59 / 46 / 61; past the line 8 experts, 4096 rows, K = 2048, N = 512 89 / 101 / 122.
    const long long met = E < R ? E : R;
    int form = 0;
    if ((R / 32 + met) * a.n_ntiles <= 400) form = 2;
    else if ((R / 128 + met / 2 + 1) * a.n_ntiles <= 256 && Kred >= 512) form = 1;
    const int cus = device_cu_count();
    if (form == 0 && cus > 0 && grid > cus) {
        a.cus = cus;
        grid += 3 * most_in_parts(cus, 2 * cus, b_kc);   // (two whole rounds: the most)
    }
    if (inter) launch_rows<false, true>(a, (int)grid, form, s);
    else if (b_kc) launch_rows<true>(a, (int)grid, form, s);
    else launch_rows<false>(a, (int)grid, form, s);
    return amoe_check_launch("grouped_gemm_f32");
}

int amoe_f32_wgrad(const void* A, const int32_t* a_row_map, const void* B, const int32_t* b_row_map,
                   const int32_t* offsets, void* C, int R, int E, int Kd, int N, hipStream_t s)
{
    GemmArgsF32 a = {};
    a.a_row_map = a_row_map;
    a.b_row_map = b_row_map;
    a.A = (const float*)A;
    a.B = (const float*)B;
    a.C = (float*)C;
    a.offsets = offsets;
    a.lda = Kd;
    a.ldb = N;
    a.ldc = N;
    a.strideC = (long long)Kd * N;
    a.E = E;
    a.M = Kd;
    a.N = N;
    // The large tile splits and stages half as much per product, where there are two of it for every compute unit and enough
    // rows to reduce over: 8 experts of 512 rows, 512 x 2048 (512 tiles) 58 against 72 us, 39 of 709, 768 x 1856 494 / 609, 44 of
    // 334, 512 x 512 67 / 65, 8 of 512, 1024 x 512 (256 tiles) 43 / 42, 38 of 13, 800 x 288 17 / 14.
    if ((long long)E * ((Kd + 127) / 128) * ((N + 127) / 128) >= 512 && R >= 128ll * E) return launch_wgrad<128, 128>(a, s);
    return launch_wgrad<64, 64>(a, s);
}
