// Expert-weight re-layout between the checkpoint format of the original MoE blocks and the
// unified ArcticMoE parameters (arctic_training/model/moe/utils.py:249-266 and :366-395):
//
//   pack    out[e][h][G*i + g] = in_g[e][i][h]     nn.Linear weights [out=I, in=H] of the gate
//                                                  (g=0) and up (g=1) projections -> the
//                                                  interleaved expert_gate_up [E, H, 2I];
//                                                  G = 1 is a plain batched transpose
//                                                  (down_proj [E, H, I] -> expert_down [E, I, H])
//   unpack  out_g[e][i][h] = in[e][h][G*i + g]     the inverse, for saving a checkpoint
//
// Pure byte movement, HBM bound: tiles go through LDS so that both the reads and the writes are 16-byte accesses along
// the contiguous dimension of their tensor, and every byte passes once: both sides bypass the caches' replacement order
// (a linear copy of 1 GB takes 5.8 TB/s with ordinary accesses and 6.35 with these).
//
// Experts that are modules of their own are read and written where their weights lie (Listed below): at E=128, H=2048,
// I=768 in bf16 a layer's 2 x 1.21 GB take 426 us in and 427 us out, 5.7 TB/s (with 64 x 64 tiles, 2-byte LDS accesses
// and ordinary loads and stores 474 and 489 us); stacked copies and copies into the parameters beside the kernels took
// 1.79 and 2.15 ms.
#include "amoe_common.h"

#include <type_traits>

namespace {

constexpr int TILE = 64;   // (of 4-byte elements)

// Where the per-expert matrices of the split side are: a strided tensor, or one address each.  The addresses of up to
// kListExperts experts travel as kernel arguments (2 KB: no copy to the device, nothing to keep alive).
constexpr int kListExperts = 128;
struct Strided {
    const void* p[2];
    long long es;   // expert stride in elements
    template <typename T>
    __device__ __forceinline__ T* at(int g, int e) const { return (T*)p[g] + (long long)e * es; }
};
struct Listed {
    const void* p[2][kListExperts];
    template <typename T>
    __device__ __forceinline__ T* at(int g, int e) const { return (T*)p[g][e]; }
};

// 2-byte elements: TH = 256 (or 128) columns h by 64 dwords of two elements that lie side by side in the joint side, (gate, up) of one
// i, or i and i + 1 of a single projection.  A thread moves two rows' 16-byte vectors, interleaved in registers, so that
// LDS sees dwords; 16-byte chunk c of LDS row h is kept at c ^ ((h / 8) % 16), which spreads a wavefront's dwords (8 rows
// apart) over all banks.  Wide tiles for long pieces: with 128 or 64 columns the split side is accessed in pieces of 256
// or 128 bytes instead of 512, and gate and up of the size above take 288 or 298 us, with 256 270.
// NT: threads.  Export of more than a few tiles takes 512, each with half of the vectors: twice the wavefronts stand on a compute
// unit, which holds two tiles either way.  A launch (32 experts) of gate and up / of down, us, 256 / 512: 2048 x 768 70.1 / 68.0 and 37.1 /
// 35.9, 2048 x 1408 123 / 121 and 66 / 65, 4096 x 14336 (8 experts) 638 / 626 and 356 / 343, 608 x 864 (1344 and 640 tiles) 26.0 /
// 25.4 and 16.4 / 16.6, 512 x 160 (192 and 128) 5.6 / 6.2 and 5.0 / 4.8, 1024 x 512 (9 experts, 288 and 144) 9.1 / 8.9 and 5.4 / 6.0.  Import so
// 70 / 71 and 36 / 37.
template <int TH, int G, bool PACK, int NT, typename SPLIT>
__global__ void __launch_bounds__(NT) remap16_kernel(SPLIT split, uint16_t* __restrict__ joint, int I, int H, long long joint_es)
{
    constexpr int W = 64, ROWS = W * 2 / G;     // dwords of a joint row, rows i
    constexpr int NS = W * TH / 8 / NT, NJ = TH * W / 4 / NT;
    __shared__ __attribute__((aligned(16))) uint32_t tile[TH * W];
    typedef uint32_t vec_t __attribute__((ext_vector_type(4)));
    const int tid = threadIdx.x;
    const int h0 = blockIdx.x * TH, i0 = blockIdx.y * ROWS, e = blockIdx.z;
    uint16_t* const row0 = split.template at<uint16_t>(0, e);
    uint16_t* const row1 = G == 2 ? split.template at<uint16_t>(1, e) : row0 + H;
    uint16_t* const j = joint + (long long)e * joint_es;
    auto at = [](int h, int d) { return h * W + (((d >> 2) ^ (h >> 3)) & 15) * 4 + (d & 3); };
    // vector n of this thread: split side, rows of dword d and column h; joint side, row h and column c
    auto split_at = [&](int n, int& d, int& hh, long long& off) {
        const int v = tid + n * NT;
        d = v / (TH / 8);
        hh = v % (TH / 8) * 8;
        const int i = i0 + (G == 2 ? d : 2 * d);
        off = (long long)i * H + h0 + hh;
        return i < I && h0 + hh < H;
    };
    auto joint_at = [&](int n, int& hh, int& d, long long& off) {
        const int v = tid + n * NT;
        hh = v / (W / 4);
        d = v % (W / 4) * 4;
        const int c = G * i0 + 2 * d;
        off = (long long)(h0 + hh) * (G * I) + c;
        return h0 + hh < H && c < G * I;
    };
    int d, hh;
    long long off;
    if (PACK) {
        vec_t a[NS], b[NS];
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            if (split_at(n, d, hh, off)) {
                a[n] = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(row0 + off));
                b[n] = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(row1 + off));
            }
        }
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            split_at(n, d, hh, off);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                tile[at(hh + 2 * k, d)] = __builtin_amdgcn_perm(b[n][k], a[n][k], 0x05040100);
                tile[at(hh + 2 * k + 1, d)] = __builtin_amdgcn_perm(b[n][k], a[n][k], 0x07060302);
            }
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NJ; ++n) {
            if (joint_at(n, hh, d, off))
                __builtin_nontemporal_store(*reinterpret_cast<const vec_t*>(&tile[at(hh, d)]), reinterpret_cast<vec_t*>(j + off));
        }
    } else {
        vec_t x[NJ];
#pragma unroll
        for (int n = 0; n < NJ; ++n) {
            const bool in = joint_at(n, hh, d, off);
            // (eight vectors without a branch, what is past the end a copy of the first: around branches the compiler keeps them as
            // one value of 232 registers)
            if (NJ <= 8 || in) x[n] = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(j + (in ? off : 0)));
        }
#pragma unroll
        for (int n = 0; n < NJ; ++n) {
            joint_at(n, hh, d, off);
            *reinterpret_cast<vec_t*>(&tile[at(hh, d)]) = x[n];
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NS; ++n) {
            const bool in = split_at(n, d, hh, off);
            vec_t a, b;
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                const uint32_t p = tile[at(hh + 2 * k, d)], q = tile[at(hh + 2 * k + 1, d)];
                a[k] = __builtin_amdgcn_perm(q, p, 0x05040100);
                b[k] = __builtin_amdgcn_perm(q, p, 0x07060302);
            }
            if (in) {
                __builtin_nontemporal_store(a, reinterpret_cast<vec_t*>(row0 + off));
                __builtin_nontemporal_store(b, reinterpret_cast<vec_t*>(row1 + off));
            }
        }
    }
}

// 4-byte elements, as raw bits; V = elements per 16-byte access
template <typename T, int G, bool PACK, typename SPLIT>
__global__ void __launch_bounds__(256)
remap_kernel(SPLIT split /* the [E,I,H] side */, T* __restrict__ joint /* the [E,H,G*I] side */, int I, int H, long long joint_es)
{
    constexpr int V = 16 / sizeof(T);
    constexpr int PAD = V;                       // keeps rows 16-byte aligned and staggers the banks
    // joint-side tile: TILE rows (h) x G*TILE columns; split-side tiles: G x TILE rows (i) x TILE columns (h)
    __shared__ __attribute__((aligned(16))) T tile[TILE][G * TILE + PAD];   // [hh][G*ii + g]
    const int tid = threadIdx.x;
    const int h0 = blockIdx.x * TILE, i0 = blockIdx.y * TILE, e = blockIdx.z;
    typedef T vec_t __attribute__((ext_vector_type(16 / sizeof(T))));

    if (PACK) {
        // read the split side: for each g, rows i, 16-byte vectors along h
        constexpr int VPR = TILE / V;            // vectors per row
        for (int g = 0; g < G; ++g) {
            const T* __restrict__ src = split.template at<const T>(g, e);
            for (int v = tid; v < TILE * VPR; v += 256) {
                const int ii = v / VPR, hv = (v % VPR) * V;
                const int i = i0 + ii, h = h0 + hv;
                if (i < I && h < H) {
                    const vec_t x = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(src + (long long)i * H + h));
#pragma unroll
                    for (int k = 0; k < V; ++k) tile[hv + k][G * ii + g] = x[k];
                }
            }
        }
        __syncthreads();
        // write the joint side: rows h, 16-byte vectors along the G*I columns
        constexpr int VPJ = G * TILE / V;
        T* dst = joint + (long long)e * joint_es;
        for (int v = tid; v < TILE * VPJ; v += 256) {
            const int hh = v / VPJ, cv = (v % VPJ) * V;
            const int h = h0 + hh, c = G * i0 + cv;
            if (h < H && c < G * I)
                __builtin_nontemporal_store(*reinterpret_cast<const vec_t*>(&tile[hh][cv]), reinterpret_cast<vec_t*>(dst + (long long)h * (G * I) + c));
        }
    } else {
        constexpr int VPJ = G * TILE / V;
        const T* src = joint + (long long)e * joint_es;
        for (int v = tid; v < TILE * VPJ; v += 256) {
            const int hh = v / VPJ, cv = (v % VPJ) * V;
            const int h = h0 + hh, c = G * i0 + cv;
            if (h < H && c < G * I)
                *reinterpret_cast<vec_t*>(&tile[hh][cv]) = __builtin_nontemporal_load(reinterpret_cast<const vec_t*>(src + (long long)h * (G * I) + c));
        }
        __syncthreads();
        constexpr int VPR = TILE / V;
        for (int g = 0; g < G; ++g) {
            T* __restrict__ dst = split.template at<T>(g, e);
            for (int v = tid; v < TILE * VPR; v += 256) {
                const int ii = v / VPR, hv = (v % VPR) * V;
                const int i = i0 + ii, h = h0 + hv;
                if (i < I && h < H) {
                    vec_t x;
#pragma unroll
                    for (int k = 0; k < V; ++k) x[k] = tile[hv + k][G * ii + g];
                    __builtin_nontemporal_store(x, reinterpret_cast<vec_t*>(dst + (long long)i * H + h));
                }
            }
        }
    }
}

template <int G, bool PACK, typename SPLIT>
void launch(bool wide, const SPLIT& split, void* joint, int E, int I, int H, hipStream_t s)
{
    const long long joint_es = (long long)H * I * G;
    if (wide) {
        const dim3 grid((H + TILE - 1) / TILE, (I + TILE - 1) / TILE, E);
        hipLaunchKernelGGL((remap_kernel<uint32_t, G, PACK, SPLIT>), grid, dim3(256), 0, s, split, (uint32_t*)joint, I, H, joint_es);
    } else {
        // Narrow tiles where wide ones would leave most of their lanes idle.  64 matrices each of gate and up, 0.6 GB in all, import /
        // export, us, narrow / wide: H = 64 201 / 248 and 206 / 220, 96 208 / 219 and 206 / 221, 288 239 / 254 and 229 / 254, 320 211 / 233 and
        // 208 / 245, 384 213 / 233 and 205 / 231; past the lines 160 262 / 219 and 248 / 219, 416 245 / 243, 512 223 / 215, 2048 218 / 208.
        // (64 x 64 tiles: 244 and 239 at 288.)  Rows that are no multiple of 64 bytes are exported
        // faster by wide tiles: 272 309 / 300, 296 346 / 308.
        const bool narrow = H <= 96 || (H > 256 && H <= 384 && (PACK || H % 32 == 0));
        auto run = [&](auto TH, auto NT) {
            const dim3 grid((H + TH - 1) / TH, (I * G + 127) / 128, E);
            hipLaunchKernelGGL((remap16_kernel<decltype(TH)::value, G, PACK, decltype(NT)::value, SPLIT>), grid, dim3(NT), 0, s, split, (uint16_t*)joint, I, H, joint_es);
        };
        typedef std::integral_constant<int, 128> N128;
        typedef std::integral_constant<int, 256> N256;
        const long long tiles = (long long)((H + 255) / 256) * ((I * G + 127) / 128) * E;
        if (narrow) run(N128{}, N256{});
        else if (PACK || tiles < 1024) run(N256{}, N256{});
        else run(N256{}, std::integral_constant<int, PACK ? 256 : 512>{});
    }
}

template <typename SPLIT>
void launch(bool pack, bool two, bool wide, const SPLIT& split, void* joint, int E, int I, int H, hipStream_t s)
{
    if (pack && two) launch<2, true>(wide, split, joint, E, I, H, s);
    else if (pack) launch<1, true>(wide, split, joint, E, I, H, s);
    else if (two) launch<2, false>(wide, split, joint, E, I, H, s);
    else launch<1, false>(wide, split, joint, E, I, H, s);
}

int launch_strided(bool pack, const void* s0, const void* s1, void* joint, int dtype, int E, int I, int H, long long es, void* stream)
{
    const Strided split = {{s0, s1}, es};
    launch(pack, s1 != nullptr, dtype == AMOE_F32, split, joint, E, I, H, (hipStream_t)stream);
    return amoe_check_launch(pack ? "remap_pack" : "remap_unpack");
}

int check(const char* what, const void* p0, const void* p1, int dtype, int E, int I, int H, long long split_es)
{
    AMOE_REQUIRE(p0 && p1, AMOE_ERR_BAD_ARG, "%s: null pointer", what);
    AMOE_REQUIRE(dtype == AMOE_F32 || dtype == AMOE_BF16 || dtype == AMOE_F16, AMOE_ERR_BAD_ARG, "%s: bad dtype %d", what, dtype);
    AMOE_REQUIRE(E > 0 && I > 0 && H > 0, AMOE_ERR_BAD_ARG, "%s: sizes must be positive (E=%d I=%d H=%d)", what, E, I, H);
    AMOE_REQUIRE(E <= 65535 && (I + TILE - 1) / TILE <= 65535, AMOE_ERR_UNSUPPORTED, "%s: grid too large", what);
    const int v = dtype != AMOE_F32 ? 8 : 4;
    AMOE_REQUIRE(I % v == 0 && H % v == 0, AMOE_ERR_UNSUPPORTED, "%s: I=%d and H=%d must be multiples of %d", what, I, H, v);
    AMOE_REQUIRE(split_es >= (long long)I * H && split_es % v == 0, AMOE_ERR_BAD_ARG,
                 "%s: expert stride %lld must be at least I*H and a multiple of %d", what, split_es, v);
    return AMOE_OK;
}

}  // namespace

AMOE_EXPORT int amoe_remap_pack(const void* in0, const void* in1, void* out, int dtype, int E, int I, int H,
                                long long in_expert_stride, void* stream)
{
    int rc = check("amoe_remap_pack", in0, out, dtype, E, I, H, in_expert_stride);
    if (rc) return rc;
    return launch_strided(true, in0, in1, out, dtype, E, I, H, in_expert_stride, stream);
}

AMOE_EXPORT int amoe_remap_unpack(const void* in, void* out0, void* out1, int dtype, int E, int I, int H,
                                  long long out_expert_stride, void* stream)
{
    int rc = check("amoe_remap_unpack", in, out0, dtype, E, I, H, out_expert_stride);
    if (rc) return rc;
    return launch_strided(false, out0, out1, const_cast<void*>(in), dtype, E, I, H, out_expert_stride, stream);
}

// The same with the split side as a list of matrices, one (or one of each of two) per expert.
static int remap_list(const char* what, bool pack, const void* const* s0, const void* const* s1, void* joint, int dtype, int E,
                      int I, int H, void* stream)
{
    int rc = check(what, s0, joint, dtype, E, I, H, (long long)I * H);
    if (rc) return rc;
    for (int e = 0; e < E; ++e)
        AMOE_REQUIRE(s0[e] && (!s1 || s1[e]), AMOE_ERR_BAD_ARG, "%s: null pointer (expert %d)", what, e);
    const size_t esz = dtype != AMOE_F32 ? 2 : 4;
    for (int e0 = 0; e0 < E; e0 += kListExperts) {
        const int n = E - e0 < kListExperts ? E - e0 : kListExperts;
        Listed split = {};
        for (int e = 0; e < n; ++e) {
            split.p[0][e] = s0[e0 + e];
            split.p[1][e] = s1 ? s1[e0 + e] : nullptr;
        }
        char* j = (char*)joint + (size_t)e0 * H * I * (s1 ? 2 : 1) * esz;
        launch(pack, s1 != nullptr, dtype == AMOE_F32, split, j, n, I, H, (hipStream_t)stream);
    }
    return amoe_check_launch(what);
}

AMOE_EXPORT int amoe_remap_pack_list(const void* const* in0, const void* const* in1, void* out, int dtype, int E, int I, int H,
                                     void* stream)
{
    return remap_list("amoe_remap_pack_list", true, in0, in1, out, dtype, E, I, H, stream);
}

AMOE_EXPORT int amoe_remap_unpack_list(const void* in, void* const* out0, void* const* out1, int dtype, int E, int I, int H,
                                       void* stream)
{
    return remap_list("amoe_remap_unpack_list", false, out0, out1, const_cast<void*>(in), dtype, E, I, H, stream);
}
