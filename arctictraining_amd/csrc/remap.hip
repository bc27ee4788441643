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
// Pure byte movement, HBM bound: 64 x 64 tiles go through LDS so that both the reads and the
// writes are 16-byte accesses along the contiguous dimension of their tensor.
//
// Experts that are modules of their own are read and written where their weights lie (Listed below): at E=128, H=2048,
// I=768 in bf16 a layer's 2 x 1.21 GB take 474 us in and 489 us out, 5.0-5.1 TB/s; stacked copies and copies into the
// parameters beside the kernels took 1.79 and 2.15 ms.
#include "amoe_common.h"

namespace {

constexpr int TILE = 64;

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

// T is the element as raw bits (uint16_t / uint32_t); V = elements per 16-byte access
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
                    const vec_t x = *reinterpret_cast<const vec_t*>(src + (long long)i * H + h);
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
                *reinterpret_cast<vec_t*>(dst + (long long)h * (G * I) + c) = *reinterpret_cast<const vec_t*>(&tile[hh][cv]);
        }
    } else {
        constexpr int VPJ = G * TILE / V;
        const T* src = joint + (long long)e * joint_es;
        for (int v = tid; v < TILE * VPJ; v += 256) {
            const int hh = v / VPJ, cv = (v % VPJ) * V;
            const int h = h0 + hh, c = G * i0 + cv;
            if (h < H && c < G * I)
                *reinterpret_cast<vec_t*>(&tile[hh][cv]) = *reinterpret_cast<const vec_t*>(src + (long long)h * (G * I) + c);
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
                    *reinterpret_cast<vec_t*>(dst + (long long)i * H + h) = x;
                }
            }
        }
    }
}

template <typename T, typename SPLIT>
void launch(bool pack, bool two, const SPLIT& split, void* joint, int E, int I, int H, hipStream_t s)
{
    const dim3 grid((H + TILE - 1) / TILE, (I + TILE - 1) / TILE, E), block(256);
    const long long joint_es = (long long)H * I * (two ? 2 : 1);
    T* j = (T*)joint;
    if (pack && two) hipLaunchKernelGGL((remap_kernel<T, 2, true, SPLIT>), grid, block, 0, s, split, j, I, H, joint_es);
    else if (pack) hipLaunchKernelGGL((remap_kernel<T, 1, true, SPLIT>), grid, block, 0, s, split, j, I, H, joint_es);
    else if (two) hipLaunchKernelGGL((remap_kernel<T, 2, false, SPLIT>), grid, block, 0, s, split, j, I, H, joint_es);
    else hipLaunchKernelGGL((remap_kernel<T, 1, false, SPLIT>), grid, block, 0, s, split, j, I, H, joint_es);
}

int launch_strided(bool pack, const void* s0, const void* s1, void* joint, int dtype, int E, int I, int H, long long es, void* stream)
{
    const Strided split = {{s0, s1}, es};
    if (dtype != AMOE_F32) launch<uint16_t>(pack, s1 != nullptr, split, joint, E, I, H, (hipStream_t)stream);
    else launch<uint32_t>(pack, s1 != nullptr, split, joint, E, I, H, (hipStream_t)stream);
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
        if (dtype != AMOE_F32) launch<uint16_t>(pack, s1 != nullptr, split, j, n, I, H, (hipStream_t)stream);
        else launch<uint32_t>(pack, s1 != nullptr, split, j, n, I, H, (hipStream_t)stream);
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
