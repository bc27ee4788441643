// The 16-bit grouped GEMMs at the default tile shape, 256 x 256 x 64 on v_mfma_f32_16x16x32, f32 accumulate.
//
// 512 threads = two groups of four wavefronts, one wavefront of each group per SIMD.  A K tile is worked off in
// four phases, one quadrant of the output each; a phase is a memory part (LDS reads of the operands the phase
// needs, direct-to-LDS loads of the K tile after the next, and, at a tile's end, the epilogue of the quadrant
// finished one phase before) and an arithmetic part (16 MFMAs back to back).  The second group runs one part
// behind the first, held there by the workgroup barrier after every part: while one wavefront of a SIMD issues
// MFMAs, the other does everything else, so reads, loads and the epilogue's conversions and stores sit under
// the matrix pipe instead of between its bursts.
#include "gemm_dma.h"
#include "wgrad_deal.h"

#ifndef AMOE_PP_PART
#define AMOE_PP_PART -1
#endif
#define AMOE_PP_PART_IS(n) (AMOE_PP_PART < 0 || AMOE_PP_PART == (n))

namespace {

constexpr int PP_BM = 256, PP_BN = 256, PP_BK = 64;
constexpr int PP_THREADS = 512;
constexpr uint32_t PP_HALF = 128 * PP_BK * 2;        // bytes of a half tile: 128 rows (or columns) of one operand
constexpr uint32_t PP_STAGE = 4 * PP_HALF;           // A0 A1 B0 B1
constexpr uint32_t PP_IDX = 2 * PP_STAGE;            // row indices of the next tile, 64 per wavefront
constexpr uint32_t PP_SCALE = PP_IDX + 8 * 64 * 4;   // row scales of two tiles
constexpr uint32_t PP_PART = PP_SCALE + 2 * PP_BM * 4;   // row-sum partials, one row of 256 per wave column
constexpr uint32_t PP_TURN = PP_PART + 4 * PP_BM * 4;    // 2 KB a wavefront for its epilogue
constexpr uint32_t PP_LDS = PP_TURN + 8 * 2048;
constexpr uint32_t PP_WIDX = 2 * PP_STAGE + 8 * 2048;         // weight gradients: behind 2 KB a wavefront for its epilogue the indices of gathered rows
constexpr uint32_t PP_WDEPTH = PP_WIDX + 8 * 512;            // the experts' depths, and how their tiles are dealt
constexpr uint32_t PP_WDEAL = PP_WDEPTH + AMOE_MAX_EXPERTS * 4;
constexpr uint32_t PP_WLOAD = 2 * PP_STAGE;                  // (while they are worked out) the workgroups' loads by number and by depth
constexpr uint32_t PP_WGRAD_LDS = PP_WDEPTH, PP_WGRAD_DEAL_LDS = PP_WDEAL + AMOE_MAX_EXPERTS * 16;

// ------------------------------------------------------------------ row-grouped products
// C[rows_e,:] = A[rows_e,:] @ B[e] (B_KC false: B [Kd,N]) or @ B[e]^T (B_KC: B [N,Kd]).
// Persistent: one workgroup per CU walks its tiles, and the K loops of consecutive tiles form one stream of
// K tiles -- the loads run two K tiles ahead, across the tile boundary.
//
// LDS: a K tile is four half tiles of 128 x 64, two stages.  K-contiguous halves are [row][8 chunks of 16 B],
// chunk c of row r at c ^ ((r >> 1) & 7); K-strided halves are [k][16 chunks], chunk c of row k at
// c ^ 2 ((k & 3) | (((k >> 3) & 1) << 2)), read with the transposing LDS read.  Either way the 32 lanes that the
// LDS serves together meet every bank once.
//
// Wave (g, wc): g = group, wc = column quarter.  Quadrant (a, b): tile rows a*128.., columns b*128 + wc*32 ..+31.
// Products that are stored as they are (LINES): columns wc*64 ..+63, with B^T b*32 ..+31 of them; with B a half tile of B is not
// 128 columns, but all of them and 32 k ([k][32 chunks]), and the quadrants of a row half one k step each.
// The rows of a half are dealt to the groups in blocks of 16 (row = (a*4 + i)*32 + g*16 + l), so that a tile with
// fewer live rows spares both groups the same MFMAs.
//
// What bounds it: the memory part of a phase has to fit into the other group's 256 cycles of MFMA, so every
// instruction in it counts (range tests on the loads, waits chosen by a branch and branches around dead rows each
// cost 4-6 % of the K loop and are gone from it).  Measured on one MI355X, 131072 rows, N = 2048, bf16 NT: K = 8192
// 1.50-1.66 PFLOP/s (operands from HBM / from L2); K = 2048 1.23-1.43, K = 768 1.03: what a tile costs beside its K loop
// is 5 to 7 us.  The gated epilogues cost more: the gate_up product of K = 2048 runs at
// 0.96-1.08 (128 uneven / even experts; the library's plain product of that size at 1.0), the gated backward one at 0.87.  The kernel this one replaced (32-wide K tiles, 32x32x16 MFMAs, all
// eight waves in step) ran at 1.0-1.1 on the same problems.
template <bool B_KC, int EPI, int ACT, bool STREAM, typename ET>
__device__ __forceinline__ void pp_rows_body()
{
    typedef typename Elem16<ET>::frag_t frag_t;
    extern __shared__ u32x4_t smem[];
    const uint32_t lds = (uint32_t)(uintptr_t)(lptr_t)smem;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, wc = wave & 3;
    const int l16 = lane & 15, lq = lane >> 4;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I4 = std::integral_constant<int, 4>;
    constexpr bool PART = EPI == EPI_PART;
    constexpr bool PAST = EPI == EPI_STORE_PAST, LINES = EPI == EPI_STORE || PAST || PART, K_HALVES = LINES && !B_KC;
    auto divide = [](int n, uint32_t inv) -> int { return inv ? (int)(((uint64_t)(uint32_t)n * inv) >> 32) : n; };
    const int Kd = pp_args().Kd;
    const int KT_all = (Kd + PP_BK - 1) / PP_BK;
    // K tiles (of a short reduction, the last are empty).  EPI_PART: a part's, and part i has those from i KT_all / splits on, one
    // fewer in some (the launch sees to it that there are four at least)
    const int KT = PART ? divide(KT_all + pp_args().splits - 1, pp_args().inv_splits) : max(4, KT_all);
    const bool ragged_k = PART || Kd < KT * PP_BK;
    // B^T whose rows lie 4, 8 or 12 KB apart (launch_pp_rows): the 128 bytes of a K tile of all rows are in a few of the memory's
    // channels, and all workgroups ask for the same K tile at about the same time.  Expert e's reduction starts at K tile 5 e and goes
    // around, so that those in flight together are spread; one expert's tiles start together and share what they load.
    constexpr bool TURNED = B_KC && !PART;
    const int first_step = TURNED ? pp_args().first_step : 0;
    struct Part { int i, k0, kd; };                                // number, first k and length
    auto part_of = [&](int& nt) -> Part {                          // N tile of all parts -> of its part
        if constexpr (PART) {
            args_t& p = pp_args();
            const int i = divide(nt, p.inv_real);
            nt -= i * p.n_real;
            const int t0 = divide(i * KT_all, p.inv_splits), t1 = divide((i + 1) * KT_all, p.inv_splits);
            return {i, t0 * PP_BK, min(t1 * PP_BK, Kd) - t0 * PP_BK};
        }
        return {0, 0, Kd};
    };
    auto first_k_of = [&](int e) -> int {                          // (K tile)
        const int k = first_step * e;
        return k - divide(k, pp_args().inv_kt) * KT;
    };

    // ------------------------------------------------------------ this workgroup's tiles
    // The tiles that there are stand in one row: groups of gm tile rows, in a group super-columns of gn tiles (the last one
    // narrower), tile row by tile row inside them.  XCD x (the hardware deals workgroups to the XCDs round-robin) takes the x-th
    // eighth of each gridDim.x of them, so that its workgroups share the gm A panels and gn B panels of a super-tile in its L2.
    // The last, partial round's tiles of more than 6 blocks of 32 rows are cut into 2 or 4 pieces of whole blocks where there are
    // workgroups for them: a round lasts as long as its tallest tile.  (Lower ones are bound by reading the weights, and each piece
    // reads them: 188 rows an expert, gated backward of 1.5 rounds of tiles 181 us whole, 182 in halves.  A piece's weights are
    // not read past the caches.)
    // Before, blocks of a padded grid were dealt, super-tile by super-tile, whether there was a tile or not: of 968 tiles, 88 x 11,
    // some workgroups got five and others three.  Steps, before / now, ms: 4001 tokens of 64 experts of 2048 x 1408 and a shared
    // one 1.653 / 1.616, 8192 tokens of 8 experts of 4096 x 14336 (4.25 rounds in two products) 13.88 / 13.80, 32768 uneven
    // ones 6.607 / 6.537; alone, us, one expert of 4001 rows: gate_up 60 / 56, down 37 / 33, gated backward 63 / 57.
    // (a product with 2^32 / d rounded up gives n / d or, past n d = 2^32, one more)
    auto divide_any = [](int n, int d, uint32_t inv) -> int {
        const int q = inv ? (int)(((uint64_t)(uint32_t)n * inv) >> 32) : n;
        return q - (int)((uint32_t)q * (uint32_t)d > (uint32_t)n);
    };
    const int n_mtiles = min(scalar_load_i32(pp_args().n_mtiles), pp_args().max_mtiles);
    int round_first = 0;                 // first tile of the round dealt next
    // the next tile: its entry of the tile map (a piece's rows in it, and in w whether it is a piece) and N tile
    auto next_tile = [&](int4& tm, int& nt) -> bool {
        args_t& p = pp_args();
        const int total = n_mtiles * p.n_ntiles, left = total - round_first, grid = gridDim.x;
        const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
        int i, piece = 0, cut = 0;
        if (left >= grid) {
            i = round_first + xcd * (grid >> 3) + slot;
        } else {
            const int share = (max(left, 0) + 7) >> 3;        // an XCD's tiles; the first pieces of all, then the second ones ..
            cut = (share * 16 <= grid) + (share * 32 <= grid);
            piece = (slot >= share) + (slot >= 2 * share) + (slot >= 3 * share);
            const int q = xcd * share + slot - piece * share;
            if (slot >= share << cut || q >= left) return false;
            i = round_first + q;
        }
        round_first += grid;
        const int per_group = p.gm * p.n_ntiles;
        const int g = divide_any(i, per_group, p.inv_group);
        int r = i - g * per_group, pm = g * p.gm;
        if (pm + p.gm <= n_mtiles) {
            const int c = divide(r, p.inv_super);
            r -= c * p.gm * p.gn;
            const bool last = c == p.sn - 1;
            const int m = divide(r, last ? p.inv_last : p.inv_gn);
            pm += m;
            nt = c * p.gn + r - m * (last ? p.n_ntiles - c * p.gn : p.gn);
        } else {
            const int m = divide_any(r, p.n_ntiles, p.inv_n);
            pm += m;
            nt = r - m * p.n_ntiles;
        }
        const int32_t* ent = reinterpret_cast<const int32_t*>(p.tile_map + pm);
        tm.x = scalar_load_i32(ent);
        tm.y = scalar_load_i32(ent + 1);
        tm.z = scalar_load_i32(ent + 2);
        tm.w = 0;
        if (cut) {
            const int blocks = (tm.z - tm.y + 31) >> 5;
            const int rows = blocks > 6 ? ((blocks + (1 << cut) - 1) >> cut) * 32 : PP_BM;
            tm.w = blocks > 6;
            tm.y += piece * rows;
            if (tm.y >= tm.z) return false;           // (the last round: this workgroup is done)
            tm.z = min(tm.z, tm.y + rows);
        }
        return true;
    };

    // ------------------------------------------------------------ loads
    // Thread tid fills chunks tid and tid + 512 of every half tile.
    // Thread tid's: K-contiguous row tid / 8 (+ 64 j), k (tid % 8 ^ (row / 2) % 8) * 8; K-strided k row tid / 16 (+ 32 j).
    uint32_t aoff[2][2], boff[2][2];
    srd_t ad, bd;
    const int lda = pp_args().lda, ldb = pp_args().ldb, N = pp_args().N;
    const bf16_t* const A = pp_args().A;
    const bool gather = pp_args().a_row_map != nullptr;
    const uint32_t bstep = B_KC ? PP_BK * 2 : (uint32_t)ldb * (PP_BK * 2);
    // STREAM: the weights of an expert whose rows are one tile are read once, those of the others by several workgroups; all
    // the tiles' weights have to be more than the caches hold
    const bool stream = STREAM && n_mtiles >= pp_args().stream_from;
    bool stream_b = false, stream_n = false;
    auto expert_b = [&](const int4& tm) {
        args_t& p = pp_args();
        if (STREAM) stream_n = stream && tm.w == 0 && scalar_load_i32(p.offsets + tm.x + 1) - scalar_load_i32(p.offsets + tm.x) <= PP_BM;
        return p.B + (long long)tm.x * p.strideB;
    };
    // a plan without rows (m0 == mend) or columns (n0 >= N) reads nothing
    auto plan_a = [&](int m0, int mend, const int32_t* map, int k0) {     // map: the row map (first tile), else the indices are in LDS
        const int th = pp_here(tid);
        const int r = th >> 3, k = ((th & 7) ^ ((r >> 1) & 7)) * 8;
        // tile row of this thread's chunk in half a: (a*4 + i)*32 + j*16 + l with i = r / 16, l = r % 16
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = m0 + (a * 4 + (r >> 4)) * 32 + j * 16 + (r & 15);
                int gr = row;
                if (gather)
                    gr = map ? map[min(row, mend - 1)] : pp_lds<int>(lds + PP_IDX + (uint32_t)(wave * 64 + a * 16 + j * 8 + (r & 7)) * 4u);
                aoff[a][j] = row < mend && k < Kd ? ((uint32_t)gr * (uint32_t)lda + k) * 2u : PP_NOWHERE;
            }
        ad = pp_srd(A);
        if constexpr (PART || TURNED) pp_advance(ad, (uint32_t)k0 * 2u);
    };
    auto plan_b = [&](const bf16_t* B, int n0, int k0) {
        const int th = pp_here(tid);
        const int r = th >> 3, kr = K_HALVES ? th >> 5 : th >> 4;
        const int k = ((th & 7) ^ ((r >> 1) & 7)) * 8;
        const int col = ((K_HALVES ? th & 31 : th & 15) ^ (2 * ((kr & 3) | (((kr >> 3) & 1) << 2)))) * 8;
        bd = pp_srd(B);
        if (STREAM) stream_b = stream_n;
        // (an expert's matrix is below 4 GiB, or the call is refused: no offset in it wraps)
        if constexpr (PART || TURNED) pp_advance(bd, B_KC ? (uint32_t)k0 * 2u : (uint32_t)k0 * ((uint32_t)ldb * 2u));
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int row = LINES ? ((th >> 8) + 2 * j) * 64 + b * 32 + (r & 31) : b * 128 + r + 64 * j;
                const int n = n0 + (B_KC ? row : K_HALVES ? col : b * 128 + col);
                const int kb = B_KC ? k : K_HALVES ? kr + 32 * b + 16 * j : kr + 32 * j;
                const uint32_t o = B_KC ? (uint32_t)n * (uint32_t)ldb + k : (uint32_t)kb * (uint32_t)ldb + n;
                boff[b][j] = n < N && kb < Kd ? o * 2u : PP_NOWHERE;
            }
    };
    // the K tile loaded next holds only `left` of its 64 k (none at all if left <= 0)
    auto cut_k = [&](int left) {
        const int th = pp_here(tid);
        const int k = ((th & 7) ^ ((th >> 4) & 7)) * 8, kr = K_HALVES ? th >> 5 : th >> 4;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                if (k >= left) aoff[h][j] = PP_NOWHERE;
                if ((B_KC ? k : K_HALVES ? kr + 32 * h + 16 * j : kr + 32 * j) >= left) boff[h][j] = PP_NOWHERE;
            }
    };
    uint32_t fill = lds + (uint32_t)wave * 1024u;                  // this wave's place in the stage being filled
    auto dma_a = [&](auto A_) {
        constexpr int a = decltype(A_)::value;
        pp_dma16<a * PP_HALF>(ad, aoff[a][0], fill);
        pp_dma16<a * PP_HALF + 8192u>(ad, aoff[a][1], fill);
    };
    auto dma_b = [&](auto B_) {
        constexpr int b = decltype(B_)::value;
        if (STREAM && stream_b) {
            pp_dma16<(2 + b) * PP_HALF, true>(bd, boff[b][0], fill);
            pp_dma16<(2 + b) * PP_HALF + 8192u, true>(bd, boff[b][1], fill);
        } else {
            pp_dma16<(2 + b) * PP_HALF>(bd, boff[b][0], fill);
            pp_dma16<(2 + b) * PP_HALF + 8192u>(bd, boff[b][1], fill);
        }
    };
    int to_wrap = 0;                     // K tiles of the tile being loaded until its last one
    auto next_k = [&]() {
        fill ^= PP_STAGE;
        pp_advance(ad, PP_BK * 2);
        pp_advance(bd, bstep);
        if constexpr (TURNED) {
            const bool wrap = --to_wrap == 0;
            pp_go_back(ad, wrap ? (uint32_t)Kd * 2u : 0u);
            pp_go_back(bd, wrap ? (uint32_t)KT * bstep : 0u);
        }
    };

    // ------------------------------------------------------------ fragments
    // B: of a half of columns two 16-column tiles by two k steps, of a half of k four 16-column tiles
    frag_t fa[4][2], fb0[4], fb1[4];
    uint32_t ra[2], rb[K_HALVES ? 4 : 2];   // LDS read addresses: A per k step; B per k step (K-contiguous) or per 16-column tile
#pragma unroll
    for (int s = 0; s < 2; ++s) {
        const int row = grp * 64 + l16;
        ra[s] = lds + (uint32_t)(row * 8 + ((s * 4 + lq) ^ ((row >> 1) & 7))) * 16u;
        if (B_KC) {
            const int n = wc * 32 + l16;
            rb[s] = lds + 2 * PP_HALF + (uint32_t)(n * 8 + ((s * 4 + lq) ^ ((n >> 1) & 7))) * 16u;
        }
    }
    if constexpr (!B_KC) {
        const int k = 8 * lq + (l16 >> 2), key = 2 * ((l16 >> 2) | ((lq & 1) << 2));
#pragma unroll
        for (int j = 0; j < (K_HALVES ? 4 : 2); ++j)
            rb[j] = lds + 2 * PP_HALF + (uint32_t)(k * (K_HALVES ? 512 : 256) + (l16 & 1) * 8) +
                    (uint32_t)(((wc * (K_HALVES ? 8 : 4)) + 2 * j + ((l16 & 3) >> 1)) ^ key) * 16u;
    }
    auto flip = [&]() {
#pragma unroll
        for (uint32_t& r : ra) r ^= PP_STAGE;
#pragma unroll
        for (uint32_t& r : rb) r ^= PP_STAGE;
    };
    auto read_a = [&](auto A_, auto N_) {
#pragma unroll
        for (int i = 0; i < decltype(N_)::value; ++i)
#pragma unroll
            for (int s = 0; s < 2; ++s)
                fa[i][s] = __builtin_bit_cast(frag_t, pp_lds<u32x4_t>(ra[s] + decltype(A_)::value * PP_HALF + i * 2048u));
    };
    auto read_b = [&](auto H_, frag_t (&fb)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            if constexpr (B_KC) {
                fb[j] = __builtin_bit_cast(frag_t, pp_lds<u32x4_t>(rb[j & 1] + decltype(H_)::value * PP_HALF + (j >> 1) * 2048u));
            } else {
                const uint32_t ad = (K_HALVES ? rb[j] : rb[j >> 1] + (j & 1) * 8192u) + decltype(H_)::value * PP_HALF;
                typedef __attribute__((address_space(3))) i16x4_t* tr_ptr;
                const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)ad));
                const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)(ad + (K_HALVES ? 2048u : 1024u))));
                fb[j] = __builtin_bit_cast(frag_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
            }
        }
    };
    // FIRST: the tile's first K tile, nothing to add to
    auto mma = [&](auto FIRST, auto H_, auto N_, mfma_f32x4 (&c)[4][4], const frag_t (&fb)[4]) {
        constexpr int h = decltype(H_)::value;
        constexpr bool first = decltype(FIRST)::value;
        if constexpr (!K_HALVES) {
#pragma unroll
            for (int s = 0; s < 2; ++s)
#pragma unroll
                for (int i = 0; i < decltype(N_)::value; ++i)
#pragma unroll
                    for (int j = 0; j < 2; ++j)
                        c[i][2 * h + j] = Mfma16<ET>::run(fb[2 * j + s], fa[i][s], first && s == 0 ? mfma_f32x4{0.f, 0.f, 0.f, 0.f} : c[i][2 * h + j]);
        } else {
#pragma unroll
            for (int i = 0; i < decltype(N_)::value; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) c[i][j] = Mfma16<ET>::run(fb[j], fa[i][h], first && h == 0 ? mfma_f32x4{0.f, 0.f, 0.f, 0.f} : c[i][j]);
        }
    };

    // ------------------------------------------------------------ tile state
    int m0, mend, nt = 0, n0;
    Part part, part_n;                   // this tile's part of the reduction, the next one's
    bool have_n, have_nn = false;        // is there a next tile, and one after it
    int nt_n = 0, nt_nn = 0;
    int4 tm_n, tm_nn = make_int4(0, 0, 0, 0);
    const bf16_t* b_n = nullptr;
    {
        int4 tm;
        if (!next_tile(tm, nt)) return;
        m0 = tm.y;
        mend = tm.z;
        have_n = next_tile(tm_n, nt_n);
        if (!have_n) tm_n = make_int4(0, 0, 0, 0);
        part = part_of(nt);
        if constexpr (TURNED) {
            to_wrap = KT - first_k_of(tm.x);
            part.k0 = (KT - to_wrap) * PP_BK;
        }
        n0 = nt * PP_BN;
        plan_a(m0, mend, pp_args().a_row_map, part.k0);
        plan_b(expert_b(tm), n0, part.k0);
    }
    int par = 0;            // row scales: which of the two LDS rows is this tile's
    bool sums_due = false;  // row-sum partials of the previous tile are complete in LDS and not yet written
    int sums_m0 = 0, sums_end = 0, sums_nt = 0;

    // ------------------------------------------------------------ epilogue of quadrant (a, b)
    // Lane (lq, l16) holds columns 4 lq ..+3 of both 16-column tiles j for row l16 of every 16-row block.
    // What the four quadrants share is worked out during the last K tile but one.
    // Blocks of 32 rows without a live row are left out: the arithmetic of the gated epilogues is 4 us (gate_up) and 13 us (gated backward)
    // of a whole tile, beside which no MFMA runs.  32 rows an expert, 128 experts of 2048 x 768, us: gate_up 165 / 156, gated backward
    // 134 / 119, down 90 / 86, with B^T 170 / 165; a training step of 509 tokens 835 / 798, a forward pass of 3001 342 / 338.
    // The gate_up epilogue asks once whether any block is (WHOLE): asked at each of its 16, a short reduction of large tiles pays for it
    // (K = 512, 180000 rows, N = 2048 398 us before, 402-405 with a test each, 396 so; K = 608, 120000 rows, N = 1792 265 / 272 / 267).
    // LINES: a wavefront's columns of the tile are 64 in a row (else 32 of either half), 128 bytes of the output.  Through 2 KB of LDS
    // of its own (chunk c of row r at c ^ (r & 7), its halves the other way round from row 8 on: no bank conflicts) eight lanes
    // come to hold a row's, and a store writes whole lines.  Adjacent lanes in adjacent rows, as the accumulators have them, are a
    // request each.  Alone, us, before / so: 131072 rows of 128 experts, 768 x 2048 453 / 425, 1536 x 2048 with B^T 737 / 706;
    // 16004 of 64, 1408 x 2048 138 / 130.  Steps, past the caches as well where launch_pp_rows says so, ms: those 3.993 / 3.922, 17484
    // tokens x 7 of 21 experts of 4288 x 480 5.03 / 4.93, 25086 rows of 55 experts of 4352 x 160 0.836 / 0.802; outputs of 45 MB
    // past them as well 0.136 / 0.141 (what reads them next finds nothing in the caches).
    // (The gated epilogues are bound by their arithmetic, and the turn through LDS comes on top: gate_up 831 / 827-860 us.)
    bf16_t *e_c, *e_c2;      // this wave's first element of the tile in the outputs (gated backward: d_gate_up, and gate_up)
    int e_ldc = 0, e_ldc2 = 0, e_cols = 0, e_rows = 0;
    uint32_t e_off = 0, e_off2 = 0;
    auto prepare_epilogue = [&]() {
        args_t& p = pp_args();
        const int le = pp_here(lane);
        const int rl = grp * 16 + (le & 15), eq = le >> 4;
        const int c0 = n0 + wc * (LINES ? 64 : 32);
        e_cols = N - c0;                 // columns of the wave's part that exist, from its first one (N is a multiple of 8)
        e_rows = mend - m0;
        if (PART) {
            e_ldc = p.N * 2;             // in elements of 16 bits, as below
            e_c = reinterpret_cast<bf16_t*>(p.split_out + ((long long)part.i * p.M + m0) * p.N + c0);
            e_off = (uint32_t)(rl * p.N + 4 * eq) * 4u;
        } else if (EPI == EPI_GATED_BWD) {
            e_ldc = p.ldg;
            e_c = p.C + (long long)m0 * e_ldc + 2 * c0;
            e_c2 = const_cast<bf16_t*>(p.G) + (long long)m0 * e_ldc + 2 * c0;
            e_off = (uint32_t)(rl * e_ldc + 8 * eq) * 2u;
        } else {
            e_ldc = p.ldc;
            e_c = p.C;
            if (LINES || e_c) e_c += (long long)m0 * e_ldc + c0;
            e_off = LINES ? (uint32_t)((grp * 16 + (le >> 3)) * e_ldc + 8 * (le & 7)) * 2u : (uint32_t)(rl * e_ldc + 8 * eq) * 2u;
            if (EPI == EPI_GATED) {
                e_ldc2 = p.ldc2;
                e_c2 = p.C2 + (long long)m0 * e_ldc2 + (c0 >> 1);
                e_off2 = (uint32_t)(rl * e_ldc2 + 4 * eq) * 2u;
            }
        }
    };
    u32x4_t gu[2][4][2];     // gated backward: gate_up of two quadrants, requested ahead of their epilogues
    auto fetch_gate_up = [&](auto A_, auto B_) {
        constexpr int a = decltype(A_)::value, b = decltype(B_)::value;
        if constexpr (EPI == EPI_GATED_BWD) {
            const int le = pp_here(lane);
            const int eq = le >> 4, rl = grp * 16 + (le & 15);
            const __amdgpu_buffer_rsrc_t g = __builtin_amdgcn_make_buffer_rsrc(e_c2, (short)0, (int)PP_DROP, 0x00020000);
#pragma unroll
            for (int i = 0; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    const bool ok = b * 128 + 16 * j + 4 * eq < e_cols && (a * 4 + i) * 32 + rl < e_rows;
                    gu[b][i][j] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(
                                                               g, ok ? e_off + j * 64u : PP_DROP, (a * 4 + i) * (uint32_t)e_ldc * 64u + b * 512u, 0));
                }
        }
    };
    float dots[4] = {0.f, 0.f, 0.f, 0.f};
    auto epilogue = [&](auto A_, auto B_, const mfma_f32x4 (&acc)[4][4], auto WHOLE) {
        constexpr int a = decltype(A_)::value, b = decltype(B_)::value;
        constexpr bool whole = decltype(WHOLE)::value;      // every block has a live row
        const int le = pp_here(lane);
        const int eq = le >> 4, rl = grp * 16 + (le & 15);
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(e_c, (short)0, (int)PP_DROP, 0x00020000);
        const uint32_t srow = (uint32_t)e_ldc * 64u;           // bytes of 32 rows
        if constexpr (LINES) {
            // (b: blocks 2 b and 2 b + 1, all columns)
#pragma unroll
            for (int i = 2 * b; i < 2 * b + 2; ++i) {
                pp_fence();
                if ((a * 4 + i) * 32 >= e_rows) break;
                const uint32_t soff = (a * 4 + i) * srow;
                const int rows = e_rows - (a * 4 + i) * 32;
                if constexpr (PART) {
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        pp_store16(d, __builtin_bit_cast(u32x4_t, acc[i][j]), 16 * j + 4 * eq < e_cols && rl < rows ? e_off + j * 64u : PP_DROP, soff);
                } else {
                    const int r16 = le & 15, r8 = le >> 3;
                    const uint32_t at = lds + PP_TURN + (uint32_t)wave * 2048u;
                    const uint32_t wr = at + (uint32_t)(r16 * 128 + (((le >> 5) ^ (r16 & 7)) * 16) + (((le >> 4) ^ (r16 >> 3)) & 1) * 8);
                    const uint32_t rd = at + (uint32_t)(r8 * 128 + ((le & 7) ^ r8) * 16);
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        *(__attribute__((address_space(3))) u32x2_t*)(uintptr_t)(wr ^ (32u * j)) =
                            u32x2_t{Elem16<ET>::pack2(acc[i][j][0], acc[i][j][1]), Elem16<ET>::pack2(acc[i][j][2], acc[i][j][3])};
                    pp_lds_turn();
                    const u32x4_t v0 = pp_lds<u32x4_t>(rd), v1 = pp_lds<u32x4_t>(rd + 1024u);
                    pp_lds_turn();
                    const bool ok = 8 * (le & 7) < e_cols;
                    pp_store16<PAST>(d, v0, ok && grp * 16 + r8 < rows ? e_off : PP_DROP, soff);
                    pp_store16<PAST>(d, u32x4_t{v1[2], v1[3], v1[0], v1[1]}, ok && grp * 16 + 8 + r8 < rows ? e_off : PP_DROP, soff + 16u * (uint32_t)e_ldc);
                }
            }
        } else if constexpr (EPI == EPI_GATED_BWD) {
            // d_inter is in the accumulators; the (gate, up) pairs of its columns come back from the forward pass
            auto place = [&](int j, int i) {
                return b * 128 + 16 * j + 4 * eq < e_cols && (a * 4 + i) * 32 + rl < e_rows ? e_off + j * 64u : PP_DROP;
            };
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pp_fence();   // (left alone, the scheduler interleaves the activation chains and their temporaries spill)
                if ((a * 4 + i) * 32 >= e_rows) break;
                const float s = pp_lds<float>(lds + PP_SCALE + (uint32_t)(par * PP_BM + (a * 4 + i) * 32 + rl) * 4u);
                float dot = 0.f;
#pragma unroll
                for (int j = 0; j < 2; ++j) {
                    u32x4_t o;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const float dd = acc[i][2 * b + j][v];
                        const float gate = Elem16<ET>::lo(gu[b][i][j][v]), up = Elem16<ET>::hi(gu[b][i][j][v]);
                        float f, df;
                        act_both_fast<ACT>(gate, f, df);
                        dot += dd * up * f;
                        const float sd = s * dd;
                        o[v] = Elem16<ET>::pack2(sd * up * df, sd * f);
                    }
                    pp_store16(d, o, place(j, i), (a * 4 + i) * srow + b * 512u);
                    pp_fence();
                }
                dots[i] = b == 0 ? dot : dots[i] + dot;
                asm volatile("" : "+v"(dots[i]));   // (summed up here: put off to its use, the sum holds on to all its terms)
                if (b == 1) {
                    const float t = pp_quarter_sum(dots[i]);
                    if (eq == 0) *(__attribute__((address_space(3))) float*)(uintptr_t)(lds + PP_PART + (uint32_t)(wc * PP_BM + (a * 4 + i) * 32 + rl) * 4u) = t;
                }
            }
            if (b == 1) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        } else {
            const __amdgpu_buffer_rsrc_t d2 = __builtin_amdgcn_make_buffer_rsrc(e_c2, (short)0, (int)PP_DROP, 0x00020000);
            const uint32_t srow2 = (uint32_t)e_ldc2 * 64u;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                pp_fence();
                if (!whole && (a * 4 + i) * 32 >= e_rows) break;
                const bool ok = b * 128 + 8 * eq < e_cols && (a * 4 + i) * 32 + rl < e_rows;
                uint32_t x[2], y[2];
#pragma unroll
                for (int v = 0; v < 2; ++v) {
                    x[v] = Elem16<ET>::pack2(acc[i][2 * b][2 * v], acc[i][2 * b][2 * v + 1]);
                    y[v] = Elem16<ET>::pack2(acc[i][2 * b + 1][2 * v], acc[i][2 * b + 1][2 * v + 1]);
                }
                // a packed pair is (gate, up) of one intermediate column
                const float s = pp_lds<float>(lds + PP_SCALE + (uint32_t)(par * PP_BM + (a * 4 + i) * 32 + rl) * 4u);
                uint32_t hx = Elem16<ET>::pack2(s * Elem16<ET>::hi(x[0]) * act_fwd_fast<ACT>(Elem16<ET>::lo(x[0])),
                                                s * Elem16<ET>::hi(x[1]) * act_fwd_fast<ACT>(Elem16<ET>::lo(x[1])));
                uint32_t hy = Elem16<ET>::pack2(s * Elem16<ET>::hi(y[0]) * act_fwd_fast<ACT>(Elem16<ET>::lo(y[0])),
                                                s * Elem16<ET>::hi(y[1]) * act_fwd_fast<ACT>(Elem16<ET>::lo(y[1])));
                pp_join(hx, hy);
                __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{hx, hy}, d2, ok ? e_off2 : PP_DROP, (a * 4 + i) * srow2 + b * 128u, 0);
                pp_join(x[0], y[0]);
                pp_join(x[1], y[1]);
                if (e_c) pp_store16(d, u32x4_t{x[0], x[1], y[0], y[1]}, ok ? e_off : PP_DROP, (a * 4 + i) * srow + b * 256u);
            }
        }
    };
    // the row sums of a finished tile: each group adds up its own rows' four wave columns
    auto write_sums = [&]() {
        if constexpr (EPI == EPI_GATED_BWD) {
            args_t& p = pp_args();
            if (sums_due && p.partials) {
                const int lane = pp_here(tid) & 63;
                const int w = wc * 32 + (lane & 31);                       // 128 rows of this group
                const int row = (w >> 4) * 32 + grp * 16 + (w & 15);
                float t = 0.f;
#pragma unroll
                for (int c = 0; c < 4; ++c) t += pp_lds<float>(lds + PP_PART + (uint32_t)(c * PP_BM + row) * 4u);
                if (lane < 32 && sums_m0 + row < sums_end) p.partials[(long long)sums_nt * p.part_stride + sums_m0 + row] = t;
            }
            sums_due = false;
        }
    };

    // ------------------------------------------------------------ one tile
    // The waits: phase n awaits the loads issued in phase n - 5, which the next phase reads after the barrier; ten younger
    // loads stay in flight.  (Epilogue stores count as well and are not allowed for: letting them stay in flight through
    // the first K tile was measured and gains nothing.)
    auto run_tile = [&]() {
        mfma_f32x4 acc[2][4][4];
        // ---- phase 0 of the first K tile
        read_a(I0{}, I4{});
        dma_a(I1{});
        next_k();
        {
            args_t& p = pp_args();
            const int le = pp_here(lane);
            if (!LINES && wave < 4) {
                const int row = wave * 64 + le;
                const uint32_t dst = lds + PP_SCALE + (uint32_t)(par * PP_BM + wave * 64) * 4u;
                if (p.row_scale) {
                    dma4_sbase(p.row_scale, (uint32_t)min(m0 + row, mend - 1) * 4u, dst);
                } else {
                    *(__attribute__((address_space(3))) float*)(uintptr_t)(dst + le * 4u) = 1.0f;
                }
            }
            if (p.a_row_map && have_n) {
                const int q = le & 31, r = wave * 8 + (q & 7);
                const int row = ((q >> 4) * 4 + (r >> 4)) * 32 + ((q >> 3) & 1) * 16 + (r & 15);
                dma4_sbase(p.a_row_map, (uint32_t)min(tm_n.y + row, tm_n.z - 1) * 4u, lds + PP_IDX + (uint32_t)wave * 256u);
            }
        }
        pp_vmwait<10>();
        pp_barrier();
        mma(T_{}, I0{}, I4{}, acc[0], fb0);
        {
            // the next tile's weights; which tile follows it, and its entry of the tile map
            b_n = expert_b(tm_n);
            part_n = part_of(nt_n);
            if constexpr (TURNED) part_n.k0 = first_k_of(tm_n.x) * PP_BK;
            have_nn = have_n && next_tile(tm_nn, nt_nn);
            if (!have_nn) tm_nn = make_int4(0, 0, 0, 0);
        }
        pp_barrier();
        write_sums();
        // K tile t (t < KT - 1): phases 1..3, and phase 0 of the next; loads K tile t + 2, with TURN (t = KT - 2) the
        // next tile's first one
        auto k_tile = [&](auto FIRST, auto TURN, auto N_) {
            constexpr bool turn = decltype(TURN)::value;
            // phase 1
            read_b(I1{}, fb1);
            if (turn) plan_b(b_n, have_n ? nt_n * PP_BN : 0x7fffff00, have_n ? part_n.k0 : 0);
            dma_b(I0{});
            pp_vmwait<10>();
            pp_barrier();
            mma(FIRST, I1{}, I4{}, acc[0], fb1);
            pp_barrier();
            // phase 2
            read_a(I1{}, N_);
            if (turn) {
                plan_a(tm_n.y, tm_n.z, nullptr, have_n ? part_n.k0 : 0);
                if constexpr (TURNED) to_wrap = KT - part_n.k0 / PP_BK;
            }
            dma_a(I0{});
            pp_vmwait<10>();
            pp_barrier();
            mma(FIRST, I0{}, N_, acc[1], fb0);
            pp_barrier();
            // phase 3
            flip();
            read_b(I0{}, fb0);
            dma_b(I1{});
            pp_vmwait<10>();
            pp_barrier();
            mma(FIRST, I1{}, N_, acc[1], fb1);
            if (turn) prepare_epilogue();
            pp_barrier();
            // phase 0 of the next K tile
            read_a(I0{}, I4{});
            dma_a(I1{});
            next_k();
            pp_vmwait<10>();
            pp_barrier();
            mma(F_{}, I0{}, I4{}, acc[0], fb0);
            pp_barrier();
        };
        if (!PART && Kd < 3 * PP_BK) cut_k(Kd - 2 * PP_BK);             // K tile 2 is loaded next
        k_tile(T_{}, F_{}, I4{});
        // The rows of the lower half beyond the last block with a live row are neither read nor multiplied: one copy of
        // the loop per number of such blocks, one after the other, all but one of them with no iterations (chosen
        // between by if and else, each copy's registers would be live across the others).
        const int n1 = min(max(((mend - m0 + 31) >> 5) - 4, 0), 4);
        int t = 1;
        for (int half = 0; half < 2; ++half) {
            const int end = KT - 3 + half;
            for (const int e = n1 == 4 ? end : 0; t < e; ++t) k_tile(F_{}, F_{}, I4{});
            for (const int e = n1 == 3 ? end : 0; t < e; ++t) k_tile(F_{}, F_{}, std::integral_constant<int, 3>{});
            for (const int e = n1 == 2 || n1 == 1 ? end : 0; t < e; ++t) k_tile(F_{}, F_{}, std::integral_constant<int, 2>{});
            for (const int e = n1 == 0 ? end : 0; t < e; ++t) k_tile(F_{}, F_{}, I0{});
            if (half == 0 && ragged_k) cut_k((PART ? part.kd : Kd) - (KT - 1) * PP_BK);    // K tile KT - 1 is loaded next
        }
        k_tile(F_{}, T_{}, I4{});
        if (!PART && Kd < 2 * PP_BK) cut_k(Kd - PP_BK);                 // the next tile's K tile 1 is loaded next
        // ---- last K tile
        read_b(I1{}, fb1);
        dma_b(I0{});
        pp_vmwait<10>();
        pp_barrier();
        mma(F_{}, I1{}, I4{}, acc[0], fb1);
        pp_barrier();
        read_a(I1{}, I4{});
        dma_a(I0{});
        if constexpr (LINES) {
            // the epilogue of a finished half in the memory parts of the phases after it
            epilogue(I0{}, I0{}, acc[0], F_{});
            pp_vmwait<10>();
            pp_barrier();
            mma(F_{}, I0{}, I4{}, acc[1], fb0);
            pp_barrier();
            flip();
            read_b(I0{}, fb0);
            dma_b(I1{});
            epilogue(I0{}, I1{}, acc[0], F_{});
            pp_vmwait<10>();
            pp_barrier();
            mma(F_{}, I1{}, I4{}, acc[1], fb1);
            pp_barrier();
            epilogue(I1{}, I0{}, acc[1], F_{});
            epilogue(I1{}, I1{}, acc[1], F_{});
        } else {
            // activations are far more vector work than one arithmetic part hides: all four quadrants together, so
            // that the two wavefronts of a SIMD share its vector unit instead of taking turns at it
            pp_vmwait<10>();
            pp_barrier();
            mma(F_{}, I0{}, I4{}, acc[1], fb0);
            pp_barrier();
            flip();
            dma_b(I1{});
            pp_vmwait<10>();
            pp_barrier();
            mma(F_{}, I1{}, I4{}, acc[1], fb1);
            fetch_gate_up(I0{}, I0{});
            fetch_gate_up(I0{}, I1{});
            pp_barrier();
            auto quadrants = [&](auto WHOLE) {
                epilogue(I0{}, I0{}, acc[0], WHOLE);
                fetch_gate_up(I1{}, I0{});
                epilogue(I0{}, I1{}, acc[0], WHOLE);
                fetch_gate_up(I1{}, I1{});
                epilogue(I1{}, I0{}, acc[1], WHOLE);
                epilogue(I1{}, I1{}, acc[1], WHOLE);
            };
            if (EPI == EPI_GATED && e_rows > PP_BM - 32) quadrants(T_{});
            else quadrants(F_{});
            read_b(I0{}, fb0);
        }
    };

    // ------------------------------------------------------------ the workgroup's tiles
    dma_b(I0{}); dma_a(I0{}); dma_b(I1{}); dma_a(I1{});
    next_k();
    if (!PART && Kd < 2 * PP_BK) cut_k(Kd - PP_BK);
    dma_b(I0{}); dma_a(I0{}); dma_b(I1{});
    pp_vmwait<12>();
    pp_barrier();
    if (grp == 1) pp_barrier();
    read_b(I0{}, fb0);
    pp_vmwait<10>();
    pp_barrier();
    pp_barrier();
    for (;;) {
        run_tile();
        if (EPI == EPI_GATED_BWD) {
            sums_due = true;
            sums_m0 = m0;
            sums_end = mend;
            sums_nt = nt;
        }
        if (!have_n) break;
        m0 = tm_n.y;
        mend = tm_n.z;
        nt = nt_n;
        part = part_n;
        n0 = nt * PP_BN;
        have_n = have_nn;
        nt_n = nt_nn;
        tm_n = tm_nn;
        par ^= 1;
    }
    pp_barrier();
    write_sums();
    if (grp == 0) pp_barrier();
    pp_vmwait<0>();   // (loads past the last tile wrote zeros into LDS: landed before the workgroup leaves)
}

// ------------------------------------------------------------------ weight gradients
// C[e] = A[rows_e,:]^T @ B[rows_e,:]: the reduction runs over the expert's rows, both operands are K-strided.  The same
// phases and the same stream of K tiles from tile to tile as the row-grouped kernel; a tile is 256 x 256 of one expert's
// gradient, its number of K tiles that of the expert's rows (three at least, the missing ones empty).  Half a is 128 columns of A,
// 64 k deep; half s of B is 32 k deep and all 256 columns wide, so that a phase is one k step of 64 x 64 a wavefront: its
// columns then are 64 in a row, and the epilogue stores whole lines.
// MAPS: 1 = the rows of A, 2 = the rows of B are gathered through a row map: the indices of a K tile are requested three K tiles ahead, by
// direct-to-LDS loads among the others, and its offsets worked out beside the MFMAs.  (By scalar loads they came back out of order with
// the LDS reads, so that every wait for those was one for all: the two parts behind the request took 420 and 460 cycles.)
// What bounds it: per tile the stores of the gradients, behind which, in order, no load of their wavefront completes, and then the MFMAs.
// With the loads between the first MFMAs and the indices out of the scalar unit's way the eight parts of a K tile take 2260 cycles
// in all, of 2048 that the MFMAs take (in the memory parts, and scalar: 2990).  The loads' place alone, with indices through LDS, gate_up's and
// down's gradient, us, in the memory parts / so: 128 experts of 2048 x 768, 1024 rows 698 / 688 and 343 / 338; 8 of 4096 x 14336, 2048 rows 2864 / 2805 and
// 1459 / 1433; 64 of 2048 x 1408, 2048 rows, uneven 1179 / 1154 and 653 / 639, 800 rows 268 / 263; nothing gathered, 32 of 7168 x 2048, 2048 rows 2804 / 2762.
// The faster the loop, the more is read again, as workgroups with a panel in common get further apart: of the 8 experts' gate_up gradient 5.9, 6.6, 6.9 GB
// by scalar indices, by these, with the loads behind the MFMAs; of the 128 experts' 1.41, 1.59, 1.57; of the 32 experts' down gradient 3.6, 4.0, 4.0.
// Both together, alone, us, the rows of one operand gathered, gate_up's / down's gradient, before / so: 64 experts of 2048 x 1408, 250 rows 277 / 143 -> 235 / 125, uneven 2048 rows 1472 / 767 -> 1316 / 749; 128 of 2048 x 768,
// 188 rows 253 / 131 -> 218 / 119, 1024 rows 769 / 439 -> 713 / 426; 8 of 4096 x 14336, 2048 rows 3024 / 1495 -> 2886 / 1457; one of 2048 x 1408, 4001
// rows 96 / 85 -> 81 / 79.  Stored as lanes 16 apart in pieces of 64 bytes, past no caches, 250 rows were 328 / 173, now 235 / 125.
// Tried and not kept: loads by one group of wavefronts and stores by the other (250 rows 257 / 147: the loading group's 16 loads a part and
// SIMD do not fit into it).
// Rows past the expert's end read as zeros: an operand that is not gathered has a descriptor that ends with them, a
// gathered one gets PP_NOWHERE for them.
// DEAL: uneven loads may be dealt by depth
template <int MAPS, bool STREAM, bool DEAL, typename ET>
__device__ __forceinline__ void pp_wgrad_body()
{
    typedef typename Elem16<ET>::frag_t frag_t;
    extern __shared__ u32x4_t smem[];
    const uint32_t lds = (uint32_t)(uintptr_t)(lptr_t)smem;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int grp = wave >> 2, wc = wave & 3;
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    using I2 = std::integral_constant<int, 2>;
    using I3 = std::integral_constant<int, 3>;
    using I4 = std::integral_constant<int, 4>;
    constexpr bool A_MAP = MAPS == 1, B_MAP = MAPS == 2;

    // ------------------------------------------------------------ this workgroup's tiles
    // Tiles are numbered expert by expert, inside an expert in strips of gn columns; XCD x (workgroups with
    // blockIdx % 8 == x) works through chunks x, x + 8, ... of 32 consecutive tiles, so that the workgroups of an XCD
    // share operand panels in its L2; the tiles left over from the last whole group of chunks are dealt one by one.
    // A workgroup takes gm tiles, one from each of gm chunks in a row.
    auto divide = [](int n, uint32_t inv) -> int { return inv ? (int)(((uint64_t)(uint32_t)n * inv) >> 32) : n; };
    struct Tile { int e, m0, n0, r0, r1; };
    auto locate = [&](int e, int i, Tile& t) {        // tile i of expert e
        args_t& p = pp_args();
        t.e = e;
        const int strip = divide(i, p.inv_sn);
        const int r = i - strip * p.n_mt * p.gn;
        const bool last = strip == p.sn - 1;
        const int mt = divide(r, last ? p.inv_gm : p.inv_gn);
        const int w = last ? p.n_ntiles - strip * p.gn : p.gn;
        t.m0 = mt * PP_BM;
        t.n0 = (strip * p.gn + r - mt * w) * PP_BN;
        t.r0 = __builtin_amdgcn_readfirstlane(scalar_load_i32(p.offsets + t.e));
        t.r1 = __builtin_amdgcn_readfirstlane(scalar_load_i32(p.offsets + t.e + 1));
    };
    // Uneven loads: by number, the deep tiles' share of the workgroups differs by a whole one (a sixteenth of 64 experts with half of the
    // rows: the most loaded workgroup has 1.22 times the mean of K tiles).  By depth (wgrad_deal.h) it has 1.01 times.  Where an expert's tiles just miss
    // whole rounds, by depth can be the worse one (8 experts, Zipf loads, 253 tiles each 1.01 / 1.08): the largest loads of both orders are
    // worked out, and the smaller one decides.  Alone, us, by number / by depth: 131072 rows as above, 2048 x 1408, gate_up's gradient 1264 / 1164,
    // down's 671 / 644; 65536 rows of 32 experts of 7168 x 2048, Zipf loads (1.06 and 1.08 times the mean / 1.04 and 1.05) 2880 / 2830 and 1478 / 1448 (within
    // the noise of a whole pass of 13 ms; 6.3 to 7.2 / 7.9 GB read); the 253 tiles 774 / 793 (768 now), 250 765 / 795 (765).  Every workgroup works the dealing out for itself,
    // some 10 us for 64 experts: only where the deepest expert has twice the mean, and the work is fifty times that.  To find that it has not takes
    // 0 to 2 us (even loads, without / with it: 64 experts of 2048 x 1408, 800 rows 264.0 / 264.4, 128 of 2048 x 768, 1024 rows 689 / 690 and 337 / 338);
    // in a kernel of its own, as the shallow tiles of two a workgroup took 1 % longer with it.
    const int my = (int)((blockIdx.x & 7) * 32 + (blockIdx.x >> 3));
    const int per = pp_args().n_mt * pp_args().n_ntiles;
    bool by_depth = false;
    if constexpr (DEAL) {
        args_t& p = pp_args();
        const int E = p.E;
        typedef __attribute__((address_space(3))) uint32_t* word_t;
        int mine = 0;
        if (tid < E) mine = min(max(3, (p.offsets[tid + 1] - p.offsets[tid] + PP_BK - 1) >> 6), 1 << 20) + 3;   // (a tile's stores: three K tiles)
        *(word_t)(uintptr_t)(lds + PP_WDEPTH + tid * 4u) = (uint32_t)mine;
        *(word_t)(uintptr_t)(lds + PP_WLOAD + tid * 4u) = 0u;
        __syncthreads();
        int sum = 0, most = 0;
#pragma unroll
        for (int k = 0; k < AMOE_MAX_EXPERTS / 64; ++k) {
            const int d = pp_lds<int>(lds + PP_WDEPTH + (lane + 64 * k) * 4u);
            sum += d;
            most = max(most, d);
        }
#pragma unroll
        for (int o = 32; o; o >>= 1) {
            sum += __shfl_xor(sum, o, 64);
            most = max(most, __shfl_xor(most, o, 64));
        }
        sum = __builtin_amdgcn_readfirstlane(sum);
        most = __builtin_amdgcn_readfirstlane(most);
        by_depth = (float)most * E > 2.f * sum && (float)sum * per >= 1024.f * E;
        if (by_depth) {
            int rank = 0;
            for (int e = 0; e < E; e += 4) {
                const u32x4_t d = pp_lds<u32x4_t>(lds + PP_WDEPTH + e * 4u);
#pragma unroll
                for (int k = 0; k < 4; ++k) rank += (int)d[k] > mine || ((int)d[k] == mine && e + k < tid);
            }
            // the workgroups' loads by number and, behind them, by depth
            auto more = [&](uint32_t at) {
                return [at](int w, int d) { __hip_atomic_fetch_add((__attribute__((address_space(3))) int*)(uintptr_t)(at + w * 4u), d, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP); };
            };
            const auto by_number = more(lds + PP_WLOAD), of_depth = more(lds + PP_WLOAD + 1024u);
            if (tid < E) {
                *(__attribute__((address_space(3))) u32x4_t*)(uintptr_t)(lds + PP_WDEAL + rank * 16u) = u32x4_t{0, 0, (uint32_t)mine, (uint32_t)tid};
                amoe_deal::add_by_number(tid, mine, per, by_number);
            }
            const int whole = E * per & ~255;
            if (tid < E * per - whole) {
                const int d = pp_lds<int>(lds + PP_WDEPTH + divide(whole + tid, p.inv_super) * 4u);
                amoe_deal::add_arc(tid, 1, -d, by_number);
                amoe_deal::add_arc(amoe_deal::last_of(tid), 1, d, by_number);
            }
            __syncthreads();
            if (wave == 0) {
                amoe_deal::Walk walk;
                for (int k = 0; k < E; ++k) {
                    const u32x4_t x = pp_lds<u32x4_t>(lds + PP_WDEAL + k * 16u);
                    const amoe_deal::Record r = walk.next(__builtin_amdgcn_readfirstlane(x[2]), per);
                    if (lane == 0) *(__attribute__((address_space(3))) u32x4_t*)(uintptr_t)(lds + PP_WDEAL + k * 16u) = u32x4_t{r.word(), (uint32_t)r.behind, (uint32_t)r.fill, x[3]};
                }
            }
            __syncthreads();
            if (tid < E) {
                const u32x4_t x = pp_lds<u32x4_t>(lds + PP_WDEAL + tid * 16u);
                amoe_deal::add_by_depth(amoe_deal::Record::of(x[0], x[1], x[2]), pp_lds<int>(lds + PP_WDEPTH + x[3] * 4u), per, of_depth);
            }
            __syncthreads();
            auto largest = [&](uint32_t at) {
                const u32x4_t x = pp_lds<u32x4_t>(at + lane * 16u);
                const int a = x[0], b = a + (int)x[1], c = b + (int)x[2], d = c + (int)x[3];
                int before = d;
#pragma unroll
                for (int o = 1; o < 64; o <<= 1) {
                    const int v = __shfl_up(before, o, 64);
                    before += lane >= o ? v : 0;
                }
                int m = before - d + max(max(a, b), max(c, d));
#pragma unroll
                for (int o = 32; o; o >>= 1) m = max(m, __shfl_xor(m, o, 64));
                return __builtin_amdgcn_readfirstlane(m);
            };
            by_depth = largest(lds + PP_WLOAD + 1024u) < largest(lds + PP_WLOAD);
        }
    }
    // this workgroup's place in the dealing: position of the expert, the expert, and its tiles
    struct { int at, e; } deal = {-1, 0};
    amoe_deal::Turns turns({0, 0, 256, 0, 0}, 0);
    // position of the last tile taken in this XCD's queue, and the end of what this workgroup takes
    int q = (int)(blockIdx.x >> 8) * 32 * pp_args().gm + (int)((blockIdx.x >> 3) & 31);
    const int q_end = q + 32 * pp_args().gm;
    q -= 32;
    auto take = [&](Tile& t) -> bool {                // this workgroup's next tile
        if (DEAL && by_depth) {
            turns.next();
            while (deal.at < 0 || turns.at >= per) {
                if (++deal.at >= pp_args().E) return false;
                const u32x4_t x = pp_lds<u32x4_t>(lds + PP_WDEAL + deal.at * 16u);
                deal.e = __builtin_amdgcn_readfirstlane(x[3]);
                turns = amoe_deal::Turns(amoe_deal::Record::of(__builtin_amdgcn_readfirstlane(x[0]), __builtin_amdgcn_readfirstlane(x[1]),
                                                               __builtin_amdgcn_readfirstlane(x[2])), my);
            }
            locate(deal.e, turns.at, t);
            return true;
        }
        args_t& p = pp_args();
        const int xcd = blockIdx.x & 7;
        const int total = p.E * per;
        const int whole = total & ~255;
        if ((q += 32) >= q_end) return false;
        int v = ((q >> 5) << 8) + (xcd << 5) + (q & 31);
        if (v >= whole) v = whole + ((q - (whole >> 3)) << 3) + xcd;
        if (v >= total) return false;
        const int e = divide(v, p.inv_super);
        locate(e, v - e * per, t);
        return true;
    };

    // ------------------------------------------------------------ loads
    // Thread tid fills k rows tid / 16 and tid / 16 + 32 of either half (128 columns) of A, and k rows tid / 32 and tid / 32 + 16 of
    // either half (32 k) of B.
    uint32_t arow[2], brow[4];        // gathered operand: byte offsets of its rows of the K tile (B: and columns; PP_NOWHERE past the last row)
    uint32_t acol[2], bcol;           // byte offsets of its columns (PP_NOWHERE outside the matrix); not gathered: of its first row's
    srd_t ad, bd;
    const uint32_t lda2 = (uint32_t)pp_args().lda * 2u, ldb2 = (uint32_t)pp_args().ldb * 2u;
    int left = 0;                     // rows of the expert from the K tile loaded next
    int row_n = 0;                    // gathered: map position of the K tile whose indices are requested next
    uint64_t map = (uint64_t)(uintptr_t)(A_MAP ? pp_args().a_row_map : pp_args().b_row_map);
    map = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)map) |
          ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(map >> 32)) << 32);
    const int last_row = pp_args().rows_total - 1;
    uint32_t slot = lds + PP_WIDX + (uint32_t)wave * 512u;        // this wavefront's indices of that K tile (two K tiles', by turns)
    auto add_sat = [](uint32_t a, uint32_t b) { return __builtin_elementwise_add_sat(a, b); };
    // A: rows 4 wave ..+3 and those 32 on; B: rows 2 wave, 2 wave + 1 and those 16, 32 and 48 on
    const int lane_row = A_MAP ? 4 * wave + (lane & 3) + 8 * (lane & 4) : 2 * wave + (lane & 1) + 8 * (lane & 6);
    // the eight indices that this wavefront's loads of a K tile need, in the order in which gather_offsets reads them
    auto fetch_idx = [&]() {
        if constexpr (MAPS != 0) {
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2"
                         :
                         : "s"(slot), "v"((uint32_t)min(row_n + lane_row, last_row) * 4u), "s"(map)
                         : "memory");
            slot ^= 256u;
        }
    };
    // the indices of the request before the last one, this thread's: read a part before its offsets are worked out beside the MFMAs
    uint32_t idx[4];
    auto read_idx = [&](uint32_t from) {
        if constexpr (MAPS != 0) {
            const int th = pp_here(tid);
            const uint32_t at = from + (uint32_t)(A_MAP ? (th >> 2) & 12 : (th >> 3) & 4);
#pragma unroll
            for (int k = 0; k < (A_MAP ? 2 : 4); ++k) idx[k] = pp_lds<uint32_t>(at + (A_MAP ? 16u : 8u) * k);
        }
    };
    // row offsets of the gathered operand for the K tile of these indices, of which `rows` rows exist
    auto gather_offsets = [&](int rows) {
        if constexpr (MAPS != 0) {
            const int th = pp_here(tid);
            const int kr = A_MAP ? th >> 4 : th >> 5;
#pragma unroll
            for (int k = 0; k < (A_MAP ? 2 : 4); ++k) {
                const uint32_t o = A_MAP ? idx[k] * lda2 : add_sat(idx[k] * ldb2, bcol);
                (A_MAP ? arow : brow)[k] = kr + (A_MAP ? 32 : 16) * k < rows ? o : PP_NOWHERE;
            }
        }
    };
    auto limit = [&]() {              // descriptors of the operands that are not gathered end with the expert's rows
        int some = max(left, 0);
        asm("" : "+s"(some));         // (a clamp in one step would be a vector instruction)
        const uint32_t rows = (uint32_t)min(some, PP_BK);
        if (!A_MAP) ad[2] = rows * lda2;
        if (!B_MAP) bd[2] = rows * ldb2;
    };
    auto plan = [&](const Tile& t) {
        args_t& p = pp_args();
        const int th = pp_here(tid);
        const int kr = th >> 4;
        const int col = ((th & 15) ^ (2 * ((kr & 3) | (((kr >> 3) & 1) << 2)))) * 8;
        ad = pp_srd(A_MAP ? p.A : p.A + (long long)t.r0 * p.lda);
        bd = pp_srd(B_MAP ? p.B : p.B + (long long)t.r0 * p.ldb);
        left = t.r1 - t.r0;
        limit();
        const int krb = th >> 5;
        const int n = t.n0 + ((th & 31) ^ (2 * ((krb & 3) | (((krb >> 3) & 1) << 2)))) * 8;
        bcol = n < p.N ? (uint32_t)n * 2u : PP_NOWHERE;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int m = t.m0 + h * 128 + col;
            acol[h] = m < p.M ? (uint32_t)m * 2u : PP_NOWHERE;
            if (!A_MAP) acol[h] = add_sat((uint32_t)kr * lda2, acol[h]);
        }
        if (!B_MAP) bcol = add_sat((uint32_t)krb * ldb2, bcol);
    };
    auto next_k = [&]() {             // on to the next K tile of the same tile
        left -= PP_BK;
        if (!A_MAP) pp_advance(ad, PP_BK * lda2);
        if (!B_MAP) pp_advance(bd, PP_BK * ldb2);
        limit();
    };
    uint32_t fill = lds + (uint32_t)wave * 1024u;
    // load J_ of the two of half H_ of A (Op_ 0) or B (1)
    auto dma = [&](auto Op_, auto H_, auto J_) {
        constexpr int h = decltype(H_)::value, j = decltype(J_)::value;
        if constexpr (decltype(Op_)::value == 0)
            pp_dma16<h * PP_HALF + j * 8192u>(ad, add_sat(A_MAP ? arow[j] : 32u * j * lda2, acol[h]), fill);
        else
            pp_dma16<(2 + h) * PP_HALF + j * 8192u>(bd, B_MAP ? brow[2 * h + j] : add_sat((32u * h + 16u * j) * ldb2, bcol), fill);
    };
    auto dma_a = [&](auto H_) { dma(I0{}, H_, I0{}); dma(I0{}, H_, I1{}); };
    auto dma_b = [&](auto H_) { dma(I1{}, H_, I0{}); dma(I1{}, H_, I1{}); };

    // ------------------------------------------------------------ fragments
    frag_t fa[4][2], fb0[4], fb1[4];
    uint32_t ra[4], rb[4];            // LDS read addresses per 16-column tile
    {
        const int l16 = lane & 15, lq = lane >> 4;
        const int k = 8 * lq + (l16 >> 2), key = 2 * ((l16 >> 2) | ((lq & 1) << 2));
        const uint32_t base = lds + (uint32_t)(k * 256 + (l16 & 1) * 8);
#pragma unroll
        for (int i = 0; i < 4; ++i) ra[i] = base + (uint32_t)((grp * 8 + 2 * i + ((l16 & 3) >> 1)) ^ key) * 16u;
#pragma unroll
        for (int j = 0; j < 4; ++j) rb[j] = base + 2 * PP_HALF + (uint32_t)(k * 256) + (uint32_t)((wc * 8 + 2 * j + ((l16 & 3) >> 1)) ^ key) * 16u;
    }
    auto flip = [&]() {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            ra[i] ^= PP_STAGE;
            rb[i] ^= PP_STAGE;
        }
    };
    auto read_tr = [&](uint32_t ad, uint32_t four_rows) -> frag_t {
        typedef __attribute__((address_space(3))) i16x4_t* tr_ptr;
        const u32x2_t lo = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)ad));
        const u32x2_t hi = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)(ad + four_rows)));
        return __builtin_bit_cast(frag_t, u32x4_t{lo[0], lo[1], hi[0], hi[1]});
    };
    auto read_a = [&](auto A_, auto N_) {
#pragma unroll
        for (int i = 0; i < decltype(N_)::value; ++i)
#pragma unroll
            for (int s = 0; s < 2; ++s) fa[i][s] = read_tr(ra[i] + decltype(A_)::value * PP_HALF + s * 8192u, 1024u);
    };
    auto read_b = [&](auto S_, frag_t (&fb)[4]) {
#pragma unroll
        for (int j = 0; j < 4; ++j) fb[j] = read_tr(rb[j] + decltype(S_)::value * PP_HALF, 2048u);
    };
    // step S_ of the K tile; FIRST: the half's first one, nothing to add to.  The phase's two loads (of half H_ of operand Op_) are issued
    // behind the first two MFMAs: a load takes the address unit, which four wavefronts share, 16 cycles.  dead: the half lies past the
    // matrix (asked once, and behind the first MFMAs: a branch around all of a phase is two, taken ones)
    auto mma = [&](auto FIRST, auto S_, bool dead, mfma_f32x4 (&c)[4][4], const frag_t (&fb)[4], auto Op_, auto H_) {
        auto one = [&](int i, int j) {
            c[i][j] = Mfma16<ET>::run(fb[j], fa[i][decltype(S_)::value], decltype(FIRST)::value ? mfma_f32x4{0.f, 0.f, 0.f, 0.f} : c[i][j]);
        };
        one(0, 0);
        pp_fence();
        dma(Op_, H_, I0{});
        pp_fence();
        one(0, 1);
        pp_fence();
        dma(Op_, H_, I1{});
        pp_fence();
        one(0, 2);
        one(0, 3);
        if (!dead) {
#pragma unroll
            for (int i = 1; i < 4; ++i)
#pragma unroll
                for (int j = 0; j < 4; ++j) one(i, j);
        }
    };

    // ------------------------------------------------------------ tile state
    Tile cur, nxt = {0, 0, 0, 0, 0}, far = {0, 0, 0, 0, 0};
    if (!take(cur)) return;
    bool have_n = take(nxt), have_nn = false;

    // Epilogue: a wavefront's columns of the tile are 64, 128 bytes of a row.  Lane (lq, l16) holds columns 16 j + 4 lq ..+3 of row
    // l16 of every 16-row block; through 2 KB of LDS of the wavefront's own (chunk c of row r at c ^ (r & 7), its halves the other way
    // round from row 8 on: no bank conflicts) eight lanes come to hold a row's 128 bytes, and a store writes whole lines.
    // (Adjacent lanes in adjacent rows, as the accumulators have them, are a request each: 128 such stores take 3.5 us on a compute
    // unit and 0.9 so.)
    bf16_t* e_c;
    int e_ldc2 = 0, e_cols = 0, e_rows = 0;
    uint32_t e_off = 0;
    auto prepare_epilogue = [&]() {
        args_t& p = pp_args();
        const int le = pp_here(lane);
        e_ldc2 = p.ldc * 2;
        e_c = p.C + (long long)cur.e * p.strideC + (long long)(cur.m0 + grp * 64) * p.ldc + cur.n0 + wc * 64;
        e_cols = p.N - cur.n0 - wc * 64;
        e_rows = p.M - cur.m0 - grp * 64;
        e_off = (uint32_t)((le >> 3) * e_ldc2 + 16 * (le & 7));
    };
    auto epilogue = [&](auto A_, auto FROM, const mfma_f32x4 (&acc)[4][4]) {      // two 16-row blocks
        constexpr int a = decltype(A_)::value, from = decltype(FROM)::value;
        const int le = pp_here(lane);
        const int r16 = le & 15, r8 = le >> 3;
        const uint32_t at = lds + 2 * PP_STAGE + (uint32_t)wave * 2048u;
        const uint32_t wr = at + (uint32_t)(r16 * 128 + (((le >> 5) ^ (r16 & 7)) * 16) + (((le >> 4) ^ (r16 >> 3)) & 1) * 8);
        const uint32_t rd = at + (uint32_t)(r8 * 128 + ((le & 7) ^ r8) * 16);
        const __amdgpu_buffer_rsrc_t d = __builtin_amdgcn_make_buffer_rsrc(e_c, (short)0, (int)PP_DROP, 0x00020000);
#pragma unroll
        for (int i = from; i < from + 2; ++i) {
            pp_fence();
#pragma unroll
            for (int j = 0; j < 4; ++j)
                *(__attribute__((address_space(3))) u32x2_t*)(uintptr_t)(wr ^ (32u * j)) =
                    u32x2_t{Elem16<ET>::pack2(acc[i][j][0], acc[i][j][1]), Elem16<ET>::pack2(acc[i][j][2], acc[i][j][3])};
            pp_lds_turn();
            u32x4_t v[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) v[t] = pp_lds<u32x4_t>(rd + t * 1024u);
            pp_lds_turn();
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                const bool ok = 8 * (le & 7) < e_cols && a * 128 + i * 16 + t * 8 + r8 < e_rows;
                pp_store16<STREAM>(d, t == 0 ? v[0] : u32x4_t{v[1][2], v[1][3], v[1][0], v[1][1]}, ok ? e_off : PP_DROP,
                                   (uint32_t)((a * 128 + i * 16 + t * 8) * e_ldc2));
            }
        }
    };

    // The waits: phase n awaits the loads issued in phase n - 5, which the next phase reads after the barrier; those of the four phases
    // since stay in flight, and a request for indices, which one of the four phases of a K tile issues behind its wait.
    // Indices of K tile t + 3 are requested in K tile t, and their offsets worked out in the next one: for A, loaded from phase 2 on, in phase 1,
    // whose memory part is the shorter one; for B, loaded from phase 1 on, in phase 0.
    constexpr int IDX = A_MAP ? 1 : B_MAP ? 0 : -1;
    auto landed = [&](auto PHASE) { pp_vmwait<8 + (MAPS != 0 && decltype(PHASE)::value != IDX)>(); };
    auto run_tile = [&]() {
        mfma_f32x4 acc[2][4][4];
        const int KT = max(3, (cur.r1 - cur.r0 + PP_BK - 1) >> 6);
        auto indices = [&](auto PHASE, int t) {
            if constexpr (decltype(PHASE)::value == IDX) {
                read_idx(slot ^ 256u);
                row_n = t == KT - 3 ? nxt.r0 : row_n + PP_BK;
                fetch_idx();
            }
        };
        auto offsets = [&](auto PHASE) {
            if constexpr (decltype(PHASE)::value == IDX) gather_offsets(left);
        };
        // ---- phase 0 of the first K tile
        read_a(I0{}, I4{});
        landed(I0{});
        indices(I0{}, 0);
        pp_barrier();
        mma(T_{}, I0{}, false, acc[0], fb0, I0{}, I1{});
        fill ^= PP_STAGE;
        next_k();
        offsets(I0{});
        have_nn = have_n && take(far);
        if (!have_nn) far = Tile{0, 0, 0, 0, 0};
        pp_barrier();
        // the lower half of the tile lies past the matrix
        const bool half = cur.m0 + 128 >= pp_args().M;
        auto k_tile = [&](auto FIRST, auto TURN, int t) {
            // phase 1
            read_b(I1{}, fb1);
            if (decltype(TURN)::value) {
                plan(nxt);
                if constexpr (B_MAP) {
                    read_idx(slot);
                    gather_offsets(left);
                }
            }
            landed(I1{});
            indices(I1{}, t);
            pp_barrier();
            mma(F_{}, I1{}, false, acc[0], fb1, I1{}, I0{});
            offsets(I1{});
            pp_barrier();
            // phase 2
            read_a(I1{}, I4{});
            landed(I2{});
            pp_barrier();
            mma(FIRST, I0{}, half, acc[1], fb0, I0{}, I0{});
            pp_barrier();
            // phase 3
            flip();
            read_b(I0{}, fb0);
            landed(I3{});
            pp_barrier();
            mma(F_{}, I1{}, half, acc[1], fb1, I1{}, I1{});
            pp_barrier();
            // phase 0 of the next K tile
            read_a(I0{}, I4{});
            landed(I0{});
            indices(I0{}, t + 1);
            pp_barrier();
            mma(F_{}, I0{}, false, acc[0], fb0, I0{}, I1{});
            fill ^= PP_STAGE;
            if (decltype(TURN)::value) prepare_epilogue();
            next_k();
            offsets(I0{});
            pp_barrier();
        };
        k_tile(T_{}, F_{}, 0);
        for (int t = 1; t < KT - 2; ++t) k_tile(F_{}, F_{}, t);
        k_tile(F_{}, T_{}, KT - 2);
        // ---- last K tile: the epilogue of each finished half in the memory parts of the phases after it
        read_b(I1{}, fb1);
        landed(I1{});
        indices(I1{}, KT - 1);
        pp_barrier();
        mma(F_{}, I1{}, false, acc[0], fb1, I1{}, I0{});
        offsets(I1{});
        pp_barrier();
        read_a(I1{}, I4{});
        epilogue(I0{}, I0{}, acc[0]);
        landed(I2{});
        pp_barrier();
        mma(F_{}, I0{}, false, acc[1], fb0, I0{}, I0{});
        pp_barrier();
        flip();
        read_b(I0{}, fb0);
        epilogue(I0{}, I2{}, acc[0]);
        landed(I3{});
        pp_barrier();
        mma(F_{}, I1{}, false, acc[1], fb1, I1{}, I1{});
        pp_barrier();
        epilogue(I1{}, I0{}, acc[1]);
        epilogue(I1{}, I2{}, acc[1]);
    };

    // ------------------------------------------------------------ the workgroup's tiles
    row_n = cur.r0;
    fetch_idx();
    row_n += PP_BK;
    fetch_idx();
    if constexpr (MAPS != 0) pp_vmwait<0>();
    plan(cur);
    read_idx(slot);
    gather_offsets(left);
    row_n += PP_BK;
    if constexpr (MAPS != 0) asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");   // (the next request takes the place of those just read)
    fetch_idx();
    dma_b(I0{}); dma_a(I0{}); dma_b(I1{}); dma_a(I1{});
    fill ^= PP_STAGE;
    next_k();
    read_idx(slot);
    gather_offsets(left);
    dma_b(I0{}); dma_a(I0{}); dma_b(I1{});
    pp_vmwait<12>();
    pp_barrier();
    if (grp == 1) pp_barrier();
    read_b(I0{}, fb0);
    pp_vmwait<8>();   // (no request for indices is among the loads since: phase 0 would await one too few)
    pp_barrier();
    pp_barrier();
    for (;;) {
        run_tile();
        if (!have_n) break;
        cur = nxt;
        nxt = far;
        have_n = have_nn;
    }
    if (grp == 0) pp_barrier();
    pp_vmwait<0>();   // (loads past the last tile wrote zeros into LDS: landed before the workgroup leaves)
}

template <bool B_KC, int EPI, int ACT, bool STREAM>
__global__ void __launch_bounds__(PP_THREADS, 2) grouped_gemm_pp_rows_bf16_kernel(GemmArgs)
{
    pp_rows_body<B_KC, EPI, ACT, STREAM, bf16_t>();
}
template <bool B_KC, int EPI, int ACT, bool STREAM>
__global__ void __launch_bounds__(PP_THREADS, 2) grouped_gemm_pp_rows_f16_kernel(GemmArgs)
{
    pp_rows_body<B_KC, EPI, ACT, STREAM, f16_t>();
}

template <int MAPS, bool STREAM, bool DEAL>
__global__ void __launch_bounds__(PP_THREADS, 2) grouped_gemm_pp_wgrad_bf16_kernel(GemmArgs)
{
    pp_wgrad_body<MAPS, STREAM, DEAL, bf16_t>();
}
template <int MAPS, bool STREAM, bool DEAL>
__global__ void __launch_bounds__(PP_THREADS, 2) grouped_gemm_pp_wgrad_f16_kernel(GemmArgs)
{
    pp_wgrad_body<MAPS, STREAM, DEAL, f16_t>();
}

}  // namespace

#include "gemm_launch.h"

// ceil(2^32 / d), 0 for a divisor of 1
static inline uint32_t tile_inverse(int d) { return d > 1 ? (uint32_t)(((1ull << 32) + d - 1) / d) : 0u; }

template <bool B_KC, int EPI, int ACT, bool STREAM>
static int launch_pp_rows(const GemmArgs& a, int grid, hipStream_t s)
{
    if (a.f16) return launch_kernel<grouped_gemm_pp_rows_f16_kernel<B_KC, EPI, ACT, STREAM>, PP_THREADS, PP_LDS>(a, grid, s);
    return launch_kernel<grouped_gemm_pp_rows_bf16_kernel<B_KC, EPI, ACT, STREAM>, PP_THREADS, PP_LDS>(a, grid, s);
}
template <bool B_KC, int EPI, int ACT>
static int launch_pp_rows(const GemmArgs& a, hipStream_t s)
{
    const int cus = device_cu_count();
    AMOE_REQUIRE(cus > 0, AMOE_ERR_LAUNCH, "grouped_gemm: cannot read the number of compute units");
    // (a multiple of 8: every XCD then runs the same number of workgroups; how many tiles there are, only the device knows)
    const int grid = (cus + 7) & ~7;
    GemmArgs b = a;
    b.inv_group = tile_inverse(a.gm * a.n_ntiles);
    b.inv_n = tile_inverse(a.n_ntiles);
    // Where expert e's reduction starts (see first_step in the kernel).  The three lengths are what was measured to gain, no more:
    // few channels alone would speak for rows 16 KB apart too, which lose, and lengths of 10240 and more were not tried.  The order in
    // which a row's products are summed depends on its expert's number there.  128 experts of N = 2048, 32 rows each, us, at 0 / at 5 e: K = 2048
    // 240 / 188, 4096 433 / 355; 16 of N = 4096, 24 rows: K = 4096 123 / 92, 6144 153 / 135; 64 of N = 2048, 300 rows: K = 2048 199 / 179.
    // Other strides have no such channels, and lose what neighbours read of one memory page: K = 1984 182 / 187, 4160 351 / 366, 8192 170 /
    // 180, 3072 276 / 280.  From 512 rows an expert on the products are not bound by the reading (600 rows 219 / 222).  With B not
    // transposed, read in rows of 512 bytes, K = 2048 180 / 183.
    b.first_step = B_KC && a.Kd % 2048 == 0 && a.Kd <= 6144 && a.M <= 512ll * a.E ? 5 : 0;
    b.inv_kt = tile_inverse(a.Kd / PP_BK);
    b.inv_last = tile_inverse(a.n_ntiles - (a.sn - 1) * a.gn);
    if (a.stream_from) return launch_pp_rows<B_KC, EPI, ACT, true>(b, grid, s);
    return launch_pp_rows<B_KC, EPI, ACT, false>(b, grid, s);
}

#if AMOE_PP_PART_IS(0)
int amoe_pp_gateup_act(const GemmArgs& a, int act, hipStream_t s)
{
    AMOE_DISPATCH_ACT(act, return (launch_pp_rows<false, EPI_GATED, ACT>(a, s)))
    return AMOE_ERR_BAD_ARG;
}
#endif
#if AMOE_PP_PART_IS(1)
int amoe_pp_part(const GemmArgs& a, bool b_kc, hipStream_t s)
{
    return b_kc ? launch_pp_rows<true, EPI_PART, 0>(a, s) : launch_pp_rows<false, EPI_PART, 0>(a, s);
}
int amoe_pp_rows(const GemmArgs& a, bool b_kc, hipStream_t s)
{
    // An output of half the last-level cache or more is stored past the caches (218 MB: 0.828 ms a step with ordinary stores, 0.801
    // so; 1 GB 5.00 / 4.94; 45 MB 0.136 / 0.141), if its rows are whole lines of 128 bytes: parts of lines meet in the L2 and not
    // past it (alone, us, ordinary / past: 120000 rows, 896 x 608 140 / 150, 80000, 544 x 1504 160 / 166).
    const bool past = a.N % 64 == 0 && 2ll * a.M * a.N >= 128ll << 20;
    if (past) return b_kc ? launch_pp_rows<true, EPI_STORE_PAST, 0>(a, s) : launch_pp_rows<false, EPI_STORE_PAST, 0>(a, s);
    return b_kc ? launch_pp_rows<true, EPI_STORE, 0>(a, s) : launch_pp_rows<false, EPI_STORE, 0>(a, s);
}
#endif
#if AMOE_PP_PART_IS(2)
int amoe_pp_gated_bwd(const GemmArgs& a, int act, hipStream_t s)
{
    AMOE_DISPATCH_ACT(act, return (launch_pp_rows<true, EPI_GATED_BWD, ACT>(a, s)))
    return AMOE_ERR_BAD_ARG;
}
#endif
#if AMOE_PP_PART_IS(3)
template <int MAPS, bool STREAM, bool DEAL>
static int launch_pp_wgrad(const GemmArgs& a, int grid, hipStream_t s)
{
    constexpr int lds = DEAL ? PP_WGRAD_DEAL_LDS : PP_WGRAD_LDS;
    if (a.f16) return launch_kernel<grouped_gemm_pp_wgrad_f16_kernel<MAPS, STREAM, DEAL>, PP_THREADS, lds>(a, grid, s);
    return launch_kernel<grouped_gemm_pp_wgrad_bf16_kernel<MAPS, STREAM, DEAL>, PP_THREADS, lds>(a, grid, s);
}
template <int MAPS>
static int launch_pp_wgrad(const GemmArgs& a, bool deal, int grid, hipStream_t s)
{
    if (a.stream_from) return deal ? launch_pp_wgrad<MAPS, true, true>(a, grid, s) : launch_pp_wgrad<MAPS, true, false>(a, grid, s);
    return deal ? launch_pp_wgrad<MAPS, false, true>(a, grid, s) : launch_pp_wgrad<MAPS, false, false>(a, grid, s);
}

int amoe_pp_wgrad(GemmArgs a, hipStream_t s)
{
    const int strips = (a.n_ntiles + 7) / 8;
    a.gn = (a.n_ntiles + strips - 1) / strips;
    a.sn = (a.n_ntiles + a.gn - 1) / a.gn;
    const long long per = (long long)a.n_mt * a.n_ntiles, total = per * a.E;
    AMOE_REQUIRE(total * per < (1ll << 32), AMOE_ERR_UNSUPPORTED, "grouped_gemm_wgrad: too many tiles");
    a.inv_super = tile_inverse((int)per);
    a.inv_sn = tile_inverse(a.n_mt * a.gn);
    a.inv_gn = tile_inverse(a.gn);
    a.inv_gm = tile_inverse(a.n_ntiles - (a.sn - 1) * a.gn);
    // Tiles a workgroup: all that fall to it from 11 K tiles an expert on (fewer workgroups then only fill their pipelines again: 1024
    // rows of 128 experts of 2048 x 768, a training step 3.80 ms, with two tiles each 3.92), below that two, so that the other stream's
    // workgroups get compute units between them.  Steps with one / two / four / all, ms, against shape 5 (to 256 rows) or all:
    //   64 experts of 2048 x 1408, 250 rows, shared expert  1.59 / 1.62 / 1.64 / 1.67, 1.67
    //   37 experts of 5568 x 1600, 221 rows                 2.08 / 2.02 / 1.99 / 1.94, 2.17
    //   24 experts of  480 x 7360, 230 rows                 0.73 / 0.73 / 0.75 / 0.76, 0.79
    //   22 experts of  832 x 11840, 615 rows                3.18 / 3.17 / 3.19 / 3.38, 3.40
    //   16 experts of 1728 x 2208, 742 rows                 0.99 / 1.01 / 1.00 / 0.98, 1.00
    // Uneven loads, both gradients alone, us, shape 5 / two tiles a workgroup: 128 experts of 2048 x 768, 175 rows, all on one expert
    // 1049 / 1057, half on the first and the last each 749 / 760 (200 rows 813 / 835), 150 rows on a quarter of the experts 522 / 356, a
    // sixteenth with half of them 440 / 367; 64 of 1024 x 2048, 150 rows, on one 581 / 502, a quarter 535 / 373, a sixteenth 319 / 245.
    const long long rounds = (total + 255) / 256;
    a.gm = (int)(a.rows_total < 11ll * PP_BK * a.E && rounds > 2 ? 2 : rounds);
    // Where a workgroup takes all that falls to it, that may be by depth (whether loads are uneven, only the device knows).
    const bool deal = a.gm == rounds && rounds > 1 && a.E > 1 && a.E <= AMOE_MAX_EXPERTS;
    const int grid = rounds == 1 ? (int)((total + 7) & ~7ll) : (int)((rounds + a.gm - 1) / a.gm * 256);
    // Gradients that the L2s (8 x 4 MB) do not hold are stored past the caches: with ordinary stores a tile's 128 KB wait for dirty
    // lines of older ones to be written out, behind which no load of the next tile completes.
    a.stream_from = 2ll * a.E * a.M * a.N > (32ll << 20);
    if (a.a_row_map) return launch_pp_wgrad<1>(a, deal, grid, s);
    if (a.b_row_map) return launch_pp_wgrad<2>(a, deal, grid, s);
    return launch_pp_wgrad<0>(a, deal, grid, s);
}
#endif
