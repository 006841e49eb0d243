// bfloat16 GEMM for the decoder's projections on gfx950: y [M, N] = x [M, K] w [N, K]^T (both
// operands K-contiguous), float32 accumulation, one rounding.
//
// What bounds it. A workgroup's tile needs (BM + BN) x 128 bytes per 64 k and BM x BN x 64 products:
// a 256 x 256 tile asks 32 bytes a clock of the CU's path to the L2 (64 a clock at most) while its
// MFMAs run, a 128 x 128 tile twice that. So large products take the largest tile and are bound
// by the MFMA (and, on random data, by the clock that the chip's power allows: 4096 x 8192 x 8192
// runs in 296 us on zeros and 384 us on normal values); short prompts are bound by how fast the
// weights stream in, which depends on bytes in flight: deep LDS rings of smaller tiles.
//   * 8 waves in every form, two per SIMD: with one wave per SIMD the step stood still at each
//     LDS wait and barrier (256 x 256 on 4 waves of 128 x 128: 530 us against 391).
//   * Tiles move global -> LDS by buffer_load_dwordx4 ... lds, one 128-byte line per row and step, into
//     rings of 2 to 6 stages. Two stages are 128 KB for the largest tile, so a slot has to be
//     refilled as early as possible: a step reads all of its fragments in its first quarter, a
//     barrier frees the slot and the refill is issued there; a second barrier at three quarters
//     publishes the next step's tiles (1.25 steps of latency covered instead of 0.5 with the refill
//     spread behind one barrier: 391 -> 371 us at 1217 x 34816 x 5120, 204 -> 180 at
//     4096 x 2560 x 9728).
//   * 16-byte chunks are permuted within a staged row so that the fragment reads meet no bank
//     twice (SQ_LDS_BANK_CONFLICT 0; half of the LDS cycles before).
//   * Blocks of one XCD take neighbouring tiles, which share rows of x and w in its L2.
//   * Products with few tiles split K; the float32 partial sums are added in order by a second
//     kernel and rounded once, so a shape's result does not depend on scheduling.
#include <algorithm>
#include <cmath>

#include "common.h"
#include "gemm_mfma.h"

namespace q35 {
namespace {

constexpr int BK = 64;        // k elements per step: one 128-byte line of every row
constexpr int ROWB = BK * 2;  // bytes of a staged row
constexpr int GROUP = 8;      // M tiles walked together along N (L2 sharing; 4 and 16 measured equal or slower)

struct GemmArgs {
    const bf16* x;
    const bf16* w;
    bf16* y;
    float* part;  // split-K partial sums
    int M, N, K, ldy;
    int tm, tn;   // tiles along M and N
    int split;    // K parts
};

// chunk permutation of staged row r: 16-byte chunk c sits at slot c ^ swz(r)
__device__ __forceinline__ int swz_x(int r) { return (r >> 1) & 7; }
__device__ __forceinline__ int swz_w(int r) { return ((r >> 1) & 1) | ((r >> 2) & 2) | ((r ^ (r >> 2)) & 4); }

// Tile number `tile` of the walk: groups of GROUP rows of tiles, along N within a group.
__device__ __forceinline__ void tile_at(int tile, int tm, int tn, int& mt, int& nt) {
    const int per = GROUP * tn, gi = tile / per, rem = tile - gi * per;
    const int gm = min(GROUP, tm - gi * GROUP);
    nt = rem / gm;
    mt = gi * GROUP + rem - nt * gm;
}

__device__ __forceinline__ u32x4 rows_rsrc(const bf16* base, int bytes) {
    const uint64_t a = (uint64_t)base;
    return u32x4{(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)a),
                 (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(a >> 32)) & 0xffffu,
                 (uint32_t)__builtin_amdgcn_readfirstlane(bytes), 0x00020000u};
}

template <int N>
__device__ __forceinline__ void wait_vm() {
    static_assert(N < 64, "vmcnt range");
    // vmcnt in bits 3:0 and 15:14; expcnt 7, lgkmcnt 15 (not waited)
    __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | 0x0f70);
}
__device__ __forceinline__ void wait_lds() { __builtin_amdgcn_s_waitcnt(0xc07f); }

template <int WM, int WN, int TM, int TN, int ST>
struct Cfg {
    static constexpr int WAVES = WM * WN, THREADS = 64 * WAVES;
    static constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
    static constexpr int XST = BM * ROWB, WST = BN * ROWB;  // bytes of a staged x / w tile
    static constexpr int STAGE = XST + WST, BYTES = ST * STAGE;  // a stage: the x rows, then the w rows
    static constexpr int XI = BM / 8, WI = BN / 8;          // 1 KB transfers per stage
    static constexpr int LX = (XI + WAVES - 1) / WAVES, LW = (WI + WAVES - 1) / WAVES;  // per wave
    static_assert(BYTES <= 160 * 1024, "LDS");
    static_assert(ST >= 2 && TN >= 2, "ring depth, one pair of n tiles");
};

template <int WM, int WN, int TM, int TN, int ST, bool SPLIT>
__global__ void __launch_bounds__(64 * WM * WN, 1) mfma_gemm_kernel(const GemmArgs a) {
    using C = Cfg<WM, WN, TM, TN, ST>;
    extern __shared__ __align__(16) unsigned char smem[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave % WM, wn = wave / WM;
    const int r16 = lane & 15, g = lane >> 4;

    // Blocks b, b + 8, b + 16, ... run on one XCD: each XCD takes a contiguous run of the tile order,
    // and when there are more tiles than blocks (one block per CU then), its blocks take turns.
    const int tiles = a.tm * a.tn;
    const int total = SPLIT ? tiles * a.split : tiles;
    int id, id_end, id_step;
    {
        const int b = blockIdx.x, xcd = b & 7, q = total >> 3, r = total & 7;
        const int first = xcd * q + min(xcd, r);
        id = first + (b >> 3);
        id_end = first + q + (xcd < r ? 1 : 0);
        id_step = ((int)gridDim.x - xcd + 7) >> 3;
    }
    if (id >= id_end) return;
    const int nk_all = a.K / BK;
    int z = 0, k_lo = 0, nk = nk_all;
    if (SPLIT) {
        z = id / tiles;
        id -= z * tiles;
        k_lo = (int)((long)nk_all * z / a.split);
        nk = (int)((long)nk_all * (z + 1) / a.split) - k_lo;
    }
    const uint32_t lds0 = (uint32_t)__builtin_amdgcn_readfirstlane(
        (int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)smem);
    // This wave's transfers of a stage: rows 8 idx .. 8 idx + 7, idx = wave + j WAVES. The offsets are
    // the same for every tile; a tile's buffers end with the matrix, so rows past it read as zero.
    int xoff[C::LX], woff[C::LW];
#pragma unroll
    for (int j = 0; j < C::LX; j++) {
        const int row = 8 * (j * C::WAVES + wave) + (lane >> 3);
        xoff[j] = row * a.K * 2 + (((lane & 7) ^ swz_x(row)) << 4);
    }
#pragma unroll
    for (int j = 0; j < C::LW; j++) {
        const int row = 8 * (j * C::WAVES + wave) + (lane >> 3);
        woff[j] = row * a.K * 2 + (((lane & 7) ^ swz_w(row)) << 4);
    }
    struct Tile {
        int m0, n0;
        u32x4 x, w;  // buffers over the rows from m0 / n0 on
    };
    auto tile_of = [&](int t) {
        Tile r;
        int mt, nt;
        tile_at(t, a.tm, a.tn, mt, nt);
        r.m0 = mt * C::BM;
        r.n0 = nt * C::BN;
        r.x = rows_rsrc(a.x + (size_t)r.m0 * a.K, min(a.M - r.m0, C::BM) * a.K * 2);
        r.w = rows_rsrc(a.w + (size_t)r.n0 * a.K, min(a.N - r.n0, C::BN) * a.K * 2);
        return r;
    };
    Tile cur = tile_of(id), nxt = cur;
    // Steps past the tile's last are the next tile's first ones, in flight while this one's results
    // are stored; after the last tile they go through empty buffers (no memory is read, zeros land
    // in a slot that is never read), so every step issues and waits alike.
    bool last = SPLIT || id + id_step >= id_end;
    auto issue = [&](int j, int step, int slot) {  // transfer j of LX + LW
        const bool is_x = j < C::LX;
        const int idx = (is_x ? j : j - C::LX) * C::WAVES + wave;
        if ((is_x ? C::XI : C::WI) % C::WAVES != 0 && idx >= (is_x ? C::XI : C::WI)) return;
        const bool over = step >= nk;
        const u32x4 r = over ? (is_x ? nxt.x : nxt.w) : (is_x ? cur.x : cur.w);
        dma16(u32x4{r[0], r[1], over && last ? 0u : r[2], r[3]},
              lds0 + slot * C::STAGE + (is_x ? 0 : C::XST) + idx * 1024, is_x ? xoff[j] : woff[j - C::LX],
              (over ? step - nk : k_lo + step) * ROWB);
    };

    // Fragment read offsets: chunk 4 h + g of the lane's row. The w rows of a pair of n tiles are
    // interleaved (tile t of pair p takes rows 32 p + 8 (l / 4) + 4 t + l % 4), so that a lane's
    // results of both tiles are 8 consecutive columns; t flips bit 2 of the slot, as h does.
    const int wb = wn * TN * 16;
    const int row_x = wm * TM * 16 + r16, row_w = wb + 8 * (r16 >> 2) + (r16 & 3), row_l = wb + (TN - 1) * 16 + r16;
    int xo[2], wo[2], wl[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        xo[h] = row_x * ROWB + (((4 * h + g) ^ swz_x(row_x)) << 4);
        wo[h] = C::XST + row_w * ROWB + (((4 * h + g) ^ swz_w(row_w)) << 4);
        wl[h] = C::XST + row_l * ROWB + (((4 * h + g) ^ swz_w(row_l)) << 4);  // an unpaired last tile
    }

    f32x4 acc[TN][TM];
    u32x4 fx[2][TM], fw[2][TN];

    constexpr int NF = TM + TN, NM = TM * TN, NL = C::LX + C::LW;
    auto read_frag = [&](int q, int h, const unsigned char* st) {
        if (q < TN) {
            if ((TN & 1) && q == TN - 1)
                fw[h][q] = *reinterpret_cast<const u32x4*>(st + wl[h]);
            else
                fw[h][q] = *reinterpret_cast<const u32x4*>(st + wo[h ^ (q & 1)] + (q >> 1) * 32 * ROWB + (q & 1) * 4 * ROWB);
        } else {
            fx[h][q - TN] = *reinterpret_cast<const u32x4*>(st + xo[h] + (q - TN) * 16 * ROWB);
        }
    };
    auto mfmas = [&](int q, int h) {
#pragma unroll
        for (int e = q * NM / NF; e < (q + 1) * NM / NF; e++) {
            const int n = e / TM, m = e % TM;
            acc[n][m] = mfma16(fw[h][n], fx[h][m], acc[n][m]);
        }
    };
    auto barrier = [] {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
    };

    // Step i lives in slot i % ST. (A wave with fewer transfers than the others waits for a little
    // more than it needs: the counts are the smallest wave's.)
    constexpr int PER = C::XI / C::WAVES + C::WI / C::WAVES;  // transfers per wave and step, at least
#pragma unroll
    for (int s = 0; s < ST; s++)
#pragma unroll
        for (int j = 0; j < NL; j++) issue(j, s, s);
    wait_vm<(ST - 1) * PER>();
    barrier();
#pragma unroll
    for (int q = 0; q < NF; q++) read_frag(q, 0, smem);

    // A step's MFMAs run in 2 NF groups (the two 32-k halves). The first QA groups also read the second
    // half's fragments; then a barrier frees the step's slot and its refill is issued, over the next
    // groups; QB groups into the second half a barrier publishes the next step's tile, whose first
    // half is read in the remaining groups. (Earlier and later barriers, and raised wave priority over
    // the MFMAs, measured equal or slower.)
    constexpr int QA = (NF + 1) / 2, QB = NF - QA;
    constexpr int RA = (NF + QA - 1) / QA, RB = (NF + NF - QB - 1) / (NF - QB);  // reads per group
    constexpr int LA = (NL + NF - QA + QB - 1) / (NF - QA + QB);                 // transfers per group
    int slot = 0;
    for (;;) {
#pragma unroll
        for (int n = 0; n < TN; n++)
#pragma unroll
            for (int m = 0; m < TM; m++) acc[n][m] = f32x4{0.f, 0.f, 0.f, 0.f};
        if (!last) nxt = tile_of(id + id_step);
        for (int i = 0; i < nk; i++) {
            const int next = slot + 1 == ST ? 0 : slot + 1;
            const unsigned char *here = smem + slot * C::STAGE, *ahead = smem + next * C::STAGE;
            auto refill = [&](int u) {
#pragma unroll
                for (int j = u * LA; j < min(NL, (u + 1) * LA); j++) issue(j, i + ST, slot);
            };
#pragma unroll
            for (int q = 0; q < NF; q++) {
#pragma unroll
                for (int r = q * RA; r < min(NF, (q + 1) * RA); r++) read_frag(r, 1, here);
                if (q == QA) {
                    wait_lds();
                    barrier();
                }
                if (q >= QA) refill(q - QA);
                __builtin_amdgcn_sched_barrier(0);
                mfmas(q, 0);
                __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int q = 0; q < NF; q++) {
                if (q < QB) refill(NF - QA + q);
                if (q == QB) {
                    wait_vm<(ST - 1) * PER>();
                    barrier();
                }
                // (past the last tile this reads a slot of zeros: never used)
                if (q >= QB) {
#pragma unroll
                    for (int r = (q - QB) * RB; r < min(NF, (q - QB + 1) * RB); r++) read_frag(r, 0, ahead);
                }
                __builtin_amdgcn_sched_barrier(0);
                mfmas(q, 1);
                __builtin_amdgcn_sched_barrier(0);
            }
            slot = next;
        }
        if constexpr (SPLIT) {
            f32x4* p = reinterpret_cast<f32x4*>(a.part) +
                       (((size_t)z * tiles + id) * C::WAVES + wave) * (TN * TM * 64) + lane;
#pragma unroll
            for (int n = 0; n < TN; n++)
#pragma unroll
                for (int m = 0; m < TM; m++) p[(n * TM + m) * 64] = acc[n][m];
        } else {
#pragma unroll
            for (int m = 0; m < TM; m++) {
                const int row = cur.m0 + (wm * TM + m) * 16 + r16;
                if (row >= a.M) continue;
                bf16* yr = a.y + (size_t)row * a.ldy;
#pragma unroll
                for (int p = 0; p < TN / 2; p++) {
                    const int col = cur.n0 + wn * TN * 16 + 32 * p + 8 * g;
                    if (col >= a.N) continue;
                    const f32x4 u = acc[2 * p][m], v = acc[2 * p + 1][m];
                    *reinterpret_cast<u32x4*>(yr + col) =
                        u32x4{pack2(u[0], u[1]), pack2(u[2], u[3]), pack2(v[0], v[1]), pack2(v[2], v[3])};
                }
                if (TN & 1) {
                    const int col = cur.n0 + wn * TN * 16 + (TN - 1) * 16 + 4 * g;
                    const f32x4 u = acc[TN - 1][m];
                    if (col < a.N) *reinterpret_cast<u32x2*>(yr + col) = u32x2{pack2(u[0], u[1]), pack2(u[2], u[3])};
                }
            }
        }
        if (last) break;
        id += id_step;
        cur = nxt;
        last = id + id_step >= id_end;
    }
    wait_vm<0>();  // the empty transfers land before the LDS is given back
}

// Sums the split partials in order and rounds once.
template <int WM, int WN, int TM, int TN>
__global__ void __launch_bounds__(256) mfma_gemm_reduce(const GemmArgs a) {
    constexpr int WAVES = WM * WN, UNITS = WAVES * TM * TN;  // 16 x 16 tiles of a block's tile
    const int lane = threadIdx.x & 63, r16 = lane & 15, g = lane >> 4;
    const int tiles = a.tm * a.tn;
    const int u = blockIdx.x * 4 + (threadIdx.x >> 6);
    if (u >= tiles * UNITS) return;
    const int tile = u / UNITS, rem = u - tile * UNITS;
    const int wave = rem / (TM * TN), nm = rem - wave * (TM * TN);
    const int n = nm / TM, m = nm - n * TM;
    const int wm = wave % WM, wn = wave / WM;
    const f32x4* src = reinterpret_cast<const f32x4*>(a.part) + (size_t)u * 64 + lane;
    const size_t zs = (size_t)tiles * UNITS * 64;
    f32x4 s = src[0];
    for (int z = 1; z < a.split; z++) s += src[z * zs];
    int mt, nt;
    tile_at(tile, a.tm, a.tn, mt, nt);
    const int row = (mt * WM + wm) * TM * 16 + m * 16 + r16;
    const bool single = (TN & 1) && n == TN - 1;
    const int col = (nt * WN + wn) * TN * 16 + (single ? 16 * n + 4 * g : 32 * (n >> 1) + 8 * g + 4 * (n & 1));
    if (row < a.M && col < a.N)
        *reinterpret_cast<u32x2*>(a.y + (size_t)row * a.ldy + col) = u32x2{pack2(s[0], s[1]), pack2(s[2], s[3])};
}

template <int WM, int WN, int TM, int TN, int ST, bool SPLIT>
int launch_part(const GemmArgs& a, hipStream_t st) {
    using C = Cfg<WM, WN, TM, TN, ST>;
    static const hipError_t configured =
        hipFuncSetAttribute(reinterpret_cast<const void*>(mfma_gemm_kernel<WM, WN, TM, TN, ST, SPLIT>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, C::BYTES);
    if (configured != hipSuccess) return configured;
    // one block per CU at most, which takes its tiles one after another: the next tile's first steps
    // are in flight while a tile's results are stored (a tile of fewer steps than stages cannot
    // look ahead like that; forms of which two fit a CU overlap by themselves)
    const int tiles = a.tm * a.tn * a.split, cus = device_cus();
    const int blocks = SPLIT || a.K / BK < ST || 2 * C::BYTES <= 160 * 1024 || cus < 8 ? tiles : std::min(tiles, cus);
    mfma_gemm_kernel<WM, WN, TM, TN, ST, SPLIT><<<blocks, C::THREADS, C::BYTES, st>>>(a);
    return hipGetLastError();
}

template <int WM, int WN, int TM, int TN, int ST>
int launch_tile(GemmArgs a, hipStream_t st) {
    using C = Cfg<WM, WN, TM, TN, ST>;
    a.tm = (a.M + C::BM - 1) / C::BM;
    a.tn = (a.N + C::BN - 1) / C::BN;
    if (a.split == 1) return launch_part<WM, WN, TM, TN, ST, false>(a, st);
    const int rc = launch_part<WM, WN, TM, TN, ST, true>(a, st);
    if (rc != hipSuccess) return rc;
    const int units = a.tm * a.tn * C::WAVES * TM * TN;
    mfma_gemm_reduce<WM, WN, TM, TN><<<(units + 3) / 4, 256, 0, st>>>(a);
    return hipGetLastError();
}

// ------------------------------------------------------------------ tile choice

// The tile forms: waves along M and N, 16-wide tiles per wave along M and N, ring stages, and
// the measured time of a 64-k step of a full device (us).
#define Q35_GEMM_TILES(X)                                                            \
    X(0, 2, 4, 8, 4, 2, 1.421f)  /* 256 x 256 */ X(1, 2, 4, 6, 4, 2, 1.111f) /* 192 x 256 */ \
    X(2, 4, 2, 4, 5, 3, 1.003f)  /* 256 x 160 */ X(3, 4, 2, 4, 4, 3, 0.808f) /* 256 x 128 */ \
    X(4, 4, 2, 3, 6, 3, 0.875f)  /* 192 x 192 */ X(5, 4, 2, 3, 5, 3, 0.805f) /* 192 x 160 */ \
    X(6, 4, 2, 2, 8, 3, 0.902f)  /* 128 x 256 */ X(7, 4, 2, 2, 5, 4, 0.625f) /* 128 x 160 */ \
    X(8, 4, 2, 2, 4, 5, 0.521f)  /* 128 x 128 */ X(9, 8, 1, 1, 5, 5, 0.399f) /* 128 x 80 */  \
    X(10, 4, 2, 1, 6, 5, 0.480f) /* 64 x 192 */  X(11, 4, 2, 1, 2, 5, 0.164f) /* 64 x 64 */ \
    X(12, 2, 4, 1, 4, 4, 0.515f) /* 32 x 256 */ X(13, 4, 2, 4, 6, 2, 1.105f) /* 256 x 192 */ \
    X(14, 4, 2, 3, 4, 4, 0.657f) /* 192 x 128 */ X(15, 4, 2, 2, 6, 4, 0.708f) /* 128 x 192 */ \
    X(16, 4, 2, 1, 4, 6, 0.347f) /* 64 x 128 */ X(17, 8, 1, 2, 9, 3, 0.960f) /* 256 x 144 */

struct TileForm {
    int bm, bn, stages;
    float step;
};
constexpr TileForm TILES[] = {
#define X(i, wm, wn, tm, tn, st, us) {wm * tm * 16, wn * tn * 16, st, us},
    Q35_GEMM_TILES(X)
#undef X
};

constexpr int FORMS = (int)(sizeof(TILES) / sizeof(TILES[0]));

size_t tiles_of(const TileForm& t, int M, int N) {
    return ((size_t)M + t.bm - 1) / t.bm * (((size_t)N + t.bn - 1) / t.bn);
}

// Time of a plan in us: ceil(blocks / CUs) rounds of (steps + start and end), the last round
// cheaper as it is emptier; against it the bytes at the rate that a partly filled device reaches;
// the split's second pass; a launch. Constants fitted to 246 shapes (M 16 to 4096, the N and K of
// the 4B- and 27B-class projections, cold weights) times up to 60 plans each. Over 5,184 other shapes
// (half of them random N and K, M 1 to 8192) and 90,109 plans the modelled times are within 12% (rms), and
// the plan chosen by them takes 1.6% longer than the best measured one on the mean, 0.79 times
// hipBLASLt's first choice (0.32 to 0.66 for 64 to 512 rows of 5120 x 17408 and 2560 x 9728).
float plan_us(const TileForm& t, int split, int M, int N, int K, int cus) {
    const float tiles = (float)((M + t.bm - 1) / t.bm) * (float)((N + t.bn - 1) / t.bn);
    const float blocks = tiles * split, q = blocks / cus, full = std::floor(q), tail = q - full;
    const float round = (float)K / BK / split * t.step + 3.74f;
    const float run = full * round + (tail > 0.f ? round * (1.f - 0.293f * (1.f - tail)) : 0.f);
    const float bytes = 2.f * ((float)M * K + (float)N * K + (float)M * N);
    const float mem = bytes / 6.06e6f / std::pow(std::min(1.f, q), 0.188f);
    const float second = split > 1 ? blocks * t.bm * t.bn * 4.f / 3.94e6f : 0.f;
    return std::sqrt(run * run + mem * mem) + second + 2.87f;
}

// Shapes that hipBLASLt runs, where the plan p measured slower than its first choice: ranges of the
// shape and of the plan's form, from 20,817 pairs of times (cold weights; M 1 to 8192, the N and K of
// the 4B- and 27B-class projections and random ones). "slower / faster" counts the shapes of a range
// by more than 2%, then the mean of this / it. Its choice among its kernels jumps from shape to shape, so
// some shapes beyond these ranges remain on the slower side: 6% of the projections' by more than 2% and
// 2.5% by more than 5% (of the random ones 4% and 2%).
bool library_faster(const MfmaPlan& p, int M, int N, int K, int cus) {
    const TileForm& t = TILES[p.tile];
    const size_t weights = (size_t)N * K;
    const bool one = p.split == 1, k128 = K % 128 == 0, k256 = K % 256 == 0, k512 = K % 512 == 0;
    const float rounds = (float)(tiles_of(t, M, N) * p.split) / cus;
    if (M <= 16) {
        // its 16-row kernels, which step through K by 128 and by 512: 770 / 17, 1.12, and 305 / 18, 1.11
        // (4 x 1024 x 1024: 7.0 us here, 5.9 there; 4 x 5120 x 6144: 18.9, 16.8)
        return (k128 && K >= 384 && K < 1600 && N > 256 && N <= 6400) ||
               (k512 && K > 4352 && K <= 8960 && N <= 8608);
    }
    if (M <= 400 && t.bm == 64) {
        // few weights and a split: the second pass costs what the split saves (149 / 6, 1.11)
        if (t.bn == 64 && p.split > 1 && p.split <= 4 && k128 && weights <= 5000000 &&
            ((K > 1088 && K <= 3648) || (K >= 768 && M <= 30 && weights <= 1080000)))
            return true;
        // 64-row tiles in one round of few steps: 172 / 8, 1.05 (128 x 12352 x 2560: 28.2, 24.8)
        if (M > 64 && M <= 256 && one && k128 && K > 2368 && K <= 3648 && weights > 30800000 && N <= 16384) return true;
        // 64 x 64 tiles, several rows of them, over a deep K: 47 / 6, 1.06 (144 x 5120 x 6144: 30.9, 28.5)
        if (M > 64 && M <= 256 && t.bn == 64 && one && k256 && K > 5824) return true;
    }
    // many parts of few rows: 35 / 1, 1.08
    if (M <= 64 && p.split >= 5 && k256 && N > 8644) return true;
    // The largest tiles: its 256 x 256 kernel takes 1.25 us a 64-k step against 1.42 here, and 10 us a round
    // against 4: slower from a depth on (358 / 58, 1.07; 4096 x 8192 x 8192: 403, 342; 4096 x 4096 x 4096:
    // 108, 90), with more weights a round the deeper (132 / 3, 1.06, and 21 / 0, 1.04).
    if (one && t.bm == 256 && t.bn == 256)
        if (K > 5312 || (K > 3424 && K < 5088) || (K >= 5088 && rounds > 1.87f && rounds <= 2.47f)) return true;
    if (one && t.bm * t.bn >= 256 * 144 && std::max(t.bm, t.bn) == 256)
        if (rounds <= 1.65f ? K > 7648 : K > 5184 && K <= 11520 && N <= 5676) return true;
    // The first rules, drawn from few shapes; what they hold beyond the ones above has always run there:
    // deep products of many rows (43 / 82, 0.95, at the projections' N and K, 118 / 536, 0.89, at random
    // ones), short K with wide N (31 / 51, 0.93), splits of a short K (78 / 76, 0.99).
    return (K > N && M > 1700) || (K <= 2560 && N > 16384 && M > 2100 && M < 4000) ||
           (p.split > 1 && K <= 4096 && M > 384);
}

}  // namespace

bool mfma_gemm_form(int tile, int* bm, int* bn, int* stages) {
    if (tile < 0 || tile >= FORMS) return false;
    *bm = TILES[tile].bm, *bn = TILES[tile].bn, *stages = TILES[tile].stages;
    return true;
}

bool mfma_gemm_takes(const MfmaPlan& p, int M, int N, int K, int ldy, size_t ws_bytes) {
    // whole 64-k steps (and 32-bit offsets within a tile), and rows of y that 16-byte stores fit
    if (K % BK != 0 || K > (1 << 20) || N % 8 != 0 || ldy % 8 != 0) return false;
    if (p.tile < 0 || p.tile >= FORMS || p.split < 1 || p.split > K / BK) return false;
    const TileForm& t = TILES[p.tile];
    const size_t tiles = tiles_of(t, M, N);
    if (p.split == 1) return tiles <= (1u << 30);
    return tiles * p.split <= (1u << 20) && tiles * p.split * t.bm * t.bn * 4 <= ws_bytes;
}

MfmaPlan mfma_gemm_model(int M, int N, int K, int ldy, size_t ws_bytes, int cus) {
    MfmaPlan best;
    if (cus <= 0) return best;
    float best_us = INFINITY;
    for (int i = 0; i < FORMS; i++) {
        const TileForm& t = TILES[i];
        for (int split = 1; split <= 12; split++) {
            // a part keeps at least 6 steps, the parts fill about two rounds, the sums fit the scratch
            if (split > 1 && (K / BK / split < 6 || tiles_of(t, M, N) * split > 2 * (size_t)cus)) break;
            if (!mfma_gemm_takes(MfmaPlan{i, split}, M, N, K, ldy, ws_bytes)) break;
            const float us = plan_us(t, split, M, N, K, cus);
            if (us < best_us) {
                best_us = us;
                best.tile = i;
                best.split = split;
            }
        }
    }
    return best;
}

MfmaPlan mfma_gemm_plan(int M, int N, int K, int ldy, size_t ws_bytes, int cus) {
    const MfmaPlan p = mfma_gemm_model(M, N, K, ldy, ws_bytes, cus);
    return p.tile >= 0 && library_faster(p, M, N, K, cus) ? MfmaPlan{} : p;
}

int mfma_gemm(const MfmaPlan& p, const void* x, const void* w, void* y, void* scratch, int M, int N, int K, int ldy,
              hipStream_t st) {
    const GemmArgs a{static_cast<const bf16*>(x), static_cast<const bf16*>(w), static_cast<bf16*>(y),
                     static_cast<float*>(scratch), M, N, K, ldy, 0, 0, p.split};
    switch (p.tile) {
#define X(i, wm, wn, tm, tn, st_, us) \
    case i:                           \
        return launch_tile<wm, wn, tm, tn, st_>(a, st);
        Q35_GEMM_TILES(X)
#undef X
    }
    return hipErrorInvalidValue;
}

}  // namespace q35
