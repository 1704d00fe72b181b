// q48_gemm.hip — token-batched Q16.48 GEMM on the int8 matrix cores (gfx950).
//
// Y[t][n] = (int64)((sum_k (int128)X[t][k] * W[n][k]) >> 48), per output
// exactly matmul_vec (llama_int.c:1014-1046) applied to each token row.
//
// Digits.  Every int64 v is written with nine signed digits,
//   v = sum_{i<=7} d_i 256^i + 2^64 d_8,
// from u = v + C mod 2^64, C = 0x0080808080808080: d_i = byte_i(u) - 128 for
// i <= 6 (in [-128, 127]), d_7 = byte_7(u) read as int8, and d_8 = 1 when v + C
// overflowed int64 (v >= 2^63 - C, so u < 0 <= v), else 0.  Zero has all digits
// zero, and so have the high digits of a small value and the low digits of a
// value with few significant bits (a bfloat16 weight in Q16.48 has three or
// four nonzero digits, an activation below 2^55 none above d_6).  Then
//   sum_k X W = sum_{a,b<=8} 256^(a+b) P_ab,   P_ab = sum_k d_a(X_k) d_b(W_k),
// an exact integer identity over any k range with no correction terms.  Only
// bits [48,112) are observable, so the pairs with a + b >= 14 are dropped and
// the rest are grouped by d = a + b into 14 int32 accumulators Q_d; |Q_d| <=
// 8 * 2^14 * K < 2^31 while K < 16384 per accumulation run (the plane-8
// products are at most 2^7 each; longer K is split across blocks and summed in
// int128).
//
// Block: 4 waves, 64 tokens x 64 rows; wave w owns 32 tokens x 32 rows as 14
// v_mfma_i32_32x32x32_i8 accumulators (224 registers, one wave per SIMD).
// Per k-step of 32 elements the block splits the int64 tiles into nine byte
// planes in LDS (double-buffered) and records which planes of each tile hold a
// nonzero digit.  k_gemm_i8 multiplies X planes 0..6 by a window of W planes
// LO..LO + 3 (28 MFMAs a step, 7 more in a step whose W tile reaches plane
// LO - 1), LO chosen from the block's first W tile; a block meeting a tile
// outside that (X digits in planes 7-8, W digits outside LO - 1 .. LO + 3)
// writes nothing and k_gemm_i8_full redoes it with every pair (63, plus the
// plane-8 pairs of a tile holding an overflowed value).  Activations below
// 2^55 and bfloat16-exact weights always fit.  The global loads run two steps
// ahead and the byte split of the next step is interleaved with the MFMAs of
// the current one.
#include "q48_digits.hpp"
#include "../../include/intllm_hip.h"

namespace {

constexpr int MT = 64;             // tokens per block
constexpr int MN = 64;             // rows per block
constexpr int MK = 32;             // k per step: one MFMA depth
constexpr int MAXK_RUN = 16320;    // k per accumulation run: |Q_d| < 2^31
constexpr int NPAIR = MK / 32;     // (row, 8 elements) pieces per thread per operand
constexpr int CH = MK / 16;        // 16-byte k chunks per row and plane
constexpr int NPL = 9;             // digit planes per operand

// Byte planes of one stage: [plane][32-row slice][k chunk][32 rows][16 bytes].
// The 64 lanes of an MFMA operand read (row l % 32, chunk 2h + l / 32) touch
// 1 KiB of consecutive bytes, and the 32 lanes of a half-wave store 256
// consecutive bytes: no bank conflicts either way.
constexpr int SLICE = CH * 512;    // one 32-row slice of one plane
constexpr int PLANE = 2 * SLICE;   // 64 rows of one plane
constexpr int STAGE = NPL * PLANE; // one operand: 18 KiB

// Piece p (0 .. 64 CH - 1) of a tile: row r, elements [k8, k8 + 8) of the
// step, and its byte offset in a plane.  Lanes 2i, 2i + 1 take one 16-byte
// chunk of row i: a half-wave covers 16 rows x 16 bytes.
struct Piece {
    int r, k8, off;
};
__device__ __forceinline__ Piece piece(int p)
{
    const int lo = p & 1, rl = (p >> 1) & 15, c = (p >> 5) % CH, rh = (p >> 5) / CH;
    const int r = rh * 16 + rl;
    return {r, (2 * c + lo) * 8, (r >> 5) * SLICE + c * 512 + (r & 31) * 16 + 8 * lo};
}

// Eight consecutive int64 of one row -> nine 8-byte digit words, digit a of
// element e in byte e of word a, stored at plane a.  Returns the planes that
// hold a nonzero digit (bit a).
__device__ __forceinline__ uint32_t split_store(uint8_t *stage, int off, const uint64_t (&v)[8])
{
    uint64_t u[8];
#pragma unroll
    for (int e = 0; e < 8; ++e)
        u[e] = v[e] + kDig;
    uint32_t l0[4], l1[4], h0[4], h1[4];
    tr4((uint32_t)u[0], (uint32_t)u[1], (uint32_t)u[2], (uint32_t)u[3], l0);
    tr4((uint32_t)u[4], (uint32_t)u[5], (uint32_t)u[6], (uint32_t)u[7], l1);
    tr4((uint32_t)(u[0] >> 32), (uint32_t)(u[1] >> 32), (uint32_t)(u[2] >> 32),
        (uint32_t)(u[3] >> 32), h0);
    tr4((uint32_t)(u[4] >> 32), (uint32_t)(u[5] >> 32), (uint32_t)(u[6] >> 32),
        (uint32_t)(u[7] >> 32), h1);
    uint2 d[NPL];
#pragma unroll
    for (int a = 0; a < 4; ++a)
        d[a] = make_uint2(l0[a] ^ 0x80808080u, l1[a] ^ 0x80808080u);
#pragma unroll
    for (int a = 0; a < 3; ++a)
        d[4 + a] = make_uint2(h0[a] ^ 0x80808080u, h1[a] ^ 0x80808080u);
    d[7] = make_uint2(h0[3], h1[3]);
    // overflow flags: bit 31 of u's high word set where v's is clear
    uint32_t f0 = 0, f1 = 0;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        f0 |= (((uint32_t)(u[e] >> 32) & ~(uint32_t)(v[e] >> 32)) >> 31) << (8 * e);
        f1 |= (((uint32_t)(u[e + 4] >> 32) & ~(uint32_t)(v[e + 4] >> 32)) >> 31) << (8 * e);
    }
    d[8] = make_uint2(f0, f1);
    uint8_t *p = stage + off;
    uint32_t m = 0;
#pragma unroll
    for (int a = 0; a < NPL; ++a) {
        *reinterpret_cast<uint2 *>(p + a * PLANE) = d[a];
        m |= ((d[a].x | d[a].y) != 0 ? 1u : 0u) << a;
    }
    return m;
}

// The window pass's split of eight consecutive int64: only planes P0..P1 are
// stored.  Returns bit 0 when a digit outside P0..P1 is nonzero or a value may
// have overflowed (v >= 2^63 - C needs v's high word >= 0x7F7F7F7F: tested on
// that word alone, so a few values below the bound are caught too), and bit 1
// when plane EXT (-1: none) holds a nonzero digit.
template <int P0, int P1, int EXT>
__device__ __forceinline__ uint32_t split_store_win(uint8_t *stage, int off,
                                                   const uint64_t (&v)[8])
{
    uint64_t u[8];
    bool big = false;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        u[e] = v[e] + kDig;
        big |= (int32_t)(uint32_t)(v[e] >> 32) >= 0x7f7f7f7f;
    }
    uint32_t l0[4], l1[4], h0[4], h1[4];
    tr4((uint32_t)u[0], (uint32_t)u[1], (uint32_t)u[2], (uint32_t)u[3], l0);
    tr4((uint32_t)u[4], (uint32_t)u[5], (uint32_t)u[6], (uint32_t)u[7], l1);
    tr4((uint32_t)(u[0] >> 32), (uint32_t)(u[1] >> 32), (uint32_t)(u[2] >> 32),
        (uint32_t)(u[3] >> 32), h0);
    tr4((uint32_t)(u[4] >> 32), (uint32_t)(u[5] >> 32), (uint32_t)(u[6] >> 32),
        (uint32_t)(u[7] >> 32), h1);
    uint2 d[8];
#pragma unroll
    for (int a = 0; a < 4; ++a)
        d[a] = make_uint2(l0[a] ^ 0x80808080u, l1[a] ^ 0x80808080u);
#pragma unroll
    for (int a = 0; a < 3; ++a)
        d[4 + a] = make_uint2(h0[a] ^ 0x80808080u, h1[a] ^ 0x80808080u);
    d[7] = make_uint2(h0[3], h1[3]);
    uint8_t *p = stage + off;
    uint32_t out = 0;
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        if (a >= P0 && a <= P1)
            *reinterpret_cast<uint2 *>(p + a * PLANE) = d[a];
        else
            out |= d[a].x | d[a].y;
    }
    uint32_t r = (out != 0 || big) ? 1u : 0u;
    if (EXT >= 0)
        r |= (d[EXT < 0 ? 0 : EXT].x | d[EXT < 0 ? 0 : EXT].y) != 0 ? 2u : 0u;
    return r;
}

// Eight elements [k, k + 8) of a row; positions at or past kend read as 0
// (all digits zero, so they add nothing to any Q_d).
template <bool VEC, bool TAIL>
__device__ __forceinline__ void load8(uint64_t (&v)[8], const int64_t *row, int k, int kend)
{
    if (!TAIL && VEC) {
        const ulonglong2 *p = reinterpret_cast<const ulonglong2 *>(row + k);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const ulonglong2 u = p[e];
            v[2 * e] = u.x;
            v[2 * e + 1] = u.y;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = (!TAIL || k + e < kend) ? (uint64_t)row[TAIL ? min(k + e, kend - 1) : k + e]
                                           : 0;
    }
}

// OR of a 32-bit value over the wave (DPP within rows of 16, then the rows)
__device__ __forceinline__ uint32_t wave_or(uint32_t v)
{
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, Q48_DPP_XOR1, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, Q48_DPP_XOR2, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, Q48_DPP_HALF_MIRROR, 0xf, 0xf, false);
    v |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, Q48_DPP_MIRROR, 0xf, 0xf, false);
    return (uint32_t)(__builtin_amdgcn_readlane((int)v, 0) | __builtin_amdgcn_readlane((int)v, 16) |
                      __builtin_amdgcn_readlane((int)v, 32) | __builtin_amdgcn_readlane((int)v, 48));
}

// Operand offset of lane l in a 32-row slice of a plane (one 32-deep half)
__device__ __forceinline__ int opnd_off(int lane) { return (lane >> 5) * 512 + (lane & 31) * 16; }

// The 28 MFMAs of a step whose X digits lie in planes 0..6 and W digits in
// planes LO..LO + 3.
template <int LO>
__device__ __forceinline__ void mfma_window(v16i (&acc)[14], const uint8_t *xs, const uint8_t *ws,
                                            int lane)
{
    static_assert(LO >= 0 && LO + 3 <= 7, "window within planes 0..7");
    const int off = opnd_off(lane);
    v4i A[7], B[4];
#pragma unroll
    for (int a = 0; a < 7; ++a)
        A[a] = *reinterpret_cast<const v4i *>(xs + a * PLANE + off);
#pragma unroll
    for (int j = 0; j < 4; ++j)
        B[j] = *reinterpret_cast<const v4i *>(ws + (LO + j) * PLANE + off);
#pragma unroll
    for (int a = 0; a < 7; ++a)
#pragma unroll
        for (int j = 0; j < 4; ++j)
            acc[a + LO + j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[a], B[j], acc[a + LO + j],
                                                                    0, 0, 0);
}

// X planes 0..6 against one more W plane B (B <= 7).
template <int B>
__device__ __forceinline__ void mfma_plane_w(v16i (&acc)[14], const uint8_t *xs,
                                             const uint8_t *ws, int lane)
{
    const int off = opnd_off(lane);
    const v4i Bv = *reinterpret_cast<const v4i *>(ws + B * PLANE + off);
#pragma unroll
    for (int a = 0; a < 7; ++a)
        if (a + B <= 13) {
            const v4i A = *reinterpret_cast<const v4i *>(xs + a * PLANE + off);
            acc[a + B] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, Bv, acc[a + B], 0, 0, 0);
        }
}

// The 63 MFMAs of planes 0..7 x 0..7 (a + b <= 13).
__device__ __forceinline__ void mfma_all(v16i (&acc)[14], const uint8_t *xs, const uint8_t *ws,
                                         int lane)
{
    const int off = opnd_off(lane);
    v4i A[8], B[8];
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        A[a] = *reinterpret_cast<const v4i *>(xs + a * PLANE + off);
        B[a] = *reinterpret_cast<const v4i *>(ws + a * PLANE + off);
    }
#pragma unroll
    for (int a = 0; a < 8; ++a)
#pragma unroll
        for (int b = 0; b < 8; ++b)
            if (a + b <= 13)
                acc[a + b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A[a], B[b], acc[a + b], 0, 0, 0);
}

// The plane-8 pairs: X planes 0..5 with W plane 8 (wide: W overflowed) and X
// plane 8 with W planes 0..5.
__device__ __forceinline__ void mfma_plane8(v16i (&acc)[14], const uint8_t *xs,
                                            const uint8_t *ws, int lane, bool w8, bool x8)
{
    const int off = opnd_off(lane);
    if (w8) {
        const v4i B8 = *reinterpret_cast<const v4i *>(ws + 8 * PLANE + off);
#pragma unroll
        for (int a = 0; a < 6; ++a) {
            const v4i A = *reinterpret_cast<const v4i *>(xs + a * PLANE + off);
            acc[a + 8] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A, B8, acc[a + 8], 0, 0, 0);
        }
    }
    if (x8) {
        const v4i A8 = *reinterpret_cast<const v4i *>(xs + 8 * PLANE + off);
#pragma unroll
        for (int b = 0; b < 6; ++b) {
            const v4i B = *reinterpret_cast<const v4i *>(ws + b * PLANE + off);
            acc[b + 8] = __builtin_amdgcn_mfma_i32_32x32x32_i8(A8, B, acc[b + 8], 0, 0, 0);
        }
    }
}

// Tile of block b in a grid of nn row tiles x nt token tiles.  Blocks go
// round-robin to the 8 XCDs (each with its own L2), so b is first renumbered
// to give every XCD a contiguous range, and that range is walked in groups of
// GROUP row tiles: a group's W tiles stay in cache while its token tiles pass.
constexpr int GROUP = 8;
__host__ __device__ __forceinline__ void tile_of(int b, int nn, int nt, int &n_tile, int &t_tile)
{
    const int total = nn * nt, q = total / 8, r = total % 8, x = b % 8, l = b / 8;
    const int pid = x < r ? x * (q + 1) + l : r * (q + 1) + (x - r) * q + l;
    const int per = GROUP * nt, g = pid / per, first = g * GROUP;
    const int gs = nn - first < GROUP ? nn - first : GROUP, in = pid - g * per;
    n_tile = first + in % gs;
    t_tile = in / gs;
}

// The block whose tile is (n_tile, t_tile): tile_of's inverse.
__host__ __device__ inline int block_of(int n_tile, int t_tile, int nn, int nt)
{
    const int total = nn * nt, q = total / 8, r = total % 8;
    const int g = n_tile / GROUP, first = g * GROUP;
    const int gs = nn - first < GROUP ? nn - first : GROUP;
    const int pid = first * nt + t_tile * gs + (n_tile - first);
    const int x = pid < r * (q + 1) ? pid / (q + 1) : r + (pid - r * (q + 1)) / (q > 0 ? q : 1);
    const int l = pid < r * (q + 1) ? pid % (q + 1) : (pid - r * (q + 1)) % (q > 0 ? q : 1);
    return 8 * l + x;
}

// Register i of the 14 digit-sum accumulators as the 128-bit sum
// S = sum_d acc[d][i] 256^d (mod 2^128, words lo and hi), where only digit
// sums D0..D1 can be nonzero.  Groups of four digit sums are exact int64
// (|g| < 2^31 (1 + 2^8 + 2^16 + 2^24) < 2^56), then
// S = g0 + 2^32 g1 + 2^64 g2 + 2^96 g3 in two words with one carry.
template <int D0, int D1>
__device__ __forceinline__ void acc_sum128(const v16i (&acc)[14], int i, uint64_t &lo,
                                           uint64_t &hi)
{
    int64_t g[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        uint64_t v = 0;
#pragma unroll
        for (int e = 3; e >= 0; --e) {
            const int d = 4 * j + e;
            v <<= 8;
            if (d >= D0 && d <= D1 && d < 14)
                v += (uint64_t)(int64_t)acc[d][i];
        }
        g[j] = (int64_t)v;
    }
    lo = (uint64_t)g[0] + ((uint64_t)g[1] << 32);
    const uint64_t carry = lo < (uint64_t)g[0] ? 1u : 0u;
    hi = (uint64_t)(g[0] >> 63) + (uint64_t)(g[1] >> 32) + carry + (uint64_t)g[2] +
         ((uint64_t)g[3] << 32);
}

// The block's tiles, loaders and accumulators, shared by the kernel's paths.
struct GemmTile {
    int64_t *Y;
    uint64_t *P;
    int T, N, n0, t0, kbeg, kend, nfull, z, S;
    bool tail;
};

// Block b's tile and k range (split z of S, spb steps each), and the rows it
// loads: piece tid of both tiles.
__device__ __forceinline__ GemmTile gemm_tile(int b, int z, int S, int64_t *Y, uint64_t *P,
                                              const int64_t *W, const int64_t *X, int T, int N,
                                              int K, int spb, Piece (&pc)[NPAIR],
                                              const int64_t *(&xrow)[NPAIR],
                                              const int64_t *(&wrow)[NPAIR])
{
    int n_tile, t_tile;
    tile_of(b, (N + MN - 1) / MN, (T + MT - 1) / MT, n_tile, t_tile);
    GemmTile g;
    g.Y = Y;
    g.P = P;
    g.T = T;
    g.N = N;
    g.n0 = n_tile * MN;
    g.t0 = t_tile * MT;
    g.z = z;
    g.S = S;
    g.kbeg = z * spb * MK;
    g.kend = max(g.kbeg, min(K, g.kbeg + spb * MK));
    g.nfull = (g.kend - g.kbeg) / MK;
    g.tail = (g.kend - g.kbeg) % MK != 0;
#pragma unroll
    for (int j = 0; j < NPAIR; ++j) {
        pc[j] = piece((int)threadIdx.x + 256 * j);
        xrow[j] = X + (size_t)min(g.t0 + pc[j].r, T - 1) * K + pc[j].k8;
        wrow[j] = W + (size_t)min(g.n0 + pc[j].r, N - 1) * K + pc[j].k8;
    }
    return g;
}

// One pass of the block's k range.  LO >= 0: X planes 0..6 against W planes
// LO..LO + 3, plus W plane LO - 1 in the steps whose tile holds it; a step
// with digits elsewhere returns false before anything is written (the caller
// then runs LO = -1).  LO = -1: every pair, never fails.  On success the
// block's outputs are written.
template <int LO, bool VEC>
__device__ __forceinline__ bool gemm_pass(const GemmTile &g, uint8_t (&lds)[2][2][STAGE],
                                          uint32_t (&pm)[2][4], const int64_t *const (&xrow)[NPAIR],
                                          const int64_t *const (&wrow)[NPAIR],
                                          const Piece (&pc)[NPAIR])
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wt = w >> 1, wn = w & 1;   // wave's token slice, row slice
    const int kbeg = g.kbeg, kend = g.kend, nfull = g.nfull;
    v16i acc[14];
#pragma unroll
    for (int d = 0; d < 14; ++d)
        acc[d] = (v16i){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};

    typedef uint64_t Regs[NPAIR][8];
    auto load = [&](Regs &gx, Regs &gw, int k) {
#pragma unroll
        for (int j = 0; j < NPAIR; ++j) {
            load8<VEC, false>(gx[j], xrow[j], k, kend);
            load8<VEC, false>(gw[j], wrow[j], k, kend);
        }
    };
    // split a step's tiles into stage st and publish the wave's plane masks
    // W planes a window pass stores and takes: LO - 1 .. LO + 3
    constexpr int WP0 = LO > 0 ? LO - 1 : 0, WP1 = LO + 3, WEXT = LO > 0 ? LO - 1 : -1;
    // split a step's tiles into stage st and publish the wave's plane masks:
    // every plane's (X in bits 0..8, W in 9..17) for the full pass; for a
    // window pass bit 0 = a digit outside the window, bit 1 = W plane LO - 1
    auto store = [&](int st, const Regs &gx, const Regs &gw) {
        uint32_t m;
        if constexpr (LO >= 0) {
            uint32_t r = 0;
#pragma unroll
            for (int j = 0; j < NPAIR; ++j)
                r |= split_store_win<0, 6, -1>(lds[st][0], pc[j].off, gx[j]) |
                     split_store_win<WP0, WP1, WEXT>(lds[st][1], pc[j].off, gw[j]);
            m = (__builtin_amdgcn_ballot_w64((r & 1u) != 0) != 0 ? 1u : 0u) |
                (__builtin_amdgcn_ballot_w64((r & 2u) != 0) != 0 ? 2u : 0u);
        } else {
            uint32_t mx = 0, mw = 0;
#pragma unroll
            for (int j = 0; j < NPAIR; ++j) {
                mx |= split_store(lds[st][0], pc[j].off, gx[j]);
                mw |= split_store(lds[st][1], pc[j].off, gw[j]);
            }
            m = wave_or(mx | (mw << 9));
        }
        if (lane == 0)
            pm[st][w] = m;
    };
    // the stage's masks (uniform over the block)
    auto planes = [&](int st) {
        const uint32_t m = pm[st][0] | pm[st][1] | pm[st][2] | pm[st][3];
        return (uint32_t)__builtin_amdgcn_readfirstlane((int)m);
    };
    bool ok = true;
    // MFMAs of stage st with the split of the next step interleaved (its data
    // arrived a step ago); the last step splits a clamped re-read, never used
    auto multiply = [&](int st, bool split_next, const Regs &cx_, const Regs &cw_) {
        const uint8_t *xs = &lds[st][0][0] + wt * SLICE, *ws = &lds[st][1][0] + wn * SLICE;
        const uint32_t m = planes(st);
        if constexpr (LO >= 0) {
            // a step outside the window still runs (its products are
            // discarded with the pass), so the loop body has no exit
            ok &= (m & 1u) == 0;
            mfma_window<LO < 0 ? 0 : LO>(acc, xs, ws, lane);
            if (split_next)
                store(st ^ 1, cx_, cw_);
            __builtin_amdgcn_sched_group_barrier(0x100, 11, 0);
#pragma unroll
            for (int i = 0; i < 28; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 5, 0);
            }
            if (LO > 0 && (m & 2u))
                mfma_plane_w<LO < 1 ? 0 : LO - 1>(acc, xs, ws, lane);
        } else {
            const uint32_t mx = m & 0x1ffu, mw = m >> 9;
            mfma_all(acc, xs, ws, lane);
            if (split_next)
                store(st ^ 1, cx_, cw_);
            __builtin_amdgcn_sched_group_barrier(0x100, 16, 0);
#pragma unroll
            for (int i = 0; i < 63; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);
            }
            if ((mw | mx) & 0x100u)
                mfma_plane8(acc, xs, ws, lane, (mw & 0x100u) != 0, (mx & 0x100u) != 0);
        }
    };
    // Steps go two ahead: step s multiplies stage s & 1, splits step s + 1
    // (loaded during step s - 1) into the other stage and loads step s + 2.
    // Register sets alternate: step s loads into set s & 1.
    // The window pass loads three steps ahead (register sets rotating by
    // step), so a step's tiles have two steps to arrive; the full pass, at
    // the register limit, two.
    constexpr int AHEAD = LO >= 0 ? 3 : 2;
    Regs gx0, gw0, gx1, gw1, gx2, gw2;
    const int last = max(nfull - 1, 0);
    __syncthreads();   // the stages and masks of an earlier pass are consumed
    if (nfull > 0) {
        load(gx0, gw0, kbeg);
        load(gx1, gw1, kbeg + min(1, last) * MK);
        if (AHEAD == 3)
            load(gx2, gw2, kbeg + min(2, last) * MK);
        store(0, gx0, gw0);
    }
    __syncthreads();
    auto step = [&](int s, Regs &lx, Regs &lw, const Regs &cx_, const Regs &cw_) {
        // step s + AHEAD's tiles (clamped to the last step: in bounds, unused)
        load(lx, lw, kbeg + min(s + AHEAD, last) * MK);
        __builtin_amdgcn_sched_barrier(0);
        multiply(s & 1, true, cx_, cw_);
        __syncthreads();
    };
    // groups with no branch inside the loop body's loads; a failed step is
    // seen by the whole block (the masks are uniform), which leaves together
    int s = 0;
    if constexpr (AHEAD == 3) {
        for (; ok && s + 2 < nfull; s += 3) {
            step(s, gx0, gw0, gx1, gw1);
            step(s + 1, gx1, gw1, gx2, gw2);
            step(s + 2, gx2, gw2, gx0, gw0);
        }
        if (ok && s < nfull)
            step(s, gx0, gw0, gx1, gw1);
        if (ok && s + 1 < nfull)
            step(s + 1, gx1, gw1, gx2, gw2);
    } else {
        for (; ok && s + 1 < nfull; s += 2) {
            step(s, gx0, gw0, gx1, gw1);
            if (ok)
                step(s + 1, gx1, gw1, gx0, gw0);
        }
        if (ok && s < nfull)
            step(s, gx0, gw0, gx1, gw1);
    }
    if (ok && g.tail) {
        const int kt = kbeg + nfull * MK;
#pragma unroll
        for (int j = 0; j < NPAIR; ++j) {
            load8<VEC, true>(gx0[j], xrow[j], kt, kend - pc[j].k8);
            load8<VEC, true>(gw0[j], wrow[j], kt, kend - pc[j].k8);
        }
        store(nfull & 1, gx0, gw0);
        __syncthreads();
        multiply(nfull & 1, false, gx0, gw0);
    }
    if (!ok)
        return false;

    // lane l, register i: token 8 (i / 4) + 4 (l / 32) + i % 4, row l % 32;
    // the window pass touches digit sums LO - 1 .. LO + 9 only
    constexpr int D0 = LO > 0 ? LO - 1 : 0, D1 = LO < 0 ? 13 : LO + 9;
    const int nl = 32 * wn + (lane & 31), n = g.n0 + nl;
    if (n >= g.N)
        return true;
#pragma unroll
    for (int i = 0; i < 16; ++i) {
        const int tl = 32 * wt + 8 * (i >> 2) + 4 * (lane >> 5) + (i & 3), t = g.t0 + tl;
        if (t >= g.T)
            continue;
        uint64_t lo, hi;
        acc_sum128<D0, D1>(acc, i, lo, hi);
        if (g.S == 1) {
            g.Y[(size_t)t * g.N + n] = (int64_t)((hi << 16) | (lo >> 48));
        } else {
            uint64_t *p = g.P + 2 * (((size_t)g.z * g.T + t) * g.N + n);
            *reinterpret_cast<ulonglong2 *>(p) = make_ulonglong2(lo, hi);
        }
    }
    return true;
}

// grid (ceil(N/64) * ceil(T/64), 1, S): split z covers k-steps [z*spb, (z+1)*spb).
// S == 1: Y gets the shifted result;
// S > 1: P[z][t][n] gets the block's int128 partial sum (two uint64, lo first).
// The window of W planes comes from the block's first W tile (its top plane
// h gives LO = h - 3, clamped to 0..4: small weights reach lower planes, the
// largest magnitudes set the top).  A block whose tiles leave the window
// writes nothing and sets redo[block] (else clears it) for k_gemm_i8_full.
template <bool VEC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
k_gemm_i8(int64_t *__restrict__ Y, uint64_t *__restrict__ P, int *__restrict__ redo,
          const int64_t *__restrict__ W, const int64_t *__restrict__ X, int T, int N, int K,
          int spb)
{
    __shared__ __align__(16) uint8_t lds[2][2][STAGE];   // [stage][X, W]
    __shared__ uint32_t pm[2][4];                         // [stage][wave]: planes, X | W << 9
    const int tid = threadIdx.x;
    Piece pc[NPAIR];
    const int64_t *xrow[NPAIR], *wrow[NPAIR];
    const GemmTile g = gemm_tile(blockIdx.x, blockIdx.z, gridDim.z, Y, P, W, X, T, N, K, spb,
                                 pc, xrow, wrow);

    // the first W tile's planes (every digit of the block's first step)
    uint32_t mw = 0;
    if (g.kend > g.kbeg) {
#pragma unroll
        for (int j = 0; j < NPAIR; ++j) {
            uint64_t v[8];
            if (g.nfull > 0)
                load8<VEC, false>(v, wrow[j], g.kbeg, g.kend);
            else
                load8<VEC, true>(v, wrow[j], g.kbeg, g.kend - pc[j].k8);
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const uint64_t u = v[e] + kDig, dz = u ^ kDig;   // digits 0..6: bytes of dz
#pragma unroll
                for (int a = 0; a < 7; ++a)
                    mw |= ((dz >> (8 * a)) & 0xffu) != 0 ? 1u << a : 0u;
                mw |= (u >> 56) != 0 ? 1u << 7 : 0u;
            }
        }
    }
    mw = wave_or(mw);
    if ((tid & 63) == 0)
        pm[0][tid >> 6] = mw;
    __syncthreads();
    mw = (uint32_t)__builtin_amdgcn_readfirstlane((int)(pm[0][0] | pm[0][1] | pm[0][2] | pm[0][3]));
    const int h = mw ? 31 - __builtin_clz(mw) : 3;
    const int lo = min(max(h - 3, 0), 4);
    bool done;
    switch (lo) {
    case 0: done = gemm_pass<0, VEC>(g, lds, pm, xrow, wrow, pc); break;
    case 1: done = gemm_pass<1, VEC>(g, lds, pm, xrow, wrow, pc); break;
    case 2: done = gemm_pass<2, VEC>(g, lds, pm, xrow, wrow, pc); break;
    case 3: done = gemm_pass<3, VEC>(g, lds, pm, xrow, wrow, pc); break;
    default: done = gemm_pass<4, VEC>(g, lds, pm, xrow, wrow, pc); break;
    }
    if (tid == 0)
        redo[blockIdx.z * gridDim.x + blockIdx.x] = done ? 0 : 1;
}

// Every pair for the blocks k_gemm_i8 left (redo set), nb blocks of S splits:
// block b of this grid takes blocks b, b + gridDim.x, ... of that grid.
template <bool VEC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
k_gemm_i8_full(int64_t *__restrict__ Y, uint64_t *__restrict__ P, const int *__restrict__ redo,
               const int64_t *__restrict__ W, const int64_t *__restrict__ X, int T, int N,
               int K, int spb, int nb, int S)
{
    __shared__ __align__(16) uint8_t lds[2][2][STAGE];
    __shared__ uint32_t pm[2][4];
    __shared__ int list[256], cnt;
    // the block's candidates i = blockIdx.x + c gridDim.x, 256 flags read at
    // once (one memory round trip when nothing is to be redone)
    const int tid = threadIdx.x, per = (nb * S - (int)blockIdx.x + gridDim.x - 1) / gridDim.x;
    for (int c0 = 0; c0 < per; c0 += 256) {
        if (tid == 0)
            cnt = 0;
        __syncthreads();
        const int i = (int)blockIdx.x + (c0 + tid) * (int)gridDim.x;
        if (c0 + tid < per && redo[i])
            list[atomicAdd(&cnt, 1)] = i;
        __syncthreads();
        const int n = cnt;
        for (int l = 0; l < n; ++l) {
            const int b = list[l];
            Piece pc[NPAIR];
            const int64_t *xrow[NPAIR], *wrow[NPAIR];
            const GemmTile g =
                gemm_tile(b % nb, b / nb, S, Y, P, W, X, T, N, K, spb, pc, xrow, wrow);
            gemm_pass<-1, VEC>(g, lds, pm, xrow, wrow, pc);
        }
        __syncthreads();   // list and cnt reused
    }
}

// Y[t][n] = (sum_z P[z][t][n]) >> 48
__global__ __launch_bounds__(256) void k_gemm_i8_reduce(int64_t *__restrict__ Y,
                                                       const uint64_t *__restrict__ P, int T,
                                                       int N, int S)
{
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)T * N)
        return;
    q48_u128 tot = 0;
    for (int z = 0; z < S; ++z) {
        const ulonglong2 u =
            *reinterpret_cast<const ulonglong2 *>(P + 2 * ((size_t)z * T * N + i));
        tot += ((q48_u128)u.y << 64) | u.x;
    }
    Y[i] = (int64_t)((q48_i128)tot >> 48);
}

// ---------------------------------------------------------------------------
// Planes path: operands split once into digit planes in HBM, then moved
// into LDS by DMA (global_load_lds), so the k loop runs no digit split.
// ---------------------------------------------------------------------------

// The shift of each 64-row tile's planes (k_planes) from its largest
// magnitude.  Block (rt, p) of grid (nn, parts) takes the p-th of the row
// tile's parts and leaves its magnitude's code in bits 20..25 of the row
// tile's p-th mask word: 8 h + 7 - shift, h the plane its largest magnitude
// fills, which grows with the magnitude, so k_planes takes the parts' largest.
// Parts of about 8192 values, one load batch a thread, fill the chip at any
// size: with a block per row tile the pass was a chain of K / 128 batches on
// N / 64 compute units (q48_gemm_prepare of 1024 x 1024 10.3 -> 7.3 us, 2048 x
// 2048 23.4 -> 18.3, 2048 x 5632 55.6 -> 40.3; 11264 x 2048 88.4 -> 87.4).
constexpr int TS_PARTS = 16;
__host__ __device__ __forceinline__ int tile_parts(int K, int nsteps)
{
    const int p = (K + 127) / 128;
    return min(min(p, nsteps), TS_PARTS);
}
__global__ __launch_bounds__(1024) void k_tile_shift(uint32_t *__restrict__ mask,
                                                    const int64_t *__restrict__ src, int R,
                                                    int K, int nsteps)
{
    __shared__ uint64_t red[16];
    const int tid = threadIdx.x, r0 = (int)blockIdx.x * MN, r1 = min(r0 + MN, R);
    const size_t all = (size_t)(r1 - r0) * K;
    // whole 8192s a part, the last takes what is left (possibly nothing)
    const size_t per = ((all + gridDim.y - 1) / gridDim.y + 8191) & ~(size_t)8191;
    const size_t b = min(all, per * blockIdx.y), n = min(all - b, per);
    const int64_t *p = src + (size_t)r0 * K + b;
    uint64_t mx = 0;
    auto add = [&](uint64_t v) {
        const uint64_t a = (int64_t)v < 0 ? (uint64_t)0 - v : v;
        mx = a > mx ? a : mx;
    };
    size_t i0 = 0;
    if ((((uintptr_t)p) & 15) == 0) {
        const ulonglong2 *q = reinterpret_cast<const ulonglong2 *>(p);
        const size_t n4 = n / 8192;   // groups of four 16-byte loads a thread
        for (size_t g = 0; g < n4; ++g) {
            ulonglong2 u[4];
#pragma unroll
            for (int e = 0; e < 4; ++e)
                u[e] = q[4096 * g + 1024 * e + tid];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                add(u[e].x);
                add(u[e].y);
            }
        }
        i0 = 8192 * n4;
    }
    for (size_t i = i0 + tid; i < n; i += 1024)
        add((uint64_t)p[i]);
    mx = (uint64_t)q48_wave_max64((int64_t)(mx >> 1));   // halved: 2^63 stays positive
    if ((tid & 63) == 0)
        red[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) {
        for (int i = 1; i < 16; ++i)
            mx = red[i] > mx ? red[i] : mx;
        mx = 2 * mx + 1;   // at least the largest magnitude
        // the lowest plane h <= 6 whose digits reach mx (values up to
        // sum_{i<=h} 127 256^i), and the largest shift that stays within it
        uint64_t lim = 127;
        uint32_t h = 0;
        for (; h < 6 && mx > lim; ++h)
            lim = lim * 256 + 127;
        uint32_t sh = 0;
        while (sh < 7 && (mx << (sh + 1)) <= lim)
            ++sh;
        mask[(size_t)blockIdx.x * nsteps + blockIdx.y] =
            (mx <= lim ? 8 * h + 7 - sh : 63u) << 20;
    }
}

// Digit planes of a row-major int64 matrix (R rows, K columns) in the LDS
// stage order of the window kernels: per row tile rt (64 rows) and k-step s
// (32 columns), block rt * nsteps + s holds planes 0..7 of the nine-digit
// form, 2 KB each ([32-row slice][16-column chunk][32 rows][16 bytes]; rows
// past R and columns past K are zero), and mask[rt * nsteps + s] has bit a
// when plane a holds a nonzero digit and bit 8 when a value may have
// overflowed v + C (high word >= 0x7F7F7F7F; plane 8 itself is not stored).
// X (!WGT) has one block more per row tile, of zero planes, for the steps that fill
// up the k loop's groups of four.
// shifted (WGT): the row tile's values are multiplied by 2^shift before the split
// (from the largest code of k_tile_shift's parts; every mask of the row tile
// keeps that code, so a block may read a part's word before or after the
// block that writes its own mask there; bits 16..18: the shift), so that the largest one fills its top plane: a
// bfloat16 weight's low bits then reach down to fewer planes (N(0, 0.02)
// weights: 10% of the 64 x 32 tiles need a fourth plane, 34% unshifted).
template <bool WGT>
__global__ __launch_bounds__(256) void k_planes(uint8_t *__restrict__ dst, uint32_t *mask,
                                               const int64_t *__restrict__ src, int R, int K,
                                               int nsteps, int shifted)
{
    __shared__ uint32_t red[4];
    const int tid = threadIdx.x, pitch = WGT ? nsteps : nsteps + 1;
    const int rt = (int)blockIdx.x / pitch, st = (int)blockIdx.x % pitch;
    const Piece pc = piece(tid);
    const int row = rt * MN + pc.r, k0 = st * MK + pc.k8;
    if (!WGT && st >= nsteps) {   // padding: zero planes, no mask
        for (int i = tid; i < PLANE / 2; i += 256)
            reinterpret_cast<uint4 *>(dst + (size_t)blockIdx.x * 8 * PLANE)[i] =
                make_uint4(0, 0, 0, 0);
        return;
    }
    uint64_t v[8];
    const int64_t *rp = src + (size_t)min(row, R - 1) * K + k0;
    if (row < R && k0 + 8 <= K && (((uintptr_t)rp) & 15) == 0) {
        const ulonglong2 *q = reinterpret_cast<const ulonglong2 *>(rp);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const ulonglong2 u = q[e];
            v[2 * e] = u.x;
            v[2 * e + 1] = u.y;
        }
    } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] = row < R && k0 + e < K ? (uint64_t)rp[e] : 0;
    }
    uint32_t sh = 0, code = 0;
    if (WGT && shifted) {
        const int part = min(tid & (TS_PARTS - 1), tile_parts(K, nsteps) - 1);
        code = (__hip_atomic_load(mask + (size_t)rt * nsteps + part, __ATOMIC_RELAXED,
                                  __HIP_MEMORY_SCOPE_AGENT) >> 20) & 63u;
        code = (uint32_t)q48_wave_max64((int64_t)code);
        sh = 7u - (code & 7u);
    }
    if (sh)
#pragma unroll
        for (int e = 0; e < 8; ++e)
            v[e] <<= sh;
    uint64_t u[8];
    bool big = false;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
        u[e] = v[e] + kDig;
        big |= (int32_t)(uint32_t)(v[e] >> 32) >= 0x7f7f7f7f;
    }
    uint32_t l0[4], l1[4], h0[4], h1[4];
    tr4((uint32_t)u[0], (uint32_t)u[1], (uint32_t)u[2], (uint32_t)u[3], l0);
    tr4((uint32_t)u[4], (uint32_t)u[5], (uint32_t)u[6], (uint32_t)u[7], l1);
    tr4((uint32_t)(u[0] >> 32), (uint32_t)(u[1] >> 32), (uint32_t)(u[2] >> 32),
        (uint32_t)(u[3] >> 32), h0);
    tr4((uint32_t)(u[4] >> 32), (uint32_t)(u[5] >> 32), (uint32_t)(u[6] >> 32),
        (uint32_t)(u[7] >> 32), h1);
    uint2 d[8];
#pragma unroll
    for (int a = 0; a < 4; ++a)
        d[a] = make_uint2(l0[a] ^ 0x80808080u, l1[a] ^ 0x80808080u);
#pragma unroll
    for (int a = 0; a < 3; ++a)
        d[4 + a] = make_uint2(h0[a] ^ 0x80808080u, h1[a] ^ 0x80808080u);
    d[7] = make_uint2(h0[3], h1[3]);
    uint8_t *p = dst + (size_t)blockIdx.x * 8 * PLANE + pc.off;
    uint32_t m = (big ? 0x100u : 0u) | (sh << 16) | (code << 20);
#pragma unroll
    for (int a = 0; a < 8; ++a) {
        if (!WGT)   // every plane, without waiting for the mask
            *reinterpret_cast<uint2 *>(p + a * PLANE) = d[a];
        m |= (d[a].x | d[a].y) != 0 ? 1u << a : 0u;
    }
    m = wave_or(m);
    if ((tid & 63) == 0)
        red[tid >> 6] = m;
    __syncthreads();
    if constexpr (!WGT) {
        if (tid == 0)
            mask[(size_t)rt * nsteps + st] = red[0] | red[1] | red[2] | red[3];
        return;
    }
    m = (uint32_t)__builtin_amdgcn_readfirstlane((int)(red[0] | red[1] | red[2] | red[3]));
    if (tid == 0)
        mask[(size_t)rt * nsteps + st] = m;
    // W planes that k_gemm_i8p never reads are not written: those above the row
    // tile's top plane, and a plane without digits that lies three or more below
    // this block's top.  (Planes TOP - 2 .. TOP are read always, TOP of a run of
    // k-steps being at least each block's top and 2, lower ones where the mask
    // has their bit.)  Of N(0, 0.02) bfloat16 weights 3 planes in 8 are left,
    // which pays for k_tile_shift's pass over W.
    const int own = (m & 0xffu) ? 31 - __builtin_clz(m & 0xffu) : 0;
    const int hi = shifted ? max((int)(code >> 3), 2) : 7;
#pragma unroll
    for (int a = 0; a < 8; ++a)
        if (a <= hi && (((m >> a) & 1u) || own < a + 3))
            *reinterpret_cast<uint2 *>(p + a * PLANE) = d[a];
}

// One LDS stage of the planes path, NW row tiles of W: X planes 0..6, then W
// planes TOP - 2 .. TOP of each row tile, then plane TOP - 3 of each; whole slots
// of four 1 KB chunks, one per wave.
constexpr int PX_BYTES = 7 * PLANE;
constexpr int stage_slots(int nw) { return (14 + 8 * nw + 3) / 4; }
constexpr int stage_bytes(int nw) { return 4096 * stage_slots(nw); }

// s_waitcnt vmcnt(n) with the other counters left alone (gfx9 encoding)
template <int N>
__device__ __forceinline__ void wait_vm()
{
    static_assert(N >= 0 && N < 64, "vmcnt");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

// Workgroup barrier without the fence of __syncthreads (whose release waits
// for every DMA still in flight); the caller's s_waitcnt before it decides
// which DMA the barrier publishes.  The empty asm keeps LDS accesses on
// their side of it.
__device__ __forceinline__ void stage_barrier()
{
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// The k loop over a ring of four LDS stages.  Step i:
//   wait for step i + 1's DMA (this wave's), barrier (every wave's);
//   DMA step i + 3 into the stage step i - 1 used (each wave moves CPW 1 KB
//   chunks: 64 lanes x 16 bytes);
//   run the MFMAs of step i on the operands read during step i - 1, while
//   reading step i + 1's.
// The stages are four LDS objects named statically in each step (the loop
// is unrolled by four), so the compiler's own waits for the reads of one
// stage do not count the DMA into another.
//
// wsrc points at plane TOP - 2 of each row tile (wext at TOP - 3, where there is
// one), and digit sums are kept relative to TOP - 4, which may be below plane
// 0: acc[j][r] is the sum of weight 256^(TOP - 4 + r), so one code
// serves every window.  A step multiplies X planes 0..6 by W planes TOP - 2
// .. TOP, 21 NW MFMAs, and by plane TOP - 3 only for a row tile that holds a
// digit there (7 more; the shift of k_planes makes that about one step in ten
// for bfloat16 weights).  ext (LDS) tells, a byte for each loop step, zero past
// the last: bit n row tile n's plane TOP - 3, bit 2 + n its plane TOP - 4.  The
// chunks of plane TOP - 3 are moved only then: otherwise their slots re-read a
// fixed line set that stays in the vector cache, so that every step issues the
// same number of DMAs with no branch around one, which would make the compiler
// wait for all of them.  Plane TOP - 4 (one step in thousands) is loaded where
// it is needed.
// acc[n][r] += A B.  The digit sums of two row tiles take 352 registers, more
// than the 256 accumulation registers the compiler keeps MFMA results in, so
// with NW = 2 the instruction is written out with the register file chosen per
// sum: the first row tile's and sums 0..3 of the second in accumulation
// registers, the rest in vector registers.  s_nop 1: the wait states a vector
// write of an operand needs before an MFMA reads it (the compiler inserts
// them only for instructions it knows).
template <bool AG>
__device__ __forceinline__ void mfma_asm(v16i &c, const v4i &a, const v4i &b)
{
    if constexpr (AG)
        asm("s_nop 1\n\tv_mfma_i32_32x32x32_i8 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
    else
        asm("s_nop 1\n\tv_mfma_i32_32x32x32_i8 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
template <int NW>
__device__ __forceinline__ void mfma_i8(v16i (&acc)[NW][11], int n, int r, const v4i &a,
                                        const v4i &b)
{
    if constexpr (NW == 1)
        acc[n][r] = __builtin_amdgcn_mfma_i32_32x32x32_i8(a, b, acc[n][r], 0, 0, 0);
    else if (n == 0 || r < 4)   // constants once unrolled
        mfma_asm<true>(acc[n][r], a, b);
    else
        mfma_asm<false>(acc[n][r], a, b);
}
// An MFMA's result may be touched by other vector instructions only after its
// passes: 12 wait states here, which the compiler keeps itself after the
// instructions it knows, but not after mfma_asm.  Nothing in the source touches
// a sum between the MFMAs, but the register allocator may put copies of sums
// at the joins of the control flow; so the waits end every path that leaves
// mfma_asm behind: the conditional MFMAs of a step, each group of four steps,
// and the loop (mfma_settle).  Inside a group the steps follow each other
// without one (12 states are about 50 cycles, the step's 42 MFMAs 1350): that no
// path of the built code touches a sum too early is checked there, by
// tests/test_device_code.py.
template <int NW>
__device__ __forceinline__ void mfma_wait()
{
    if constexpr (NW > 1) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 11");
        __builtin_amdgcn_sched_barrier(0);
    }
}
// The sums after the k loop, what reads them depending on this (mad_shl_asm is
// as unknown to the compiler as mfma_asm).
template <int NW>
__device__ __forceinline__ void mfma_settle(v16i (&acc)[NW][11])
{
    asm volatile("s_nop 15\n\ts_nop 15"
                 : "+a"(acc[0][0]), "+a"(acc[0][1]), "+a"(acc[0][2]), "+a"(acc[0][3]),
                   "+a"(acc[0][4]), "+a"(acc[0][5]), "+a"(acc[0][6]), "+a"(acc[0][7]),
                   "+a"(acc[0][8]), "+a"(acc[0][9]), "+a"(acc[0][10]));
    if constexpr (NW > 1)
        asm volatile(""
                     : "+a"(acc[1][0]), "+a"(acc[1][1]), "+a"(acc[1][2]), "+a"(acc[1][3]),
                       "+v"(acc[1][4]), "+v"(acc[1][5]), "+v"(acc[1][6]), "+v"(acc[1][7]),
                       "+v"(acc[1][8]), "+v"(acc[1][9]), "+v"(acc[1][10]));
}

// The X chunks of slots 0 .. XSLOTS - 1 (which hold no W) of the loop's steps
// 0..2, before the masks are known.
constexpr int XSLOTS = 3;   // chunks 0 .. 11 of 14
template <int PS>
__device__ __forceinline__ void planes_first_x(uint8_t (&s0)[PS], uint8_t (&s1)[PS],
                                               uint8_t (&s2)[PS], const uint8_t *xsrc, int ns,
                                               int xz, bool rev)
{
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    auto one = [&](int s, uint8_t(&dst)[PS]) {
        const uint32_t at = (uint32_t)(s < ns ? (rev ? ns - 1 - s : s) : xz) * (8u * PLANE);
#pragma unroll
        for (int j = 0; j < XSLOTS; ++j) {
            const int c = w + 4 * j;
            __builtin_amdgcn_global_load_lds(xsrc + c * 1024 + (at + (uint32_t)lane * 16u),
                                             dst + c * 1024, 16, 0, 0);
        }
    };
    one(0, s0);
    one(1, s1);
    one(2, s2);
}

template <int NW>
__device__ __forceinline__ void planes_pass(uint8_t (&s0)[stage_bytes(NW)],
                                            uint8_t (&s1)[stage_bytes(NW)],
                                            uint8_t (&s2)[stage_bytes(NW)],
                                            uint8_t (&s3)[stage_bytes(NW)],
                                            const uint8_t *ext, const uint8_t *xsrc,
                                            const uint8_t *const (&wsrc)[NW],
                                            const uint8_t *const (&wext)[NW],
                                            const bool (&has5)[NW], int ns, int xz,
                                            bool rev, v16i (&acc)[NW][11])
{
    constexpr int PSTAGE = stage_bytes(NW);
    constexpr int DENSE = 14 + 6 * NW;                 // chunks every step moves
    constexpr int ALL = DENSE + 2 * NW;                // and the conditional ones
    constexpr int CPW = stage_slots(NW);
    constexpr int XB = PX_BYTES + 3 * NW * PLANE;      // plane TOP - 3
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6), wt = w >> 1, wn = w & 1;
    const int off = opnd_off(lane);
    // this wave's slot j moves chunk w + 4 j: its source in the first k-step (a
    // scalar address; the k-step's offset is one vector addition a step), and
    // the ext bit it needs (0: none; 16: past the last chunk)
    const uint8_t *base[CPW];
    uint32_t need[CPW];
#pragma unroll
    for (int j = 0; j < CPW; ++j) {
        const int c = w + 4 * j, d = c - 14, x = c - DENSE;
        const uint8_t *wd = NW > 1 && d >= 6 ? wsrc[NW - 1] : wsrc[0];
        const uint8_t *wx = NW > 1 && x >= 2 ? wext[NW - 1] : wext[0];
        need[j] = c < DENSE ? 0u : c < ALL ? 1u << (x >> 1) : 16u;
        base[j] = c < 14 ? xsrc + c * 1024
                  : c < DENSE ? wd + (NW > 1 && d >= 6 ? d - 6 : d) * 1024
                  : c < ALL ? wx + (x & 1) * 1024 : xsrc;
    }
    // plane TOP - 4, and TOP - 2 where there is none
    const uint8_t *wlow[NW];
#pragma unroll
    for (int n = 0; n < NW; ++n)
        wlow[n] = (has5[n] ? wsrc[n] - 2 * PLANE : wsrc[n]) + wn * SLICE + off;
    // Step s of the loop is k-step rev ? ns - 1 - s : s of the block's range.
    // The loop runs whole groups of four: steps past the last take the zero X
    // planes that follow the row tile's (k-step xz), with the last k-step of W.
    // A conditional slot that is not needed moves its own first k-step.
    struct Src {
        uint32_t x, w;   // byte offsets of a step's X and W planes
    };
    auto src_of = [&](int s) {
        const int c = min(s, ns - 1), k = rev ? ns - 1 - c : c;
        return Src{(uint32_t)(s < ns ? k : xz) * (8u * PLANE), (uint32_t)k * (8u * PLANE)};
    };
    const uint32_t lane16 = (uint32_t)lane * 16u;
    auto dma1 = [&](int j, Src f, uint32_t e, uint8_t(&dst)[PSTAGE]) {
        const int c = w + 4 * j;
        uint32_t at = 4 * j + 3 < 14 ? f.x : 4 * j >= 14 ? f.w : c < 14 ? f.x : f.w;
        if (4 * j + 3 >= DENSE)
            at = need[j] == 0 || (need[j] & e) != 0 ? at : 0u;
        __builtin_amdgcn_global_load_lds(base[j] + (at + lane16), dst + c * 1024, 16, 0, 0);
    };
    auto dma = [&](int s, uint32_t e, uint8_t(&dst)[PSTAGE]) {   // all but the first X slots
#pragma unroll
        for (int j = XSLOTS; j < CPW; ++j)
            dma1(j, src_of(s), e, dst);
    };
    // The operands of a step: X planes (A), and the dense W planes and TOP - 3
    // of each row tile (B).  They are read one step ahead, one LDS read per
    // MFMA or two from the step's start, so the reads finish under the MFMAs.
    struct Opnd {
        v4i A[7], B[NW][3], E[NW];
    };
    auto rdA = [&](const uint8_t(&src)[PSTAGE], int a) {
        return *reinterpret_cast<const v4i *>(src + wt * SLICE + a * PLANE + off);
    };
    auto rdB = [&](const uint8_t(&src)[PSTAGE], int k) {   // k = 3 n + j
        return *reinterpret_cast<const v4i *>(src + PX_BYTES + k * PLANE + wn * SLICE + off);
    };
    auto rdX = [&](const uint8_t(&src)[PSTAGE], int n) {
        return *reinterpret_cast<const v4i *>(src + XB + n * PLANE + wn * SLICE + off);
    };
    auto rd = [&](const uint8_t(&src)[PSTAGE], Opnd &o) {
#pragma unroll
        for (int a = 0; a < 7; ++a)
            o.A[a] = rdA(src, a);
#pragma unroll
        for (int n = 0; n < NW; ++n) {
#pragma unroll
            for (int j = 0; j < 3; ++j)
                o.B[n][j] = rdB(src, 3 * n + j);
            o.E[n] = rdX(src, n);
        }
    };
    // Step i with operands o (e: its ext bits), leaving the next
    // step's operands, read from nxt, in the same registers as they come free:
    // A[a] is read again once plane a's MFMAs are issued.  Step i + 3's DMA into
    // ldst (el: its ext bits) goes out between the MFMAs too: one wave runs per
    // SIMD, so its address arithmetic ahead of the MFMAs leaves the matrix core
    // idle.  The order is fixed by scheduling barriers.
    auto step = [&](int i, uint32_t e, Opnd &o, const uint8_t(&nxt)[PSTAGE], uint32_t el,
                    uint8_t(&ldst)[PSTAGE]) {
        const Src f = src_of(i + 3);
        constexpr int EVERY = 21 * NW / CPW;
        if (e) {
#pragma unroll
            for (int n = 0; n < NW; ++n)
                if ((e >> n) & 1u)
#pragma unroll
                    for (int a = 0; a < 7; ++a)
                        mfma_i8(acc, n, a + 1, o.A[a], o.E[n]);
            if (e >> 2) {
                // in bounds for every tile, used by those whose bit is set; the
                // loads end in this branch, or the compiler waits for them, and
                // for the DMAs, on the way without them too
                v4i Bx[NW];
#pragma unroll
                for (int n = 0; n < NW; ++n)
                    Bx[n] = *reinterpret_cast<const v4i *>(wlow[n] + src_of(i).w);
#pragma unroll
                for (int n = 0; n < NW; ++n)
                    asm volatile("" : "+v"(Bx[n]));
#pragma unroll
                for (int n = 0; n < NW; ++n)
                    if ((e >> (2 + n)) & 1u)
#pragma unroll
                        for (int a = 0; a < 7; ++a)
                            mfma_i8(acc, n, a, o.A[a], Bx[n]);
            }
            mfma_wait<NW>();
        }
        v4i nb[NW][3], a6;
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int a = 0; a < 7; ++a) {
#pragma unroll
            for (int j = 0; j < 3; ++j)
#pragma unroll
                for (int n = 0; n < NW; ++n) {
                    const int m = (a * 3 + j) * NW + n;   // MFMA of the step
                    mfma_i8(acc, n, a + 2 + j, o.A[a], o.B[n][j]);
                    // a read or two under the MFMAs of a plane, the last one
                    // (A[5]) six MFMAs or three from the step's end
                    if (j == 0 && n == 0) {
                        if (a < 3 * NW)
                            nb[a / 3][a % 3] = rdB(nxt, a);
                        if (a > 0)
                            o.A[a - 1] = rdA(nxt, a - 1);
                    }
                    if (j == 1 && n == 0) {
                        if (a < NW)
                            o.E[a] = rdX(nxt, a);
                        if (a == 5)
                            a6 = rdA(nxt, 6);
                    }
                    if (m % EVERY == EVERY / 2 && m / EVERY < CPW)
                        dma1(m / EVERY, f, el, ldst);
                    __builtin_amdgcn_sched_barrier(0);
                }
        }
        o.A[6] = a6;
#pragma unroll
        for (int n = 0; n < NW; ++n)
#pragma unroll
            for (int j = 0; j < 3; ++j)
                o.B[n][j] = nb[n][j];
    };
    // ext bits of loop steps i .. i + 3, from their bytes in a word
    auto ext4 = [&](uint32_t v, uint32_t &f0, uint32_t &f1, uint32_t &f2, uint32_t &f3) {
        const uint32_t f = (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
        f0 = f & 15u;
        f1 = (f >> 8) & 15u;
        f2 = (f >> 16) & 15u;
        f3 = f >> 24;
    };
    auto ext_word = [&](int i) { return *reinterpret_cast<const uint32_t *>(ext + i); };
    // prologue: steps 0..2 landed (their X chunks are in flight already), step 0
    // read.  e0..e3: ext bits of the group's steps; en: the next group's word,
    // read a group ahead.
    uint32_t e0, e1, e2, e3;
    ext4(ext_word(0), e0, e1, e2, e3);
    uint32_t en = ext_word(4);
    dma(0, e0, s0);
    dma(1, e1, s1);
    dma(2, e2, s2);
    wait_vm<0>();
    stage_barrier();
    Opnd o;
    rd(s0, o);
    for (int i = 0; i < ns; i += 4) {
        uint32_t e4, e5, e6, e7;
        ext4(en, e4, e5, e6, e7);
        wait_vm<CPW>();
        stage_barrier();
        en = ext_word(i + 8);
        step(i, e0, o, s1, e3, s3);
        wait_vm<CPW>();
        stage_barrier();
        step(i + 1, e1, o, s2, e4, s0);
        wait_vm<CPW>();
        stage_barrier();
        step(i + 2, e2, o, s3, e5, s1);
        wait_vm<CPW>();
        stage_barrier();
        step(i + 3, e3, o, s0, e6, s2);
        e0 = e4;
        e1 = e5;
        e2 = e6;
        e3 = e7;
        mfma_wait<NW>();   // the next group's first wait and barrier follow anyway
    }
    wait_vm<0>();   // no DMA in flight when the block gives its LDS back
}

// mad_shl as assembly, for the settled sums: the compiler's own form of it here
// spills in k_gemm_i8p<2>.
template <int S>
__device__ __forceinline__ int64_t mad_shl_asm(int a, int64_t c)
{
    int64_t r;
    uint64_t cy;
    asm("v_mad_i64_i32 %0, %1, %2, %3, %4" : "=v"(r), "=s"(cy) : "v"(a), "s"(1 << S), "v"(c));
    return r;
}

// Register i of the 11 window digit sums as the 128-bit sum S = sum_r acc[r][i]
// 256^r (two words; |S| < 2^112): groups of four are exact int64 (|g| < 2^31
// (1 + 2^8 + 2^16 + 2^24) < 2^56), S = g0 + 2^32 g1 + 2^64 g2 with one carry.
__device__ __forceinline__ void win_sum128(const v16i (&acc)[11], int i, uint64_t &lo,
                                           uint64_t &hi)
{
    int64_t g[3];
#pragma unroll
    for (int j = 0; j < 3; ++j) {
        g[j] = mad_shl_asm<8>(acc[4 * j + 1][i], (int64_t)acc[4 * j][i]);
        g[j] = mad_shl_asm<16>(acc[4 * j + 2][i], g[j]);
        if (j < 2)
            g[j] = mad_shl_asm<24>(acc[4 * j + 3][i], g[j]);
    }
    lo = (uint64_t)g[0] + ((uint64_t)g[1] << 32);
    const uint64_t carry = lo < (uint64_t)g[0] ? 1u : 0u;
    hi = (uint64_t)(g[0] >> 63) + (uint64_t)(g[1] >> 32) + carry + (uint64_t)g[2];
}

// Words of the signed 128-bit (lo, hi), Z zero words put below it, from bit b
// (uniform, below 96) on, sign words above: word selects and funnel shifts.
template <int N, int Z>
__device__ __forceinline__ void words_from(uint64_t lo, uint64_t hi, int b, uint32_t (&o)[N])
{
    const uint32_t s = (uint32_t)((int64_t)hi >> 63);
    const uint32_t w[8] = {(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi,
                           (uint32_t)(hi >> 32), s, s, s, s};
    const int q = b >> 5;
    uint32_t a[N + 1];
#pragma unroll
    for (int k = 0; k <= N; ++k)
        a[k] = q == 0 ? (k < Z ? 0u : w[k - Z]) : q == 1 ? w[k + 1 - Z] : w[k + 2 - Z];
#pragma unroll
    for (int k = 0; k < N; ++k)
        o[k] = __builtin_amdgcn_alignbit(a[k + 1], a[k], b & 31);
}

// grid (ceil(ceil(N/64) / NW) * ceil(T/64), 1, S) over operands split by
// k_planes (nsteps k-steps): split z covers steps [z spb, (z + 1) spb), and a
// block NW row tiles of W.  The block ORs its tiles' masks over its steps; a
// row tile's TOP is its top plane (at least 2).  A row tile whose digits leave
// TOP - 4 .. TOP, and all of a block whose X digits reach plane 7 (or may
// overflow), are not written and have their redo flags set (the others'
// cleared; the flag of a 64 x 64 tile is that of its block in k_gemm_i8_full's
// numbering).  S == 1: Y gets the shifted
// result; S > 1: P[z][t][n] the int128 partial.  Row tiles whose planes are
// shifted (prepared weights) give sums 2^shift too large: exact multiples,
// shifted back.
//
// Two row tiles (NW = 2) halve the X traffic and the barriers per product: a
// step moves 26 KB for 42 MFMAs a wave, where NW = 1 moves 20 KB for 21.
//
// What bounds it: the matrix cores at the clock their power allows.  A loop of
// nothing but these MFMAs on random digits runs at 3.1 to 3.5 POP/s (4.3-4.8 on
// zeros); 2048 x 11264 x 2048 takes 22 digit products per Q16.48 MAC here, 2.8
// POP/s over 735 us, with the matrix cores busy two thirds of the time at 1.75
// GHz.  With a four-plane window always multiplied (28 products), the DMA ahead
// of the MFMAs and a 64-bit vector address per chunk the call took 931 us.
template <int NW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void
k_gemm_i8p(int64_t *__restrict__ Y, uint64_t *__restrict__ P, int *__restrict__ redo,
           const uint8_t *__restrict__ Xp, const uint32_t *__restrict__ Xm,
           const uint8_t *__restrict__ Wp, const uint32_t *__restrict__ Wm, int T, int N,
           int nsteps, int spb, int cpx)
{
    constexpr int PSTAGE = stage_bytes(NW);
    __shared__ __align__(16) uint8_t st0[PSTAGE];
    __shared__ __align__(16) uint8_t st1[PSTAGE];
    __shared__ __align__(16) uint8_t st2[PSTAGE];
    __shared__ __align__(16) uint8_t st3[PSTAGE];
    __shared__ uint32_t red[1 + NW][4];
    // a byte per loop step, and the groups' words a group ahead
    constexpr int EXT_BYTES = 512;
    static_assert(MAXK_RUN / MK <= 510 && 256 * 2 == EXT_BYTES, "two steps a thread");
    __shared__ __align__(4) uint8_t ext[EXT_BYTES + 12];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int nn = (N + MN - 1) / MN, nt = (T + MT - 1) / MT;
    int n_blk, t_tile;
    tile_of(blockIdx.x, (nn + NW - 1) / NW, nt, n_blk, t_tile);
    // a split past the last k-step is empty, at nsteps
    const int s0 = min((int)blockIdx.z * spb, nsteps), ns = min(nsteps, s0 + spb) - s0;
    int n_tile[NW];   // past the last row tile: that one again, not stored
#pragma unroll
    for (int j = 0; j < NW; ++j)
        n_tile[j] = min(NW * n_blk + j, nn - 1);
    // Blocks run in rounds of one per compute unit; each XCD's round holds 8
    // row blocks x 4 token tiles (tile_of), and the next round's blocks take
    // the same row blocks with the next token tiles.  Odd rounds walk k
    // downwards, so they start on the W planes the round before ended on,
    // which are still in L2.
    const bool rev = ((((int)blockIdx.x >> 3) / cpx) & 1) != 0;
    // the masks of loop steps tid and tid + 256 (ns <= 510)
    uint32_t mx = 0, mw[NW] = {}, wk[2][NW];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = tid + 256 * u, k = s0 + (rev ? ns - 1 - i : i);
#pragma unroll
        for (int j = 0; j < NW; ++j)
            wk[u][j] = i < ns ? Wm[(size_t)n_tile[j] * nsteps + k] & 0xffffu : 0u;
        mx |= i < ns ? Xm[(size_t)t_tile * nsteps + k] : 0u;
    }
    const uint8_t *xsrc = Xp + ((size_t)t_tile * (nsteps + 1) + s0) * 8 * PLANE;
    planes_first_x(st0, st1, st2, xsrc, ns, nsteps - s0, rev);
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int j = 0; j < NW; ++j)
            mw[j] |= wk[u][j];
    mx = wave_or(mx);
#pragma unroll
    for (int j = 0; j < NW; ++j)
        mw[j] = wave_or(mw[j]);
    if (lane == 0) {
        red[0][w] = mx;
#pragma unroll
        for (int j = 0; j < NW; ++j)
            red[1 + j][w] = mw[j];
    }
    __syncthreads();
    auto block_or = [&](int i) {
        return (uint32_t)__builtin_amdgcn_readfirstlane(
            (int)(red[i][0] | red[i][1] | red[i][2] | red[i][3]));
    };
    mx = block_or(0);
    // Every row tile has its own window: with one for both, two of different
    // magnitude would both be redone (1024 x 4096 x 2048 with every other row
    // tile's weights 2^-24 of the rest: 430 us, now 204; equal ones 143)
    int low[NW];   // TOP - 4: -2 .. 3
    bool fit[NW], any = false;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        mw[j] = block_or(1 + j);
        low[j] = max((mw[j] & 0xffu) ? 31 - __builtin_clz(mw[j] & 0xffu) : 0, 2) - 4;
        fit[j] = (mx & ~0x7fu) == 0 && mw[j] < 0x100u &&
                 (mw[j] & ((1u << max(low[j], 0)) - 1u)) == 0;
        any = any || fit[j];
        if (tid == 0 && NW * n_blk + j < nn)
            redo[blockIdx.z * nn * nt + (NW == 1 ? (int)blockIdx.x
                                                 : block_of(NW * n_blk + j, t_tile, nn, nt))] =
                fit[j] ? 0 : 1;
    }
    if (!any) {
        wait_vm<0>();   // no DMA in flight when the block gives its LDS back
        return;         // uniform over the block
    }

    v16i acc[NW][11];
#pragma unroll
    for (int j = 0; j < NW; ++j)
#pragma unroll
        for (int d = 0; d < 11; ++d)
            acc[j][d] = (v16i){0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    const uint8_t *wsrc[NW], *wext[NW];
    bool has5[NW];
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        wsrc[j] = Wp + ((size_t)n_tile[j] * nsteps + s0) * 8 * PLANE + (low[j] + 2) * PLANE;
        wext[j] = wsrc[j] - (low[j] > -2 ? PLANE : 0);
        has5[j] = low[j] >= 0;
    }
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        const int i = tid + 256 * u;
        uint32_t b = 0;
#pragma unroll
        for (int j = 0; j < NW; ++j) {
            const uint32_t m = fit[j] ? (wk[u][j] << 2) >> (low[j] + 2) : 0u;   // from TOP - 4
            b |= ((m >> 1) & 1u) << j | (m & 1u) << (2 + j);
        }
        if (i < EXT_BYTES)
            ext[i] = (uint8_t)b;
    }
    if (tid < 3)   // the words read a group ahead, past the last step
        reinterpret_cast<uint32_t *>(ext + EXT_BYTES)[tid] = 0;
    __syncthreads();
    if (ns > 0)   // an empty split has its X slots' zeros in flight: waited for below
        planes_pass<NW>(st0, st1, st2, st3, ext, xsrc, wsrc, wext, has5, ns, nsteps - s0, rev,
                        acc);
    else
        wait_vm<0>();
    mfma_settle<NW>(acc);
    // lane l, register i: token 8 (i / 4) + 4 (l / 32) + i % 4, row l % 32
    const int wt = w >> 1, wn = w & 1;
#pragma unroll
    for (int j = 0; j < NW; ++j) {
        if (!fit[j])
            continue;
        const int n = (NW * n_blk + j) * MN + 32 * wn + (lane & 31);
        const int t0 = t_tile * MT + 32 * wt + 4 * (lane >> 5);
        const int wsh = (int)((Wm[(size_t)n_tile[j] * nsteps] >> 16) & 7u);
        // bits b .. b + 63 of the sum are bits 48 .. 111 of the result's
        const int b = 48 + wsh - 8 * low[j];   // 24 .. 71
        if (gridDim.z == 1) {
            int64_t y[16];
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                uint64_t lo, hi;
                win_sum128(acc[j], i, lo, hi);
                uint32_t o[2];
                words_from<2, 0>(lo, hi, b, o);
                y[i] = (int64_t)(((uint64_t)o[1] << 32) | o[0]);
            }
            int64_t *p = Y + (size_t)t0 * N + n;
            if ((t_tile + 1) * MT <= T && (NW * n_blk + j + 1) * MN <= N) {   // whole tile
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    p[(size_t)(8 * (i >> 2) + (i & 3)) * N] = y[i];
            } else if (n < N) {
#pragma unroll
                for (int i = 0; i < 16; ++i)
                    if (t0 + 8 * (i >> 2) + (i & 3) < T)
                        p[(size_t)(8 * (i >> 2) + (i & 3)) * N] = y[i];
            }
        } else if (n < N) {
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int t = t0 + 8 * (i >> 2) + (i & 3);
                if (t >= T)
                    continue;
                uint64_t lo, hi;
                win_sum128(acc[j], i, lo, hi);
                uint32_t u[4];
                words_from<4, 1>(lo, hi, b - 16, u);   // from a zero word on: 8 .. 55
                uint64_t *p = P + 2 * (((size_t)blockIdx.z * T + t) * N + n);
                *reinterpret_cast<uint4 *>(p) = make_uint4(u[0], u[1], u[2], u[3]);
            }
        }
    }
}

} // namespace

int q48_gemm_auto_kernel(int T, int N, int K)
{
    // measured on MI355X: the int8 kernel is 7-30x faster than the VALU
    // kernel at every T >= 16 of the TinyLlama shapes
    (void)T;
    (void)N;
    (void)K;
    return Q48_GEMM_I8;
}

// K splits by an estimate of the time (ns): rounds of blocks over the compute
// units, each a block's k-steps (0.6 us from planes, 1.3 with the split inside
// the loop) and its 5 us of prologue and epilogue, then for S > 1 the
// reduction's launch and its traffic (32 bytes an output and split at about
// 4.5 TB/s).  Doubling S while the grid was under one block per unit gave two
// rounds, the second nearly empty, where the tiles divide badly: 128 tokens x
// 2560 x 2048 took 320 blocks at S = 4, 52.8 us (38.7 prepared), and takes 240 at S
// = 3, 38.7 us (30.5).
static int i8_splits(int T, int N, int K, int cu_count, bool planes, int64_t *ns = nullptr)
{
    const int64_t base = (int64_t)((N + MN - 1) / MN) * ((T + MT - 1) / MT);
    const int steps = (K + MK - 1) / MK;
    const int min_s = (steps + MAXK_RUN / MK - 1) / (MAXK_RUN / MK);
    const int64_t step = planes ? 600 : 1300;
    int best = min_s;
    int64_t cost = INT64_MAX;
    // 256 x 2048: 16 splits 2-4% faster than 8 to 32 tokens, 2-4% slower from 96
    const int few = T <= 32 ? 4 : 8;
    for (int s = min_s; s <= min_s + 63 && (s == min_s || steps / s >= few); ++s) {
        const int64_t rounds = (base * s + cu_count - 1) / cu_count;
        const int64_t t = rounds * ((steps + s - 1) / s * step + 5000) +
                          (s > 1 ? 4500 + 32ll * s * T * N / 4500 : 0);
        if (t < cost) {
            cost = t;
            best = s;
        }
    }
    if (ns)
        *ns = cost;
    return best;
}

// Whether splitting both operands into planes first pays for weights that are
// not prepared, by the estimate above: the planes' k-steps are shorter, and
// two launches (5.5 us) and 16 bytes a value at 5 TB/s come before them.
// Measured (us, split in the loop / planes): 96 tokens x 11264 x 2048 120 /
// 126, 128 x 2560 x 2048 37 / 42, 256 x 1024 x 1024 22 / 28, 2048 x 256 x 2048
// 45 / 45; 160 x 11264 x 2048 197 / 163, 192 x 5632 x 2048 116 / 89, 256 x
// 2560 x 2048 65 / 51, 2048 x 512 x 2048 69 / 57, 2048 x 11264 x 2048 1433 /
// 820.  Over 150 shapes (64 to 2048 tokens, N 128 to 11264, K 256 to 5632) the choice
// costs 0.25% on average and 10% at most over the better one; at least 256
// tokens and N >= 1024, the line before, 2.5% and 30%.
static bool planes_pay(int T, int N, int K, int cu_count)
{
    int64_t fused, planes;
    i8_splits(T, N, K, cu_count, false, &fused);
    i8_splits(T, N, K, cu_count, true, &planes);
    return planes + 5500 + 16ll * ((int64_t)T + N) * K / 5000 < fused;
}

size_t q48_gemm_planes_size(int N, int K)
{
    const size_t tiles = (size_t)((N + MN - 1) / MN) * ((K + MK - 1) / MK);
    return tiles * 8 * PLANE + ((tiles * 4 + 255) & ~(size_t)255);
}

int q48_launch_gemm_prepare(q48_ctx *c, void *Wp, const int64_t *W, int N, int K)
{
    const int steps = (K + MK - 1) / MK, nn = (N + MN - 1) / MN;
    if ((size_t)nn * steps > 0x7fffffff)
        return Q48_EINVAL;
    uint8_t *p = (uint8_t *)Wp;
    uint32_t *m = (uint32_t *)(p + (size_t)nn * steps * 8 * PLANE);
    hipLaunchKernelGGL(k_tile_shift, dim3(nn, tile_parts(K, steps)), dim3(1024), 0, c->stream, m,
                       W, N, K, steps);
    hipLaunchKernelGGL(k_planes<true>, dim3(nn * steps), dim3(256), 0, c->stream, p, m, W, N, K,
                       steps, 1);
    return (int)hipGetLastError();
}

int q48_launch_gemm_i8(q48_ctx *c, int64_t *Y, const int64_t *W, const int64_t *X, int T,
                       int N, int K, int kernel, const void *Wpre)
{
    const int steps = (K + MK - 1) / MK;
    const int nt = (T + MT - 1) / MT, nn = (N + MN - 1) / MN, nb = nn * nt;
    // with W prepared, planes win from 2 tokens on: the GEMM streams W then, and
    // 3 to 4 planes hold a value's 8 bytes
    const bool fits = (size_t)max(nt, nn) * (steps + 1) <= 0x7fffffff;
    const bool choose =
        fits && !Wpre && kernel != Q48_GEMM_I8_PLANES && kernel != Q48_GEMM_I8_FUSED;
    bool planes = fits && (kernel == Q48_GEMM_I8_PLANES ||
                           (kernel != Q48_GEMM_I8_FUSED && Wpre && T >= 2 && N >= 1024) ||
                           (choose && planes_pay(T, N, K, c->cu_count)));
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    int S, spb, rc;
    size_t flags, part, xpl, wpl, xms;
    for (bool again = false;; again = true) {
        S = i8_splits(T, N, K, c->cu_count, planes);
        spb = (steps + S - 1) / S;
        // planes_pass reaches a row tile's zero X planes by a 32-bit offset from
        // the split's start.  Where that can pass 4 GB only the last split, which
        // they follow directly, may need them: whole groups of four steps elsewhere
        if (planes && (size_t)steps * 8 * PLANE > 0xffffffffu) {
            spb = min((spb + 3) & ~3, MAXK_RUN / MK & ~3);
            S = (steps + spb - 1) / spb;
        }
        // workspace: the blocks' redo flags, (S > 1) the int128 partials, then
        // (planes path) X and W digit planes and their masks
        flags = al((size_t)nb * S * sizeof(int));
        part = S > 1 ? 16 * (size_t)S * T * N : 0;
        xpl = planes ? (size_t)nt * (steps + 1) * 8 * PLANE : 0;
        wpl = planes && !Wpre ? (size_t)nn * steps * 8 * PLANE : 0;
        xms = planes ? al((size_t)nt * steps * 4) : 0;
        const size_t wms = planes && !Wpre ? al((size_t)nn * steps * 4) : 0;
        // blocks (and their redo flags) are numbered in int
        rc = (size_t)nn * nt * S > 0x7fffffff
                 ? Q48_EINVAL
                 : q48_ws_reserve(c, flags + part + xpl + wpl + xms + wms);
        if (!rc)
            break;
        // no room for the chosen form (nor, in a capture, a way to make some):
        // the other one may fit
        if (!choose || again)
            return rc;
        planes = !planes;
    }
    char *ws = (char *)c->ws;
    int *redo = (int *)ws;
    uint64_t *P = S > 1 ? (uint64_t *)(ws + flags) : nullptr;
    const dim3 grid(nb, 1, S);
    const int fgrid = min(nb * S, c->cu_count);
    const bool vec = K % 2 == 0 && (((uintptr_t)W | (uintptr_t)X) & 15) == 0;
    if (planes) {
        uint8_t *Xp = (uint8_t *)(ws + flags + part), *Wp = Xp + xpl;
        uint32_t *Xm = (uint32_t *)(Wp + wpl), *Wm = (uint32_t *)((char *)Xm + xms);
        hipLaunchKernelGGL(k_planes<false>, dim3(nt * (steps + 1)), dim3(256), 0, c->stream, Xp,
                           Xm, X, T, K, steps, 0);
        if (Wpre) {
            // planes from q48_launch_gemm_prepare: masks after the planes
            Wp = (uint8_t *)Wpre;
            Wm = (uint32_t *)(Wp + (size_t)nn * steps * 8 * PLANE);
        } else {
            hipLaunchKernelGGL(k_planes<true>, dim3(nn * steps), dim3(256), 0, c->stream, Wp, Wm,
                               W, N, K, steps, 0);
        }
        // one or two row tiles a block, by rounds of blocks over the compute
        // units: a block of two takes 1.78 to 1.87 times one of one (2048 x 11264
        // x 2048: 22 rounds in 794 us, 11 in 740), so two win from 11 rounds
        // against 6 on (us, one / two: 11 and 6 rounds 396 / 385, 17 and 9 592 /
        // 572, 19 and 10 672 / 643), and lose where the last round is emptier
        // (7 and 4 252 / 255, 3 and 2 123 / 136).  Split K keeps one: its runs
        // are short, and the part that fills the device is what it is for (128
        // tokens x 2560 x 2048: 39.0 against 41.6 us).
        const int cu = c->cu_count, cpx = max(1, cu / 8), nb2 = (nn + 1) / 2 * nt;
        const int rounds1 = (nb + cu - 1) / cu, rounds2 = (nb2 + cu - 1) / cu;
        if (S == 1 && 11 * rounds2 <= 6 * rounds1)
            hipLaunchKernelGGL(k_gemm_i8p<2>, dim3(nb2, 1, 1), dim3(256), 0, c->stream, Y, P,
                               redo, Xp, Xm, Wp, Wm, T, N, steps, spb, cpx);
        else
            hipLaunchKernelGGL(k_gemm_i8p<1>, grid, dim3(256), 0, c->stream, Y, P, redo, Xp, Xm,
                               Wp, Wm, T, N, steps, spb, cpx);
    } else if (vec) {
        hipLaunchKernelGGL((k_gemm_i8<true>), grid, dim3(256), 0, c->stream, Y, P, redo, W, X, T,
                           N, K, spb);
    } else {
        hipLaunchKernelGGL((k_gemm_i8<false>), grid, dim3(256), 0, c->stream, Y, P, redo, W, X,
                           T, N, K, spb);
    }
    if (vec)
        hipLaunchKernelGGL((k_gemm_i8_full<true>), dim3(fgrid), dim3(256), 0, c->stream, Y, P,
                           redo, W, X, T, N, K, spb, nb, S);
    else
        hipLaunchKernelGGL((k_gemm_i8_full<false>), dim3(fgrid), dim3(256), 0, c->stream, Y, P,
                           redo, W, X, T, N, K, spb, nb, S);
    if (S > 1) {
        const size_t tn = (size_t)T * N;
        hipLaunchKernelGGL(k_gemm_i8_reduce, dim3((unsigned)((tn + 255) / 256)), dim3(256), 0,
                           c->stream, Y, P, T, N, S);
    }
    return (int)hipGetLastError();
}
