// q48_pfattn.hip — causal attention of a batched prefill on the int8 matrix
// cores: T query rows at positions p0 .. p0 + T - 1, row t over the cache rows
// 0 .. p0 + t, each row bit-identical to the reference's exact attention path
// at its position (llama_int.c:1502-1529 with softmax, 1060-1072).
//
// Scores.  s_j = fp_mul((sum_d q_d k_j,d) >> 48, scale): the int128 dot
//   product from the digit identity over d (q48_digits.hpp), 63
//   v_mfma_i32_16x16x64_i8 per 16 x 16 tile and 64 dims.
// Weights.  The softmax on the VALU: exact maximum, fp_safe_exp of the
//   wrapped difference, wrapping sum, fp_div when the sum is positive.
// Values.  o_d = sum_j fp_mul(p_j, v_j,d) truncates every product: one FP64
//   operation per (row, position, dim), rounding down (q48_fsum4x4), for
//   values in [-2^51, 2^51).  A block whose span holds a larger value splits
//   v = v1 + 2^48 v2 (v1 = v mod 2^48) and the weight p = pa + 2^24 pb, and
//   makes three such sums, o = sum floor(p v1 / 2^48) + sum pa v2 + 2^24 sum
//   pb v2, the last two exact integers below 2^51; one whose weights are not
//   a plain softmax (wrapped score differences) multiplies in integers.
//
// A block owns 16 consecutive query rows of one head.  k_pfa_prep first
// writes the layer's keys and values as digit planes once per KV head; the
// scores go to a workspace region of the block (16 rows x its position span)
// and are overwritten by the exponentials.
#include "q48_digits.hpp"

namespace {

constexpr int PF_ROWS = 16;   // query rows per block: one MFMA tile
constexpr int PF_STEP = 64;   // positions per value step: one MFMA depth

// Accumulation runs stay below 16320 positions: |digit-product sum| < 2^31.
constexpr int PF_MAX_POS = 16320;

__host__ __device__ inline int pf_round64(int x) { return (x + 63) & ~63; }

// positions the block of rows [16 tile, 16 tile + 16) reads, rounded up to 64
__host__ __device__ inline int pf_span(int tile, int p0, int T)
{
    const int end = PF_ROWS * (tile + 1) < T ? PF_ROWS * (tile + 1) : T;
    return pf_round64(p0 + end);
}

__device__ __forceinline__ int64_t row16_max64(int64_t v)
{
    int64_t o = (int64_t)q48_dpp64<Q48_DPP_XOR1>((uint64_t)v);
    v = o > v ? o : v;
    o = (int64_t)q48_dpp64<Q48_DPP_XOR2>((uint64_t)v);
    v = o > v ? o : v;
    o = (int64_t)q48_dpp64<Q48_DPP_HALF_MIRROR>((uint64_t)v);
    v = o > v ? o : v;
    o = (int64_t)q48_dpp64<Q48_DPP_MIRROR>((uint64_t)v);
    return o > v ? o : v;
}

__device__ __forceinline__ q48_u128 ld128(const uint64_t *p)
{
    return ((q48_u128)p[1] << 64) | p[0];
}

__device__ __forceinline__ void st128(uint64_t *p, q48_u128 v)
{
    p[0] = (uint64_t)v;
    p[1] = (uint64_t)(v >> 64);
}

// Digit planes of the layer's keys, and its values as doubles, at positions
// [64 c, 64 c + 64) of KV head kh (grid (Ppad / 64, n_kv)); keys at or past P
// read as C (all digits zero), values as 0:
//  KD[kh][a][j][HDP]   digit a of k_j,d (HDP: head_dim rounded up to 64, the
//                      pad dims zero digits)
//  CK[kh][j]           C sum_d k_j,d - hd C^2 (int128, low word first)
//  VF[kh][j][d]        v_j,d (where it is within [-2^51, 2^51))
//  VB[kh][c]           1 when some v of the 64 positions is outside [-2^51, 2^51)
template <int HD>
__global__ __launch_bounds__(256) void k_pfa_prep(uint8_t *__restrict__ KD,
                                                 uint64_t *__restrict__ CK,
                                                 double *__restrict__ VF,
                                                 int *__restrict__ VB,
                                                 const int64_t *__restrict__ kcache,
                                                 const int64_t *__restrict__ vcache, int layer,
                                                 int P, int Ppad, int n_kv, int max_seq)
{
    constexpr int HDP = HD < 64 ? 64 : HD;
    const int c = blockIdx.x, kh = blockIdx.y, tid = threadIdx.x, j0 = PF_STEP * c;
    const size_t kvd = (size_t)n_kv * HD;
    const int64_t *kb = kcache + (size_t)layer * max_seq * kvd + (size_t)kh * HD;
    const int64_t *vb = vcache + (size_t)layer * max_seq * kvd + (size_t)kh * HD;
    uint8_t *kd = KD + (size_t)kh * 8 * Ppad * HDP;

    // keys: (position, 4 dims) per item
    for (int it = tid; it < PF_STEP * (HDP / 4); it += 256) {
        const int j = j0 + it / (HDP / 4), d = 4 * (it % (HDP / 4));
        uint64_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e)
            v[e] = (j < P && d + e < HD) ? (uint64_t)kb[(size_t)j * kvd + d + e] : kDig;
        uint32_t w[8];
        digits4(v, w);
#pragma unroll
        for (int a = 0; a < 8; ++a)
            *reinterpret_cast<uint32_t *>(kd + ((size_t)a * Ppad + j) * HDP + d) = w[a];
    }
    uint32_t big = 0;
#pragma unroll 4
    for (int it = tid; it < PF_STEP * HD; it += 256) {
        const int j = j0 + it / HD, d = it % HD;
        const int64_t v = j < P ? vb[(size_t)j * kvd + d] : 0;
        VF[((size_t)kh * Ppad + j) * HD + d] = q48_f51(v, big);
    }
    const int any = __syncthreads_or(q48_f51_big(big));
    if (tid == 0)
        VB[(size_t)kh * (Ppad / PF_STEP) + c] = any ? 1 : 0;
    if (tid < PF_STEP) {
        const int j = j0 + tid;
        q48_u128 s = 0;
        if (j < P) {
            for (int d = 0; d < HD; ++d)
                s += (q48_u128)(q48_i128)kb[(size_t)j * kvd + d];
            s = s * kDig - (q48_u128)kDig * kDig * (q48_u128)HD;
        }
        st128(CK + 2 * ((size_t)kh * Ppad + j), s);
    }
}

// Attention of 16 query rows of one head.  Blocks go round-robin to the 8
// XCDs; when n_kv divides 8, XCD x takes KV head x % n_kv only, so each L2
// holds the digit planes of one KV head.  Within an XCD the longest row
// blocks (the last rows) start first.
//  phase 1: scores by MFMA (wave w: position tiles w, w + 4, ...), written to
//           the block's workspace rows, and the row maxima;
//  phase 2: exponentials in place and the row sums;
//  phase 3: wave w takes the 16-position chunks w, w + 4, ... by itself, with
//           no barrier: the weights of its 16 rows (fp_div, four a lane) go
//           through LDS so that lane l of each row of 16 lanes holds position
//           l % 16 of every query row, and row_newbcast hands them to the
//           lanes, which hold one dim each (head_dim 128: two; 32: 32
//           positions a chunk, 16 for each half of the wave) of the chunk's
//           values and the sums of all 16 rows: 256 FP64 operations a chunk
//           on 16 value loads and 16 LDS reads;
//  then the four waves' sums are added in LDS.
// TinyLlama heads, rows 0..1499: 1028 -> 474 us a launch against digit
// products of weights and values on the matrix cores with six integer
// operations per term for the truncations (and two barriers per 64
// positions); rows 512..1023: 390 -> 205 us.  158 VGPRs (228) and 17 KB of
// LDS (59) let three blocks run on a compute unit (two).
template <int HD>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(HD == 128 ? 1 : 2))) void
k_pfa(int64_t *__restrict__ out, const int64_t *__restrict__ QKV,
      const uint8_t *__restrict__ KD, const uint64_t *__restrict__ CK,
      const double *__restrict__ VF, const int *__restrict__ VB,
      const int64_t *__restrict__ vcache, int64_t *__restrict__ SCR,
      const int64_t *__restrict__ scale_p, int p0, int T, int n_heads, int n_kv, int Ppad,
      size_t per_head)
{
    q48_round_down();
    constexpr int HDP = HD < 64 ? 64 : HD, KS = HDP / 64;
    constexpr int DL = HD == 128 ? 2 : 1;          // dims per lane
    constexpr int PG = HD == 32 ? 2 : 1;           // 16-position groups per chunk
    constexpr int CP = 16 * PG;                    // positions per chunk
    __shared__ double pw[4][PF_ROWS][CP];          // a wave's weights of a chunk
    __shared__ uint64_t lam[PF_ROWS][HD];          // the sums
    __shared__ q48_u128 cq[PF_ROWS];
    __shared__ int64_t mxs[4][PF_ROWS], sums[PF_ROWS];
    __shared__ int form;                           // see phase 3

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int rl = lane & 15, kq = lane >> 4;
    const int G = n_heads / n_kv, nt = (T + PF_ROWS - 1) / PF_ROWS;
    int tile, h;
    if (8 % n_kv == 0) {
        const int x = (int)blockIdx.x & 7, item = ((int)blockIdx.x >> 3) * (8 / n_kv) + x / n_kv;
        if (item >= G * nt)
            return;   // uniform over the block
        tile = nt - 1 - item / G;
        h = (x % n_kv) * G + item % G;
    } else {
        if ((int)blockIdx.x >= n_heads * nt)
            return;
        tile = nt - 1 - (int)blockIdx.x / n_heads;
        h = (int)blockIdx.x % n_heads;
    }
    const int kh = h / G;
    const int t0 = PF_ROWS * tile, nrow = min(PF_ROWS, T - t0);
    const int J = pf_span(tile, p0, T);
    size_t off = 0;
    for (int i = 0; i < tile; ++i)
        off += (size_t)pf_span(i, p0, T);
    int64_t *sc = SCR + (size_t)h * per_head + (size_t)PF_ROWS * off;   // [16][J]
    const int64_t scale = *scale_p;

    // query digits: lane (row rl, dims 64 ks + 16 kq .. + 15), the A operand
    v4i A[KS][8];
    {
        const int64_t *q = QKV + (size_t)min(t0 + rl, T - 1) * ((size_t)(n_heads + 2 * n_kv) * HD) +
                           (size_t)h * HD;
        q48_u128 qs = 0;
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) {
            const int d0 = 64 * ks + 16 * kq;
            uint64_t v[16];
            if (d0 < HD) {   // head_dim is a multiple of 16: all 16 dims real
                const ulonglong2 *q2 = reinterpret_cast<const ulonglong2 *>(q + d0);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const ulonglong2 u = q2[e];
                    v[2 * e] = u.x;
                    v[2 * e + 1] = u.y;
                }
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    qs += (q48_u128)(q48_i128)(int64_t)v[e];
            } else {
#pragma unroll
                for (int e = 0; e < 16; ++e)
                    v[e] = kDig;
            }
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const uint64_t v4[4] = {v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
                uint32_t wd[8];
                digits4(v4, wd);
#pragma unroll
                for (int a = 0; a < 8; ++a)
                    A[ks][a][g] = (int)wd[a];
            }
        }
        qs += shfl_xor128(qs, 16);
        qs += shfl_xor128(qs, 32);
        if (w == 0 && kq == 0)
            cq[rl] = qs * kDig;
    }
    if (tid == 0)
        form = 0;
    for (int i = tid; i < PF_ROWS * HD; i += 256)
        (&lam[0][0])[i] = 0;
    __syncthreads();

    // phase 1: lane holds position j0 + rl of rows 4 kq + i
    int64_t mx[4] = {INT64_MIN, INT64_MIN, INT64_MIN, INT64_MIN};
    uint32_t far = 0;   // bit 31: a score outside [-2^62, 2^62)
    // a scale that is a power of two (head_dim 64: 2^45) multiplies by a shift
    const bool pow2 = scale > 0 && scale <= Q48_ONE && (scale & (scale - 1)) == 0;
    const int sshr = 48 - (63 - __builtin_clzll((uint64_t)(scale > 0 ? scale : 1)));
    {
        const uint8_t *kd = KD + (size_t)kh * 8 * Ppad * HDP;
        const uint64_t *ck = CK + 2 * (size_t)kh * Ppad;
        for (int jt = w; jt < J / 16; jt += 4) {
            const int j = 16 * jt + rl;
            v4i B[KS][8];
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int b = 0; b < 8; ++b)
                    B[ks][b] = *reinterpret_cast<const v4i *>(kd + ((size_t)b * Ppad + j) * HDP +
                                                              64 * ks + 16 * kq);
            v4i acc[14];
#pragma unroll
            for (int d = 0; d < 14; ++d)
                acc[d] = (v4i){0, 0, 0, 0};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int a = 0; a < 8; ++a)
#pragma unroll
                    for (int b = 0; b < 8; ++b)
                        if (a + b <= 13)
                            acc[a + b] = __builtin_amdgcn_mfma_i32_16x16x64_i8(
                                A[ks][a], B[ks][b], acc[a + b], 0, 0, 0);
            const q48_u128 ckj = ld128(ck + 2 * (size_t)j);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = 4 * kq + i;
                const int64_t dot = digits_shr48(acc, i, cq[m] + ckj);
                const int64_t s = pow2 ? dot >> sshr : q48_mul(dot, scale);
                sc[(size_t)m * J + j] = s;
                far |= (uint32_t)((uint64_t)s >> 32) + 0x40000000u;
                if (m < nrow && j <= p0 + t0 + m)
                    mx[i] = s > mx[i] ? s : mx[i];
            }
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        mx[i] = row16_max64(mx[i]);
    if (rl == 0)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            mxs[w][4 * kq + i] = mx[i];
    if (far & 0x80000000u)
        atomicOr(&form, 4);
    __syncthreads();

    // phase 2: row r = tid / 16, positions tid % 16 + 16 k.  With every score
    // (of any tile position, masked ones too) within 2^62 of zero no difference
    // to the maximum wraps and q48_exp_neg serves; else q48_safe_exp.
    {
        const int r = tid >> 4, jj = tid & 15;
        int64_t sum = 0;
        int odd = 0;   // an exponential outside [0, ONE]: a wrapped difference
        if (r < nrow) {
            int64_t m = mxs[0][r];
#pragma unroll
            for (int u = 1; u < 4; ++u)
                m = mxs[u][r] > m ? mxs[u][r] : m;
            const int S = p0 + t0 + r + 1;
            int64_t *srow = sc + (size_t)r * J;
            if ((form & 4) == 0) {
                auto ex = [&](int64_t s) { return q48_exp_neg((uint64_t)m - (uint64_t)s); };
                int j = jj;
                for (; j + 48 < S; j += 64) {
                    const int64_t s0 = srow[j], s1 = srow[j + 16], s2 = srow[j + 32],
                                  s3 = srow[j + 48];
                    const int64_t e0 = ex(s0), e1 = ex(s1), e2 = ex(s2), e3 = ex(s3);
                    srow[j] = e0;
                    srow[j + 16] = e1;
                    srow[j + 32] = e2;
                    srow[j + 48] = e3;
                    sum += e0 + e1 + e2 + e3;   // at most 16320 ONE
                }
                for (; j < S; j += 16) {
                    const int64_t e = ex(srow[j]);
                    srow[j] = e;
                    sum += e;
                }
            } else {
                for (int j = jj; j < S; j += 16) {
                    const int64_t e = q48_safe_exp((int64_t)((uint64_t)srow[j] - (uint64_t)m));
                    srow[j] = e;
                    odd |= (uint64_t)e > (uint64_t)Q48_ONE ? 1 : 0;
                    sum = (int64_t)((uint64_t)sum + (uint64_t)e);
                }
            }
        }
        sum = (int64_t)group_sum64<16>((uint64_t)sum);
        if (jj == 0)
            sums[r] = sum;
        // a value outside [-2^51, 2^51) somewhere in the span
        const int *vbig = VB + (size_t)kh * (Ppad / PF_STEP);
        for (int c = tid; c < J / PF_STEP; c += 256)
            odd |= vbig[c] ? 2 : 0;
        if (odd)
            atomicOr(&form, odd);
    }
    __syncthreads();

    // phase 3.  form 0: every exponential is in [0, ONE], so each row's sum is
    // exact, at least ONE, and its weights add up to at most ONE; every value
    // of the span is in [-2^51, 2^51).  2: the same weights, larger values.
    // Bit 0: weights of any kind.
    const int vform = form & 3;
    const int Smax = p0 + t0 + nrow;
    const size_t kvd = (size_t)n_kv * HD;
    const int64_t *vraw = vcache + (size_t)kh * HD;
    if (vform & 1) {
        // the weights in place of the exponentials, then integer products
        {
            const int r = tid >> 4;
            if (r < nrow) {
                const int64_t den = sums[r];
                const q48_divisor dv = q48_divisor_of(den);
                if (den > 0)
                    for (int j = tid & 15; j < p0 + t0 + r + 1; j += 16)
                        sc[(size_t)r * J + j] = q48_div_by(sc[(size_t)r * J + j], dv);
            }
        }
        __syncthreads();
        for (int i = tid; i < nrow * HD; i += 256) {
            const int r = i / HD, d = i % HD;
            uint64_t a = 0;
            for (int j = 0; j < p0 + t0 + r + 1; ++j)
                a += (uint64_t)q48_mul(sc[(size_t)r * J + j], vraw[(size_t)j * kvd + d]);
            lam[r][d] = a;
        }
    } else {
        const int g = lane >> 4;
        double y48[4];
        uint64_t den[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const q48_divisor dv = q48_divisor_of(4 * i + g < nrow ? sums[4 * i + g] : Q48_ONE);
            y48[i] = dv.y48;
            den[i] = dv.d;
        }
        const double *vf = VF + (size_t)kh * Ppad * HD;
        const int vd = HD == 32 ? lane & 31 : lane;         // this lane's dim (and + 64)
        const int vp = HD == 32 ? 16 * (lane >> 5) : 0;     // its positions in the chunk
        // one set of sums over the span: the weights and values as this pass
        // takes them (0: p 2^-48 and v; 1: p 2^-48 and v mod 2^48; 2, 3: the
        // low 24 bits and the rest of p, and v >> 48), shifted left by sh
        auto pass = [&](auto split, int mode) {
            constexpr bool SPLIT = decltype(split)::value;
            double acc[DL][PF_ROWS];
#pragma unroll
            for (int l = 0; l < DL; ++l)
#pragma unroll
                for (int r = 0; r < PF_ROWS; ++r)
                    acc[l][r] = Q48_FSUM0;
            uint64_t er[4 * PG];
            auto load_e = [&](int j0) {
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int u = 0; u < PG; ++u)
                        er[PG * i + u] =
                            (uint64_t)sc[(size_t)(4 * i + g) * J + j0 + 16 * u + rl];
            };
            if (CP * w < Smax)
                load_e(CP * w);
            for (int j0 = CP * w; j0 < Smax; j0 += 4 * CP) {
                double v[DL][16];
#pragma unroll
                for (int n = 0; n < 16; ++n)
#pragma unroll
                    for (int l = 0; l < DL; ++l) {
                        const int j = j0 + vp + n;
                        if constexpr (SPLIT) {
                            const int64_t x = vraw[(size_t)min(j, Smax - 1) * kvd + vd + 64 * l];
                            uint32_t any = 0;
                            v[l][n] = q48_f51(mode == 1 ? x & (Q48_ONE - 1) : x >> 48, any);
                        } else {
                            v[l][n] = vf[(size_t)j * HD + vd + 64 * l];
                        }
                    }
                // fp_div(e, sum), as q48_div_by (0 <= e <= ONE <= sum, so its
                // estimate settles), as p 2^-48; 0 past the row's position
#pragma unroll
                for (int i = 0; i < 4; ++i)
#pragma unroll
                    for (int u = 0; u < PG; ++u) {
                        const uint64_t e = er[PG * i + u];
                        const int j = j0 + 16 * u + rl, r = 4 * i + g;
                        const double ed =
                            __builtin_bit_cast(double, e | 0x4330000000000000ull) - 0x1p52;
                        const uint64_t q0 =
                            q48_word_m52(__builtin_fma(ed, y48[i], 0x1p52 - 0.5));
                        const uint64_t rem = (e << 48) - q0 * den[i];
                        const double p = q48_pscaled((int64_t)(q0 + (rem >= den[i] ? 1 : 0)));
                        pw[w][r][16 * u + rl] = r < nrow && j < p0 + t0 + r + 1 ? p : 0.0;
                    }
                if (j0 + 4 * CP < Smax)
                    load_e(j0 + 4 * CP);
                // the wave's own LDS writes before its reads (in order; the
                // fence keeps the compiler's order)
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
                for (int r = 0; r < PF_ROWS; r += 4) {
                    double p[4];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        p[i] = pw[w][r + i][vp + rl];
                        if constexpr (SPLIT)
                            if (mode >= 2) {
                                const double pb = __builtin_fma(p[i], 0x1p24, 0x1p52) - 0x1p52;
                                p[i] = mode == 3 ? pb
                                                 : __builtin_fma(p[i], 0x1p48, -pb * 0x1p24);
                            }
                    }
#pragma unroll
                    for (int l = 0; l < DL; ++l) {
                        auto f4 = [&](auto base) {
                            constexpr int B = decltype(base)::value;
                            const double x[4] = {v[l][B], v[l][B + 1], v[l][B + 2], v[l][B + 3]};
                            q48_fsum4x4<B>(acc[l][r], acc[l][r + 1], acc[l][r + 2], acc[l][r + 3],
                                           p, x);
                        };
                        f4(std::integral_constant<int, 0>{});
                        f4(std::integral_constant<int, 4>{});
                        f4(std::integral_constant<int, 8>{});
                        f4(std::integral_constant<int, 12>{});
                    }
                }
                __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
                __builtin_amdgcn_wave_barrier();
                __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
            }
#pragma unroll
            for (int r = 0; r < PF_ROWS; ++r)
#pragma unroll
                for (int l = 0; l < DL; ++l) {
                    uint64_t t = (uint64_t)q48_fsum_total(acc[l][r]);
                    if (SPLIT && mode == 3)
                        t <<= 24;
                    atomicAdd(reinterpret_cast<unsigned long long *>(&lam[r][vd + 64 * l]),
                              (unsigned long long)t);
                }
        };
        if (vform == 0)
            pass(std::false_type{}, 0);
        else
            for (int mode = 1; mode <= 3; ++mode)
                pass(std::true_type{}, mode);
    }
    __syncthreads();
    for (int i = tid; i < nrow * HD; i += 256)
        out[(size_t)(t0 + i / HD) * n_heads * HD + (size_t)h * HD + i % HD] =
            (int64_t)lam[i / HD][i % HD];
}

} // namespace

bool q48_pf_attn_mfma_ok(int p0, int T, int hd)
{
    return (hd == 32 || hd == 64 || hd == 128) && T > 0 && p0 >= 0 && p0 + T <= PF_MAX_POS;
}

int q48_pf_attn_mfma_max_pos() { return PF_MAX_POS; }

int q48_launch_pf_attn_mfma(q48_ctx *c, int64_t *out, const int64_t *QKV, int64_t *kcache,
                            int64_t *vcache, int layer, int p0, int T, int n_heads, int n_kv,
                            int hd, int max_seq)
{
    const int P = p0 + T, Ppad = pf_round64(P), HDP = hd < 64 ? 64 : hd;
    const int nt = (T + PF_ROWS - 1) / PF_ROWS, G = n_heads / n_kv;
    size_t span = 0;
    for (int i = 0; i < nt; ++i)
        span += (size_t)pf_span(i, p0, T);
    const size_t per_head = PF_ROWS * span;
    size_t o = 0;
    auto take = [&](size_t bytes) {
        const size_t at = o;
        o += (bytes + 255) & ~(size_t)255;
        return at;
    };
    const size_t o_kd = take((size_t)n_kv * 8 * Ppad * HDP);
    const size_t o_ck = take((size_t)n_kv * Ppad * 16);
    const size_t o_vf = take((size_t)n_kv * Ppad * hd * sizeof(double));
    const size_t o_vb = take((size_t)n_kv * (Ppad / PF_STEP) * sizeof(int));
    const size_t o_sc = take((size_t)n_heads * per_head * sizeof(int64_t));
    int rc = q48_ws_reserve(c, o);
    if (rc)
        return rc;
    uint8_t *ws = (uint8_t *)c->ws;
    uint8_t *KD = ws + o_kd;
    uint64_t *CK = (uint64_t *)(ws + o_ck);
    double *VF = (double *)(ws + o_vf);
    int *VB = (int *)(ws + o_vb);
    int64_t *SCR = (int64_t *)(ws + o_sc);
    const int64_t *vl = vcache + (size_t)layer * max_seq * n_kv * hd;
    const int64_t *scale_p = c->rope_sin + (size_t)c->rope_max_seq * (c->rope_head_dim / 2);
    const dim3 pgrid(Ppad / PF_STEP, n_kv);
    const unsigned grid = 8 % n_kv == 0
                              ? 8u * (unsigned)((G * nt + 8 / n_kv - 1) / (8 / n_kv))
                              : (unsigned)(n_heads * nt);
#define PFA_LAUNCH(HDV)                                                                       \
    do {                                                                                      \
        hipLaunchKernelGGL(k_pfa_prep<HDV>, pgrid, dim3(256), 0, c->stream, KD, CK, VF, VB,   \
                           kcache, vcache, layer, P, Ppad, n_kv, max_seq);                    \
        hipLaunchKernelGGL(k_pfa<HDV>, dim3(grid), dim3(256), 0, c->stream, out, QKV, KD, CK, \
                           VF, VB, vl, SCR, scale_p, p0, T, n_heads, n_kv, Ppad, per_head);   \
    } while (0)
    if (hd == 64)
        PFA_LAUNCH(64);
    else if (hd == 32)
        PFA_LAUNCH(32);
    else
        PFA_LAUNCH(128);
#undef PFA_LAUNCH
    return (int)hipGetLastError();
}
