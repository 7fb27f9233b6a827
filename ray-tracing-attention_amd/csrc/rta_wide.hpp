// rta_wide.hpp -- the K-quant readout over more than one matrix-core batch tile (prompt
// chunks, large decode batches): y[b, r] = sum_k W[r, k] x[b, k] for up to kWideBatch rows
// in one pass over the weights.
//
// The narrow readouts (rta_gemm.hpp, rta_tiled.hpp) keep a slab of x in LDS and build the
// weight operands in the wave that multiplies them, which suits one tile of up to 32 rows;
// for a batch of 256 they read and decode the weights eight times.  Here the weights are
// what the workgroup shares:
//   - a workgroup (8 waves: 4 along the batch x 2 along the rows) computes 64 NB batch rows
//     x 32 TN weight rows over its K slab;
//   - each half superblock (4 matrix-core steps of 32 columns) of the 2 TN row tiles is
//     decoded once, by the wave owning the tile, into binary16 B operands in LDS (two
//     buffers, one barrier per half superblock), and read by all waves;
//   - x comes as matrix-core fragments (wide_xprep_kernel: 64 lanes x 16 bytes per 16 rows,
//     32 columns and plane), read straight into registers: a wave's loads are whole
//     contiguous KB and only the wave pair of a SIMD shares them.
// Arithmetic per superblock, operand values and scales are those of the narrow readouts
// (rta_gemm.hpp): x s as hi + lo binary16, exact code x sub-block scale products, the group
// sums in one more MFMA, then d, the minimum / offset and 1 / s on the fp32 results.
// GGUF rows and packed tiles differ only in where a lane's bytes lie (LaneSource).
//
// Bound: matrix cores (two MFMAs per weight tile, 16 rows and 32 columns) where the grid
// fills the chip; per superblock of TN = 8, NB = 2 a wave issues 272 MFMAs (4352 cycles)
// and ~450 VALU instructions, and two waves share a SIMD.
#pragma once
#include "rta_tiled.hpp"

namespace rta {

constexpr int kWideBatch = 256;   // batch rows of one launch
constexpr int kWideThreads = 512;

// x as matrix-core fragments (workspace): for row tile t (16 rows), superblock sb, step j
// (0..7) and plane p (hi, lo) 64 lanes x 8 binary16 at frag[(((t nsb + sb) 8 + j) 2 + p) 64],
// lane (s, li) holding row li, columns of (step j, segment s) of the tile format; the group
// sums at g[(t nsb + sb) 64] and 1 / s of the 16 rows at inv[(t nsb + sb) 16].
struct WideX {
    uint4* frag;
    uint4* g;
    float* inv;
};

// Steps of a superblock.  With one row tile per wave (NB = 1, 33 to 64 rows) step j is column
// offset m = j of the tile format and the K slabs are those of the narrow tiles, so that a
// row's result is bit for bit that of a call of 17 to 32 rows.  With two the order is split:
// each half superblock (j < 4, j >= 4) uses one half of a lane's quant bytes, which frees
// their registers early (256 are all in use).
template <int NB>
constexpr bool kWideSplit = NB == 2;
__device__ __forceinline__ int wide_step(bool q4, bool split, int m) {
    return !split ? m : q4 ? 4 * ((m >> 1) & 1) + (m & 1) + 2 * (m >> 2) : 4 * (m & 1) + (m >> 1);
}

// Block: 16 rows x 32 threads of 8 columns, one superblock (grid: superblocks x row tiles).
// With nw, x is a residual row and its RMSNorm (op 1: x nw / sqrt(mean(x^2) + eps)) is taken
// here, every block summing its rows' squares itself: the rows are read once per superblock
// from the cache, for the launch of a norm kernel saved (64-sequence step of 17 norms: 986 ->
// 964 us).
template <int FMT, bool SPLIT>
__global__ void __launch_bounds__(512) wide_xprep_kernel(const float* __restrict__ x, int cols, int batch, WideX p,
                                                         const float* __restrict__ nw, float eps) {
    constexpr bool kQ4 = FMT == RTA_Q4_K;
    __shared__ uint4 frag[16][64];
    __shared__ h8_t gs[16][4];
    const int tid = threadIdx.x, r = tid >> 5, t = tid & 31;
    const int sb = blockIdx.x, nsb = gridDim.x, row = blockIdx.y * 16 + r;
    float v[8];
    {
        const bool live = row < batch;
        const float4* src = reinterpret_cast<const float4*>(x + (int64_t)(live ? row : batch - 1) * cols + sb * 256 + 8 * t);
        const float4 a = src[0], c = src[1];
        v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = c.x; v[5] = c.y; v[6] = c.z; v[7] = c.w;
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = live ? v[i] : 0.0f;
    }
    if (nw) {   // uniform
        const float4* xr = reinterpret_cast<const float4*>(x + (int64_t)min(row, batch - 1) * cols);
        float ss = 0.0f;
#pragma unroll 8
        for (int i = t; i < cols >> 2; i += 32) {
            const float4 a = xr[i];
            ss += (a.x * a.x + a.y * a.y) + (a.z * a.z + a.w * a.w);
        }
        ss += dpp_mov<0xB1>(ss);
        ss += dpp_mov<0x4E>(ss);
        ss += dpp_mov<0x141>(ss);
        ss += dpp_mov<0x140>(ss);
        const float inv = 1.0f / sqrtf(add_xor16(ss) / (float)cols + eps);
        const float4* g = reinterpret_cast<const float4*>(nw + sb * 256 + 8 * t);
        const float4 g0 = g[0], g1 = g[1];
        const float gw[8] = {g0.x, g0.y, g0.z, g0.w, g1.x, g1.y, g1.z, g1.w};
#pragma unroll
        for (int i = 0; i < 8; ++i) v[i] = v[i] * inv * gw[i];
    }
    float m = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) m = fmaxf(m, fabsf(v[i]));
    m = group_max(m, 32);
    const int e = operand_exponent(m);
    const float sc = ldexpf(1.0f, 14 - e);   // max |x s| in [2^13, 2^14)
    const int64_t at = (int64_t)blockIdx.y * nsb + sb;
    if (t == 0) p.inv[at * 16 + r] = row < batch ? ldexpf(1.0f, e - 14) : 0.0f;
    constexpr int perm[8] = {0, 2, 1, 3, 4, 6, 5, 7};
    h8_t hi, lo;
    float sum8 = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const float w = v[perm[i]] * sc;
        hi[i] = (_Float16)w;
        lo[i] = (_Float16)(w - (float)hi[i]);
        sum8 += v[i] * sc;
    }
    // this thread's 8 columns are (segment, column offset) of the tile format
    const int seg = kQ4 ? t >> 3 : 2 * (t >> 4) + ((t >> 1) & 1);
    const int mo = kQ4 ? t & 7 : 2 * ((t >> 2) & 3) + (t & 1);
    const int j = wide_step(kQ4, SPLIT, mo);
    frag[2 * j][16 * seg + r] = __builtin_bit_cast(uint4, hi);
    frag[2 * j + 1][16 * seg + r] = __builtin_bit_cast(uint4, lo);
    _Float16* g = reinterpret_cast<_Float16*>(&gs[r][0]);
    const float s16 = sum8 + dpp_mov<0xB1>(sum8);
    const float s32 = s16 + dpp_mov<0x4E>(s16);
    if constexpr (kQ4) {
        const int q = t >> 2;   // 32-group: segment q / 2, slots 2 (q % 2), + 1; zeros at + 4, + 5
        if ((t & 3) == 0) {
            const float w = s32 * (1.0f / 32.0f);
            const _Float16 h = (_Float16)w;
            g[8 * (q >> 1) + 2 * (q & 1)] = h;
            g[8 * (q >> 1) + 2 * (q & 1) + 1] = (_Float16)(w - (float)h);
        } else if ((t & 3) == 1) {
            g[8 * (q >> 1) + 4 + 2 * (q & 1)] = (_Float16)0.0f;
            g[8 * (q >> 1) + 5 + 2 * (q & 1)] = (_Float16)0.0f;
        }
    } else if ((t & 1) == 0) {   // 16-group u = 8 hh + 2 q + sg -> segment 2 hh + sg, slot 2 q
        const int u = t >> 1, sg = 2 * (u >> 3) + (u & 1), q = (u >> 1) & 3;
        const float w = s16 * (1.0f / 16.0f);
        const _Float16 h = (_Float16)w;
        g[8 * sg + 2 * q] = h;
        g[8 * sg + 2 * q + 1] = (_Float16)(w - (float)h);
    }
    __syncthreads();
    uint4* dst = p.frag + at * 1024;
#pragma unroll
    for (int i = 0; i < 2; ++i) dst[tid + 512 * i] = (&frag[0][0])[tid + 512 * i];
    if (tid < 64) p.g[at * 64 + tid] = __builtin_bit_cast(uint4, gs[tid & 15][tid >> 4]);
}

struct WideArgs {
    const uint8_t* w;
    const uint8_t* w2;       // DUAL: the up matrix
    int64_t row_bytes;       // GGUF rows; 0: packed tiles
    int rows, nsbt;
    WideX x;
    int batch, rt;           // batch rows of the launch, their row tiles of x
    float* y;                // [batch, rows]
    float* part;             // K slabs [slab][batch][DUAL ? 2 rows : rows] when gridDim.z > 1
    float* pmax;             // kLogits: [batch][row tiles] maxima
    int sb_per_slab;
    int mode;
};

template <int TN>
struct WideLds {
    uint4 w[2 * TN][4][64];      // B operands of half a superblock: tile, step, lane
};
template <int TN>
struct WideMeta {
    uint2 bm[2][2 * TN][64];     // group-sum operand of the superblock (two buffers)
    float2 d[2][2 * TN][16];     // d terms per row
};

// Grid: (row blocks of 2 TN tiles, batch blocks of 64 NB rows, K slabs).
template <int FMT, bool DUAL, int NB, int TN>
__global__ void __launch_bounds__(kWideThreads, 2) wide_kernel(const WideArgs a) {
    constexpr bool kQ4 = FMT == RTA_Q4_K, kSplit = kWideSplit<NB>;
    using Source = LaneSource<FMT>;
    using Raw = typename Source::Raw;
    constexpr int DT = (2 * TN + 7) / 8;   // tiles a wave decodes (the last only while they last)
    __shared__ WideLds<TN> buf0;
    __shared__ WideLds<TN> buf1;
    __shared__ WideMeta<TN> meta;
    const int tid = threadIdx.x, lane = tid & 63, li = lane & 15, s = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), mg = wave & 3, nh = wave >> 2;
    const int nsbt = a.nsbt, sb0 = blockIdx.z * a.sb_per_slab, nsb = min(a.sb_per_slab, nsbt - sb0);
    const int ntile = (a.rows + 15) >> 4;
    const bool tiled = a.row_bytes == 0;

    // Row tile of workgroup-local tile t.  DUAL: each wave half holds TN / 2 gate tiles, then
    // the TN / 2 up tiles of the same rows.  Tiles past the end repeat the last one.
    auto tile_of = [&](int t) {
        if constexpr (DUAL) return ((int)blockIdx.x * 2 + t / TN) * (TN / 2) + t % (TN / 2);
        else return (int)blockIdx.x * 2 * TN + t;
    };
    const Source src(tiled, lane);
    const uint8_t* wp[DT];
#pragma unroll
    for (int i = 0; i < DT; ++i) {
        const int t = min(wave + 8 * i, 2 * TN - 1);
        const uint8_t* m = DUAL && (t % TN) >= TN / 2 ? a.w2 : a.w;
        const int T = min(tile_of(t), ntile - 1);
        if (tiled) wp[i] = m + ((int64_t)T * nsbt + sb0) * src.stride;
        else wp[i] = m + (int64_t)min(16 * T + li, a.rows - 1) * a.row_bytes + (int64_t)sb0 * src.stride;
    }
    auto load_raw = [&](int sb, Raw* r) {
#pragma unroll
        for (int i = 0; i < DT; ++i)
            if (8 * i + 7 < 2 * TN || wave + 8 * i < 2 * TN) src.load(wp[i] + (int64_t)sb * src.stride, r[i]);
    };

    // x fragments of this wave's NB row tiles: contiguous over superblocks and steps
    const uint4* xp[NB];
    int rtile[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        rtile[b] = ((int)blockIdx.y * 4 + mg) * NB + b;
        xp[b] = a.x.frag + ((int64_t)min(rtile[b], a.rt - 1) * nsbt + sb0) * 1024 + lane;
    }
    const int nstep = 8 * nsb;
    h8_t xa[2][NB][2];
    auto load_x = [&](int j, h8_t(*dst)[2]) {
        const int at = min(j, nstep - 1) * 128;
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            dst[b][0] = __builtin_bit_cast(h8_t, xp[b][at]);
            dst[b][1] = __builtin_bit_cast(h8_t, xp[b][at + 64]);
        }
    };

    const Q4kSegment seg(s);
    uint32_t sc[DT][kQ4 ? 2 : 4];   // binary16 pairs of a lane's sub-block scales
    // Scales of a superblock, its d terms and group-sum operand (into meta[par])
    auto decode_header = [&](const Raw* r, int par) {
#pragma unroll
        for (int i = 0; i < DT; ++i) {
            const int t = wave + 8 * i;
            if (8 * i + 7 >= 2 * TN && t >= 2 * TN) continue;   // uniform
            if constexpr (kQ4) {
                uint32_t sc0, sc1, m0, m1;
                if (tiled) q4k_tile_scale_min(r[i].hdr, seg, sc0, sc1, m0, m1);
                else q4k_row_scale_min(r[i].hdr, s, sc0, sc1, m0, m1);
                sc[i][0] = h2dup_scaled(sc0, 1024.0f);
                sc[i][1] = h2dup_scaled(sc1, 64.0f);
                meta.bm[par][t][lane] = uint2{h2dup_scaled(m0, 1.0f), h2dup_scaled(m1, 1.0f)};
                // codes carry 2^-14; group sums are staged / 32
                if (s == 0) meta.d[par][t][li] = make_float2(half_lo(r[i].hdr.x) * 16384.0f, half_hi(r[i].hdr.x) * -32.0f);
            } else {
                const int hh = s >> 1, sg = s & 1;
                const uint32_t wa = hh ? r[i].sc.z : r[i].sc.x, wb = hh ? r[i].sc.w : r[i].sc.y;
                float f[4];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    f[q] = (float)(int)(int8_t)(((q < 2 ? wa : wb) >> (8 * (2 * (q & 1) + sg))) & 255u);
                    sc[i][q] = h2dup(f[q] * 256.0f);
                }
                meta.bm[par][t][lane] = uint2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(-f[0], -f[1])),
                                              __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(-f[2], -f[3]))};
                const float d = (float)__builtin_bit_cast(_Float16, (uint16_t)r[i].d);
                if (s == 0) meta.d[par][t][li] = make_float2(d * 16384.0f, d * 512.0f);   // sums staged / 16
            }
        }
    };
    // B operands of step k (0..3) of half hf of a superblock -> dst
    auto decode_step = [&](const Raw* r, int hf, int k, WideLds<TN>& dst) {
#pragma unroll
        for (int i = 0; i < DT; ++i) {
            const int t = wave + 8 * i;
            if (8 * i + 7 >= 2 * TN && t >= 2 * TN) continue;   // uniform
            uint4 v;
            if constexpr (kQ4) {
                const bool second = kSplit ? hf : k >> 1, high = kSplit ? k >> 1 : hf;   // quant run, nibble
                const uint4& q = second ? r[i].q1 : r[i].q0;
                const uint32_t w0 = word_of(q, 2 * (k & 1)), w1 = word_of(q, 2 * (k & 1) + 1);
                const uint32_t M = high ? 0x00F000F0u : 0x000F000Fu, sp = sc[i][high ? 1 : 0];
                v = uint4{pk_mul_f16(w0 & M, sp), pk_mul_f16((w0 >> 8) & M, sp), pk_mul_f16(w1 & M, sp),
                          pk_mul_f16((w1 >> 8) & M, sp)};
            } else {
                const int q = kSplit ? k : 2 * hf + (k >> 1), half = kSplit ? hf : k & 1;   // scale group, word pair
                const uint4& run = (q & 1) ? r[i].b : r[i].a;
                uint32_t o[4];
#pragma unroll
                for (int d2 = 0; d2 < 2; ++d2) {
                    const uint32_t rw = word_of(run, 2 * half + d2), hw = word_of(r[i].h, 2 * half + d2);
                    // 4 c per byte: nibble at bits 2..5, the two high bits at 6..7
                    const uint32_t nb = (q >> 1) ? (rw >> 2) : (rw << 2);
                    const uint32_t code = (nb & 0x3C3C3C3Cu) | ((hw << (6 - 2 * q)) & 0xC0C0C0C0u);
                    o[2 * d2] = pk_mul_f16(code & 0x00FF00FFu, sc[i][q]);
                    o[2 * d2 + 1] = pk_mul_f16((code >> 8) & 0x00FF00FFu, sc[i][q]);
                }
                v = uint4{o[0], o[1], o[2], o[3]};
            }
            dst.w[t][k][lane] = v;
        }
    };

    f4_t acc[TN][NB], C[TN][NB];
    const f4_t zero = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int b = 0; b < NB; ++b) acc[j][b] = zero;

    // MFMAs of one step: hi plane then lo plane of a tile pair, so that an accumulator's two
    // are 2 NB apart
    auto multiply = [&](const WideLds<TN>& from, int k, const h8_t(*x)[2], bool first) {
#pragma unroll
        for (int j0 = 0; j0 < TN; j0 += 2) {
            h8_t bw[2];
#pragma unroll
            for (int t = 0; t < 2; ++t) bw[t] = __builtin_bit_cast(h8_t, from.w[nh * TN + j0 + t][k][lane]);
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int b = 0; b < NB; ++b)
                        C[j0 + t][b] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                            x[b][p], bw[t], first && p == 0 ? zero : C[j0 + t][b], 0, 0, 0);
        }
    };

    Raw cur[DT], nxt[DT];
    load_raw(0, cur);
    load_x(0, xa[0]);
    load_x(1, xa[1]);
    decode_header(cur, 0);
#pragma unroll
    for (int k = 0; k < 4; ++k) decode_step(cur, 0, k, buf0);
    __syncthreads();

    for (int sb = 0; sb < nsb; ++sb) {
        load_raw(min(sb + 1, nsb - 1), nxt);
        // first half from buf0; the second half is decoded meanwhile
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            decode_step(cur, 1, k, buf1);
            multiply(buf0, k, xa[k & 1], k == 0);
            load_x(8 * sb + k + 2, xa[k & 1]);
        }
        // the superblock's group sums and 1 / s, needed at its end
        h8_t am[NB];
        float4 inv[NB];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const int64_t at = (int64_t)min(rtile[b], a.rt - 1) * nsbt + sb0 + sb;
            am[b] = __builtin_bit_cast(h8_t, a.x.g[at * 64 + lane]);
            inv[b] = *reinterpret_cast<const float4*>(a.x.inv + at * 16 + 4 * s);
        }
        __syncthreads();
        // second half from buf1; the next superblock's first half is decoded meanwhile (at
        // the end a repeat of the last superblock, never read)
        decode_header(nxt, (sb + 1) & 1);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            decode_step(nxt, 0, k, buf0);
            multiply(buf1, k, xa[k & 1], false);
            load_x(8 * sb + k + 6, xa[k & 1]);
        }
        const int par = sb & 1;
#pragma unroll
        for (int j = 0; j < TN; ++j) {
            const int t = nh * TN + j;
            const uint2 m = meta.bm[par][t][lane];
            const float2 d = meta.d[par][t][li];
            uint4 bm;
            if constexpr (kQ4) bm = uint4{m.x, m.y, 0u, 0u};
            else   // each group's negated scale twice (the sum's hi and lo)
                bm = uint4{(m.x & 0xffffu) * 0x10001u, (m.x >> 16) * 0x10001u, (m.y & 0xffffu) * 0x10001u,
                           (m.y >> 16) * 0x10001u};
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                const f4_t Cm = __builtin_amdgcn_mfma_f32_16x16x32_f16(am[b], __builtin_bit_cast(h8_t, bm), zero, 0, 0, 0);
                const float iv[4] = {inv[b].x, inv[b].y, inv[b].z, inv[b].w};
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    acc[j][b][e] = fmaf(fmaf(d.y, Cm[e], d.x * C[j][b][e]), iv[e], acc[j][b][e]);
            }
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < DT; ++i) cur[i] = nxt[i];
    }

    // ---- results: lane (s, li) holds batch rows 4 s + e of each row tile, weight row li
    const int total = DUAL ? 2 * a.rows : a.rows;
    const bool slabs = gridDim.z > 1;
#pragma unroll
    for (int j = 0; j < (DUAL ? TN / 2 : TN); ++j) {
        const int T = tile_of(nh * TN + j), row = 16 * T + li;
        const bool ok = row < a.rows;
        auto batch_row = [&](int b, int e) { return 16 * rtile[b] + 4 * s + e; };
        float old[NB][4];   // kAccumulate: every load of the tile before the first store
        if (!DUAL && !slabs && a.mode == kAccumulate) {
#pragma unroll
            for (int b = 0; b < NB; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    old[b][e] = a.y[(int64_t)min(batch_row(b, e), a.batch - 1) * a.rows + min(row, a.rows - 1)];
        }
#pragma unroll
        for (int b = 0; b < NB; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int br = batch_row(b, e);
                const bool live = ok && br < a.batch;
                const float v = acc[j][b][e];
                if constexpr (DUAL) {
                    const float up = acc[j + TN / 2][b][e];
                    if (slabs) {
                        if (live)
                            *reinterpret_cast<float2*>(a.part + ((int64_t)blockIdx.z * a.batch + br) * total + 2 * row) =
                                make_float2(v, up);
                    } else if (live) {
                        a.y[(int64_t)br * a.rows + row] = swiglu(v, up);
                    }
                } else {
                    if (slabs) {
                        if (live) a.part[((int64_t)blockIdx.z * a.batch + br) * total + row] = v;
                    } else if (a.mode == kAccumulate) {
                        if (live) a.y[(int64_t)br * a.rows + row] = old[b][e] + v;
                    } else {
                        if (live) a.y[(int64_t)br * a.rows + row] = v;
                        if (a.mode == kLogits) {   // per-tile maxima for the argmax
                            const float mx = group_max(ok ? v : -INFINITY, 16);
                            if (li == 0 && br < a.batch && T < ntile) a.pmax[(int64_t)br * ntile + T] = mx;
                        }
                    }
                }
            }
    }
}

}  // namespace rta
