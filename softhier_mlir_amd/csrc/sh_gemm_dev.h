// Device code shared by the GEMM kernels (sh_gemm.hip, sh_gemm_small.hip): the launch arguments, the tile order, the
// LayerNorm fold and the epilogue chain. Not part of the C ABI.
#pragma once
#include "sh_common.h"
#include "sh_ln_pair.h"

constexpr int BK = 64;

struct GemmArgs {
    const uint16_t *x, *w;
    uint16_t *z;
    float *part;                 // split-K partials [splits][M][N] (fp32), or null
    const void *bias;            // null, fp16 or fp32 row of N
    const uint16_t *res;         // null or fp16 [M, ldr]
    uint64_t ldx, ldw, ldz, ldr;
    uint32_t M, N, K;
    uint32_t kps;                // K per split (multiple of BK)
    uint32_t tiles_m, tiles_n, splits;
    uint32_t accumulate, bias_fp32, act;
    uint32_t xcd_groups;         // > 1: XCD-aware block remap with this many XCDs (requires divisibility)
    uint32_t group_m;            // > 1: tiles ordered in bands of this many tile rows, column by column within a band
    uint32_t per_xcd;            // workgroups per XCD of the remap, and tile_of's divisors (set_tile_order): by the XCDs,
    ShDiv d_xcd, d_tiles, d_band, d_rows, d_last;    // the tiles of one split, a band's tiles, a band's rows, the last band's
    const float *ln_stats;       // LayerNorm fold (or null): (mu, r) per row, fp32 [M][2], or ln_parts partials ...
    const float *ln_c;           // ... and c per column (fp32 [N]); the fp32 bias row is then d
    uint32_t ln_parts;           // > 0: ln_stats holds ln_parts (sum, M2) pairs of 32 columns per row (row_partials)
    float ln_eps;                // ... and the statistics are formed with this eps
    float *stats_out;            // or null: the (sum, M2) pairs of every 32 columns of each stored row, [M][N / 32]
};

namespace {

// (mu, r = 1 / sqrt(var + eps)) of row gm for the LayerNorm fold: given (ln_parts == 0), or formed from the row's
// ln_parts partials (s_b, M2_b) of 32 columns each (Chan, Golub and LeVeque, "Algorithms for computing the sample
// variance", 1983): mu = sum s_b / n, M2 = sum_b (M2_b + 32 (s_b / 32 - mu)^2), var = M2 / n, n = 32 ln_parts,
// sums in block order. Up to 32 partials (K <= 1024) of a 16-byte aligned array are loaded at once into registers,
// 16 bytes per load (only the P / 2 loads the row has: the partials are re-read by every column tile, so their volume
// is what this costs), and summed twice; more, or an array that is only 8-byte aligned, are read twice from memory
// 8 bytes at a time (the same sums in the same order). Every consumer (register epilogues, split-K reduction) forms
// the statistics with this one function.
__device__ __forceinline__ bool ln_in_registers(const GemmArgs &a) {
    return a.ln_parts <= 32 && a.ln_parts % 2 == 0 && ((uintptr_t)a.ln_stats & 15u) == 0;
}
__device__ __forceinline__ float2 ln_row(const GemmArgs &a, uint32_t gm) {
    if (a.ln_parts == 0) return ((const float2 *)a.ln_stats)[gm];
    const uint32_t P = a.ln_parts;
    const float2 *pp = (const float2 *)a.ln_stats + (uint64_t)gm * P;
    const float inv_n = 1.f / (32.f * (float)P);
    float s = 0.f, m2 = 0.f;
    if (ln_in_registers(a)) {
        const uint32_t last = P / 2 - 1;             // wave-uniform: the branches below skip whole loads
        float4 q[16];
#pragma unroll
        for (int h = 0; h < 16; ++h)
            if ((uint32_t)h <= last) q[h] = ((const float4 *)pp)[h];
#pragma unroll
        for (int h = 0; h < 16; ++h)
            if ((uint32_t)h <= last) s += q[h].x + q[h].z;
        const float mu = s * inv_n;
#pragma unroll
        for (int h = 0; h < 16; ++h) {
            if ((uint32_t)h > last) continue;
            const float d0 = fmaf(q[h].x, 1.f / 32.f, -mu), d1 = fmaf(q[h].z, 1.f / 32.f, -mu);
            m2 += fmaf(32.f * d0, d0, q[h].y) + fmaf(32.f * d1, d1, q[h].w);
        }
        return make_float2(mu, sh_fast_rsq(fmaf(m2, inv_n, a.ln_eps)));
    }
    for (uint32_t b = 0; b < P; b += 2) s += pp[b].x + (b + 1 < P ? pp[b + 1].x : 0.f);
    const float mu = s * inv_n;
    for (uint32_t b = 0; b < P; b += 2) {
        const float2 q0 = pp[b], q1 = b + 1 < P ? pp[b + 1] : make_float2(32.f * mu, 0.f);
        const float d0 = fmaf(q0.x, 1.f / 32.f, -mu), d1 = fmaf(q1.x, 1.f / 32.f, -mu);
        m2 += fmaf(32.f * d0, d0, q0.y) + fmaf(32.f * d1, d1, q1.y);
    }
    return make_float2(mu, sh_fast_rsq(fmaf(m2, inv_n, a.ln_eps)));
}

// The same for 32 rows of a wavefront, lanes r32 and r32 + 32 sharing row gm, in two halves so that work can go between the
// loads and their use: each lane requests half of its row's partials, and the upper lane carries the lower lane's
// running sums on, so the order of every sum (and its bits) is ln_row's. pair_form: (mu, r) in both lanes.
struct LnPair { float4 q[8]; };
__device__ __forceinline__ void ln_pair_load(const GemmArgs &a, uint32_t gm, LnPair &l) {
    if (a.ln_parts == 0) {
        const float2 v = ((const float2 *)a.ln_stats)[gm];
        l.q[0] = make_float4(v.x, v.y, 0.f, 0.f);
        return;
    }
    if (!ln_in_registers(a)) return;
    const uint32_t n = a.ln_parts / 2, up = (threadIdx.x >> 5) & 1;
    const float4 *pp = (const float4 *)((const float2 *)a.ln_stats + (uint64_t)gm * a.ln_parts);
#pragma unroll
    for (int h = 0; h < 8; ++h)
        if ((uint32_t)h < ln_pair_count(n, 0)) l.q[h] = pp[ln_pair_at(n, up, h)];           // (n odd: the upper lane's last is unused)
}
__device__ __forceinline__ float2 ln_pair_form(const GemmArgs &a, uint32_t gm, const LnPair &l) {
    if (a.ln_parts == 0) return make_float2(l.q[0].x, l.q[0].y);
    if (!ln_in_registers(a)) return ln_row(a, gm);
    const uint32_t up = (threadIdx.x >> 5) & 1, mine = ln_pair_count(a.ln_parts / 2, up);
    const int lower = (int)(threadIdx.x & 31), upper = lower + 32;
    const float inv_n = 1.f / (32.f * (float)a.ln_parts);
    float s = 0.f, m2 = 0.f;
#pragma unroll
    for (int p = 0; p < 2; ++p) {                       // pass 0: the lower lane's sums, pass 1: the upper lane's after them
        if (p == 1) s = __shfl(s, lower, 64);
        if (p == (int)up) {
#pragma unroll
            for (int h = 0; h < 8; ++h)
                if ((uint32_t)h < mine) s += l.q[h].x + l.q[h].z;
        }
    }
    s = __shfl(s, upper, 64);
    const float mu = s * inv_n;
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        if (p == 1) m2 = __shfl(m2, lower, 64);
        if (p == (int)up) {
#pragma unroll
            for (int h = 0; h < 8; ++h) {
                if ((uint32_t)h >= mine) continue;
                const float d0 = fmaf(l.q[h].x, 1.f / 32.f, -mu), d1 = fmaf(l.q[h].z, 1.f / 32.f, -mu);
                m2 += fmaf(32.f * d0, d0, l.q[h].y) + fmaf(32.f * d1, d1, l.q[h].w);
            }
        }
    }
    m2 = __shfl(m2, upper, 64);
    return make_float2(mu, sh_fast_rsq(fmaf(m2, inv_n, a.ln_eps)));
}

// A wavefront's rows' fold factors (r and r mu of rows mrow + 32 i + r32), formed once at the start of a tile so
// the loads overlap its first DMAs and the epilogue waits on nothing: lane l forms rows mrow + l + 64 k, and each
// lane takes its rows' factors from those lanes.
template <int FM>
struct LnRows { float r[FM], rm[FM]; };
template <int FM>
__device__ __forceinline__ LnRows<FM> ln_rows(const GemmArgs &a, uint32_t mrow) {
    constexpr int RPL = (FM + 1) / 2;                // rows formed per lane
    LnRows<FM> l;
    const int lane = threadIdx.x & 63, r32 = lane & 31;
    if (!a.ln_stats) {
#pragma unroll
        for (int i = 0; i < FM; ++i) { l.r[i] = 0.f; l.rm[i] = 0.f; }
        return l;
    }
    float2 st[RPL];
#pragma unroll
    for (int k = 0; k < RPL; ++k) st[k] = ln_row(a, min(mrow + 64 * k + lane, a.M - 1));
#pragma unroll
    for (int i = 0; i < FM; ++i) {                   // row 32 i + r32 was formed by lane 32 (i % 2) + r32, k = i / 2
        const float mu = __shfl(st[i / 2].x, 32 * (i % 2) + r32, 64), r = __shfl(st[i / 2].y, 32 * (i % 2) + r32, 64);
        l.r[i] = r;
        l.rm[i] = mu * r;
    }
    return l;
}

// LayerNorm folded into the product (sh_gemm_epi.ln_stats): p -> r p - (r mu) c + d in fp32, before the fp16
// rounding; the bias (d) is part of this step, so the chain below skips it. st = ln_row(a, gm).
__device__ __forceinline__ float ln_apply(const GemmArgs &a, float2 st, float p, uint32_t gn) {
    return fmaf(st.y, p, fmaf(-(st.x * st.y), a.ln_c[gn], ((const float *)a.bias)[gn]));
}

// Logical tile of block b -> (split, tile row, tile column). Dispatch deals workgroups round-robin over the
// XCDs, so block b becomes logical index (b % X) (T / X) + b / X: each XCD walks a contiguous run of the tile
// order and the operand panels it shares stay in that XCD's L2. The order is row-major, or (group_m > 1) in bands
// of group_m tile rows taken column by column, so the tiles an XCD runs at once span group_m row panels of X and
// a few column panels of W instead of every column panel (a bijection: a band's last, short one included).
// (Divisions by the host's multiply-highs: four by hardware reciprocal were ~150 dependent instructions before a
// workgroup's first load, 0.5 us of a 5.6 us kernel at 256 x 768 x 768.)
__device__ __forceinline__ void tile_of(const GemmArgs &a, uint32_t b, uint32_t &tm, uint32_t &tn, uint32_t &split) {
    uint32_t L = b;
    if (a.xcd_groups > 1) { const uint32_t j = sh_div(b, a.d_xcd); L = (b - j * a.xcd_groups) * a.per_xcd + j; }
    split = a.splits > 1 ? sh_div(L, a.d_tiles) : 0u;
    const uint32_t l = L - split * (a.tiles_m * a.tiles_n);
    const uint32_t band = sh_div(l, a.d_band), first = band * a.group_m, w = l - band * a.d_band.d;
    const bool whole = first + a.group_m <= a.tiles_m;
    const ShDiv d = whole ? a.d_rows : a.d_last;
    tn = sh_div(w, d);
    tm = first + (w - tn * d.d);
}
// Host: the divisors of tile_of (tiles_m, tiles_n, splits, xcd_groups and group_m set; nblk workgroups). group_m = 1 is
// the row-major order: bands of one row.
static inline void set_tile_order(GemmArgs &a, uint32_t nblk) {
    a.per_xcd = nblk / (a.xcd_groups ? a.xcd_groups : 1);
    a.d_xcd = sh_make_div(a.xcd_groups);
    a.d_tiles = sh_make_div(a.tiles_m * a.tiles_n);
    a.d_band = sh_make_div(a.group_m * a.tiles_n);
    a.d_rows = sh_make_div(a.group_m);
    a.d_last = sh_make_div(a.tiles_m % a.group_m ? a.tiles_m % a.group_m : a.group_m);
}

__device__ __forceinline__ uint32_t swz(uint32_t r) { return (r ^ (r >> 3)) & 7u; }

__device__ __forceinline__ uint4 zero4() { return make_uint4(0, 0, 0, 0); }

__device__ __forceinline__ uint32_t comp(const uint4 &q, int i) { return i == 0 ? q.x : i == 1 ? q.y : i == 2 ? q.z : q.w; }

// The epilogue chain applied to one fp16 product value, each step rounded to fp16 exactly as the unfused
// library sequence sh_gemm -> (accumulate) -> sh_add_bias -> sh_gelu -> sh_add would store it:
// z = r16(z_old + p) [accumulate]; z = r16(z + bias); z = r16(gelu(z)); z = r16(z + residual).
__device__ __forceinline__ uint16_t epi_chain(const GemmArgs &a, uint16_t p, uint32_t gm, uint32_t gn) {
    float v = sh_dev_h2f(p);
    if (a.accumulate) v = sh_dev_h2f(sh_dev_f2h_rr(v + sh_dev_h2f(a.z[(uint64_t)gm * a.ldz + gn])));
    if (a.bias && !a.ln_stats) {
        const float b = a.bias_fp32 ? ((const float *)a.bias)[gn] : sh_dev_h2f(((const uint16_t *)a.bias)[gn]);
        v = sh_dev_h2f(sh_dev_f2h_rr(v + b));
    }
    if (a.act == SH_ACT_GELU) { const uint16_t h = sh_dev_f2h(v); v = sh_dev_h2f((uint16_t)sh_gelu_u32(h | ((uint32_t)h << 16))); }
    if (a.res) v += sh_dev_h2f(a.res[(uint64_t)gm * a.ldr + gn]);
    return sh_dev_f2h(v);
}

// The same chain on 8 consecutive columns, with z_old / bias / residual already loaded (16-byte chunks; an
// fp32 bias is b0:b1). fp16 + fp16 steps use packed fp16 adds, which round exactly like the fp32 form above.
__device__ __forceinline__ uint4 epi_chain8(const GemmArgs &a, uint4 q, const uint4 &zo, const uint4 &b0, const uint4 &b1,
                                            const uint4 &rq) {
    uint32_t w[4] = {q.x, q.y, q.z, q.w};
    if (a.accumulate) {
#pragma unroll
        for (int p = 0; p < 4; ++p) w[p] = sh_hadd2(comp(zo, p), w[p]);
    }
    if (a.bias && !a.ln_stats) {
        if (a.bias_fp32) {
#pragma unroll
            for (int p = 0; p < 4; ++p) {
                const sh_h2 h = __builtin_bit_cast(sh_h2, w[p]);
                const uint4 &bb = p < 2 ? b0 : b1;
                const float lo = (float)h.x + __uint_as_float(comp(bb, (2 * p) & 3));
                const float hi = (float)h.y + __uint_as_float(comp(bb, (2 * p + 1) & 3));
                w[p] = (uint32_t)sh_dev_f2h_rr(lo) | ((uint32_t)sh_dev_f2h_rr(hi) << 16);
            }
        } else {
#pragma unroll
            for (int p = 0; p < 4; ++p) w[p] = sh_hadd2(w[p], comp(b0, p));
        }
    }
    if (a.act == SH_ACT_GELU) {
#pragma unroll
        for (int p = 0; p < 4; ++p) w[p] = sh_gelu_u32(w[p]);
    }
    if (a.res) {
#pragma unroll
        for (int p = 0; p < 4; ++p) w[p] = sh_hadd2(w[p], comp(rq, p));
    }
    return make_uint4(w[0], w[1], w[2], w[3]);
}

template <int BN>
__device__ __forceinline__ uint32_t fw(uint32_t k) {
    return ((BN / 8) % 16 == 0) ? 4u * (k & 3u) : 4u * ((k >> 1) & 1u);
}

// ---- epilogue from registers (Z^T accumulator layout) ------------------------------------------------------
// Kernels that pass the MFMA operands swapped (first = W fragment, second = X fragment) hold every 32 x 32
// accumulator as a block of Z^T: lane l has row l % 32 of Z and columns 8 q + 4 g + e in register 4 q + e
// (q, e = 0..3, g = l / 32). One permlane32 swap per register pair hands each lane 8 consecutive columns of its
// row, which pass through the epilogue chain and leave as one 16-byte store: no LDS staging and no barrier.
// The products are the same k-ordered sums as with the operands in X, W order (the tests check every
// configuration stores the same bits). The helpers take the wavefront's position (wm, wn) in the 2 x 2 grid of
// (BM/2) x (BN/2) sub-tiles.

// x's upper 32 lanes <-> y's lower 32 lanes (v_permlane32_swap_b32).
__device__ __forceinline__ void swap_halves(uint32_t &x, uint32_t &y) {
    const auto r = __builtin_amdgcn_permlane32_swap(x, y, false, false);
    x = r[0];
    y = r[1];
}

__device__ __forceinline__ uint32_t pack_h2(float lo, float hi) {     // (fp32 values rounded to fp16 once more)
    asm volatile("" : "+v"(lo), "+v"(hi));           // (as sh_dev_f2h_rr: no conversion folded into the producer)
    return __builtin_bit_cast(uint32_t, sh_h2{(_Float16)lo, (_Float16)hi});
}

// The LayerNorm fold on a wavefront's Z^T accumulators (block (i, j) of lane l: the row of ln's entry i, columns
// ncol + 32 j + 8 q + 4 g + e in register 4 q + e), in place, before they are rounded.
template <int FM, int FN, bool OFF32 = false>
__device__ __forceinline__ void ln_fold_zt(const GemmArgs &a, sh_f16v (&acc)[FM][FN], const LnRows<FM> &ln, uint32_t ncol) {
    const int lane = threadIdx.x & 63, g = lane >> 5;
    const float *rr = ln.r, *rm = ln.rm;
    const float *d = (const float *)a.bias;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
        float cj[16], dj[16];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t n = min(ncol + 32 * j + 8 * q + 4 * g, a.N - 4);
            // (OFF32: scalar base plus a 32-bit byte offset, N < 2^24)
            const float4 c4 = OFF32 ? *(const float4 *)((const char *)a.ln_c + n * 4u) : *(const float4 *)(a.ln_c + n);
            const float4 d4 = OFF32 ? *(const float4 *)((const char *)d + n * 4u) : *(const float4 *)(d + n);
            cj[4 * q] = c4.x; cj[4 * q + 1] = c4.y; cj[4 * q + 2] = c4.z; cj[4 * q + 3] = c4.w;
            dj[4 * q] = d4.x; dj[4 * q + 1] = d4.y; dj[4 * q + 2] = d4.z; dj[4 * q + 3] = d4.w;
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][j][r] = fmaf(rr[i], acc[i][j][r], fmaf(-rm[i], cj[r], dj[r]));
    }
}

// Row partials of a wavefront's finished chunks (Z^T layout: chunk (i, j, p) of a lane is row rbase + 32 i + r32,
// columns cbase + 32 j + 16 p + 8 g): for each row and each 32-column block, the sum s of its 32 stored fp16 values
// and M2 = sum (v - s / 32)^2 (two passes in fp32; lanes g = 0, 1 hold 16 values each), written as a float2 to
// stats_out[row][block] (the consumer combines a row's blocks with ln_row). Stores the same bits in every
// register-epilogue tile (the same 32 values, the same order).
template <int FM, int FN, bool OFF32 = false>
__device__ __forceinline__ void stats_zt(const GemmArgs &a, const uint4 (&q)[FM][FN][2], uint32_t rbase, uint32_t cbase) {
    const int lane = threadIdx.x & 63, g = lane >> 5, r32 = lane & 31;
    const uint32_t P = a.N / 32;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const uint32_t row = rbase + 32 * i + r32;
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            float x[16], sum = 0.f;
#pragma unroll
            for (int p = 0; p < 2; ++p)
#pragma unroll
                for (int w = 0; w < 4; ++w) {
                    const sh_h2 h = __builtin_bit_cast(sh_h2, comp(q[i][j][p], w));
                    x[8 * p + 2 * w] = (float)h.x;
                    x[8 * p + 2 * w + 1] = (float)h.y;
                }
#pragma unroll
            for (int e = 0; e < 16; ++e) sum += x[e];
            sum += __shfl_xor(sum, 32, 64);
            const float mb = sum * (1.f / 32.f);
            float m2 = 0.f;
#pragma unroll
            for (int e = 0; e < 16; ++e) { const float d = x[e] - mb; m2 = fmaf(d, d, m2); }
            m2 += __shfl_xor(m2, 32, 64);
            const uint32_t col = cbase + 32 * j;
            if (g == 0 && row < a.M && col < a.N) {
                if constexpr (OFF32)           // (M N / 4 bytes of partials < 4 GiB: the launch checks it)
                    *(float2 *)((char *)a.stats_out + (__umul24(row, P) + col / 32) * 8u) = make_float2(sum, m2);
                else
                    ((float2 *)a.stats_out)[(uint64_t)row * P + col / 32] = make_float2(sum, m2);
            }
        }
    }
}

// 8 consecutive fp16 products of row block i, column block j, half p of one lane, in the Z^T layout above.
// Both 16-byte chunks (p = 0, 1) of the 32 x 32 block come out of the same four swaps.
template <int FM, int FN>
__device__ __forceinline__ void zt_chunks(const sh_f16v (&acc)[FM][FN], int i, int j, uint4 (&q)[2]) {
    uint32_t P[4][2];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        P[u][0] = pack_h2(acc[i][j][4 * u], acc[i][j][4 * u + 1]);
        P[u][1] = pack_h2(acc[i][j][4 * u + 2], acc[i][j][4 * u + 3]);
    }
#pragma unroll
    for (int p = 0; p < 2; ++p) {
        swap_halves(P[2 * p][0], P[2 * p + 1][0]);
        swap_halves(P[2 * p][1], P[2 * p + 1][1]);
        q[p] = make_uint4(P[2 * p][0], P[2 * p][1], P[2 * p + 1][0], P[2 * p + 1][1]);
    }
}

// The epilogue chain on a tile's chunks in place (q from zt_chunks of every block; chunk (i, j, p) of a lane is
// row m0 + wm TM + 32 i + r32, columns n0 + wn TN + 32 j + 16 p + 8 g). Converting every accumulator first
// halves the registers the epilogue holds. For the common chains (fp16 or no bias, optional residual) every
// operand load of the tile is issued in one batch, so the epilogue waits for one memory latency.
template <int BM, int BN, int FM, int FN>
__device__ __forceinline__ void chain_chunks(const GemmArgs &a, uint4 (&q)[FM][FN][2], uint32_t m0, uint32_t n0, int wm, int wn) {
    constexpr int TM = BM / 2, TN = BN / 2;
    const int lane = threadIdx.x & 63, g = lane >> 5, r32 = lane & 31;
    if (!a.accumulate && (!a.bias || a.ln_stats) && !a.res && a.act == SH_ACT_NONE) return;
    if (!a.accumulate && (!(a.bias && a.bias_fp32) || a.ln_stats)) {
        uint4 bq[FN][2];
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t gn = n0 + wn * TN + 32 * j + 16 * p + 8 * g, gc = min(gn, a.N - 8);
                bq[j][p] = (a.bias && !a.ln_stats) ? *(const uint4 *)((const uint16_t *)a.bias + gc) : zero4();
            }
        uint4 rq[FM][FN][2];
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const uint32_t gm = m0 + wm * TM + 32 * i + r32;
            const uint64_t rowr = (uint64_t)min(gm, a.M - 1) * a.ldr;
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    const uint32_t gn = n0 + wn * TN + 32 * j + 16 * p + 8 * g, gc = min(gn, a.N - 8);
                    rq[i][j][p] = a.res ? *(const uint4 *)(a.res + rowr + gc) : zero4();
                }
        }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j)
#pragma unroll
                for (int p = 0; p < 2; ++p) q[i][j][p] = epi_chain8(a, q[i][j][p], zero4(), bq[j][p], zero4(), rq[i][j][p]);
        return;
    }
    // z_old (accumulate) or a 32-byte fp32 bias per chunk: one (row block, column block) at a time
#pragma unroll
    for (int i = 0; i < FM; ++i) {
        const uint32_t gm = m0 + wm * TM + 32 * i + r32;
        const uint32_t gmc = min(gm, a.M - 1);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
            uint4 zo[2], b0[2], b1[2], rq[2];
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t gn = n0 + wn * TN + 32 * j + 16 * p + 8 * g, gc = min(gn, a.N - 8);
                zo[p] = a.accumulate ? *(const uint4 *)(a.z + (uint64_t)gmc * a.ldz + gc) : zero4();
                if (a.bias && a.bias_fp32) {
                    b0[p] = *(const uint4 *)((const float *)a.bias + gc);
                    b1[p] = *(const uint4 *)((const float *)a.bias + gc + 4);
                } else {
                    b0[p] = a.bias ? *(const uint4 *)((const uint16_t *)a.bias + gc) : zero4();
                    b1[p] = zero4();
                }
                rq[p] = a.res ? *(const uint4 *)(a.res + (uint64_t)gmc * a.ldr + gc) : zero4();
            }
#pragma unroll
            for (int p = 0; p < 2; ++p) q[i][j][p] = epi_chain8(a, q[i][j][p], zo[p], b0[p], b1[p], rq[p]);
        }
    }
}

// Store a finished tile's chunks (origin m0, n0).
template <int BM, int BN, int FM, int FN>
__device__ __forceinline__ void store_all(const GemmArgs &a, const uint4 (&q)[FM][FN][2], uint32_t m0, uint32_t n0, int wm, int wn) {
    constexpr int TM = BM / 2, TN = BN / 2;
    const int lane = threadIdx.x & 63, g = lane >> 5, r32 = lane & 31;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t gm = m0 + wm * TM + 32 * i + r32, gn = n0 + wn * TN + 32 * j + 16 * p + 8 * g;
                if (gm < a.M && gn < a.N) *(uint4 *)(a.z + (uint64_t)gm * a.ldz + gn) = q[i][j][p];
            }
}

}  // namespace
