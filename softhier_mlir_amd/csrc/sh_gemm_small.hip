// GEMM kernels for problems that do not fill the chip with the tile table's workgroups, and for operands without
// 16-byte alignment (sh_gemm.hip decides which calls come here: small_plan).
//
// What bounds such a product is latency: at M = 256 a 64 x 64 tiling of a 768-wide layer is 48 workgroups, each a chain
// of k-slices that waits for memory two slices at a time. Here R slices of 64 k per workgroup or wavefront are requested
// ahead into registers (plain 16-byte loads: one wavefront moves 25 B/clk with them, 11 with
// global -> LDS DMA, whose issue takes a wavefront ~90 cycles each; measured on resident data), tiles go down to 32 x 32
// so that every CU has work, each slice is written to LDS once its loads have landed, and the fragments of slice kt are
// read while the MFMAs of the one before run. The epilogue's operands are loaded before the k-loop.
// As compiled, only the R = 4 build (64 x 64) keeps loads in flight through a wait (its waits stop at vmcnt 8). In the R = 2
// builds the waits before the first of two slices' LDS writes go down to vmcnt 0 (14, 12, ... 0 for 32 x 32, 22 ... 0 for 64 x 32,
// 5 ... 0 for 128 x 64), so both slices land together and a memory latency is exposed every 128 k.
// The products are summed in the order of the direct-to-LDS kernels (16-k blocks in sequence through one MFMA chain per
// output; with K ranges, which only a call with splits = 0 or two equal ranges gets, the ranges' sums added in range order), so
// they store those kernels' bits.
#include "sh_gemm_dev.h"
#include "sh_gemm_small.h"
#include <type_traits>
#include <utility>

namespace {

template <bool EDGE>
__device__ __forceinline__ uint4 ld16(const uint16_t *p) {
    if constexpr (EDGE) return sh_ld16_any(p);
    else return *(const uint4 *)p;
}

// W slice swizzle ([K, N] layout): as fw, but a 32-column row (4 chunks) needs none (4 rows span the banks).
template <int BN>
__device__ __forceinline__ uint32_t fws(uint32_t k) { return BN == 32 ? 0u : fw<BN>(k); }

template <typename F, int... I>
__device__ __forceinline__ void unroll_impl(F &f, std::integer_sequence<int, I...>) { (f(std::integral_constant<int, I>{}), ...); }
template <int N, typename F>
__device__ __forceinline__ void unroll(F &&f) { unroll_impl(f, std::make_integer_sequence<int, N>{}); }

// One BM x BN tile per workgroup.
//  - KS = false: four wavefronts load the slices together into two LDS stages (one barrier per slice), each computes FM
//    32 x 32 blocks of Z^T.
//  - KS = true: wavefront s computes K range s of the whole tile from a stage of its own, without a barrier, and wavefront 0
//    adds the ranges' fp32 sums in range order. A single wavefront issues an LDS read or a 16-byte load only every ~35-40
//    cycles, so at these sizes the ranges' parallel instruction streams are what shortens the kernel.
// MODE: ALIGNED: 16-byte operands and K % 64 == 0; ALIGNED_FOLD: the same with the LayerNorm fold (its own build: the
// rows' partials and the c / d rows take ~60 registers); ANY_ALIGN: operands, leading dims, N and K of any alignment
// (ldx, ldw >= 8 and tensors of at least 8 elements: small_plan); the chunks of the last slice that would reach past the
// tensor's last element are loaded from its end and shifted. WT: W given as [N, K].
enum { ALIGNED = 0, ALIGNED_FOLD = 1, ANY_ALIGN = 2 };
template <int BM, int BN, int FM, int R, bool WT, int MODE, bool KS>
__global__ __launch_bounds__(KS && FM == 1 ? 512 : 256, KS ? 1 : 2) void k_gemm_small(GemmArgs a) {
    constexpr bool EDGE = MODE == ANY_ALIGN, FOLD = MODE == ALIGNED_FOLD;
    constexpr int NTH = KS ? 64 : 256;                     // threads that load one slice
    constexpr int WGM = BM / (32 * FM), WGN = BN / 32, CW = WGM * WGN, TM = 32 * FM;
    constexpr int XR = BM * 8 / NTH, WR = BN * 8 / NTH;    // 16-byte chunks per thread per slice
    constexpr int XCH = BM * 8, STAGE = (BM + BN) * 8;     // chunks per stage: X then W
    constexpr int WCPR = BN / 8;                           // chunks per W row ([K, N] layout)
    static_assert(!KS || FM * 4 * 64 <= STAGE, "a range's sums fit in its stage");
    static_assert(R % 2 == 0 && FM <= 2 && CW == (KS ? 1 : 4) && BM * 8 % NTH == 0 && BN * 8 % NTH == 0, "tile");
    extern __shared__ uint4 smem[];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int t = KS ? lane : (int)threadIdx.x;
    const int g = lane >> 5, r32 = lane & 31, q4 = lane >> 4, iq = lane & 15;
    const int wm = KS ? 0 : wave / WGN, wn = KS ? 0 : wave % WGN;

    // (the launch pads the fast grid dimension to whole XCD rounds: a workgroup past its tiles has nothing to do)
    const uint32_t tm = a.group_m ? blockIdx.x : blockIdx.y, tn = a.group_m ? blockIdx.y : blockIdx.x;
    if (tm >= a.tiles_m || tn >= a.tiles_n) return;
    const uint32_t m0 = tm * BM, n0 = tn * BN;
    const uint32_t kbeg = KS ? wave * a.kps : 0u, kend = KS ? min(a.K, kbeg + a.kps) : a.K;
    const int KT = kend > kbeg ? (int)((kend - kbeg + BK - 1) / BK) : 0;
    const uint32_t rem = EDGE && KT > 0 ? (kend - kbeg) - (uint32_t)(KT - 1) * BK : BK;     // (aligned: K % 64 == 0)

    // Addresses: a wave-uniform base per operand and slice plus each lane's 32-bit byte offset of its chunk (the launch
    // checks the leading dims). xo / wo: any slice but the last; xl / wl: the last one, from a base 16 bytes lower, where a
    // chunk (or row) past kend is replaced by the first one and, with EDGE, a chunk that would reach past the tensor's last
    // element is loaded from its end (sh halves before its own place); nv: its valid halves.
    const char *const xb = (const char *)(a.x + (uint64_t)m0 * a.ldx + kbeg);
    const char *const wb = WT ? (const char *)(a.w + (uint64_t)n0 * a.ldw + kbeg) : (const char *)(a.w + (uint64_t)kbeg * a.ldw + n0);
    const uint64_t xadv = BK * 2, wadv = WT ? (uint64_t)BK * 2 : (uint64_t)BK * a.ldw * 2;
    const char *const xbl = xb + (uint64_t)max(KT - 1, 0) * xadv - 16, *const wbl = wb + (uint64_t)max(KT - 1, 0) * wadv - 16;
    auto k_valid = [&](uint32_t c8) -> uint32_t { return (uint32_t)min(max((int)rem - 8 * (int)c8, 0), 8); };
    auto clamp_end = [&](const char *base, uint32_t off, const uint16_t *last8, uint32_t &sh) -> uint32_t {
        sh = 0;
        if constexpr (EDGE) {
            const char *p = base + off;
            if (p > (const char *)last8) { sh = (uint32_t)(p - (const char *)last8) / 2; off -= 2 * sh; }
        }
        return off;
    };
    auto last_x = [&](int r, uint32_t &sh, uint32_t &nv) -> uint32_t {
        const uint32_t c = t + NTH * r, m = min(m0 + (c >> 3), a.M - 1) - m0;
        nv = k_valid(c & 7);
        return clamp_end(xbl, 16 + (m * (uint32_t)a.ldx + (nv ? 8 * (c & 7) : 0u)) * 2, a.x + (uint64_t)(a.M - 1) * a.ldx + a.K - 8, sh);
    };
    auto last_w = [&](int r, uint32_t &sh, uint32_t &nv) -> uint32_t {
        const uint32_t c = t + NTH * r;
        if constexpr (WT) {
            const uint32_t n = min(n0 + (c >> 3), a.N - 1) - n0;
            nv = k_valid(c & 7);
            return clamp_end(wbl, 16 + (n * (uint32_t)a.ldw + (nv ? 8 * (c & 7) : 0u)) * 2, a.w + (uint64_t)(a.N - 1) * a.ldw + a.K - 8, sh);
        } else {
            const uint32_t k = c / WCPR, n = min(n0 + 8 * (c % WCPR), EDGE ? a.N - 1 : a.N - 8) - n0;
            nv = k < rem ? 8u : 0u;
            return clamp_end(wbl, 16 + ((nv ? k : 0u) * (uint32_t)a.ldw + n) * 2, a.w + (uint64_t)(a.K - 1) * a.ldw + a.N - 8, sh);
        }
    };
    uint32_t xo[XR], xl[XR], wo[WR], wl[WR];
#pragma unroll
    for (int r = 0; r < XR; ++r) {
        const uint32_t c = t + NTH * r;
        uint32_t sh, nv;
        xo[r] = (__umul24(min(m0 + (c >> 3), a.M - 1) - m0, (uint32_t)a.ldx) + 8 * (c & 7)) * 2;
        xl[r] = EDGE ? last_x(r, sh, nv) : xo[r];
    }
#pragma unroll
    for (int r = 0; r < WR; ++r) {
        const uint32_t c = t + NTH * r;
        uint32_t sh, nv;
        if constexpr (WT) wo[r] = (__umul24(min(n0 + (c >> 3), a.N - 1) - n0, (uint32_t)a.ldw) + 8 * (c & 7)) * 2;
        else wo[r] = (__umul24(c / WCPR, (uint32_t)a.ldw) + min(n0 + 8 * (c % WCPR), EDGE ? a.N - 1 : a.N - 8) - n0) * 2;
        wl[r] = EDGE ? last_w(r, sh, nv) : wo[r];
    }
    // Slice kt into register set u. Always the same number of loads: a slice past the end re-reads the last one (a few
    // cached lines).
    uint4 rx[R][XR], rw[R][WR];
    auto gload = [&](int kt, auto uc) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        const int src = min(kt, KT - 1);
        const bool last = EDGE && src == KT - 1;
        const char *xp = last ? xbl : xb + (uint64_t)src * xadv, *wp = last ? wbl : wb + (uint64_t)src * wadv;
#pragma unroll
        for (int r = 0; r < XR; ++r) rx[u][r] = ld16<EDGE>((const uint16_t *)(xp + (last ? xl[r] : xo[r])));
#pragma unroll
        for (int r = 0; r < WR; ++r) rw[u][r] = ld16<EDGE>((const uint16_t *)(wp + (last ? wl[r] : wo[r])));
    };
    uint4 *const mine = KS ? smem + wave * STAGE : smem;
    auto sstore = [&](int kt, auto uc) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value;
        uint4 *st = mine + (KS ? 0 : (u & 1) * STAGE);
        if (EDGE && kt == KT - 1) {
            uint32_t sh, nv;
#pragma unroll
            for (int r = 0; r < XR; ++r) { (void)last_x(r, sh, nv); rx[u][r] = sh_fix8(rx[u][r], sh, nv); }
#pragma unroll
            for (int r = 0; r < WR; ++r) { (void)last_w(r, sh, nv); rw[u][r] = sh_fix8(rw[u][r], sh, nv); }
        }
#pragma unroll
        for (int r = 0; r < XR; ++r) {
            const uint32_t c = t + NTH * r, m = c >> 3;
            st[m * 8 + ((c & 7) ^ swz(m))] = rx[u][r];
        }
#pragma unroll
        for (int r = 0; r < WR; ++r) {
            const uint32_t c = t + NTH * r;
            if constexpr (WT) { const uint32_t n = c >> 3; st[XCH + n * 8 + ((c & 7) ^ swz(n))] = rw[u][r]; }
            else { const uint32_t k = c / WCPR; st[XCH + k * WCPR + ((c % WCPR) ^ fws<BN>(k))] = rw[u][r]; }
        }
    };

    // Fragments of NSB 16-k substeps, two sets: set `b` of stage so. While one set's reads are under way the MFMAs of the
    // set before it run. A set is a whole slice, or half of one where the registers are short.
    constexpr int NSB = FM > 1 || KS ? 2 : 4, NPH = 4 / NSB;
    sh_h8 xf[2][NSB][FM], wf[2][NSB];
    const uint32_t lds0 = sh_lds_addr(mine);
    auto frags = [&](auto soc, auto phc, auto bc) __attribute__((always_inline)) {
        constexpr int so = decltype(soc)::value, ph = decltype(phc)::value, b = decltype(bc)::value;
        const uint4 *st = mine + so;
#pragma unroll
        for (int q = 0; q < NSB; ++q) {
            const int s = ph * NSB + q;
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const uint32_t m = (uint32_t)(wm * TM + 32 * i + r32);
                xf[b][q][i] = __builtin_bit_cast(sh_h8, st[m * 8 + ((2 * s + g) ^ swz(m))]);
            }
            if constexpr (WT) {
                const uint32_t n = (uint32_t)(wn * 32 + r32);
                wf[b][q] = __builtin_bit_cast(sh_h8, st[XCH + n * 8 + ((2 * s + g) ^ swz(n))]);
            } else {
                const uint32_t n = (uint32_t)(wn * 32 + 16 * (q4 & 1) + 4 * (iq & 3)), k0 = 16 * s + 8 * g + (iq >> 2), k1 = k0 + 4;
                const uint32_t wb = lds0 + (so + XCH) * 16;
                const sh_s4 lo = sh_ds_read_tr(wb + k0 * (BN * 2) + 16 * ((n >> 3) ^ fws<BN>(k0)) + 2 * (n & 7));
                const sh_s4 hi = sh_ds_read_tr(wb + k1 * (BN * 2) + 16 * ((n >> 3) ^ fws<BN>(k1)) + 2 * (n & 7));
                wf[b][q] = __builtin_bit_cast(sh_h8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
            }
        }
    };
    sh_f16v acc[FM][1];
#pragma unroll
    for (int i = 0; i < FM; ++i) acc[i][0] = sh_f16v{};
    auto mfmas = [&](auto bc) __attribute__((always_inline)) {
        constexpr int b = decltype(bc)::value;
#pragma unroll
        for (int q = 0; q < NSB; ++q)
#pragma unroll
            for (int i = 0; i < FM; ++i) acc[i][0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(wf[b][q], xf[b][q][i], acc[i][0], 0, 0, 0);
    };

    __builtin_amdgcn_sched_barrier(0);
    if (KT > 0) unroll<R>([&](auto uc) __attribute__((always_inline)) { gload(decltype(uc)::value, uc); });
    __builtin_amdgcn_sched_barrier(0);
    // The epilogue's operands, requested behind the first slices: c and d of the LayerNorm fold and its rows' factors, the
    // fp16 bias, z_old and the residual (chunk (i, p) of a lane: row m0 + wm TM + 32 i + r32, columns ncol + 16 p + 8 g).
    const bool fin = !KS || wave == 0;                      // this wavefront finishes (and stores) a block
    const uint32_t mrow = m0 + wm * TM, ncol = n0 + wn * 32;
    float4 c4[4], d4[4];
    uint4 bq[2] = {zero4(), zero4()}, zo[FM][2], rq[FM][2];
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int p = 0; p < 2; ++p) { zo[i][p] = zero4(); rq[i][p] = zero4(); }
    const bool bias16 = !FOLD && a.bias && !a.bias_fp32;
    auto col_ok = [&](int p) -> bool { return ncol + 16 * p + 8 * g + 8 <= a.N; };     // (EDGE: a whole chunk)
    LnPair lnl[FM];
    if (fin) {
        if constexpr (FOLD) {
#pragma unroll
            for (int i = 0; i < FM; ++i) ln_pair_load(a, min(mrow + 32 * i + r32, a.M - 1), lnl[i]);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t n = min(ncol + 8 * q + 4 * g, a.N - 4);
                c4[q] = *(const float4 *)(a.ln_c + n);
                d4[q] = *(const float4 *)((const float *)a.bias + n);
            }
        }
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            if (EDGE && !col_ok(p)) continue;               // (a ragged last chunk goes element by element below)
            const uint32_t gc = EDGE ? ncol + 16 * p + 8 * g : min(ncol + 16 * p + 8 * g, a.N - 8);
            if (bias16) bq[p] = ld16<EDGE>((const uint16_t *)a.bias + gc);
#pragma unroll
            for (int i = 0; i < FM; ++i) {
                const uint32_t gm = min(mrow + 32 * i + r32, a.M - 1);
                if (!FOLD && a.accumulate) zo[i][p] = ld16<EDGE>(a.z + (uint64_t)gm * a.ldz + gc);
                if (a.res) rq[i][p] = ld16<EDGE>(a.res + (uint64_t)gm * a.ldr + gc);
            }
        }
    }
    __builtin_amdgcn_sched_barrier(0);

    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int q = 0; q < NSB; ++q) {                         // before slice 0: zeros (acc stays +0)
        wf[1][q] = sh_h8{};
#pragma unroll
        for (int i = 0; i < FM; ++i) xf[1][q][i] = sh_h8{};
    }
    // Step kt: the fragment reads of slice kt, the LDS writes of slice kt + 1 and the MFMAs of slice kt - 1 are under way
    // together; one barrier ends the step (slice kt + 1 is in its stage, and every wavefront has slice kt in registers, so
    // its stage is free). KS: one wavefront's LDS instructions execute in order, so a single stage and no barrier do.
    auto step = [&](int kt, auto uc, auto more) __attribute__((always_inline)) {
        constexpr int u = decltype(uc)::value, un = (u + 1) % R;
        unroll<NPH>([&](auto phc) __attribute__((always_inline)) {
            constexpr int ph = decltype(phc)::value, b = NPH == 1 ? u & 1 : ph;
            frags(std::integral_constant<int, KS ? 0 : (u & 1) * STAGE>{}, phc, std::integral_constant<int, b>{});
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ph == NPH - 1) {
                if (decltype(more)::value || kt + 1 < KT) sstore(kt + 1, std::integral_constant<int, un>{});
                __builtin_amdgcn_sched_barrier(0);
                if constexpr (decltype(more)::value) gload(kt + 1 + R, std::integral_constant<int, un>{});
                __builtin_amdgcn_sched_barrier(0);
            }
            mfmas(std::integral_constant<int, b ^ 1>{});
            __builtin_amdgcn_sched_barrier(0);
        });
        asm volatile("" ::: "memory");
        if constexpr (!KS) {
            sh_wait_lgkm0();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    int kt0 = 0;
    if (KT > 0) {
        sstore(0, std::integral_constant<int, 0>{});
        gload(R, std::integral_constant<int, 0>{});
        asm volatile("" ::: "memory");
        if constexpr (!KS) {
            sh_wait_lgkm0();
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
        }
        __builtin_amdgcn_sched_barrier(0);
    }
    for (; kt0 + R < KT; kt0 += R)
        unroll<R>([&](auto uc) __attribute__((always_inline)) { step(kt0 + decltype(uc)::value, uc, std::true_type{}); });
    unroll<R>([&](auto uc) __attribute__((always_inline)) {
        if (kt0 + decltype(uc)::value < KT) step(kt0 + decltype(uc)::value, uc, std::false_type{});
    });
    if (KT > 0) {
        if (NPH > 1 || ((KT - 1) & 1)) mfmas(std::integral_constant<int, 1>{});
        else mfmas(std::integral_constant<int, 0>{});
    }
    float lnr[FM], lnrm[FM];                                // r and r mu of rows mrow + 32 i + r32
    if (FOLD && fin) {
#pragma unroll
        for (int i = 0; i < FM; ++i) {
            const float2 st = ln_pair_form(a, min(mrow + 32 * i + r32, a.M - 1), lnl[i]);
            lnr[i] = st.y;
            lnrm[i] = st.x * st.y;
        }
    }
    if constexpr (KS) {                                     // the ranges' sums, added in range order from 0
        float4 *park = (float4 *)mine;
        if (wave > 0) {
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    park[(4 * i + e) * 64 + lane] = make_float4(acc[i][0][4 * e], acc[i][0][4 * e + 1], acc[i][0][4 * e + 2], acc[i][0][4 * e + 3]);
        }
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[i][0][r] += 0.f;
        for (uint32_t s = 1; s < blockDim.x / 64; ++s) {
            const float4 *p = (const float4 *)(smem + s * STAGE);
#pragma unroll
            for (int i = 0; i < FM; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float4 v = p[(4 * i + e) * 64 + lane];
                    acc[i][0][4 * e] += v.x; acc[i][0][4 * e + 1] += v.y; acc[i][0][4 * e + 2] += v.z; acc[i][0][4 * e + 3] += v.w;
                }
        }
    }

    if constexpr (FOLD) {                                   // (the expressions of ln_fold_zt)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float cc[4] = {c4[q].x, c4[q].y, c4[q].z, c4[q].w}, dd[4] = {d4[q].x, d4[q].y, d4[q].z, d4[q].w};
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[i][0][4 * q + e] = fmaf(lnr[i], acc[i][0][4 * q + e], fmaf(-lnrm[i], cc[e], dd[e]));
            }
    }
    uint4 qc[FM][1][2];
#pragma unroll
    for (int i = 0; i < FM; ++i) zt_chunks<FM, 1>(acc, i, 0, qc[i][0]);
    if constexpr (EDGE) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int p = 0; p < 2; ++p) {
                const uint32_t gm = mrow + 32 * i + r32, gn = ncol + 16 * p + 8 * g;
                if (gm >= a.M || gn >= a.N) continue;
                uint16_t *z = a.z + (uint64_t)gm * a.ldz + gn;
                if (col_ok(p)) {
                    uint4 b0 = bq[p], b1 = zero4();
                    if (a.bias && a.bias_fp32) {
                        b0 = ld16<true>((const uint16_t *)((const float *)a.bias + gn));
                        b1 = ld16<true>((const uint16_t *)((const float *)a.bias + gn + 4));
                    }
                    const uint4 v = epi_chain8(a, qc[i][0][p], zo[i][p], b0, b1, rq[i][p]);
                    sh_st8_any(z, v, 8);
                } else {
#pragma unroll
                    for (int e = 0; e < 8; ++e)
                        if (gn + e < a.N) z[e] = epi_chain(a, (uint16_t)(comp(qc[i][0][p], e >> 1) >> (16 * (e & 1))), gm, gn + e);
                }
            }
    } else {
#pragma unroll
        for (int p = 0; p < 2; ++p) {
            uint4 b0 = bq[p], b1 = zero4();
            if (!FOLD && a.bias && a.bias_fp32) {
                const float *b = (const float *)a.bias + min(ncol + 16 * p + 8 * g, a.N - 8);
                b0 = *(const uint4 *)b;
                b1 = *(const uint4 *)(b + 4);
            }
#pragma unroll
            for (int i = 0; i < FM; ++i) qc[i][0][p] = epi_chain8(a, qc[i][0][p], zo[i][p], b0, b1, rq[i][p]);
        }
        if (a.stats_out) stats_zt<FM, 1>(a, qc, mrow, ncol);
        store_all<2 * TM, 64, FM, 1>(a, qc, m0, n0, wm, wn);
    }
}

}  // namespace

void sh_gemm_small_enqueue(const GemmArgs &a, SmallTile v, bool wt, bool any, uint32_t ranges, hipStream_t st) {
    typedef void (*Fn)(GemmArgs);
    // [tile][WT][mode]; the 64-row range tile has no fold build (registers), the shared tiles only serve ANY_ALIGN
    static const Fn fns[SMALL_ANY_TILES][2][3] = {
        {{k_gemm_small<32, 32, 1, 2, false, ALIGNED, true>, k_gemm_small<32, 32, 1, 2, false, ALIGNED_FOLD, true>, k_gemm_small<32, 32, 1, 2, false, ANY_ALIGN, true>},
         {k_gemm_small<32, 32, 1, 2, true, ALIGNED, true>, k_gemm_small<32, 32, 1, 2, true, ALIGNED_FOLD, true>, k_gemm_small<32, 32, 1, 2, true, ANY_ALIGN, true>}},
        {{k_gemm_small<64, 32, 2, 2, false, ALIGNED, true>, nullptr, k_gemm_small<64, 32, 2, 2, false, ANY_ALIGN, true>},
         {k_gemm_small<64, 32, 2, 2, true, ALIGNED, true>, nullptr, k_gemm_small<64, 32, 2, 2, true, ANY_ALIGN, true>}},
        {{nullptr, nullptr, k_gemm_small<64, 64, 1, 4, false, ANY_ALIGN, false>}, {nullptr, nullptr, k_gemm_small<64, 64, 1, 4, true, ANY_ALIGN, false>}},
        {{nullptr, nullptr, k_gemm_small<128, 64, 2, 2, false, ANY_ALIGN, false>}, {nullptr, nullptr, k_gemm_small<128, 64, 2, 2, true, ANY_ALIGN, false>}},
    };
    const bool ks = v == SMALL_RANGES_32 || v == SMALL_RANGES_64;
    const uint32_t stage = (kSmallDims[v].bm + kSmallDims[v].bn) * BK * 2;
    const uint32_t threads = ks ? 64 * ranges : 256, lds = ks ? ranges * stage : 2 * stage;
    const Fn fn = fns[v][wt][any || !ks ? ANY_ALIGN : a.ln_stats ? ALIGNED_FOLD : ALIGNED];
    // The fast grid dimension runs over the larger operand's tiles, in whole rounds of the XCDs (dispatch deals workgroups
    // round-robin over them): each of its panels is then read by one XCD's L2 only.
    GemmArgs g = a;
    g.group_m = a.M > a.N;
    uint32_t fast = g.group_m ? a.tiles_m : a.tiles_n;
    const uint32_t slow = g.group_m ? a.tiles_n : a.tiles_m, X = (uint32_t)sh_num_xcds();
    if (X > 1 && fast >= X) fast = sh_cdiv(fast, X) * X;
    hipLaunchKernelGGL(fn, dim3(fast, slow), dim3(threads), lds, st, g);
}
