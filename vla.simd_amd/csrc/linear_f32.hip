// linear_f32.hip - fp32 linear layers on the matrix cores (gfx950).
//
// out[m, n] (+)= act(sum_k x[m, k] * W[n, k] + bias[n])
//
// The layers the reference keeps in fp32 around the int8 path go through this
// kernel: Linear::Role::Generic (dense_linear, src/hal/common/gemm.cpp) and the
// Gemm-role layers a model leaves out of its int8 mask - ACT's state_proj and
// action head (src/models/act/act_transformer.cpp:127-128), Octo's token
// projections outside OCTO_INT8 bit 8 (src/models/octo/octo_transformer.cpp:60-62),
// SmolVLA's flow-matching projections (src/models/smolvla/action_expert.cpp:196-211).
// fp32 results differ from the reference's only by summation order.
//
// More than 128 rows take linear_f32_tiled (two fp16 parts of every operand on
// the fp16 matrix cores); up to 128 rows, and few tiles over a long K without a
// workspace, linear_f32_skinny on v_mfma_f32_16x16x4f32: lane l supplies A[row
// l % 16][k l / 16] and B[col l % 16][k l / 16]; output lane l holds column
// l % 16, rows 4 * (l / 16) + r.

#include "act.h"
#include "common.h"
#include "fp16parts.h"
#include "wave.h"

#include <cstdlib>

#pragma clang fp contract(off)

namespace vla {
namespace hip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

// max over the N = 8 or 16 lanes that hold a row
template <int N>
__device__ __forceinline__ float lanes_max(float v) {
    v = fmaxf(v, dpp_f32<0xb1, 0xf>(v, v));    // quad_perm [1,0,3,2]
    v = fmaxf(v, dpp_f32<0x4e, 0xf>(v, v));    // quad_perm [2,3,0,1]
    v = fmaxf(v, dpp_f32<0x141, 0xf>(v, v));   // row_half_mirror
    return N == 8 ? v : fmaxf(v, dpp_f32<0x140, 0xf>(v, v));  // row_mirror
}

// Block barrier that orders LDS only: __syncthreads' release fence would also
// wait for the global loads of the slab after next.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

__device__ __forceinline__ float act_of(float v, int act) {
    switch (act) {
    case 1: return act_relu(v);
    case 2: return act_gelu_tanh(v);
    case 3: return act_gelu_erf(v);
    case 4: return act_silu(v);
    default: return v;
    }
}

// The tiled form for M > 128 (the conv GEMMs of ACT's fp32 backbone and Octo's
// stems, the fp32 projections) on the fp16 matrix cores: x W^T from the products
// hh, hm and mh of the operands' two parts. Three v_mfma_f32_16x16x32_f16 take
// 48 cycles of a SIMD where eight v_mfma_f32_16x16x4f32 take 256, and their
// fp32 sums round once per 32 terms: against 64 bits the results are closer
// (2-norm, N(0, 1) rows, K = 768: 3.6e-7 against 5.8e-7).
//
// Every row of x and of W has a scale of its own, a power of two taken out of
// the sums exactly (both at once and by the exponent: the product of the two
// need not be a float). It is guessed from the row's values in one slab (the first;
// a convolution's centre tap, which always lies inside the image), so that they
// reach 2^6, or from the tile's where the row has none; the maxima of all
// slabs are kept, and a tile some row of which ends up outside [2^3, 2^15] is
// computed once more with the scales of the true maxima. So no part overflows
// and an operand loses no more than 2^-22 of itself or 2^-28 of its row's largest
// value. (Hence a row's last bits can depend on the other rows of its tile.)
// Infinities are left to plain fmaf chains. Aimed at 2^12, a channel at 30 times the
// others took the second pass: 690 x 768 x 3072 44.8 us against 27.1, 177 x 960 x 960
// 16.9 against 10.0; at 2^6 rows 512 times their slab's maximum still do, at less
// than twice the time.
//
// BM x BN tiles, four waves in a 2 x 2 grid. A K slab, KS steps of 32, is loaded as
// float4 runs (whole 128-byte row segments per 8 lanes, 256 per 16 with KS = 2) into registers while
// the slab before it computes, and split once per block on its way to LDS:
// [part][k step][row][32 k] with the 16-byte chunks of a row permuted by its number, so
// the 16 rows of one fragment read fall on distinct banks. The weights are the
// first operand: a lane then holds four consecutive output columns.
// CONV: x is an NHWC map and row m of A is output pixel m's k x k patch,
// column (ky * k + kx) * Cin + ci (im2col's order), gathered by the A loads
// themselves: with Cin % 32 == 0 a thread's float4 of a slab always lies in
// one tap, and its tap advances by the slab's channels. Same scales and
// products in the same order as im2col + this kernel; no column matrix.
// VEC: rows are 16-byte aligned runs; otherwise elements are loaded one by one.
// resid (a block's skip map, rows as out's): out = relu(v + resid), the pass
// that would read both again.
// G = 2: two groups of four waves take half of the block's K slabs each, with
// slabs, scales and sums of their own; the sums meet in LDS and each group
// finishes half of the tile. Twice the waves where the tiles alone leave a CU
// one block (4800 x 1152 x 128 21.6 -> 18.3 us).
template <int BM, int BN, int KS, int G, bool CONV, bool VEC>
__global__ __launch_bounds__(256 * G) void linear_f32_tiled(float* __restrict__ out, int ldo,
                                                        const float* __restrict__ x, int ldx,
                                                        const float* __restrict__ W, int ldw,
                                                        const float* __restrict__ bias, int M, int N,
                                                        int K, int act, int accumulate, float alpha,
                                                        ConvGeom cg, int gcol, int gn,
                                                        const float* __restrict__ resid,
                                                        float* __restrict__ part, int kchunk) {
    constexpr int BK = 32 * KS, LR = 8 * KS, ROWS = BM + BN;  // LR lanes hold a row of a slab
    constexpr int TM = BM / 2, TN = BN / 2, FM = TM / 16, FN = TN / 16;
    constexpr int AV = BM * BK / 4 / 256, BV = BN * BK / 4 / 256;  // float4 loads per thread
    static_assert(AV >= 1 && BV >= 1 && TM % 16 == 0 && TN % 16 == 0 && FM % G == 0, "tile");
    __shared__ __attribute__((aligned(16))) char smem[G][2][2][KS][ROWS * 64];
    __shared__ int units[G][ROWS];  // the power of two a row's sums are multiplied by in the end
    __shared__ uint32_t guesses[G][2];  // the tile's largest value of x and of W in the guess slab
    const int grp = G == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 8);
    auto& sm = smem[grp];
    auto& unit = units[grp];
    auto& guess = guesses[grp];
    const int tid = G == 1 ? threadIdx.x : threadIdx.x & 255, lane = tid & 63, wave = tid >> 6;
    const int wm = wave >> 1, wn = wave & 1;
    const int m0 = blockIdx.y * BM, n0 = blockIdx.x * BN;
    // split K (part != null): chunk blockIdx.z of kchunk columns, raw sums into
    // its slice of part; K becomes the chunk's length
    const int kblk = part ? blockIdx.z * kchunk : 0;
    if (part) K = K - kblk < kchunk ? K - kblk : kchunk;
    const int kall = K;  // the block's columns; from here on kbeg, K: the group's
    const int nk = ((K + BK - 1) / BK + G - 1) / G;
    const int kbeg = G > 1 ? kblk + grp * nk * BK : kblk;
    if constexpr (G > 1) K = K - grp * nk * BK < nk * BK ? K - grp * nk * BK : nk * BK;  // (0 or less: no columns)

    // float4 v of a slab: row v / LR, k 4 (v % LR); rows past the matrix clamped
    const float* ap[AV];
    const float* bp[BV];
    int iy0[AV], ix0[AV];  // CONV: the patch origin of each loaded row
#pragma unroll
    for (int j = 0; j < AV; j++) {
        const int v = tid + 256 * j, r = v / LR, k = (v % LR) * 4;
        const int m = m0 + r < M ? m0 + r : M - 1;
        if (CONV) {
            const int oy = m / cg.Wout, ox = m - oy * cg.Wout;
            iy0[j] = oy * cg.stride - cg.pad;
            ix0[j] = ox * cg.stride - cg.pad;
            ap[j] = x;
        } else {
            ap[j] = x + (size_t)m * ldx + kbeg + k;
        }
    }
#pragma unroll
    for (int j = 0; j < BV; j++) {
        const int v = tid + 256 * j, r = v / LR, k = (v % LR) * 4;
        const int n = n0 + r < N ? n0 + r : N - 1;
        bp[j] = W + (size_t)n * ldw + kbeg + k;
    }
    const int kq = (tid % LR) * 4;  // this thread's k offset within a slab (same for every load)
    float4 ra[AV], rb[BV];
    auto ld4 = [&](const float* p, int k) {
        if (VEC && k + 4 <= K) return *reinterpret_cast<const float4*>(p);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k < K) v.x = p[0];
        if (k + 1 < K) v.y = p[1];
        if (k + 2 < K) v.z = p[2];
        if (k + 3 < K) v.w = p[3];
        return v;
    };
    // CONV: the tap of this thread's next A slab (kbeg is a multiple of 32)
    int ci, kx, ky;
    auto first_tap = [&] {
        const int t = (kbeg + kq) / cg.Cin;
        ci = kbeg + kq - t * cg.Cin;
        ky = t / cg.k;
        kx = t - ky * cg.k;
    };
    auto gload = [&](int k0) {
        const bool whole = VEC && k0 + BK <= K;  // wave-uniform: no lane meets the end of a row
        if (CONV) {  // called for k0 = 0, BK, 2 BK, ... in order
#pragma unroll
            for (int j = 0; j < AV; j++) {
                const int iy = iy0[j] + ky, ix = ix0[j] + kx;
                ra[j] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (iy >= 0 && iy < cg.H && ix >= 0 && ix < cg.Wd && ((KS == 1 && G == 1) || k0 + kq < K))
                    ra[j] = *reinterpret_cast<const float4*>(x + ((size_t)iy * cg.Wd + ix) * cg.Cin + ci);
            }
            ci += BK;
            while (ci >= cg.Cin) {  // (once, but for KS * 32 channels past a tap of 32)
                ci -= cg.Cin;
                if (++kx == cg.k) {
                    kx = 0;
                    ++ky;
                }
            }
        } else if (whole) {
#pragma unroll
            for (int j = 0; j < AV; j++) ra[j] = *reinterpret_cast<const float4*>(ap[j] + k0);
        } else {
#pragma unroll
            for (int j = 0; j < AV; j++) ra[j] = ld4(ap[j] + k0, k0 + kq);
        }
        if (whole) {
#pragma unroll
            for (int j = 0; j < BV; j++) rb[j] = *reinterpret_cast<const float4*>(bp[j] + k0);
        } else {
#pragma unroll
            for (int j = 0; j < BV; j++) rb[j] = ld4(bp[j] + k0, k0 + kq);
        }
    };
    float ma[AV], mb[BV];       // this thread's part of its rows' maxima
    uint32_t ea[AV], eb[BV];    // the rows' scales (biased exponents)
    // row r's 16-byte chunk q lies at chunk q ^ (-(r / 4) % 4): rows that share
    // banks (4 apart) take different chunks, in the 16 lanes 0-3, 12-15, 20-23
    // and 24-27 (and their like) that a ds_read_b128 serves at once
    auto at = [](int r, int q) { return r * 64 + ((q ^ -(r >> 2)) & 3) * 16; };
    auto lstore = [&](int buf) {
        const int ks = (tid % LR) >> 3, q = (tid & 7) >> 1, half = (tid & 1) * 8;
        auto put = [&](int r, const float4& v, uint32_t e) {
            const float s = exp_float(e);
            uint2 h, m;
            split2(v.x * s, v.y * s, h.x, m.x);
            split2(v.z * s, v.w * s, h.y, m.y);
            const int o = at(r, q) + half;
            *reinterpret_cast<uint2*>(&sm[buf][0][ks][o]) = h;
            *reinterpret_cast<uint2*>(&sm[buf][1][ks][o]) = m;
        };
#pragma unroll
        for (int j = 0; j < AV; j++) {
            ma[j] = absmax4(ma[j], ra[j]);
            put((tid + 256 * j) / LR, ra[j], ea[j]);
        }
#pragma unroll
        for (int j = 0; j < BV; j++) {
            mb[j] = absmax4(mb[j], rb[j]);
            put(BM + (tid + 256 * j) / LR, rb[j], eb[j]);
        }
    };

    v4f acc[FM][FN];
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
    const int r16 = lane & 15, g = lane >> 4;
    auto compute = [&](int buf) {
#pragma unroll
        for (int ks = 0; ks < KS; ks++) {
            f16x8 af[FM][2], bf[FN][2];
#pragma unroll
            for (int p = 0; p < 2; p++) {
#pragma unroll
                for (int i = 0; i < FM; i++)
                    af[i][p] = *reinterpret_cast<const f16x8*>(&sm[buf][p][ks][at(wm * TM + i * 16 + r16, g)]);
#pragma unroll
                for (int j = 0; j < FN; j++)
                    bf[j][p] = *reinterpret_cast<const f16x8*>(&sm[buf][p][ks][at(BM + wn * TN + j * 16 + r16, g)]);
            }
            auto mul = [&](int pa, int pb) {
#pragma unroll
                for (int i = 0; i < FM; i++)
#pragma unroll
                    for (int j = 0; j < FN; j++)
                        acc[i][j] =
                            __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[j][pb], af[i][pa], acc[i][j], 0, 0, 0);
            };
            mul(0, 1);
            mul(1, 0);
            mul(0, 0);
        }
    };

    // the guess: rows' maxima in the first slab, x's of a convolution from the
    // centre tap: the map's pixel, or im2col's columns gcol .. gcol + gn - 1 (the
    // same values, so both forms take the same scales)
    if (tid < 2) guess[tid] = 0;
    const bool tap = CONV || (VEC && gn > 0);
    if (CONV) first_tap();
    if (tap) {
#pragma unroll
        for (int j = 0; j < AV; j++) {
            const float* p = nullptr;
            if (CONV) {
                const int t = min(cg.pad, cg.k - 1), o = guess_offset(cg, iy0[j] + t, ix0[j] + t, kq);
                if (o >= 0) p = x + o;
            } else if (kq < gn) {
                p = ap[j] - kbeg + gcol;
            }
            ma[j] = absmax4(0.0f, p ? *reinterpret_cast<const float4*>(p) : make_float4(0.f, 0.f, 0.f, 0.f));
        }
    }
    gload(0);
#pragma unroll
    for (int j = 0; j < AV; j++) ma[j] = lanes_max<LR>(tap ? ma[j] : absmax4(0.0f, ra[j]));
#pragma unroll
    for (int j = 0; j < BV; j++) mb[j] = lanes_max<LR>(absmax4(0.0f, rb[j]));
    bool none = false;  // a row without values in the guess slab takes the tile's guess
#pragma unroll
    for (int j = 0; j < AV; j++) none = none || ma[j] == 0.0f;
#pragma unroll
    for (int j = 0; j < BV; j++) none = none || mb[j] == 0.0f;
    if (__syncthreads_or(none)) {
        float ta = 0.0f, tb = 0.0f;
#pragma unroll
        for (int j = 0; j < AV; j++) ta = fmaxf(ta, ma[j]);
#pragma unroll
        for (int j = 0; j < BV; j++) tb = fmaxf(tb, mb[j]);
        ta = wave_max_f32(ta);
        tb = wave_max_f32(tb);
        if (lane == 0) {  // floats >= 0 order as their bits
            atomicMax(&guess[0], __float_as_uint(ta));
            atomicMax(&guess[1], __float_as_uint(tb));
        }
        __syncthreads();
#pragma unroll
        for (int j = 0; j < AV; j++) ma[j] = ma[j] > 0.0f ? ma[j] : __uint_as_float(guess[0]);
#pragma unroll
        for (int j = 0; j < BV; j++) mb[j] = mb[j] > 0.0f ? mb[j] : __uint_as_float(guess[1]);
    }
#pragma unroll
    for (int j = 0; j < AV; j++) ea[j] = scale_exp(ma[j], 6);
#pragma unroll
    for (int j = 0; j < BV; j++) eb[j] = scale_exp(mb[j], 6);

    bool again = false, bad;
    for (;;) {
#pragma unroll
        for (int j = 0; j < AV; j++) ma[j] = 0.0f;
#pragma unroll
        for (int j = 0; j < BV; j++) mb[j] = 0.0f;
        lstore(0);
        if (nk > 1) gload(BK);
        lds_barrier();
        for (int kt = 0; kt < nk; kt++) {
            const int buf = kt & 1;
            compute(buf);
            if (kt + 1 < nk) {
                lstore(buf ^ 1);  // slab kt + 1, loaded during this compute
                if (kt + 2 < nk) gload((kt + 2) * BK);
            }
            lds_barrier();
        }
        // the rows' true maxima under the scales used; what the sums are
        // multiplied by, for the epilogue
        bool off = false, inf = false;
        auto check = [&](float& mx, uint32_t e, int r) {
            mx = lanes_max<LR>(mx);
            const float t = mx * exp_float(e);
            off = off || !(mx == 0.0f || (t >= 8.0f && t <= 32768.0f));
            inf = inf || !(mx <= 3.4028235e38f);
            if (tid % LR == 0) unit[r] = 127 - (int)e;
        };
#pragma unroll
        for (int j = 0; j < AV; j++) check(ma[j], ea[j], (tid + 256 * j) / LR);
#pragma unroll
        for (int j = 0; j < BV; j++) check(mb[j], eb[j], BM + (tid + 256 * j) / LR);
        // a second pass can only find values that are not finite, or rows so
        // small that 2^126 leaves them below 2^3
        bad = __syncthreads_or(again ? inf : off);
        if (!bad || again) break;
        again = true;
#pragma unroll
        for (int j = 0; j < AV; j++) ea[j] = scale_exp(ma[j], 14);
#pragma unroll
        for (int j = 0; j < BV; j++) eb[j] = scale_exp(mb[j], 14);
#pragma unroll
        for (int i = 0; i < FM; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) acc[i][j] = v4f{0.f, 0.f, 0.f, 0.f};
        if (CONV) first_tap();
        gload(0);
    }

    float* dst = part ? part + (size_t)blockIdx.z * M * N : out;
    const int ldd = part ? N : ldo;
    if (bad) {  // one fmaf chain per output; its speed does not matter
        for (int e = threadIdx.x; e < BM * BN; e += 256 * G) {
            const int m = m0 + e / BN, n = n0 + e % BN;
            if (m >= M || n >= N) continue;
            const float* wr = W + (size_t)n * ldw + kblk;
            float v = 0.0f;
            if (CONV) {
                const int oy = m / cg.Wout, ox = m - oy * cg.Wout;
                for (int k = 0; k < kall; k++) {
                    const int t = (kblk + k) / cg.Cin, c = kblk + k - t * cg.Cin;
                    const int iy = oy * cg.stride - cg.pad + t / cg.k, ix = ox * cg.stride - cg.pad + t % cg.k;
                    const bool in = iy >= 0 && iy < cg.H && ix >= 0 && ix < cg.Wd;
                    v = fmaf(in ? x[((size_t)iy * cg.Wd + ix) * cg.Cin + c] : 0.0f, wr[k], v);
                }
            } else {
                const float* xr = x + (size_t)m * ldx + kblk;
                for (int k = 0; k < kall; k++) v = fmaf(xr[k], wr[k], v);
            }
            float* o = dst + (size_t)m * ldd + n;
            if (!part) v = act_of(v + (bias ? bias[n] : 0.0f), act);
            if (resid && !part) v = relu_gt(v + resid[(size_t)m * ldd + n]);
            *o = !part && accumulate ? fmaf(alpha, v, *o) : v;
        }
        return;
    }

    // the groups' sums of the tile: group g finishes fragment rows g FM / G ..
    constexpr int FG = FM / G;
    if constexpr (G == 2) {
        // (the barrier of `bad` lies after the last read of the slabs)
        v4f* mine = reinterpret_cast<v4f*>(&smem[grp][0][0][0][0]) + tid;
        const v4f* other = reinterpret_cast<const v4f*>(&smem[grp ^ 1][0][0][0][0]) + tid;
#pragma unroll
        for (int i = 0; i < FG; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
                v4f v = grp ? acc[i][j] : acc[FG + i][j];  // the other group's half
                const int ua = unit[wm * TM + (grp ? i : FG + i) * 16 + r16];
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = ldexpf(v[r], ua + unit[BM + wn * TN + j * 16 + 4 * g + r]);
                mine[(i * FN + j) * 256] = v;
            }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < FG; i++)
#pragma unroll
            for (int j = 0; j < FN; j++) {
                v4f v = grp ? acc[FG + i][j] : acc[i][j];
                const int ua = unit[wm * TM + (grp ? FG + i : i) * 16 + r16];
#pragma unroll
                for (int r = 0; r < 4; r++) v[r] = ldexpf(v[r], ua + unit[BM + wn * TN + j * 16 + 4 * g + r]);
                acc[i][j] = v + other[(i * FN + j) * 256];
            }
    }

    // lane: row m = r16 of a fragment, columns n = 4 g .. 4 g + 3
    const bool vec = (ldd & 3) == 0 && (reinterpret_cast<uintptr_t>(dst) & 15) == 0;
    const bool rvec = (ldd & 3) == 0 && (reinterpret_cast<uintptr_t>(resid) & 15) == 0;
#pragma unroll
    for (int j = 0; j < FN; j++) {
        const int n = n0 + wn * TN + j * 16 + 4 * g;
        if (n >= N) continue;
        float b[4] = {0.f, 0.f, 0.f, 0.f};
        if (bias && !part)
            for (int r = 0; r < 4; r++)
                if (n + r < N) b[r] = bias[n + r];
#pragma unroll
        for (int i = 0; i < FG; i++) {
            const int fr = wm * TM + (grp * FG + i) * 16 + r16, m = m0 + fr;
            if (m >= M) continue;
            float* o = dst + (size_t)m * ldd + n;
            const int ua = unit[fr];
            float v[4];
#pragma unroll
            for (int r = 0; r < 4; r++) {
                v[r] = G > 1 ? acc[i][j][r] : ldexpf(acc[i][j][r], ua + unit[BM + wn * TN + j * 16 + 4 * g + r]);
                if (!part) v[r] = act_of(v[r] + b[r], act);
            }
            if (resid && !part) {
                const float* q = resid + (size_t)m * ldd + n;
                if (rvec && n + 4 <= N) {
                    const float4 d = *reinterpret_cast<const float4*>(q);
                    v[0] = relu_gt(v[0] + d.x);
                    v[1] = relu_gt(v[1] + d.y);
                    v[2] = relu_gt(v[2] + d.z);
                    v[3] = relu_gt(v[3] + d.w);
                } else {
                    for (int r = 0; r < 4; r++)
                        if (n + r < N) v[r] = relu_gt(v[r] + q[r]);
                }
            }
            if (vec && n + 4 <= N) {
                if (!part && accumulate) {
                    const float4 d = *reinterpret_cast<const float4*>(o);
                    v[0] = fmaf(alpha, v[0], d.x);
                    v[1] = fmaf(alpha, v[1], d.y);
                    v[2] = fmaf(alpha, v[2], d.z);
                    v[3] = fmaf(alpha, v[3], d.w);
                }
                *reinterpret_cast<float4*>(o) = make_float4(v[0], v[1], v[2], v[3]);
            } else {
                for (int r = 0; r < 4 && n + r < N; r++) o[r] = !part && accumulate ? fmaf(alpha, v[r], o[r]) : v[r];
            }
        }
    }
}

// M <= 128 (the batch-1 action heads and flow-matching projections): a block
// owns 16 output columns and every row; its W waves split K in 16-wide steps
// and stream both operands from global memory as float4 runs. A step's 16 rows
// of 64 bytes are loaded four neighbouring lanes to a row and cross to the
// matrix operand's order (row l % 16, k 4 (l / 16) ..) through the wave's own
// LDS: loaded in that order, each lane of a quad on another row, the address
// unit takes a cycle per lane and a CU pulls 14.7 bytes per clock instead of
// 40. 100 x 512 x 3200 13.5 -> 9.7 us, 128 x 768 x 3072 20.4 -> 14.3,
// 1 x 960 x 2560 4.7 -> 4.1; what is left is the fp32 MFMAs (3 us of the first)
// after the fill (2.7). Lane group g takes k = 4g .. 4g+3 of a step; A and B use
// the same k order, so each MFMA sums matching products. The waves' partial sums
// meet in LDS before the epilogue.
template <int FM, int W, bool VEC>
__global__ __launch_bounds__(W * 64) void linear_f32_skinny(float* __restrict__ out, int ldo,
                                                            const float* __restrict__ x, int ldx,
                                                            const float* __restrict__ Wt, int ldw,
                                                            const float* __restrict__ bias, int M,
                                                            int N, int K, int act, int accumulate,
                                                            float alpha) {
    __shared__ __attribute__((aligned(16))) float red[W * (FM + 1) * 256];
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n0 = blockIdx.x * 16, mb = blockIdx.y * 16 * FM;  // row tile blockIdx.y of 16 * FM rows
    const int lr = lane >> 2, lk = 4 * (lane & 3);              // the row and k of a step this lane loads
    const float* brow = Wt + (size_t)min(n0 + lr, N - 1) * ldw;
    const float* arow[FM];
#pragma unroll
    for (int i = 0; i < FM; i++) arow[i] = x + (size_t)min(mb + 16 * i + lr, M - 1) * ldx;
    auto load4 = [&](const float* row, int k) {
        if (VEC && k + 4 <= K) return *reinterpret_cast<const float4*>(row + k);
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (k < K) v.x = row[k];
        if (k + 1 < K) v.y = row[k + 1];
        if (k + 2 < K) v.z = row[k + 2];
        if (k + 3 < K) v.w = row[k + 3];
        return v;
    };
    // a fragment's 64 chunks in LDS: row r's chunk q at 4 r + (q ^ (-(r / 4) % 4)),
    // distinct banks for the 16 lanes an access serves at once
    auto slot = [](int r, int q) { return 4 * r + ((q ^ -(r >> 2)) & 3); };
    float4* tr = reinterpret_cast<float4*>(red) + wave * (FM + 1) * 64;
    const int put = slot(lr, lane & 3), get = slot(lane & 15, lane >> 4);
    v4f acc[FM];
#pragma unroll
    for (int i = 0; i < FM; i++) acc[i] = v4f{0.f, 0.f, 0.f, 0.f};
    // P of the wave's K steps per round: all their loads are issued before the
    // first MFMA (one wait per round instead of one per step); the MFMAs run
    // in the same step order, so the sums are the same
    constexpr int P = FM <= 4 ? 4 : 2;
    for (int k16r = wave * 16; k16r < K; k16r += P * W * 16) {
        float4 b[P], a[P][FM];
#pragma unroll
        for (int p = 0; p < P; p++) {
            const int k16 = k16r + p * W * 16;
            if (k16 < K) {  // wave-uniform
                const int k = k16 + lk;
                b[p] = load4(brow, k);
#pragma unroll
                for (int i = 0; i < FM; i++) a[p][i] = load4(arow[i], k);
            }
        }
#pragma unroll
        for (int p = 0; p < P; p++) {
            if (k16r + p * W * 16 < K) {
                // a wave's LDS accesses run in order: the compiler must keep it
                asm volatile("" ::: "memory");
                tr[put] = b[p];
#pragma unroll
                for (int i = 0; i < FM; i++) tr[64 * (i + 1) + put] = a[p][i];
                asm volatile("" ::: "memory");
                const float4 bv = tr[get];
#pragma unroll
                for (int i = 0; i < FM; i++) {
                    const float4 av = tr[64 * (i + 1) + get];
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.x, bv.x, acc[i], 0, 0, 0);
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.y, bv.y, acc[i], 0, 0, 0);
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.z, bv.z, acc[i], 0, 0, 0);
                    acc[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(av.w, bv.w, acc[i], 0, 0, 0);
                }
            }
        }
    }
    __syncthreads();  // the partial sums take the fragments' place
#pragma unroll
    for (int i = 0; i < FM; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) red[((wave * FM + i) * 4 + r) * 64 + lane] = acc[i][r];
    __syncthreads();
    // thread e sums element e of the FM x 4 x 64 lane-major tile over the waves
    for (int e = tid; e < FM * 256; e += W * 64) {
        float v = 0.0f;
#pragma unroll
        for (int w = 0; w < W; w++) v += red[w * FM * 256 + e];
        const int l = e & 63, r = (e >> 6) & 3, i = e >> 8;
        const int m = mb + 16 * i + 4 * (l >> 4) + r, nn = n0 + (l & 15);
        if (m >= M || nn >= N) continue;
        v = act_of(v + (bias ? bias[nn] : 0.0f), act);
        float* o = out + (size_t)m * ldo + nn;
        *o = accumulate ? fmaf(alpha, v, *o) : v;
    }
}

template <int FM, bool VEC>
void launch_skinny_fm(float* out, int ldo, const float* x, int ldx, const float* W, int ldw,
                      const float* bias, int M, int N, int K, int act, int accumulate, float alpha,
                      hipStream_t st) {
    const int steps = (K + 15) / 16;
    // row groups of 16 * FM rows (grid.y): as the int8 skinny GEMM, the fewest
    // that give every CU a block; each output's sum is unchanged
    const dim3 blocks((N + 15) / 16, (M + 16 * FM - 1) / (16 * FM));
    // about four K steps per wave, at most 8 waves
    const int w = steps >= 32 ? 8 : steps >= 16 ? 4 : steps >= 8 ? 2 : 1;
    switch (w) {
    case 8: linear_f32_skinny<FM, 8, VEC><<<blocks, 512, 0, st>>>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha); break;
    case 4: linear_f32_skinny<FM, 4, VEC><<<blocks, 256, 0, st>>>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha); break;
    case 2: linear_f32_skinny<FM, 2, VEC><<<blocks, 128, 0, st>>>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha); break;
    default: linear_f32_skinny<FM, 1, VEC><<<blocks, 64, 0, st>>>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha); break;
    }
}

template <bool VEC>
void launch_skinny(float* out, int ldo, const float* x, int ldx, const float* W, int ldw,
                   const float* bias, int M, int N, int K, int act, int accumulate, float alpha,
                   hipStream_t st) {
    const int nfrag = (M + 15) / 16, nb = (N + 15) / 16;
    int g = (256 + nb - 1) / nb;  // 256 CUs
    if (const char* e = std::getenv("VLA_HIP_SKINNY_R")) g = *e ? std::atoi(e) : g;
    g = g < 1 ? 1 : g > nfrag ? nfrag : g;
    switch ((nfrag + g - 1) / g) {
    case 1: launch_skinny_fm<1, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    case 2: launch_skinny_fm<2, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    case 3: launch_skinny_fm<3, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    case 4: launch_skinny_fm<4, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    case 5: launch_skinny_fm<5, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    case 6: launch_skinny_fm<6, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    case 7: launch_skinny_fm<7, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    default: launch_skinny_fm<8, VEC>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st); break;
    }
}

// The split-K partial sums of linear_f32_tiled: out = act(sum_z part[z] + bias)
// with the chunks added in z order, then the epilogue of the unsplit kernel.
__global__ __launch_bounds__(256) void linear_f32_split_reduce(float* __restrict__ out, int ldo,
                                                               const float* __restrict__ part, int S, int M, int N,
                                                               const float* __restrict__ bias, int act,
                                                               int accumulate, float alpha,
                                                               const float* __restrict__ resid) {
    const int64_t MN = (int64_t)M * N;
    for (int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; e < MN; e += (int64_t)gridDim.x * blockDim.x) {
        float v = part[e];
        for (int z = 1; z < S; z++) v += part[z * MN + e];
        const int m = (int)(e / N), n = (int)(e - (int64_t)m * N);
        v = act_of(v + (bias ? bias[n] : 0.0f), act);
        if (resid) v = relu_gt(v + resid[(size_t)m * ldo + n]);
        float* o = out + (size_t)m * ldo + n;
        *o = accumulate ? fmaf(alpha, v, *o) : v;
    }
}

constexpr int kCUs = 256;  // MI355X compute units

struct F32Call {
    float* out;
    int ldo;
    const float* x;
    int ldx;
    const float* W;
    int ldw;
    const float* bias;
    int M, N, K, act, accumulate;
    float alpha;
    ConvGeom cg;
    const float* resid = nullptr;
    int gcol = 0, gn = 0;  // the columns of x that a row's scale is guessed from (gn 0: the first slab's)
};

// Split-K plan for M > 128 over K >= 1024 when 64 x 64 tiles number < 128
// (ResNet's last stages): S chunks of K (multiples of 32, >= 256) so that
// S x tiles reaches about two blocks per CU, S <= 8.
struct F32Split {
    int S = 1, kchunk = 0;
};
F32Split f32_split_plan(int M, int N, int K) {
    F32Split p;
    const long t64 = (long)((M + 63) / 64) * ((N + 63) / 64);
    if (M <= 128 || t64 >= 128 || K < 1024) return p;
    int S = (int)((2 * kCUs + t64 - 1) / t64);
    S = S < 8 ? S : 8;
    int kc = ((K + S - 1) / S + 31) / 32 * 32;
    kc = kc > 256 ? kc : 256;
    p.S = (K + kc - 1) / kc;
    p.kchunk = kc;
    if (p.S < 2) p = F32Split{};
    return p;
}

template <int BM, int BN, int KS, int G, bool CONV, bool VEC>
void launch_tile(const F32Call& c, float* part, int S, int kchunk, hipStream_t st) {
    const dim3 grid((c.N + BN - 1) / BN, (c.M + BM - 1) / BM, S);
    linear_f32_tiled<BM, BN, KS, G, CONV, VEC><<<grid, 256 * G, 0, st>>>(c.out, c.ldo, c.x, c.ldx, c.W, c.ldw, c.bias, c.M, c.N,
                                                              c.K, c.act, c.accumulate, c.alpha, c.cg, c.gcol, c.gn,
                                                                     c.resid, part, kchunk);
    VLA_LAUNCH_CHECK();
}

// The largest tile that still gives the CUs enough waves: a group's slabs are a
// serial chain of LDS round trips, splitting and products, and two or three
// groups on a CU fill each other's gaps. From two blocks of 64 x 64 per CU those
// are blocks; from half a block per CU, two groups of one block that share its
// K; below, 32 x 32 tiles, with 64-wide slabs, half the round trips (177 x 960 x
// 960 17.5 -> 13.1 us); on the larger ones the second step costs residency (690
// x 768 x 3072 on 64 x 64 29.0 -> 39.6). Measured, us (fp32 matrix cores | 32 x
// 32, 64 x 64, 64 x 64 by two groups, 128 x 64):
// 690 x 768 x 3072 64.5 | 39.3 28.6 30.8 32; 1024 x 768 x 3072 64.1 | 49.3 30.9 33.6 34;
// 2048 x 2048 x 2048 156 | 140 89.8 90.6 80.7; 19200 x 576 x 64 29.2 | 22.8 19.2 17.5 23;
// 4800 x 1152 x 128 33.3 | 21.4 26.2 18.3 34; 690 x 768 x 768 23.8 | 14.2 19.4 13.9 26;
// 690 x 3072 x 768 78 | 42.6 57.2 37.0; 302 x 512 x 3200 18.8 | 14.7 16.0 12.5;
// 256 x 768 x 512 (32 blocks of 64 x 64) 9.6 | 8.9 16.2 12.3; 177 x 960 x 960 (45) 14.3 | 13.0 21.9 15.2.
template <bool CONV, bool VEC>
void launch_tiles(const F32Call& c, hipStream_t st) {
    auto blocks = [&](int bm, int bn) { return (long)((c.M + bm - 1) / bm) * ((c.N + bn - 1) / bn); };
    if (blocks(128, 64) >= 2 * kCUs) launch_tile<128, 64, 1, 1, CONV, VEC>(c, nullptr, 1, 0, st);
    else if (blocks(64, 64) >= 2 * kCUs) launch_tile<64, 64, 1, 1, CONV, VEC>(c, nullptr, 1, 0, st);
    else if (2 * blocks(64, 64) >= kCUs) launch_tile<64, 64, 1, 2, CONV, VEC>(c, nullptr, 1, 0, st);
    else launch_tile<32, 32, 2, 1, CONV, VEC>(c, nullptr, 1, 0, st);
}

// Shapes whose 32 x 32 tiles leave CUs idle while each walks a long K.
bool few_tiles(int M, int N, int K) { return K >= 1024 && (long)((M + 31) / 32) * ((N + 31) / 32) < kCUs; }

void launch_f32_split(const F32Call& c, bool conv, const F32Split& p, float* part, hipStream_t st) {
    if (conv) launch_tile<64, 64, 1, 1, true, true>(c, part, p.S, p.kchunk, st);
    else launch_tile<64, 64, 1, 1, false, true>(c, part, p.S, p.kchunk, st);
    const int64_t MN = (int64_t)c.M * c.N;
    const int blocks = (int)((MN + 255) / 256 < 4096 ? (MN + 255) / 256 : 4096);
    linear_f32_split_reduce<<<blocks, 256, 0, st>>>(c.out, c.ldo, part, p.S, c.M, c.N, c.bias, c.act, c.accumulate,
                                                    c.alpha, c.resid);
    VLA_LAUNCH_CHECK();
}

}  // namespace

size_t linear_f32_split_floats(int M, int N, int K) {
    const F32Split p = f32_split_plan(M, N, K);
    return p.S > 1 ? (size_t)p.S * M * N : 0;
}

void launch_linear_f32(float* out, int ldo, const float* x, int ldx, const float* W, int ldw,
                       const float* bias, int M, int N, int K, int act, int accumulate, float alpha,
                       hipStream_t st, float* work, size_t work_floats, bool taps, const ConvGeom* cols) {
    VLA_REQUIRE(M >= 0 && N > 0 && K > 0, "linear_f32: need M >= 0, N > 0, K > 0");
    VLA_REQUIRE((ldx >= K || (taps && ldx > 0)) && ldw >= K && ldo >= N,
                "linear_f32: row strides shorter than the rows");
    VLA_REQUIRE(out && x && W, "linear_f32: null buffer");
    VLA_REQUIRE(act >= 0 && act <= 4, "linear_f32: unknown activation");
    if (M == 0) return;
    if (M <= 128) {
        const bool vec = ldx % 4 == 0 && ldw % 4 == 0 && aligned(x, 16) && aligned(W, 16);
        if (vec) launch_skinny<true>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st);
        else launch_skinny<false>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, st);
        VLA_LAUNCH_CHECK();
        return;
    }
    F32Call c{out, ldo, x, ldx, W, ldw, bias, M, N, K, act, accumulate, alpha, ConvGeom{}};
    if (cols && cols->Cin % 32 == 0) {  // as the implicit form guesses (which takes no other widths)
        const int t = cols->pad < cols->k ? cols->pad : cols->k - 1;
        c.gcol = (t * cols->k + t) * cols->Cin;
        c.gn = cols->Cin;
        VLA_REQUIRE(c.gcol + c.gn <= K, "linear_f32: the columns are not these patches'");
    }
    const bool vec = ldx % 4 == 0 && ldw % 4 == 0 && aligned(x, 16) && aligned(W, 16);
    if (!vec) {
        launch_tiles<false, false>(c, st);
        return;
    }
    const F32Split sp = f32_split_plan(M, N, K);
    if (sp.S > 1 && work && work_floats >= (size_t)sp.S * M * N && aligned(work, 16)) {
        // few tiles over a long K with a workspace: 64 x 64 tiles split over K
        launch_f32_split(c, false, sp, work, st);
        return;
    }
    if (few_tiles(M, N, K)) {
        // few tiles over a long K (ResNet's last stages): the split-K form,
        // 64-row x 16-column blocks whose 8 waves share K, so the chain of
        // dependent loads per wave is an eighth of K (300 x 4608 x 512, 160
        // tiles of 32 x 32, 35.6 us against 43.3 in tiles; 177 x 2560 x 960, 180
        // tiles, 21.7 against 26.3; 500 x 2048 x 448, 224, 18.2 against 22.1; near
        // even at 302 x 2048 x 768, 240, 17.5 and 17.1; at 1200 x 2304 x 256, 304, the
        // tiles are ahead, 26.7 against 35.0)
        const dim3 grid((N + 15) / 16, (M + 63) / 64);
        linear_f32_skinny<4, 8, true><<<grid, 512, 0, st>>>(out, ldo, x, ldx, W, ldw, bias, M, N, K, act,
                                                             accumulate, alpha);
        VLA_LAUNCH_CHECK();
        return;
    }
    launch_tiles<false, true>(c, st);
}

bool launch_conv_f32_implicit(float* out, const float* x, int H, int Wd, int Cin, int k, int stride, int pad,
                              int Hout, int Wout, const float* W, const float* bias, int Cout, int act,
                              hipStream_t st, float* work, size_t work_floats, const float* resid) {
    const char* e = std::getenv("VLA_CONV_F32_IMPLICIT");  // 0: im2col + GEMM (A/B runs)
    if (e && e[0] == '0' && e[1] == '\0') return false;
    VLA_REQUIRE(out && x && W && H > 0 && Wd > 0 && Cin > 0 && k > 0 && stride > 0 && pad >= 0 && Cout > 0 &&
                    Hout > 0 && Wout > 0 && act >= 0 && act <= 4,
                "conv_f32: bad arguments");
    const int64_t K64 = (int64_t)k * k * Cin, M64 = (int64_t)Hout * Wout;
    // the output pixels' patches stay inside the padded input
    VLA_REQUIRE((int64_t)(Hout - 1) * stride + k <= (int64_t)H + 2 * pad &&
                    (int64_t)(Wout - 1) * stride + k <= (int64_t)Wd + 2 * pad,
                "conv_f32: output larger than the padded input allows");
    if (Cin % 32 || K64 > INT32_MAX || M64 > INT32_MAX || (int64_t)H * Wd * Cin > INT32_MAX) return false;
    if (!aligned(x, 16) || !aligned(W, 16)) return false;
    const int M = (int)M64, K = (int)K64, N = Cout;
    if (M <= 128) return false;
    const ConvGeom cg{H, Wd, Cin, k, stride, pad, Wout};
    const F32Split sp = f32_split_plan(M, N, K);
    const F32Call c{out, N, x, K, W, K, bias, M, N, K, act, 0, 1.0f, cg, resid};
    if (sp.S > 1) {  // as launch_linear_f32: split over K with a workspace, else not here
        if (!(work && work_floats >= (size_t)sp.S * M * N && aligned(work, 16))) return false;
        launch_f32_split(c, true, sp, work, st);
        return true;
    }
    if (few_tiles(M, N, K)) return false;  // the skinny route of launch_linear_f32
    launch_tiles<true, true>(c, st);
    return true;
}

}  // namespace hip
}  // namespace vla
