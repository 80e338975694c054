// attn.hip - fused masked GQA attention (QK^T -> online softmax -> PV) on gfx950.
//
// Semantics are the reference's gqa_attention_masked (src/ops/lm_ops.h:33;
// scalar reference src/hal/scalar/attn.cpp:22-87, AVX2 engine
// src/hal/avx2/attn.cpp:266-447):
//   score = (q . k) * scale + mask;  a key whose mask entry is lowest() or whose
//   score is -inf gets weight exactly 0;  out = sum_j softmax_j * v_j;  a row
//   with every key blocked is the uniform mean of V over all seq_k keys
//   (attn_uniform_row, avx2/attn.cpp:45-52).
// fp32 operands, sums and softmax; results are tolerance-class against the
// reference (its exp is a Cephes polynomial, its sums run in another order).
//
// Two kernels: attn_split (below, head_dim <= 128) forms both products from
// two fp16 parts of the fp32 values, 22 bits of each, attn_fwd from the values
// themselves on the fp32 matrix cores; it keeps head_dim 129 to 256 and the calls
// the split form does not take (scales that are not finite, strides or lengths past
// its offsets).
//
// attn_fwd: a block owns 16 queries of one head; its W waves split the key range: wave w
// takes key tiles w, w + W, ... (KT keys each), stages each tile in its own
// LDS region (no block barrier in the main loop) and keeps its own online
// softmax state; at the end the waves merge their (max, sum, output) through
// LDS. Small problems (the batch-1 action chunks) thereby still occupy many
// waves, and large ones get W-fold more waves than query tiles.
// Both products run on the fp32 matrix cores (v_mfma_f32_16x16x4_f32, one
// float per lane per operand):
//   S^T = K Q^T : A = K tile rows (keys), B = Q^T; lane l's result holds
//                 S[q = l%16][key = 16*kt + 4*(l/16) + r], r = 0..3;
//   O^T = V^T P^T: A = V^T, B = P^T. The B operand lane l must supply is
//                 P[q = l%16][key = 16*kt + 4*(l/16) + r] - exactly the value
//                 lane l already holds from S^T, so P never moves between lanes.
// The head dimension is walked as d = g*(HDP/4) + s for lane group g = l/16,
// so each lane's Q slice and each K row read are contiguous (ds_read_b128).
// LDS rows are HDP+4 floats: the 16 rows of one read land on distinct banks,
// and the four lane groups of a V read land 16 banks apart. The next tile's
// K/V rows are loaded into registers while the current tile computes.
// Scores and the running max stay in the natural domain (dot*scale + mask, as
// the reference forms them); exp(x) is evaluated as v_exp_f32(x * log2 e).

#include "common.h"
#include "fp16parts.h"
#include "wave.h"

#include <cfloat>
#include <cmath>

namespace vla {
namespace hip {
namespace {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr float kLog2e = 1.44269504088896340736f;

__device__ __forceinline__ v4f mfma_f32(float a, float b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }

// max / sum of x over the lanes l, l^16, l^32, l^48 (the four 16-lane rows of
// a wave) with gfx950's row-swap permutes, VALU ops instead of LDS round trips.
// permlane16_swap(x, x) returns, in every lane, the values of the lane pair
// {l, l^16} (one from the even row, one from the odd row); permlane32_swap the
// pair {l, l^32}. The sum adds each pair in either order, which is the same
// float: the results equal those of x op shfl_xor(x, 16), then 32.
__device__ __forceinline__ float rows_max(float x) {
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const float y = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const unsigned v = __float_as_uint(y);
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float rows_sum(float x) {
    const unsigned u = __float_as_uint(x);
    const auto a = __builtin_amdgcn_permlane16_swap(u, u, false, false);
    const float y = __uint_as_float(a[0]) + __uint_as_float(a[1]);
    const unsigned v = __float_as_uint(y);
    const auto b = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    return __uint_as_float(b[0]) + __uint_as_float(b[1]);
}

// Orders this wave's LDS accesses (its writes before other lanes' reads) with
// no block barrier.
__device__ __forceinline__ void wave_lds_sync() {
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt((15) | (3 << 14) | (7 << 4));  // lgkmcnt(0) only
    __builtin_amdgcn_wave_barrier();
    asm volatile("" ::: "memory");
}

template <int HDP, int KT, int W>
struct AttnCfg {
    static constexpr int SK = HDP + 4;               // LDS row, floats
    static constexpr int TILE = 2 * KT * SK;         // K + V of one wave, floats
    static constexpr int F4 = KT * HDP / 4 / 64;     // float4 loads per lane per K (or V) tile
    static constexpr int MO = HDP + 4;               // merge row, floats: the 16 rows of one
                                                     // float4 access fall on distinct banks
    static constexpr int MERGE = W * (32 + 16 * MO);
    static constexpr int MAIN = 4 * (W * TILE > MERGE ? W * TILE : MERGE);  // bytes
    static constexpr int ALLOW = 4096;  // group table bytes kept in LDS (n_groups <= 64)
    static constexpr int LDS = MAIN + ALLOW;
    static_assert(KT % 16 == 0 && (KT * HDP / 4) % 64 == 0, "tile shape");
};

// MKC: the mask class compiled in - 1 dense, 3 group table (per-key data
// prefetched with each tile), 0 for kinds 0 and 2 (none, causal), which read
// no per-key data.
template <int HDP, int KT, int W, int MKC>
__global__ __launch_bounds__(W * 64) void attn_fwd(AttnArgs a) {
    constexpr bool KD = MKC != 0;
    using C = AttnCfg<HDP, KT, W>;
    constexpr int SK = C::SK, F4 = C::F4;
    constexpr int NT = KT / 16;
    constexpr int QS = HDP / 4;
    constexpr int DT = HDP / 16;
    extern __shared__ __attribute__((aligned(16))) float smem[];

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = tid >> 6;
    const int g = lane >> 4, c = lane & 15;
    // XCD-aware block order for grids of at most one round (256 blocks): the
    // hardware deals workgroup i to XCD i % 8, so each XCD is given a contiguous
    // run of (head, query tile) pairs and its L2 holds the K/V rows of a few
    // heads instead of every head's. Larger grids measured slower that way;
    // they take the balanced order below.
    const int nqt = gridDim.x, total = nqt * gridDim.y;
    const int bid = blockIdx.y * nqt + blockIdx.x;
    int qt, h;
    if (total <= 256) {
        const int xcd = bid & 7, per = total >> 3, rem = total & 7;
        const int logical = xcd * per + (xcd < rem ? xcd : rem) + (bid >> 3);
        qt = logical % nqt;
        h = logical / nqt;
    } else {
        // rounds of 256 blocks put one block on every CU (block b and b + 256
        // share a CU); under causal and block-causal masks a query tile's work grows
        // with its index, so tiles are dealt heaviest first with every other
        // round reversed: a CU's heavy block meets a light one, and a last
        // partial round gets the lightest
        const int r = bid >> 8, p = bid & 255, start = r << 8;
        const int len = total - start < 256 ? total - start : 256;
        const int i = total - 1 - (start + ((r & 1) ? len - 1 - p : p));
        qt = i / gridDim.y;
        h = i - qt * gridDim.y;
    }
    const int kvh = h / (a.n_q / a.n_kv);
    const int HD = a.head_dim;
    const int qi = qt * 16 + c;
    const bool qok = qi < a.seq_q;
    const bool qfull = qt * 16 + 16 <= a.seq_q;  // every query of the tile exists
    float* Ks = smem + wave * C::TILE;
    float* Vs = Ks + KT * SK;

    float qreg[QS];
#pragma unroll
    for (int s = 0; s < QS; s += 4) {
        const int d = g * QS + s;
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        if (qok && d < HD) v = *reinterpret_cast<const float4*>(a.Q + (size_t)qi * a.ldq + h * HD + d);
        qreg[s] = v.x;
        qreg[s + 1] = v.y;
        qreg[s + 2] = v.z;
        qreg[s + 3] = v.w;
    }

    const float scale = a.scale;
    const int mk = a.mask_kind;
    const int qg = (MKC == 3 && qok) ? a.q_group[qi] : 0;
    const int G = a.n_groups;
    // small group tables live in LDS, so the per-key test is an LDS read. The
    // main loop reads the table through `al` (derived from the shared array,
    // so its reads compile to ds_read_u8) or straight from global memory; one
    // pointer that could be either compiles to flat loads, whose waits
    // (vmcnt(0) as well) also drain the next key tile's prefetch.
    const bool allow_lds = MKC == 3 && G * G <= C::ALLOW;
    const uint8_t* al = reinterpret_cast<const uint8_t*>(smem) + C::MAIN;
    if (allow_lds) {
        uint8_t* alw = reinterpret_cast<uint8_t*>(smem) + C::MAIN;
        for (int i = tid; i < G * G; i += W * 64) alw[i] = a.allow[i];
        __syncthreads();
    }

    // keys past kv_end are blocked for every query of the block (causal bound)
    int kv_end = a.seq_k;
    if (mk == 2) {
        const int qlast = (qt * 16 + 16 < a.seq_q ? qt * 16 + 16 : a.seq_q) - 1;
        const int e = qlast + a.causal_offset + 1;
        kv_end = e < 0 ? 0 : (e < kv_end ? e : kv_end);
    }

    const bool vec_kg = MKC == 3 && (reinterpret_cast<uintptr_t>(a.k_group) & 3) == 0;
    const bool vec_mask = MKC == 1 && (reinterpret_cast<uintptr_t>(a.mask) & 15) == 0 && (a.ldm & 3) == 0;

    // this lane's share of a tile load: float4 number e = lane + 64 * i of the
    // KT x HDP/4 tile is row e / (HDP/4), dims 4 * (e % (HDP/4))
    float4 kr[F4], vr[F4];
    // with the tile: the mask data of the lane's keys kv0 + 16 kt + 4 g + r
    // (dense mask values or key groups), so the masking step waits on nothing.
    // A run of 4 key groups read as one word stays packed (gword) until the
    // tile is used: unpacking it here would make the wave wait for that load,
    // and with it for the whole K/V prefetch issued just before.
    float mnext[4 * NT];
    int gnext[4 * NT] = {};
    uint32_t gword[NT] = {};
    bool gpacked[NT] = {};
    auto gload = [&](int kv0, int end) {
        if (kv0 + KT <= end && HD == HDP) {  // wave-uniform: every row and column is in range
#pragma unroll
            for (int i = 0; i < F4; i++) {
                const int e = lane + 64 * i, row = e / (HDP / 4), d = 4 * (e % (HDP / 4));
                const int j = kv0 + row;
                kr[i] = *reinterpret_cast<const float4*>(a.K + (size_t)j * a.ldk + kvh * HD + d);
                vr[i] = *reinterpret_cast<const float4*>(a.V + (size_t)j * a.ldv + kvh * HD + d);
            }
        } else {
#pragma unroll
            for (int i = 0; i < F4; i++) {
                const int e = lane + 64 * i, row = e / (HDP / 4), d = 4 * (e % (HDP / 4));
                const int j = kv0 + row;
                kr[i] = vr[i] = make_float4(0.f, 0.f, 0.f, 0.f);
                if (j < end && d < HD) {
                    kr[i] = *reinterpret_cast<const float4*>(a.K + (size_t)j * a.ldk + kvh * HD + d);
                    vr[i] = *reinterpret_cast<const float4*>(a.V + (size_t)j * a.ldv + kvh * HD + d);
                }
            }
        }
        if (!KD) return;
        // a lane's keys come in runs of 4 consecutive (4 g .. 4 g + 3 of each
        // 16): whole in-range runs take one 4-byte group load or one float4
        // mask load when the table allows it
#pragma unroll
        for (int kt = 0; kt < NT; kt++) {
            const int j0 = kv0 + kt * 16 + 4 * g;
            if (MKC == 3) gpacked[kt] = j0 + 4 <= end && vec_kg;
            if (MKC == 3 && j0 + 4 <= end && vec_kg) {
                gword[kt] = *reinterpret_cast<const uint32_t*>(a.k_group + j0);
            } else if (MKC == 1 && j0 + 4 <= end && vec_mask) {
                float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                if (qok) v = *reinterpret_cast<const float4*>(a.mask + (size_t)qi * a.ldm + j0);
                mnext[kt * 4] = v.x;
                mnext[kt * 4 + 1] = v.y;
                mnext[kt * 4 + 2] = v.z;
                mnext[kt * 4 + 3] = v.w;
            } else {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const int j = j0 + r;
                    mnext[kt * 4 + r] = 0.0f;
                    gnext[kt * 4 + r] = 0;
                    if (j < end) {
                        if (MKC == 1 && qok) mnext[kt * 4 + r] = a.mask[(size_t)qi * a.ldm + j];
                        else if (MKC == 3) gnext[kt * 4 + r] = a.k_group[j];
                    }
                }
            }
        }
    };
    auto lstore = [&]() {
#pragma unroll
        for (int i = 0; i < F4; i++) {
            const int e = lane + 64 * i, row = e / (HDP / 4), d = 4 * (e % (HDP / 4));
            *reinterpret_cast<float4*>(Ks + row * SK + d) = kr[i];
            *reinterpret_cast<float4*>(Vs + row * SK + d) = vr[i];
        }
    };

    float m = -INFINITY, lsum = 0.0f;
    v4f oacc[DT];
#pragma unroll
    for (int i = 0; i < DT; i++) oacc[i] = v4f{0.f, 0.f, 0.f, 0.f};

    const int nkt = (kv_end + KT - 1) / KT;
    if (wave < nkt) gload(wave * KT, a.seq_k);
    for (int t = wave; t < nkt; t += W) {
        const int kv0 = t * KT;
        lstore();
        float mcur[4 * NT];
        int gcur[4 * NT];
        if (KD) {
#pragma unroll
            for (int x = 0; x < 4 * NT; x++) {
                mcur[x] = mnext[x];
                gcur[x] = gpacked[x >> 2] ? (int)((gword[x >> 2] >> (8 * (x & 3))) & 0xffu) : gnext[x];
            }
        }
        wave_lds_sync();
        if (t + W < nkt) gload((t + W) * KT, a.seq_k);  // next tile, under this one's math

        // group masks: which of this lane's scores the table blocks, decided
        // before the products; a tile the table blocks for every query of the
        // wave adds p = 0 everywhere and leaves (m, l, O) as they are, so it
        // is skipped (Octo's later timesteps for earlier queries)
        bool mblk[4 * NT];
        if (MKC == 3) {
            bool live = false;
            if (allow_lds) {
#pragma unroll
                for (int x = 0; x < 4 * NT; x++) {
                    const int j = kv0 + (x >> 2) * 16 + 4 * g + (x & 3);
                    const bool b = !qok || j >= kv_end || !al[qg * G + gcur[x]];
                    mblk[x] = b;
                    live = live || !b;
                }
            } else {
#pragma unroll
                for (int x = 0; x < 4 * NT; x++) {
                    const int j = kv0 + (x >> 2) * 16 + 4 * g + (x & 3);
                    const bool b = !qok || j >= kv_end || !a.allow[qg * G + gcur[x]];
                    mblk[x] = b;
                    live = live || !b;
                }
            }
            if (!__any(live)) continue;
        }

        v4f sacc[NT];
#pragma unroll
        for (int kt = 0; kt < NT; kt++) {
            sacc[kt] = v4f{0.f, 0.f, 0.f, 0.f};
            const float* krow = Ks + (kt * 16 + c) * SK + g * QS;
#pragma unroll
            for (int s = 0; s < QS; s += 4) {
                const float4 kv = *reinterpret_cast<const float4*>(krow + s);
                sacc[kt] = mfma_f32(kv.x, qreg[s], sacc[kt]);
                sacc[kt] = mfma_f32(kv.y, qreg[s + 1], sacc[kt]);
                sacc[kt] = mfma_f32(kv.z, qreg[s + 2], sacc[kt]);
                sacc[kt] = mfma_f32(kv.w, qreg[s + 3], sacc[kt]);
            }
        }

        // scale, mask, tile max; a whole tile of keys for a whole query tile
        // with no mask (wave-uniform) only scales
        float mt = -INFINITY;
        if (MKC == 0 && mk == 0 && qfull && kv0 + KT <= kv_end) {
#pragma unroll
            for (int kt = 0; kt < NT; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float x = sacc[kt][r] * scale;
                    sacc[kt][r] = x;
                    mt = fmaxf(mt, x);
                }
        } else
#pragma unroll
        for (int kt = 0; kt < NT; kt++)
#pragma unroll
            for (int r = 0; r < 4; r++) {
                const int j = kv0 + kt * 16 + 4 * g + r;
                float x = sacc[kt][r] * scale;
                bool blocked;
                if (MKC == 3) {
                    blocked = mblk[kt * 4 + r];
                } else if (MKC == 1) {
                    const float mv = mcur[kt * 4 + r];
                    blocked = !qok || j >= kv_end || mv == -FLT_MAX;
                    if (!blocked) x = x + mv;
                } else {
                    blocked = !qok || j >= kv_end || (mk == 2 && j > qi + a.causal_offset);
                }
                x = blocked ? -INFINITY : x;
                sacc[kt][r] = x;
                mt = fmaxf(mt, x);
            }
        mt = rows_max(mt);
        const float mnew = fmaxf(m, mt);

        float alpha = 1.0f;
        if (mnew == -INFINITY) {
#pragma unroll
            for (int kt = 0; kt < NT; kt++) sacc[kt] = v4f{0.f, 0.f, 0.f, 0.f};
        } else {
            // mnew == m gives alpha = exp2(0) = 1 exactly
            alpha = mnew == m ? 1.0f : fast_exp2((m - mnew) * kLog2e);
            float ps = 0.0f;
#pragma unroll
            for (int kt = 0; kt < NT; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const float p = fast_exp2((sacc[kt][r] - mnew) * kLog2e);
                    sacc[kt][r] = p;
                    ps += p;
                }
            lsum = lsum * alpha + ps;
            m = mnew;
        }
        // the accumulators are rescaled only when some query's running max
        // moved (multiplying by alpha = 1 changes nothing)
        if (__any(alpha != 1.0f)) {
#pragma unroll
            for (int dt = 0; dt < DT; dt++) oacc[dt] *= alpha;
        }
#pragma unroll
        for (int dt = 0; dt < DT; dt++) {
#pragma unroll
            for (int kt = 0; kt < NT; kt++)
#pragma unroll
                for (int r = 0; r < 4; r++)
                    oacc[dt] = mfma_f32(Vs[(kt * 16 + 4 * g + r) * SK + dt * 16 + c], sacc[kt][r], oacc[dt]);
        }
        wave_lds_sync();  // this tile's reads are done before the next lstore
    }

    lsum = rows_sum(lsum);

    // merge the waves' partial states: m*, then sum_w e^(m_w - m*) (l_w, O_w)
    __syncthreads();
    float* Mm = smem;               // [W][16]
    float* Ml = smem + 16 * W;      // [W][16]
    float* Mo = smem + 32 * W;      // [W][16][MO]
    if (g == 0) {
        Mm[wave * 16 + c] = m;
        Ml[wave * 16 + c] = lsum;
    }
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
        *reinterpret_cast<float4*>(Mo + (wave * 16 + c) * C::MO + dt * 16 + 4 * g) =
            make_float4(oacc[dt][0], oacc[dt][1], oacc[dt][2], oacc[dt][3]);
    __syncthreads();
    // every wave's (m, l) for this lane's query, in registers: the uniform pass
    // below reuses this LDS for V tiles
    float mw[W], lw[W], mstar = -INFINITY;
#pragma unroll
    for (int w = 0; w < W; w++) {
        mw[w] = Mm[w * 16 + c];
        lw[w] = Ml[w * 16 + c];
        mstar = fmaxf(mstar, mw[w]);
    }
    const bool masked = qok && mstar == -INFINITY;
    // rows with every key blocked: uniform mean of V over all seq_k keys
    // (attn_uniform_row); the waves sum V over their tiles with p = 1
    if (__syncthreads_or(masked)) {
        // a row that is not masked keeps its softmax partial (it adds p = 0 below)
        if (masked)
#pragma unroll
            for (int i = 0; i < DT; i++) oacc[i] = v4f{0.f, 0.f, 0.f, 0.f};
        const int nall = (a.seq_k + KT - 1) / KT;
        for (int t = wave; t < nall; t += W) {
            const int kv0 = t * KT;
            gload(kv0, a.seq_k);
            lstore();
            wave_lds_sync();
#pragma unroll
            for (int dt = 0; dt < DT; dt++)
#pragma unroll
                for (int kt = 0; kt < NT; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const int j = kv0 + kt * 16 + 4 * g + r;
                        const float p = (masked && j < a.seq_k) ? 1.0f : 0.0f;
                        oacc[dt] = mfma_f32(Vs[(kt * 16 + 4 * g + r) * SK + dt * 16 + c], p, oacc[dt]);
                    }
            wave_lds_sync();
        }
        __syncthreads();
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
            *reinterpret_cast<float4*>(Mo + (wave * 16 + c) * C::MO + dt * 16 + 4 * g) =
                make_float4(oacc[dt][0], oacc[dt][1], oacc[dt][2], oacc[dt][3]);
        __syncthreads();
    }
    // wave w writes the 16-dim output slices w, w + W, ... (every wave holds
    // all (m, l) already; the sums over waves run in the same order for each)
    if (wave >= DT || !qok) return;

    float f[W], l = 0.0f;
#pragma unroll
    for (int w = 0; w < W; w++) {
        f[w] = masked ? 1.0f : (mw[w] == -INFINITY ? 0.0f : fast_exp2((mw[w] - mstar) * kLog2e));
        l += f[w] * lw[w];
    }
    const float inv = masked ? 1.0f / (float)a.seq_k : 1.0f / l;
    for (int dt = wave; dt < DT; dt += W) {
        const int d = dt * 16 + 4 * g;
        if (d < HD) {
            float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int w = 0; w < W; w++) {
                const float4 v = *reinterpret_cast<const float4*>(Mo + (w * 16 + c) * C::MO + d);
                o.x += f[w] * v.x;
                o.y += f[w] * v.y;
                o.z += f[w] * v.z;
                o.w += f[w] * v.w;
            }
            o.x *= inv;
            o.y *= inv;
            o.z *= inv;
            o.w *= inv;
            *reinterpret_cast<float4*>(a.out + (size_t)qi * a.ldo + h * HD + d) = o;
        }
    }
}

template <int HDP, int KT, int W, int MKC>
void launch_kd(const AttnArgs& a, hipStream_t st) {
    using C = AttnCfg<HDP, KT, W>;
    static const bool attr = [] {
        if (C::LDS > 65536)
            VLA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_fwd<HDP, KT, W, MKC>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
        return true;
    }();
    (void)attr;
    attn_fwd<HDP, KT, W, MKC><<<dim3((a.seq_q + 15) / 16, a.n_q), W * 64, C::LDS, st>>>(a);
}

template <int HDP, int KT, int W>
void launch_w(const AttnArgs& a, hipStream_t st) {
    if (a.mask_kind == 1) launch_kd<HDP, KT, W, 1>(a, st);
    else if (a.mask_kind == 3) launch_kd<HDP, KT, W, 3>(a, st);
    else launch_kd<HDP, KT, W, 0>(a, st);
}

// ---------------------------------------------------------------------------
// attn_split: the same attention with both products on the fp16 matrix cores.
//
// The operands' two parts (fp16parts.h) hold them to 2^-22 (2^-24.5 in the mean)
// or to 2^-40 of the largest value that shares the scale, whichever is more (a
// weight under 2^-41 of its query's largest adds nothing to the values' sum). So three
// v_mfma_f32_16x16x32_f16 (16 cycles each, exact products, fp32 sums over 32
// terms at once) replace the eight v_mfma_f32_16x16x4_f32 (32 cycles each) of a
// 16 x 16 x 32 product, and the sums round an eighth as often: against 64 bits
// the outputs are closer than the fp32 matrix cores' (2-norm, 1024 x 1024 x 12 heads of 64,
// N(0, 1): 2.3e-7 against 4.1e-7; 50 x 227 x 15: 2.0e-7 against 3.0e-7).
// Scales: one per query row, running ones per wave for K and V (V's accumulators
// are rescaled with it, as for a new maximum), 2^15 for the weights; all powers
// of two, taken out again exactly.
//
// What a shared scale does not carry goes to attn_block_f32, which computes the
// block again from the inputs in plain fp32, 15 to 60 times slower (50 x 227 x 15
// heads 9 -> 142 us): infinities in an operand and outputs that are not finite;
// where a scale is set, a key's four columns of V 2^17 below the value that sets it
// (as beside a masked row of padding that holds anything) and a largest query times
// largest key that could add 2^14 to a score; at every tile, a column of V over a
// lane's keys 2^18 below the scale. Of 400 calls with columns lognormal to 1.5, at most 6
// take it. These checks, scores in the natural domain and masks after the scale cost
// 4 to 7% (50 x 227 x 15 heads 8.5 -> 9.0 us, 690 x 690 x 12 block-causal 18.2 -> 19.2,
// 1024 x 1024 x 12 22.8 -> 24.4).
//
// A block owns 16 * QF queries of one head and its W waves split the key
// range in tiles of 32 keys (tile t, t + W, ...), each wave for all of the
// block's queries, so every K and V value is loaded and split once per block.
// Every global load puts the 16 lanes of a group on 256 contiguous bytes of a
// key row. (Loading K in the matrix cores' operand order, 16 rows by 16 bytes
// across neighbouring lanes, costs the address unit a cycle per lane: 14.7
// bytes per clock and CU against 40, measured from L2.) K's parts cross the
// lanes through a wave's own LDS rows; V's do not have to, since the k index of
// a product may run over its terms in any order as long as both operands use
// the same one:
//   S^T = K Q^T   : lane (g = l / 16, c = l % 16) supplies key c, dims 8 g ..
//                   8 g + 7 of a 32-dim step;
//   O^T = V^T P^T : element i of lane group g is key 16 (i / 4) + 4 g + i % 4,
//                   which is the probability the lane already holds from S^T
//                   (sub-tile i / 4, register i % 4), and V's row index c of
//                   16-row tile dt stands for dim 4 c + dt, so a lane's own
//                   float4 loads of eight key rows are its operands.
// The loads of a wave's next tile are issued as soon as the registers of this
// one are split.

struct Split8 {
    f16x8 h, m;
};

__device__ __forceinline__ Split8 split8(const float4& x, const float4& y) {
    uint4 h, m;
    split2(x.x, x.y, h.x, m.x);
    split2(x.z, x.w, h.y, m.y);
    split2(y.x, y.y, h.z, m.z);
    split2(y.z, y.w, h.w, m.w);
    return Split8{__builtin_bit_cast(f16x8, h), __builtin_bit_cast(f16x8, m)};
}
__device__ __forceinline__ Split8 split8(const float4& x, const float4& y, float s) {
    return split8(make_float4(x.x * s, x.y * s, x.z * s, x.w * s), make_float4(y.x * s, y.y * s, y.z * s, y.w * s));
}

// max over eight values (NaN is passed over)
__device__ __forceinline__ float max4(v4f x, v4f y) {
    float m;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(m) : "v"(x[0]), "v"(x[1]), "v"(x[2]));
    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(m) : "v"(x[3]), "v"(y[0]));
    asm("v_max3_f32 %0, %0, %1, %2" : "+v"(m) : "v"(y[1]), "v"(y[2]));
    return fmaxf(m, y[3]);
}

__device__ __forceinline__ bool not_finite(float mx) { return ((__float_as_uint(mx) >> 23) & 0xffu) == 255u; }

// n / d for 0 <= n < 2^20, given the float nearest 1 / d: (n + 0.5) / d is at
// least 0.5 / d away from the whole numbers, the rounding below n 2^-23 / d
struct AttnInv {
    float nqt, heads, group;  // 1 / query tiles, 1 / query heads, 1 / (query heads per kv head)
};
__device__ __forceinline__ int quotient(int n, float inv) {
    return __builtin_amdgcn_readfirstlane((int)(((float)n + 0.5f) * inv));
}

__device__ __forceinline__ v4f mfma_f16(const f16x8& a, const f16x8& b, v4f c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0);
}

// whether query qi may not see key j (qi < seq_q, j < seq_k); *add is the
// additive mask value of a key it may see
__device__ __forceinline__ bool mask_blocks(const AttnArgs& a, int qi, int j, float* add) {
    *add = 0.0f;
    if (a.mask_kind == 1) {
        const float mv = a.mask[(size_t)qi * a.ldm + j];
        *add = mv;
        return mv <= -FLT_MAX;  // lowest() or -inf
    }
    if (a.mask_kind == 2) return j > qi + a.causal_offset;
    if (a.mask_kind == 3) return !a.allow[(int)a.q_group[qi] * a.n_groups + a.k_group[j]];
    return false;
}

// The block's queries [q0, q0 + nq) of head h in plain fp32, one query per wave
// at a time, lanes over keys, then over dims: for operands the split kernel
// does not carry, whose speed does not matter. Keys a query may not see are
// left out, whatever they hold.
template <int HDP>
__device__ __forceinline__ void attn_block_f32(const AttnArgs& a, int q0, int nq, int h, int kvh) {
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, nw = blockDim.x >> 6;
    const int HD = a.head_dim;
    for (int q = wave; q < nq; q += nw) {
        const int qi = q0 + q;
        if (qi >= a.seq_q) break;
        const float* qp = a.Q + (size_t)qi * a.ldq + h * HD;
        auto score = [&](int j) {
            float add;
            if (mask_blocks(a, qi, j, &add)) return -INFINITY;
            const float* kp = a.K + (size_t)j * a.ldk + kvh * HD;
            float4 s4 = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll 4
            for (int d = 0; d < HD; d += 4) {
                const float4 k = *reinterpret_cast<const float4*>(kp + d);
                s4 = make_float4(fmaf(qp[d], k.x, s4.x), fmaf(qp[d + 1], k.y, s4.y), fmaf(qp[d + 2], k.z, s4.z),
                                 fmaf(qp[d + 3], k.w, s4.w));
            }
            const float s = ((s4.x + s4.y) + (s4.z + s4.w)) * a.scale;
            return a.mask_kind == 1 ? s + add : s;
        };
        float m = -INFINITY;
        for (int j = lane; j < a.seq_k; j += 64) m = fmaxf(m, score(j));
        for (int o = 32; o; o >>= 1) m = fmaxf(m, __shfl_xor(m, o));
        const bool masked = m == -INFINITY;
        float l = 0.0f;
        float o[4][HDP / 64];  // four sums of every fourth key
#pragma unroll
        for (int t = 0; t < 4; t++)
#pragma unroll
            for (int u = 0; u < HDP / 64; u++) o[t][u] = 0.0f;
        for (int j0 = 0; j0 < a.seq_k; j0 += 64) {
            const int j = j0 + lane;
            float p = 0.0f, add;
            const bool seen = j < a.seq_k && (masked || !mask_blocks(a, qi, j, &add));
            if (seen) p = masked ? 1.0f : fast_exp2((score(j) - m) * kLog2e);
            l += p;
            // eight keys' loads in flight (past the last key: the last again, weight 0)
            const uint64_t take = __ballot(seen);
            for (int t0 = 0; t0 < 64 && j0 + t0 < a.seq_k; t0 += 8) {
                float v[8][HDP / 64];
#pragma unroll
                for (int t = 0; t < 8; t++)
#pragma unroll
                    for (int u = 0; u < HDP / 64; u++) {
                        const int d = u * 64 + lane;
                        v[t][u] = d < HD ? a.V[(size_t)min(j0 + t0 + t, a.seq_k - 1) * a.ldv + kvh * HD + d] : 0.0f;
                    }
#pragma unroll
                for (int t = 0; t < 8; t++) {
                    const float pt = __shfl(p, t0 + t);
#pragma unroll
                    for (int u = 0; u < HDP / 64; u++)
                        o[t & 3][u] = (take >> (t0 + t)) & 1u ? fmaf(pt, v[t][u], o[t & 3][u]) : o[t & 3][u];
                }
            }
        }
        for (int x = 32; x; x >>= 1) l += __shfl_xor(l, x);
#pragma unroll
        for (int u = 0; u < HDP / 64; u++) {
            const int d = u * 64 + lane;
            if (d < HD) a.out[(size_t)qi * a.ldo + h * HD + d] = ((o[0][u] + o[1][u]) + (o[2][u] + o[3][u])) / l;
        }
    }
}

template <int HDP, int QF, int W>
struct SplitCfg {
    static constexpr int S = HDP / 32;             // 32-dim steps of Q K^T
    static constexpr int U = HDP / 64;             // 64-dim column groups of V
    static constexpr int MO = HDP + 4;             // merge row, floats
    static constexpr bool QLDS = QF > 2;           // the query fragments live in LDS
    static constexpr int QB = QLDS ? QF * S * 2 * 1024 : 0;
    static constexpr int KG = 4096;                // key groups kept in LDS behind them
    static constexpr int FSB = QB + KG + 32;       // (a last tile reads groups past seq_k)
    static constexpr int KROW = 2 * HDP + 16;      // bytes of one part of a key row: 16 rows'
                                                   // 16-byte reads fall on distinct banks
    static constexpr int KB = FSB + (QLDS ? 64 * QF : 0);  // 32 keys' two parts per wave
    static constexpr int MAINB = KB + W * 32 * 2 * KROW;
    static constexpr int MERGE = 4 * W * 16 * QF * (MO + 2);
    static constexpr int MEAN = 4 * (W * 4 + 1) * HDP;  // partial means of V, then the mean
    static constexpr int MAX0 = MERGE > MAINB ? MERGE : MAINB;
    static constexpr int LDS = (MAX0 > MEAN ? MAX0 : MEAN) + 16;
    static_assert(LDS <= 160 * 1024, "LDS");
};

template <int HDP, int QF, int W, int MKC, bool FULL>
__global__ __launch_bounds__(W * 64, HDP == 64 ? 2 : 1) void attn_split(AttnArgs a, AttnInv inv) {
    using C = SplitCfg<HDP, QF, W>;
    constexpr int S = C::S, U = C::U, MO = C::MO, NQ = 16 * QF;
    extern __shared__ __attribute__((aligned(16))) float smem[];
    uint32_t* flags = reinterpret_cast<uint32_t*>(reinterpret_cast<char*>(smem) + C::LDS - 16);

    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // wave-uniform: scalar addresses
    const int g = lane >> 4, c = lane & 15;
    // block order: as attn_fwd (XCD-contiguous up to one round of 256 blocks,
    // else heaviest query tiles first with every other round reversed). The
    // quotients are taken with the launch's reciprocals: exact for the block
    // counts the launch allows, and four integer divisions ahead of the first
    // load are not.
    const int nqt = gridDim.x, total = nqt * gridDim.y;
    const int bid = blockIdx.y * nqt + blockIdx.x;
    int qt, h;
    if (total <= 256) {
        const int xcd = bid & 7, per = total >> 3, rem = total & 7;
        const int logical = xcd * per + (xcd < rem ? xcd : rem) + (bid >> 3);
        h = quotient(logical, inv.nqt);
        qt = logical - h * nqt;
    } else {
        const int r = bid >> 8, p = bid & 255, start = r << 8;
        const int len = total - start < 256 ? total - start : 256;
        const int i = total - 1 - (start + ((r & 1) ? len - 1 - p : p));
        qt = quotient(i, inv.heads);
        h = i - qt * gridDim.y;
    }
    const int kvh = quotient(h, inv.group);
    const int HD = a.head_dim;
    const int q0 = qt * NQ;
    const bool qfull = q0 + NQ <= a.seq_q;
    const float* Kb = a.K + kvh * HD;
    const float* Vb = a.V + kvh * HD;
    if (tid == 0) *flags = 0;

    // this lane's share of a tile: K rows 4 jj + g, V rows of keys
    // 16 (jj / 4) + 4 g + jj % 4, dims 64 u + 4 c .. (rows past the last key
    // repeat it, their scores are blocked; dims past the head read as zero)
    float4 kr[8][U], vr[8][U];
    const int jmax = a.seq_k - 1;
    // base + a 32-bit byte offset per lane: rows are clamped as offsets, so a
    // tile's last rows take no branch and no 64-bit address per lane
    auto rload = [&](float4 (&dst)[U], const float* base, uint32_t off) {
        const char* p = reinterpret_cast<const char*>(base);
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (FULL) {
                dst[u] = *reinterpret_cast<const float4*>(p + off + 256 * u);
            } else {
                const int d = 64 * u + 4 * c;
                dst[u] = *reinterpret_cast<const float4*>(p + (off - 16u * c + 4u * min(d, HD - 4)));
                if (d >= HD) dst[u] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
    };
    const uint32_t kld = 4u * a.ldk, vld = 4u * a.ldv;
    const uint32_t koff = g * kld + 16u * c, voff = 4 * g * vld + 16u * c;
    auto kload = [&](int kv0) {
        const uint32_t last = min(jmax - kv0, 31) * kld + 16u * c;
        uint32_t o = koff;
        asm volatile("" : "+v"(o));  // eight sums here, not eight registers kept over the loop
#pragma unroll
        for (int jj = 0; jj < 8; jj++) rload(kr[jj], Kb + (size_t)kv0 * a.ldk, min(o + 4 * jj * kld, last));
    };
    auto vload = [&](int kv0) {
        const uint32_t last = min(jmax - kv0, 31) * vld + 16u * c;
        uint32_t o = voff;
        asm volatile("" : "+v"(o));
#pragma unroll
        for (int jj = 0; jj < 8; jj++)
            rload(vr[jj], Vb + (size_t)kv0 * a.ldv, min(o + (16 * (jj >> 2) + (jj & 3)) * vld, last));
    };
    char* kw = reinterpret_cast<char*>(smem) + C::KB + wave * (32 * 2 * C::KROW);

    // keys past kv_end are blocked for every query of the block (causal bound)
    int kv_end = a.seq_k;
    const int mk = a.mask_kind;
    if (mk == 2) {
        const int qlast = (q0 + NQ < a.seq_q ? q0 + NQ : a.seq_q) - 1;
        const int e = qlast + a.causal_offset + 1;
        kv_end = e < 0 ? 0 : (e < kv_end ? e : kv_end);
    }
    const int nkt = (kv_end + 31) / 32;

    // the query fragments: query 16 f + c, dims 32 s + 8 g ..
    Split8 qreg[C::QLDS ? 1 : QF][C::QLDS ? 1 : S];
    float fs[QF];  // scores' unit of a query, times the softmax scale
    f16x8* qlds = reinterpret_cast<f16x8*>(smem);
    float* fsl = reinterpret_cast<float*>(reinterpret_cast<char*>(smem) + C::FSB);
    auto qload = [&](int f, float4 (&x)[S][2]) {
        const int qi = min(q0 + 16 * f + c, a.seq_q - 1);
        const float* p = a.Q + (size_t)qi * a.ldq + h * HD;
#pragma unroll
        for (int s = 0; s < S; s++)
#pragma unroll
            for (int e = 0; e < 2; e++) {
                const int d = 32 * s + 8 * g + 4 * e;
                x[s][e] = *reinterpret_cast<const float4*>(p + (FULL ? d : min(d, HD - 4)));
                if (!FULL && d >= HD) x[s][e] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
    };
    bool bad = false;
    // splits a query fragment; returns its scores' unit times the softmax scale
    auto qsplit = [&](const float4 (&x)[S][2], Split8 (&q)[S]) {
        float mx = 0.0f;
#pragma unroll
        for (int s = 0; s < S; s++)
#pragma unroll
            for (int e = 0; e < 2; e++) mx = absmax4(mx, x[s][e]);
        mx = rows_max(mx);
        bad = bad || not_finite(mx);
        const uint32_t e = scale_exp(mx, 14);
#pragma unroll
        for (int s = 0; s < S; s++) q[s] = split8(x[s][0], x[s][1], a.scale < 0.0f ? -exp_float(e) : exp_float(e));
        return exp_float(254u - e) * fabsf(a.scale);
    };
    // the queries' loads ahead of the first tile's: loads return in order
    const bool qmine = !C::QLDS || wave < QF;
    float4 qx[C::QLDS ? 1 : QF][S][2];
    static_assert(!C::QLDS || W >= QF, "a wave per query fragment");
    if (qmine) {
#pragma unroll
        for (int f = 0; f < (C::QLDS ? 1 : QF); f++) qload(C::QLDS ? wave : f, qx[f]);
    }
    if (MKC != 3 && wave < nkt) {  // group masks first find a tile with something to see
        kload(wave * 32);
        vload(wave * 32);
    }
    if constexpr (C::QLDS) {
        if (qmine) {
            Split8 q[S];
            const float u = qsplit(qx[0], q);
#pragma unroll
            for (int s = 0; s < S; s++) {
                qlds[((wave * S + s) * 2 + 0) * 64 + lane] = q[s].h;
                qlds[((wave * S + s) * 2 + 1) * 64 + lane] = q[s].m;
            }
            if (g == 0) fsl[16 * wave + c] = u;
        }
    } else {
#pragma unroll
        for (int f = 0; f < QF; f++) fs[f] = qsplit(qx[f], qreg[f]);
    }

    // group masks: the key groups a query's group may see, as two words for up
    // to 64 groups (more are read from the table per score), and the keys'
    // groups in LDS where they fit
    const int G = a.n_groups;
    uint32_t am0[QF], am1[QF];
    int qg[QF];
    uint8_t* kgl = reinterpret_cast<uint8_t*>(smem) + C::QB;
    if constexpr (MKC == 3) {
        for (int j = tid; j < a.seq_k && a.seq_k <= C::KG; j += W * 64) kgl[j] = a.k_group[j];
#pragma unroll
        for (int f = 0; f < QF; f++) {
            const int qi = q0 + 16 * f + c;
            qg[f] = qi < a.seq_q ? a.q_group[qi] : 0;
            uint32_t lo = 0, hi = 0;
            if (G <= 64 && qi < a.seq_q)
                for (int x = g; x < G; x += 4) {  // the four lanes of a query read a quarter of its row each
                    const uint32_t b = a.allow[qg[f] * G + x] ? 1u : 0u;
                    if (x < 32) lo |= b << x;
                    else hi |= b << (x - 32);
                }
            lo |= __shfl_xor(lo, 16);
            hi |= __shfl_xor(hi, 16);
            am0[f] = lo | __shfl_xor(lo, 32);
            am1[f] = hi | __shfl_xor(hi, 32);
        }
    }
    const bool vec_mask = MKC == 1 && (reinterpret_cast<uintptr_t>(a.mask) & 15) == 0 && (a.ldm & 3) == 0;
    __syncthreads();
    if constexpr (C::QLDS)
#pragma unroll
        for (int f = 0; f < QF; f++) fs[f] = fsl[16 * f + c];

    float M[QF], lsum[QF];  // running max and sum per query 16 f + c
    v4f oacc[QF][U][4];     // O^T: dim 64 u + 4 (4 g + r) + dt of query 16 f + c,
                            // in units of 1 / sv (both sums carry the weights' 2^15)
    // K's and V's scales: the first tile's, until a value outgrows them (V's
    // accumulators are then rescaled; a tile of smaller values keeps the unit)
    float sk = 0.0f, uk = 0.0f, sv = 0.0f, uv = 0.0f, klim = -1.0f, vlim = -1.0f;
#pragma unroll
    for (int f = 0; f < QF; f++) {
        M[f] = -INFINITY;
        lsum[f] = 0.0f;
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int dt = 0; dt < 4; dt++) oacc[f][u][dt] = v4f{0.f, 0.f, 0.f, 0.f};
    }

    // group masks: bit 8 f + 4 kt + r says whether this lane's score of tile t
    // is blocked. A tile the table blocks for every query would add p = 0
    // everywhere: it is neither loaded nor computed.
    constexpr uint32_t kAll = QF == 4 ? 0xffffffffu : (1u << (8 * QF)) - 1u;
    auto dead_of = [&](int kv0) {
        uint32_t dead = 0;
#pragma unroll
        for (int kt = 0; kt < 2; kt++) {
            const int j0 = kv0 + 16 * kt + 4 * g;
            uint32_t kg = 0;
            if (a.seq_k <= C::KG) kg = *reinterpret_cast<const uint32_t*>(kgl + j0);
            else
                for (int r = 0; r < 4; r++) kg |= (uint32_t)a.k_group[min(j0 + r, jmax)] << (8 * r);
            if (G <= 64) {
#pragma unroll
                for (int r = 0; r < 4; r++) {
                    const uint32_t v = (kg >> (8 * r)) & 0xffu;
#pragma unroll
                    for (int f = 0; f < QF; f++) {
                        const uint32_t w = v < 32 ? am0[f] : am1[f];
                        dead |= (~(w >> (v & 31)) & 1u) << (8 * f + 4 * kt + r);
                    }
                }
            } else {
#pragma unroll
                for (int f = 0; f < QF; f++)
                    for (int r = 0; r < 4; r++)
                        if (!a.allow[qg[f] * G + (int)((kg >> (8 * r)) & 0xffu)]) dead |= 1u << (8 * f + 4 * kt + r);
            }
            // keys past the last one
            const int past = j0 + 4 - a.seq_k;
            const uint32_t out = past <= 0 ? 0u : (0xf0u >> (past > 4 ? 4 : past)) & 0xfu;
#pragma unroll
            for (int f = 0; f < QF; f++) dead |= out << (8 * f + 4 * kt);
        }
#pragma unroll
        for (int f = 0; f < QF; f++)
            if (q0 + 16 * f + c >= a.seq_q) dead |= 0xffu << (8 * f);
        return dead;
    };
    // the first tile from t on (in steps of W) with something to see
    auto next_tile = [&](int t, uint32_t* dead) {
        if constexpr (MKC == 3) {
            for (; t < nkt; t += W) {
                *dead = dead_of(t * 32);
                if (__any(*dead != kAll)) break;
            }
        }
        return t;
    };

    uint32_t dead = 0;
    int t = next_tile(wave, &dead);
    if (MKC == 3 && t < nkt) {
        kload(t * 32);
        vload(t * 32);
    }
    while (t < nkt) {
        const int kv0 = t * 32;
        uint32_t dead_next = 0;
        const int tn = next_tile(t + W, &dead_next);
        const bool more = tn < nkt;
        float mval[MKC == 1 ? QF : 1][2][4];
        if constexpr (MKC == 1) {
#pragma unroll
            for (int f = 0; f < QF; f++)
#pragma unroll
                for (int kt = 0; kt < 2; kt++) {
                    const int qi = q0 + 16 * f + c, j0 = kv0 + 16 * kt + 4 * g;
                    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
                    if (qi < a.seq_q) {
                        const float* mp = a.mask + (size_t)qi * a.ldm + j0;
                        if (j0 + 4 <= a.seq_k && vec_mask) {
                            v = *reinterpret_cast<const float4*>(mp);
                        } else {
                            if (j0 < a.seq_k) v.x = mp[0];
                            if (j0 + 1 < a.seq_k) v.y = mp[1];
                            if (j0 + 2 < a.seq_k) v.z = mp[2];
                            if (j0 + 3 < a.seq_k) v.w = mp[3];
                        }
                    }
                    mval[f][kt][0] = v.x;
                    mval[f][kt][1] = v.y;
                    mval[f][kt][2] = v.z;
                    mval[f][kt][3] = v.w;
                }
        }

        float kmax = 0.0f;
#pragma unroll
        for (int jj = 0; jj < 8; jj++)
#pragma unroll
            for (int u = 0; u < U; u++)
                kmax = absmax4(kmax, kr[jj][u]);
        if (__any(kmax > klim)) {
            kmax = wave_max_f32(kmax);
            bad = bad || not_finite(kmax);
            const uint32_t e = scale_exp(kmax, 14);
            sk = exp_float(e);
            uk = exp_float(254u - e);
            klim = 32768.0f * uk;
            // queries and keys, seen or not, whose largest product could add 2^14 to
            // a score: 2^-40 of that is no longer below the rounding of an ordinary one
#pragma unroll
            for (int f = 0; f < QF; f++) bad = bad || fs[f] * kmax > 1.0f;
        }

        // K's parts to the operand's lanes through this wave's LDS rows
#pragma unroll
        for (int jj = 0; jj < 8; jj++)
#pragma unroll
            for (int u = 0; u < U; u++) {
                uint2 kh, km;
                split2(kr[jj][u].x * sk, kr[jj][u].y * sk, kh.x, km.x);
                split2(kr[jj][u].z * sk, kr[jj][u].w * sk, kh.y, km.y);
                char* p = kw + (4 * jj + g) * (2 * C::KROW) + 128 * u + 8 * c;
                *reinterpret_cast<uint2*>(p) = kh;
                *reinterpret_cast<uint2*>(p + C::KROW) = km;
            }
        if (more) kload(tn * 32);
        wave_lds_sync();

        // S^T = K Q^T
        v4f sacc[QF][2];
#pragma unroll
        for (int f = 0; f < QF; f++) sacc[f][0] = sacc[f][1] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < S; s++) {
            Split8 kp[2], q[QF];
#pragma unroll
            for (int kt = 0; kt < 2; kt++) {
                const char* p = kw + (16 * kt + c) * (2 * C::KROW) + 64 * s + 16 * g;
                kp[kt].h = *reinterpret_cast<const f16x8*>(p);
                kp[kt].m = *reinterpret_cast<const f16x8*>(p + C::KROW);
            }
#pragma unroll
            for (int f = 0; f < QF; f++) {
                if constexpr (C::QLDS) {
                    q[f].h = qlds[((f * S + s) * 2 + 0) * 64 + lane];
                    q[f].m = qlds[((f * S + s) * 2 + 1) * 64 + lane];
                } else {
                    q[f] = qreg[f][s];
                }
            }
#define VLA_QK(KP, QP)                                       \
    _Pragma("unroll") for (int f = 0; f < QF; f++)           \
        _Pragma("unroll") for (int kt = 0; kt < 2; kt++)     \
            sacc[f][kt] = mfma_f16(kp[kt].KP, q[f].QP, sacc[f][kt]);
            VLA_QK(m, h)
            VLA_QK(h, m)
            VLA_QK(h, h)
#undef VLA_QK
        }
        // the largest of the lane's columns, and the least that is not zero (as
        // bits less one)
        float vmax = 0.0f, resc = 1.0f;
        uint32_t vmin = ~0u;
#pragma unroll
        for (int u = 0; u < U; u++) {
            float m[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int jj = 0; jj < 8; jj += 2) {
                const float4 &p = vr[jj][u], &q = vr[jj + 1][u];
                m[0] = absmax(m[0], p.x, q.x);
                m[1] = absmax(m[1], p.y, q.y);
                m[2] = absmax(m[2], p.z, q.z);
                m[3] = absmax(m[3], p.w, q.w);
            }
            vmax = absmax(absmax(vmax, m[0], m[1]), m[2], m[3]);
#pragma unroll
            for (int dt = 0; dt < 4; dt++) vmin = min(vmin, __float_as_uint(m[dt]) - 1u);
        }
        if (__any(vmax > vlim)) {
            vmax = wave_max_f32(vmax);
            bad = bad || not_finite(vmax);
            // a key's four columns (that are not zero, hence the bits less one) 2^17
            // below the largest of a tile, as beside a row of padding that holds
            // anything: a scale for both leaves those too few bits
#pragma unroll
            for (int jj = 0; jj < 8; jj++)
#pragma unroll
                for (int u = 0; u < U; u++) {
                    const float m = absmax4(0.0f, vr[jj][u]);
                    bad = bad || __float_as_uint(m) - 1u < __float_as_uint(vmax * 0x1p-17f);
                }
            const uint32_t e = scale_exp(vmax, 14);
            sv = exp_float(e);
            resc = uv * sv;  // the old unit over the new one (0 before any tile, whose sums are 0)
            uv = exp_float(254u - e);
            vlim = 32768.0f * uv;
        }
        // a column of the lane's keys 2^18 below the scale. (Not of fewer than four, the
        // last ones, where the lane's others lie past them: of 64 ordinary values one
        // is that small every few hundred calls, of four keys' none.)
        bad = bad || (kv0 + 4 * g + 3 < a.seq_k && vmin < __float_as_uint(0.125f * uv));

        // scale, mask and online softmax: x = acc f + mask in the natural domain
        // (times log2 e a mask between lowest() / log2 e and lowest(), bf16's
        // lowest among them, would overflow), rounded once; the maximum and the
        // weights p = e^(x - M) are taken from the same x, so no weight passes 1
        // (a mask of -1e9 leaves x and M whole multiples of 64, the unrounded
        // score is not)
        Split8 pp[QF];
        const bool plain = MKC == 0 && mk == 0 && qfull && kv0 + 32 <= kv_end;  // wave-uniform
#pragma unroll
        for (int f = 0; f < QF; f++) {
            const int qi = q0 + 16 * f + c;
            const float fq = fs[f] * uk;
            float mt;
            if constexpr (MKC == 1) {
                mt = -INFINITY;
#pragma unroll
                for (int kt = 0; kt < 2; kt++)
#pragma unroll
                    for (int r = 0; r < 4; r++) {
                        const float v = mval[f][kt][r];
                        const bool blocked =
                            qi >= a.seq_q || kv0 + 16 * kt + 4 * g + r >= kv_end || v <= -FLT_MAX;
                        const float x = blocked ? -INFINITY : fmaf(sacc[f][kt][r], fq, v);
                        sacc[f][kt][r] = x;
                        mt = fmaxf(mt, x);
                    }
            } else {
                sacc[f][0] *= fq;
                sacc[f][1] *= fq;
                if (!plain) {  // (after the product: fq underflows to 0 under zero or tiny operands)
#pragma unroll
                    for (int kt = 0; kt < 2; kt++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const int j = kv0 + 16 * kt + 4 * g + r;
                            const bool blocked =
                                MKC == 3 ? (dead >> (8 * f + 4 * kt + r)) & 1u
                                         : qi >= a.seq_q || j >= kv_end || (mk == 2 && j > qi + a.causal_offset);
                            sacc[f][kt][r] = blocked ? -INFINITY : sacc[f][kt][r];
                        }
                }
                mt = max4(sacc[f][0], sacc[f][1]);
            }
            const float mnew = fmaxf(M[f], rows_max(mt));
            // a query that has seen nothing yet keeps M = -inf; its weights are
            // e^-inf = 0 against any finite reference
            const float mref = fmaxf(mnew, -FLT_MAX);
            const float decay = fast_exp2((M[f] - mref) * kLog2e), alpha = decay * resc;
            float4 x[2];
#pragma unroll
            for (int kt = 0; kt < 2; kt++) {
                auto weight = [&](int r) {
                    // times 2^15 after the exponential: 15 in the exponent would coarsen it
                    return fast_exp2((sacc[f][kt][r] - mref) * kLog2e) * 32768.0f;
                };
                x[kt] = make_float4(weight(0), weight(1), weight(2), weight(3));
            }
            const float ps = ((x[0].x + x[0].y) + (x[0].z + x[0].w)) + ((x[1].x + x[1].y) + (x[1].z + x[1].w));
            lsum[f] = fmaf(lsum[f], decay, ps);
            M[f] = mnew;
            if (__any(alpha != 1.0f)) {
#pragma unroll
                for (int u = 0; u < U; u++)
#pragma unroll
                    for (int dt = 0; dt < 4; dt++) oacc[f][u][dt] *= alpha;
            }
            pp[f] = split8(x[0], x[1]);
        }

        // O^T += V^T P^T
#pragma unroll
        for (int u = 0; u < U; u++) {
            Split8 vp[4];
#pragma unroll
            for (int dt = 0; dt < 4; dt++) {
                float4 e[2];
#pragma unroll
                for (int kt = 0; kt < 2; kt++) {
                    auto at = [&](int r) {
                        const float4& v = vr[4 * kt + r][u];
                        return dt == 0 ? v.x : dt == 1 ? v.y : dt == 2 ? v.z : v.w;
                    };
                    e[kt] = make_float4(at(0), at(1), at(2), at(3));
                }
                vp[dt] = split8(e[0], e[1], sv);
            }
            if (u == U - 1 && more) vload(tn * 32);
#define VLA_PV(VP, PP)                                       \
    _Pragma("unroll") for (int f = 0; f < QF; f++)           \
        _Pragma("unroll") for (int dt = 0; dt < 4; dt++)     \
            oacc[f][u][dt] = mfma_f16(vp[dt].VP, pp[f].PP, oacc[f][u][dt]);
            VLA_PV(m, h)
            VLA_PV(h, m)
            VLA_PV(h, h)
#undef VLA_PV
        }
        wave_lds_sync();  // this tile's reads of kw are done before the next tile's writes
        t = tn;
        dead = dead_next;
    }

    if (__any(bad) && lane == 0) atomicOr(flags, 1u);
#pragma unroll
    for (int f = 0; f < QF; f++) lsum[f] = rows_sum(lsum[f]);

    // merge the waves' partial states: M*, then sum_w e^(M_w - M*) (l_w, O_w)
    __syncthreads();
    float* Mm = smem;                   // [W][NQ]
    float* Ml = smem + W * NQ;          // [W][NQ]
    float* Mo = smem + 2 * W * NQ;      // [W][NQ][MO]
    // V's unit and the weights' 2^15 out of the sums, by the exponent: their
    // quotient need not be a float
    const int ve = (int)(__float_as_uint(uv) >> 23) - 127 - 15;
#pragma unroll
    for (int f = 0; f < QF; f++) {
        if (g == 0) {
            Mm[wave * NQ + 16 * f + c] = M[f];
            Ml[wave * NQ + 16 * f + c] = lsum[f] * 0x1p-15f;
        }
#pragma unroll
        for (int u = 0; u < U; u++)
#pragma unroll
            for (int r = 0; r < 4; r++)
                *reinterpret_cast<float4*>(Mo + (wave * NQ + 16 * f + c) * MO + 64 * u + 16 * g + 4 * r) =
                    make_float4(ldexpf(oacc[f][u][0][r], ve), ldexpf(oacc[f][u][1][r], ve),
                                ldexpf(oacc[f][u][2][r], ve), ldexpf(oacc[f][u][3][r], ve));
    }
    __syncthreads();
    // thread x finishes float4 column x % (HDP / 4) of queries x / (HDP / 4), ...:
    // whole 16-byte runs of an output row per wave
    constexpr int QPT = W * 64 / (HDP / 4);  // queries per step of the block
    constexpr int NO = (NQ + QPT - 1) / QPT;
    const int d4 = tid % (HDP / 4), part = tid / (HDP / 4);
    float4 o[NO];
    uint32_t masked = 0;  // bit n: no key of query part + n QPT counts
    bool odd = *flags != 0;
#pragma unroll
    for (int n = 0; n < NO; n++) {
        const int q = part + n * QPT;
        o[n] = make_float4(0.f, 0.f, 0.f, 0.f);
        if (q >= NQ || q0 + q >= a.seq_q) continue;
        float mw[W], ms = -INFINITY;
#pragma unroll
        for (int w = 0; w < W; w++) {
            mw[w] = Mm[w * NQ + q];
            ms = fmaxf(ms, mw[w]);
        }
        if (ms == -INFINITY) {
            masked |= 1u << n;
            continue;
        }
        float l = 0.0f;
#pragma unroll
        for (int w = 0; w < W; w++) {
            const float fw = mw[w] == -INFINITY ? 0.0f : fast_exp2((mw[w] - ms) * kLog2e);
            l += fw * Ml[w * NQ + q];
            const float4 v = *reinterpret_cast<const float4*>(Mo + (w * NQ + q) * MO + 4 * d4);
            o[n].x += fw * v.x;
            o[n].y += fw * v.y;
            o[n].z += fw * v.z;
            o[n].w += fw * v.w;
        }
        const float inv = 1.0f / l;
        o[n] = make_float4(o[n].x * inv, o[n].y * inv, o[n].z * inv, o[n].w * inv);
        odd = odd || !(fabsf(o[n].x) + fabsf(o[n].y) + fabsf(o[n].z) + fabsf(o[n].w) < INFINITY);
    }
    if (__syncthreads_or(odd || masked)) {
        // not finite: from an input that this query sees, or 0 times one that
        // it does not
        if (__syncthreads_or(odd)) {
            attn_block_f32<HDP>(a, q0, NQ, h, kvh);
            return;
        }
        // rows with every key blocked: the uniform mean of V over all seq_k keys,
        // the same for each of them, from partial sums over 4 W strided key sets
        // (in Mm's place: every thread is past it)
        float4 sum = make_float4(0.f, 0.f, 0.f, 0.f);
        if (4 * d4 < HD)
            for (int j = part; j < a.seq_k; j += QPT) {
                const float4 v = *reinterpret_cast<const float4*>(Vb + (size_t)j * a.ldv + 4 * d4);
                sum.x += v.x;
                sum.y += v.y;
                sum.z += v.z;
                sum.w += v.w;
            }
        *reinterpret_cast<float4*>(smem + part * HDP + 4 * d4) = sum;
        __syncthreads();
        float4 mean = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int x = 0; x < QPT; x++) {
            const float4 v = *reinterpret_cast<const float4*>(smem + x * HDP + 4 * d4);
            mean.x += v.x;
            mean.y += v.y;
            mean.z += v.z;
            mean.w += v.w;
        }
        const float inv = 1.0f / (float)a.seq_k;
#pragma unroll
        for (int n = 0; n < NO; n++)
            if ((masked >> n) & 1u) o[n] = make_float4(mean.x * inv, mean.y * inv, mean.z * inv, mean.w * inv);
    }
#pragma unroll
    for (int n = 0; n < NO; n++) {
        const int q = part + n * QPT;
        if (q < NQ && q0 + q < a.seq_q && 4 * d4 < HD)
            *reinterpret_cast<float4*>(a.out + (size_t)(q0 + q) * a.ldo + h * HD + 4 * d4) = o[n];
    }
}

template <int HDP, int QF, int W, int MKC, bool FULL>
void launch_split_kd(const AttnArgs& a, hipStream_t st) {
    using C = SplitCfg<HDP, QF, W>;
    static const bool attr = [] {
        if (C::LDS > 65536)
            VLA_HIP_CHECK(hipFuncSetAttribute(reinterpret_cast<const void*>(&attn_split<HDP, QF, W, MKC, FULL>),
                                              hipFuncAttributeMaxDynamicSharedMemorySize, C::LDS));
        return true;
    }();
    (void)attr;
    attn_split<HDP, QF, W, MKC, FULL>
        <<<dim3((a.seq_q + 16 * QF - 1) / (16 * QF), a.n_q), W * 64, C::LDS, st>>>(a, {1.0f / (float)((a.seq_q + 16 * QF - 1) / (16 * QF)), 1.0f / (float)a.n_q,
                                      1.0f / (float)(a.n_q / a.n_kv)});
}

template <int HDP, int QF, int W, bool FULL>
void launch_split_w(const AttnArgs& a, hipStream_t st) {
    if (a.mask_kind == 1) launch_split_kd<HDP, QF, W, 1, FULL>(a, st);
    else if (a.mask_kind == 3) launch_split_kd<HDP, QF, W, 3, FULL>(a, st);
    else launch_split_kd<HDP, QF, W, 0, FULL>(a, st);
}

// Query fragments and waves per block, from the sizes alone (a dense mask of
// zeros must take the same waves as no mask: the merge order is theirs).
// QF: the fewest 16-query fragments whose blocks fit one round of the 256 CUs
// (a block of 8 waves, or of 4 at head_dim 128, fills a CU's registers), else
// the most: every fragment more divides the K/V traffic and the splitting, a
// second round costs as much as the first. Measured, us (fp32 matrix cores |
// QF 1, 2, 3, 4 at 8 waves): 1024 x 1024 x 12 heads 39.6 | 38.1 33.3 35.2 24.5; 690 x
// 690 x 12, block-causal 26.1 | 27.7 23.5 19.1 25.6; 512 x 512 x 12 16.9 | 17.6
// 12.3 13.0 15.3; 302 x 302 x 8 8.1 | 8.3 10.4 10.2 13.6; heads of 32: 1024 x 1024 x
// 12 QF 1, 2, 4 37.6 33.2 25.2, 512 x 512 x 12 17.5 12.2 15.7; heads of 48: 1024 x 1024
// x 8 26.6 18.2 24.4.
// W: 8 waves from 9 tiles of 32 keys on, 4 for 3 to 8 (50 x 227 x 15 heads 9.0
// against 9.2, heads of 32 x 8 7.0 against 7.4), 2 below (50 x 64 x 8 4.85 against
// 4.98). head_dim 128 has the registers for 4: QF 1 or 2 at 4 waves | at 2, 302 x 302
// x 8 13.3 17.0 | 17.2 21.8; 512 x 512 x 16 29.1 20.2 | 25.1 30.2; 1024 x 1024 x 8 45.3
// 31.5 | 40.8 52.2; 50 x 64 x 8 7.2 9.8 | 7.0 9.4.
template <int HDP, bool FULL>
void run_split(const AttnArgs& a, hipStream_t st) {
    const int tiles = (a.seq_k + 31) / 32;
    const long frags = (a.seq_q + 15) / 16;
    auto fits = [&](int qf) { return (frags + qf - 1) / qf * a.n_q <= 256; };
    if constexpr (HDP == 128) {
        if (fits(1)) launch_split_w<HDP, 1, 4, FULL>(a, st);
        else launch_split_w<HDP, 2, 4, FULL>(a, st);
    } else if (tiles <= 2) {
        launch_split_w<HDP, 1, 2, FULL>(a, st);
    } else if (tiles <= 8) {
        if (fits(1)) launch_split_w<HDP, 1, 4, FULL>(a, st);
        else launch_split_w<HDP, 2, 4, FULL>(a, st);
    } else {
        if (fits(1)) launch_split_w<HDP, 1, 8, FULL>(a, st);
        else if (fits(2)) launch_split_w<HDP, 2, 8, FULL>(a, st);
        else if (FULL && fits(3)) launch_split_w<HDP, FULL ? 3 : 4, 8, FULL>(a, st);
        else launch_split_w<HDP, 4, 8, FULL>(a, st);
    }
    VLA_LAUNCH_CHECK();
}

// attn_fwd's waves, for heads of 129 to 256: enough that each walks a few key tiles,
// at most 4 (LDS).
void run_attn(const AttnArgs& a, hipStream_t st) {
    int kv = a.seq_k;
    if (a.mask_kind == 2) {  // keys no query of the problem can see are never walked
        const int e = a.seq_q + a.causal_offset;
        kv = e < 1 ? 1 : (e < kv ? e : kv);
    }
    const int tiles = (kv + 15) / 16;
    if (tiles <= 1) launch_w<256, 16, 1>(a, st);
    else if (tiles <= 2) launch_w<256, 16, 2>(a, st);
    else launch_w<256, 16, 4>(a, st);
    VLA_LAUNCH_CHECK();
}

}  // namespace

void launch_attention(const AttnArgs& a, hipStream_t st) {
    VLA_REQUIRE(a.seq_q >= 0 && a.seq_k > 0 && a.n_q > 0 && a.n_kv > 0,
                "attention: need seq_q >= 0, seq_k > 0, n_q > 0, n_kv > 0");
    VLA_REQUIRE(a.n_q % a.n_kv == 0, "attention: n_q must be a multiple of n_kv");
    VLA_REQUIRE(a.head_dim > 0 && a.head_dim <= 256 && a.head_dim % 4 == 0,
                "attention: head_dim must be a multiple of 4 in [4, 256]");
    VLA_REQUIRE(a.ldq % 4 == 0 && a.ldk % 4 == 0 && a.ldv % 4 == 0 && a.ldo % 4 == 0,
                "attention: row strides must be multiples of 4 floats");
    VLA_REQUIRE(aligned(a.Q, 16) && aligned(a.K, 16) && aligned(a.V, 16) && aligned(a.out, 16),
                "attention: Q, K, V and out must be 16-byte aligned");
    VLA_REQUIRE(a.ldq >= a.n_q * a.head_dim && a.ldo >= a.n_q * a.head_dim &&
                    a.ldk >= a.n_kv * a.head_dim && a.ldv >= a.n_kv * a.head_dim,
                "attention: row stride shorter than heads * head_dim");
    VLA_REQUIRE(a.mask_kind >= 0 && a.mask_kind <= 3, "attention: unknown mask kind");
    VLA_REQUIRE(a.mask_kind != 1 || (a.mask && a.ldm >= a.seq_k), "attention: dense mask missing");
    VLA_REQUIRE(a.mask_kind != 3 || (a.q_group && a.k_group && a.allow && a.n_groups > 0 &&
                                     a.n_groups <= 256),
                "attention: group mask needs q_group, k_group, allow and 1..256 groups");
    if (a.seq_q == 0) return;
    // (lengths and strides past the block index's and offsets' range)
    const bool split = std::isfinite(a.scale) && a.head_dim <= 128 && a.ldk < (1 << 24) && a.ldv < (1 << 24) &&
                       (long)((a.seq_q + 15) / 16) * a.n_q < (1 << 20);
    if (!split) run_attn(a, st);
    else if (a.head_dim == 64) run_split<64, true>(a, st);
    else if (a.head_dim < 64) run_split<64, false>(a, st);
    else if (a.head_dim == 128) run_split<128, true>(a, st);
    else run_split<128, false>(a, st);
}

}  // namespace hip
}  // namespace vla
