// attn.hip — the gated full-attention layer of the Qwen3.5/3.6 engine
// (engines/qwen.c:366-425, attn_step), the layer that every fourth block runs
// beside the GDN layers, for T new tokens of one sequence at positions
// pos .. pos+T-1.
//
// After the qkv projection (one launch_proj over the concatenated rows
// [H x (q | gate), KV x k, KV x v], qwen.c:370-374) three launches:
//  1. attn_prep_kernel, one workgroup per token (its RoPE cos / sin computed
//     once, then a wave per head row; decode steps do this inside the split
//     kernel instead): RMSNorm of q and k with
//     (1 + w) weights (qwen.c:148-152, 385-386), partial RoPE over the first
//     rot dims as two non-interleaved halves (qwen.c:388-398, inverse
//     frequencies computed on the host as there), then q into a scratch row
//     and k, v into the sequence's cache rows pos + t (qwen.c:400-404).
//  2. the split kernel, flash-decoding: a workgroup reads the K and V rows of
//     one key split of one kv head once for the query heads of its group
//     (GQA, qwen.c:408-409), keeps a running max and sum per head (online
//     softmax) and writes unnormalised partials.  Head widths of 64 and
//     more: attn_split_mfma_kernel, K and V from HBM straight into fp32 MFMA
//     operands whose 16 columns are (token, head) pairs of the group.  Width
//     32: attn_split_kernel, a workgroup per token, 64-key tiles
//     staged through LDS, lane = key for the scores (q broadcast from LDS),
//     lane = 4 output columns for P.V (each key's weight by readlane).
//  3. attn_combine_kernel, per (token, head, 64 columns): merges the splits,
//     normalises, and applies the output gate sigmoid(gate) (qwen.c:421).
// The o_proj is a second launch_proj.
//
// Decode is HBM-bound on the visible cache: 2 * KV * n * hd * 4 bytes for
// n = pos + 1 keys; the splits fill the CUs once (one workgroup per CU, as
// the LDS footprint allows).  Token t
// sees keys 0 .. pos+t (causal), and the key tiles beyond that are masked.
#include "omh_internal.h"
#include "omh_device.h"

#include <algorithm>
#include <cmath>

namespace omh {
namespace {

template <int HD>
struct AttnShape {
    static constexpr int KT = 64;                 // keys per tile
    static constexpr int KS = HD + 4;             // padded K row in LDS (floats)
    static constexpr int NG4 = HD / 4;            // float4 groups per row
    static constexpr int R4 = (NG4 + OMH_WAVE - 1) / OMH_WAVE;   // groups per lane in P.V
    static constexpr int NW = 8;                  // waves (two per SIMD)
    static constexpr size_t LDS = (size_t)(kAttnMaxGroup * HD + KT * KS + KT * HD) * sizeof(float);
};

__device__ __forceinline__ float wave_max(float v) { return omh_lane_max(v); }

// cos and sin of p * inv[j] for j < rot / 2 into LDS tables, by the threads
// of a workgroup.  One out-of-line function computes them wherever a kernel
// needs them, so every kernel rotates with the same bits.
__device__ __attribute__((noinline)) void rope_cos_sin(float ang, float *c, float *s) {
    *c = cosf(ang);
    *s = sinf(ang);
}
__device__ __forceinline__ void rope_table(const AttnArgs &a, int p, float *cs, float *sn, int tid, int nthreads) {
    for (int j = tid; j < a.rot / 2; j += nthreads) rope_cos_sin((float)p * a.inv[j], cs + j, sn + j);
}

// One q or k row of the prep (RMSNorm with 1 + w, then partial RoPE as two
// non-interleaved halves), or a v row (no weights: copied), by one wave,
// into an LDS row (the RoPE pairs are read back from it).  cs_t / sn_t: the
// token's rope_table.  prep_row_regs takes the row (v, element lane + 64 i
// in v[i]) and the weights (wv, likewise) already in registers, so a caller
// can issue those loads ahead of others; prep_row loads them itself.  On
// return v holds the row as written (its fences order LDS only, so global
// loads a caller issued ahead stay in flight).
template <int HD>
__device__ __forceinline__ void prep_row_regs(const AttnArgs &a, float (&v)[(HD + OMH_WAVE - 1) / OMH_WAVE],
                                              const float (&wv)[(HD + OMH_WAVE - 1) / OMH_WAVE], bool norm, float *row,
                                              int lane, const float *cs_t, const float *sn_t) {
    constexpr int NE = (HD + OMH_WAVE - 1) / OMH_WAVE;
    if (norm) {
        float ss = 0.f;
#pragma unroll
        for (int i = 0; i < NE; i++) ss += v[i] * v[i];
        ss = omh_xor_sum_from<1>(ss);
        const float rr = 1.f / sqrtf(ss / (float)HD + a.eps);   // qwen.c:148-152
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int j = lane + OMH_WAVE * i;
            if (j < HD) {
                v[i] = v[i] * rr * (1.f + wv[i]);
                row[j] = v[i];
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");   // the wave's row is in LDS
        __builtin_amdgcn_wave_barrier();
        const int half = a.rot / 2;
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int j = lane + OMH_WAVE * i;
            if (j < a.rot) {                                     // qwen.c:388-398
                const int jj = j < half ? j : j - half;
                const float cs = cs_t[jj], sn = sn_t[jj];
                const float a0 = row[jj], b0 = row[jj + half];
                v[i] = j < half ? a0 * cs - b0 * sn : b0 * cs + a0 * sn;
            }
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup", "local");   // every lane has read its pair
        __builtin_amdgcn_wave_barrier();
    }
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const int j = lane + OMH_WAVE * i;
        if (j < HD) row[j] = v[i];
    }
}
template <int HD>
__device__ __forceinline__ void prep_row(const AttnArgs &a, const float *src, const float *w, float *row, int lane,
                                         const float *cs_t, const float *sn_t) {
    constexpr int NE = (HD + OMH_WAVE - 1) / OMH_WAVE;
    float v[NE], wv[NE];
#pragma unroll
    for (int i = 0; i < NE; i++) {
        const int j = lane + OMH_WAVE * i;
        v[i] = j < HD ? src[j] : 0.f;
        wv[i] = w && j < HD ? w[j] : 0.f;
    }
    prep_row_regs<HD>(a, v, wv, w != nullptr, row, lane, cs_t, sn_t);
}

// Whether v is finite and rounds to a finite bf16; and where in a token's
// projection row the prep leaves word of a v row (kv head g) that has a value
// of which this is not so: at the row's own first element, copied by then.
__device__ __forceinline__ bool bf16_finite(float v) { return fabsf(v) < 0x1.ffp127f; }
__device__ __forceinline__ int odd_flag_at(int H, int KV, int g, int hd) { return (2 * H + KV + g) * hd; }

// The prep: one workgroup of kPrepWaves waves per token (gridDim.y of them
// where tokens are few, each with its share of the rows).  The token's RoPE
// cos and sin (rot / 2 frequencies) go into LDS once, then wave w takes rows
// w, w + kPrepWaves, ... of [H q heads, KV k heads, KV v heads]: q into the
// scratch, k and v into the cache rows pos + t.  A wave's next row (and its
// norm weights) is requested before the current one is formed, and its
// first before the RoPE table, so the rows' HBM round trips overlap.
constexpr int kPrepWaves = 4;
template <int HD>
__global__ __launch_bounds__(kPrepWaves * OMH_WAVE) void attn_prep_kernel(const AttnArgs a) {
    constexpr int NE = (HD + OMH_WAVE - 1) / OMH_WAVE;
    __shared__ float cs[HD / 2], sn[HD / 2], sv[kPrepWaves][HD];
    const int H = a.H, KV = a.KV, nr = H + 2 * KV;
    const int t = blockIdx.x, tid = threadIdx.x, lane = tid % OMH_WAVE;
    const int wv = __builtin_amdgcn_readfirstlane(tid / OMH_WAVE);
    const int r0 = wv + kPrepWaves * blockIdx.y, rs = kPrepWaves * gridDim.y;   // this wave's first row, and the step
    const int p = a.pos + t;
    const float *row = a.qkv + (size_t)t * a.ld_qkv;
    // row r's source and norm weights (null: a v row, copied)
    auto src_of = [&](int r, const float *&w) -> const float * {
        if (r < H) { w = a.qn; return row + (size_t)r * 2 * HD; }                          // q of head r (then its gate)
        if (r < H + KV) { w = a.kn; return row + (size_t)2 * H * HD + (size_t)(r - H) * HD; }   // k of kv head r - H
        w = nullptr;
        return row + (size_t)2 * H * HD + (size_t)(r - H) * HD;                          // v of kv head r - H - KV
    };
    float v[NE], wt[NE];
    auto fetch = [&](int r) __attribute__((always_inline)) {
        const float *w;
        const float *src = src_of(r, w);
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int j = lane + OMH_WAVE * i;
            v[i] = j < HD ? src[j] : 0.f;
            wt[i] = w && j < HD ? w[j] : 0.f;
        }
    };
    if (r0 < nr) fetch(r0);
    rope_table(a, p, cs, sn, tid, kPrepWaves * OMH_WAVE);
    __syncthreads();
    for (int r = r0; r < nr; r += rs) {
        float cv[NE], cw[NE];
#pragma unroll
        for (int i = 0; i < NE; i++) {
            cv[i] = v[i];
            cw[i] = wt[i];
        }
        if (r + rs < nr) fetch(r + rs);
        float *dst;
        if (r < H) dst = a.qb + ((size_t)t * H + r) * HD;
        else if (r < H + KV) dst = a.Kc + (((size_t)a.seq * KV + (r - H)) * a.max_t + p) * HD;
        else dst = a.Vc + (((size_t)a.seq * KV + (r - H - KV)) * a.max_t + p) * HD;
        prep_row_regs<HD>(a, cv, cw, r < H + KV, sv[wv], lane, cs, sn);
#pragma unroll
        for (int i = 0; i < NE; i++) {
            const int j = lane + OMH_WAVE * i;
            if (j < HD) dst[j] = cv[i];
        }
        if (gridDim.y == 1 && r >= H + KV) {       // (flash steps among them)
            bool odd = false;
#pragma unroll
            for (int i = 0; i < NE; i++) odd |= !bf16_finite(cv[i]);
            const bool any = __builtin_amdgcn_ballot_w64(odd) != 0;
            if (lane == 0) a.qkv[(size_t)t * a.ld_qkv + odd_flag_at(H, KV, r - H - KV, HD)] = any ? 1.f : 0.f;
        }
    }
}


// GPW = query heads per wave (the group's heads grp spread over the NW
// waves: head wave + NW*i).  The hot loops carry no per-head conditions (a
// branch there serialises every LDS read behind its own wait): a wave
// whose head index runs past grp computes a copy of head grp-1 and does not
// write it.
// PREP (decode steps, T = 1): the prep kernel's work is done here instead
// of in a launch of its own: every workgroup forms its group's q rows
// straight into LDS, and the workgroup whose split holds position pos writes
// the new k and v rows into the cache before it reads any tile.
template <int HD, int GPW, bool PREP = false>
__global__ __launch_bounds__(AttnShape<HD>::NW * OMH_WAVE) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_split_kernel(const AttnArgs a) {   // one workgroup per CU (LDS): all of each SIMD's registers
    using S = AttnShape<HD>;
    constexpr int R4 = S::R4, NG4 = S::NG4, KT = S::KT, NW = S::NW, NT = NW * OMH_WAVE;
    extern __shared__ float smem[];
    float *qs = smem;                              // [group heads][HD]
    float *Ks = qs + kAttnMaxGroup * HD;           // [KT][KS]
    float *Vs = Ks + KT * S::KS;                   // [KT][HD]

    const int H = a.H, KV = a.KV, grp = H / KV, ns = a.ns;
    const int s = blockIdx.x % ns, g = (blockIdx.x / ns) % KV, t = blockIdx.x / (ns * KV);
    const int tid = threadIdx.x, lane = tid % OMH_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / OMH_WAVE);
    const int n = a.pos + t + 1;                   // keys token t sees
    const int k0 = s * a.kps, k1 = min(n, k0 + a.kps);
    // partial of query head g*grp + i: index pb + i*ns
    const size_t pb = ((size_t)t * H + (size_t)g * grp) * ns + s;
    if (k0 >= k1) {                                // an empty split: weight zero in the merge
        for (int e = tid; e < grp * NG4; e += NT) {
            const size_t pi = pb + (size_t)(e / NG4) * ns;
            *reinterpret_cast<float4 *>(a.po + pi * HD + 4 * (e % NG4)) = f4_zero();
            if (e % NG4 == 0) {
                a.pml[2 * pi] = -INFINITY;
                a.pml[2 * pi + 1] = 0.f;
            }
        }
        return;
    }
    if constexpr (PREP) {
        const int p = a.pos + t;
        const float *row = a.qkv + (size_t)t * a.ld_qkv;
        float *cs = Ks + HD, *sn = cs + HD / 2;     // (the K tile region is free until the first tile)
        rope_table(a, p, cs, sn, tid, NT);
        __syncthreads();
        if (k0 <= p && p < k1) {
            // the new k (wave 0, normed and rotated through a scratch LDS row)
            // and v (wave 1) of kv head g go into the cache rows p
            const size_t crow = (((size_t)a.seq * KV + g) * a.max_t + p) * HD;
            if (wave == 0) {
                prep_row<HD>(a, row + (size_t)2 * H * HD + (size_t)g * HD, a.kn, Ks, lane, cs, sn);
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                __builtin_amdgcn_wave_barrier();
                for (int j = lane; j < HD; j += OMH_WAVE) a.Kc[crow + j] = Ks[j];
            } else if (wave == 1) {
                for (int j = lane; j < HD; j += OMH_WAVE) a.Vc[crow + j] = row[(size_t)2 * H * HD + (size_t)(KV + g) * HD + j];
            }
            __threadfence();                       // the rows are in memory before any tile load reads them
            __syncthreads();
        }
        for (int i = wave; i < grp; i += NW)
            prep_row<HD>(a, row + (size_t)(g * grp + i) * 2 * HD, a.qn, qs + i * HD, lane, cs, sn);
    } else {
        for (int e = tid; e < grp * NG4; e += NT) {
            const int i = e / NG4, c = e % NG4;
            *reinterpret_cast<float4 *>(qs + i * HD + 4 * c) =
                *reinterpret_cast<const float4 *>(a.qb + ((size_t)t * H + (size_t)g * grp + i) * HD + 4 * c);
        }
    }
    const float *qh[GPW];                          // this wave's heads' q rows in LDS
#pragma unroll
    for (int i = 0; i < GPW; i++) qh[i] = qs + min(wave + NW * i, grp - 1) * HD;
    float m[GPW], l[GPW];
    float4 o[GPW][R4];
#pragma unroll
    for (int i = 0; i < GPW; i++) {
        m[i] = -INFINITY;
        l[i] = 0.f;
#pragma unroll
        for (int r = 0; r < R4; r++) o[i][r] = f4_zero();
    }
    const size_t cache0 = ((size_t)a.seq * KV + g) * a.max_t;
    const float *Kg = a.Kc + cache0 * HD, *Vg = a.Vc + cache0 * HD;

    // K and V tiles go HBM -> registers -> LDS: every thread's PER pieces of
    // a tile are in flight at once, and the next tile's loads are issued as
    // soon as the current one is in LDS, so they overlap its compute.  Rows
    // past the split's end repeat the tile's first row, so every LDS row
    // holds finite values (their weights are zero).
    constexpr int PER = KT * NG4 / NT;
    static_assert(KT * NG4 % NT == 0, "tile pieces per thread");
    omh_v4f kr[PER], vr[PER];                      // native vectors: HIP's float4 copies stay in scratch
#define OMH_ATTN_LOAD_PIECE(I, KT0, NK)                                                   \
    {                                                                                     \
        const int e = tid + NT * (I), kk = e / NG4, c = e % NG4;                          \
        const size_t off = (size_t)((KT0) + (kk < (NK) ? kk : 0)) * HD + 4 * c;           \
        kr[I] = *reinterpret_cast<const omh_v4f *>(Kg + off);                             \
        vr[I] = *reinterpret_cast<const omh_v4f *>(Vg + off);                             \
    }
#pragma unroll
    for (int i = 0; i < PER; i++) OMH_ATTN_LOAD_PIECE(i, k0, min(KT, k1 - k0))
    for (int kt = k0; kt < k1; kt += KT) {
        const int nk = min(KT, k1 - kt);
        omh_lds_barrier();                         // the previous tile's readers are done
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int e = tid + NT * i, kk = e / NG4, c = e % NG4;
            *reinterpret_cast<omh_v4f *>(Ks + kk * S::KS + 4 * c) = kr[i];
            *reinterpret_cast<omh_v4f *>(Vs + kk * HD + 4 * c) = vr[i];
        }
        omh_lds_barrier();
        // the next tile's pieces are issued spread over the score blocks
        // below; after the last tile they re-read this one (cache hits)
        const bool more = kt + KT < k1;
        const int kn = more ? kt + KT : kt, nkn = more ? min(KT, k1 - kt - KT) : nk;

        // scores q.k * hd^-1/2 (qwen.c:410-414), lane = key
        const bool valid = lane < nk;
        const float *kr_l = Ks + lane * S::KS;
        float acc[GPW], pl[GPW];
#pragma unroll
        for (int i = 0; i < GPW; i++) acc[i] = 0.f;
        constexpr int CB = 8, NB = NG4 / CB, PPB = (PER + NB - 1) / NB;
        static_assert(NG4 % CB == 0, "score blocks");
#pragma unroll
        for (int b = 0; b < NB; b++) {
#pragma unroll
            for (int u = 0; u < PPB; u++)
                if (b * PPB + u < PER) OMH_ATTN_LOAD_PIECE(b * PPB + u, kn, nkn)
#pragma unroll
            for (int cc = 0; cc < CB; cc++) {
                const int c = b * CB + cc;
                const float4 kv = *reinterpret_cast<const float4 *>(kr_l + 4 * c);
#pragma unroll
                for (int i = 0; i < GPW; i++) {
                    const float4 q = *reinterpret_cast<const float4 *>(qh[i] + 4 * c);
                    acc[i] = fmaf(q.x, kv.x, acc[i]);
                    acc[i] = fmaf(q.y, kv.y, acc[i]);
                    acc[i] = fmaf(q.z, kv.z, acc[i]);
                    acc[i] = fmaf(q.w, kv.w, acc[i]);
                }
            }
        }
        // online softmax (qwen.c:413 softmax_ over all keys, merged per tile)
#pragma unroll
        for (int i = 0; i < GPW; i++) {
            const float sc = valid ? acc[i] * a.scale : -INFINITY;
            const float mn = fmaxf(m[i], wave_max(sc));
            const float corr = expf(m[i] - mn);
            const float pe = valid ? expf(sc - mn) : 0.f;
            l[i] = l[i] * corr + omh_xor_sum_from<1>(pe);
#pragma unroll
            for (int r = 0; r < R4; r++) o[i][r] = f4_scale(o[i][r], corr);
            pl[i] = pe;
            m[i] = mn;
        }

        // P.V (qwen.c:415-419), lane = 4 columns; the weight of key kk is
        // lane kk's pl (zero past nk), broadcast by readlane
#pragma unroll 8
        for (int kk = 0; kk < KT; kk++) {
            float4 vv[R4];
#pragma unroll
            for (int r = 0; r < R4; r++) {
                const int c = min(lane + OMH_WAVE * r, NG4 - 1);
                vv[r] = *reinterpret_cast<const float4 *>(Vs + kk * HD + 4 * c);
            }
#pragma unroll
            for (int i = 0; i < GPW; i++) {
                const float pv = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, pl[i]), kk));
#pragma unroll
                for (int r = 0; r < R4; r++) o[i][r] = f4_fma(vv[r], pv, o[i][r]);
            }
        }
    }
#pragma unroll
    for (int i = 0; i < GPW; i++) {
        const int h = wave + NW * i;
        if (h < grp) {
            const size_t pi = pb + (size_t)h * ns;
#pragma unroll
            for (int r = 0; r < R4; r++) {
                const int c = lane + OMH_WAVE * r;
                if (c < NG4) *reinterpret_cast<float4 *>(a.po + pi * HD + 4 * c) = o[i][r];
            }
            if (lane == 0) {
                a.pml[2 * pi] = m[i];
                a.pml[2 * pi + 1] = l[i];
            }
        }
    }
}
#undef OMH_ATTN_LOAD_PIECE

// ---------------------------------------------------------------- decode on the matrix cores
// The split kernel for head widths of 64 and more: one workgroup takes one
// key split of one kv head for a column tile of 16 (token, query head) pairs
// of its group (a decode step: the one token's heads, the prep folded in),
// with K and V going from HBM straight into fp32 MFMA operands, so every key
// row is read once for the 16 columns (no LDS staging, no per-head re-reads).
// Steps of 2 to 63 tokens took a workgroup per token before, 8 of the 16
// columns in use at 8 heads a group and the cache read again for every token:
// 5 tokens at position 8001 (16 heads on 2 kv heads, width 256) 47.3 us (260
// workgroups, two rounds of the CUs), as column tiles 21.3 us (252).  Tried:
// a block's K and V rows in registers of their own, the next block's loads
// ahead: 25.5 us (and a decode step at position 32767 37.0 us for 34.4).
// Each of the NW waves streams its own 16-key blocks (blocks w, w + NW, ...) and keeps its own online softmax.
// A wave holds one operand set: a block's K rows, then (once the scores are
// formed) its V rows in the same registers; the two waves of a SIMD overlap
// one's loads with the other's products:
//   S^T = K Q^T   (v_mfma_f32_16x16x4_f32; A = K rows, lane l16 = key;
//                  B = q from LDS, lane l16 = column, columns past
//                  the tile's last zero; head dims taken in the order 16 i + 4 g + s
//                  on both operands, one 16-byte K load per 4 products),
//   O += P V      (A = the probabilities as the score product left them:
//                  key 4 g + s of lane group g is register s; B = V rows
//                  4 g + s, lane l16 = output columns 64 q + 4 l16 + c of
//                  tile 4 q + c, so one 16-byte V load serves 4 tiles).
// The waves' (max, sum, O) then merge through LDS into the split's partial,
// which the combine kernel merges with the other splits as before.  Keys
// past the split's end (their rows repeat its last one) and keys past a
// column's own position are masked; values that are not finite reach only
// the tokens that see them.
template <int HD>
struct MfmaSplitShape {
    static constexpr int NW = 8;                   // waves, two per SIMD
    static constexpr int QS = HD + 4;              // padded q row in LDS
    static constexpr int NI = HD / 16;             // K float4s per lane per block (4 k-steps each)
    static constexpr int NQ = HD / 64;             // V float4s per lane per key step
    static constexpr size_t LDS = (size_t)(kAttnMaxGroup * QS + NW * 16 * HD + 2 * NW * 16) * sizeof(float);
    static_assert(HD % 64 == 0, "64-column V groups");
};

// The token p / grp of (token, head) pair p without a division (five of them
// before a step's first load cost 0.3 us): the high half of p times
// r = ceil(2^32 / grp), exact while p (r grp - 2^32) < 2^32, so below 2^32 / 15
// pairs; a cache of 2^31 bytes holds 2^23 tokens of width 64, 2^27 pairs.
constexpr unsigned group_recip(int grp) { return grp > 1 ? 0xffffffffu / (unsigned)grp + 1 : 0; }
__host__ __device__ constexpr int pair_token(int p, unsigned r) { return r ? (int)((uint64_t)(unsigned)p * r >> 32) : p; }
constexpr bool pair_tokens_exact() {
    for (int grp = 1; grp <= kAttnMaxGroup; grp++)
        for (int t : {1, 2, 63, 155697, 339538, 1048576, (1 << 23) - 1}) {
            const unsigned r = group_recip(grp);
            if (pair_token(t * grp - 1, r) != t - 1 || pair_token(t * grp, r) != t || pair_token(t * grp + grp - 1, r) != t) return false;
        }
    return true;
}
static_assert(pair_tokens_exact(), "pair_token at the ends of a token's heads");

// NT: streamed past the caches (one reader)
template <bool NT>
__device__ __forceinline__ omh_v4f ld_buf_v4(__amdgpu_buffer_rsrc_t r, int off) {
    return __builtin_bit_cast(omh_v4f, __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, NT ? kOmhNT : 0));
}

template <int HD, bool PREP>
__global__ __launch_bounds__(MfmaSplitShape<HD>::NW * OMH_WAVE, 1) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_split_mfma_kernel(const AttnArgs a) {
    using S = MfmaSplitShape<HD>;
    constexpr int NW = S::NW, NT = NW * OMH_WAVE, QS = S::QS, NI = S::NI, NQ = S::NQ;
    extern __shared__ float smem[];
    float *qs = smem;                              // [kAttnMaxGroup][QS] the columns' q rows
    float *mo = qs + kAttnMaxGroup * QS;           // [NW][16][HD] the waves' outputs (the prep's scratch before)
    float *mm = mo + NW * 16 * HD;                 // [NW][16] running max, then [NW][16] sums

    const int H = a.H, KV = a.KV, grp = H / KV, ns = a.ns;
    // unit (key split s, kv head g) and column tile ct; a unit's tiles run
    // side by side on one XCD (workgroup i on XCD i mod 8), which then reads
    // the unit's keys from memory once.  (A decode step is one tile of one
    // token, and knows it: with the general form's quotients before its first
    // load a step at position 57 took 17.1 us for 16.9, 8 heads on 2 kv heads
    // of 128, and 26.7 for 26.4, 16 on 2 of 256.)
    const int nct = PREP ? 1 : (a.T * grp + 15) / 16, nu = ns * KV;
    const bool spread = !PREP && nu % 8 == 0;
    const int ct = PREP ? 0 : spread ? (int)blockIdx.x / 8 % nct : (int)blockIdx.x % nct;
    const int unit = spread ? (int)blockIdx.x / (8 * nct) * 8 + (int)blockIdx.x % 8 : (int)blockIdx.x / nct;
    const int s = unit % ns, g = unit / ns;
    const int tid = threadIdx.x, lane = tid % OMH_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / OMH_WAVE);
    const int l16 = lane % 16, g4 = lane / 16;
    // column c of the tile is (token, head) pair c0 + c of the group's
    // T * grp, head fastest
    const unsigned rgrp = PREP ? 0 : a.rgrp;
    auto token_of = [&](int c) __attribute__((always_inline)) { return PREP ? 0 : pair_token(c, rgrp); };
    const int c0 = 16 * ct, ncol = PREP ? grp : min(16, a.T * grp - c0);
    const int tlast = token_of(c0 + ncol - 1);
    const int n = a.pos + tlast + 1;               // keys the tile's last token sees
    const int k0 = s * a.kps, k1 = min(n, k0 + a.kps);
    // partial and q row of column c
    auto row_of = [&](int c) __attribute__((always_inline)) {
        const int t = token_of(c0 + c);
        return (size_t)(t * H + g * grp + c0 + c - t * grp);
    };
    if (k0 >= k1) {                                // an empty split: weight zero in the merge
        for (int e = tid; e < ncol * (HD / 4); e += NT) {
            const size_t pi = row_of(e / (HD / 4)) * ns + s;
            *reinterpret_cast<float4 *>(a.po + pi * HD + 4 * (e % (HD / 4))) = f4_zero();
            if (e % (HD / 4) == 0) {
                a.pml[2 * pi] = -INFINITY;
                a.pml[2 * pi + 1] = 0.f;
            }
        }
        return;
    }
    const size_t cache0 = ((size_t)a.seq * KV + g) * a.max_t * HD;
    const int cbytes = a.max_t * HD * (int)sizeof(float);          // (launch_attn_d checks the range)
    const __amdgpu_buffer_rsrc_t krs = omh_rsrc(a.Kc + cache0, cbytes), vrs = omh_rsrc(a.Vc + cache0, cbytes);
    const int nb = (k1 - k0 + 15) / 16;            // 16-key blocks of the split
    // one operand set: a block's K rows (lane (l16, g4): key l16, dims
    // 16 i + 4 g4 .. +3 in kv[i]), then its V rows (key 4 g4 + st, columns
    // 64 q + 4 l16 .. +3 in kv[NQ st + q])
    static_assert(NI == 4 * NQ, "K and V fill the same registers");
    omh_v4f kv[NI];
    auto load_k = [&](int b) __attribute__((always_inline)) {
        const int kk = min(k0 + 16 * b + l16, k1 - 1);
#pragma unroll
        for (int i = 0; i < NI; i++) kv[i] = ld_buf_v4<PREP>(krs, (kk * HD + 16 * i + 4 * g4) * 4);
    };
    auto load_v = [&](int b) __attribute__((always_inline)) {
#pragma unroll
        for (int st = 0; st < 4; st++) {
            const int kr = min(k0 + 16 * b + 4 * g4 + st, k1 - 1);
#pragma unroll
            for (int q = 0; q < NQ; q++) kv[NQ * st + q] = ld_buf_v4<PREP>(vrs, (kr * HD + 64 * q + 4 * l16) * 4);
        }
    };
    // Prologue.  A decode step's RoPE table comes first (its out-of-line
    // cos / sin call waits for every load the wave has in flight), and the
    // split holding the step's position writes the new k / v cache rows.
    // Then the loads the q prep needs (the group's q rows, the norm weights)
    // and the first K / V block of the wave go out, in that order, in
    // straight-line code: loads complete in issue order, so the prep's waits
    // leave the block's loads in flight.  A prompt step's prepared q rows go
    // to LDS before the block loads.
    // (decode steps: one token, its group's heads in one tile)
    const int p = a.pos;
    if constexpr (PREP) {
        const float *row = a.qkv;
        float *krow = mo, *cs = mo + HD, *sn = cs + HD / 2;
        rope_table(a, p, cs, sn, tid, NT);
        __syncthreads();
        if (k0 <= p && p < k1) {
            // the new k (wave 0, normed and rotated through a scratch LDS row)
            // and v (wave 1) of kv head g go into the cache rows p
            const size_t crow = (((size_t)a.seq * KV + g) * a.max_t + p) * HD;
            if (wave == 0) {
                prep_row<HD>(a, row + (size_t)2 * H * HD + (size_t)g * HD, a.kn, krow, lane, cs, sn);
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                __builtin_amdgcn_wave_barrier();
                for (int j = lane; j < HD; j += OMH_WAVE) a.Kc[crow + j] = krow[j];
            } else if (wave == 1) {
                for (int j = lane; j < HD; j += OMH_WAVE) a.Vc[crow + j] = row[(size_t)2 * H * HD + (size_t)(KV + g) * HD + j];
            }
            __threadfence();                       // the rows are in memory before any block load reads them
            __syncthreads();
        }
        constexpr int NE = HD / OMH_WAVE, MAXH = (kAttnMaxGroup + NW - 1) / NW;
        float xv[MAXH][NE], wn[NE];
#pragma unroll
        for (int k = 0; k < MAXH; k++) {
            const int i = min(wave + NW * k, grp - 1);
#pragma unroll
            for (int e = 0; e < NE; e++) xv[k][e] = row[(size_t)(g * grp + i) * 2 * HD + lane + OMH_WAVE * e];
        }
#pragma unroll
        for (int e = 0; e < NE; e++) wn[e] = a.qn[lane + OMH_WAVE * e];
#pragma unroll
        for (int k = 0; k < MAXH; k++) {
            const int i = wave + NW * k;
            if (i < grp) prep_row_regs<HD>(a, xv[k], wn, true, qs + i * QS, lane, cs, sn);
        }
        load_k(wave);
    } else {
        for (int e = tid; e < ncol * (HD / 4); e += NT) {
            const int i = e / (HD / 4), c = e % (HD / 4);
            *reinterpret_cast<float4 *>(qs + i * QS + 4 * c) =
                *reinterpret_cast<const float4 *>(a.qb + row_of(i) * HD + 4 * c);
        }
        load_k(wave);
    }
    // (LDS-only barriers from here on: a full __syncthreads would also wait
    // for the block loads in flight)
    omh_lds_barrier();
    // q as the B operand: lane (g4, column l16) reads q[l16][16 i + 4 g4 .. +3]
    // (columns past the tile's last read as zero)
    if (ncol < 16) {
        for (int e = tid; e < (16 - ncol) * (HD / 4); e += NT)
            *reinterpret_cast<float4 *>(qs + (ncol + e / (HD / 4)) * QS + 4 * (e % (HD / 4))) = f4_zero();
        omh_lds_barrier();
    }
    const int kend = min(k1, a.pos + token_of(c0 + min(l16, ncol - 1)) + 1);   // keys this lane's column sees end here
    const float *qrow = qs + l16 * QS + 4 * g4;

    float m = -INFINITY, l = 0.f;                  // of column l16 (the same in the four lane groups)
    omh_v4f o[NI];                                 // O rows 4 g4 + r, columns 64 q + 4 l16 + c of tile 4 q + c
#pragma unroll
    for (int dt = 0; dt < NI; dt++) o[dt] = omh_v4f{0.f, 0.f, 0.f, 0.f};

    auto step = [&](int b) __attribute__((always_inline)) {
        // scores of keys kb + 4 g4 + r for column l16 (two product chains)
        omh_v4f sa = omh_v4f{0.f, 0.f, 0.f, 0.f}, sb = sa;
#pragma unroll
        for (int i = 0; i < NI; i++) {
            const omh_v4f qf = *reinterpret_cast<const omh_v4f *>(qrow + 16 * i);
#pragma unroll
            for (int st = 0; st < 4; st++) {
                if (i & 1) sb = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i][st], qf[st], sb, 0, 0, 0);
                else sa = __builtin_amdgcn_mfma_f32_16x16x4f32(kv[i][st], qf[st], sa, 0, 0, 0);
            }
        }
        load_v(b);                                 // (into the registers the scores have read)
        const int kb = k0 + 16 * b;
        float sc[4], mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            sc[r] = kb + 4 * g4 + r < kend ? (sa[r] + sb[r]) * a.scale : -INFINITY;   // qwen.c:410-414
            mx = fmaxf(mx, sc[r]);
        }
        mx = omh_swap32_max(omh_swap16_max(mx));
        // online softmax (qwen.c:413 softmax_ over all keys, merged per block);
        // a decode step's blocks begin with a visible key, so mn is finite;
        // with more tokens an early one may have seen none yet (weights 0)
        const float mn = fmaxf(m, mx), ref = PREP || mn > -INFINITY ? mn : 0.f;
        const float corr = expf(m - ref);
        float pr[4], ps = 0.f;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            pr[r] = kb + 4 * g4 + r < kend ? expf(sc[r] - ref) : 0.f;
            ps += pr[r];
        }
        ps = omh_swap32_sum(omh_swap16_sum(ps));
        l = l * corr + ps;
        m = mn;
        // the output rows are columns 4 g4 + r: their corrections from lanes 4 g4 + r
        float cr[4];
#pragma unroll
        for (int r = 0; r < 4; r++) cr[r] = __shfl(corr, 4 * g4 + r, OMH_WAVE);
#pragma unroll
        for (int dt = 0; dt < NI; dt++)
#pragma unroll
            for (int r = 0; r < 4; r++) o[dt][r] *= cr[r];
        // A block that some of the tile's tokens see only in part, and whose
        // values are not all finite: a weight of zero would not hide those
        // from the tokens before them, so this block's sums run key by key
        // over the keys each column sees, O in the wave's LDS rows meanwhile.
        if constexpr (!PREP) {
            if (kb + 15 > a.pos) {
                bool odd = false;
#pragma unroll
                for (int i = 0; i < NI; i++)
#pragma unroll
                    for (int c = 0; c < 4; c++) odd |= !(fabsf(kv[i][c]) < INFINITY);
                if (__ballot(odd)) {
                    float *ow = mo + wave * 16 * HD;
#pragma unroll
                    for (int q = 0; q < NQ; q++)
#pragma unroll
                        for (int r = 0; r < 4; r++)
                            *reinterpret_cast<omh_v4f *>(ow + (4 * g4 + r) * HD + 64 * q + 4 * l16) =
                                omh_v4f{o[4 * q][r], o[4 * q + 1][r], o[4 * q + 2][r], o[4 * q + 3][r]};
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                    __builtin_amdgcn_wave_barrier();
#pragma unroll 1
                    for (int c = 0; c < ncol; c++) {
                        const int ke = min(kb + 16, min(k1, a.pos + token_of(c0 + c) + 1)), d = 4 * lane % HD;
                        omh_v4f acc = *reinterpret_cast<const omh_v4f *>(ow + c * HD + d);
#pragma unroll 1
                        for (int k = kb; k < ke; k++) {
                            const int r = (k - kb) % 4;
                            const float w = __shfl(r < 2 ? (r ? pr[1] : pr[0]) : (r > 2 ? pr[3] : pr[2]), (k - kb) / 4 * 16 + c, OMH_WAVE);
                            acc += w * ld_buf_v4<false>(vrs, (k * HD + d) * 4);
                        }
                        __builtin_amdgcn_wave_barrier();     // (lanes past HD / 4 repeat the row)
                        *reinterpret_cast<omh_v4f *>(ow + c * HD + d) = acc;
                    }
                    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
                    __builtin_amdgcn_wave_barrier();
#pragma unroll
                    for (int q = 0; q < NQ; q++)
#pragma unroll
                        for (int r = 0; r < 4; r++) {
                            const omh_v4f x = *reinterpret_cast<const omh_v4f *>(ow + (4 * g4 + r) * HD + 64 * q + 4 * l16);
#pragma unroll
                            for (int c = 0; c < 4; c++) o[4 * q + c][r] = x[c];
                        }
                    return;
                }
            }
        }
        // P.V (qwen.c:415-419)
#pragma unroll
        for (int q = 0; q < NQ; q++)
#pragma unroll
            for (int c = 0; c < 4; c++)
#pragma unroll
                for (int st = 0; st < 4; st++)
                    o[4 * q + c] = __builtin_amdgcn_mfma_f32_16x16x4f32(pr[st], kv[NQ * st + q][c], o[4 * q + c], 0, 0, 0);
    };
    // the wave's blocks wave, wave + NW, ... (block wave's loads went out above)
    for (int b = wave; b < nb; b += NW) {
        if (b != wave) load_k(b);
        step(b);
    }

    // merge the waves: the workgroup's max per column, each wave's output scaled to it
    if (g4 == 0) {
        mm[wave * 16 + l16] = m;
        mm[NW * 16 + wave * 16 + l16] = l;
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < 4; r++) {
        const int h = 4 * g4 + r;
        float M = -INFINITY;
#pragma unroll
        for (int w = 0; w < NW; w++) M = fmaxf(M, mm[w * 16 + h]);
        // 0 for a wave without blocks, or one whose column saw no key (its m is -inf)
        const float f = PREP || M > -INFINITY ? expf(mm[wave * 16 + h] - M) : 0.f;
#pragma unroll
        for (int q = 0; q < NQ; q++)
            *reinterpret_cast<omh_v4f *>(mo + (wave * 16 + h) * HD + 64 * q + 4 * l16) =
                omh_v4f{o[4 * q][r] * f, o[4 * q + 1][r] * f, o[4 * q + 2][r] * f, o[4 * q + 3][r] * f};
    }
    __syncthreads();
    for (int e = tid; e < ncol * (HD / 4); e += NT) {
        const int i = e / (HD / 4), c = e % (HD / 4);
        omh_v4f acc = *reinterpret_cast<const omh_v4f *>(mo + i * HD + 4 * c);
#pragma unroll
        for (int w = 1; w < NW; w++) acc += *reinterpret_cast<const omh_v4f *>(mo + (w * 16 + i) * HD + 4 * c);
        *reinterpret_cast<omh_v4f *>(a.po + (row_of(i) * ns + s) * HD + 4 * c) = acc;
    }
    if (tid < ncol) {
        float M = -INFINITY, L = 0.f;
#pragma unroll
        for (int w = 0; w < NW; w++) M = fmaxf(M, mm[w * 16 + tid]);
        if (PREP || M > -INFINITY)
#pragma unroll
            for (int w = 0; w < NW; w++) L += mm[NW * 16 + w * 16 + tid] * expf(mm[w * 16 + tid] - M);
        const size_t pi = row_of(tid) * ns + s;
        a.pml[2 * pi] = M;
        a.pml[2 * pi + 1] = L;
    }
}

// ---------------------------------------------------------------- prompt steps
// Flash attention on the matrix cores for prompt steps of at least
// kFlashMinT tokens (attn_flash3_kernel below: bf16 x 3 products, the
// default; this one with fp32 products, v_mfma_f32_16x16x4f32, kept for
// comparison, OMH_ATTN_FLASH=fp32): the same fp32 scores, online
// softmax and P.V as the split kernel, as dense products.  A wave owns one
// unit, 16 consecutive tokens of one query head; a workgroup of 8 waves
// takes 8 units of one kv group (the group's heads of a token block, then
// the next block), so the K and V tiles it stages in LDS (32 keys, double
// buffered, HBM -> registers -> LDS one tile ahead) serve 8 waves.  Per
// wave, S^T = K Q^T (A = a K row from LDS, B = the wave's q, held in
// registers for the whole sweep), so each lane's scores belong to its own
// query row (lane % 16): the row max and sum need two exchanges and the
// rescale of the output is lane-local; O^T = V^T P^T (A = V from LDS, B =
// the probabilities as the score product left them: key 16 n + 4 g + s of
// lane group g is register s).  The head dims of q.k are taken in the order
// 16 c + 4 g + s on both operands (one 16-byte K read per 4 products).  The
// workgroups holding the most keys (the prompt's end) start first.  Keys
// past a token's position are masked; rows of the last tile past the
// visible keys repeat the tile's first row, so every LDS value is finite.
template <int HD>
struct FlashShape {
    static constexpr int KT = 32;                  // keys per tile
    static constexpr int LD = HD + 4;              // padded row in LDS (floats)
    static constexpr int STAGE = 2 * KT * LD;      // one stage: K rows, then V rows
    static constexpr size_t LDS = 2 * (size_t)STAGE * sizeof(float);
    static constexpr int NC = HD / 16;             // 16-dim groups (q registers; output tiles)
    static constexpr int PER = KT * HD / 4 / (8 * OMH_WAVE);   // float4 pieces of K (and of V) per thread
};
constexpr int kFlashMinT = 64;
// decode steps fold the prep into the split kernel unless OMH_ATTN_FUSE=0 (comparison)
bool fuse_prep() {
    const char *e = getenv("OMH_ATTN_FUSE");
    return !(e && e[0] == '0');
}
// the fp32-product flash kernel instead of the bf16 x 3 one (OMH_ATTN_FLASH=fp32, for comparison)
bool flash_fp32() {
    const char *e = getenv("OMH_ATTN_FLASH");
    return e && e[0] == 'f';
}
// the bf16 x 3 kernel converting every tile itself instead of copying tile
// images (OMH_ATTN_FLASH=reg, for comparison)
bool flash_reg() {
    const char *e = getenv("OMH_ATTN_FLASH");
    return e && e[0] == 'r';
}
// prompt steps of at least this many tokens stage their tiles from images
constexpr int kFlashImageMinT = 256;

template <int HD>
__global__ __launch_bounds__(8 * OMH_WAVE) __attribute__((amdgpu_waves_per_eu(2, 2)))
void attn_flash_kernel(const AttnArgs a) {
    using F = FlashShape<HD>;
    constexpr int KT = F::KT, LD = F::LD, NC = F::NC, PER = F::PER, NT = 8 * OMH_WAVE;
    extern __shared__ float smem[];
    const int H = a.H, KV = a.KV, grp = H / KV;
    const int nunit = (a.T + 15) / 16 * grp, wpg = (nunit + 7) / 8;
    const int g = blockIdx.x % KV, wi = wpg - 1 - (int)blockIdx.x / KV;
    const int tid = threadIdx.x, lane = tid % OMH_WAVE;
    const int w = __builtin_amdgcn_readfirstlane(tid / OMH_WAVE);
    const int l16 = lane % 16, gq = lane / 16;
    const bool own = 8 * wi + w < nunit;
    const int u = min(8 * wi + w, nunit - 1);
    const int tb = u / grp, h = g * grp + u % grp;
    const int tq = 16 * tb + l16;                  // this lane's query token (may be past T: not written)
    const int tlast = min(16 * (min(8 * wi + 7, nunit - 1) / grp) + 15, a.T - 1);
    const int nkeys = a.pos + tlast + 1;           // keys the workgroup's last token sees
    const int kmax = a.pos + tq;                   // the last key this lane's token sees

    omh_v4f q[NC];                                 // dims 16 c + 4 gq .. +3 of token tq
    {
        const float *qr = a.qb + ((size_t)min(tq, a.T - 1) * H + h) * HD + 4 * gq;
#pragma unroll
        for (int c = 0; c < NC; c++) q[c] = *reinterpret_cast<const omh_v4f *>(qr + 16 * c);
    }
    const size_t cache0 = ((size_t)a.seq * KV + g) * a.max_t;
    const float *Kg = a.Kc + cache0 * HD, *Vg = a.Vc + cache0 * HD;
    omh_v4f kr[PER], vr[PER];
    auto load = [&](int kt) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int e = tid + NT * i, kk = e / (HD / 4), c = e % (HD / 4);
            const size_t off = (size_t)(kt + kk < nkeys ? kt + kk : kt) * HD + 4 * c;
            kr[i] = *reinterpret_cast<const omh_v4f *>(Kg + off);
            vr[i] = *reinterpret_cast<const omh_v4f *>(Vg + off);
        }
    };
    auto put = [&](int stage) __attribute__((always_inline)) {
        float *Ks = smem + stage * F::STAGE, *Vs = Ks + KT * LD;
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int e = tid + NT * i, kk = e / (HD / 4), c = e % (HD / 4);
            *reinterpret_cast<omh_v4f *>(Ks + kk * LD + 4 * c) = kr[i];
            *reinterpret_cast<omh_v4f *>(Vs + kk * LD + 4 * c) = vr[i];
        }
    };

    omh_v4f o[NC];                                     // O^T: o[j][i] = O[token tq][dim 16 j + 4 gq + i]
#pragma unroll
    for (int j = 0; j < NC; j++) o[j] = omh_v4f{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    load(0);
    put(0);
    __syncthreads();
    for (int kt = 0, st = 0; kt < nkeys; kt += KT, st ^= 1) {
        if (kt + KT < nkeys) load(kt + KT);
        const float *Ks = smem + st * F::STAGE, *Vs = Ks + KT * LD;
        // S^T for keys kt + 16 n + 4 gq + i (register i of sc[n]), query row tq
        omh_v4f sc[KT / 16];
#pragma unroll
        for (int n = 0; n < KT / 16; n++) {
            sc[n] = omh_v4f{0.f, 0.f, 0.f, 0.f};
            const float *kp = Ks + (16 * n + l16) * LD + 4 * gq;
#pragma unroll
            for (int c = 0; c < NC; c++) {
                const omh_v4f kf = *reinterpret_cast<const omh_v4f *>(kp + 16 * c);
#pragma unroll
                for (int s = 0; s < 4; s++) sc[n] = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[s], q[c][s], sc[n], 0, 0, 0);
            }
        }
        // scores * hd^-1/2, causal mask, online softmax (qwen.c:410-414)
        float mx = -INFINITY;
#pragma unroll
        for (int n = 0; n < KT / 16; n++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int key = kt + 16 * n + 4 * gq + i;
                sc[n][i] = key <= kmax ? sc[n][i] * a.scale : -INFINITY;
                mx = fmaxf(mx, sc[n][i]);
            }
        mx = omh_swap32_max(omh_swap16_max(mx));
        const float mn = fmaxf(m, mx);             // finite: key 0 is in every token's first tile
        const float corr = expf(m - mn);
        float ps = 0.f;
#pragma unroll
        for (int n = 0; n < KT / 16; n++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                sc[n][i] = expf(sc[n][i] - mn);
                ps += sc[n][i];
            }
        ps = omh_swap32_sum(omh_swap16_sum(ps));
        l = fmaf(l, corr, ps);
        m = mn;
        // O^T = corr O^T + V^T P^T (qwen.c:415-419)
#pragma unroll
        for (int j = 0; j < NC; j++) {
            o[j] = o[j] * corr;
#pragma unroll
            for (int n = 0; n < KT / 16; n++) {
                const float *vp = Vs + (16 * n + 4 * gq) * LD + 16 * j + l16;
#pragma unroll
                for (int s = 0; s < 4; s++) o[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(vp[s * LD], sc[n][s], o[j], 0, 0, 0);
            }
        }
        if (kt + KT < nkeys) put(st ^ 1);
        __syncthreads();
    }
    // normalise and gate (qwen.c:420-421)
    if (!own || tq >= a.T) return;
    const float il = 1.f / l;
    const float *gate = a.qkv + (size_t)tq * a.ld_qkv + (size_t)h * 2 * HD + HD + 4 * gq;
    float *dst = a.ctx + ((size_t)tq * H + h) * HD + 4 * gq;
#pragma unroll
    for (int j = 0; j < NC; j++) {
        const float4 gv = *reinterpret_cast<const float4 *>(gate + 16 * j);
        float4 r;
        r.x = o[j][0] * il * omh_sigmoid(gv.x);
        r.y = o[j][1] * il * omh_sigmoid(gv.y);
        r.z = o[j][2] * il * omh_sigmoid(gv.z);
        r.w = o[j][3] * il * omh_sigmoid(gv.w);
        *reinterpret_cast<float4 *>(dst + 16 * j) = r;
    }
}

// The default flash attention, on the bf16 matrix cores
// (v_mfma_f32_32x32x16_bf16, fp32 accumulation) with every product as three:
// each fp32 operand x splits as hi = bf16(x), lo = bf16(x - hi), so
// x = hi + lo to 2^-16 relative, and a.b = hi.hi + hi.lo + lo.hi with the
// dropped lo.lo term below 2^-16 |a||b|.
//
// A wave owns one unit, 32 consecutive tokens of one query head, with q and
// the output (128 registers each at HD = 256) in registers; a workgroup is 4
// waves, one per SIMD, and 4 units of one kv group (the group's heads of a
// token block, then the next block).  What bounds the kernel is the matrix
// cores against the LDS reads of the K and V tiles: per 32-key tile a wave
// reads the whole 64 KiB and issues 96 products of 32 cycles, 256 KiB per CU
// (2048 cycles at 128 B per clock) against 3072 cycles of products on every
// SIMD.  (16-token units on 8 waves, the form before, read 512 KiB per tile.)
//
// Tiles sit in LDS in MFMA operand order: fragment f is the 1 KiB that the
// 64 lanes of one A operand read as 16 contiguous bytes each, so no read has
// a bank conflict and no padding is needed.  K fragment (s, plane): lane l
// holds key l % 32 at dims 16 s + 8 (l / 32) + j.  The score product S^T =
// K Q^T leaves token l % 32, key 8 (i / 4) + 4 (l / 32) + i % 4 in register i,
// which P^T as the B operand of O^T = V^T P^T takes as it stands (16-key step
// u: registers 8 u + j), so V fragment (d / 2, u, d % 2, plane) holds, in lane l, dim
// 32 d + l % 32 at the keys 16 u + 8 (j / 4) + 4 (l / 32) + j % 4.
//
// K runs one tile ahead of V: an iteration forms the next tile's scores, then
// adds its own tile's P V while the next tile's softmax (VALU) runs beside
// those products.  One barrier per tile.
//
// Steps whose units leave CUs idle (a turn appended to a long conversation)
// split the keys over ns workgroups per unit group (attn_flash_plan); each
// writes its unnormalised output, and attn_flash_merge_kernel merges them.
template <int HD>
struct Flash3Shape {
    static constexpr int KT = 32;                  // keys per tile
    static constexpr int NW = 4;                   // waves (units) per workgroup
    static constexpr int NS = HD / 16;             // 16-dim steps of q.k
    static constexpr int ND = HD / 32;             // 32-dim output tiles
    static constexpr int KB = NS * 2 * 1024;       // bytes of a tile's K fragments: (s, plane)
    static constexpr int VB = ND * 2 * 2 * 1024;   // of its V fragments: (d / 2, u, d % 2, plane)
    static constexpr int TILE = KB + VB;           // a tile image: K, then V
    static constexpr size_t LDS = 2 * (size_t)TILE;   // two K stages, then two V stages
    static constexpr int EU = HD > 128 ? 1 : 2;    // waves per SIMD the registers allow
    static_assert(LDS <= 160 * 1024 && KB == VB, "two stages in a CU's LDS");
};
typedef __bf16 omh_v8bf __attribute__((ext_vector_type(8)));
typedef float omh_v16f __attribute__((ext_vector_type(16)));

// a and b as bf16 pairs: *hi = their roundings, *lo = the roundings of what those leave
__device__ __forceinline__ void bf16_split2(float a, float b, uint32_t &hi, uint32_t &lo) {
    typedef __bf16 v2bf __attribute__((ext_vector_type(2)));
    hi = __builtin_bit_cast(uint32_t, v2bf{(__bf16)a, (__bf16)b});
    const float ra = a - __builtin_bit_cast(float, hi << 16), rb = b - __builtin_bit_cast(float, hi & 0xffff0000u);
    lo = __builtin_bit_cast(uint32_t, v2bf{(__bf16)ra, (__bf16)rb});
}
typedef uint32_t omh_v4u32 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void bf16_split8(const float (&v)[8], omh_v8bf &hi, omh_v8bf &lo) {
    omh_v4u32 h, l;
#pragma unroll
    for (int j = 0; j < 4; j++) {
        uint32_t x, y;
        bf16_split2(v[2 * j], v[2 * j + 1], x, y);
        h[j] = x;
        l[j] = y;
    }
    hi = __builtin_bit_cast(omh_v8bf, h);
    lo = __builtin_bit_cast(omh_v8bf, l);
}

// K or V fragments of the tile of keys kt .. kt + 31 on their way to LDS (or
// to a tile image in memory), 4 waves: wave w takes fragment pairs (hi, lo)
// w, w + 4, ...  Rows past nkeys repeat the tile's first row, so every value
// is a visible one.
template <int HD>
struct Flash3Frags {
    using F = Flash3Shape<HD>;
    static constexpr int N = F::NS / F::NW;        // fragment pairs per wave (of K, and of V)
    static_assert(F::NS % F::NW == 0 && F::NS == 2 * F::ND, "whole fragments per wave");
    float x[N][8];
    __device__ __forceinline__ void load_k(const float *Kg, int kt, int nkeys, int w, int lane) {
        const int kk = kt + lane % 32 < nkeys ? kt + lane % 32 : kt;
#pragma unroll
        for (int i = 0; i < N; i++) {
            const float *src = Kg + (size_t)kk * HD + 16 * (w + F::NW * i) + 8 * (lane / 32);
            const omh_v4f a = *reinterpret_cast<const omh_v4f *>(src), b = *reinterpret_cast<const omh_v4f *>(src + 4);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                x[i][j] = a[j];
                x[i][4 + j] = b[j];
            }
        }
    }
    __device__ __forceinline__ void load_v(const float *Vg, int kt, int nkeys, int w, int lane) {
#pragma unroll
        for (int i = 0; i < N; i++) {
            const int f = w + F::NW * i, d = 2 * (f / 4) + f % 2, u = f / 2 % 2;
#pragma unroll
            for (int j = 0; j < 8; j++) {
                const int k = kt + 16 * u + 8 * (j / 4) + 4 * (lane / 32) + j % 4;
                x[i][j] = Vg[(size_t)(k < nkeys ? k : kt) * HD + 32 * d + lane % 32];
            }
        }
    }
    // (the pairs' order is the fragments': (s, plane) and (d / 2, u, d % 2, plane))
    __device__ __forceinline__ void put(unsigned char *dst, int w, int lane) const {
#pragma unroll
        for (int i = 0; i < N; i++) {
            omh_v8bf hi, lo;
            bf16_split8(x[i], hi, lo);
            unsigned char *p = dst + (size_t)(w + F::NW * i) * 2048 + 16 * lane;
            *reinterpret_cast<omh_v8bf *>(p) = hi;
            *reinterpret_cast<omh_v8bf *>(p + 1024) = lo;
        }
    }
};

// The tile images of keys 0 .. pos + T - 1 of the step's sequence, one
// workgroup per (kv head, tile): image (g, i) at a.img + (g * a.img_tiles +
// i) * TILE holds exactly what attn_flash3_kernel stages in LDS for tile i.
template <int HD>
__global__ __launch_bounds__(Flash3Shape<HD>::NW * OMH_WAVE) void attn_tile_image_kernel(const AttnArgs a) {
    using F = Flash3Shape<HD>;
    const int g = blockIdx.x % a.KV, ti = blockIdx.x / a.KV;
    const int lane = threadIdx.x % OMH_WAVE, w = __builtin_amdgcn_readfirstlane(threadIdx.x / OMH_WAVE);
    const size_t cache0 = ((size_t)a.seq * a.KV + g) * a.max_t * HD;
    unsigned char *dst = a.img + ((size_t)g * a.img_tiles + ti) * F::TILE;
    Flash3Frags<HD> k, v;
    k.load_k(a.Kc + cache0, ti * F::KT, a.pos + a.T, w, lane);
    v.load_v(a.Vc + cache0, ti * F::KT, a.pos + a.T, w, lane);
    k.put(dst, w, lane);
    v.put(dst + F::KB, w, lane);
}

// The products of the one-wave-per-SIMD form, with its output in accumulation
// registers for the whole sweep and everything else in vector registers (the
// form that stages its tiles itself has about 50 values too many for those and
// keeps them in accumulation registers between uses): through the builtin the
// compiler puts all results in accumulation registers and moves 128 of them to
// vector registers and back on every tile.  It does not see what these
// instructions are, so their waits are here (test_flash_waits.py follows them
// through the compiled code): two states
// before each (an operand may just have been written by a VALU instruction,
// a move between the register files among them; they pass while the product
// before still runs), and acc_settle and vec_settle (a product's write lands
// within 18 states) between the products and any other use of their results.
__device__ __forceinline__ void acc_product(omh_v16f &c, const omh_v8bf &a, const omh_v8bf &b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void vec_product(omh_v16f &c, const omh_v8bf &a, const omh_v8bf &b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void vec_product0(omh_v16f &c, const omh_v8bf &a, const omh_v8bf &b) {   // c = a b
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, 0" : "=&v"(c) : "v"(a), "v"(b));
}
__device__ __forceinline__ void vec_settle(omh_v16f &c, omh_v16f &d) { asm volatile("s_nop 15\n\ts_nop 3" : "+v"(c), "+v"(d)); }
template <int N>
__device__ __forceinline__ void acc_settle(omh_v16f (&c)[N]) {
    asm volatile("s_nop 15\n\ts_nop 3" : "+a"(c[0]));
#pragma unroll
    for (int d = 1; d < N; d++) asm volatile("" : "+a"(c[d]));
}
// (no instruction: where control flow joins, a value whose only use is one
// that wants accumulation registers stays in them)
template <int N>
__device__ __forceinline__ void acc_keep(omh_v16f (&c)[N]) {
#pragma unroll
    for (int d = 0; d < N; d++) asm volatile("" : "+a"(c[d]));
}
__device__ __forceinline__ void acc_scale(omh_v16f &c, float f) {
#pragma unroll
    for (int i = 0; i < 16; i++) {
        float t, r;
        asm volatile("v_accvgpr_read_b32 %0, %1" : "=v"(t) : "a"(c[i]));
        t *= f;
        asm volatile("v_accvgpr_write_b32 %0, %1" : "=a"(r) : "v"(t));
        c[i] = r;
    }
}

// IMG: each tile goes from its image (attn_tile_image_kernel) into LDS as
// whole 1 KiB runs (buffer loads to LDS), with no conversion in the kernel.
template <int HD, bool IMG>
__global__ __launch_bounds__(Flash3Shape<HD>::NW * OMH_WAVE)
__attribute__((amdgpu_waves_per_eu(Flash3Shape<HD>::EU, Flash3Shape<HD>::EU)))
void attn_flash3_kernel(const AttnArgs a) {
    using F = Flash3Shape<HD>;
    constexpr int KT = F::KT, NS = F::NS, ND = F::ND, NW = F::NW;
    extern __shared__ __attribute__((aligned(16))) unsigned char smem3[];
    unsigned char *const Ks = smem3, *const Vs = smem3 + 2 * F::KB;
    const int H = a.H, KV = a.KV, grp = H / KV;
    const int nunit = (a.T + 31) / 32 * grp, wpg = (nunit + NW - 1) / NW;
    // the workgroups of one (kv head, key split) read the same tiles
    const int gs = blockIdx.x % (KV * a.ns), g = gs % KV, sp = gs / KV;
    const int wi = wpg - 1 - (int)(blockIdx.x / (KV * a.ns));   // the most keys first
    const int tid = threadIdx.x, lane = tid % OMH_WAVE;
    const int w = __builtin_amdgcn_readfirstlane(tid / OMH_WAVE);
    const int l32 = lane % 32, g2 = lane / 32;
    const bool own = NW * wi + w < nunit;
    const int u = min(NW * wi + w, nunit - 1);
    const int tb = u / grp, h = g * grp + u % grp;
    const int tq = 32 * tb + l32;                  // this lane's query token (may be past T: not written)
    const int tlast = min(32 * (min(NW * wi + NW - 1, nunit - 1) / grp) + 31, a.T - 1);
    const int nkeys = a.pos + tlast + 1;           // keys the workgroup's last token sees
    const int k0 = sp * a.kps, k1 = min(nkeys, k0 + a.kps);   // (kps is whole tiles)
    if (k0 >= k1) return;                          // (the merge reads no such split)
    const int kmax = a.pos + tq;                   // the last key this lane's token sees

    // Values that are not finite must reach only the tokens that see them,
    // and a weight of zero does not hide them from the others.  From key ka on
    // the tiles hold keys that some of the workgroup's tokens do not see, rows
    // of this step.  Where the prep left word that one of those is odd, the
    // tiles from ka on are taken with such values as zeros, and at the end a
    // token that sees one gets NaN in that dim.
    const int ka = max(k0, (a.pos + 32 * (NW * wi / grp) + 1) / KT * KT);
    const int kz = min(a.pos + a.T, (k1 + KT - 1) / KT * KT);
    const float *Vk = a.Vc + (((size_t)a.seq * KV + g) * a.max_t + ka) * HD;
    const int tf = max(ka - a.pos, 0) + lane;      // (requested ahead of q: their round trips overlap)
    const float *flags = a.qkv + odd_flag_at(H, KV, g, HD);
    float flag = flags[(size_t)min(tf, a.T - 1) * a.ld_qkv];

    // q as the B operand of S^T: dims 16 s + 8 g2 .. +7 of token tq, hi and lo
    omh_v8bf qh[NS], ql[NS];
    {
        const float *qr = a.qb + ((size_t)min(tq, a.T - 1) * H + h) * HD + 8 * g2;
#pragma unroll
        for (int s = 0; s < NS; s++) {
            const float4 x0 = *reinterpret_cast<const float4 *>(qr + 16 * s);
            const float4 x1 = *reinterpret_cast<const float4 *>(qr + 16 * s + 4);
            const float v[8] = {x0.x, x0.y, x0.z, x0.w, x1.x, x1.y, x1.z, x1.w};
            bf16_split8(v, qh[s], ql[s]);
        }
    }
    flag = tf < kz - a.pos ? flag : 0.f;
    for (int t = tf + OMH_WAVE; t < kz - a.pos; t += OMH_WAVE) flag += flags[(size_t)t * a.ld_qkv];   // (several token blocks)
    const bool odd = __builtin_amdgcn_ballot_w64(flag != 0.f) != 0;   // (the same in every wave)
    const size_t cache0 = ((size_t)a.seq * KV + g) * a.max_t * HD;
    const float *Kg = a.Kc + cache0, *Vg = a.Vc + cache0;
    Flash3Frags<HD> fk, fv;
    const __amdgpu_buffer_rsrc_t irs =
        omh_rsrc(IMG ? a.img + (size_t)g * a.img_tiles * F::TILE : a.img, IMG ? a.img_tiles * F::TILE : 0);
    // IMG: half an image (K at 0, V at KB) of the tile at key kt into dst
    auto copy = [&](int kt, int half, unsigned char *dst) __attribute__((always_inline)) {
        const int src = kt / KT * F::TILE + half;
#pragma unroll
        for (int i = 0; i < F::KB / 1024 / NW; i++) {
            const int c = (w + NW * i) * 1024;
            __builtin_amdgcn_raw_ptr_buffer_load_lds(irs, (__attribute__((address_space(3))) void *)(dst + c), 16,
                                                     16 * lane, src + c, 0, 0);
        }
    };
    // fetch: request K of tile kt into K stage st (reg form: into registers,
    // land() stores them once the stage is free)
    auto fetch_k = [&](int kt, int st) __attribute__((always_inline)) {
        if constexpr (IMG) copy(kt, 0, Ks + st * F::KB);
        else fk.load_k(Kg, kt, nkeys, w, lane);
    };
    auto fetch_v = [&](int kt, int st) __attribute__((always_inline)) {
        if constexpr (IMG) copy(kt, F::KB, Vs + st * F::VB);
        else fv.load_v(Vg, kt, nkeys, w, lane);
    };
    auto land_k = [&](int st) __attribute__((always_inline)) {
        if constexpr (!IMG) fk.put(Ks + st * F::KB, w, lane);
    };
    auto land_v = [&](int st) __attribute__((always_inline)) {
        if constexpr (!IMG) fv.put(Vs + st * F::VB, w, lane);
    };
    auto arrive = [&]() __attribute__((always_inline)) {
        if constexpr (IMG) __builtin_amdgcn_s_waitcnt(0x0f70);   // vmcnt(0): this wave's copies have landed
        __syncthreads();
    };

    // the V stage's values that are not finite as zeros: of the pieces that
    // this wave has brought
    auto scrub = [&](unsigned char *stage) __attribute__((always_inline)) {
#pragma unroll 1
        for (int i = 0; i < F::VB / 1024 / NW; i++) {
            const int c = IMG ? w + NW * i : 2 * (w + NW * (i / 2)) + i % 2;
            uint32_t *p = reinterpret_cast<uint32_t *>(stage + c * 1024 + 16 * lane);
#pragma unroll
            for (int j = 0; j < 4; j++) {
                uint32_t v = p[j];
                if ((v & 0x7f80u) == 0x7f80u) v &= 0xffff0000u;
                if ((v & 0x7f800000u) == 0x7f800000u) v &= 0xffffu;
                p[j] = v;
            }
        }
        __builtin_amdgcn_s_waitcnt(0xc07f);       // lgkmcnt(0): in place before the barrier that follows
    };

    omh_v16f o[ND];                                // O^T: o[d][i] = O[token tq][dim 32 d + 8 (i / 4) + 4 g2 + i % 4]
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int i = 0; i < 16; i++) o[d][i] = 0.f;
    float m = -INFINITY, l = 0.f;                  // reference of the raw scores (q.k), sum of the weights
    const float sl2 = a.scale * 1.4426950408889634f;   // hd^-1/2 log2 e (qwen.c:410-414)

    // The work of one iteration, in a fixed order (sched_barriers between
    // the steps: left to itself the compiler reads each fragment right
    // before its products, and a lone wave then waits out every LDS read).
    // Step i of a block takes fragment pairs (hi, lo) 2 i and 2 i + 1 through
    // their three products each, on two accumulators in turn (a product on
    // the accumulator of the one right before it waits twice as long),
    // requests pairs 2 i + AHEAD and the next, and does a piece of the softmax.
    constexpr int AHEAD = 4;
    omh_v8bf rh[AHEAD], rl[AHEAD];                 // the pairs in flight
    const int l16 = 16 * lane;
    omh_v16f sc, sd;                               // S^T of a tile: even and odd steps' sums
    omh_v8bf ph[2], pl[2];                         // P^T as the B operand of 16-key step u
    omh_v4u32 nh[2], nl[2];                        // the next tile's
    float mx, ps, ref, corr = 1.f;
    auto ask = [&](const unsigned char *base, auto pair) __attribute__((always_inline)) {
        constexpr int P = decltype(pair)::value;
        rh[P % AHEAD] = *reinterpret_cast<const omh_v8bf *>(base + l16 + 2048 * P);
        rl[P % AHEAD] = *reinterpret_cast<const omh_v8bf *>(base + l16 + 2048 * P + 1024);
    };
    auto product = [&](omh_v16f &c, const omh_v8bf &x, const omh_v8bf &y) __attribute__((always_inline)) {
        if constexpr (F::EU == 1) vec_product(c, x, y);
        else c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    };
    auto product0 = [&](omh_v16f &c, const omh_v8bf &x, const omh_v8bf &y) __attribute__((always_inline)) {
        if constexpr (F::EU == 1) vec_product0(c, x, y);
        else {
            const omh_v16f zero = {};
            c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, zero, 0, 0, 0);
        }
    };
    auto add_product = [&](omh_v16f &c, const omh_v8bf &x, const omh_v8bf &y) __attribute__((always_inline)) {
        if constexpr (F::EU == 1) acc_product(c, x, y);
        else c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x, y, c, 0, 0, 0);
    };
    // step s of the scores of the K tile at kb; with then_v the last steps
    // ask for the first V pairs at vb
    auto score_step = [&](auto step, const unsigned char *kb, auto then_v, const unsigned char *vb) __attribute__((always_inline)) {
        constexpr int S = 2 * decltype(step)::value, R = S % AHEAD;
        const omh_v8bf h0 = rh[R], l0 = rl[R], h1 = rh[R + 1], l1 = rl[R + 1];
        if constexpr (S == 0) {
            product0(sc, l0, qh[S]);
            product0(sd, l1, qh[S + 1]);
        } else {
            product(sc, l0, qh[S]);
            product(sd, l1, qh[S + 1]);
        }
        product(sc, h0, ql[S]);
        product(sd, h1, ql[S + 1]);
        product(sc, h0, qh[S]);
        product(sd, h1, qh[S + 1]);
        if constexpr (S + AHEAD < NS) {
            ask(kb, std::integral_constant<int, S + AHEAD>{});
            ask(kb, std::integral_constant<int, S + AHEAD + 1>{});
        } else if constexpr (decltype(then_v)::value) {
            ask(vb, std::integral_constant<int, S + AHEAD - NS>{});
            ask(vb, std::integral_constant<int, S + AHEAD + 1 - NS>{});
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    // Causal mask and online softmax of the tile at key kt (qwen.c:410-414),
    // in pieces 0 .. NP - 1.  The reference moves only where a score exceeds
    // it by 2^kSlack (the weights then stay below 2^kSlack, well inside fp32
    // and its bf16 pairs), so o is hardly ever rescaled: with the running max
    // itself some of a wave's 32 rows move on most of a prompt's tiles.
    constexpr int NP = 14;
    constexpr float kSlack = 8.f;
    auto soften = [&](auto piece, int kt) __attribute__((always_inline)) {
        constexpr int P = decltype(piece)::value;
        if constexpr (P == 0 && F::EU == 1) {
            vec_settle(sc, sd);
        }
        if constexpr (P < 4) {
            const int left = kmax - kt - 4 * g2;   // key 8 (i / 4) + i % 4 of this lane is visible up to here
#pragma unroll
            for (int i = 4 * P; i < 4 * P + 4; i++) sc[i] = 8 * (i / 4) + i % 4 <= left ? sc[i] + sd[i] : -INFINITY;
            const float m4 = fmaxf(fmaxf(sc[4 * P], sc[4 * P + 1]), fmaxf(sc[4 * P + 2], sc[4 * P + 3]));
            mx = P == 0 ? m4 : fmaxf(mx, m4);
        } else if constexpr (P == 4) {
            mx = omh_swap32_max(mx);
            const bool none = m == -INFINITY, moves = none | ((mx - m) * sl2 > kSlack);
            const float shrink = __builtin_amdgcn_exp2f((m - mx) * sl2);
            corr = (moves & !none) ? shrink : 1.f;
            m = moves ? mx : m;
            // (a split may begin past some of its tokens' keys: nothing seen
            // yet, and every weight 2^-inf = 0 against any finite reference)
            ref = m == -INFINITY ? 0.f : m * sl2;
            ps = 0.f;
        } else if constexpr (P < 13) {
            constexpr int E = 2 * (P - 5);
            const float p0 = __builtin_amdgcn_exp2f(fmaf(sc[E], sl2, -ref));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(sc[E + 1], sl2, -ref));
            ps += p0;
            ps += p1;
            uint32_t hi, lo;
            bf16_split2(p0, p1, hi, lo);
            nh[E / 8][E % 8 / 2] = hi;
            nl[E / 8][E % 8 / 2] = lo;
            // (formed here, not behind the rescale's branch)
            if constexpr (P == 8 || P == 12) asm volatile("" : "+v"(nh[P / 4 - 2]), "+v"(nl[P / 4 - 2]));
        } else {
            l = fmaf(l, corr, omh_swap32_sum(ps));
        }
    };
    auto turn = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int u = 0; u < 2; u++) {
            ph[u] = __builtin_bit_cast(omh_v8bf, nh[u]);
            pl[u] = __builtin_bit_cast(omh_v8bf, nl[u]);
        }
    };
    // step i of O^T += V^T P^T for the V tile at vb: output tiles 2 (i / 2)
    // and the next, 16-key step i % 2
    auto weigh_step = [&](auto step, const unsigned char *vb) __attribute__((always_inline)) {
        constexpr int I = decltype(step)::value, d = 2 * (I / 2), u = I % 2, R = 2 * I % AHEAD;
        const omh_v8bf h0 = rh[R], l0 = rl[R], h1 = rh[R + 1], l1 = rl[R + 1];
        add_product(o[d], l0, ph[u]);
        add_product(o[d + 1], l1, ph[u]);
        add_product(o[d], h0, pl[u]);
        add_product(o[d + 1], h1, pl[u]);
        add_product(o[d], h0, ph[u]);
        add_product(o[d + 1], h1, ph[u]);
        if constexpr (2 * I + AHEAD < 2 * ND) {
            ask(vb, std::integral_constant<int, 2 * I + AHEAD>{});
            ask(vb, std::integral_constant<int, 2 * I + AHEAD + 1>{});
        }
    };
    // O^T = corr O^T (qwen.c:415-419), where some row's reference moved
    auto rescale = [&]() __attribute__((always_inline)) {
        if (!__builtin_amdgcn_ballot_w64(corr != 1.f)) return;
        if constexpr (F::EU == 1) {
            acc_settle(o);
#pragma unroll
            for (int d = 0; d < ND; d++) acc_scale(o[d], corr);
            acc_settle(o);
        } else {
#pragma unroll
            for (int d = 0; d < ND; d++) o[d] = o[d] * corr;
        }
    };
    fetch_k(k0, 0);
    fetch_v(k0, 0);
    land_k(0);
    if (k0 + KT < k1) fetch_k(k0 + KT, 1);
    land_v(0);
    if (k0 + KT < k1) land_k(1);
    arrive();
    if (odd && ka < k0 + KT) {
        scrub(Vs);
        __syncthreads();
    }
    static_assert(NS % AHEAD == 0 && NS == 2 * ND && AHEAD % 2 == 0, "pairs in flight");
    constexpr int STEPS = NS / 2;
    omh_static_for<AHEAD>([&](auto i) { ask(Ks, i); });
    omh_static_for<STEPS>([&](auto i) { score_step(i, Ks, std::false_type{}, nullptr); });
    omh_static_for<NP>([&](auto i) { soften(i, k0); });   // (o is still zero: nothing to rescale)
    turn();
    if constexpr (F::EU == 1) acc_keep(o);
    int kt = k0, st = 0;
    for (; kt + KT < k1; kt += KT, st ^= 1) {
        // K stage st held tile kt, whose scores every wave has formed, and V
        // stage st ^ 1 the tile before it, which every wave has added
        if constexpr (F::EU == 1) acc_keep(o);
        __syncthreads();
        const unsigned char *kb = Ks + (st ^ 1) * F::KB, *vb = Vs + st * F::VB;
        omh_static_for<AHEAD>([&](auto i) { ask(kb, i); });
        __builtin_amdgcn_sched_barrier(0);
        if (kt + 2 * KT < k1) fetch_k(kt + 2 * KT, st);
        fetch_v(kt + KT, st ^ 1);
        __builtin_amdgcn_sched_barrier(0);
        omh_static_for<STEPS>([&](auto i) { score_step(i, kb, std::true_type{}, vb); });
        omh_static_for<STEPS>([&](auto i) {
            constexpr int I = decltype(i)::value, PER = (NP + STEPS - 2) / (STEPS - 1);   // (the scores land during step 0)
            weigh_step(i, vb);
            if constexpr (I > 0)
                omh_static_for<PER>([&](auto j) {
                    constexpr int P = PER * (I - 1) + decltype(j)::value;
                    if constexpr (P < NP) soften(std::integral_constant<int, P>{}, kt + KT);
                });
            __builtin_amdgcn_sched_barrier(0);
        });
        turn();
        rescale();
        if constexpr (F::EU == 1) acc_keep(o);
        if (kt + 2 * KT < k1) land_k(st);
        land_v(st ^ 1);
        // this wave's copies (IMG: vmcnt(0)) or LDS stores (lgkmcnt(0): this
        // compiler leaves the wait for stores before a loop's back edge out
        // of the barrier at its head) have landed
        __builtin_amdgcn_s_waitcnt(IMG ? 0x0f70 : 0xc07f);
        if (odd && ka < kt + 2 * KT) scrub(Vs + (st ^ 1) * F::VB);
    }
    if constexpr (F::EU == 1) acc_keep(o);
    __syncthreads();
    const unsigned char *vb = Vs + st * F::VB;
    omh_static_for<AHEAD>([&](auto i) { ask(vb, i); });
    omh_static_for<STEPS>([&](auto i) { weigh_step(i, vb); });
    if constexpr (F::EU == 1) acc_settle(o);

    if (!own || tq >= a.T) return;
    // NaN over the dims of a written row in which its token sees a value that
    // is not finite (after the row: o stays where the products left it)
    auto mark = [&](float *row) __attribute__((always_inline)) {
        if (!odd) return;
#pragma unroll 1
        for (int k = ka; k < min(kz, kmax + 1); k++)
#pragma unroll 1
            for (int d = 0; d < HD; d += 8)
#pragma unroll
                for (int j = 0; j < 4; j++)
                    if (!bf16_finite(Vk[(size_t)(k - ka) * HD + 4 * g2 + d + j])) row[d + j] = __builtin_nanf("");
    };
    if (a.ns > 1) {
        // unnormalised partial of split sp (the reference in the scaled scores' units)
        const size_t pi = ((size_t)tq * H + h) * a.ns + sp;
        float *dst = a.po + pi * HD + 4 * g2;
#pragma unroll
        for (int d = 0; d < ND; d++)
#pragma unroll
            for (int k = 0; k < 4; k++)
                *reinterpret_cast<float4 *>(dst + 32 * d + 8 * k) =
                    make_float4(o[d][4 * k], o[d][4 * k + 1], o[d][4 * k + 2], o[d][4 * k + 3]);
        if (g2 == 0) {
            a.pml[2 * pi] = m * a.scale;
            a.pml[2 * pi + 1] = l;
        }
        mark(dst);
        return;
    }
    // normalise and gate (qwen.c:420-421)
    const float il = 1.f / l;
    const float *gate = a.qkv + (size_t)tq * a.ld_qkv + (size_t)h * 2 * HD + HD + 4 * g2;
    float *dst = a.ctx + ((size_t)tq * H + h) * HD + 4 * g2;
#pragma unroll
    for (int d = 0; d < ND; d++)
#pragma unroll
        for (int k = 0; k < 4; k++) {
            const float4 gv = *reinterpret_cast<const float4 *>(gate + 32 * d + 8 * k);
            float4 r;
            r.x = o[d][4 * k] * il * omh_sigmoid(gv.x);
            r.y = o[d][4 * k + 1] * il * omh_sigmoid(gv.y);
            r.z = o[d][4 * k + 2] * il * omh_sigmoid(gv.z);
            r.w = o[d][4 * k + 3] * il * omh_sigmoid(gv.w);
            *reinterpret_cast<float4 *>(dst + 32 * d + 8 * k) = r;
        }
    mark(dst);
}

// The flash kernel's splits merged, normalised and gated: a wave per (token,
// head) row (two at HD = 128), lane = 4 columns.  Token t has a partial in
// every split that begins at or before its position.
template <int HD>
__global__ __launch_bounds__(256) void attn_flash_merge_kernel(const AttnArgs a) {
    constexpr int LR = HD / 4;                     // lanes per row
    const size_t th = (size_t)blockIdx.x * (256 / LR) + threadIdx.x / LR;
    if (th >= (size_t)a.T * a.H) return;
    const int c = 4 * (threadIdx.x % LR), t = (int)(th / a.H), h = (int)(th % a.H);
    const int nl = (a.pos + t) / a.kps + 1;        // live splits
    const float *ml = a.pml + 2 * th * a.ns, *po = a.po + th * a.ns * HD + c;
    float M = -INFINITY;
    for (int s = 0; s < nl; s++) M = fmaxf(M, ml[2 * s]);
    float L = 0.f;
    float4 o = f4_zero();
#pragma unroll 4
    for (int s = 0; s < nl; s++) {
        const float f = expf(ml[2 * s] - M);
        L = fmaf(ml[2 * s + 1], f, L);
        o = f4_fma(*reinterpret_cast<const float4 *>(po + (size_t)s * HD), f, o);
    }
    const float il = 1.f / L;
    const float4 gv = *reinterpret_cast<const float4 *>(a.qkv + (size_t)t * a.ld_qkv + (size_t)h * 2 * HD + HD + c);
    float4 r;
    r.x = o.x * il * omh_sigmoid(gv.x);
    r.y = o.y * il * omh_sigmoid(gv.y);
    r.z = o.z * il * omh_sigmoid(gv.z);
    r.w = o.w * il * omh_sigmoid(gv.w);
    *reinterpret_cast<float4 *>(a.ctx + th * HD + c) = r;
}

// One workgroup per (token, head, 64 columns): the CW waves take every
// CW-th split, lane = column, then sum through LDS.
constexpr int kCombineWaves = 8;
template <int HD>
__global__ __launch_bounds__(kCombineWaves * OMH_WAVE) void attn_combine_kernel(const AttnArgs a) {
    constexpr int NCB = HD < OMH_WAVE ? 1 : HD / OMH_WAVE;     // column blocks per head
    constexpr int CW = kCombineWaves;
    __shared__ float so[CW][OMH_WAVE], sl[CW];
    const int th = blockIdx.x / NCB, cb = blockIdx.x % NCB;
    const int t = th / a.H, h = th % a.H, ns = a.ns;
    const int tid = threadIdx.x, lane = tid % OMH_WAVE;
    const int wave = __builtin_amdgcn_readfirstlane(tid / OMH_WAVE);
    const int j = cb * OMH_WAVE + lane;
    const size_t pb = (size_t)th * ns;
    float M = -INFINITY;
    for (int s = lane; s < ns; s += OMH_WAVE) M = fmaxf(M, a.pml[2 * (pb + s)]);
    M = wave_max(M);
    float L = 0.f, o = 0.f;
    const int jc = j < HD ? j : HD - 1;
#pragma unroll 8
    for (int s = wave; s < ns; s += CW) {          // an empty split: m = -inf, weight 0, zero partial
        const float wgt = expf(a.pml[2 * (pb + s)] - M);
        L = fmaf(a.pml[2 * (pb + s) + 1], wgt, L);
        o = fmaf(a.po[(pb + s) * HD + jc], wgt, o);
    }
    so[wave][lane] = o;
    if (lane == 0) sl[wave] = L;
    __syncthreads();
    if (wave == 0 && j < HD) {
        float ls = 0.f, os = 0.f;                  // split 0 always holds key 0: ls > 0
#pragma unroll
        for (int w = 0; w < CW; w++) {
            ls += sl[w];
            os += so[w][lane];
        }
        const float g = a.qkv[(size_t)t * a.ld_qkv + (size_t)h * 2 * HD + HD + j];
        a.ctx[((size_t)t * a.H + h) * HD + j] = os / ls * omh_sigmoid(g);
    }
}

template <int HD>
hipError_t launch_attn_d(const AttnArgs &a, hipStream_t st) {
    static const bool lds_ok = [] {
        bool ok = true;
        if constexpr (HD >= 64) {
            for (const void *f : {(const void *)attn_split_mfma_kernel<HD, false>, (const void *)attn_split_mfma_kernel<HD, true>})
                ok = ok && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)MfmaSplitShape<HD>::LDS) == hipSuccess;
        } else {
            for (const void *f : {(const void *)attn_split_kernel<HD, 1>, (const void *)attn_split_kernel<HD, 2>,
                                  (const void *)attn_split_kernel<HD, 3>, (const void *)attn_split_kernel<HD, 4>,
                                  (const void *)attn_split_kernel<HD, 1, true>, (const void *)attn_split_kernel<HD, 2, true>,
                                  (const void *)attn_split_kernel<HD, 3, true>, (const void *)attn_split_kernel<HD, 4, true>})
                ok = ok && hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, (int)AttnShape<HD>::LDS) == hipSuccess;
        }
        return ok;
    }();
    if (!lds_ok) return hipErrorInvalidValue;
    static_assert(kAttnMaxGroup <= 4 * AttnShape<HD>::NW, "heads per wave");
    // decode steps: the prep is done inside the split kernel (OMH_ATTN_FUSE=0: its own launch, for comparison)
    const bool flash = HD >= 128 && attn_uses_flash(a.T, HD);
    const bool fuse = a.T == 1 && !flash && fuse_prep();
    // (few tokens: a token's rows over several workgroups, one row per wave)
    if (!fuse) {
        const int ny = a.T < 64 ? (a.H + 2 * a.KV + kPrepWaves - 1) / kPrepWaves : 1;
        hipLaunchKernelGGL((attn_prep_kernel<HD>), dim3((unsigned)a.T, (unsigned)ny), dim3(kPrepWaves * OMH_WAVE), 0, st, a);
    }
    if constexpr (HD >= 128) {
        if (attn_uses_flash(a.T, HD)) {
            if (flash_fp32()) {
                const int wpg = ((a.T + 15) / 16 * (a.H / a.KV) + 7) / 8;
                static const bool ok = hipFuncSetAttribute((const void *)attn_flash_kernel<HD>,
                                                           hipFuncAttributeMaxDynamicSharedMemorySize,
                                                           (int)FlashShape<HD>::LDS) == hipSuccess;
                if (!ok) return hipErrorInvalidValue;
                hipLaunchKernelGGL((attn_flash_kernel<HD>), dim3((unsigned)(a.KV * wpg)), dim3(8 * OMH_WAVE),
                                   FlashShape<HD>::LDS, st, a);
                return hipGetLastError();
            }
            using F = Flash3Shape<HD>;
            const int wpg = ((a.T + 31) / 32 * (a.H / a.KV) + F::NW - 1) / F::NW;
            if (a.kps % F::KT != 0) return hipErrorInvalidValue;
            static const bool ok =
                hipFuncSetAttribute((const void *)attn_flash3_kernel<HD, false>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)F::LDS) == hipSuccess &&
                hipFuncSetAttribute((const void *)attn_flash3_kernel<HD, true>,
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)F::LDS) == hipSuccess;
            if (!ok) return hipErrorInvalidValue;
            const dim3 grid((unsigned)(a.KV * a.ns * wpg)), blk(F::NW * OMH_WAVE);
            if (a.img) {
                // the images of every tile of keys 0 .. pos + T - 1, then the kernel copying them
                const long tiles = ((long)a.pos + a.T + F::KT - 1) / F::KT;
                if (a.img_tiles != tiles || (size_t)tiles * F::TILE > (size_t)INT32_MAX) return hipErrorInvalidValue;
                hipLaunchKernelGGL((attn_tile_image_kernel<HD>), dim3((unsigned)(a.KV * tiles)), blk, 0, st, a);
                hipLaunchKernelGGL((attn_flash3_kernel<HD, true>), grid, blk, F::LDS, st, a);
            } else {
                hipLaunchKernelGGL((attn_flash3_kernel<HD, false>), grid, blk, F::LDS, st, a);
            }
            if (a.ns > 1) {
                constexpr int rows = 256 / (HD / 4);
                hipLaunchKernelGGL((attn_flash_merge_kernel<HD>), dim3((unsigned)(((size_t)a.T * a.H + rows - 1) / rows)),
                                   dim3(256), 0, st, a);
            }
            return hipGetLastError();
        }
    }
    if constexpr (HD >= 64) {
        // the K / V slices of a (sequence, kv head) are addressed by 32-bit byte offsets
        if ((size_t)a.max_t * HD * sizeof(float) > (size_t)INT32_MAX) return hipErrorInvalidValue;
        const int nct = (a.T * (a.H / a.KV) + 15) / 16;
        const dim3 grid((unsigned)(a.ns * a.KV * nct)), blk(MfmaSplitShape<HD>::NW * OMH_WAVE);
        const size_t lds = MfmaSplitShape<HD>::LDS;
        if (fuse) hipLaunchKernelGGL((attn_split_mfma_kernel<HD, true>), grid, blk, lds, st, a);
        else hipLaunchKernelGGL((attn_split_mfma_kernel<HD, false>), grid, blk, lds, st, a);
    } else {
        const dim3 grid((unsigned)(a.ns * a.KV * a.T)), blk(AttnShape<HD>::NW * OMH_WAVE);
        const size_t lds = AttnShape<HD>::LDS;
        const int gpw = (a.H / a.KV + AttnShape<HD>::NW - 1) / AttnShape<HD>::NW;
        if (fuse) {
            switch (gpw) {
            case 1: hipLaunchKernelGGL((attn_split_kernel<HD, 1, true>), grid, blk, lds, st, a); break;
            case 2: hipLaunchKernelGGL((attn_split_kernel<HD, 2, true>), grid, blk, lds, st, a); break;
            case 3: hipLaunchKernelGGL((attn_split_kernel<HD, 3, true>), grid, blk, lds, st, a); break;
            default: hipLaunchKernelGGL((attn_split_kernel<HD, 4, true>), grid, blk, lds, st, a); break;
            }
        } else {
            switch (gpw) {
            case 1: hipLaunchKernelGGL((attn_split_kernel<HD, 1>), grid, blk, lds, st, a); break;
            case 2: hipLaunchKernelGGL((attn_split_kernel<HD, 2>), grid, blk, lds, st, a); break;
            case 3: hipLaunchKernelGGL((attn_split_kernel<HD, 3>), grid, blk, lds, st, a); break;
            default: hipLaunchKernelGGL((attn_split_kernel<HD, 4>), grid, blk, lds, st, a); break;
            }
        }
    }
    constexpr int NCB = HD < OMH_WAVE ? 1 : HD / OMH_WAVE;
    hipLaunchKernelGGL((attn_combine_kernel<HD>), dim3((unsigned)(a.T * a.H * NCB)), dim3(kCombineWaves * OMH_WAVE), 0, st, a);
    return hipGetLastError();
}

}  // namespace

bool attn_uses_flash(int T, int hd) {
    if (const char *e = getenv("OMH_ATTN_FLASH"))
        if (e[0] == '0') return false;
    return T >= kFlashMinT && (hd == 128 || hd == 256);
}

template <int HD>
size_t flash_image_bytes_d(int KV, int pos, int T, int *tiles) {
    using F = Flash3Shape<HD>;
    const size_t n = ((size_t)pos + T + F::KT - 1) / F::KT;
    // one kv head's images are addressed with 32-bit buffer offsets: longer
    // steps stage their tiles in the kernel
    if (n * F::TILE > (size_t)INT32_MAX) return 0;
    *tiles = (int)n;
    return (size_t)KV * n * F::TILE;
}

size_t attn_flash_image_bytes(int hd, int KV, int pos, int T, int *tiles) {
    *tiles = 0;
    if (!attn_uses_flash(T, hd) || T < kFlashImageMinT || flash_fp32() || flash_reg()) return 0;
    return hd == 256 ? flash_image_bytes_d<256>(KV, pos, T, tiles) : flash_image_bytes_d<128>(KV, pos, T, tiles);
}

bool attn_supported(int hd, int H, int KV, int rot) {
    return (hd == 32 || hd == 64 || hd == 128 || hd == 256) && KV >= 1 && H >= KV && H % KV == 0 &&
           H / KV <= kAttnMaxGroup && rot >= 0 && rot <= hd && rot % 2 == 0;
}

void attn_plan(int pos, int T, int H, int KV, int hd, int &ns, int &kps) {
    const long nmax = (long)pos + T;                       // keys the last token sees
    // workgroups per key split: a column tile of 16 (token, head) pairs each (width 32: a token each)
    const long per = hd >= 64 ? (long)KV * (((long)T * (H / KV) + 15) / 16) : (long)KV * T;
    // as many splits as leave every workgroup resident at once, one per CU
    // (T = 5 at position 8001 with 260 workgroups, a token each: 47.7 us)
    const long want = std::max(1L, 256 / per);
    long k = (nmax + want - 1) / want;
    k = (k + 63) / 64 * 64;
    kps = (int)k;
    ns = (int)((nmax + k - 1) / k);
}

// Key splits of a prompt step on the flash kernel, by an estimate of its time
// in 32-key tiles of one workgroup: the workgroups of a split sweep their
// tiles with kEnds tiles' worth of prologue and epilogue, one per CU at a time
// (two at head width 128); partials cost a tile per kBytesPerTile written and
// read, and the merge two.  One split where the unsplit workgroups fill the
// chip.  A tile is 2.5 us in a step of 333 tokens at position 6000 (5 splits of
// 40 tiles, 107 us) and 3.6 us at 4096 tokens, where 6.4 MB a tile are 2.6 and
// 1.8 TB/s: a price above what partials cost, on the side of fewer splits.
void attn_flash_plan(int pos, int T, int H, int KV, int hd, long most, int &ns, int &kps) {
    constexpr int KT = 32, NW = 4, kMaxSplits = 64;
    constexpr double kEnds = 3, kBytesPerTile = 6.4e6;
    const long nt = ((long)pos + T + KT - 1) / KT;
    const long wpg = ((long)(T + 31) / 32 * (H / KV) + NW - 1) / NW;
    const double avg = 0.5 * ((double)nt + (double)(pos / KT + 1));   // tiles of a workgroup, unsplit
    const double slots = hd > 128 ? 256 : 512;
    most = std::min(most, (long)(kFlashPartialBytes / ((size_t)T * H * hd * sizeof(float))));   // (0: unsplit)
    double best = 0;
    ns = 1;
    kps = (int)(nt * KT);
    if (flash_fp32()) return;
    for (int s = 1; s <= kMaxSplits && s <= nt && s <= most; s++) {
        const long tps = (nt + s - 1) / s;
        if ((nt + tps - 1) / tps != s) continue;              // the same split as an earlier s
        const double per = s == 1 ? 1 : std::min((double)s, avg / tps + 0.5);   // live splits of a workgroup
        const double units = (double)KV * wpg * per, sum = (double)KV * wpg * avg;
        double cost = tps + kEnds;
        if (units > slots)
            cost = std::max(std::ceil(units / slots) * (sum / units + kEnds),
                            (sum + kEnds * units) / slots + 0.25 * (tps + kEnds));
        if (s > 1) cost += 2 + (double)T * H * per * hd * 8 / kBytesPerTile;
        if (s == 1 || cost < best) {
            best = cost;
            ns = s;
            kps = (int)(tps * KT);
        }
    }
}

hipError_t launch_attn(const AttnArgs &a, int hd, hipStream_t st) {
    if (a.T <= 0) return hipSuccess;
    if (!attn_supported(hd, a.H, a.KV, a.rot) || a.ns < 1 || a.kps < 1 || (long)a.ns * a.kps < (long)a.pos + a.T ||
        a.pos < 0 || (long)a.pos + a.T > a.max_t)
        return hipErrorInvalidValue;
    AttnArgs b = a;
    b.rgrp = group_recip(a.H / a.KV);
    switch (hd) {
    case 32: return launch_attn_d<32>(b, st);
    case 64: return launch_attn_d<64>(b, st);
    case 128: return launch_attn_d<128>(b, st);
    default: return launch_attn_d<256>(b, st);
    }
}

}  // namespace omh
