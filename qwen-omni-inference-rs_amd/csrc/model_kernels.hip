// model_kernels.hip -- decoder kernels around the Q8_0 linears (gfx950).
//
// Orders follow the CPU oracle exactly:
//   SUM64   lane l (of one 64-lane wave) accumulates elements l, l+64, ... from
//           0; the partials fold at distances 32, 16, 8, 4, 2, 1.  Used for the
//           RMSNorm sum of squares and the softmax denominator.
//   scores  q.k sequential over head_dim (src/tensor.rs:2846-2915), then
//           times 1/sqrt(head_dim).
//   ATTN    positions in segments of 64: per segment m_c = max s, e = exp(s - m_c),
//           l_c = SUM64(e), o_c = sum_j e_j v_j (j in order); then the running
//           (m, num, den) update m' = max(m, m_c), a = exp(m - m'),
//           b = exp(m_c - m'), num = num a + b o_c, den = den a + b l_c; the
//           output is num / den.
#include <type_traits>

#include "attn_device.h"
#include "lq8_internal.h"
#include "lq8_numerics.h"

namespace lq8 {

namespace {

// q/k RmsNorm per head, RoPE and KV-cache append for n rows (prefill).
// grid (n, num_heads + num_kv_heads), block 64.
__global__ __launch_bounds__(64) void k_qk_rope_kv(QkRopeLaunch a) {
    const int i = blockIdx.x, h = blockIdx.y, lane = threadIdx.x;
    const int QD = a.num_heads * 128, KD = a.num_kv_heads * 128, row = QD + 2 * KD;
    const int pos = (a.d_pos ? *a.d_pos : a.pos_base) + i;
    const bool isq = h < a.num_heads;
    const float* src = a.qkv + (size_t)i * row + (isq ? h * 128 : QD + (h - a.num_heads) * 128);
    const float* cs = a.cos_t + (size_t)pos * 64;
    const float* sn = a.sin_t + (size_t)pos * 64;
    if (isq) {
        head_norm_rope(src, a.q_norm, cs, sn, a.eps, a.q_out + (size_t)i * QD + h * 128);
    } else {
        const int kvh = h - a.num_heads;
        head_norm_rope(src, a.k_norm, cs, sn, a.eps, a.k_cache + ((size_t)kvh * a.max_pos + pos) * 128);
        const float* v = a.qkv + (size_t)i * row + QD + KD + kvh * 128;
        float* vc = a.v_cache + ((size_t)kvh * a.max_pos + pos) * 128;
        vc[lane] = v[lane];
        vc[lane + 64] = v[lane + 64];
    }
}


// Decode attention, one workgroup per (kv head, group of HG of its G query
// heads, segment slot y), which takes the segments of 64 positions y, y +
// gridDim.y, ... in use (ROUNDS; otherwise there are as many slots as
// segments of capacity, and the instance without the loop keeps its
// registers: 73 VGPRs against 148).  Every workgroup normalizes and rotates its HG query
// heads; the workgroups of the last segment also normalize and rotate the
// new key and use key and value from LDS, and the one of head group 0
// appends them to the cache at the position.  Output: per (segment, q head)
// o_c[128], m_c, l_c at part[(c * H + h) * ATT_PART_STRIDE].
template <bool ROUNDS>
__global__ __launch_bounds__(ATT_THREADS) void k_attn_seg(AttnSegLaunch a) {
    extern __shared__ float sm[];
    const int G = a.num_heads / a.num_kv_heads, HG = a.head_group, NG = G / HG;
    const int kvh = blockIdx.x / NG, hg = blockIdx.x - kvh * NG, c0 = blockIdx.y, b = blockIdx.z;
    const int h0 = kvh * G + hg * HG;  // this workgroup's first query head
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int QD = a.num_heads * 128, KD = a.num_kv_heads * 128;
    a.qkv += b * a.qkv_stride;
    a.k_cache += b * a.kv_stride;
    a.v_cache += b * a.kv_stride;
    a.part += b * a.part_stride;
    const float* Kc = a.k_cache + (size_t)kvh * a.max_pos * 128;
    const float* Vc = a.v_cache + (size_t)kvh * a.max_pos * 128;
    // Loads that do not depend on the position go out before it arrives: the
    // K/V rows of the first ATT_EARLY_SEGS segments of a single sequence
    // (almost always in use; later segments, and batches, whose idle
    // workgroups would multiply the waste, wait) and this wave's first head
    // vector (q head `wave`, or the new k / v).
    float4 kreg[ATT_F4], vreg[ATT_F4];
    const bool early = c0 < ATT_EARLY_SEGS && gridDim.z == 1;
    if (early) seg_load_capacity(Kc, Vc, c0 * SEG, a.max_pos, kreg, vreg);
    float x0 = 0.0f, x1 = 0.0f, n0 = 0.0f, n1 = 0.0f;
    if (wave < HG + 2) {
        const float* src = wave < HG ? a.qkv + (h0 + wave) * 128
                                     : a.qkv + QD + (wave == HG ? 0 : KD) + kvh * 128;
        x0 = src[lane];
        x1 = src[lane + 64];
        if (wave <= HG) {
            const float* w = wave < HG ? a.q_norm : a.k_norm;
            n0 = w[lane];
            n1 = w[lane + 64];
        }
    }
    const int pos = a.d_pos ? a.d_pos[b] : a.pos_base;
    const int L = pos + 1;
    const int C = (L + SEG - 1) / SEG;
    // before any barrier: the whole workgroup leaves (a position outside the
    // cache writes nothing)
    if (c0 >= C || pos < 0 || pos >= a.max_pos) return;
    float* qs = sm;                      // [HG][128]
    float* kn = qs + HG * 128;           // [128]
    float* vn = kn + 128;                // [128]
    float* sc = vn + 128;                // [HG][64]
    float* mlc = sc + HG * SEG;          // [HG][2]
    float* ks = sm + seg_ks_off(HG);     // [64][KPAD], later vs [64][128]
    const float* cs = a.cos_t + (size_t)pos * 64;
    const float* sn = a.sin_t + (size_t)pos * 64;
    // segments c0, c0 + gridDim.y, ... (every workgroup of the launch takes
    // the same number of rounds of its own; the rounds after the first wait
    // for the previous one's reads of the LDS regions)
    for (int c = c0;;) {
        const int js = c * SEG;
        const int nj = min(SEG, L - js);
        const bool last = c == C - 1;
        const int newrow = last ? pos - js : -1;
        if (!(early && c == c0)) seg_load(Kc, Vc, js, nj, kreg, vreg);
        for (int t = wave; t < HG + 2; t += ATT_THREADS / 64) {
            if (t < HG) {
                if (t == wave) head_norm_rope_vals(x0, x1, n0, n1, cs, sn, a.eps, qs + t * 128);
                else head_norm_rope(a.qkv + (h0 + t) * 128, a.q_norm, cs, sn, a.eps, qs + t * 128);
            } else if (t == HG && last) {
                if (t == wave) head_norm_rope_vals(x0, x1, n0, n1, cs, sn, a.eps, kn);
                else head_norm_rope(a.qkv + QD + kvh * 128, a.k_norm, cs, sn, a.eps, kn);
                if (hg == 0) {
                    float* kr = a.k_cache + ((size_t)kvh * a.max_pos + pos) * 128;
                    kr[lane] = kn[lane];
                    kr[lane + 64] = kn[lane + 64];
                }
            } else if (t == HG + 1 && last) {
                const float* v = a.qkv + QD + KD + kvh * 128;
                const float v0 = t == wave ? x0 : v[lane], v1 = t == wave ? x1 : v[lane + 64];
                vn[lane] = v0;
                vn[lane + 64] = v1;
                if (hg == 0) {
                    float* vr = a.v_cache + ((size_t)kvh * a.max_pos + pos) * 128;
                    vr[lane] = v0;
                    vr[lane + 64] = v1;
                }
            }
        }
        __syncthreads();
        seg_scores(kreg, nj, newrow, kn, qs, HG, a.scale, ks, sc, mlc);
        __syncthreads();
        seg_stage_v(vreg, nj, newrow, vn, ks);
        __syncthreads();
        for (int t = tid; t < HG * 128; t += ATT_THREADS) {
            const int h = t >> 7, d = t & 127;
            const float o = pv_chain(sc + h * SEG, ks, d, nj);
            float* p = a.part + ((size_t)c * a.num_heads + h0 + h) * ATT_PART_STRIDE;
            p[d] = o;
            if (d == 0) {
                p[128] = mlc[2 * h];
                p[129] = mlc[2 * h + 1];
            }
        }
        if (!ROUNDS) break;
        c += gridDim.y;
        if (c >= C) break;
        __syncthreads();  // the next round's writes wait for this round's reads of the LDS regions
    }
}

// Attention output of one sequence's head from its per-segment partials,
// one thread per head dimension d: the running update over the segments in
// order, m' = max(m, m_c), a = exp(m - m'), b = exp(m_c - m'),
// num = num * a + b * o_c, den = den * a + b * l_c; out = num / den (the
// arithmetic of the o-projection's XS_ATTN staging, thread by thread).
__global__ __launch_bounds__(128) void k_attn_combine(const float* __restrict__ part, size_t part_stride,
                                                      const int* __restrict__ d_pos, int H, int cmax,
                                                      float* __restrict__ out) {
    const int h = blockIdx.x, b = blockIdx.y, d = threadIdx.x;
    const int C = min(max(d_pos[b], 0) / SEG + 1, cmax);
    const float* pb = part + b * part_stride;
    float m = -__builtin_huge_valf(), den = 0.0f, num = 0.0f;
    for (int c = 0; c < C; c++) {
        const float* p = pb + ((size_t)c * H + h) * ATT_PART_STRIDE;
        const float mc = p[128], lc = p[129];
        const float mn = m > mc ? m : mc;
        const float ea = expf_cr(m - mn), eb = expf_cr(mc - mn);
        den = den * ea + eb * lc;
        num = num * ea + eb * p[d];
        m = mn;
    }
    out[(size_t)b * H * 128 + h * 128 + d] = __fdiv_rn(num, den);
}

// Attention over n query rows with a filled cache (prefill), its output
// quantized into the o projection's operand.  One workgroup of 4 waves per (kv
// head, NV = 16 NVT query vectors): vector v is query head v % G of row i0 +
// v / G.  The 64-position segments run in order, one per step, with the
// running update of each vector.
//
// The chains round every product before it is added, so a multiply-accumulate
// is no fma; the matrix cores take the products: v_mfma_f32_16x16x1_4b_f32
// with C = 0 gives four 16 x 16 outer products, each element round(a * b)
// exactly as v_mul_f32 rounds it (each is fma(a, b, +0): 4e8 products over all
// exponents, subnormal ones among them, agree; a zero factor gives +0 where a
// multiply may give -0, which no sum that starts from +0 can tell), at twice the
// VALU's rate, and the VALU only adds them in the order of the chain.  Operand
// lane l is row (column) l % 16 of block l / 16, and the blocks are four terms
// of the chain: a float4 of 16 consecutive terms per lane group feeds 4
// instructions (component c, block p: term 4 p + c), whose 64 products per
// lane are then added term by term.  Result lane l holds column l % 16, rows
// 4 (l / 16) .. + 3 of every block.
//   scores  rows = 16 keys (wave w: keys 16 w .. of the segment, straight from
//           the cache), columns = 16 query vectors (LDS), terms = d
//   P.V     rows = 16 d (wave w: d 32 w .. + 31, even and odd d as two tiles),
//           columns = 16 query vectors, terms = the segment's 64 positions
//   softmax a thread takes 4 NVT positions of one vector, part + PARTS i, so
//           that SUM64's distances >= PARTS are sums inside the thread
//   output  a wave's 32 d of a vector are one Q8_0 block of the operand
// Positions past a row's own enter P.V with e = 0; their products are zeros
// unless V is not finite there, and a segment where that is so takes the adds
// one by one under the row's length.
//
// Bound: instruction issue.  For 951 rows behind 2048 positions of Qwen3-1.7B
// the VALU instructions (840k cycles per SIMD, about 600k of them the chains'
// adds) and the f32 matrix instructions (303k; they use the same fp32 units, and
// issuing the next group's products between a group's adds changed nothing) fill
// the 1.13M cycles the kernel runs (496 us).  Against one chain per thread from
// LDS followed by the separate quantizer, per layer of Qwen3-0.6B: 1283 -> 398 us
// at 2048 rows, 370 -> 125 at 1024, 109 -> 48 at 512, 20 -> 15 at 128 (where a
// wave's chain latencies bound it), and 5 us of quantizer less.  64 vectors per
// workgroup (256 VGPRs) measured 553 us at 2048 rows.
typedef float v16f __attribute__((ext_vector_type(16)));
constexpr int AR_THREADS = 256;
constexpr int AR_QPAD = 132, AR_SPAD = 68;  // LDS row strides: 16-byte aligned, 4 banks apart

// exp's constants in memory: read by scalar loads where they are used (as
// literals in a loop they are hoisted into 26 VGPRs)
__constant__ const double exp_consts[EXP_CONSTS] = LQ8_EXP_CONSTS;
typedef const double __attribute__((address_space(4))) * ExpConsts;
__device__ __forceinline__ ExpConsts exp_consts_here() {
    ExpConsts c = (ExpConsts)exp_consts;
    asm volatile("" : "+s"(c));
    return c;
}

__device__ __forceinline__ v16f products(float a, float b) {
    const v16f z = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
    return __builtin_amdgcn_mfma_f32_16x16x1f32(a, b, z, 0, 0, 0);
}

// s[v] += the 16 terms of (a, b) in order; MASKED: only terms j0 + t < nj.
// The empty asm statements keep one group's 64 products in registers at a
// time (a pure value is otherwise computed at its use).
template <bool MASKED>
__device__ __forceinline__ void add_terms(const float (&a)[4], float4 b, float (&s)[4], int j0, int nj) {
    asm volatile("" : "+v"(b.x), "+v"(b.y), "+v"(b.z), "+v"(b.w));
    const v16f p0 = products(a[0], b.x), p1 = products(a[1], b.y), p2 = products(a[2], b.z), p3 = products(a[3], b.w);
#pragma unroll
    for (int p = 0; p < 4; p++) {
#pragma unroll
        for (int c = 0; c < 4; c++) {
            const v16f& q = c == 0 ? p0 : c == 1 ? p1 : c == 2 ? p2 : p3;
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const float t = s[v] + q[4 * p + v];
                s[v] = !MASKED || j0 + 4 * p + c < nj ? t : s[v];
            }
        }
    }
    asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s[2]), "+v"(s[3]));
    __builtin_amdgcn_sched_barrier(0);
}

// 8 codes of a Q8_0 block as the two dwords of its operand bytes
__device__ __forceinline__ uint2 codes8(const float (&y)[8], float id) {
    uint32_t w[2];
#pragma unroll
    for (int i = 0; i < 2; i++)
        w[i] = (uint32_t)(quant_code(y[4 * i], id) & 0xFF) | ((uint32_t)(quant_code(y[4 * i + 1], id) & 0xFF) << 8) |
               ((uint32_t)(quant_code(y[4 * i + 2], id) & 0xFF) << 16) | ((uint32_t)(quant_code(y[4 * i + 3], id) & 0xFF) << 24);
    return make_uint2(w[0], w[1]);
}

template <int NVT>
__global__ __launch_bounds__(AR_THREADS) __attribute__((amdgpu_waves_per_eu(2))) void k_attn_rows(AttnRowsLaunch a) {
    static_assert(NVT == 1 || NVT == 2, "16 or 8 threads per softmax vector");
    constexpr int NV = 16 * NVT, PARTS = AR_THREADS / NV, KPT = SEG / PARTS;
    __shared__ __attribute__((aligned(16))) float qs[NV * AR_QPAD];
    __shared__ __attribute__((aligned(16))) float sbuf[2][NV * AR_SPAD];  // scores, then exps
    __shared__ float coef[2][NV * 2];                                     // the step's a, b of each vector
    __shared__ float dens[NV];
    const int tid = threadIdx.x, lane = tid & 63, r = lane & 15, p = lane >> 4;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int G = a.num_heads / a.num_kv_heads, R = NV / G;
    const int QD = a.num_heads * 128;
    // the rows with the most positions first
    const int kvh = blockIdx.x, i0 = ((int)gridDim.y - 1 - (int)blockIdx.y) * R;
    const int nr = min(R, a.n - i0);
    const int L0 = a.pos_base + i0 + 1;   // positions of the first row
    const int Lmax = L0 + nr - 1;         // and of the last
    const float* Kc = a.k_cache + (size_t)kvh * a.max_pos * 128;
    const float* Vc = a.v_cache + (size_t)kvh * a.max_pos * 128;
    float4 kr[8];
    float2 vr[4][4];
    // a whole segment loads from a uniform base with constant lane offsets; in
    // the last one the rows past the last row's position read that row
    const unsigned ko = ((16 * w + r) * 128 + 4 * p) * 4, vo = (4 * p * 128 + 32 * w + 2 * r) * 4;
    auto load_k = [&](int js) {
        if (js + SEG <= Lmax) {
            const char* kp = (const char*)(Kc + (size_t)js * 128);
#pragma unroll
            for (int i = 0; i < 8; i++) kr[i] = *(const float4*)(kp + ko + 64 * i);
        } else if (js < Lmax) {
            const float* kp = Kc + (size_t)min(js + 16 * w + r, Lmax - 1) * 128 + 4 * p;
#pragma unroll
            for (int i = 0; i < 8; i++) kr[i] = *(const float4*)(kp + 16 * i);
        }
    };
    auto load_v = [&](int js) {
        if (js + SEG <= Lmax) {
            const char* vp = (const char*)(Vc + (size_t)js * 128);
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int c = 0; c < 4; c++) vr[i][c] = *(const float2*)(vp + 16 * 512 * i + vo + 512 * c);
        } else if (js < Lmax) {
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int c = 0; c < 4; c++)
                    vr[i][c] = *(const float2*)(Vc + (size_t)min(js + 16 * i + 4 * p + c, Lmax - 1) * 128 + 32 * w + 2 * r);
        }
    };
    load_k(0);
    for (int e = tid; e < NV * 32; e += AR_THREADS) {
        const int v = e >> 5, c4 = e & 31, rr = min(v / G, nr - 1), h = v % G;  // spare vectors repeat the last row
        *(float4*)(qs + v * AR_QPAD + 4 * c4) =
            *(const float4*)(a.q_rows + (size_t)(i0 + rr) * QD + (kvh * G + h) * 128 + 4 * c4);
    }
    load_v(0);
    int lenv[NVT];  // positions of the lane's column vectors
    float num[NVT][2][4];
#pragma unroll
    for (int vt = 0; vt < NVT; vt++) {
        lenv[vt] = L0 + min((16 * vt + r) / G, nr - 1);
#pragma unroll
        for (int v = 0; v < 4; v++) num[vt][0][v] = num[vt][1][v] = 0.0f;
    }
    const int sv = tid / PARTS, part = tid % PARTS;  // this thread's softmax vector
    const int slen = L0 + min(sv / G, nr - 1);
    float mrun = -__builtin_huge_valf(), den = 0.0f;
    __syncthreads();
    int buf = 0;
    for (int js = 0; js < Lmax; js += SEG, buf ^= 1) {
        float* S = sbuf[buf];
        const bool full = js + SEG <= L0;  // every row has the whole segment
        // scores of the wave's 16 keys
#pragma unroll
        for (int vt = 0; vt < NVT; vt++) {
            float s[4] = {0.0f, 0.0f, 0.0f, 0.0f};
            const float* qp = qs + (16 * vt + r) * AR_QPAD + 4 * p;
            float4 q = *(const float4*)qp;
#pragma unroll
            for (int i = 0; i < 8; i++) {
                const float ka[4] = {kr[i].x, kr[i].y, kr[i].z, kr[i].w};
                const float4 qn = *(const float4*)(qp + 16 * min(i + 1, 7));  // the next group's, ahead of the adds
                add_terms<false>(ka, q, s, 0, 0);
                q = qn;
            }
            *(float4*)(S + (16 * vt + r) * AR_SPAD + 16 * w + 4 * p) =
                make_float4(s[0] * a.scale, s[1] * a.scale, s[2] * a.scale, s[3] * a.scale);
        }
        load_k(js + SEG);
        lds_sync();
        {
            // m_c, e, l_c of the thread's vector, then its running update
            const ExpConsts ec = exp_consts_here();
            const int nj = min(SEG, slen - js);
            float* row = S + sv * AR_SPAD + part;
            float x[KPT + 1];  // the thread's scores and the update's exponent
            float mc = -__builtin_huge_valf();
#pragma unroll
            for (int i = 0; i < KPT; i++) x[i] = row[PARTS * i];
            if (!full) {
#pragma unroll
                for (int i = 0; i < KPT; i++) x[i] = part + PARTS * i < nj ? x[i] : -__builtin_huge_valf();
            }
#pragma unroll
            for (int i = 0; i < KPT; i++) mc = fmaxf(mc, x[i]);
            mc = fmaxf(mc, lane_xor<1>(mc));
            mc = fmaxf(mc, lane_xor<2>(mc));
            mc = fmaxf(mc, lane_xor<4>(mc));
            if (PARTS > 8) mc = fmaxf(mc, lane_xor<8>(mc));
#pragma unroll
            for (int i = 0; i < KPT; i++) x[i] = x[i] - mc;
            if (!full) {
                // (a row with no position here has mc = -inf)
#pragma unroll
                for (int i = 0; i < KPT; i++) x[i] = part + PARTS * i < nj ? x[i] : -__builtin_huge_valf();
            }
            const float mn = mrun > mc ? mrun : mc;
            x[KPT] = (part & 1 ? mc : mrun) - mn;
            expf_le0(x, ec);
#pragma unroll
            for (int i = 0; i < KPT; i++) row[PARTS * i] = x[i];
#pragma unroll
            for (int d = KPT / 2; d > 0; d /= 2)
#pragma unroll
                for (int i = 0; i < d; i++) x[i] = x[i] + x[i + d];
            float lc = x[0];
            if (PARTS > 8) lc = lc + lane_xor<8>(lc);
            lc = lc + lane_xor<4>(lc);
            lc = lc + lane_xor<2>(lc);
            lc = lc + lane_xor<1>(lc);
            const float ex = x[KPT], ey = lane_xor<1>(ex);
            if (part < 2) coef[buf][2 * sv + part] = ex;
            const float dn = (part & 1 ? den * ey : den * ex) + (part & 1 ? ex * lc : ey * lc);
            den = nj > 0 ? dn : den;
            mrun = nj > 0 ? mn : mrun;
        }
        lds_sync();
        // WHOLE: the step is full; M: V is not finite somewhere in the segment
        auto pv = [&](auto whole, auto masked) {
            constexpr bool WHOLE = decltype(whole)::value, M = decltype(masked)::value;
#pragma unroll
            for (int vt = 0; vt < NVT; vt++) {
                float o[2][4] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
                const int nj = lenv[vt] - js;
                const float* ep = S + (16 * vt + r) * AR_SPAD + 4 * p;
                float4 e = *(const float4*)ep;
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    if (!WHOLE && js + 16 * i >= Lmax) break;  // no row has these positions
                    const float4 en = *(const float4*)(ep + 16 * min(i + 1, 3));
                    const float v0[4] = {vr[i][0].x, vr[i][1].x, vr[i][2].x, vr[i][3].x};
                    const float v1[4] = {vr[i][0].y, vr[i][1].y, vr[i][2].y, vr[i][3].y};
                    add_terms<M>(v0, e, o[0], 16 * i, nj);
                    add_terms<M>(v1, e, o[1], 16 * i, nj);
                    e = en;
                }
                const float ca = coef[buf][2 * (16 * vt + r)], cb = coef[buf][2 * (16 * vt + r) + 1];
#pragma unroll
                for (int t = 0; t < 2; t++)
#pragma unroll
                    for (int v = 0; v < 4; v++) {
                        const float y = num[vt][t][v] * ca + cb * o[t][v];
                        num[vt][t][v] = WHOLE || nj > 0 ? y : num[vt][t][v];
                    }
            }
        };
        if (full) {
            pv(std::true_type{}, std::false_type{});
        } else {
            uint32_t top = 0;
#pragma unroll
            for (int i = 0; i < 4; i++)
#pragma unroll
                for (int c = 0; c < 4; c++) {
                    top = max(top, __float_as_uint(vr[i][c].x) & 0x7FFFFFFFu);
                    top = max(top, __float_as_uint(vr[i][c].y) & 0x7FFFFFFFu);
                }
            if (__all(top < 0x7F800000u)) pv(std::false_type{}, std::false_type{});
            else pv(std::false_type{}, std::true_type{});
        }
        load_v(js + SEG);
    }
    if (part == 0) dens[sv] = den;
    __syncthreads();
    // lane (r, p): values 8 p .. + 7 of block 4 head + w of vector 16 vt + r
    const int nb = a.num_heads * 4, np = nb / 2, nbp4 = 2 * ((nb + GEMM_GROUP - 1) / GEMM_GROUP);
#pragma unroll
    for (int vt = 0; vt < NVT; vt++) {
        const int v = 16 * vt + r, rr = v / G, head = kvh * G + v - rr * G, row = i0 + rr;
        const float dn = dens[v];
        float y[8], amax = 0.0f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            y[i] = __fdiv_rn(num[vt][i & 1][i >> 1], dn);
            amax = fmaxf(amax, fabsf(y[i]));
        }
        amax = fmaxf(amax, lane_xor<16>(amax));
        amax = fmaxf(amax, lane_xor<32>(amax));
        const QBlock qb = block_scale(amax);
        const uint2 c = codes8(y, block_inv(qb.d));
        if (rr < nr) {  // (not the spare vectors)
            const int b = head * 4 + w;
            *(uint2*)(a.codes + code_off(row / TILE_ROWS, np, b, p >> 1, row % TILE_ROWS) + 8 * (p & 1)) = c;
            if ((p & 1) == 0) {
                uint32_t* xs = a.scales + ((size_t)((row >> 5) * nbp4 + (b >> 2)) * 64 + 16 * p + (row & 31)) * 4;
                xs[w] = p ? 0u : qb.d16;
                // an odd head count: the operand's last 4 blocks are padding
                if (w == 3 && head == a.num_heads - 1 && (nb >> 2) < nbp4) *(uint4*)(xs + 256) = make_uint4(0, 0, 0, 0);
            }
        }
    }
}

// RmsNorm of each row (src/rms_norm.rs:143-176), one wave per row.
template <int U>
__global__ __launch_bounds__(64) void k_rms_norm_rows(const float* __restrict__ x, const float* __restrict__ w, int dim,
                                                      float eps, float* __restrict__ y) {
    // U <= 32: the row and the norm weights stay in registers (loaded together);
    // U == 0: longer rows, two passes of 16 loads in flight per lane.
    const int r = blockIdx.x, lane = threadIdx.x;
    const float* xr = x + (size_t)r * dim;
    float* yr = y + (size_t)r * dim;
    if (U > 0) {
        constexpr int UU = U > 0 ? U : 1;
        float v[UU], wn[UU];
#pragma unroll
        for (int u = 0; u < UU; u++) {
            v[u] = xr[min(lane + 64 * u, dim - 1)];
            wn[u] = w[min(lane + 64 * u, dim - 1)];
        }
        float acc = 0.0f;
#pragma unroll
        for (int u = 0; u < UU; u++)
            if (lane + 64 * u < dim) {
                const float b = bf16_round(v[u]);
                acc = acc + b * b;
            }
        acc = wave_sum64(acc);
        const float inv = __fdiv_rn(1.0f, __builtin_sqrtf(__fdiv_rn(acc, (float)dim) + eps));
#pragma unroll
        for (int u = 0; u < UU; u++)
            if (lane + 64 * u < dim) yr[lane + 64 * u] = bf16_round((bf16_round(v[u]) * inv) * bf16_round(wn[u]));
        return;
    }
    constexpr int L = 16;  // loads in flight per lane
    float acc = 0.0f;
    for (int i0 = lane; i0 < dim; i0 += 64 * L) {
        float v[L];
#pragma unroll
        for (int u = 0; u < L; u++) v[u] = xr[min(i0 + 64 * u, dim - 1)];
#pragma unroll
        for (int u = 0; u < L; u++)
            if (i0 + 64 * u < dim) {
                const float b = bf16_round(v[u]);
                acc = acc + b * b;
            }
    }
    acc = wave_sum64(acc);
    const float mean = __fdiv_rn(acc, (float)dim);
    const float inv = __fdiv_rn(1.0f, __builtin_sqrtf(mean + eps));
    for (int i0 = lane; i0 < dim; i0 += 64 * L) {
        float v[L], wv[L];
#pragma unroll
        for (int u = 0; u < L; u++) {
            const int i = min(i0 + 64 * u, dim - 1);
            v[u] = xr[i];
            wv[u] = w[i];
        }
#pragma unroll
        for (int u = 0; u < L; u++)
            if (i0 + 64 * u < dim) yr[i0 + 64 * u] = bf16_round((bf16_round(v[u]) * inv) * bf16_round(wv[u]));
    }
}

// act = silu(gate) * up (src/mlp.rs:151-164; silu src/tensor.rs:1978).
__global__ void k_silu_mul(const float* __restrict__ gu, int rows, int inter, float* __restrict__ act) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (size_t)rows * inter) return;
    const size_t r = idx / inter, j = idx % inter;
    const float g = gu[r * 2 * inter + j], u = gu[r * 2 * inter + inter + j];
    const float s = __fdiv_rn(g, 1.0f + expf_cr(-g));
    act[idx] = s * u;
}

// Tensor::silu f32 branch (src/tensor.rs:1978): x / (1 + exp(-x)).
__global__ void k_silu(const float* __restrict__ x, size_t n, float* __restrict__ y) {
    const size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= n) return;
    const float v = x[idx];
    y[idx] = __fdiv_rn(v, 1.0f + expf_cr(-v));
}

inline unsigned grid1(size_t n, unsigned block) { return (unsigned)((n + block - 1) / block); }

constexpr int ATT_WG_TARGET = 512;  // decode attention workgroups sought per launch (2 per CU)
constexpr int ATT_MIN_SLOTS = 8;    // segment slots at least (512 positions without a second round)

size_t seg_smem(int G) { return ((size_t)seg_ks_off(G) + (size_t)SEG * KPAD) * sizeof(float); }

}  // namespace

bool attention_supported(int num_heads, int num_kv_heads, int head_dim) {
    return head_dim == 128 && num_kv_heads > 0 && num_heads % num_kv_heads == 0 &&
           num_heads / num_kv_heads <= ATT_MAX_GROUP;
}

lq8_status launch_qk_rope_kv(hipStream_t s, const QkRopeLaunch& a) {
    if (a.head_dim != 128) return fail(LQ8_ERR_SHAPE_MISMATCH, "head_dim must be 128");
    const dim3 grid((unsigned)a.n, (unsigned)(a.num_heads + a.num_kv_heads));
    hipLaunchKernelGGL(k_qk_rope_kv, grid, dim3(64), 0, s, a);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

lq8_status launch_attention_seg(hipStream_t s, const AttnSegLaunch& a) {
    if (!attention_supported(a.num_heads, a.num_kv_heads, 128))
        return fail(LQ8_ERR_SHAPE_MISMATCH, "attention: unsupported head layout");
    const int G = a.num_heads / a.num_kv_heads;
    const int cmax = (a.max_pos + SEG - 1) / SEG;
    if (a.batch <= 0) return fail(LQ8_ERR_INVALID_ARG, "attention: batch must be positive");
    AttnSegLaunch b = a;
    if (b.head_group <= 0 || G % b.head_group) b.head_group = G;
    const int NG = G / b.head_group;
    // segment slots: all cmax segments up to about ATT_WG_TARGET workgroups
    // (at least ATT_MIN_SLOTS slots); a long max_positions (Qwen3's 40960:
    // 640 segments) no longer launches a workgroup per segment of capacity,
    // almost all of them idle, and a workgroup loops over its segments
    const int per_slot = a.num_kv_heads * NG * a.batch;
    const int slots = std::min(cmax, std::max(ATT_MIN_SLOTS, (ATT_WG_TARGET + per_slot - 1) / per_slot));
    const dim3 grid((unsigned)(a.num_kv_heads * NG), (unsigned)slots, (unsigned)a.batch);
    if (slots < cmax) hipLaunchKernelGGL(k_attn_seg<true>, grid, dim3(ATT_THREADS), seg_smem(b.head_group), s, b);
    else hipLaunchKernelGGL(k_attn_seg<false>, grid, dim3(ATT_THREADS), seg_smem(b.head_group), s, b);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

lq8_status launch_attention_combine(hipStream_t s, const float* part, size_t part_stride, const int* d_pos,
                                    int batch, int num_heads, int cmax, float* out) {
    if (batch <= 0 || num_heads <= 0 || cmax <= 0) return LQ8_OK;
    hipLaunchKernelGGL(k_attn_combine, dim3((unsigned)num_heads, (unsigned)batch), dim3(128), 0, s, part, part_stride,
                       d_pos, num_heads, cmax, out);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

lq8_status launch_attention_rows(hipStream_t s, const AttnRowsLaunch& a) {
    if (!attention_supported(a.num_heads, a.num_kv_heads, 128))
        return fail(LQ8_ERR_SHAPE_MISMATCH, "attention: unsupported head layout");
    const int G = a.num_heads / a.num_kv_heads;
    // 32 query vectors per workgroup where that still leaves four workgroups a
    // CU (the per-step work is shared by more rows: 398 against 415 us at 2048
    // rows of Qwen3-0.6B), else 16 (the rows' lengths balance better: 125
    // against 152 us at 1024 rows, 48 against 72 at 512, 15 against 24 at 128).
    // Behind a cache the lengths differ less and 16 loses that: 1024 rows behind
    // 1024 positions 293 against 291, behind 2048 472 against 444
    auto tiles = [&](int nv) { return (a.n + nv / G - 1) / (nv / G); };
    const bool two = a.num_kv_heads * tiles(32) >= 1024;
    const dim3 grid((unsigned)a.num_kv_heads, (unsigned)tiles(two ? 32 : 16));
    if (two) hipLaunchKernelGGL(k_attn_rows<2>, grid, dim3(AR_THREADS), 0, s, a);
    else hipLaunchKernelGGL(k_attn_rows<1>, grid, dim3(AR_THREADS), 0, s, a);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

lq8_status launch_rms_norm_rows(hipStream_t s, const float* x, const float* w, int rows, int dim, float eps, float* y) {
    const dim3 grid((unsigned)rows);
    const int u = (dim + 63) / 64;
    if (u <= 4) hipLaunchKernelGGL(k_rms_norm_rows<4>, grid, dim3(64), 0, s, x, w, dim, eps, y);
    else if (u <= 8) hipLaunchKernelGGL(k_rms_norm_rows<8>, grid, dim3(64), 0, s, x, w, dim, eps, y);
    else if (u <= 16) hipLaunchKernelGGL(k_rms_norm_rows<16>, grid, dim3(64), 0, s, x, w, dim, eps, y);
    else if (u <= 32) hipLaunchKernelGGL(k_rms_norm_rows<32>, grid, dim3(64), 0, s, x, w, dim, eps, y);
    else hipLaunchKernelGGL(k_rms_norm_rows<0>, grid, dim3(64), 0, s, x, w, dim, eps, y);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

lq8_status launch_silu_mul(hipStream_t s, const float* gu, int rows, int inter, float* act) {
    const size_t n = (size_t)rows * inter;
    if (!n) return LQ8_OK;
    hipLaunchKernelGGL(k_silu_mul, dim3(grid1(n, 256)), dim3(256), 0, s, gu, rows, inter, act);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

lq8_status launch_silu(hipStream_t s, const float* x, size_t n, float* y) {
    if (!n) return LQ8_OK;
    hipLaunchKernelGGL(k_silu, dim3(grid1(n, 256)), dim3(256), 0, s, x, n, y);
    LQ8_HIP(hipGetLastError());
    return LQ8_OK;
}

}  // namespace lq8
