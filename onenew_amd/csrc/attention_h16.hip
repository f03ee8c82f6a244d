// Attention with 16-bit operands (bf16 / fp16 q, k, v and result in memory, fp32 scores and Softmax): the 16-bit storage
// form of attention.hip, same chain of reference operators (device/x86/MatMul/mat_mul.c:10-102, device/x86/Softmax/
// softmax.c:26-59, Transposes folded into strides), same trick: a wavefront computes the TRANSPOSED scores S^T = k q^T
// with v_mfma_f32_32x32x16_{bf16,f16}, so a lane owns one query and, per 32-key tile, the 16 keys 8 (r / 4) + 4 (lane / 32)
// + r % 4, the Softmax is a reduction inside the lane, and the probabilities feed the second product out^T = v^T P^T from
// the registers they are in.  An MFMA step of the second product takes 8 reduction indices per lane half: registers
// 8 g .. 8 g + 7 of a tile, i.e. the keys 32 t + 16 g + 8 (j / 4) + 4 (lane / 32) + j % 4, rounded to the 16-bit type and
// packed; the A operand for them is two 8-byte reads of v that transpose on their way out of LDS (ds_read_b64_tr_b16).  What is
// rounded to the operand type before the second product is exp(x - max), and the result is divided by their sum: the relative rounding of
// a probability, which is what 16-bit operands mean for a MatMul, without a product for each of them; everything before it (scores,
// maximum, exponentials, sum) is fp32.  Head dimension 64, at most 256 tokens.
//
// What bounds it: one copy of k and v a head, one trip to memory, 3 us of a launch with its start; then the Softmax, 20 vector cycles and 16 of
// the exponential a score, two wavefronts a SIMD where heads have seven tiles of queries, the matrix instructions behind them.
// 64 x 3 heads of 197 tokens 10.0 -> 8.9 us (their 19 MB are 4 of a large copy), 48 x 3 of 225 11.1 -> 9.3, 24 x 3 of 256 9.5 -> 7.3, 128 x 3 of 100
// 9.8 -> 7.4 (with v transposed by registers, q and the result a row a lane and the probabilities normalised one by one before), the error
// against 64 bits 0.65-0.95 of what it was.
#include "igemm_kernel.hpp"

namespace onhip {

struct AttnH16Params {
    const unsigned short *q, *k, *v;
    unsigned short *o;
    long long qs[3], ks[3], vs[3], os[3];   // element strides of (batch, head, token); the head dimension is contiguous
    int heads, tokens;
    float scale;
};

// NW wavefronts of 32 queries each share one copy of k and v in LDS
template <int DT, int NKT, int NW>
__global__ __launch_bounds__(64 * NW, 2) void attention_h16_kernel(const AttnH16Params p) {
    constexpr int HD = 64, KEYS = NKT * 32, NT = 64 * NW;
    __shared__ uint4 Ks[KEYS * HD / 8];   // rows of k, by `unit` below
    // rows of v as they are, the two halves of rows 2 and 3 of four swapped: a transposing read takes 64 bytes of four rows, every bank once
    __shared__ __attribute__((aligned(16))) unsigned short Vs[KEYS * HD];
    // a wavefront's rows of q, later of the result: memory is read and written eight lanes to a row of 128 bytes (a row a lane, 64 cycles of
    // the compute unit's address path each, were 2 us of a launch)
    __shared__ uint4 Ws[NW][32 * HD / 8];

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int bh = blockIdx.y, b = bh / p.heads, h = bh - b * p.heads;
    const int T = p.tokens;
    const unsigned short *kb = p.k + b * p.ks[0] + h * p.ks[1];
    const unsigned short *vb = p.v + b * p.vs[0] + h * p.vs[1];

    // where the 16 bytes `u` of a row of 128 lie: neither 32 lanes that take one `u` of 32 rows each nor eight that take a row meet in a bank
    auto unit = [](int row, int u) { return row * 8 + (u ^ (row >> 1 & 7)); };
    // all loads first; rows past the last token as zeros
    constexpr int PARTS = HD / 8, NK = (KEYS * PARTS + NT - 1) / NT;
    const int q0 = (blockIdx.x * NW + wave) * 32;
    const unsigned short *qb = p.q + b * p.qs[0] + h * p.qs[1];
    uint4 kq[NK], vq[NK], qf[HD / 16];
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int key = (tid + i * NT) / PARTS, part = tid % PARTS;
        kq[i] = make_uint4(0u, 0u, 0u, 0u);
        if (key < T) kq[i] = *reinterpret_cast<const uint4 *>(kb + key * p.ks[2] + part * 8);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int query = q0 + i * 8 + lane / 8;
        qf[i] = make_uint4(0u, 0u, 0u, 0u);
        if (query < T) qf[i] = *reinterpret_cast<const uint4 *>(qb + query * p.qs[2] + lane % 8 * 8);
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int key = (tid + i * NT) / PARTS, part = tid % PARTS;
        vq[i] = make_uint4(0u, 0u, 0u, 0u);
        if (key < T) vq[i] = *reinterpret_cast<const uint4 *>(vb + key * p.vs[2] + part * 8);
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int f = tid + i * NT;
        if (f < KEYS * PARTS) Ks[unit(f / PARTS, f % PARTS)] = kq[i];
    }
    // this lane's query row: the channels 16 s + 8 (lane / 32) .. + 7 of MFMA step s
    uint4 *const mine = Ws[wave];
#pragma unroll
    for (int i = 0; i < 4; ++i) mine[unit(i * 8 + lane / 8, lane % 8)] = qf[i];
#pragma unroll
    for (int st = 0; st < HD / 16; ++st) qf[st] = mine[unit(li, 2 * st + lh)];
    if (p.scale < 0.0f) {   // uniform: the scale's sign is the query's, so that the largest score stays it when scaled
#pragma unroll
        for (int st = 0; st < HD / 16; ++st) {
            qf[st].x ^= 0x80008000u; qf[st].y ^= 0x80008000u; qf[st].z ^= 0x80008000u; qf[st].w ^= 0x80008000u;
        }
    }
#pragma unroll
    for (int i = 0; i < NK; ++i) {
        const int f = tid + i * NT, key = f / PARTS, part = f % PARTS;
        if (f < KEYS * PARTS) *reinterpret_cast<uint4 *>(Vs + key * HD + (part ^ (key >> 1 & 1) * 4) * 8) = vq[i];
    }
    __syncthreads();
    if (q0 >= T) return;   // a wavefront without queries (uniform); nothing below synchronises

    auto mfma = [](const uint4 &a, const uint4 &bq, f32x16 c) __attribute__((always_inline)) {
        if constexpr (DT == DT_BF16)
            return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, bq), c, 0, 0, 0);
        else
            return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, bq), c, 0, 0, 0);
    };

    // S^T = k q^T, and the largest score of a query over the keys there are
    f32x16 s[NKT];
    float mx = -INFINITY;
#pragma unroll
    for (int t = 0; t < NKT; ++t) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[t][r] = 0.0f;
#pragma unroll
        for (int st = 0; st < HD / 16; ++st)
            s[t] = mfma(Ks[unit(32 * t + li, 2 * st + lh)], qf[st], s[t]);
    }
#pragma unroll
    for (int t = 0; t < NKT; ++t)
        if (32 * t + 32 <= T) {   // uniform: every key of the tile exists
#pragma unroll
            for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[t][r]);
        } else {
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * t + 8 * (r / 4) + 4 * lh + (r % 4) < T) mx = fmaxf(mx, s[t][r]);
        }
    mx = fmaxf(mx, __shfl_xor(mx, 32, 64));

    // Softmax over the keys in fp32 (softmax.c:26-59), exp(scale (s - max)) as one fused product into the exponential base 2, and behind each tile
    // its part of out^T = v^T P^T.  bf16 has fp32's range, and a sum of 256 of its largest values leaves it: 2^-8 of them.
    const float c = __fmul_rn(fabsf(p.scale), 1.44269504088896340736f);
    const float shift = DT == DT_BF16 ? -__fadd_rn(__fmul_rn(mx, c), 8.0f) : -__fmul_rn(mx, c);
    f32x16 o[2];
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
    // of 16 lanes, four read the 32 bytes of 16 channels of one key, and each gets four keys of one channel
    typedef short s16x4 __attribute__((ext_vector_type(4)));
    typedef __attribute__((address_space(3))) s16x4 *lds_s16x4_t;
    const int j = lane & 15;
    const unsigned short *vr[2];
#pragma unroll
    for (int d = 0; d < 2; ++d) vr[d] = Vs + (4 * lh + j / 4) * HD + (d ^ (j >> 3)) * 32 + li / 16 * 16 + j % 4 * 4;
    float sum = 0.0f;
#pragma unroll
    for (int t = 0; t < NKT; ++t) {
        float e[16];
#pragma unroll
        for (int r = 0; r < 16; ++r) e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[t][r], c, shift));
        if (32 * t + 32 > T)   // uniform
#pragma unroll
            for (int r = 0; r < 16; ++r)
                if (32 * t + 8 * (r / 4) + 4 * lh + (r % 4) >= T) e[r] = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) sum += e[r];
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            const uint4 pq = make_uint4(pack_h16<DT>(e[8 * g], e[8 * g + 1]), pack_h16<DT>(e[8 * g + 2], e[8 * g + 3]),
                                        pack_h16<DT>(e[8 * g + 4], e[8 * g + 5]), pack_h16<DT>(e[8 * g + 6], e[8 * g + 7]));
#pragma unroll
            for (int d = 0; d < 2; ++d) {   // keys 4 lh .. + 3 and 8 + 4 lh .. + 3 of the 16
                const unsigned short *at = vr[d] + (32 * t + 16 * g) * HD;
                const uint2 lo = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t) at));
                const uint2 hi = __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t) (at + 8 * HD)));
                o[d] = mfma(make_uint4(lo.x, lo.y, hi.x, hi.y), pq, o[d]);
            }
        }
    }
    sum += __shfl_xor(sum, 32, 64);
    const float inv = 1.0f / sum;

#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            reinterpret_cast<uint2 *>(mine + unit(li, 4 * d + g))[lh] =
                make_uint2(pack_h16<DT>(__fmul_rn(o[d][4 * g], inv), __fmul_rn(o[d][4 * g + 1], inv)),
                           pack_h16<DT>(__fmul_rn(o[d][4 * g + 2], inv), __fmul_rn(o[d][4 * g + 3], inv)));
    unsigned short *ob = p.o + b * p.os[0] + h * p.os[1];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int query = q0 + i * 8 + lane / 8;
        if (query < T) *reinterpret_cast<uint4 *>(ob + query * p.os[2] + lane % 8 * 8) = mine[unit(i * 8 + lane / 8, lane % 8)];
    }
}

template <int DT>
static int attention_h16_launch_dt(const AttnH16Params &p, int batch, hipStream_t stream) {
    const int nkt = (p.tokens + 31) / 32;
    const unsigned heads = (unsigned) (batch * p.heads);
    // Eight wavefronts share a copy of k and v where four would make a second copy for the same head, and the heads alone give
    // half of the CUs a workgroup (fewer heads: two workgroups on two CUs do the staging side by side).
    const bool wide = nkt > 4 && heads >= 128;
    const dim3 grid(wide ? 1u : (unsigned) ((p.tokens + 127) / 128), heads);
    // one wavefront where there is one tile (24 heads of one token 4.4 us in four wavefronts with two tiles, 3.8 here; one head of five tokens 3.4 and 2.8)
    if (nkt == 1) hipLaunchKernelGGL((attention_h16_kernel<DT, 1, 1>), grid, dim3(64), 0, stream, p);
    else if (nkt <= 2) hipLaunchKernelGGL((attention_h16_kernel<DT, 2, 4>), grid, dim3(256), 0, stream, p);
    else if (nkt <= 4) hipLaunchKernelGGL((attention_h16_kernel<DT, 4, 4>), grid, dim3(256), 0, stream, p);
    else if (nkt <= 7 && wide) hipLaunchKernelGGL((attention_h16_kernel<DT, 7, 8>), grid, dim3(512), 0, stream, p);
    else if (nkt <= 7) hipLaunchKernelGGL((attention_h16_kernel<DT, 7, 4>), grid, dim3(256), 0, stream, p);
    else if (wide) hipLaunchKernelGGL((attention_h16_kernel<DT, 8, 8>), grid, dim3(512), 0, stream, p);
    else hipLaunchKernelGGL((attention_h16_kernel<DT, 8, 4>), grid, dim3(256), 0, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}

int attention_h16_launch(int dt, const onhip_attention_desc_t &d, const void *q, const void *k, const void *v, void *out,
                         hipStream_t stream) {
    AttnH16Params p;
    p.q = reinterpret_cast<const unsigned short *>(q);
    p.k = reinterpret_cast<const unsigned short *>(k);
    p.v = reinterpret_cast<const unsigned short *>(v);
    p.o = reinterpret_cast<unsigned short *>(out);
    for (int i = 0; i < 3; ++i) {
        p.qs[i] = d.q_strides[i]; p.ks[i] = d.k_strides[i]; p.vs[i] = d.v_strides[i]; p.os[i] = d.out_strides[i];
    }
    p.heads = d.heads;
    p.tokens = d.tokens;
    p.scale = d.scale;
    return dt == DT_BF16 ? attention_h16_launch_dt<DT_BF16>(p, d.batch, stream) : attention_h16_launch_dt<DT_F16>(p, d.batch, stream);
}

}  // namespace onhip
