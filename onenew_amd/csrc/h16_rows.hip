// 16-bit products with a short K: C[N, M] = act(B[N, K] * A[M, K]^T + bias), rows of B and C in memory as they are multiplied (a linear layer, a
// 1x1 convolution on NHWC), K of 64, 128, 192 or 256.  With so few steps igemm_dma_kernel's workgroups are a chain of trips to memory, the operands', then
// the activation table's, and the store behind them, with two or three of them a compute unit to cover it.  Here a workgroup of eight
// wavefronts keeps 256 rows of B in registers (a wavefront 32 rows, all of K) and the activation table in LDS, and walks over panels of 64 rows of
// A, the next one on its way while this one is multiplied and stored: the trips at the start are made once, side by side.
// What bounds it: those trips (4000 cycles), then the store's vector work: a panel of 192 deep is 770 cycles of matrix instructions a wavefront and, with a
// table, 1500 of vector instructions and LDS, two wavefronts a SIMD in step.  12608 rows, 192 -> 576 11.2 -> 9.2 us, 192 -> 768 with GELU 17.7 -> 13.4,
// 192 -> 192 with an addend 7.1 -> 6.7; 25088 rows, 128 -> 512 with an addend 16.3 -> 13.8; 100000 rows, 64 -> 256 with a table 29.8 -> 23.3.
//
// Same instructions over K in the same order as igemm_dma_kernel, and the store's operations are its: same bits.
#include "igemm_kernel.hpp"

namespace onhip {

struct RowsH16Params {
    const void *A, *B;
    void *C;
    const void *res;
    const float *bias, *lut;
    int M, N, lda, ldb, pitch;     // bytes between rows of A and of B, elements between rows of C
    unsigned a_bytes, b_bytes;
    int panels, subs;              // of 64 rows of A; runs of them
    int relu;                      // behind the residual operand
};

template <int DT, int KS, bool TABLE>
__global__ __launch_bounds__(512, 2) void rows_h16_kernel(const RowsH16Params p) {
    constexpr int NW = 8, NT = 64 * NW, PM = 64, U = 2 * KS;   // U: 16-byte units of a row
    constexpr int A_PER_T = PM * U / NT;
    static_assert(PM * U % NT == 0);
    constexpr int PITCH = 2 * PM + 16;                          // of a staged row of C, in bytes
    __shared__ uint4 s_a[2][PM * U];
    __shared__ __attribute__((aligned(16))) unsigned char s_out[NW][32 * PITCH];
    __shared__ __attribute__((aligned(16))) float s_bias[2][PM];
    __shared__ __attribute__((aligned(16))) unsigned short s_table[8 + (TABLE ? 8192 : 0)];   // entry -1 in front of the first

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    // an XCD gets a contiguous run of workgroups: those of the same rows of B next to each other
    int rows, sub;
    {
        const int nb = (int) gridDim.x, bid = (int) blockIdx.x, per = nb >> 3, rmd = nb & 7, xcd = bid & 7, idx = bid >> 3;
        const int lid = xcd * per + (xcd < rmd ? xcd : rmd) + idx;
        rows = lid / p.subs;
        sub = lid - rows * p.subs;
    }
    const int first = sub * p.panels / p.subs, last = (sub + 1) * p.panels / p.subs;
    const int n_wave = (rows * NW + wave) * 32;

    // where unit u of row r of a panel lies: units exchanged by the row, so that 16 rows' reads of one unit cover the banks
    auto slot = [](int r, int u) { return r * U + (u ^ (U % 16 ? r >> 1 & 7 : r & 15)); };
    const rsrc_t ra = make_rsrc(p.A, p.a_bytes), rb = make_rsrc(p.B, p.b_bytes), rbias = make_rsrc(p.bias, p.bias ? (unsigned) (p.M * 4) : 0u);
    uint4 aq[A_PER_T];
    unsigned a_from[A_PER_T], a_to[A_PER_T];
#pragma unroll
    for (int t = 0; t < A_PER_T; ++t) {
        const int f = tid + t * NT;
        a_from[t] = (unsigned) (f / U * p.lda + f % U * 16);
        a_to[t] = (unsigned) slot(f / U, f % U);
    }
    float bias_q = 0.0f;
    auto load_panel = [&](int panel) __attribute__((always_inline)) {   // rows beyond M read as zero
#pragma unroll
        for (int t = 0; t < A_PER_T; ++t) aq[t] = buf_load_b128(ra, a_from[t], (unsigned) (panel * PM * p.lda));
        if (wave == 0) bias_q = buf_load_f32(rbias, (unsigned) lane * 4u, (unsigned) panel * PM * 4u);   // uniform
    };
    auto stage_panel = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < A_PER_T; ++t) s_a[buf][a_to[t]] = aq[t];
        if (wave == 0) s_bias[buf][lane] = bias_q;
    };

    load_panel(first);
    constexpr int PER = TABLE ? 8192 / 4 / NT : 1;
    float4 t[PER];
    if constexpr (TABLE)
#pragma unroll
        for (int i = 0; i < PER; ++i) t[i] = reinterpret_cast<const float4 *>(p.lut)[tid + i * NT];
    __builtin_amdgcn_sched_barrier(0);
    // This wavefront's rows of B, eight lanes to the 128 bytes of a row, and from there through the wavefront's part of LDS to the lanes that multiply
    // with them.  (Loaded in that order, 32 rows an instruction, they were 64 cycles of the compute unit's address path each, two microseconds of
    // a launch.)
    uint4 b[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) {
        const int n = n_wave + s % 4 * 8 + lane / 8;
        b[s] = buf_load_b128(rb, n < p.N ? (unsigned) n * (unsigned) p.ldb + (unsigned) (lane % 8) * 16u : OOB, s / 4 * 128u);
    }
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (TABLE)   // rounded to the output type, as what is stored of an entry
#pragma unroll
        for (int i = 0; i < PER; ++i)
            reinterpret_cast<uint2 *>(s_table + 8)[tid + i * NT] = make_uint2(pack_h16<DT>(t[i].x, t[i].y), pack_h16<DT>(t[i].z, t[i].w));
    {
        uint4 *mine = reinterpret_cast<uint4 *>(s_out[wave]);
        auto at = [](int r, int u) { return r * 8 + (u ^ (r >> 1 & 7)); };
#pragma unroll
        for (int c = 0; c < KS / 4; ++c) {
#pragma unroll
            for (int i = 0; i < 4; ++i) mine[at(i * 8 + lane / 8, lane % 8)] = b[4 * c + i];
#pragma unroll
            for (int i = 0; i < 4; ++i) b[4 * c + i] = mine[at(li, 2 * i + lh)];
        }
    }
    if (TABLE && tid == 0) s_table[7] = 0;
    stage_panel(0);
    __syncthreads();

    const rsrc_t rc = make_rsrc(p.C, RSRC_RANGE), rr = make_rsrc(p.res, p.res ? RSRC_RANGE : 0u);
    unsigned char *const out = s_out[wave];
    // this lane's 16-byte pieces of the wavefront's 32 rows of a panel of C
    unsigned at[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int n = n_wave + (i * 64 + lane) / 8;
        at[i] = n < p.N ? (unsigned) (n * p.pitch + lane % 8 * 8) * 2u : OOB;
    }
#pragma unroll 1
    for (int panel = first; panel < last; ++panel) {
        const int buf = (panel - first) & 1, m0 = panel * PM;
        if (panel + 1 < last) load_panel(panel + 1);   // uniform
        u32x4 addend[4];
        if (p.res) {   // uniform
#pragma unroll
            for (int i = 0; i < 4; ++i) addend[i] = __builtin_amdgcn_raw_buffer_load_b128(rr, m0 + lane % 8 * 8 < p.pitch ? at[i] : OOB, (unsigned) m0 * 2u, 0);
        }
        f32x16 acc[2];
#pragma unroll
        for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][r] = 0.0f;
        uint4 av[3][2];   // operands two steps ahead
        auto read_a = [&](int s) __attribute__((always_inline)) {
#pragma unroll
            for (int a = 0; a < 2; ++a) av[s % 3][a] = s_a[buf][slot(32 * a + li, 2 * s + lh)];
        };
        read_a(0);
        read_a(1);
#pragma unroll
        for (int s = 0; s < KS; ++s) {
            if (s + 2 < KS) read_a(s + 2);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                if constexpr (DT == DT_BF16) acc[a] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, av[s % 3][a]), __builtin_bit_cast(bf16x8, b[s]), acc[a], 0, 0, 0);
                else acc[a] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, av[s % 3][a]), __builtin_bit_cast(f16x8, b[s]), acc[a], 0, 0, 0);
            }
        }
        if (panel + 1 < last) stage_panel(buf ^ 1);
        auto store = [&](auto at_edge, auto with_res) __attribute__((always_inline)) {
            constexpr bool EDGE = decltype(at_edge)::value, RES = decltype(with_res)::value;
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                // sixteen columns of C: their table entries are requested together
                float y[16];
                unsigned w[8];
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 bias = *reinterpret_cast<const float4 *>(&s_bias[buf][32 * a + 8 * q + 4 * lh]);
                    const float bv[4] = {bias.x, bias.y, bias.z, bias.w};
#pragma unroll
                    for (int j = 0; j < 4; ++j) y[4 * q + j] = __fadd_rn(acc[a][4 * q + j], bv[j]);   // zero without a bias
                }
                if constexpr (TABLE) table_h16<DT>(y, w, (lds_u16_t) (s_table + 8));
                else
#pragma unroll
                    for (int i = 0; i < 8; ++i) w[i] = pack_h16<DT>(y[2 * i], y[2 * i + 1]);
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int ml = 32 * a + 8 * q + 4 * lh;   // first of the lane's four columns of C
                    if constexpr (EDGE)
#pragma unroll
                        for (int i = 2 * q; i < 2 * q + 2; ++i) {
                            const int m = m0 + ml + i % 2 * 2;
                            w[i] = (m < p.M ? w[i] & 0xffffu : 0u) | (m + 1 < p.M ? w[i] & 0xffff0000u : 0u);
                        }
                    *reinterpret_cast<uint2 *>(out + li * PITCH + ml * 2) = make_uint2(w[2 * q], w[2 * q + 1]);
                }
            }
            uint4 v[4];   // the wavefront's own: in order behind its writes
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = *reinterpret_cast<const uint4 *>(out + (i * 64 + lane) / 8 * PITCH + lane % 8 * 16);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                if constexpr (RES) {
                    unsigned *w = reinterpret_cast<unsigned *>(&v[i]);
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        float lo = __fadd_rn(unpack_h16<DT>(w[j], 0), unpack_h16<DT>(addend[i][j], 0));
                        float hi = __fadd_rn(unpack_h16<DT>(w[j], 1), unpack_h16<DT>(addend[i][j], 1));
                        if (p.relu) { lo = lo > 0.0f ? lo : 0.0f; hi = hi > 0.0f ? hi : 0.0f; }
                        w[j] = pack_h16<DT>(lo, hi);
                    }
                }
                // (the panel's place in the vector offset: with a scalar register there the compiler leaves no wait before the data registers' next use)
                __builtin_amdgcn_raw_buffer_store_b128(u32x4{v[i].x, v[i].y, v[i].z, v[i].w}, rc, m0 + lane % 8 * 8 < p.pitch ? at[i] + (unsigned) m0 * 2u : OOB, 0, 0);
            }
        };
        // the columns beyond M in the last panel alone; the addend asked once
        if (m0 + PM > p.M) {
            if (p.res) store(std::true_type{}, std::true_type{});
            else store(std::true_type{}, std::false_type{});
        } else {
            if (p.res) store(std::false_type{}, std::true_type{});
            else store(std::false_type{}, std::false_type{});
        }
        __syncthreads();   // the next panel is staged, and everybody has read this one
    }
}

template <int DT, int KS>
static int rows_h16_launch_one(const RowsH16Params &p, bool table, hipStream_t stream) {
    const dim3 grid((unsigned) ((p.N + 255) / 256 * p.subs));
    if (table) hipLaunchKernelGGL((rows_h16_kernel<DT, KS, true>), grid, dim3(512), 0, stream, p);
    else hipLaunchKernelGGL((rows_h16_kernel<DT, KS, false>), grid, dim3(512), 0, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}
template <int DT>
static int rows_h16_launch_dt(const RowsH16Params &p, int ks, bool table, hipStream_t stream) {
    switch (ks) {
        case 4: return rows_h16_launch_one<DT, 4>(p, table, stream);
        case 8: return rows_h16_launch_one<DT, 8>(p, table, stream);
        case 12: return rows_h16_launch_one<DT, 12>(p, table, stream);
        default: return rows_h16_launch_one<DT, 16>(p, table, stream);
    }
}

// runs of panels that the 64-row panels of A (the channels that pad a row of C as well) are cut into: a workgroup a compute unit
int rows_h16_subs(const IgemmParams &p) {
    const int blocks = (p.N + 255) / 256, panels = ((int) p.c_stride_n + 63) / 64;
    return blocks >= 256 ? 1 : 256 / blocks < panels ? 256 / blocks : panels;
}

// Which problems there is a form for (which of them it is faster for: rows_h16_faster).  Not with a Relu or a Clip alone, the narrow layers in front of a
// filter, where neither is ahead (100352 rows, 256 -> 64 15.2 and 15.6).
bool rows_h16_ok(const IgemmLaunch &cfg, const IgemmParams &p) {
    if ((cfg.dtype != DT_BF16 && cfg.dtype != DT_F16) || cfg.bl != BL_KVEC || cfg.batch != 1 || !p.out_h16 || p.out_mode != OUT_PLAIN || p.c_stride_m != 1) return false;
    // rows of B as they lie: one tap, no stride, no padding
    if (p.khkw != 1 || p.tap_spans_pixels || p.sh != 1 || p.sw != 1 || p.pt || p.pl || p.OHW != p.HW || p.pix_stride != p.k_units * 16 || p.lda != p.k_units * 16) return false;
    if (p.ep.act != NOT_ACT && p.ep.act != SILU && p.ep.act != ONHIP_ACT_GELU_LUT) return false;
    return p.k_units == 8 || p.k_units == 16 || p.k_units == 24 || p.k_units == 32;
}

int rows_h16_launch(const IgemmLaunch &cfg, const IgemmParams &q, hipStream_t stream) {
    RowsH16Params p;
    p.A = q.A; p.B = q.B; p.C = q.C; p.res = q.res16; p.bias = q.bias_mode == BIAS_M ? q.bias : nullptr;
    const bool table = q.ep.act == SILU || q.ep.act == ONHIP_ACT_GELU_LUT;
    p.lut = table ? q.ep.lut : nullptr;
    p.M = q.M; p.N = q.N; p.lda = q.lda; p.ldb = q.pix_stride; p.pitch = (int) q.c_stride_n;
    p.a_bytes = (unsigned) q.a_slice_bytes; p.b_bytes = (unsigned) q.b_slice_bytes;
    p.relu = q.res_relu;
    p.panels = (p.pitch + 63) / 64;
    p.subs = rows_h16_subs(q);
    return cfg.dtype == DT_BF16 ? rows_h16_launch_dt<DT_BF16>(p, q.k_units / 2, table, stream) : rows_h16_launch_dt<DT_F16>(p, q.k_units / 2, table, stream);
}

}  // namespace onhip
