// fp32 implicit GEMM for launches with few tiles (gfx950): K cut over the wavefronts of a workgroup.
//
// A tile of 32 x 32, 64 x 32 or 16 x 16 belongs to one workgroup of four wavefronts (32 x 32: or eight); wavefront w takes the K steps w,
// w + NW, w + 2 NW ... of it, with both operands straight from memory in registers: no LDS, no barrier and no neighbour to wait
// for in the K loop.  The wavefronts' sums meet in LDS once, and every thread finishes one to eight outputs.
//
// Why: a batch-1 layer has 4 to 200 tiles of 64 x 64.  The kernels that stage tiles through LDS reach the other compute units by
// K slices in memory and a second launch that adds them up (3.9 us each on ResNet-50 at batch 1, 33 of its 91 launches), and run
// one wavefront per SIMD in lock step.  Here the slices are wavefronts: small tiles reach the compute units, four wavefronts per
// SIMD cover each other's loads.  What bounds it: the operands of a 32 x 32 tile are not shared with anyone, so a compute unit
// moves 64 bytes a clock from its L2 for 12 (16 x 16: 6) multiply-adds a byte, which is why larger problems stay with the others.
//
// Measured (one launch, against two launches in slices or one of 64 x 64 tiles): 64 x 3136 x 576 13.4 -> 7.6 us, 256 x 196 x 1024
// 11.4 -> 6.4, 1024 x 196 x 256 8.4 -> 5.0, 512 x 784 x 128 5.8 -> 5.2; 512 x 49 x 4608 15 against 13, so not there.  Eight
// wavefronts on 16 x 16 tiles, sixteen anywhere and a ring of two steps are not faster: the cache lines a compute unit asks for
// set the pace, not the latency.
//
// Arithmetic, by what the weights are:
//   F3   split into bf16 parts ahead of time: that of igemm_f3_kernel.hpp, the activations split in registers, a third of the
//        matrix time of fp32 instructions against 52 vector instructions a step.  Sums that are not finite are made again with
//        fp32 matrix instructions.
//   F32  fp32 as given: fp32 matrix instructions.
// A wavefront's sum is in the order of K, the wavefronts' sums are added in their order: the same bits on every run.
//
// Replaces, for the dense fp32 cases with few tiles (kw_choice in api.hip): device/x86/Conv/conv.c im2col (:168,:260) +
// opt_gemm.h SGEMM (:17) + bias sweep (:405) + do_act (:1216); device/x86/MatMul/mat_mul.c:10.
#include "igemm_f3_kernel.hpp"

namespace onhip {

enum { KW_F32 = 0, KW_F3 = 1 };

// one matrix instruction over the 8 (bf16) values a lane holds, tile edge 32 or 16
__device__ __forceinline__ void kw_mma(f32x16 &c, const uint4 &a, const uint4 &b) { mma_bf16(c, a, b); }
__device__ __forceinline__ void kw_mma(f32x4 &c, const uint4 &a, const uint4 &b) {
    c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// and over one fp32 value
__device__ __forceinline__ void kw_mma1(f32x16 &c, float a, float b) { c = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
__device__ __forceinline__ void kw_mma1(f32x4 &c, float a, float b) { c = __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <int MODE, int BL, int T, int TM, int NW>
__global__ __launch_bounds__(64 * NW) void igemm_kw_kernel(const IgemmProblem p) {
    static_assert(T == 32 || (T == 16 && TM == 1), "blocks of 32 x 32 or 16 x 16");
    constexpr int BM = T * TM, GROUPS = 64 / T;   // lanes of a row: each holds 8 consecutive K of a step
    constexpr int KS = 8 * GROUPS;                // K of a step
    constexpr int R = T * T / 64, VALS = TM * R * 64, NT = 64 * NW, PER = (VALS + NT - 1) / NT;
    constexpr int NA = MODE == KW_F3 ? 3 : 2;     // 16-byte loads of A per row block and step
    constexpr int RING = TM == 2 ? 2 : 3;         // steps in flight: a third one of 64 rows costs a wavefront per SIMD
    typedef std::conditional_t<T == 32, f32x16, f32x4> acc_t;
    __shared__ float s_sum[NW * VALS];            // [wavefront][row block][register][lane]
    __shared__ int s_again;

    warm_params<sizeof(IgemmProblem)>();
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lc = lane % T, lg = lane / T;
    const TilePlace tp = place_tile<BM, T>(p);
    const int m0 = tp.m0, n0 = tp.n0;
    const int steps = (p.K + KS - 1) / KS;        // of the whole tile

    const char *b_base = reinterpret_cast<const char *>(p.B) - (size_t) p.b_shift_bytes;
    const unsigned b_bytes = (unsigned) (p.b_slice_bytes + p.b_shift_bytes);
    const char *a_base = reinterpret_cast<const char *>(MODE == KW_F3 ? p.a_split : p.A);
    const unsigned a_bytes = (unsigned) (MODE == KW_F3 ? p.a_split_bytes : p.a_slice_bytes);

    // A: this lane's share of a step.  Split weights lie [32 rows][16 of K][part][row, half][8 bf16]: a 32-row block's share is the
    // lane's own 16 bytes, that of 16 rows covers two such groups of K.  fp32 weights: two 16-byte loads of the row.
    unsigned a_voff[TM];
#pragma unroll
    for (int t = 0; t < TM; ++t) {
        if constexpr (MODE == KW_F3) {
            const unsigned block = (unsigned) ((m0 + t * T) / 32) * (unsigned) ((p.K + 15) / 16) * 3072u;
            a_voff[t] = block + (T == 32 ? (unsigned) lane * 16u : (unsigned) (lg / 2) * 3072u + (unsigned) (lg % 2 * 32 + m0 % 32 + lc) * 16u);
        } else {
            const int m = m0 + t * T + lc;
            a_voff[t] = m < p.M ? (unsigned) (m * p.lda + 8 * lg) * 4u : OOB;
        }
    }
    // B: this lane's column, moved to its 8 of K
    ColState col = f3_col<BL>(p, n0 + lc);
    const unsigned hw4 = (unsigned) p.HW * 4u;
    if (col.pixoff != OOB) col.pixoff += (unsigned) lg * 8u * hw4;

    // what the finished outputs of this thread need, requested ahead of the operands
    int row[PER];
    unsigned at[PER];
    float bias[PER], res[PER];
    const rsrc_t rbias = make_rsrc(p.bias, p.bias_mode == BIAS_NONE ? 0u : (unsigned) ((p.bias_mode == BIAS_M ? p.M : p.N) * 4));
    const rsrc_t rres = make_rsrc(p.res, p.res ? RSRC_RANGE : 0u);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int v = tid + i * NT, ln = v % 64, r = v / 64 % R, t = v / 64 / R;
        row[i] = m0 + t * T + (T == 32 ? 8 * (r / 4) + 4 * (ln / 32) + r % 4 : 4 * (ln / 16) + r);
        const int n = n0 + ln % T;
        const bool on = v < VALS && row[i] < p.M && n < p.N;
        at[i] = on ? out_col_offset(p, n, 4) + (unsigned) row[i] * (unsigned) p.c_stride_m * 4u : OOB;
        bias[i] = buf_load_f32(rbias, on ? (unsigned) (p.bias_mode == BIAS_N ? n : row[i]) * 4u : OOB, 0);
        res[i] = buf_load_f32(rres, at[i], 0);
    }

    acc_t acc[TM];
#pragma unroll
    for (int t = 0; t < TM; ++t)
#pragma unroll
        for (int r = 0; r < R; ++r) acc[t][r] = 0.0f;

    struct Step { uint4 a[NA][TM]; float b[8]; };
    // where B starts in a step, taken into the descriptor so that the eight loads have fixed offsets (a scalar instruction less
    // each); a step past the end reads through empty descriptors (zeros, no traffic)
    auto b_from = [&](unsigned off, bool live) __attribute__((always_inline)) {
        return make_rsrc(b_base + off, (unsigned) max(live ? (int) (b_bytes - off) : 0, 0));
    };
    auto load = [&](Step &s, int step) __attribute__((always_inline)) {
        const bool live = step < steps;
        const rsrc_t ra = make_rsrc(a_base, live ? a_bytes : 0u);
        const unsigned a_soff = (unsigned) step * (MODE == KW_F3 ? KS / 16 * 3072u : KS * 4u);
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int z = 0; z < NA; ++z) s.a[z][t] = buf_load_b128(ra, a_voff[t] + (MODE == KW_F3 ? z * 1024u : z * 16u), a_soff);
        // a step lies inside one filter tap (kw_ok): its place in the image is scalar
        const F3Prep q = f3_prep<BL>(p, step * (KS / 4), 0);
        const unsigned voff = f3_voff<BL>(col, q.tap);
        const rsrc_t rb = b_from(q.soff, live);
#pragma unroll
        for (int e = 0; e < 8; ++e) s.b[e] = buf_load_f32(rb, voff, (unsigned) e * hw4);
    };
    auto multiply = [&](const Step &s) __attribute__((always_inline)) {
        if constexpr (MODE == KW_F3) {
            uint4 part[3];
            SplitUnit u, w;
            static_for<4>([&](auto q) __attribute__((always_inline)) {
                u.phase<decltype(q)::value>(s.b[0], s.b[1], s.b[2], s.b[3]);
                w.phase<decltype(q)::value>(s.b[4], s.b[5], s.b[6], s.b[7]);
            });
            part[0] = make_uint4(u.h0, u.h1, w.h0, w.h1);
            part[1] = make_uint4(u.m0, u.m1, w.m0, w.m1);
            part[2] = make_uint4(u.l0, u.l1, w.l0, w.l1);
            static_for<F3_PRODUCTS>([&](auto q) __attribute__((always_inline)) {
                constexpr int i = decltype(q)::value;
#pragma unroll
                for (int t = 0; t < TM; ++t) kw_mma(acc[t], s.a[f3_pa(i)][t], part[f3_pb(i)]);
            });
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
#pragma unroll
                for (int t = 0; t < TM; ++t) {
                    const uint4 &q = s.a[e / 4][t];
                    kw_mma1(acc[t], __uint_as_float(e % 4 == 0 ? q.x : e % 4 == 1 ? q.y : e % 4 == 2 ? q.z : q.w), s.b[e]);
                }
        }
    };
    Step ring[RING];
    static_for<RING - 1>([&](auto j) __attribute__((always_inline)) { load(ring[decltype(j)::value], wave + NW * decltype(j)::value); });
    for (int s = wave; s < steps; s += NW * RING)
        static_for<RING>([&](auto j) __attribute__((always_inline)) {
            constexpr int J = decltype(j)::value;
            load(ring[(J + RING - 1) % RING], s + NW * (J + RING - 1));
            __builtin_amdgcn_sched_barrier(0);   // the loads stay in front: left alone they sink to their first use
            if (J == 0 || s + NW * J < steps) multiply(ring[J]);
            __builtin_amdgcn_sched_barrier(0);
        });

    float sum[PER];
    auto reduce = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TM; ++t)
#pragma unroll
            for (int r = 0; r < R; ++r) s_sum[((wave * TM + t) * R + r) * 64 + lane] = acc[t][r];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int v = tid + i * NT;
            sum[i] = 0.0f;
            if (v < VALS) {
                sum[i] = s_sum[v];
#pragma unroll
                for (int w = 1; w < NW; ++w) sum[i] = __fadd_rn(sum[i], s_sum[w * VALS + v]);
            }
        }
    };
    if (MODE == KW_F3 && tid == 0) s_again = 0;   // ordered against its readers by the barriers of reduce
    reduce();
    if constexpr (MODE == KW_F3) {
        bool again = false;
#pragma unroll
        for (int i = 0; i < PER; ++i) again |= sum[i] * 0.0f != 0.0f;   // true for an infinity and a NaN
        if (again) s_again = 1;
        __syncthreads();
        if (s_again) {   // uniform.  The same steps with fp32 matrix instructions (see igemm_f3_kernel.hpp: unscale_fix_nonfinite)
            const rsrc_t ra = make_rsrc(a_base, a_bytes);
#pragma unroll
            for (int t = 0; t < TM; ++t)
#pragma unroll
                for (int r = 0; r < R; ++r) acc[t][r] = 0.0f;
#pragma unroll 1
            for (int s = wave; s < steps; s += NW) {
                uint4 a[3][TM];
#pragma unroll
                for (int t = 0; t < TM; ++t)
#pragma unroll
                    for (int z = 0; z < 3; ++z) a[z][t] = buf_load_b128(ra, a_voff[t], (unsigned) s * (KS / 16 * 3072u) + z * 1024u);
                const F3Prep q = f3_prep<BL>(p, s * (KS / 4), 0);
                const unsigned voff = f3_voff<BL>(col, q.tap);
                const rsrc_t rb = b_from(q.soff, true);
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    // beyond K the weights are zero and what B brings in need not be finite
                    const float bv = buf_load_f32(rb, s * KS + 8 * lg + e < p.K ? voff : OOB, (unsigned) e * hw4);
#pragma unroll
                    for (int t = 0; t < TM; ++t) {
                        auto up = [&](const uint4 &x) __attribute__((always_inline)) {
                            const unsigned w = e / 2 == 0 ? x.x : e / 2 == 1 ? x.y : e / 2 == 2 ? x.z : x.w;
                            return __uint_as_float(e % 2 ? w & 0xffff0000u : w << 16);
                        };
                        const float hi = up(a[0][t]), mid = up(a[1][t]), low = up(a[2][t]);
                        const float whole = __uint_as_float(__float_as_uint(mid) | __float_as_uint(low) >> 16);
                        kw_mma1(acc[t], hi - hi == 0.0f ? ((hi + mid) + low) * (1.0f / F3_SCALE) : whole, bv);
                    }
                }
            }
            float scaled[PER];
#pragma unroll
            for (int i = 0; i < PER; ++i) scaled[i] = sum[i];
            reduce();   // every thread has read its first sums before the barrier above
#pragma unroll
            for (int i = 0; i < PER; ++i) sum[i] = scaled[i] * 0.0f != 0.0f ? sum[i] : scaled[i] * F3_UNSCALE;
        } else {
#pragma unroll
            for (int i = 0; i < PER; ++i) sum[i] *= F3_UNSCALE;
        }
    }
    const rsrc_t rc = make_rsrc(p.C, RSRC_RANGE);
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        float v = p.bias_mode == BIAS_NONE ? sum[i] : __fadd_rn(sum[i], bias[i]);
        if (at[i] != OOB) v = apply_act(v, p.ep);   // the table's loads for outputs that exist
        if (p.res) v = add_res(v, res[i], p.res_relu, at[i] >> 2, p.res_body);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rc, at[i], 0, 0);
    }
}

template <int MODE, int BL, int T, int TM, int NW>
static int kw_launch_one(const IgemmLaunch &cfg, const IgemmProblem &p_in, hipStream_t stream) {
    IgemmProblem p = p_in;
    dim3 grid;
    const int rc = tile_grid<T * TM, T>(cfg, p, &grid);
    if (rc) return rc;
    hipLaunchKernelGGL((igemm_kw_kernel<MODE, BL, T, TM, NW>), grid, dim3(64 * NW), 0, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}
template <int MODE, int BL>
static int kw_launch_tile(const IgemmLaunch &cfg, const IgemmProblem &p, int waves, hipStream_t stream) {
    switch (cfg.bm * 100 + waves) {
        case 1604: return kw_launch_one<MODE, BL, 16, 1, 4>(cfg, p, stream);
        case 3204: return kw_launch_one<MODE, BL, 32, 1, 4>(cfg, p, stream);
        case 3208: return kw_launch_one<MODE, BL, 32, 1, 8>(cfg, p, stream);
        case 6404: return kw_launch_one<MODE, BL, 32, 2, 4>(cfg, p, stream);
        default: return set_error(ONHIP_ERR_ARG, "igemm kw: no kernel for %d rows and %d wavefronts", cfg.bm, waves);
    }
}

bool kw_ok(const IgemmLaunch &cfg, const IgemmProblem &p, int bm, bool split) {
    if (cfg.dtype != DT_F32 || cfg.batch != 1 || p.M < 1 || p.N < 1 || p.K < 1) return false;
    if (p.a_slice_bytes >= (1LL << 31) || p.b_slice_bytes + 2 * p.b_shift_bytes >= (1LL << 31) || p.c_slice_bytes >= (1LL << 31)) return false;
    const int ks = bm == 16 ? 32 : 16;
    if ((long long) (p.K + ks) * p.HW >= (1LL << 29)) return false;   // a step's place in B as a signed number of bytes
    if (cfg.bl == BL_TAPC) return p.use_tapmask && p.units_per_tap % (ks / 4) == 0;   // a step inside one tap
    // fp32 weights end with the row: whole steps.  Split ones are padded with zeros to 16
    return cfg.bl == BL_PLAIN && (split && bm != 16 ? true : p.K % ks == 0);
}

int kw_launch(const IgemmLaunch &cfg, const IgemmProblem &p_in, int waves, hipStream_t stream) {
    const bool split = p_in.a_split != nullptr;
    if (!kw_ok(cfg, p_in, cfg.bm, split) || cfg.bn != (cfg.bm == 16 ? 16 : 32) || cfg.split != 1)
        return set_error(ONHIP_ERR_ARG, "igemm kw: not a problem of this kernel");
    IgemmProblem p = p_in;
    // an XCD keeps a band of the larger operand and sweeps the smaller one
    p.n_fast = (long long) p.M * p.K * (split ? 6 : 4) > p.b_slice_bytes;
    if (split) return cfg.bl == BL_PLAIN ? kw_launch_tile<KW_F3, BL_PLAIN>(cfg, p, waves, stream) : kw_launch_tile<KW_F3, BL_TAPC>(cfg, p, waves, stream);
    return cfg.bl == BL_PLAIN ? kw_launch_tile<KW_F32, BL_PLAIN>(cfg, p, waves, stream) : kw_launch_tile<KW_F32, BL_TAPC>(cfg, p, waves, stream);
}

}  // namespace onhip
