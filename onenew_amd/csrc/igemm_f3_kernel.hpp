// fp32 implicit GEMM on the 16-bit matrix cores (gfx950): C[M, N] = A[M, K] * B[K, N], operands and result fp32.
//
// Arithmetic.  Every fp32 operand is written as the sum of three bf16 numbers, x = h + m + l: h = bf16(x), m = bf16(x - h),
// l = x - h - m, each rounded to nearest.  The two differences are exact, and so is the sum: 24 significant bits are three
// times eight (|m| <= 2^-8 |h|, |l| <= 2^-8 |m|).  Of the nine
// partial products six are formed, each exact in the matrix core and added to the fp32 accumulator: l h, m m, m h, h l, h m,
// h h.  The three left out, m l, l m and l l, are at most 2^-23 and typically 2^-26 of |a b|, below the rounding that a chain
// of fp32 multiply-adds makes at every step.  Measured against 64-bit sums over K = 48 ... 4608,
// root mean square of the error as a share of sum |a b|: 0.73 ... 0.88 of v_mfma_f32_32x32x2_f32's on normal operands, 0.63 ... 0.82 on
// all-positive ones, 0.77 ... 0.82 on operands spread over 2^+-4; 1.10 ... 1.19 where they spread over 2^+-24 and one term decides a sum.
// The nine products give the same errors as the six.
// The parts are those of x 2^24 (F3_SCALE): every fp32 number, subnormals included, is a multiple of 2^-149, so the parts are
// multiples of 2^-125 and none falls below bf16's smallest normal number (unscaled, an operand below 2^-110 lost low bits: a relative
// 2^-14 of it at 2^-120, all of it at 2^-134).  The sum is of a 2^24 times b 2^24 and loses 2^48 again when the K loop is over.
// What differs from an fp32 multiply: an infinity, a NaN and an operand of 2^104 or more have no finite parts, and sums of 2^80
// or more may overflow on the way; either leaves a sum that is not finite.  A wavefront that holds one when its K loop is over
// computes its tile again with fp32 matrix instructions (unscale_fix_nonfinite), so all of these come out as they do in fp32 arithmetic.
//
// Why: v_mfma_f32_32x32x16_bf16 does the multiply-adds of eight v_mfma_f32_32x32x2_f32 in a sixteenth of their time.  On
// random operands the card holds its power limit by its clock (1.2 to 1.7 GHz in these loops), so what counts is energy: six
// products reach 200-210 TFLOP/s of fp32 multiply-adds on 1024 x 32768 x 1024 and on a 3x3 convolution over 256 channels,
// where fp32 matrix instructions reach 146-155 on their own and 116 in igemm_kernel.
//
// Work decomposition: as igemm_kernel.hpp, whose column state, scalar load descriptions, store and split-K pieces this
// kernel uses; K in tiles of 4 units of 4 floats = one 16-deep MFMA step.  What differs:
//   * A, the weights, is split ahead of time (split_weights_launch) into the order the matrix instructions read it, and goes
//     from memory straight into operand registers, one contiguous KiB per load: no LDS, no vector instruction.  The
//     wavefronts of a tile lie along M (the 64 x 64, 192 x 64 and 128 x 128 tiles apart), so no two of them load the same rows;
//   * B is split on its way into LDS, [part][k / 8][column][8 bf16], a unit per thread and K tile, in four phases of four to
//     ten vector instructions each behind an MFMA of its own: 26 vector instructions per 12 to 24 MFMAs and wavefront.
// Per K tile of the 128 x 64 tile a wavefront issues 12 MFMAs, 3 A loads, 4 B loads, 3 LDS stores and 6 LDS reads.
//
// Replaces, for the dense fp32 cases with enough work (f3_choice in api.hip): device/x86/Conv/conv.c im2col (:168,:260) +
// opt_gemm.h SGEMM (:17) + bias sweep (:405) + do_act (:1216); device/x86/MatMul/mat_mul.c:10.
#pragma once
#include "igemm_kernel.hpp"
#include "row_norm.hpp"

namespace onhip {

// f(integral_constant<int, 0>), ..., f(integral_constant<int, N - 1>): indices the front end knows, so that every register
// array of the kernel is taken apart before anything else happens to it
template <int N, class F> __device__ __forceinline__ void static_for(F &&f) {
    [&]<int... I>(std::integer_sequence<int, I...>) __attribute__((always_inline)) { (f(std::integral_constant<int, I>{}), ...); }(std::make_integer_sequence<int, N>{});
}

constexpr float F3_SCALE = 0x1p24f, F3_UNSCALE = 0x1p-48f;   // of each operand, and of a sum of their products

// two floats, each rounded to bf16, packed
__device__ __forceinline__ unsigned cvt_pk_bf16(float a, float b) {
    unsigned d;   // the conversion of a pair; from C the compiler converts some of the values twice
    asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(d) : "v"(a), "v"(b));
    return d;
}
// A unit of four floats on its way to three parts, in four phases of four to ten vector instructions, each behind an MFMA while it
// runs.
struct SplitUnit {
    float r0, r1, r2, r3, u0, u1, u2, u3;   // what is left to split; the part taken last
    unsigned h0, h1, m0, m1, l0, l1;   // the parts, packed in pairs
    __device__ __forceinline__ void unpack(unsigned a, unsigned b) {
        u0 = __uint_as_float(a << 16); u1 = __uint_as_float(a & 0xffff0000u);
        u2 = __uint_as_float(b << 16); u3 = __uint_as_float(b & 0xffff0000u);
    }
    template <int Q, bool SCALED = true> __device__ __forceinline__ void phase(float x0, float x1, float x2, float x3) {
        if constexpr (Q == 0) {
            constexpr float scale = SCALED ? F3_SCALE : 1.0f;
            r0 = x0 * scale; r1 = x1 * scale; r2 = x2 * scale; r3 = x3 * scale;
            h0 = cvt_pk_bf16(r0, r1); h1 = cvt_pk_bf16(r2, r3);
            unpack(h0, h1);
        } else if constexpr (Q == 1) {
            r0 -= u0; r1 -= u1; r2 -= u2; r3 -= u3;
            m0 = cvt_pk_bf16(r0, r1); m1 = cvt_pk_bf16(r2, r3);
        } else if constexpr (Q == 2) {
            unpack(m0, m1);
        } else {
            l0 = cvt_pk_bf16(r0 - u0, r1 - u1); l1 = cvt_pk_bf16(r2 - u2, r3 - u3);
        }
    }
};
__device__ __forceinline__ void mma_bf16(f32x16 &c, const uint4 &a, const uint4 &b) {
    c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}
// the six partial products, (part of a, part of b) with 0 = h, 1 = m, 2 = l, smallest first
constexpr int F3_PRODUCTS = 6;
__device__ constexpr int f3_pa(int i) { constexpr int t[F3_PRODUCTS] = {2, 1, 1, 0, 0, 0}; return t[i]; }
__device__ constexpr int f3_pb(int i) { constexpr int t[F3_PRODUCTS] = {0, 1, 0, 2, 1, 0}; return t[i]; }

// column n's share of the B addresses
template <int BL>
__device__ __forceinline__ ColState f3_col(const IgemmProblem &p, int n) {
    if constexpr (BL == BL_ROWS) return {n < p.N ? (unsigned) (n * p.ldb) * 4u : OOB, 0, 0, 0u, 0u};
    else {
        ColState c = make_col<BL>(p, n);
        if constexpr (BL == BL_GATHER)
            if (!p.use_tapmask) c.mask_lo = c.mask_hi = ~0u;   // every window lies inside the image (f3_ok)
        return c;
    }
}

// prep_b and b_voff for the K loop: filters of at most 64 taps, or windows inside the image (f3_ok), and no test of the reduction index, so nothing that a
// branch could come of (those stood between the MFMAs of every K tile).  Beyond K the tap's bit is clear, or another tap's:
// what is read there meets zero weights.
struct F3Prep { unsigned soff, tap; };
template <int BL>
__device__ __forceinline__ F3Prep f3_prep(const IgemmProblem &p, int u, int e) {
    if constexpr (BL == BL_PLAIN) {
        return {(unsigned) (u * 4 + e) * (unsigned) p.HW * 4u, 0u};
    } else if constexpr (BL == BL_GATHER) {
        const unsigned k = (unsigned) (u * 4 + e), ch = fast_div(k, p.magic_khkw, p.pass_khkw), tap = k - ch * (unsigned) p.khkw;
        const unsigned i = fast_div(tap, p.magic_kw, p.pass_kw), j = tap - i * (unsigned) p.kw;
        return {(ch * (unsigned) p.HW + i * (unsigned) p.W + j) * 4u, tap};
    } else {
        const unsigned tap = fast_div((unsigned) u, p.magic_upt, p.pass_upt), cb = (unsigned) u - tap * (unsigned) p.units_per_tap;
        const unsigned i = fast_div(tap, p.magic_kw, p.pass_kw), j = tap - i * (unsigned) p.kw;
        return {(cb * 4u * (unsigned) p.HW + i * (unsigned) p.W + j) * 4u, tap};
    }
}
template <int BL>
__device__ __forceinline__ unsigned f3_voff(const ColState &c, unsigned tap) {
    if constexpr (BL == BL_PLAIN) return c.pixoff;
    const unsigned long long taps = (unsigned long long) c.mask_hi << 32 | c.mask_lo;
    const unsigned keep = 0u - ((unsigned) (taps >> (tap & 63u)) & 1u);
    return (c.pixoff & keep) | (OOB & ~keep);
}

// Byte offset of element (k, column) of B for unscale_fix_nonfinite, where k differs between lanes; OOB beyond the column's taps.
template <int BL>
__device__ __forceinline__ unsigned f3_element(const IgemmProblem &p, const ColState &c, unsigned k) {
    if constexpr (BL == BL_ROWS) return c.pixoff == OOB ? OOB : c.pixoff + k * 4u;
    if constexpr (BL == BL_PLAIN) return c.pixoff == OOB ? OOB : c.pixoff + k * (unsigned) p.HW * 4u;
    const F3Prep q = BL == BL_GATHER ? f3_prep<BL_GATHER>(p, (int) (k / 4), (int) (k % 4)) : f3_prep<BL_TAPC>(p, (int) (k / 4), 0);
    const unsigned at = f3_voff<BL>(c, q.tap);
    return at == OOB ? OOB : at + q.soff + (BL == BL_TAPC ? (k % 4) * (unsigned) p.HW * 4u : 0u);
}

// Element j of eight split values: its parts add up to the scaled value exactly, or are a marker and the value's two halves
// (split_weights_kernel).
__device__ __forceinline__ float f3_whole(const uint4 (&part)[3], int j) {
    auto up = [&](const uint4 &q) __attribute__((always_inline)) {
        const unsigned w = j / 2 == 0 ? q.x : j / 2 == 1 ? q.y : j / 2 == 2 ? q.z : q.w;
        return __uint_as_float(j % 2 ? w & 0xffff0000u : w << 16);
    };
    const float hi = up(part[0]), mid = up(part[1]), low = up(part[2]);
    const float whole = __uint_as_float(__float_as_uint(mid) | __float_as_uint(low) >> 16);
    return hi - hi == 0.0f ? ((hi + mid) + low) * (1.0f / F3_SCALE) : whole;
}

// Sums with the operands' scale taken out, and those that are not finite computed again in fp32 (see the head of the file): a wavefront that holds one multiplies its whole tile
// again with v_mfma_f32_32x32x2_f32, operands straight from memory, and takes the elements that were not finite from there.
// Sixteen of K a step, 8 (lane / 32) + j in MFMA j.  Units u_begin .. of the reduction up to klim elements.
// A product of 4099 x 1031 x 2053 takes 0.127 ms, with a NaN in one row of the left operand 0.23, all of it NaN 0.54; a 3x3 convolution
// 256 -> 256 over 32 x 14 x 14 0.075, and 0.22 with a NaN in one plane of each image.  (One element a lane and multiply-add: 4.6 and
// 15 ms, 2.7 ms.)
template <int BL, int TM, int TN>
__device__ __forceinline__ void unscale_fix_nonfinite(const IgemmProblem &p, f32x16 (&acc)[TM][TN], rsrc_t ra, rsrc_t rb, int m_wave, int n_wave, int lane,
                                              int u_begin, int klim) {
    float probe = 0.0f;   // stays zero while every sum is finite: 0 * inf and 0 * NaN are NaN
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(acc[a][b][r], 0.0f, probe);
    if (__builtin_amdgcn_ballot_w64(probe != probe) == 0ull) {
#pragma unroll
        for (int a = 0; a < TM; ++a)
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) acc[a][b][r] *= F3_UNSCALE;
        return;
    }
    const int li = lane & 31, lh = lane >> 5;
    ColState col[TN];
#pragma unroll
    for (int b = 0; b < TN; ++b) col[b] = f3_col<BL>(p, n_wave + b * 32 + li);
    // a row block at a time: no more registers than the K loop has given up
#pragma unroll
    for (int a = 0; a < TM; ++a) {
        f32x16 s[TN];
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[b][r] = 0.0f;
        const unsigned a_row = (unsigned) (m_wave / 32 + a) * (unsigned) ((p.K + 15) / 16) * 3072u;
#pragma unroll 1
        for (int k0 = u_begin * 4; k0 < klim; k0 += 16) {
            uint4 part[3];
#pragma unroll
            for (int z = 0; z < 3; ++z) part[z] = buf_load_b128(ra, (unsigned) lane * 16u, a_row + (unsigned) (k0 / 16) * 3072u + z * 1024u);
            float bv[TN][8];
#pragma unroll
            for (int b = 0; b < TN; ++b)
#pragma unroll
                for (int j = 0; j < 8; ++j) {
                    const int k = k0 + 8 * lh + j;
                    bv[b][j] = buf_load_f32(rb, k < klim ? f3_element<BL>(p, col[b], (unsigned) k) : OOB, 0);
                }
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const float av = f3_whole(part, j);
#pragma unroll
                for (int b = 0; b < TN; ++b) s[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv[b][j], s[b], 0, 0, 0);
            }
        }
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = acc[a][b][r] * 0.0f != 0.0f ? s[b][r] : acc[a][b][r] * F3_UNSCALE;
    }
}

// The store for B given as rows (a product's left operand): C is row-major with the tile's columns as its rows, so the four
// consecutive rows of the tile that a lane holds in registers 4 q .. 4 q + 3 are 16 contiguous bytes of C.  A block of 32 x 32 at a time goes
// through 4 KB of LDS of the wavefront's own to eight lanes a row of 128 bytes, as which the residual operand arrives too: a row a lane was
// 64 cycles of the compute unit's address path for each of the four stores and loads, 16 now.  Residual and bias as in write_tile.
// norm: LDS for the rows of C as well, M + 1 floats apart, at row n_wave (the variant that normalises the rows), or nullptr.
template <int EPI, int TM, int TN, bool RES, bool NORM = false>
__device__ __forceinline__ void write_tile_rows(const IgemmProblem &p, f32x16 (&acc)[TM][TN], int m_wave, int n_wave, int li, int lh,
                                                const float *sbias, lds_f32_t table, uint4 *turn, float *norm = nullptr) {
    const rsrc_t rc = make_rsrc(p.C, (unsigned) p.c_slice_bytes), rr = make_rsrc(RES ? p.res : nullptr, RES ? (unsigned) p.c_slice_bytes : 0u);
    const int lane = lh * 32 + li, row8 = lane / 8, u8 = lane % 8;
    auto unit = [](int row, int u) { return row * 8 + (u ^ (row >> 1 & 7)); };
    // this lane's piece i of block (a, b): row 8 i + lane / 8, columns 4 (lane % 8) .. + 3
    auto place = [&](int a, int b, int i) __attribute__((always_inline)) {
        const int n = n_wave + b * 32 + 8 * i + row8;
        unsigned base = (unsigned) (n * (int) p.c_stride_n + m_wave + a * 32 + 4 * u8) * 4u;
        if (p.c_part) {   // several products: a block of 32 rows lies inside one of them
            const int row = m_wave + a * 32, part = (row >= p.c_part) + (row >= 2 * p.c_part) + (row >= 3 * p.c_part);
            base += (unsigned) part * (p.c_part_step - (unsigned) p.c_part * 4u);
        }
        return n < p.N ? base : OOB;
    };
    u32x4 rv[2][4];   // a block ahead
    auto load_res = [&](int blk) __attribute__((always_inline)) {
        if constexpr (RES)
#pragma unroll
            for (int i = 0; i < 4; ++i) rv[blk & 1][i] = __builtin_amdgcn_raw_buffer_load_b128(rr, place(blk % TM, blk / TM, i), 0, 0);
    };
    load_res(0);
#pragma unroll
    for (int b = 0; b < TN; ++b) {
#pragma unroll
        for (int a = 0; a < TM; ++a) {
            const int blk = b * TM + a;
            if (blk + 1 < TM * TN) load_res(blk + 1);
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const float4 bias = *reinterpret_cast<const float4 *>(sbias + a * 32 + 8 * q + 4 * lh);
                const float bv[4] = {bias.x, bias.y, bias.z, bias.w};
                float v[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) v[j] = __fadd_rn(acc[a][b][4 * q + j], bv[j]);
                act_store<EPI, true>(v, p.ep, table);
                turn[unit(li, 2 * q + lh)] = make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3]));
            }
            const int m = m_wave + a * 32 + 4 * u8, left = p.M - m;   // columns of C from this lane's on
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const uint4 t = turn[unit(8 * i + row8, u8)];
                u32x4 o = {t.x, t.y, t.z, t.w};
                if constexpr (RES)
#pragma unroll
                    for (int j = 0; j < 4; ++j) o[j] = __float_as_uint(__fadd_rn(__uint_as_float(o[j]), __uint_as_float(rv[blk & 1][i][j])));
                if constexpr (NORM)
                    if (left > 0)   // rows of a multiple of four
#pragma unroll
                        for (int j = 0; j < 4; ++j) norm[(b * 32 + 8 * i + row8) * (p.M + 1) + m + j] = __uint_as_float(o[j]);
                const unsigned at = place(a, b, i);
                if (left >= 4) {
                    __builtin_amdgcn_raw_buffer_store_b128(o, rc, at, 0, 0);
                } else {
#pragma unroll
                    for (int j = 0; j < 3; ++j)
                        if (j < left) __builtin_amdgcn_raw_buffer_store_b32(o[j], rc, at + 4u * j, 0, 0);
                }
            }
        }
    }
}

// A problem whose rows of C are normalised as well (RowNorm): what the kernel takes of it.
struct IgemmNormProblem : IgemmProblem {
    const float *norm_w, *norm_b;
    float *norm_y, inv_n;
};

// ---- LayerNormalization of the finished tile's rows (the NORM variant, rows of B, one tile over all columns of C) ------------------------
// The tile holds whole rows of C, so their LayerNormalization needs no launch of its own and no trip to memory in between: the store leaves
// a copy in LDS (odd pitch), a wavefront adds up the 64 rows, another one their squares, all of them normalise.  Same operations in the same
// order as layernorm_rows4_kernel: the same bits.  A chain of M additions and a pass over LDS are 3 to 4 us more on the product (12544 rows of
// 192 columns from K = 192 15.8 -> 19.0, from K = 768 34.4 -> 38.6) instead of a launch of 6.8; ViT-Tiny at batch 64 1866 -> 1756 us.
template <int NT>
__device__ __forceinline__ void normalise_rows(const IgemmNormProblem &p, const float *tile, float *stats, int n0, int tid) {
    const int pitch = p.M + 1, rows = min(64, p.N - n0), groups = p.M / 4, lane = tid & 63, wave = tid >> 6;
    // a thread keeps its four columns and walks down the rows
    const int per_pass = NT / groups, r0 = tid / groups, c = tid - r0 * groups;
    const float4 w = reinterpret_cast<const float4 *>(p.norm_w)[c], b = reinterpret_cast<const float4 *>(p.norm_b)[c];
    __syncthreads();
    if (wave < 2 && lane < rows) stats[wave * 64 + lane] = wave == 0 ? ln_chain<false>(tile + lane * pitch, p.M) : ln_chain<true>(tile + lane * pitch, p.M);
    __syncthreads();
    if (tid < rows) ln_stats(stats[tid], stats[64 + tid], p.inv_n, &stats[tid], &stats[64 + tid]);
    __syncthreads();
    if (r0 >= per_pass) return;
    for (int r = r0; r < rows; r += per_pass) {
        const float *t = tile + r * pitch + 4 * c;
        const float m = stats[r], s = stats[64 + r];
        const float4 o = make_float4(ln_one(t[0], m, s, w.x, b.x), ln_one(t[1], m, s, w.y, b.y), ln_one(t[2], m, s, w.z, b.z), ln_one(t[3], m, s, w.w, b.w));
        reinterpret_cast<float4 *>(p.norm_y + (size_t) (n0 + r) * p.M)[c] = o;
    }
}

// ---- a second, 1x1 product over the finished tile (the PW2 variant of the kernel, tile 64 x 64) --------------------------------
// As pw2_stage of igemm_kernel.hpp, on the 16-bit matrix cores: the workgroup's tile, with bias and activation applied in fp32, is
// split into its three parts and goes to LDS as the B operand of out[m2][64] = w2[m2][M] * tile ([part][row / 8][column][8 bf16]; a lane's
// accumulator registers 4 q .. 4 q + 3 are half of such a slot).  Every wavefront then walks w2, split ahead of time like the first weights,
// 32 rows at a time, four steps of 16 rows of the tile each: six matrix instructions a step, A two steps ahead from memory, B a step ahead
// from LDS, no barrier.  A value that is not finite when scaled is kept as split_weights_kernel keeps one, so sums that are not finite
// are computed again in fp32 from the same operands.
// Bound by HBM in the first stage of a ResNet (the addend and the result): 3x3 64 -> 64 and 1x1 64 -> 256 with the Add on 56 x 56 at batch 32 take 95 us (231 MB;
// 130 on fp32 matrix instructions), without it 87 (124).
// tl: LDS of at least 3 * 8 * 64 * 16 bytes that no wavefront reads any more (the caller has synchronised).
template <bool RES>
__device__ __forceinline__ void pw2_split_stage(const IgemmProblem &p, const f32x16 &acc1, uint4 *tl, const float *sbias, int n0, int wm, int wn,
                                                int li, int lh) {
    const int cmid = p.M;
    constexpr int STEPS = 4;   // 64 rows of the tile; those beyond cmid are zero
    const int ksteps = (cmid + 15) / 16, lane = lh * 32 + li;
    const rsrc_t rw2 = make_rsrc(p.w2, (unsigned) ((p.m2 + 31) / 32 * ksteps) * 3072u);
    const unsigned pitch = (unsigned) ksteps * 3072u, lane16 = (unsigned) lane * 16u;
    const int mblocks = (p.m2 + 63) / 64;
    struct Step { uint4 part[3]; };
    // nothing is read of steps beyond ksteps (their rows of the tile are zero as well) and of blocks of rows beyond m2
    auto load_a = [&](Step &o, int mb, int s, int z) __attribute__((always_inline)) {
        const bool on = s < ksteps && (mb * 2 + wm) * 32 < p.m2;   // uniform
        o.part[z] = buf_load_b128(rw2, on ? lane16 : OOB, on ? (unsigned) (mb * 2 + wm) * pitch + (unsigned) s * 3072u + (unsigned) z * 1024u : 0u);
    };
    Step wa[2];
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
        for (int z = 0; z < 3; ++z) load_a(wa[s], 0, s, z);
    // none, Relu or Clip (the launcher refuses others): apply_act's comparisons as selects under two uniform flags
    const bool lo_on = p.ep.act == RELU || p.ep.act == CLIP, hi_on = p.ep.act == CLIP;
    const float lo = p.ep.act == CLIP ? p.ep.clip_min : 0.0f, hi = p.ep.clip_max;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float4 t = *reinterpret_cast<const float4 *>(sbias + wm * 32 + 8 * q + 4 * lh);
        const float b1[4] = {t.x, t.y, t.z, t.w};
        float v[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            float x = __fadd_rn(acc1[4 * q + j], b1[j]);
            x = (lo_on & !(x > lo)) ? lo : x;
            x = (hi_on & !(x < hi)) ? hi : x;
            v[j] = wm * 32 + 8 * q + 4 * lh + j < cmid ? x : 0.0f;
        }
        SplitUnit u;
        u.phase<0>(v[0], v[1], v[2], v[3]);
        const float probe = __builtin_fmaf(u.u0, 0.0f, __builtin_fmaf(u.u1, 0.0f, __builtin_fmaf(u.u2, 0.0f, u.u3 * 0.0f)));
        const float first[4] = {u.u0, u.u1, u.u2, u.u3};
        u.phase<1>(v[0], v[1], v[2], v[3]);
        u.phase<2>(v[0], v[1], v[2], v[3]);
        u.phase<3>(v[0], v[1], v[2], v[3]);
        if (probe != probe) {
            unsigned *h[2] = {&u.h0, &u.h1}, *m[2] = {&u.m0, &u.m1}, *l[2] = {&u.l0, &u.l1};
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if (first[j] - first[j] == 0.0f) continue;
                const unsigned raw = __float_as_uint(v[j]), keep = j % 2 ? 0xffffu : 0xffff0000u, at = j % 2 * 16;
                *h[j / 2] = (*h[j / 2] & keep) | 0x7f80u << at;
                *m[j / 2] = (*m[j / 2] & keep) | (raw >> 16) << at;
                *l[j / 2] = (*l[j / 2] & keep) | (raw & 0xffffu) << at;
            }
        }
        uint2 *base = reinterpret_cast<uint2 *>(&tl[(wm * 4 + q) * 64 + wn * 32 + li]) + lh;
        base[0] = make_uint2(u.h0, u.h1);
        base[2 * 8 * 64] = make_uint2(u.m0, u.m1);
        base[4 * 8 * 64] = make_uint2(u.l0, u.l1);
    }
    __syncthreads();
    const uint4 *tbp = tl + lh * 64 + wn * 32 + li;
    auto read_b = [&](Step &o, int s, int z) __attribute__((always_inline)) { o.part[z] = tbp[(z * 8 + 2 * s) * 64]; };
    Step tb;
#pragma unroll
    for (int z = 0; z < 3; ++z) read_b(tb, 0, z);

    const rsrc_t rc = make_rsrc(p.C, RSRC_RANGE);
    const rsrc_t rres = make_rsrc(RES ? p.res : nullptr, RES ? RSRC_RANGE : 0u);
    const rsrc_t rb2 = make_rsrc(p.bias2, p.bias2 ? (unsigned) (p.m2 * 4) : 0u);
    const bool bias2_on = p.bias2 != nullptr, lo2_on = p.ep2.act == RELU || p.ep2.act == CLIP, hi2_on = p.ep2.act == CLIP;
    const float lo2 = p.ep2.act == CLIP ? p.ep2.clip_min : 0.0f, hi2 = p.ep2.clip_max;
    const unsigned row_bytes = (unsigned) p.c_stride_m * 4u, lh16 = (unsigned) lh * 16u;
    const int n = n0 + wn * 32 + li, lh4 = 4 * lh;
    const unsigned col_voff = n < p.N ? out_col_offset(p, n, 4) + (unsigned) lh4 * row_bytes : OOB;
    // rows in groups of four: a lane's are inside or beyond m2 by group and remainder, asked again for the store
    auto row_voff = [&](int m_uni, auto edge) __attribute__((always_inline)) { return !decltype(edge)::value || lh4 < p.m2 - m_uni ? col_voff : OOB; };
    // relu.c's rule by element index: row offsets of this lane's column that lie in its body (one register, not sixteen sums)
    const unsigned body = p.res_body * 4u > col_voff ? p.res_body * 4u - col_voff : 0u;
    auto finish = [&](float v, float bias, float addend, int m_uni, auto edge) __attribute__((always_inline)) {
        if (!row_there<decltype(edge)::value>(m_uni, p.m2)) return;   // uniform
        v = bias2_on ? __fadd_rn(v, bias) : v;
        v = (lo2_on & !(v > lo2)) ? lo2 : v;
        v = (hi2_on & !(v < hi2)) ? hi2 : v;
        if constexpr (RES) v = add_res(v, addend, p.res_relu, (unsigned) m_uni * row_bytes, body);
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), rc, row_voff(m_uni, edge), (unsigned) m_uni * row_bytes, 0);
    };
    bool fine = true;   // every sum of the wavefront so far is finite (uniform)
    for (int mb = 0; mb < mblocks; ++mb) {
        const int m_wave = mb * 64 + wm * 32;   // uniform
        const bool m_edge = m_wave + 32 > p.m2;
        float b2[16], rv[RES ? 16 : 1];
        auto addends = [&](auto edge) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m_uni = m_wave + 8 * (r / 4) + (r % 4);
                rv[r] = 0.0f;
                if (row_there<decltype(edge)::value>(m_uni, p.m2)) rv[r] = buf_load_f32(rres, row_voff(m_uni, edge), (unsigned) m_uni * row_bytes);
            }
        };
        if constexpr (RES) {
            if (m_edge) addends(std::true_type{});
            else addends(std::false_type{});
        }
        __builtin_amdgcn_sched_barrier(0);
        f32x16 acc2;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc2[r] = 0.0f;
        static_for<STEPS>([&](auto step) __attribute__((always_inline)) {
            constexpr int s = decltype(step)::value;
            static_for<F3_PRODUCTS>([&](auto product) __attribute__((always_inline)) {
                constexpr int pr = decltype(product)::value;
                mma_bf16(acc2, wa[s & 1].part[f3_pa(pr)], tb.part[f3_pb(pr)]);
                // two steps on, into the registers whose products are done
                if constexpr (pr == 0 || pr == 2 || pr == 5) load_a(wa[s & 1], s + 2 < STEPS ? mb : mb + 1, (s + 2) % STEPS, f3_pa(pr));
                if constexpr (pr >= 3) read_b(tb, (s + 1) % STEPS, f3_pb(pr));
                __builtin_amdgcn_sched_barrier(0);
            });
            if constexpr (s == STEPS - 2) {
#pragma unroll
                for (int r = 0; r < 16; ++r) b2[r] = buf_load_f32(rb2, lh16, (unsigned) (m_wave + 8 * (r / 4) + (r % 4)) * 4u);
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        float probe = 0.0f;   // as in unscale_fix_nonfinite
#pragma unroll
        for (int r = 0; r < 16; ++r) probe = __builtin_fmaf(acc2[r], 0.0f, probe);
        fine &= __builtin_amdgcn_ballot_w64(probe != probe) == 0ull;
        auto store = [&](auto edge) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) finish(acc2[r] * F3_UNSCALE, b2[r], RES ? rv[r] : 0.0f, m_wave + 8 * (r / 4) + (r % 4), edge);
        };
        if (m_edge) store(std::true_type{});
        else store(std::false_type{});
    }
    if (fine) return;
    // All blocks once more, sums that are not finite from fp32 matrix instructions: a pass of its own, so that the one above
    // keeps no registers for it.  Behind the stores that it writes over.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#pragma unroll 1
    for (int mb = 0; mb < mblocks; ++mb) {
        f32x16 acc2, again;
#pragma unroll
        for (int r = 0; r < 16; ++r) acc2[r] = again[r] = 0.0f;
#pragma unroll 1
        for (int s = 0; s < STEPS; ++s) {
            Step a;
#pragma unroll
            for (int z = 0; z < 3; ++z) { load_a(a, mb, s, z); read_b(tb, s, z); }
            static_for<F3_PRODUCTS>([&](auto pr) __attribute__((always_inline)) { mma_bf16(acc2, a.part[f3_pa(pr)], tb.part[f3_pb(pr)]); });
#pragma unroll
            for (int j = 0; j < 8; ++j) again = __builtin_amdgcn_mfma_f32_32x32x2f32(f3_whole(a.part, j), f3_whole(tb.part, j), again, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const int m_uni = mb * 64 + wm * 32 + 8 * (r / 4) + (r % 4);
            const float bias = buf_load_f32(rb2, lh16, (unsigned) m_uni * 4u);
            if (!row_there<true>(m_uni, p.m2)) continue;   // uniform
            const float addend = RES ? buf_load_f32(rres, row_voff(m_uni, std::true_type{}), (unsigned) m_uni * row_bytes) : 0.0f;
            finish(acc2[r] * 0.0f != 0.0f ? again[r] : acc2[r] * F3_UNSCALE, bias, addend, m_uni, std::true_type{});
        }
    }
}

// (the second bound: wavefronts a SIMD that the registers leave room for.  128 of them are four; with a residual operand in tiles of 128 rows the
// compiler took one more, and 21 -> 1430 channels under 3x3 on 83 x 83 with an Add 52 us instead of 47)
template <int BL, int BM, int BN, int WM, int WN, bool RES, bool PW2 = false, bool NORM = false>
__global__ __launch_bounds__(64 * WM * WN, (BM / WM) * (BN / WN) >= 32 * 128 ? 2 : (BM / WM) * (BN / WN) > 32 * 64 ? 3 : 4)
void igemm_f3_kernel(const std::conditional_t<NORM, IgemmNormProblem, IgemmProblem> p) {
    static_assert(!NORM || (BL == BL_ROWS && WM * WN >= 4 && BN == 64 && RES), "rows are normalised behind a residual operand, 64 rows a tile");
    static_assert(BM % (WM * 32) == 0 && BN % (WN * 32) == 0, "wavefronts of 32 x 32 blocks");
    constexpr int TM = BM / WM / 32, TN = BN / WN / 32;
    constexpr int UPT = 4, NT = 64 * WM * WN;
    constexpr bool ALL = BN * UPT == NT;   // a thread stages one unit of B per K tile, or the first wavefronts' do
    static_assert(ALL || (BN * UPT < NT && BN * UPT % 64 == 0));
    constexpr int LD = BL == BL_ROWS ? BN + 1 : BN;   // 16-byte slots per 8 elements of K; rows arrive from neighbouring lanes
    constexpr int PLANE = 2 * LD, SLOTS = 3 * PLANE;
    static_assert(!PW2 || (BM == 64 && BN == 64 && WM == 2 && WN == 2), "the second product exists for tiles of 64 x 64");
    // two K tiles; with PW2 then the first product as three parts, for rows 4 KB a wavefront for their store
    constexpr int AFTER = PW2 ? 3 * 8 * 64 : BL == BL_ROWS ? WM * WN * 256 : 0;
    __shared__ uint4 lds[AFTER > 2 * SLOTS ? AFTER : 2 * SLOTS];
    static_assert(sizeof(lds) >= 2 * SLOTS * sizeof(uint4));
    __shared__ __attribute__((aligned(16))) float s_bias[BM];

    warm_params<(sizeof(p) < 640 ? sizeof(p) : 640)>();
    const int tid = threadIdx.x;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    const int wm = wave / WN, wn = wave % WN;

    extern __shared__ __attribute__((aligned(1024))) float s_table[];   // TABLE_BYTES where table_in_lds says so
    if (!PW2 && !NORM && table_in_lds(p)) request_table(p.ep.lut, s_table, wave, lane, NT);   // NORM: s_table is the rows' copy

    const TilePlace tp = place_tile<BM, BN>(p);
    const int m0 = tp.m0, n0 = tp.n0, slice = tp.slice;
    const int u_begin = slice * p.k_split_units, u_end = min(p.k_units, u_begin + p.k_split_units);
    const int k_tiles = (u_end - u_begin + UPT - 1) / UPT;
    const int klim = min(p.K, u_end * 4);

    const char *b_base = reinterpret_cast<const char *>(p.B) - (size_t) p.b_shift_bytes;
    const unsigned b_bytes = (unsigned) (p.b_slice_bytes + p.b_shift_bytes);

    // A: [32 rows][16 of K][part][lane][16 bytes], row block, K tile and part in the scalar offset
    const rsrc_t ra = make_rsrc(p.a_split, (unsigned) p.a_split_bytes);
    const unsigned a_pitch = (unsigned) ((p.K + 15) / 16) * 3072u;
    const unsigned a_block0 = (unsigned) ((m0 + wm * (BM / WM)) / 32) * a_pitch + (unsigned) (u_begin / UPT) * 3072u;
    const unsigned lane16 = (unsigned) lane * 16u;

    // B: this thread's column and its unit of every K tile.  From NCHW activations lanes run along the columns and the unit
    // is the wavefront's; from rows four neighbouring lanes hold the four units of a row (64 contiguous bytes)
    const int bcol = BL == BL_ROWS ? tid / UPT : tid % BN;
    const int bunit = BL == BL_ROWS ? tid % UPT : __builtin_amdgcn_readfirstlane(tid / BN);
    const ColState col = f3_col<BL>(p, n0 + bcol);
    const bool stages = ALL || wave < BN * UPT / 64;   // uniform

    f32x16 acc[TM][TN];
#pragma unroll
    for (int a = 0; a < TM; ++a)
#pragma unroll
        for (int b = 0; b < TN; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[a][b][r] = 0.0f;

    constexpr int BE = BL == BL_GATHER ? 4 : 1;         // scalar descriptions per B unit
    constexpr int STEPS = F3_PRODUCTS * TM * TN;        // MFMAs per K tile and wavefront
    constexpr int BAR = STEPS / 2 + 1;                  // the barrier stands before this step
    constexpr int READS = 3 * TN;
    struct Operands { uint4 a[3][TM], b[3][TN]; };
    RawUnit<DT_F32> qb[2];                              // two K tiles in flight between memory and LDS
    F3Prep bp[BE];
    const unsigned hw4 = (unsigned) p.HW * 4u;

    auto prep_unit = [&](int kt) __attribute__((always_inline)) {
        if constexpr (BL != BL_ROWS)
#pragma unroll
            for (int e = 0; e < BE; ++e) bp[e] = f3_prep<BL>(p, u_begin + kt * UPT + bunit, e);
    };
    // the loads of B for K tile kt; a tile past the end reads through an empty descriptor (zeros, no traffic)
    auto issue_b = [&](int kt, auto slot) __attribute__((always_inline)) {
        RawUnit<DT_F32> &q = qb[decltype(slot)::value];
        const rsrc_t rb = make_rsrc(b_base, kt < k_tiles ? b_bytes : 0u);
        if constexpr (BL == BL_ROWS) {
            const uint4 t = buf_load_b128(rb, col.pixoff + (unsigned) bunit * 16u, (unsigned) (u_begin + kt * UPT) * 16u);
            q.v[0] = __uint_as_float(t.x); q.v[1] = __uint_as_float(t.y); q.v[2] = __uint_as_float(t.z); q.v[3] = __uint_as_float(t.w);
        } else if constexpr (BL == BL_TAPC) {
            const unsigned voff = f3_voff<BL>(col, bp[0].tap);
#pragma unroll
            for (int e = 0; e < 4; ++e) q.v[e] = buf_load_f32(rb, voff, bp[0].soff + (unsigned) e * hw4);
        } else if constexpr (BL == BL_PLAIN) {
#pragma unroll
            for (int e = 0; e < 4; ++e) q.v[e] = buf_load_f32(rb, col.pixoff, bp[0].soff + (unsigned) e * hw4);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) q.v[e] = buf_load_f32(rb, f3_voff<BL>(col, bp[e].tap), bp[e].soff);
        }
    };
    auto load_a = [&](Operands &o, int kt, int part) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < TM; ++t) o.a[part][t] = buf_load_b128(ra, lane16, a_block0 + (unsigned) t * a_pitch + (unsigned) kt * 3072u + part * 1024u);
    };
    SplitUnit work;   // the unit being split
    auto stage_b = [&](int buf, auto phase, auto slot) __attribute__((always_inline)) {
        constexpr int Q = decltype(phase)::value;
        const RawUnit<DT_F32> &q = qb[decltype(slot)::value];
        work.phase<Q>(q.v[0], q.v[1], q.v[2], q.v[3]);
        if constexpr (Q == 3) {
            uint2 *base = reinterpret_cast<uint2 *>(&lds[buf + bunit / 2 * LD + bcol]) + bunit % 2;
            base[0] = make_uint2(work.h0, work.h1);
            base[2 * PLANE] = make_uint2(work.m0, work.m1);
            base[4 * PLANE] = make_uint2(work.l0, work.l1);
        }
    };
    // LDS reads in the order the products need them
    auto read_operand = [&](Operands &o, int buf, auto idx) __attribute__((always_inline)) {
        constexpr int pb = decltype(idx)::value / TN, t = decltype(idx)::value % TN;
        o.b[pb][t] = lds[buf + pb * PLANE + lh * LD + wn * (BN / WN) + t * 32 + li];
    };

    Operands op0, op1;
    constexpr std::integral_constant<int, 0> S0{};
    constexpr std::integral_constant<int, 1> S1{};
    prep_unit(0);
    if (stages) issue_b(0, S0);
#pragma unroll
    for (int z = 2; z >= 0; --z) load_a(op0, 0, z);
    prep_unit(1);
    if (stages) issue_b(1, S1);
#pragma unroll
    for (int z = 2; z >= 0; --z) load_a(op1, 1, z);
    // One workgroup a compute unit and a long K: nothing but this workgroup's own loads, two K tiles ahead, covers the trip its part of A
    // makes to the L2, and all workgroups of an XCD ask for the same K tile at the same time, so each of them is that trip again.  A touch of
    // every cache line of A up front, shared out among the XCD's workgroups with the same rows, makes them one trip (rows 192 x 768, 196
    // workgroups: 39.0 -> 34.7 us a launch; 64 x 384 and 96 x 576, 196 of 128 x 64: 16.4 -> 14.0 and 24.2 -> 20.3).  Not for a short K (one trip as
    // well), not for several workgroups a unit (4099 x 1031 x 2053 106 -> 115), nor for more of A than leaves the L2 room (512 x 1024 43.6 -> 47.4).
    constexpr int TOUCH = BM > 64 ? 2 : 0;   // (64 x 64 tiles would lose a wavefront a SIMD to the registers)
    unsigned touch[TOUCH + 1];
    if constexpr (TOUCH) {
        constexpr int ROW = BM / 32 * 24;   // cache lines of a K tile
        unsigned at[TOUCH];
#pragma unroll
        for (int i = 0; i < TOUCH; ++i) at[i] = OOB;
        if (gridDim.x <= 256 && gridDim.y == 1 && !p.n_fast && k_tiles >= 24 && p.a_split_bytes <= (2 << 20)) {   // uniform
            const int share = max(1, (int) div31(gridDim.x >> 3, p.div_tiles_m)), turn = (int) div31(blockIdx.x >> 3, p.div_tiles_m);
#pragma unroll
            for (int i = 0; i < TOUCH; ++i) {
                const int l = (i * share + turn) * NT + tid, kt = l / ROW, r = l - kt * ROW;
                if (kt < k_tiles) at[i] = (unsigned) (r / 24) * a_pitch + (unsigned) kt * 3072u + (unsigned) (r % 24) * 128u;
            }
        }
#pragma unroll
        for (int i = 0; i < TOUCH; ++i) touch[i] = __builtin_amdgcn_raw_buffer_load_b32(ra, at[i], (unsigned) (m0 / 32) * a_pitch, 0);
    }
    float bias_row[(BM + NT - 1) / NT];   // the tile's rows of the bias, for LDS when the K loop is over; -0.0f changes nothing
#pragma unroll
    for (int i = 0; i < (BM + NT - 1) / NT; ++i) {
        const bool on = p.bias_mode == BIAS_M;
        const int row = tid + i * NT;
        const float bv = buf_load_f32(make_rsrc(p.bias, on ? (unsigned) (p.M * 4) : 0u), row < BM ? (unsigned) (m0 + row) * 4u : OOB, 0);
        bias_row[i] = on ? bv : -0.0f;
    }
    if (stages) static_for<4>([&](auto ph) __attribute__((always_inline)) { stage_b(0, ph, S0); });
    prep_unit(2);
    if (stages) issue_b(2, S0);
    prep_unit(3);
    __syncthreads();
    static_for<READS>([&](auto i) __attribute__((always_inline)) { read_operand(op0, 0, i); });

    // Body kt: the MFMAs of tile kt, whose operands are in registers.  Behind them, a phase at a time over the steps before the
    // barrier, B of tile kt + 1 goes through the split to LDS, with the loads of tile kt + 3 into the registers that frees;
    // after the barrier the LDS reads of tile kt + 1.  A of tile kt + 2 is loaded into the operand registers of tile kt as
    // its products retire them (l first, h last).
    auto body = [&](Operands &cur, Operands &nxt, int kt, auto wr, auto stager) __attribute__((always_inline)) {
        constexpr int WR = decltype(wr)::value * SLOTS;
        __builtin_amdgcn_sched_barrier(0);
        static_for<STEPS>([&](auto step) __attribute__((always_inline)) {
            constexpr int st = decltype(step)::value, pr = st / (TM * TN), a = (st / TN) % TM, b = st % TN;
            mma_bf16(acc[a][b], cur.a[f3_pa(pr)][a], cur.b[f3_pb(pr)][b]);
            static_for<4>([&](auto phase) __attribute__((always_inline)) {
                constexpr int ph = decltype(phase)::value;
                if constexpr (decltype(stager)::value && ph * (BAR - 1) / 4 == st) {
                    stage_b(WR, phase, wr);
                    if constexpr (ph == 1) {   // the unit's floats are used up
                        issue_b(kt + 3, wr);
                        prep_unit(kt + 4);
                    }
                }
            });
            if constexpr (st == 1 * TM * TN - 1) load_a(cur, kt + 2, 2);
            if constexpr (st == 3 * TM * TN - 1) load_a(cur, kt + 2, 1);
            if constexpr (st == 6 * TM * TN - 1) load_a(cur, kt + 2, 0);
            static_for<READS>([&](auto i) __attribute__((always_inline)) {
                if constexpr (st >= BAR && BAR + decltype(i)::value * (STEPS - BAR) / READS == st) read_operand(nxt, WR, i);
            });
            if constexpr (st == BAR - 1) __syncthreads();
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // Two tiles a trip; behind an odd last tile runs one more, whose B is zero.  No test of reduction indices anywhere: beyond
    // K the split weights are zero, and what B brings in there (the next row or image, zeros behind the tensor) is multiplied
    // by that; should it not be finite, unscale_fix_nonfinite sums the elements over K alone.
    auto loop = [&](auto stager) __attribute__((always_inline)) {
        for (int kt = 0; kt < k_tiles; kt += 2) {
            body(op0, op1, kt, S1, stager);
            body(op1, op0, kt + 1, S0, stager);
        }
    };
    if (ALL || stages) loop(std::true_type{});
    else loop(std::false_type{});   // as many barriers
#pragma unroll
    for (int i = 0; i < TOUCH; ++i) asm volatile("" :: "v"(touch[i]));   // kept until here
#pragma unroll
    for (int i = 0; i < (BM + NT - 1) / NT; ++i)
        if (tid + i * NT < BM) s_bias[tid + i * NT] = bias_row[i];
    if (!PW2 && !NORM && table_in_lds(p)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's part of the table
    __syncthreads();

    const int m_wave = m0 + wm * (BM / WM), n_wave = n0 + wn * (BN / WN);
    unscale_fix_nonfinite<BL, TM, TN>(p, acc, ra, make_rsrc(b_base, b_bytes), m_wave, n_wave, lane, u_begin, klim);
    if constexpr (PW2) {   // the launcher gives this variant one row tile and all of K
        pw2_split_stage<RES>(p, acc[0][0], lds, s_bias, n0, wm, wn, li, lh);
        return;
    }
    if (p.partial) {   // a finishing launch adds the slices up
        write_partial<TM, TN, false>(p, acc, slice, m_wave, n_wave, li, lh);
        return;
    }
    const float *sb = s_bias + wm * (BM / WM);
    if constexpr (NORM) {   // the launcher gives this variant no activation and a tile over all of M
        write_tile_rows<EPI_NONE, TM, TN, RES, true>(p, acc, m_wave, n_wave, li, lh, sb, (lds_f32_t) nullptr, lds + wave * 256, s_table + wn * (BN / WN) * (p.M + 1));
        static_assert(TN == 1 && BM >= 128, "a lane holds one row; the bias's LDS takes the statistics");
        normalise_rows<NT>(p, s_table, s_bias, n0, tid);
        return;
    }
    auto store = [&](auto epi) __attribute__((always_inline)) {
        constexpr int EPI = decltype(epi)::value;
        if constexpr (BL == BL_ROWS) write_tile_rows<EPI, TM, TN, RES>(p, acc, m_wave, n_wave, li, lh, sb, (lds_f32_t) s_table, lds + wave * 256);
        else write_tile<DT_F32, EPI, TM, TN, RES, true, true>(p, acc, 0, m_wave, n_wave, li, lh, sb, nullptr, nullptr, 0, (lds_f32_t) s_table);
    };
    switch (p.ep.act) {
        case NOT_ACT:
        case RELU6: store(std::integral_constant<int, EPI_NONE>{}); break;
        case RELU: store(std::integral_constant<int, EPI_RELU>{}); break;
        case CLIP: store(std::integral_constant<int, EPI_CLIP>{}); break;
        case SILU:
        case ONHIP_ACT_GELU_LUT: store(std::integral_constant<int, EPI_LUT>{}); break;
        default: store(std::integral_constant<int, EPI_GENERIC>{}); break;
    }
}

template <int BL, int BM, int BN, int WM, int WN, bool RES>
static int f3_launch_one(const IgemmLaunch &cfg, const IgemmProblem &p_in, hipStream_t stream) {
    IgemmProblem p = p_in;
    dim3 grid;
    const int rc = tile_grid<BM, BN>(cfg, p, &grid);
    if (rc) return rc;
    if (RES != (p.res != nullptr)) return set_error(ONHIP_ERR_ARG, "igemm: residual operand and kernel variant do not match");
    hipLaunchKernelGGL((igemm_f3_kernel<BL, BM, BN, WM, WN, RES>), grid, dim3(64 * WM * WN), table_lds_bytes(p), stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return finish_launch<false>(cfg, p, stream);
}

// Up to one workgroup a compute unit: a tile of 192 x 64 in twelve wavefronts of one 32 x 32 block each instead of four of three, three a SIMD where
// there was one to wait for each barrier and each trip of A (196 workgroups, 192 x 12544 x 768 with rows normalised 36.4 -> 32.2 us, from K = 192 15.8 ->
// 12.8, 192 x 12544 x 768 from 16 x 16 pixels 50.1 -> 46.3; in slices, 160 x 3136 x 960 13.7 -> 12.9); with more of them they stand in for each
// other.  The other tiles stay as they are: 128 x 64 in eight and 256 x 64 in eight took 6 % and 14 % less a launch (256 x 6272 x 1024 30.0 -> 28.2, 512 x
// 1568 x 4608 in slices 46.5 -> 39.6) and ResNet-50 at batch 32 as long as before, its clock lower by as much; 128 x 128 in sixteen was slower
// (128 x 25088 x 576 56 -> 66).  Same products in the
// same order: same bits.
inline bool f3_alone(const IgemmLaunch &cfg, const IgemmProblem &p) {
    const long long slices = p.k_split_units ? (p.k_units + p.k_split_units - 1) / p.k_split_units : 1;
    return (long long) ((p.M + cfg.bm - 1) / cfg.bm) * ((p.N + cfg.bn - 1) / cfg.bn) * slices <= 256;
}

template <int BL, bool RES>
int f3_launch_tile(const IgemmLaunch &cfg, const IgemmProblem &p, hipStream_t stream) {
    switch (cfg.bm * 1000 + cfg.bn) {
        case 256128: return f3_launch_one<BL, 256, 128, 8, 1, RES>(cfg, p, stream);
        case 256064: return f3_launch_one<BL, 256, 64, 4, 1, RES>(cfg, p, stream);
        case 192064: return f3_alone(cfg, p) ? f3_launch_one<BL, 192, 64, 6, 2, RES>(cfg, p, stream) : f3_launch_one<BL, 192, 64, 2, 2, RES>(cfg, p, stream);
        case 128128: return f3_launch_one<BL, 128, 128, 4, 2, RES>(cfg, p, stream);
        case 128064: return f3_launch_one<BL, 128, 64, 4, 1, RES>(cfg, p, stream);
        case 64064: return f3_launch_one<BL, 64, 64, 2, 2, RES>(cfg, p, stream);
        default: return set_error(ONHIP_ERR_ARG, "igemm f32: no kernel for tile %dx%d", cfg.bm, cfg.bn);
    }
}

}  // namespace onhip
