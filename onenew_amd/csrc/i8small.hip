// int8 convolution with few output pixels in one launch (gfx950), from fp32 NCHW or int8 NHWC to either, with the Add of a residual block: the
// activations go once into LDS, quantised on their way where they are fp32, and K is cut over the wavefronts of a workgroup.
//
// Why: the general form of these layers is a launch that writes the activations as int8 NHWC (3.1-3.5 us at batch 1), the product
// (6-8 us, its K loop behind two dependent trips to memory), and for a long K on few tiles a launch that adds up slices (4.5 us) or, for an
// int8 result, which is never cut, a tile's whole K one step behind the other (16 us for 512 channels under a 3x3 filter).
//
// A workgroup of eight wavefronts owns 32 WM output channels x a rectangle of up to 32 NB output pixels of one image:
//   * the input rows and columns under that rectangle, all channels, go ONCE from fp32 NCHW through the quantiser into LDS as
//     [pixel][channel] int8: a thread takes 16 channels of one pixel (16 loads in flight, neighbouring lanes neighbouring pixels) and
//     stores 16 bytes; int8 activations are copied; a pixel takes an odd number of 16-byte units so that neighbours start in different banks;
//   * 32 of K at a time are one v_mfma_i32_32x32x32_i8 per 32 pixels.  WM wavefronts lie along the rows, the others take 64 of K in turn:
//     the weights come from memory four lanes to a row, the first three turns of them requested before the activations, and go through
//     a corner of LDS of the wavefront's own into the matrix instruction's order; the pixels lie in LDS at their place plus the offset
//     of the 16 of K (filter tap and channels), which a table holds: any filter, stride and padding;
//   * the wavefronts' sums meet in LDS (int32, exact), every thread finishes 2 NB WM outputs, a table activation from LDS.
// What bounds it: a launch, one trip to memory, the quantiser (six vector instructions a value), which runs once per 32 WM output channels
// and again where rectangles overlap, and the outputs a thread finishes: larger problems stay with the staged form (i8small_ok).
//
// Measured, us a layer in a graph, staged form -> this: 64 -> 64 channels 1x1 on 20 x 20 pixels 5.3 -> 3.9, 3x3 7.6 -> 4.5, 3x3 on 80 x 80
// 7.9 -> 5.7; 128 -> 128 3x3 on 40 x 40 9.3 -> 6.2; 256 -> 256 3x3 on 20 x 20 11.2 -> 6.7; 512 -> 512 1x1 on 20 x 20 7.8 -> 5.6, 256 -> 128
// on 80 x 80 8.6 -> 6.7; the 63 layers of YOLOv8s at batch 1 580 -> 441.  From int8 to int8 256 -> 256
// 3x3 on 20 x 20 10.3 -> 5.2, 512 -> 512 3x3 on 7 x 7 at batch 8 16.1 -> 6.4, 128 -> 128 on 40 x 40 6.4 -> 4.8; with an Add and the int8 form 960 ->
// 160 1x1 on 7 x 7 at batch 8 6.9 -> 4.8, 384 -> 64 on 14 x 14 5.2 -> 4.6.  On the way: a lane a row for the weights 494 (64 separate pieces a
// load), the table activation gathered from memory 484 (a compute unit takes a cycle for each of a load's 64 lines).
//
// Arithmetic: conv.c:961-973 (quantiser), :1024-1056 (acc * s, + bias, * (aux / 127), activation), the same bits as every other kernel
// of the W8A32 form.
#include <algorithm>
#include <atomic>
#include <cstring>

#include "igemm_kernel.hpp"

namespace onhip {

// quant_s8 in five instructions: rounded before it is clamped, by a conversion that saturates and makes 0 of a NaN (so does the cast in
// quant_s8).  Below 128.5 in magnitude the same rounding as there; beyond, both are past the clamp.
__device__ __forceinline__ int quant_s8_sat(float x, float inv_scale) {
    const float t = __fmul_rn(x, inv_scale);
    const float half = __uint_as_float((__float_as_uint(t) & 0x80000000u) | 0x3effffffu);
    int i;
    asm("v_cvt_i32_f32 %0, %1" : "=v"(i) : "v"(__fadd_rn(t, half)));
    return min(max(i, -128), 127);
}

constexpr int I8S_WAVES = 8, I8S_THREADS = 64 * I8S_WAVES, I8S_RING = 3;
constexpr int I8S_TURN_ROW = 80, I8S_TURN = 32 * I8S_TURN_ROW;   // bytes of 64 of K of a row, of a wavefront's chunk (rows 20 banks apart)
constexpr int I8S_LDS = 160 * 1024;

struct I8SmallParams {
    const float *x;                 // fp32 NCHW, or
    const int8_t *xq;               // int8 NHWC, cu * 16 channels a pixel
    const int8_t *w;                // [M][units * 16]: K = (filter tap, channel padded to 16)
    void *y;                        // fp32 NCHW or int8 NHWC
    const float *res;               // the other operand of a residual block's Add, laid out like y; then the Relu
    int res_relu;
    unsigned res_body;
    int8_t *twin;                   // the finished fp32 result once more as int8 NHWC, M channels a pixel
    float twin_inv_scale, out_inv_scale;
    const float *aux;
    const int32_t *bias32;
    Epilogue ep;
    float in_scale, inv_scale;
    int M, cin, H, W, HW, OH, OW, OHW;
    int stride, sw, pad_t, pad_l, kw;
    int cu, units;                  // 16-channel units of a pixel, of K
    int tr, tw, pr, pw;             // rectangle of output pixels, of input pixels under it
    int pitch, turn_at, table_at;   // bytes of a pixel in LDS; places of the weights' chunks and of the offset table
    Div31 div_m, div_tx, div_ty, div_pix, div_pw, div_tw, div_cu, div_kw;
};

// SRC8: int8 NHWC in; OUT: what leaves
enum { I8S_F32 = 0, I8S_ADD = 1, I8S_S8 = 2 };   // fp32; fp32 after a residual block's Add, perhaps its int8 twin as well; int8 NHWC

template <int NB, int WM, bool TABLE, bool SRC8, int OUT>
__global__ __launch_bounds__(I8S_THREADS) void i8small_kernel(const I8SmallParams p) {
    constexpr int BM = 32 * WM, WK = I8S_WAVES / WM, PER = 2 * NB * WM;   // rows, wavefronts along K, outputs of a thread
    constexpr int AT = TABLE ? TABLE_BYTES : 0;
    extern __shared__ __attribute__((aligned(1024))) unsigned char i8s_all[];   // the activation's table, then what follows it
    unsigned char *const i8s_lds = i8s_all + AT;
    warm_params<sizeof(I8SmallParams)>();
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    if constexpr (TABLE) request_table(p.ep.lut, reinterpret_cast<float *>(i8s_all), wave, lane, I8S_THREADS);
    const int wk = wave / WM, mw = wave % WM * 32;   // this wavefront's part of K and of the rows
    // an XCD takes a contiguous run of (image, rectangle, row block): the row blocks of a rectangle read its pixels through one L2
    const int nb = (int) gridDim.x, per = nb >> 3, rmd = nb & 7, xcd = (int) blockIdx.x & 7;
    unsigned id = (unsigned) (xcd * per + min(xcd, rmd) + ((int) blockIdx.x >> 3));
    auto take = [&](const Div31 &d, int n) { const unsigned q = div31(id, d), r = id - q * (unsigned) n; id = q; return (int) r; };
    const int m0 = take(p.div_m, (p.M + BM - 1) / BM) * BM;
    const int ox0 = take(p.div_tx, (p.OW + p.tw - 1) / p.tw) * p.tw;
    const int oy0 = take(p.div_ty, (p.OH + p.tr - 1) / p.tr) * p.tr;
    const long long img = (long long) id;
    const int iy0 = oy0 * p.stride - p.pad_t, ix0 = ox0 * p.sw - p.pad_l;

    // The weights' first chunks: 64 of K of the wavefront's 32 rows, four lanes a row (a lane a row would be 64 separate 16-byte pieces a
    // load, 64 cycles of the address path instead of 16)
    const int chunks = (p.units + 3) / 4;
    const unsigned w_bytes = (unsigned) p.M * (unsigned) p.units * 16u;
    unsigned a_voff[2];
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const int row = m0 + mw + h * 16 + lane / 4;
        a_voff[h] = row < p.M ? (unsigned) row * (unsigned) p.units * 16u + (unsigned) (lane & 3) * 16u : OOB;
    }
    struct Chunk { uint4 q[2]; };
    auto load_a = [&](Chunk &c, int chunk) __attribute__((always_inline)) {
        const rsrc_t ra = make_rsrc(p.w, chunk < chunks ? w_bytes : 0u);
        const bool in = chunk * 4 + (lane & 3) < p.units;
#pragma unroll
        for (int h = 0; h < 2; ++h) c.q[h] = buf_load_b128(ra, in ? a_voff[h] : OOB, (unsigned) chunk * 64u);
    };
    Chunk ring[I8S_RING];
#pragma unroll
    for (int j = 0; j < I8S_RING; ++j) load_a(ring[j], wk + WK * j);

    // what this thread's outputs need: value v of the workgroup is register (v / 64) % 16 of lane v % 64, pixel block
    // (v / 1024) % NB, row block v / (1024 NB)
    unsigned at[PER];
    float aux[PER], b32[PER], res[OUT == I8S_ADD ? PER : 1];
    const long long y_img = img * (long long) p.M * p.OHW;   // elements in front of the image in an NCHW result
    {
        const rsrc_t rres = make_rsrc(OUT == I8S_ADD ? p.res + y_img : nullptr, OUT == I8S_ADD ? (unsigned) p.M * (unsigned) p.OHW * 4u : 0u);
        const rsrc_t raux = make_rsrc(p.aux, (unsigned) p.M * 4u), rb = make_rsrc(p.bias32, p.bias32 ? (unsigned) p.M * 4u : 0u);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            const int v = tid + i * I8S_THREADS, r = v / 64 % 16, j = v / 1024 % NB * 32 + li;
            const int row = m0 + v / (1024 * NB) * 32 + 8 * (r / 4) + 4 * lh + r % 4;
            const int ty = (int) div31((unsigned) j, p.div_tw), tx = j - ty * p.tw;
            const bool on = row < p.M && ty < p.tr && oy0 + ty < p.OH && ox0 + tx < p.OW;
            at[i] = on ? (unsigned) (row * p.OHW + (oy0 + ty) * p.OW + ox0 + tx) * 4u : OOB;
            if constexpr (OUT == I8S_ADD) res[i] = buf_load_f32(rres, at[i], 0);
            aux[i] = buf_load_f32(raux, (unsigned) row * 4u, 0);
            const float f = (float) (int) __builtin_amdgcn_raw_buffer_load_b32(rb, (unsigned) row * 4u, 0, 0);
            b32[i] = p.bias32 ? f : -0.0f;   // the addend that changes nothing
        }
    }

    // the pixels under the rectangle
    const int pixels = p.pr * p.pw, items = pixels * p.cu;
    if constexpr (SRC8) {   // copied, neighbouring lanes the units of a pixel
        const rsrc_t rx = make_rsrc(p.xq + img * (long long) p.HW * p.cu * 16, (unsigned) p.HW * (unsigned) p.cu * 16u);
        constexpr int N = 4;   // in flight
        for (int i0 = tid; i0 < items; i0 += N * I8S_THREADS) {
            uint4 v[N];
            unsigned to[N];
#pragma unroll
            for (int j = 0; j < N; ++j) {
                const int i = i0 + j * I8S_THREADS;
                const unsigned px = div31((unsigned) i, p.div_cu), unit = (unsigned) i - px * (unsigned) p.cu, py = div31(px, p.div_pw);
                const int iy = iy0 + (int) py, ix = ix0 + (int) (px - py * (unsigned) p.pw);
                const bool on = i < items && (unsigned) iy < (unsigned) p.H && (unsigned) ix < (unsigned) p.W;
                v[j] = buf_load_b128(rx, on ? ((unsigned) (iy * p.W + ix) * (unsigned) p.cu + unit) * 16u : OOB, 0);
                to[j] = px * (unsigned) p.pitch + unit * 16u;
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < N; ++j)
                if (i0 + j * I8S_THREADS < items) *reinterpret_cast<uint4 *>(i8s_lds + to[j]) = v[j];
        }
    } else {
        const unsigned hw4 = (unsigned) p.HW * 4u;
        const rsrc_t rx = make_rsrc(p.x + img * (long long) p.cin * p.HW, (unsigned) p.cin * hw4);   // channels past the last come as zeros
        struct Item { float v[16]; unsigned to; };
        auto load = [&](Item &q, int i) __attribute__((always_inline)) {
            const unsigned unit = div31((unsigned) i, p.div_pix), px = (unsigned) i - unit * (unsigned) pixels;
            const unsigned py = div31(px, p.div_pw);
            const int iy = iy0 + (int) py, ix = ix0 + (int) (px - py * (unsigned) p.pw);
            const bool on = i < items && (unsigned) iy < (unsigned) p.H && (unsigned) ix < (unsigned) p.W;
            const unsigned voff = on ? unit * 16u * hw4 + (unsigned) (iy * p.W + ix) * 4u : OOB;
            q.to = px * (unsigned) p.pitch + unit * 16u;
#pragma unroll
            for (int e = 0; e < 16; ++e) q.v[e] = buf_load_f32(rx, voff, (unsigned) e * hw4);
        };
        auto put = [&](const Item &q) __attribute__((always_inline)) {
            unsigned w[4];
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                int b[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) b[e] = quant_s8_sat(q.v[4 * g + e], p.inv_scale);
                const unsigned p01 = __builtin_amdgcn_perm((unsigned) b[1], (unsigned) b[0], 0x0c0c0400u);
                const unsigned p23 = __builtin_amdgcn_perm((unsigned) b[3], (unsigned) b[2], 0x0c0c0400u);
                w[g] = __builtin_amdgcn_perm(p23, p01, 0x05040100u);
            }
            *reinterpret_cast<uint4 *>(i8s_lds + q.to) = make_uint4(w[0], w[1], w[2], w[3]);
        };
        for (int i = tid; i < items; i += 2 * I8S_THREADS) {
            Item q[2];
            load(q[0], i);
            // the second item's loads only where some lane has one: sent out with nothing to fetch they take the address path as long as the
            // others (YOLOv8s at batch 1 538 -> 531 us)
            const bool two = i + I8S_THREADS - lane < items;   // uniform
            if (two) load(q[1], i + I8S_THREADS);
            __builtin_amdgcn_sched_barrier(0);   // both items' loads in front
            put(q[0]);
            if (two && i + I8S_THREADS < items) put(q[1]);
        }
    }
    // where unit u of K lies from a pixel's place on (past the last: somewhere, the weights there are zeros)
    unsigned *table = reinterpret_cast<unsigned *>(i8s_lds + p.table_at);
    for (int u = tid; u < 4 * chunks; u += I8S_THREADS) {
        const unsigned tap = div31((unsigned) u, p.div_cu), c = (unsigned) u - tap * (unsigned) p.cu;
        const unsigned ti = div31(tap, p.div_kw), tj = tap - ti * (unsigned) p.kw;
        table[u] = u < p.units ? (ti * (unsigned) p.pw + tj) * (unsigned) p.pitch + c * 16u : 0u;
    }
    // this wavefront's chunk on its way from rows of lanes to the matrix instruction's order: its own, so nothing to wait for
    unsigned char *turn = i8s_lds + p.turn_at + wave * I8S_TURN;
    unsigned from[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        const unsigned j = (unsigned) (b * 32 + li), ty = div31(j, p.div_tw), tx = j - ty * (unsigned) p.tw;
        from[b] = (int) ty < p.tr ? (ty * (unsigned) p.stride * (unsigned) p.pw + tx * (unsigned) p.sw) * (unsigned) p.pitch : 0u;
    }
    __syncthreads();

    i32x16 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[b][r] = 0;
    for (int c = wk; c < chunks; c += WK * I8S_RING) {
#pragma unroll
        for (int j = 0; j < I8S_RING; ++j) {
            const int chunk = c + WK * j;
            if (j == 0 || chunk < chunks) {
                unsigned off[2];
#pragma unroll
                for (int z = 0; z < 2; ++z) off[z] = table[4 * chunk + 2 * z + lh];
#pragma unroll
                for (int h = 0; h < 2; ++h) *reinterpret_cast<uint4 *>(turn + (h * 16 + lane / 4) * I8S_TURN_ROW + (lane & 3) * 16) = ring[j].q[h];
                load_a(ring[j], chunk + WK * I8S_RING);
#pragma unroll
                for (int z = 0; z < 2; ++z) {
                    const uint4 w = *reinterpret_cast<const uint4 *>(turn + li * I8S_TURN_ROW + z * 32 + lh * 16);
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        const uint4 v = *reinterpret_cast<const uint4 *>(i8s_lds + from[b] + off[z]);
                        acc[b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, w), __builtin_bit_cast(i32x4, v), acc[b], 0, 0, 0);
                    }
                }
            }
        }
    }

    int *sums = reinterpret_cast<int *>(i8s_lds);   // [part of K][row block][pixel block][register][lane]
    __syncthreads();   // nobody reads pixels or the table any more
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) sums[((wave * NB + b) * 16 + r) * 64 + lane] = acc[b][r];
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this wavefront's part of the activation's table
    __syncthreads();
    float f[PER];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        int sum = 0;
#pragma unroll
        for (int w = 0; w < WK; ++w) sum += sums[w * WM * NB * 1024 + tid + i * I8S_THREADS];
        f[i] = __fmul_rn(__fadd_rn(__fmul_rn((float) sum, p.in_scale), b32[i]), __fdiv_rn(aux[i], 127.0f));
    }
    act_store<TABLE ? EPI_LUT : EPI_GENERIC, TABLE>(f, p.ep, (lds_f32_t) reinterpret_cast<const float *>(i8s_all));
    if constexpr (OUT != I8S_S8) {
        const rsrc_t ry = make_rsrc(reinterpret_cast<float *>(p.y) + y_img, (unsigned) p.M * (unsigned) p.OHW * 4u);
#pragma unroll
        for (int i = 0; i < PER; ++i) {
            if constexpr (OUT == I8S_ADD) f[i] = add_res(f[i], res[i], p.res_relu, (unsigned) y_img + (at[i] >> 2), p.res_body);
            __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(f[i]), ry, at[i], 0, 0);
        }
    }
    if constexpr (OUT == I8S_F32) return;
    if (OUT == I8S_ADD && !p.twin) return;   // uniform
    // int8 NHWC: the workgroup's bytes are turned in LDS so that 16 channels of a pixel leave as one store
    constexpr int ROW = BM + 16;
    const int8_t *out = OUT == I8S_S8 ? reinterpret_cast<const int8_t *>(p.y) : p.twin;
    const float inv = OUT == I8S_S8 ? p.out_inv_scale : p.twin_inv_scale;
    __syncthreads();   // the sums have been read
#pragma unroll
    for (int i = 0; i < PER; ++i) {
        const int v = tid + i * I8S_THREADS, r = v / 64 % 16, j = v / 1024 % NB * 32 + li, ml = v / (1024 * NB) * 32 + 8 * (r / 4) + 4 * lh + r % 4;
        i8s_lds[j * ROW + ml] = (unsigned char) (m0 + ml < p.M ? requant_s8(f[i], inv) : 0);   // padding channels are zeros
    }
    __syncthreads();
    const int groups = (p.M + 15) / 16;
    const rsrc_t ro = make_rsrc(out + img * (long long) p.OHW * groups * 16, (unsigned) p.OHW * (unsigned) groups * 16u);
    for (int u = tid; u < 32 * NB * (BM / 16); u += I8S_THREADS) {
        const int j = u / (BM / 16), g = u % (BM / 16);
        const int ty = (int) div31((unsigned) j, p.div_tw), tx = j - ty * p.tw;
        const bool on = m0 / 16 + g < groups && ty < p.tr && oy0 + ty < p.OH && ox0 + tx < p.OW;
        const uint4 q = *reinterpret_cast<const uint4 *>(i8s_lds + j * ROW + g * 16);
        __builtin_amdgcn_raw_buffer_store_b128(u32x4{q.x, q.y, q.z, q.w}, ro,
                                               on ? ((unsigned) ((oy0 + ty) * p.OW + ox0 + tx) * (unsigned) groups + (unsigned) (m0 / 16 + g)) * 16u : OOB, 0, 0);
    }
}

// The rectangle and the rows: of the shapes with a workgroup for each compute unit at most, the one expected to be fastest.  The terms are
// the values a workgroup quantises or copies, the steps of K one behind the other and all of them, the outputs a thread finishes, and what all
// workgroups together read through the caches: least squares over 390 launches from fp32 (YOLOv8s at batch 1, 2 and 4, 6 % off on average)
// and 585 from int8 (the same, and the 1x1 layers of ResNet-50 and MobileNetV2 at batch 1, 8 and 32, 3 %).
static bool i8small_plan(const onhip_conv_desc_t &d, int OH, int OW, const I8SmallIO &io, I8SmallPlan *out) {
    static const int shapes[4][2] = {{1, 1}, {1, 2}, {1, 4}, {2, 2}};   // pixel blocks, row blocks (2 x 1 and 2 x 4 were never the fastest)
    const int cu = (d.cin + 15) / 16, units = cu * d.kh * d.kw, chunks = (units + 3) / 4;
    const int pitch = (cu | 1) * 16;
    const size_t table = d.has_bias && d.act_type == SILU ? TABLE_BYTES : 0;
    out->us = 1e300;
    for (const auto &shape : shapes) {
        const int nb = shape[0], wm = shape[1], area = 32 * nb, row_tiles = (d.cout + 32 * wm - 1) / (32 * wm), chain = nb * ((chunks + 8 / wm - 1) / (8 / wm));
        if (wm > 1 && 32 * wm >= d.cout + 32) continue;
        const int widths[] = {4, 8, 16, 32, 64, OW, (OW + 1) / 2, (OW + 2) / 3, (OW + 3) / 4};
        for (int tw : widths) {
            tw = std::min(tw, OW);
            if (tw > area) continue;
            const int tr = std::min(area / tw, OH);
            const long long wgs = (long long) d.n * ((OH + tr - 1) / tr) * ((OW + tw - 1) / tw) * row_tiles;
            const long long pixels = ((long long) (tr - 1) * d.stride_h + d.kh) * ((long long) (tw - 1) * d.stride_w + d.kw);
            const long long lds = (long long) table + std::max(pixels * pitch + I8S_WAVES * I8S_TURN + (units + 3LL) * 4, nb * 32768LL);
            if (wgs > 256 || lds > I8S_LDS) continue;
            const double values = (double) (pixels * cu * 16);
            const double us = io.xq ? 3.42 + 0.154e-4 * values + 0.087 * chain + 0.0125 * wm * chunks + (io.res ? 0.70 : 0.49) * nb * wm + wgs * 3e-5 * wm * chunks -
                                          (io.res || io.out_s8 ? 0.0 : 0.2)
                                    : 3.6 + 0.81e-4 * values + 0.149 * chain + 0.0095 * wm * chunks + 0.38 * nb * wm + wgs * (7.3e-8 * values + 4.8e-5 * wm * chunks);
            if (us < out->us) *out = I8SmallPlan{nb, wm, tr, tw, wgs, (size_t) lds, us};
        }
    }
    return out->us < 1e299;
}

// Where one launch takes the place of the other kernels', with a margin of 8 to 10 % against the time expected of those.  From fp32: two or
// three launches of 5.9 us, the K loop of a tile up to where it is cut into slices, fp32 in and out at 4.4 TB/s; a microsecond less without
// a table.  From int8: a launch of 3.4 us (4.3 with a residual operand, half a microsecond more with a table) and a tile's K loop, 2 ns an
// element on the kernel that loads into LDS and 2.9 on the register-staged one, which runs few tiles with a long K (whole: its int8 results are
// never cut).  More workgroups than compute units were never ahead by more than the timing repeats and up to twice as slow.
bool i8small_ok(const onhip_conv_desc_t &d, int OH, int OW, const I8SmallIO &io, I8SmallPlan *plan) {
    const long long in = (long long) d.cin * d.h * d.w, out = (long long) d.cout * OH * OW, units = (long long) (d.cin + 15) / 16 * d.kh * d.kw;
    const bool table = d.has_bias && d.act_type == SILU;
    if (d.group != 1 || d.n > 65535 || in * 4 >= (1LL << 31) || out * 4 >= (1LL << 31) || d.cout * units * 16 >= (1LL << 31) || (io.res && (table || !io.xq)) ||
        !i8small_plan(d, OH, OW, io, plan))
        return false;
    const double k = 16.0 * units;
    if (!io.xq) return plan->us < 0.9 * (5.9 + std::min(0.002 * k, 5.0) + 4e-6 * d.n * (in + out) / 4.4 - (table ? 0.0 : 1.0));
    const long long tiles = (d.cout + 63LL) / 64 * (((long long) d.n * OH * OW + 63) / 64);
    const double other = io.res ? 4.3 + 0.0027 * k : 3.4 + (table ? 0.5 : 0.0) + (tiles < 96 && units >= 128 ? 0.0029 * k : std::min(0.002 * k, 6.6));
    // From a K of some 7000 on, the longer the more tiles there are (130 tiles from 26000), the other kernels cut it into slices, which a launch more
    // adds up (not with a residual operand).  What that takes is fitted to 605 launches (4 % off), and this kernel's own time there, where more than
    // 3 MB of weights go past every workgroup, to 532 (7 %); the choices within 20 % of the faster one and 0.2 % on average (16 % without the rule).
    // 1198 channels under a 7x7 filter, stride 3, on 5 x 5 at batch 4 48 us, 15 in slices; 832 -> 35, 7x7 on 11 x 11, 24 and 12; 154 -> 1146, 7x7
    // and stride 2 on 11 x 11, K 7840 and not cut, 8.0 and 31.6.
    if (k > 7000.0 + 90.0 * (double) tiles && !io.res) {
        const double sliced = 8.55 + 7.7e-5 * k + 1.3e-5 * k * (double) tiles - 0.0836 * (double) tiles + 3.6e-5 * d.cout * ((double) d.n * OH * OW);
        if (1.193 * plan->us - 1.02 + 0.183 * std::max(0.0, 1e-6 * d.cout * k - 3.0) > 0.98 * sliced) return false;
    }
    return plan->us < 0.92 * other;
}

template <int NB, int WM, bool TABLE, bool SRC8, int OUT>
static int i8small_launch_as(const I8SmallParams &p, const I8SmallPlan &plan, hipStream_t stream) {
    static std::atomic<bool> allowed{false};
    if (plan.lds > 64 * 1024 && !allowed.load()) {
        ONHIP_CHECK_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(i8small_kernel<NB, WM, TABLE, SRC8, OUT>), hipFuncAttributeMaxDynamicSharedMemorySize, I8S_LDS));
        allowed.store(true);
    }
    hipLaunchKernelGGL((i8small_kernel<NB, WM, TABLE, SRC8, OUT>), dim3((unsigned) plan.wgs), dim3(I8S_THREADS), plan.lds, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}

template <int NB, int WM>
static int i8small_launch_one(const I8SmallParams &p, const I8SmallIO &io, const I8SmallPlan &plan, hipStream_t stream) {
    const bool table = p.ep.act == SILU;
    if (!p.xq && io.out_s8) return table ? i8small_launch_as<NB, WM, true, false, I8S_S8>(p, plan, stream) : i8small_launch_as<NB, WM, false, false, I8S_S8>(p, plan, stream);
    if (!p.xq) return table ? i8small_launch_as<NB, WM, true, false, I8S_F32>(p, plan, stream) : i8small_launch_as<NB, WM, false, false, I8S_F32>(p, plan, stream);
    if (p.res) return i8small_launch_as<NB, WM, false, true, I8S_ADD>(p, plan, stream);
    if (io.out_s8) return table ? i8small_launch_as<NB, WM, true, true, I8S_S8>(p, plan, stream) : i8small_launch_as<NB, WM, false, true, I8S_S8>(p, plan, stream);
    return table ? i8small_launch_as<NB, WM, true, true, I8S_F32>(p, plan, stream) : i8small_launch_as<NB, WM, false, true, I8S_F32>(p, plan, stream);
}

int i8small_launch(const onhip_conv_desc_t &d, int OH, int OW, const I8SmallPlan &plan, const I8SmallIO &io, const int8_t *packed, const int32_t *bias32,
                   const float *weight_aux, const Epilogue &ep, hipStream_t stream) {
    I8SmallParams p;
    memset(&p, 0, sizeof(p));
    p.x = io.x; p.xq = io.xq; p.y = io.y; p.res = io.res; p.res_relu = io.res_relu; p.res_body = io.res_body; p.twin = io.twin;
    p.twin_inv_scale = io.twin ? 1.0f / d.output_scale : 0.0f; p.out_inv_scale = io.out_s8 ? 1.0f / d.output_scale : 0.0f;
    p.w = packed; p.aux = weight_aux; p.bias32 = d.has_bias ? bias32 : nullptr; p.ep = ep;
    p.in_scale = d.input_scale; p.inv_scale = 1.0f / d.input_scale;
    p.M = d.cout; p.cin = d.cin; p.H = d.h; p.W = d.w; p.HW = d.h * d.w; p.OH = OH; p.OW = OW; p.OHW = OH * OW;
    p.stride = d.stride_h; p.sw = d.stride_w; p.pad_t = d.pad_t; p.pad_l = d.pad_l; p.kw = d.kw;
    p.cu = (d.cin + 15) / 16; p.units = p.cu * d.kh * d.kw;
    p.tr = plan.tr; p.tw = plan.tw;
    p.pr = (plan.tr - 1) * d.stride_h + d.kh; p.pw = (plan.tw - 1) * d.stride_w + d.kw;
    p.pitch = (p.cu | 1) * 16; p.turn_at = p.pr * p.pw * p.pitch; p.table_at = p.turn_at + I8S_WAVES * I8S_TURN;
    p.div_m = make_div31((unsigned) ((d.cout + 32 * plan.wm - 1) / (32 * plan.wm)));
    p.div_tx = make_div31((unsigned) (OW + plan.tw - 1) / plan.tw);
    p.div_ty = make_div31((unsigned) (OH + plan.tr - 1) / plan.tr);
    p.div_pix = make_div31((unsigned) (p.pr * p.pw));
    p.div_pw = make_div31((unsigned) p.pw); p.div_tw = make_div31((unsigned) p.tw);
    p.div_cu = make_div31((unsigned) p.cu); p.div_kw = make_div31((unsigned) p.kw);
    if (plan.nb == 2) return i8small_launch_one<2, 2>(p, io, plan, stream);
    return plan.wm == 1 ? i8small_launch_one<1, 1>(p, io, plan, stream) : plan.wm == 2 ? i8small_launch_one<1, 2>(p, io, plan, stream) : i8small_launch_one<1, 4>(p, io, plan, stream);
}

}  // namespace onhip
