// Attention of one (batch, head) on the 16-bit matrix cores, operands and result fp32, head dimension 64, 65 to 256 tokens: the
// chain of attention.hip (scores = q k^T * scale, Softmax over the keys, context = scores v) with every product as the six partial
// products of three bf16 parts (igemm_f3_kernel.hpp: same parts, same order).
//
// A wavefront owns 32 queries, whose parts it keeps in registers, and walks the keys in tiles of 32: TRANSPOSED scores S^T = k q^T with
// v_mfma_f32_32x32x16_bf16, so that a lane holds one query (column lane % 32) and the 16 keys 8 (r / 4) + 4 (lane / 32) + r % 4 of the tile.
// Registers 8 g .. 8 g + 7 then are, as exponentials, split in place, the B operand of a step of the second product
// out^T += v^T P^T.  k and v come through LDS a tile at a time as three bf16 parts, split by the thread that loads them; v transposed,
// with the keys of a tile in the order that makes a lane half's eight keys of a step one 16-byte read, and its channel rows taken in an order
// that leaves a lane with 32 consecutive channels of its query.  What is subtracted before the exponential is the largest score so far;
// results and sums are only rescaled when a tile exceeds it by 2^8 (the exponentials stay below that), and divided by the sum once.
//
// A pass of the loop is 48 matrix instructions (the scores of tile t + 1, then the second product of tile t) with everything else
// behind them a piece at a time, up to six vector instructions a matrix instruction being free: the split of tile t's exponentials and of
// the next k and v behind the former, the exponentials of tile t + 1 and the loads behind the latter; one barrier.  It is a loop, not unrolled
// over the tiles with all scores in registers, whose 40 KB of code run once and are not there in time.
// What bounds it: two wavefronts a SIMD, whose 21500 cycles of matrix instructions (196 keys) are half of a launch's 45000, because the barrier keeps
// them in step (0.39 of their time is waiting) and nothing covers what lies before the first of them: loads, the split of the queries and the first tile.
// 64 x 3 heads of 196 tokens 22.0 us (23.5
// with q and the result a row a lane), on fp32 matrix instructions (attention.hip) 30.2.  Error against 64 bits (relative, 2-norm; normal operands of a spread of 1 to 3,
// 100 to 256 tokens) 2.5e-7 ... 7.2e-7, there 3.1e-7 ... 9.5e-7; on operands spread over 2^+-4 0.71-0.80 of there, on operands of one sign 0.99-1.03;
// where one key has all the weight, 5e-8 (v as its three parts' sum, rounded on the way) instead of v itself.
//
// Results that are not finite (an operand that is not, or of 2^104 and more, sums of 2^80 and more) are made again from the tensors in
// memory with fp32 matrix instructions, as in igemm_f3_kernel.hpp: a score that is not finite makes its query's results NaN.
#include "igemm_f3_kernel.hpp"

namespace onhip {

struct AttnF3Params {
    const float *q, *k, *v;
    float *o;
    long long qs[3], ks[3], vs[3], os[3];   // element strides of (batch, head, token); the head dimension is contiguous
    int heads, tokens, qblocks;             // qblocks: workgroups per head
    float scale;
};

template <int NW>
__global__ __launch_bounds__(64 * NW, 2) void attention_f3_kernel(const AttnF3Params p) {
    static_assert(NW == 4 || NW == 8, "a tile is staged in two units or one a thread, of k and of v");
    constexpr int NT = 64 * NW, HD = 64, STEPS = HD / 16, UNITS = 8 / NW;
    constexpr int PART = 32 * HD / 8, TILE = 3 * PART;   // 16-byte slots of one part of a tile of k or v, and of a tile
    __shared__ uint4 lds[4 * TILE];                      // two tiles of k, two of v
    // a wavefront's rows of q, later of the result: memory is read and written sixteen lanes to a row of 256 bytes (a row a lane, 64 cycles of
    // the compute unit's address path each, were 2 us of a launch)
    __shared__ uint4 rows[NW][32 * HD / 4];

    // k: [part][key][8 slots of 8 channels], slots exchanged by the row so that 16 rows' reads of one slot cover the banks
    auto k_slot = [](int key, int u) { return key * 8 + (u ^ (key >> 1 & 7)); };
    // v^T: [part][4 slots of 8 keys][channel], channels in an order in which the 16 that a read takes together ({0..7} and {32..39}, or 8, 16, 24
    // more) cover the banks
    auto v_slot = [](int ch, int u) { return u * HD + ((ch & 7) | (ch >> 2 & 8) | (ch << 1 & 48)); };

    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int li = lane & 31, lh = lane >> 5;
    // as attention_f32_kernel: an XCD gets a contiguous run of (head, query block) pairs
    int qblock, bh;
    {
        const int nb = (int) gridDim.x, bid = (int) blockIdx.x;
        const int per = nb >> 3, rmd = nb & 7, xcd = bid & 7, idx = bid >> 3;
        const int lid = xcd * per + (xcd < rmd ? xcd : rmd) + idx;
        bh = lid / p.qblocks;
        qblock = lid - bh * p.qblocks;
    }
    const int b = bh / p.heads, h = bh - b * p.heads;
    const int T = p.tokens, tiles = (T + 31) / 32;
    // the launcher has checked that tokens * token stride stays below 2 GiB
    const rsrc_t rk = make_rsrc(p.k + b * p.ks[0] + h * p.ks[1], RSRC_RANGE);
    const float *v_base = p.v + b * p.vs[0] + h * p.vs[1];
    const unsigned kstride = (unsigned) p.ks[2] * 4, vstride = (unsigned) p.vs[2] * 4;

    // a thread's share of a tile: 4 channels of a key of k, 4 keys of a channel of v; rows past the last key are zeros
    // (two tiles on their way at a time; a tile's parity, where it is given, is that of t: which registers and which part of LDS are then known)
    uint4 kq[2][UNITS];
    float vq[2][UNITS][4];
    auto load_k = [&](int t, auto parity) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < UNITS; ++i) {
            const int key = 32 * t + (tid + i * NT) / 16;
            kq[decltype(parity)::value][i] = buf_load_b128(rk, key < T ? (unsigned) key * kstride + tid % 16 * 16u : OOB, 0);
        }
    };
    auto load_v1 = [&](int t, auto parity, int i, int j) __attribute__((always_inline)) {
        const int key = 32 * t + (wave + i * NW) * 4 + j;   // uniform
        vq[decltype(parity)::value][i][j] = buf_load_f32(make_rsrc(v_base, key < T ? RSRC_RANGE : 0u), (unsigned) lane * 4u, (unsigned) key * vstride);
    };
    auto load_v = [&](int t, auto parity) __attribute__((always_inline)) {
#pragma unroll
        for (int i = 0; i < UNITS; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) load_v1(t, parity, i, j);
    };
    SplitUnit su, sw;
    auto stage_k = [&](auto parity, auto unit, auto phase) __attribute__((always_inline)) {
        constexpr int i = decltype(unit)::value, Q = decltype(phase)::value, P = decltype(parity)::value;
        su.phase<Q>(__uint_as_float(kq[P][i].x), __uint_as_float(kq[P][i].y), __uint_as_float(kq[P][i].z), __uint_as_float(kq[P][i].w));
        if constexpr (Q == 3) {
            uint2 *to = reinterpret_cast<uint2 *>(&lds[P * TILE + k_slot((tid + i * NT) / 16, tid % 16 / 2)]) + tid % 2;
            to[0] = make_uint2(su.h0, su.h1);
            to[2 * PART] = make_uint2(su.m0, su.m1);
            to[4 * PART] = make_uint2(su.l0, su.l1);
        }
    };
    // keys 4 n .. 4 n + 3 of a tile, n = 4 g + 2 a + half, are half a of slot 2 g + half
    auto stage_v = [&](auto parity, auto unit, auto phase) __attribute__((always_inline)) {
        constexpr int i = decltype(unit)::value, Q = decltype(phase)::value, P = decltype(parity)::value;
        sw.phase<Q>(vq[P][i][0], vq[P][i][1], vq[P][i][2], vq[P][i][3]);
        if constexpr (Q == 3) {
            const int n = wave + i * NW;   // uniform
            uint2 *to = reinterpret_cast<uint2 *>(&lds[(2 + P) * TILE + v_slot(lane, n / 4 * 2 + n % 2)]) + n / 2 % 2;
            to[0] = make_uint2(sw.h0, sw.h1);
            to[2 * PART] = make_uint2(sw.m0, sw.m1);
            to[4 * PART] = make_uint2(sw.l0, sw.l1);
        }
    };
    auto stage_all = [&](auto &&stage, auto parity) __attribute__((always_inline)) {
        static_for<UNITS>([&](auto unit) __attribute__((always_inline)) { static_for<4>([&](auto ph) __attribute__((always_inline)) { stage(parity, unit, ph); }); });
    };
    constexpr std::integral_constant<int, 0> EVEN{};
    constexpr std::integral_constant<int, 1> ODD{};

    load_k(0, EVEN);
    __builtin_amdgcn_sched_barrier(0);   // the loads in this order, so that a pass waits for the older ones alone
    const int q0 = (qblock * NW + wave) * 32, query = q0 + li;
    const bool active = q0 < T;   // uniform: a wavefront without queries only helps with the operands
    const float *qb = p.q + b * p.qs[0] + h * p.qs[1] + (long long) (query < T ? query : T - 1) * p.qs[2];   // rows past the last: unused
    uint4 *const mine = rows[wave];
    auto row_slot = [](int row, int u) { return row * 16 + (u ^ (row & 15)); };   // 16 bytes `u` of a row
    uint4 qf[2 * STEPS];
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i) {
        const int row = q0 + 4 * i + lane / 16;
        qf[i] = *reinterpret_cast<const uint4 *>(p.q + b * p.qs[0] + h * p.qs[1] + (long long) (row < T ? row : T - 1) * p.qs[2] + lane % 16 * 4);
    }
    __builtin_amdgcn_sched_barrier(0);
    load_k(1, ODD);
    load_v(0, EVEN);
    load_v(1, ODD);
    __builtin_amdgcn_sched_barrier(0);
    stage_all(stage_k, EVEN);
    load_k(2, EVEN);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i) mine[row_slot(4 * i + lane / 16, lane % 16)] = qf[i];
#pragma unroll
    for (int i = 0; i < 2 * STEPS; ++i) qf[i] = mine[row_slot(li, i / 2 * 4 + 2 * lh + i % 2)];
    uint4 qp[STEPS][3];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
        SplitUnit u, w;
        const float4 lo = __builtin_bit_cast(float4, qf[2 * s]), hi = __builtin_bit_cast(float4, qf[2 * s + 1]);
        static_for<4>([&](auto ph) __attribute__((always_inline)) {
            u.phase<decltype(ph)::value>(lo.x, lo.y, lo.z, lo.w);
            w.phase<decltype(ph)::value>(hi.x, hi.y, hi.z, hi.w);
        });
        qp[s][0] = make_uint4(u.h0, u.h1, w.h0, w.h1);
        qp[s][1] = make_uint4(u.m0, u.m1, w.m0, w.m1);
        qp[s][2] = make_uint4(u.l0, u.l1, w.l0, w.l1);
    }
    stage_all(stage_k, ODD);
    load_k(3, ODD);
    __builtin_amdgcn_sched_barrier(0);
    stage_all(stage_v, EVEN);
    load_v(2, EVEN);
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    f32x16 o[2], x, e;   // results; scores of a tile; exponentials of the tile before it
    uint4 f[2][3], pp[2][3];
    float run = 0.0f, sum = 0.0f, factor = 1.0f;
    bool grown = false;
    const float c = p.scale * 1.44269504088896340736f * F3_UNSCALE;   // exp(x) as exp2(x log2 e) with the hardware's exp2
    auto channel = [](int m, int d) { return 32 * (m / 4 % 2) + 16 * d + 4 * (m / 8) + m % 4; };   // that row m of tile d stands for
    auto key_of = [&](int t, int r) __attribute__((always_inline)) { return 32 * t + 8 * (r / 4) + 4 * lh + r % 4; };
    auto read_k = [&](uint4 (&to)[3], int parity, int st) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 3; ++z) to[z] = lds[parity * TILE + z * PART + k_slot(li, 2 * st + lh)];
    };
    auto read_v = [&](uint4 (&to)[3], int parity, int g, int d) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 3; ++z) to[z] = lds[(2 + parity) * TILE + z * PART + v_slot(channel(li, d), 2 * g + lh)];
    };
    auto largest = [&](int t) __attribute__((always_inline)) {
        if (32 * t + 32 > T) {   // uniform: keys past the last count as minus infinity
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = key_of(t, r) < T ? x[r] : -INFINITY;
        }
        float mx = x[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) mx = fmaxf(mx, x[r]);
        return __fmul_rn(fmaxf(mx, __shfl_xor(mx, 32, 64)), c);
    };
    auto exponential = [&](int r) __attribute__((always_inline)) {
        e[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(x[r], c, -run));
        sum += e[r];
    };
    // phases 0 .. 15: the four units of e
    auto split_e = [&](auto phase) __attribute__((always_inline)) {
        constexpr int Q = decltype(phase)::value % 4, u = decltype(phase)::value / 4, g = u / 2;
        su.phase<Q, false>(e[4 * u], e[4 * u + 1], e[4 * u + 2], e[4 * u + 3]);
        if constexpr (Q == 3 && u % 2 == 0) {
            pp[g][0].x = su.h0; pp[g][0].y = su.h1; pp[g][1].x = su.m0; pp[g][1].y = su.m1; pp[g][2].x = su.l0; pp[g][2].y = su.l1;
        } else if constexpr (Q == 3) {
            pp[g][0].z = su.h0; pp[g][0].w = su.h1; pp[g][1].z = su.m0; pp[g][1].w = su.m1; pp[g][2].z = su.l0; pp[g][2].w = su.l1;
        }
    };
    if (active) {
#pragma unroll
        for (int r = 0; r < 16; ++r) o[0][r] = o[1][r] = x[r] = 0.0f;
        read_k(f[0], 0, 0);
        static_for<STEPS>([&](auto step) __attribute__((always_inline)) {
            constexpr int st = decltype(step)::value;
            if constexpr (st + 1 < STEPS) read_k(f[(st + 1) & 1], 0, st + 1);
            static_for<F3_PRODUCTS>([&](auto pr) __attribute__((always_inline)) { mma_bf16(x, f[st & 1][f3_pa(pr)], qp[st][f3_pb(pr)]); });
        });
        run = largest(0);
#pragma unroll
        for (int r = 0; r < 16; ++r) exponential(r);
        read_k(f[0], 1, 0);
    }
    __syncthreads();   // k of the first tile is read: the first pass writes over it
    // Everything of a pass but its products: k of tile t + 2 and v of tile t + 1 into the buffers of k of tile t and v of tile t - 1, which everybody has
    // read before the last barrier, and the loads behind them.  Tiles past the last are zeros.
    auto stage = [&](int t, auto parity, auto slot) __attribute__((always_inline)) {
        constexpr int S = decltype(slot)::value;   // 0 .. 7
        constexpr std::integral_constant<int, 1 - decltype(parity)::value> next{};
        if constexpr (UNITS == 1) {
            if constexpr (S < 4) stage_k(parity, EVEN, slot);
            else stage_v(next, EVEN, std::integral_constant<int, S - 4>{});
        } else {
            stage_k(parity, std::integral_constant<int, S / 4>{}, std::integral_constant<int, S % 4>{});
            stage_v(next, std::integral_constant<int, S / 4>{}, std::integral_constant<int, S % 4>{});
        }
        if constexpr (S == 4) load_k(t + 4, parity);
    };
    // v's loads one at a time: all wavefronts' at once are some hundred cycles in which none of them goes on
    auto load_behind = [&](int t, auto parity, auto slot) __attribute__((always_inline)) {
        constexpr int S = decltype(slot)::value, EACH = 16 / (4 * UNITS);
        constexpr std::integral_constant<int, 1 - decltype(parity)::value> next{};
        if constexpr (S < 16 && S % EACH == 0) load_v1(t + 3, next, S / EACH / 4, S / EACH % 4);
    };
    constexpr int HALF = STEPS * F3_PRODUCTS;   // products of either kind a pass
    // two passes a trip, the second one's parity odd
    auto passes = [&](auto &&pass) __attribute__((always_inline)) {
        for (int t = 0; t + 1 < tiles; t += 2) {
            pass(t, EVEN);
            if (t + 2 >= tiles) break;
            pass(t + 1, ODD);
        }
    };
    if (!active) {   // a loop of its own: next to the other, what both do first would wait for its loads at the head of a pass
        passes([&](int t, auto parity) __attribute__((always_inline)) {
            static_for<8>([&](auto s) __attribute__((always_inline)) { stage(t, parity, s); });
            static_for<16>([&](auto s) __attribute__((always_inline)) { load_behind(t, parity, s); });
            __syncthreads();
        });
        return;
    }
    passes([&](int t, auto parity) __attribute__((always_inline)) {
        constexpr int P = decltype(parity)::value;
#pragma unroll
        for (int r = 0; r < 16; ++r) x[r] = 0.0f;
        static_for<HALF>([&](auto slot) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value, st = S / F3_PRODUCTS, pr = S % F3_PRODUCTS;
            __builtin_amdgcn_sched_barrier(0);
            mma_bf16(x, f[st & 1][f3_pa(pr)], qp[st][f3_pb(pr)]);
            if constexpr (pr == 0) {
                if constexpr (st + 1 < STEPS) read_k(f[(st + 1) & 1], 1 - P, st + 1);
                else read_v(f[0], P, 0, 0);
            }
            if constexpr (S < 16) split_e(slot);
            else stage(t, parity, std::integral_constant<int, S - 16>{});
        });
        static_for<HALF>([&](auto slot) __attribute__((always_inline)) {
            constexpr int S = decltype(slot)::value, m = S / F3_PRODUCTS, pr = S % F3_PRODUCTS, d = m % 2;
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (S == HALF - F3_PRODUCTS) {   // the last operands are read, k of tile t + 2 and v of tile t + 1 written
                __syncthreads();
                __builtin_amdgcn_sched_barrier(0);
            }
            mma_bf16(o[d], f[m & 1][f3_pa(pr)], pp[m / 2][f3_pb(pr)]);
            if constexpr (pr == 0) {
                if constexpr (m < 3) read_v(f[(m + 1) & 1], P, (m + 1) / 2, (m + 1) % 2);
                else read_k(f[0], P, 0);
            }
            if constexpr (S == 2) {
                const float top = largest(t + 1);
                grown = __builtin_amdgcn_ballot_w64(top > run + 8.0f) != 0ull;
                if (grown) {   // uniform
                    const float next = fmaxf(run, top);
                    factor = __builtin_amdgcn_exp2f(__fsub_rn(run, next));
                    sum = __fmul_rn(sum, factor);
                    run = next;
                }
            }
            if constexpr (S >= 4 && S < 20) exponential(S - 4);
            load_behind(t, parity, slot);
        });
        __builtin_amdgcn_sched_barrier(0);
        if (grown) {
#pragma unroll
            for (int d = 0; d < 2; ++d)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[d][r] = __fmul_rn(o[d][r], factor);
        }
    });
    // the last tile's second product
    static_for<16>([&](auto phase) __attribute__((always_inline)) { split_e(phase); });
    read_v(f[0], (tiles - 1) & 1, 0, 0);
    static_for<4>([&](auto mini) __attribute__((always_inline)) {
        constexpr int m = decltype(mini)::value;
        if constexpr (m < 3) read_v(f[(m + 1) & 1], (tiles - 1) & 1, (m + 1) / 2, (m + 1) % 2);
        static_for<F3_PRODUCTS>([&](auto pr) __attribute__((always_inline)) { mma_bf16(o[m % 2], f[m & 1][f3_pa(pr)], pp[m / 2][f3_pb(pr)]); });
    });
    sum += __shfl_xor(sum, 32, 64);
    const float inv = 1.0f / sum;
    float probe = (sum + inv) * 0.0f;   // stays zero while everything is finite
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            probe = __builtin_fmaf(o[d][r], 0.0f, probe);
            o[d][r] = __fmul_rn(o[d][r] * (1.0f / F3_SCALE), inv);   // v alone was scaled
        }
    if (__builtin_amdgcn_ballot_w64(probe != probe) != 0ull) {   // uniform
        // scores made anew for the maximum, the sum and the product
        auto scores = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = 0.0f;
            const int key = 32 * t + li;
#pragma unroll 1
            for (int j = 0; j < HD; j += 2) {
                const float kv = buf_load_f32(rk, key < T ? (unsigned) key * kstride + (unsigned) (j + lh) * 4u : OOB, 0);
                x = __builtin_amdgcn_mfma_f32_32x32x2f32(kv, qb[j + lh], x, 0, 0, 0);
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) x[r] = key_of(t, r) < T ? __fmul_rn(x[r], p.scale) : -INFINITY;
        };
        f32x16 again[2];
        float top = -INFINITY, total = 0.0f;
#pragma unroll 1
        for (int t = 0; t < tiles; ++t) {
            scores(t);
#pragma unroll
            for (int r = 0; r < 16; ++r) top = fmaxf(top, x[r]);
        }
        top = fmaxf(top, __shfl_xor(top, 32, 64));
        auto shifted = [&](float v) __attribute__((always_inline)) { return __builtin_amdgcn_exp2f(__fmul_rn(__fsub_rn(v, top), 1.44269504088896340736f)); };
#pragma unroll 1
        for (int t = 0; t < tiles; ++t) {
            scores(t);
#pragma unroll
            for (int r = 0; r < 16; ++r) total += shifted(x[r]);
        }
        total += __shfl_xor(total, 32, 64);
        const float inv2 = 1.0f / total;
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) again[d][r] = 0.0f;
#pragma unroll 1
        for (int t = 0; t < tiles; ++t) {
            scores(t);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = key_of(t, r);   // the two lane halves hold one key each
                const float prob = __fmul_rn(shifted(x[r]), inv2);
#pragma unroll
                for (int d = 0; d < 2; ++d) {
                    const float vv = buf_load_f32(make_rsrc(v_base, RSRC_RANGE), key < T ? (unsigned) key * vstride + (unsigned) channel(li, d) * 4u : OOB, 0);
                    again[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(vv, prob, again[d], 0, 0, 0);
                }
            }
        }
#pragma unroll
        for (int d = 0; d < 2; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[d][r] = o[d][r] * 0.0f != 0.0f ? again[d][r] : o[d][r];
    }
#pragma unroll
    for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < 4; ++i)
            mine[row_slot(li, 8 * lh + 4 * d + i)] = make_uint4(__float_as_uint(o[d][4 * i]), __float_as_uint(o[d][4 * i + 1]),
                                                                __float_as_uint(o[d][4 * i + 2]), __float_as_uint(o[d][4 * i + 3]));
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int row = q0 + 4 * i + lane / 16;
        if (row < T)
            *reinterpret_cast<uint4 *>(p.o + b * p.os[0] + h * p.os[1] + (long long) row * p.os[2] + lane % 16 * 4) = mine[row_slot(4 * i + lane / 16, lane % 16)];
    }
}

template <int NW>
static int attention_f3_launch_one(AttnF3Params &p, int batch, hipStream_t stream) {
    p.qblocks = (p.tokens + 32 * NW - 1) / (32 * NW);
    hipLaunchKernelGGL((attention_f3_kernel<NW>), dim3((unsigned) (p.qblocks * batch * p.heads)), dim3(64 * NW), 0, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}

// Head dimension 64; a scale for which neither it nor its product with the sums' unscaling leaves the normal numbers; more than 64 tokens; and more
// 64-query workgroups of attention.hip than compute units.  Up to one each, that kernel's 16 queries a wavefront reach four times the SIMDs: 16 x 3
// heads of 129 tokens 9.9 us there and 12.7 here, 3 heads of 196 11.7 and 14.5; 48 x 3 of 100 12.3 and 10.5, 64 x 3 of 196 30.2 and 22.0,
// 48 x 3 of 225 36.2 and 22.9.  Up to 64 tokens half of the wavefronts here and more have no queries, and two tiles of keys do not pay for the start: 260
// heads of 64 tokens 9.0 us there and 10.7 here, 768 of 64 14.1 and 17.1, of 33 11.4 and 15.4, of 16 7.4 and 11.1, 1536 of one 9.1 and 17.1 (17 to 32
// tokens of 260 to 512 heads are level); of more than 64, 130 to 2048 heads take 0.55-0.99 of the time here.
bool attention_f3_ok(const onhip_attention_desc_t &d) {
    return d.head_dim == 64 && d.tokens > 64 && d.scale >= 0x1p-60f && d.scale <= 0x1p60f && (long long) d.batch * d.heads * ((d.tokens + 63) / 64) > 256;
}

int attention_f3_launch(const onhip_attention_desc_t &d, const float *q, const float *k, const float *v, float *out, hipStream_t stream) {
    AttnF3Params p;
    p.q = q; p.k = k; p.v = v; p.o = out;
    for (int i = 0; i < 3; ++i) {
        p.qs[i] = d.q_strides[i]; p.ks[i] = d.k_strides[i]; p.vs[i] = d.v_strides[i]; p.os[i] = d.out_strides[i];
    }
    p.heads = d.heads;
    p.tokens = d.tokens;
    p.scale = d.scale;
    // Eight wavefronts share the tiles where the heads alone give half of the compute units a workgroup (64 x 3 heads of 196 tokens 23.5 us before the
    // rows went through LDS, with four 25.3); fewer heads take four, for twice the workgroups (24 x 3 of 256 tokens 19.0 and 22.6).
    const bool wide = d.tokens > 128 && d.batch * d.heads >= 128;
    return wide ? attention_f3_launch_one<8>(p, d.batch, stream) : attention_f3_launch_one<4>(p, d.batch, stream);
}

}  // namespace onhip
