// Gemm  out[m][n] = sum_k a[m][k] * w[n][k] + bias[n]  in fp32 for the rows of a batch (gfx950): a classifier's last layer.
// Reference: device/x86/Gemm/gemm.c:9-79.
//
// What bounds it: the weights, read once (8 MB for 2048 -> 1000 features, 2 us), behind one trip to memory and a launch.  So every
// compute unit gets a share of them, K is cut over the wavefronts of a workgroup instead of walked by one, and a wavefront asks for
// several steps of both operands before its first multiply-add.  Sums in a fixed order: the same bits on every run.
//
// Measured, us a launch in a graph of twenty, 2048 -> 1000 (1280 -> 1000) features: up to 8 rows, against one wavefront per column with
// a step in flight: 1 row 2.7 (2.6); in a pass of ResNet-50 at batch 1 7.8 before, 8 rows of MobileNetV2 16 before, 4.1 now.  More rows,
// against the convolution kernels on one-pixel images, whose loads of 16 images touch 16 cache lines for 4 bytes each: 9 rows
// 14.5 -> 7.7 (10.2 -> 6.1), 32 rows 20.6 -> 9.0 (14.1 -> 7.0), 64 rows 20.7 -> 9.2; 192 -> 1000 at 64 rows 4.8 -> 3.4.
#include <algorithm>

#include "igemm_kernel.hpp"

namespace onhip {

// ---- up to 8 rows of A: vector arithmetic.  A workgroup owns COLS columns, its four wavefronts take 256 of K in turn, two turns in
// flight; the COLS * ROWS sums of a lane meet in a tree that halves their number with every exchange.
constexpr int NT_COLS = 4;

template <int ROWS, bool VEC>
__global__ __launch_bounds__(256) void gemm_nt_kernel(int M, int K, int N, const float *a, const float *w, const float *bias, float *out) {
    constexpr int S = NT_COLS * ROWS;
    __shared__ float s_sum[4][S];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n0 = blockIdx.x * NT_COLS;
    a += (long long) blockIdx.y * ROWS * K;
    out += (long long) blockIdx.y * ROWS * N;
    M -= blockIdx.y * ROWS;
    struct Turn { float w[NT_COLS][4], a[ROWS][4]; };
    // rows are scalar: each has a descriptor of what is left of it from k on, so operands of any size are in reach and what is past
    // the end comes as zeros
    auto get = [&](float *v, const float *base, int row, int rows, long long k) __attribute__((always_inline)) {
        const rsrc_t r = make_rsrc(base + (long long) row * K + k, row < rows && k < K ? (unsigned) min(K - k, 256LL) * 4u : 0u);
        if constexpr (VEC) {
            const uint4 q = buf_load_b128(r, lane * 16, 0);
            v[0] = __uint_as_float(q.x); v[1] = __uint_as_float(q.y); v[2] = __uint_as_float(q.z); v[3] = __uint_as_float(q.w);
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = buf_load_f32(r, lane * 4, 256 * e);
        }
    };
    auto load = [&](Turn &t, long long k) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < NT_COLS; ++c) get(t.w[c], w, n0 + c, N, k);
#pragma unroll
        for (int r = 0; r < ROWS; ++r) get(t.a[r], a, r, M, k);
    };
    float acc[S];
#pragma unroll
    for (int i = 0; i < S; ++i) acc[i] = 0.0f;
    for (long long k0 = wave * 256; k0 < K; k0 += 2048) {
        Turn t[2];
        load(t[0], k0);
        load(t[1], k0 + 1024);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay in front
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int i = 0; i < S; ++i) acc[i] = fmaf(t[j].a[i / NT_COLS][e], t[j].w[i % NT_COLS][e], acc[i]);
    }
    // after step s a lane keeps the half of its sums that its bit s names; with one sum left, the rest is a butterfly
    int mine = 0;
#pragma unroll
    for (int s = 0; s < 6; ++s) {
        const int bit = 1 << s, have = S >> s;
        const bool up = lane & bit;
        if (have > 1) {
#pragma unroll
            for (int i = 0; i < have / 2; ++i) {
                // values, not places: a choice between two elements would be an index at run time
                const float lo = acc[i], hi = acc[i + have / 2];
                const float give = up ? +lo : +hi, keep = up ? +hi : +lo;
                acc[i] = keep + __shfl_xor(give, bit, 64);
            }
            mine += up ? have / 2 : 0;
        } else {
            acc[0] += __shfl_xor(acc[0], bit, 64);
        }
    }
    if (lane < S) s_sum[wave][mine] = acc[0];
    __syncthreads();
    const int i = threadIdx.x, m = i / NT_COLS, n = n0 + i % NT_COLS;
    if (i < S && m < M && n < N)
        out[(long long) m * N + n] = __fadd_rn(__fadd_rn(__fadd_rn(s_sum[0][i], s_sum[1][i]), __fadd_rn(s_sum[2][i], s_sum[3][i])), bias[n]);
}

// ---- more rows: 16 columns x 16 rows on fp32 matrix instructions.  A workgroup of 16 wavefronts owns such a tile, wavefront v the
// steps v, v + 16, ... of 32 K; a lane's 16-byte loads are four of K of its row, so the rows of a step are whole 128-byte lines.
constexpr int MT_WAVES = 16, MT_RING = 4;

__global__ __launch_bounds__(64 * MT_WAVES) void gemm_nt_mfma_kernel(int M, int K, int N, const float *a, const float *w, const float *bias, float *out,
                                                                     int m_tiles) {
    __shared__ float s_sum[MT_WAVES][256 + 16];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    // workgroups go round the eight XCDs: those that read the same weights are neighbours on one of them
    const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
    const int m0 = slot % m_tiles * 16, n0 = (slot / m_tiles * 8 + xcd) * 16;
    if (n0 >= N) return;
    const int lc = lane & 15, lg = lane >> 4;
    const rsrc_t ra = make_rsrc(a, (unsigned) M * (unsigned) K * 4u), rw = make_rsrc(w, (unsigned) N * (unsigned) K * 4u);
    struct Step { uint4 w[2], a[2]; };
    auto load = [&](Step &s, int step) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 2; ++z) {
            const int k = step * 32 + z * 16 + lg * 4;   // K is a multiple of 4: inside the row or past it as a whole
            s.w[z] = buf_load_b128(rw, k < K && n0 + lc < N ? ((unsigned) (n0 + lc) * (unsigned) K + (unsigned) k) * 4u : OOB, 0);
            s.a[z] = buf_load_b128(ra, k < K && m0 + lc < M ? ((unsigned) (m0 + lc) * (unsigned) K + (unsigned) k) * 4u : OOB, 0);
        }
    };
    f32x4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
    auto multiply = [&](const Step &s) __attribute__((always_inline)) {
#pragma unroll
        for (int z = 0; z < 2; ++z)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                auto f = [&](const uint4 &q) { return __uint_as_float(e == 0 ? q.x : e == 1 ? q.y : e == 2 ? q.z : q.w); };
                acc = __builtin_amdgcn_mfma_f32_16x16x4f32(f(s.w[z]), f(s.a[z]), acc, 0, 0, 0);
            }
    };
    const int steps = (K + 31) / 32;
    for (int s = wave; s < steps; s += MT_WAVES * MT_RING) {
        Step ring[MT_RING];
#pragma unroll
        for (int j = 0; j < MT_RING; ++j) load(ring[j], s + MT_WAVES * j);
        __builtin_amdgcn_sched_barrier(0);   // the loads stay in front
#pragma unroll
        for (int j = 0; j < MT_RING; ++j)
            if (j == 0 || s + MT_WAVES * j < steps) multiply(ring[j]);
    }
    // a lane holds four neighbouring columns of one row
#pragma unroll
    for (int r = 0; r < 4; ++r) s_sum[wave][lc * 17 + lg * 4 + r] = acc[r];
    __syncthreads();
    const int i = threadIdx.x, m = m0 + i / 16, n = n0 + i % 16;
    if (i < 256 && m < M && n < N) {
        const int at = i / 16 * 17 + i % 16;
        float v = s_sum[0][at];
#pragma unroll
        for (int j = 1; j < MT_WAVES; ++j) v = __fadd_rn(v, s_sum[j][at]);
        out[(long long) m * N + n] = __fadd_rn(v, bias[n]);
    }
}

template <int ROWS, bool VEC>
static void gemm_nt_rows(int m, int k, int n, const float *a, const float *w, const float *bias, float *out, hipStream_t stream) {
    constexpr int MOST = ROWS * 32768;   // rows a launch's second grid dimension holds
    for (; m > 0; m -= MOST, a += (long long) MOST * k, out += (long long) MOST * n)
        hipLaunchKernelGGL((gemm_nt_kernel<ROWS, VEC>), dim3((n + NT_COLS - 1) / NT_COLS, (std::min(m, MOST) + ROWS - 1) / ROWS), dim3(256), 0, stream,
                           std::min(m, MOST), k, n, a, w, bias, out);
}
template <bool VEC>
static void gemm_nt_few(int m, int k, int n, const float *a, const float *w, const float *bias, float *out, hipStream_t stream) {
    if (m == 1) gemm_nt_rows<1, VEC>(m, k, n, a, w, bias, out, stream);
    else if (m == 2) gemm_nt_rows<2, VEC>(m, k, n, a, w, bias, out, stream);
    else if (m <= 4) gemm_nt_rows<4, VEC>(m, k, n, a, w, bias, out, stream);
    else gemm_nt_rows<8, VEC>(m, k, n, a, w, bias, out, stream);
}

// The kernel on matrix instructions: 16-byte loads of whole operands by 32-bit offsets, and a compute unit for each workgroup.  With a
// second round of workgroups the other kernels, which share operands among more columns, are ahead: 2048 -> 1000 at 96 rows (378
// workgroups) 16.6 against 14.7 us, 4096 -> 4096 at 16 rows (256) 17.4 against 38, at 24 rows (512) 31 against 24.5.  Up to 8 rows it
// takes 6.3 to 7.6 us where the vector kernel takes 2.7 to 4.1.
// A workgroup walks all of K, 1.4 to 3 ns an element, slowest with rows that start at the same place of a cache line; the convolution kernels
// cut a long K into slices and are then bound by the weights: 25088 -> 512 at 16 rows 88 against 25 us, 8192 -> 2048 31 against 25, 4096 -> 512 at
// 64 rows 16.9 against 12.4, but 4096 -> 4096 at 16 rows 19.3 and 25.1, 2544 -> 1641 at 21 rows 10.0 and 13.2, 3992 -> 706 at 65 12.7 and 23.3.
// Both are fitted to 1121 launches of 9 to 160 rows, 10 to 5000 columns and K of 1025 to 26000, on weights in the L2s and beyond them; the
// choices are 0.4 % above the faster one.
bool gemm_nt_mfma_ok(int m, int k, int n, const float *a, const float *w) {
    const long long lim = 1LL << 29;
    if (k % 4 || ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) & 15) || (long long) m * k >= lim || (long long) n * k >= lim ||
        (long long) m * n >= lim || (long long) ((m + 15) / 16) * ((n + 15) / 16) > 256)
        return false;
    const double mb = 4e-6 * n * k, lines = k % 32 ? 1.0 : k <= 2048 ? 1.15 : 1.25;
    const double us = lines * (3.0 + k * (0.00141 + 6.3e-5 * std::min(m, 16)) + 0.088 * mb), other = 6.85 + 0.00054 * k + mb * (0.17 + 0.0058 * m) + 0.0123 * m;
    return k <= 1024 || us < other;
}

int gemm_nt_launch(int m, int k, int n, const float *a, const float *w, const float *bias, float *out, hipStream_t stream) {
    if (m > 8 && gemm_nt_mfma_ok(m, k, n, a, w)) {
        const int m_tiles = (m + 15) / 16, n_groups = ((n + 15) / 16 + 7) / 8;
        hipLaunchKernelGGL(gemm_nt_mfma_kernel, dim3(n_groups * 8 * m_tiles), dim3(64 * MT_WAVES), 0, stream, m, k, n, a, w, bias, out, m_tiles);
    } else if (k % 4 == 0 && (reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(w)) % 16 == 0) {
        gemm_nt_few<true>(m, k, n, a, w, bias, out, stream);
    } else {
        gemm_nt_few<false>(m, k, n, a, w, bias, out, stream);
    }
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}

}  // namespace onhip
