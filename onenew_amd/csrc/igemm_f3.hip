// fp32 implicit GEMM on the 16-bit matrix cores: dispatch, and the kernels for a 1x1 convolution's input and for rows.
#include "igemm_f3_kernel.hpp"

namespace onhip {

int f3_launch_tapc(const IgemmLaunch &cfg, const IgemmProblem &p, hipStream_t stream);     // igemm_f3_conv.hip
int f3_launch_gather(const IgemmLaunch &cfg, const IgemmProblem &p, hipStream_t stream);

// The rows of C normalised in the product's launch: the tile covers all columns, results and parameters are whole 16-byte pieces.
static bool f3_norm_ok(const IgemmLaunch &cfg, const IgemmProblem &p) {
    const RowNorm *r = p.norm;
    return r && cfg.bl == BL_ROWS && cfg.bm == 192 && cfg.bn == 64 && p.res && !p.partial && !p.c_part && p.M <= 192 && p.M >= 32 && p.M % 4 == 0 &&
           p.c_stride_n == p.M && p.ep.act == NOT_ACT &&
           ((reinterpret_cast<uintptr_t>(r->w) | reinterpret_cast<uintptr_t>(r->b) | reinterpret_cast<uintptr_t>(r->y)) & 15) == 0;
}
// (here and not in the header: what launches a kernel there puts a copy of it into every file that includes it)
static int f3_launch_norm(const IgemmLaunch &cfg, const IgemmProblem &p_in, hipStream_t stream) {
    IgemmNormProblem p;
    static_cast<IgemmProblem &>(p) = p_in;
    dim3 grid;
    const int rc = tile_grid<192, 64>(cfg, p, &grid);
    if (rc) return rc;
    p.norm_w = p_in.norm->w; p.norm_b = p_in.norm->b; p.norm_y = p_in.norm->y; p.inv_n = 1.0f / p.M;
    if (f3_alone(cfg, p)) hipLaunchKernelGGL((igemm_f3_kernel<BL_ROWS, 192, 64, 6, 2, true, false, true>), grid, dim3(768), 64 * (p.M + 1) * 4, stream, p);
    else hipLaunchKernelGGL((igemm_f3_kernel<BL_ROWS, 192, 64, 2, 2, true, false, true>), grid, dim3(256), 64 * (p.M + 1) * 4, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    p_in.norm->done = true;
    return ONHIP_OK;
}

int f3_launch(const IgemmLaunch &cfg, const IgemmProblem &p, hipStream_t stream) {
    if (p.M < 1 || p.N < 1 || p.K < 1 || cfg.batch != 1 || cfg.split < 1 || p.dp_tiles || p.arrive || !p.a_split || p.a_split_bytes >= (1LL << 31) ||
        p.b_slice_bytes + 2 * p.b_shift_bytes >= (1LL << 31) || p.c_slice_bytes >= (1LL << 31))
        return set_error(ONHIP_ERR_ARG, "igemm f3: not a problem of this kernel");
    switch (cfg.bl) {
        case BL_GATHER: return f3_launch_gather(cfg, p, stream);
        case BL_PLAIN: return p.res ? f3_launch_tile<BL_PLAIN, true>(cfg, p, stream) : f3_launch_tile<BL_PLAIN, false>(cfg, p, stream);
        case BL_TAPC: return f3_launch_tapc(cfg, p, stream);
        case BL_ROWS:
            if (p.partial) return set_error(ONHIP_ERR_ARG, "igemm f3: no split along K for rows");
            if (f3_norm_ok(cfg, p)) return f3_launch_norm(cfg, p, stream);
            return p.res ? f3_launch_tile<BL_ROWS, true>(cfg, p, stream) : f3_launch_tile<BL_ROWS, false>(cfg, p, stream);
        default: return set_error(ONHIP_ERR_ARG, "igemm f3: unsupported loader %d", cfg.bl);
    }
}

// ---- weights -> the split form ---------------------------------------------------------------------------------------
// element (row, k) of the weights at w[row * s_row + k * s_k]; out [32 rows][16 of K][part][lane (row, half of 8)][8 bf16], zeros beyond
// M rows and K.  A weight that is not finite when scaled has an infinity for its first part, which makes every sum it takes part in
// infinite or NaN, and its own upper and lower half for the others, from which those sums are computed again.
__global__ __launch_bounds__(256) void split_weights_kernel(const float *w, int M, int K, long long s_row, long long s_k, int ksteps, uint4 *out,
                                                            long long total) {
    const long long i = (long long) blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= total) return;
    const int lane = (int) (i % 64);
    const long long t = i / 64;
    const int step = (int) (t % ksteps), blk = (int) (t / ksteps);
    const int row = blk * 32 + lane % 32, k = step * 16 + lane / 32 * 8;
    float x[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) x[j] = row < M && k + j < K ? w[row * s_row + (k + j) * s_k] : 0.0f;
    unsigned part[3][4];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
        const float v = x[j] * F3_SCALE, h = (float) (__bf16) v, r = v - h, m = (float) (__bf16) r;
        const bool finite = h - h == 0.0f;
        const unsigned raw = __float_as_uint(x[j]);
        const unsigned hml[3] = {finite ? __float_as_uint(h) >> 16 : 0x7f80u, finite ? __float_as_uint(m) >> 16 : raw >> 16,
                                 finite ? __float_as_uint((float) (__bf16) (r - m)) >> 16 : raw & 0xffffu};
#pragma unroll
        for (int z = 0; z < 3; ++z) part[z][j / 2] = j % 2 ? part[z][j / 2] | hml[z] << 16 : hml[z];
    }
    uint4 *o = out + t * 192 + lane;
#pragma unroll
    for (int z = 0; z < 3; ++z) o[z * 64] = make_uint4(part[z][0], part[z][1], part[z][2], part[z][3]);
}

int split_weights_launch(const float *w, int M, int K, long long s_row, long long s_k, void *out, hipStream_t stream) {
    const long long total = split_weights_bytes(M, K) / 48;
    hipLaunchKernelGGL(split_weights_kernel, dim3((unsigned) ((total + 255) / 256)), dim3(256), 0, stream, w, M, K, s_row, s_k, (K + 15) / 16,
                       reinterpret_cast<uint4 *>(out), total);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}

}  // namespace onhip
