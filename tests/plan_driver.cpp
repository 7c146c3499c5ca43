// Test driver: plain-C doors onto the rules by which libtfq.so chooses kernels, which need no GPU.  Built by
// __graft_entry__.build() with hipcc, host side only.
#include "../transformers-fusion_amd/csrc/tfq_internal.hpp"

namespace {
// a matrix as the rules see it: no memory behind it
tfq_weight matrix(int fmt, int64_t N, int64_t K) {
    tfq_weight w{};
    w.fmt = (uint8_t)fmt;
    w.N = N;
    w.K = K;
    const int f = tfq::canonical(fmt);
    w.layout = f == TFQ_Q_4 || f == TFQ_Q_G_6 ? TFQ_LAYOUT_WIRE : TFQ_LAYOUT_TILED16;
    size_t block = 0;
    tfq_block_bytes((uint8_t)fmt, 256, &block);
    w.bytes = (size_t)N * (size_t)(K / 256) * block;
    w.dev_bytes = (size_t)(N + 15) / 16 * 16 * (size_t)(K / 256) * block;
    return w;
}
}  // namespace

extern "C" {

// the integer tile kernel's plans with this much scratch, at most `cap` of them, and the one that is taken
int drv_gemm_exact_plans(int fmt, int64_t N, int64_t K, int x_dtype, int M, size_t scratch, int matrices, int cap, tfq::GemmExactPlan* all,
                         tfq::GemmExactPlan* taken) {
    const tfq_weight w = matrix(fmt, N, K);
    *taken = tfq::gemm_exact_plan(&w, x_dtype, M, scratch, matrices);
    const std::vector<tfq::GemmExactPlan> v = tfq::gemm_exact_plans(&w, x_dtype, M, scratch, matrices);
    for (int i = 0; i < cap && i < (int)v.size(); ++i) all[i] = v[i];
    return (int)v.size();
}

int drv_gemm_takes_exact(int fmt, int64_t N, int64_t K, int x_dtype, int M, size_t scratch) {
    const tfq_weight w = matrix(fmt, N, K);
    return tfq::gemm_takes_exact(&w, x_dtype, M, scratch);
}

size_t drv_gemm_scratch_bytes(int fmt, int64_t N, int64_t K, int x_dtype, int M) {
    const tfq_weight w = matrix(fmt, N, K);
    return tfq::gemm_scratch_bytes(&w, x_dtype, M);
}

// whether tfq_mlp_step of these sizes has gate and up in one launch of the integer tile kernel
int drv_mlp_pairs(int fmt, int64_t N, int64_t K, int x_dtype, int M) {
    const tfq_weight w = matrix(fmt, N, K);
    return M > 4 && tfq::gemm_exact_pair_serves(&w, &w, x_dtype, M) && tfq::gemm_pair_pays(&w, x_dtype, M);
}

// one to sixteen rows: what serves best, and what the decode kernels alone use
size_t drv_gemv_rows_scratch_bytes(int fmt, int64_t N, int64_t K, int x_dtype, int B, size_t* decode) {
    const tfq_weight w = matrix(fmt, N, K);
    *decode = tfq::gemv_split_bytes(&w);
    return tfq::gemv_rows_scratch_bytes(&w, x_dtype, B);
}

}  // extern "C"
