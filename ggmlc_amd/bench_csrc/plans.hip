// libgq's size-dependent launch plans for tests on the host (libgqbench.so, outside libgq's
// ABI): the same headers, asked without a device.
#include "../csrc/plans.h"

// out: 32-token tiles per workgroup, K splits, stages per split, stages per segment
extern "C" void gqbench_gemm_q8_plan(int type, int64_t N, int64_t K, int64_t M, size_t part_bytes, int64_t ncu,
                                     int* out) {
    const gq::GemmQ8Plan p = gq::plan_gemm_q8(type, N, K, M, part_bytes, ncu);
    out[0] = p.mt, out[1] = p.ks, out[2] = p.sps, out[3] = p.seg;
}

extern "C" double gqbench_fp16_pair_chain(int64_t N, int64_t K, int64_t M, int64_t ncu) {
    return gq::fp16_pair_sums(N, K, M, ncu).chain;
}

// out: 32-query sub-tiles per workgroup, key splits over workgroups
extern "C" void gqbench_attn_pre_plan(int64_t NQ, int64_t Hkv, int64_t n_kv, int64_t most, int* out) {
    const gq::AttnPrePlan p = gq::plan_attn_pre(NQ, Hkv, n_kv, most);
    out[0] = p.nqw, out[1] = p.ks;
}
