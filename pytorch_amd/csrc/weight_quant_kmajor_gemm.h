// Internal interface of the tiled weight-only GEMM for int8 weights with one scale per column, stored [N, K] or [K, N] (more than
// 32 activation rows); not part of the C ABI.
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace mi355 {

struct WqKmGemmPlan {
    bool ok;                               // the kernel accepts this problem
    bool n_major;                          // the weight is [K, N]
    double us;                             // estimated time
    int wtm;                               // 64 * wtm activation rows per workgroup tile
    int S;                                 // workgroups that share the K range of a tile
    size_t counter_bytes, partial_bytes;   // workspace when S > 1: [arrival counters | partial sums]
};

// `n_major`: the weight is [K, N].  `ldw`: bytes between its columns, of a [K, N] weight between its rows.  Null pointers (the workspace query) count as aligned.  `room`: the workspace that a split of K
// may use.  `own_chunk_counts`: the estimate of a split as if the collecting workgroup read its own chunk back.
__attribute__((visibility("hidden"))) WqKmGemmPlan make_wq_kmajor_gemm_plan(int64_t M, int64_t N, int64_t K, int64_t group_size, int64_t ldw,
                                                                            int64_t ldx, const void *x, const void *w,
                                                                            const void *scale, const void *offset,
                                                                            size_t room = ~(size_t)0, bool n_major = false,
                                                                            bool own_chunk_counts = false);

// Whether the kernel takes such a problem.  Strides that it takes change the plan only where they rule out tall tiles, and its request then
// never grows (200,000 shapes, activation rows 2^22 and more apart).
__attribute__((visibility("hidden"))) bool wq_kmajor_gemm_accepts(int64_t M, int64_t N, int64_t K, int64_t group_size, int64_t ldw, int64_t ldx,
                                                                  const void *x, const void *w, const void *scale, const void *offset,
                                                                  bool n_major = false);

// Launches the kernel; `workspace` holds counter_bytes + partial_bytes when plan.S > 1.
__attribute__((visibility("hidden"))) int launch_wq_kmajor_gemm(const WqKmGemmPlan &plan, const void *x, int act_f16, const void *w,
                                                                const void *scale, const void *offset, const void *bias, void *out, int64_t M,
                                                                int64_t N, int64_t K, int64_t ldx, int64_t ldw, int64_t ldo, void *workspace,
                                                                void *stream);

} // namespace mi355
