// Attention of a DiT block on one wave, shared by its kernels.
#pragma once

#include "common.h"

namespace ming {

constexpr int kMaxL = 8;  // positions per sequence (attention)

// Attention of one (sequence, head) over its L positions on the wave, lane d
// holding dimension d of q, k and v (lanes past head_dim: on = false, adding
// zeros): scores sum_d (q/8) k in f32 (wave sums), p = exp(s - max),
// l = sum p, o[i] = (sum_j p_j v_j) / l, to be rounded once by the caller.
__device__ __forceinline__ void attn_math(const float (&qv)[kMaxL], const float (&kv)[kMaxL],
                                          const float (&vv)[kMaxL], int L, bool on, float (&o)[kMaxL]) {
    const float scale = 1.0f / 8.0f;
#pragma unroll
    for (int i = 0; i < kMaxL; i++)
        if (i < L) {
            const float qd = on ? scale * qv[i] : 0.0f;
            float sc[kMaxL], m = -INFINITY;
#pragma unroll
            for (int j = 0; j < kMaxL; j++)
                if (j < L) {
                    sc[j] = team_sum<kWave>(qd * kv[j]);
                    m = fmaxf(m, sc[j]);
                }
            float l = 0.0f, acc = 0.0f;
#pragma unroll
            for (int j = 0; j < kMaxL; j++)
                if (j < L) {
                    const float p = exp_rep(sc[j] - m);
                    l += p;
                    acc += p * vv[j];
                }
            o[i] = acc / l;
        }
}

}  // namespace ming
