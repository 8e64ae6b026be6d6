// The order in which the flow head's residual GEMM (flow_res_kernel, dit_batch.hip) walks a K
// slice, with the rule on K that it needs.  Plain C++: the host runs the same code on counters.
#pragma once

namespace ming {

// K slices of a sum for the bias, residual and gelu epilogues: a function of K alone.
constexpr int k_slices(int K) {
    return K >= 2048 && K % (4 * 64) == 0 ? 4 : (K >= 1024 && K % (2 * 64) == 0 ? 2 : 1);
}

// Steps of 32 k in one of a wave's two register sets, by its row and column tiles: what the registers hold.
constexpr int flow_set_steps(int mt, int nt) { return mt * nt > 2 ? 4 : 8; }

// A slice is whole register sets, whatever the tile (the tile is a function of the rows).
constexpr int kFlowSetSteps = 8;
constexpr bool flow_k_fits(int K) { return K % k_slices(K) == 0 && K / k_slices(K) % (32 * kFlowSetSteps) == 0; }

// S steps, a multiple of CH, in two register sets: set 0 takes the even runs of CH steps, set 1 the odd ones, each
// loaded again as soon as it is worked.  flow_first issues the first loads (a single run is loaded twice: no branch
// before the loop).  An odd number of runs ends in the middle of the last turn; runs of four steps never do, and are
// spared the tests (64 sequences: 3803 us with them, 3731 without).
template <int CH>
constexpr bool kWholeTurns = kFlowSetSteps % (2 * CH) == 0;

template <int CH, class Load>
[[gnu::always_inline]] constexpr void flow_first(int S, Load load) {
    load(0, 0);
    load(1, kWholeTurns<CH> || CH < S ? CH : 0);
}
template <int CH, class Load, class Work>
[[gnu::always_inline]] constexpr void flow_turns(int S, Load load, Work work) {
#pragma unroll 1
    for (int s = 0; s < S; s += 2 * CH) {
        work(0);
        if (s + 2 * CH < S) load(0, s + 2 * CH);
        if (kWholeTurns<CH> || s + CH < S) {
            work(1);
            if (s + 3 * CH < S) load(1, s + 3 * CH);
        }
    }
}

}  // namespace ming
