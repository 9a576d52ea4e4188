// How the wavefronts of a few-rows product share the k-steps (32 values of k each) of a tile of W, or its pairs of k-steps.  Plain
// arithmetic, the same on the host.
#pragma once

// Wavefront `wave` of `waves` takes k-steps [first_k_step(wave), first_k_step(wave + 1)) of `steps`; with
// fewer steps than wavefronts some have none.
constexpr int first_k_step(int steps, int wave, int waves) { return (int)((long long)steps * wave / waves); }

// What a wavefront of [first, behind) asks for ahead of its loop: load(u, k) for the first N of its k-steps, the last one again past
// its end; nothing where it has none.
template <int N, class Load> constexpr void ask_ahead(int first, int behind, Load load) {
  if (first >= behind) return;
#pragma unroll
  for (int u = 0; u < N; ++u) load(u, first + u < behind ? first + u : behind - 1);
}
