// The tile loop of a prefill workgroup (context_attention.hip), whose waves
// may decide, after any tile, to start again.  Host and device code, so that
// the waves' agreement can be checked without a GPU.
#pragma once

#include <type_traits>

namespace akv {

#if defined(__HIPCC__)
#define AKV_LOOP __device__ __forceinline__
#else
#define AKV_LOOP inline
#endif

constexpr int kRestartWords = 2;

// The word in which tile `it` asks for a restart: one for each pair of tiles,
// and another for the next pair.
AKV_LOOP int restart_word(int begin, int it) { return ((it - begin) >> 1) & 1; }

// Every wave runs tiles [begin, end) in pairs, one tile buffer each (`half`,
// a compile-time 0 or 1).  step(it, half) ends in a barrier; before it a wave
// may set the pair's word.  asked(it) reads that word behind the pair's last
// barrier; restart() makes further requests impossible and the loop starts
// again.  Nothing stands between the read and the next pair, so a wave that is
// late for it can meet waves already inside the next tile.  They cannot pass
// that tile's barrier without the late wave, and their word is the other one,
// so all waves read the same answer.  With one word for all tiles the late
// wave could see the next tile's request, restart alone, and leave the
// others' barriers unpaired.
template <typename Step, typename Asked, typename Restart>
AKV_LOOP void run_tiles(int begin, int end, Step step, Asked asked, Restart restart) {
  const std::integral_constant<int, 0> even{};
  const std::integral_constant<int, 1> odd{};
  for (int it = begin; it < end; it += 2) {
    step(it, even);
    if (it + 1 < end) step(it + 1, odd);
    if (asked(it)) {
      restart();
      it = begin - 2;
    }
  }
}

}  // namespace akv
