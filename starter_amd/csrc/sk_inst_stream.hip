// Stream-path kernel instances (sk_stream.hpp) for one epilogue (-DSK_EPI=<0, 1, 2, 3, 11, 12>).
#include "sk_registry.hpp"

#ifndef SK_EPI
#error "build with -DSK_EPI=<epilogue id>"
#endif

#define SK_CAT2(a, b) a##b
#define SK_CAT(a, b) SK_CAT2(a, b)

namespace sk {

#if SK_EPI == 0 || SK_EPI == 2   // persistent tiles: logits and the fused argmax
template <int MT, int EPI>
__global__ void __launch_bounds__(64 * kTilesMG * kTilesNG) stream_tiles_entry(Args p) {
  stream_tiles_body<MT, EPI>(p);
}

KernelFn SK_CAT(stream_tiles_for_epi, SK_EPI)(int MT) {
  return MT == 1 ? &stream_tiles_entry<1, SK_EPI> : MT == 2 ? &stream_tiles_entry<2, SK_EPI> : nullptr;
}
#endif

#if SK_EPI != 2
template <int KG, int MG, int MT, int NT, int UC, int EPI>
__global__ void __launch_bounds__(64 * KG * MG) stream_entry(Args p) {
  stream_body<KG, MG, MT, NT, UC, EPI>(p);
}

#define SK_ST(KG, MG, MT, NT, UC) \
  case stream_key(KG, MG, MT, NT, UC): return &stream_entry<KG, MG, MT, NT, UC, SK_EPI>;
// The wave shapes: up to 16 rows (four waves split K), 32 and 64 (two K groups
// of two; 64 with 128-column units for low tiles), 128 (four row groups of one
// K group, 128-column units).
#define SK_ST_NT(NT) \
  SK_ST(4, 1, 1, NT, 64) SK_ST(2, 2, 1, NT, 64) SK_ST(2, 2, 2, NT, 64) SK_ST(1, 4, 2, NT, 128)

KernelFn SK_CAT(stream_for_epi, SK_EPI)(int KG, int MG, int MT, int NT, int UC) {
  switch (stream_key(KG, MG, MT, NT, UC)) {
    SK_ST(2, 2, 2, 1, 128) SK_ST(2, 2, 2, 2, 128)
    SK_ST_NT(1) SK_ST_NT(2) SK_ST_NT(3) SK_ST_NT(4) SK_ST_NT(5)
    default: break;
  }
  return nullptr;
}
#endif

}  // namespace sk
