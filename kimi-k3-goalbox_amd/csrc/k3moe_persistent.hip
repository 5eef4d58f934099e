// The persistent kernels, in a translation unit and so a code object of their
// own, each at a multiple of kPersistentAlign: the time of a decode step of 10 to
// 60 us depends on where in its code object the kernel lies, by up to 2 % with the
// same instructions, so no other kernel may move them. (By which mechanism is not
// known; where the buffers lie moves a time by up to 1 % too, so that layouts are
// compared on the same buffers.) us of 64 experts x 2048 at 8 / 32 tokens, a TP8
// rank at 8 / 64 tokens, the Kimi rank's block at 1 / 6, medians of four runs in
// turn (of one layout they differ by 0.1 %; lines of other runs by their difference
// from the first):
//   the library before the grouped and latent GEMMs joined it
//                             30.57  38.21  60.75  183.3  52.39  100.6
//   beside those GEMMs        30.84  38.27  60.87  183.4  52.64  100.2
//   here, aligned to  256 B   31.00  38.86  61.20  183.5  52.55  100.5
//                     512 B   30.62  38.51  60.72  183.4  52.69  100.4
//                     1 KiB   30.75  38.20  61.05  183.5  52.48  100.3
//                     2 KiB   30.85  38.30  60.93  183.2  52.63  100.2
//                     4 KiB   30.62  38.45  60.81  183.7  52.59  100.2
//                     8 KiB   30.75  38.52  60.92  183.7  52.64  100.3
//                    16 KiB   30.53  38.40  60.86  182.8  52.65  100.3
//                    32 KiB   30.63  38.33  60.84  183.2  52.52  100.2
//                    64 KiB   30.84  38.27  61.12  183.1  52.73  100.3
// 32 KiB with the single-token kernels first: 30.61, 38.25, 60.87, 183.9, 52.72, 100.4.
// Over nine placements of the buffers, 64 experts at 8 / 32, a TP8 rank at 8, the block at
// 1: before those GEMMs 30.47, 38.22, 59.40, 51.25; beside them 30.74, 38.27, 59.56, 51.46;
// here 30.55, 38.25, 59.59, 51.34.
#include <hip/hip_runtime.h>

#include "k3moe_persistent.hpp"
#include "k3moe_single.hpp"

namespace k3moe {

// (The kernels lie in the order of their first mention.)
PersistentKernel persistent_kernel(const Plan &p, int &slot) {
  // The latent block's phases (Plan::lat_in) have instantiations of their own.
  // decode: whole gate/up super-steps (AL: K a multiple of 512; lat_in plans are pinned, so they
  // have them) and the expert-major down variant of the plan's I
  static const PersistentKernel decode[3][4] = {
      {k_moe_decode<false, 0, false>, k_moe_decode<false, 2, false>, k_moe_decode<false, 3, false>,
       k_moe_decode<false, 4, false>},
      {k_moe_decode<true, 0, false>, k_moe_decode<true, 2, false>, k_moe_decode<true, 3, false>,
       k_moe_decode<true, 4, false>},
      {k_moe_decode<true, 0, true>, k_moe_decode<true, 2, true>, k_moe_decode<true, 3, true>,
       k_moe_decode<true, 4, true>}};
  // single: chosen experts per wave in the down phase (1: k <= 8, 2: k <= 16), its k-steps (2: I <= 256, 4: I <= 512)
  static const PersistentKernel single[2][2][2] = {
      {{k_moe_single<1, 2, false>, k_moe_single<1, 4, false>}, {k_moe_single<2, 2, false>, k_moe_single<2, 4, false>}},
      {{k_moe_single<1, 2, true>, k_moe_single<1, 4, true>}, {k_moe_single<2, 2, true>, k_moe_single<2, 4, true>}}};
  if (p.single) {
    const int lat = p.lat_in ? 1 : 0, je2 = p.k > kDecWaves ? 1 : 0, ks4 = p.I > 256 ? 1 : 0;
    slot = 12 + lat * 4 + je2 * 2 + ks4;
    return single[lat][je2][ks4];
  }
  const int row = p.lat_in ? 2 : (p.K / kBlockK) % 16 == 0 ? 1 : 0;
  const int v = p.I == 256 ? 1 : p.I == 384 ? 2 : p.I == 512 ? 3 : 0;
  slot = row * 4 + v;
  return decode[row][v];
}

}  // namespace k3moe
