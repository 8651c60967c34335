// launch_pass refuses a pass whose output codes it would not write: every
// width but 1, 2, 4 and 8 bytes, and any wider than the input's.  The refusal
// comes before any device call; an accepted width ends in the launch's own
// error where there is no device.  Host code only.
#include <cstdio>
#include <string>

#include "internal.hpp"

using namespace ecl::lib;

int main() {
  int bad = 0;
  alignas(16) static unsigned char out[64];
  for (int cw : {1, 2, 4, 8})
    for (int dst_cw = -1; dst_cw <= 9; ++dst_cw) {
      PassParams p{};
      p.cw = cw;
      p.tile_rows = 4;
      p.tile_codes = static_cast<uint32_t>(pass_tile_codes(cw, 4));
      p.k = 1;
      p.num_tiles = 1;
      p.tiles_per_wg = 1;
      p.dst = out;
      p.dst_cw = dst_cw;
      const bool fits = (dst_cw == 1 || dst_cw == 2 || dst_cw == 4 || dst_cw == 8) && dst_cw <= cw;
      if (fits) continue;  // would launch
      bool refused = false;
      try {
        launch_pass(p, nullptr);
      } catch (const Error& e) {
        refused = e.status == ECL_ERROR_INTERNAL &&
                  std::string(e.what()).find("codes of this width") != std::string::npos;
      }
      if (!refused) {
        std::printf("cw %d, dst_cw %d: not refused\n", cw, dst_cw);
        ++bad;
      }
    }
  std::printf(bad ? "FAILED\n" : "ALL OK\n");
  return bad != 0;
}
