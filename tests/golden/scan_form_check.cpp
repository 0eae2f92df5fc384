// Prints the scan's form for a volume of X x Y x Z points (scan_form,
// mdmc_tilemap.h), with the classify's tiling: 256-cell x-tiles for rows of up
// to 256 cells, 512-cell ones for longer rows, blocks of 7 cell rows.
#include "mdmc_tilemap.h"

#include <cstdio>
#include <cstdlib>

int main(int argc, char **argv) {
  if (argc != 4) return 2;
  const uint64_t cx = std::strtoull(argv[1], nullptr, 10) - 1, cy = std::strtoull(argv[2], nullptr, 10) - 1,
                 cz = std::strtoull(argv[3], nullptr, 10) - 1;
  const uint64_t cap = cx <= 256 ? 256 : 512, XT = (cx + cap - 1) / cap;
  const mdmc::ScanForm f = mdmc::scan_form(XT * cy * cz, XT * cy, XT * ((cy + 6) / 7));
  std::puts(f == mdmc::ScanForm::planes ? "planes" : f == mdmc::ScanForm::tiles ? "tiles" : "lookback");
  return 0;
}
