// Walks of crm_index.hpp on the host: argv rows, tile, blocks; prints how many tiles all blocks
// take together, the first row of the last tile and whether an index ever fell or went below 0.
// With four arguments (row nrad 0 0): the level of a row.
#include <cstdio>
#include <cstdlib>

#include "crm_index.hpp"

int main(int argc, char** argv) {
  if (argc == 5) {
    std::printf("%d\n", level_of(std::atol(argv[1]), std::atoi(argv[2])));
    return 0;
  }
  const long rows = std::atol(argv[1]);
  const int tile = std::atoi(argv[2]);
  const unsigned blocks = (unsigned)std::atol(argv[3]);
  long taken = 0, last = -1;
  bool wrapped = false;
  for (unsigned b = 0; b < blocks; b++) {
    long before = -1;
    for (Strided t = tiles_of(rows, tile, b, blocks); t.more() && !wrapped; t.next()) {
      wrapped = t.at < 0 || t.at <= before;
      before = t.at;
      last = t.at * tile > last ? t.at * tile : last;
      taken++;
    }
  }
  std::printf("%ld %ld %d\n", taken, last, (int)wrapped);
}
