// coef_bytes over a recording whose windows' needs wander upwards: how often the buffer grows, and the largest share
// of the device's memory it takes. Arguments: windows, first need, growth per window (per mille), device memory.
#include <cstdio>
#include <cstdlib>

#include "coefs.h"

int main(int argc, char** argv) {
  if (argc < 5) return 2;
  const int windows = std::atoi(argv[1]);
  double need = std::atof(argv[2]);
  const double growth = 1.0 + std::atof(argv[3]) / 1000.0;
  const size_t device = static_cast<size_t>(std::atof(argv[4]));
  size_t have = 0, most = 0;
  int grown = 0, without = 0;
  for (int w = 0; w < windows; ++w, need *= growth) {
    const size_t n = static_cast<size_t>(need);
    const size_t got = bsx::coef_bytes(n, have, device - have);
    if (got == 0) {
      ++without;
      continue;
    }
    if (got < n || got < have) return 1;
    grown += got > have;
    have = got;
    most = have > most ? have : most;
  }
  std::printf("grown %d without %d share %.4f\n", grown, without, static_cast<double>(most) / static_cast<double>(device));
  return 0;
}
