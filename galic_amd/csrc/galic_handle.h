// galic_handle.h -- the opaque galic_ctx of the C ABI: device state plus the
// host copies the driver sequences and the file writers read.
#pragma once
#include <vector>

#include "../../include/galic_hip.h"
#include "galic_ctx.h"

struct galic_ctx {
  galic::Ctx c;
  // host copies of the geometry
  std::vector<double> distance, cellsize;
  bool initial_done = false;
  bool fp32_initial_done = false;
};
