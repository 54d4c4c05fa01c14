// Population synthesis on the device (init.hip): the agent draws, the public-transport
// cap, the starting-infection selection, the start cells and the occupancy grid, written
// straight into the SoA and grid of every simulation of a batch.
#pragma once
#include <hip/hip_runtime_api.h>

#include <cstdint>
#include <string>
#include <vector>

#include "config.hpp"
#include "population.hpp"

namespace epi {

// One simulation: what to build, and its slices of the batch's concatenated arrays. The grid
// (strips of `strip` bytes) must be clear.
struct InitJob {
  const Config* cfg;
  uint64_t seed;
  const Geometry* geo;
  uint32_t *pos, *st, *tm, *wsa;
  uint8_t* occ;
  uint32_t strip;
};

// Fills the jobs' slices with the same agents synthesize_population builds on the host, on
// `stream`. The configs must have passed prepare_population. Returns hipSuccess or the first
// HIP error; `err` names the failing step.
hipError_t synthesize_on_device(const std::vector<InitJob>& jobs, hipStream_t stream, std::string& err);

// One simulation's office layout (model.hpp) from its home-layout state words `st` (n agents).
struct OfficeJob {
  uint32_t n, n_offices, n_houses;
  const uint32_t* st;
  uint32_t *office_agent, *office_slot;
};

// Slot maps of every simulation, office_agent[slot] = id and office_slot[id] = slot, with the
// number of Normal and Essential workers of each office, on `stream`.
hipError_t build_office_maps_on_device(const std::vector<OfficeJob>& jobs,
                                       std::vector<std::vector<uint32_t>>& workers_per_office, hipStream_t stream,
                                       std::string& err);

}  // namespace epi
