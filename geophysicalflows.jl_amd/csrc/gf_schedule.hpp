// Radix schedules chosen by the autotuner, per (model, nlayers, nx, ny, dtype), shared by the
// contexts of a process and persisted as a JSON table.
#pragma once
#include <array>
#include <string>

namespace gf {

using SchedKey = std::array<int, 5>;   // model, nlayers, nx, ny, dtype

struct Sched {
  int p[3] = {0, 0, 0};         // FFT points per thread of K1, K2, K3 (0: built-in choice)
  int split[3] = {0, 0, 0};     // K1 one field per workgroup row, K2 u q / v q in two rows,
                                // K3 one column per workgroup
  double step_us = 0;           // measured time of one step under this schedule, microseconds
};

bool sched_lookup(const SchedKey& key, Sched& out);
// For a single-layer problem without an entry of its own: K1 and K3 transform columns of ny points
// and K2 rows of nx, so each takes what the table has for square grids of that length, of the same
// model and precision if there is one, else of the same precision, else any. False where the table
// has no square grid of either length (the built-in choice then); where it has one of them, the other
// takes the next longer length's.
bool sched_by_length(const SchedKey& key, Sched& out);
void sched_store(const SchedKey& key, const Sched& s);
void sched_clear();
// Writes every entry; throws std::runtime_error naming the problem.
void sched_save(const std::string& path);
// Reads a table written by sched_save and stores its entries; returns the number read.
// Throws std::runtime_error on a malformed file or an entry whose schedule is not offered.
int sched_load(const std::string& path);

}  // namespace gf
