// Weights that the next launch reads, fetched into the caches by `blocks`
// workgroups behind those of this one: `chunks` runs of `pieces` KiB, a run for
// each of the next launch's workgroups.
#pragma once

struct Ahead {
  const char* from;
  int blocks, chunks, pieces;
};
