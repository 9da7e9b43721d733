// Stable grouping of labels [P][n] by cluster (defined in group.hip).
#pragma once
#include "common.hpp"

namespace eac {

// The counting table's shape for n points, P partitions, ktot clusters.
struct GroupShape {
  int64_t chunk;  // points a wavefront places
  int64_t nch;    // chunks per partition
  int64_t table;  // table entries (int32)
};
GroupShape group_shape(int64_t n, int P, int64_t ktot);

// Workspace bytes group_by_cluster takes beyond its outputs.
size_t group_ws_bytes(int64_t n, int P, int64_t ktot);

// members: point ids by global cluster (k_off[p] + label), ascending inside a
// cluster; start[ktot + 1]: each cluster's first position (uint32), then the
// number of assigned points. Labels < 0 are left out; labels >= k of their
// partition are left out and set *bad (nullable). pos (nullable, [P][n]):
// each point's position in members, -1 when left out. P * n < 2^32.
int group_by_cluster(const int32_t* labels, int64_t n, int P, const int64_t* d_koff,
                     const int64_t* h_koff, uint32_t* members, uint32_t* start, int32_t* pos,
                     unsigned int* bad, Arena& ar, hipStream_t s);

}  // namespace eac
