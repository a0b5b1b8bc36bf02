// What a pass builder (pass.hip) launches in one go for several kernel maps:
// the launches themselves live beside the single-map forms in query.hip (maps
// and rank tables) and conv.hip (offset groups).
#pragma once

#include <vector>

#include "common.h"

namespace mnt {

constexpr int kPassMaps = 12;             // maps of one batched launch

// ---- kernel-map queries (query.hip) ----

// One dense map to look up.  Addresses are device memory; batch dims are null
// for a single cloud.
struct QueryWork {
  const void *sources, *targets;
  const void *source_batch_dims, *target_batch_dims;
  int64_t num_sources, num_targets;
  int *kernel_map;
  int plan;                               // index into the plans of the batch
};

// Frame, offset groups and members of a map as the batched query reads them
// from device memory; `ints` is empty when the frame does not fit a packed key.
struct QueryTables {
  std::vector<int> ints;
  int num_groups, num_offsets, last_width;
  bool groups_in_rows;
};
QueryTables make_query_tables(const long long *source_bounds, const long long *target_bounds,
                              const int64_t *offsets, int64_t num_offsets, int ndim, int64_t num_batches);
// tables_at[i]: where the ints of plan i start inside `tables` (device memory).
void enqueue_queries(const std::vector<QueryWork> &work, const std::vector<QueryTables> &plans,
                     const std::vector<int> &tables_at, const int *tables, int ndim, int coord_dtype,
                     int batch_dtype, int64_t num_batches, hipStream_t stream);

// ---- sizes, stable size order, rank tables and pair lists (query.hip) ----

struct TableWork {
  const int *kernel_map;
  int num_sources, num_targets, num_offsets, reorder;
  int *source_masks, *target_masks, *in_idx, *out_idx, *sizes, *order;
  // filled in by enqueue_tables: where the host finds sizes and order
  int host_at;
};
// Scratch comes from `scope`; source_masks must hold -1 already.  Order and sizes
// of every map go to pinned memory, its flag word there takes the value
// `sequence` once they are complete.
void enqueue_tables(std::vector<TableWork> &work, Scope &scope, unsigned long long sequence, hipStream_t stream);
void collect_tables(const TableWork &work, Arena &arena, unsigned long long sequence, int64_t *sizes_host,
                    int64_t *order_host);

// ---- offset groups of 3 x 3 x 3 maps (conv.hip) ----

struct GroupWork {
  const int *kernel_map;
  int num_targets;
  const int32_t *offsets_host;            // [3][9][3]
  int *rank, *src, *head;
};
void enqueue_offset_groups(const std::vector<GroupWork> &work, Scope &scope, hipStream_t stream);

}  // namespace mnt
