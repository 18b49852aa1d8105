// Packed-chunk MLA attention (mla_chunk.hip): host interface used by mla_run.
#pragma once
#include <stdint.h>

namespace ifattn {

struct MlaChunkCall {
  const void *q, *cache;
  const int32_t *block_tables;
  int32_t table_stride;
  const int32_t *cu_q, *kv_lens;
  int32_t num_seqs, num_rows, window;
  const void *sink_k, *sink_v;
  int32_t n_sinks;
  void *out;
  int32_t heads, block_size;
  int64_t num_blocks;
  int32_t max_context;
  float scale;
  void *workspace;
  uint64_t workspace_bytes;
  void *stream;
};

// Workspace of a call of num_rows packed rows (0: too few rows for this path).
uint64_t mla_chunk_workspace(int32_t num_rows);
// Whether a (validated) bf16 window call runs on the chunk kernel.
bool mla_chunk_takes(const MlaChunkCall &c);
void launch_mla_chunk(const MlaChunkCall &c);

}  // namespace ifattn
