// The steps of the module's forward as module_fwd.hip strings them together; the library's single-step entry points run the
// same functions.  All arguments have been validated by the caller.
#pragma once
#include "linear_common.h"

namespace sla {

// mask builder (block_map.hip); sparse_map may be null where only the look-up table is wanted
int64_t block_map_workspace_bytes(int dtype, int BH, int L, int D, int BLKQ, int BLKK);
int block_map_check(const void* q, const void* k, const int64_t* strides, int dtype, int B, int H, int L, int D, int BLKQ,
                    int BLKK, int topk, const void* workspace, int64_t workspace_bytes, const int8_t* sparse_map, bool want_map,
                    const void* lut, int lut_elem_bytes, RowLayout* lay);
// Where the parts of its workspace lie: chunk sums and column mean of k, block means of q and k (tiled: in operand order), scores.
struct MapParts {
  float *chunk_sums, *group_sums;
  void *colmean, *pq, *pk, *score;
  int tiled, M, N, nchunk;
};
MapParts block_map_parts(int dtype, int BH, int L, int D, int BLKQ, int BLKK, void* workspace, int64_t workspace_bytes);
void block_map_select(int dtype, const MapParts& m, int BH, int D, int topk, int8_t* sparse_map, void* lut, int lut64,
                      hipStream_t st);
int block_map_run(const void* q, const void* k, const RowLayout& lay, int dtype, const MapParts& m, int BH, int L, int D, int BLKQ,
                  int BLKK, int topk, int8_t* sparse_map, void* lut, int lut64, bool first_pass, hipStream_t st);
int block_map_entry(const void* q, const void* k, const int64_t* strides, int dtype, int B, int H, int L, int D, int BLKQ,
                    int BLKK, int topk, void* workspace, int64_t workspace_bytes, int8_t* sparse_map, bool want_map, void* lut,
                    int lut_elem_bytes, void* stream);

// per-head states of the linear branch (linear.hip): `states` receives what linear_states_bytes() counts, `parts` (the
// slices' partial sums, linear_parts_bytes()) is scratch
int64_t linear_states_bytes(int BH, int L, int D);
int64_t linear_parts_bytes(int BH, int L, int D);
int linear_state_run(const void* k, const void* v, const RowLayout& lay, const float* weight, int dtype, int fmap, int BH, int L,
                     int D, char* states, char* parts, hipStream_t st);

// attention with the linear branch in its epilogue (sparse_fwd.hip)
int attn_linear_run(const void* q, const void* k, const void* v, const RowLayout& lin, const void* lut, int lut_elem_bytes,
                    const char* states, const float* bias, void* o_s, void* out, const RowLayout& lout, float* lse, int dtype,
                    int fmap, int BH, int L, int D, int BLKQ, int topk, float qk_scale, hipStream_t st);

int validate_attn_shape(int dtype, int B, int H, int L, int D, int BLKQ, int BLKK, int topk, int lut_elem_bytes);

}  // namespace sla
