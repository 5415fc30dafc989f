// The prebuilt layer (moe_layer): its stages on one set of buffers.
//
// Under an expert map (expert parallelism) most slots belong to experts on
// other devices.  align then also writes the list of the local experts' blocks
// (local_blocks) and the GEMMs run over that list: the tile map deals the local
// blocks out over the XCDs evenly, where the plain map deals out all blocks in
// expert order and leaves the local experts -- usually a run of consecutive
// ids -- to one or two XCDs.  Blocks of other devices are not visited, their
// slots have no row in D, and the top-k sum passes them over.  The tile height
// follows the slots per routed expert, not per local one (the former gave 256-row
// tiles to experts of 62 rows).  Measured on one rank of eight of the DeepSeek-V3
// shape (32 of 256 experts, 1999 tokens): 1548 us a layer over all blocks (W13
// 923, W2 562: one XCD did the work), 329 us over the list.
#include "internal.hpp"

using namespace moe;

static LocalBlocks local_of(const moe_layer* l) {
  LocalBlocks r;
  r.E_routed = l->E_routed;
  if (l->expert_map) r.blocks = local_blk(l->local_blocks);
  if (l->T * l->top_k <= kRunsMaxSlots) r.runs = l->runs;
  r.share = l->share;
  return r;
}

extern "C" int64_t moe_layer_local_blocks_bytes(int64_t T, int64_t max_padded, int32_t BM) {
  if (T < 0 || max_padded < 0 || !block_m_ok(BM)) return -1;
  return 4 * (1 + 2 * ((max_padded + BM - 1) / BM) + T);
}

extern "C" int64_t moe_layer_share_bytes(void) { return (4 + 2 * 128 * kShareRows) * (int64_t)kShareTiles; }

extern "C" int64_t moe_layer_runs_bytes(int32_t E_routed) { return E_routed < 0 ? -1 : 16 * ((int64_t)E_routed + 1); }

static int layer_quant_align(const moe_layer* l, const moe_layer* shared, const void* hidden, const int32_t* topk_ids,
                             void* stream) {
  if (!l || (l->expert_map && !l->local_blocks)) return kErrNullPointer;
  return quant_align(hidden, hidden ? l->T : 0, l->H, l->q1, l->Hp, l->s1, topk_ids, l->T * l->top_k, l->E_routed,
                     l->block_size_m, l->expert_map, l->sorted_ids, l->expert_ids, l->ntpp, l->max_padded,
                     l->workspace, l->local_blocks,
                     l->T * l->top_k <= kRunsMaxSlots ? l->runs : nullptr, l->share,
                     shared ? shared->share : nullptr, l->top_k, stream);
}

extern "C" int moe_layer_quant_align(const moe_layer* l, const void* hidden, const int32_t* topk_ids, void* stream) {
  return layer_quant_align(l, nullptr, hidden, topk_ids, stream);
}

extern "C" int moe_layer_scales(const moe_layer* l, void* stream) {
  if (!l) return kErrNullPointer;
  if (!l->s1_pos) return kOk;
  return moe_gather_scales_by_position(l->s1, l->T, l->Hp / 128, l->sorted_ids, l->ntpp, l->T * l->top_k, l->top_k,
                                       l->max_padded, l->s1_pos, stream);
}

extern "C" int moe_layer_w13(const moe_layer* l, void* stream) {
  if (!l || (l->expert_map && !l->local_blocks)) return kErrNullPointer;
  if (l->expert_map && l->E >> kLocalExpertBits) return kErrBadExperts;
  return w13_gemm(l->q1, l->s1_pos ? l->s1_pos : l->s1, l->w13, l->w13_scale, l->sorted_ids,
                  l->expert_map ? local_eid(l->local_blocks, l->max_padded, l->block_size_m) : l->expert_ids,
                  l->expert_map ? local_rows(l->local_blocks) : l->ntpp, l->T * l->top_k, l->top_k, l->Hp, l->I, l->E,
                  l->block_size_m, l->max_padded, l->tile_m, l->s1_pos != nullptr, l->exact_dot != 0, l->hq, l->hs,
                  stream, local_of(l));
}

extern "C" int moe_layer_w2(const moe_layer* l, const float* topk_weights, void* stream) {
  if (!l || (l->expert_map && !l->local_blocks)) return kErrNullPointer;
  if (l->expert_map && l->E >> kLocalExpertBits) return kErrBadExperts;
  return plain_gemm(l->hq, l->hs, l->w2, l->w2_scale, l->sorted_ids,
                    l->expert_map ? local_eid(l->local_blocks, l->max_padded, l->block_size_m) : l->expert_ids,
                    l->expert_map ? local_rows(l->local_blocks) : l->ntpp, topk_weights, l->T * l->top_k, 1, 1, l->Hp,
                    l->I, l->E, l->block_size_m, l->max_padded, 0, l->tile_m, l->s1_pos != nullptr, l->D, stream,
                    local_of(l));
}

extern "C" int moe_layer_reduce(const moe_layer* l, const void* addend, int64_t addend_ld, int64_t cols, void* y,
                                void* stream) {
  if (!l || (l->expert_map && !l->local_blocks)) return kErrNullPointer;
  return reduce_topk(l->D, l->Hp, addend, addend_ld, l->T, l->top_k, cols,
                     l->expert_map ? local_mask(l->local_blocks, l->max_padded, l->block_size_m) : nullptr, y, stream);
}

extern "C" int moe_layer_run(const moe_layer* l, const moe_layer* shared, const void* hidden,
                             const float* topk_weights, const int32_t* topk_ids, int64_t cols, void* y,
                             void* stream) {
  if (!l) return kErrNullPointer;
  if (shared && (shared->T != l->T || shared->Hp != l->Hp || shared->top_k != 1)) return kErrBadShape;
  if (l->T > 0 && !hidden) return kErrNullPointer;
  int rc = layer_quant_align(l, shared, hidden, topk_ids, stream);
  if (rc == kOk) rc = moe_layer_scales(l, stream);
  if (rc == kOk) rc = moe_layer_w13(l, stream);
  if (rc == kOk) rc = moe_layer_w2(l, topk_weights, stream);
  if (rc == kOk && shared) rc = moe_layer_w13(shared, stream);
  if (rc == kOk && shared) rc = moe_layer_w2(shared, nullptr, stream);
  if (rc == kOk) rc = moe_layer_reduce(l, shared ? shared->D : nullptr, shared ? shared->Hp : 0, cols, y, stream);
  return rc;
}
