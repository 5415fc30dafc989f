// Host functions shared by the C entry points and the layer (layer.hip).
#pragma once

#include "common.hpp"

namespace moe {

// What the layer knows of its blocks beyond the align outputs.  blocks: the list
// of local blocks that align writes under an expert map (moe_layer's
// local_blocks), null without one.  runs: the table of runs, or null.  share:
// moe_layer's share buffer, or null.
// E_routed: the experts the slots are spread over, for the choice of the tile
// height and a bound on the blocks (0: E, and what fits in max_padded, which
// with few slots allows for more).  A map may send several of them to one
// local expert, so the local ones bound nothing.
struct LocalBlocks {
  const int32_t* blocks = nullptr;
  const int32_t* runs = nullptr;
  int32_t* share = nullptr;
  int64_t E_routed = 0;
};

// The table of runs that the one-launch align writes: [0] the experts with
// slots here, then from [4] four words for each of them by descending rows
// (equal ones by ascending expert): first position, rows, local expert id,
// rows with padding.
constexpr int64_t kRunsMaxSlots = 16384;

// S slots over E experts fill at most this many blocks of BM: m <= min(S, E)
// experts with c >= 1 slots have ceil(c/BM) <= 1 + (c-1)/BM blocks each.
inline int64_t blocks_bound(int64_t S, int64_t E, int64_t BM) {
  const int64_t m = S < E ? S : E;
  return m + (S - m) / BM;
}

// moe_layer's share: a counter for each of kShareTiles tiles that several
// workgroups compute together, zero between launches (align clears them, which
// runs on the layer's stream before the GEMMs), then kShareRows rows of 128 bf16
// for each.
constexpr int kShareTiles = 128;
constexpr int kShareRows = 64;

// local_blocks holds [0] local blocks * BM, then the blocks, then a word for each
// with its expert, then a word per token whose bit i says that slot i's expert
// is local.  A block's word has the local expert in its low bits and the expert
// before the map above them: a map may send several to one local expert, whose
// blocks, one after another in the list, are still runs of their own with other
// blocks or padding between their slots.  One word holds both, so that a tile
// has its run and its expert from one load.
constexpr int kLocalExpertBits = 20;
MOE_HOST_DEVICE int32_t block_word(int32_t e, int32_t local) {
  const int32_t most = (1 << kLocalExpertBits) - 1;  // a local expert that is not here stays none
  return e << kLocalExpertBits | (local < most ? local : most);
}
MOE_HOST_DEVICE int32_t local_of_word(int32_t w) { return w & ((1 << kLocalExpertBits) - 1); }
inline const int32_t* local_rows(const int32_t* l) { return l; }
template <class T>
MOE_HOST_DEVICE T* local_blk(T* l) { return l + 1; }
template <class T>
MOE_HOST_DEVICE T* local_eid(T* l, int64_t max_padded, int32_t BM) { return l + 1 + (max_padded + BM - 1) / BM; }

template <class T>
MOE_HOST_DEVICE T* local_mask(T* l, int64_t max_padded, int32_t BM) { return l + 1 + 2 * ((max_padded + BM - 1) / BM); }

int plain_gemm(const void* A, const float* A_scale, const void* B, const float* B_scale, const int32_t* sorted_ids,
               const int32_t* expert_ids, const int32_t* ntpp, const float* topk_weights, int64_t S, int32_t top_k,
               int32_t a_by_pos, int64_t N, int64_t K, int32_t E, int32_t BM, int64_t max_padded, int32_t tile_order,
               int32_t tile_m, bool scales_by_pos, void* C, void* stream, LocalBlocks local = {});

int w13_gemm(const void* Aq, const float* A_scale, const void* W13, const float* W13_scale, const int32_t* sorted_ids,
             const int32_t* expert_ids, const int32_t* ntpp, int64_t S, int32_t top_k, int64_t H, int64_t I, int32_t E,
             int32_t BM, int64_t max_padded, int32_t tile_m, bool scales_by_pos, bool exact, void* hq, float* hs,
             void* stream, LocalBlocks local = {});

// T == 0: align alone.  local: the lists to write under an expert map, or null;
// runs: the table of runs to write (S <= kRunsMaxSlots), or null; share, share2:
// the counters to clear (the layer's and its shared expert's), or null; top_k:
// the slots of a token (for its mask).
int quant_align(const void* x, int64_t T, int64_t H, void* q, int64_t ldq, float* scales, const int32_t* topk_ids,
                int64_t S, int32_t E, int32_t BM, const int32_t* expert_map, int32_t* sorted_ids, int32_t* expert_ids,
                int32_t* ntpp, int64_t max_padded, void* workspace, int32_t* local, int32_t* runs, int32_t* share,
                int32_t* share2, int32_t top_k, void* stream);

// The top-k sum of rows of H columns in D (row stride ldd) into y (row stride
// H); addend rows (row stride lda) or null; with mask (a word per token) the
// slots without a set bit are passed over.
int reduce_topk(const void* D, int64_t ldd, const void* addend, int64_t lda, int64_t T, int32_t top_k, int64_t H,
                const int32_t* mask, void* y, void* stream);

}  // namespace moe
