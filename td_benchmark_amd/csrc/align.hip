// A3: moe_align_block_size -- sort token slots by expert and pad every
// expert's run to a multiple of the GEMM block size BM.
//
// Semantics (reference call sites overlap/overlap_forward.py:165-169, padded
// cumsum of tdx/kernels/moe_utils.py:168-217, pad value = number of valid
// slots as overlap/kernels.py:108-110 masks it):
//   c_e = #slots with expert e, p_e = ceil(c_e/BM)*BM, off_e = sum_{e'<e} p_e'
//   sorted_ids[off_e + j] = j-th slot (flat t*top_k+i, ascending) of expert e
//   sorted_ids[...]      = S at every padding position and in the tail
//   expert_ids[b]        = e for the blocks of e, -1 for blocks >= ntpp/BM
//   ntpp                 = sum_e p_e
// The within-expert order is the stable (ascending slot) order, so the result
// is deterministic and bit-exact against the CPU restatement.
//
// Up to 16384 slots (fewer from 768 experts on, but for a layer) one launch with
// a workgroup per expert (align_expert) computes everything, alone or beside the
// activation quant in the same launch (the two do not depend on each other);
// above that three launches, none of which waits on another workgroup:
//   1. count:  1024 slots per workgroup.  Slots with equal expert inside a wave
//      are found with log2(E) ballots (a match-any built from per-bit ballots),
//      giving each slot its rank among equal-expert slots of its wave; per-wave
//      counts in LDS are prefix-summed across the 16 waves, giving each slot its
//      rank within the chunk and each chunk its per-expert count.
//   2. scan:   one workgroup scans the chunk counts per expert (column-wise,
//      from LDS), pads, scans across experts, and writes the expert offsets,
//      counts and ntpp; the chunk counts become within-expert chunk bases.
//   3. place:  a wide pass: sorted_ids[off[e] + chunk_base[chunk][e] + rank[s]]
//      = s for every slot, S at every padding position, and expert_ids for
//      every block (the expert of a position comes from a binary search over
//      the offsets held in LDS).
// Align moves well under 2 MB at every configuration, so it is latency-bound.
#include <mutex>
#include <type_traits>

#include "common.hpp"
#include "internal.hpp"
#include "quant_group.hpp"

namespace moe {

constexpr int kAlignChunk = 1024;   // slots per count workgroup (16 waves)
constexpr int kAlignMaxExperts = 1024;
constexpr int64_t kAlignStageLimit = 32768;  // chunk counts staged in LDS up to 128 KiB

__global__ __launch_bounds__(kAlignChunk) void align_count_kernel(
    const int32_t* __restrict__ ids, int64_t S, int E, int nbits,
    int32_t* __restrict__ chunk_count, int32_t* __restrict__ rank) {
  extern __shared__ int32_t wcnt[];  // [16][E]
  const int tid = threadIdx.x;
  const int wave = tid >> 6;
  const int lane = tid & 63;
  const int64_t s = (int64_t)blockIdx.x * kAlignChunk + tid;
  for (int i = tid; i < 16 * E; i += kAlignChunk) wcnt[i] = 0;
  int e = -1;
  if (s < S) e = ids[s];
  const bool valid = (e >= 0) && (e < E);
  uint64_t m = __ballot(valid);
  for (int b = 0; b < nbits; ++b) {
    const bool bit = (e >> b) & 1;
    const uint64_t bb = __ballot(bit);
    m &= bit ? bb : ~bb;
  }
  const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
  const int rank_in_wave = __popcll(m & lt);
  __syncthreads();
  if (valid && rank_in_wave == 0) wcnt[wave * E + e] = __popcll(m);
  __syncthreads();
  for (int x = tid; x < E; x += kAlignChunk) {
    int run = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      int t = wcnt[w * E + x];
      wcnt[w * E + x] = run;
      run += t;
    }
    chunk_count[(int64_t)blockIdx.x * E + x] = run;
  }
  __syncthreads();
  if (valid) rank[s] = wcnt[wave * E + e] + rank_in_wave;
}

// One workgroup: per-expert totals and the within-expert base of every chunk
// (column prefix sums of the chunk counts, staged in LDS when they fit), then
// padded sizes and their exclusive scan across experts.  Writes off[0..E]
// (off[E] = ntpp), cnt[0..E) and ntpp; every fill is left to the wide place
// kernel.
__global__ __launch_bounds__(kAlignMaxExperts) void align_scan_kernel(
    int32_t* __restrict__ chunk_count, int64_t n_chunks, int E, int BM, int use_lds,
    int32_t* __restrict__ off_out, int32_t* __restrict__ cnt_out, int32_t* __restrict__ ntpp_out, int32_t* share,
    int32_t* share2) {
  extern __shared__ int32_t staged[];  // [n_chunks][E] when use_lds
  __shared__ int32_t wave_tot[kAlignMaxExperts / 64];
  const int tid = threadIdx.x;
  const int e = tid;
  if (share && tid < kShareTiles) share[tid] = 0;
  if (share2 && tid < kShareTiles) share2[tid] = 0;
  if (use_lds) {
    for (int64_t i = tid; i < n_chunks * E; i += kAlignMaxExperts) staged[i] = chunk_count[i];
    __syncthreads();
  }
  int cnt = 0;
  if (e < E) {
    if (use_lds) {
      for (int64_t c = 0; c < n_chunks; ++c) {
        const int v = staged[c * E + e];
        chunk_count[c * E + e] = cnt;
        cnt += v;
      }
    } else {
      int64_t c = 0;
      for (; c + 8 <= n_chunks; c += 8) {
        int v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = chunk_count[(c + j) * E + e];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          chunk_count[(c + j) * E + e] = cnt;
          cnt += v[j];
        }
      }
      for (; c < n_chunks; ++c) {
        const int v = chunk_count[c * E + e];
        chunk_count[c * E + e] = cnt;
        cnt += v;
      }
    }
  }
  const int padded = (e < E) ? (cnt + BM - 1) / BM * BM : 0;
  // Block-wide exclusive scan of `padded` (wave inclusive scan + wave totals).
  const int lane = tid & 63, wave = tid >> 6;
  int incl = padded;
#pragma unroll
  for (int o = 1; o < 64; o <<= 1) {
    const int y = __shfl_up(incl, o);
    if (lane >= o) incl += y;
  }
  if (lane == 63) wave_tot[wave] = incl;
  __syncthreads();
  if (tid < 64) {
    // exclusive scan of the 16 wave totals by the first wave
    const int t = tid < kAlignMaxExperts / 64 ? wave_tot[tid] : 0;
    int x = t;
#pragma unroll
    for (int o = 1; o < 16; o <<= 1) {
      const int y = __shfl_up(x, o);
      if (lane >= o) x += y;
    }
    if (tid < kAlignMaxExperts / 64) wave_tot[tid] = x - t;
    if (tid == kAlignMaxExperts / 64 - 1) {
      off_out[E] = x;
      *ntpp_out = x;
    }
  }
  __syncthreads();
  if (e < E) {
    off_out[e] = wave_tot[wave] + incl - padded;
    cnt_out[e] = cnt;
  }
}

// Wide pass over max(S, max_padded) indices: slot i goes to
// off[e] + chunk_base[chunk][e] + rank[i]; position i is set to S when it is
// padding (inside an expert's run past its count, or past ntpp), and the first
// position of every block writes that block's expert (-1 past ntpp).  Valid
// and padding positions are disjoint, so no two threads write one element.
__global__ __launch_bounds__(256) void align_place_kernel(
    const int32_t* __restrict__ ids, int64_t S, int E, int BM, const int32_t* __restrict__ chunk_base,
    const int32_t* __restrict__ rank, const int32_t* __restrict__ off, const int32_t* __restrict__ cnt,
    const int32_t* __restrict__ expert_map, int32_t* __restrict__ sorted_ids,
    int32_t* __restrict__ expert_ids, int64_t max_padded) {
  __shared__ int32_t s_off[kAlignMaxExperts + 1];
  __shared__ int32_t s_cnt[kAlignMaxExperts];
  for (int i = threadIdx.x; i <= E; i += 256) s_off[i] = off[i];
  for (int i = threadIdx.x; i < E; i += 256) s_cnt[i] = cnt[i];
  __syncthreads();
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < S) {
    const int e = ids[i];
    if (e >= 0 && e < E) {
      const int64_t chunk = i / kAlignChunk;
      sorted_ids[s_off[e] + chunk_base[chunk * E + e] + rank[i]] = (int32_t)i;
    }
  }
  if (i < max_padded) {
    const int total = s_off[E];
    int e = -1;
    bool pad = true;
    if (i < total) {
      int lo = 0, hi = E - 1;  // largest e with off[e] <= i
      while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (s_off[mid] <= i) lo = mid;
        else hi = mid - 1;
      }
      e = lo;
      pad = (i - s_off[e]) >= s_cnt[e];
    }
    if (pad) sorted_ids[i] = (int32_t)S;
    // With an expert map (global -> local id, -1 = not on this device) the
    // block's expert is reported as its local id.
    if (i % BM == 0) expert_ids[i / BM] = (expert_map && e >= 0) ? expert_map[e] : e;
  }
}

// One launch, a workgroup per expert: every workgroup reads all slot ids (at
// most 64 KiB, from L2 after the first reader), counts every expert's slots in
// LDS, sums the padded sizes before its own expert, and compacts its expert's
// slots in ascending order (each wave owns a contiguous stretch of the slots;
// ballots give a slot its rank).  No workgroup waits on another one.
// Bound by its chain of about four dependent steps, not by bytes.  Against the
// three launches it replaces (kernel time, with the table of runs and the other
// notes that a layer's align leaves): S = 8192, E = 64: 7.8 us with the quant in
// the same launch, 19 us before (quant 5.0, count, scan and place 4.7 each);
// S = 2408, E = 128: 5.1 us, before 17; against the former single workgroup for
// S <= 1024 with the quant: S = 128, E = 8: 3.9 us, before 6.6.
struct AlignArgs {
  const int32_t* ids;
  const int32_t* expert_map;  // or null
  int32_t* sorted;
  int32_t* eids;
  int32_t* ntpp;
  int32_t* local;  // the lists of local blocks and slots, or null (see internal.hpp)
  int32_t* runs;   // the table of runs, or null (see internal.hpp)
  int32_t* share;  // the counters of shared tiles to clear, of two layers, or null
  int32_t* share2;
  int max_padded, S, top_k;
  uint16_t E, BM;  // at most 1024 and 256
};

// Bit i: the expert of token t's slot i is local.
MOE_DEVICE int32_t local_slots(const int32_t* ids, const int32_t* expert_map, int E, int top_k, int t) {
  uint32_t m = 0;
  for (int i0 = 0; i0 < top_k && i0 < 32; i0 += 8) {  // eight at a time: two round trips, not sixteen
    int x[8], here[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = i0 + i < top_k ? ids[(int64_t)t * top_k + i0 + i] : -1;
#pragma unroll
    for (int i = 0; i < 8; ++i) here[i] = (unsigned)x[i] < (unsigned)E ? expert_map[x[i]] : -1;
#pragma unroll
    for (int i = 0; i < 8; ++i) m |= here[i] >= 0 ? 1u << (i0 + i) : 0u;
  }
  return (int32_t)m;
}

// Each expert's count is kept in COPIES words, by lane: a wave's slots of one
// expert add to eight words at a time, where 64 adds to one word follow each
// other.  A call of align alone with every slot on one expert took, with one
// word, with eight, and in three launches (us; the smallest launch takes 6 to 7
// so): S = 8192, E = 64: 12.8, 7.0, 13.0; S = 16384, E = 64: 19.0, 7.3, 13.0;
// S = 16384, E = 256, Zipf: 9.1, 7.2, 13.0.  Up to 1024 slots the few adds cost
// less than the longer sums (0.15 us).
constexpr int kAlignThreads = 512;
constexpr int kAlignWaves = kAlignThreads / 64;

// IT: ids a lane holds (IT * 512 >= S).
template <int IT>
MOE_DEVICE void align_expert(const AlignArgs& a, int e) {
  constexpr int COPIES = IT > 2 ? 8 : 1;
  __shared__ __attribute__((aligned(16))) int32_t hist[kAlignMaxExperts * COPIES];
  auto count_of = [&](int x) {
    if constexpr (COPIES == 1) {
      return hist[x];
    } else {
      const v4i* c = reinterpret_cast<const v4i*>(hist + x * COPIES);
      const v4i s = c[0] + c[1];
      return s[0] + s[1] + s[2] + s[3];
    }
  };
  __shared__ int32_t wave_cnt[kAlignWaves], wave_before[kAlignWaves], wave_total[kAlignWaves];
  __shared__ int32_t wave_lbefore[kAlignWaves], wave_ltotal[kAlignWaves];
  __shared__ int32_t wave_rank[kAlignWaves], wave_runs[kAlignWaves];
  const int sh = __builtin_ctz(a.BM);  // BM is a power of two
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  // wave w takes slots [w*IT*64, (w+1)*IT*64), 64 consecutive ones a step
  const int first = wave * IT * 64 + lane;
  int id[IT];
#pragma unroll
  for (int i = 0; i < IT; ++i) id[i] = first + 64 * i < a.S ? a.ids[first + 64 * i] : -1;
  for (int i = tid; i < a.E * COPIES; i += kAlignThreads) hist[i] = 0;
  __syncthreads();
  int mine = 0;  // this wave's slots of expert e
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    if ((unsigned)id[i] < (unsigned)a.E) atomicAdd(&hist[id[i] * COPIES + lane % COPIES], 1);
    mine += __popcll(__ballot(id[i] == e));
  }
  if (lane == 0) wave_cnt[wave] = mine;
  __syncthreads();
  int before = 0, total = 0;    // padded sizes of the experts before e, and of all
  int lbefore = 0, ltotal = 0;  // and of the local ones among them
  int place = 0, n_runs = 0;    // experts here with more slots than e (or as many and before it), and with any
  const int own = count_of(e);
  for (int x = tid; x < a.E; x += kAlignThreads) {
    const int c = count_of(x);
    const int p = (c + a.BM - 1) >> sh << sh;
    total += p;
    if (x < e) before += p;
    if (!a.expert_map || a.expert_map[x] >= 0) {
      ltotal += p;
      if (x < e) lbefore += p;
      n_runs += p > 0;
      place += c > own || (c == own && x < e);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    before += __shfl_xor(before, o);
    total += __shfl_xor(total, o);
    lbefore += __shfl_xor(lbefore, o);
    ltotal += __shfl_xor(ltotal, o);
    place += __shfl_xor(place, o);
    n_runs += __shfl_xor(n_runs, o);
  }
  if (lane == 0) {
    wave_before[wave] = before;
    wave_total[wave] = total;
    wave_lbefore[wave] = lbefore;
    wave_ltotal[wave] = ltotal;
    wave_rank[wave] = place;
    wave_runs[wave] = n_runs;
  }
  __syncthreads();
  before = total = lbefore = ltotal = place = n_runs = 0;
  int rank = 0;  // of this wave's first slot of e
#pragma unroll
  for (int w = 0; w < kAlignWaves; ++w) {
    before += wave_before[w];
    total += wave_total[w];
    lbefore += wave_lbefore[w];
    ltotal += wave_ltotal[w];
    place += wave_rank[w];
    n_runs += wave_runs[w];
    rank += w < wave ? wave_cnt[w] : 0;
  }
  const int cnt = own;
  const int padded = (cnt + a.BM - 1) >> sh << sh;
  const uint64_t lt = lane == 0 ? 0ull : ~0ull >> (64 - lane);
#pragma unroll
  for (int i = 0; i < IT; ++i) {
    const uint64_t m = __ballot(id[i] == e);
    if (id[i] == e) a.sorted[before + rank + __popcll(m & lt)] = first + 64 * i;
    rank += __popcll(m);
  }
  for (int i = cnt + tid; i < padded; i += kAlignThreads) a.sorted[before + i] = a.S;
  const int local = a.expert_map ? a.expert_map[e] : e;
  for (int i = tid; i < padded >> sh; i += kAlignThreads) a.eids[(before >> sh) + i] = local;
  if (a.local && local >= 0) {
    for (int i = tid; i < padded >> sh; i += kAlignThreads) {
      local_blk(a.local)[(lbefore >> sh) + i] = (before >> sh) + i;
      local_eid(a.local, a.max_padded, a.BM)[(lbefore >> sh) + i] = block_word(e, local);
    }
  }
  // the tokens' local slots, and the positions and blocks past ntpp, shared out over the workgroups
  if (a.local) {
    int32_t* mask = local_mask(a.local, a.max_padded, a.BM);
    for (int t = e * kAlignThreads + tid; t < a.S / a.top_k; t += a.E * kAlignThreads)
      mask[t] = local_slots(a.ids, a.expert_map, a.E, a.top_k, t);
  }
  for (int64_t i = total + (int64_t)e * kAlignThreads + tid; i < a.max_padded; i += (int64_t)a.E * kAlignThreads) {
    a.sorted[i] = a.S;
    if ((i & (a.BM - 1)) == 0) a.eids[i >> sh] = -1;
  }
  if (a.runs && tid == 0 && cnt > 0 && local >= 0)
    reinterpret_cast<v4i*>(a.runs + 4)[place] = (v4i){before, cnt, local, padded};
  if (a.share && e == 0 && tid < kShareTiles) a.share[tid] = 0;
  if (a.share2 && e == 0 && tid < kShareTiles) a.share2[tid] = 0;
  if (e == 0 && tid == 0) {
    *a.ntpp = total;
    if (a.local) *a.local = ltotal;
    if (a.runs) *a.runs = n_runs;
  }
}

template <int IT>
__global__ __launch_bounds__(kAlignThreads) void align_expert_kernel(AlignArgs a) {
  align_expert<IT>(a, blockIdx.x);
}

// The same lists after the three launches: the first workgroup compacts the
// blocks whose (local) expert id is not -1, 1024 at a time (a block's first
// position always holds a slot, whose id is the expert before the map), the
// others mark the tokens' local slots.
__global__ __launch_bounds__(1024) void local_blocks_kernel(const int32_t* __restrict__ ids, int64_t S, int E,
                                                            int top_k, const int32_t* __restrict__ expert_map,
                                                            const int32_t* __restrict__ sorted,
                                                            const int32_t* __restrict__ eids,
                                                            const int32_t* __restrict__ ntpp, int BM,
                                                            int64_t max_padded, int32_t* __restrict__ local) {
  __shared__ int32_t wave_cnt[16];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  if (blockIdx.x > 0) {
    const int64_t t = (int64_t)(blockIdx.x - 1) * 1024 + tid;
    if (t < S / top_k) local_mask(local, max_padded, BM)[t] = local_slots(ids, expert_map, E, top_k, (int)t);
    return;
  }
  const int n = *ntpp / BM;
  const uint64_t lt = lane == 0 ? 0ull : ~0ull >> (64 - lane);
  int done = 0;
  for (int b0 = 0; b0 < n; b0 += 1024) {
    const int b = b0 + tid;
    const int e = b < n ? eids[b] : -1;
    const uint64_t m = __ballot(e >= 0);
    if (lane == 0) wave_cnt[wave] = __popcll(m);
    __syncthreads();
    int at = done;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      at += w < wave ? wave_cnt[w] : 0;
      done += wave_cnt[w];
    }
    if (e >= 0) {
      local_blk(local)[at + __popcll(m & lt)] = b;
      local_eid(local, max_padded, BM)[at + __popcll(m & lt)] = block_word(ids[sorted[(int64_t)b * BM]], e);
    }
    __syncthreads();
  }
  if (tid == 0) *local = done * BM;
}

// The same workgroups followed by those of the 1x128 activation quant, one
// launch for the layer's two first stages (they are independent, and each alone
// leaves most of the chip idle at the sizes taken here).
template <int IT, bool WHOLE>
__global__ __launch_bounds__(kAlignThreads) void quant_align_kernel(AlignArgs a, QuantArgs q) {
  if ((int)blockIdx.x < a.E)
    align_expert<IT>(a, blockIdx.x);
  else
    quant_chunks<kAlignThreads, 1, false, WHOLE>(q, (int64_t)blockIdx.x - a.E);
}

// The one-launch form holds up to 32 ids a lane.  Every workgroup reads every
// slot: with near 1024 experts and all 16384 slots align alone takes 16.5 to
// 18.6 us so and 16 in three launches (1024 experts, 8192 slots: 11.2 to 12.4
// and 14; 256, 16384: 7.2 and 13), which only the layer's table of runs outweighs.
constexpr int64_t kAlignOneLaunchReads = (int64_t)12 << 20;
constexpr int64_t kAlignOneLaunchSlots = 32 * kAlignThreads;
static_assert(kAlignOneLaunchSlots == kRunsMaxSlots, "the one-launch form writes the table of runs");
// Chunks (16 B of input) up to which the quant runs beside align; larger ones
// are bound by HBM and take the quant kernel's own block and unroll.
constexpr int64_t kQuantBesideAlign = (int64_t)1 << 22;

}  // namespace moe

using namespace moe;

extern "C" int64_t moe_align_max_padded(int64_t S, int32_t E, int32_t BM) {
  if (S < 0 || E <= 0 || BM <= 0) return -1;
  int64_t m = S + (int64_t)E * (BM - 1);
  if (S < E) m = (S * BM < m) ? S * BM : m;
  return m;
}

extern "C" int64_t moe_align_workspace_bytes(int64_t S, int32_t E) {
  if (S < 0 || E <= 0) return -1;
  const int64_t n_chunks = (S + kAlignChunk - 1) / kAlignChunk;
  // chunk counts [n_chunks][E], rank [S], off [E+1], cnt [E]
  return 4 * (n_chunks * E + S + 2 * (int64_t)E + 1) + 256;
}

// Every argument check of an align call, before any device work; the
// workspace pointer is checked only when the caller supplies one.
static int align_args(const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM, int32_t* sorted_ids,
                      int32_t* expert_ids, int32_t* ntpp, int64_t max_padded, bool need_ws, const void* workspace) {
  if (S < 0) return kErrBadShape;
  if (E <= 0 || E > kAlignMaxExperts) return kErrBadExperts;
  if (!block_m_ok(BM)) return kErrBadBlockSize;
  if (!sorted_ids || !expert_ids || !ntpp || (need_ws && !workspace) || (S > 0 && !topk_ids))
    return kErrNullPointer;
  if (max_padded < moe_align_max_padded(S, E, BM)) return kErrCapacity;
  if (S > 0x7FFFFFFF - 1 || max_padded > 0x7FFFFFFF) return kErrBadShape;
  return kOk;
}

static bool align_one_launch(int64_t S, int32_t E, const int32_t* runs) {
  return S <= kAlignOneLaunchSlots && (runs || S * E <= kAlignOneLaunchReads);
}

// f(ids a lane holds) for the one-launch form.
template <class F>
static void by_slots(int64_t S, F&& f) {
  if (S <= 2 * kAlignThreads) f(std::integral_constant<int, 2>{});
  else if (S <= 8 * kAlignThreads) f(std::integral_constant<int, 8>{});
  else if (S <= 16 * kAlignThreads) f(std::integral_constant<int, 16>{});
  else f(std::integral_constant<int, 32>{});
}

static int align_impl(const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM, const int32_t* expert_map,
                      int32_t* sorted_ids, int32_t* expert_ids, int32_t* ntpp, int64_t max_padded,
                      void* workspace, void* stream, int32_t* local = nullptr, int32_t* runs = nullptr,
                      int32_t* share = nullptr, int32_t* share2 = nullptr, int32_t top_k = 1) {
  const int arg_rc = align_args(topk_ids, S, E, BM, sorted_ids, expert_ids, ntpp, max_padded, true, workspace);
  if (arg_rc != kOk) return arg_rc;
  if (!expert_map) local = nullptr;
  hipStream_t st = (hipStream_t)stream;
  if (align_one_launch(S, E, runs)) {
    const AlignArgs a{topk_ids, expert_map, sorted_ids, expert_ids, ntpp, local, runs, share, share2,
                      (int)max_padded, (int)S, (int)top_k, (uint16_t)E, (uint16_t)BM};
    by_slots(S, [&](auto it) {
      hipLaunchKernelGGL(align_expert_kernel<decltype(it)::value>, dim3((unsigned)E), dim3(kAlignThreads), 0, st, a);
    });
    return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
  }
  const int64_t n_chunks = (S + kAlignChunk - 1) / kAlignChunk;
  int32_t* chunk_count = (int32_t*)workspace;
  int32_t* rank = chunk_count + n_chunks * E;
  int32_t* off = rank + S;
  int32_t* cnt = off + E + 1;
  int nbits = 0;
  while ((1 << nbits) < E) ++nbits;
  if (n_chunks > 0) {
    hipLaunchKernelGGL(align_count_kernel, dim3((unsigned)n_chunks), dim3(kAlignChunk),
                       16 * E * sizeof(int32_t), st, topk_ids, S, (int)E, nbits, chunk_count,
                       rank);
  }
  // Stage the chunk counts in LDS when they fit (128 KiB of the 160 KiB).
  // Set once per process (thread-safe initialisation of a function-local static).
  static const hipError_t lds_attr_rc = hipFuncSetAttribute(
      (const void*)align_scan_kernel, hipFuncAttributeMaxDynamicSharedMemorySize,
      (int)(kAlignStageLimit * sizeof(int32_t)));
  if (lds_attr_rc != hipSuccess) return kErrLaunch;
  const int use_lds = n_chunks * E <= kAlignStageLimit ? 1 : 0;
  hipLaunchKernelGGL(align_scan_kernel, dim3(1), dim3(kAlignMaxExperts),
                     use_lds ? (size_t)(n_chunks * E * sizeof(int32_t)) : 0, st, chunk_count, n_chunks,
                     (int)E, (int)BM, use_lds, off, cnt, ntpp, share, share2);
  const int64_t wide = S > max_padded ? S : max_padded;
  if (wide > 0) {
    hipLaunchKernelGGL(align_place_kernel, dim3((unsigned)((wide + 255) / 256)), dim3(256), 0, st,
                       topk_ids, S, (int)E, (int)BM, chunk_count, rank, off, cnt, expert_map,
                       sorted_ids, expert_ids, max_padded);
  }
  if (local)
    hipLaunchKernelGGL(local_blocks_kernel, dim3((unsigned)(1 + (S / top_k + 1023) / 1024)), dim3(1024), 0, st,
                       topk_ids, S, (int)E, (int)top_k, expert_map, sorted_ids, expert_ids, ntpp, (int)BM, max_padded, local);
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

int moe::quant_align(const void* x_bf16, int64_t T, int64_t H, void* q_fp8, int64_t ldq, float* scales,
                     const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM, const int32_t* expert_map,
                     int32_t* sorted_ids, int32_t* expert_ids, int32_t* ntpp, int64_t max_padded, void* workspace,
                     int32_t* local, int32_t* runs, int32_t* share, int32_t* share2, int32_t top_k, void* stream) {
  // both halves' arguments before either is launched
  if (top_k <= 0) return kErrBadTopK;
  if (T < 0 || H < 0 || ldq < (H + 127) / 128 * 128) return kErrBadShape;
  if (T > 0 && H > 0) {
    if (!x_bf16 || !q_fp8 || !scales) return kErrNullPointer;
    if (((uintptr_t)x_bf16 & 1) != 0) return kErrBadShape;
  }
  const int rc = align_args(topk_ids, S, E, BM, sorted_ids, expert_ids, ntpp, max_padded, true, workspace);
  if (rc != kOk) return rc;
  const QuantArgs q = quant_args(x_bf16, T, H, q_fp8, ldq, scales);
  if (!align_one_launch(S, E, runs) || q.n_chunks == 0 || q.n_chunks > kQuantBesideAlign ||
      !quant_vectorised(x_bf16, H, q_fp8, ldq)) {
    const int qrc = moe_quant_group128_padded(x_bf16, T, H, q_fp8, ldq, scales, stream);
    if (qrc != kOk) return qrc;
    return align_impl(topk_ids, S, E, BM, expert_map, sorted_ids, expert_ids, ntpp, max_padded, workspace, stream,
                      local, runs, share, share2, top_k);
  }
  if (!expert_map) local = nullptr;
  const AlignArgs a{topk_ids, expert_map, sorted_ids, expert_ids, ntpp, local, runs, share, share2,
                      (int)max_padded, (int)S, (int)top_k, (uint16_t)E, (uint16_t)BM};
  const unsigned grid = (unsigned)(E + (q.n_chunks + kAlignThreads - 1) / kAlignThreads);
  by_slots(S, [&](auto it) {
    constexpr int IT = decltype(it)::value;
    if (quant_whole(q))
      hipLaunchKernelGGL((quant_align_kernel<IT, true>), dim3(grid), dim3(kAlignThreads), 0, (hipStream_t)stream, a, q);
    else
      hipLaunchKernelGGL((quant_align_kernel<IT, false>), dim3(grid), dim3(kAlignThreads), 0, (hipStream_t)stream, a, q);
  });
  return hipGetLastError() == hipSuccess ? kOk : kErrLaunch;
}

extern "C" int moe_quant_align(const void* x_bf16, int64_t T, int64_t H, void* q_fp8, int64_t ldq, float* scales,
                               const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM,
                               const int32_t* expert_map, int32_t* sorted_ids, int32_t* expert_ids, int32_t* ntpp,
                               int64_t max_padded, void* workspace, void* stream) {
  return quant_align(x_bf16, T, H, q_fp8, ldq, scales, topk_ids, S, E, BM, expert_map, sorted_ids, expert_ids, ntpp,
                     max_padded, workspace, nullptr, nullptr, nullptr, nullptr, 1, stream);
}

extern "C" int moe_align_block_size(const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM,
                                    int32_t* sorted_ids, int32_t* expert_ids, int32_t* ntpp,
                                    int64_t max_padded, void* workspace, void* stream) {
  return align_impl(topk_ids, S, E, BM, nullptr, sorted_ids, expert_ids, ntpp, max_padded, workspace, stream);
}

extern "C" int moe_align_block_size_mapped(const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM,
                                           const int32_t* expert_map, int32_t* sorted_ids,
                                           int32_t* expert_ids, int32_t* ntpp, int64_t max_padded,
                                           void* workspace, void* stream) {
  if (!expert_map) return kErrNullPointer;
  return align_impl(topk_ids, S, E, BM, expert_map, sorted_ids, expert_ids, ntpp, max_padded, workspace,
                    stream);
}

// ---------------------------------------------------------------------------
// Allocation-free align: the same kernels, the three launches with their
// workspace in a file-scope device array instead of caller memory, for callers
// that cannot allocate (code under graph capture, tight serving loops).  Each
// GPU holds its own copy of the array until the process ends; every call on a
// GPU that takes three launches shares it, so such calls race where they
// overlap.  Nothing in the workspace needs clearing: every call writes each
// chunk count, rank, offset and count that it later reads.  (The one launch
// uses no workspace.)

namespace moe {

constexpr int64_t kNoAllocScratchBytes = MOE_ALIGN_NOALLOC_SCRATCH_BYTES;
constexpr int kMaxDevices = 64;

static __device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

// The array's device address on the current GPU, looked up once per device
// with that device current (the host-side name is only a stand-in).
static int scratch_for_current_device(void** out) {
  static std::mutex mu;
  static void* ptr[kMaxDevices] = {};
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return kErrLaunch;
  std::lock_guard<std::mutex> lock(mu);
  if (!ptr[dev]) {
    void* p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return kErrLaunch;
    ptr[dev] = p;
  }
  *out = ptr[dev];
  return kOk;
}

}  // namespace moe

extern "C" int moe_align_block_size_noalloc(const int32_t* topk_ids, int64_t S, int32_t E, int32_t BM,
                                            int32_t* sorted_ids, int32_t* expert_ids, int32_t* ntpp,
                                            int64_t max_padded, void* stream) {
  // every argument is checked before the device is touched (symbol lookup)
  const int arg_rc = align_args(topk_ids, S, E, BM, sorted_ids, expert_ids, ntpp, max_padded, false, nullptr);
  if (arg_rc != kOk) return arg_rc;
  if (moe_align_workspace_bytes(S, E) > kNoAllocScratchBytes) return kErrCapacity;
  void* ws = nullptr;
  const int rc = scratch_for_current_device(&ws);
  if (rc != kOk) return rc;
  return align_impl(topk_ids, S, E, BM, nullptr, sorted_ids, expert_ids, ntpp, max_padded, ws, stream);
}
