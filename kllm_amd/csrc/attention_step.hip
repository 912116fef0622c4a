// Attention of a step that has both kinds of tokens, those of short spans (attention_decode.hpp) and blocks of longer ones (attention_prompt.hpp), in one
// launch: the former wait for memory, the latter for their products, each on a part of the chip (see step_workgroups for when and what it gives).
// A step of 20 tokens and 480 of a prompt at 7B Llama sizes: 10,240 -> 9,640 us.
#include <math.h>

#include "attention_decode.hpp"
#include "attention_merge.hpp"
#include "attention_prompt.hpp"
#include "common.hpp"
#include "kllm_kernels.h"

namespace kllm {

constexpr int kStepWaves = 8;       // of a workgroup, whichever it takes

// Workgroups 0 ... items - 1 take a block of queries and a head each, longest first (their chains of tiles are what a step waits for), the rest
// a token, a KV head and a share of its keys each.
template <int HDT>   // head_dim = 32 * HDT
__global__ __launch_bounds__(64 * kStepWaves) __attribute__((amdgpu_waves_per_eu(2))) void attn_step_kernel(
    const bf16_t* __restrict__ cache, const int* __restrict__ positions, const int* __restrict__ span_of_token,
    const int* __restrict__ block_table, const int* __restrict__ token_list, const bf16_t* __restrict__ q, int max_pages, int KV,
    bf16_t* __restrict__ out, float* __restrict__ part, int H, int G, int page16, int wgs, unsigned page_magic, unsigned slice_magic, int window, int chunk,
    const float* __restrict__ sinks, float scale, int head_tiles, int count, int items, const int* __restrict__ query_tiles, int n_tiles,
    const int* __restrict__ span_start, const int* __restrict__ span_pos, unsigned prompt_page_magic, const OutGate gate) {
  const int id = blockIdx.x;
  if (id < items) {
    attn_prompt_block<HDT, kStepWaves / 4>(q, out, cache, query_tiles, n_tiles, span_start, span_pos, block_table, max_pages, 16 * page16,
                                           prompt_page_magic, H, KV, window, chunk, sinks, 0, scale, nullptr, gate, id, 0, 1);
    return;
  }
  const int place = id - items, rest = place / count;          // token fastest
  attn_decode_block<2 * HDT, kStepWaves, false, false, false>(cache, positions, span_of_token, block_table, token_list, q, max_pages, KV, out, part, H, G,
                                                              page16, wgs, page_magic, slice_magic, window, chunk, sinks, 0, scale, nullptr,
                                                              head_tiles, gate, place - rest * count, rest / wgs, rest % wgs);
}

template <int HDT>
static int launch_step(const void* q, void* out, float* part, const void* cache, const int* positions, const int* span_of_token, const int* block_table,
                       int max_pages, int page_size, int H, int KV, int window, int chunk, const float* sinks, float scale, int wgs, const int* token_list,
                       int count, const int* query_tiles, int n_tiles, const int* span_start, const int* span_pos, const OutGate& gate, hipStream_t stream) {
  typedef PromptShape<HDT> S;
  constexpr size_t prompt_lds = (size_t)(kStepWaves / 4) * S::RING * 2 * S::TB, decode_lds = (size_t)kStepWaves * 16 * (32 * HDT + 4) * sizeof(float);
  constexpr size_t lds = prompt_lds > decode_lds ? prompt_lds : decode_lds;
  static int raised = 0;
  if (!raised) {
    const hipError_t e = hipFuncSetAttribute((const void*)attn_step_kernel<HDT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) KLLM_FAIL((int)e, "attn_step: cannot raise the LDS limit: %s", hipGetErrorString(e));
    raised = 1;
  }
  const int head_tiles = (H / KV + 15) / 16, items = n_tiles * H;
  const unsigned page16 = page_size / 16, slices = wgs * kStepWaves;
  const unsigned page_magic = page16 == 1 ? 0xFFFFFFFFu : (unsigned)((1ull << 32) / page16), slice_magic = (unsigned)((1ull << 32) / slices);
  const unsigned prompt_page_magic = (unsigned)(((1UL << 35) + page_size - 1) / page_size);
  hipLaunchKernelGGL((attn_step_kernel<HDT>), dim3(items + count * KV * head_tiles * wgs), dim3(64 * kStepWaves), lds, stream, (const bf16_t*)cache, positions,
                     span_of_token, block_table, token_list, (const bf16_t*)q, max_pages, KV, (bf16_t*)out, part, H, H / KV, (int)page16, wgs, page_magic,
                     slice_magic, window, chunk, sinks, scale, head_tiles, count, items, query_tiles, n_tiles, span_start, span_pos, prompt_page_magic, gate);
  KLLM_CHECK_LAUNCH("attn_step");
  if (wgs > 1) {
    launch_attn_merge<bf16_t>((bf16_t*)out, part, count, H, 32 * HDT, wgs, token_list, gate, stream);
    KLLM_CHECK_LAUNCH("attn_merge");
  }
  return 0;
}

// Workgroups to a token and KV head in the one launch, or 0 where two launches are faster.
//
// Apart, the tokens' kernel waits for memory while the blocks' one multiplies on what are often a quarter of the CUs; together the shorter of the two
// hides behind the other.  And since the step waits for the blocks' chains of tiles anyway, a token's keys go to so few workgroups that theirs take
// about as long (3 us more at most, which their results' way through memory and the merge's launch would take): mostly one, and no merge.  us,
// two launches / one (operands in the caches): 20 tokens at 560 keys and 480 of a prompt behind 1,440, 32 KV heads of 128 59 / 43, behind none 43 / 33;
// 4 at 300 and 300 33.5 / 25.8 behind 900; 20 at 500 and 500 with 8 KV heads 28 / 17; 4 KV heads of 64: 32 at 1,400 and 640 23 / 18, 10 at 700 and
// 300 14 / 8.2, 2 at 100 and 40 8.5 / 6.0, 256 at 600 and 200 31.5 / 29.9.
// Two launches: where the blocks' keys go in slices and their chain whole would take longer than their sliced launch, its merge and the tokens' one (4 at
// 300 and 100 behind 2,000, 32 KV heads of 128 29 / 36; behind 1,200 25.6 / 26.3; 20 at 400 and 100 behind 2,000 42 / 38, behind 3,400 47 / 56; 12 at
// 400 and 500 behind 2,000, 8 KV heads 45 / 42, behind 6,000 77 / 95); where more blocks than half the CUs are better off with one group of waves
// each, several to a CU, which this kernel has no room for (16 at 1,000 and four prompts of 300, 8 KV heads of 128 31.3 / 32.4; 4 at 900 and eight prompts
// of 30 12 / 19; but four prompts of 100 15.5 / 14.6).
static int step_workgroups(int hdt, int n_tiles, int H, int KV, int count, int max_pages, int page_size, int nslices, long keys_total, int keys_longest,
                           int block_slices) {
  const long cus = device_cus(), items = (long)n_tiles * H, groups = (long)count * KV * ((H / KV + 15) / 16);
  const float chain = 6.f + keys_longest / 64.f * (hdt > 2 ? 0.9f : 0.55f);
  if (block_slices > 1 && keys_longest >= kPrefillSliceFromKeys) {
    const float sliced = 11.f + keys_longest / (64.f * block_slices) * 1.05f + 0.77f * n_tiles * block_slices;
    if (chain + 3.f > sliced + fmaxf(7.f, 8.f * groups / cus)) return 0;
  }
  long pages = 8;                       // (a table's width, rounded as for recorded steps: both cut the keys alike)
  while (pages < max_pages) pages *= 2;
  const float keys = (float)(pages * page_size) / (32 * kStepWaves);
  int wgs = 1;
  while (wgs < (nslices + 1) / 2 && 4.f + 0.7f * keys / wgs > chain + 3.f) wgs *= 2;
  if (wgs > (nslices + 1) / 2) wgs = (nslices + 1) / 2;      // (the workspace has room for nslices; two workgroups of four waves each are one here)
  if (2 * items > cus && items + groups * wgs > cus && prompt_groups(hdt, (int)items, H, keys_total, keys_longest) != 2) return 0;
  return wgs;
}

}  // namespace kllm

using namespace kllm;

extern "C" int kllm_attn_step(const void* q, void* out, float* part, long part_floats, const void* cache, const int* positions, const int* span_of_token,
                              const int* block_table, int max_pages, int page_size, int n, int H, int KV, int hd, int window, int chunk, const float* sinks,
                              int keep_first, float scale, const float* slopes, int nslices, int dtype, const int* token_list, int n_listed,
                              const int* query_tiles, int n_tiles, const int* span_start, const int* span_pos, long keys_total, int keys_longest,
                              float* block_part, long block_part_floats, int block_slices, const float* gate_sums, int gate_nsplit, long gate_stride,
                              long gate_row, int gate_width, int out_side, hipStream_t stream) {
  const bool built = dtype == DT_BF16 && (hd == 64 || hd == 128) && !slopes && keep_first == 0 && out_side == 0 && token_list;
  const bool fits = built && q && out && part && cache && positions && span_of_token && block_table && query_tiles && span_start && span_pos &&
                    (((uintptr_t)q | (uintptr_t)out | (uintptr_t)cache | (uintptr_t)part) & 15) == 0 && direct_pages(cache, KV, hd, page_size, sizeof(bf16_t)) &&
                    n > 0 && H > 0 && KV > 0 && H % KV == 0 &&
                    page_size > 0 && page_size % 16 == 0 && page_size <= kPrefillMaxPage && max_pages > 0 && (long)max_pages * page_size <= kPrefillMaxKeys &&
                    window >= 0 && chunk >= 0 && nslices >= 1 && nslices <= 256 && part_floats >= (long)n * H * nslices * (hd + 2) && n_listed > 0 &&
                    n_listed <= n && n_tiles > 0 && keys_total > 0 && keys_longest > 0 &&
                    (!gate_sums || (gate_nsplit >= 1 && gate_width > 0 && gate_width <= hd && gate_row >= (long)H * gate_width)) &&
                    (long)n_tiles * H + (long)n_listed * (KV + H) * nslices < (1L << 31);
  const int wgs = fits ? step_workgroups(hd / 32, n_tiles, H, KV, n_listed, max_pages, page_size, nslices, keys_total, keys_longest, block_slices) : 0;
  if (wgs) {
    const OutGate gate = {gate_sums, gate_nsplit, gate_width, gate_stride, gate_row, 0};
    return hd == 64 ? launch_step<2>(q, out, part, cache, positions, span_of_token, block_table, max_pages, page_size, H, KV, window, chunk, sinks, scale, wgs,
                                     token_list, n_listed, query_tiles, n_tiles, span_start, span_pos, gate, stream)
                    : launch_step<4>(q, out, part, cache, positions, span_of_token, block_table, max_pages, page_size, H, KV, window, chunk, sinks, scale, wgs,
                                     token_list, n_listed, query_tiles, n_tiles, span_start, span_pos, gate, stream);
  }
  if (int rc = kllm_attn_decode(q, out, part, part_floats, cache, positions, span_of_token, block_table, max_pages, page_size, n, H, KV, hd, window, chunk, sinks,
                                keep_first, scale, slopes, nslices, dtype, token_list, n_listed, gate_sums, gate_nsplit, gate_stride, gate_row, gate_width,
                                out_side, stream))
    return rc;
  return kllm_attn_prefill(q, out, cache, query_tiles, n_tiles, span_start, span_pos, block_table, max_pages, page_size, H, KV, hd, window, chunk, sinks,
                           keep_first, scale, slopes, keys_total, keys_longest, block_part, block_part_floats, block_slices, n, dtype, gate_sums, gate_nsplit,
                           gate_stride, gate_row, gate_width, out_side, stream);
}
