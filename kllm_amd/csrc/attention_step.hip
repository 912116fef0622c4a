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
// hides behind the other.  A workgroup of a token takes about 2.1 us for 256 keys of a KV head of 64, 3.5 of 128 (its eight waves' loads from one CU),
// and 5 beside them; several leave partial results and a merge, 4 us.  As many as make the launch shortest, by the longest chain of tiles, the longest
// token's keys and the CUs' rounds of workgroups (a CU holds one): one where the chain is
// longer anyway, up to what two launches would take where it is short.  us, two launches / one with one, two, four ... workgroups: one token at 4,400 keys and 45 of
// a prompt, 8 KV heads of 128 14.8 / 55, 37, 22, 14, 12; 4 at 4,088 and 184, 4 KV heads of 128 21.8 / 63, 38, 24, 17.7, 16.7; 16 at 1,492 behind a window of 1,024 and
// 75, 2 of 128 16.0 / 24.5, 23.6, 16.6, 12.0; 20 at 560 and 480 of a prompt behind 1,440, 32 KV heads of 128 77 / 58, 8 of 128 51 / 36; 32 at 1,400 and 640, 4 KV heads of
// 64 34.7 / 29.9; 2 at 100 and 40, 32 of 128 13.4 / 7.4.  (When a round of 256 keys of a table's width was taken for 0.7 us, whatever the head and the
// window: in 34 of 500 drawn steps the one launch was more than 3 % slower than two, by up to 2.5 times; now in 3, by up to 1.06.)
// Two launches: where the blocks' keys go in slices and this launch would take longer than theirs, its merge and the tokens' one (8 at 17 and
// one block of 2,224 keys, 12 heads of 128 27 / 36; 27 at 53 and 2,184, 16 heads 33 / 39; 20 at 400 and 100 behind 3,400, 32 KV heads 47 / 56); where
// more blocks than half the CUs are better off with one group of waves
// each, several to a CU, which this kernel has no room for (16 at 1,000 and four prompts of 300, 8 KV heads of 128 31.3 / 32.4; 4 at 900 and eight prompts
// of 30 12 / 19; but four prompts of 100 15.5 / 14.6).
static int step_workgroups(int hdt, int n_tiles, int H, int KV, int count, int max_pages, int page_size, int nslices, long keys_total, int keys_longest,
                           int keys_token, int block_slices, int window, int chunk) {
  const float cus = device_cus(), chain = 6.f + keys_longest / 64.f * (hdt > 2 ? 0.9f : 0.55f), merge = 4.f;
  const long items = (long)n_tiles * H, groups = (long)count * KV * ((H / KV + 15) / 16);
  long keys = keys_token > 0 ? keys_token : (long)max_pages * page_size;
  if (window > 0 && keys > window + 32) keys = window + 32;
  if (chunk > 0 && keys > chunk) keys = chunk;
  const float round = (hdt > 2 ? 3.5f : 2.1f) * keys / (32.f * kStepWaves);   // a token's keys in one workgroup
  const int most = (nslices + 1) / 2;   // (the workspace has room for nslices; two workgroups of four waves each are one here)
  int wgs = 1;
  float best = INFINITY;
  for (int w = 1;; w *= 2) {
    const int n = w < most ? w : most;
    const float token = 5.f + round / n;
    float t = fmaxf(chain, token);
    const float rounds = (groups * n + items * chain / token) / cus;           // (the last one as if half of what it leaves idle were)
    if (items + groups * n > cus) t = fmaxf(t, token * 0.5f * (rounds + ceilf(rounds)));
    if (n > 1) t += merge;
    if (t < best - 0.01f) {
      best = t;
      wgs = n;
    }
    if (w >= most) break;
  }
  if (block_slices > 1 && keys_longest >= kPrefillSliceFromKeys) {
    const float sliced = 11.f + keys_longest / (64.f * block_slices) * 1.05f + 0.4f * n_tiles * block_slices;
    const float token = 5.f + (nslices == 1 ? round : 2.f * round / nslices);            // (four waves to a workgroup, two of them to a CU)
    const float tokens = fmaxf(token, groups * token * (nslices == 1 ? 1.f : 0.5f * nslices) / cus) + (nslices > 1 ? merge : 0.f);
    if (best + 4.f > sliced + tokens) return 0;
  }
  if (2 * items > cus && items + groups * wgs > cus && prompt_groups(hdt, (int)items, H, keys_total, keys_longest) != 2) return 0;
  return wgs;
}

}  // namespace kllm

using namespace kllm;

extern "C" int kllm_attn_step_workgroups(int hd, int n_tiles, int H, int KV, int count, int max_pages, int page_size, int nslices, long keys_total,
                                         int keys_longest, int keys_token, int block_slices, int window, int chunk) {
  if ((hd != 64 && hd != 128) || n_tiles <= 0 || KV <= 0 || H % KV || count <= 0 || max_pages <= 0 || page_size <= 0 || nslices < 1 || keys_total <= 0 ||
      keys_longest <= 0)
    return 0;
  return step_workgroups(hd / 32, n_tiles, H, KV, count, max_pages, page_size, nslices, keys_total, keys_longest, keys_token, block_slices, window,
                         chunk);
}

extern "C" int kllm_attn_step(const void* q, void* out, float* part, long part_floats, const void* cache, const int* positions, const int* span_of_token,
                              const int* block_table, int max_pages, int page_size, int n, int H, int KV, int hd, int window, int chunk, const float* sinks,
                              int keep_first, float scale, const float* slopes, int nslices, int dtype, const int* token_list, int n_listed,
                              const int* query_tiles, int n_tiles, const int* span_start, const int* span_pos, long keys_total, int keys_longest,
                              int keys_token, float* block_part, long block_part_floats, int block_slices, const float* gate_sums, int gate_nsplit, long gate_stride,
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
  const int wgs = fits ? step_workgroups(hd / 32, n_tiles, H, KV, n_listed, max_pages, page_size, nslices, keys_total, keys_longest, keys_token,
                                          block_slices, window, chunk) : 0;
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
