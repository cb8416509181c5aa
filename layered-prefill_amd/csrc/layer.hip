// The expert MLP from routing to combine as one call: moe_layer enqueues whatever kernels suit the
// batch: the router, the alignment of the ids by expert and moe_fused_experts.
//
// Replaces the sequence of nanovllm/layers/fused_moe.py:163-216 (select_experts, fused_experts) and
// nanovllm/layers/for_moe/fused_moe.py:547-631 of the reference, whose host enqueues the steps apart.
#include "common.h"

namespace {

struct Carver {   // places regions of a workspace one behind the other
  char* base;
  int64_t at = 0;
  void* take(int64_t bytes) {
    void* p = base + at;
    at += moe_align_up(bytes, 256);
    return p;
  }
};

// Where everything sits in the workspace of a call.
struct Layout {
  int block;
  int64_t sorted_cap, expert_cap, align_bytes, fused_bytes, bytes;
  float* topk_w;
  int32_t *topk_ids, *sorted, *experts, *npp;
  void *align_ws, *fused_ws;
};
Layout layout_of(const MoeLayerArgs* a) {
  Layout l{};
  Carver c{static_cast<char*>(a->workspace)};
  const int64_t numel = static_cast<int64_t>(a->T) * a->K;
  if (a->router_logits) {
    l.topk_w = static_cast<float*>(c.take(numel * 4));
    l.topk_ids = static_cast<int32_t*>(c.take(numel * 4));
  } else {
    l.topk_w = a->topk_weights;
    l.topk_ids = a->topk_ids;
  }
  l.block = a->block_size ? a->block_size
                          : moe_call_block_size(a->T, a->H, a->I, a->E, a->K, a->act_dtype, a->weight_dtype, a->weight_layout);
  l.sorted_cap = numel + static_cast<int64_t>(a->E) * (l.block - 1);
  l.expert_cap = (l.sorted_cap + l.block - 1) / l.block;
  l.align_bytes = moe_align_workspace_bytes(numel, a->E);
  l.fused_bytes = moe_fused_experts_workspace_bytes(a->T, a->H, a->I, a->E, a->K, l.block, a->act_dtype, a->weight_dtype);
  l.sorted = static_cast<int32_t*>(c.take(l.sorted_cap * 4));
  l.experts = static_cast<int32_t*>(c.take(l.expert_cap * 4));
  l.npp = static_cast<int32_t*>(c.take(4));
  l.align_ws = c.take(l.align_bytes);
  l.fused_ws = c.take(l.fused_bytes);
  l.bytes = c.at;
  return l;
}

int check_layer_args(const MoeLayerArgs* a) {
  if (!a) return moe_fail(MOE_ERR_ARG, "layer: null argument block");
  if (a->T < 0 || a->H < 1 || a->I < 1 || a->E < 1 || a->K < 1 || a->block_size < 0)
    return moe_fail(MOE_ERR_ARG, "layer: bad sizes T=%d H=%d I=%d E=%d K=%d block_size=%d", a->T, a->H, a->I, a->E, a->K,
                    a->block_size);
  if (static_cast<int64_t>(a->T) * a->K > INT32_MAX) return moe_fail(MOE_ERR_ARG, "layer: T*K overflows int32");
  return MOE_OK;
}

}  // namespace

// Block size of a call that does not name one: 256 (large-tile kernel) or 32 (streaming kernel, with the large tile's
// roundings where that would do as well: passes bit 64 of moe_fused_experts).  The streaming kernel reads the weights
// again for every 32 rows of an expert; the large tile leaves CUs idle where there are few tiles, and its blocks half empty
// where experts have few rows.  What decides between them is the call's matrix work, T * K * H * I, with 40000 beside H * I
// for what a routed row costs outside its products (rows of narrow layers).  Measured over 1233 points, whole layer, Zipf
// routing: 1 to 128 experts, H 128 to 4096, I 128 to 1440, 16 to 4000 routed rows per expert.  Mean and worst excess over the
// faster of the two, by this rule and by rows and tiles (moe_layer_block_size):
//   16 bit, plain weights, line 3.4e9: 0.5 % and 15 %; 8.3 % and 118 %
//   16 bit, tiled weights, line 3.2e9: 0.5 % and 16 %; 3.1 % and 51 %
//   16 bit, I 1440, line 1e10: 1.1 % and 22 %; 12.9 % and 68 %
//   e4m3, line 6e9: 0.7 % and 23 %; 8.4 % and 86 %.  e4m3, I 1440, line 2e10: 0.7 % and 19 %; 16 % and 67 %
// (H or I that is no whole number of the large tile's K units, as 1440 is not: that pass runs on the register-staged
// kernel at blocks of 256, and the line lies where it lies with that.)  For instance, us with blocks of 256 and of 32: 128
// experts, H 1024, I 512, 640 tokens top-4: 70.8 and 54.8; 128, H 2880, I 1440, 640 tokens: 489 and 407; 128, H 2048, I 768,
// 256 tokens top-8: plain 171 and 161, tiled 152 and 156; 16, H 2048, I 768, 384 tokens top-4: 1.25 times.  Fewer than 16
// (e4m3: 32) rows per expert always stream, as under the older rules.
// Every caller that enqueues a call's steps asks here, so that a call runs on the same kernels whichever way it is entered.
MOE_EXPORT int moe_call_block_size(int M, int H, int I, int E, int K, int act_dtype, int weight_dtype, int weight_layout) {
  const bool e4m3 = weight_dtype == MOE_E4M3;
  const int es = e4m3 ? 1 : 2;
  // rows that are no whole 32-byte steps run on the register-staged kernels with either block: the rule by rows and tiles
  if (E < 1 || H < 1 || I < 1 || act_dtype == MOE_F32 || weight_dtype == MOE_F32 || H * static_cast<int64_t>(es) % 32 ||
      I * static_cast<int64_t>(es) % 32)
    return moe_layer_block_size(M, I, E, K, act_dtype, weight_dtype);
  const int64_t numel = static_cast<int64_t>(M) * K;
  if (numel / E < (e4m3 ? 32 : 16)) return 32;
  const int unit = e4m3 ? 128 : 64;  // elements of a K unit of the large tile
  const bool whole = H % unit == 0 && I % unit == 0;
  const double line = e4m3 ? (whole ? 6e9 : 2e10) : !whole ? 1e10 : weight_layout == MOE_WEIGHTS_TILED ? 3.2e9 : 3.4e9;
  return static_cast<double>(numel) * (static_cast<double>(H) * I + 40000.) >= line ? 256 : 32;
}

// The rule for callers that know neither H nor the weights' layout; moe_call_block_size is the better one and the one that
// calls of this library take.
// Blocks of 256 slots (large-tile kernel) or of 32 (streaming kernel, with the large tile's roundings from its old
// line on: passes bit 64 of moe_fused_experts).  What the large tile costs below its crossover
// is idle CUs: an expert's weights are walked by I / 128 + H / 256 workgroups, each a serial chain of K tiles, and with
// `tiles` = E * ceil(I / 128) gate-up tiles for the 256 CUs a layer of few experts leaves the chip half empty, however
// many rows an expert has.  What the streaming kernel costs above it is re-reading the weights for every 32 rows.
// The crossover as measured when the line was drawn, in routed rows per expert, both GEMM passes and the combine, Zipf
// routing:
//   bf16 tiles 768 (E 128, I 768): 24; 384 (E 64): 44; 256 (E 32, I 1024): 64; 96 (E 16, I 768; E 32, I 384): 97 and 115;
//   64 (E 16, I 512): beyond 128.  e4m3 tiles 768: 34; 256: 84; 64: beyond 96.  The 16-bit line lies lower than these
//   because tiled weights favour the large tile.
// On the present kernels it gives calls to the large tile too early where weights are plain or the layer is narrow, by 3 to
// 16 % in the mean and up to 118 % (the figures at moe_call_block_size).
MOE_EXPORT int moe_layer_block_size(int M, int I, int E, int K, int act_dtype, int weight_dtype) {
  if (act_dtype == MOE_F32 || E < 1 || I < 0) return moe_preferred_block_size(M, E, K, act_dtype, weight_dtype);
  // An expert counts as six tiles at least: a caller that passes 0 for a size it does not know gets the line of I = 768.
  // (So do narrower experts, whose crossovers lie higher.)
  const int64_t per_expert = (static_cast<int64_t>(I) + 127) / 128;
  const int64_t tiles = static_cast<int64_t>(E) * (per_expert > 6 ? per_expert : 6);
  const int64_t rows = static_cast<int64_t>(M) * K / E;
  const int64_t line = weight_dtype == MOE_E4M3 ? 22528 : 12288, least = weight_dtype == MOE_E4M3 ? 32 : 16;
  if (rows < least) return 32;
  return rows >= 96 || rows * tiles >= line ? 256 : 32;
}

MOE_EXPORT int64_t moe_layer_workspace_bytes(const MoeLayerArgs* a) {
  if (check_layer_args(a)) return 0;
  return a->T == 0 ? 0 : layout_of(a).bytes;
}

MOE_EXPORT int moe_layer(const MoeLayerArgs* a) {
  if (int rc = check_layer_args(a)) return rc;
  if (a->T == 0) return MOE_OK;
  if (!a->x || !a->out || !a->w13 || !a->w2) return moe_fail(MOE_ERR_ARG, "layer: null tensor pointer");
  if (!a->router_logits && (!a->topk_weights || !a->topk_ids))
    return moe_fail(MOE_ERR_ARG, "layer: neither router_logits nor topk_weights and topk_ids");
  const Layout l = layout_of(a);
  if (!a->workspace || a->workspace_bytes < l.bytes)
    return moe_fail(MOE_ERR_WORKSPACE, "layer: workspace %lld B, needs %lld B", static_cast<long long>(a->workspace_bytes),
                    static_cast<long long>(l.bytes));
  if (reinterpret_cast<uintptr_t>(a->workspace) & 255u)
    return moe_fail(MOE_ERR_WORKSPACE, "layer: workspace must be 256-byte aligned");
  const int64_t numel = static_cast<int64_t>(a->T) * a->K;
  int rc = MOE_OK;
  if (moe_layer_few(a, l.topk_w, l.topk_ids, l.sorted, l.fused_ws, &rc)) return rc;
  // what the expert passes will be given (the routing of an e4m3 call leaves the codes of x in their workspace)
  MoeFusedExpertsArgs f{};
  f.workspace = l.fused_ws; f.workspace_bytes = l.fused_bytes;
  f.T = a->T; f.H = a->H; f.I = a->I; f.E = a->E; f.K = a->K;
  f.block_size = l.block; f.act_dtype = a->act_dtype; f.weight_dtype = a->weight_dtype;
  f.x = a->x; f.out = a->out; f.w13 = a->w13; f.w2 = a->w2;
  f.w13_bias = a->w13_bias; f.w2_bias = a->w2_bias; f.w13_scale = a->w13_scale; f.w2_scale = a->w2_scale;
  f.topk_weights = l.topk_w;
  f.sorted_token_ids = l.sorted; f.expert_ids = l.experts; f.num_tokens_post_pad = l.npp;
  f.w13_stride_e = a->w13_stride_e; f.w13_stride_n = a->w13_stride_n;
  f.w2_stride_e = a->w2_stride_e; f.w2_stride_n = a->w2_stride_n;
  f.sorted_cap = l.sorted_cap;
  f.activation = a->activation;
  f.apply_router_weight_on_input = a->apply_router_weight_on_input;
  f.swiglu_alpha = a->swiglu_alpha; f.swiglu_limit = a->swiglu_limit;
  f.weight_layout = a->weight_layout;
  f.stream = a->stream;
  // A few hundred ids are aligned by the gate-up pass itself; the launch that routes and aligns in one workgroup is for calls
  // whose gate-up pass does not.  Layer with the norm, us, that launch and this way: 128 experts, 12 tokens 62.8 and 60.0,
  // 14 65.2 and 62.4, e4m3 8 tokens 41.0 and 38.7, 16 49.1 and 47.0; 64 experts, 30 tokens 80.2 and 75.8; 32 experts, 60
  // tokens 71.0 and 69.3.
  const bool aligns = !a->block_size && moe_experts_align(&f);
  MoeXCodes xc{a->x, a->H, nullptr, nullptr};
  moe_experts_x_codes(&f, &xc.codes, &xc.scales);
  const bool code_x = a->router_logits && a->weight_dtype == MOE_E4M3 && a->logits_dtype == a->act_dtype && moe_x_codes_ok(xc);
  const bool routed = a->router_logits && !aligns &&
                      moe_layer_route_align(a->router_logits, a->logits_dtype, l.topk_w, a->T, a->E, a->K, a->renormalize, l.block,
                                            l.sorted, l.sorted_cap, l.experts, l.expert_cap, l.npp, code_x ? &xc : nullptr,
                                            static_cast<hipStream_t>(a->stream), &rc);
  if (rc) return rc;
  bool x_coded = routed && code_x;
  if (code_x && !routed)
    x_coded = moe_layer_route_quant(a->router_logits, a->logits_dtype, l.topk_w, l.topk_ids, a->T, a->E, a->K, a->renormalize, xc,
                                    static_cast<hipStream_t>(a->stream), &rc);
  if (rc) return rc;
  if (a->router_logits && !routed && !x_coded) {
    if (int rc = moe_topk_softmax_typed(a->router_logits, a->logits_dtype, l.topk_w, l.topk_ids, nullptr, a->T, a->E, a->K,
                                        a->renormalize, a->stream))
      return rc;
  }
  // align, with the large-tile kernel's plan left in its workspace when the sizes allow
  int64_t bounds_off = 0, done_off = 0;
  int32_t num_done = 0, cap_mb = 0;
  const bool plan = l.block == 256 && moe_align_can_plan(numel, a->E) &&
                    moe_fused_experts_plan_layout(a->T, a->H, a->I, a->E, a->K, l.block, a->act_dtype, a->weight_dtype,
                                                  &bounds_off, &done_off, &num_done, &cap_mb);
  char* fws = static_cast<char*>(l.fused_ws);
  f.passes = plan ? 16 : 0;
  // a block of 32 of the library's own choice where the large tile would also do: same roundings as that
  if (!a->block_size && l.block < moe_preferred_block_size(a->T, a->E, a->K, a->act_dtype, a->weight_dtype)) f.passes |= 64;
  if (plan)
    rc = moe_align_block_size_planned(l.topk_ids, MOE_ID_I32, numel, a->E, l.block, l.sorted, l.sorted_cap, l.experts,
                                      l.expert_cap, l.npp, l.align_ws, l.align_bytes, a->stream,
                                      reinterpret_cast<int32_t*>(fws + bounds_off), reinterpret_cast<int32_t*>(fws + done_off),
                                      num_done, cap_mb);
  else if (!routed && !aligns)
    rc = moe_align_block_size(l.topk_ids, MOE_ID_I32, numel, a->E, l.block, l.sorted, l.sorted_cap, l.experts, l.expert_cap,
                              l.npp, l.align_ws, l.align_bytes, a->stream);
  if (rc) return rc;
  return moe_fused_experts_of_codes(&f, x_coded, aligns ? l.topk_ids : nullptr);
}
