/*
 * prunepath_moe.h -- C ABI of the MI355X (gfx950) PrunePath sparse-MoE MLP path.
 *
 * Library: prune_path_openpangu-embedded-1b_amd/libprunepath_moe.so (hipcc, gfx950 only).
 * Every entry point takes plain device pointers, sizes and a hipStream_t passed as
 * void* (NULL = the null stream). Work is enqueued on that stream without any host
 * synchronisation and without allocating memory, so calls can be captured in a
 * hipGraph. Return value: PP_OK or an error code; pp_last_error() gives the message
 * of the last failure on the calling thread. Invalid shapes are rejected before any
 * launch.
 *
 * Shapes: H hidden size, E experts, G neurons per expert (I = E*G FFN width),
 * N tokens. Supported: H % 128 == 0 and 128 <= H <= 4096, 1 <= E <= 256,
 * G % 32 == 0 and 32 <= G <= 8192.
 *
 * Reference interfaces replaced (paths relative to the reference repository root):
 *   src/tl_kernel_optimized_Ultimate_PanGU.py  -- TauSparseMoE and its Triton kernels
 *   src/MoEBlock_origin.py                     -- softmax_thresholding / MoELayer routing
 *   src/openpangu_moe.py                       -- physical_reorder_for_inference
 */
#ifndef PRUNEPATH_MOE_H
#define PRUNEPATH_MOE_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define PP_OK 0
#define PP_ERR_INVALID 1     /* bad shape / pointer / argument */
#define PP_ERR_HIP 2         /* a HIP runtime call failed */
#define PP_ERR_UNSUPPORTED 3 /* shape outside the supported range */

#define PP_DTYPE_F32 0
#define PP_DTYPE_BF16 1

#define PP_MAX_EXPERTS 256

/* Message of the last error on this thread ("" if none). */
const char* pp_last_error(void);
/* ABI version (incremented on any signature or workspace-layout change): 3. */
int pp_abi_version(void);

/* ------------------------------------------------------------------------- *
 * Rearrangement: one-time physical reorder of the expert weights.
 * Replaces physical_reorder_for_inference (src/openpangu_moe.py:212-256), which
 * argsorts neuron->expert ids and mounts W_gate/W_up [H,I], W_down [I,H] and
 * router [H,E] in bf16 on TauSparseMoE (src/tl_kernel_optimized_Ultimate_PanGU.py:483-486).
 *
 * Packed expert buffer (bf16), two regions:
 *   rows   [E*G][3][H]  for rearranged neuron j: gate row, up row, down column,
 *                       each H contiguous values (one 6*H-byte record per neuron);
 *   down_t [E][H][G]    the down projection of each expert with its G neurons
 *                       contiguous (K-contiguous operand of the prefill down GEMM).
 * Source element (neuron n, hidden h) is read at src[n*s_n + h*s_h] for gate and up
 * and at down[n*d_n + h*d_h] for down, so both the nn.Linear layout
 * (gate/up [I,H]: s_n=H, s_h=1; down [H,I]: d_n=1, d_h=I) and the TauSparseMoE
 * layout (W_gate [H,I]: s_n=1, s_h=I; W_down [I,H]: d_n=H, d_h=1) are accepted.
 * perm[j] (device int32 [I], may be NULL = identity) names the source neuron of
 * rearranged neuron j; expert e owns rearranged neurons e*G .. e*G+G-1.
 * ------------------------------------------------------------------------- */
size_t pp_packed_expert_bytes(int H, int E, int G);
int pp_pack_experts(const void* w_gate, const void* w_up, int64_t s_n, int64_t s_h,
                    const void* w_down, int64_t d_n, int64_t d_h, int src_dtype,
                    const int32_t* perm, int H, int E, int G, void* packed, void* stream);

/* Router weights to the fp32 [Epad][H] layout the kernels read (Epad = E rounded up
 * to 16, zero rows). Source element (expert e, hidden h) at src[e*s_e + h*s_h]:
 * MoELayer.mlp_router[0].weight [E,H] (src/MoEBlock_origin.py:127-129) or
 * TauSparseMoE.router [H,E] (src/tl_kernel_optimized_Ultimate_PanGU.py:486). */
size_t pp_packed_router_bytes(int H, int E);
int pp_pack_router(const void* w_router, int64_t s_e, int64_t s_h, int src_dtype,
                   int H, int E, float* router_packed, void* stream);

/* ------------------------------------------------------------------------- *
 * Routing: tau cumulative-probability expert selection.
 * Replaces softmax_thresholding (src/MoEBlock_origin.py:50-97) and the prefill
 * moe_router_kernel + torch.sort + moe_select_expert_kernel + scatter
 * (src/tl_kernel_optimized_Ultimate_PanGU.py:40-124, 550-564).
 * Semantics (bit-exact with torch CPU given the same fp32 logits):
 *   p = softmax(logits); order = torch.sort(p, descending) order; cum = fp32 of
 *   the float64 running sum of p in that order; selected = ranks r with
 *   cum[r] < (float)tau, and rank 0 always; gate = sigmoid(logit) on selected
 *   experts, 0 elsewhere.
 * Outputs (NULL = not written): logits/probs/gates fp32 [N,E]; mask uint8 [N,E];
 * count int32 [N] (selected experts per token).
 * ------------------------------------------------------------------------- */
int pp_route(const void* x, int x_dtype, int64_t n_tokens, int H,
             const float* router_packed, const float* bias, int E, float tau,
             float* logits_out, float* probs_out, float* gates_out,
             uint8_t* mask_out, int32_t* count_out, void* stream);
int pp_route_logits(const float* logits, int64_t n_tokens, int E, float tau,
                    float* probs_out, float* gates_out, uint8_t* mask_out,
                    int32_t* count_out, void* stream);

/* ------------------------------------------------------------------------- *
 * Bucketing: token -> expert CSR layout, experts ascending, tokens ascending
 * inside each expert (the order moe_local_scan_kernel / moe_global_scan_kernel /
 * moe_dispatch_kernel produce, src/tl_kernel_optimized_Ultimate_PanGU.py:133-266,
 * without the 16-row padding and without the total_tiles host sync at :581).
 *   offsets     int32 [E+1]
 *   token_ids   int32 [N*E] capacity, first offsets[E] used
 *   pair_gates  fp32  [N*E] capacity
 *   token_pairs int32 [N,E]: pair positions of token t in ascending expert id, -1 padded
 *   tiles       int32 [pp_max_tiles(N,E,tile_m)][4]: {expert, first pair, rows, 0}
 *   meta        int32 [4]: {number of tiles, number of pairs P, 0, 0}
 * workspace: pp_bucket_workspace_bytes(N, E) bytes of device scratch.
 * mask must be 4-byte aligned (it is read as 32-bit words); PP_ERR_INVALID otherwise.
 * ------------------------------------------------------------------------- */
size_t pp_bucket_workspace_bytes(int64_t n_tokens, int E);
/* Row-tile height the grouped GEMMs (pp_expert_gateup / pp_expert_down) expect
 * in the tile map; pass it as tile_m. */
int pp_gemm_tile_m(void);
int64_t pp_max_tiles(int64_t n_tokens, int E, int tile_m);
int pp_bucket(const uint8_t* mask, const float* gates, int64_t n_tokens, int E, int tile_m,
              int32_t* offsets, int32_t* token_ids, float* pair_gates, int32_t* token_pairs,
              int32_t* tiles, int32_t* meta, void* workspace, void* stream);

/* ------------------------------------------------------------------------- *
 * Decode (N == 1): one fused kernel -- router GEMV (fp32), selection, gate/up
 * GEMVs over the selected experts' neurons, silu(g)*u*gate, down GEMV, bf16 output.
 * Replaces TauSparseMoE.forward_decode with moe_router_select_kernel_decode and
 * moe_decode_swiglu_fused_kernel (src/tl_kernel_optimized_Ultimate_PanGU.py:335-462, 494-530).
 * Three kernels, by shape:
 *   E = 16, H % 512 == 0, G <= 512 (the configured shape): two phases in one launch.
 *     The gate/up records are spread over all workgroups and every act
 *     silu(g.x)*(u.x)*gate is published to the workspace; each workgroup then writes
 *     its own rows of the output as a fixed-order sum over the selected experts' down
 *     rows. Every workgroup waits for acts from all the others, so the grid is clamped
 *     to the workgroups the device holds at once (occupancy calculator) and to 1024;
 *     the automatic grid is one workgroup per CU.
 *   other shapes with E*G <= 8192 and G <= 512 (the checkpoint's E = 192, G = 32 among
 *     them): the same two phases; with E > 16 or 16*H > 32768 each logit is computed
 *     and published by its own workgroup and every workgroup gathers all E of them.
 *   the rest: each workgroup accumulates its records' act * down into a partial
 *     output, partials are summed in 64-bit fixed point (value * 2^32) and the last
 *     workgroup writes bf16.
 *   Where logits are published, the E router workgroups must be resident together:
 *   checked from the occupancy calculator before the launch (PP_ERR_UNSUPPORTED
 *   otherwise).
 * Both sum in an order that does not depend on timing: the bf16 output is the same bits
 * on every call. A wait that cannot finish (e.g. other work holding the device) ends
 * after a bounded spin with error bit 1 and NaN outputs, never a hang.
 * The workspace (pp_decode_workspace_bytes) must be zeroed once with
 * pp_decode_workspace_init before the first call; every call leaves it ready for
 * the next one. The init call also writes a layout tag into the workspace (the
 * library's workspace layout and the H it was sized for, pp_decode_layout_tag): a call
 * whose tag differs (a workspace initialised by another build of the library or for
 * another H, or never initialised) writes nothing into the workspace but error bit 8,
 * and NaN outputs. Calls that share a workspace must be ordered (same stream);
 * overlapping calls on one workspace race. After a call the workspace holds the
 * call's logits, selected experts and gates (struct pp_decode_state below).
 * grid = number of workgroups (0 = automatic).
 * ------------------------------------------------------------------------- */
typedef struct pp_decode_state {
  uint32_t router_ticket; /* internal: call epoch of the general kernel, advanced by one per call */
  uint32_t epoch16;       /* internal: call epoch of the E = 16 kernel, advanced by one per call */
  uint32_t epochb;        /* internal: call epoch of the batch kernel (pp_moe_decode_batch) */
  uint32_t error;         /* sticky error bits, 0 = none: 1 a logit-slot wait timed out
                             (every later call on the workspace writes NaN), 2 the selection
                             was not a permutation of the experts, 4 a workgroup partial sum
                             was not finite or reached 2^30 (beyond the fixed-point
                             reduction), 8 the workspace's layout tag did not match the call
                             (nothing else written); stays set until pp_decode_workspace_init
                             clears it */
  int32_t k;              /* experts selected by the last call */
  uint32_t error_call;    /* call epoch + 1 of the last failed call: that call wrote NaN outputs */
  uint32_t layout;        /* layout tag written by pp_decode_workspace_init (pp_decode_layout_tag) */
  int32_t pad;
  float logits[PP_MAX_EXPERTS];
  int32_t sel_ids[PP_MAX_EXPERTS];   /* selected experts, descending probability */
  float sel_gates[PP_MAX_EXPERTS];   /* sigmoid(logit) of each selected expert */
} pp_decode_state;

size_t pp_decode_workspace_bytes(int H, int E);
int pp_decode_workspace_init(void* workspace, int H, int E, void* stream);
/* The layout tag pp_decode_workspace_init writes for hidden size H (0 for an H outside
 * the shape limits). No counterpart in the reference (its decode keeps no workspace). */
uint32_t pp_decode_layout_tag(int H);
/* Checks a host copy of a workspace's state header against this library's layout for H:
 * PP_OK, or PP_ERR_INVALID (with the tags in pp_last_error) when the kernels would refuse
 * the workspace. No counterpart in the reference. */
int pp_decode_state_check(const pp_decode_state* state, int H);
int pp_moe_decode(const void* x, int x_dtype, int H, const float* router_packed,
                  const float* bias, int E, int G, float tau, const void* packed,
                  void* out_bf16, void* workspace, int grid, void* stream);

/* Allocation-free decode. No counterpart in the reference: for callers that cannot
 * allocate device memory (code under hipGraph capture, serving loops or harnesses that
 * forbid hipMalloc). Same arguments and results as pp_moe_decode without the workspace:
 * the library's own 596 KB device array is the workspace (one per GPU, zeroed by a fill
 * kernel on the caller's stream at the first call on that GPU, held until the process
 * ends). Limits: H <= 4096, E <= 256 (the library's shape limits; PP_ERR_UNSUPPORTED
 * beyond). Every call on a GPU shares that GPU's array: calls that overlap on one GPU
 * (different streams, threads or processes' graphs replayed concurrently) race; calls
 * ordered on one stream of any shapes are safe. The call allocates and frees nothing.
 * The first call on a GPU initialises the array and must not be captured into a graph
 * (PP_ERR_INVALID while the stream is capturing, nothing launched): make one eager call,
 * or call pp_decode_noalloc_reset, before capturing. Error bits 1, 2 and 8 of the
 * array's state are sticky as in a caller's workspace (every later call writes NaN);
 * pp_decode_noalloc_reset clears them. */
int pp_moe_decode_noalloc(const void* x, int x_dtype, int H, const float* router_packed,
                          const float* bias, int E, int G, float tau, const void* packed,
                          void* out_bf16, int grid, void* stream);
/* Re-initialises the current GPU's pp_moe_decode_noalloc array (a fill kernel on `stream`,
 * no allocation; initialises it on first use). No counterpart in the reference: for the
 * callers of pp_moe_decode_noalloc, which cannot reach the array to re-initialise it
 * after an error. error_out (may be NULL): the error bits the array held, read before
 * the reset (a synchronous copy: waits for the stream's earlier work). error_in: error
 * bits the array holds after the reset; 0, except to test a caller's error handling
 * (bit 1 makes every later call write NaN until the next reset). PP_ERR_INVALID while
 * `stream` is capturing. Must not overlap decode calls on the same GPU. */
int pp_decode_noalloc_reset(uint32_t* error_out, uint32_t error_in, void* stream);

/* Small-batch decode: 1 <= N <= 64 tokens in one launch. Replaces, for such batches,
 * TauSparseMoE.forward_prefill (src/tl_kernel_optimized_Ultimate_PanGU.py:532-604: route,
 * bucket, fused expert kernel, scatter-add), which the reference forward takes for every
 * N > 1 (:606-615); same selection and output semantics as pp_moe_prefill on the same
 * tokens, for the E = 16 family (E == 16, H % 512 == 0, G <= 512; PP_ERR_UNSUPPORTED
 * otherwise, so a caller can fall back to pp_moe_prefill). Every token's routing, the
 * gate/up MFMA over the union of the selected experts, the down projection and the fold
 * run in one kernel whose workgroups exchange data through the two workspaces:
 * workspace is a decode workspace (pp_decode_workspace_bytes, zeroed once by
 * pp_decode_workspace_init; it carries the call epoch, the tagged gates and the
 * per-workgroup flags, and may be the one the layer's pp_moe_decode calls use),
 * batch_workspace pp_decode_batch_workspace_bytes(H, E, G) bytes needing no initialisation
 * (untagged data only: one batch workspace may serve several decode workspaces). Calls that
 * share either must be ordered on one stream. logits_out ([N][16] fp32) and mask_out
 * ([N][16] uint8) receive the routing when not null. The output is the same bits on
 * every call (fixed summation orders). Error reporting as pp_moe_decode (error bit 1: a
 * wait timed out, every later call writes NaN until pp_decode_workspace_init).
 * grid = number of workgroups (0 = automatic; rounded down to a multiple of 16 and to
 * what the device holds at once). */
size_t pp_decode_batch_workspace_bytes(int H, int E, int G);
int pp_moe_decode_batch(const void* x, int x_dtype, int64_t n_tokens, int H, const float* router_packed,
                        const float* bias, int E, int G, float tau, const void* packed, void* out_bf16,
                        float* logits_out, uint8_t* mask_out, void* workspace, void* batch_workspace,
                        int grid, void* stream);

/* ------------------------------------------------------------------------- *
 * Prefill / N > 1. Replaces TauSparseMoE.forward_prefill
 * (src/tl_kernel_optimized_Ultimate_PanGU.py:532-604) and moe_fused_expert_kernel (:271-328).
 * No host synchronisation; hand-written kernels only. Two forms, by the expert width G:
 *   G % 64 == 0: route -> bucket -> grouped gate/up GEMM with fused SwiGLU epilogue
 *     (bf16 MFMA) -> grouped down GEMM -> per-token combine in fp32 -> bf16. The pair
 *     buffers are sized for every token selecting every expert, so the call runs in
 *     consecutive passes of at most max(64, 512 MiB / (E * H * 4)) tokens (2048 tokens in
 *     one pass at E = 16, H = 1536). At E = 16, calls longer than that (and from 2048 tokens
 *     on with tau >= 0.9) may instead take one down GEMM over every expert, the acts of the
 *     experts a token does not select being 0: chosen on the device, per pass, from the
 *     number of selected pairs; passes of up to 8192 tokens on the same workspace, where their
 *     buffers fit it and the call is large enough (pp_prefill_pass tells both).
 *   G % 64 != 0 (e.g. the checkpoint's E = 192 experts of G = 32 neurons, narrower than an
 *     MFMA column tile): router logits (fp32 MFMA, one fixed summation order per
 *     (token, expert): a token routes the same way in any batch) -> selection -> dense
 *     gate/up GEMM over every (token, neuron) with act = bf16(silu(g) * u * gate), 0 for the
 *     experts a token does not select -> dense down GEMM over all neurons, fp32
 *     accumulation, one rounding to bf16. Small batches (E != 16; up to 224 tokens at
 *     512 <= H <= 1536, 64 above, below 192, or 160 with E <= 64; and buffers that fit the
 *     GEMMs' split workspace) take the same arithmetic, summed in another order, in three
 *     launches that stream the weights (four with E <= 64: the selection apart). Passes of up
 *     to ~256 MiB of per-token buffers (about 15000 tokens at H = 1536, E = 192, G = 32).
 * Either way every token's routing is the same as in one pass over all N (its sums may be
 * taken in another order), and the output is the same bits on every call with the same N.
 * workspace: pp_prefill_workspace_bytes(N, H, E, G) bytes of device scratch.
 * ------------------------------------------------------------------------- */
size_t pp_prefill_workspace_bytes(int64_t n_tokens, int H, int E, int G);
int pp_moe_prefill(const void* x, int x_dtype, int64_t n_tokens, int H,
                   const float* router_packed, const float* bias, int E, int G, float tau,
                   const void* packed, void* out_bf16, void* workspace, void* stream);
/* pp_moe_prefill that also returns the routing it used: logits_out fp32 [N,E] (the
 * router's logits, bias included) and mask_out uint8 [N,E] (4-byte aligned), each NULL =
 * not written. The selection in mask_out is bit-exact with softmax_thresholding
 * (src/MoEBlock_origin.py:50-97) applied to logits_out. Same reference interface as
 * pp_moe_prefill (the reference's forward_prefill keeps its routing in locals, :550-564). */
int pp_moe_prefill_routed(const void* x, int x_dtype, int64_t n_tokens, int H,
                          const float* router_packed, const float* bias, int E, int G, float tau,
                          const void* packed, void* out_bf16, void* workspace,
                          float* logits_out, uint8_t* mask_out, void* stream);

/* How pp_moe_prefill cuts such a call: returns its number of passes (0: arguments out of range
 * or G % 64 != 0) and writes for pass `index`, each where not NULL, its tokens, the number of
 * selected pairs from which it takes the down GEMM over every expert (-1: not offered), and the
 * bytes of workspace it lays out, at most pp_prefill_workspace_bytes. Host arithmetic. No
 * counterpart in the reference. */
int64_t pp_prefill_pass(int64_t n_tokens, int H, int E, int G, float tau, int64_t index, int64_t* tokens,
                        int64_t* min_pairs, size_t* workspace_bytes);

/* Stages of pp_moe_prefill, exposed for testing and for callers that route
 * elsewhere. x is bf16 [N,H]. act is bf16 [N*E][G] capacity (row = pair), y is
 * fp32 [N*E][H] capacity (row = pair). */
int pp_expert_gateup(const void* x_bf16, int H, int G, const void* packed, int E,
                     const int32_t* token_ids, const float* pair_gates,
                     const int32_t* tiles, const int32_t* meta, int64_t max_tiles,
                     void* act_bf16, void* stream);
int pp_expert_down(const void* act_bf16, int H, int G, const void* packed, int E,
                   const int32_t* tiles, const int32_t* meta, int64_t max_tiles,
                   float* y_f32, void* stream);
int pp_combine(const float* y_f32, const int32_t* token_pairs, const int32_t* count,
               int64_t n_tokens, int H, int E, void* out_bf16, void* stream);

/* ------------------------------------------------------------------------- *
 * Masked training path: the expert gating of MoELayer.forward
 * (src/MoEBlock_origin.py:205-212: self_moe_mask = experts_prob @ experts_masks;
 * intermediate * self_moe_mask) and its backward, for the dense masked MLP that
 * IntegratedOpenPanguMoEMLP trains (src/openpangu_moe_origin.py:83-120).
 *   forward:  out[n,d] = inter[n,d] * gates[n, expert_ids[d]]
 *   backward: d_inter[n,d] = d_out[n,d] * gates[n, expert_ids[d]] (d_inter may be NULL);
 *             d_gates[n,e] = sum of d_out[n,d] * inter[n,d] over the neurons d of expert e
 *             (fp32, fixed order: repeated calls give the same bits).
 * inter / out / d_out / d_inter are [n_rows, I] fp32 or bf16 (dtype), 16-byte aligned;
 * gates / d_gates fp32 [n_rows, E]; expert_ids int32 [I] (16-byte aligned, values in
 * [0, E)); perm int32 [I]: the neurons sorted by expert id (stable), seg int32 [E+1]:
 * expert e owns perm[seg[e] .. seg[e+1]). bf16 activations: the gate is rounded to
 * bf16 before the multiply and the product to bf16 (the all-bf16 reference).
 * Supported: 1 <= E <= 256, I % 8 == 0, 8 <= I <= 16384. out may alias inter.
 * ------------------------------------------------------------------------- */
int pp_masked_gate_fwd(const void* inter, int dtype, const float* gates, const int32_t* expert_ids,
                       int64_t n_rows, int I, int E, void* out, void* stream);
int pp_masked_gate_bwd(const void* d_out, const void* inter, int dtype, const float* gates,
                       const int32_t* expert_ids, const int32_t* perm, const int32_t* seg, int64_t n_rows,
                       int I, int E, void* d_inter, float* d_gates, void* stream);

#ifdef __cplusplus
}
#endif
#endif /* PRUNEPATH_MOE_H */
