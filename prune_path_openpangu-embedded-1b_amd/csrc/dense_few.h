// Small batches of the dense form (a few dozen tokens at G % 64 != 0, e.g. the checkpoint's
// E = 192, G = 32): the layer is a stream of its weights (56.6 MB at I = 6144, H = 1536)
// past a few token rows, so the GEMM tiles of dense.hip (256 token rows, most of them
// padding, operands through LDS) are the wrong shape. Here the weights go straight from
// memory into MFMA A operands (16 rows x 32 k per instruction, each weight loaded by one
// wave of the launch), every load of a wave issued before the first MFMA, and the tokens
// are the B operand (16 columns at a time):
//   route_logits_few_kernel   one 16 token x 16 expert tile of logits per workgroup, in the
//                             summation order of route_logits_kernel (the same bits)
//   dense_few_gateup_kernel   h[t, n] = silu(x_t . Wg_n) * (x_t . Wu_n), fp32, before the
//                             router's gate is known: the selection (E > 64) runs in
//                             workgroups of the same launch, one token each
//   dense_few_down_kernel     act = bf16(h * gate), 0 where the expert is not selected (as
//                             dense_gemm_kernel<0>'s epilogue), out = bf16(act . Wd)
// What bounds it: at 16 tokens the three launches take about 9.5 us each, 28 in all (82 us before,
// on the GEMM tiles), of which a stream of the weights at the rate of a large copy would be 9 us:
// the logits are one latency chain (router rows from memory, 96 dependent MFMAs), the other
// two a launch, a cold stream and the sums of the waves. Beyond, each 16 tokens cost ~2.9 us:
// x and h pass once per workgroup through L2, and the sums once through LDS. Two token tiles per
// logits workgroup (router rows shared, two MFMA chains) took 4 us more, 49.1 -> 53.3 us a layer
// at 128 tokens: the chain is bound by the fp32 MFMA, not by its loads.
#pragma once
#include "pp_common.h"

__device__ __forceinline__ f32x4_t mfma16b(uint4 a, uint4 b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_bf16x8(a), as_bf16x8(b), c, 0, 0, 0);
}

__device__ __forceinline__ uint4 pack_bf16x8(const float (&v)[8]) {
  bf16x8_t r;
#pragma unroll
  for (int i = 0; i < 8; ++i) r[i] = (__bf16)v[i];
  return __builtin_bit_cast(uint4, r);
}

// Eight consecutive values of a row as a bf16 MFMA operand.
template <typename XT>
struct Row8;
template <>
struct Row8<bf16_t> {
  uint4 u;
  __device__ __forceinline__ void load(const bf16_t* p) { u = *(const uint4*)p; }
  __device__ __forceinline__ uint4 bf() const { return u; }
  __device__ __forceinline__ void f32(float (&v)[8]) const {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};
template <>
struct Row8<float> {
  float4 a, b;
  __device__ __forceinline__ void load(const float* p) {
    a = *(const float4*)p;
    b = *(const float4*)(p + 4);
  }
  __device__ __forceinline__ void f32(float (&v)[8]) const {
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  __device__ __forceinline__ uint4 bf() const {
    float v[8];
    f32(v);
    return pack_bf16x8(v);
  }
};

// ------------------------------------------------------------------ router logits
// Wave kq takes the 32-wide K block kq of every 128-wide chunk, lane (t = l % 16, g = l / 16)
// x[t][k + 8 g + j] and W[expert l % 16][k + 8 g + j], one fp32 MFMA per j; the chain runs in
// chunk order, j order, the four K-block partials are added in block order, then the bias:
// route_logits_kernel's order, so a token's logits are the same bits from either kernel.
// There a workgroup walks 12 chunks through LDS for 32 x 48 logits, and a few tokens fill a
// few CUs; here the loads of up to RLF_C chunks are in flight at once.
#define RLF_C 12
template <typename XT>
__global__ __launch_bounds__(256, 1) void route_logits_few_kernel(const XT* __restrict__ x, int64_t N, int H,
                                                                  const float* __restrict__ router,
                                                                  const float* __restrict__ bias, int E,
                                                                  float* __restrict__ logits_out,
                                                                  bf16_t* __restrict__ xbf_out,
                                                                  bf16_t* __restrict__ xfrag_out,
                                                                  uint32_t* __restrict__ zero, int nzero) {
  __shared__ float part[4][16][17];
  const int tid = threadIdx.x, lane = tid & 63, kq = tid >> 6;
  const int t_l = lane & 15, g = lane >> 4;
  const int64_t tok0 = (int64_t)blockIdx.x * 16;
  const int e0 = (int)blockIdx.y * 16;
  if (zero && blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = tid; i < nzero; i += 256) zero[i] = 0u;
  const bool real = tok0 + t_l < N;
  const int64_t xo = min(tok0 + t_l, N - 1) * H + kq * 32 + 8 * g;
  const XT* xp = x + xo;
  const float* wp = router + (int64_t)(e0 + t_l) * H + kq * 32 + 8 * g;  // router_packed has Epad rows
  const int nch = H / 128;
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  for (int c0 = 0; c0 < nch; c0 += RLF_C) {
    Row8<XT> xr[RLF_C];
    Row8<float> wr[RLF_C];
#pragma unroll
    for (int c = 0; c < RLF_C; ++c)
      if (c0 + c < nch) {
        xr[c].load(xp + (c0 + c) * 128);
        wr[c].load(wp + (c0 + c) * 128);
      }
#pragma unroll
    for (int c = 0; c < RLF_C; ++c)
      if (c0 + c < nch) {
        float xv[8], wv[8];
        xr[c].f32(xv);
        wr[c].f32(wv);
#pragma unroll
        for (int j = 0; j < 8; ++j) acc = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[j], wv[j], acc, 0, 0, 0);
        if (sizeof(XT) == 4 && xbf_out && blockIdx.y == 0 && real)
          *(uint4*)(xbf_out + xo + (c0 + c) * 128) = xr[c].bf();
        if (xfrag_out && blockIdx.y == 0)  // K step 4 (c0 + c) + kq of the small-batch gate/up's B operand
          *(uint4*)(xfrag_out + (((int64_t)((c0 + c) * 4 + kq) * gridDim.x + blockIdx.x) * 64 + lane) * 8) = xr[c].bf();
      }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) part[kq][4 * g + q][t_l] = acc[q];
  __syncthreads();
  const int r = tid >> 4, ce = tid & 15;
  const int64_t t = tok0 + r;
  const int e = e0 + ce;
  if (t < N && e < E) {
    float l = part[0][r][ce];
#pragma unroll
    for (int ww = 1; ww < 4; ++ww) l = __fadd_rn(l, part[ww][r][ce]);
    if (bias) l = __fadd_rn(l, bias[e]);
    logits_out[t * E + e] = l;
  }
}

// ------------------------------------------------------------------ gate/up
#define DF_MAX 224  // tokens at most (dense_few_max)

struct FewArgs {
  const bf16_t* xfrag;    // x as bf16: [H / 32][token block][lane][8]
  const bf16_t* rows;     // packed neuron records [I][3][H]
  const bf16_t* down_t;   // [E][H][G]
  const float* logits;    // [N][E]
  float* gates;           // [N][E], 0 where not selected
  uint8_t* mask;          // [N][E]
  float* h;               // silu(g) u of every (token, neuron), few_h order
  float* part;            // down: K-part partial sums [parts][N][H]
  uint32_t* tick;         // down: one ticket per 16-row block, zero at launch, left zero
  bf16_t* out;            // [N][H]
  float tau;
  int N, H, E, G, I;
  int n_sel;              // selection workgroups at the front of the gate/up grid (N or 0)
};

// h in the down projection's B operand order: K step n / 32, token block tb, two halves of 64
// lanes x 4 values (lane 16 q + token: neurons 8 q + 4 half ..), so a wave's load is 1 KB
// contiguous.
__device__ __forceinline__ int64_t few_h(int n, int tb, int tok, int ntb) {
  return ((((int64_t)(n >> 5) * ntb + tb) * 2 + ((n >> 2) & 1)) * 64 + ((n >> 3) & 3) * 16 + tok) * 4 + (n & 3);
}

// U units of eight neurons per workgroup (a unit's A rows: the gate rows, then the up rows of
// its neurons); wave w takes the K steps (32 wide) [w per, (w + 1) per) of H, at most KS of
// them loaded at a time. The eight waves' partial sums are added in wave order through LDS.
// ONE: every wave has exactly KS K steps (H = 256 KS), so the weights stay in registers over all
// token blocks. U = 3 there: at I = 6144 one workgroup per CU (and the selection's beside them in
// the 128 VGPRs that leave room for two), H = 1536, N = 16 / 64 / 128: 28.7 / 37.7 / 49.2 us a layer
// against 30.4 / 40.4 / 52.7 with U = 2 and 30.8 / 40.8 / 54.2 with U = 1. x in operand order
// instead of token rows (each load 16 rows x 64 B): 46 -> 40 us at N = 64.
template <int U, int KS, bool ONE>
__global__ __launch_bounds__(512, 4) void dense_few_gateup_kernel(FewArgs p) {
  constexpr int PR = 16 * U + 4;  // LDS row of a token: U units of 16 sums, padded
  __shared__ __align__(16) union {
    float part[2][8][16][PR];
    SelWgScratch sel;
  } sm;
  if ((int)blockIdx.x < p.n_sel) {
    route_select_wg_token<512>(p.logits, blockIdx.x, p.E, p.tau, nullptr, nullptr, p.gates, p.mask, nullptr, &sm.sel);
    return;
  }
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int n0 = ((int)blockIdx.x - p.n_sel) * U * 8;
  const int steps = p.H / 32, per = (steps + 7) / 8;
  const int s0 = w * per, ns = max(0, min(per, steps - s0));
  const int nch = (per + KS - 1) / KS;  // uniform over the waves
  const bf16_t* wr[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int n = min(n0 + u * 8 + (r & 7), p.I - 1);
    wr[u] = p.rows + ((int64_t)n * 3 + (r >> 3)) * p.H + s0 * 32 + q * 8;
  }
  auto in = [&](int c, int s) { return ONE || c * KS + s < ns; };  // uniform
  uint4 wf[U][KS], xf[KS];
  auto load_w = [&](int c) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const bf16_t* wp = wr[u] + c * KS * 32;
#pragma unroll
      for (int s = 0; s < KS; ++s)
        if (in(c, s)) wf[u][s] = *(const uint4*)(wp + s * 32);
    }
  };
  const int ntb = (p.N + 15) / 16;
  auto load_x = [&](int tb, int c) {
    const char* xb = (const char*)p.xfrag + ((int64_t)(s0 + c * KS) * ntb + tb) * 1024;  // uniform
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (in(c, s)) xf[s] = *(const uint4*)(xb + lane * 16);
      xb += ntb * 1024;
    }
  };
  // the eight waves' sums of token block tb, and h (lane: token r, rows 4 q .. 4 q + 3 of a unit)
  auto finish = [&](int tb, const f32x4_t(&acc)[U]) {
    float(*pt)[16][PR] = sm.part[tb & 1];
#pragma unroll
    for (int u = 0; u < U; ++u) *(f32x4_t*)&pt[w][r][u * 16 + q * 4] = acc[u];
    wg_lds_barrier();  // (two buffers: the next block's writes cannot reach these reads)
    for (int i = tid; i < 16 * U * 8; i += 512) {
      const int tl = i / (U * 8), nl = i % (U * 8), n = n0 + nl;
      const int o = (nl >> 3) * 16 + (nl & 7);
      float sg = pt[0][tl][o], su = pt[0][tl][o + 8];
#pragma unroll
      for (int k = 1; k < 8; ++k) {
        sg = __fadd_rn(sg, pt[k][tl][o]);
        su = __fadd_rn(su, pt[k][tl][o + 8]);
      }
      if (n < p.I) p.h[few_h(n, tb, tl, ntb)] = dg_silu(sg) * su;
    }
  };
  if constexpr (ONE) {
    load_x(0, 0);
    load_w(0);
    for (int tb = 0; tb < ntb; ++tb) {
      f32x4_t acc[U];
#pragma unroll
      for (int u = 0; u < U; ++u) acc[u] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int u = 0; u < U; ++u) acc[u] = mfma16b(wf[u][s], xf[s], acc[u]);
      if (tb + 1 < ntb) load_x(tb + 1, 0);  // in flight under this block's sums
      finish(tb, acc);
    }
  } else {
    constexpr int TG = 4;  // token blocks whose sums are kept while the K chunks pass
    for (int t0 = 0; t0 < ntb; t0 += TG) {
      f32x4_t acc[TG][U];
#pragma unroll
      for (int g = 0; g < TG; ++g)
#pragma unroll
        for (int u = 0; u < U; ++u) acc[g][u] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
      for (int c = 0; c < nch; ++c) {
        if (nch > 1 || t0 == 0) load_w(c);
#pragma unroll
        for (int g = 0; g < TG; ++g)
          if (t0 + g < ntb) {
            load_x(t0 + g, c);
#pragma unroll
            for (int s = 0; s < KS; ++s)
              if (in(c, s)) {
#pragma unroll
                for (int u = 0; u < U; ++u) acc[g][u] = mfma16b(wf[u][s], xf[s], acc[g][u]);
              }
          }
      }
#pragma unroll
      for (int g = 0; g < TG; ++g)
        if (t0 + g < ntb) finish(t0 + g, acc[g]);
    }
  }
}

// ------------------------------------------------------------------ down
// R 16-row blocks of the output's H per workgroup and one of `parts` ranges of the K steps
// (32 neurons of one expert each): wave w of part p takes KW steps. Waves add in order
// through LDS; parts > 1: the fp32 sums of a part go to memory (agent-scope stores) and the
// part drawing a block's last ticket adds them in part order (nobody waits). R = 2, KW = 3 (at
// I = 6144, H = 1536 eight parts of 48 row blocks): N = 16 / 64 / 128 32.2 / 46.2 / 71.8 us a
// layer, measured before the x order above, against 34.0 / 49.7 / 77.8 with R = 1, KW = 6 and
// 34.1 / 53.9 / 86.2 with R = 4, KW = 2; no parts at all (R = 1, KW = 24) 45 / 103.
template <int R, int KW>
__global__ __launch_bounds__(512, 4) void dense_few_down_kernel(FewArgs p) {
  constexpr int PR = 16 * R + 4;
  constexpr int NE = 8 * KW + 1;  // experts a part's K steps can touch (G >= 32)
  __shared__ __align__(16) float part_s[2][8][16][PR];
  __shared__ float gate_s[DF_MAX][NE];
  __shared__ int role_s;
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const int nrb = p.H / (16 * R), parts = (int)gridDim.x / nrb;
  const int rb = (int)blockIdx.x % nrb, pi = (int)blockIdx.x / nrb;
  const int spe = p.G / 32, steps = p.I / 32;
  const int s0 = (pi * 8 + w) * KW, ns = min(KW, steps - s0);
  uint4 wf[R][KW];
#pragma unroll
  for (int s = 0; s < KW; ++s)
    if (s < ns) {
      const int e = (s0 + s) / spe, g0 = (s0 + s - e * spe) * 32;
#pragma unroll
      for (int b = 0; b < R; ++b)
        wf[b][s] = *(const uint4*)(p.down_t + ((int64_t)e * p.H + (rb * R + b) * 16 + r) * p.G + g0 + q * 8);
    }
  const int ntb = (p.N + 15) / 16;
  float4 hf[KW][2];
  auto load_h = [&](int tb) {
#pragma unroll
    for (int s = 0; s < KW; ++s)
      if (s < ns) {
        const float4* hp = (const float4*)p.h + ((int64_t)(s0 + s) * ntb + tb) * 128 + lane;
        hf[s][0] = hp[0];
        hf[s][1] = hp[64];
      }
  };
  load_h(0);
  // the part's router gates
  const int e_lo = pi * 8 * KW / spe, ne = min(p.E, (min(steps, (pi + 1) * 8 * KW) - 1) / spe + 1) - e_lo;
  for (int i = tid; i < p.N * ne; i += 512) {
    const int t = i / ne, e = i - t * ne;
    gate_s[t][e] = p.gates[(int64_t)t * p.E + e_lo + e];
  }
  __syncthreads();
  for (int tb = 0; tb < ntb; ++tb) {
    const float* gp = gate_s[min(tb * 16 + r, p.N - 1)];
    f32x4_t acc[R];
#pragma unroll
    for (int b = 0; b < R; ++b) acc[b] = (f32x4_t){0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KW; ++s)
      if (s < ns) {
        const float gt = gp[(s0 + s) / spe - e_lo];
        const float hv[8] = {hf[s][0].x, hf[s][0].y, hf[s][0].z, hf[s][0].w,
                             hf[s][1].x, hf[s][1].y, hf[s][1].z, hf[s][1].w};
        float v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) v[j] = gt == 0.0f ? 0.0f : hv[j] * gt;
        const uint4 a = pack_bf16x8(v);
#pragma unroll
        for (int b = 0; b < R; ++b) acc[b] = mfma16b(wf[b][s], a, acc[b]);
      }
    if (tb + 1 < ntb) load_h(tb + 1);
    float(*pt)[16][PR] = part_s[tb & 1];
#pragma unroll
    for (int b = 0; b < R; ++b) *(f32x4_t*)&pt[w][r][b * 16 + q * 4] = acc[b];
    wg_lds_barrier();
    for (int i = tid; i < 256 * R; i += 512) {
      const int tl = i / (16 * R), hl = i % (16 * R), to = tb * 16 + tl;
      float s = pt[0][tl][hl];
#pragma unroll
      for (int k = 1; k < 8; ++k) s = __fadd_rn(s, pt[k][tl][hl]);
      if (to < p.N) {
        const int64_t o = (int64_t)to * p.H + rb * 16 * R + hl;
        if (parts == 1)
          p.out[o] = f32_to_bf16(s);
        else
          __hip_atomic_store(p.part + (int64_t)pi * p.N * p.H + o, s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
    }
  }
  if (parts == 1) return;
  asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory");  // every thread's stores performed
  if (tid == 0)
    role_s = (int)__hip_atomic_fetch_add(p.tick + rb, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  if (role_s != parts - 1) return;
  for (int i = tid; i < p.N * 16 * R; i += 512) {
    const int64_t o = (int64_t)(i / (16 * R)) * p.H + rb * 16 * R + i % (16 * R);
    float s = 0.0f;
    for (int k0 = 0; k0 < parts; k0 += 8) {  // eight parts' loads in flight at a time
      float v[8];
#pragma unroll
      for (int k = 0; k < 8; ++k)
        v[k] = k0 + k < parts ? __hip_atomic_load(p.part + (int64_t)(k0 + k) * p.N * p.H + o, __ATOMIC_RELAXED,
                                                  __HIP_MEMORY_SCOPE_AGENT)
                              : 0.0f;
#pragma unroll
      for (int k = 0; k < 8; ++k)
        if (k0 + k < parts) s = k0 + k == 0 ? v[0] : __fadd_rn(s, v[k]);
    }
    p.out[o] = f32_to_bf16(s);
  }
  if (tid == 0) __hip_atomic_store(p.tick + rb, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
