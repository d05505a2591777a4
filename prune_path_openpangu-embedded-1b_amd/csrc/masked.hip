// Masked training path: the expert gating of MoELayer.forward (src/MoEBlock_origin.py:205-212),
//   self_moe_mask = experts_prob @ experts_masks      ([N,E] x [E,I] one-hot)
//   intermediate  = intermediate * self_moe_mask
// and its backward, as two HBM-bound kernels over rows of the [N, I] activations.
//
// experts_masks is one-hot per neuron, so the matmul picks gates[n, eid[d]] exactly
// (one product by 1.0 plus zeros: no rounding), and the forward is one multiply per
// element: out[n,d] = inter[n,d] * gates[n, eid[d]] -- bit-identical to the fp32
// reference ops. With bf16 activations the gate is rounded to bf16 first and the
// product rounded to bf16, as the all-bf16 reference (bf16 experts_prob @ bf16 masks,
// bf16 multiply) computes it.
//
// Backward (the autograd of the two ops):
//   d_inter[n,d] = d_out[n,d] * gates[n, eid[d]]
//   d_gates[n,e] = sum over the neurons d of expert e of d_out[n,d] * inter[n,d]
// accumulated in fp32 in a fixed order, so repeated calls give the same bits: the
// products are staged in LDS in the expert-sorted neuron order (perm, seg) and summed in
// that order, TPE interleaved partial sums per expert then an xor tree, whatever the partition.
//
// Workgroups of 256 threads; each thread moves 8 consecutive elements per step (16-byte
// bf16 / 32-byte fp32 vectors).
#include <algorithm>

#include "pp_common.h"

#define MG_THREADS 256
#define MG_MAX_I 16384  // LDS holds one row's fp32 products; places in the expert-sorted order are 16-bit

// 16-byte loads and stores, non-temporal (NT) or not. A non-temporal result does not take the
// place of rows that the launch still has to read, but the kernel that reads it next finds it in
// memory, not in the cache.
// Forward: NT where a result is larger than half of the 256 MB last-level cache (MG_NT_BYTES), so
// that rows and results together do not fit. I = 6144, us, rows normal / NT: forward alone bf16
// 1024 4.7 / 4.0, 16384 77 / 57; with an elementwise kernel before and a product with a [1536][I]
// matrix after it bf16 512 30.6 / 34.0, 1024 41.9 / 46.4, 4096 106 / 111, 8192 202 / 204, 16384
// 407 / 409 (followed by an elementwise kernel alone 183 / 178), fp32 6144 931 / 932 (142 / 140).
// Backward: NT loads and stores at every size. It is its rows' last reader and stores as it reads;
// between an elementwise kernel that writes d_out and one that reads d_inter, bf16 rows, normal
// and NT: 512 24.2 / 20.0, 1024 31.2 / 32.5, 4096 80.6 / 81.7, 8192 168 / 153, 16384 332 / 313.
#define MG_NT_BYTES ((int64_t)128 << 20)
typedef uint32_t mg_u4 __attribute__((ext_vector_type(4)));
template <bool NT>
__device__ __forceinline__ uint4 mg_ld(const void* p) {
  const mg_u4 v = NT ? __builtin_nontemporal_load((const mg_u4*)p) : *(const mg_u4*)p;
  return make_uint4(v.x, v.y, v.z, v.w);
}
template <bool NT>
__device__ __forceinline__ void mg_st(void* p, uint4 u) {
  const mg_u4 v = {u.x, u.y, u.z, u.w};
  if (NT)
    __builtin_nontemporal_store(v, (mg_u4*)p);
  else
    *(mg_u4*)p = v;
}

template <typename T>
struct MgVec;
template <>
struct MgVec<float> {
  static __device__ __forceinline__ void load(const float* p, float (&v)[8]) {
    const float4 a = *(const float4*)p, b = *(const float4*)(p + 4);
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
  template <bool NT>
  static __device__ __forceinline__ void store(float* p, const float (&v)[8]) {
    mg_st<NT>(p, make_uint4(__float_as_uint(v[0]), __float_as_uint(v[1]), __float_as_uint(v[2]), __float_as_uint(v[3])));
    mg_st<NT>(p + 4, make_uint4(__float_as_uint(v[4]), __float_as_uint(v[5]), __float_as_uint(v[6]), __float_as_uint(v[7])));
  }
  static __device__ __forceinline__ float gate(float g) { return g; }
};
template <>
struct MgVec<bf16_t> {
  static __device__ __forceinline__ void load(const bf16_t* p, float (&v)[8]) {
    const uint4 u = *(const uint4*)p;
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
  template <bool NT>
  static __device__ __forceinline__ void store(bf16_t* p, const float (&v)[8]) {
    uint4 u;
    u.x = (uint32_t)f32_to_bf16(v[0]) | ((uint32_t)f32_to_bf16(v[1]) << 16);
    u.y = (uint32_t)f32_to_bf16(v[2]) | ((uint32_t)f32_to_bf16(v[3]) << 16);
    u.z = (uint32_t)f32_to_bf16(v[4]) | ((uint32_t)f32_to_bf16(v[5]) << 16);
    u.w = (uint32_t)f32_to_bf16(v[6]) | ((uint32_t)f32_to_bf16(v[7]) << 16);
    mg_st<NT>(p, u);
  }
  static __device__ __forceinline__ float gate(float g) { return bf16_to_f32(f32_to_bf16(g)); }
};

// one row's elements of a thread in the storage type
template <typename T, int NI>
struct MgRow {
  static constexpr int W = 8 * (int)sizeof(T) / 16;  // 16-byte words per 8 elements
  uint4 v[NI][W];
  template <bool NT>
  __device__ __forceinline__ void load(const T* row, int tid, int I) {
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int d = 8 * tid + it * 8 * MG_THREADS;
      if (d < I) {
#pragma unroll
        for (int q = 0; q < W; ++q) v[it][q] = mg_ld<NT>((const char*)(row + d) + 16 * q);
      }
    }
  }
  __device__ __forceinline__ void get(int it, float (&f)[8]) const {
    T t[8];
#pragma unroll
    for (int q = 0; q < W; ++q) *(uint4*)((char*)t + 16 * q) = v[it][q];
    MgVec<T>::load(t, f);
  }
};

// The forward takes one row per workgroup (no barrier between rows; the ids come through L2 as
// int32): 57 us for 16384 x 6144 bf16, 7.0 TB/s. The persistent form with the ids in LDS was a
// little slower (85 against 80 us, both with normal stores).
__device__ __forceinline__ void mg_eids(const int32_t* eid, int d, int E, int (&e)[8]) {
  const int4 a = *(const int4*)(eid + d), b = *(const int4*)(eid + d + 4);
  const int v[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
  for (int i = 0; i < 8; ++i) e[i] = (int)min((unsigned)v[i], (unsigned)(E - 1));  // clamped
}

template <typename T, bool NT>
__global__ __launch_bounds__(MG_THREADS) void masked_gate_fwd_kernel(const T* __restrict__ inter,
                                                                     const float* __restrict__ gates,
                                                                     const int32_t* __restrict__ eid, int I, int E,
                                                                     T* __restrict__ out) {
  __shared__ float g_s[PP_MAX_EXPERTS];
  const int64_t n = blockIdx.x;
  const int tid = threadIdx.x;
  for (int e = tid; e < E; e += MG_THREADS) g_s[e] = MgVec<T>::gate(gates[n * E + e]);
  __syncthreads();
  for (int d = 8 * tid; d < I; d += 8 * MG_THREADS) {
    float v[8];
    int e[8];
    MgRow<T, 1> xr;
    xr.template load<false>(inter + n * I + d, 0, 8);
    xr.get(0, v);
    mg_eids(eid, d, E, e);
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = __fmul_rn(v[i], g_s[e[i]]);
    MgVec<T>::template store<NT>(out + n * I + d, v);
  }
}

// ------------------------------------------------------------------ backward
// Persistent over rows. A thread's elements are the same in every row (8 tid + 2048 it, NI
// steps), so their expert ids and their places in the expert-sorted order are registers, and a
// row is: products scattered to their sorted places in LDS, barrier, per-expert sums, barrier.
// The next row's loads are issued before the first barrier and land under the sums (LDS-only
// barriers: __syncthreads would wait for them).
// Place k of the order sits at word MG_SKEW(k) = k + k / 32: the lanes of a wave sum segments 32 E' apart
// (E = 192: 32 neurons each, one lane per expert), which would all start in two banks.
// The earlier form kept the order and the ids in LDS (45 KB: three workgroups per CU), gathered
// the products through the order (a dependent pair of LDS reads per term) and had no loads in
// flight during the sums: 16384 x 6144 bf16, E = 16 / 192, 146 / 209 us, this form 126 / 132 with
// the same loads and 111 / 117 with the non-temporal ones (5.4 / 5.2 TB/s); 6144 x 6144 fp32,
// E = 192, 113 -> 93 us. Bound: memory (a copy of such rows reaches 5.1 to 6.2 TB/s).
#define MG_SKEW(k) ((k) + ((k) >> 5))

static size_t mg_bwd_lds(int I, int E) { return ((size_t)MG_SKEW(I) + 1 + 2 * E + E + 1) * 4; }

// workgroups per CU (waves per SIMD) that the registers of NI steps leave room for
template <typename T>
constexpr int mg_bwd_wpc(int ni) {
  return ni == 1 ? 6 : ni == 2 ? 5 : ni == 3 ? 4 : ni == 4 ? 3 : ni == 6 || sizeof(T) == 2 ? 2 : 1;
}

// tpe: threads per expert for the sums (a power of two <= 64, E * tpe <= MG_THREADS).
template <typename T, int NI>
__global__ __launch_bounds__(MG_THREADS, mg_bwd_wpc<T>(NI)) void masked_gate_bwd_kernel(
    const T* __restrict__ d_out, const T* __restrict__ inter, const float* __restrict__ gates,
    const int32_t* __restrict__ eid, const int32_t* __restrict__ perm, const int32_t* __restrict__ seg,
    int64_t n_rows, int I, int E, int tpe, T* __restrict__ d_inter, float* __restrict__ d_gates) {
  extern __shared__ __align__(16) float mg_smem[];
  const int np = MG_SKEW(I) + 1;  // sorted places, and one nobody sums
  float* prod_s = mg_smem;
  float* g_s = prod_s + np;        // [2][E]
  int* seg_s = (int*)(g_s + 2 * E);
  const int tid = threadIdx.x;
  // the inverse of the order (ids, order and segments come from the caller: clamped)
  uint16_t* inv_s = (uint16_t*)prod_s;
  for (int k = tid; k < I; k += MG_THREADS) inv_s[k] = (uint16_t)(np - 1);
  for (int e = tid; e <= E; e += MG_THREADS) seg_s[e] = min(max(seg[e], 0), I);
  wg_lds_barrier();
  for (int k = tid; k < I; k += MG_THREADS) inv_s[min((unsigned)perm[k], (unsigned)(I - 1))] = (uint16_t)MG_SKEW(k);
  wg_lds_barrier();
  uint32_t inv[NI][4];  // eight 16-bit places
  uint32_t ids[NI][2];  // eight 8-bit expert ids
#pragma unroll
  for (int it = 0; it < NI; ++it) {
    const int d = 8 * tid + it * 8 * MG_THREADS;
    if (d < I) {
      const uint4 p = *(const uint4*)(inv_s + d);
      inv[it][0] = p.x, inv[it][1] = p.y, inv[it][2] = p.z, inv[it][3] = p.w;
      int e[8];
      mg_eids(eid, d, E, e);
#pragma unroll
      for (int h = 0; h < 2; ++h)
        ids[it][h] = (uint32_t)e[4 * h] | (uint32_t)e[4 * h + 1] << 8 | (uint32_t)e[4 * h + 2] << 16 |
                     (uint32_t)e[4 * h + 3] << 24;
    }
  }
  wg_lds_barrier();
  for (int k = tid; k < np; k += MG_THREADS) prod_s[k] = 0.0f;
  const int ex = tid / tpe, j = tid - ex * tpe;
  MgRow<T, NI> go, x;
  float gr = 0.0f;
  auto load = [&](int64_t n) {
    go.template load<true>(d_out + n * I, tid, I);
    x.template load<true>(inter + n * I, tid, I);
    if (tid < E) gr = gates[n * E + tid];
  };
  int64_t n = blockIdx.x;
  if (n < n_rows) load(n);
  for (int par = 0; n < n_rows; n += gridDim.x, par ^= 1) {
    float* g = g_s + par * E;
    if (tid < E) g[tid] = MgVec<T>::gate(gr);
    wg_lds_barrier();  // gates visible; the previous row's sums done
#pragma unroll
    for (int it = 0; it < NI; ++it) {
      const int d = 8 * tid + it * 8 * MG_THREADS;
      if (d < I) {
        float a[8], b[8], gi[8];
        go.get(it, a);
        x.get(it, b);
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          gi[i] = __fmul_rn(a[i], g[(ids[it][i >> 2] >> (8 * (i & 3))) & 0xff]);
          prod_s[(inv[it][i >> 1] >> (16 * (i & 1))) & 0xffff] = __fmul_rn(a[i], b[i]);
        }
        if (d_inter) MgVec<T>::template store<true>(d_inter + n * I + d, gi);
      }
    }
    if (n + gridDim.x < n_rows) load(n + gridDim.x);
    wg_lds_barrier();
    // expert ex, partial j over its places k = seg[ex] + j, + tpe, ... in four interleaved
    // sums, ((a0 + a1) + (a2 + a3)), then the xor tree inside the tpe-lane group
    float s = 0.0f;
    if (ex < E) {
      const int k1 = seg_s[ex + 1];
      int k = seg_s[ex] + j;
      float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f, a3 = 0.0f;
#pragma unroll 2
      for (; k + 3 * tpe < k1; k += 4 * tpe) {
        a0 = __fadd_rn(a0, prod_s[MG_SKEW(k)]);
        a1 = __fadd_rn(a1, prod_s[MG_SKEW(k + tpe)]);
        a2 = __fadd_rn(a2, prod_s[MG_SKEW(k + 2 * tpe)]);
        a3 = __fadd_rn(a3, prod_s[MG_SKEW(k + 3 * tpe)]);
      }
      for (; k < k1; k += tpe) a0 = __fadd_rn(a0, prod_s[MG_SKEW(k)]);
      s = __fadd_rn(__fadd_rn(a0, a1), __fadd_rn(a2, a3));
    }
    for (int o = 1; o < tpe; o <<= 1) s = __fadd_rn(s, __shfl_xor(s, o, PP_WAVE));
    if (ex < E && j == 0) d_gates[n * E + ex] = s;
  }
}

// Workgroups per launch: as many as fit the CUs by registers (wpc) and LDS, no more than
// there are rows.
static unsigned mg_grid(int64_t n_rows, size_t lds, int wpc) {
  const int per_cu = std::max(1, std::min(wpc, (int)((160 * 1024) / (lds + 1024))));
  return (unsigned)std::min<int64_t>(n_rows, (int64_t)pp_device_cus() * per_cu);
}

template <typename T>
static void mg_bwd_launch(const void* d_out, const void* inter, const float* gates, const int32_t* eid,
                          const int32_t* perm, const int32_t* seg, int64_t n_rows, int I, int E, void* d_inter,
                          float* d_gates, hipStream_t st) {
  int tpe = 64;
  while (tpe > 1 && tpe * E > MG_THREADS) tpe >>= 1;
  const size_t lds = mg_bwd_lds(I, E);
  const int ni = (I + 8 * MG_THREADS - 1) / (8 * MG_THREADS);
#define MG_BWD(NI)                                                                                                 \
  masked_gate_bwd_kernel<T, NI><<<mg_grid(n_rows, lds, mg_bwd_wpc<T>(NI)), MG_THREADS, lds, st>>>(                 \
      (const T*)d_out, (const T*)inter, gates, eid, perm, seg, n_rows, I, E, tpe, (T*)d_inter, d_gates)
  if (ni <= 1) MG_BWD(1);
  else if (ni <= 2) MG_BWD(2);
  else if (ni <= 3) MG_BWD(3);
  else if (ni <= 4) MG_BWD(4);
  else if (ni <= 6) MG_BWD(6);
  else MG_BWD(8);
#undef MG_BWD
}

static int mg_check(const void* a, const void* b, int dtype, int64_t n_rows, int I, int E, const char* what) {
  PP_REQUIRE(dtype == PP_DTYPE_F32 || dtype == PP_DTYPE_BF16, PP_ERR_INVALID, "%s: dtype %d", what, dtype);
  PP_REQUIRE(E >= 1 && E <= PP_MAX_EXPERTS, PP_ERR_UNSUPPORTED, "%s: E=%d unsupported (1..256)", what, E);
  PP_REQUIRE(I >= 8 && I % 8 == 0 && I <= MG_MAX_I, PP_ERR_UNSUPPORTED,
             "%s: I=%d unsupported (need I %% 8 == 0, 8 <= I <= %d)", what, I, MG_MAX_I);
  PP_REQUIRE(n_rows >= 0 && n_rows <= 0x7fffffff, PP_ERR_UNSUPPORTED, "%s: n_rows %lld", what, (long long)n_rows);
  PP_REQUIRE(((uintptr_t)a & 15) == 0 && ((uintptr_t)b & 15) == 0, PP_ERR_INVALID,
             "%s: activations must be 16-byte aligned", what);
  return PP_OK;
}

extern "C" int pp_masked_gate_fwd(const void* inter, int dtype, const float* gates, const int32_t* expert_ids,
                                  int64_t n_rows, int I, int E, void* out, void* stream) {
  int rc = mg_check(inter, out, dtype, n_rows, I, E, "pp_masked_gate_fwd");
  if (rc) return rc;
  if (n_rows == 0) return PP_OK;
  PP_REQUIRE(inter && gates && expert_ids && out, PP_ERR_INVALID, "pp_masked_gate_fwd: null pointer");
  PP_REQUIRE(((uintptr_t)expert_ids & 15) == 0, PP_ERR_INVALID, "pp_masked_gate_fwd: expert_ids not 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  const bool nt = n_rows * I * (dtype == PP_DTYPE_F32 ? 4 : 2) > MG_NT_BYTES;
#define MG_FWD(T, NT)                                                                                                \
  masked_gate_fwd_kernel<T, NT>                                                                                      \
      <<<(unsigned)n_rows, MG_THREADS, 0, st>>>((const T*)inter, gates, expert_ids, I, E, (T*)out)
  if (dtype == PP_DTYPE_F32) {
    if (nt) MG_FWD(float, true);
    else MG_FWD(float, false);
  } else {
    if (nt) MG_FWD(bf16_t, true);
    else MG_FWD(bf16_t, false);
  }
#undef MG_FWD
  return pp_check_launch("pp_masked_gate_fwd");
}

extern "C" int pp_masked_gate_bwd(const void* d_out, const void* inter, int dtype, const float* gates,
                                  const int32_t* expert_ids, const int32_t* perm, const int32_t* seg, int64_t n_rows,
                                  int I, int E, void* d_inter, float* d_gates, void* stream) {
  int rc = mg_check(d_out, inter, dtype, n_rows, I, E, "pp_masked_gate_bwd");
  if (rc) return rc;
  if (n_rows == 0) return PP_OK;
  PP_REQUIRE(d_out && inter && gates && expert_ids && perm && seg && d_gates, PP_ERR_INVALID,
             "pp_masked_gate_bwd: null pointer");
  PP_REQUIRE(((uintptr_t)d_inter & 15) == 0 && ((uintptr_t)expert_ids & 15) == 0, PP_ERR_INVALID,
             "pp_masked_gate_bwd: d_inter / expert_ids not 16-byte aligned");
  hipStream_t st = (hipStream_t)stream;
  if (dtype == PP_DTYPE_F32)
    mg_bwd_launch<float>(d_out, inter, gates, expert_ids, perm, seg, n_rows, I, E, d_inter, d_gates, st);
  else
    mg_bwd_launch<bf16_t>(d_out, inter, gates, expert_ids, perm, seg, n_rows, I, E, d_inter, d_gates, st);
  return pp_check_launch("pp_masked_gate_bwd");
}
