// The attention side of one decode step, for the caller of the MoE hook: what sits between two
// MoE layers when every sequence of the batch advances by one token. In the reference this is
// a few dozen PyTorch launches per layer (switchyard/model.py:14-17 rmsnorm, :61-84
// _attention, :117-121 attention_block); at decode each of them is a launch that moves a few
// kilobytes, so the step is bound by launches, not by the 34 MB of attention weights and the
// KV cache it has to read. A few kernels replace them (the projections themselves go through
// the weight-stream kernel with a single "expert"):
//
//   row_kernel            one token per workgroup: x += delta; h = w * f16(x * rsqrt(mean(x^2) + eps)).
//                         x may be an embedding lookup (embed_rmsnorm), delta may be the combine
//                         of the MoE layer's rows (combine_add_rmsnorm, which also applies
//                         the router weights to rows that were left unscaled), and the router's
//                         logits of h may come out of the same launch (add_rmsnorm_logits); with
//                         them route and the sort as well (add_rmsnorm_route_sort, and
//                         router_route_sort for rows that need no norm: front_core.h), the whole
//                         front of the MoE layer in the launch that the step needs anyway
//   qk_norm_rope_cache    q/k RMS norm over the whole projection, clamp, rotary embedding, and
//                         the new keys and values written into the cache from `slot` on (one
//                         token per sequence at decode, the whole prompt at prefill)
//   decode_attention      one query per (sequence, head) against the cache: a single pass over
//                         the keys and values with a running softmax, HBM-bound; its _qkv form
//                         does the work of qk_norm_rope_cache in its own prologue
//   greedy_advance        arg-max of the logits, the token appended to the output, rotary
//                         positions and cache slot advanced
//
// Everything a replayed HIP graph must not bake in (the cache slot, the rotary positions, the
// output column) is read from device memory, so the same launches serve every step.
//
// Rounding follows the PyTorch graph on fp16 tensors where it is cheap to do so: the norm is
// taken in fp32, rounded to fp16 and then scaled in fp16; rotary products and their sum are
// each rounded to fp16. Attention scores and the softmax stay in fp32 (the reference rounds
// the scores to fp16 first), which is the more exact of the two.
#include <mutex>

#include "combine_core.h"
#include "common.h"
#include "front_core.h"
#include "../../include/switchyard_decode.h"
#include "passes.h"

namespace {

constexpr int ROW_THREADS = 256;
constexpr int MAX_CHUNKS = 4;  // 8-half chunks per thread: rows of up to 8192 halves

__device__ __forceinline__ float block_sum(float v, float* lds, int slot_base) {
  // sum over the wavefronts of the workgroup (at most 16); every thread gets the total
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6, nwaves = blockDim.x >> 6;
  if ((threadIdx.x & 63) == 0) lds[slot_base + wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < nwaves; ++w) total += lds[slot_base + w];
  return total;
}

// The same where the values are those of the workgroup's first four wavefronts (the others' are zero): one
// read of four sums, not a loop over them.
__device__ __forceinline__ float block_sum_of_four(float v, float* lds) {
  v = wave_sum(v);
  const int wave = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0 && wave < 4) lds[wave] = v;
  __syncthreads();
  const float4_t p = *reinterpret_cast<const float4_t*>(lds);
  return p[0] + p[1] + p[2] + p[3];
}

constexpr int FEW_ROWS = 64;   // up to these the row kernels are built for a short chain of waits, not for many wavefronts
constexpr int FEW_MIN_K = 4;   // ... where a token has at least so many rows to combine: it asks for AT_ONCE rows, used or not
constexpr int ROW_MAX_K = 64;  // choices per token the combining variant ranks in one wavefront

// One workgroup per token (row). The residual `delta` is either a tensor, or (COMBINE) the
// token's k expert outputs summed in fp32 in ascending expert id and rounded to f16 once,
// exactly as the combine kernel leaves it (`delta` then holds the router weights [N, k] of rows
// that the down projection left unscaled, or is null); then x_out = f16(x + delta) and h = the RMS norm
// of x_out. With LOGITS the normalised row stays in LDS and the four wavefronts also take its
// dot products with the E rows of the router (fp32 sums, one rounding to f16), so that the
// router needs no launch of its own; that variant runs 16 wavefronts, each with the loads of
// four experts in flight at once, because the router's rows come from L2 one round trip at a
// time and the trips, not the bytes, are what it waits for.
// With FRONT (and LOGITS) the workgroup then routes its token from the logits in LDS; with FRONT
// == FRONT_SORT the last workgroup of the launch to get there also sorts every token's choices
// (front_core.h): the layer's router GEMM, route and sort in one launch.
// FROM says where a row's inputs are, and each answer is an instance of its own, so that the rows of a
// layer pay for neither of the others (as run-time questions they cost every instance 23 to 37
// instructions, and the logits one a wavefront of occupancy): EMBEDDED looks row t up in x by gather[t], and
// its first workgroup sets the `nclear` counters at `clear` to zero for the launches behind it; TWINNED
// (with COMBINE) takes the expert outputs of token twin[t] (front.hip).
// FEW (with COMBINE): a launch of few rows is a chain of waits. The norm's weights and the row are asked for
// first, and a token's choices are ranked without LDS and their rows of y asked for together (combine_core.h):
// one row 5.2 -> 4.4 us a launch, 8 rows 5.6 -> 5.0. (A replayed graph of such launches, 8 rows of 2048: top-8 4.20 -> 3.73, top-5
// 3.71 -> 3.58, top-4 3.48 -> 3.53 and rows of 3072 4.31 -> 4.13; top-2 would be 3.11 -> 3.42, top-1 3.01 -> 3.35.) It takes 26 more registers, and with many rows it is
// the wavefronts in flight that count: 437 rows 6.7 -> 7.3, 4096 rows 31.9 -> 33.2.
// COUNTED (and PACKED, which is EMBEDDED for such rows): only the first *count of the launch's rows exist (prompt.hip);
// PACKED looks up row t by gather[map[t]].
constexpr int FRONT_ROUTE = 1, FRONT_SORT = 2;
constexpr int OWN_ROWS = 0, EMBEDDED = 1, TWINNED = 2, COUNTED = 3, PACKED = 4;
template <bool COMBINE, bool LOGITS, int FRONT = 0, int FROM = OWN_ROWS, bool FEW = false>
__global__ void __launch_bounds__(LOGITS ? 1024 : ROW_THREADS)
row_kernel(const half_t* x, const half_t* __restrict__ delta, const half_t* __restrict__ y,
           const int* __restrict__ pos_of, const int* __restrict__ idx, int k, const half_t* __restrict__ weight,
           float eps, const half_t* __restrict__ router, int E, int H, half_t* x_out, half_t* h_out,
           half_t* __restrict__ logits, const int64_t* __restrict__ gather, int src_rows,
           front_core::Outputs front = front_core::Outputs{}, const int* __restrict__ twin = nullptr,
           unsigned* __restrict__ clear = nullptr, int nclear = 0, const int* __restrict__ count = nullptr,
           const int* __restrict__ map = nullptr) {  // x_out or h_out may be x
  extern __shared__ __attribute__((aligned(16))) half_t hs[];  // LOGITS: the normalised row [H]; FRONT: the tail's LDS behind it
  __shared__ __attribute__((aligned(16))) float part[16];
  __shared__ int rows[ROW_MAX_K];
  __shared__ float wts[ROW_MAX_K];   // COMBINE: the router weight of each row, 1 where y is already scaled
  const int t = blockIdx.x, tid = threadIdx.x, nthreads = blockDim.x;
  if ((FROM == COUNTED || FROM == PACKED) && t >= *count) return;
  const size_t row = (size_t)t * H;
  const int chunks = H >> 3;
  half8_t v[MAX_CHUNKS], wn[MAX_CHUNKS];
  combine_core::Choices own;
  if (FEW) {
#pragma unroll
    for (int i = 0; i < MAX_CHUNKS; ++i) {
      const int c = tid + i * nthreads;
      if (c < chunks) {
        wn[i] = *reinterpret_cast<const half8_t*>(weight + c * 8);
        v[i] = *reinterpret_cast<const half8_t*>(x + row + c * 8);
      }
    }
    own = combine_core::ranked(idx, pos_of, delta, (size_t)t * k, k);
  }
  const half_t* xrow = x + row;
  if (FROM == EMBEDDED || FROM == PACKED) {
    long g = (long)gather[FROM == PACKED ? map[t] : t];
    g = g < 0 ? 0 : g >= src_rows ? src_rows - 1 : g;
    xrow = x + (size_t)g * H;
    if (FROM == EMBEDDED && t == 0)
      for (int i = tid; i < nclear; i += nthreads) clear[i] = 0;
  }
  if (COMBINE && !FEW) {
    // rank the k choices by (expert id, slot); rows[] lists their rows of y in that order
    if (tid < WAVE) {
      const int of = FROM == TWINNED ? twin[t] : t;
      const int mine = tid < k ? idx[(size_t)of * k + tid] : 0x7fffffff;
      const int src = tid < k ? pos_of[(size_t)of * k + tid] : 0;
      int rank = 0;
      for (int j = 0; j < k; ++j) {
        const int other = read_lane(mine, j);
        rank += (other < mine) || (other == mine && j < tid);
      }
      if (tid < k) {
        rows[rank] = src;
        wts[rank] = delta ? (float)delta[(size_t)of * k + tid] : 1.f;
      }
    }
    __syncthreads();
  }
  float ss = 0.f;
#pragma unroll
  for (int i = 0; i < MAX_CHUNKS; ++i) {
    const int c = tid + i * nthreads;
    if (c < chunks) {
      if (!FEW) v[i] = *reinterpret_cast<const half8_t*>(xrow + c * 8);
      if (COMBINE) {
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        auto fetch = [&](int r) { return __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(y + (size_t)r * H + c * 8)); };   // read once
        // the rounding of the down projection's scaled epilogue (times 1 it changes nothing)
        auto add = [&](half8_t e, float wt) {
#pragma unroll
          for (int q = 0; q < 8; ++q) acc[q] += (float)(half_t)((float)e[q] * wt);
        };
        if (FEW) {
          half8_t e[combine_core::AT_ONCE];
#pragma unroll
          for (int j = 0; j < combine_core::AT_ONCE; ++j) e[j] = fetch(own.row[j]);
#pragma unroll
          for (int j = 0; j < combine_core::AT_ONCE; ++j)
            if (j < k) add(e[j], own.weight[j]);
        } else {
          for (int j = 0; j < k; ++j) add(fetch(rows[j]), wts[j]);
        }
#pragma unroll
        for (int q = 0; q < 8; ++q) v[i][q] = (half_t)((float)v[i][q] + (float)(half_t)acc[q]);
      } else if (delta) {
        const half8_t d = *reinterpret_cast<const half8_t*>(delta + row + c * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) v[i][j] = (half_t)((float)v[i][j] + (float)d[j]);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) ss += (float)v[i][j] * (float)v[i][j];
    }
  }
  if (LOGITS && !weight) {
    // no norm asked for: the logits of the rows as they are (the router GEMM alone)
#pragma unroll
    for (int i = 0; i < MAX_CHUNKS; ++i) {
      const int c = tid + i * nthreads;
      if (c < chunks) *reinterpret_cast<half8_t*>(hs + c * 8) = v[i];
    }
  } else {
    const float rs = rsqrtf((FEW ? block_sum_of_four(ss, part) : block_sum(ss, part, 0)) / (float)H + eps);
#pragma unroll
    for (int i = 0; i < MAX_CHUNKS; ++i) {
      const int c = tid + i * nthreads;
      if (c < chunks) {
        const half8_t w = FEW ? wn[i] : *reinterpret_cast<const half8_t*>(weight + c * 8);
        half8_t h;
#pragma unroll
        for (int j = 0; j < 8; ++j) h[j] = (half_t)((float)w[j] * (float)(half_t)((float)v[i][j] * rs));
        if (x_out) *reinterpret_cast<half8_t*>(x_out + row + c * 8) = v[i];
        *reinterpret_cast<half8_t*>(h_out + row + c * 8) = h;
        if (LOGITS) *reinterpret_cast<half8_t*>(hs + c * 8) = h;
      }
    }
  }
  if (!LOGITS) return;
  __syncthreads();
  // wavefront w takes experts w, w + nwaves, ...: four at a time with every load issued before
  // the first is used (rows of 2048: 16 loads of 16 bytes per lane)
  const int wave = tid >> 6, lane = tid & 63, nwaves = nthreads >> 6;
  for (int e0 = wave; e0 < E; e0 += 4 * nwaves) {
    const half_t* r[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int e = e0 + nwaves * u;
      r[u] = router + (size_t)(e < E ? e : e0) * H;
    }
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    if (chunks == 4 * WAVE) {
      half8_t rv[4][4];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int u = 0; u < 4; ++u) rv[u][i] = *reinterpret_cast<const half8_t*>(r[u] + (lane + WAVE * i) * 8);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const half8_t hv = *reinterpret_cast<const half8_t*>(hs + (lane + WAVE * i) * 8);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[u] += (float)hv[j] * (float)rv[u][i][j];
      }
    } else {
      for (int c = lane; c < chunks; c += WAVE) {
        const half8_t hv = *reinterpret_cast<const half8_t*>(hs + c * 8);
        half8_t rv[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) rv[u] = *reinterpret_cast<const half8_t*>(r[u] + c * 8);
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int j = 0; j < 8; ++j) acc[u] += (float)hv[j] * (float)rv[u][j];
      }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const float total = wave_sum(acc[u]);
      const int e = e0 + nwaves * u;
      if (lane == 0 && e < E) {
        logits[(size_t)t * E + e] = (half_t)total;
        if (FRONT) hs[H + e] = (half_t)total;
      }
    }
  }
  if (FRONT) {
    __syncthreads();
    unsigned char* tail = reinterpret_cast<unsigned char*>(hs + H);
    if (FRONT == FRONT_ROUTE) {
      if (E <= 64) front_core::route_own<1>(t, E, front, tail);
      else front_core::route_own<2>(t, E, front, tail);
    } else if (E <= 64) {
      front_core::route_own_sort_last<1>(t, (int)gridDim.x, E, front, tail);
    } else {
      front_core::route_own_sort_last<2>(t, (int)gridDim.x, E, front, tail);
    }
  }
}

// The router's logits of a few rows for a launch that routes by itself (gemv.hip), with NORM behind the residual add and the
// norm: every token's experts are dealt to E / 4 workgroups, one to a wavefront. A workgroup that has a token's whole router to
// read waits for 256 KB at the 55 to 57 bytes a clock that a compute unit pulls from L2, then routes: 6.9 us a launch with one
// row and 7.6 with 8. Here the router's rows are asked for with the token's, and the norm, which every workgroup of the token
// computes for itself, runs while they are on their way: 2.8 and 4.8, and the stream behind it takes 1.0 and 2.2 more to
// route. x_out must not be x: other workgroups may still have x to read.
constexpr int SPREAD_THREADS = ROW_THREADS, SPREAD_WAVES = SPREAD_THREADS / WAVE, SPREAD_H = SPREAD_THREADS * 8, SPREAD_ROWS = 8;
template <bool NORM>
__global__ void __launch_bounds__(SPREAD_THREADS)
logits_spread_kernel(const half_t* __restrict__ x, const half_t* __restrict__ delta, const half_t* __restrict__ weight, float eps,
                     const half_t* __restrict__ router, int E, half_t* __restrict__ x_out, half_t* __restrict__ h_out,
                     half_t* __restrict__ logits) {
  constexpr int H = SPREAD_H, PER_LANE = H / (WAVE * 8);
  __shared__ __attribute__((aligned(16))) half_t hs[NORM ? H : 8];
  __shared__ __attribute__((aligned(16))) float part[4];
  const int t = blockIdx.y, tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int e = blockIdx.x * SPREAD_WAVES + wave;
  const size_t row = (size_t)t * H;
  half8_t v, d, w, hv[PER_LANE], rv[PER_LANE];
  if (NORM) {
    v = *reinterpret_cast<const half8_t*>(x + row + tid * 8);
    d = *reinterpret_cast<const half8_t*>(delta + row + tid * 8);
    w = *reinterpret_cast<const half8_t*>(weight + tid * 8);
  } else {
#pragma unroll
    for (int i = 0; i < PER_LANE; ++i) hv[i] = *reinterpret_cast<const half8_t*>(x + row + (lane + WAVE * i) * 8);
  }
#pragma unroll
  for (int i = 0; i < PER_LANE; ++i)
    rv[i] = *reinterpret_cast<const half8_t*>(router + (size_t)min(e, E - 1) * H + (lane + WAVE * i) * 8);
  if (NORM) {
    float ss = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = (half_t)((float)v[j] + (float)d[j]);
#pragma unroll
    for (int j = 0; j < 8; ++j) ss += (float)v[j] * (float)v[j];
    const float rs = rsqrtf(block_sum_of_four(ss, part) / (float)H + eps);
    half8_t h;
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = (half_t)((float)w[j] * (float)(half_t)((float)v[j] * rs));
    *reinterpret_cast<half8_t*>(hs + tid * 8) = h;
    if (blockIdx.x == 0) {
      *reinterpret_cast<half8_t*>(x_out + row + tid * 8) = v;
      *reinterpret_cast<half8_t*>(h_out + row + tid * 8) = h;
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < PER_LANE; ++i) hv[i] = *reinterpret_cast<const half8_t*>(hs + (lane + WAVE * i) * 8);
  }
  float acc = 0.f;
#pragma unroll
  for (int i = 0; i < PER_LANE; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc += (float)hv[i][j] * (float)rv[i][j];
  acc = wave_sum(acc);
  if (lane == 0 && e < E) logits[(size_t)t * E + e] = (half_t)acc;
}

__device__ __forceinline__ half_t clamp_f16(half_t v, float clip) {
  if (clip > 0.f) {
    const float f = (float)v;
    return (half_t)(f < -clip ? -clip : f > clip ? clip : f);
  }
  return v;
}

// out = f16(f16(y * cos) + f16(rot * sin)): three roundings, as three PyTorch operators on
// fp16 tensors make them. Contraction is switched off here, or the compiler narrows the
// arithmetic to fp16 and fuses product and sum into one fma with a single rounding.
__device__ __forceinline__ half_t rotary_f16(half_t y, half_t rot, half_t cos_v, half_t sin_v) {
#pragma clang fp contract(off)
  const half_t t1 = (half_t)((float)y * (float)cos_v);
  const half_t t2 = (half_t)((float)rot * (float)sin_v);
  return (half_t)((float)t1 + (float)t2);
}

// The same for eight elements, and the RMS norm's scaling and clamp before it. The product of two f16 numbers is exact
// in fp32, and their sum is rounded to f16 alike from fp32 or at once (24 bits are twice 11 and two more), so f16
// arithmetic, two elements to an instruction, has the roundings that fp32 arithmetic followed by a conversion has. The
// scaling by an fp32 number is the one product that is not exact: elsewhere it is compiled to v_fma_mixlo_f16, which
// rounds once, and over a vector to a product and a conversion, which round twice; the instruction is named here so
// that every kernel's keys are the same. These kernels are bound by the instructions in front of their loops: decode
// attention of 8 sequences 13.7 -> 12.7 us a launch, of 64 45.6 -> 44.0, the prompts' q/k norm of 8 x 512 23.7 -> 19.3.
__device__ __forceinline__ half8_t norm_f16x8(half8_t x, half8_t w, float rs, float clip) {
  typedef int i4_t __attribute__((ext_vector_type(4)));
  i4_t in = __builtin_bit_cast(i4_t, x), out;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    int pair;
    asm("v_fma_mixlo_f16 %0, %1, %2, 0 op_sel_hi:[1,0,0]" : "=v"(pair) : "v"(in[j]), "v"(rs));
    asm("v_fma_mixhi_f16 %0, %1, %2, 0 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "+v"(pair) : "v"(in[j]), "v"(rs));
    out[j] = pair;
  }
  half8_t h = w * __builtin_bit_cast(half8_t, out);
  if (clip > 0.f) {
#pragma unroll
    for (int j = 0; j < 8; ++j) h[j] = clamp_f16(h[j], clip);
  }
  return h;
}
__device__ __forceinline__ half8_t rotary_f16x8(half8_t y, half8_t rot, half8_t cos_v, half8_t sin_v) {
#pragma clang fp contract(off)
  const half8_t t1 = y * cos_v;
  const half8_t t2 = rot * sin_v;
  return t1 + t2;
}

// One workgroup per token. qkv row = [q (heads*D) | k (kv_heads*D) | v (kv_heads*D)].
// PROMPT: the first token goes to cache position `first`. With `place`, rows of padding that are the same in every layer
// exist once (prompt.hip): position r is row place[r], or, where it is one of those but not the first of them,
// row ~place[r], of which only key and value are made again, for its own place in the cache.
template <bool PROMPT>
__global__ void __launch_bounds__(ROW_THREADS)
qk_norm_rope_cache_kernel(const half_t* __restrict__ qkv, const half_t* __restrict__ q_norm,
                          const half_t* __restrict__ k_norm, float eps, float clip, const half_t* __restrict__ cos_t,
                          const half_t* __restrict__ sin_t, int max_positions, const int64_t* __restrict__ positions,
                          const int64_t* __restrict__ slot_ptr, int T, int heads, int kv_heads, int D, int capacity,
                          half_t* __restrict__ q_out, half_t* __restrict__ kcache, half_t* __restrict__ vcache,
                          const int* __restrict__ place = nullptr, int first = 0) {
  extern __shared__ __attribute__((aligned(16))) half_t normed[];  // [qd + kvd] after norm and clamp
  __shared__ float part[32];
  // row r of qkv is token t = r % T of sequence b = r / T; it goes to cache position slot + t
  const int r = blockIdx.x, b = r / T;
  const int qd = heads * D, kvd = kv_heads * D;
  int at = r;
  if (PROMPT && place) at = place[r];
  const bool own = at >= 0;   // the same in the whole workgroup
  at = own ? at : ~at;
  const half_t* row = qkv + (size_t)at * (qd + 2 * kvd);
  const int qchunks = own ? qd >> 3 : 0, kchunks = kvd >> 3;
  const long slot = (PROMPT ? (long)first : (long)*slot_ptr) + (r - b * T);
  long pos = (long)positions[r];
  pos = pos < 0 ? 0 : pos >= max_positions ? max_positions - 1 : pos;
  const bool slot_ok = slot >= 0 && slot < capacity;

  half8_t q[MAX_CHUNKS], k[MAX_CHUNKS];
  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int i = 0; i < MAX_CHUNKS; ++i) {
    const int c = threadIdx.x + i * ROW_THREADS;
    if (c < qchunks) {
      q[i] = *reinterpret_cast<const half8_t*>(row + c * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) sq += (float)q[i][j] * (float)q[i][j];
    }
    if (c < kchunks) {
      k[i] = *reinterpret_cast<const half8_t*>(row + qd + c * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) sk += (float)k[i][j] * (float)k[i][j];
    }
  }
  const float rq = rsqrtf(block_sum(sq, part, 0) / (float)qd + eps);
  const float rk = rsqrtf(block_sum(sk, part, 16) / (float)kvd + eps);
#pragma unroll
  for (int i = 0; i < MAX_CHUNKS; ++i) {
    const int c = threadIdx.x + i * ROW_THREADS;
    if (c < qchunks) {
      const half8_t w = *reinterpret_cast<const half8_t*>(q_norm + c * 8);
      half8_t o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = clamp_f16((half_t)((float)w[j] * (float)(half_t)((float)q[i][j] * rq)), clip);
      *reinterpret_cast<half8_t*>(normed + c * 8) = o;
    }
    if (c < kchunks) {
      const half8_t w = *reinterpret_cast<const half8_t*>(k_norm + c * 8);
      half8_t o;
#pragma unroll
      for (int j = 0; j < 8; ++j)
        o[j] = clamp_f16((half_t)((float)w[j] * (float)(half_t)((float)k[i][j] * rk)), clip);
      *reinterpret_cast<half8_t*>(normed + qd + c * 8) = o;
    }
  }
  __syncthreads();

  // rotary embedding: out[d] = f16(y[d] * cos[d]) + f16(rot[d] * sin[d]), rot = [-y[D/2:], y[:D/2]]
  const int half_d = D >> 1;
  const half_t* cs = cos_t + (size_t)pos * D;
  const half_t* sn = sin_t + (size_t)pos * D;
  for (int c = (own ? 0 : qd >> 3) + threadIdx.x; c < (qd >> 3) + kchunks; c += ROW_THREADS) {
    const int d0 = (c * 8) % D;  // qd is a multiple of D, so this also holds in the k part
    const half8_t y = *reinterpret_cast<const half8_t*>(normed + c * 8);
    const bool low = d0 < half_d;
    const half8_t other = *reinterpret_cast<const half8_t*>(normed + c * 8 + (low ? half_d : -half_d));
    const half8_t cc = *reinterpret_cast<const half8_t*>(cs + d0);
    const half8_t ssn = *reinterpret_cast<const half8_t*>(sn + d0);
    half8_t o;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      o[j] = rotary_f16(y[j], low ? -other[j] : other[j], cc[j], ssn[j]);
    }
    if (c < qchunks) {
      *reinterpret_cast<half8_t*>(q_out + (size_t)at * qd + c * 8) = o;
    } else if (slot_ok) {
      const int e = (c - (qd >> 3)) * 8, h = e / D;
      *reinterpret_cast<half8_t*>(kcache + (((size_t)b * kv_heads + h) * capacity + slot) * D + (e - h * D)) = o;
    }
  }
  if (slot_ok) {
    for (int c = threadIdx.x; c < kchunks; c += ROW_THREADS) {
      half8_t v = *reinterpret_cast<const half8_t*>(row + qd + kvd + c * 8);
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = clamp_f16(v[j], clip);
      const int e = c * 8, h = e / D;
      *reinterpret_cast<half8_t*>(vcache + (((size_t)b * kv_heads + h) * capacity + slot) * D + (e - h * D)) = v;
    }
  }
}

// qk_norm_rope_cache_kernel<true> for projections of at most 2048 and heads of 64 or 128: a thread has one 16-byte chunk each
// of q, k and v, and everything it reads is asked for at once. With six waits one after the other (row, sums, norm
// weights, rotary table, values) a workgroup took 11 us whatever the batch, and 2048 workgroups are all that fit:
// 437 rows 7.1 -> 5.5 us a launch, 8 prompts of 256 to 512 26.7 -> 22.5, 3 of 1000 to 2000 35.6 -> 28.9. The chunk half a head further on, which the rotary embedding mixes in, is in a lane
// of the same wavefront, so nothing but the sums goes through LDS. The same bits.
template <int D>
__global__ void __launch_bounds__(ROW_THREADS)
qk_norm_rope_prompt_kernel(const half_t* __restrict__ qkv, const half_t* __restrict__ q_norm, const half_t* __restrict__ k_norm,
                           float eps, float clip, const half_t* __restrict__ cos_t, const half_t* __restrict__ sin_t,
                           int max_positions, const int64_t* __restrict__ positions, int first, const int* __restrict__ place, int T,
                           int qd, int kvd, int capacity, half_t* __restrict__ q_out, half_t* __restrict__ kcache,
                           half_t* __restrict__ vcache) {
  constexpr int PARTNER = D / 16;   // chunks to the other half of the head
  __shared__ __attribute__((aligned(16))) float part[8];
  const int r = blockIdx.x, b = r / T, tid = threadIdx.x, e = tid * 8;
  long pos = (long)positions[r];
  int at = place ? place[r] : r;
  const bool own = at >= 0;   // the same in the whole workgroup
  at = own ? at : ~at;
  pos = pos < 0 ? 0 : pos >= max_positions ? max_positions - 1 : pos;
  const half_t* row = qkv + (size_t)at * (qd + 2 * kvd);
  const half8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const bool has_q = own && e < qd, has_k = e < kvd;
  half8_t q = zero8, k = zero8, v = zero8, wq = zero8, wk = zero8;
  if (has_q) {
    q = *reinterpret_cast<const half8_t*>(row + e);
    wq = *reinterpret_cast<const half8_t*>(q_norm + e);
  }
  if (has_k) {
    k = *reinterpret_cast<const half8_t*>(row + qd + e);
    wk = *reinterpret_cast<const half8_t*>(k_norm + e);
  }
  const int d0 = e % D;
  const half8_t cc = *reinterpret_cast<const half8_t*>(cos_t + (size_t)pos * D + d0);
  const half8_t ss = *reinterpret_cast<const half8_t*>(sin_t + (size_t)pos * D + d0);
  if (has_k) v = *reinterpret_cast<const half8_t*>(row + qd + kvd + e);

  float sq = 0.f, sk = 0.f;
#pragma unroll
  for (int j = 0; j < 8; ++j) sq += (float)q[j] * (float)q[j];
#pragma unroll
  for (int j = 0; j < 8; ++j) sk += (float)k[j] * (float)k[j];
  sq = wave_sum(sq);
  sk = wave_sum(sk);
  if ((tid & 63) == 0) {
    part[tid >> 6] = sq;
    part[4 + (tid >> 6)] = sk;
  }
  __syncthreads();
  const float4_t pq = *reinterpret_cast<const float4_t*>(part), pk = *reinterpret_cast<const float4_t*>(part + 4);
  const float rq = rsqrtf((pq[0] + pq[1] + pq[2] + pq[3]) / (float)qd + eps);
  const float rk = rsqrtf((pk[0] + pk[1] + pk[2] + pk[3]) / (float)kvd + eps);
  const bool low = d0 < D / 2;
  auto rotate = [&](half8_t x, half8_t w, float rs) {
    typedef int i4_t __attribute__((ext_vector_type(4)));
    const half8_t y = norm_f16x8(x, w, rs, clip);
    i4_t words = __builtin_bit_cast(i4_t, y);
#pragma unroll
    for (int j = 0; j < 4; ++j) words[j] = __shfl_xor(words[j], PARTNER, WAVE);
    const half8_t other = __builtin_bit_cast(half8_t, words);
    return rotary_f16x8(y, low ? -other : other, cc, ss);
  };
  const half8_t qo = rotate(q, wq, rq), ko = rotate(k, wk, rk);
  if (has_q) *reinterpret_cast<half8_t*>(q_out + (size_t)at * qd + e) = qo;
  const int slot = first + (r - b * T);
  if (has_k && slot < capacity) {
    const int h = e / D;
    const size_t to = (((size_t)b * (kvd / D) + h) * capacity + slot) * D + d0;
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = clamp_f16(v[j], clip);
    *reinterpret_cast<half8_t*>(kcache + to) = ko;
    *reinterpret_cast<half8_t*>(vcache + to) = v;
  }
}

// Sum over the LPK lanes that share a key (LPK = 16: one DPP row; 8: half a row).
template <int LPK>
__device__ __forceinline__ float key_sum(float v) {
  if (LPK == 16) return row_allreduce(v, [](float a, float b) { return a + b; });
  v += __shfl_xor(v, 4, WAVE);
  v += __shfl_xor(v, 2, WAVE);
  v += __shfl_xor(v, 1, WAVE);
  return v;
}

constexpr float MASKED = -1.0e30f;   // running maximum before any key was seen
constexpr int ATT_WAVES = 16;   // wavefronts of a (sequence, head) pair where there are few pairs

// One workgroup per (sequence, query head), NW wavefronts. A load instruction covers KPL =
// 64 / LPK consecutive keys (LPK = D / 8 lanes per key, 16 bytes per lane: whole 256-byte rows
// for D = 128), so the cache is read as long contiguous runs. Each group of LPK lanes keeps its
// own running softmax (maximum, sum, 8 output dimensions per lane) over the keys it meets, so
// the key loop has no cross-lane traffic except the score's sum; the KPL x NW partial results
// are merged once at the end.
// What the fused variant needs beyond the plain one: the projections' output and what
// qk_norm_rope_cache takes.
struct NewToken {
  const half_t* qkv;      // [B, (heads + 2 kv_heads) D]
  const half_t* q_norm;   // [heads D]
  const half_t* k_norm;   // [kv_heads D]
  const half_t* cos_t;    // [max_positions, D]
  const half_t* sin_t;
  const int64_t* positions;
  half_t* kcache_w;       // the caches again, writable
  half_t* vcache_w;
  uint8_t* real_w;        // the mask again, writable: the new token's position becomes real
  float eps, clip;
  int max_positions;
};

// A head's 16-byte chunk c of a projection, loaded with everything its norm and rotary
// embedding need, so that the loads are in flight before the norm's scale is known.
template <int LPK>
struct HeadChunk {
  half8_t mine, other, wm, wo;
  __device__ __forceinline__ void load(const half_t* head, const half_t* norm_w, int c) {
    const int partner = c ^ (LPK / 2);
    mine = *reinterpret_cast<const half8_t*>(head + c * 8);
    other = *reinterpret_cast<const half8_t*>(head + partner * 8);
    wm = *reinterpret_cast<const half8_t*>(norm_w + c * 8);
    wo = *reinterpret_cast<const half8_t*>(norm_w + partner * 8);
  }
  // RMS norm (scale rs), clamp and rotary embedding, with the roundings of qk_norm_rope_cache
  __device__ __forceinline__ half8_t finish(float rs, float clip, half8_t cc, half8_t ss, int c) const {
    const half8_t a = norm_f16x8(mine, wm, rs, clip), r = norm_f16x8(other, wo, rs, clip);
    return rotary_f16x8(a, c < LPK / 2 ? -r : r, cc, ss);
  }
};

// A batch of UNROLL key groups of one wavefront: 16 bytes of key and of value per lane each, and the key's byte of the
// mask (0 where there is no key). The byte stays as it is loaded until the batch is used: compared to zero where it
// is asked for, it is waited for there, and with it every load before, one group after the other.
template <int UNROLL>
struct KeyBatch {
  half8_t kk[UNROLL], vv[UNROLL];
  unsigned mask[UNROLL];
};

// FUSED: the query is taken from the projections' output (norm over the whole q and k rows of
// the sequence, clamp, rotary embedding: the work of qk_norm_rope_cache, redone by every
// workgroup for its own head, which costs two 4 KB reads from L2), the new key and value are
// used from registers as the last key, and the first query head of each kv head writes them
// into the cache; the loop then covers the cached keys before `slot` only.
// The first batch of keys and values is requested before any of that. (Requesting each further
// batch while the previous one is multiplied costs registers, hence resident wavefronts, and
// with them bandwidth: 67.5 us against 55.3 us at 64 sequences x 16 heads x 536 keys.)
// LW wavefronts per (sequence, head) pair, each with a batch of UNROLL key groups in flight: 16 when
// there are few pairs, so that the cache is still read by many, 4 when the pairs fill the chip.
// Batches in front of the sequence's first real key (left padding) are not read: every wavefront looks
// for that key in the mask itself. At 64 sequences of 288 to 576 keys, 16 heads: 52.6 us a launch with them,
// 45.6 without.
// NW < LW: the pair's wavefronts are dealt to LW / NW workgroups, so that a pair's keys and values (358 KB
// at 700 keys of 128) come through four compute units and not one: 17.2 -> 14.6 us for one sequence of
// 700 keys, 15.5 -> 14.7 for 8 of 256 to 512 (16 workgroups of one wavefront, each with the whole of
// the norms to do: 16.0 for one sequence).
// Every workgroup leaves its wavefronts' results in `parts` and draws a number from the pair's
// ticket; the one that draws the last merges them, as a workgroup of LW wavefronts would have done (the
// same bits), and sets the ticket back to zero. Nobody waits for anybody. The results travel by
// agent-scope atomic stores and loads, which go past the XCDs' own L2s, and the store counter is
// waited for before the draw: a release fence would write back the whole L2 of the XCD each time
// (22 us a launch at 1024 workgroups).
template <int LPK, bool FUSED, int NW, int UNROLL, int LW = NW>
__global__ void __launch_bounds__(NW * WAVE)
decode_attention_kernel(const half_t* __restrict__ q, const half_t* kcache, const half_t* vcache,
                                        const uint8_t* __restrict__ real, const int64_t* __restrict__ slot_ptr,
                                        int heads, int kv_heads, int capacity, float scale_log2e,
                                        half_t* __restrict__ out, NewToken nt, float* __restrict__ parts,
                                        unsigned* __restrict__ tickets) {
  constexpr int D = LPK * 8, KPL = WAVE / LPK;
  constexpr int SPLITS = LW / NW;   // workgroups per pair
  constexpr bool SPLIT = SPLITS > 1;
  extern __shared__ float merge[];  // [NW][D + 2]: accumulators, maximum, sum
  __shared__ float part[32];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int sub = lane / LPK, c = lane % LPK;
  const int pair = blockIdx.x / SPLITS, vwave = blockIdx.x % SPLITS * NW + wave;   // the wavefront's number in its pair
  const int b = pair / heads, qh = pair % heads;
  const int group = heads / kv_heads, kvh = qh / group;
  const half8_t zero8 = {0, 0, 0, 0, 0, 0, 0, 0};
  const int qd = heads * D, kvd = kv_heads * D;
  const bool owner = vwave < NW;   // the workgroup of the pair's first wavefronts takes the new key
  const half_t* row = nt.qkv + (size_t)b * (qd + 2 * kvd);
  HeadChunk<LPK> hq, hk;
  half8_t knew = zero8, vnew = zero8, cc = zero8, ss = zero8;
  half8_t eq[SPLITS], ek[SPLITS];   // 16-byte chunks of the q row and of the k row, for their norms
  long pos = FUSED ? (long)nt.positions[b] : 0;
  auto new_row = [&] {
#pragma unroll
    for (int u = 0; u < SPLITS; ++u) {
      const int i = (u * NW + wave) * WAVE + lane;
      eq[u] = ek[u] = zero8;
      if (i < (qd >> 3)) eq[u] = *reinterpret_cast<const half8_t*>(row + i * 8);
      if (owner && i < (kvd >> 3)) ek[u] = *reinterpret_cast<const half8_t*>(row + qd + i * 8);
    }
    hq.load(row + qh * D, nt.q_norm + qh * D, c);
    hk.load(row + qd + kvh * D, nt.k_norm + kvh * D, c);
    vnew = *reinterpret_cast<const half8_t*>(row + qd + kvd + kvh * D + c * 8);
    pos = pos < 0 ? 0 : pos >= nt.max_positions ? nt.max_positions - 1 : pos;
    cc = *reinterpret_cast<const half8_t*>(nt.cos_t + (size_t)pos * D + c * 8);
    ss = *reinterpret_cast<const half8_t*>(nt.sin_t + (size_t)pos * D + c * 8);
  };
  // Loads return in order, so what stands behind the keys and values is waited for with them: the new
  // token's row, which does not depend on the slot, goes first (64 sequences 46.8 -> 45.6 us), except
  // where 16 wavefronts ask at once and the keys are late enough as it is (17.2 against 18.0 at one).
  constexpr bool ROW_FIRST = NW < ATT_WAVES;
  if (FUSED && ROW_FIRST) new_row();
  const long slot = (long)*slot_ptr;
  long n = FUSED ? slot : slot + 1;   // cached keys the loop visits
  n = n < 0 ? 0 : n > capacity ? capacity : n;
  const size_t base = ((size_t)b * kv_heads + kvh) * (size_t)capacity * D + c * 8;
  const uint8_t* rl = real + (size_t)b * capacity;
  const int groups = ((int)n + KPL - 1) / KPL;
  constexpr int STRIDE = LW * UNROLL;   // key groups of one batch of all the pair's wavefronts
  // the first batch that holds a real key, found 512 positions at a time (few pairs wait for the
  // look at the mask longer than for the batches it would spare)
  int from = LW > 4 ? 0 : groups;
  for (int p0 = LW > 4 ? (int)n : 0; p0 < (int)n; p0 += 8 * WAVE) {
    uint8_t at[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) at[u] = rl[min(p0 + u * WAVE + lane, (int)n - 1)];
    int first = 8 * WAVE;
#pragma unroll
    for (int u = 7; u >= 0; --u) {
      const uint64_t seen = __ballot(at[u] != 0);
      if (seen) first = u * WAVE + __builtin_ctzll(seen);
    }
    if (first < 8 * WAVE) {
      from = (p0 + first) / (STRIDE * KPL) * STRIDE;
      break;
    }
  }
  auto fetch = [&](KeyBatch<UNROLL>& kb, int g0) {
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const int key = (g0 + u * LW) * KPL + sub;
      kb.mask[u] = 0;
      kb.kk[u] = zero8;
      kb.vv[u] = zero8;
      if (key < n) {
        kb.kk[u] = __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(kcache + base + (size_t)key * D));   // the cache is
        kb.vv[u] = __builtin_nontemporal_load(reinterpret_cast<const half8_t*>(vcache + base + (size_t)key * D));   // read once a step
        kb.mask[u] = rl[key];
      }
    }
  };
  KeyBatch<UNROLL> ka;
  fetch(ka, from + vwave);   // requested before the rest of the prologue, so that the two waits overlap

  float qf[8];
  if (FUSED && !ROW_FIRST) new_row();
  if (FUSED) {
    // The sums of squares as LW wavefronts would take them, whose sums are then added in order: a
    // workgroup of fewer takes the others' shares one after the other.
    float sq = 0.f, sk = 0.f;
#pragma unroll
    for (int u = 0; u < SPLITS; ++u) {
      const int v = u * NW + wave;
      float q2 = 0.f, k2 = 0.f;
      auto square = [](float& sum, half8_t e) {
#pragma unroll
        for (int j = 0; j < 8; ++j) sum += (float)e[j] * (float)e[j];
      };
      // the chunk that was asked for first (zero where the row has none), then those of longer rows
      square(q2, eq[u]);
      for (int i = (LW + v) * WAVE + lane; i < (qd >> 3); i += LW * WAVE) square(q2, *reinterpret_cast<const half8_t*>(row + i * 8));
      if (owner) {
        square(k2, ek[u]);
        for (int i = (LW + v) * WAVE + lane; i < (kvd >> 3); i += LW * WAVE)
          square(k2, *reinterpret_cast<const half8_t*>(row + qd + i * 8));
      }
      q2 = wave_sum(q2);
      k2 = wave_sum(k2);
      if (lane == 0) {
        part[v] = q2;
        part[16 + v] = k2;
      }
    }
    // both sums through one barrier
    __syncthreads();
    for (int w = 0; w < LW; ++w) {
      sq += part[w];
      sk += part[16 + w];
    }
    const float rq = rsqrtf(sq / (float)qd + nt.eps), rk = rsqrtf(sk / (float)kvd + nt.eps);
    const half8_t qv = hq.finish(rq, nt.clip, cc, ss, c);
#pragma unroll
    for (int j = 0; j < 8; ++j) qf[j] = (float)qv[j] * scale_log2e;
    if (vwave == 0) {   // the same in the whole wavefront
      knew = hk.finish(rk, nt.clip, cc, ss, c);
#pragma unroll
      for (int j = 0; j < 8; ++j) vnew[j] = clamp_f16(vnew[j], nt.clip);
    }
    if (slot >= 0 && slot < capacity && qh % group == 0 && vwave == 0 && sub == 0) {
      const size_t at = (((size_t)b * kv_heads + kvh) * capacity + slot) * D + c * 8;
      *reinterpret_cast<half8_t*>(nt.kcache_w + at) = knew;
      *reinterpret_cast<half8_t*>(nt.vcache_w + at) = vnew;
      // no workgroup of this launch reads the mask at `slot`: the loop stops before it
      if (qh == 0 && c == 0) nt.real_w[(size_t)b * capacity + slot] = 1;
    }
  } else {
    const half8_t qv = *reinterpret_cast<const half8_t*>(q + ((size_t)b * heads + qh) * D + c * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) qf[j] = (float)qv[j] * scale_log2e;
  }

  float m = MASKED, l = 0.f, acc[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] = 0.f;

  auto consume = [&](const KeyBatch<UNROLL>& kb) {
    float s[UNROLL], mx = m;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      float d = 0.f;
#pragma unroll
      for (int j = 0; j < 8; ++j) d += qf[j] * (float)kb.kk[u][j];
      s[u] = key_sum<LPK>(d);
      if (kb.mask[u] != 0) mx = fmaxf(mx, s[u]);
    }
    const float alpha = __builtin_amdgcn_exp2f(m - mx);
    m = mx;
    l *= alpha;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] *= alpha;
#pragma unroll
    for (int u = 0; u < UNROLL; ++u) {
      const float p = kb.mask[u] != 0 ? __builtin_amdgcn_exp2f(s[u] - mx) : 0.f;
      l += p;
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[j] += p * (float)kb.vv[u][j];
    }
  };
  if (SPLIT) {   // few wavefronts on a compute unit, registers to spare: a batch ahead
    KeyBatch<UNROLL> kb;
    for (int g0 = from + vwave; g0 < groups; g0 += 2 * STRIDE) {
      fetch(kb, g0 + STRIDE);
      consume(ka);
      if (g0 + STRIDE >= groups) break;
      fetch(ka, g0 + 2 * STRIDE);
      consume(kb);
    }
  } else {
    for (int g0 = from + vwave; g0 < groups; g0 += STRIDE) {
      if (g0 != from + vwave) fetch(ka, g0);
      consume(ka);
    }
  }

  if (FUSED && vwave == 0 && slot >= 0 && slot < capacity) {
    // the new token's own key and value, from registers: one more key for the first key group
    float d = 0.f;
#pragma unroll
    for (int j = 0; j < 8; ++j) d += qf[j] * (float)knew[j];
    const float sc = key_sum<LPK>(d);
    const bool ok = sub == 0;   // the new token is real
    const float mx = ok ? fmaxf(m, sc) : m;
    const float alpha = __builtin_amdgcn_exp2f(m - mx);
    const float p = ok ? __builtin_amdgcn_exp2f(sc - mx) : 0.f;
    m = mx;
    l = l * alpha + p;
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] = acc[j] * alpha + p * (float)vnew[j];
  }

  // ---- merge the KPL key groups of the wavefront (lanes with equal c)
  float mw = m;
#pragma unroll
  for (int off = LPK; off < WAVE; off <<= 1) mw = fmaxf(mw, __shfl_xor(mw, off, WAVE));
  const float a = __builtin_amdgcn_exp2f(m - mw);
  l *= a;
#pragma unroll
  for (int j = 0; j < 8; ++j) acc[j] *= a;
#pragma unroll
  for (int off = LPK; off < WAVE; off <<= 1) {
    l += __shfl_xor(l, off, WAVE);
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[j] += __shfl_xor(acc[j], off, WAVE);
  }
  float* mine = merge + wave * (D + 2);
  if (sub == 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) mine[c * 8 + j] = acc[j];
    if (c == 0) {
      mine[D] = mw;
      mine[D + 1] = l;
    }
  }
  __syncthreads();
  // ---- merge the wavefronts: lane i of the first one finishes output dimensions i, i + 64
  if (wave != 0) return;
  constexpr int DIMS = D / WAVE;
  float pm[LW], pl[LW], pa[LW][DIMS];   // every wavefront's maximum, sum and accumulators
  if (SPLIT) {
    float* all = parts + (size_t)pair * LW * (D + 2);
    for (int i = lane; i < NW * (D + 2); i += WAVE)
      __hip_atomic_store(all + vwave * (D + 2) + i, merge[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // they are where every XCD's atomic loads find them
    unsigned drawn = 0;
    if (lane == 0) drawn = __hip_atomic_fetch_add(tickets + pair, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (__builtin_amdgcn_readfirstlane(drawn) != (unsigned)(SPLITS - 1)) return;
    asm volatile("" ::: "memory");
    if (lane == 0) __hip_atomic_store(tickets + pair, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    auto get = [&](int i) { return __hip_atomic_load(all + i, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT); };
#pragma unroll
    for (int w = 0; w < LW; ++w) {
      pm[w] = get(w * (D + 2) + D);
      pl[w] = get(w * (D + 2) + D + 1);
#pragma unroll
      for (int i = 0; i < DIMS; ++i) pa[w][i] = get(w * (D + 2) + i * WAVE + lane);
    }
  } else {
#pragma unroll
    for (int w = 0; w < LW; ++w) {
      pm[w] = merge[w * (D + 2) + D];
      pl[w] = merge[w * (D + 2) + D + 1];
#pragma unroll
      for (int i = 0; i < DIMS; ++i) pa[w][i] = merge[w * (D + 2) + i * WAVE + lane];
    }
  }
  float M = MASKED, den = 0.f, num[DIMS] = {};
#pragma unroll
  for (int w = 0; w < LW; ++w) M = fmaxf(M, pm[w]);
#pragma unroll
  for (int w = 0; w < LW; ++w) {
    const float f = __builtin_amdgcn_exp2f(pm[w] - M);
    den += f * pl[w];
#pragma unroll
    for (int i = 0; i < DIMS; ++i) num[i] += f * pa[w][i];
  }
#pragma unroll
  for (int i = 0; i < DIMS; ++i)
    out[((size_t)b * heads + qh) * D + i * WAVE + lane] = (half_t)(den > 0.f ? num[i] / den : 0.f);
}

// One workgroup per sequence: the arg-max of its logits (the lowest index among equal maxima)
// becomes its next token, is appended to its output row, and its rotary position advances;
// the first workgroup also advances the cache slot, which nothing in this launch reads.
constexpr int PICK_THREADS = 1024;

__global__ void __launch_bounds__(PICK_THREADS)
greedy_advance_kernel(const half_t* __restrict__ logits, int V, int64_t* __restrict__ tok, int64_t* __restrict__ out,
                      int out_stride, const int64_t* __restrict__ base_position, int64_t* __restrict__ next_position,
                      int64_t* __restrict__ slot) {
  __shared__ float best_v[PICK_THREADS / WAVE];
  __shared__ int best_i[PICK_THREADS / WAVE];
  const int b = blockIdx.x, tid = threadIdx.x;
  const half_t* row = logits + (size_t)b * V;
  float bv = -INFINITY;
  int bi = 0x7fffffff;
  const int chunks = V % 8 == 0 ? V >> 3 : 0;   // 16-byte loads need rows that start on 16 bytes
  for (int c = tid; c < chunks; c += PICK_THREADS) {
    const half8_t v = *reinterpret_cast<const half8_t*>(row + c * 8);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float f = (float)v[j];
      if (f > bv) {           // ascending indices per thread: the first of equal values is kept
        bv = f;
        bi = c * 8 + j;
      }
    }
  }
  for (int i = chunks * 8 + tid; i < V; i += PICK_THREADS) {
    const float f = (float)row[i];
    if (f > bv) {
      bv = f;
      bi = i;
    }
  }
  // wavefront, then workgroup: larger value wins, equal values go to the lower index
  for (int off = 32; off > 0; off >>= 1) {
    const float ov = __shfl_xor(bv, off, WAVE);
    const int oi = __shfl_xor(bi, off, WAVE);
    if (ov > bv || (ov == bv && oi < bi)) {
      bv = ov;
      bi = oi;
    }
  }
  if ((tid & 63) == 0) {
    best_v[tid >> 6] = bv;
    best_i[tid >> 6] = bi;
  }
  __syncthreads();
  if (tid == 0) {
    for (int w = 1; w < PICK_THREADS / WAVE; ++w)
      if (best_v[w] > bv || (best_v[w] == bv && best_i[w] < bi)) {
        bv = best_v[w];
        bi = best_i[w];
      }
    if (bi == 0x7fffffff) bi = 0;   // a row of NaNs or -inf: token 0
    tok[b] = bi;
    const long col = (long)(next_position[b] - base_position[b]);
    if (col >= 0 && col < out_stride) out[(size_t)b * out_stride + col] = bi;
    next_position[b] += 1;
    if (b == 0) *slot += 1;
  }
}

}  // namespace

#define ROW_LIMITS(what)                                                                          \
  SY_REQUIRE(N >= 0 && H >= 8 && H % 8 == 0 && H <= 8 * ROW_THREADS * MAX_CHUNKS,                \
             what ": N = %d, H = %d (a multiple of 8 up to %d)", N, H, 8 * ROW_THREADS * MAX_CHUNKS)

extern "C" SY_API int sy_add_rmsnorm(const void* x, const void* delta, const void* weight, float eps, int N, int H,
                                     void* x_out, void* h_out, void* stream) {
  ROW_LIMITS("add_rmsnorm");
  if (N == 0) return SY_OK;
  SY_REQUIRE(x && weight && h_out, "add_rmsnorm: null pointer");
  row_kernel<false, false><<<N, ROW_THREADS, 0, (hipStream_t)stream>>>(
      (const half_t*)x, (const half_t*)delta, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps, nullptr, 0, H,
      (half_t*)x_out, (half_t*)h_out, nullptr, nullptr, 0);
  return sy_check_launch("add_rmsnorm");
}

int sy_embed_rmsnorm_step(const int64_t* tokens, const void* embed, int vocab, const void* weight, float eps, int N, int H,
                          void* x_out, void* h_out, unsigned* clear, int nclear, void* stream) {
  ROW_LIMITS("embed_rmsnorm");
  SY_REQUIRE(vocab >= 1, "embed_rmsnorm: vocab = %d", vocab);
  if (N == 0) return SY_OK;
  SY_REQUIRE(tokens && embed && weight && x_out && h_out && (clear || !nclear), "embed_rmsnorm: null pointer");
  row_kernel<false, false, 0, EMBEDDED><<<N, ROW_THREADS, 0, (hipStream_t)stream>>>(
      (const half_t*)embed, nullptr, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps, nullptr, 0, H,
      (half_t*)x_out, (half_t*)h_out, nullptr, tokens, vocab, front_core::Outputs{}, nullptr, clear, nclear);
  return sy_check_launch("embed_rmsnorm");
}

extern "C" SY_API int sy_embed_rmsnorm(const int64_t* tokens, const void* embed, int vocab, const void* weight, float eps,
                                       int N, int H, void* x_out, void* h_out, void* stream) {
  return sy_embed_rmsnorm_step(tokens, embed, vocab, weight, eps, N, H, x_out, h_out, nullptr, 0, stream);
}

// The rows of a packed batch of prompts (prompt.hip): the first *count of N, row t from tokens[map[t]].
int sy_embed_rmsnorm_packed(const int64_t* tokens, const int32_t* map, const int32_t* count, const void* embed, int vocab,
                            const void* weight, float eps, int N, int H, void* x_out, void* h_out, void* stream) {
  ROW_LIMITS("embed_rmsnorm");
  SY_REQUIRE(vocab >= 1, "embed_rmsnorm: vocab = %d", vocab);
  if (N == 0) return SY_OK;
  SY_REQUIRE(tokens && map && count && embed && weight && x_out && h_out, "embed_rmsnorm: null pointer");
  row_kernel<false, false, 0, PACKED><<<N, ROW_THREADS, 0, (hipStream_t)stream>>>(
      (const half_t*)embed, nullptr, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps, nullptr, 0, H, (half_t*)x_out,
      (half_t*)h_out, nullptr, tokens, vocab, front_core::Outputs{}, nullptr, nullptr, 0, count, map);
  return sy_check_launch("embed_rmsnorm");
}

int sy_add_rmsnorm_counted(const void* x, const void* delta, const void* weight, float eps, int N, const int32_t* count, int H,
                           void* x_out, void* h_out, void* stream) {
  if (!count) return sy_add_rmsnorm(x, delta, weight, eps, N, H, x_out, h_out, stream);
  ROW_LIMITS("add_rmsnorm");
  if (N == 0) return SY_OK;
  SY_REQUIRE(x && weight && h_out, "add_rmsnorm: null pointer");
  row_kernel<false, false, 0, COUNTED><<<N, ROW_THREADS, 0, (hipStream_t)stream>>>(
      (const half_t*)x, (const half_t*)delta, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps, nullptr, 0, H,
      (half_t*)x_out, (half_t*)h_out, nullptr, nullptr, 0, front_core::Outputs{}, nullptr, nullptr, 0, count, nullptr);
  return sy_check_launch("add_rmsnorm");
}

extern "C" SY_API int sy_add_rmsnorm_logits(const void* x, const void* delta, const void* weight, float eps,
                                            const void* router, int E, int N, int H, void* x_out, void* h_out,
                                            void* logits, void* stream) {
  ROW_LIMITS("add_rmsnorm_logits");
  SY_REQUIRE(E >= 1 && E <= 1024, "add_rmsnorm_logits: 1 <= E <= 1024 (got %d)", E);
  if (N == 0) return SY_OK;
  SY_REQUIRE(x && weight && h_out && router && logits, "add_rmsnorm_logits: null pointer");
  row_kernel<false, true><<<N, 1024, (size_t)H * sizeof(half_t), (hipStream_t)stream>>>(
      (const half_t*)x, (const half_t*)delta, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps,
      (const half_t*)router, E, H, (half_t*)x_out, (half_t*)h_out, (half_t*)logits, nullptr, 0);
  return sy_check_launch("add_rmsnorm_logits");
}

extern "C" SY_API int sy_router_logits(const void* h, const void* router, int N, int H, int E, void* logits, void* stream) {
  ROW_LIMITS("router_logits");
  SY_REQUIRE(E >= 1 && E <= 1024, "router_logits: 1 <= E <= 1024 (got %d)", E);
  if (N == 0) return SY_OK;
  SY_REQUIRE(h && router && logits, "router_logits: null pointer");
  row_kernel<false, true><<<N, 1024, (size_t)H * sizeof(half_t), (hipStream_t)stream>>>(
      (const half_t*)h, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 0.f, (const half_t*)router, E, H, nullptr, nullptr,
      (half_t*)logits, nullptr, 0);
  return sy_check_launch("router_logits");
}

// The counters of the launches that end in front_core's tail. Every GPU the library runs on
// holds its own copy, all zero when the module is loaded and again after every launch. In host
// code the array's name is only a handle for hipGetSymbolAddress: launches take next_ticket()'s
// pointer.
static __device__ unsigned front_tickets[front_core::FRONT_TICKETS];

namespace {
constexpr int TICKET_DEVICES = 64;
std::mutex ticket_mutex;
unsigned* ticket_base[TICKET_DEVICES] = {nullptr};
unsigned ticket_next[TICKET_DEVICES][2] = {{0, 0}};

// The counter for the next launch on the current device. Slots are handed out in turn, the
// lower half of the pool to launches that run now and the upper half to launches that a stream
// capture records: a captured launch keeps its slot for every replay of its graph, so no launch
// outside a capture may ever be given it, and two captured launches share a slot only if half
// the pool's size in launches was captured between them.
int next_ticket(unsigned** out, hipStream_t stream) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= TICKET_DEVICES)
    return sy_fail(SY_ERR_LAUNCH, "router_route_sort: no current device below %d", TICKET_DEVICES);
  std::lock_guard<std::mutex> hold(ticket_mutex);
  if (!ticket_base[dev]) {
    void* p = nullptr;
    const hipError_t err = hipGetSymbolAddress(&p, HIP_SYMBOL(front_tickets));
    if (err != hipSuccess || !p)
      return sy_fail(SY_ERR_LAUNCH, "router_route_sort: hipGetSymbolAddress: %s", hipGetErrorString(err));
    ticket_base[dev] = static_cast<unsigned*>(p);
  }
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(stream, &status) != hipSuccess) {
    (void)hipGetLastError();
    status = hipStreamCaptureStatusNone;
  }
  constexpr unsigned HALF = front_core::FRONT_TICKETS / 2;
  const int captured = status == hipStreamCaptureStatusActive ? 1 : 0;
  *out = ticket_base[dev] + captured * HALF + ticket_next[dev][captured]++ % HALF;
  return SY_OK;
}

int front_outputs(const char* what, int N, int E, int k, int norm, int32_t* idx, void* w, int32_t* counts, int32_t* offsets,
                  int32_t* token, void* wsorted, int32_t* pos_of, hipStream_t stream, front_core::Outputs* out) {
  SY_REQUIRE(N <= front_core::TAIL_MAX_TOKENS, "%s: at most %d tokens (got %d)", what, front_core::TAIL_MAX_TOKENS, N);
  SY_REQUIRE(E <= 128 && k >= 1 && k <= front_core::TAIL_MAX_K && k <= E, "%s: at most 128 experts and top-8 (got E = %d, k = %d)",
             what, E, k);
  SY_REQUIRE(idx && w && counts && offsets && token && wsorted && pos_of, "%s: null pointer", what);
  unsigned* ticket = nullptr;
  const int rc = next_ticket(&ticket, stream);
  if (rc) return rc;
  int nbits = 0;
  while ((1 << nbits) < E) ++nbits;
  *out = front_core::Outputs{idx, (half_t*)w, counts, offsets, token, (half_t*)wsorted, pos_of, ticket, k, norm, nbits};
  return SY_OK;
}
}  // namespace

extern "C" SY_API int sy_router_route_sort(const void* h, const void* router, int N, int H, int E, int k, int norm, void* logits,
                                           int32_t* idx, void* w, int32_t* counts, int32_t* offsets, int32_t* token,
                                           void* wsorted, int32_t* pos_of, void* stream) {
  ROW_LIMITS("router_route_sort");
  SY_REQUIRE(E >= 1, "router_route_sort: E = %d", E);
  if (N == 0) return SY_OK;
  SY_REQUIRE(h && router && logits, "router_route_sort: null pointer");
  front_core::Outputs front;
  const int rc = front_outputs("router_route_sort", N, E, k, norm, idx, w, counts, offsets, token, wsorted, pos_of, (hipStream_t)stream, &front);
  if (rc) return rc;
  const size_t lds = (size_t)H * sizeof(half_t) + front_core::tail_lds_bytes(N, E, k);
  row_kernel<false, true, FRONT_SORT><<<N, 1024, lds, (hipStream_t)stream>>>(
      (const half_t*)h, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 0.f, (const half_t*)router, E, H, nullptr, nullptr,
      (half_t*)logits, nullptr, 0, front);
  return sy_check_launch("router_route_sort");
}

// The router GEMM and route for a few rows, one workgroup per row and no sort: what
// sy_router_route does for a decode step (front.hip hands such calls over).
int sy_router_route_rows(const void* h, const void* router, int N, int H, int E, int k, int norm, void* logits, int32_t* idx,
                         void* w, void* stream) {
  ROW_LIMITS("router_route");
  SY_REQUIRE(E >= 1 && E <= 128 && k >= 1 && k <= front_core::TAIL_MAX_K && k <= E,
             "router_route: at most 128 experts and top-8 (got E = %d, k = %d)", E, k);
  if (N == 0) return SY_OK;
  SY_REQUIRE(h && router && logits && idx && w, "router_route: null pointer");
  front_core::Outputs front{idx, (half_t*)w, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, k, norm, 0};
  const size_t lds = (size_t)H * sizeof(half_t) + sizeof(half_t) * ((size_t)(E + 7) / 8 * 8);
  row_kernel<false, true, FRONT_ROUTE><<<N, 1024, lds, (hipStream_t)stream>>>(
      (const half_t*)h, nullptr, nullptr, nullptr, nullptr, 0, nullptr, 0.f, (const half_t*)router, E, H, nullptr, nullptr,
      (half_t*)logits, nullptr, 0, front);
  return sy_check_launch("router_route");
}

int sy_logits_spread(const void* x, const void* delta, const void* weight, float eps, const void* router, int E, int N, int H,
                     void* x_out, void* h_out, void* logits, void* stream) {
  SY_REQUIRE(N >= 1 && N <= SPREAD_ROWS && E >= 1 && E <= 128 && H == SPREAD_H, "logits_spread: N = %d, E = %d, H = %d", N, E, H);
  SY_REQUIRE(x && router && logits && (!weight || (delta && x_out && h_out && x_out != x)), "logits_spread: null pointer, or x_out is x");
  const dim3 grid((unsigned)((E + SPREAD_WAVES - 1) / SPREAD_WAVES), (unsigned)N);
  void (*kern)(const half_t*, const half_t*, const half_t*, float, const half_t*, int, half_t*, half_t*, half_t*) =
      weight ? logits_spread_kernel<true> : logits_spread_kernel<false>;
  kern<<<grid, SPREAD_THREADS, 0, (hipStream_t)stream>>>((const half_t*)x, (const half_t*)delta, (const half_t*)weight, eps,
                                                         (const half_t*)router, E, (half_t*)x_out, (half_t*)h_out, (half_t*)logits);
  return sy_check_launch("logits_spread");
}

int sy_add_rmsnorm_route(const void* x, const void* delta, const void* weight, float eps, const void* router, int E, int N,
                         int H, int k, int norm, void* x_out, void* h_out, void* logits, int32_t* idx, void* w, void* stream) {
  ROW_LIMITS("add_rmsnorm_route");
  SY_REQUIRE(E >= 1 && E <= 128 && k >= 1 && k <= front_core::TAIL_MAX_K && k <= E,
             "add_rmsnorm_route: at most 128 experts and top-8 (got E = %d, k = %d)", E, k);
  if (N == 0) return SY_OK;
  SY_REQUIRE(x && weight && h_out && router && logits && idx && w, "add_rmsnorm_route: null pointer");
  front_core::Outputs front{idx, (half_t*)w, nullptr, nullptr, nullptr, nullptr, nullptr, nullptr, k, norm, 0};
  const size_t lds = (size_t)H * sizeof(half_t) + sizeof(half_t) * ((size_t)(E + 7) / 8 * 8);
  row_kernel<false, true, FRONT_ROUTE><<<N, 1024, lds, (hipStream_t)stream>>>(
      (const half_t*)x, (const half_t*)delta, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps,
      (const half_t*)router, E, H, (half_t*)x_out, (half_t*)h_out, (half_t*)logits, nullptr, 0, front);
  return sy_check_launch("add_rmsnorm_route");
}

extern "C" SY_API int sy_add_rmsnorm_route_sort(const void* x, const void* delta, const void* weight, float eps,
                                                const void* router, int E, int N, int H, int k, int norm, void* x_out,
                                                void* h_out, void* logits, int32_t* idx, void* w, int32_t* counts,
                                                int32_t* offsets, int32_t* token, void* wsorted, int32_t* pos_of,
                                                void* stream) {
  ROW_LIMITS("add_rmsnorm_route_sort");
  SY_REQUIRE(E >= 1, "add_rmsnorm_route_sort: E = %d", E);
  if (N == 0) return SY_OK;
  SY_REQUIRE(x && weight && h_out && router && logits, "add_rmsnorm_route_sort: null pointer");
  front_core::Outputs front;
  const int rc = front_outputs("add_rmsnorm_route_sort", N, E, k, norm, idx, w, counts, offsets, token, wsorted, pos_of, (hipStream_t)stream, &front);
  if (rc) return rc;
  const size_t lds = (size_t)H * sizeof(half_t) + front_core::tail_lds_bytes(N, E, k);
  row_kernel<false, true, FRONT_SORT><<<N, 1024, lds, (hipStream_t)stream>>>(
      (const half_t*)x, (const half_t*)delta, nullptr, nullptr, nullptr, 0, (const half_t*)weight, eps,
      (const half_t*)router, E, H, (half_t*)x_out, (half_t*)h_out, (half_t*)logits, nullptr, 0, front);
  return sy_check_launch("add_rmsnorm_route_sort");
}

int sy_combine_add_rmsnorm_twins(const void* y, const int32_t* pos_of, const int32_t* idx, const void* w, int k,
                                 const int32_t* twin, const int32_t* count, const void* x, const void* weight, float eps, int N,
                                 int H, void* x_out, void* h_out, void* stream) {
  ROW_LIMITS("combine_add_rmsnorm");
  SY_REQUIRE(k >= 1 && k <= ROW_MAX_K, "combine_add_rmsnorm: 1 <= k <= %d (got %d)", ROW_MAX_K, k);
  if (N == 0) return SY_OK;
  SY_REQUIRE(y && pos_of && idx && x && weight && h_out, "combine_add_rmsnorm: null pointer");
  SY_REQUIRE(!twin || !count, "combine_add_rmsnorm: rows that exist once have no twins");
  auto kern = twin ? row_kernel<true, false, 0, TWINNED>
              : count ? row_kernel<true, false, 0, COUNTED>
              : N <= FEW_ROWS && k >= FEW_MIN_K && k <= combine_core::AT_ONCE ? row_kernel<true, false, 0, OWN_ROWS, true> : row_kernel<true, false>;
  kern<<<N, ROW_THREADS, 0, (hipStream_t)stream>>>(
      (const half_t*)x, (const half_t*)w, (const half_t*)y, pos_of, idx, k, (const half_t*)weight, eps, nullptr, 0, H,
      (half_t*)x_out, (half_t*)h_out, nullptr, nullptr, 0, front_core::Outputs{}, twin, nullptr, 0, count, nullptr);
  return sy_check_launch("combine_add_rmsnorm");
}

extern "C" SY_API int sy_combine_add_rmsnorm(const void* y, const int32_t* pos_of, const int32_t* idx, const void* w, int k,
                                             const void* x, const void* weight, float eps, int N, int H, void* x_out,
                                             void* h_out, void* stream) {
  return sy_combine_add_rmsnorm_twins(y, pos_of, idx, w, k, nullptr, nullptr, x, weight, eps, N, H, x_out, h_out, stream);
}

// One workgroup per sequence of a batch of prompts. A row in front of its sequence's first real token
// holds the same numbers in every layer as any other such row with the same token: no query but its
// own sees it, and it sees itself alone, so nothing but its token's embedding ever reaches it. All
// of them are made twins of the first such row of the batch whose token they share; every
// other row is its own. What it saves is the experts' work for the padding, which is all on the same
// eight of them: 8 prompts of 256 to 512 tokens, gate/up 264 -> 217 us a layer, down 154 -> 126.
__global__ void __launch_bounds__(ROW_THREADS)
padding_twins_kernel(const int64_t* __restrict__ tokens, const uint8_t* __restrict__ real, int B, int T, int* __restrict__ twin) {
  __shared__ int s_row, s_first;
  const int b = blockIdx.x;
  if (threadIdx.x == 0) {
    s_row = B;     // the first sequence that starts with padding
    s_first = T;   // this sequence's first real token
  }
  __syncthreads();
  for (int r = threadIdx.x; r < B; r += ROW_THREADS)
    if (!real[(size_t)r * T]) {
      atomicMin(&s_row, r);
      break;
    }
  for (int t = threadIdx.x; t < T; t += ROW_THREADS)
    if (real[(size_t)b * T + t]) {
      atomicMin(&s_first, t);
      break;
    }
  __syncthreads();
  const int first = s_first, row = s_row < B ? s_row * T : 0;
  for (int t = threadIdx.x; t < T; t += ROW_THREADS) {
    const int at = b * T + t;
    twin[at] = t < first && tokens[at] == tokens[row] ? row : at;
  }
}

extern "C" SY_API int sy_padding_twins(const int64_t* tokens, const uint8_t* real, int B, int T, int32_t* twin, void* stream) {
  SY_REQUIRE(B >= 0 && T >= 1 && (long)B * T < (1l << 31), "padding_twins: B = %d, T = %d", B, T);
  if (B == 0) return SY_OK;
  SY_REQUIRE(tokens && real && twin, "padding_twins: null pointer");
  padding_twins_kernel<<<B, ROW_THREADS, 0, (hipStream_t)stream>>>(tokens, real, B, T, twin);
  return sy_check_launch("padding_twins");
}

static int qk_norm_check(const void* qkv, const void* q_norm, const void* k_norm, const void* cos_table, const void* sin_table,
                         int max_positions, const int64_t* positions, int B, int T, int heads, int kv_heads, int D, int capacity,
                         const void* q_out, const void* kcache, const void* vcache) {
  SY_REQUIRE(B >= 0 && T >= 1 && (long)B * T < (1l << 31) && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
             "qk_norm_rope_cache: B = %d, T = %d, heads = %d, kv_heads = %d", B, T, heads, kv_heads);
  SY_REQUIRE(D >= 16 && D % 16 == 0 && (long)heads * D <= 8 * ROW_THREADS * MAX_CHUNKS,
             "qk_norm_rope_cache: head_dim = %d must be a multiple of 16 and heads * head_dim at most %d", D,
             8 * ROW_THREADS * MAX_CHUNKS);
  SY_REQUIRE(capacity >= 1 && max_positions >= 1, "qk_norm_rope_cache: capacity = %d, max_positions = %d", capacity,
             max_positions);
  if (B == 0) return SY_OK;
  SY_REQUIRE(qkv && q_norm && k_norm && cos_table && sin_table && positions && q_out && kcache && vcache,
             "qk_norm_rope_cache: null pointer");
  return SY_OK;
}

extern "C" SY_API int sy_qk_norm_rope_cache(const void* qkv, const void* q_norm, const void* k_norm, float eps, float clip,
                                            const void* cos_table, const void* sin_table, int max_positions,
                                            const int64_t* positions, const int64_t* slot, int B, int T, int heads,
                                            int kv_heads, int D, int capacity, void* q_out, void* kcache, void* vcache,
                                            void* stream) {
  if (int rc = qk_norm_check(qkv, q_norm, k_norm, cos_table, sin_table, max_positions, positions, B, T, heads, kv_heads, D, capacity,
                             q_out, kcache, vcache))
    return rc;
  if (B == 0) return SY_OK;
  SY_REQUIRE(slot, "qk_norm_rope_cache: null pointer");
  const size_t lds = (size_t)(heads + kv_heads) * D * sizeof(half_t);
  qk_norm_rope_cache_kernel<false><<<B * T, ROW_THREADS, lds, (hipStream_t)stream>>>(
      (const half_t*)qkv, (const half_t*)q_norm, (const half_t*)k_norm, eps, clip, (const half_t*)cos_table,
      (const half_t*)sin_table, max_positions, positions, slot, T, heads, kv_heads, D, capacity, (half_t*)q_out,
      (half_t*)kcache, (half_t*)vcache);
  return sy_check_launch("qk_norm_rope_cache");
}

// The same for a prompt whose first token goes to position `first`, with the rows that exist (`place`, or null: all).
int sy_qk_norm_rope_prompt(const void* qkv, const void* q_norm, const void* k_norm, float eps, float clip, const void* cos_table,
                           const void* sin_table, int max_positions, const int64_t* positions, int first, const int32_t* place, int B,
                           int T, int heads, int kv_heads, int D, int capacity, void* q_out, void* kcache, void* vcache, void* stream) {
  if (int rc = qk_norm_check(qkv, q_norm, k_norm, cos_table, sin_table, max_positions, positions, B, T, heads, kv_heads, D, capacity,
                             q_out, kcache, vcache))
    return rc;
  if (B == 0) return SY_OK;
  if ((D == 64 || D == 128) && heads * D <= 8 * ROW_THREADS) {
    const auto kern = D == 128 ? qk_norm_rope_prompt_kernel<128> : qk_norm_rope_prompt_kernel<64>;
    kern<<<B * T, ROW_THREADS, 0, (hipStream_t)stream>>>(
        (const half_t*)qkv, (const half_t*)q_norm, (const half_t*)k_norm, eps, clip, (const half_t*)cos_table, (const half_t*)sin_table,
        max_positions, positions, first, place, T, heads * D, kv_heads * D, capacity, (half_t*)q_out, (half_t*)kcache, (half_t*)vcache);
    return sy_check_launch("qk_norm_rope_prompt");
  }
  const size_t lds = (size_t)(heads + kv_heads) * D * sizeof(half_t);
  qk_norm_rope_cache_kernel<true><<<B * T, ROW_THREADS, lds, (hipStream_t)stream>>>(
      (const half_t*)qkv, (const half_t*)q_norm, (const half_t*)k_norm, eps, clip, (const half_t*)cos_table,
      (const half_t*)sin_table, max_positions, positions, nullptr, T, heads, kv_heads, D, capacity, (half_t*)q_out,
      (half_t*)kcache, (half_t*)vcache, place, first);
  return sy_check_launch("qk_norm_rope_prompt");
}

// Whether the (sequence, head) pairs are too few to fill the chip with four wavefronts each: they then
// get 16, in one workgroup or, with room for their results, in four.
extern "C" SY_API int sy_decode_attention_shares(int B, int heads) { return (long)B * heads < 2l * sy_compute_units(); }

extern "C" SY_API int sy_decode_attention(const void* q, const void* kcache, const void* vcache, const uint8_t* real,
                                          const int64_t* slot, int B, int heads, int kv_heads, int D, int capacity,
                                          void* out, void* stream) {
  SY_REQUIRE(B >= 0 && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
             "decode_attention: B = %d, heads = %d, kv_heads = %d", B, heads, kv_heads);
  SY_REQUIRE(D == 64 || D == 128, "decode_attention: head_dim must be 64 or 128 (got %d)", D);
  SY_REQUIRE(capacity >= 1, "decode_attention: capacity = %d", capacity);
  if (B == 0) return SY_OK;
  SY_REQUIRE(q && kcache && vcache && real && slot && out, "decode_attention: null pointer");
  const long pairs = (long)B * heads;
  const int waves = sy_decode_attention_shares(B, heads) ? ATT_WAVES : 4;
  const size_t lds = (size_t)waves * (D + 2) * sizeof(float);
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)D);
  auto kern = D == 128 ? (waves == 4 ? decode_attention_kernel<16, false, 4, 4> : decode_attention_kernel<16, false, 16, 4>)
                       : (waves == 4 ? decode_attention_kernel<8, false, 4, 4> : decode_attention_kernel<8, false, 16, 4>);
  kern<<<(unsigned)pairs, waves * WAVE, lds, (hipStream_t)stream>>>((const half_t*)q, (const half_t*)kcache,
                                                                   (const half_t*)vcache, real, slot, heads, kv_heads,
                                                                   capacity, scale_log2e, (half_t*)out, NewToken{}, nullptr,
                                                                   nullptr);
  return sy_check_launch("decode_attention");
}

extern "C" SY_API int sy_decode_attention_qkv_split(const void* qkv, const void* q_norm, const void* k_norm, float eps,
                                                    float clip, const void* cos_table, const void* sin_table,
                                                    int max_positions, const int64_t* positions, const int64_t* slot,
                                                    uint8_t* real, int B, int heads, int kv_heads, int D, int capacity,
                                                    void* kcache, void* vcache, void* out, void* parts, void* tickets,
                                                    void* stream) {
  SY_REQUIRE(B >= 0 && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
             "decode_attention_qkv: B = %d, heads = %d, kv_heads = %d", B, heads, kv_heads);
  SY_REQUIRE(D == 64 || D == 128, "decode_attention_qkv: head_dim must be 64 or 128 (got %d)", D);
  SY_REQUIRE(capacity >= 1 && max_positions >= 1, "decode_attention_qkv: capacity = %d, max_positions = %d", capacity,
             max_positions);
  if (B == 0) return SY_OK;
  SY_REQUIRE(qkv && q_norm && k_norm && cos_table && sin_table && positions && slot && real && kcache && vcache && out,
             "decode_attention_qkv: null pointer");
  const long pairs = (long)B * heads;
  NewToken nt{(const half_t*)qkv, (const half_t*)q_norm, (const half_t*)k_norm, (const half_t*)cos_table,
              (const half_t*)sin_table, positions, (half_t*)kcache, (half_t*)vcache, real, eps, clip, max_positions};
  const float scale_log2e = 1.4426950408889634f / sqrtf((float)D);
  const bool few = sy_decode_attention_shares(B, heads), split = few && parts && tickets;
  const int waves = few && !split ? ATT_WAVES : 4, splits = split ? ATT_WAVES / waves : 1;
  const size_t lds = (size_t)waves * (D + 2) * sizeof(float);
  auto kern = D == 128 ? (split   ? decode_attention_kernel<16, true, 4, 4, ATT_WAVES>
                          : few ? decode_attention_kernel<16, true, ATT_WAVES, 4>
                                : decode_attention_kernel<16, true, 4, 4>)
                       : (split   ? decode_attention_kernel<8, true, 4, 4, ATT_WAVES>
                          : few ? decode_attention_kernel<8, true, ATT_WAVES, 4>
                                : decode_attention_kernel<8, true, 4, 4>);
  kern<<<(unsigned)(pairs * splits), waves * WAVE, lds, (hipStream_t)stream>>>(
      nullptr, (const half_t*)kcache, (const half_t*)vcache, real, slot, heads, kv_heads, capacity, scale_log2e, (half_t*)out,
      nt, (float*)parts, (unsigned*)tickets);
  return sy_check_launch("decode_attention_qkv");
}

extern "C" SY_API int sy_decode_attention_qkv(const void* qkv, const void* q_norm, const void* k_norm, float eps, float clip,
                                              const void* cos_table, const void* sin_table, int max_positions,
                                              const int64_t* positions, const int64_t* slot, uint8_t* real, int B,
                                              int heads, int kv_heads, int D, int capacity, void* kcache, void* vcache,
                                              void* out, void* stream) {
  return sy_decode_attention_qkv_split(qkv, q_norm, k_norm, eps, clip, cos_table, sin_table, max_positions, positions, slot,
                                       real, B, heads, kv_heads, D, capacity, kcache, vcache, out, nullptr, nullptr, stream);
}

extern "C" SY_API int sy_greedy_advance(const void* logits, int B, int V, int64_t* tok, int64_t* out, int out_stride,
                                        const int64_t* base_position, int64_t* next_position, int64_t* slot,
                                        void* stream) {
  SY_REQUIRE(B >= 0 && V >= 1 && out_stride >= 0, "greedy_advance: B = %d, V = %d, out_stride = %d", B, V, out_stride);
  if (B == 0) return SY_OK;
  SY_REQUIRE(logits && tok && out && base_position && next_position && slot, "greedy_advance: null pointer");
  greedy_advance_kernel<<<B, PICK_THREADS, 0, (hipStream_t)stream>>>((const half_t*)logits, V, tok, out, out_stride,
                                                                    base_position, next_position, slot);
  return sy_check_launch("greedy_advance");
}
