// prefill_attention: the prompt's attention. T new queries per sequence against the keys and
// values that the cache holds for the sequence, the new ones included (qk_norm_rope_cache has
// written them): query t sits at cache position first + t and sees the real positions up to its
// own; a padding query, which may see nothing, then takes its own value.
//
// Replaces the scores, mask, softmax and value product of the reference's forward pass
// (switchyard/model.py:78-84).
//
// One pass over the keys with a running softmax, on v_mfma_f32_32x32x16_f16. A wavefront owns 32
// queries, which stay in registers, and takes 64 keys at a time; everything is computed transposed
// (S^T = K Q^T, then O^T = V^T P^T), so that a lane always holds one query: the softmax's maximum
// and sum are reductions over the lane's own registers (one exchange with the lane 32 further on),
// rescaling the output is a multiply by a scalar of the lane, and the probabilities are already in
// the operand layout of the second product, because that product may visit the keys in any order
// as long as both operands agree: lane half h holds keys 8 j + 4 h .. + 3 of a block as the MFMA
// leaves them, and the values are read to match, four keys of one column at a time, by the LDS
// transpose read (ds_read_b64_tr_b16).
//
// Keys and values reach LDS by direct loads (no staging registers), a tile ahead of its use, in
// 16-byte chunks whose position inside a row is swizzled by the row: the key operand reads (16
// bytes of 32 rows) and the transposed value reads (32 bytes of 4 rows) both spread over the banks.
// A tile's mask is one 64-bit word, computed once per workgroup: tiles without a real key (left
// padding) are skipped whole, and only tiles that touch the diagonal or hold padding pay for
// masking.
//
// Precision. The first product's sums, the softmax and the output stay in fp32. For the second product
// probabilities are rounded to f16, relative to the maximum of the keys up to the end of their step: against
// that exact maximum the largest probability is 1 and has no rounding error. (A maximum rounded up to a
// whole power of two, with rescaling put off until it grew by 2^8, was faster - 13.8, 22.8 and 68 us
// at the sizes below - and had 9 to 37 % more error against 64 bits.) A step's length matters in the same
// way, less: 32 keys have 0.3 to 0.8 % more error than 16, 64 again 0.3 to 0.6 % more, and each takes 5 to 11 %
// less time. launch_steps below picks the longest that is no less precise than PyTorch's fused call, which
// this kernel replaces. With fewer key heads than query heads what it replaces held the probabilities in
// 32 bits, and so does WIDE: the sum of two f16 numbers, each with a product of its own, 2^14 times as
// large as above so that the second one stays normal. One prompt of 437 tokens, 16 heads over 4: 16.7 us.
//
// Measured (16 heads of 128, us a launch; before: PyTorch's fused call with a mask tensor, beside which
// the mask's conversion, a workspace fill and a transposed copy were launches of their own): one
// prompt of 437 tokens 15.8 (43 before), 8 of 512 24.6 (64), 3 of 2000 67.5 (643). At 3 x 2000 that is 730
// Tflop/s of the causal half; matrix pipes, LDS reads and the exponentials each need about a third
// of the time, and what is lost is their overlap. 128 queries per workgroup at every size: with the
// power-of-two rule 64 were never faster (437 tokens 14.6 against 14.2, 8 x 512 27.2 against 22.2, 3 x
// 2000 105 against 68) and 256 only at 16 x 128 (9.0 against 10.0; 3 x 2000 72 against 68).
#include "common.h"
#include "passes.h"

namespace {

constexpr int ATT_KEYS = 64;           // keys per tile
constexpr int ATT_QROWS = 32;          // queries per wavefront
constexpr int ATT_WAVES = 4;           // wavefronts per workgroup, of one head of one sequence
constexpr float ATT_NONE = -1.0e30f;   // running maximum before any key was seen

typedef int att_int4 __attribute__((ext_vector_type(4)));
typedef short att_short4 __attribute__((__vector_size__(8)));

__device__ __forceinline__ att_int4 att_descriptor(const void* base, unsigned bytes) {
  const uint64_t a = (uint64_t)base;
  att_int4 d;
  d[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)a);
  d[1] = __builtin_amdgcn_readfirstlane((int)((unsigned)(a >> 32) & 0xffffu));
  d[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  d[3] = 0x00020000;
  return d;
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 carries the LDS address
// 16 bytes per lane from buffer offset `voffset` (0 where it is past the end) to LDS address lds_addr + 16 * lane
__device__ __forceinline__ void att_load_to_lds(att_int4 rsrc, unsigned voffset, unsigned lds_addr) {
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, 0 offen lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voffset), "s"(rsrc)
      : "memory", "m0");
}
#pragma clang diagnostic pop

// The maximum (or sum) over the two lanes that hold a query.
__device__ __forceinline__ float other_half(float v) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  // r[0]: the lower half's value in every lane, r[1]: the upper half's
  return (threadIdx.x & 32) ? __uint_as_float(r[0]) : __uint_as_float(r[1]);
}

// STEP: keys per step of the running softmax (16, 32 or 64). WIDE: probabilities of 22 bits instead of 11.
template <int D, int STEP, bool WIDE>
__global__ void __launch_bounds__(ATT_WAVES * WAVE, 2)
prefill_attention_kernel(const half_t* __restrict__ q, const half_t* __restrict__ kcache, const half_t* __restrict__ vcache,
                         const uint8_t* __restrict__ real, int first, int T, int pairs, int heads, int kv_heads, int capacity,
                         float scale_log2e, half_t* __restrict__ out, const int* __restrict__ place) {
  constexpr int NW = ATT_WAVES;
  constexpr int ROW_BYTES = D * 2, CHUNKS = D / 8;        // 16-byte chunks of a row
  constexpr int TILE_BYTES = ATT_KEYS * ROW_BYTES;
  constexpr int QSTEPS = D / 16, DBLOCKS = D / 32;
  constexpr int ROWS_PER_LOAD = 1024 / ROW_BYTES;         // rows that one wavefront's load brings
  constexpr int LOADS = ATT_KEYS / ROWS_PER_LOAD / NW;    // loads of a tile per wavefront, of keys and of values each
  extern __shared__ __attribute__((aligned(1024))) char lds[];   // [2][keys | values], then the tiles' masks
  uint64_t* masks = reinterpret_cast<uint64_t*>(lds + 4 * TILE_BYTES);
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int l32 = lane & 31, half = lane >> 5;

  // Consecutive workgroups are different (sequence, head) pairs, so the query blocks of a pair land
  // on one XCD (workgroups are dealt to the 8 XCDs in turn; the pairs are a multiple of 8 in
  // earnest) and share its keys and values in that L2; the longest query blocks go first.
  const int pair = blockIdx.x % pairs, nblocks = gridDim.x / pairs, block = nblocks - 1 - blockIdx.x / pairs;
  const int b = pair / heads, h = pair - b * heads, kvh = h / (heads / kv_heads);
  const int t0 = block * (NW * ATT_QROWS), t_end = min(t0 + NW * ATT_QROWS, T);
  const int keys = first + t_end;                         // cache positions that the block's last query may see
  const int ntiles = (keys + ATT_KEYS - 1) / ATT_KEYS;
  const uint8_t* rl = real + (size_t)b * capacity;
  const size_t cache_at = ((size_t)b * kv_heads + kvh) * (size_t)capacity * D;

  // ---- the tiles' masks: bit j of tile i is whether position 64 i + j holds a real token
  for (int i = wave; i < ntiles; i += NW) {
    const int key = i * ATT_KEYS + lane;
    const uint64_t m = __ballot(key < keys && rl[key] != 0);
    if (lane == 0) masks[i] = m;
  }

  // ---- the wavefront's queries: lane (half, l32) holds 8 halves of query l32 per K step
  const int tw = t0 + wave * ATT_QROWS, t = tw + l32;     // this lane's query
  const int tq = min(t, T - 1);
  // with `place`, position r of the batch is row place[r], or (negative) one of the rows that exist once, ~place[r], of
  // which another position writes the output (prompt.hip)
  int row = b * T + tq;
  if (place) row = place[row];
  const bool own = row >= 0;
  row = own ? row : ~row;
  half8_t qf[QSTEPS];
  const half_t* qrow = q + (size_t)row * ((size_t)heads * D) + (size_t)h * D + half * 8;
#pragma unroll
  for (int s = 0; s < QSTEPS; ++s) qf[s] = *reinterpret_cast<const half8_t*>(qrow + 16 * s);
  const int slot = first + tq;
  const int wave_last = first + min(tw + ATT_QROWS, t_end) - 1;   // the last position any query of the wavefront sees
  const bool wave_live = tw < T;

  // ---- loader: a load brings 1 KB, ROWS_PER_LOAD whole rows; chunk c of row r goes to position c ^ swz(r)
  auto swz = [](int r) { return D == 128 ? (((r & 3) << 2) | ((r >> 2) & 3)) : (((r & 3) << 1) | ((r >> 2) & 1)); };
  const att_int4 krsrc = att_descriptor(kcache + cache_at, (unsigned)keys * ROW_BYTES);
  const att_int4 vrsrc = att_descriptor(vcache + cache_at, (unsigned)keys * ROW_BYTES);
  const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds;
  unsigned voff[LOADS];
#pragma unroll
  for (int i = 0; i < LOADS; ++i) {
    const int r = (i * NW + wave) * ROWS_PER_LOAD + lane / CHUNKS;
    voff[i] = (unsigned)(r * ROW_BYTES + ((lane % CHUNKS) ^ swz(r)) * 16);
  }
  auto issue = [&](int tile, int stage) {
    const unsigned base = (unsigned)tile * TILE_BYTES;
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      att_load_to_lds(krsrc, base + voff[i], lds_base + (unsigned)(2 * stage) * TILE_BYTES + (unsigned)(i * NW + wave) * 1024u);
#pragma unroll
    for (int i = 0; i < LOADS; ++i)
      att_load_to_lds(vrsrc, base + voff[i], lds_base + (unsigned)(2 * stage + 1) * TILE_BYTES + (unsigned)(i * NW + wave) * 1024u);
  };
  __syncthreads();
  auto next_tile = [&](int i) {   // the first tile from i on that holds a real key
    while (i < ntiles && masks[i] == 0) ++i;
    return __builtin_amdgcn_readfirstlane(i);
  };

  float16_t o[DBLOCKS];
#pragma unroll
  for (int d = 0; d < DBLOCKS; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.f;
  float m = ATT_NONE, l = 0.f;   // in units of the exponent (score * scale * log2 e)

  // operand addresses inside a tile. Keys: row l32 (+ 32 for the second block), chunk 2 s + half.
  unsigned kread[QSTEPS];
#pragma unroll
  for (int s = 0; s < QSTEPS; ++s) kread[s] = (unsigned)(l32 * ROW_BYTES + (((2 * s + half) ^ swz(l32)) * 16));
  // Values: a group of 16 lanes reads 4 keys x 16 columns; lane i of it supplies the address of key
  // i / 4, columns 4 (i % 4) .. + 3, and receives the 4 keys of column i
  const int vkey = 4 * half + ((lane & 15) >> 2), vcol = ((lane >> 4) & 1) * 16 + (lane & 3) * 4;
  unsigned vread[DBLOCKS];   // the swizzle of a row depends on the row modulo 16, of which keys + 8 changes one bit
  unsigned vread8[DBLOCKS];
#pragma unroll
  for (int d = 0; d < DBLOCKS; ++d) {
    const int c = (32 * d + vcol) >> 3, in = (vcol & 7) * 2;
    vread[d] = (unsigned)(vkey * ROW_BYTES + ((c ^ swz(vkey)) * 16) + in);
    vread8[d] = (unsigned)((vkey + 8) * ROW_BYTES + ((c ^ swz(vkey + 8)) * 16) + in);
  }

  int tile = next_tile(0), stage = 0;
  if (tile < ntiles) issue(tile, 0);
  while (tile < ntiles) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();   // the tile has landed for everybody, and everybody is done with the other buffer
    const int after = next_tile(tile + 1);
    if (after < ntiles) issue(after, stage ^ 1);
    const int key0 = tile * ATT_KEYS;
    if (wave_live && key0 <= wave_last) {
      const char* kt = lds + 2 * stage * TILE_BYTES;
      float16_t s[2];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[kb][r] = 0.f;
#pragma unroll
        for (int st = 0; st < QSTEPS; ++st) {
          const half8_t kf = *reinterpret_cast<const half8_t*>(kt + kb * 32 * ROW_BYTES + kread[st]);
          s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[st], s[kb], 0, 0, 0);
        }
      }
      // register r of block kb: key 32 kb + 8 (r / 4) + 4 half + r % 4
      const uint64_t tm = masks[tile];
      if (tm != ~0ull || key0 + ATT_KEYS - 1 > first + tw) {   // padding, or the diagonal (the same in the whole wavefront)
        const int n = slot - key0;
        uint64_t seen = n >= 63 ? ~0ull : n < 0 ? 0ull : (2ull << n) - 1;
        seen = (seen & tm) >> (4 * half);
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const unsigned word = kb ? (unsigned)(seen >> 32) : (unsigned)seen;
            s[kb][r] = (word >> (8 * (r / 4) + r % 4)) & 1 ? s[kb][r] : -INFINITY;
          }
      }
      // one step of the running softmax over registers r0 .. r1 - 1 of blocks k0 .. k1 - 1
      half8_t p[2][2], rest[2][2];
      auto softmax = [&](int k0, int k1, int r0, int r1) {
        float mx = -INFINITY;
#pragma unroll
        for (int kb = k0; kb < k1; ++kb)
#pragma unroll
          for (int r = r0; r < r1; ++r) mx = fmaxf(mx, s[kb][r]);
        mx = fmaxf(mx, other_half(mx)) * scale_log2e;
        if (__any(mx > m)) {
          const float mn = fmaxf(m, mx);
          const float alpha = __builtin_amdgcn_exp2f(m - mn);
          m = mn;
          l *= alpha;
#pragma unroll
          for (int d = 0; d < DBLOCKS; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
        }
#pragma unroll
        for (int kb = k0; kb < k1; ++kb)
#pragma unroll
          for (int r = r0; r < r1; ++r) {
            const float e = __builtin_amdgcn_exp2f(s[kb][r] * scale_log2e - (m - (WIDE ? 14.f : 0.f)));
            l += e;
            const half_t rounded = (half_t)e;
            p[kb][r >> 3][r & 7] = rounded;
            if (WIDE) rest[kb][r >> 3][r & 7] = (half_t)(e - (float)rounded);
          }
      };
      const unsigned vt = lds_base + (unsigned)(2 * stage + 1) * TILE_BYTES;
      auto values = [&](int kb, int st) {   // 16 keys of block kb
#pragma unroll
        for (int d = 0; d < DBLOCKS; ++d) {
          const unsigned at = vt + (unsigned)(kb * 32 + st * 16) * ROW_BYTES;
          typedef __attribute__((address_space(3))) att_short4 lds_short4;
          const half4_t lo = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(size_t)(at + vread[d])));
          const half4_t hi = __builtin_bit_cast(half4_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(size_t)(at + vread8[d])));
          const half8_t vf = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, p[kb][st], o[d], 0, 0, 0);
          if (WIDE) o[d] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, rest[kb][st], o[d], 0, 0, 0);
        }
      };
      if (STEP == 64) softmax(0, 2, 0, 16);
#pragma unroll
      for (int kb = 0; kb < 2; ++kb) {
        if (STEP == 32) softmax(kb, kb + 1, 0, 16);
#pragma unroll
        for (int st = 0; st < 2; ++st) {
          if (STEP == 16) softmax(kb, kb + 1, 8 * st, 8 * st + 8);
          values(kb, st);
        }
      }
    }
    tile = after;
    stage ^= 1;
  }

  // ---- the lane holds columns 32 d + 8 g + 4 half + 0..3 of its query; after swapping with the lane 32
  // further on it holds 8 consecutive ones (group g of the lower half's two, g + 1 of the upper's)
  l += other_half(l);
  // A query that saw no key takes its own value (a padding query; a real one sees itself). A sum of zero alone
  // does not say so: scores of minus infinity leave it too, and their softmax is NaN.
  bool alone = l == 0.f;
  for (int i = 0, last = slot / ATT_KEYS; alone && i <= last; ++i)
    alone = (i < last ? masks[i] : masks[i] & ((2ull << (slot - last * ATT_KEYS)) - 1)) == 0;
  const float inv = 1.f / l;
  if (!wave_live) return;
  half_t* orow = out + (size_t)row * ((size_t)heads * D) + (size_t)h * D;
  const half_t* own_value = vcache + cache_at + (size_t)slot * D;
#pragma unroll
  for (int d = 0; d < DBLOCKS; ++d)
#pragma unroll
    for (int g = 0; g < 4; g += 2) {
      typedef unsigned u2_t __attribute__((ext_vector_type(2)));
      typedef unsigned u4_t __attribute__((ext_vector_type(4)));
      half4_t v0, v1;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        v0[r] = (half_t)(o[d][4 * g + r] * inv);
        v1[r] = (half_t)(o[d][4 * (g + 1) + r] * inv);
      }
      const u2_t a = __builtin_bit_cast(u2_t, v0), c = __builtin_bit_cast(u2_t, v1);
      const auto x0 = __builtin_amdgcn_permlane32_swap(a[0], c[0], false, false);
      const auto x1 = __builtin_amdgcn_permlane32_swap(a[1], c[1], false, false);
      const u4_t w = {x0[0], x1[0], x0[1], x1[1]};
      half8_t v = __builtin_bit_cast(half8_t, w);
      const int col = 32 * d + 8 * (g + half);
      if (alone) v = *reinterpret_cast<const half8_t*>(own_value + col);
      if (t < T && own) *reinterpret_cast<half8_t*>(orow + col) = v;
    }
}

// LDS of a launch over `positions` positions: two stages of keys and values, and a mask per tile
size_t att_lds_bytes(int positions, int D) {
  return (size_t)4 * ATT_KEYS * D * 2 + sizeof(uint64_t) * (((size_t)positions + ATT_KEYS - 1) / ATT_KEYS);
}

template <int D, int STEP, bool WIDE>
int launch_prefill_attention(const half_t* q, const half_t* kc, const half_t* vc, const uint8_t* real, int first, int B, int T,
                             int heads, int kv_heads, int capacity, const int* place, half_t* out, hipStream_t st) {
  const int pairs = B * heads, rows = ATT_WAVES * ATT_QROWS, nblocks = (T + rows - 1) / rows;
  const size_t lds = att_lds_bytes(first + T, D);
  const auto kern = prefill_attention_kernel<D, STEP, WIDE>;
  if (lds > 48 * 1024 && hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return sy_fail(SY_ERR_LAUNCH, "prefill_attention: cannot reserve %zu bytes of LDS", lds);
  kern<<<(unsigned)(pairs * nblocks), ATT_WAVES * WAVE, lds, st>>>(q, kc, vc, real, first, T, pairs, heads, kv_heads, capacity,
                                                          1.4426950408889634f / sqrtf((float)D), out, place);
  return sy_check_launch("prefill_attention");
}

// PyTorch's fused call (its results were compared with each step's, over queries and positions from 1 to
// 3000 on this card) takes 16 keys at a time up to 256 positions and, for 33 to 64 queries, up to 1024; 32 at
// 257 to 1024 queries and as many positions, and for heads of 64 up to 2048 queries; 64 or more otherwise.
// So a query's last bits may differ with the number of tokens that share its call: the step changes behind 256
// and 1024 positions and behind 64 queries. What a step rounds by is the exact maximum so far at every length,
// and a probability below 2^-14 of it is rounded to a multiple of 2^-24, as f16 is. 1 in 600 to 1 in 7000
// results differ from the call's where the steps are alike, by their last place, and the error
// against 64 bits is the call's to four digits. (With a mask the call is off by up to 1.0 in some rows at 1100
// and 1500 positions, heads of 128; this kernel is not.)
template <int D>
int launch_steps(const half_t* q, const half_t* kc, const half_t* vc, const uint8_t* real, int first, int B, int T, int heads,
                 int kv_heads, int capacity, const int* place, half_t* out, hipStream_t st) {
  const int positions = first + T;
#define SY_PREFILL(STEP_, WIDE_) \
  launch_prefill_attention<D, STEP_, WIDE_>(q, kc, vc, real, first, B, T, heads, kv_heads, capacity, place, out, st)
  if (kv_heads != heads) return SY_PREFILL(64, true);
  if (positions <= 256 || (T <= 64 && positions <= 1024)) return SY_PREFILL(16, false);
  if constexpr (D == 128) {
    if (positions > 1024) return SY_PREFILL(64, false);
  }
  return SY_PREFILL(32, false);
#undef SY_PREFILL
}

}  // namespace

extern "C" SY_API int sy_prefill_attention_takes(int positions, int capacity, int D) {
  return (D == 64 || D == 128) && positions >= 1 && positions <= capacity && (long)capacity * D * 2 < (1l << 31) &&
         att_lds_bytes(positions, D) <= 160 * 1024;
}

extern "C" SY_API int sy_prefill_attention(const void* q, const void* kcache, const void* vcache, const uint8_t* real, int first,
                                           int B, int T, int heads, int kv_heads, int D, int capacity, void* out, void* stream) {
  return sy_prefill_attention_rows(q, kcache, vcache, real, first, B, T, heads, kv_heads, D, capacity, nullptr, out, stream);
}

int sy_prefill_attention_rows(const void* q, const void* kcache, const void* vcache, const uint8_t* real, int first, int B, int T,
                              int heads, int kv_heads, int D, int capacity, const int32_t* place, void* out, void* stream) {
  SY_REQUIRE(B >= 0 && T >= 1 && heads >= 1 && kv_heads >= 1 && heads % kv_heads == 0,
             "prefill_attention: B = %d, T = %d, heads = %d, kv_heads = %d", B, T, heads, kv_heads);
  SY_REQUIRE(D == 64 || D == 128, "prefill_attention: head_dim must be 64 or 128 (got %d)", D);
  SY_REQUIRE(first >= 0 && capacity >= 1 && (long)first + T <= capacity, "prefill_attention: positions %d .. %ld of %d", first,
             (long)first + T - 1, capacity);
  SY_REQUIRE(sy_prefill_attention_takes(first + T, capacity, D), "prefill_attention: %d positions of %d are too many", first + T,
             capacity);
  if (B == 0) return SY_OK;
  SY_REQUIRE((long)B * heads * ((T + 127) / 128) < (1l << 31), "prefill_attention: too many queries (B = %d, heads = %d, T = %d)", B, heads, T);
  SY_REQUIRE(q && kcache && vcache && real && out, "prefill_attention: null pointer");
  const half_t *qh = (const half_t*)q, *kc = (const half_t*)kcache, *vc = (const half_t*)vcache;
  half_t* o = (half_t*)out;
  hipStream_t st = (hipStream_t)stream;
  return D == 128 ? launch_steps<128>(qh, kc, vc, real, first, B, T, heads, kv_heads, capacity, place, o, st)
                  : launch_steps<64>(qh, kc, vc, real, first, B, T, heads, kv_heads, capacity, place, o, st);
}
