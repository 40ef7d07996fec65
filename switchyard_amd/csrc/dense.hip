// dense_tiles: x [rows, K] @ weight [Nout, K]^T for a few dozen rows: the projections around the MoE layer where a
// step has more sequences than the weight stream (gemv.hip) is for, and of short prompts.
//
// What bounds such a product is the latency of a launch's first loads, weights out of HBM among them, and the barriers of its
// K loop: the tiles get 20 to 25 bytes a clock and compute unit of the 55 to 57 that loads straight to LDS bring from L2 in a
// loop of nothing else. The MFMAs need a fraction of the time. So the tile is chosen to put one tile on each compute unit with as few rows and columns together as
// possible (pick_tile below), and the whole of LDS is a ring of K slices: rows and weight rows in slices of 64
// (128 bytes: whole lines), up to fourteen deep, by buffer loads that write LDS directly, XOR-swizzled by row so that
// the operand reads spread over the banks, two slices to a barrier. The waits for the loads are counted by hand: the
// compiler is not told about them. Weights out of HBM, us a launch, against the library's GEMM: [6144, 2048] 17 to 32
// rows 8.8 to 9.1 (11.8), 33 to 64 rows 11.4 to 11.7 (12.5); [2048, 2048] up to 64 rows 6.7 to 6.9 (10.7 to 11.0), 128 rows
// 8.3 (11.0), 256 rows 11.2 (11.7). Larger tiles gain nothing: 64 x 64 takes 14 to 17 us, 128 x 96 16 to 24 where the
// library takes 13.5 at 100 rows and 22.8 at 437.
//
// K is summed in order with one accumulator per output on v_mfma_f32_16x16x32_f16 (the bits of sy_grouped_gemm with
// one expert), except in the smallest tile, where four accumulators take every fourth step of 32. The library's GEMM gives
// the same bits for 17 to 64 rows of [6144, 2048] and 17 to 256 of [2048, 2048]; for other weights (K = 512, 1024, 3072) about
// 0.15 % of the results differ at some numbers of rows, by their last place.
//
// Replaces F.linear in the reference's attention block (switchyard/model.py:61-76,84).
#include "common.h"
#include "passes.h"

namespace {

constexpr int DT_WAVES = 8, DT_THREADS = DT_WAVES * WAVE;
constexpr int DT_BK = 64, DT_ROW_BYTES = DT_BK * 2;
constexpr int DT_XCDS = 8;
constexpr unsigned DT_OUT_OF_RANGE = 0x80000000u;

typedef int dt_int4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ dt_int4 dt_descriptor(const void* base, unsigned bytes) {
  const uint64_t a = (uint64_t)base;
  dt_int4 d;
  d[0] = __builtin_amdgcn_readfirstlane((int)(unsigned)a);
  d[1] = __builtin_amdgcn_readfirstlane((int)((unsigned)(a >> 32) & 0xffffu));
  d[2] = __builtin_amdgcn_readfirstlane((int)bytes);
  d[3] = 0x00020000;
  return d;
}

#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"   // m0 carries the LDS address
// 16 bytes per lane from buffer offset voffset + soffset to LDS address lds_addr + 16 * lane; only voffset is checked
// against the size of the buffer
__device__ __forceinline__ void dt_load_to_lds(dt_int4 rsrc, unsigned voffset, unsigned soffset, unsigned lds_addr) {
#pragma unroll
  for (int c = 0; c < 4; ++c) rsrc[c] = __builtin_amdgcn_readfirstlane(rsrc[c]);
  asm volatile(
      "s_mov_b32 m0, %0\n\t"
      "s_nop 0\n\t"
      "buffer_load_dwordx4 %1, %2, %3 offen lds"
      :
      : "s"(__builtin_amdgcn_readfirstlane(lds_addr)), "v"(voffset), "s"(rsrc), "s"(__builtin_amdgcn_readfirstlane(soffset))
      : "memory", "m0");
}
#pragma clang diagnostic pop

constexpr int dt_slice_bytes(int BR, int BC) { return (BR + BC) * DT_ROW_BYTES; }
constexpr int DT_PAIR = 2;   // slices to a barrier
constexpr int dt_loads(int BR, int BC) { return ((BR + BC) / 8 + DT_WAVES - 1) / DT_WAVES; }   // of a slice, per wavefront
// slices in the ring: what fits 152 KB of LDS, up to 14, in pairs
constexpr int dt_stages(int BR, int BC) {
  const int fit = 152 * 1024 / dt_slice_bytes(BR, BC) / DT_PAIR * DT_PAIR;
  return fit > 14 ? 14 : fit;
}

// One workgroup: BR rows (fewer where the tiles are lower or the rows end) x BC weight rows, all of K.
template <int BR, int BC>
__global__ void __launch_bounds__(DT_THREADS)
dense_tiles_kernel(const half_t* __restrict__ A, const half_t* __restrict__ B, int M, int Nout, int K, int height,
                   half_t* __restrict__ C) {
  constexpr int P = DT_PAIR, S = dt_stages(BR, BC), SLICE = dt_slice_bytes(BR, BC);
  constexpr int NG = (BR + BC) / 8;                                   // loads of a slice: 8 rows each
  constexpr int EACH = dt_loads(BR, BC);                              // of a wavefront, one fewer from wavefront NG % 8 on
  constexpr int NBR = BR / 16, NBC = BC / 16;                         // blocks of 16 rows, of 16 weight rows
  // A tile of fewer blocks than wavefronts: four wavefronts to a block, each with every fourth K step (32), and their
  // sums added in order at the end.
  constexpr int KS = NBR * NBC * 4 == DT_WAVES ? 4 : 1;
  constexpr int WC = KS > 1 ? NBC : NBC % 4 == 0 ? 4 : NBC % 2 == 0 ? 2 : 1, WR = DT_WAVES / KS / WC;
  constexpr int RBW = (NBR + WR - 1) / WR, CBW = NBC / WC;            // blocks of a wavefront
  static_assert(S >= 3 * P && (S - P) * EACH < 64, "loads in flight that the wait can count");
  extern __shared__ __attribute__((aligned(1024))) char lds[];
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;

  // Consecutive tiles share weight rows and go to one XCD (workgroups are dealt round-robin to the XCDs), so that they
  // meet in its L2.
  const int row_tiles = (M + height - 1) / height, per_xcd = gridDim.x / DT_XCDS;
  const int place = (int)(blockIdx.x % DT_XCDS) * per_xcd + (int)(blockIdx.x / DT_XCDS);
  const int col = place / row_tiles, n0 = col * BC, row0 = (place - col * row_tiles) * height;
  if (n0 >= Nout) return;
  const int nrows = min(height, M - row0);

  // ---- loader: group g of a slice is 8 rows (of A, then of B); a lane fetches the chunk that its place holds
  const dt_int4 arsrc = dt_descriptor(A, (unsigned)((size_t)M * K * 2)), brsrc = dt_descriptor(B, (unsigned)((size_t)Nout * K * 2));
  const unsigned lds_base = (unsigned)(size_t)(__attribute__((address_space(3))) char*)lds;
  unsigned voff[EACH];
#pragma unroll
  for (int i = 0; i < EACH; ++i) {
    const int r = (i * DT_WAVES + wave) * 8 + (lane >> 3);
    const unsigned chunk = (unsigned)((lane & 7) ^ ((r >> 1) & 7)) * 16u;
    voff[i] = DT_OUT_OF_RANGE;
    if (r < BR) {
      if (r < nrows) voff[i] = (unsigned)(row0 + r) * (unsigned)K * 2u + chunk;
    } else if (r < BR + BC && n0 + r - BR < Nout) {
      voff[i] = (unsigned)(n0 + r - BR) * (unsigned)K * 2u + chunk;
    }
  }
  const int nk = K / DT_BK;
  // slices past the end are asked for too, out of range: they keep the count of loads in flight the same and
  // bring nothing
  auto issue = [&](int s, int stage) {
#pragma unroll
    for (int i = 0; i < EACH; ++i) {
      const int g = i * DT_WAVES + wave;
      if (i < EACH - 1 || NG % DT_WAVES == 0 || g < NG)
        dt_load_to_lds(g < BR / 8 ? arsrc : brsrc, s < nk ? voff[i] : DT_OUT_OF_RANGE, (unsigned)(s < nk ? s : 0) * DT_ROW_BYTES,
                       lds_base + (unsigned)stage * SLICE + (unsigned)g * 1024u);
    }
  };
  const bool full = NG % DT_WAVES == 0 || wave < NG % DT_WAVES;

  const int ks = wave / (WR * WC), wr = wave / WC % WR, wc = wave % WC, l16 = lane & 15, lg = lane >> 4;
  float4_t acc[RBW][CBW];
#pragma unroll
  for (int i = 0; i < RBW; ++i)
#pragma unroll
    for (int j = 0; j < CBW; ++j) acc[i][j] = float4_t{0.f, 0.f, 0.f, 0.f};
  unsigned aread[2], bread[2];   // of K step 0 and 1 of a slice; a block of 16 rows further on is 2 KB
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    const unsigned chunk = (unsigned)((4 * s + lg) ^ (l16 >> 1)) * 16u;
    aread[s] = (unsigned)(wr * 16 + l16) * DT_ROW_BYTES + chunk;
    bread[s] = (unsigned)(BR + wc * CBW * 16 + l16) * DT_ROW_BYTES + chunk;
  }

  for (int s = 0; s < S - P; ++s) issue(s, s);
  int at = 0, fill = S - P;   // the buffer of slice s, and the one the next load fills
  for (int s = 0; s < nk; s += P) {
    // this wavefront's loads of slices s .. s + P - 1 have landed when only those of the S - 2 P after them are in flight
    if (full) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2 * P) * EACH) : "memory");
    else asm volatile("s_waitcnt vmcnt(%0)" ::"n"((S - 2 * P) * (EACH - 1)) : "memory");
    __syncthreads();   // everybody's have, and everybody has read the P slices before, whose buffers the next loads fill
#pragma unroll
    for (int p = 0; p < P; ++p) issue(s + S - P + p, fill + p);
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const char* stage = lds + (at + p) * SLICE;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (KS > 1 && 2 * p + st != ks) continue;   // the same in the whole wavefront
        half8_t wf[CBW];
#pragma unroll
        for (int j = 0; j < CBW; ++j) wf[j] = *reinterpret_cast<const half8_t*>(stage + bread[st] + j * 16 * DT_ROW_BYTES);
#pragma unroll
        for (int i = 0; i < RBW; ++i) {
          if ((wr + i * WR) * 16 >= nrows) continue;   // the same in the whole wavefront
          const half8_t xf = *reinterpret_cast<const half8_t*>(stage + aread[st] + i * WR * 16 * DT_ROW_BYTES);
#pragma unroll
          for (int j = 0; j < CBW; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(wf[j], xf, acc[i][j], 0, 0, 0);
        }
      }
    }
    fill = at;   // pairs never wrap inside the ring
    at = at + P == S ? 0 : at + P;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // no load may land in LDS after this workgroup has given it back

  if (KS > 1) {
    float4_t* parts = reinterpret_cast<float4_t*>(lds);   // nothing of the slices is needed any more
    __syncthreads();
    if (ks > 0) parts[wave * WAVE + lane] = acc[0][0];
    __syncthreads();
    if (ks > 0) return;
#pragma unroll
    for (int u = 1; u < KS; ++u) acc[0][0] += parts[(u * WR * WC + wave) * WAVE + lane];
  }

  // ---- lane (lg, l16) holds columns 4 lg .. + 3 of row l16 of each block
#pragma unroll
  for (int i = 0; i < RBW; ++i) {
    const int r = (wr + i * WR) * 16 + l16;
    if (r >= nrows) continue;
#pragma unroll
    for (int j = 0; j < CBW; ++j) {
      const int c = n0 + (wc * CBW + j) * 16 + 4 * lg;
      const half4_t o = __builtin_convertvector(acc[i][j], half4_t);
      half_t* dst = C + (size_t)(row0 + r) * Nout + c;
      if (Nout % 4 == 0) {
        if (c < Nout) *reinterpret_cast<half4_t*>(dst) = o;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e)
          if (c + e < Nout) dst[e] = o[e];
      }
    }
  }
}

struct Tile {
  int br, bc;
  void (*kern)(const half_t*, const half_t*, int, int, int, int, half_t*);
};
const Tile TILES[] = {{32, 16, dense_tiles_kernel<32, 16>}, {32, 32, dense_tiles_kernel<32, 32>}, {64, 32, dense_tiles_kernel<64, 32>}};

// The smallest tile that makes no more tiles than compute units, or null: a second round of tiles costs as much as the first
// (64 rows by 2048 columns in tiles of 32 x 16: 6.9 us, 6144 columns in 768 of them: 18.2).
const Tile* pick_tile(int rows, int Nout) {
  for (const Tile& t : TILES)
    if ((long)((rows + t.br - 1) / t.br) * ((Nout + t.bc - 1) / t.bc) <= sy_compute_units()) return &t;
  return nullptr;
}

}  // namespace

extern "C" SY_API int sy_dense_tiles_takes(int rows, int Nout, int K) {
  return rows >= 1 && Nout >= 1 && K >= 128 && K % 128 == 0 && (long)Nout * K * 2 < (1l << 31) && (long)rows * K * 2 < (1l << 31) &&
         pick_tile(rows, Nout) != nullptr;
}

extern "C" SY_API int sy_dense_tiles(const void* x, const void* weight, int rows, int Nout, int K, void* out, void* stream) {
  SY_REQUIRE(rows >= 0, "dense_tiles: rows = %d", rows);
  if (rows == 0) return SY_OK;
  SY_REQUIRE(sy_dense_tiles_takes(rows, Nout, K), "dense_tiles: rows = %d, Nout = %d, K = %d: K a multiple of 128, operands under 2 GiB, "
             "no more tiles than compute units", rows, Nout, K);
  SY_REQUIRE(x && weight && out, "dense_tiles: null pointer");
  const Tile& t = *pick_tile(rows, Nout);
  const int row_tiles = (rows + t.br - 1) / t.br, height = ((rows + row_tiles - 1) / row_tiles + 15) / 16 * 16;
  const int tiles = (rows + height - 1) / height * ((Nout + t.bc - 1) / t.bc);
  const size_t lds = (size_t)dt_stages(t.br, t.bc) * dt_slice_bytes(t.br, t.bc);
  if (hipFuncSetAttribute((const void*)t.kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds) != hipSuccess)
    return sy_fail(SY_ERR_LAUNCH, "dense_tiles: cannot reserve %zu bytes of LDS", lds);
  t.kern<<<(tiles + DT_XCDS - 1) / DT_XCDS * DT_XCDS, DT_THREADS, lds, (hipStream_t)stream>>>((const half_t*)x, (const half_t*)weight, rows,
                                                                                         Nout, K, height, (half_t*)out);
  return sy_check_launch("dense_tiles");
}
