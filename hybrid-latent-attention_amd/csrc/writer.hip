// Writer of the S6 terminal block: the per-loop candidate projection, its register accumulation and the
// committed-row store (hla/latent/register.py:45-61, hla/vllm_latent/s6_layer.py:124-147,
// hla/vllm_latent/ouro_latent.py:127-129), as one kernel.
//
//   u[t, n]   = bf16( sum_k h[t, k] * W[n, k] )                 (nn.Linear, bf16 output)
//   reg[t, n] = prev ? bf16(prev[t, n] + u[t, n]) : u[t, n]      (write_step: previous + update)
//   commit:     cache row slots[t] <- [RoPE_lat(reg[t, :w]) | reg[t, w:]]
//
// W is the nn.Linear weight [2w, hidden] (rows = output columns), so both MFMA operands are k-contiguous and come
// straight from global memory with 16-byte loads: lane l takes A = h[row l%16][k + 8(l/16) ..] and B = W[column
// l%16][k + 8(l/16) ..]. A workgroup computes 16 or 64 tokens x 16 output columns; its eight waves (four when hidden
// is not a multiple of 1024) take one slice of the hidden dimension each, with two batches of four
// v_mfma_f32_16x16x32_bf16 k steps in flight, so every operand byte of a decode step's workgroup is requested at once
// (the kernel is latency-bound at decode sizes); the per-wave fp32 partials are summed in LDS in a fixed order. A
// key-half tile holds 8 rotation pairs (columns c and c + w/2), so each thread of the epilogue has both partners of a
// RoPE pair; value-half tiles hold 16 consecutive columns. More than 128 tokens take the tiled kernel below.
#include "common.h"

namespace hla {
namespace {

struct WriterParams {
  const uint16_t* h;
  int64_t h_st;
  const uint16_t* w;
  int64_t w_st;
  const uint16_t* prev;
  int64_t prev_st;
  uint16_t* reg;
  int64_t reg_st;
  const int64_t* slots;
  const int64_t* pos;
  const uint16_t* table;
  int table_rows;
  int64_t table_stride;
  uint16_t* cache;
  int64_t page_stride, row_stride;
  int block;
  int64_t num_slots;
  int T, K, width;
};

// Output column of MFMA column j (0..15) of column tile x.
__device__ __forceinline__ int writer_col(int x, int j, int width) {
  const int key_tiles = width / 16;
  return x < key_tiles ? 8 * x + (j & 7) + (j >> 3) * (width / 2) : width + 16 * (x - key_tiles) + j;
}

template <int WAVES, int MT>
__global__ __launch_bounds__(WAVES * 64) void writer_kernel(WriterParams a) {
  __shared__ float red[WAVES][16 * MT][17];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int l16 = lane & 15, g = lane >> 4;
  const int x = blockIdx.x, t0 = blockIdx.y * 16 * MT;
  const int kw = a.K / WAVES, k0 = wave * kw;
  const int msub = min(MT, (a.T - t0 + 15) / 16);  // row tiles holding tokens (wave-uniform)

  const uint16_t* wrow = a.w + (int64_t)writer_col(x, l16, a.width) * a.w_st + k0 + 8 * g;
  const uint16_t* hrow[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) hrow[m] = a.h + (int64_t)min(t0 + 16 * m + l16, a.T - 1) * a.h_st + k0 + 8 * g;

  floatx4 acc[MT];
#pragma unroll
  for (int m = 0; m < MT; ++m) acc[m] = floatx4{0.f, 0.f, 0.f, 0.f};
  // kw is a multiple of 128: batches of four 32-wide k steps, two batches in flight (the second batch's loads
  // are issued before the first batch's MFMAs)
  u32x4 b0[4], a0[4][MT], b1[4], a1[4][MT];
  auto issue = [&](u32x4(&bv)[4], u32x4(&av)[4][MT], int k) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      bv[i] = ld16(wrow + k + 32 * i);
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (m < msub) av[i][m] = ld16(hrow[m] + k + 32 * i);
    }
  };
  auto compute = [&](const u32x4(&bv)[4], const u32x4(&av)[4][MT]) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int m = 0; m < MT; ++m)
        if (m < msub) acc[m] = mfma16x16x32(av[i][m], bv[i], acc[m]);
  };
  issue(b0, a0, 0);
  for (int k = 0; k < kw; k += 256) {
    const bool second = k + 128 < kw;
    if (second) issue(b1, a1, k + 128);
    compute(b0, a0);
    if (k + 256 < kw) issue(b0, a0, k + 256);
    if (second) compute(b1, a1);
  }
  // lane holds D[4g + r][l16] of row tile m: token t0 + 16m + 4g + r, tile column l16
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < 4; ++r) red[wave][16 * m + 4 * g + r][l16] = acc[m][r];
  __syncthreads();

  // thread: token t0 + tid/4, tile columns q, q+4, q+8, q+12 (q = tid % 4): two rotation pairs in a key tile
  const int row = tid >> 2, q = tid & 3, t = t0 + row;
  if (row >= 16 * MT || t >= a.T) return;
  float v[4];
  int col[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int j = q + 4 * i;
    col[i] = writer_col(x, j, a.width);
    float sum = red[0][row][j];
#pragma unroll
    for (int v2 = 1; v2 < WAVES; ++v2) sum += red[v2][row][j];
    float u = rbf(sum);
    if (a.prev) u = rbf(bf2f(a.prev[(int64_t)t * a.prev_st + col[i]]) + u);
    v[i] = u;
    if (a.reg) a.reg[(int64_t)t * a.reg_st + col[i]] = f2bf(u);
  }
  if (!a.cache) return;
  const int64_t slot = a.slots[t];
  if (slot < 0 || slot >= a.num_slots) return;
  uint16_t* crow = a.cache + (slot / a.block) * a.page_stride + (slot % a.block) * a.row_stride;
  if (x < a.width / 16) {
    const int half = a.width / 2;
    const uint16_t* tr =
        a.table + min(max(a.pos[t], (int64_t)0), (int64_t)a.table_rows - 1) * a.table_stride;
#pragma unroll
    for (int p = 0; p < 2; ++p) {  // pair (col[p], col[p] + w/2) = (v[p], v[p + 2])
      const int c = col[p];
      const float cs = bf2f(tr[c]), sn = bf2f(tr[half + c]);
      const float x1 = v[p], x2 = v[p + 2];
      crow[c] = f2bf(rbf(x1 * cs) - rbf(x2 * sn));
      crow[c + half] = f2bf(rbf(x2 * cs) + rbf(x1 * sn));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) crow[col[i]] = f2bf(v[i]);
  }
}

// ---- many tokens: LDS-tiled GEMM ---------------------------------------------------------------------------------
// out^T[column][token] = W h^T on 16x16x32 MFMA: a workgroup of 2 x 2 waves computes 32 MT tokens x 32 NT columns, a
// wave 16 MT x 16 NT of them, over the whole hidden dimension in steps of 64. A step's rows of h and W (128 bytes
// each) go global -> LDS directly into a ring of three stages, two steps ahead, one barrier per step; the 16-byte
// chunk c of row r sits at position c ^ (r % 8), so the MFMA operands' row reads meet no bank conflict (the copy's
// lanes take their source chunk through the same swizzle). A lane holds four consecutive columns of one token; in a
// key-half tile the column blocks f and f + NT / 2 of a wave are the two halves of the same rotation pairs, so the
// RoPE stays in registers. h comes from one XCD's L2 for all its column tiles (token blocks are dealt to the XCDs in
// turn).
// Bound: about 5 us of launch, first copies and epilogue, then the chain of steps (LDS copies, operand reads,
// MFMAs, barrier). Per launch with hidden 2048, MI355X, against the kernel above, one layer's weights again and
// again: 2048 tokens 17.0 us at width 512 (506 TFLOP/s) and 12.8 at 256, from 89.7 and 46.4; 300 tokens 11.0 and
// 10.4, from 20.7 and 12.5. In a model's layers, each with weights of its own (kernel trace): 2048 tokens 20.4 and
// 15.3 us. Rings of four and six stages, fragments read a half step ahead of their MFMAs, and eight waves splitting a
// step's two halves measured within 8 % of this either way; 64 x 128 tiles are slower up to 2048 tokens (18.6 us) and
// faster at 8192 (50.5 against 56.5), 128 x 128 ones slower everywhere.
constexpr int kStages = 3, kStep = 64;

template <int MT, int NT>
__global__ __launch_bounds__(256) void writer_gemm(WriterParams a, int tblocks, int ctiles) {
  constexpr int BM = 32 * MT, BN = 32 * NT, ROWS = BM + BN, COPIES = ROWS / 32;
  __shared__ __attribute__((aligned(16))) uint16_t ring[kStages][ROWS * kStep];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, l16 = lane & 15, g = lane >> 4;
  const int wm = wave & 1, wn = wave >> 1;
  // workgroup id -> (token block, column tile): XCD id % 8 takes the token blocks = its index mod 8
  const int slot = (int)blockIdx.x / 8, tb = (int)blockIdx.x % 8 + 8 * (slot / ctiles), x = slot % ctiles;
  if (tb >= tblocks) return;
  const int t0 = tb * BM;
  const int key_tiles = a.width / BN;
  const bool key_tile = x < key_tiles;
  // output column of column 0 of block f of wave column w
  auto col_of = [&](int w, int f) {
    if (key_tile) return 8 * NT * (2 * x + w) + 16 * (f % (NT / 2)) + (f >= NT / 2 ? a.width / 2 : 0);
    return a.width + BN * (x - key_tiles) + 16 * NT * w + 16 * f;
  };

  // this wave's copies: rows 8 (wave + 4 i) .. + 8 of the stage (h rows first, then W rows), 8 lanes per row
  const uint16_t* src[COPIES];
#pragma unroll
  for (int i = 0; i < COPIES; ++i) {
    const int r = 8 * (wave + 4 * i) + (lane >> 3), c = (lane & 7) ^ (r & 7);
    const uint16_t* row;
    if (r < BM) {
      row = a.h + (int64_t)min(t0 + r, a.T - 1) * a.h_st;
    } else {
      const int n = r - BM, f = (n / 16) % NT, w = n / (16 * NT);
      row = a.w + (int64_t)(col_of(w, f) + n % 16) * a.w_st;
    }
    src[i] = row + 8 * c;
  }
  auto copy_stage = [&](int step) {
    uint16_t* dst = ring[step % kStages];
#pragma unroll
    for (int i = 0; i < COPIES; ++i)
      copy16_to_lds_v(src[i] + step * kStep, dst + __builtin_amdgcn_readfirstlane(8 * (wave + 4 * i) * kStep));
  };

  floatx4 acc[MT][NT];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int f = 0; f < NT; ++f) acc[m][f] = floatx4{0.f, 0.f, 0.f, 0.f};
  const int steps = a.K / kStep;  // at least 8
  copy_stage(0);
  copy_stage(1);
  for (int i = 0; i < steps; ++i) {
    // stage i has landed once only the copies of stage i + 1 are outstanding, and this wave's reads of stage i - 1,
    // whose buffer takes stage i + 2, have returned; the barrier makes both true of every wave
    if (i + 1 < steps)
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(COPIES, 0));
    else
      __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    plain_barrier();
    if (i + 2 < steps) copy_stage(i + 2);
    const uint16_t* st = ring[i % kStages];
#pragma unroll
    for (int kk = 0; kk < kStep / 32; ++kk) {
      const int off = ((4 * kk + g) ^ (l16 & 7)) * 8;  // (block bases are multiples of 16 rows: r % 8 = l16 % 8)
      u32x4 hv[MT], wv[NT];
#pragma unroll
      for (int m = 0; m < MT; ++m) hv[m] = ld16(st + (16 * (MT * wm + m) + l16) * kStep + off);
#pragma unroll
      for (int f = 0; f < NT; ++f) wv[f] = ld16(st + (BM + 16 * (NT * wn + f) + l16) * kStep + off);
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int f = 0; f < NT; ++f) acc[m][f] = mfma16x16x32(wv[f], hv[m], acc[m][f]);
    }
  }

  // lane: columns col_of(wn, f) + 4 g .. + 4 of token t0 + 16 (MT wm + m) + l16
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const int t = t0 + 16 * (MT * wm + m) + l16;
    if (t >= a.T) continue;
    float v[NT][4];
#pragma unroll
    for (int f = 0; f < NT; ++f) {
      const int c = col_of(wn, f) + 4 * g;
#pragma unroll
      for (int r = 0; r < 4; ++r) v[f][r] = rbf(acc[m][f][r]);
      if (a.prev) {
        const u32x2 p = *reinterpret_cast<const u32x2*>(a.prev + (int64_t)t * a.prev_st + c);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[f][r] = rbf((r % 2 ? hi_bf(p[r / 2]) : lo_bf(p[r / 2])) + v[f][r]);
      }
      if (a.reg)
        *reinterpret_cast<u32x2*>(a.reg + (int64_t)t * a.reg_st + c) =
            u32x2{pack2(v[f][0], v[f][1]), pack2(v[f][2], v[f][3])};
    }
    if (!a.cache) continue;
    const int64_t row = a.slots[t];
    if (row < 0 || row >= a.num_slots) continue;
    uint16_t* crow = a.cache + (row / a.block) * a.page_stride + (row % a.block) * a.row_stride;
    if (key_tile) {
      const int half = a.width / 2;
      const uint16_t* tr = a.table + min(max(a.pos[t], (int64_t)0), (int64_t)a.table_rows - 1) * a.table_stride;
#pragma unroll
      for (int f = 0; f < NT / 2; ++f) {
        const int c = col_of(wn, f) + 4 * g;
        const u32x2 cw = *reinterpret_cast<const u32x2*>(tr + c), sw = *reinterpret_cast<const u32x2*>(tr + half + c);
        float lo[4], hi[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float cs = r % 2 ? hi_bf(cw[r / 2]) : lo_bf(cw[r / 2]), sn = r % 2 ? hi_bf(sw[r / 2]) : lo_bf(sw[r / 2]);
          const float x1 = v[f][r], x2 = v[f + NT / 2][r];
          lo[r] = rbf(x1 * cs) - rbf(x2 * sn);
          hi[r] = rbf(x2 * cs) + rbf(x1 * sn);
        }
        *reinterpret_cast<u32x2*>(crow + c) = u32x2{pack2(lo[0], lo[1]), pack2(lo[2], lo[3])};
        *reinterpret_cast<u32x2*>(crow + half + c) = u32x2{pack2(hi[0], hi[1]), pack2(hi[2], hi[3])};
      }
    } else {
#pragma unroll
      for (int f = 0; f < NT; ++f)
        *reinterpret_cast<u32x2*>(crow + col_of(wn, f) + 4 * g) =
            u32x2{pack2(v[f][0], v[f][1]), pack2(v[f][2], v[f][3])};
    }
  }
}

template <int MT, int NT>
void launch_gemm(const WriterParams& p, hipStream_t st) {
  const int tblocks = (p.T + 32 * MT - 1) / (32 * MT), ctiles = 2 * p.width / (32 * NT);
  const unsigned grid = 8u * (unsigned)((tblocks + 7) / 8) * (unsigned)ctiles;
  hipLaunchKernelGGL((writer_gemm<MT, NT>), dim3(grid), dim3(256), 0, st, p, tblocks, ctiles);
}

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool aligned8(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 7u) == 0; }

}  // namespace
}  // namespace hla

extern "C" int hla_s6_write_rows(const void* h, int32_t num_tokens, int32_t hidden, int64_t h_st, const void* weight,
                                 int32_t width, int64_t w_st, const void* prev, int64_t prev_st, void* reg,
                                 int64_t reg_st, const int64_t* slots, const int64_t* positions,
                                 const void* rope_table, int32_t table_rows, int64_t table_stride, void* cache,
                                 int64_t page_stride, int64_t row_stride, int32_t block_size, int64_t num_blocks,
                                 void* stream) {
  using namespace hla;
  HLA_REQUIRE(num_tokens >= 0 && num_tokens <= 65535 * 64, HLA_S6_EINVAL, "write_rows: bad token count %d",
              num_tokens);
  HLA_REQUIRE(width >= 16 && width % 16 == 0 && width <= 4096, HLA_S6_EUNSUPPORTED,
              "write_rows: width %d must be a multiple of 16 (at most 4096)", width);
  HLA_REQUIRE(hidden >= 512 && hidden % 512 == 0, HLA_S6_EUNSUPPORTED,
              "write_rows: hidden %d must be a positive multiple of 512", hidden);
  HLA_REQUIRE(reg || cache, HLA_S6_EINVAL, "write_rows: neither a register output nor a cache to commit to");
  if (num_tokens == 0) return HLA_S6_OK;
  HLA_REQUIRE(h && weight, HLA_S6_EINVAL, "write_rows: null input");
  HLA_REQUIRE(aligned16(h) && h_st % 8 == 0 && aligned16(weight) && w_st % 8 == 0 && h_st >= hidden &&
                  w_st >= hidden,
              HLA_S6_EINVAL, "write_rows: h and weight rows must be 16-byte aligned with a unit last stride");
  HLA_REQUIRE(!prev || prev_st >= 2 * width, HLA_S6_EINVAL, "write_rows: prev rows shorter than 2 * width");
  HLA_REQUIRE(!reg || reg_st >= 2 * width, HLA_S6_EINVAL, "write_rows: reg rows shorter than 2 * width");
  if (cache) {
    HLA_REQUIRE(slots && positions && rope_table && table_rows > 0 && table_stride >= width, HLA_S6_EINVAL,
                "write_rows: a commit needs slots, positions and a [rows, width] RoPE table");
    HLA_REQUIRE(block_size > 0 && num_blocks > 0 && row_stride >= 2 * width && page_stride >= row_stride,
                HLA_S6_EINVAL, "write_rows: bad cache geometry");
  }
  WriterParams p = {};
  p.h = static_cast<const uint16_t*>(h);
  p.h_st = h_st;
  p.w = static_cast<const uint16_t*>(weight);
  p.w_st = w_st;
  p.prev = static_cast<const uint16_t*>(prev);
  p.prev_st = prev_st;
  p.reg = static_cast<uint16_t*>(reg);
  p.reg_st = reg_st;
  p.slots = slots;
  p.pos = positions;
  p.table = static_cast<const uint16_t*>(rope_table);
  p.table_rows = table_rows;
  p.table_stride = table_stride;
  p.cache = static_cast<uint16_t*>(cache);
  p.page_stride = page_stride;
  p.row_stride = row_stride;
  p.block = block_size;
  p.num_slots = cache ? num_blocks * (int64_t)block_size : 0;
  p.T = num_tokens;
  p.K = hidden;
  p.width = width;
  hipStream_t st = as_stream(stream);
  // Up to 128 tokens the operands' latency decides: a workgroup takes 16 tokens x 16 columns and splits the hidden
  // dimension over its waves (6.7-10.5 us against 10-10.9 for the tiled kernel at 16-128 tokens). Beyond, the tiled
  // kernel, in 32 x 64 tiles while 64 x 64 ones would number at most one per CU (1000 tokens, width 512: 12.6 against
  // 13.3 us; 2048 tokens, 512 large tiles: 22.2 against 17.0). It moves 8 bytes of every register, cache and table row
  // at a time and takes whole 64-column tiles: other geometries keep the first kernel in blocks of 64 tokens.
  const bool small = num_tokens <= 128;
  const bool tiled = !small && width % 64 == 0 && aligned8(prev) && prev_st % 4 == 0 && aligned8(reg) &&
                     reg_st % 4 == 0 && aligned8(cache) && page_stride % 4 == 0 && row_stride % 4 == 0 &&
                     aligned8(rope_table) && table_stride % 4 == 0;
  if (tiled) {
    const int64_t large_tiles = (int64_t)((num_tokens + 63) / 64) * (2 * width / 64);
    if (large_tiles <= 256)
      launch_gemm<1, 2>(p, st);
    else
      launch_gemm<2, 2>(p, st);
    return check_launch("write_rows");
  }
  const int rows = small ? 16 : 64;
  const dim3 grid((unsigned)(width / 8), (unsigned)((num_tokens + rows - 1) / rows));
  if (hidden % 1024 == 0) {
    if (small)
      hipLaunchKernelGGL((writer_kernel<8, 1>), grid, dim3(512), 0, st, p);
    else
      hipLaunchKernelGGL((writer_kernel<8, 4>), grid, dim3(512), 0, st, p);
  } else {
    if (small)
      hipLaunchKernelGGL((writer_kernel<4, 1>), grid, dim3(256), 0, st, p);
    else
      hipLaunchKernelGGL((writer_kernel<4, 4>), grid, dim3(256), 0, st, p);
  }
  return check_launch("write_rows");
}
