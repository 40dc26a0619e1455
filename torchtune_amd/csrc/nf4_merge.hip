// Dequantise an NF4 weight and fold the LoRA update into it in one pass:
//
//     out[n][k] = bf16( D(W)[n][k] + bf16( scale * bf16( sum_r B[n][r] * A[r][k] ) ) )
//
// which is the rounding sequence of the eager checkpoint path: the state-dict hook first turns the NF4 weight into
// a bf16 tensor (torchtune/modules/common_utils.py:55-59), then get_merged_lora_ckpt adds
// `(alpha / rank) * lora_b @ lora_a` in bf16 (torchtune/modules/peft/_utils.py:264-266).  The rank-r sum is
// accumulated in fp32 in ascending r with fused multiply-adds.
//
// HBM-bound: 0.5625 B/element read (codes + fp32 block scalers), 2 B/element written.  A workgroup owns a strip of
// 2048 columns and 16 rows: each lane keeps A[0..R)[its 8 columns] in registers for all rows of the strip, so the
// adapter matrices are read from L2 once per workgroup, not once per output.
#include "common.h"
#include "nf4_math.h"

namespace ttamd {
namespace {

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __constant__ float kNF4Merge[16] = TT_NF4_TABLE;

__device__ __forceinline__ uint32_t pack2(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}

constexpr int kRowsPerWg = 16;

template <int R8>  // R8 = rank / 8
__global__ __launch_bounds__(256) void nf4_dequant_merge_kernel(const uint32_t* __restrict__ qdata,
                                                                const float* __restrict__ block_scalers,
                                                                const uint16_t* __restrict__ A,
                                                                const uint16_t* __restrict__ B, float scale, int N, int K,
                                                                uint16_t* __restrict__ out) {
  constexpr int R = 8 * R8;
  __shared__ float2 lut[256];
  __shared__ float bsh[kRowsPerWg][R];
  const int t = threadIdx.x;
  lut[t] = make_float2(round_to_bf16(kNF4Merge[t >> 4]), round_to_bf16(kNF4Merge[t & 15]));
  const int n0 = blockIdx.y * kRowsPerWg;
  for (int i = t; i < kRowsPerWg * R; i += 256) {
    const int n = n0 + i / R;
    bsh[i / R][i % R] = n < N ? bf16_bits_to_f32(B[(int64_t)n * R + i % R]) : 0.f;
  }
  const int k = blockIdx.x * 2048 + t * 8;
  const bool live = k < K;  // K % 8 == 0
  // adapter columns of this lane, as packed bf16 pairs: a[r][d] = (A[r][k + 2d], A[r][k + 2d + 1])
  u32x4_t a[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    a[r] = u32x4_t{0, 0, 0, 0};
    if (live) a[r] = *reinterpret_cast<const u32x4_t*>(A + (int64_t)r * K + k);
  }
  __syncthreads();
  if (!live) return;
  for (int i = 0; i < kRowsPerWg; ++i) {
    const int n = n0 + i;
    if (n >= N) break;  // uniform over the workgroup
    const int64_t e = (int64_t)n * K + k;
    const uint32_t code = __builtin_nontemporal_load(qdata + (e >> 3));
    const float sc = block_scalers[e >> 6];
    float m[8];
#pragma unroll
    for (int d = 0; d < 8; ++d) m[d] = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const float b = bsh[i][r];
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        uint32_t ar = a[r][d];
        // ranks above 32: keep the pair packed inside the row loop; unpacked ahead of it (which the compiler does when it
        // can) the adapter columns take twice the registers and the kernel spills
        if constexpr (R8 > 4) asm volatile("" : "+v"(ar));
        m[2 * d] = __builtin_fmaf(b, bits_f32(ar << 16), m[2 * d]);
        m[2 * d + 1] = __builtin_fmaf(b, bits_f32(ar & 0xffff0000u), m[2 * d + 1]);
      }
    }
    u32x4_t o;
#pragma unroll
    for (int d = 0; d < 4; ++d) {
      const float2 pr = lut[(code >> (8 * d)) & 0xffu];
      const float w0 = round_to_bf16(pr.x * sc), w1 = round_to_bf16(pr.y * sc);
      const float u0 = round_to_bf16(scale * round_to_bf16(m[2 * d])), u1 = round_to_bf16(scale * round_to_bf16(m[2 * d + 1]));
      o[d] = pack2(w0 + u0, w1 + u1);
    }
    __builtin_nontemporal_store(o, reinterpret_cast<u32x4_t*>(out + e));
  }
}

// Sum of squares of every row of the merged weight bf16(D(W) + bf16(scale * bf16(B . A))) over a strip of 1024 columns,
// norm_part[strip][n] (DoRA's weight norm; finished by dora_norm_finish_kernel).
//
// Bound by the vector ALU, about eleven operations per element (expansion, three roundings, the square), once the rank-r
// product runs on the matrix cores: as r fused multiply-adds per element, the way the merge above forms it, it took three
// quarters of the time (rank 16: 4096 x 14336 64 us, the six other layers of an 8B decoder layer 37 us each on average; now
// 31 and 15).  A wave owns 128 columns and keeps
// their r x 128 piece of A as the row operand of eight v_mfma_f32_16x16x32_bf16 (contraction = the ranks, zeros beyond r),
// then walks over tiles of 16 weight rows, whose r values of B are the column operand.  Row i of product t stands for
// column 8 i + t of the piece: a lane loads its operands of A as 16-byte pieces, and the 32 products it receives belong to
// the 32 consecutive elements of one row whose codes it loads as one 16-byte piece.
constexpr int kNormWaves = 8;
constexpr int kNormStrip = 128 * kNormWaves;
constexpr int kNormMaxTiles = 16;

template <int RG>  // groups of 32 ranks
__global__ __launch_bounds__(64 * kNormWaves) void dora_norm_kernel(const uint32_t* __restrict__ qdata,
                                                                    const float* __restrict__ block_scalers,
                                                                    const uint16_t* __restrict__ A,
                                                                    const uint16_t* __restrict__ B, float scale, int N, int K, int R,
                                                                    int tiles_per_wg, float* __restrict__ norm_part) {
  __shared__ float2 lut[256];
  __shared__ float ssq[kNormMaxTiles][kNormWaves][16];
  const int t = threadIdx.x, lane = t & 63;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  const int i = lane & 15, g = lane >> 4;
  const int kb = (int)blockIdx.x * kNormStrip + 128 * wave;
  const int n_begin = (int)blockIdx.y * tiles_per_wg * 16;
  if (t < 256) lut[t] = make_float2(round_to_bf16(kNF4Merge[t >> 4]), round_to_bf16(kNF4Merge[t & 15]));

  const int k = kb + 32 * g;  // this lane's 32 elements of a row
  const bool live = k < K;    // K % 64 == 0
  struct Piece {
    u32x4_t codes;
    float sc;
    u32x4_t b[RG];
  };
  auto request = [&](int tile) {
    Piece p;
    int n = n_begin + 16 * tile + i;
    n = n < N ? n : N - 1;  // rows beyond N repeat the last one and are never stored
    const int64_t e = (int64_t)n * K + (live ? k : 0);
    p.codes = *reinterpret_cast<const u32x4_t*>(qdata + (e >> 3));
    p.sc = block_scalers[e >> 6];
#pragma unroll
    for (int h = 0; h < RG; ++h) {
      p.b[h] = u32x4_t{0, 0, 0, 0};
      if (32 * h + 8 * g < R) p.b[h] = *reinterpret_cast<const u32x4_t*>(B + (int64_t)n * R + 32 * h + 8 * g);
    }
    return p;
  };
  Piece next = request(0);
  // a[h][t]: ranks 32 h + 8 g .. + 7 of column kb + 8 i + t
  u32x4_t a[RG][8];
#pragma unroll
  for (int h = 0; h < RG; ++h) {
    u32x4_t x[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = u32x4_t{0, 0, 0, 0};
      if (32 * h + 8 * g < R && kb + 8 * i < K) x[e] = *reinterpret_cast<const u32x4_t*>(A + (int64_t)(32 * h + 8 * g + e) * K + kb + 8 * i);
    }
#pragma unroll
    for (int c = 0; c < 8; ++c)
#pragma unroll
      for (int d = 0; d < 4; ++d)
        a[h][c][d] = __builtin_amdgcn_perm(x[2 * d + 1][c >> 1], x[2 * d][c >> 1], (c & 1) ? 0x07060302u : 0x05040100u);
  }
  __syncthreads();
  int tiles = (N - n_begin + 15) / 16;
  tiles = tiles < tiles_per_wg ? tiles : tiles_per_wg;
  for (int tile = 0; tile < tiles; ++tile) {
    const Piece p = next;
    if (tile + 1 < tiles) next = request(tile + 1);
    f32x4_t m[8];
#pragma unroll
    for (int c = 0; c < 8; ++c) {
      m[c] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int h = 0; h < RG; ++h)
        m[c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a[h][c]), __builtin_bit_cast(bf16x8_t, p.b[h]), m[c], 0, 0, 0);
    }
    // m[c][v] = (B . A)[n][k + 8 v + c]
    float ss = 0.f;
#pragma unroll
    for (int v = 0; v < 4; ++v)
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float2 pr = lut[(p.codes[v] >> (8 * d)) & 0xffu];
        const uint32_t w = pack2(pr.x * p.sc, pr.y * p.sc);
        const uint32_t ba = pack2(m[2 * d][v], m[2 * d + 1][v]);
        const uint32_t u = pack2(scale * bits_f32(ba << 16), scale * bits_f32(ba & 0xffff0000u));
        const uint32_t r = pack2(bits_f32(w << 16) + bits_f32(u << 16), bits_f32(w & 0xffff0000u) + bits_f32(u & 0xffff0000u));
        const float v0 = bits_f32(r << 16), v1 = bits_f32(r & 0xffff0000u);
        ss = __builtin_fmaf(v0, v0, ss);
        ss = __builtin_fmaf(v1, v1, ss);
      }
    if (!live) ss = 0.f;
    ss += __shfl_xor(ss, 16, kWave);
    ss += __shfl_xor(ss, 32, kWave);
    if (g == 0) ssq[tile][wave][i] = ss;
  }
  __syncthreads();
  for (int e = t; e < tiles * 16; e += 64 * kNormWaves) {
    const int n = n_begin + e;
    if (n >= N) continue;
    float s = 0.f;
#pragma unroll
    for (int w = 0; w < kNormWaves; ++w) s += ssq[e >> 4][w][e & 15];
    norm_part[(int64_t)blockIdx.x * N + n] = s;
  }
}

// Row tiles per workgroup: a workgroup per CU where the weight has that many, so that the piece of A is loaded for as
// many rows as possible.
int norm_tiles_per_wg(int64_t N, int64_t K) {
  const int64_t strips = (K + kNormStrip - 1) / kNormStrip;
  const int64_t tiles = strips * ((N + 15) / 16) / 256;
  return (int)(tiles < 1 ? 1 : (tiles > kNormMaxTiles ? kNormMaxTiles : tiles));
}

// norm[n] = bf16(sqrt(sum over strips of norm_part[strip][n])), and optionally mag_norm_scale[n] = bf16(magnitude[n] / norm[n])
__global__ __launch_bounds__(256) void dora_norm_finish_kernel(const float* __restrict__ norm_part, int strips, int N,
                                                               const uint16_t* __restrict__ magnitude,
                                                               uint16_t* __restrict__ norm, uint16_t* __restrict__ mns) {
  const int n = blockIdx.x * 256 + threadIdx.x;
  if (n >= N) return;
  float s = 0.f;
  for (int p = 0; p < strips; ++p) s += norm_part[(int64_t)p * N + n];
  const float nv = round_to_bf16(__builtin_sqrtf(s));
  norm[n] = f32_to_bf16_bits(nv);
  if (mns) mns[n] = f32_to_bf16_bits(bf16_bits_to_f32(magnitude[n]) / nv);
}

// DoRA backward prologue, one pass over gy and the layer's saved output:
//   gy0 = bf16(gy * mns)              (the gradient reaching the LoRA-fused linear)
//   gmag_part[slice][n] = sum over the rows of a slice of gy * out   (d out / d magnitude = out / magnitude)
// A workgroup owns 512 columns (8 per lane) and a slice of rows; its 4 waves take rows in turn and add their sums in wave
// order.  Bound by its three streams: 2048 x 14336 37 us = 4.8 TB/s.
__global__ __launch_bounds__(256) void dora_bwd_prologue_kernel(const uint16_t* __restrict__ gy, const uint16_t* __restrict__ out,
                                                                const uint16_t* __restrict__ mns, uint16_t* __restrict__ gy0,
                                                                float* __restrict__ gmag_part, int M, int N,
                                                                int rows_per_split) {
  __shared__ float red[4][512];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = blockIdx.x * 512 + lane * 8;
  const bool live = col < N;  // N % 8 == 0
  const int m_begin = blockIdx.y * rows_per_split;
  int m_end = m_begin + rows_per_split;
  m_end = m_end < M ? m_end : M;
  float acc[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) acc[e] = 0.f;
  if (live) {
    const u32x4_t sv = *reinterpret_cast<const u32x4_t*>(mns + col);
    for (int m = m_begin + wave; m < m_end; m += 4) {
      const int64_t e0 = (int64_t)m * N + col;
      const u32x4_t g = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(gy + e0));
      const u32x4_t o = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(out + e0));
      u32x4_t r;
#pragma unroll
      for (int d = 0; d < 4; ++d) {
        const float g0 = bits_f32(g[d] << 16), g1 = bits_f32(g[d] & 0xffff0000u);
        acc[2 * d] += g0 * bits_f32(o[d] << 16);
        acc[2 * d + 1] += g1 * bits_f32(o[d] & 0xffff0000u);
        r[d] = pack2(g0 * bits_f32(sv[d] << 16), g1 * bits_f32(sv[d] & 0xffff0000u));
      }
      __builtin_nontemporal_store(r, reinterpret_cast<u32x4_t*>(gy0 + e0));
    }
  }
  *reinterpret_cast<f32x4_t*>(&red[wave][lane * 8]) = f32x4_t{acc[0], acc[1], acc[2], acc[3]};
  *reinterpret_cast<f32x4_t*>(&red[wave][lane * 8 + 4]) = f32x4_t{acc[4], acc[5], acc[6], acc[7]};
  __syncthreads();
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int c = threadIdx.x + 256 * h, n = blockIdx.x * 512 + c;
    if (n < N) gmag_part[(int64_t)blockIdx.y * N + n] = ((red[0][c] + red[1][c]) + red[2][c]) + red[3][c];
  }
}

// gmag[n] = bf16(sum over the slices of gmag_part[slice][n] / magnitude[n]), fixed order: a thread adds every eighth slice of
// its column, then the eight sums of a column are added in turn.  (One thread per column over 256 partial rows: 11 - 13 us
// a call, a serial chain of loads on a handful of workgroups; now 4.)
__global__ __launch_bounds__(256) void dora_gmag_finish_kernel(const float* __restrict__ part, int n_parts, int N,
                                                               const uint16_t* __restrict__ magnitude,
                                                               uint16_t* __restrict__ gmag) {
  __shared__ float red[8][32];
  const int c = threadIdx.x & 31, q = threadIdx.x >> 5;
  const int n = blockIdx.x * 32 + c;
  float s = 0.f;
  if (n < N) {
#pragma unroll 8
    for (int p = q; p < n_parts; p += 8) s += part[(int64_t)p * N + n];
  }
  red[q][c] = s;
  __syncthreads();
  if (q != 0 || n >= N) return;
#pragma unroll
  for (int p = 1; p < 8; ++p) s += red[p][c];
  gmag[n] = f32_to_bf16_bits(s / bf16_bits_to_f32(magnitude[n]));
}

constexpr int kDoraBwdSplits = 64;  // most row slices of the backward prologue

void launch_merge(int rank, dim3 grid, hipStream_t s, const uint32_t* q, const float* bs, const uint16_t* a, const uint16_t* b,
                  float scale, int N, int K, uint16_t* o) {
  const dim3 block(256);
  switch (rank / 8) {
    case 1: nf4_dequant_merge_kernel<1><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    case 2: nf4_dequant_merge_kernel<2><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    case 3: nf4_dequant_merge_kernel<3><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    case 4: nf4_dequant_merge_kernel<4><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    case 5: nf4_dequant_merge_kernel<5><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    case 6: nf4_dequant_merge_kernel<6><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    case 7: nf4_dequant_merge_kernel<7><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
    default: nf4_dequant_merge_kernel<8><<<grid, block, 0, s>>>(q, bs, a, b, scale, N, K, o); break;
  }
}

}  // namespace
}  // namespace ttamd

using namespace ttamd;

extern "C" int ttamd_nf4_dequantize_merge_bf16(const uint8_t* quantized_data, const void* block_scalers, const void* lora_a,
                                               const void* lora_b, int rank, float scale, void* out, int64_t N, int64_t K,
                                               void* stream) {
  TT_REQUIRE(quantized_data && block_scalers && lora_a && lora_b && out, "nf4_dequantize_merge: null pointer argument");
  TT_REQUIRE(aligned16(quantized_data) && aligned16(lora_a) && aligned16(out) &&
                 (reinterpret_cast<uintptr_t>(block_scalers) & 3u) == 0,
             "nf4_dequantize_merge: quantized_data, lora_a and out must be 16-byte aligned");
  TT_REQUIRE(N > 0 && K > 0 && N < (1 << 30) && K < (1 << 30) && K % 64 == 0,
             "nf4_dequantize_merge: bad shape N=%lld K=%lld (K must be a multiple of the NF4 block size 64)", (long long)N,
             (long long)K);
  TT_REQUIRE(rank > 0 && rank <= 64 && rank % 8 == 0, "nf4_dequantize_merge: rank (%d) must be a multiple of 8 in [8, 64]", rank);
  const dim3 grid((unsigned)((K + 2047) / 2048), (unsigned)((N + kRowsPerWg - 1) / kRowsPerWg));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const uint32_t* q = reinterpret_cast<const uint32_t*>(quantized_data);
  const float* bs = reinterpret_cast<const float*>(block_scalers);
  const uint16_t* a = reinterpret_cast<const uint16_t*>(lora_a);
  const uint16_t* b = reinterpret_cast<const uint16_t*>(lora_b);
  uint16_t* o = reinterpret_cast<uint16_t*>(out);
  launch_merge(rank, grid, s, q, bs, a, b, scale, (int)N, (int)K, o);
  return check_launch("nf4_dequantize_merge");
}

extern "C" size_t ttamd_dora_weight_norm_workspace_bytes(int64_t N, int64_t K) {
  if (N <= 0 || K <= 0) return 0;
  return (size_t)((K + kNormStrip - 1) / kNormStrip) * (size_t)N * sizeof(float);
}

extern "C" int ttamd_nf4_dora_weight_norm_bf16(const uint8_t* quantized_data, const void* block_scalers, const void* lora_a,
                                               const void* lora_b, int rank, float scale, const void* magnitude,
                                               void* weight_norm, void* mag_norm_scale, int64_t N, int64_t K, void* workspace,
                                               size_t workspace_bytes, void* stream) {
  TT_REQUIRE(quantized_data && block_scalers && lora_a && lora_b && weight_norm && workspace,
             "nf4_dora_weight_norm: null pointer argument");
  TT_REQUIRE((magnitude == nullptr) == (mag_norm_scale == nullptr),
             "nf4_dora_weight_norm: magnitude and mag_norm_scale must both be given or both be null");
  TT_REQUIRE(aligned16(quantized_data) && aligned16(lora_a) && aligned16(lora_b) && aligned16(workspace) &&
                 (reinterpret_cast<uintptr_t>(block_scalers) & 3u) == 0,
             "nf4_dora_weight_norm: quantized_data, lora_a, lora_b and workspace must be 16-byte aligned");
  TT_REQUIRE(N > 0 && K > 0 && N < (1 << 30) && K < (1 << 30) && K % 64 == 0,
             "nf4_dora_weight_norm: bad shape N=%lld K=%lld (K must be a multiple of the NF4 block size 64)", (long long)N,
             (long long)K);
  TT_REQUIRE(rank > 0 && rank <= 64 && rank % 8 == 0, "nf4_dora_weight_norm: rank (%d) must be a multiple of 8 in [8, 64]", rank);
  if (workspace_bytes < ttamd_dora_weight_norm_workspace_bytes(N, K))
    return fail(TTAMD_EWORKSPACE, "nf4_dora_weight_norm: workspace has %zu bytes, needs %zu", workspace_bytes,
                ttamd_dora_weight_norm_workspace_bytes(N, K));
  const int strips = (int)((K + kNormStrip - 1) / kNormStrip), tiles = norm_tiles_per_wg(N, K);
  const dim3 grid((unsigned)strips, (unsigned)((N + 16 * tiles - 1) / (16 * tiles))), block(64 * kNormWaves);
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  float* part = reinterpret_cast<float*>(workspace);
  const uint32_t* q = reinterpret_cast<const uint32_t*>(quantized_data);
  const float* bs = reinterpret_cast<const float*>(block_scalers);
  const uint16_t* a = reinterpret_cast<const uint16_t*>(lora_a);
  const uint16_t* b = reinterpret_cast<const uint16_t*>(lora_b);
  if (rank <= 32)
    dora_norm_kernel<1><<<grid, block, 0, s>>>(q, bs, a, b, scale, (int)N, (int)K, rank, tiles, part);
  else
    dora_norm_kernel<2><<<grid, block, 0, s>>>(q, bs, a, b, scale, (int)N, (int)K, rank, tiles, part);
  dora_norm_finish_kernel<<<dim3((unsigned)((N + 255) / 256)), dim3(256), 0, s>>>(
      part, strips, (int)N, reinterpret_cast<const uint16_t*>(magnitude), reinterpret_cast<uint16_t*>(weight_norm),
      reinterpret_cast<uint16_t*>(mag_norm_scale));
  return check_launch("nf4_dora_weight_norm");
}

extern "C" size_t ttamd_dora_bwd_workspace_bytes(int64_t N) {
  return N > 0 ? (size_t)kDoraBwdSplits * (size_t)N * sizeof(float) : 0;
}

extern "C" int ttamd_dora_bwd_prologue_bf16(const void* gy, const void* out, const void* mag_norm_scale, const void* magnitude,
                                            void* gy0, void* gmagnitude, int64_t M, int64_t N, void* workspace,
                                            size_t workspace_bytes, void* stream) {
  TT_REQUIRE(gy && out && mag_norm_scale && magnitude && gy0 && gmagnitude && workspace, "dora_bwd_prologue: null pointer argument");
  TT_REQUIRE(aligned16(gy) && aligned16(out) && aligned16(mag_norm_scale) && aligned16(gy0) && aligned16(workspace),
             "dora_bwd_prologue: pointers must be 16-byte aligned");
  TT_REQUIRE(M > 0 && N > 0 && N % 8 == 0 && M < (1 << 30) && N < (1 << 30), "dora_bwd_prologue: bad shape M=%lld N=%lld (N must be a multiple of 8)",
             (long long)M, (long long)N);
  if (workspace_bytes < ttamd_dora_bwd_workspace_bytes(N))
    return fail(TTAMD_EWORKSPACE, "dora_bwd_prologue: workspace has %zu bytes, needs %zu", workspace_bytes,
                ttamd_dora_bwd_workspace_bytes(N));
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int64_t rows_per_split = (M + kDoraBwdSplits - 1) / kDoraBwdSplits;
  rows_per_split = (rows_per_split + 3) / 4 * 4;
  const int splits = (int)((M + rows_per_split - 1) / rows_per_split);
  float* part = reinterpret_cast<float*>(workspace);
  dora_bwd_prologue_kernel<<<dim3((unsigned)((N + 511) / 512), (unsigned)splits), dim3(256), 0, s>>>(
      reinterpret_cast<const uint16_t*>(gy), reinterpret_cast<const uint16_t*>(out), reinterpret_cast<const uint16_t*>(mag_norm_scale),
      reinterpret_cast<uint16_t*>(gy0), part, (int)M, (int)N, (int)rows_per_split);
  dora_gmag_finish_kernel<<<dim3((unsigned)((N + 31) / 32)), dim3(256), 0, s>>>(
      part, splits, (int)N, reinterpret_cast<const uint16_t*>(magnitude), reinterpret_cast<uint16_t*>(gmagnitude));
  return check_launch("dora_bwd_prologue");
}
