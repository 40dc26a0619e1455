// NF4 double-quantisation codec for gfx950: to_nf4 (quantise) and get_original_weight (dequantise).
//
// Both directions are HBM-bound streaming kernels.  Algorithmic traffic per weight element for a bf16
// tensor with block 64 / scaler block 256:  0.5 B codes + 1/64 B int8 scaler + 2/16384 B factor on the
// packed side, 2 B on the dense side = 2.515747 B.
//
// Layout (all row-major, flattened):
//   quantized_data   u8  [numel/2]        byte b = code(2b) << 4 | code(2b+1)
//   quantized_scalers i8 [numel/bs]       one per block of `bs` consecutive elements
//   quantization_factor T [numel/bs/SB]   one per `SB` consecutive blocks
//   scaler_mean      T   [1]
#include <type_traits>

#include "common.h"
#include "nf4_math.h"

namespace ttamd {
namespace {

__device__ __constant__ float kNF4Dev[16] = TT_NF4_TABLE;

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ uint32_t pack_bf16x2(float lo, float hi) {
  bf16x2_t v;
  v.x = (__bf16)lo;
  v.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, v);
}

// max that propagates NaN the way torch.max does
__device__ __forceinline__ float nanmax(float a, float b) { return (a != a) ? a : ((b != b) ? b : (a > b ? a : b)); }

template <bool BF16>
__device__ __forceinline__ float load1(const void* base, int64_t i) {
  if constexpr (BF16)
    return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(base)[i]);
  else
    return reinterpret_cast<const float*>(base)[i];
}

template <bool BF16>
__device__ __forceinline__ void store1(void* base, int64_t i, float v) {
  if constexpr (BF16)
    reinterpret_cast<uint16_t*>(base)[i] = f32_to_bf16_bits(v);
  else
    reinterpret_cast<float*>(base)[i] = v;
}

// ---------------------------------------------------------------------------------------------------
// quantise, pass 1: per-block absmax and the 4-bit codes.  One lane owns 8 consecutive elements (128 bits of bf16, twice
// that of float); a block of `bs` elements is spread over bs/8 neighbouring lanes of one wave.
//
// Vector-ALU bound when every element took a division and a search, so the work per element is what counts:
// * the maximum is one of bit patterns without signs (a NaN is above every number, as torch.max has it), for bf16 two
//   elements at a time, and for blocks of 64 travels between lanes as DPP operands instead of through the LDS;
// * the block's elements share one reciprocal, and a code is one read of a 64-word table, whose entries lie in banks of
//   their own, and one comparison (nf4_math.h says why that is exact);
// * a thread's four chunks are all requested before the first is used.
// 9 vector-ALU instructions per bf16 element (about 15 and a byte read from a 1.3 KB table before): 14336 x 4096 in bf16
// takes 25 us = 6.0 TB/s, what a streaming copy reaches; quantising and dequantising it, with the passes below, 59 us.
// An absmax outside the range where the shared reciprocal is exact (zero, denormal, huge, infinite, NaN) takes the
// division and the search of the 16 codes.
// ---------------------------------------------------------------------------------------------------
constexpr int kQuantChunksPerThread = 4;

typedef uint16_t u16x2_t __attribute__((ext_vector_type(2)));

template <int CTRL>
__device__ __forceinline__ uint32_t dpp_max(uint32_t m) {
  const uint32_t o = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)m, CTRL, 0xf, 0xf, true);
  return m > o ? m : o;
}

// LPB: lanes per block, 0 = the argument (any power of two up to 64)
template <bool BF16, int LPB>
__global__ __launch_bounds__(256) void nf4_quantize_blocks_kernel(const u32x4_t* __restrict__ w, int64_t n_chunks, int lpb_arg,
                                                                  int log2_lpb, uint32_t fast_low, uint32_t fast_high,
                                                                  uint32_t* __restrict__ qdata, float* __restrict__ absmax,
                                                                  double* __restrict__ partial, const Nf4BinTable<BF16> table) {
  constexpr int U = kQuantChunksPerThread;
  constexpr int V = BF16 ? 1 : 2;  // 128-bit words per chunk
  __shared__ uint32_t tab[Nf4BinTable<BF16>::kWords];
  const int64_t chunk0 = (int64_t)blockIdx.x * (U * 256) + threadIdx.x;
  u32x4_t raw[U][V];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t chunk = chunk0 + u * 256;
    const int64_t at = chunk < n_chunks ? chunk : n_chunks - 1;  // past the end: any valid chunk, not stored
#pragma unroll
    for (int h = 0; h < V; ++h) raw[u][h] = w[V * at + h];
  }
  if (threadIdx.x < Nf4BinTable<BF16>::kWords) tab[threadIdx.x] = table.words[threadIdx.x];
  __shared__ double wave_sum[4];
  __syncthreads();
  const int lpb = LPB ? LPB : lpb_arg;
  double sum = 0.0;  // of the maxima of this lane's blocks
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int64_t chunk = chunk0 + u * 256;
    uint32_t m_bits;
    if constexpr (BF16) {
      u16x2_t mm = __builtin_bit_cast(u16x2_t, raw[u][0][0] & 0x7fff7fffu);
#pragma unroll
      for (int i = 1; i < 4; ++i) mm = __builtin_elementwise_max(mm, __builtin_bit_cast(u16x2_t, raw[u][0][i] & 0x7fff7fffu));
      const uint32_t lo = mm[0], hi = mm[1];
      m_bits = (lo > hi ? lo : hi) << 16;
    } else {
      m_bits = 0;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t a = raw[u][(i >> 2) * (V - 1)][i & 3] & 0x7fffffffu;
        m_bits = m_bits > a ? m_bits : a;
      }
    }
    if constexpr (LPB == 8) {
      m_bits = dpp_max<0xb1>(m_bits);   // quad_perm [1, 0, 3, 2]
      m_bits = dpp_max<0x4e>(m_bits);   // quad_perm [2, 3, 0, 1]
      m_bits = dpp_max<0x141>(m_bits);  // row_half_mirror: the other four lanes
    } else {
      for (int off = 1; off < lpb; off <<= 1) {
        const uint32_t o = (uint32_t)__shfl_xor((int)m_bits, off, kWave);
        m_bits = m_bits > o ? m_bits : o;
      }
    }
    if (chunk >= n_chunks) continue;  // a whole block of lanes: n_chunks is a multiple of lpb
    const float m = bits_f32(m_bits);
    if ((threadIdx.x & (lpb - 1)) == 0) {
      absmax[chunk >> log2_lpb] = m;
      sum += (double)m;
    }
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      if constexpr (BF16)
        v[i] = bits_f32((i & 1) ? raw[u][0][i >> 1] & 0xffff0000u : raw[u][0][i >> 1] << 16);
      else
        v[i] = bits_f32(raw[u][(i >> 2) * (V - 1)][i & 3]);
    }
    uint32_t packed = 0;
    if (m_bits >= fast_low && m_bits < fast_high) {
      const float y = BF16 ? __builtin_amdgcn_rcpf(m) : 1.0f / m;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float t = BF16 ? v[i] * y : nf4_shared_quotient(v[i], m, y);
        const uint32_t* entry = reinterpret_cast<const uint32_t*>(reinterpret_cast<const char*>(tab) + nf4_bin_offset(t));
        uint32_t code;
        if constexpr (BF16)
          code = nf4_code_below(entry[0]) + (nf4_above_edge_bf16(t, entry[0]) ? 1u : 0u);
        else
          code = entry[kNf4Bins] + (t >= bits_f32(entry[0]) ? 1u : 0u);
        packed |= code << (8 * (i >> 1) + ((i & 1) ? 0 : 4));
      }
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        packed |= (uint32_t)nf4_nearest_code<BF16>(Arith<BF16>::rnd(v[i] / m)) << (8 * (i >> 1) + ((i & 1) ? 0 : 4));
    }
    qdata[chunk] = packed;
  }
  for (int off = lpb; off < kWave; off <<= 1) sum += __shfl_xor(sum, off, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) wave_sum[threadIdx.x >> 6] = sum;
  __syncthreads();
  if (threadIdx.x == 0) partial[blockIdx.x] = (wave_sum[0] + wave_sum[1]) + (wave_sum[2] + wave_sum[3]);
}

int64_t quantize_workgroups(int64_t n_chunks) { return (n_chunks + 256 * kQuantChunksPerThread - 1) / (256 * kQuantChunksPerThread); }

// The table, filled and verified once per process.
template <bool BF16>
struct Nf4BinTableHost {
  Nf4BinTable<BF16> table;
  bool ok;
  Nf4BinTableHost() { ok = nf4_fill_bins<BF16>(table); }
};

template <bool BF16>
void launch_quantize_blocks(const void* w, int64_t n_chunks, int lpb, int log2_lpb, uint8_t* qdata, float* absmax, double* partial,
                            hipStream_t s) {
  static const Nf4BinTableHost<BF16> host;
  const uint32_t low = host.ok ? Nf4FastRange<BF16>::low : 0u, high = host.ok ? Nf4FastRange<BF16>::high : 0u;
  const dim3 grid((unsigned)quantize_workgroups(n_chunks));
  auto launch = [&](auto kernel) {
    kernel<<<grid, dim3(256), 0, s>>>(reinterpret_cast<const u32x4_t*>(w), n_chunks, lpb, log2_lpb, low, high,
                                      reinterpret_cast<uint32_t*>(qdata), absmax, partial, host.table);
  };
  if (lpb == 8)
    launch(nf4_quantize_blocks_kernel<BF16, 8>);
  else
    launch(nf4_quantize_blocks_kernel<BF16, 0>);
}

// ---------------------------------------------------------------------------------------------------
// quantise, pass 2: mean of the block absmaxes.  Summed in fp64 in a fixed order (pass 1 leaves one sum per workgroup, pass 3 adds
// them by a fixed strided walk and a fixed LDS tree) so the result does not depend on scheduling; for realistic dynamic
// ranges the fp64 sum is exact.  mean = dtype(float(sum / n)).  Every workgroup of pass 3 reads all the sums: 57 KB of them at
// 14336 x 4096, where a launch that summed the maxima took 5.4 us and reading the sums takes 3 (the quantisation 38.7 -> 37.7, that of
// 4096 x 4096 19.5 -> 16.8; fewer workgroups in pass 3 read less and are slower, 43.6 with 256); beyond kDirectPartials they are added up to
// kMeanPartials by a launch of its own first (28672 x 8192 134 -> 124).
// ---------------------------------------------------------------------------------------------------
constexpr int kMeanPartials = 256;
constexpr int64_t kDirectPartials = 8192;

__device__ __forceinline__ double block_sum_256(double s, double* sh) {  // sh: four
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) s += __shfl_xor(s, off, kWave);
  if ((threadIdx.x & (kWave - 1)) == 0) sh[threadIdx.x >> 6] = s;
  __syncthreads();
  return (sh[0] + sh[1]) + (sh[2] + sh[3]);
}

__global__ __launch_bounds__(256) void nf4_partial_sum_kernel(const double* __restrict__ sums, int64_t n, double* __restrict__ partial) {
  __shared__ double sh[4];
  double s = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)kMeanPartials * 256) s += sums[i];
  s = block_sum_256(s, sh);
  if (threadIdx.x == 0) partial[blockIdx.x] = s;
}

// ---------------------------------------------------------------------------------------------------
// quantise, pass 3: double quantisation of the block scalers.  One wave per scaler block of SB blocks.  Every workgroup
// finishes the mean for itself (the partial sums in the same order: the same bits), which saves a launch of one workgroup.
// The first also writes the sixteen code values where they are asked for.
// ---------------------------------------------------------------------------------------------------
template <bool BF16>
__global__ __launch_bounds__(256) void nf4_quantize_scalers_kernel(const float* __restrict__ absmax,
                                                                   const double* __restrict__ partial, int n_partial, int64_t n_blocks,
                                                                   int64_t n_sb, int SB, int8_t* __restrict__ qscalers,
                                                                   void* __restrict__ qfactor, void* __restrict__ scaler_mean,
                                                                   void* __restrict__ code_values) {
  __shared__ double sh[4];
  double sum = 0.0;
#pragma unroll 8
  for (int i = threadIdx.x; i < n_partial; i += 256) sum += partial[i];
  const float mean = Arith<BF16>::rnd((float)(block_sum_256(sum, sh) / (double)n_blocks));
  if (code_values && blockIdx.x == 0 && threadIdx.x < 16) store1<BF16>(code_values, threadIdx.x, kNF4Dev[threadIdx.x]);
  if (blockIdx.x == 0 && threadIdx.x == 0) store1<BF16>(scaler_mean, 0, mean);
  const int64_t sb = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (sb >= n_sb) return;  // whole wave leaves together
  const int lane = threadIdx.x & 63;
  const float* a = absmax + sb * SB;
  float m = 0.f;
  for (int i = lane; i < SB; i += kWave) m = nanmax(m, __builtin_fabsf(Arith<BF16>::rnd(a[i] - mean)));
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) m = nanmax(m, __shfl_xor(m, off, kWave));
  const float factor = Arith<BF16>::rnd(256.0f / Arith<BF16>::rnd(2.0f * m));
  if (lane == 0) store1<BF16>(qfactor, sb, factor);
  for (int i = lane; i < SB; i += kWave) {
    float s1 = Arith<BF16>::rnd(a[i] - mean);
    float q = __builtin_rintf(Arith<BF16>::rnd(s1 * factor));  // torch.round: half to even
    q = (q != q) ? 0.f : (q < -128.f ? -128.f : (q > 127.f ? 127.f : q));
    qscalers[sb * SB + i] = (int8_t)(int)q;
  }
}

// ---------------------------------------------------------------------------------------------------
// dequantise.  A workgroup expands 256 * DW * 8 elements (DW = dwords of codes per lane).  It first evaluates the
// block scalers of its span once (one thread per block, into LDS: the division is done once per block, not once per
// lane), then every lane turns one dword of codes (8 elements) into one 128-bit bf16 store (two for fp32), so each load and
// store instruction of a wave covers one contiguous span.  Code pairs are looked up a byte at a time in a
// 256-entry LDS table of (nf4[hi], nf4[lo]) in fp32; for bf16 the product is rounded once, by the packing
// conversion (round to nearest even, the same rounding the eager reference applies to the product).
//
// DW is chosen by the launch: 8 (16384 elements per workgroup) while codes and output together fit the 256 MB
// last-level cache, where fewer, longer workgroups win (measured 5.9 against 5.6 TB/s on 14336 x 4096), and 4 beyond
// it, where twice the number of workgroups keeps more HBM requests in flight (6.1 against 5.4 TB/s on 28672 x 8192
// with the cache defeated by rotating over four weights).
// ---------------------------------------------------------------------------------------------------
constexpr int64_t kDequantCacheResidentBytes = int64_t(192) << 20;

template <bool BF16, int DW>
__global__ __launch_bounds__(256) void nf4_dequantize_kernel(const uint32_t* __restrict__ qdata,
                                                             const int8_t* __restrict__ qscalers,
                                                             const void* __restrict__ qfactor,
                                                             const void* __restrict__ scaler_mean, int64_t n_dwords,
                                                             int log2_dwords_per_block, int SB, int log2_SB,
                                                             int64_t n_blocks, void* __restrict__ out) {
  __shared__ float2 lut[256];
  __shared__ float scal[256 * DW];  // smallest block size is 8 elements = one dword
  const int t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * (256 * DW) + t;
  uint32_t code[DW];
#pragma unroll
  for (int u = 0; u < DW; ++u) {
    const int64_t idx = base + u * 256;
    code[u] = idx < n_dwords ? __builtin_nontemporal_load(qdata + idx) : 0u;
  }
  lut[t] = make_float2(Arith<BF16>::rnd(kNF4Dev[t >> 4]), Arith<BF16>::rnd(kNF4Dev[t & 15]));
  {
    const float mean = load1<BF16>(scaler_mean, 0);
    const int blocks_per_wg = (256 * DW) >> log2_dwords_per_block;
    const int64_t blk0 = (int64_t)blockIdx.x * blocks_per_wg;
    for (int i = t; i < blocks_per_wg; i += 256) {
      const int64_t blk = blk0 + i;
      if (blk >= n_blocks) break;
      const int64_t sb = log2_SB >= 0 ? (blk >> log2_SB) : (blk / SB);
      scal[i] = nf4_block_scaler<BF16>((int)qscalers[blk], load1<BF16>(qfactor, sb), mean);
    }
  }
  __syncthreads();
#pragma unroll
  for (int u = 0; u < DW; ++u) {
    const int64_t idx = base + u * 256;
    if (idx >= n_dwords) continue;
    const float sc = scal[(u * 256 + t) >> log2_dwords_per_block];
    float v[8];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
      const float2 pr = lut[(code[u] >> (8 * b)) & 0xffu];
      v[2 * b] = pr.x * sc;
      v[2 * b + 1] = pr.y * sc;
    }
    if constexpr (BF16) {
      u32x4_t o;
      o.x = pack_bf16x2(v[0], v[1]);
      o.y = pack_bf16x2(v[2], v[3]);
      o.z = pack_bf16x2(v[4], v[5]);
      o.w = pack_bf16x2(v[6], v[7]);
      __builtin_nontemporal_store(o, reinterpret_cast<u32x4_t*>(out) + idx);
    } else {
      f32x4_t* o = reinterpret_cast<f32x4_t*>(out) + 2 * idx;
      f32x4_t a = {v[0], v[1], v[2], v[3]}, b = {v[4], v[5], v[6], v[7]};
      __builtin_nontemporal_store(a, o);
      __builtin_nontemporal_store(b, o + 1);
    }
  }
}

int log2_exact(int64_t v) {
  int l = 0;
  while ((int64_t(1) << l) < v) ++l;
  return l;
}

struct QuantWorkspace {
  float* absmax;    // [n_blocks]
  double* partial;  // [kMeanPartials], then one per workgroup of pass 1
};

size_t quant_ws_bytes(int64_t numel, int64_t n_blocks) {
  size_t absmax_bytes = ((size_t)n_blocks * sizeof(float) + 255) & ~size_t(255);
  return absmax_bytes + (kMeanPartials + (size_t)quantize_workgroups(numel / 8)) * sizeof(double) + 256;
}

int check_nf4_shape(int64_t numel, int block_size, int scaler_block_size) {
  TT_REQUIRE(numel > 0, "nf4: numel must be positive (got %lld)", (long long)numel);
  TT_REQUIRE(block_size >= 8 && block_size <= 512 && is_pow2(block_size),
             "nf4: block_size must be a power of two in [8, 512] (got %d)", block_size);
  TT_REQUIRE(scaler_block_size >= 1, "nf4: scaler_block_size must be positive (got %d)", scaler_block_size);
  TT_REQUIRE(numel % block_size == 0, "nf4: numel (%lld) must be divisible by block_size (%d)", (long long)numel,
             block_size);
  TT_REQUIRE((numel / block_size) % scaler_block_size == 0,
             "nf4: number of blocks (%lld) must be divisible by scaler_block_size (%d)",
             (long long)(numel / block_size), scaler_block_size);
  return TTAMD_OK;
}

}  // namespace
}  // namespace ttamd

using namespace ttamd;

extern "C" size_t ttamd_nf4_quantize_workspace_bytes(int64_t numel, int block_size) {
  if (numel <= 0 || block_size <= 0) return 0;
  return quant_ws_bytes(numel, numel / block_size);
}

extern "C" int ttamd_nf4_quantize_with_codes(const void* w, int dtype, int64_t numel, int block_size, int scaler_block_size,
                                             uint8_t* quantized_data, int8_t* quantized_scalers, void* quantization_factor,
                                             void* scaler_mean, void* code_values, void* workspace,
                                             size_t workspace_bytes, void* stream) {
  if (int rc = check_nf4_shape(numel, block_size, scaler_block_size)) return rc;
  TT_REQUIRE(dtype == TTAMD_BF16 || dtype == TTAMD_F32, "nf4_quantize: unknown dtype code %d", dtype);
  TT_REQUIRE(w && quantized_data && quantized_scalers && quantization_factor && scaler_mean && workspace,
             "nf4_quantize: null pointer argument");
  TT_REQUIRE(aligned16(w) && (reinterpret_cast<uintptr_t>(quantized_data) & 3u) == 0 && aligned16(workspace),
             "nf4_quantize: w/workspace must be 16-byte aligned and quantized_data 4-byte aligned");
  const int64_t n_blocks = numel / block_size;
  const int64_t n_sb = n_blocks / scaler_block_size;
  if (workspace_bytes < quant_ws_bytes(numel, n_blocks))
    return fail(TTAMD_EWORKSPACE, "nf4_quantize: workspace has %zu bytes, needs %zu", workspace_bytes,
                quant_ws_bytes(numel, n_blocks));
  QuantWorkspace ws;
  ws.absmax = reinterpret_cast<float*>(workspace);
  size_t absmax_bytes = ((size_t)n_blocks * sizeof(float) + 255) & ~size_t(255);
  ws.partial = reinterpret_cast<double*>(reinterpret_cast<char*>(workspace) + absmax_bytes);

  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int64_t n_chunks = numel / 8;
  const int lpb = block_size / 8;
  const int64_t grid1 = (n_chunks + 255) / 256;
  TT_REQUIRE(grid1 < (int64_t(1) << 31), "nf4_quantize: tensor too large for one launch");
  const int64_t grid3 = (n_sb + 3) / 4;
  auto run = [&](auto bf16) {
    constexpr bool BF16 = decltype(bf16)::value;
    const int64_t sums = quantize_workgroups(n_chunks);
    double* const by_workgroup = ws.partial + kMeanPartials;
    launch_quantize_blocks<BF16>(w, n_chunks, lpb, log2_exact(lpb), quantized_data, ws.absmax, by_workgroup, s);
    const bool direct = sums <= kDirectPartials;
    if (!direct) nf4_partial_sum_kernel<<<dim3(kMeanPartials), dim3(256), 0, s>>>(by_workgroup, sums, ws.partial);
    nf4_quantize_scalers_kernel<BF16><<<dim3((unsigned)grid3), dim3(256), 0, s>>>(
        ws.absmax, direct ? by_workgroup : ws.partial, direct ? (int)sums : kMeanPartials, n_blocks, n_sb, scaler_block_size,
        quantized_scalers, quantization_factor, scaler_mean, code_values);
  };
  if (dtype == TTAMD_BF16)
    run(std::true_type{});
  else
    run(std::false_type{});
  return check_launch("nf4_quantize");
}

extern "C" int ttamd_nf4_quantize(const void* w, int dtype, int64_t numel, int block_size, int scaler_block_size,
                                  uint8_t* quantized_data, int8_t* quantized_scalers, void* quantization_factor,
                                  void* scaler_mean, void* workspace, size_t workspace_bytes, void* stream) {
  return ttamd_nf4_quantize_with_codes(w, dtype, numel, block_size, scaler_block_size, quantized_data, quantized_scalers,
                                       quantization_factor, scaler_mean, nullptr, workspace, workspace_bytes, stream);
}

extern "C" int ttamd_nf4_dequantize(const uint8_t* quantized_data, const int8_t* quantized_scalers,
                                    const void* quantization_factor, const void* scaler_mean, int dtype, int64_t numel,
                                    int block_size, int scaler_block_size, void* out, void* stream) {
  if (int rc = check_nf4_shape(numel, block_size, scaler_block_size)) return rc;
  TT_REQUIRE(dtype == TTAMD_BF16 || dtype == TTAMD_F32, "nf4_dequantize: unknown dtype code %d", dtype);
  TT_REQUIRE(quantized_data && quantized_scalers && quantization_factor && scaler_mean && out,
             "nf4_dequantize: null pointer argument");
  TT_REQUIRE((reinterpret_cast<uintptr_t>(quantized_data) & 3u) == 0 && aligned16(out),
             "nf4_dequantize: quantized_data must be 4-byte aligned and out 16-byte aligned");
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  const int64_t n_dwords = numel / 8;
  const int l2dpb = log2_exact(block_size / 8);
  const int l2sb = is_pow2(scaler_block_size) ? log2_exact(scaler_block_size) : -1;
  const int64_t bytes_moved = numel / 2 + numel * (dtype == TTAMD_BF16 ? 2 : 4);
  const int dw = bytes_moved <= kDequantCacheResidentBytes ? 8 : 4;
  const int64_t per_wg = 256 * dw;
  const int64_t grid = (n_dwords + per_wg - 1) / per_wg;
  TT_REQUIRE(grid < (int64_t(1) << 31), "nf4_dequantize: tensor too large for one launch");
  auto launch = [&](auto kernel) {
    kernel<<<dim3((unsigned)grid), dim3(256), 0, s>>>(reinterpret_cast<const uint32_t*>(quantized_data), quantized_scalers,
                                                      quantization_factor, scaler_mean, n_dwords, l2dpb, scaler_block_size,
                                                      l2sb, numel / block_size, out);
  };
  if (dtype == TTAMD_BF16) {
    if (dw == 8) launch(nf4_dequantize_kernel<true, 8>); else launch(nf4_dequantize_kernel<true, 4>);
  } else {
    if (dw == 8) launch(nf4_dequantize_kernel<false, 8>); else launch(nf4_dequantize_kernel<false, 4>);
  }
  return check_launch("nf4_dequantize");
}
