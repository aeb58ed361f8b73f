// Few-row projections y[M, N] = x[M, K] W[N, K]^T that stream their weights
// past resident rows: 17 to 64 rows, and the K of fewer rows for which that
// measured faster than gemm_skinny.hip (rows_form in api.hip; bf16 in, fp32
// accumulate, bf16 out).
//
// What bounds a few-row projection is how fast a compute unit takes in
// operands: about 25-30 bytes per nanosecond (measured, HBM and L2 alike), and
// in a kernel where every 16-column tile loads its rows again the rows are
// most of it (24 rows are 1.5 times a tile's weight bytes).  Here one
// workgroup per compute unit keeps its rows' fragments in registers (KS
// K-steps of 32 for each of MT 16-row tiles and wavefront) and walks the
// column tiles t, t + C, ..., the next tile's weights in flight while the
// current one is multiplied; its eight wavefronts split K and the tile is
// summed through LDS.  A K that does not fit the registers, or few column
// tiles with a long K, is split over `splits` groups of C workgroups, whose
// fp32 partial tiles rows_reduce_kernel adds.
//
// Measured on MI355X with weights from HBM (graph replay; gemm_skinny.hip's
// generic loop before -> here): 24 rows, N x K 151936 x 2560 311 -> 154 us
// (5.0 TB/s of weights), 6144 x 2560 19.4 -> 12, 2 x 9728 x 2560 with SiLU
// 40 -> 24, 2560 x 4096 19.2 -> 9.7 (4 splits), 2560 x 9728 42 -> 15.7 (8
// splits); 64 rows, 2560 x 9728 60 -> 20; 8 rows, 151936 x 2560 192 -> 141.
//
// With SILU (gate rows, then up rows in W: the merged gate/up projection) a
// tile is 8 gate columns and the 8 matching up columns, so the pair meets in
// one wavefront.  The residual-add RMSNorm is not folded in here: every
// workgroup would normalise all rows (24 rows x 6144 x 2560: 24 us against 15
// with the norm as its own launch; 24 x 4096 x 1024: 8.5 against 8.0).
#include "kernels.hpp"

namespace aios {
namespace {

constexpr int kRowsThreads = 512;  // one workgroup per compute unit
constexpr int kRowsWaves = kRowsThreads / 64;
constexpr int kRowsMaxSplits = 8;
constexpr int kRsrcWord3 = 0x00020000;     // raw buffer descriptor word 3 (32-bit data format)
constexpr int kOut = (int)0x80000000;      // an offset past every buffer's range: reads zero,
                                           // writes nothing, touches no memory
constexpr int64_t kRange = 0x7fffffff;

typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rows_buffer(const void* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)kRange, kRsrcWord3);
}
__device__ __forceinline__ bf16x8 rows_load(__amdgpu_buffer_rsrc_t r, int voff, int soff) {
  return __builtin_bit_cast(bf16x8, __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, 0));
}

// The register steps built for a row tile count, 0 when the K steps per
// wavefront do not fit, and the steps that every wavefront has of KS
// (its share is `need` or one less).
int rows_ks(int mt, int need, bool silu) {
  if (need <= 3) return 3;
  if (need <= 4) return 4;
  if (need <= 6) return silu ? 8 : 6;
  if (need <= 8) return 8;
  if (need <= 10) return 10;
  if (need <= 12 && mt <= 2 && !silu) return 12;
  return 0;
}
constexpr int rows_whole(int ks, bool silu) {
  return ks == 3 ? 1 : ks == 4 ? 3 : ks == 8 && silu ? 4 : ks - 2;
}

// NH = 2: a tile's weights in two halves, so that two buffers of KS / 2 steps
// serve where MT * KS fragments leave no room for two of KS.
// Register use at two wavefronts per SIMD (256): 4 * (MT * KS + 2 * KS / NH)
// for the fragments, at most 240.
template <int MT, int KS, int NH, bool SILU, bool PART>
__global__ __launch_bounds__(kRowsThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void rows_gemm_kernel(
    const bf16* __restrict__ x, const bf16* __restrict__ w, bf16* __restrict__ y, int32_t x_stride,
    int32_t w_stride, int32_t y_stride, int32_t M, int32_t K, int32_t N, int32_t splits,
    float* __restrict__ part) {
  static_assert(!PART || !SILU, "partial tiles are sums only");
  static_assert(NH <= 2 && KS % NH == 0, "one or two halves");
  constexpr int KH = KS / NH;
  constexpr int NC = SILU ? 8 : 16;  // output columns of a tile
  __shared__ f32x4 red[2][kRowsWaves][MT][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int l16 = lane & 15;
  const int lg = lane >> 4;
  const int split = PART ? blockIdx.x % splits : 0;
  const int C = PART ? gridDim.x / splits : gridDim.x;
  int t = PART ? blockIdx.x / splits : blockIdx.x;
  const int tiles = N / NC;
  // This wavefront's K steps s0 .. s0 + ns - 1 (1 <= ns <= KS: the launcher's
  // choice of splits); steps past them read zeros on both sides (weights read
  // there would meet the zero x, but 0 * Inf is NaN).
  const int T = K >> 5;
  const int unit = split * kRowsWaves + wave, units = (PART ? splits : 1) * kRowsWaves;
  const int s0 = unit * T / units;
  const int ns = (unit + 1) * T / units - s0;
  const __amdgpu_buffer_rsrc_t rw = rows_buffer(w);
  const int wrow = SILU ? (l16 < 8 ? l16 : N + l16 - 8) : l16;
  const int wvoff = (wrow * w_stride + lg * 8) * 2;
  const int tile_b = NC * w_stride * 2;
  auto load = [&](bf16x8 (&f)[KH], int tile, int half) {
    // (the count made opaque for each tile: hoisted out of the loop, the steps'
    // offsets would take a register each)
    int n = ns;
    asm volatile("" : "+s"(n));
#pragma unroll
    for (int u = 0; u < KH; ++u) {
      const int step = half * KH + u;
      const bool pad = step >= rows_whole(KS, SILU) && step >= n;
      f[u] = rows_load(rw, pad ? kOut : wvoff, tile * tile_b + (s0 + (pad ? 0 : step)) * 64);
    }
  };
  bf16x8 wa[KH], wb[KH];
  load(wa, t, 0);

  // The rows: fragment u of row tile mt is K step s0 + u of row 16 mt + l16.
  bf16x8 xb[MT][KS];
  {
    const __amdgpu_buffer_rsrc_t rx = rows_buffer(x);
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int m = mt * 16 + l16;
      const int off = m < M ? (m * x_stride + lg * 8) * 2 : kOut;
#pragma unroll
      for (int u = 0; u < KS; ++u)
        xb[mt][u] = rows_load(rx, u < ns ? off : kOut, (s0 + min(u, ns - 1)) * 64);
    }
  }
  f32x4 acc[MT];
  auto mma = [&](const bf16x8 (&f)[KH], int half) {
#pragma unroll
    for (int u = 0; u < KH; ++u)
#pragma unroll
      for (int mt = 0; mt < MT; ++mt)
        acc[mt] = mfma16x16x32(f[u], xb[mt][half * KH + u],
                               half == 0 && u == 0 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[mt]);
  };
  const __amdgpu_buffer_rsrc_t ry =
      rows_buffer(PART ? (const void*)(part + (int64_t)split * M * N) : (const void*)y);
  // Sums the wavefronts' tiles (acc[mt][i]: row 16 mt + l16, W row lg * 4 + i)
  // and stores: wavefront mt takes row tile mt.  The stores carry no branch
  // per lane (rows past M get an offset out of range), so the next tile's
  // loads stay in flight past them; the parity of red orders its reuse two
  // barriers apart.
  auto finish = [&](int tile, int par) {
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) red[par][wave][mt][lane] = acc[mt];
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    asm volatile("s_barrier" ::: "memory");
    if (wave >= MT) return;
    f32x4 v = red[par][0][wave][lane];
#pragma unroll
    for (int q = 1; q < kRowsWaves; ++q) v += red[par][q][wave][lane];
    const int m = wave * 16 + l16;
    if constexpr (PART) {
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), ry,
                                             m < M ? (m * N + lg * 4) * 4 : kOut, tile * NC * 4, 0);
    } else {
      bool ok = m < M;
      if constexpr (SILU) {
        // lanes lg 0, 1: gate columns 4 lg ..; the up columns are 32 lanes on
        ok = ok && lg < 2;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const float up = round_bf16(__shfl_xor(v[i], 32));
          const float g = round_bf16(v[i]);
          v[i] = round_bf16(g / (1.f + expf(-g))) * up;
        }
      }
      const u32x2 o = {pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3])};
      __builtin_amdgcn_raw_buffer_store_b64(o, ry, ok ? (m * y_stride + lg * 4) * 2 : kOut,
                                            tile * NC * 2, 0);
    }
  };
  // Every load so far has landed before the loop: with loads of unknown
  // count pending at its header the compiler would wait for all of them in
  // every iteration.
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)
  int par = 0;
  while (true) {
    if constexpr (NH == 2) {
      load(wb, t, 1);
      mma(wa, 0);
      const int n = t + C;
      if (n >= tiles) {
        mma(wb, 1);
        finish(t, par);
        break;
      }
      load(wa, n, 0);
      mma(wb, 1);
      finish(t, par);
      t = n;
      par ^= 1;
    } else {
      int n = t + C;
      if (n >= tiles) {
        mma(wa, 0);
        finish(t, 0);
        break;
      }
      load(wb, n, 0);
      mma(wa, 0);
      finish(t, 0);
      t = n;
      n = t + C;
      if (n >= tiles) {
        mma(wb, 0);
        finish(t, 1);
        break;
      }
      load(wa, n, 0);
      mma(wb, 0);
      finish(t, 1);
      t = n;
    }
  }
}

// y = bf16(sum of the splits' partial products), in split order.
__global__ __launch_bounds__(256) void rows_reduce_kernel(const float* __restrict__ part,
                                                          bf16* __restrict__ y, int32_t splits,
                                                          int32_t M, int32_t N, int32_t y_stride) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  const int nq = N / 4;
  if (i >= M * nq) return;
  const int m = i / nq;
  const int n = (i - m * nq) * 4;
  const f32x4* p = reinterpret_cast<const f32x4*>(part + (int64_t)m * N + n);
  const int64_t step = (int64_t)M * N / 4;
  f32x4 v[kRowsMaxSplits];
#pragma unroll
  for (int s = 0; s < kRowsMaxSplits; ++s)
    v[s] = s < splits ? p[s * step] : f32x4{0.f, 0.f, 0.f, 0.f};
  f32x4 o = v[0];
#pragma unroll
  for (int s = 1; s < kRowsMaxSplits; ++s) o += v[s];
  *reinterpret_cast<uint2*>(y + (int64_t)m * y_stride + n) =
      make_uint2(pack_bf16x2(o[0], o[1]), pack_bf16x2(o[2], o[3]));
}

template <int MT, int KS, int NH = 1>
hipError_t launch_rows(const LinearArgs& a, bool silu, const RowsPlan& p, float* part,
                       hipStream_t stream) {
#define AIOS_ROWS(SILU, PART)                                                                    \
  hipLaunchKernelGGL((rows_gemm_kernel<MT, KS, NH, SILU, PART>), dim3((unsigned)p.grid),         \
                     dim3(kRowsThreads), 0, stream, a.x, a.w, a.y, (int32_t)a.x_stride,          \
                     (int32_t)a.w_stride, (int32_t)a.y_stride, a.M, a.K, (int32_t)a.N, p.splits, \
                     part)
  if (p.splits > 1) {
    AIOS_ROWS(false, true);
    const int64_t quads = (int64_t)a.M * (a.N / 4);
    hipLaunchKernelGGL(rows_reduce_kernel, dim3((unsigned)((quads + 255) / 256)), dim3(256), 0,
                       stream, part, a.y, p.splits, a.M, (int32_t)a.N, (int32_t)a.y_stride);
    return hipGetLastError();
  }
  if constexpr (KS != 6 && KS != 12) {
    if (silu) {
      AIOS_ROWS(true, false);
      return hipGetLastError();
    }
  }
  AIOS_ROWS(false, false);
#undef AIOS_ROWS
  return hipGetLastError();
}

template <int MT>
hipError_t launch_rows_mt(const LinearArgs& a, bool silu, const RowsPlan& p, float* part,
                          hipStream_t stream) {
  switch (p.ks) {
    case 3: return launch_rows<MT, 3>(a, silu, p, part, stream);
    case 4: return launch_rows<MT, 4>(a, silu, p, part, stream);
    case 6: return launch_rows<MT, 6>(a, silu, p, part, stream);
    case 8: return launch_rows<MT, 8>(a, silu, p, part, stream);
    case 10: return launch_rows<MT, 10, MT == 4 ? 2 : 1>(a, silu, p, part, stream);
    case 12:
      if constexpr (MT <= 2) return launch_rows<MT, 12>(a, silu, p, part, stream);
      break;
    default: break;
  }
  return hipErrorInvalidValue;
}

}  // namespace

// The split of K: the estimate below, in nanoseconds of the busiest compute
// unit, over the splits whose K steps fit the registers.  25 bytes per
// nanosecond taken in (its tiles' weights and its rows), 250 ns per tile
// (barrier, LDS sum, store), and for more than one split the second launch
// (3.5 us) and the partial tiles written and read (3 TB/s).  At 24 rows it
// takes 1 split for 6144 x 2560 (12 us, 2 splits 12.7), 6 for 2560 x 4096
// (9.6; 2 splits 10.9), 8 for 2560 x 9728 (15.7; 4 splits 17.7) and 4 for
// 1024 x 3072 (6.7 us; unsplit 9 in the eight-column skinny form).
bool rows_gemm_plan(int64_t M, int64_t N, int64_t K, bool silu, bool workspace, int cus,
                    RowsPlan* plan) {
  if (M < 1 || M > 64 || N < 16 || N % 16 != 0 || K < 256 || K % 32 != 0 || K > (1 << 20))
    return false;
  const int mt = (int)((M + 15) / 16);
  const int64_t T = K / 32, nc = silu ? 8 : 16, tiles = N / nc;
  double best = 0.0;
  plan->splits = 0;
  for (int s = 1; s <= (workspace && !silu ? kRowsMaxSplits : 1); ++s) {
    if (T < kRowsWaves * s) break;
    const int ks = rows_ks(mt, (int)((T + kRowsWaves * s - 1) / (kRowsWaves * s)), silu);
    if (ks == 0) continue;
    const int64_t C = tiles < cus / s ? tiles : cus / s;
    const int64_t walk = (tiles + C - 1) / C;
    double ns = (double)(walk * 16 + M) * (K / s) * 2 / 25.0 + 250.0 * walk;
    if (s > 1) ns += 3500.0 + (double)s * M * N * 8 / 3000.0;
    if (plan->splits == 0 || ns < best) {
      best = ns;
      plan->splits = s;
      plan->ks = ks;
      plan->grid = (int32_t)(C * s);
    }
  }
  if (plan->splits == 0) return false;
  plan->bytes = plan->splits > 1 ? (int64_t)plan->splits * M * N * 4 : 0;
  return plan->bytes < kRange;
}

hipError_t rows_gemm(const LinearArgs& a, bool silu, const RowsPlan& p, void* workspace, hipStream_t stream) {
  float* part = static_cast<float*>(workspace);
  switch ((a.M + 15) / 16) {
    case 1: return launch_rows_mt<1>(a, silu, p, part, stream);
    case 2: return launch_rows_mt<2>(a, silu, p, part, stream);
    case 3: return launch_rows_mt<3>(a, silu, p, part, stream);
    case 4: return launch_rows_mt<4>(a, silu, p, part, stream);
    default: return hipErrorInvalidValue;
  }
}

// Offsets inside each operand are 32-bit.
bool rows_gemm_fits(const LinearArgs& a, bool silu) {
  const int64_t w_rows = (silu ? 2 : 1) * a.N;
  return a.x_stride <= (1 << 23) && a.y_stride <= (1 << 23) &&
         w_rows * a.w_stride * 2 < kRange && a.N <= (1 << 23);
}

}  // namespace aios
