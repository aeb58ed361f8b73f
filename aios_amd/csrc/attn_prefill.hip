// Varlen causal paged prefill (kernel (b)), also used for cross-keystroke
// LCP extension (a few new tokens against a cached prefix).
//
// One workgroup owns (request r, kv-head h, query tile): q_tile consecutive
// query tokens times the G query heads of h, packed into the 128 MFMA rows
// (row = token * G + head), and streams KV positions [0, cached_len +
// last token of the tile] of r through the tile engine with the offset
// causal mask key_pos <= cached_len + i (python/aios/attention/
// flashinfer.py:67-80).  Tiles entirely below the diagonal are unmasked; the
// mask only bites in the last sub-tiles.  Batches with few tiles split each
// tile's KV range over several workgroups (prefill_split_kernel below).
#include "engine.hpp"

namespace aios {

template <int D>
__global__ __launch_bounds__(kEngineThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_kernel(PrefillArgs a) {
  __shared__ __align__(16) uint8_t lds[KVTile<D>::LDS_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int G = a.group;
  // One flat grid: consecutive workgroups take consecutive kv-heads (the
  // hardware deals workgroups round-robin to the XCDs, so with 8 kv-heads
  // each XCD's L2 holds one head's K/V, read by all of that head's query
  // tiles), and the query tiles run from the last (the longest causal KV
  // range) to the first, so the short tiles fill in behind the long ones
  // instead of the long ones forming the tail.
  const int flat = blockIdx.x;
  const int h = flat % a.num_kv_heads;
  const int rest = flat / a.num_kv_heads;
  const int r = rest % a.batch;
  const int qt = a.q_tiles - 1 - rest / a.batch;
  const int q_start = a.cu_q[r];
  const int q_len = a.cu_q[r + 1] - q_start;
  if (qt * a.q_tile >= q_len) return;
  const int kv_base = a.cu_k[r];
  const int kv_len = a.cu_k[r + 1] - kv_base;
  const int cached = kv_len - q_len;
  const int q_hi = min(q_len, (qt + 1) * a.q_tile);

  TileEngine32<D, true> eng;
  // The lane's query row (lanes l and l ^ 32 share it).
  const int m = wave * 32 + (lane & 31);
  const int i = qt * a.q_tile + m / G;
  const int g = m - (m / G) * G;
  const bool ok = (m < a.q_tile * G) && (i < q_len);
  const bf16* qr = a.q + (int64_t)(q_start + i) * a.q_tok_stride + (int64_t)(h * G + g) * D;
  const int64_t out_off = ((int64_t)(q_start + i) * a.num_qo_heads + (h * G + g)) * D;
  eng.limit = cached + i;
  eng.min_limit = cached + qt * a.q_tile;
  // A wavefront whose 32 rows are all past the tile's tokens only helps
  // stream K/V; it skips the math.
  const int m0 = wave * 32;
  const bool active = m0 < a.q_tile * G && qt * a.q_tile + m0 / G < q_len;
  eng.run(lds, reinterpret_cast<const uint8_t*>(a.k_cache) + (int64_t)h * D * 2,
          reinterpret_cast<const uint8_t*>(a.v_cache) + (int64_t)h * D * 2, a.kv_tok_stride * 2,
          a.num_pages, a.indices + kv_base, 0, min(kv_len, cached + q_hi), a.scale_log2,
          [&] { eng.load_q(qr, ok); }, active);

  if (!ok) return;
  const float l_tot = eng.l_run;
  const float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
  bf16* po = a.out + out_off + 4 * (lane >> 5);
  // o[nt] register 4j + i: dim 32 nt + 8j + 4h + i of the lane's row
#pragma unroll
  for (int nt = 0; nt < D / 32; ++nt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      uint2 packed;
      packed.x = pack_bf16x2(eng.o[nt][4 * j] * inv, eng.o[nt][4 * j + 1] * inv);
      packed.y = pack_bf16x2(eng.o[nt][4 * j + 2] * inv, eng.o[nt][4 * j + 3] * inv);
      *reinterpret_cast<uint2*>(po + nt * 32 + 8 * j) = packed;
    }
}

// ---------------------------------------------------------------------------
// KV split.  One workgroup per (tile, kv-head) leaves the chip idle when the
// batch has few tiles (an extension of a cached prefix has one: 8 workgroups
// on 256 compute units, each streaming the whole prefix) or when the longest
// of few causal tiles outlasts the others.  Here a workgroup owns one part of
// a tile's KV range and writes the part's fp32 state (o, m, l);
// prefill_combine_kernel merges them.  Bound: a part's latency chain (page
// ids, gathers, one sub-tile's math per wavefront, merge) and the states'
// traffic.  Measured per layer on MI355X (graph replay), one workgroup per
// tile -> split (main launch + combine): 6 tokens against 4,099 positions,
// 32q/8kv x 128: 94.7 -> 16.2 us; 100 against 4,100: 102 -> 28 us; a
// 2,048-token prompt, 16q/8kv x 128: 57 -> 42 us.
//
// A tile of at most 64 rows fills one or two of the four 32-row wavefront
// tiles; its wavefronts then also share the part's sub-tiles (all resident
// in the LDS ring): with one row tile wavefront w takes sub-tile w, with two
// wavefronts w and w + 2 take the two halves of row tile w, and the states
// of a row tile are merged through the ring once every sub-tile is consumed.

// The parts of a tile of `rows` MFMA rows over kv positions: one, written
// directly, where it has more rows than the plan gave each part room for
// (lengths on the device other than the planned ones).
__device__ __forceinline__ PrefillParts tile_parts(const PrefillArgs& a, int rows, int kv) {
  return prefill_parts(kv, a.part_sub, rows <= a.part_rows ? a.n_parts : 1);
}

// Dims 8 dg .. 8 dg + 7 of row m in a part's o.
template <int D>
__device__ __forceinline__ int64_t prefill_part_o(const PrefillArgs& a, int64_t part, int dg, int m) {
  return ((part * (D / 8) + dg) * a.part_rows + m) * 8;
}

template <int D>
__global__ __launch_bounds__(kEngineThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) void prefill_split_kernel(PrefillArgs a) {
  using T = KVTile<D, true>;
  __shared__ __align__(16) uint8_t lds[T::LDS_BYTES];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int G = a.group;
  // Consecutive workgroups: consecutive kv-heads (as above), then the tiles,
  // longest first, then the parts.  (The parts must not come before the
  // tiles: short tiles lack the later ones, and workgroup i runs on XCD i %
  // 8, so with kv-heads x parts a multiple of 8 some XCDs would get only
  // missing parts.)
  const int flat = blockIdx.x;
  const int h = flat % a.num_kv_heads;
  int rest = flat / a.num_kv_heads;
  const int r = rest % a.batch;
  rest /= a.batch;
  const int qt = a.q_tiles - 1 - rest % a.q_tiles;
  const int s = rest / a.q_tiles;
  const int q_start = a.cu_q[r];
  const int q_len = a.cu_q[r + 1] - q_start;
  if (qt * a.q_tile >= q_len) return;
  const int kv_base = a.cu_k[r];
  const int kv_len = a.cu_k[r + 1] - kv_base;
  const int cached = kv_len - q_len;
  const int q_hi = min(q_len, (qt + 1) * a.q_tile);
  const int kv_hi = min(kv_len, cached + q_hi);
  const int rows = (q_hi - qt * a.q_tile) * G;
  const PrefillParts pp = tile_parts(a, rows, kv_hi);
  if (s >= pp.n) return;
  const int kv_begin = s * pp.per * kSubTok;
  const int kv_end = min(kv_hi, kv_begin + pp.per * kSubTok);

  // Wavefront -> (row tile, share of the sub-tiles).
  const int nr = rows <= 32 ? 1 : rows <= 64 ? 2 : 4;
  const int rt = wave & (nr - 1);
  const int share = nr == 4 ? 0 : nr == 2 ? wave >> 1 : wave;
  const int m = rt * 32 + (lane & 31);
  const int i = qt * a.q_tile + m / G;
  const int g = m - (m / G) * G;
  const bool ok = m < rows;
  const int hl = lane >> 5;
  const bf16* qr = a.q + (int64_t)(q_start + i) * a.q_tok_stride + (int64_t)(h * G + g) * D;
  const uint8_t* kc = reinterpret_cast<const uint8_t*>(a.k_cache) + (int64_t)h * D * 2;
  const uint8_t* vc = reinterpret_cast<const uint8_t*>(a.v_cache) + (int64_t)h * D * 2;

  TileEngine32<D, true> eng;
  eng.limit = cached + i;
  eng.min_limit = cached + qt * a.q_tile;
  const int64_t slot = ((int64_t)r * a.q_tiles + qt) * a.num_kv_heads + h;
  const int64_t part = slot * a.n_parts + s;
  bf16* out_row = a.out + ((int64_t)(q_start + i) * a.num_qo_heads + (h * G + g)) * D;

  if (nr == 4) {
    eng.run(lds, kc, vc, a.kv_tok_stride * 2, a.num_pages, a.indices + kv_base, kv_begin, kv_end,
            a.scale_log2, [&] { eng.load_q(qr, ok); }, rt * 32 < rows);
    if (!ok) return;
    if (pp.n == 1) {
      const float inv = eng.l_run > 0.f ? 1.f / eng.l_run : 0.f;
#pragma unroll
      for (int nt = 0; nt < D / 32; ++nt)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint2 packed;
          packed.x = pack_bf16x2(eng.o[nt][4 * j] * inv, eng.o[nt][4 * j + 1] * inv);
          packed.y = pack_bf16x2(eng.o[nt][4 * j + 2] * inv, eng.o[nt][4 * j + 3] * inv);
          *reinterpret_cast<uint2*>(out_row + nt * 32 + 8 * j + 4 * hl) = packed;
        }
      return;
    }
#pragma unroll
    for (int nt = 0; nt < D / 32; ++nt)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        *reinterpret_cast<f32x4*>(a.part_o + prefill_part_o<D>(a, part, nt * 4 + j, m) + 4 * hl) =
            f32x4{eng.o[nt][4 * j], eng.o[nt][4 * j + 1], eng.o[nt][4 * j + 2],
                  eng.o[nt][4 * j + 3]};
    if (hl == 0) a.part_ml[part * a.part_rows + m] = make_float2(eng.m_run, eng.l_run);
    return;
  }

  // Few rows: the sub-tiles of a part of at most kRing are all in LDS before
  // the math.  (A longer part -- more KV positions than the plan was built
  // for -- streams through the ring, share 0 of each row tile computing.)
  eng.reset();
  const auto lo = eng.lane_offsets(lds);
  const int ng = 4 / nr;
  stream_kv<T, 0, true>(
      lds, kc, vc, a.kv_tok_stride * 2, a.num_pages, a.indices + kv_base, kv_begin, kv_end,
      [&] { eng.load_q(qr, ok); },
      [&](uint32_t sb, int kv0) {
        if (share == 0) eng.compute_at(lo, sb, kv0, kv_end, a.scale_log2);
      },
      true,
      [&](auto&& wait_sub, int n_sub) {
        wait_sub(kRing - 1);
        for (int it = share; it < n_sub; it += ng)
          eng.compute_at(lo, (uint32_t)(it * T::SUB_BYTES), kv_begin + it * kSubTok, kv_end,
                         a.scale_log2);
      });

  // Merge: each wavefront's o to its own sub-tile's worth of the ring
  // ([D / 8][32 rows][8] fp32 is exactly one sub-tile), (m, l) behind it.
  static_assert(T::SUB_BYTES == 32 * D * 4, "a row tile's fp32 o fills one sub-tile");
  lds_barrier();  // every wavefront is done with K/V
  float* so = reinterpret_cast<float*>(lds + wave * T::SUB_BYTES);
  float2* sml = reinterpret_cast<float2*>(lds + T::RING_BYTES);  // [wave][32]
#pragma unroll
  for (int nt = 0; nt < D / 32; ++nt)
#pragma unroll
    for (int j = 0; j < 4; ++j)
      *reinterpret_cast<f32x4*>(so + ((nt * 4 + j) * 32 + (lane & 31)) * 8 + 4 * hl) =
          f32x4{eng.o[nt][4 * j], eng.o[nt][4 * j + 1], eng.o[nt][4 * j + 2], eng.o[nt][4 * j + 3]};
  if (hl == 0) sml[wave * 32 + (lane & 31)] = make_float2(eng.m_run, eng.ol[0]);
  __syncthreads();
  const int nrow = nr * 32;
  for (int e = threadIdx.x; e < nrow * (D / 8); e += kEngineThreads) {
    const int dg = e / nrow;
    const int row = e - dg * nrow;
    if (row >= rows) continue;
    const int w0 = row >> 5;  // the row tile; its shares are wavefronts w0 + k * nr
    float mx = kNegInf;
    for (int w = w0; w < 4; w += nr) mx = vmax(mx, sml[w * 32 + (row & 31)].x);
    const float mu = mx == kNegInf ? 0.f : mx;
    f32x4 acc0 = f32x4{0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
    float l = 0.f;
    for (int w = w0; w < 4; w += nr) {
      const float2 ml = sml[w * 32 + (row & 31)];
      const float f = fast_exp2(ml.x - mu);
      l += ml.y * f;
      const f32x4* po = reinterpret_cast<const f32x4*>(lds + w * T::SUB_BYTES) +
                        (dg * 32 + (row & 31)) * 2;
      acc0 += po[0] * f;
      acc1 += po[1] * f;
    }
    if (pp.n == 1) {
      const float inv = l > 0.f ? 1.f / l : 0.f;
      acc0 *= inv;
      acc1 *= inv;
      const int qi = q_start + qt * a.q_tile + row / G;
      bf16* po = a.out + ((int64_t)qi * a.num_qo_heads + h * G + row % G) * D + dg * 8;
      *reinterpret_cast<uint4*>(po) =
          make_uint4(pack_bf16x2(acc0[0], acc0[1]), pack_bf16x2(acc0[2], acc0[3]),
                     pack_bf16x2(acc1[0], acc1[1]), pack_bf16x2(acc1[2], acc1[3]));
    } else {
      f32x4* po = reinterpret_cast<f32x4*>(a.part_o + prefill_part_o<D>(a, part, dg, row));
      po[0] = acc0;
      po[1] = acc1;
      if (dg == 0) a.part_ml[part * a.part_rows + row] = make_float2(mx, l);
    }
  }
}

// Merges the parts of each row: out = sum_j 2^(m_j - m) o_j / sum_j 2^(m_j -
// m) l_j, m = max_j m_j.  A wavefront takes RB rows, one (row, 8-dim group)
// per lane, so that few-row tiles still spread over many workgroups and a
// part's loads of a wavefront are whole 128-byte lines; NW wavefronts share a
// row block's parts, NB of them in flight per wavefront.
template <int D, int NW, int NB>
__global__ __launch_bounds__(NW * 64) void prefill_combine_kernel(PrefillArgs a, int32_t row_blocks) {
  constexpr int DG = D / 8;
  constexpr int RB = 64 / DG;
  const int lane = threadIdx.x & 63;
  const int wave = threadIdx.x >> 6;
  const int flat = blockIdx.x;
  const int h = flat % a.num_kv_heads;
  int rest = flat / a.num_kv_heads;
  const int rb = rest % row_blocks;
  rest /= row_blocks;
  const int r = rest % a.batch;
  const int qt = a.q_tiles - 1 - rest / a.batch;
  const int q_start = a.cu_q[r];
  const int q_len = a.cu_q[r + 1] - q_start;
  if (qt * a.q_tile >= q_len) return;
  const int kv_len = a.cu_k[r + 1] - a.cu_k[r];
  const int q_hi = min(q_len, (qt + 1) * a.q_tile);
  const int rows = (q_hi - qt * a.q_tile) * a.group;
  const PrefillParts pp = tile_parts(a, rows, min(kv_len, kv_len - q_len + q_hi));
  if (pp.n == 1 || rb * RB >= rows) return;  // (uniform)
  const int dg = lane % DG;
  const int m = rb * RB + lane / DG;
  const bool ok = lane < RB * DG && m < rows;
  const int64_t part0 = (((int64_t)r * a.q_tiles + qt) * a.num_kv_heads + h) * a.n_parts;
  const f32x4* po =
      reinterpret_cast<const f32x4*>(a.part_o + prefill_part_o<D>(a, part0, dg, ok ? m : 0));
  const int64_t part_stride = (int64_t)D / 4 * a.part_rows;
  const float2* ml = a.part_ml + part0 * a.part_rows + (ok ? m : 0);
  float mx = kNegInf, l = 0.f;
  f32x4 acc0 = f32x4{0.f, 0.f, 0.f, 0.f}, acc1 = acc0;
  for (int j0 = wave; j0 < pp.n; j0 += NW * NB) {
    float2 w[NB];
    f32x4 x0[NB], x1[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const int j = j0 + k * NW;
      if (j < pp.n) {  // (uniform per wavefront)
        w[k] = ml[(int64_t)j * a.part_rows];
        x0[k] = po[j * part_stride];
        x1[k] = po[j * part_stride + 1];
      } else {
        w[k] = make_float2(kNegInf, 0.f);
        x0[k] = x1[k] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
    float mb = mx;
#pragma unroll
    for (int k = 0; k < NB; ++k) mb = vmax(mb, w[k].x);
    const float mu = mb == kNegInf ? 0.f : mb;
    const float f0 = fast_exp2(mx - mu);
    acc0 *= f0;
    acc1 *= f0;
    l *= f0;
#pragma unroll
    for (int k = 0; k < NB; ++k) {
      const float f = fast_exp2(w[k].x - mu);
      l += w[k].y * f;
      acc0 += x0[k] * f;
      acc1 += x1[k] * f;
    }
    mx = mb;
  }
  if constexpr (NW > 1) {
    __shared__ f32x4 so[2][NW][64];
    __shared__ float2 sml[NW][64];
    so[0][wave][lane] = acc0;
    so[1][wave][lane] = acc1;
    sml[wave][lane] = make_float2(mx, l);
    __syncthreads();
    if (wave > 0) return;
#pragma unroll
    for (int w = 1; w < NW; ++w) mx = vmax(mx, sml[w][lane].x);
    const float mu = mx == kNegInf ? 0.f : mx;
    l = 0.f;
    acc0 = acc1 = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < NW; ++w) {
      const float2 s = sml[w][lane];
      const float f = fast_exp2(s.x - mu);
      l += s.y * f;
      acc0 += so[0][w][lane] * f;
      acc1 += so[1][w][lane] * f;
    }
  }
  if (!ok) return;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  acc0 *= inv;
  acc1 *= inv;
  const int qi = q_start + qt * a.q_tile + m / a.group;
  bf16* out = a.out + ((int64_t)qi * a.num_qo_heads + h * a.group + m % a.group) * D + dg * 8;
  *reinterpret_cast<uint4*>(out) =
      make_uint4(pack_bf16x2(acc0[0], acc0[1]), pack_bf16x2(acc0[2], acc0[3]),
                 pack_bf16x2(acc1[0], acc1[1]), pack_bf16x2(acc1[2], acc1[3]));
}

template <int D>
static hipError_t launch_split_d(const PrefillArgs& a, hipStream_t s) {
  const int tiles = a.q_tiles * a.num_kv_heads * a.batch;
  if (tiles == 0) return hipSuccess;
  hipLaunchKernelGGL(prefill_split_kernel<D>, dim3(tiles * a.n_parts), dim3(kEngineThreads), 0, s,
                     a);
  if (a.n_parts > 1) {
    constexpr int RB = 64 / (D / 8);
    const int row_blocks = (a.part_rows + RB - 1) / RB;
    const dim3 grid(tiles * row_blocks);
    if (a.n_parts <= 4)
      hipLaunchKernelGGL((prefill_combine_kernel<D, 1, 4>), grid, dim3(64), 0, s, a, row_blocks);
    else
      hipLaunchKernelGGL((prefill_combine_kernel<D, 4, 8>), grid, dim3(256), 0, s, a, row_blocks);
  }
  return hipGetLastError();
}

hipError_t launch_prefill_split(int D, const PrefillArgs& a, hipStream_t s) {
  switch (D) {
    case 64: return launch_split_d<64>(a, s);
    case 96: return launch_split_d<96>(a, s);
    case 128: return launch_split_d<128>(a, s);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_prefill(int D, int NW, const PrefillArgs& a, int q_tiles, int batch,
                          hipStream_t s) {
  (void)NW;
  const dim3 grid(q_tiles * a.num_kv_heads * batch);
  if (q_tiles == 0 || batch == 0) return hipSuccess;
  switch (D) {
    case 64: hipLaunchKernelGGL(prefill_kernel<64>, grid, dim3(kEngineThreads), 0, s, a); break;
    case 96: hipLaunchKernelGGL(prefill_kernel<96>, grid, dim3(kEngineThreads), 0, s, a); break;
    case 128: hipLaunchKernelGGL(prefill_kernel<128>, grid, dim3(kEngineThreads), 0, s, a); break;
    default: return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace aios
