// Weight-streaming product of many rows (9..128), everything in registers:
// one workgroup per CU, four waves splitting its k range.
//
// Between the calls of up to 8 rows (which stay in a workgroup's LDS) and
// the prefill's 64 x 64 tiles a projection is still bound by its weights, but
// the direct path re-reads the whole activation matrix for every 16-column
// tile (64 rows: 200 MB beside gate/up's 100), and at 64 rows its ring is
// down to four slots.  Here a workgroup takes U output units
// (16-column tiles, or half pairs with GLU) at all MT row tiles, and each
// wave a quarter of the k range of all of them: a k step is U weight
// fragments and MT activation fragments, 1 KiB loads straight into MFMA
// operands, for U MT products.  No operand is shared between waves, so there
// is no LDS traffic and no barrier until the four waves' sums are added, in
// wave order, through LDS.  One wave per SIMD has 512 registers: the
// accumulators and a ring of RING k steps (32 to 91 KiB per wave, of which the
// 6-bit load counter lets 63 be in flight).
//
// Sums and order are those of the direct path at four waves (gemm_dev.h):
// the same bits.  gate/up at 64 rows 30.7 -> 22.5 us per launch (3.2 -> 4.4
// TB/s), at 13 rows 20.3 -> 19.3 (5.2 TB/s); what is left at many rows is the
// activations each workgroup streams through its CU's L1 beside the weights.
#include "gemm_dev.h"

namespace qdec {
namespace {

// Ring slots (k steps): what the accumulators leave of the registers of one
// wave per SIMD, or of two (ARGMAX).
constexpr int wide_ring(int mt, int u, bool two) {
  const int slots = ((two ? 216 : 400) - 4 * mt * u) / (4 * (mt + u));
  return slots > 16 ? 16 : slots;
}

// ARGMAX (the lm_head) has many more output tiles than one round takes, so
// two workgroups share a CU: one's first loads and last sums run beside the
// other's stream.  The keys are those of gemm_body.inc, first folded over the
// workgroup in LDS.
template <int MT, int U, uint32_t FLAGS>
__global__ void __launch_bounds__(256, (FLAGS & QDEC_ARGMAX) ? 2 : 1) wide_kernel(const GemmParams p) {
  constexpr bool GLU = (FLAGS & QDEC_GLU) != 0;
  constexpr bool RES = (FLAGS & QDEC_RES_OUT) != 0;
  constexpr bool ARG = (FLAGS & QDEC_ARGMAX) != 0;
  constexpr int RING = wide_ring(MT, U, ARG);
  static_assert(RING >= 3 && MT * U * 4096 <= 163840, "registers and LDS of one wave per SIMD");
  __shared__ __align__(16) float4 red[4][MT * U][64];  // [wave][accumulator][lane]
  __shared__ uint64_t s_key[ARG ? MT * 16 : 1];        // the workgroup's best of each row
  __shared__ uint32_t s_flag[1];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int S = p.ksplit, KS = p.KS, ksw = p.ksw, nmt = p.xt;
  const int part = blockIdx.x % S, g = blockIdx.x / S;
  const int T = GLU ? p.n >> 3 : p.n >> 4;  // units
  const int G = gridDim.x / S;
  const int u0 = (int)((int64_t)g * T / G), nu = (int)((int64_t)(g + 1) * T / G) - u0;

  // Unit u: a weight tile; with GLU half pair h: columns 8h .. 8h+7 of gate
  // (operand rows 0..7) and up (rows 8..15).
  const int k0 = part * (KS / S) + wave * ksw;
  const char *wq[U];
#pragma unroll
  for (int u = 0; u < U; ++u) {
    const int unit = u0 + min(u, nu - 1);  // a unit past the last repeats it and is not stored
    const size_t tile = GLU ? unit >> 1 : unit;
    wq[u] = reinterpret_cast<const char *>(p.w) + (tile * KS + k0) * 1024 + (GLU ? (unit & 1) * 128 : 0);
  }
  const uint32_t xoff = lane * 16;
  const uint32_t woff = GLU ? (col < 8 ? 0u : (uint32_t)p.up_tiles * KS * 1024u) + (col & 7) * 16 + grp * 256 : xoff;
  const char *xq = reinterpret_cast<const char *>(p.x) + (size_t)k0 * nmt * 1024;

  f32x4_t acc[U][MT];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < MT; ++t) acc[u][t] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  uint4 w[RING][U], x[RING][MT];
  auto load = [&](int r, int i) {  // k step i into slot r
#pragma unroll
    for (int t = 0; t < MT; ++t) x[r][t] = *reinterpret_cast<const uint4 *>(xq + ((size_t)i * nmt + t) * 1024 + xoff);
#pragma unroll
    for (int u = 0; u < U; ++u) w[r][u] = ldw(reinterpret_cast<const uint4 *>(wq[u] + (size_t)i * 1024 + woff));
  };
  auto mma = [&](int r) {
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int t = 0; t < MT; ++t) acc[u][t] = mfma16x16x32(w[r][u], x[r][t], acc[u][t]);
  };
#pragma unroll
  for (int r = 0; r < RING; ++r) load(r, min(r, ksw - 1));
  int i = 0;
  for (; i + 2 * RING <= ksw; i += RING) {
#pragma unroll
    for (int r = 0; r < RING; ++r) {
      mma(r);
      load(r, i + RING + r);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the last RING .. 2 RING - 1 steps (or all of a shorter range)
#pragma unroll
  for (int r = 0; r < RING; ++r) {
    if (i + r < ksw) mma(r);
    if (i + RING + r < ksw) load(r, i + RING + r);
  }
#pragma unroll
  for (int r = 0; r < RING - 1; ++r)
    if (i + RING + r < ksw) mma(r);

  // ---- the four waves in order: wave v adds up accumulators v, v + 4, ...
  if constexpr (ARG) {
    if (threadIdx.x < MT * 16) s_key[threadIdx.x] = 0ull;
  }
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int t = 0; t < MT; ++t)
      red[wave][u * MT + t][lane] = make_float4(acc[u][t][0], acc[u][t][1], acc[u][t][2], acc[u][t][3]);
  __syncthreads();
  for (int f = wave; f < nu * MT; f += 4) {
    const int u = f / MT, t = f - u * MT, unit = u0 + u;
    const int m = t * 16 + col;
    float4 s = red[0][f][lane];
#pragma unroll
    for (int v = 1; v < 4; ++v) {
      const float4 r = red[v][f][lane];
      s.x += r.x; s.y += r.y; s.z += r.z; s.w += r.w;
    }
    if constexpr (ARG) {
      const int n0 = unit * 16 + grp * 4;
      const float v4[4] = {rbf(s.x), rbf(s.y), rbf(s.z), rbf(s.w)};
      if (p.out && m < p.rows)
        *reinterpret_cast<uint2 *>(reinterpret_cast<uint16_t *>(p.out) + (size_t)m * p.n + n0) =
            make_uint2(pack2(v4[0], v4[1]), pack2(v4[2], v4[3]));
      float bv = -__builtin_huge_valf();
      int bi = 0x7fffffff;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (v4[e] > bv) {
          bv = v4[e];
          bi = n0 + e;
        }
      if (m < p.rows)
        __hip_atomic_fetch_max(&s_key[m], argmax_key(bv, bi), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
    } else if constexpr (GLU) {
      // lanes 32..63 hold the up columns of lanes 0..31's gate columns
      const float4 up = make_float4(shfl_xor(s.x, 32), shfl_xor(s.y, 32), shfl_xor(s.z, 32), shfl_xor(s.w, 32));
      if (m >= p.rows || grp >= 2) continue;
      const float g4[4] = {rbf(s.x), rbf(s.y), rbf(s.z), rbf(s.w)}, u4[4] = {rbf(up.x), rbf(up.y), rbf(up.z), rbf(up.w)};
      float o4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o4[e] = swiglu(g4[e], u4[e]);
      const int n0 = unit * 8 + grp * 4;
      uint16_t *out = reinterpret_cast<uint16_t *>(p.out);
      *reinterpret_cast<uint2 *>(p.ofrag ? out + frag_off(m, n0, p.ofrag) : out + (size_t)m * p.n + n0) =
          make_uint2(pack2(o4[0], o4[1]), pack2(o4[2], o4[3]));
    } else {
      if (m >= p.rows) continue;
      const int n0 = unit * 16 + grp * 4;
      if (RES && p.parts_out) {
        *reinterpret_cast<float4 *>(p.parts_out + ((size_t)part * p.rows + m) * p.n + n0) = s;
      } else if constexpr (RES) {
        uint16_t *rp = reinterpret_cast<uint16_t *>(p.res) + (size_t)m * p.n + n0;
        const uint2 r = *reinterpret_cast<const uint2 *>(rp);
        *reinterpret_cast<uint2 *>(rp) = make_uint2(pack2(lo16(r.x) + rbf(s.x), hi16(r.x) + rbf(s.y)),
                                                    pack2(lo16(r.y) + rbf(s.z), hi16(r.y) + rbf(s.w)));
      } else {
        uint16_t *out = reinterpret_cast<uint16_t *>(p.out);
        *reinterpret_cast<uint2 *>(p.ofrag ? out + frag_off(m, n0, p.ofrag) : out + (size_t)m * p.n + n0) =
            make_uint2(pack2(s.x, s.y), pack2(s.z, s.w));
      }
    }
  }
  if constexpr (ARG) {
    uint64_t *keys = reinterpret_cast<uint64_t *>(p.counters + 2);  // [rows][kArgSlots]
    __syncthreads();
    if ((int)threadIdx.x < p.rows)
      __hip_atomic_fetch_max(keys + (size_t)threadIdx.x * kArgSlots + (blockIdx.x & (kArgSlots - 1)), s_key[threadIdx.x],
                             __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    if (!arrive_last(p.counters, gridDim.x, s_flag)) return;
    argmax_finish(keys, p.rows, 4, wave, lane, p.ids_out, p.lens_inc);
  }
}

template <int MT, uint32_t FLAGS>
hipError_t launch_wide_mt(const GemmParams &p, hipStream_t s) {
  constexpr bool GLU = (FLAGS & QDEC_GLU) != 0;
  const int T = GLU ? p.n / 8 : p.n / 16;
  // The fewest units per workgroup that run in one round of the CUs (a unit
  // more costs its own loads; a second round costs the whole first again).
  auto rounds = [&](int u) { return ((T + u - 1) / u * p.ksplit + kWideWorkgroups - 1) / kWideWorkgroups; };
  auto go = [&](auto kernel, int u) {
    hipLaunchKernelGGL(kernel, dim3((T + u - 1) / u * p.ksplit), dim3(256), 0, s, p);
    return hipSuccess;
  };
  if constexpr ((FLAGS & QDEC_ARGMAX) != 0) {
    if constexpr (MT > 4) return hipErrorInvalidValue;
    else return go(wide_kernel<MT, 3, FLAGS>, 3);
  } else if constexpr (GLU) {
    // gate/up has more units than one round of few takes, and where the 256
    // CUs do not divide them a last round runs for a few: the least of rounds
    // x (units + row tiles / 2 beyond the first, whose fragments the
    // workgroups share through L2).  MI355X, us at 9 / 24 / 48 / 64 rows of
    // 12288 x 4096: per-tile kernels 32.7 / 36.7 / 41.4 / 46.2; units 2 32.7 /
    // 38.3 / 44.1 / 49.3, 3 34.0 / 36.2 / 39.6 / 43.6, 5 (308 workgroups) 43.9
    // / 47.4 / 50.2 / 53.9, 6 35.4 / 36.2 / 37.0 / 38.0; of 3072 x 1024: 5.9 /
    // 6.6 / 7.5 / 8.3; 6.3 / 6.9 / 8.0 / 8.8, 3 7.3 / 8.1 / 9.4 / 9.8.
    int best = rounds(1) == 1 ? 1 : 0, least = 0;
    if (!best)
      for (const int u : {2, 3, 5, 6}) {
        if (u == 6 && MT > 6) continue;  // beyond the LDS
        const int cost = rounds(u) * (25 * u + 13 * (MT - 1));
        if (!best || cost < least) best = u, least = cost;
      }
    switch (best) {
      case 1: return go(wide_kernel<MT, 1, FLAGS>, 1);
      case 2: return go(wide_kernel<MT, 2, FLAGS>, 2);
      case 3: return go(wide_kernel<MT, 3, FLAGS>, 3);
      case 6:
        if constexpr (MT <= 6) return go(wide_kernel<MT, 6, FLAGS>, 6);
      default: return go(wide_kernel<MT, 5, FLAGS>, 5);
    }
  } else {
    // A k split of wide outputs (Qwen3-8B's down, 256 tiles x 4) fills a
    // round at 4 units: us at 9 / 24 / 48 / 64 rows, per-tile kernels 22.4 /
    // 28.9 / 32.3 / 37.2, units 3 23.8 / 26.1 / 29.0 / 32.1, 4 19.1 / 19.2 /
    // 20.7 / 22.4.
    return rounds(1) == 1           ? go(wide_kernel<MT, 1, FLAGS>, 1)
           : rounds(2) == 1         ? go(wide_kernel<MT, 2, FLAGS>, 2)
           : rounds(3) <= rounds(4) ? go(wide_kernel<MT, 3, FLAGS>, 3)
                                    : go(wide_kernel<MT, 4, FLAGS>, 4);
  }
}

template <uint32_t FLAGS>
hipError_t launch_wide_flags(const GemmParams &p, hipStream_t s) {
  switch ((p.rows + 15) / 16) {
    case 1: return launch_wide_mt<1, FLAGS>(p, s);
    case 2: return launch_wide_mt<2, FLAGS>(p, s);
    case 3: return launch_wide_mt<3, FLAGS>(p, s);
    case 4: return launch_wide_mt<4, FLAGS>(p, s);
    case 5: return launch_wide_mt<5, FLAGS>(p, s);
    case 6: return launch_wide_mt<6, FLAGS>(p, s);
    case 7: return launch_wide_mt<7, FLAGS>(p, s);
    case 8: return launch_wide_mt<8, FLAGS>(p, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace

hipError_t launch_wide(const GemmParams &p, uint32_t flags, hipStream_t s) {
  if (p.waves != 4 || !p.xt || p.ksw * 4 * p.ksplit != p.KS || (p.ksplit > 1 && !p.parts_out)) return hipErrorInvalidValue;
  switch (flags & ~QDEC_NORM_IN) {
    case 0u: return launch_wide_flags<0u>(p, s);
    case QDEC_RES_OUT: return launch_wide_flags<QDEC_RES_OUT>(p, s);
    case QDEC_GLU: return launch_wide_flags<QDEC_GLU>(p, s);
    case QDEC_ARGMAX: return launch_wide_flags<QDEC_ARGMAX>(p, s);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace qdec
