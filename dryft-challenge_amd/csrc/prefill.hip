// Prompt-processing (prefill) kernels for gfx950: the large-M product on the
// matrix cores, the batched head norm / RoPE / cache fill, and causal GQA
// flash attention over the cache.
//
// Reference behaviour replaced: engine/engine.py:448-490 (_layers_forward,
// _attend_prefill, _prefill: F.linear, ops.qkv_post_rows, SDPA flash
// attention), engine/kernels/ops.py:149-205 (_qkv_post_rows_kernel) and
// :242-267 (_silu_mul_kernel).
#include "qdec_common.h"
#include "qdec_kernels.h"

namespace qdec {
namespace {

// ------------------------------------------------------------------ product
// The transposed product D = W . x^T: a weight fragment (16 weight rows x 32
// k) is the A operand and an activation fragment (32 k x 16 rows) the B
// operand of v_mfma_f32_16x16x32_bf16, and both are one contiguous KiB in
// their layouts.  Every fragment moves from global memory straight into LDS
// (global_load_lds_dwordx4: one instruction per 1 KiB fragment, no
// registers) through a ring of stages, RING - 1 in flight while one computes.
// Two kernels: pgemm_kernel for tiles of 256 rows (below), and
// pgemm_small_kernel for few rows: 4 waves of 2 x 2 fragments on 64 x 64
// tiles, stages of two k steps (16 KiB), three workgroups per CU.
constexpr int kPgGroupN = 4;  // column tiles walked together (x reuse in L2)

__device__ __forceinline__ uint4 ld16(const uint16_t *p) { return *reinterpret_cast<const uint4 *>(p); }

// 16 bytes per lane from global memory into LDS at byte address lds_addr +
// 16 * lane (global_load_lds_dwordx4; M0 holds the wave's LDS address).
// Issued from inline assembly so the compiler does not make every later LDS
// read wait for all of these loads; the caller waits (vmcnt) and
// synchronises the workgroup itself.
// M0 is saved and restored around the load.
__device__ __forceinline__ void dma16(const void *g, uint32_t lds_addr) {
  uint32_t saved;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\ts_mov_b32 m0, %0"
      : "=&s"(saved)
      : "v"(g), "s"(__builtin_amdgcn_readfirstlane(lds_addr))
      : "memory");
}
// The same from a wave-uniform base and a lane offset, without saving M0
// (for kernels none of whose other instructions read it).
__device__ __forceinline__ void dma16s(const char *base, uint32_t lane_off, uint32_t lds_addr) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1"
               :: "v"(lane_off), "s"(base), "s"(lds_addr)
               : "memory");
}
__device__ __forceinline__ uint32_t lds_addr(const void *p) { return (uint32_t)reinterpret_cast<uintptr_t>(p); }

// Keeps the computation of v where it stands among other pins and volatile
// assembly (the compiler moves plain arithmetic and MFMAs past scheduling
// barriers before it schedules).
template <class V>
__device__ __forceinline__ void pin(V &v) {
  asm volatile("" : "+v"(v));
}

// Maximum of v over the lane pairs (l, l ^ 16) and then (l, l ^ 32), with
// gfx950's row swaps instead of LDS permutes: after v_permlane16_swap the two
// outputs hold the odd / even 16-lane rows exchanged, after
// v_permlane32_swap the two halves, so the maximum of both outputs is the
// pairwise maximum in every lane.
__device__ __forceinline__ float max_xor16_32(float v) {
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// s_waitcnt encodings (gfx9 family): vmcnt in bits 3:0 and 15:14, expcnt
// 6:4, lgkmcnt 11:8; the other counters at their maximum (no wait).
constexpr int vmcnt_enc(int n) { return (n & 15) | ((n >> 4) << 14) | (7 << 4) | (15 << 8); }
constexpr int kVmcnt0 = vmcnt_enc(0);

template <int V>
struct Int {
  static constexpr int value = V;
};

// Tiles of 256 rows x (32 WN) columns, eight waves as 2 (columns) x 4 (rows),
// each WN weight x 4 activation fragments: 256 x 256 (WN 8, 32 KiB stages,
// RING 5), 256 x 160 (WN 5, 26 KiB, RING 6) and 256 x 128 (WN 4, 24 KiB,
// RING 6).  One workgroup per CU walks its tiles with the ring running on:
// the next tile's first stages load while this one ends and stores.
//
// What bounds it is the matrix cores' power: at 32K rows the same code runs
// gate/up at 1310 TFLOP/s on random data and 1650 on zeros.  A step's
// fragment reads, loads and MFMAs are interleaved by hand (each group of 4
// MFMAs between scheduling barriers): left to the compiler, the 12 reads
// came first and the MFMAs of both waves of a SIMD waited together (1150).
// The loads of a step are spread the same way; PRE groups of MFMAs run
// ahead of the barrier, so the matrix cores are busy while the waves meet.
template <int WN>
struct PgTile {
  static constexpr int XW = 4, NW = 8;
  static constexpr int Wf = 2 * WN, Xf = 4 * XW;  // fragments per k step
  static constexpr int Frags = Wf + Xf;
  static constexpr int Loads = Frags / NW;        // per wave and k step; waves below LoadsRem one more
  static constexpr int LoadsRem = Frags % NW;
  static constexpr int LoadsMax = Loads + (LoadsRem ? 1 : 0);
  static constexpr int RING = 163840 / (Frags * 1024) > 6 ? 6 : 163840 / (Frags * 1024);
  static constexpr int PRE = (3 * WN) / 8;        // MFMA groups ahead of the barrier
};

constexpr uint32_t kPgParts = 1u << 8;  // template flag beside the QDEC_* ones

template <uint32_t FLAGS, int WN>
__global__ void __launch_bounds__(512, 2) pgemm_kernel(const PgemmParams p) {
  using S = PgTile<WN>;
  constexpr bool GLU = (FLAGS & QDEC_GLU) != 0;
  constexpr bool RES = (FLAGS & QDEC_RES_OUT) != 0;
  constexpr bool PARTS = (FLAGS & kPgParts) != 0;  // k parts, their sums left in p.parts
  constexpr int XW = S::XW, RING = S::RING;
  static_assert(!GLU || WN % 2 == 0, "gate and up fragments pair up within a wave");
  __shared__ uint4 lds[RING * S::Frags * 64];  // [ring slot][fragment][lane]
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, grp = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;
  const int KSW = p.k >> 5, KS = PARTS ? KSW / p.ksplit : KSW;  // k steps of the weights and of a part (even)

  // Tile order: workgroup i runs on XCD i % 8, so each XCD gets a contiguous
  // range of the sequence, dealt to its workgroups in turn; the sequence
  // walks groups of kPgGroupN column tiles across all row tiles (the group's
  // weights stay in L2, each row tile of x is read by the group's workgroups
  // together).
  const int ntm = p.tiles / S::Xf, T1 = ntm * p.wg_n, T = PARTS ? T1 * p.ksplit : T1;
  const int G = gridDim.x, xcd = blockIdx.x & 7;
  const int per = G >> 3;  // workgroups on this XCD (the grid is a multiple of 8)
  const int seq_end = (int)((int64_t)T * (xcd + 1) / 8);
  int seq = (int)((int64_t)T * xcd / 8) + (blockIdx.x >> 3);
  if (seq >= seq_end) return;
  auto place = [&](int id, int &tm, int &tn) -> int {  // and the k part
    const int part = PARTS ? __builtin_amdgcn_readfirstlane(id / T1) : 0;
    id -= part * T1;
    const int gsz = kPgGroupN * ntm;
    const int g = __builtin_amdgcn_readfirstlane(id / gsz), r = id - g * gsz;
    const int gn = min(kPgGroupN, p.wg_n - g * kPgGroupN);
    tm = __builtin_amdgcn_readfirstlane(r / gn);
    tn = g * kPgGroupN + (r - tm * gn);
    return part;
  };
  // Weight tile of workgroup fragment f (GLU: WN gate tiles, then the WN
  // matching up tiles).
  auto wtile = [&](int tn, int f) -> int {
    if constexpr (GLU)
      return f < WN ? tn * WN + f : p.up_tiles + tn * WN + f - WN;
    else
      return tn * S::Wf + f;
  };
  // This wave's weight fragments (GLU: gate i pairs with up i + WN/2).
  auto wf = [&](int i) -> int {
    if constexpr (GLU)
      return i < WN / 2 ? wn * (WN / 2) + i : WN + wn * (WN / 2) + i - WN / 2;
    else
      return wn * WN + i;
  };

  // Loads: wave w moves fragments w + 8 q of every k step (weights first).
  // The load cursor (lseq, lk) runs RING - 1 stages ahead of the compute;
  // past this workgroup's last tile it loads that tile's stages again, which
  // nothing reads.
  const bool hi = wave < S::LoadsRem;
  const size_t xks = (size_t)p.tiles * 1024;  // bytes per k step of x
  const uint32_t voff = lane * 16, lds0 = lds_addr(lds);
  const char *src[S::LoadsMax];
  auto aim = [&](int id) {
    int tm, tn;
    const size_t k0 = (size_t)place(id, tm, tn) * KS;
#pragma unroll
    for (int q = 0; q < S::LoadsMax; ++q) {
      const int f = min(wave + S::NW * q, S::Frags - 1);
      src[q] = f < S::Wf ? reinterpret_cast<const char *>(p.w) + ((size_t)wtile(tn, f) * KSW + k0) * 1024
                         : reinterpret_cast<const char *>(p.x) + k0 * xks + (size_t)(tm * S::Xf + f - S::Wf) * 1024;
    }
  };
  auto load = [&](int q, uint32_t slot_base) {
    const int f = wave + S::NW * q;
    dma16s(src[q], voff, slot_base + f * 1024);
    src[q] += f < S::Wf ? (size_t)1024 : xks;
  };
  int lseq = seq, lk = 0;
  aim(seq);
  auto next_pair = [&]() {  // before the loads of stages lk and lk + 1
    if (lk == KS) {
      lk = 0;
      if (lseq + per < seq_end) lseq += per;
      aim(lseq);
    }
    lk += 2;
  };
#pragma unroll
  for (int st = 0; st < RING - 1; ++st) {
    if (st % 2 == 0) next_pair();
#pragma unroll
    for (int q = 0; q < S::LoadsMax; ++q)
      if (q < S::Loads || hi) load(q, lds0 + st * S::Frags * 1024);
  }
  // Waits until at most `stages` whole stages of this wave's loads (and
  // `after` younger stores) are outstanding.
  auto wait_stages = [&](auto stages, auto after) {
    constexpr int n = decltype(stages)::value * S::Loads + decltype(after)::value;
    constexpr int nh = n + decltype(stages)::value;
    static_assert(nh <= 63, "vmcnt");
    if (S::LoadsRem != 0 && hi)
      __builtin_amdgcn_s_waitcnt(vmcnt_enc(nh));
    else
      __builtin_amdgcn_s_waitcnt(vmcnt_enc(n));
  };
  wait_stages(Int<RING - 2>{}, Int<0>{});
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");

  f32x4_t acc[WN][XW];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < WN; ++i)
#pragma unroll
      for (int q = 0; q < XW; ++q) acc[i][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  };
  clear();
  // Two register sets of fragments: step t + 1's are read while step t's
  // MFMAs run.
  uint4 a[2][WN], b[2][XW];
#pragma unroll
  for (int q = 0; q < XW; ++q) b[0][q] = lds[(S::Wf + wm * XW + q) * 64 + lane];
#pragma unroll
  for (int i = 0; i < WN; ++i) a[0][i] = lds[wf(i) * 64 + lane];
  int rslot = 1, fslot = RING - 1;  // ring slots read and filled next
  bool stored = false;              // the last tile's stores are younger than the stages waited for

  // One k step: the MFMAs of the fragments in set `cur`; behind PRE groups of
  // them the barrier that makes stage t + 1 visible and frees the slot of
  // stage t - 1 (all of whose fragments are in registers) for the loads.
  constexpr int kStores = GLU ? WN * XW / 2 : WN * XW;
  auto step = [&](auto curc) {
    constexpr int cur = decltype(curc)::value, nx = cur ^ 1;
    auto mma = [&](int i) {
#pragma unroll
      for (int q = 0; q < XW; ++q) acc[i][q] = mfma16x16x32(a[cur][i], b[cur][q], acc[i][q]);
    };
#pragma unroll
    for (int i = 0; i < S::PRE; ++i) mma(i);
    __builtin_amdgcn_sched_barrier(0);
    if (stored)
      wait_stages(Int<RING - 3>{}, Int<kStores>{});
    else
      wait_stages(Int<RING - 3>{}, Int<0>{});
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    const uint4 *L = lds + rslot * S::Frags * 64 + lane;
    const uint32_t fill = lds0 + fslot * S::Frags * 1024;
    __builtin_amdgcn_sched_barrier(0);
    constexpr int REM = WN - S::PRE, RD = XW + WN;
#pragma unroll
    for (int i = S::PRE; i < WN; ++i) {
      const int j = i - S::PRE;
      const int r0 = (RD * j + REM - 1) / REM, r1 = (RD * (j + 1) + REM - 1) / REM;
      const int d0 = (S::Loads * j + REM - 1) / REM, d1 = (S::Loads * (j + 1) + REM - 1) / REM;
#pragma unroll
      for (int r = r0; r < r1; ++r) {
        if (r < XW)
          b[nx][r] = L[(S::Wf + wm * XW + r) * 64];
        else
          a[nx][r - XW] = L[wf(r - XW) * 64];
      }
#pragma unroll
      for (int q = d0; q < d1; ++q) load(q, fill);
      if (i == WN - 1 && S::LoadsRem != 0 && hi) load(S::Loads, fill);
      __builtin_amdgcn_sched_barrier(0);
      mma(i);
      __builtin_amdgcn_sched_barrier(0);
    }
    rslot = rslot + 1 == RING ? 0 : rslot + 1;
    fslot = fslot + 1 == RING ? 0 : fslot + 1;
  };

  for (;;) {
    for (int t = 0; t < KS; t += 2) {
      if (RING & 1) next_pair();
      step(Int<0>{});
      if (!(RING & 1)) next_pair();
      step(Int<1>{});
      stored = false;
    }
    // Epilogue: lane holds columns n0 .. n0+3 of row m for every fragment
    // pair.  A tile whose rows are all real stores through inline assembly,
    // so the number of stores the next tile's first waits let pass is known.
    int tm, tn;
    const int part = place(seq, tm, tn);
    auto residual = [&](int m, int n0) -> uint2 {
      if constexpr (RES) return *reinterpret_cast<const uint2 *>(p.res + (size_t)m * p.n_out + n0);
      return make_uint2(0u, 0u);
    };
    auto value = [&](int i, int q, uint2 rv) -> uint2 {
      if constexpr (GLU) {
        float o4[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) o4[e] = swiglu(rbf(acc[i][q][e]), rbf(acc[i + WN / 2][q][e]));
        return make_uint2(pack2(o4[0], o4[1]), pack2(o4[2], o4[3]));
      } else if constexpr (RES) {
        return make_uint2(pack2(lo16(rv.x) + rbf(acc[i][q][0]), hi16(rv.x) + rbf(acc[i][q][1])),
                          pack2(lo16(rv.y) + rbf(acc[i][q][2]), hi16(rv.y) + rbf(acc[i][q][3])));
      } else {
        return make_uint2(pack2(acc[i][q][0], acc[i][q][1]), pack2(acc[i][q][2], acc[i][q][3]));
      }
    };
    auto dst = [&](int m, int n0) -> uint16_t * {
      return p.ofrag ? p.out + frag_off(m, n0, p.tiles) : p.out + (size_t)m * p.n_out + n0;
    };
    constexpr int NI = GLU ? WN / 2 : WN;
    const int m_base = (tm * S::Xf + wm * XW) * 16 + col;
    if constexpr (PARTS) {
      // a k part's sums, merged by the row norm that reads the residual next
#pragma unroll
      for (int q = 0; q < XW; ++q) {
        const int m = m_base + q * 16;
        if (m >= p.rows) continue;
#pragma unroll
        for (int i = 0; i < WN; ++i)
          *reinterpret_cast<f32x4_t *>(p.parts + ((size_t)part * p.rows + m) * p.n_out + wtile(tn, wf(i)) * 16 + 4 * grp) =
              acc[i][q];
      }
    } else if ((tm + 1) * S::Xf * 16 <= p.rows) {
#pragma unroll
      for (int q0 = 0; q0 < XW; q0 += 2) {
        uint2 rv[2][NI];  // residuals of two row fragments, loaded together
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < NI; ++i) rv[u][i] = residual(m_base + (q0 + u) * 16, wtile(tn, wf(i)) * 16 + 4 * grp);
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            const int m = m_base + (q0 + u) * 16, n0 = wtile(tn, wf(i)) * 16 + 4 * grp;
            const uint2 o = value(i, q0 + u, rv[u][i]);
            asm volatile("global_store_dwordx2 %0, %1, off" ::"v"(dst(m, n0)), "v"(__builtin_bit_cast(uint64_t, o))
                         : "memory");
          }
      }
      stored = true;
    } else {
#pragma unroll
      for (int q = 0; q < XW; ++q) {
        const int m = m_base + q * 16;
        if (m >= p.rows) continue;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
          const int n0 = wtile(tn, wf(i)) * 16 + 4 * grp;
          *reinterpret_cast<uint2 *>(dst(m, n0)) = value(i, q, residual(m, n0));
        }
      }
    }
    seq += per;
    if (seq >= seq_end) break;
    clear();
  }
  // The loads past the last tile still write this workgroup's LDS.
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
}

// ---- few rows
constexpr int kPsFrags = 4 + 4;           // weight + activation fragments per k step
constexpr int kPsSteps = 2, kPsRing = 3;  // k steps per stage, stage buffers
constexpr int kPsStage = kPsSteps * kPsFrags;
constexpr int kPsLoads = kPsStage / 4;    // loads per wave per stage

template <uint32_t FLAGS>
__global__ void __launch_bounds__(256, 1) pgemm_small_kernel(const PgemmParams p) {
  constexpr bool GLU = (FLAGS & QDEC_GLU) != 0;
  constexpr bool RES = (FLAGS & QDEC_RES_OUT) != 0;
  __shared__ uint4 lds[kPsRing * kPsStage * 64];  // [ring slot][k step][fragment][lane]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int wn = wave & 1, wm = wave >> 1;

  // Tile order as in pgemm_kernel, one tile per workgroup; row tiles of the
  // padding beyond the rows are left out.
  int id = blockIdx.x;
  const int G = gridDim.x;
  if ((G & 7) == 0) id = (id & 7) * (G >> 3) + (id >> 3);
  const int ntm = pg_small_row_tiles(p.rows);
  const int gsz = kPgGroupN * ntm;
  const int g = id / gsz, r = id - g * gsz;
  const int gn = min(kPgGroupN, p.wg_n - g * kPgGroupN);
  const int tm = r / gn, tn = g * kPgGroupN + (r - (r / gn) * gn);

  const int KS = p.k >> 5;
  auto wtile = [&](int f) -> int {
    if constexpr (GLU)
      return f < 2 ? tn * 2 + f : p.up_tiles + tn * 2 + f - 2;
    else
      return tn * 4 + f;
  };
  const uint16_t *wb = p.w + (size_t)wtile(wave) * KS * 512 + lane * 8;
  const uint16_t *xb = p.x + (size_t)(tm * 4 + wave) * 512 + lane * 8;
  const size_t xks = (size_t)p.tiles * 512;  // elements per k step of x
  const uint32_t lds0 = lds_addr(lds);
  auto dma = [&](int s, int slot) {
#pragma unroll
    for (int j = 0; j < kPsSteps; ++j) {
      const int ks = s * kPsSteps + j;
      const uint32_t dst = lds0 + (uint32_t)(((slot * kPsSteps + j) * kPsFrags + wave) * 1024);
      dma16(wb + (size_t)ks * 512, dst);
      dma16(xb + ks * xks, dst + 4 * 1024);
    }
  };
  // This wave's weight fragments (GLU: gate 0 pairs with up 1).
  auto wf = [&](int i) -> int {
    if constexpr (GLU)
      return i < 1 ? wn + i : 2 + wn + i - 1;
    else
      return wn * 2 + i;
  };

  f32x4_t acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int q = 0; q < 2; ++q) acc[i][q] = f32x4_t{0.f, 0.f, 0.f, 0.f};

  const int nst = p.k / (32 * kPsSteps);
#pragma unroll
  for (int s = 0; s < kPsRing - 1; ++s)
    if (s < nst) dma(s, s);
  int slot = 0;
  for (int s = 0; s < nst; ++s) {
    // this wave's loads of stage s are done once at most the younger stage's
    // are outstanding; the barrier makes every wave's visible and frees the
    // slot of stage s-1 for stage s + 2
    if (s + 1 < nst)
      __builtin_amdgcn_s_waitcnt(vmcnt_enc(kPsLoads));
    else
      __builtin_amdgcn_s_waitcnt(kVmcnt0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + kPsRing - 1 < nst) dma(s + kPsRing - 1, slot == 0 ? kPsRing - 1 : slot - 1);
#pragma unroll
    for (int j = 0; j < kPsSteps; ++j) {
      const uint4 *L = lds + (size_t)(slot * kPsSteps + j) * kPsFrags * 64 + lane;
      uint4 a[2], bx[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) a[i] = L[wf(i) * 64];
#pragma unroll
      for (int q = 0; q < 2; ++q) bx[q] = L[(4 + wm * 2 + q) * 64];
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int q = 0; q < 2; ++q) acc[i][q] = mfma16x16x32(a[i], bx[q], acc[i][q]);
    }
    slot = slot == kPsRing - 1 ? 0 : slot + 1;
  }

  // Epilogue: lane holds columns n0 .. n0+3 of row m for every fragment pair.
  auto store = [&](int m, int n0, uint2 o) {
    uint16_t *dst = p.ofrag ? p.out + frag_off(m, n0, p.tiles) : p.out + (size_t)m * p.n_out + n0;
    *reinterpret_cast<uint2 *>(dst) = o;
  };
  const int m_base = (tm * 4 + wm * 2) * 16 + col;
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int m = m_base + q * 16;
    if (m >= p.rows) continue;
    if constexpr (GLU) {
      float o4[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) o4[e] = swiglu(rbf(acc[0][q][e]), rbf(acc[1][q][e]));
      store(m, wtile(wf(0)) * 16 + 4 * grp, make_uint2(pack2(o4[0], o4[1]), pack2(o4[2], o4[3])));
    } else {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int n0 = wtile(wf(i)) * 16 + 4 * grp;
        uint2 o;
        if constexpr (RES) {
          const uint2 rv = *reinterpret_cast<const uint2 *>(p.res + (size_t)m * p.n_out + n0);
          o.x = pack2(lo16(rv.x) + rbf(acc[i][q][0]), hi16(rv.x) + rbf(acc[i][q][1]));
          o.y = pack2(lo16(rv.y) + rbf(acc[i][q][2]), hi16(rv.y) + rbf(acc[i][q][3]));
        } else {
          o.x = pack2(acc[i][q][0], acc[i][q][1]);
          o.y = pack2(acc[i][q][2], acc[i][q][3]);
        }
        store(m, n0, o);
      }
    }
  }
}

// ------------------------------------------------------- head norm + RoPE
// 16 lanes hold a head, 8 channels each, so a wave normalises and rotates 4
// heads at once with one reciprocal square root for all of them: the sum of
// squares is 3 additions in a lane, then the 16 lanes of a DPP row (the
// pairing of the full butterfly over 2-channel lanes that the decode kernels
// use, so the bits are theirs), and RoPE's partner channel i +- 64 is the
// lane 8 further round the row.  With 2 channels per lane the vector units
// bounded it: 8192 rows of 32 + 8 heads took 75 us.
constexpr int kPqBatch = 5;  // heads per lane loaded before the first is reduced
typedef uint32_t u32x4a4_t __attribute__((ext_vector_type(4), aligned(4)));

// Tables and norm weights are only promised to be aligned to 4 bytes.
__device__ __forceinline__ uint4 ld16a4(const uint16_t *p) {
  const u32x4a4_t v = *reinterpret_cast<const u32x4a4_t *>(p);
  return make_uint4(v.x, v.y, v.z, v.w);
}

__device__ __forceinline__ uint4 head_norm_rope8(const uint4 &raw, const uint4 &w, const uint4 &cw, const uint4 &sw,
                                                 bool first_half, float eps) {
  float x[8], g[8], c[8], s[8], y[8], o[8];
  unpack8(raw, x);
  unpack8(w, g);
  unpack8(cw, c);
  unpack8(sw, s);
  float q[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    q[e] = x[2 * e] * x[2 * e] + x[2 * e + 1] * x[2 * e + 1];
    pin(q[e]);
  }
  float ss = (q[0] + q[1]) + (q[2] + q[3]);
  ss += dpp_f<0xB1>(ss);   // quad_perm [1,0,3,2]
  ss += dpp_f<0x4E>(ss);   // quad_perm [2,3,0,1]
  ss += dpp_f<0x141>(ss);  // row_half_mirror
  ss += dpp_f<0x140>(ss);  // row_mirror
  const float rstd = 1.0f / sqrtf(ss / 128.0f + eps);
#pragma unroll
  for (int e = 0; e < 8; ++e) y[e] = rbf(g[e] * rbf(x[e] * rstd));
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float r = dpp_f<0x128>(y[e]);  // row_ror:8
    o[e] = rbf(y[e] * c[e]) + rbf((first_half ? -r : r) * s[e]);
  }
  return pack8(o);
}

// ROWS = 1: a workgroup per row, its waves taking 4 heads each in turn.
// ROWS = 8: a workgroup takes the positions of one sequence that share a
// group of 8 slots, each wave two of them.  The values move in groups of 8
// slots, the channel-major V cache's 16-byte cells: two channels of a kv head
// per thread, 4 bytes of each of the group's rows, element by element at the
// call's ragged ends.  With ROWS = 1 the row that starts a whole group writes
// its 8 rows; at the ragged ends each row writes its own elements (left to
// one row of the group, that work met on one XCD where t_rows is a multiple
// of 8: 40 sequences of 32 rows from slot 3 17.3 us, so 10.8).
template <int ROWS>
__global__ void __launch_bounds__(256) pqk_kernel(const PqkParams p) {
  constexpr int D = 128;
  const int T = p.t_rows;
  const int off = p.pos0 & (ROWS - 1);  // groups start on multiples of 8 slots
  const int ngrp = (T + off + ROWS - 1) / ROWS;
  const int b = blockIdx.x / ngrp, g0 = (blockIdx.x - b * ngrp) * ROWS - off;
  const int t0 = max(g0, 0);
  const int nrow = min(g0 + ROWS, T) - t0;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ch8 = (lane & 15) * 8;
  const bool first_half = (lane & 15) < 8;
  const int width = (p.nq + 2 * p.nkv) * D;
  uint16_t *rows = p.qkv + (size_t)(b * T + t0) * width;
  const uint4 qw = ld16a4(p.q_norm_w + ch8), kw = ld16a4(p.k_norm_w + ch8);
  constexpr int RW = ROWS == 1 ? 1 : ROWS / 4;  // rows of a wave
  constexpr int HS = ROWS == 1 ? 16 : 4;        // heads normalised at once on a row
  const int h0 = (lane >> 4) + (ROWS == 1 ? 4 * wave : 0);
  const int nh = p.nq + p.nkv;
  for (int i = 0; i < RW; ++i) {
    const int r = ROWS == 1 ? 0 : wave * RW + i;
    if (r >= nrow) break;
    const int pos = p.pos0 + t0 + r;
    uint16_t *row = rows + (size_t)r * width + ch8;
    uint16_t *kc = p.k_cache + ((size_t)b * p.nkv * p.cap + pos) * D + ch8;
    const uint4 cw = ld16a4(p.cos_tab + (size_t)pos * D + ch8), sw = ld16a4(p.sin_tab + (size_t)pos * D + ch8);
    for (int hb = 0; hb < nh; hb += HS * kPqBatch) {
      uint4 raw[kPqBatch];
#pragma unroll
      for (int j = 0; j < kPqBatch; ++j) {
        const int h = hb + h0 + HS * j;
        raw[j] = h < nh ? ld16(row + (size_t)h * D) : zero4();
      }
#pragma unroll
      for (int j = 0; j < kPqBatch; ++j) {
        if (hb + HS * j >= nh) break;  // no head left for any lane
        const int h = hb + h0 + HS * j;
        const uint4 o = head_norm_rope8(raw[j], h < p.nq ? qw : kw, cw, sw, first_half, p.eps);
        if (h < nh)
          *reinterpret_cast<uint4 *>(h < p.nq ? row + (size_t)h * D : kc + (size_t)(h - p.nq) * p.cap * D) = o;
      }
    }
  }
  const int slot0 = p.pos0 + t0;
  int n = nrow;  // rows to move, from slot0
  if (ROWS == 1) {
    const int g = slot0 & ~7;
    if (g >= p.pos0 && g + 8 <= p.pos0 + T) {
      if (slot0 != g) return;  // the group's first row writes it
      n = 8;
    }
  }
  const bool whole = n == 8 && (slot0 & 7) == 0;
  for (int i = threadIdx.x; i < p.nkv * (D / 2); i += blockDim.x) {
    const int kvh = i >> 6, ch = (i & 63) * 2;
    const uint16_t *src = rows + (size_t)(p.nq + p.nkv + kvh) * D + ch;
    uint16_t *vb = p.v_cache + ((size_t)b * p.nkv + kvh) * p.cap * D;
    if (whole) {
      uint32_t v[8];
#pragma unroll
      for (int r = 0; r < 8; ++r) v[r] = *reinterpret_cast<const uint32_t *>(src + (size_t)r * width);
      uint32_t lo[4], hi[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        lo[r] = (v[2 * r] & 0xffffu) | (v[2 * r + 1] << 16);
        hi[r] = (v[2 * r] >> 16) | (v[2 * r + 1] & 0xffff0000u);
      }
      uint4 *dst = reinterpret_cast<uint4 *>(vb + ((size_t)(slot0 >> 3) * D + ch) * 8);
      dst[0] = make_uint4(lo[0], lo[1], lo[2], lo[3]);
      dst[1] = make_uint4(hi[0], hi[1], hi[2], hi[3]);
    } else {
      for (int r = 0; r < n; ++r) {
        const int slot = slot0 + r;
        const uint32_t v = *reinterpret_cast<const uint32_t *>(src + (size_t)r * width);
        uint16_t *cell = vb + ((size_t)(slot >> 3) * D + ch) * 8 + (slot & 7);
        cell[0] = (uint16_t)v;
        cell[8] = (uint16_t)(v >> 16);
      }
    }
  }
}

// ------------------------------------------------------------ row norm
// RMSNorm of 16 rows (one M tile) per workgroup into fragment order.  A wave
// loads two rows whole, NG 1 KiB vectors of each, sums and rounds them as rownorm_kernel does (the same bits), and leaves the 16-byte cells in
// LDS; then every wave stores whole fragments.  A cell's row is swapped with
// its vector's number so that neither the writes (64 vectors of one row) nor
// the reads (16 rows of 4 vectors) meet in a bank.  A lane that read its
// row's cells in fragment order instead touched 64 cache lines per load: 8192
// rows of 2560 25.2 us, here 17.8 (84 MB, the card's copy rate), 32768 rows
// 95 / 64, of 4096 channels 36 / 32.  Two rows per wave: with four, 128 KiB
// of LDS left 4096 channels one wave per SIMD (38 us).  Rows past `rows` are
// zeros.
constexpr int kPnRpw = 2, kPnWaves = 16 / kPnRpw;  // rows per wave, waves
template <int NG>
__global__ void __launch_bounds__(64 * kPnWaves) pnorm_kernel(const uint16_t *__restrict__ X, const uint16_t *__restrict__ norm_w,
                                                    uint16_t *__restrict__ out, int k, float eps, int rows, int tiles) {
  __shared__ uint4 xs[NG * 64 * 16];  // [vector][row ^ vector % 16]
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int mt = blockIdx.x, nvec = k >> 3;
  uint4 xv[kPnRpw][NG], nw[NG];
#pragma unroll
  for (int j = 0; j < kPnRpw; ++j) {
    const uint16_t *row = X + (size_t)min(mt * 16 + wave * kPnRpw + j, rows - 1) * k;
#pragma unroll
    for (int q = 0; q < NG; ++q) xv[j][q] = ld16(row + 8 * min(q * 64 + lane, nvec - 1));
  }
  if (norm_w) {
#pragma unroll
    for (int q = 0; q < NG; ++q) nw[q] = ld16(norm_w + 8 * min(q * 64 + lane, nvec - 1));
  }
#pragma unroll
  for (int j = 0; j < kPnRpw; ++j) {
    const int r = wave * kPnRpw + j;
    const bool real = mt * 16 + r < rows;
    float rs = 0.f;
    if (norm_w) {
      float tot = 0.f;
#pragma unroll
      for (int a = 0; a < (NG < 4 ? NG : 4); ++a) {  // thread 64 a + lane of rownorm_kernel
        float ss = 0.f;
#pragma unroll
        for (int q = a; q < NG; q += 4)
          if (q * 64 + lane < nvec) {
            float f[8];
            unpack8(xv[j][q], f);
#pragma unroll
            for (int e = 0; e < 8; ++e) ss += f[e] * f[e];
          }
        tot += wave_sum(ss);
      }
      rs = 1.0f / sqrtf(tot / (float)k + eps);
    }
#pragma unroll
    for (int q = 0; q < NG; ++q) {
      const int v = q * 64 + lane;
      if (v < nvec) xs[v * 16 + (r ^ (v & 15))] = !real ? zero4() : norm_w ? norm8(xv[j][q], nw[q], rs) : xv[j][q];
    }
  }
  __syncthreads();
  for (int ks = wave; ks < k >> 5; ks += kPnWaves) {
    const int v = ks * 4 + (lane >> 4);
    *reinterpret_cast<uint4 *>(out + ((size_t)ks * tiles + mt) * 512 + lane * 8) = xs[v * 16 + ((lane & 15) ^ (v & 15))];
  }
}

// ---------------------------------------------------------------- attention
// A workgroup takes kPaRows positions of G = 2 or 4 query heads of one kv
// head of one sequence; wave w takes head w % G of them and half of the
// positions, 2 M tiles of 16 rows (4 or 8 waves).  Blocks of 32 cache slots
// go from global memory straight into LDS (global_load_lds_dwordx4 with
// per-lane gather addresses, so every fragment lands in MFMA operand
// order), kPaRing blocks in a ring shared by the waves:
//   K fragment (s, h): lane (c, g) holds slot 8*(c >> 2) + (c & 3) + 4h,
//     channels 32s + 8g .. +8: the slot order that makes the score registers
//     of S^T = K . Q^T exactly the B operand of O^T += V^T . P^T (each lane
//     ends up with 8 consecutive slots of one query row);
//   V fragment dt: lane (c, g) holds channel 16dt + c, slots 8g .. 8g+7 --
//     16 contiguous bytes of the channel-major cache.
// The loop is pipelined by hand: while block j's softmax runs on the vector
// units, the matrix cores form block j + 1's scores (one MFMA every few
// vector instructions), and block j's P.V product covers the LDS reads of
// block j + 2's keys.  Before that every wave of a workgroup met at the
// block's barrier, multiplied, then exponentiated, so the two units took
// turns: 8 x 1024 rows after 3072 cached slots 575 -> 516 us, 503 now that
// the last block leaves out the scores of none to follow (840 -> 960
// TFLOP/s; short prompts were 2 to 12% slower with them: 13 x 187 26.0 ->
// 27.2, now 26.0), and two heads per kv head 513 -> 269 us.  What bounds it
// is shared: LDS reads (a wave's 32 rows take every K/V fragment for two
// MFMAs), the vector units and the matrix cores each cost about a fifth of
// the time when left out.
// Online softmax in base 2 with fp32 state per row (running max kept in
// score units, exp2(s * scale - m * scale) as one FMA), probabilities rounded
// to bf16 for the P.V product.  Each lane compares its own scores with the
// running maximum; the cross-lane maximum and the rescaling of the
// accumulators run only for a tile some row's maximum moves in.
// Only blocks that cross some row's position are masked.  Slots past the
// block's last row are zeroed in V after the LDS read (the cache may hold
// anything there, and 0 * NaN would poison the product).
constexpr int kPaKFrags = 8, kPaVFrags = 8;
constexpr int kPaBlockVec = (kPaKFrags + kPaVFrags) * 64;  // uint4 per staged block
constexpr int kPaRing = 4;
// Waves per query head: two, each taking 2 M tiles.
constexpr int kPaWph = 2;

// G query heads per workgroup out of GS per kv head: GS / G workgroups per
// (kv head, row block), each reading the kv head's K/V (8 heads in one
// workgroup would need 64 accumulator rows per wave and spill).
template <int G, int GS, int MT>
__global__ void __launch_bounds__(64 * G * kPaWph, 2) pattn_kernel(const PattnParams p) {
  constexpr int D = 128;
  constexpr int ROWS = 16 * MT * kPaWph;       // positions per workgroup
  constexpr int NWV = G * kPaWph;              // waves
  constexpr int NSUB = GS / G;                 // workgroups per (kv head, row block)
  static_assert((MT == 1 || MT == 2) && GS % G == 0 && 16 % NWV == 0, "whole fragments per wave");
  constexpr int FPW = (kPaKFrags + kPaVFrags) / NWV;  // fragments each wave loads per block
  __shared__ uint4 lds[kPaRing * kPaBlockVec];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int col = lane & 15, grp = lane >> 4;
  const int head = wave % G, half = wave / G;  // query head of the group, which 16*MT positions
  const int T = p.t_rows;
  const int nqb = (T + ROWS - 1) / ROWS;
  const int cells = p.batch * p.nkv * NSUB;
  const int qb = nqb - 1 - (int)(blockIdx.x / cells);  // longest rows first
  const int cell = (int)(blockIdx.x % cells);
  const int bk = cell / NSUB, sub = cell - bk * NSUB;
  const int b = bk / p.nkv, kvh = bk - b * p.nkv;
  const int hq = kvh * GS + sub * G + head;
  const int width = (p.nq + 2 * p.nkv) * D;
  const int t0 = qb * ROWS;
  const int tw = t0 + half * 16 * MT;  // this wave's first position
  const int tlast = min(T, t0 + ROWS) - 1;
  const int last = p.pos0 + tlast;  // highest slot any row of the block sees
  const int nb = last / 32 + 1;
  const size_t slab = ((size_t)b * p.nkv + kvh) * (size_t)p.cap * D;
  const uint16_t *kc = p.k_cache + slab;
  const uint16_t *vc = p.v_cache + slab;
  const float NEG_INF = -__builtin_huge_valf();
  const float scale = p.scale_log2;
  const bool rows_full = t0 + ROWS - 1 <= tlast;  // all rows are real

  // Queries as B operands: row col of M tile mt, channels 32s + 8*grp.
  uint4 qf[MT][4];
  int qpos[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int t = tw + mt * 16 + col;
    const bool valid = t <= tlast;
    qpos[mt] = valid ? p.pos0 + t : -1;
    const uint16_t *qrow = p.qkv + (size_t)(b * T + min(t, tlast)) * width + (size_t)hq * D + grp * 8;
#pragma unroll
    for (int s = 0; s < 4; ++s) qf[mt][s] = valid ? ld16(qrow + s * 32) : zero4();
  }

  // Block j into its ring slot: this wave gathers K fragments wave + NWV*i
  // (index 2s + h) and V fragments wave + NWV*i.
  const uint32_t lds0 = lds_addr(lds);
  const uint16_t *kg = kc + (size_t)(8 * (col >> 2) + (col & 3)) * D + 8 * grp;
  const uint16_t *vg = vc + (size_t)grp * D * 8 + col * 8;
  auto dma_block = [&](int j) {
    const int s0 = j * 32;
    const uint32_t base = lds0 + (uint32_t)((j & (kPaRing - 1)) * kPaBlockVec * 16);
#pragma unroll
    for (int i = 0; i < FPW / 2; ++i) {
      const int f = wave + NWV * i;
      dma16(kg + (size_t)(s0 + 4 * (f & 1)) * D + 32 * (f >> 1), base + f * 1024);
    }
#pragma unroll
    for (int i = 0; i < FPW / 2; ++i) {
      const int dt = wave + NWV * i;
      dma16(vg + (size_t)(s0 >> 3) * D * 8 + dt * 128, base + (kPaKFrags + dt) * 1024);
    }
  };

  f32x4_t acc[MT][8];
  float m_run[MT], l_run[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    m_run[mt] = NEG_INF;
    l_run[mt] = 0.f;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) acc[mt][dt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  uint4 kf[8];  // keys of the next block to score: fragment 2s + h
  auto read_k = [&](int j) {
    const uint4 *B = lds + (j & (kPaRing - 1)) * kPaBlockVec + lane;
#pragma unroll
    for (int f = 0; f < 8; ++f) kf[f] = B[f * 64];
  };
  struct Scores {
    f32x4_t a[MT], b[MT];  // slots sb .. sb+3 and sb+4 .. sb+7 of a lane
  };
  // k step s of tile u's scores, slots sb .. +3 (h = 0) or sb+4 .. +7
  auto score1 = [&](Scores &S, int s, int u, int h) {
    f32x4_t &d = h ? S.b[u] : S.a[u];
    d = mfma16x16x32(kf[2 * s + h], qf[u][s], s ? d : f32x4_t{0.f, 0.f, 0.f, 0.f});
  };
  // Waits until this wave's loads of block j are done (blocks up to `newest`
  // have been issued), then meets the other waves: block j is in LDS, and
  // every wave has read what it needs of the blocks before.
  auto await = [&](int j, int newest) {
    const int younger = min(newest, nb - 1) - j;
    if (younger >= 2)
      __builtin_amdgcn_s_waitcnt(vmcnt_enc(2 * FPW) & ~(15 << 8));
    else if (younger == 1)
      __builtin_amdgcn_s_waitcnt(vmcnt_enc(FPW) & ~(15 << 8));
    else
      __builtin_amdgcn_s_waitcnt(kVmcnt0 & ~(15 << 8));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };

  // The query loads complete here, so no wait inside the loop (where it
  // would also wait for the blocks in flight) is needed for them.
  __builtin_amdgcn_s_waitcnt(kVmcnt0);
#pragma unroll
  for (int j = 0; j < kPaRing - 1; ++j)
    if (j < nb) dma_block(j);
  await(0, kPaRing - 2);
  read_k(0);
  Scores s0, s1;
#pragma unroll
  for (int i = 0; i < 8 * MT; ++i) score1(s0, i / (2 * MT), (i >> 1) % MT, i & 1);
  await(min(1, nb - 1), kPaRing - 2);
  if (kPaRing - 1 < nb) dma_block(kPaRing - 1);
  read_k(1);

  // Block j from its scores S; leaves block j + 1's in N (kf holds its keys)
  // unless it is the last.
  auto block = [&](int j, Scores &S, Scores &N, auto lastc) {
    constexpr bool LAST = decltype(lastc)::value != 0;
    const int sb = j * 32 + 8 * grp;  // first of this lane's 8 slots
    if (!(rows_full && j * 32 + 31 <= p.pos0 + t0)) {
      // the block crosses some row's position (the diagonal, rows past the end)
#pragma unroll
      for (int u = 0; u < MT; ++u)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (sb + i > qpos[u]) S.a[u][i] = NEG_INF;
          if (sb + 4 + i > qpos[u]) S.b[u][i] = NEG_INF;
        }
    }
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      const float bmax = fmaxf(fmaxf(fmaxf(S.a[u][0], S.a[u][1]), fmaxf(S.a[u][2], S.a[u][3])),
                               fmaxf(fmaxf(S.b[u][0], S.b[u][1]), fmaxf(S.b[u][2], S.b[u][3])));
      if (!__any(bmax > m_run[u])) continue;  // no row's maximum moves
      const float m_new = fmaxf(m_run[u], max_xor16_32(bmax));
      const float alpha = __builtin_amdgcn_exp2f((m_run[u] - m_new) * scale);
      l_run[u] *= alpha;
      m_run[u] = m_new;
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) acc[u][dt] *= alpha;
    }
    uint4 vf[8];
    const uint4 *B = lds + (j & (kPaRing - 1)) * kPaBlockVec + lane;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) vf[dt] = B[(kPaKFrags + dt) * 64];
    // Block j + 1's scores between the exponentials of block j: one MFMA
    // per probability, in this order.
    uint4 pf[MT];
    float pj[MT][8], mc[MT], psum[MT];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      mc[u] = m_run[u] * scale;
      psum[u] = 0.f;
    }
#pragma unroll
    for (int u = 0; u < MT; ++u)
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int i = u * 8 + e;  // MFMA i of the scores: k step, tile, slot half
        float x = e < 4 ? S.a[u][e] : S.b[u][e - 4];
        pin(x);
        pj[u][e] = __builtin_amdgcn_exp2f(__builtin_fmaf(x, scale, -mc[u]));
        if constexpr (!LAST) {
          score1(N, i / (2 * MT), (i >> 1) % MT, i & 1);
          pin((i & 1) ? N.b[(i >> 1) % MT] : N.a[(i >> 1) % MT]);
        }
        if (i > 0) psum[(i - 1) >> 3] += pj[(i - 1) >> 3][(i - 1) & 7];
        pin(pj[u][e]);
      }
    psum[MT - 1] += pj[MT - 1][7];
#pragma unroll
    for (int u = 0; u < MT; ++u) {
      l_run[u] += psum[u];
      pf[u] = pack8(pj[u]);
    }
    // Block j + 2 in LDS; slot j (whose V every wave holds) takes block j + kPaRing.
    if constexpr (!LAST) {
      await(min(j + 2, nb - 1), j + kPaRing - 1);
      if (j + kPaRing < nb) dma_block(j + kPaRing);
    }
    if (j * 32 + 31 > last) {  // slots past the last row: zero V
      uint32_t keep[4];
#pragma unroll
      for (int d = 0; d < 4; ++d)
        keep[d] = (sb + 2 * d <= last ? 0x0000ffffu : 0u) | (sb + 2 * d + 1 <= last ? 0xffff0000u : 0u);
#pragma unroll
      for (int dt = 0; dt < 8; ++dt) {
        vf[dt].x &= keep[0];
        vf[dt].y &= keep[1];
        vf[dt].z &= keep[2];
        vf[dt].w &= keep[3];
      }
    }
    if constexpr (!LAST) read_k(j + 2);
#pragma unroll
    for (int dt = 0; dt < 8; ++dt)
#pragma unroll
      for (int u = 0; u < MT; ++u) acc[u][dt] = mfma16x16x32(vf[dt], pf[u], acc[u][dt]);
  };
  int j = 0;
  if (!(nb & 1)) {  // pairs, then the last block by itself
    block(0, s0, s1, Int<0>{});
    s0 = s1;
    j = 1;
  }
  for (; j + 1 < nb; j += 2) {
    block(j, s0, s1, Int<0>{});
    block(j + 1, s1, s0, Int<0>{});
  }
  block(j, s0, s1, Int<1>{});

  // Rows in fragment order for the O projection: lane holds channels
  // 16dt + 4*grp .. +3 of its row.
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (tw + mt * 16 > tlast) continue;
    float l = l_run[mt] + shfl_xor(l_run[mt], 16);
    l += shfl_xor(l, 32);
    const int t = tw + mt * 16 + col;
    if (t > tlast) continue;
    const int m = b * T + t;
#pragma unroll
    for (int dt = 0; dt < 8; ++dt) {
      uint2 o;
      o.x = pack2(acc[mt][dt][0] / l, acc[mt][dt][1] / l);
      o.y = pack2(acc[mt][dt][2] / l, acc[mt][dt][3] / l);
      *reinterpret_cast<uint2 *>(p.out + frag_off(m, hq * D + dt * 16 + 4 * grp, p.tiles)) = o;
    }
  }
}

}  // namespace

namespace {
template <int WN>
hipError_t launch_pgemm_tile(const PgemmParams &p, uint32_t flags, hipStream_t s) {
  const int T = p.wg_n * (p.tiles / PgTile<WN>::Xf) * p.ksplit;
  // A whole number per XCD: an XCD's tiles never outnumber its workgroups
  // while the launch has fewer tiles than CUs.
  const dim3 grid(T < kPgWorkgroups ? (T + 7) / 8 * 8 : kPgWorkgroups), block(512);
  switch (flags) {
    case 0u: hipLaunchKernelGGL((pgemm_kernel<0u, WN>), grid, block, 0, s, p); return hipSuccess;
    case QDEC_RES_OUT: hipLaunchKernelGGL((pgemm_kernel<QDEC_RES_OUT, WN>), grid, block, 0, s, p); return hipSuccess;
    case kPgParts:
      if constexpr (WN == 4) {
        hipLaunchKernelGGL((pgemm_kernel<kPgParts, WN>), grid, block, 0, s, p);
        return hipSuccess;
      }
      return hipErrorInvalidValue;
    case QDEC_GLU:
      if constexpr (WN % 2 == 0) {
        hipLaunchKernelGGL((pgemm_kernel<QDEC_GLU, WN>), grid, block, 0, s, p);
        return hipSuccess;
      }
      return hipErrorInvalidValue;
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_pgemm_small(const PgemmParams &p, uint32_t flags, hipStream_t s) {
  const dim3 grid(p.wg_n * pg_small_row_tiles(p.rows)), block(256);
  switch (flags) {
    case 0u: hipLaunchKernelGGL(pgemm_small_kernel<0u>, grid, block, 0, s, p); break;
    case QDEC_RES_OUT: hipLaunchKernelGGL(pgemm_small_kernel<QDEC_RES_OUT>, grid, block, 0, s, p); break;
    case QDEC_GLU: hipLaunchKernelGGL(pgemm_small_kernel<QDEC_GLU>, grid, block, 0, s, p); break;
    default: return hipErrorInvalidValue;
  }
  return hipSuccess;
}
}  // namespace

hipError_t launch_pgemm(const PgemmParams &p, uint32_t flags, hipStream_t s) {
  if (p.tile_rows == 64) return launch_pgemm_small(p, flags, s);
  if (p.parts) flags = kPgParts;
  switch (p.tile_cols) {
    case 256: return launch_pgemm_tile<8>(p, flags, s);
    case 160: return launch_pgemm_tile<5>(p, flags, s);
    default: return launch_pgemm_tile<4>(p, flags, s);
  }
}

// Row norms by whole 16-row tiles from this many rows (below it the tiles
// leave the GPU short of workgroups: a 512-token prompt measured 10.0 ms with
// the per-row kernels and 11.8 with the grouped ones; 32 x 1024-row chunks 5%
// faster with the grouped ones).
constexpr int kGroupedRows = 4096;
// Head norms and RoPE by groups of 8 slots from this many rows: us grouped /
// per row with 32 + 8 heads: 512 rows 12.7 / 7.4, 1500 14.3 / 12.0, 3000 22.7
// / 20.2, 4000 23.7 / 25.7, 6000 30.9 / 35.7; with 16 + 8 heads 1500 11.1 /
// 10.0, 3000 15.2 / 16.9, 4000 17.7 / 20.7; whatever the rows per sequence
// (1296 rows of 8 13.8 / 11.0).  Before a lane left out the heads that its
// row does not have, 16 + 8 heads took 10.1 us at 1000 rows (now 8.4) and 26.9
// at 6000 (21.7).
constexpr int kPqGroupedRows = 3584;

hipError_t launch_prefill_qk(const PqkParams &p, hipStream_t s) {
  if (p.batch * p.t_rows < kPqGroupedRows) {
    hipLaunchKernelGGL(pqk_kernel<1>, dim3(p.batch * p.t_rows), dim3(256), 0, s, p);
    return hipSuccess;
  }
  hipLaunchKernelGGL(pqk_kernel<8>, dim3(p.batch * (((p.pos0 & 7) + p.t_rows + 7) / 8)), dim3(256), 0, s, p);
  return hipSuccess;
}

bool pnorm_fits(int k, int rows) { return k <= 4096 && rows >= kGroupedRows; }

hipError_t launch_pnorm(const void *x, const void *norm_w, void *out, float eps, int rows, int k, int tiles,
                        hipStream_t s) {
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(tiles), dim3(64 * kPnWaves), 0, s, reinterpret_cast<const uint16_t *>(x),
                       reinterpret_cast<const uint16_t *>(norm_w), reinterpret_cast<uint16_t *>(out), k, eps, rows,
                       tiles);
    return hipSuccess;
  };
  return k <= 1024 ? go(pnorm_kernel<2>) : k <= 2048 ? go(pnorm_kernel<4>) : k <= 2560 ? go(pnorm_kernel<5>)
                                                                         : go(pnorm_kernel<8>);
}

namespace {
// One M tile per wave (32 positions per workgroup) instead of two: for calls
// of at most 32 positions; while 64 leave more than half of the CUs idle -- a
// block takes a wave about as long as its latencies, however few rows it
// carries; and, up to a workgroup per CU, where the positions cover most of
// the slots they see (pos0 < t_rows), so that the workgroups' lengths differ
// and two short ones share a CU.  MI355X, us (64 positions / 32): one sequence
// of 300 tokens 19.2 / 12.3, 512 28.2 / 18.0, 1024 49.5 / 31.7; 128 positions
// after 2000 cached 88 / 52; 8 x 128 13.6 / 10.4; 64 sequences of 20 on 16
// heads 10.9 / 8.3; 10 x 67 13.0 / 9.5; 1791 78 / 56; but 5 x 258 after 1479
// 73 / 84.
template <int G, int GS>
void launch_pattn(const PattnParams &p, hipStream_t s) {
  const int cells = p.batch * p.nkv * (GS / G);
  const int b64 = (p.t_rows + kPaRows - 1) / kPaRows * cells, b32 = (p.t_rows + kPaRows / 2 - 1) / (kPaRows / 2) * cells;
  const bool few = b64 <= 128 || p.t_rows <= kPaRows / 2 || (b64 <= 256 && p.pos0 < p.t_rows);
  if (few)
    hipLaunchKernelGGL((pattn_kernel<G, GS, 1>), dim3(b32), dim3(64 * G * kPaWph), 0, s, p);
  else
    hipLaunchKernelGGL((pattn_kernel<G, GS, 2>), dim3(b64), dim3(64 * G * kPaWph), 0, s, p);
}
}  // namespace

hipError_t launch_prefill_attn(const PattnParams &p, hipStream_t s) {
  switch (p.nq / p.nkv) {
    case 2: launch_pattn<2, 2>(p, s); break;
    case 4: launch_pattn<4, 4>(p, s); break;
    case 8: launch_pattn<4, 8>(p, s); break;
    default: return hipErrorInvalidValue;
  }
  return hipSuccess;
}

}  // namespace qdec
