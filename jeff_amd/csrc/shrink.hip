// The LoRA first factor ("shrink"): mid[p, rho_j + q] = bf16( sum_k x[perm[p], k] A_j[a][q, k] ) for every sorted
// token position p of an adapter segment, matrix j of the group and live rank q. Summed in float32 in a fixed
// order and rounded once to bf16, as the reference rounds its first factor before the second product
// (engine/fast_path.py:159-177,196; engine/int4_kernels.py:67-82,120). Three kernels, chosen by segment length and size:
//  - shrink_seg: few tokens per adapter (decode). One workgroup per (segment, 32-rank block) streams those 32 rows
//    of A once into MFMA operands, the segment's rows as the other operand; its waves split the inputs and add their
//    sums in a fixed order. Memory-bound on A.
//  - shrink_rows: long segments, few rows. One workgroup per 32 sorted rows and 32 stacked ranks, the inputs sliced over
//    its 16 waves.
//  - shrink_tile: long segments (prefill). Workgroups per 128 sorted positions, 4 waves of 32 rows; the x rows and
//    the adapter's A rows stream through LDS rings two steps ahead, A shared by the waves; each wave sums its rows
//    over all the inputs in order.
#include <type_traits>

#include "shrink_seg.h"
#include "tile_common.h"

namespace {

using namespace mlora;

constexpr int kSChunk = 64;   // inputs per staged chunk (128-byte rows)

__device__ __forceinline__ void drain_lds() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }

template <int RB, int D>
__global__ __launch_bounds__(256) void shrink_tile_kernel(mlora_lora_t L, mlora_route_t r,
                                                          const uint16_t* __restrict__ x, int64_t x_stride, int32_t k,
                                                          uint16_t* __restrict__ mid) {
  constexpr int kRows = 128;
  constexpr int kLoads = 4 + RB;  // memory instructions per lane and step: x rows, then A rows
  static_assert(RB >= 1 && RB <= 4, "at most 4 blocks of A per pass");
  static_assert(D >= 3 && D <= 5, "rings of 3 to 5 slots");
  // rings of D x buffers (128 rows x 64 inputs) and D A buffers (RB blocks of 32 stacked ranks x 64 inputs), distinct
  // arrays so each slot is known at compile time; only the first D of each are used (and allocated). The host picks
  // D for the LDS a workgroup may take: two per CU, or one with more steps in flight.
  __shared__ __attribute__((aligned(16))) uint16_t t_x0[kRows * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_x1[kRows * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_x2[kRows * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_x3[kRows * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_x4[kRows * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_a0[RB * 32 * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_a1[RB * 32 * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_a2[RB * 32 * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_a3[RB * 32 * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t t_a4[RB * 32 * kSChunk];
  auto xslot = [&](auto slot) __attribute__((always_inline)) {
    constexpr int S = decltype(slot)::value % D;
    if constexpr (S == 0) return t_x0;
    else if constexpr (S == 1) return t_x1;
    else if constexpr (S == 2) return t_x2;
    else if constexpr (S == 3) return t_x3;
    else return t_x4;
  };
  auto aslot = [&](auto slot) __attribute__((always_inline)) {
    constexpr int S = decltype(slot)::value % D;
    if constexpr (S == 0) return t_a0;
    else if constexpr (S == 1) return t_a1;
    else if constexpr (S == 2) return t_a2;
    else if constexpr (S == 3) return t_a3;
    else return t_a4;
  };
  const int64_t T = r.tokens;
  const int64_t p0 = (int64_t)blockIdx.x * kRows;
  if (p0 >= T) return;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s_first = r.seg_of[p0], s_last = r.seg_of[min(p0 + kRows, T) - 1];
  const int s_lo = blockIdx.y == 0 ? s_first : s_first + 1, s_hi = blockIdx.y == 0 ? s_first : s_last;
  if (s_lo > s_hi) return;
  // x staging: instruction i of wave w fills rows 8 (4 i + w) .. +7; lane l writes 16-byte slot l & 7 of row
  // +(l >> 3), which holds logical chunk swz_slot(row, l & 7). Rows past the tokens read the tile's first row.
  const uint16_t* xsrc[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * (4 * i + wave) + (lane >> 3);
    const int64_t p = p0 + row;
    xsrc[i] = x + (int64_t)r.tok_perm[p < T ? p : p0] * x_stride + 8 * swz_slot(row, lane & 7);
  }
  const int nk = k / kSChunk;
  const int R = L.rank_cap, nblk = (R + 31) / 32;
  const int orow = wave * 32 + (lane & 31);  // the lane's x operand row (and token of its accumulators)
  const int64_t prow = p0 + orow;
  for (int s = s_lo; s <= s_hi; ++s) {
    const int a = r.seg_adapter[s];
    if (a == 0) continue;  // the base row: no first factor is read
    const int64_t sb = r.seg_start[s], se = r.seg_start[s + 1];
    const uint16_t* Abase = L.pool + (int64_t)a * L.pool_stride + L.off_a;
    const int passes = (nblk + RB - 1) / RB;
    for (int pass = 0; pass < passes; ++pass) {
      const int b0 = pass * RB;
      // A staging: instruction i of wave w fills stacked rows 32 b0 + 8 (4 i + w) .. +7 (rows past R re-read row
      // R - 1, never written out)
      // (a fixed-size array: captured by the lambdas below, an array sized by RB kept the compiler from emitting the
      // kernel's host-side launch stubs)
      const uint16_t* asrc[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * (4 * i + wave) + (lane >> 3);
        asrc[i] = Abase + (int64_t)min(32 * b0 + row, R - 1) * k + 8 * swz_slot(row, lane & 7);
      }
      // a step's loads into ring slot (xs, as); past the last step they re-read it (the same number of loads in
      // flight at every wait)
      auto issue = [&](uint16_t* xs, uint16_t* as, int c) __attribute__((always_inline)) {
        const int kc = min(c, nk - 1) * kSChunk;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          __builtin_amdgcn_global_load_lds(xsrc[i] + kc, (lds_void*)(xs + 8 * (4 * i + wave) * kSChunk), 16, 0, 0);
#pragma unroll
        for (int i = 0; i < RB; ++i)
          __builtin_amdgcn_global_load_lds(asrc[i] + kc, (lds_void*)(as + 8 * (4 * i + wave) * kSChunk), 16, 0, 0);
      };
      f32x16_t acc[RB];
#pragma unroll
      for (int bi = 0; bi < RB; ++bi) acc[bi] = f32x16_t{};
      auto compute = [&](const uint16_t* xs, const uint16_t* as) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int c = 2 * t + (lane >> 5);
          const uint4 xv = *reinterpret_cast<const uint4*>(&xs[swz(orow, c)]);
#pragma unroll
          for (int bi = 0; bi < RB; ++bi) {
            const uint4 av = *reinterpret_cast<const uint4*>(&as[swz(bi * 32 + (lane & 31), c)]);
            acc[bi] = mfma32(av, xv, acc[bi]);
          }
        }
      };
      // Step i reads slot i % D. Its loads landed (the wave's own: at most those of the D - 2 steps after it are in
      // flight), then the barrier (every wave's have, and every wave is done reading step i - 1's slot), then step
      // i + D - 1's loads into that slot, then the MFMAs of step i.
      using I0 = std::integral_constant<int, 0>;
      using I1 = std::integral_constant<int, 1>;
      using I2 = std::integral_constant<int, 2>;
      using I3 = std::integral_constant<int, 3>;
      using I4 = std::integral_constant<int, 4>;
      __syncthreads();  // the previous pass (or segment) is done reading the rings
      issue(xslot(I0{}), aslot(I0{}), 0);
      issue(xslot(I1{}), aslot(I1{}), 1);
      if constexpr (D > 3) issue(xslot(I2{}), aslot(I2{}), 2);
      if constexpr (D > 4) issue(xslot(I3{}), aslot(I3{}), 3);
      auto step = [&](auto slot, int i) __attribute__((always_inline)) {
        constexpr int S = decltype(slot)::value;
        MLORA_WAIT_VM((D - 2) * kLoads);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        issue(xslot(std::integral_constant<int, S + D - 1>{}), aslot(std::integral_constant<int, S + D - 1>{}),
              i + D - 1);
        compute(xslot(slot), aslot(slot));
        drain_lds();  // this step's LDS reads are done before the next barrier
      };
      for (int i = 0; i < nk; i += D) {
        step(I0{}, i);
        if (i + 1 >= nk) break;
        step(I1{}, i + 1);
        if (i + 2 >= nk) break;
        step(I2{}, i + 2);
        if constexpr (D > 3) {
          if (i + 3 >= nk) break;
          step(I3{}, i + 3);
        }
        if constexpr (D > 4) {
          if (i + 4 >= nk) break;
          step(I4{}, i + 4);
        }
      }
      MLORA_WAIT_VM(0);
      // lane l holds, for token p0 + orow and block bi, stacked ranks 32 (b0 + bi) + 8 g + 4 (l >> 5) + e
      if (prow >= sb && prow < se && prow < T) {
        uint16_t* mrow = mid + prow * R;
#pragma unroll
        for (int bi = 0; bi < RB; ++bi) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int n0 = 32 * (b0 + bi) + 8 * g + 4 * (lane >> 5);
            if (n0 >= R) continue;
            // the matrix holding rank n0 (capacities are multiples of 8, so the four ranks n0..n0+3 share it)
            int j = 0, rho = 0;
            while (j + 1 < L.n_mats && n0 >= rho + L.cap[j]) rho += L.cap[j++];
            const int live = live_rank(L, a, j) - (n0 - rho);  // ranks n0.. of matrix j below its live rank
            const uint32_t lo = pack_bf16x2(acc[bi][4 * g], acc[bi][4 * g + 1]);
            const uint32_t hi = pack_bf16x2(acc[bi][4 * g + 2], acc[bi][4 * g + 3]);
            if (live >= 4) {
              *reinterpret_cast<uint2*>(mrow + n0) = make_uint2(lo, hi);
            } else {
              const uint16_t h[4] = {(uint16_t)lo, (uint16_t)(lo >> 16), (uint16_t)hi, (uint16_t)(hi >> 16)};
              for (int e = 0; e < live; ++e) mrow[n0 + e] = h[e];
            }
          }
        }
      }
    }
  }
}

// Long segments in a small or medium pass: one workgroup per (32 sorted rows, 32 stacked ranks), its 16 waves slicing
// the inputs (wave w the 64-input chunks w, w + 16, ...), as slice_kernel (sliced.hip) slices the base product's: a
// pass of few row tiles has few workgroups, and with all the inputs in one wave each would walk them in one long chain.
// A wave stages its chunk's x rows and A rows in two LDS slots of its own (loads that write LDS directly, whole
// 128-byte rows), takes the operands into registers, re-fills the slots and multiplies; there is no barrier before the
// waves' sums are added in wave order. Segments crossing the rows are taken in turn.
constexpr int kRowWaves = 16;
__global__ __launch_bounds__(kRowWaves * 64) void shrink_rows_kernel(mlora_lora_t L, mlora_route_t r,
                                                                    const uint16_t* __restrict__ x, int64_t x_stride,
                                                                    int32_t k, uint16_t* __restrict__ mid) {
  __shared__ __attribute__((aligned(16))) uint16_t w_x[kRowWaves * 32 * kSChunk];
  __shared__ __attribute__((aligned(16))) uint16_t w_a[kRowWaves * 32 * kSChunk];
  const int tid = threadIdx.x, lane = tid & 63, h = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int T = (int)r.tokens, R = L.rank_cap;
  const int p0 = (int)blockIdx.x * 32, p1 = min(p0 + 32, T), b0 = (int)blockIdx.y * 32;
  // instruction i fills rows 8 i + (lane >> 3); lane l writes slot l & 7 of its row, which holds the row's 16-byte
  // chunk swz_slot(row, l & 7); rows past the pass re-read its last row, ranks past the stack the last rank
  const uint16_t* xsrc[4];
  int aoff[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = 8 * i + (lane >> 3);
    xsrc[i] = x + (int64_t)r.tok_perm[min(p0 + row, T - 1)] * x_stride + 8 * swz_slot(row, lane & 7);
    aoff[i] = min(row, R - 1 - b0) * k + 8 * swz_slot(row, lane & 7);
  }
  const int nk = k / kSChunk;
  const int n = wave < nk ? (nk - wave + kRowWaves - 1) / kRowWaves : 0;
  auto issue_x = [&](int i) __attribute__((always_inline)) {
    const int kc = (wave + kRowWaves * i) * kSChunk;
#pragma unroll
    for (int q = 0; q < 4; ++q)
      __builtin_amdgcn_global_load_lds(xsrc[q] + kc, (lds_void*)(w_x + (wave * 32 + q * 8) * kSChunk), 16, 0, 0);
  };
  // the first chunk's rows are asked for before the segments' bookkeeping is read (a layer over 384 tokens 163.9 -> 162.7 us)
  if (n > 0) issue_x(0);
  bool staged = true;
  const int s_lo = r.seg_of[p0], s_hi = r.seg_of[p1 - 1];
  for (int s = s_lo; s <= s_hi; ++s) {
    const int a = r.seg_adapter[s];
    if (a == 0) continue;  // the base row: no first factor
    const int sb = r.seg_start[s], se = r.seg_start[s + 1];
    bool any = false;  // the adapter has a live rank in this block
    for (int j = 0, rho = 0; j < L.n_mats; rho += L.cap[j++])
      any = any || (rho < b0 + 32 && rho + live_rank(L, a, j) > b0);
    if (!any) continue;
    const uint16_t* Ablk = L.pool + (int64_t)a * L.pool_stride + L.off_a + (int64_t)b0 * k;
    auto issue_a = [&](int i) __attribute__((always_inline)) {
      const int kc = (wave + kRowWaves * i) * kSChunk;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        __builtin_amdgcn_global_load_lds(Ablk + aoff[q] + kc, (lds_void*)(w_a + (wave * 32 + q * 8) * kSChunk), 16, 0,
                                         0);
    };
    f32x16_t acc = f32x16_t{};
    if (n > 0) {
      if (!staged) issue_x(0);
      issue_a(0);
    }
    staged = false;
    for (int i = 0; i < n; ++i) {
      uint4 xv[4], av[4];
      const uint4* xs = reinterpret_cast<const uint4*>(w_x);
      const uint4* as = reinterpret_cast<const uint4*>(w_a);
      MLORA_WAIT_VM(0);
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        const int at = (wave * 32 * kSChunk + swz(lane & 31, 2 * u + h)) >> 3;
        xv[u] = xs[at];
        av[u] = as[at];
      }
      drain_lds();  // the slots' reads are done
      if (i + 1 < n) {
        issue_x(i + 1);
        issue_a(i + 1);
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) acc = mfma32(av[u], xv[u], acc);
    }
    // lane l holds row p0 + (l & 31), stacked ranks b0 + 8 g + 4 (l >> 5) + e: the waves' sums added in wave order
    float4* red = reinterpret_cast<float4*>(w_x);
    __syncthreads();  // every wave is done with its slots
#pragma unroll
    for (int g = 0; g < 4; ++g)
      red[(wave * 4 + g) * 64 + lane] = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
    __syncthreads();
    if (tid < 256) {
      float4 v = red[tid];
#pragma unroll
      for (int q = 1; q < kRowWaves; ++q) {
        const float4 t = red[q * 256 + tid];
        v.x += t.x, v.y += t.y, v.z += t.z, v.w += t.w;
      }
      const int p = p0 + (lane & 31), n0 = b0 + 8 * wave + 4 * h;
      if (p >= sb && p < se && p < T && n0 < R) {
        int j = 0, rho = 0;  // the matrix holding rank n0 (capacities are multiples of 8: n0 .. n0 + 3 share it)
        while (j + 1 < L.n_mats && n0 >= rho + L.cap[j]) rho += L.cap[j++];
        const int live = live_rank(L, a, j) - (n0 - rho);
        uint16_t* mrow = mid + (int64_t)p * R + n0;
        const uint32_t lo = pack_bf16x2(v.x, v.y), hi = pack_bf16x2(v.z, v.w);
        if (live >= 4) {
          *reinterpret_cast<uint2*>(mrow) = make_uint2(lo, hi);
        } else {
          const uint16_t o[4] = {(uint16_t)lo, (uint16_t)(lo >> 16), (uint16_t)hi, (uint16_t)(hi >> 16)};
          for (int e = 0; e < live; ++e) mrow[e] = o[e];
        }
      }
    }
    __syncthreads();  // the sums are read before the next segment's slots are filled
  }
  MLORA_WAIT_VM(0);  // (a tile of base rows ends with its first chunk's rows still in flight)
}

// Short segments (decode): one workgroup per (segment, 32-rank block), the body in shrink_seg.h.
__global__ __launch_bounds__(kDWaves * 64) void shrink_seg_kernel(mlora_lora_t L, mlora_route_t r,
                                                                 const uint16_t* __restrict__ x, int64_t x_stride,
                                                                 int32_t k, uint16_t* __restrict__ mid,
                                                                 int32_t max_blocks) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[kSegLds];
  shrink_seg_block(L, r, x, x_stride, k, mid, max_blocks, blockIdx.x, lds, lds + kSegLds / 2);
}

}  // namespace

int launch_shrink(const mlora_lora_t& L, const mlora_route_t& r, const uint16_t* x, int64_t x_stride, int32_t k,
                    uint16_t* mid, bool mfma, hipStream_t stream) {
  if (r.tokens == 0 || r.max_segs == 0) return MLORA_OK;
  if (mfma) {
    // 32-rank blocks of the stacked capacity, in passes of at most 4 (as even as the count allows)
    const int nblk = (L.rank_cap + 31) / 32;
    if (nblk == 0) return MLORA_OK;
    // Rows of 32 with the inputs sliced over 16 waves, where its estimate (a workgroup a CU: 9 us a round and one per
    // chunk of a wave) is below the 128-row tiles' (their waves walk every chunk: 5.5 us and 0.335 a chunk). 2311 rows,
    // K 2048 and 6144: 13 and 16 us against 22 and 34; 32 rows: 5 to 7 against 12 to 37; 8855 rows, K 1024: the tiles,
    // 10 us against 12.
    const int64_t wgs = (r.tokens + 31) / 32 * nblk, nk = k / kSChunk;
    if ((double)((wgs + device_cus() - 1) / device_cus()) * (9.0 + (double)((nk + kRowWaves - 1) / kRowWaves)) <
        5.5 + 0.335 * (double)nk) {
      const dim3 rows((unsigned)((r.tokens + 31) / 32), (unsigned)nblk);
      hipLaunchKernelGGL(shrink_rows_kernel, rows, dim3(kRowWaves * 64), 0, stream, L, r, x, x_stride, k, mid);
      return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
    }
    const int passes = (nblk + 3) / 4, rb = (nblk + passes - 1) / passes;
    const dim3 grid((unsigned)((r.tokens + 127) / 128), 2);
    // ring slots: 20 KB a slot at one block (4 slots, two workgroups per CU), 24 KB at two (3 slots, two per CU),
    // 28 and 32 KB at three and four (5 and 4 slots, one per CU)
    if (rb == 1)
      hipLaunchKernelGGL((shrink_tile_kernel<1, 4>), grid, dim3(256), 0, stream, L, r, x, x_stride, k, mid);
    else if (rb == 2)
      hipLaunchKernelGGL((shrink_tile_kernel<2, 3>), grid, dim3(256), 0, stream, L, r, x, x_stride, k, mid);
    else if (rb == 3)
      hipLaunchKernelGGL((shrink_tile_kernel<3, 5>), grid, dim3(256), 0, stream, L, r, x, x_stride, k, mid);
    else
      hipLaunchKernelGGL((shrink_tile_kernel<4, 4>), grid, dim3(256), 0, stream, L, r, x, x_stride, k, mid);
  } else {
    int max_blocks = 0;  // 32-rank blocks of an adapter using every matrix's capacity
    for (int j = 0; j < L.n_mats; ++j) max_blocks += (L.cap[j] + 31) / 32;
    const int64_t blocks = (int64_t)r.max_segs * max_blocks;
    if (blocks == 0) return MLORA_OK;
    hipLaunchKernelGGL(shrink_seg_kernel, dim3((unsigned)blocks), dim3(kDWaves * 64), 0, stream, L, r, x, x_stride, k,
                       mid, max_blocks);
  }
  return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
}
