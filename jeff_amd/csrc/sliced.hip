// INT4 product of a small or medium pass, its inputs sliced over a workgroup's waves:
//   y[perm[p], c] = bf16( sum_k x[perm[p], k] W[c, k] + sum_q mid[p, rho_j + q] sB_j[a(p)][c - o_j, q] )
// The same arithmetic as the prefill kernel (gemm256.hip). A workgroup of 8 waves owns a tile of 32 RB sorted rows x CW
// groups of 64 columns; wave (cw, ks) sums group cw over slice ks of the inputs (the 64-input chunks ks, ks + KW, ...) and
// over the adapter segments ks, ks + KW, ... crossing the tile, and the slices' float32 tiles are added in slice order
// through LDS, rounded once and written (plain, added to the residual, or silu(gate) * up). Why this split: at these
// sizes a product is a chain of latencies, not a stream. 256 x 256 tiles over all the inputs leave most CUs idle (384
// rows of 2048 -> 2048: 16 tiles, 45 us); slicing the inputs inside the workgroup fills the CUs with short chains and
// needs no float32 partials in memory and no second launch (16 us).
//
// What bounds it: the conversion of the packed weights (19 vector instructions a word of eight, RB MFMAs beside them), so
// a step of 64 inputs a slice takes about 1.1 us whether RB is 1 or 3, plus 7 to 13 us of fixed time a round (launch,
// first loads, LoRA term, exchange). The four forms (RB, CW, KW) trade rows per conversion against workgroups: (1, 1, 8)
// and (2, 1, 8) for few columns, (2, 2, 4) and (3, 4, 2) for many; slice_form below picks by estimate.
//
// Per step, the x rows of the slices' chunks go straight from memory to LDS (buffer loads with the LDS flag, whole
// 128-byte rows in, MFMA operands out), staged once for a chunk's CW column waves; each lane loads the packed words it
// uses and dequantises them in registers while the products of the word before run. A lane of the plain form takes
// columns 2 i and 2 i + 1 (i = lane & 31), so its two words come in one 8-byte load and its sums of one row are eight
// consecutive columns; the gated form takes gate column i and up column i.
#include <type_traits>

#include "tile_common.h"

namespace {

using namespace mlora;
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

constexpr int kSlCols = 64;       // columns of a tile: two 32-column MFMA blocks
constexpr int kSlRanks = 64;      // ranks of a matrix per LoRA pass

// Eight consecutive output columns (four packed bf16 pairs) of one row, as store4 (mlora_common.h); wide: 16-byte
// stores are aligned.
__device__ __forceinline__ void store8(uint16_t* yr, uint16_t* last, const uint32_t (&v)[4], int left, int32_t flags,
                                       bool wide) {
  if (wide && left >= 8) {
    uint4 o = make_uint4(v[0], v[1], v[2], v[3]);
    if (flags & kStoreResidual) {
      const uint4 rv = *reinterpret_cast<const uint4*>(yr);
      o = make_uint4(add_bf16x2(rv.x, o.x), add_bf16x2(rv.y, o.y), add_bf16x2(rv.z, o.z), add_bf16x2(rv.w, o.w));
    }
    *reinterpret_cast<uint4*>(yr) = o;
    if (last != nullptr) *reinterpret_cast<uint4*>(last) = o;
    return;
  }
  store4(yr, last, v[0], v[1], left, flags);
  if (left > 4) store4(yr + 4, last != nullptr ? last + 4 : nullptr, v[2], v[3], left - 4, flags);
}

// A wave's weights of one chunk as loaded: the words of its two columns for the four 16-input slices, raw scales and
// zero points (converted when used).
struct SliceW {
  uint32_t w[4][2];
  uint32_t s[2], z[2];
};

// The four operand chunks of a 32-row block staged in LDS, read in one statement with their wait: the compiler does not
// see which loads in flight fill the block, and would otherwise wait for all of them before each read.
__device__ __forceinline__ void read_block(uint4 (&a)[4], const uint32_t (&at)[4], uint32_t base) {
  typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
  u32x4_t v[4];
  const uint32_t a0 = at[0] + base, a1 = at[1] + base, a2 = at[2] + base, a3 = at[3] + base;
  asm volatile(
      "ds_read_b128 %0, %4\n ds_read_b128 %1, %5\n ds_read_b128 %2, %6\n ds_read_b128 %3, %7\n"
      "s_waitcnt lgkmcnt(0)"
      : "=&v"(v[0]), "=&v"(v[1]), "=&v"(v[2]), "=&v"(v[3])
      : "v"(a0), "v"(a1), "v"(a2), "v"(a3)
      : "memory");
#pragma unroll
  for (int u = 0; u < 4; ++u) a[u] = make_uint4(v[u].x, v[u].y, v[u].z, v[u].w);
}

template <int RB, int CW, int KW, bool GATED>
__global__ __launch_bounds__(CW* KW * 64) void slice_kernel(mlora_int4_t w, mlora_lora_t L, mlora_route_t r,
                                                           const uint16_t* __restrict__ x, int64_t x_stride,
                                                           uint16_t* __restrict__ y, int64_t y_stride,
                                                           uint16_t* __restrict__ last_out, int32_t n_out,
                                                           const uint16_t* __restrict__ mid, int32_t n_tiles,
                                                           int32_t m_tiles, int32_t vec, int32_t wide,
                                                           int32_t inter) {
  constexpr int W = CW * KW;
  constexpr int kRows = 32 * RB;
  constexpr int kXI = 4 * RB / CW;  // a wave's x instructions per step, 8 rows each
  static_assert(kXI * CW == 4 * RB, "the column waves share a chunk's rows evenly");
  constexpr int kWI = GATED ? 12 : 8;           // weight instructions per step
  constexpr int kChunkB = kRows * 128;          // bytes of one staged chunk
  constexpr int kSlotB = KW * kChunkB;          // one step's chunks: a slot of the ring
  constexpr int kLds = kSlotB > W * 4096 ? kSlotB : W * 4096;  // (and a 4 KB LoRA slot a wave)
  constexpr int D = 3 * kLds <= 160 * 1024 ? 3 : 2;            // slots of the ring (and weight sets)
  static_assert(D * kLds <= 160 * 1024, "LDS");
  // the ring's slots, distinct arrays chosen at compile time (the third is unused, and not allocated, at D = 2): the
  // compiler then knows which one a read touches and does not wait for the loads in flight into the others
  __shared__ __attribute__((aligned(16))) uint8_t sl_x0[kLds];
  __shared__ __attribute__((aligned(16))) uint8_t sl_x1[kLds];
  __shared__ __attribute__((aligned(16))) uint8_t sl_x2[kLds];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int cw = wave % CW, ks = wave / CW;  // the wave's columns and input slice
  const int li = lane & 31, h = lane >> 5;
  // block -> (row tile, column tile): groups of about 512 rows, the group's row tiles innermost, so the workgroups of an
  // XCD share a few column tiles' weights and a group's x rows stay in its L2 over the column tiles
  constexpr int GM = 16 / RB;
  const int b = xcd_tile(blockIdx.x, n_tiles * m_tiles);
  const int grp = b / (GM * n_tiles), rest = b - grp * (GM * n_tiles);
  const int gm = min(GM, m_tiles - grp * GM);
  const int nt = rest / gm, mt = grp * GM + rest - nt * gm;
  const int T = (int)r.tokens;
  const int p0 = mt * kRows, p1 = min(p0 + kRows, T);
  // the wave's 64 columns: MFMA block cb's row index i is plain column n0 + 2 i + cb, gated gate (cb 0) or up (cb 1)
  // column g0 + i; a wave past the layout's columns computes the last ones again and writes nothing
  const int n0 = min((nt * CW + cw) * kSlCols, w.columns - kSlCols), g0 = n0 / 2;
  const bool wout = GATED ? (nt * CW + cw) * 32 < inter : (nt * CW + cw) * kSlCols < n_out;

  // x: the chunk's instruction q = cw kXI + i fills its rows 8 q + (lane >> 3); lane l writes slot l & 7 of its row, which
  // holds the row's 16-byte chunk swz_slot(row, l & 7). Rows past the pass re-read its last row (never written out).
  uint32_t xoff[16];  // (kXI of them: captured by a lambda, an array sized by it loses the kernel's host launch stub)
#pragma unroll
  for (int i = 0; i < kXI; ++i) {
    const int row = 8 * (cw * kXI + i) + (lane >> 3);
    xoff[i] = (uint32_t)(((int64_t)r.tok_perm[min(p0 + row, T - 1)] * x_stride + (swz_slot(row, lane & 7) << 3)) * 2);
  }
  const int nk = w.k / kTK;
  const int steps = (nk + KW - 1) / KW;  // step i: chunk KW i + ks of this wave's slice, while below nk
  const int64_t groups = w.k / w.group;
  const int gshift = w.group == 128 ? 7 : 6;  // the host accepts groups of 64 and 128 inputs
  const bool asym = w.zeros != nullptr;
  const int col0 = GATED ? g0 + li : n0 + 2 * li;
  const int col1 = GATED ? inter + g0 + li : col0 + 1;
  const uint32_t woff0 = (uint32_t)(col0 + h * w.columns) * 4, woff1 = (uint32_t)(col1 + h * w.columns) * 4;
  const uint32_t zmul = asym ? 1 : 2;
  // Loads past the slice's last chunk go through resources of no bytes: they read nothing, and the number of loads in
  // flight at every wait stays the same.
  auto fetch_w = [&](SliceW& st, int i) __attribute__((always_inline)) {
    const int in = __builtin_amdgcn_readfirstlane((KW * i + ks - nk) >> 31);  // all ones for a chunk of the slice's
    const int kc = ((KW * i + ks) * kTK) & in;
    const __amdgpu_buffer_rsrc_t wres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)w.words, (short)0, (int)((int64_t)(w.k / 8) * w.columns * 4) & in, 0x00020000);
    const __amdgpu_buffer_rsrc_t sres = __builtin_amdgcn_make_buffer_rsrc(
        (void*)w.scales, (short)0, (int)(groups * w.columns * 2) & in, 0x00020000);
    const __amdgpu_buffer_rsrc_t zres = __builtin_amdgcn_make_buffer_rsrc(
        asym ? (void*)w.zeros : (void*)w.scales, (short)0,
        __builtin_amdgcn_readfirstlane((int)(groups * w.columns) & in), 0x00020000);
    const int wbase = (kc / 8) * w.columns * 4;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const int so = wbase + u * w.columns * 8;
      if constexpr (GATED) {
        st.w[u][0] = __builtin_amdgcn_raw_buffer_load_b32(wres, woff0, so, 0);
        st.w[u][1] = __builtin_amdgcn_raw_buffer_load_b32(wres, woff1, so, 0);
      } else {
        const u32x2_t v = __builtin_bit_cast(u32x2_t, __builtin_amdgcn_raw_buffer_load_b64(wres, woff0, so, 0));
        st.w[u][0] = v.x;
        st.w[u][1] = v.y;
      }
    }
    const int g = (kc >> gshift) * w.columns;
    st.s[0] = __builtin_amdgcn_raw_buffer_load_b16(sres, col0 * 2, g * 2, 0);
    st.s[1] = __builtin_amdgcn_raw_buffer_load_b16(sres, col1 * 2, g * 2, 0);
    const int gz = __builtin_amdgcn_readfirstlane(g * zmul);
    st.z[0] = __builtin_amdgcn_raw_buffer_load_b8(zres, col0 * zmul, gz, 0);
    st.z[1] = __builtin_amdgcn_raw_buffer_load_b8(zres, col1 * zmul, gz, 0);
  };
  using I0 = std::integral_constant<int, 0>;
  using I1 = std::integral_constant<int, 1>;
  using I2 = std::integral_constant<int, 2>;
  auto slot_of = [&](auto slot) __attribute__((always_inline)) {
    constexpr int S = decltype(slot)::value % D;
    if constexpr (S == 0)
      return (uint8_t*)sl_x0;
    else if constexpr (S == 1)
      return (uint8_t*)sl_x1;
    else
      return (uint8_t*)sl_x2;
  };
  auto dma_x = [&](auto slot, int i0) __attribute__((always_inline)) {
    const int in = __builtin_amdgcn_readfirstlane((KW * i0 + ks - nk) >> 31);
    const int kb = ((KW * i0 + ks) * (kTK * 2)) & in;
    const __amdgpu_buffer_rsrc_t xres = __builtin_amdgcn_make_buffer_rsrc((void*)x, (short)0, in, 0x00020000);
    uint8_t* dst = slot_of(slot) + ks * kChunkB + cw * kXI * 1024;
#pragma unroll
    for (int i = 0; i < kXI; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xres, (lds_void*)(dst + i * 1024), 16, xoff[i], kb, 0, 0);
  };
  // the operands of 16-input slice u of the wave's chunk, read as one index into the LDS array
  auto read_x = [&](auto slot, int u, uint4 (&a)[RB]) __attribute__((always_inline)) {
    const uint4* xv = reinterpret_cast<const uint4*>(slot_of(slot));
#pragma unroll
    for (int rb = 0; rb < RB; ++rb) a[rb] = xv[(ks * kRows * kTK + swz(rb * 32 + li, 2 * u + h)) >> 3];
  };
  uint32_t at[4];  // the lane's operands in a 32-row block of 128-byte rows
#pragma unroll
  for (int u = 0; u < 4; ++u) at[u] = 2 * swz(li, 2 * u + h);
  auto lds_of = [&](auto slot) __attribute__((always_inline)) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)slot_of(slot);
  };

  // The segments crossing the tile, s_lo .. s_hi; this wave's are s_lo + ks + KW i. Their bookkeeping is read before the
  // chunks: lane i holds the wave's segment i (adapter, bounds relative to the tile, live ranks of the first matrix of
  // the wave's columns, or of gate and up), and each thread the output rows it will write.
  const bool lora = L.n_mats > 0 && mid != nullptr;
  const int jlo = GATED || !lora ? 0 : matrix_of(L, min(n0, n_out - 1));
  int s_lo = 0, ns = 0, ta = 0, tb = 0, te = 0, tl0 = 0, tl1 = 0;
  auto table = [&](int t0) __attribute__((always_inline)) {
    const int s = s_lo + ks + KW * min(t0 + lane, ns - 1);
    ta = r.seg_adapter[s];
    tb = r.seg_start[s] - p0;
    te = r.seg_start[s + 1] - p0;
  };
  if (lora) {
    s_lo = __builtin_amdgcn_readfirstlane(r.seg_of[p0]);
    const int left = __builtin_amdgcn_readfirstlane(r.seg_of[p1 - 1]) - s_lo - ks;
    ns = left >= 0 ? left / KW + 1 : 0;
    if (ns > 0) table(0);
  }
  int orow[4], olast[4];  // (RB of them)
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    const int row = min(p0 + q * 32 + li, T - 1);
    orow[q] = r.tok_perm[row];
    olast[q] = last_out != nullptr ? r.last_of[row] : -1;
  }

  f32x16_t acc[RB][2];
#pragma unroll
  for (int rb = 0; rb < RB; ++rb) acc[rb][0] = acc[rb][1] = f32x16_t{};

  // Step i reads ring slot i % D and weight set i % D, in eight units e: the products of word e (16-input slice e / 2,
  // block e % 2) run while word e + 1 is dequantised and, at each even unit, the next slice's x operands are read. The
  // step's barrier sits before its last slice (a lone column wave needs none: it reads only what it staged, and the waves
  // drift apart: 384 rows of 6144 -> 2048 30 -> 26 us): past it every wave has the step's last operands in registers, so the
  // slot takes step i + D's rows, and the next step's first operands are read while the last products run. Words are
  // loaded D steps ahead too, once the step's last word is converted. Loads complete in order; past the last step
  // they read nothing, so the number in flight at every wait stays the same.
  SliceW w0, w1, w2;
  uint4 a0[RB], a1[RB], bw;  // operands of the even and odd 16-input slices; the next word's weights
  auto scale_of = [&](const SliceW& st, int cb, float& sv, float& zs) __attribute__((always_inline)) {
    sv = bf16_to_f32(st.s[cb]);
    zs = (asym ? (float)st.z[cb] : 8.0f) * sv;
  };
  auto step = [&](auto slot, SliceW& st, const SliceW& nst, int i) __attribute__((always_inline)) {
    constexpr int S = decltype(slot)::value;
    using Next = std::integral_constant<int, (S + 1) % D>;
    float sv[2], zs[2], nsv, nzs;
    scale_of(st, 0, sv[0], zs[0]);
    scale_of(st, 1, sv[1], zs[1]);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int u = e >> 1, cb = e & 1;
      if (e == 6) {
        __builtin_amdgcn_sched_barrier(0);
        MLORA_WAIT_VM((D - 2) * kXI + (D - 1) * kWI);  // x(i + 1) has landed, and the step's operands are read
        if constexpr (CW > 1) step_sync();             // (a lone column wave reads only the chunks it staged itself)
        dma_x(slot, i + D);
        __builtin_amdgcn_sched_barrier(0);
      }
      const uint4 cur = bw;
      if (e < 7) {
        bw = dequant_word(st.w[(e + 1) >> 1][(e + 1) & 1], sv[(e + 1) & 1], zs[(e + 1) & 1]);
      } else {
        scale_of(nst, 0, nsv, nzs);
        bw = dequant_word(nst.w[0][0], nsv, nzs);
      }
      if (cb == 0) {
        if (u < 3)
          read_x(slot, u + 1, (u & 1) ? a0 : a1);
        else
          read_x(Next{}, 0, a0);
      }
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) acc[rb][cb] = mfma32(cur, (u & 1) ? a1[rb] : a0[rb], acc[rb][cb]);
#pragma unroll
      for (int rb = 0; rb < RB; ++rb) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);                   // one MFMA
        if (cb == 0) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);      // one LDS read
        __builtin_amdgcn_sched_group_barrier(0x002, (19 + RB - 1) / RB, 0);  // a share of the conversion
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    fetch_w(st, i + D);
    __builtin_amdgcn_sched_barrier(0);
  };
  dma_x(I0{}, 0);
  __builtin_amdgcn_sched_barrier(0);
  fetch_w(w0, 0);
  __builtin_amdgcn_sched_barrier(0);
  dma_x(I1{}, 1);
  __builtin_amdgcn_sched_barrier(0);
  fetch_w(w1, 1);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (D == 3) {
    dma_x(I2{}, 2);
    __builtin_amdgcn_sched_barrier(0);
    fetch_w(w2, 2);
    __builtin_amdgcn_sched_barrier(0);
  }
  if (ns > 0 && ta != 0) {
    tl0 = live_rank(L, ta, jlo);
    if constexpr (GATED) tl1 = live_rank(L, ta, 1);
  }
  __builtin_amdgcn_sched_barrier(0);
  MLORA_WAIT_VM((D - 1) * (kXI + kWI));  // x(0) and its words have landed
  step_sync();
  read_x(I0{}, 0, a0);
  {
    float sv, zs;
    scale_of(w0, 0, sv, zs);
    bw = dequant_word(w0.w[0][0], sv, zs);
  }
  // whole rounds of D steps in a loop with no other exit, then the rest
  const int full = steps - steps % D;
  for (int i = 0; i < full; i += D) {
    step(I0{}, w0, w1, i);
    if constexpr (D == 3) {
      step(I1{}, w1, w2, i + 1);
      step(I2{}, w2, w0, i + 2);
    } else {
      step(I1{}, w1, w0, i + 1);
    }
  }
  if (full < steps) {
    step(I0{}, w0, w1, full);
    if constexpr (D == 3) {
      if (full + 1 < steps) step(I1{}, w1, w2, full + 1);
    }
  }
  MLORA_WAIT_VM(0);

  // LoRA second factor: the wave's segments. A segment's sB rows (32 columns x ranks rc .. rc + 63, rows of 128 bytes
  // swizzled like x) are staged in a slot of the wave's own by loads that write LDS directly, two segments ahead of the
  // products; the first factors of the tile's rows are operands in registers, rows outside the segment and ranks past
  // the adapter's live rank set to zero (the first factors past a live rank are not written).
  lds_sync();  // every wave is done with the ring
  if (ns > 0 && wout) {
    const int jhi = GATED ? 1 : matrix_of(L, min(n0 + kSlCols, n_out) - 1);
    auto lora_matrix = [&](int j, auto first) __attribute__((always_inline)) {
      const int oj = col_offset(L, j), cj = L.cols[j], capj = L.cap[j], rho = rank_offset(L, j);
      const bool allin = GATED || (n0 >= oj && n0 + kSlCols <= oj + cj);
      for (int rc = 0; rc < capj; rc += kSlRanks) {
        uint4 m[RB][4];
        for (int t0 = 0; t0 < ns; t0 += kWave) {
          if (ns > kWave) table(t0);
          const int tl = t0 == 0 && j == jlo ? tl0 : GATED && t0 == 0 ? tl1 : ta == 0 ? 0 : live_rank(L, ta, j);
          const int cnt = min(kWave, ns - t0);
          // segment i's sB rows of block q into the wave's slot of sl_x0 or sl_x1 (past the last: the last again)
          auto load_b = [&](auto slot, int q, int i) __attribute__((always_inline)) {
            const int ic = min(i, cnt - 1);
            const int a = __builtin_amdgcn_readlane(ta, ic), live = __builtin_amdgcn_readlane(tl, ic);
            const int sbs = sb_stride(live, capj);  // at least 8: capj > rc >= 0
            const __amdgpu_buffer_rsrc_t bres = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(L.pool + (int64_t)a * L.pool_stride + L.off_b[j]), (short)0, cj * sbs * 2, 0x00020000);
            uint8_t* dst = slot_of(slot) + wave * 4096;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int row = 8 * e + (lane >> 3);
              const int col = GATED ? g0 + row : n0 + 2 * row + q - oj;
              const int cc = col >= 0 && col < cj ? col : 0;
              const uint32_t off = (uint32_t)((cc * sbs + min(rc + 8 * swz_slot(row, lane & 7), sbs - 8)) * 2);
              __builtin_amdgcn_raw_ptr_buffer_load_lds(bres, (lds_void*)(dst + e * 1024), 16, off, 0, 0, 0);
            }
          };
          // its products of block q, once the slot's rows have landed (the other slot's 4 loads in flight); the slot
          // then takes segment `next`
          auto apply = [&](auto slot, auto block, int i, int next) __attribute__((always_inline)) {
            constexpr int q = decltype(block)::value;
            MLORA_WAIT_VM(4);
            uint4 bv[4];
            read_block(bv, at, lds_of(slot) + wave * 4096);
            load_b(slot, q, next);
            const int ic = min(i, cnt - 1);
            const int rk = i < cnt ? min(__builtin_amdgcn_readlane(tl, ic) - rc, kSlRanks) : 0;
            if (rk <= 0) return;
            const int sb = __builtin_amdgcn_readlane(tb, ic), se = __builtin_amdgcn_readlane(te, ic);
            const bool ragged = (rk & 15) != 0;
            const int cc = GATED ? 0 : n0 + 2 * li + q - oj;
            const bool cin = cc >= 0 && cc < cj;
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              if (ragged) bv[u] = keep_first(bv[u], rk - (16 * u + 8 * h));
              if (!allin) bv[u] = cin ? bv[u] : make_uint4(0, 0, 0, 0);
            }
#pragma unroll
            for (int rb = 0; rb < RB; ++rb) {
              if (rb * 32 >= se || rb * 32 + 32 <= sb) continue;
              const int row = rb * 32 + li;
              const bool rin = row >= sb && row < se;
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                if (16 * u >= rk) break;
                uint4 v = rin ? m[rb][u] : make_uint4(0, 0, 0, 0);
                if (ragged) v = keep_first(v, rk - (16 * u + 8 * h));
                acc[rb][q] = mfma32(bv[u], v, acc[rb][q]);
              }
            }
          };
          // (each segment's rows are asked for before the first factors, which then arrive with them)
          load_b(I0{}, GATED ? decltype(first)::value : 0, 0);
          load_b(I1{}, GATED ? decltype(first)::value : 1, GATED ? 1 : 0);
          if (t0 == 0) {
#pragma unroll
            for (int rb = 0; rb < RB; ++rb)
#pragma unroll
              for (int u = 0; u < 4; ++u) {
                const int row = p0 + rb * 32 + li, q = rc + 16 * u + 8 * h;
                m[rb][u] = (row < p1 && q < capj)
                               ? *reinterpret_cast<const uint4*>(mid + (int64_t)row * L.rank_cap + rho + q)
                               : make_uint4(0, 0, 0, 0);
              }
          }
          if constexpr (GATED) {
            using G = decltype(first);
            for (int i = 0; i < cnt; i += 2) {
              apply(I0{}, G{}, i, i + 2);
              apply(I1{}, G{}, i + 1, i + 3);
            }
          } else {
            for (int i = 0; i < cnt; ++i) {
              apply(I0{}, I0{}, i, i + 1);
              apply(I1{}, I1{}, i, i + 1);
            }
          }
          MLORA_WAIT_VM(0);  // the last slot loads have landed before the slots are used again
        }
      }
    };
    if constexpr (GATED) {
      lora_matrix(0, I0{});  // gate: the products of block 0
      lora_matrix(1, I1{});  // up: block 1
    } else {
      for (int j = jlo; j <= jhi; ++j) lora_matrix(j, I0{});
    }
  }

  // The slices' tiles added in slice order, one row block at a time: block 0's sums through sl_x0, block 1's through
  // sl_x1, as float4 [wave][g][lane] (lane l holds row l & 31 and index 8 g + 4 (l >> 5) .. +3 of the block); a thread adds
  // one position (column wave, g, lane) of both blocks, of every slice, at a time.
  float4* r0 = reinterpret_cast<float4*>(sl_x0);
  float4* r1 = reinterpret_cast<float4*>(sl_x1);
#pragma unroll
  for (int q = 0; q < RB; ++q) {
    lds_sync();  // every wave is done with its slots (and the previous block's sums are read)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const f32x16_t& c0 = acc[q][0];
      const f32x16_t& c1 = acc[q][1];
      r0[(wave * 4 + e) * 64 + lane] = make_float4(c0[4 * e], c0[4 * e + 1], c0[4 * e + 2], c0[4 * e + 3]);
      r1[(wave * 4 + e) * 64 + lane] = make_float4(c1[4 * e], c1[4 * e + 1], c1[4 * e + 2], c1[4 * e + 3]);
    }
    lds_sync();
    for (int pos = tid; pos < CW * 256; pos += W * 64) {
      const int c = pos >> 8, g = (pos >> 6) & 3, ln = pos & 63;
      const int row = p0 + q * 32 + (ln & 31);
      const int colw = nt * CW + c;  // the position's column wave
      if (row >= T || (GATED ? colw * 32 >= inter : colw * kSlCols >= n_out)) continue;
      const int64_t orig = orow[q], lq = olast[q];
      float4 u0 = r0[pos], u1 = r1[pos];
#pragma unroll 3
      for (int v = 1; v < KW; ++v) {
        const float4 t0 = r0[v * CW * 256 + pos], t1 = r1[v * CW * 256 + pos];
        u0.x += t0.x, u0.y += t0.y, u0.z += t0.z, u0.w += t0.w;
        u1.x += t1.x, u1.y += t1.y, u1.z += t1.z, u1.w += t1.w;
      }
      if constexpr (GATED) {
        const uint2 v = silu_mul4(make_uint2(pack_bf16x2(u0.x, u0.y), pack_bf16x2(u0.z, u0.w)),
                                  make_uint2(pack_bf16x2(u1.x, u1.y), pack_bf16x2(u1.z, u1.w)));
        const int col = colw * 32 + g * 8 + (ln >> 5) * 4;
        store4(y + orig * y_stride + col, lq >= 0 ? last_out + lq * inter + col : nullptr, v.x, v.y, 4,
               vec & kStoreVec);
      } else {
        const int col = colw * kSlCols + g * 16 + (ln >> 5) * 8;
        if (col >= n_out) continue;
        const uint32_t v[4] = {pack_bf16x2(u0.x, u1.x), pack_bf16x2(u0.y, u1.y), pack_bf16x2(u0.z, u1.z),
                               pack_bf16x2(u0.w, u1.w)};
        store8(y + orig * y_stride + col, lq >= 0 ? last_out + lq * n_out + col : nullptr, v, n_out - col, vec, wide);
      }
    }
  }
}

}  // namespace

// The form of a product over `tokens` rows with the least estimated time, and that estimate in microseconds. A workgroup
// takes a CU (its LDS): a round of them lasts a fixed time (launch, first loads, the sums' exchange and the stores) plus a
// time per step, both measured on full rounds.
SliceForm slice_form(int64_t tokens, int32_t columns, int32_t k, double* us) {
  // measured with K = 2048 and 6144 over 32, 384 and 2311 rows of 2048 to 12288 columns: 10.8 and 18.5 us a round,
  // 15.6 and 25.6, 18.5 and 36.4, 35 and 78
  struct Cost {
    SliceForm f;
    double fixed, step;
  };
  static const Cost costs[] = {{{1, 1, 8}, 7.0, 0.95}, {{2, 1, 8}, 10.6, 1.25}, {{2, 2, 4}, 9.5, 1.12}, {{3, 4, 2}, 13.5, 1.34}};
  const int cus = device_cus();
  SliceForm best = costs[0].f;
  double least = 0.0;
  for (const Cost& c : costs) {
    const int64_t wgs = ((tokens + 32 * c.f.rb - 1) / (32 * c.f.rb)) * ((columns / kSlCols + c.f.cw - 1) / c.f.cw);
    const int64_t rounds = (wgs + cus - 1) / cus, steps = (k / kTK + c.f.kw - 1) / c.f.kw;
    const double t = (double)rounds * (c.fixed + c.step * (double)steps);
    if (least == 0.0 || t < least) {
      least = t;
      best = c.f;
    }
  }
  if (us != nullptr) *us = least;
  return best;
}

int launch_slice(const mlora_int4_t& w, const mlora_lora_t& L, const mlora_route_t& r, const uint16_t* x,
                 int64_t x_stride, uint16_t* y, int64_t y_stride, uint16_t* last_out, int32_t n_out,
                 const uint16_t* mid, hipStream_t stream, int32_t inter, bool residual) {
  if (r.tokens == 0 || n_out == 0) return MLORA_OK;
  if (w.columns % kSlCols || (residual && inter > 0)) return MLORA_EINVAL;
  if (inter > 0 && (inter % 32 || n_out != 2 * inter)) return MLORA_EINVAL;
  const SliceForm f = slice_form(r.tokens, w.columns, w.k, nullptr);
  const int n_tiles = (w.columns / kSlCols + f.cw - 1) / f.cw;
  const int m_tiles = (int)((r.tokens + 32 * f.rb - 1) / (32 * f.rb));
  if ((int64_t)n_tiles * m_tiles > INT_MAX) return MLORA_EOVERFLOW;
  const int out_cols = inter > 0 ? inter : n_out;
  auto aligned = [&](int bytes) {
    return reinterpret_cast<uintptr_t>(y) % bytes == 0 && y_stride % (bytes / 2) == 0 &&
           (last_out == nullptr ||
            (reinterpret_cast<uintptr_t>(last_out) % bytes == 0 && out_cols % (bytes / 2) == 0));
  };
  const int32_t vec = (aligned(8) ? kStoreVec : 0) | (residual ? kStoreResidual : 0);
  const int32_t wide = aligned(16) ? 1 : 0;
  auto launch = [&](auto kernel, int waves) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)(n_tiles * m_tiles)), dim3(waves * 64), 0, stream, w, L, r, x, x_stride,
                       y, y_stride, last_out, n_out, mid, n_tiles, m_tiles, vec, wide, inter);
  };
#define SLICE_CASE(RB, CW, KW)                                        \
  if (f.rb == RB && f.cw == CW && f.kw == KW) {                       \
    if (inter > 0)                                                    \
      launch(slice_kernel<RB, CW, KW, true>, CW * KW);                \
    else                                                              \
      launch(slice_kernel<RB, CW, KW, false>, CW * KW);               \
  }
  SLICE_CASE(1, 1, 8)
  SLICE_CASE(2, 1, 8)
  SLICE_CASE(2, 2, 4)
  SLICE_CASE(3, 4, 2)
#undef SLICE_CASE
  return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
}
