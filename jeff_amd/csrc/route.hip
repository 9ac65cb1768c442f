// Adapter routing: request rows -> segments of the sorted order, one segment per adapter present.
// Replaces the reference's per-tile lookup adp[t // row_len] (engine/fast_path.py:167,189;
// engine/int4_kernels.py:72,113) with a stable order, so every adapter's tokens are contiguous.
#include "mlora_common.h"

namespace {

constexpr int kRouteThreads = 1024;
constexpr int kRouteWaves = kRouteThreads / 64;
constexpr int kWaveRequests = 2;                           // request rows per wave
constexpr int kRouteRequests = kRouteWaves * kWaveRequests;  // ... per workgroup
constexpr int kLongRow = 1024;                             // rows of more tokens are written by the whole workgroup
constexpr int kIndexBits = 13;  // request index in the low bits of a sort key: MLORA_MAX_REQUESTS = 2^13
static_assert((1 << kIndexBits) == MLORA_MAX_REQUESTS, "key layout");
static_assert(MLORA_MAX_POOL_ROWS <= (1 << (31 - kIndexBits)), "a key must stay below the padding key");

__device__ __forceinline__ int wave_total(int v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// More than 64 request rows: a workgroup per 32 of them, and no sort. The keys (adapter, request) are all distinct, so a
// request's sorted position is the number of smaller keys, its first token the sum of their lengths, and its segment the
// number of adapters below its own among those present (a bit map's population count): every workgroup reads all the
// requests (at most 8192) into LDS, and a wave counts for two of them at a time, then writes their tokens. One workgroup
// sorting the keys in LDS and writing every token took 14 us at 256 requests of one token, 27 at 643, 117 at 4096 and
// 47 at 512 requests of 159,488 tokens.
__global__ __launch_bounds__(kRouteThreads) void route_kernel(const int32_t* __restrict__ adp,
                                                             const int32_t* __restrict__ cu, int32_t row_len,
                                                             mlora_route_t r, int32_t pool_rows) {
  __shared__ uint32_t keys[MLORA_MAX_REQUESTS];
  __shared__ int32_t lens[MLORA_MAX_REQUESTS];
  __shared__ uint32_t present[MLORA_MAX_POOL_ROWS / 32];  // a bit per pool row
  __shared__ int32_t l_start[kRouteRequests], l_len[kRouteRequests], l_ps[kRouteRequests], l_seg[kRouteRequests];
  __shared__ int32_t status, seq_ok;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int B = r.requests;
  const int64_t T = r.tokens;
  const int words = (pool_rows + 31) / 32;
  if (tid == 0) {
    status = 0;
    seq_ok = 1;
  }
  if (tid < kRouteRequests) l_len[tid] = 0;
  for (int i = tid; i < words; i += kRouteThreads) present[i] = 0;
  __syncthreads();
  // the offsets must start at 0, never decrease and end at the token count
  bool bad = cu != nullptr && tid == 0 && (cu[0] != 0 || (int64_t)cu[B] != T);
  bool bad_adapter = false;
  for (int i = tid; i < B; i += kRouteThreads) {
    int a = adp[i];
    // (offsets are compared, not subtracted: two more than 2^31 apart differ by a wrapped length of either sign)
    int len = row_len;
    if (cu != nullptr) {
      const int c0 = cu[i], c1 = cu[i + 1];
      bad |= c1 < c0;
      len = c1 < c0 ? 0 : (int)((uint32_t)c1 - (uint32_t)c0);
    }
    if (a < 0 || a >= pool_rows) {
      a = 0;
      bad_adapter = true;
    }
    keys[i] = ((uint32_t)a << kIndexBits) | (uint32_t)i;
    lens[i] = len;
    atomicOr(&present[a >> 5], 1u << (a & 31));
  }
  if (bad) atomicAnd(&seq_ok, 0);
  if (bad_adapter) atomicOr(&status, MLORA_ROUTE_BAD_ADAPTER);
  __syncthreads();
  if (!seq_ok) {  // unusable offsets: identity routing through row 0 (no LoRA), flagged
    for (int64_t p = (int64_t)blockIdx.x * kRouteThreads + tid; p < T; p += (int64_t)gridDim.x * kRouteThreads) {
      r.tok_perm[p] = (int32_t)p;
      r.last_of[p] = -1;
      r.seg_of[p] = 0;
    }
    if (blockIdx.x != 0) return;
    for (int i = tid; i < B; i += kRouteThreads) r.req_order[i] = i;
    if (tid == 0) {
      *r.num_segs = 1;
      r.seg_start[0] = 0;
      r.seg_start[1] = (int32_t)T;
      r.seg_adapter[0] = 0;
      *r.status = MLORA_ROUTE_BAD_SEQLENS;
    }
    return;
  }
  const int q0 = blockIdx.x * kRouteRequests + wave * kWaveRequests;  // the wave's requests q0, q0 + 1
  uint32_t key[kWaveRequests], base[kWaveRequests];
  int rank[kWaveRequests], ps[kWaveRequests];
  bool seen[kWaveRequests];  // an earlier request of the same adapter
#pragma unroll
  for (int e = 0; e < kWaveRequests; ++e) {
    key[e] = q0 + e < B ? keys[q0 + e] : 0u;
    base[e] = key[e] & ~((1u << kIndexBits) - 1);
    rank[e] = ps[e] = 0;
    seen[e] = false;
  }
  for (int j = lane; j < B; j += 64) {
    const uint32_t k = keys[j];
    const int l = lens[j];
#pragma unroll
    for (int e = 0; e < kWaveRequests; ++e) {
      const bool less = k < key[e];
      rank[e] += less ? 1 : 0;
      ps[e] += less ? l : 0;
      seen[e] = seen[e] || (less && k >= base[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < kWaveRequests; ++e) {
    const int q = q0 + e;
    if (q >= B) break;
    const int a = (int)(key[e] >> kIndexBits);
    int below = 0;  // adapters present below a
    for (int i = lane; i <= (a >> 5); i += 64)
      below += __popc(i < (a >> 5) ? present[i] : present[i] & ((1u << (a & 31)) - 1));
    const int pos = wave_total(rank[e]), p0 = wave_total(ps[e]), seg = wave_total(below);
    const bool first = __ballot(seen[e]) == 0;
    const int l = lens[q], start = cu != nullptr ? cu[q] : q * row_len;
    if (lane == 0) {
      r.req_order[pos] = q;
      if (first) {
        r.seg_adapter[seg] = a;
        r.seg_start[seg] = p0;
      }
    }
    if (l > kLongRow) {
      if (lane == 0) {
        const int at = wave * kWaveRequests + e;
        l_start[at] = start;
        l_len[at] = l;
        l_ps[at] = p0;
        l_seg[at] = seg;
      }
      continue;
    }
    for (int t = lane; t < l; t += 64) {
      r.tok_perm[p0 + t] = start + t;
      r.last_of[p0 + t] = t == l - 1 ? q : -1;
      r.seg_of[p0 + t] = seg;
    }
  }
  if (blockIdx.x == 0 && wave == 0) {
    int n = 0;
    for (int i = lane; i < words; i += 64) n += __popc(present[i]);
    n = wave_total(n);
    if (lane == 0) {
      *r.num_segs = n;
      r.seg_start[n] = (int32_t)T;
      *r.status = status;
    }
  }
  __syncthreads();
  for (int i = 0; i < kRouteRequests; ++i) {  // the long rows
    const int l = l_len[i];
    if (l == 0) continue;
    const int q = blockIdx.x * kRouteRequests + i;
    for (int t = tid; t < l; t += kRouteThreads) {
      r.tok_perm[l_ps[i] + t] = l_start[i] + t;
      r.last_of[l_ps[i] + t] = t == l - 1 ? q : -1;
      r.seg_of[l_ps[i] + t] = l_seg[i];
    }
  }
}

// Passes of at most 64 request rows: one workgroup per request. Wave 0 of every workgroup routes all of them in
// registers (one request per lane, a bitonic sort of the same keys by lane shuffles, prefix sums by shuffles; a few
// hundred instructions, cheaper than sharing the result between workgroups); workgroup 0 writes the per-request and
// per-segment outputs, and after one barrier workgroup b writes the tokens of the request at sorted position b, so
// the token stores spread over as many CUs as there are requests. The outputs are the block kernel's, bit for bit.
constexpr int kSmallRequests = 64;
constexpr int kSmallThreads = 256;

__global__ __launch_bounds__(kSmallThreads) void route_small_kernel(const int32_t* __restrict__ adp,
                                                                   const int32_t* __restrict__ cu, int32_t row_len,
                                                                   mlora_route_t r, int32_t pool_rows) {
  __shared__ int32_t s_start[kSmallRequests], s_len[kSmallRequests], s_ps[kSmallRequests];
  __shared__ int32_t s_seg[kSmallRequests], s_q[kSmallRequests];
  __shared__ int32_t s_ok;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int B = r.requests;
  const int64_t T = r.tokens;
  if (wave == 0) {
    const bool live = lane < B;
    int c0 = 0, c1 = 0;
    bool bad = false;
    if (cu != nullptr) {
      if (live) {
        c0 = cu[lane];
        c1 = cu[lane + 1];
        bad = c1 < c0;
      }
      if (lane == 0) bad = bad || cu[0] != 0 || (int64_t)cu[B] != T;
    }
    const bool seq_ok = __ballot(bad) == 0;
    int a = live ? adp[lane] : 0;
    const bool bad_a = live && (a < 0 || a >= pool_rows);
    if (bad_a) a = 0;
    const int len = cu != nullptr ? c1 - c0 : row_len;
    const int start = cu != nullptr ? c0 : lane * row_len;
    uint32_t key = live ? (((uint32_t)a << kIndexBits) | (uint32_t)lane) : 0xFFFFFFFFu;  // padding sorts last
#pragma unroll
    for (int k = 2; k <= 64; k <<= 1)
#pragma unroll
      for (int j = k >> 1; j > 0; j >>= 1) {
        const uint32_t other = __shfl_xor(key, j);
        const bool up = (lane & k) == 0, lower = (lane & j) == 0;
        key = (lower == up) ? min(key, other) : max(key, other);
      }
    const int q = (int)(key & ((1u << kIndexBits) - 1));  // the request at sorted position `lane`
    const int ada = (int)(key >> kIndexBits);
    const int qlen_any = __shfl(len, q & 63);  // every lane takes part in the shuffle
    const int qlen = live ? qlen_any : 0;
    const int qstart = __shfl(start, q & 63);
    const int prev = __shfl_up(ada, 1);
    const bool first = live && (lane == 0 || prev != ada);
    int lsum = qlen, fsum = first ? 1 : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int yl = __shfl_up(lsum, o), yf = __shfl_up(fsum, o);
      if (lane >= o) {
        lsum += yl;
        fsum += yf;
      }
    }
    const int pstart = lsum - qlen, seg = fsum - 1;
    const int nseg = __shfl(fsum, 63), total = __shfl(lsum, 63);
    const bool any_bad_adapter = __ballot(bad_a) != 0;  // every lane takes part in the vote
    const bool lead = blockIdx.x == 0;  // the one workgroup that writes the per-request and per-segment outputs
    if (seq_ok) {
      if (live) {
        if (lead) {
          r.req_order[lane] = q;
          if (first) {
            r.seg_adapter[seg] = ada;
            r.seg_start[seg] = pstart;
          }
        }
        s_start[lane] = qstart;
        s_len[lane] = qlen;
        s_ps[lane] = pstart;
        s_seg[lane] = seg;
        s_q[lane] = q;
      }
      if (lane == 0 && lead) {
        *r.num_segs = nseg;
        r.seg_start[nseg] = total;
        *r.status = any_bad_adapter ? MLORA_ROUTE_BAD_ADAPTER : 0;
      }
    }
    if (lane == 0) s_ok = seq_ok ? 1 : 0;
  }
  __syncthreads();
  if (!s_ok) {  // unusable offsets: identity routing through row 0 (no LoRA), flagged
    for (int64_t p = (int64_t)blockIdx.x * kSmallThreads + tid; p < T; p += (int64_t)gridDim.x * kSmallThreads) {
      r.tok_perm[p] = (int32_t)p;
      r.last_of[p] = -1;
      r.seg_of[p] = 0;
    }
    if (blockIdx.x != 0) return;
    for (int i = tid; i < B; i += kSmallThreads) r.req_order[i] = i;
    if (tid == 0) {
      *r.num_segs = 1;
      r.seg_start[0] = 0;
      r.seg_start[1] = (int32_t)T;
      r.seg_adapter[0] = 0;
      *r.status = MLORA_ROUTE_BAD_SEQLENS;
    }
    return;
  }
  for (int i = blockIdx.x; i < B; i += gridDim.x) {  // one request per workgroup, its tokens across the threads
    const int start = s_start[i], l = s_len[i], ps = s_ps[i], sg = s_seg[i], q = s_q[i];
    for (int t = tid; t < l; t += kSmallThreads) {
      r.tok_perm[ps + t] = start + t;
      r.last_of[ps + t] = t == l - 1 ? q : -1;
      r.seg_of[ps + t] = sg;
    }
  }
}

__global__ __launch_bounds__(256) void dequant_kernel(mlora_int4_t w, uint16_t* __restrict__ out) {
  const int64_t idx = (int64_t)blockIdx.x * 256 + threadIdx.x;
  const int words_per_col = w.k / 8;
  if (idx >= (int64_t)words_per_col * w.out) return;
  const int c = (int)(idx / words_per_col), i = (int)(idx % words_per_col);
  const int g = (8 * i) / w.group;
  const float s = mlora::bf16_to_f32(w.scales[(int64_t)g * w.columns + c]);
  const float z = w.zeros != nullptr ? (float)w.zeros[(int64_t)g * w.columns + c] : 8.0f;
  const uint32_t word = (uint32_t)w.words[(int64_t)i * w.columns + c];
  *reinterpret_cast<uint4*>(out + (int64_t)c * w.k + 8 * i) = mlora::dequant_word(word, s, z * s);
}

}  // namespace

int launch_route(const int32_t* adp, const int32_t* cu, int32_t row_len, const mlora_route_t& r, int32_t pool_rows,
                 hipStream_t stream) {
  if (r.requests <= kSmallRequests)
    hipLaunchKernelGGL(route_small_kernel, dim3((unsigned)(r.requests > 1 ? r.requests : 1)), dim3(kSmallThreads), 0, stream, adp,
                       cu, row_len, r, pool_rows);
  else
    hipLaunchKernelGGL(route_kernel, dim3((unsigned)((r.requests + kRouteRequests - 1) / kRouteRequests)),
                       dim3(kRouteThreads), 0, stream, adp, cu, row_len, r, pool_rows);
  return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
}

int launch_dequant(const mlora_int4_t& w, uint16_t* out, hipStream_t stream) {
  const int64_t n = (int64_t)(w.k / 8) * w.out;
  if (n == 0) return MLORA_OK;
  hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, w, out);
  return hipGetLastError() == hipSuccess ? MLORA_OK : MLORA_ELAUNCH;
}
