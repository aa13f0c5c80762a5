// Backward of the candidate-list sparse attention (replaces fastseg.py:81-110 _attn_bwd and its caller
// fastseg.py:158-170 _SparseAttnFn.backward).  With p_j the softmax weight of valid slot j (from the
// forward's log-sum-exp), Dq = do . o, dp_j = do . v_j and ds_j = p_j (dp_j - Dq):
//   dq = scale * sum_j ds_j k_j,   dk[cand_j] += scale * ds_j q,   dv[cand_j] += p_j do.
//
// bwd_query_kernel, one wavefront per query: the valid slots of a round of 64 are compacted (typically a quarter of
// a candidate row names a key), then 64 / L slots at a time are worked on by L lanes each (L lanes of 8 dimensions
// hold a row): the key and value rows are read once, in whole lines, the two dot products are finished inside the
// group, and dq takes the key row that is still in registers.  dk and dv then take one of two routes:
//  * with a workspace (the Python binding's default up to 131072 positions): every valid slot's ds and p are written
//    there, the slots are sorted by key in a stable order (queries ascending, slots ascending) and
//    bwd_keys_kernel adds each key's contributions from its own consecutive list.  Which entries a lane adds, and
//    how the lanes' and wavefronts' parts are added, follows from the list alone: dk and dv are bit-reproducible.
//  * without one, each slot's dk and dv rows receive float32 atomic adds (the reference's scheme, whose order
//    depends on scheduling: reproducible to float32 rounding only).
//
// The sort is one stable most-significant-digit pass over chunks of queries (bwd_count_kernel, bwd_scan_kernel,
// bwd_scatter_kernel) into at most 2048 buckets of 16 (or more) consecutive keys; bwd_keys_kernel lists a bucket's
// entries key by key in LDS.  The cost is linear in the slots but for the buckets' finding of their keys (wider buckets
// past 32768 keys).  Past 2^26 slots, 2^22 queries or 2^21 keys the pairs and queries are sorted, and the keys summed,
// in parts one after another, which keeps the order.  Scanning all candidate rows once per block of keys instead (one
// wavefront per block, a serial chain over the queries, quadratic in T) took 6.2 ms of the 7.0 ms forward and backward
// of a (2, 6, 4096, 64) float16 layer with 52 candidates a row (12 valid); this takes 0.13 ms:
// count 9, scan 14, scatter 19 and keys 82 us.  What is left in the key kernel is latency (about 8 us per bucket, six
// rounds of workgroups) and the bucket of the sink, which every query names: its workgroups are started first and
// take 82 us.  8 or 32 keys per bucket, 4 or 16 wavefronts, tiles of 1024 entries: 0.19-0.25 against 0.19 ms for the
// whole backward.  bwd_query_kernel: 42 us (85 with a lane per slot and a second pass over the key rows).
#include "common.hpp"

namespace ta {

struct BwdParams {
  const void *q, *k, *v, *o, *dout;
  int64_t qsb, qsh, qst, ksb, ksh, kst, vsb, vsh, vst, osb, osh, ost, dsb, dsh, dst;
  const int32_t* cand;   // (B,H,T,KC) contiguous
  const float* lse;      // (B,H,T) contiguous
  void* dq;              // (B,H,T,D) rows, input dtype
  float *dk, *dv;        // (B,H,Tk,D) rows, float32: accumulated into (atomics) or written (workspace)
  // the sorted route's workspace, for the `pairs` (b,h) from bh0 on and their queries [t0, t0 + Ts):
  float2* dsp;           // (pairs,Ts,KC) per-slot (ds, p), written where the slot is valid, or null
  uint2* ent;            // (pairs,Ts*KC) sorted entries: slot index, query << kLowBits | key within its bucket
  int32_t* cnt;          // per pair: [bucket][chunk] counts, then starts; one more word: the number of entries
  int B, H, T, Tk, KC, D;
  int bh0, t0, Ts;       // this launch's pairs and queries
  int j0, Tj;            // the keys being summed: [j0, j0 + Tj)
  float scale;
  int rows_al;           // q, o and do rows, dq, dk and dv are 16-byte aligned
  int CQ, NC;            // queries per chunk, chunks of the Ts queries
  int wlog, NB;          // log2 of a bucket's keys, buckets
  int64_t gq[3], gk[3], gv[3];   // strides (b, h, row) of dq, dk, dv
};

constexpr int kBwdMaxD = 256;
constexpr int kLowBits = 10;          // bits of the key within its bucket
constexpr int kMaxBuckets = 2048;
constexpr int kChunkSlots = 4096;     // slots per chunk (at least one query)
// At most this many chunks, larger ones past it (from about 20,000 queries of 52 slots on): the scan of a pair's counts
// is one workgroup's, and with chunks of 4096 slots throughout it grew with the square of the queries: 6.2 of the
// 17.7 ms of (1, 1, 262144, 64), against 0.5 of 12.1
constexpr int kMaxChunks = 256;
constexpr int kBwdWaves = 4;          // wavefronts of the query, count and scatter kernels
constexpr int kKeyWaves = 8;
constexpr int kTile = 2048;           // entries sorted in LDS at a time
constexpr int64_t kSortSlots = 1 << 26;
constexpr int kHeavy = 96;            // a key with more entries in a tile is shared by the workgroup's wavefronts

// Lanes per row: the power of two of 8-dimension slices that covers D (lanes past D hold zeros).
__host__ __device__ constexpr int bwd_lanes(int D) {
  int l = 1;
  while (l * 8 < D) l *= 2;
  return l;
}

// 8 elements at p (zeros past the row); vector loads where rows are aligned
template <typename T>
__device__ __forceinline__ void load8(const T* p, bool in, bool al, float (&x)[8]) {
  if (!in) {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = 0.0f;
  } else if (al) {
    load_row<T, 8>(p, x);
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) x[i] = to_f32(p[i]);
  }
}

template <typename T>
__device__ __forceinline__ void store8(T* p, bool al, const float (&x)[8]) {
  if (al) {
    if constexpr (sizeof(T) == 4) {
      reinterpret_cast<float4*>(p)[0] = make_float4(x[0], x[1], x[2], x[3]);
      reinterpret_cast<float4*>(p)[1] = make_float4(x[4], x[5], x[6], x[7]);
    } else {
      union { T e[8]; uint4 u; } r;
#pragma unroll
      for (int i = 0; i < 8; ++i) r.e[i] = from_f32<T>(x[i]);
      *reinterpret_cast<uint4*>(p) = r.u;
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) p[i] = from_f32<T>(x[i]);
  }
}

// Sum over the lanes that hold the same slice of different slots (lane ^ multiples of L), in a fixed order.  The
// exchanges of 8, 16 and 32 lanes are register moves: a row rotation, and the row and half swaps whose two results
// hold a lane's own and its partner's value.
__device__ __forceinline__ float xor16_sum(float x) {
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float xor32_sum(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
template <int L>
__device__ __forceinline__ float across_groups(float x) {
#pragma unroll
  for (int o = L; o < 8; o *= 2) x += __shfl_xor(x, o, kWave);
  if constexpr (L <= 8) x += dpp_f<0x128>(x);   // row_ror:8
  if constexpr (L <= 16) x = xor16_sum(x);
  return xor32_sum(x);
}

template <typename T, int L, bool ATOMIC>
__global__ __launch_bounds__(kWave * kBwdWaves) void bwd_query_kernel(BwdParams p) {
  constexpr int G = kWave / L;   // slots worked on together
  constexpr int M = (L * 8 + kWave - 1) / kWave;   // atomic adds: dimensions lane, lane + 64, ...
  __shared__ int s_row[kBwdWaves][kWave], s_slot[kBwdWaves][kWave];
  const int lane = lane_id(), wv = wave_id();
  const int ts = blockIdx.x * kBwdWaves + wv;
  if (ts >= p.Ts) return;   // a whole wavefront leaves; no workgroup barrier follows
  const int t = p.t0 + ts, bh = p.bh0 + blockIdx.y;
  const int b = bh / p.H, h = bh - b * p.H;
  const int D = p.D;
  const int g = lane / L, d0 = (lane % L) * 8;
  const bool in = d0 < D;
  const bool al = p.rows_al != 0;
  const T* kb = reinterpret_cast<const T*>(p.k) + b * p.ksb + h * p.ksh + d0;
  const T* vb = reinterpret_cast<const T*>(p.v) + b * p.vsb + h * p.vsh + d0;
  const int64_t row = (int64_t)bh * p.T + t;
  const int32_t* cr = p.cand + row * p.KC;
  float2* dsp = p.dsp + ((int64_t)blockIdx.y * p.Ts + ts) * p.KC;
  const float lse = p.lse[row];
  float qa[M], da[M];
  if constexpr (ATOMIC) {
    const T* qr = reinterpret_cast<const T*>(p.q) + b * p.qsb + h * p.qsh + (int64_t)t * p.qst;
    const T* dr = reinterpret_cast<const T*>(p.dout) + b * p.dsb + h * p.dsh + (int64_t)t * p.dst;
#pragma unroll
    for (int m = 0; m < M; ++m) {
      const int d = lane + kWave * m;
      qa[m] = d < D ? to_f32(qr[d]) : 0.0f;
      da[m] = d < D ? to_f32(dr[d]) : 0.0f;
    }
  }
  float qf[8], df[8], of[8];
  load8(reinterpret_cast<const T*>(p.q) + b * p.qsb + h * p.qsh + (int64_t)t * p.qst + d0, in, al, qf);
  load8(reinterpret_cast<const T*>(p.dout) + b * p.dsb + h * p.dsh + (int64_t)t * p.dst + d0, in, al, df);
  load8(reinterpret_cast<const T*>(p.o) + b * p.osb + h * p.osh + (int64_t)t * p.ost + d0, in, al, of);
  float Dq = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) Dq += df[i] * of[i];
  Dq = group_sum<L>(Dq);
  float dq[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) dq[i] = 0.0f;
  const uint64_t below = (1ull << lane) - 1;
  for (int c0 = 0; c0 < p.KC; c0 += kWave) {
    const int c = c0 + lane;
    const int j = c < p.KC ? cr[c] : -1;
    const bool ok = j >= 0 && j < p.Tk;
    const uint64_t m = __ballot(ok);
    const int n = __popcll(m);
    if (ok) {
      const int r = __popcll(m & below);
      s_row[wv][r] = j;
      s_slot[wv][r] = c;
    }
    wave_sync();
    for (int i = g; i - g < n; i += G) {
      const bool live = i < n;
      const int jr = live ? s_row[wv][i] : 0;
      float kf[8], vf[8];
      load8(kb + (int64_t)jr * p.kst, in && live, true, kf);
      load8(vb + (int64_t)jr * p.vst, in && live, true, vf);
      float s = 0.0f, dp = 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        s += qf[e] * kf[e];
        dp += df[e] * vf[e];
      }
      s = group_sum<L>(s);
      dp = group_sum<L>(dp);
      const float pw = live ? __expf(s * p.scale - lse) : 0.0f;
      const float ds = live ? pw * (dp - Dq) : 0.0f;
#pragma unroll
      for (int e = 0; e < 8; ++e) dq[e] += ds * kf[e];
      if constexpr (ATOMIC) {
        // slot by slot, consecutive lanes on consecutive dimensions: a row's 128-byte lines are asked for once per
        // instruction.  Every group adding its own slot's slices, 8 dimensions a lane, took 7 to 8 times as long:
        // (2, 6, 4096, 64) float16 5481 us against 689
        for (int u = 0; u < G && i - g + u < n; ++u) {
          const int j = __builtin_amdgcn_readlane(jr, u * L);
          const float a = p.scale * __int_as_float(__builtin_amdgcn_readlane(__float_as_int(ds), u * L));
          const float w = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(pw), u * L));
          float* dkr = p.dk + b * p.gk[0] + h * p.gk[1] + j * p.gk[2];
          float* dvr = p.dv + b * p.gv[0] + h * p.gv[1] + j * p.gv[2];
#pragma unroll
          for (int m = 0; m < M; ++m) {
            const int d = lane + kWave * m;
            if (d < D) {
              atomicAdd(dkr + d, a * qa[m]);
              atomicAdd(dvr + d, w * da[m]);
            }
          }
        }
      } else if (live && d0 == 0) {
        dsp[s_slot[wv][i]] = make_float2(ds, pw);
      }
    }
    wave_sync();
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) dq[e] = p.scale * across_groups<L>(dq[e]);
  if (g == 0 && in) store8(reinterpret_cast<T*>(p.dq) + b * p.gq[0] + h * p.gq[1] + t * p.gq[2] + d0, al, dq);
}

// ---------------------------------------------------------------------------------- sorting the slots by key
// A chunk's slots are consecutive: queries [ch * CQ, ...) of the Ts, KC slots each.
__device__ __forceinline__ void chunk_range(const BwdParams& p, int ch, int& s0, int& s1) {
  const int t0 = ch * p.CQ, t1 = t0 + p.CQ < p.Ts ? t0 + p.CQ : p.Ts;
  s0 = t0 * p.KC;
  s1 = t1 * p.KC;
}

// A candidate's key counted from the first one being summed: below Tj where it is one of them (unused slots, which
// are negative, wrap to the top).
__device__ __forceinline__ uint32_t key_of(const BwdParams& p, int32_t cand) { return (uint32_t)cand - (uint32_t)p.j0; }

// The candidate slots of pair `pair`'s queries from t0 on.
__device__ __forceinline__ const int32_t* pair_slots(const BwdParams& p, int pair) {
  return p.cand + ((int64_t)(p.bh0 + pair) * p.T + p.t0) * p.KC;
}

__global__ __launch_bounds__(kWave * kBwdWaves) void bwd_count_kernel(BwdParams p) {
  __shared__ int s_n[kMaxBuckets];
  const int ch = blockIdx.x, bh = blockIdx.y;
  for (int i = threadIdx.x; i < p.NB; i += blockDim.x) s_n[i] = 0;
  __syncthreads();
  int s0, s1;
  chunk_range(p, ch, s0, s1);
  const int32_t* cr = pair_slots(p, bh);
  for (int s = s0 + threadIdx.x; s < s1; s += blockDim.x) {
    const uint32_t j = key_of(p, cr[s]);
    if (j < (uint32_t)p.Tj) atomicAdd(&s_n[j >> p.wlog], 1);
  }
  __syncthreads();
  int32_t* cnt = p.cnt + (int64_t)bh * ((int64_t)p.NB * p.NC + 1);
  for (int i = threadIdx.x; i < p.NB; i += blockDim.x) cnt[(int64_t)i * p.NC + ch] = s_n[i];
}

// Exclusive sums of one (b,h)'s counts, in place, and the number of entries after them: 8 counts per thread and step.
__global__ __launch_bounds__(1024) void bwd_scan_kernel(BwdParams p) {
  __shared__ int s_w[16];
  const int n = p.NB * p.NC;
  int32_t* cnt = p.cnt + (int64_t)blockIdx.x * ((int64_t)n + 1);
  const int lane = lane_id(), wv = wave_id();
  int base = 0;
  for (int i0 = 0; i0 < n; i0 += 8192) {
    int x[8], sum = 0;
    const int i = i0 + (int)threadIdx.x * 8;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      x[e] = i + e < n ? cnt[i + e] : 0;
      sum += x[e];
    }
    int inc = sum;   // inclusive over the wavefront
#pragma unroll
    for (int o = 1; o < kWave; o *= 2) {
      const int y = __shfl_up(inc, o, kWave);
      if (lane >= o) inc += y;
    }
    if (lane == kWave - 1) s_w[wv] = inc;
    __syncthreads();
    int before = base, all = 0;
#pragma unroll
    for (int w = 0; w < 16; ++w) {
      if (w < wv) before += s_w[w];
      all += s_w[w];
    }
    int at = before + inc - sum;
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      if (i + e < n) cnt[i + e] = at;
      at += x[e];
    }
    base += all;
    __syncthreads();
  }
  if (threadIdx.x == 0) cnt[n] = base;
}

// Lanes of the wavefront that hold the same digit (`bits` wide) as this one, among the valid ones.
__device__ __forceinline__ uint64_t same_digit(int digit, bool ok, int bits) {
  uint64_t m = __ballot(ok);
  for (int b = 0; b < bits; ++b) {
    const bool one = (digit >> b) & 1;
    const uint64_t y = __ballot(one);
    m &= one ? y : ~y;
  }
  return m;
}

// Each chunk's valid slots to their places: bucket starts from the scan, then wavefronts (a consecutive quarter of
// the chunk each), rounds of 64 slots and lanes in order -- a stable order.
__global__ __launch_bounds__(kWave * kBwdWaves) void bwd_scatter_kernel(BwdParams p) {
  __shared__ int s_n[kBwdWaves][kMaxBuckets];
  const int ch = blockIdx.x, bh = blockIdx.y;
  const int lane = lane_id(), wv = wave_id();
  int* mine = s_n[wv];
  for (int i = lane; i < p.NB; i += kWave) mine[i] = 0;
  wave_sync();
  int s0, s1;
  chunk_range(p, ch, s0, s1);
  const int part = (s1 - s0 + kBwdWaves - 1) / kBwdWaves;
  const int a0 = s0 + wv * part, a1 = a0 + part < s1 ? a0 + part : s1;
  const int32_t* cr = pair_slots(p, bh);
  for (int s = a0 + lane; s < a1; s += kWave) {
    const uint32_t j = key_of(p, cr[s]);
    if (j < (uint32_t)p.Tj) atomicAdd(&mine[j >> p.wlog], 1);
  }
  __syncthreads();
  const int32_t* cnt = p.cnt + (int64_t)bh * ((int64_t)p.NB * p.NC + 1);
  for (int i = threadIdx.x; i < p.NB; i += blockDim.x) {
    int at = cnt[(int64_t)i * p.NC + ch];
#pragma unroll
    for (int w = 0; w < kBwdWaves; ++w) {
      const int n = s_n[w][i];
      s_n[w][i] = at;
      at += n;
    }
  }
  __syncthreads();
  uint2* ent = p.ent + (int64_t)bh * p.Ts * p.KC;
  const int bits = 32 - __clz(p.NB - 1 | 1);
  const uint64_t below = (1ull << lane) - 1;
  const uint32_t low = (1u << p.wlog) - 1;
  for (int sb = a0; sb < a1; sb += kWave) {
    const int s = sb + lane;
    const uint32_t j = s < a1 ? key_of(p, cr[s]) : ~0u;
    const bool ok = j < (uint32_t)p.Tj;
    const int d = ok ? (int)(j >> p.wlog) : 0;
    const uint64_t m = same_digit(d, ok, bits);
    int at = 0;
    if (ok) at = mine[d] + __popcll(m & below);
    wave_sync();
    if (ok) {
      ent[at] = make_uint2((uint32_t)s, (uint32_t)(s / p.KC) << kLowBits | (j & low));
      if ((m >> lane) == 1) mine[d] = at + 1;   // the last lane of the digit
    }
    wave_sync();
  }
}

// ------------------------------------------------------------------------------------------------ dk and dv
// 8 elements of a row as they lie in memory, converted when they are used (fewer registers for rows in flight)
template <typename T>
struct Raw8 {
  T e[8];
  __device__ __forceinline__ void load(const T* p, bool vec) {
    if (vec) {
#pragma unroll
      for (int i = 0; i < (int)sizeof(T) / 2; ++i)
        reinterpret_cast<uint4*>(e)[i] = reinterpret_cast<const uint4*>(p)[i];
    } else {
#pragma unroll
      for (int i = 0; i < 8; ++i) e[i] = p[i];
    }
  }
};

// Contributions of entries list[g], list[g + G], ... < n of one key to its dk and dv slices (this lane's group's
// part), then their sum over the groups.  BATCH entries' rows are requested together (past the end the last entry's,
// with weight 0), so that a list pays one round trip per BATCH * G entries.
template <typename T, int L, bool VEC, int BATCH>
__device__ __forceinline__ void key_part(const BwdParams& p, const T* qb, const T* db, const float2* dsp,
                                         const uint2* s_e, const uint16_t* list, int n, int g, float (&dk)[8],
                                         float (&dv)[8]) {
  constexpr int G = kWave / L;
#pragma unroll
  for (int i = 0; i < 8; ++i) dk[i] = dv[i] = 0.0f;
  for (int i0 = 0; i0 < n; i0 += G * BATCH) {
    float2 c[BATCH];
    Raw8<T> qr[BATCH], dr[BATCH];
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const int i = i0 + u * G + g;
      const uint2 e = s_e[list[i < n ? i : n - 1]];
      const int64_t t = e.y >> kLowBits;
      c[u] = dsp[e.x];
      qr[u].load(qb + t * p.qst, VEC);
      dr[u].load(db + t * p.dst, VEC);
    }
#pragma unroll
    for (int u = 0; u < BATCH; ++u) {
      const bool live = i0 + u * G + g < n;
      const float a = live ? p.scale * c[u].x : 0.0f, w = live ? c[u].y : 0.0f;
#pragma unroll
      for (int x = 0; x < 8; ++x) {
        dk[x] += a * (live ? to_f32(qr[u].e[x]) : 0.0f);
        dv[x] += w * (live ? to_f32(dr[u].e[x]) : 0.0f);
      }
    }
  }
#pragma unroll
  for (int x = 0; x < 8; ++x) {
    dk[x] = across_groups<L>(dk[x]);
    dv[x] = across_groups<L>(dv[x]);
  }
}

// dk and dv of one bucket's keys of one (sequence, head).  The bucket's entries come through LDS a tile at a time;
// per round every wavefront takes one key, lists the tile's entries of that key (ballots over the tile, which keeps
// their order) and adds their contributions, 64 / L entries at a time (the q and do rows in whole lines, the groups'
// partial sums in a fixed order).  A key that many queries name (the sink) is shared by all wavefronts, their parts
// added in order.  Each row is written by the first tile of the first queries and added to by later ones.
template <typename T, int L, bool VEC>
__global__ __launch_bounds__(kWave * kKeyWaves, 4) void bwd_keys_kernel(BwdParams p) {
  __shared__ uint2 s_e[kTile];
  __shared__ uint16_t s_list[kKeyWaves][kTile];
  __shared__ uint8_t s_heavy[1 << kLowBits];
  __shared__ float s_part[kKeyWaves][2][L * 8];
  const int lane = lane_id(), wv = wave_id(), tid = threadIdx.x;
  const int bh = blockIdx.x, bk = blockIdx.y;   // first buckets first: they hold the sink, the longest list
  const int b = (p.bh0 + bh) / p.H, h = p.bh0 + bh - b * p.H;
  const int D = p.D;
  const int g = lane / L, d0 = (lane % L) * 8;
  const bool in = d0 < D;
  const int j0 = p.j0 + (bk << p.wlog);
  const int W = 1 << p.wlog;
  const int nk = p.j0 + p.Tj - j0 < W ? p.j0 + p.Tj - j0 : W;
  const int32_t* cnt = p.cnt + (int64_t)bh * ((int64_t)p.NB * p.NC + 1);
  const int first = cnt[(int64_t)bk * p.NC], last = cnt[(int64_t)(bk + 1) * p.NC];
  const uint2* ent = p.ent + (int64_t)bh * p.Ts * p.KC;
  const float2* dsp = p.dsp + (int64_t)bh * p.Ts * p.KC;
  const int dl = in ? d0 : 0;   // lanes past the row read its first slice and write nothing
  const T* qb = reinterpret_cast<const T*>(p.q) + b * p.qsb + h * p.qsh + p.t0 * p.qst + dl;
  const T* db = reinterpret_cast<const T*>(p.dout) + b * p.dsb + h * p.dsh + p.t0 * p.dst + dl;
  float* dkb = p.dk + b * p.gk[0] + h * p.gk[1] + j0 * p.gk[2];
  float* dvb = p.dv + b * p.gv[0] + h * p.gv[1] + j0 * p.gv[2];
  const uint64_t below = (1ull << lane) - 1;
  constexpr uint32_t kLow = (1u << kLowBits) - 1;
  uint16_t* list = s_list[wv];
  // this wavefront's list of the entries i0 <= i < i1 of the tile that name `key`
  auto find = [&](int key, int i0, int i1) {
    int len = 0;
#pragma unroll 4
    for (; i0 < i1; i0 += kWave) {
      const int i = i0 + lane;
      const bool mine = i < i1 && (s_e[i].y & kLow) == (uint32_t)key;
      const uint64_t m = __ballot(mine);
      if (mine) list[len + __popcll(m & below)] = (uint16_t)i;
      len += __popcll(m);
    }
    wave_sync();
    return len;
  };
  float dk[8], dv[8];
  int at = first;
  do {
    const bool fresh = at == first && p.t0 == 0;
    const int n = last - at < kTile ? last - at : kTile;
    for (int i = tid; i < n; i += kWave * kKeyWaves) s_e[i] = ent[at + i];
    __syncthreads();
    for (int key = wv; key < W; key += kKeyWaves) {
      const int len = key < nk ? find(key, 0, n) : 0;
      if (lane == 0) s_heavy[key] = len > kHeavy;
      if (key >= nk || len > kHeavy || (len == 0 && !fresh)) continue;
      key_part<T, L, VEC, 2>(p, qb, db, dsp, s_e, list, len, g, dk, dv);
      if (g == 0 && in) {
        float* dkr = dkb + key * p.gk[2] + d0;
        float* dvr = dvb + key * p.gv[2] + d0;
        if (!fresh) {
#pragma unroll
          for (int x = 0; x < 8; ++x) {
            dk[x] += dkr[x];
            dv[x] += dvr[x];
          }
        }
        store8(dkr, VEC, dk);
        store8(dvr, VEC, dv);
      }
    }
    __syncthreads();
    for (int key = 0; key < nk; ++key) {   // the keys with many entries: a consecutive part of the tile per wavefront
      if (!s_heavy[key]) continue;
      const int part = (n + kKeyWaves - 1) / kKeyWaves;
      const int i0 = wv * part, i1 = i0 + part < n ? i0 + part : n;
      const int len = find(key, i0, i1);
      key_part<T, L, VEC, sizeof(T) == 4 ? 4 : 8>(p, qb, db, dsp, s_e, list, len, g, dk, dv);
      if (g == 0) {
#pragma unroll
        for (int x = 0; x < 8; ++x) {
          s_part[wv][0][d0 + x] = dk[x];
          s_part[wv][1][d0 + x] = dv[x];
        }
      }
      __syncthreads();
      for (int d = tid; d < 2 * D; d += kWave * kKeyWaves) {
        const int which = d >= D, dd = which ? d - D : d;
        float sum = 0.0f;
#pragma unroll
        for (int u = 0; u < kKeyWaves; ++u) sum += s_part[u][which][dd];
        float* r = (which ? dvb + key * p.gv[2] : dkb + key * p.gk[2]) + dd;
        *r = fresh ? sum : *r + sum;
      }
      __syncthreads();
    }
    at += n;
    __syncthreads();   // the tile is rewritten
  } while (at < last);
}

__global__ void bwd_zero_kernel(float* a, float* b, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    a[i] = b[i] = 0.0f;
}

// How the sorted route is cut: `pairs` (b,h) and Ts queries of each at a time, so that the workspace stays within
// kSortSlots slots (1 GiB; more only where a single query has more slots) and a slot and a query fit an entry's words.
// The pieces of a key's list come in order of the queries, so the cut does not disturb the fixed order of the sums.
struct BwdPlan {
  int pairs, Ts;
  int CQ, NC;            // queries per chunk, chunks
  int64_t slots, words;  // of a pair: slots of the Ts queries, words of the counts
};

static BwdPlan bwd_plan(int B, int H, int T, int KC) {
  BwdPlan r;
  const int64_t fit = kSortSlots / KC > 1 ? kSortSlots / KC : 1;
  const int64_t most = fit < (1 << (32 - kLowBits)) ? fit : 1 << (32 - kLowBits);
  r.Ts = (int)(T < most ? T : most);
  r.CQ = KC >= kChunkSlots ? 1 : kChunkSlots / KC;
  if (r.CQ < (r.Ts + kMaxChunks - 1) / kMaxChunks) r.CQ = (r.Ts + kMaxChunks - 1) / kMaxChunks;
  r.NC = (r.Ts + r.CQ - 1) / r.CQ;
  r.slots = (int64_t)r.Ts * KC;
  r.words = (int64_t)kMaxBuckets * r.NC + 1;
  const int64_t bh = (int64_t)B * H, together = kSortSlots / (r.slots + r.words / 4 + 1);
  r.pairs = (int)(bh < together ? bh : together > 1 ? together : 1);
  return r;
}

template <typename T, int L, bool ATOMIC>
static void launch_query(const BwdParams& p, int pairs, hipStream_t st) {
  hipLaunchKernelGGL((bwd_query_kernel<T, L, ATOMIC>), dim3((unsigned)((p.Ts + kBwdWaves - 1) / kBwdWaves), (unsigned)pairs),
                     dim3(kWave * kBwdWaves), 0, st, p);
}

template <typename T, int L>
static void launch_bwd(BwdParams p, const BwdPlan* pl, hipStream_t st) {
  const int bh = p.B * p.H;
  if (pl == nullptr) {   // atomic adds
    launch_query<T, L, true>(p, bh, st);
    return;
  }
  const dim3 block(kWave * kBwdWaves);
  constexpr int kMaxKeys = kMaxBuckets << kLowBits;   // sorted at a time
  for (p.bh0 = 0; p.bh0 < bh; p.bh0 += pl->pairs) {
    const int pairs = bh - p.bh0 < pl->pairs ? bh - p.bh0 : pl->pairs;
    for (int64_t t0 = 0; t0 < p.T; t0 += pl->Ts) {
      p.t0 = (int)t0;
      p.Ts = p.T - p.t0 < pl->Ts ? p.T - p.t0 : pl->Ts;
      p.NC = (p.Ts + p.CQ - 1) / p.CQ;
      launch_query<T, L, false>(p, pairs, st);
      for (int64_t j0 = 0; j0 < p.Tk; j0 += kMaxKeys) {
        p.j0 = (int)j0;
        p.Tj = p.Tk - p.j0 < kMaxKeys ? p.Tk - p.j0 : kMaxKeys;
        p.wlog = 4;   // 16 keys: two per wavefront of the key kernel
        while (((p.Tj - 1) >> p.wlog) + 1 > kMaxBuckets) ++p.wlog;
        p.NB = ((p.Tj - 1) >> p.wlog) + 1;
        const dim3 cgrid((unsigned)p.NC, (unsigned)pairs);
        hipLaunchKernelGGL(bwd_count_kernel, cgrid, block, 0, st, p);
        hipLaunchKernelGGL(bwd_scan_kernel, dim3((unsigned)pairs), dim3(1024), 0, st, p);
        hipLaunchKernelGGL(bwd_scatter_kernel, cgrid, block, 0, st, p);
        const dim3 kgrid((unsigned)pairs, (unsigned)p.NB), kblock(kWave * kKeyWaves);
        if (p.rows_al)
          hipLaunchKernelGGL((bwd_keys_kernel<T, L, true>), kgrid, kblock, 0, st, p);
        else
          hipLaunchKernelGGL((bwd_keys_kernel<T, L, false>), kgrid, kblock, 0, st, p);
      }
    }
  }
}

template <typename T>
static void launch_bwd_d(const BwdParams& p, const BwdPlan* pl, hipStream_t st) {
  switch (bwd_lanes(p.D)) {
    case 1: launch_bwd<T, 1>(p, pl, st); break;
    case 2: launch_bwd<T, 2>(p, pl, st); break;
    case 4: launch_bwd<T, 4>(p, pl, st); break;
    case 8: launch_bwd<T, 8>(p, pl, st); break;
    case 16: launch_bwd<T, 16>(p, pl, st); break;
    default: launch_bwd<T, 32>(p, pl, st); break;
  }
}

}  // namespace ta

using namespace ta;

static int sparse_attn_bwd_impl(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                  int dtype, int64_t qsb, int64_t qsh, int64_t qst, int64_t ksb, int64_t ksh,
                                  int64_t kst, int64_t vsb, int64_t vsh, int64_t vst, int64_t osb, int64_t osh,
                                  int64_t ost, int64_t dsb, int64_t dsh, int64_t dst, const int32_t* cand,
                                  const float* lse, int B, int H, int T, int Tk, int KC, int D, float scale,
                                  void* dq, float* dk, float* dv, float* ws, const int64_t* gs, void* stream) {
  if (B < 0 || H < 0 || T < 0 || Tk <= 0 || KC < 0 || D <= 0 || D > kBwdMaxD || D % 8) {
    set_error("ta_sparse_attn_bwd: bad sizes (D a multiple of 8, at most 256)");
    return TA_ERR_ARG;
  }
  if (dtype != TA_F32 && dtype != TA_F16 && dtype != TA_BF16) {
    set_error("ta_sparse_attn_bwd: unknown dtype");
    return TA_ERR_ARG;
  }
  if ((uintptr_t)ws % sizeof(float) != 0) {
    set_error("ta_sparse_attn_bwd: workspace not aligned to float32");
    return TA_ERR_ARG;
  }
  const int es = dtype == TA_F32 ? 4 : 2;
  // key and value rows are read 8 elements at a time
  if (((uintptr_t)k | (uintptr_t)v) % 16 || (ksb * es) % 16 || (ksh * es) % 16 || (kst * es) % 16 ||
      (vsb * es) % 16 || (vsh * es) % 16 || (vst * es) % 16) {
    set_error("ta_sparse_attn_bwd: k and v rows must be 16-byte aligned");
    return TA_ERR_ARG;
  }
  if (B == 0 || H == 0 || T == 0) return TA_OK;
  if ((int64_t)B * H > 65535) {
    set_error("ta_sparse_attn_bwd: B * H above 65535");
    return TA_ERR_UNSUPPORTED;
  }
  // rows of q, o, dout, dq, dk and dv are moved 8 elements at a time where all are aligned, else one by one
  const int al = !(((uintptr_t)q | (uintptr_t)o | (uintptr_t)dout | (uintptr_t)dq | (uintptr_t)dk | (uintptr_t)dv) % 16 ||
                   (qsb * es) % 16 || (qsh * es) % 16 || (qst * es) % 16 || (osb * es) % 16 || (osh * es) % 16 ||
                   (ost * es) % 16 || (dsb * es) % 16 || (dsh * es) % 16 || (dst * es) % 16 ||
                   ((gs[0] | gs[1] | gs[2]) * es) % 16 ||
                   ((gs[3] | gs[4] | gs[5] | gs[6] | gs[7] | gs[8]) * 4) % 16);
  BwdParams p{};
  p.q = q, p.k = k, p.v = v, p.o = o, p.dout = dout;
  p.qsb = qsb, p.qsh = qsh, p.qst = qst, p.ksb = ksb, p.ksh = ksh, p.kst = kst, p.vsb = vsb, p.vsh = vsh, p.vst = vst;
  p.osb = osb, p.osh = osh, p.ost = ost, p.dsb = dsb, p.dsh = dsh, p.dst = dst;
  p.cand = cand, p.lse = lse, p.dq = dq, p.dk = dk, p.dv = dv;
  p.B = B, p.H = H, p.T = T, p.Tk = Tk, p.KC = KC, p.D = D, p.Ts = T;
  p.scale = scale;
  p.rows_al = al;
  for (int i = 0; i < 3; ++i) p.gq[i] = gs[i], p.gk[i] = gs[3 + i], p.gv[i] = gs[6 + i];
  hipStream_t st = (hipStream_t)stream;
  BwdPlan pl;
  const bool sorted = ws != nullptr && KC > 0;
  if (sorted) {
    pl = bwd_plan(B, H, T, KC);
    const int64_t slots = pl.pairs * pl.slots;
    float* w = ws + ((uintptr_t)ws % 8 != 0);   // pairs of words; the size has room for the step
    p.dsp = reinterpret_cast<float2*>(w);
    p.ent = reinterpret_cast<uint2*>(w + 2 * slots);
    p.cnt = reinterpret_cast<int32_t*>(w + 4 * slots);
    p.CQ = pl.CQ;
  } else if (ws != nullptr) {   // no slots: every row is zero
    const int64_t n = (int64_t)B * H * Tk * D;
    const int64_t wgs = (n + 255) / 256;
    hipLaunchKernelGGL(bwd_zero_kernel, dim3((unsigned)(wgs < 4096 ? wgs : 4096)), dim3(256), 0, st, dk, dv, n);
  }
  const BwdPlan* plan = sorted ? &pl : nullptr;
  switch (dtype) {
    case TA_F32: launch_bwd_d<float>(p, plan, st); break;
    case TA_F16: launch_bwd_d<f16_t>(p, plan, st); break;
    default: launch_bwd_d<bf16_t>(p, plan, st); break;
  }
  return check_launch("ta_sparse_attn_bwd");
}

extern "C" int ta_sparse_attn_bwd(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                  int dtype, int64_t qsb, int64_t qsh, int64_t qst, int64_t ksb, int64_t ksh,
                                  int64_t kst, int64_t vsb, int64_t vsh, int64_t vst, int64_t osb, int64_t osh,
                                  int64_t ost, int64_t dsb, int64_t dsh, int64_t dst, const int32_t* cand,
                                  const float* lse, int B, int H, int T, int Tk, int KC, int D, float scale,
                                  void* dq, float* dk, float* dv, float* ws, int, void* stream) {
  const int64_t hq = (int64_t)T * D, hk = (int64_t)Tk * D;
  const int64_t gs[9] = {H * hq, hq, D, H * hk, hk, D, H * hk, hk, D};
  return sparse_attn_bwd_impl(q, k, v, o, dout, dtype, qsb, qsh, qst, ksb, ksh, kst, vsb, vsh, vst, osb, osh, ost, dsb,
                              dsh, dst, cand, lse, B, H, T, Tk, KC, D, scale, dq, dk, dv, ws, gs, stream);
}

extern "C" int ta_sparse_attn_bwd_strided(const void* q, const void* k, const void* v, const void* o, const void* dout,
                                          int dtype, int64_t qsb, int64_t qsh, int64_t qst, int64_t ksb, int64_t ksh,
                                          int64_t kst, int64_t vsb, int64_t vsh, int64_t vst, int64_t osb,
                                          int64_t osh, int64_t ost, int64_t dsb, int64_t dsh, int64_t dst,
                                          const int32_t* cand, const float* lse, int B, int H, int T, int Tk, int KC,
                                          int D, float scale, void* dq, float* dk, float* dv, float* ws, int,
                                          const int64_t* grad_strides, void* stream) {
  if (grad_strides == nullptr) {
    set_error("ta_sparse_attn_bwd_strided: no strides of the gradients");
    return TA_ERR_ARG;
  }
  return sparse_attn_bwd_impl(q, k, v, o, dout, dtype, qsb, qsh, qst, ksb, ksh, kst, vsb, vsh, vst, osb, osh, ost, dsb,
                              dsh, dst, cand, lse, B, H, T, Tk, KC, D, scale, dq, dk, dv, ws, grad_strides, stream);
}

// Workspace of the sorted dk / dv route of ta_sparse_attn_bwd: per-slot (ds, p), the sorted entries, and the counts of
// at most kMaxBuckets buckets per chunk of queries (whatever the number of keys), for what bwd_plan sorts at a time.
extern "C" int64_t ta_sparse_attn_bwd_workspace_size(int B, int H, int T, int KC) {
  if (B <= 0 || H <= 0 || T <= 0 || KC <= 0) return 0;
  const BwdPlan pl = bwd_plan(B, H, T, KC);
  return (pl.pairs * (4 * pl.slots + pl.words) + 1) * (int64_t)sizeof(float);
}
