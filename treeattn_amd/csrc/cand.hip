// The candidate list of the module forward (fastseg.py:367-381, attention_dyn.py:12-17 and 74-96), in one
// launch: for every query row, the candidates in the reference's order -- the tree leaves' keys (leaf groups of
// `leaf` positions: entry r * wl + j is position r of leaf j), the neighbour leaves' keys, the static keys (0, t,
// t - 1, ..., t - Lw + 1 with Lw = max(local, 3)) and, for leaf > 2, the query's own leaf group up to t -- each
// valid where the reference's mask says so (a tree entry: its leaf is among the first n_tree found ones and
// the position is not -1; every other entry: not -1), then only the first valid copy of each position kept
// (the dedupe, selection.dedupe_fast), written as the masked row (position or -1, int32) that the sparse
// attention takes, with the row's counts for the module's statistics: kept entries in all, among the tree
// entries and among the neighbour entries, and the leaves used.
//
// One wavefront per query row: the row's candidates and validity go to LDS, and lane e tests its entries e, e +
// 64, ... against every earlier valid entry (a row holds at most kCandMax entries).
#include "common.hpp"

namespace ta {

constexpr int kCandMax = 320;   // candidates per row
constexpr int kCandRows = 4;    // rows (wavefronts) per workgroup

__global__ __launch_bounds__(kWave * kCandRows) void assemble_candidates_kernel(
    const int64_t* __restrict__ tree_pos, const uint8_t* __restrict__ leaf_ok, const int64_t* __restrict__ n_tree,
    const int64_t* __restrict__ nb_pos, const int64_t* __restrict__ tq, int tq_batched, int B, int H, int N, int wl,
    int leaf, int nbk, int local, int KC, int32_t* __restrict__ cm, int32_t* __restrict__ counts) {
  __shared__ int32_t s_pos[kCandRows][kCandMax];
  __shared__ uint8_t s_val[kCandRows][kCandMax];
  const int lane = lane_id(), wv = wave_id();
  const int64_t row = (int64_t)blockIdx.x * kCandRows + wv;
  if (row >= (int64_t)B * H * N) return;   // a whole wavefront leaves; no workgroup barrier follows
  const int64_t b = row / ((int64_t)H * N), n = row % N;
  const int64_t t = tq[tq_batched ? b * N + n : n];
  const int ntr = (int)n_tree[row];
  const int lw = local > 3 ? local : 3, ntp = leaf * wl, ns = 1 + lw;
  int32_t* pos = s_pos[wv];
  uint8_t* val = s_val[wv];
  // the row's candidates and validity
  for (int e = lane; e < KC; e += kWave) {
    int64_t p = -1;
    bool v = false;
    if (e < ntp) {
      const int j = e % wl;
      p = tree_pos[row * ntp + e];
      v = p >= 0 && leaf_ok[row * wl + j] != 0 && j < ntr;
    } else if (e < ntp + nbk) {
      p = nb_pos[row * nbk + (e - ntp)];
      v = p >= 0;
    } else if (e < ntp + nbk + ns) {
      const int s = e - ntp - nbk;
      p = s == 0 ? 0 : t - (s - 1);
      if (p < 0) p = -1;
      v = p >= 0;
    } else {
      const int r = e - ntp - nbk - ns;
      p = (t / leaf) * leaf + r;
      if (p > t) p = -1;
      v = p >= 0;
    }
    pos[e] = (int32_t)p;
    val[e] = v ? 1 : 0;
  }
  wave_sync();
  // first valid copy of each position
  int kept = 0, kept_tree = 0, kept_nb = 0;
  for (int e = lane; e < KC; e += kWave) {
    const int32_t p = pos[e];
    bool keep = val[e] != 0;
    for (int j = 0; j < e && keep; ++j) keep = !(val[j] != 0 && pos[j] == p);
    cm[row * KC + e] = keep ? p : -1;
    kept += keep ? 1 : 0;
    kept_tree += keep && e < ntp ? 1 : 0;
    kept_nb += keep && e >= ntp && e < ntp + nbk ? 1 : 0;
  }
  int used = 0;
  for (int j = lane; j < wl; j += kWave) used += leaf_ok[row * wl + j] != 0 && j < ntr ? 1 : 0;
  for (int o = 32; o >= 1; o >>= 1) {
    kept += __shfl_xor(kept, o);
    kept_tree += __shfl_xor(kept_tree, o);
    kept_nb += __shfl_xor(kept_nb, o);
    used += __shfl_xor(used, o);
  }
  if (lane == 0) {
    int32_t* c = counts + row * 4;
    c[0] = kept;
    c[1] = kept_tree;
    c[2] = kept_nb;
    c[3] = used;
  }
}

// The same list from the leaves themselves (what a descent and a neighbour pass write), in one launch: the leaf budget
// (seg.py:111-117) from lhat and the distinct matched leaves nL, the masked row, and the sums behind the module's
// statistics.  A leaf's positions are all listed or none, so the dedupe compares leaves: one wavefront per row holds a
// tree leaf and a neighbour leaf per lane and walks the valid ones (about a dozen) with scalar reads; static keys and
// the query's own leaf group are tested against the same leaves.  The next row is requested before the current one is
// worked on.  For a (2, 6, 4096) selection of 8 leaves and 16 stored ones, 52 entries a row: 30 us; building
// the row from expanded int64 position lists (assemble_candidates_kernel) took 74 us and the concatenations, masks and
// sums around it about 160 us more.
constexpr int kLeafRows = 8;    // rows (wavefronts) per workgroup

__device__ __forceinline__ int leaf_budget(int64_t L, int nl, int wmax) {
  // signed 64-bit like the reference's, clamped before it is narrowed; half rounds down for negative budgets too
  const int64_t need = L - nl > 0 ? L - nl : 0, half = (L + 1 - ((L + 1) < 0 && ((L + 1) & 1))) / 2;
  const int64_t least = nl < half ? 2 : 1;
  const int64_t want = nl >= L ? 0 : (need > least ? need : least);
  return (int)(want < wmax ? want : wmax);
}

__device__ __forceinline__ void store_sums(int (&sum)[5], int32_t (*s_sum)[5], int32_t* sums) {
  if (lane_id() == 0) {
#pragma unroll
    for (int i = 0; i < 5; ++i) s_sum[wave_id()][i] = sum[i];
  }
  __syncthreads();
  if (threadIdx.x < 5) {
    int x = 0;
#pragma unroll
    for (int w = 0; w < kLeafRows; ++w) x += s_sum[w][threadIdx.x];
    sums[(int64_t)blockIdx.x * 5 + threadIdx.x] = x;
  }
}

// Budgets and statistics only (the structural attention needs no list): a row per lane, its flags read four at a time
// where rows are whole words.
__global__ __launch_bounds__(kWave * kLeafRows) void count_leaves_kernel(
    const uint8_t* __restrict__ vld, const int64_t* __restrict__ lhat, const int32_t* __restrict__ nL, int64_t rows,
    int wl, int wmax, int words, int32_t* __restrict__ n_tree, int32_t* __restrict__ sums) {
  __shared__ int32_t s_sum[kLeafRows][5];
  int used = 0, nls = 0;
  const int64_t step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t row = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; row < rows; row += step) {
    const int nl = nL != nullptr ? nL[row] : 0;
    const int ntr = leaf_budget(lhat[row], nl, wmax);
    nls += nl;
    if (n_tree != nullptr) n_tree[row] = ntr;
    const uint8_t* v = vld + row * wl;
    if (words) {
      for (int j = 0; j < wl; j += 4) {
        const uint32_t u = *reinterpret_cast<const uint32_t*>(v + j);
#pragma unroll
        for (int i = 0; i < 4; ++i) used += ((u >> (8 * i)) & 0xff) != 0 && j + i < ntr ? 1 : 0;
      }
    } else {
      for (int j = 0; j < wl; ++j) used += v[j] != 0 && j < ntr ? 1 : 0;
    }
  }
  for (int o = 32; o >= 1; o >>= 1) {
    used += __shfl_xor(used, o);
    nls += __shfl_xor(nls, o);
  }
  int sum[5] = {0, 0, 0, used, nls};
  store_sums(sum, s_sum, sums);
}

struct LeafRow {   // one row's inputs, a leaf of each kind per lane
  int id_t, id_n, nl, t;
  bool ok_t, ok_n;
  int64_t L;
};

__global__ __launch_bounds__(kWave * kLeafRows) void assemble_leaves_kernel(
    const int32_t* __restrict__ ids, const uint8_t* __restrict__ vld, const int64_t* __restrict__ lhat,
    const int32_t* __restrict__ nL, const int32_t* __restrict__ nid, const uint8_t* __restrict__ match,
    const int32_t* __restrict__ tq, int64_t tq_sb, int64_t HN, int N, int64_t rows, int wl, int S, int llog, int local,
    int wmax, int KC, int32_t* __restrict__ n_tree, int32_t* __restrict__ cm, int32_t* __restrict__ sums) {
  __shared__ int32_t s_leaf[kLeafRows][2][kWave];
  __shared__ int32_t s_sum[kLeafRows][5];
  const int lane = lane_id(), wv = wave_id();
  const int leaf = 1 << llog, lw = local > 3 ? local : 3, ns = 1 + lw;
  const float inv_wl = 1.0f / wl, inv_s = S > 0 ? 1.0f / S : 0.0f;
  int32_t* lt = s_leaf[wv][0];
  int32_t* ln = s_leaf[wv][1];
  int kept = 0, kept_tree = 0, kept_nb = 0, used_n = 0, nl_sum = 0;
  auto read = [&](int64_t row) {
    LeafRow r;
    r.id_t = lane < wl ? ids[row * wl + lane] : -1;
    r.ok_t = lane < wl && vld[row * wl + lane] != 0;
    r.id_n = lane < S ? nid[row * S + lane] : -1;
    r.ok_n = lane < S && match[row * S + lane] != 0;
    r.nl = nL != nullptr ? nL[row] : 0;
    r.L = lhat[row];
    r.t = tq[(row / HN) * tq_sb + row % N];
    return r;
  };
  const int64_t step = (int64_t)gridDim.x * kLeafRows;
  int64_t row = (int64_t)blockIdx.x * kLeafRows + wv;
  LeafRow next = read(row < rows ? row : rows - 1);
  for (; row < rows; row += step) {
    const LeafRow cur = next;
    next = read(row + step < rows ? row + step : row);
    const int id_t = cur.id_t, id_n = cur.id_n, nl = cur.nl, t = cur.t;
    const bool ok_n = cur.ok_n;
    const int ntr = leaf_budget(cur.L, nl, wmax);
    const bool used = cur.ok_t && lane < ntr;
    used_n += __popcll(__ballot(used));
    nl_sum += nl;
    if (n_tree != nullptr && lane == 0) n_tree[row] = ntr;
    const int own = t >> llog;
    const int ps = lane == 0 ? 0 : t - (lane - 1);
    bool keep_t = used, keep_n = ok_n, keep_s = lane < ns && ps >= 0 && (lane == 0 || ps != 0), own_in = false;
    const int sleaf = ps >> llog;
    for (uint64_t m = __ballot(used); m != 0; m &= m - 1) {
      const int k = __ffsll((unsigned long long)m) - 1;
      const int id = __builtin_amdgcn_readlane(id_t, k);
      keep_t = keep_t && !(lane > k && id_t == id);
      keep_n = keep_n && id_n != id;
      keep_s = keep_s && sleaf != id;
      own_in = own_in || own == id;
    }
    for (uint64_t m = __ballot(ok_n); m != 0; m &= m - 1) {
      const int k = __ffsll((unsigned long long)m) - 1;
      const int id = __builtin_amdgcn_readlane(id_n, k);
      keep_n = keep_n && !(lane > k && id_n == id);
      keep_s = keep_s && sleaf != id;
      own_in = own_in || own == id;
    }
    lt[lane] = keep_t ? id_t << llog : -1;
    ln[lane] = keep_n ? id_n << llog : -1;
    wave_sync();
    int32_t* c = cm + row * KC;
    for (int e = lane; e < wl << llog; e += kWave) {   // entry r * wl + j: position r of leaf j
      const int r = (int)(((float)e + 0.5f) * inv_wl), v = lt[e - r * wl];
      c[e] = v < 0 ? -1 : v + r;
    }
    c += wl << llog;
    for (int e = lane; e < S << llog; e += kWave) {
      const int r = (int)(((float)e + 0.5f) * inv_s), v = ln[e - r * S];
      c[e] = v < 0 ? -1 : v + r;
    }
    c += S << llog;
    if (lane < ns) c[lane] = keep_s ? ps : -1;
    c += ns;
    int own_n = 0;
    if (leaf > 2) {   // the own leaf group up to t, without the static keys (0 and the last lw positions)
      for (int e = lane; e - lane < leaf; e += kWave) {
        const int p = (own << llog) + e;
        const bool k = e < leaf && p <= t && !own_in && p != 0 && t - p >= lw;
        if (e < leaf) c[e] = k ? p : -1;
        own_n += __popcll(__ballot(k));
      }
    }
    const int kt = __popcll(__ballot(keep_t)) << llog, kn = __popcll(__ballot(keep_n)) << llog;
    kept_tree += kt;
    kept_nb += kn;
    kept += kt + kn + __popcll(__ballot(keep_s)) + own_n;
    wave_sync();
  }
  int sum[5] = {kept, kept_tree, kept_nb, used_n, nl_sum};
  store_sums(sum, s_sum, sums);
}

}  // namespace ta

using namespace ta;

extern "C" int ta_assemble_candidates(const int64_t* tree_pos, const uint8_t* leaf_ok, const int64_t* n_tree,
                                      const int64_t* nb_pos, const int64_t* tq, int tq_batched, int B, int H, int N,
                                      int wl, int leaf, int nbk, int local, int32_t* cm, int32_t* counts,
                                      void* stream) {
  const int lw = local > 3 ? local : 3;
  const int64_t KC = (int64_t)leaf * wl + nbk + 1 + lw + (leaf > 2 ? leaf : 0);
  if (tree_pos == nullptr || leaf_ok == nullptr || n_tree == nullptr || tq == nullptr || cm == nullptr ||
      counts == nullptr || (nbk > 0 && nb_pos == nullptr) || B <= 0 || H <= 0 || N <= 0 || wl < 1 || leaf < 2 ||
      nbk < 0 || local < 0 || KC > kCandMax) {
    set_error("ta_assemble_candidates: bad arguments (at most 320 candidates per row: leaf * wl + nbk + 1 + "
              "max(local, 3) (+ leaf when leaf > 2))");
    return TA_ERR_ARG;
  }
  const int64_t rows = (int64_t)B * H * N;
  const int64_t grid = (rows + kCandRows - 1) / kCandRows;
  if (grid > 0x7fffffff) {
    set_error("ta_assemble_candidates: too many rows");
    return TA_ERR_ARG;
  }
  hipLaunchKernelGGL(assemble_candidates_kernel, dim3((unsigned)grid), dim3(kWave * kCandRows), 0,
                     (hipStream_t)stream, tree_pos, leaf_ok, n_tree, nb_pos, tq, tq_batched, B, H, N, wl, leaf, nbk,
                     local, (int)KC, cm, counts);
  return check_launch("ta_assemble_candidates");
}

extern "C" int ta_assemble_leaves(const int32_t* ids, const uint8_t* vld, const int64_t* lhat, const int32_t* nL,
                                  const int32_t* nid, const uint8_t* match, const int32_t* tq, int64_t tq_sb, int B,
                                  int H, int N, int wl, int S, int leaf, int local, int wmax, int32_t* n_tree,
                                  int32_t* cm, int32_t* sums, int sum_rows, void* stream) {
  const int lw = local > 3 ? local : 3;
  if (ids == nullptr || vld == nullptr || lhat == nullptr || sums == nullptr || B <= 0 || H <= 0 || N <= 0 || wl < 1 ||
      wl > kWave || S < 0 || S > kWave || (S > 0 && (nid == nullptr || match == nullptr)) || leaf < 2 ||
      (leaf & (leaf - 1)) || local < 0 || lw >= kWave || wmax < 0 || sum_rows < 1 ||
      (cm != nullptr && (tq == nullptr || leaf > 65536))) {
    set_error("ta_assemble_leaves: bad arguments (at most 64 tree leaves and 64 stored ones per row, leaf a power of "
              "two, at most 65536 for the list, local below 64)");
    return TA_ERR_ARG;
  }
  const int64_t rows = (int64_t)B * H * N;
  const int64_t KC = ((int64_t)wl + S) * leaf + 1 + lw + (leaf > 2 ? leaf : 0);
  // rows that one row of sums adds up, and the most that one of them adds
  const int64_t per_wave = (rows + (int64_t)sum_rows * kLeafRows - 1) / ((int64_t)sum_rows * kLeafRows);
  const int64_t most = cm != nullptr ? per_wave * kLeafRows * KC : (per_wave + kWave) * kLeafRows * kWave;
  if (most > 0x7fffffff) {
    set_error("ta_assemble_leaves: too many rows for the sums");
    return TA_ERR_ARG;
  }
  int llog = 0;
  while ((1 << llog) < leaf) ++llog;
  // every row of sums is written: as many workgroups as rows of sums, whatever the number of candidate rows
  const dim3 grid((unsigned)sum_rows), block(kWave * kLeafRows);
  if (cm == nullptr)
    hipLaunchKernelGGL(count_leaves_kernel, grid, block, 0, (hipStream_t)stream, vld, lhat, nL, rows, wl, wmax,
                       wl % 4 == 0 && (uintptr_t)vld % 4 == 0, n_tree, sums);
  else
    hipLaunchKernelGGL(assemble_leaves_kernel, grid, block, 0, (hipStream_t)stream, ids, vld, lhat, nL, nid, match, tq,
                       tq_sb, (int64_t)H * N, N, rows, wl, S, llog, local, wmax, (int)KC, n_tree, cm, sums);
  return check_launch("ta_assemble_leaves");
}
