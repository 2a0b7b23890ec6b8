// prefill_split.h - the even split of a chunked prefill over workgroups,
// shared by the 16-bit and the fp32 MFMA kernels, and the merge of what it
// cuts.
//
// A prefill's work items are (sequence, kv head, query tile); an item runs
// over the K/V tiles its last row sees. One workgroup per item leaves the
// chip idle where items are few or uneven: 24 sequences of 0..6000 cached
// tokens (28/4 heads, 40 % of them bringing 1..300 tokens, the rest one) ran
// 357 us at 156 TFLOP/s, most of it a few long items alone. Here `groups`
// workgroups split the items' flattened K/V tiles evenly, as the decode's
// stream kernel does: group w takes the units [bound(w), bound(w + 1)),
// crossing item borders, and an item cut by a bound leaves one partial per
// group in the workspace, which prefill_merge combines.
//
// Units: an item costs Cfg::kItemUnits (its Q loads and the fill of the tile
// ring) plus Cfg::tile_units(rows) per K/V tile. The items of one kv head
// follow each other, a sequence's query tiles in folded order (heaviest,
// lightest, second heaviest, ...), so that equal shares of a uniform batch
// tend to end at item borders; a bound within Cfg::snap() units of an item
// border moves onto it, as a cut costs two partials and their merge. snap() is
// at least kItemUnits and the units of a tile, so that every group between
// an item's first and last one holds at least one of its tiles. Where every
// group gets at most one item and the longest is not far above the even
// share, nothing is cut at all: the cuts (kCutUnits: what a cut group loses to
// its two partials and their merge) would cost more than the evenness gives.
#pragma once

#include <algorithm>

#include "attn_common.h"

namespace clv {

// The decision behind the split shapes: `rows` query rows per workgroup, `bk`
// K/V tokens per tile, `per_cu` workgroups per compute unit, at most
// `tile_units` units per tile; no split up to `min_tiles` tiles, nor (with
// `even_rounds`) of equal chunks whose items fill whole rounds of the device.
//
// It sees sizes, not lengths. What that costs: where a table is much wider than
// the contexts, the schedule and an empty merge launch are 5 to 7 us of a call
// that is not cut (28/4 heads, bf16, 512 blocks wide: a prompt of 100 tokens 12.3
// and 18.6 us, one of 777 31.8 and 38.6), against what long contexts gain (one
// row over 4000 tokens 104 -> 25, three chunks of 100 over 2000 70 -> 40).
inline PrefillSplitShape prefill_split_shape(const PrefillParams &p, int rows, int bk, int per_cu,
                                             int tile_units, int min_tiles, bool even_rounds) {
  const PrefillSplitShape none = {rows, 0};
  const int64_t bq = rows / p.group;
  const int64_t n_q = std::max<int64_t>(1, ((int64_t)p.max_query_len + bq - 1) / bq);
  const int64_t max_tiles = (((int64_t)p.max_blocks_per_seq << p.block_shift) + bk - 1) / bk;
  // The table width bounds every context: up to min_tiles tiles the longest
  // item is short, and the split would cost its merge launch.
  if (max_tiles <= min_tiles || p.cus_per_xcd <= 0) return none;
  // Every sequence has an entry in LDS for each tile of the longest chunk, also
  // those that bring less. Past the table (28/4 heads in 16 bits: 64 sequences
  // with a chunk of over 576 tokens, 128 with one of over 288) the call runs
  // unsplit, however uneven it is.
  const int64_t entries = (int64_t)p.num_seqs * n_q;
  if (entries > kPrefillSplitItems) return none;
  // Units are 32-bit on the device (an item's own are at most four tiles').
  if (entries * p.num_kv_heads * (max_tiles + 4) * tile_units >= (int64_t)1 << 30) return none;
  // Chunks of one length that fill whole rounds of the device: over equal cached
  // lengths the 16-bit kernel's natural order (dispatch_slot) makes them even
  // already (8 x 512 over 4096, 32/8 heads, 292 us, split 303). The lengths are not
  // known here: over 0..8192 cached tokens the same chunks take 489 us unsplit and
  // would take 364 split.
  const int groups = per_cu * p.cus_per_xcd * 8;
  if (even_rounds && (int64_t)p.num_tokens == (int64_t)p.num_seqs * p.max_query_len &&
      entries * p.num_kv_heads % groups == 0)
    return none;
  return {rows, groups};
}

// Wave operations of the schedule. It also compiles for the host, where one
// thread stands for the wave (tests/host/prefill_split_check.h).
__host__ __device__ __forceinline__ int first_lane(int x) {
#ifdef __HIP_DEVICE_COMPILE__
  return __builtin_amdgcn_readfirstlane(x);
#else
  return x;
#endif
}
__host__ __device__ __forceinline__ bool is_first_lane() {
#ifdef __HIP_DEVICE_COMPILE__
  return (threadIdx.x & 63) == 0;
#else
  return true;
#endif
}

// What a group left in the workspace: the item whose first part it holds
// (rows 0: none; partial slot 2w + 1), and whether its first item was begun
// by an earlier group (cont, partial slot 2w) and ends here. The item is
// described by what the merge needs, so that it reads nothing else first.
struct __attribute__((aligned(16))) PrefillDesc {
  int32_t rows;  // query rows of the item (tokens x query heads)
  int32_t row0;  // token row of q / out of its first token
  int32_t q0;    // that token's index in its chunk
  int32_t kvh;
  int32_t cont;  // 0: none, 1: goes on in the next group, 2: ends here
  int32_t unused[3];
};
static_assert(sizeof(PrefillDesc) == kPrefillDescBytes, "the workspace layout");

// One work item.
struct PrefillItem {
  int s, kvh, qt;
  int qs, n_new;         // first query row of the sequence, its rows
  int q0, q_hi;          // rows [q0, q_hi) of the chunk
  int ctx, base_pos;     // cached tokens; position of row 0
  int kv_end;            // tokens the last row sees

  __host__ __device__ __forceinline__ void set(const PrefillParams &p, int bq, int s_, int kvh_,
                                               int qt_) {
    s = s_;
    kvh = kvh_;
    qt = qt_;
    qs = p.query_start_loc[s];
    n_new = p.query_start_loc[s + 1] - qs;
    const int cap = p.max_blocks_per_seq << p.block_shift;
    ctx = max(0, min(p.context_lens[s], cap));
    base_pos = ctx - n_new;
    q0 = qt * bq;
    q_hi = min(q0 + bq, n_new);
    kv_end = max(0, min(ctx, base_pos + q_hi));
  }
};

template <class Cfg>
struct PrefillSched {
  static constexpr int kCursorInts = 5;
  const int *pre;  // LDS: exclusive prefix of the units of one kv head's items
  int n;           // entries: num_seqs * nq
  int nq;          // query tiles per sequence the entries allow for
  int C, N, W;     // units per kv head, units in all, groups in use
  int tol;
  bool whole;      // nothing is cut: one item per group, one unit per item

  // Query tile at position pos of a sequence's nqs tiles.
  static __host__ __device__ __forceinline__ int folded(int pos, int nqs) {
    return (pos & 1) ? pos >> 1 : nqs - 1 - (pos >> 1);
  }
  static __host__ __device__ __forceinline__ int tiles(int kv_end) {
    return max(1, (kv_end + Cfg::kBK - 1) / Cfg::kBK);
  }
  static __host__ __device__ __forceinline__ int seq_tiles(int n_new, int bq, int nq) {
    return min(nq, (max(0, n_new) + bq - 1) / bq);
  }

  // Units of entry i (0: no tile there).
  __host__ __device__ __forceinline__ int entry_units(const PrefillParams &p, int bq, int i) const {
    const int s = i / nq, pos = i - s * nq;
    PrefillItem it;
    it.set(p, bq, s, 0, 0);
    const int nqs = seq_tiles(it.n_new, bq, nq);
    if (pos >= nqs) return 0;
    it.set(p, bq, s, 0, folded(pos, nqs));
    return Cfg::kItemUnits + tiles(it.kv_end) * Cfg::tile_units((it.q_hi - it.q0) * p.group);
  }

  // The rest of the schedule from one kv head's units, its items and the
  // longest of them.
  __host__ __device__ __forceinline__ void set_totals(int heads, int groups, int units, int items,
                                                      int most) {
    const int share = units * heads / min(groups, max(1, units * heads / Cfg::kMinShare));
    whole = items * heads <= groups && most <= share + share / 4 + Cfg::kCutUnits;
    C = first_lane(whole ? items : units);
    N = C * heads;
    W = whole ? max(1, N) : min(groups, max(1, N / Cfg::kMinShare));
    tol = whole ? 0 : Cfg::snap(share);
  }

  // Fills buf (kPrefillSplitItems + 1 ints of LDS; tmp: 3 per wave) and the
  // totals; every thread of the workgroup (NT of them) calls it.
  template <int NT>
  __device__ __forceinline__ void init(const PrefillParams &p, int bq, int nq_, int groups,
                                       int *buf, int *tmp) {
    nq = nq_;
    n = p.num_seqs * nq;
    pre = buf;
    const int tid = threadIdx.x;
    const int per = (n + NT - 1) / NT;
    const int b = min(n, tid * per), e = min(n, b + per);
    int units = 0, count = 0, most = 0;
    for (int i = b; i < e; ++i) {
      const int u = entry_units(p, bq, i);
      buf[i] = u;
      units += u;
      count += u > 0 ? 1 : 0;
      most = max(most, u);
    }
    // Inclusive scans over the wave, then over the waves' totals.
    int xu = units, xc = count;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int yu = __shfl_up(xu, off, 64), yc = __shfl_up(xc, off, 64);
      if ((tid & 63) >= off) {
        xu += yu;
        xc += yc;
      }
      most = max(most, __shfl_xor(most, off, 64));
    }
    if ((tid & 63) == 63) {
      tmp[3 * (tid >> 6)] = xu;
      tmp[3 * (tid >> 6) + 1] = xc;
      tmp[3 * (tid >> 6) + 2] = most;
    }
    __syncthreads();
    int ru = xu - units, rc = xc - count;
    int tu = 0, tc = 0;
    most = 0;
#pragma unroll
    for (int w = 0; w < NT / 64; ++w) {
      if (w < (tid >> 6)) {
        ru += tmp[3 * w];
        rc += tmp[3 * w + 1];
      }
      tu += tmp[3 * w];
      tc += tmp[3 * w + 1];
      most = max(most, tmp[3 * w + 2]);
    }
    set_totals(p.num_kv_heads, groups, tu, tc, most);
    int run = whole ? rc : ru;
    for (int i = b; i < e; ++i) {
      const int u = buf[i];
      buf[i] = run;
      run += whole ? (u > 0 ? 1 : 0) : u;
    }
    if (tid == 0) buf[n] = whole ? tc : tu;
    __syncthreads();
  }

  // Group of workgroup `block`, or -1. Consecutive ids go round-robin over the
  // 8 XCDs: each takes a contiguous run of the W groups in use (query tiles of
  // one kv head then share its L2), the idle workgroups spread over all of them.
  __host__ __device__ __forceinline__ int group_of(int block) const {
    const int per_xcd = (W + 7) / 8;
    const int w = (block % 8) * per_xcd + block / 8;
    return block / 8 < per_xcd && w < W ? w : -1;
  }

  // Clears the descriptor of group w, and those past W between all groups.
  __device__ __forceinline__ void clear_desc(const PrefillSplit &sp, int w) const {
    for (int i = w; i < sp.groups; i += W)
      reinterpret_cast<PrefillDesc *>(sp.desc)[i] = PrefillDesc{0, 0, 0, 0, 0, {0, 0, 0}};
  }

  // Entry holding unit rem of a kv head (0 <= rem < C): the last one with
  // pre[i] <= rem; 64 candidates a round, as in the decode's stream kernel.
  __host__ __device__ __forceinline__ int find(int rem) const {
#ifdef __HIP_DEVICE_COMPILE__
    const int lane = threadIdx.x & 63;
    int lo = 0, len = n;
    while (len > 1) {
      const int stride = (len + 63) / 64;
      const bool le = lane * stride < len && pre[lo + lane * stride] <= rem;
      const int k = 63 - __builtin_clzll(__ballot(le));
      lo += k * stride;
      len = min(stride, len - k * stride);
    }
    return first_lane(lo);
#else
    return (int)(std::upper_bound(pre, pre + n, rem) - pre) - 1;
#endif
  }

  // First unit of group w. Never decreases in w: a bound only moves onto the
  // item border nearest to it.
  __host__ __device__ __forceinline__ int bound(int w) const {
    if (w <= 0) return 0;
    if (w >= W) return N;
    const int x = (int)((int64_t)w * N / W);
    const int kvh = x / C, rem = x - kvh * C;
    const int i = find(rem);
    const int lo = first_lane(pre[i]);
    const int hi = first_lane(pre[i + 1]);
    const int dl = rem - lo, dh = hi - rem;
    if (min(dl, dh) > tol) return x;
    return kvh * C + (dl <= dh ? lo : hi);
  }

  // Writes the cursor of group w, kCursorInts ints of LDS that only this
  // wave uses.
  __host__ __device__ __forceinline__ void start(int w, int *cur) const {
    int x = 0, x_end = 0, entry = 0;
    if (N > 0 && w < W) {
      x = bound(w);
      x_end = bound(w + 1);
      if (x < x_end) entry = find(x % C);
    }
    if (is_first_lane()) {
      cur[0] = x;
      cur[1] = x_end;
      cur[2] = entry;
      cur[3] = C;
      cur[4] = whole ? 1 : 0;
    }
  }

  // Next piece of the group: tiles [t0, t1) of the nt tiles of item it (an
  // item of no tokens counts one); false when the group is done. The cursor
  // lives in LDS because the kernels' tile loops leave it no registers.
  static __host__ __device__ __forceinline__ bool next(const PrefillParams &p, int bq, int nq,
                                                       const int *pre, int *cur, PrefillItem &it,
                                                       int &t0, int &t1, int &nt) {
    int x = first_lane(cur[0]);
    const int x_end = first_lane(cur[1]);
    int entry = first_lane(cur[2]);
    const int C = first_lane(cur[3]);
    const bool whole = first_lane(cur[4]) != 0;
    bool found = false;
    while (!found && x < x_end) {
      const int kvh = x / C;
      const int rem = x - kvh * C;
      if (rem == 0) entry = 0;  // a kv head's first item
      while (first_lane(pre[entry + 1]) <= rem) ++entry;
      const int s = entry / nq;
      const int lo = kvh * C + first_lane(pre[entry]);
      const int hi = kvh * C + first_lane(pre[entry + 1]);
      const int n_new = p.query_start_loc[s + 1] - p.query_start_loc[s];
      it.set(p, bq, s, kvh, folded(entry - s * nq, seq_tiles(n_new, bq, nq)));
      nt = tiles(it.kv_end);
      const int u = Cfg::tile_units((it.q_hi - it.q0) * p.group);
      const int end = min(x_end, hi);
      const int first = lo + Cfg::kItemUnits;
      t0 = whole ? 0 : min((max(0, x - first) + u - 1) / u, nt);
      t1 = whole ? nt : min((max(0, end - first) + u - 1) / u, nt);
      x = end;
      ++entry;
      found = t0 < t1;
    }
    if (is_first_lane()) {
      cur[0] = x;
      cur[2] = entry;
    }
    return found;
  }
};

// The kernel's argument, read again from where the launch left it: values
// that a long loop does not use are then not kept (or spilled) across it.
// `args` must be the kernel's first and only argument.
__device__ __forceinline__ PrefillArgs reload_args() {
  typedef const PrefillArgs __attribute__((address_space(4))) *args_t;
  args_t a = (args_t)__builtin_amdgcn_kernarg_segment_ptr();
  asm volatile("" : "+s"(a));
  PrefillArgs r;
  __builtin_memcpy(&r, (const PrefillArgs *)a, sizeof(r));
  return r;
}

// Records the partial that group w leaves of item `it`: its first part, or a
// later one that ends the item or not. One thread writes all of a group's.
__device__ __forceinline__ void prefill_note(const PrefillSplit &sp, int w, const PrefillItem &it,
                                             int group, bool begins, bool ends) {
  PrefillDesc *d = reinterpret_cast<PrefillDesc *>(sp.desc) + w;
  if (begins) {
    d->rows = (it.q_hi - it.q0) * group;
    d->row0 = it.qs + it.q0;
    d->q0 = it.q0;
    d->kvh = it.kvh;
  } else {
    d->cont = ends ? 2 : 1;
  }
}

// Merges the partials of the items that the split cut: workgroup (w, y)
// takes rows [y * merge_rows(ROWS), ..) of the item that group w begins and
// does not finish. Bound by memory latency for a few partials, by their bytes
// for many; so the descriptors of w and of the groups after it are read
// together, then the weights and contexts of a row's first four partials.
// LPR lanes share a row (16 bytes each), lane k of them weighs partial k.
//
// Rows of a workgroup: 16 of 256, so that one long item cut into many pieces
// still fills the chip (64 rows over 4000 cached tokens, 28/4 heads, bf16: 40 us
// a call against 52 at 32 rows and 54 at 64; the mixed step 115.5, 116.6 and
// 115.8); 32 of the fp32 kernel's 64 (OPT-125m prompts 40.0 us, at 16 40.8).
constexpr int merge_rows(int rows) { return rows > 64 ? 16 : 32; }

template <typename T, int D, int ROWS>
__global__ void __launch_bounds__(256)
prefill_merge(const PrefillArgs args) {
  constexpr int LPR = D / 4;
  constexpr int RPP = 256 / LPR;
  constexpr int kChunk = merge_rows(ROWS);
  static_assert(ROWS % kChunk == 0, "row chunks");
  const PrefillParams &p = args.p;
  const PrefillSplit &sp = args.sp;
  const PrefillDesc *desc = (const PrefillDesc *)sp.desc;
  const int w = blockIdx.x;
  const int lane = threadIdx.x & 63;
  const int32_t cont0 = desc[min(w + 1 + lane, sp.groups - 1)].cont;
  const PrefillDesc d = desc[w];
  const int r_end = min(d.rows, (int)(blockIdx.y + 1) * kChunk);
  if ((int)blockIdx.y * kChunk >= r_end) return;
  int n = 1;
  for (int b = w + 1; b < sp.groups; b += 64) {
    const int32_t c = b == w + 1 ? cont0 : desc[min(b + lane, sp.groups - 1)].cont;
    const uint64_t ends = __ballot(b + lane < sp.groups && c == 2);
    if (ends != 0) {
      n = b - w + __builtin_ctzll(ends) + 1;
      break;
    }
  }
  const int G = p.group;
  const int sub = threadIdx.x % LPR;
  const float c = fmaxf(fabsf(p.scale_log2), 0x1p-126f);  // as the kernels scale scores
  for (int r = blockIdx.y * kChunk + threadIdx.x / LPR; r < r_end; r += RPP) {
    auto row_of = [&](int k) {  // row of partial k in the workspace
      return (int64_t)(k == 0 ? 2 * w + 1 : 2 * (w + k)) * ROWS + r;
    };
    auto load4 = [&](int k0, f32x4 (&v)[4]) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        v[u] = load_vec<f32x4>(sp.ws_o + row_of(min(k0 + u, n - 1)) * D + 4 * sub);
    };
    const float m0 = sub < n ? sp.ws_m[row_of(sub)] : kNegInf;
    const float l0 = sub < n ? sp.ws_l[row_of(sub)] : 0.f;
    f32x4 v[4];
    load4(0, v);
    float M = m0;
    for (int k = sub + LPR; k < n; k += LPR) M = fmaxf(M, sp.ws_m[row_of(k)]);
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) M = fmaxf(M, __shfl_xor(M, off, LPR));
    const float Msub = M == kNegInf ? 0.f : M;
    float L = 0.f;
    f32x4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < n; k0 += LPR) {
      const int cnt = min(LPR, n - k0);
      float wk = 0.f;
      if (sub < cnt) {
        wk = fast_exp2(((k0 == 0 ? m0 : sp.ws_m[row_of(k0 + sub)]) - Msub) * c);
        L += (k0 == 0 ? l0 : sp.ws_l[row_of(k0 + sub)]) * wk;
      }
      for (int k = 0; k < cnt; k += 4) {  // four rows' loads in flight
        if (k0 + k > 0) load4(k0 + k, v);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const float f = __shfl(wk, min(k + u, LPR - 1), LPR);
          if (k + u < cnt) acc += v[u] * f;
        }
      }
    }
#pragma unroll
    for (int off = 1; off < LPR; off <<= 1) L += __shfl_xor(L, off, LPR);
    const int tok = r / G;
    const float inv =
        d.q0 + tok >= p.max_query_len ? __builtin_nanf("") : L > 0.f ? 1.f / L : 0.f;
    T *dst = (T *)p.out + (int64_t)(d.row0 + tok) * p.out_stride_token +
             (int64_t)(d.kvh * G + r % G) * p.out_stride_head + 4 * sub;
    if constexpr (sizeof(T) == 4) {
      store_vec<f32x4>(dst, acc * inv);
    } else {
      uint32_t h[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) h[e] = __builtin_bit_cast(uint16_t, (T)(acc[e] * inv));
      store_vec<u32x2>(dst, (u32x2){h[0] | (h[1] << 16), h[2] | (h[3] << 16)});
    }
  }
}

// Rows past the grid's query tiles (a chunk longer than max_query_len, a
// caller error) are filled with NaN by the workgroup of the last tile, so
// that the error shows in the output instead of stale memory.
template <typename T, int D, int NT>
__device__ __forceinline__ void prefill_nan_tail(const PrefillParams &p, const PrefillItem &it) {
  const T nan = (T)__builtin_nanf("");
  const int G = p.group;
  for (int idx = threadIdx.x; idx < (it.n_new - it.q_hi) * G * D; idx += NT) {
    const int d = idx % D;
    const int h = (idx / D) % G;
    const int tok = it.q_hi + idx / (D * G);
    ((T *)p.out)[(int64_t)(it.qs + tok) * p.out_stride_token +
                 (int64_t)(it.kvh * G + h) * p.out_stride_head + d] = nan;
  }
}

}  // namespace clv
