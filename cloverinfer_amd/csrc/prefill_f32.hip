// prefill_f32.hip - chunked prefill over paged KV with fp32 MFMAs.
//
// Semantics as in prefill.hip: query row i of sequence s sees cached
// positions p <= context_lens[s] - n_s + i; fp32 operands and accumulation
// throughout (v_mfma_f32_16x16x4f32, 256 FLOP per clock and CU, the bound of
// this kernel).
//
// A workgroup (4 waves; two per CU, three at head_dim 64) takes 64 query rows = bq
// tokens x G query heads of one kv head, 16 rows per wave, and streams
// 32-token K/V tiles through a two-stage LDS ring; the global loads of tile
// k + 1 are in flight while tile k is computed. 64 rows: a prompt of a few
// hundred tokens still gives each (sequence, head) several items, and the
// fp32 MFMA is slow enough (32 cycles) that 16 rows per wave already hide the
// LDS reads. Items are split evenly over the workgroups (prefill_split.h)
// where the launcher has a workspace.
//
// Measured against the VALU form (one workgroup per query row and kv head):
// 8 prompts of 54..500 tokens, 12 heads of 64, 174 -> 40 us; 4 x 512 tokens
// over 2048 cached, 12 heads of 64, 1584 -> 192 us (76 TFLOP/s), 32/8 heads of
// 128, 5069 -> 843 us (92 of the 154 TFLOP/s of a large fp32 product). The
// matrix pipes are busy half the time: waves wait on each other's issue and
// on LDS; short prompts are bound by the items' start and the merge. Batches of
// one-token rows stay with the VALU form (valu_is_faster).
//
// Fragments (lane = 16j + n16): the score MFMAs take K as A (row = token) and
// Q as B (column = query row), so that the lane ends up with the scores of
// row n16 at tokens 16h + 4j + e, which are its A operands of P.V as they
// are. The order of the sum over d and the placement of output columns are
// free: score MFMA (i, e) takes d = 16i + 4j + e and o[4w + e] holds columns
// 64w + 4 n16 + e, so every LDS read is 16 bytes and conflict-free.
//
// Accuracy: against 64 bits this kernel must not be further off than the
// VALU form it replaces, whose sums are short per-lane chains joined by
// trees. A score is therefore a tree over chains of two MFMAs (eight
// products), and P.V of a tile likewise, added to the running accumulator
// once per tile (which also folds the rescale into that add). Scores and row
// maxima stay raw: (s - m) * c rounds an exponent once, by its own size.
#include "prefill_split.h"

namespace clv {
namespace {

constexpr int kWaves = 4;
constexpr int kThreads = kWaves * 64;
constexpr int kRows = kWaves * 16;  // query rows per workgroup
constexpr int kBK = 32;             // K/V tokens per tile
static_assert(kWaves == 4, "the per-wave flags are read as one word");

// Workgroups (and so waves per SIMD) of a compute unit: what the registers
// allow. At head_dim 64 (162 VGPRs) three against two: 8 x 512 tokens, 12 heads
// 69.8 -> 65.1 us, 4 x 512 over 2048 cached 210 -> 192, one prompt of 512
// 26.2 -> 25.8; four (128 VGPRs, spilled) 85 us on the first.
constexpr int per_cu(int head_dim) { return head_dim == 64 ? 3 : 2; }

struct SplitCfg {
  static constexpr int kBK = clv::kBK;
  static constexpr int kItemUnits = 1;
  static constexpr int kMinShare = 3;
  static constexpr int kCutUnits = 3;
  static __host__ __device__ __forceinline__ int tile_units(int) { return 1; }
  static __host__ __device__ __forceinline__ int snap(int share) { return max(1, share / 16); }
};

__device__ __forceinline__ f32x4 mfma(uint32_t a, uint32_t b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(__builtin_bit_cast(float, a),
                                              __builtin_bit_cast(float, b), c, 0, 0, 0);
}

// Table width in tiles up to which a call is not split (measured as in
// prefill_mfma.hip, sum of 24 to 28 batches' times unsplit and split): 4 tiles 491
// and 586 us, 6 759 and 762, 7 933 and 800, 8 1200 and 981, 12 2065 and 1395.
constexpr int kSplitMinTiles = 6;

// Most items of a call (above, prefill_f32_chosen sends it to the VALU form).
constexpr int64_t kMaxItems = (int64_t)1 << 30;

// Item of workgroup `block` in the unsplit form. Consecutive ids go round-robin
// over the 8 XCDs: runs of `run` items are dealt to them in turn, each turn
// starting one XCD further, as a run's place among a sequence's query tiles may
// be the same every turn. A permutation of every 8 * run items.
__host__ __device__ inline int dealt_item(int block, int run) {
  const int xcd = block % 8, i = block / 8;
  const int turn = i / run;
  return (turn * 8 + ((xcd + turn + (turn >> 3)) & 7)) * run + i % run;
}

template <int D, bool SPLIT>
__global__ void __launch_bounds__(kThreads, per_cu(D))
chunked_prefill_f32(const PrefillArgs args) {
  constexpr int NQK = D / 16;            // 16-byte Q / K words per lane
  constexpr int CH = D / 16;             // output blocks
  constexpr int ROW = D + 4;             // LDS row stride (floats)
  constexpr int CPR = D / 4;             // 16-byte chunks per row
  constexpr int RPP = kThreads / CPR;    // rows per load pass
  constexpr int PASSES = kBK / RPP;
  constexpr int WROWS = 64 / CPR;        // rows of one load instruction of a wave
  __shared__ __attribute__((aligned(16))) float sK[2][kBK * ROW];
  __shared__ __attribute__((aligned(16))) float sV[2][kBK * ROW];
  __shared__ __attribute__((aligned(4))) uint8_t sValid[2][kBK];
  // Per wave: the V rows it staged hold a value that is not finite.
  __shared__ __attribute__((aligned(4))) uint8_t sInf[2][kWaves];
  __shared__ int s_pre[SPLIT ? kPrefillSplitItems + 1 : 1];
  __shared__ int s_tmp[3 * kWaves];
  __shared__ int s_cur[kWaves][PrefillSched<SplitCfg>::kCursorInts];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n16 = lane & 15;
  const int j = lane >> 4;
  typedef PrefillSched<SplitCfg> Sched;
  int L = SPLIT ? 0 : dealt_item(blockIdx.x, args.xcd_run);
  if constexpr (SPLIT) {
    Sched sched;
    sched.init<kThreads>(args.p, args.bq, args.n_qtiles, args.sp.groups, s_pre, s_tmp);
    L = sched.group_of(blockIdx.x);
    if (L < 0) return;
    sched.start(L, s_cur[wave]);
    if (tid == 0) sched.clear_desc(args.sp, L);
  } else if (L >= args.total) {
    return;
  }

  for (bool first = true;; first = false) {
    const PrefillArgs ar0 = SPLIT ? reload_args() : args;
    const PrefillParams &p = ar0.p;
    const int bq = ar0.bq, n_qtiles = ar0.n_qtiles;
    PrefillItem it;
    int t0 = 0, t1, nt;  // this workgroup's tiles of the item, and all of them
    if constexpr (SPLIT) {
      if (!Sched::next(p, bq, n_qtiles, s_pre, s_cur[wave], it, t0, t1, nt)) break;
    } else {
      if (!first) break;
      const int qt = n_qtiles - 1 - L % n_qtiles;  // longest query tiles first
      const int rest = L / n_qtiles;
      it.set(p, bq, rest / p.num_kv_heads, rest % p.num_kv_heads, qt);
      if (it.q0 >= it.n_new) break;
      nt = t1 = Sched::tiles(it.kv_end);
    }
    const int G = p.group;
    // A negative scale flips the sign of Q, a zero one becomes 2^-126 (weights
    // of 1 to far below fp32 resolution, 0 for masked scores): the softmax
    // multiplies by c > 0 only.
    const float c = fmaxf(fabsf(p.scale_log2), 0x1p-126f);
    const uint32_t qflip = p.scale_log2 < 0.f ? 0x80000000u : 0u;

    const char *kbase = (const char *)p.k_cache + (int64_t)it.kvh * p.kv_stride_head * 4;
    const char *vbase = (const char *)p.v_cache + (int64_t)it.kvh * p.kv_stride_head * 4;
    const int kv_end = it.kv_end;
    const int te = min(t1, (kv_end + kBK - 1) / kBK);  // 0 tokens: no tile at all

    // Q (B operand) of this lane's row 16 wave + n16.
    u32x4 q[NQK];
    int lim;  // last visible position of the row (-1: no row)
    {
      const int r = 16 * wave + n16;
      const int tok = it.q0 + r / G;
      const bool ok = r < bq * G && tok < it.n_new;
      lim = ok ? it.base_pos + tok : -1;
      const float *qrow = (const float *)p.q + (int64_t)(it.qs + (ok ? tok : it.q0)) * p.q_stride_token +
                          (int64_t)(it.kvh * G + (ok ? r % G : 0)) * p.q_stride_head + 4 * j;
#pragma unroll
      for (int i = 0; i < NQK; ++i) {
        q[i] = load_vec<u32x4>(qrow + 16 * i);
        q[i] ^= qflip;
        if (!ok) q[i] = (u32x4){0u, 0u, 0u, 0u};
      }
    }
    // Causal limits of the wave's first and last real rows: tiles at or below
    // the first need no mask, tiles past the last are left out by this wave.
    const int rows = (it.q_hi - it.q0) * G;
    int lim_first = -1, te_w = t0;
    if (16 * wave < rows) {
      lim_first = it.base_pos + it.q0 + 16 * wave / G;
      const int lim_last = it.base_pos + it.q0 + min(16 * wave + 15, rows - 1) / G;
      te_w = max(t0, min(te, lim_last < 0 ? 0 : lim_last / kBK + 1));
    }

    // Tile loader: thread handles chunk tid % CPR of rows tid / CPR + RPP * i;
    // the rows of one load instruction lie in one block (block_size >= WROWS).
    const int lchunk = tid % CPR;
    const int lrow = tid / CPR;
    const int wrow = WROWS * wave;
    const uint32_t sblk32 = (uint32_t)(p.kv_stride_block * 4), stok32 = (uint32_t)(p.kv_stride_token * 4);
    const uint32_t bmask = (1u << p.block_shift) - 1u;
    const uint32_t lane_off = (uint32_t)(lrow - wrow) * stok32 + (uint32_t)lchunk * 16u;
    typedef const int32_t __attribute__((address_space(4))) *cint_t;
    const cint_t brow = (cint_t)(p.block_tables + (int64_t)it.s * p.max_blocks_per_seq);
    u32x4 kreg[PASSES], vreg[PASSES];
    bool rvalid[PASSES];
    int rblk[PASSES];
    auto fetch_blocks = [&](int tile) {
#pragma unroll
      for (int i = 0; i < PASSES; ++i) {
        const int t = tile * kBK + wrow + RPP * i;
        rblk[i] = (tile < te && t < kv_end) ? brow[t >> p.block_shift] : -1;
      }
    };
    // Lanes whose token is not readable (past the context, or in an unmapped
    // block) read zeros from the buffer resource's range check. The range is
    // the bytes from a block's first row to the end of its last one, also
    // where rows overlap.
    auto load_tile = [&](int tile) {
#pragma unroll
      for (int i = 0; i < PASSES; ++i) {
        const uint32_t t = (uint32_t)(tile * kBK + wrow + RPP * i);
        const bool bok = (unsigned)rblk[i] < (unsigned)p.num_blocks;
        const bool ok = bok && (int)t + (lrow - wrow) < kv_end;
        rvalid[i] = ok;
        const uint64_t boff = (uint64_t)(uint32_t)(bok ? rblk[i] : 0) * sblk32;
        const int nrec = bok ? (int)(stok32 * bmask) + D * 4 : 0;
        const uint32_t voff = ok ? (t & bmask) * stok32 + lane_off : 0x80000000u;
        kreg[i] = buf_load<u32x4>(make_rsrc_range(kbase + boff, nrec), voff);
        vreg[i] = buf_load<u32x4>(make_rsrc_range(vbase + boff, nrec), voff);
      }
    };
    auto store_tile = [&](int buf) {
      bool bad = false;
#pragma unroll
      for (int i = 0; i < PASSES; ++i) {
        const int row = lrow + RPP * i;
        store_vec<u32x4>(&sK[buf][row * ROW + lchunk * 4], kreg[i]);
        store_vec<u32x4>(&sV[buf][row * ROW + lchunk * 4], vreg[i]);
        if (lchunk == 0) sValid[buf][row] = rvalid[i] ? 1 : 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) bad |= (vreg[i][e] & 0x7f800000u) == 0x7f800000u;
      }
      const bool any_bad = __any(bad);
      if (lane == 0) sInf[buf][wave] = any_bad ? 1 : 0;
    };

    f32x4 o[CH];
    float m_run = kNegInf, l_run = 0.f;
#pragma unroll
    for (int m = 0; m < CH; ++m) o[m] = (f32x4){0.f, 0.f, 0.f, 0.f};

    fetch_blocks(t0);
    if (t0 < te) {
      load_tile(t0);
      fetch_blocks(t0 + 1);
      store_tile(t0 & 1);  // the item before this one ended with a barrier
    }
    __syncthreads();

    for (int tile = t0; tile < te; ++tile) {
      const int buf = tile & 1;
      const bool more = tile + 1 < te;
      if (more) {
        load_tile(tile + 1);
        fetch_blocks(tile + 2);
      }
      if (tile < te_w) {
        // Scores: chains of two MFMAs (eight products), joined by a tree.
        f32x4 sacc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          f32x4 part[NQK / 4];  // the tree's level above four words of K
#pragma unroll
          for (int i4 = 0; i4 < NQK; i4 += 4) {
            f32x4 ch[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) ch[u] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const u32x4 k =
                  load_vec<u32x4>(&sK[buf][(16 * h + n16) * ROW + 16 * (i4 + i) + 4 * j]);
#pragma unroll
              for (int e = 0; e < 4; ++e)
                ch[4 * (i & 1) + e] = mfma(k[e], q[i4 + i][e], ch[4 * (i & 1) + e]);
            }
            part[i4 / 4] = ((ch[0] + ch[1]) + (ch[2] + ch[3])) + ((ch[4] + ch[5]) + (ch[6] + ch[7]));
          }
          sacc[h] = NQK == 8 ? part[0] + part[NQK / 4 - 1] : part[0];
        }
        const bool full = __all(sValid[buf][lane & 31] != 0) && tile * kBK + kBK - 1 <= lim_first;
        // Bit 4h + e: the row sees token 16h + 4j + e. Hidden scores become -inf.
        uint32_t vis = 0xffu;
        if (!full) {
          vis = 0;
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            const uint32_t vf = *reinterpret_cast<const uint32_t *>(&sValid[buf][16 * h + 4 * j]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const uint32_t seen = ((vf >> (8 * e)) & 1u) &
                                    (tile * kBK + 16 * h + 4 * j + e <= lim ? 1u : 0u);
              vis |= seen << (4 * h + e);
              if (seen == 0) sacc[h][e] = kNegInf;
            }
          }
        }
        float mx = kNegInf;
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) mx = fmaxf(mx, sacc[h][e]);
        mx = fmaxf(mx, shfl_xor(mx, 16));
        mx = fmaxf(mx, shfl_xor(mx, 32));
        const float m_new = fmaxf(m_run, mx);
        const float msub = m_new == kNegInf ? 0.f : m_new;
        const float alpha = fast_exp2((m_run - msub) * c);
        m_run = m_new;
        float pr[2][4];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int e = 0; e < 4; ++e) pr[h][e] = fast_exp2((sacc[h][e] - msub) * c);
        l_run = l_run * alpha + (((pr[0][0] + pr[0][1]) + (pr[0][2] + pr[0][3])) +
                                 ((pr[1][0] + pr[1][1]) + (pr[1][2] + pr[1][3])));
        float ar[4];  // alpha of the accumulator's rows 4j + r
#pragma unroll
        for (int r = 0; r < 4; ++r) ar[r] = shfl(alpha, 4 * j + r);

        if (full || *reinterpret_cast<const uint32_t *>(&sInf[buf][0]) == 0) {
#pragma unroll
          for (int w = 0; w < CH / 4; ++w) {
            u32x4 v[2][4];
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int k = 0; k < 4; ++k)
                v[h][k] = load_vec<u32x4>(&sV[buf][(16 * h + 4 * j + k) * ROW + 64 * w + 4 * n16]);
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              f32x4 t[2][2];
#pragma unroll
              for (int h = 0; h < 2; ++h)
#pragma unroll
                for (int k = 0; k < 2; ++k) t[h][k] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
              for (int k = 0; k < 4; ++k)
#pragma unroll
                for (int h = 0; h < 2; ++h)
                  t[h][k & 1] = mfma(__builtin_bit_cast(uint32_t, pr[h][k]), v[h][k][e], t[h][k & 1]);
              const f32x4 sum = (t[0][0] + t[0][1]) + (t[1][0] + t[1][1]);
#pragma unroll
              for (int r = 0; r < 4; ++r)
                o[4 * w + e][r] = __builtin_fmaf(o[4 * w + e][r], ar[r], sum[r]);
            }
          }
        } else {
          // A masked tile with an infinity or NaN in V: a row must not take
          // 0 * inf from tokens it does not see, so its tokens are added one
          // by one.
#pragma unroll
          for (int m = 0; m < CH; ++m)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[m][r] *= ar[r];
          for (int t = 0; t < kBK; ++t) {
            float pv = 0.f;
            uint32_t seen = 0;
#pragma unroll
            for (int h = 0; h < 2; ++h)
#pragma unroll
              for (int e = 0; e < 4; ++e)
                if (t == 16 * h + 4 * j + e) {
                  pv = pr[h][e];
                  seen = (vis >> (4 * h + e)) & 1u;
                }
            const int src = 16 * ((t >> 2) & 3);  // lanes that hold token t
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float a = shfl(pv, src + 4 * j + r);
              const bool s = __shfl((int)seen, src + 4 * j + r, 64) != 0;
#pragma unroll
              for (int m = 0; m < CH; ++m) {
                const float v = sV[buf][t * ROW + 64 * (m >> 2) + 4 * n16 + (m & 3)];
                o[m][r] = s ? __builtin_fmaf(a, v, o[m][r]) : o[m][r];
              }
            }
          }
        }
      }
      if (more) store_tile(buf ^ 1);
      __syncthreads();
    }

    l_run += shfl_xor(l_run, 16);
    l_run += shfl_xor(l_run, 32);
    // The rest of the arguments are read only now.
    const PrefillArgs ar1 = SPLIT ? reload_args() : args;
    const bool whole = !SPLIT || (t0 == 0 && t1 == nt);
    const int64_t prow = (int64_t)(2 * L + (t0 == 0 ? 1 : 0)) * kRows;  // partial's first row
    if constexpr (SPLIT) {
      if (!whole) {
        if (tid == 0) prefill_note(ar1.sp, L, it, G, t0 == 0, t1 == nt);
        if (j == 0 && 16 * wave + n16 < rows) {
          ar1.sp.ws_m[prow + 16 * wave + n16] = m_run;
          ar1.sp.ws_l[prow + 16 * wave + n16] = l_run;
        }
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int row = 16 * wave + 4 * j + r;
      const float l = shfl(l_run, 4 * j + r);
      if (row >= rows) continue;
      const int tok = it.q0 + row / G;
      float *dst;
      float inv;
      if (whole) {
        // A row at or past max_query_len (a caller error) is marked with NaN.
        inv = tok >= ar1.p.max_query_len ? __builtin_nanf("") : l > 0.f ? 1.f / l : 0.f;
        dst = (float *)ar1.p.out + (int64_t)(it.qs + tok) * ar1.p.out_stride_token +
              (int64_t)(it.kvh * G + row % G) * ar1.p.out_stride_head;
      } else {
        inv = 1.f;
        dst = ar1.sp.ws_o + (prow + row) * D;
      }
#pragma unroll
      for (int w = 0; w < CH / 4; ++w)
        store_vec<f32x4>(dst + 64 * w + 4 * n16,
                         (f32x4){o[4 * w][r] * inv, o[4 * w + 1][r] * inv, o[4 * w + 2][r] * inv,
                                 o[4 * w + 3][r] * inv});
    }
    if (t1 == nt && it.qt == ar1.n_qtiles - 1 && it.q_hi < it.n_new)
      prefill_nan_tail<float, D, kThreads>(ar1.p, it);
  }
}

template <int D>
hipError_t launch_td(const PrefillParams &p, const PrefillSplit *sp, hipStream_t stream) {
  PrefillArgs args{};
  args.p = p;
  args.bq = kRows / p.group;
  args.n_qtiles = max(1, (p.max_query_len + args.bq - 1) / args.bq);
  const int64_t total = (int64_t)p.num_seqs * p.num_kv_heads * args.n_qtiles;
  if (total > kMaxItems) return hipErrorInvalidValue;
  if (sp != nullptr) {
    args.sp = *sp;
    hipLaunchKernelGGL((chunked_prefill_f32<D, true>), dim3((unsigned)sp->groups), dim3(kThreads),
                       0, stream, args);
    hipLaunchKernelGGL((prefill_merge<float, D, kRows>),
                       dim3((unsigned)sp->groups, kRows / merge_rows(kRows)), dim3(256), 0, stream,
                       args);
    return hipGetLastError();
  }
  args.total = (int)total;
  // Query tiles of one kv head share the L2 of their XCD. Where most of the
  // (sequence, query tile) pairs hold rows, each XCD takes an eighth of the
  // items in a row. Where most are empty (one long chunk among one-token rows)
  // that eighth can be all the work there is, and short runs are dealt: 24
  // sequences over 0..4000 tokens, one bringing 2048, 32/8 heads 12808 -> 2199
  // us; 8 x 180 tokens, 28/4 heads, 44 us in eighths and 50 dealt.
  const int64_t filled = p.num_seqs + p.num_tokens / args.bq;
  const bool dense = 2 * filled >= (int64_t)p.num_seqs * args.n_qtiles;
  args.xcd_run = (int)std::max<int64_t>(1, dense ? (total + 7) / 8 : std::min(8, args.n_qtiles));
  const int64_t turn = 8 * (int64_t)args.xcd_run;
  hipLaunchKernelGGL((chunked_prefill_f32<D, false>),
                     dim3((unsigned)((total + turn - 1) / turn * turn)), dim3(kThreads), 0, stream,
                     args);
  return hipGetLastError();
}

}  // namespace

// Calls of few rows per (sequence, kv head) that the VALU form does faster: a
// workgroup of 64 rows spends its time on an item's start, and on few tokens, or
// once the items fill the device (`slots` workgroups), nothing hides it. Batches
// over ragged contexts up to the given length, us of the MFMA form and of the
// VALU form:
//   one token a sequence, not split:
//     12/12 heads of 64: 1 x 190 15.4, 9.3; 64 x 190 17.8, 15.2; 1200 x 190 235, 153;
//     32/32 of 128: 4 x 100 17.4, 10.2; 64 x 60 38.9, 16.9; 1200 x 60 619, 246;
//     16/8 of 128: 4 x 100 14.2, 12.5; 32 x 190 25.2, 28.4; 128 x 190 47.6, 32.5;
//     24/12 of 64: 16 x 100 11.2, 9.2; 64 x 190 19.3, 20.1;
//     32/8 of 128: 16 x 60 11.1, 13.8; 64 x 190 27.8, 41.0; 128 x 60 22.9, 20.0;
//       512 x 60 76.2, 44.1;
//     28/4 of 128: 512 x 60 42.8, 79.4;
//   split:
//     12/12 of 64: 128 x 500 58.8, 45.1; 128 x 1000 105, 124; 128 x 4000 288, 465;
//     32/32 of 128: 16 x 500 45.9, 56.9; 64 x 500 165, 142;
//     16/8 of 128: 128 x 500 81.5, 75.4; 32/8 of 128: 128 x 500 94.0, 127;
//   every 32nd sequence brings 33 tokens:
//     12/12 of 64: 64 x 190 (split) 37.7, 20.1; 1200 x 60 126, 95;
//     16/8 of 128: 1200 x 190 632, 323;
//   2.8 tokens a sequence on average: 12/12 of 64, 256 x 500 142, 150.
static bool valu_is_faster(const PrefillParams &p, int64_t entries) {
  const int64_t tokens = p.num_tokens, seqs = p.num_seqs, items = seqs * p.num_kv_heads;
  const int64_t slots = per_cu(p.head_dim) * 8 * (int64_t)p.cus_per_xcd;
  const int64_t tiles = (((int64_t)p.max_blocks_per_seq << p.block_shift) + kBK - 1) / kBK;
  if (tiles <= kSplitMinTiles || entries > kPrefillSplitItems)
    return p.group <= 4 && 2 * tokens <= 5 * seqs &&
           (p.group == 1 || (p.group == 2 && tiles <= 4) || items >= 2 * slots);
  return tiles <= 16 && p.group <= 2 && tokens <= 2 * seqs &&
         items >= (p.group * p.head_dim == 64 ? 1 : 2) * slots;
}

bool prefill_f32_chosen(const PrefillParams &p, int block_size) {
  // One load instruction of a wave covers 256 / head_dim rows of one block,
  // and offsets inside a block are 32-bit bytes. The grid of the unsplit form
  // has a workgroup per (sequence, kv head, query tile).
  const uint64_t lim = (uint64_t)1 << 31;
  if (!((p.head_dim == 64 || p.head_dim == 128) && block_size >= 4 && p.group <= kRows &&
        (uint64_t)p.kv_stride_block * 4 < lim &&
        ((uint64_t)p.kv_stride_token * 4 << p.block_shift) < lim))
    return false;
  const int64_t bq = kRows / p.group;
  const int64_t entries =
      p.num_seqs * std::max<int64_t>(1, ((int64_t)p.max_query_len + bq - 1) / bq);
  return entries * p.num_kv_heads <= kMaxItems && !valu_is_faster(p, entries);
}

PrefillSplitShape prefill_f32_split_shape(const PrefillParams &p) {
  return prefill_split_shape(p, kRows, kBK, per_cu(p.head_dim), 1, kSplitMinTiles, false);
}

hipError_t launch_prefill_f32(const PrefillParams &p, const PrefillSplit *sp, hipStream_t stream) {
  if (p.head_dim == 128) return launch_td<128>(p, sp, stream);
  if (p.head_dim == 64) return launch_td<64>(p, sp, stream);
  return hipErrorInvalidValue;
}

}  // namespace clv
