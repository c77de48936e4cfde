// Stage 2: block-sparse flash attention on bf16/fp16 MFMA (v_mfma_f32_32x32x16_*).
//
// Exact softmax attention of each 128-row query block over the key blocks its row of the
// kernel mask selects, with natural-log LSE -- the semantics of the external
// block_sparse_attn_func call at recap/kernels/block_sparse.py:111-138.  Same kernel, all
// blocks kept, is the dense attention + LSE of a refresh (recap/operator.py:254-256).
//
// Workgroup = one (bank, query block): 4 waves x 32 query rows.  Each wave computes
// S^T = K Q^T (keys x queries) so that a lane owns one query row: the row max needs one
// lane-pair exchange per key tile and the row sum none until the end.  The fp32 S^T
// registers become the B operand P^T of O^T = V^T P^T directly; the packed V^T tile stores
// its keys in the matching order (swap23), so no shuffle is needed.  K and V^T tiles are
// verbatim images in HBM (written once per call by pack_pool) copied into XOR-swizzled
// LDS.  Q rows and the output rows go through the Hilbert row map, i.e. the reorder and
// restore of recap/operator.py:496-498, 527 are fused into the loads and stores.
//
// Epilogues:
//   head   (oh, lh) in reordered order, oh rounded to the query type as the external
//          kernel's bf16 output is -- the head branch a refresh capture needs;
//   dense  output + LSE in native order -- a refresh's dense call;
//   dense-head  both of a refresh in one pass: the kept blocks are walked first, the head
//          branch is stored when they are done, then the remaining blocks complete the
//          dense output;
//   merge  head (+) [coarse tail + drift-weighted refinement] in LSE space for rows < R,
//          the head alone above (recap/kernels/detail_cache.py:220-301), written in
//          native order: the whole corrected sparse output in one pass.  The head enters
//          the merge rounded to the query type, as the reference's head tensor does.
// The masked modes walk their kept blocks in one order (a kept ragged last block first,
// then ascending), and dense-head stores its head branch before the first block after the
// kept ones can move the running max, so the head branch of head, dense-head and merge
// modes is the same bit for bit; a long row that head or merge mode walks in segments (below)
// differs from it by the order of its sums.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "kernels.hpp"

namespace recap {

constexpr int kMaxTiles = 2048;

// Rows whose running max grows by less than this (log2 units) keep their stale max: p then
// stays below 2^8, exact in fp32 and bf16, and the O rescale is skipped.
constexpr float kRescaleSlack = 8.0f;

// At d = 64 a step has half the MFMA work of d = 128 for the same softmax work per score,
// so the VALU bounds it.  There the running max is instead raised only when a sub-tile's
// probabilities, taken against the current max, sum to more than kSumCap in some lane (or
// are not finite): the sub-tile is then redone against its own max, and no row max is taken
// on the common path (every accepted p is <= kSumCap, exact in fp32 and bf16).
constexpr float kSumCap = 4096.0f;

// s_waitcnt immediate (gfx9 encoding: vmcnt bits 3:0 and 15:14, expcnt 6:4, lgkmcnt 11:8)
// that waits for all vector memory operations of this wave -- the tile copies into LDS --
// and all its LDS reads.
constexpr int kWaitVmLgkm0 = 0x7 << 4;

// Wait for this wave's copies into LDS and its LDS reads, then for every wave of the
// workgroup: afterwards the copied sub-tiles are visible and the slots read so far may be
// overwritten.  The copies count on vmcnt only, so the wait is spelled out.
__device__ inline void tile_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(kWaitVmLgkm0);
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Wait for this wave's LDS accesses, then for every wave, with its global loads (the Q rows)
// left in flight.
__device__ inline void lds_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(0xf | (0x7 << 4) | (0x3 << 14));  // lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Each wave owns kGroups groups of 32 query rows, so every K/V fragment it reads from LDS
// feeds kGroups MFMAs; a 128-row query block then takes kThreads threads.  kGroups = 2
// halves the LDS reads and is correct, but at d = 128 it needs one wave per SIMD and the
// compiler then keeps every MFMA result in AGPRs: it measured slower.
constexpr int kGroups = 1;
constexpr int kRowsPerWave = 32 * kGroups;
constexpr int kThreads = 64 * (kBlock / kRowsPerWave);

// A bank's drift centre from the coarse tail's partial sums, in drift_center's order (256
// threads' runs, then its halving tree), by one whole wave: a launch of its own less per call.
__device__ inline float drift_centre(const float* part, int tiles, int rows) {
  const int lane = threadIdx.x & 63, per = (tiles + 255) / 256;
  float v[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int t = lane + 64 * k;
    v[k] = 0.0f;
    for (int i = t * per; i < min((t + 1) * per, tiles); ++i) v[k] += part[i];
  }
  float x = (v[0] + v[2]) + (v[1] + v[3]);
  for (int off = 32; off >= 1; off >>= 1) x += __shfl_down(x, off, 64);
  return __uint_as_float((unsigned)__builtin_amdgcn_readfirstlane((int)__float_as_uint(x))) / (float)rows;
}

// Final normalisation and store of one query row per lane pair, in the layout of the kernel's
// mode.  Lane (g, l32) holds columns 32 dt + 8 q4 + 4 g .. +3 of its row; one exchange of
// packed words within the lane pair gives it 8 consecutive ones, 32 dt + 16 j + 8 g .., so that
// every access moves 16 bytes.  In merge mode the row's coarse output and refinement are all
// requested before the first of them is used: with the loads between the stores (which the
// compiler must keep in order: the output might be one of the inputs) each 8-byte load waited
// out the memory's latency, 16-18 us a work item of 100-200 us; now 5-7.
template <class T, int D, int MODE>
__device__ inline void store_rows(const AttnArgs& a, int bank, int b, int h, int r, int nat,
                                  int g, const f32x16 (&oacc)[D / 32], float m, float lt) {
  constexpr int NV = D / 16;  // 16-byte vectors of a lane
  const float inv = 1.0f / lt;
  const float lse = (m + log2f(lt)) * kLn2;
  auto col = [&](int i) { return 16 * i + 8 * g; };
  // The output rounded to the query type, columns col(i) .. col(i) + 7.
  auto packed = [&](int i) {
    const f32x16& o = oacc[i >> 1];
    const int e = 8 * (i & 1);
    u32x4 v;
#pragma unroll
    for (int w = 0; w < 2; ++w) {
      const unsigned lo = pack2<T>(o[e + 2 * w] * inv, o[e + 2 * w + 1] * inv);
      const unsigned hi = pack2<T>(o[e + 4 + 2 * w] * inv, o[e + 4 + 2 * w + 1] * inv);
      const auto x = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
      v[w] = x[0];
      v[2 + w] = x[1];
    }
    return v;
  };

  if constexpr (MODE == kModeHead) {
    // Head branch in the query type (the reference's head is the bf16 tensor its attention
    // kernel returns, recap/operator.py:366-370); the capture reads it back from here.
    uint16_t* orow = a.head_out + ((int64_t)bank * a.n_tokens + r) * D;
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<u32x4*>(orow + col(i)) = packed(i);
    if (g == 0) a.head_lse[(int64_t)bank * a.n_tokens + r] = lse;
    return;
  }

  uint16_t* orow = a.out + b * a.osB + h * a.osH + (int64_t)nat * a.osN;
  if constexpr (MODE == kModeDense) {
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<u32x4*>(orow + col(i)) = packed(i);
    if (g == 0) a.lse_native[(int64_t)bank * a.n_tokens + nat] = lse;
    return;
  }

  // Merge epilogue (recap/kernels/detail_cache.py:228-301): rows < R get the drift-weighted
  // tail.  The head is rounded to the query type first: the reference merges the head
  // tensor its attention kernel stored in that type (recap/operator.py:500-509, loaded with
  // .to(float32) at recap/kernels/detail_cache.py:228-234).
  if (r < a.rows) {
    const int64_t ri = (int64_t)bank * a.rows + r;
    const uint16_t* gorow = a.go + ri * D;
    const uint16_t* drow = a.det + ri * D;
    u32x4 gv[NV], dv[NV];
    const float glv = a.gl[ri], dlv = a.dl[ri];
    float move = 0.0f;
    if (!a.use_override) {
      // Every lane is here: r < R for all 128 rows of a query block or for none.
      const int tiles = a.rows / kBlock;
      const float centre = a.center != nullptr
                               ? a.center[bank]
                               : drift_centre(a.drift_part + (int64_t)bank * tiles, tiles, a.rows);
      move = glv - a.glref[ri] - centre;
    }
#pragma unroll
    for (int i = 0; i < NV; ++i) gv[i] = *reinterpret_cast<const u32x4*>(gorow + col(i));
#pragma unroll
    for (int i = 0; i < NV; ++i) dv[i] = *reinterpret_cast<const u32x4*>(drow + col(i));
    asm volatile("" ::: "memory");  // all of them before the first store
    const float admit = a.use_override ? a.alpha_override : expf(-fabsf(move));
    const float cl = glv + dlv;
    const float tc = fmaxf(glv, cl);
    const float sm = (1.0f - admit) * expf(glv - tc);
    const float cm = admit * expf(cl - tc);
    const float den = fmaxf(sm + cm, 1.0e-30f);
    const float tl = tc + logf(den);
    const float common = fmaxf(lse, tl);
    const float wh = expf(lse - common);
    const float wt = expf(tl - common);
    const float den2 = fmaxf(wh + wt, 1.0e-30f);
    // One reciprocal per denominator and row instead of a division per element.
    const float rden = 1.0f / den, rden2 = 1.0f / den2;
#pragma unroll
    for (int i = 0; i < NV; ++i) {
      const u32x4 hv = packed(i);
      u32x4 v;
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        float res[2];
#pragma unroll
        for (int e = 0; e < 2; ++e) {
          const float gov = T::to_f((uint16_t)(e ? gv[i][w] >> 16 : gv[i][w] & 0xffff));
          const float detv = f16_to_f((uint16_t)(e ? dv[i][w] >> 16 : dv[i][w] & 0xffff));
          const float ohv = T::to_f((uint16_t)(e ? hv[w] >> 16 : hv[w] & 0xffff));
          const float to = (gov * sm + (gov + detv) * cm) * rden;
          res[e] = (ohv * wh + to * wt) * rden2;
        }
        v[w] = pack2<T>(res[0], res[1]);
      }
      *reinterpret_cast<u32x4*>(orow + col(i)) = v;
    }
  } else {
#pragma unroll
    for (int i = 0; i < NV; ++i) *reinterpret_cast<u32x4*>(orow + col(i)) = packed(i);
  }
}

// The segments of a long row: each one's state (O^T, running max, row sum) goes to the
// workspace, and the last one to arrive combines them all, in segment order, so the result
// does not depend on which one that is.  True for the workgroup that then holds the row's
// state.  The segments run on different XCDs, whose L2 caches are not coherent within a
// launch: the state is written and read with the SC1 bit (agent scope), past those caches, and
// every store has been acknowledged (vmcnt) before its segment is counted.
template <int D>
__device__ inline bool merge_segments(const AttnArgs& a, int item, int seg, int nseg, int* shared,
                                      f32x16 (&oacc)[D / 32], float& m, float& lt) {
  static_assert(kGroups == 1, "one query group per wave");
  constexpr int NDT = D / 32;
  constexpr int kAgent = 16;             // SC1
  constexpr int kVec = 16 * kThreads;    // bytes of one 16-byte vector of every thread
  constexpr int kState = 4 * NDT * kVec; // O^T of a segment; max and sum follow it
  constexpr int kBytes = attn_part_words(D) * 8;
  int t = threadIdx.x;
  asm volatile("" : "+v"(t));  // keeps the addresses below out of the registers of the walk
  const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(a.part + (int64_t)item * nseg * attn_part_words(D)), 0, nseg * kBytes, kBufferRsrcWord3);
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
    for (int e = 0; e < 16; e += 4) {
      const f32x4 x = {oacc[dt][e], oacc[dt][e + 1], oacc[dt][e + 2], oacc[dt][e + 3]};
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, x), rs,
                                             16 * t + (4 * dt + e / 4) * kVec, seg * kBytes, kAgent);
    }
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u32x2, f32x2{m, lt}), rs, kState + 8 * t,
                                        seg * kBytes, kAgent);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(kWaitVmLgkm0);
  __syncthreads();
  if (t == 0)
    *shared = (int)__hip_atomic_fetch_add(a.tickets + item, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __syncthreads();
  if (__builtin_amdgcn_readfirstlane(*shared) != nseg - 1) return false;
  float ms[kMaxSplit], ls[kMaxSplit];
#pragma unroll
  for (int s = 0; s < kMaxSplit; ++s) {
    ms[s] = -INFINITY;
    ls[s] = 0.0f;
    if (s < nseg) {
      const f32x2 x = __builtin_bit_cast(f32x2, __builtin_amdgcn_raw_buffer_load_b64(rs, kState + 8 * t, s * kBytes, kAgent));
      ms[s] = x[0];
      ls[s] = x[1];
    }
  }
  float top = ms[0];
#pragma unroll
  for (int s = 1; s < kMaxSplit; ++s) top = fmaxf(top, ms[s]);
#pragma unroll
  for (int dt = 0; dt < NDT; ++dt) oacc[dt] = f32x16{};
  m = top;
  lt = 0.0f;
#pragma unroll
  for (int s = 0; s < kMaxSplit; ++s) {
    if (s < nseg) {
      // The whole state requested before its first use.
      u32x4 x[4 * NDT];
#pragma unroll
      for (int i = 0; i < 4 * NDT; ++i)
        x[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, 16 * t + i * kVec, s * kBytes, kAgent);
      __builtin_amdgcn_sched_barrier(0);
      const float w = ms[s] == -INFINITY ? 0.0f : __builtin_amdgcn_exp2f(ms[s] - top);
      lt = fmaf(w, ls[s], lt);
#pragma unroll
      for (int i = 0; i < 4 * NDT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          oacc[i / 4][4 * (i % 4) + e] = fmaf(w, __uint_as_float(x[i][e]), oacc[i / 4][4 * (i % 4) + e]);
    }
  }
  return true;
}

// Starts on a multiple of 16 KB: with cold caches a short launch otherwise depends on where the
// linker puts the code (the same 40 KB at 0x3600 past such a boundary 83-85 us, at 0x0, 0x1600 and
// 0x2000 72-76, at 12 heads x 4,856 tokens in fp16; no difference once the code is warm).
template <class T, int D, int MODE>
__global__ __launch_bounds__(kThreads, 2) __attribute__((aligned(16384)))
void attention_kernel(AttnArgs a) {
  using G = TileGeom<D>;
  constexpr int NS = D / 16;                  // k-steps over the head dimension
  constexpr int NDT = D / 32;                 // 32-row tiles of O^T
  constexpr int HALF = G::kHalfBytes;         // K or V^T image of a 64-key sub-tile
  constexpr int NDMA = HALF / (16 * kThreads);  // 16-byte copies per thread per image
  // LDS: K images of sub-tiles 2k / 2k+1 in k_lds0 / k_lds1, V^T images likewise.  Four
  // separate arrays, each access naming one of them at compile time (the step parity is
  // static): the compiler can then tell that a step's fragment reads do not touch the slots
  // its copies are filling, and does not wait for those copies before the reads.
  __shared__ __attribute__((aligned(16))) char k_lds0[HALF];
  __shared__ __attribute__((aligned(16))) char k_lds1[HALF];
  __shared__ __attribute__((aligned(16))) char v_lds0[HALF];
  __shared__ __attribute__((aligned(16))) char v_lds1[HALF];
  __shared__ int list[MODE == kModeDense ? 1 : kMaxTiles];
  __shared__ int counts[kMaxTiles / 64];  // kept blocks per 64 blocks of the mask row

  const int t = threadIdx.x, lane = t & 63, g = lane >> 5, l32 = lane & 31;
  const int wave = __builtin_amdgcn_readfirstlane(t >> 6);
  // Work items.  The long rows of every bank (query blocks ds .. tb-1: the text rows and a
  // ragged last video block, all dense) come first, dealt round-robin over the XCDs
  // (workgroup i runs on XCD i % 8): they start before the short ones and every XCD gets an
  // equal share.  The other rows follow in runs of 64 query blocks per XCD (about the
  // workgroups one XCD holds at once): the neighbouring Hilbert-ordered blocks in flight on
  // an XCD share many key tiles in its L2, and all XCDs together stay within ~512 blocks of
  // one bank, whose K/V images (58 MB at the HunyuanVideo shape) stay in the 256 MB
  // Infinity Cache.
  //
  // With a queue the workgroups are persistent (about two per CU) and claim their items:
  // XCD x holds the positions p = x, x + 8, x + 16, ... in that order, and a workgroup takes
  // the next one of its own XCD (one atomic increment) or, once those are all taken, of the
  // next XCD that still has one; it stops when every queue is empty.  XCDs that run faster
  // then process the slower ones' last items instead of idling.  Every increment below an
  // XCD's count claims a distinct position, so each item is processed exactly once.
  //
  // In the masked modes each long row is `split` items, segments of its list of kept blocks:
  // a long row alone takes as long as tb / keep of the others, which bounds a launch with few
  // rounds of items (see attn_split).
  __shared__ int claimed;
  // The arguments that only one part of an item needs are read again there from the kernel's
  // argument segment: kept over the walk they would take registers from it.
  auto reread = []() -> const AttnArgs& {
    typedef const __attribute__((address_space(4))) AttnArgs KernelArgs;
    KernelArgs* args = (KernelArgs*)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(args));
    return *(const AttnArgs*)args;
  };
  constexpr bool kSplits = MODE == kModeHead || MODE == kModeMerge;
  const int split = kSplits ? a.split : 1;
  const int nlong = a.tb - a.ds, nshort = a.ds;
  const int n_long_items = a.banks * nlong * split;
  const int n_items = n_long_items + a.banks * nshort;
  const bool persistent = a.queue != nullptr;
  for (int round = 0;; ++round) {
  int pos = blockIdx.x;
  if (persistent) {
    if (t == 0) {
      const int own = blockIdx.x & 7;
      int got = -1;
      for (int k = 0; k < 8 && got < 0; ++k) {
        const int x = (own + k) & 7;
        const int count = (n_items - x + 7) >> 3;  // positions on XCD x
        const int i = (int)atomicAdd(a.queue + kQueueStride * x, 1u);
        if (i < count) got = 8 * i + x;
      }
      claimed = got;  // -1: every queue is empty
    }
    __syncthreads();
    pos = __builtin_amdgcn_readfirstlane(claimed);
    if (pos < 0) break;
  } else if (round > 0) {
    break;
  }
  int bank, qt, seg = 0, nseg = 1;
  if (pos < n_long_items) {
    const int li = pos / split;
    bank = li / nlong;
    qt = a.ds + li % nlong;
    seg = pos % split;
    nseg = split;
  } else {
    const int lin = xcd_runs(pos - n_long_items, n_items - n_long_items, 64);
    bank = lin / nshort;
    qt = lin % nshort;
  }
  const int b = bank / a.heads, h = bank % a.heads;

  const AttnArgs& early = reread();
  // Query group q of this wave: rows 32 q .. 32 q + 31 of the wave's kRowsPerWave.  The row
  // map, the mask row and the Q rows are all requested before the first of them is used.
  int row[kGroups], nat[kGroups];
  bool valid[kGroups];
#pragma unroll
  for (int q = 0; q < kGroups; ++q) {
    row[q] = qt * kBlock + wave * kRowsPerWave + 32 * q + l32;
    valid[q] = row[q] < a.n_tokens;
    nat[q] = valid[q] ? early.rowmap[row[q]] : 0;
  }
  // A copy of the thread index that the compiler cannot see through: what is derived from it
  // is computed per item instead of being kept in registers over all items.
  int tt = t;
  asm volatile("" : "+v"(tt));
  constexpr int kChunks = MODE == kModeDense ? 1 : kMaxTiles / kThreads;
  const int nchunks = (a.tb + kThreads - 1) / kThreads;
  uint8_t cell[kChunks];
  bool lead = false;
  if constexpr (MODE != kModeDense) {
    const uint8_t* mrow = early.kmask + ((int64_t)bank * a.tb + qt) * a.tb;
#pragma unroll
    for (int i = 0; i < kChunks; ++i)
      if (i < nchunks) cell[i] = mrow[min(kThreads * i + tt, a.tb - 1)];
    // A kept ragged last block goes first, so its masked steps open the walk (in dense-head
    // mode the blocks that are not kept follow the kept ones, and the ragged block would
    // otherwise fall in the middle); every masked mode uses the same order.
    lead = (a.n_tokens % kBlock) != 0 && mrow[a.tb - 1] != 0;
  }
  u32x4 qreg[kGroups][NS];
#pragma unroll
  for (int q = 0; q < kGroups; ++q) {
    const uint16_t* qrow = early.q + b * early.qsB + h * early.qsH + (int64_t)nat[q] * early.qsN;
#pragma unroll
    for (int s = 0; s < NS; ++s)
      qreg[q][s] = valid[q] ? *reinterpret_cast<const u32x4*>(qrow + 16 * s + 8 * g)
                            : u32x4{0u, 0u, 0u, 0u};
  }

  int nkeep = a.tb, first = 0;  // blocks of this item's walk: list[first ..]
  if constexpr (MODE != kModeDense) {
    // Kept blocks in ascending order; in dense-head mode the other blocks follow them.  Block
    // j's place is the number of kept blocks before it: the counts of the earlier groups of
    // 64 blocks, scanned by every wave for itself, plus the kept lanes below it in its
    // ballot.  Two barriers a row (a scan over the 256 threads took 18).
    const int ln = tt & 63;
    unsigned kept = 0;
#pragma unroll
    for (int i = 0; i < kChunks; ++i)
      if (i < nchunks) {
        const bool on = kThreads * i + tt < a.tb && cell[i] != 0;
        const unsigned long long bal = __ballot(on);
        kept |= (unsigned)on << i;
        if (ln == 0) counts[kThreads / 64 * i + wave] = (int)__popcll(bal);
      }
    lds_barrier();
    const int own = ln < kThreads / 64 * nchunks ? counts[ln] : 0;
    int upto = own;  // inclusive
#pragma unroll
    for (int off = 1; off < kMaxTiles / 64; off <<= 1) {
      const int u = __shfl_up(upto, off, 64);
      if (ln >= off) upto += u;
    }
    nkeep = __builtin_amdgcn_readlane(upto, kMaxTiles / 64 - 1);
#pragma unroll
    for (int i = 0; i < kChunks; ++i)
      if (i < nchunks) {
        const bool on = (kept >> i) & 1u;
        const unsigned long long bal = __ballot(on);
        const int j = kThreads * i + tt;
        const int before = __shfl(upto - own, kThreads / 64 * i + wave, 64) +
                           (int)__popcll(bal & ((1ull << ln) - 1ull));
        if (on)
          list[lead ? (j == a.tb - 1 ? 0 : before + 1) : before] = j;
        else if (MODE == kModeDenseHead && j < a.tb)
          list[nkeep + (j - before)] = j;
      }
    lds_barrier();
    if constexpr (kSplits) {
      if (nseg > 1) {
        first = nkeep * seg / nseg;
        nkeep = nkeep * (seg + 1) / nseg - first;
      }
    }
  }
  int nsub = MODE == kModeDenseHead ? 2 * a.tb : 2 * nkeep;  // 64-key sub-tiles
  // Opaque: told that nsub is 2 nkeep, the compiler rewrites the d = 64 walk's loop over both
  // and spills 90 registers in it.
  asm volatile("" : "+s"(nsub));

  // Sub-tile `it` = half (it & 1) of kept tile (it >> 1): its K rows and its V^T half are
  // each HALF contiguous bytes of the packed images, copied verbatim into LDS slot it & 1
  // by buffer loads into LDS (each lane moves 16 bytes; one wave instruction fills 1 KB in
  // lane order) over this bank's images, whose byte size bounds the buffer resource.
  const int bank_bytes = a.tb * G::kTileBytes;
  const __amdgpu_buffer_rsrc_t krs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(early.kp + (int64_t)bank * a.tb * G::kTileElems), 0, bank_bytes, kBufferRsrcWord3);
  const __amdgpu_buffer_rsrc_t vrs = __builtin_amdgcn_make_buffer_rsrc(
      (void*)(early.vp + (int64_t)bank * a.tb * G::kTileElems), 0, bank_bytes, kBufferRsrcWord3);
  auto image = [&](int it) {  // byte offset of sub-tile `it` within the bank's images
    const int j = MODE == kModeDense ? (it >> 1) : list[first + (it >> 1)];
    return __builtin_amdgcn_readfirstlane(j * G::kTileBytes + (it & 1) * HALF);
  };
  auto copy = [&](__amdgpu_buffer_rsrc_t rs, int off, char* dst) {
#pragma unroll
    for (int i = 0; i < NDMA; ++i)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          rs, (lds_void*)(dst + 16 * kThreads * i + 1024 * wave), 16,
          16 * kThreads * i + 16 * t, off, 0, 0);
  };

  const float inv_scale_log2 = 1.0f / a.scale_log2;
  const bool ragged = (a.n_tokens % kBlock) != 0;

  // S^T (64 keys x 32 queries of each group) of the sub-tile whose K image is in `kl`, by the lane's
  // row and half (l32 and g; captured, they had the compiler compute eight of the main walk's LDS
  // addresses anew in every pair of steps, 1% at 24 heads x 119,056 tokens).
  auto qk = [&](const char* kl, f32x16 (&s)[kGroups][2], int lr, int lg) {
#pragma unroll
    for (int st = 0; st < NS; ++st)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt) {
        const u32x4 ka = lds_load16(kl, G::k_off(32 * kt + lr, 2 * st + lg));
#pragma unroll
        for (int q = 0; q < kGroups; ++q)
          s[q][kt] = T::mfma32(ka, qreg[q][st], st == 0 ? f32x16{} : s[q][kt]);
      }
  };
  // Keys past the sequence end in a sub-tile of the last (ragged) block.
  auto mask_tail = [&](f32x16 (&s)[kGroups][2], int it) {
    int limit = a.n_tokens - ((a.tb - 1) * kBlock + 64 * (it & 1)) - 4 * g;
    asm volatile("" : "+v"(limit));  // keeps the compares in this rare branch
#pragma unroll
    for (int q = 0; q < kGroups; ++q)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) {
          // At d = 64 also one at a time: 32 masks at once took the scalar registers that the walk
          // keeps its copies' LDS addresses in (0.8% at 48 heads x 45,106 tokens; at d = 128 the
          // walk is scheduled better with them at once, 0.5% at 24 x 119,056).
          if constexpr (D == 64) asm volatile("" : "+v"(limit));
          if (32 * kt + mfma_row(rr, 0) >= limit) s[q][kt][rr] = -INFINITY;
        }
  };
  auto lane_max = [](f32x16 (&s)[2]) {
    float mx = -INFINITY;
#pragma unroll
    for (int kt = 0; kt < 2; ++kt)
#pragma unroll
      for (int rr = 0; rr < 16; ++rr) mx = __builtin_elementwise_maximum(mx, s[kt][rr]);
    return mx;
  };
  float m[kGroups], mraw[kGroups], lsum[kGroups];
  f32x16 oacc[kGroups][NDT];
#pragma unroll
  for (int q = 0; q < kGroups; ++q) {
    m[q] = -INFINITY;
    mraw[q] = -INFINITY;
    lsum[q] = 0.0f;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt) oacc[q][dt] = f32x16{};
  }
  // Lazy running-max update of group q from a per-lane candidate raw score: moves only when
  // the row max grows by more than kRescaleSlack, rescaling O and l.  The test is on raw
  // scores against mraw = (m + slack) / (scale log2 e), kept with m (scale > 0).
  auto update_max = [&](int q, float mx) {
    const float pm = pair_max(mx);
    const bool grow = pm > mraw[q];
    if (__any(grow)) {
      const float mnew = grow ? pm * a.scale_log2 : m[q];
      const float alpha = __builtin_amdgcn_exp2f(m[q] - mnew);
      lsum[q] *= alpha;
#pragma unroll
      for (int dt = 0; dt < NDT; ++dt) oacc[q][dt] *= alpha;
      m[q] = mnew;
      mraw[q] = (mnew + kRescaleSlack) * inv_scale_log2;
    }
  };

  // Dense-head mode: the head branch of the kept blocks (the list's first 2 * nkeep
  // sub-tiles), stored from the running state once their last PV is done and before the
  // next sub-tile's scores may raise the running max -- the state head mode ends with.
  const int kept_end = 2 * nkeep;
  auto store_head = [&]() __attribute__((always_inline)) {
    if constexpr (MODE == kModeDenseHead) {
#pragma unroll
      for (int q = 0; q < kGroups; ++q) {
        const float lt = pair_sum(lsum[q]);
        if (valid[q])
          store_rows<T, D, kModeHead>(a, bank, b, h, row[q], nat[q], g, oacc[q], m[q], lt);
      }
    }
  };

  // One pipeline step, written as slices that the scheduler may not reorder: slice n reads
  // one LDS fragment (of slice n+2) and issues one MFMA per query group with the fragment
  // of slice n -- first the 2*NS of S_{it+1} (head-dimension chunk n/2, key tile n%2),
  // then the 4*NDT of PV_it (P chunk (kt, hh), O^T tile dt) -- plus a fixed share of VALU
  // work: while S_{it+1} runs, pairs of P_it = exp2(S_it scale log2e - m) values (two exp,
  // packed for the PV MFMAs); while PV_it runs, the row max over pairs of S_{it+1} scores.
  // The matrix core then works while the VALU does, instead of one after the other.
  // `it` is even at every call with parity tag 0 and odd with tag 1.
  auto step = [&](int it, f32x16 (&cur)[kGroups][2], f32x16 (&nxt)[kGroups][2], bool mask,
                  auto next_tag, auto parity_tag) __attribute__((always_inline)) {
    constexpr bool kNext = decltype(next_tag)::value;
    constexpr bool kOdd = decltype(parity_tag)::value;
    if (it + 1 < nsub) copy(vrs, image(it + 1), kOdd ? v_lds0 : v_lds1);
    if (it + 2 < nsub) copy(krs, image(it + 2), kOdd ? k_lds1 : k_lds0);
    const char* kl = kOdd ? k_lds0 : k_lds1;   // K_{it+1}
    const char* vl = kOdd ? v_lds1 : v_lds0;   // V_it
    constexpr int NQK = kNext ? 2 * NS : 0;  // S fragments of this step
    constexpr int NPV = 4 * NDT;             // PV fragments
    constexpr int NN = NQK + NPV;
    constexpr int NPAIR = 16 * kGroups;      // P pairs (16 per group)
    constexpr int PPS = kNext ? (NPAIR + NQK - 1) / (kNext ? NQK : 1) : NPAIR;  // P pairs per slice
    constexpr int MPS = 16 * kGroups / NPV;  // score pairs of the row max per PV slice
    auto frag = [&](int n) -> u32x4 {
      if (n < NQK) return lds_load16(kl, G::k_off(32 * (n & 1) + l32, 2 * (n >> 1) + g));
      const int i = n - NQK;
      return lds_load16(vl, G::vt_off(32 * (i % NDT) + l32, 2 * (i / NDT) + g));
    };
    unsigned w[kGroups][2][2][4];
    float part[kGroups][2];
    float mx[kGroups];
#pragma unroll
    for (int q = 0; q < kGroups; ++q) mx[q] = -INFINITY;
    u32x4 fr[3];
    fr[0] = frag(0);
    fr[1] = frag(1);
#pragma unroll
    for (int n = 0; n < NN; ++n) {
      if (n + 2 < NN) fr[(n + 2) % 3] = frag(n + 2);
      // P pairs first (the PV MFMAs need them); pair pr is pair pr / kGroups of group
      // pr % kGroups, so every group's chunk (kt, hh) is complete by the same slice.
      if (n * PPS < NPAIR) {
#pragma unroll
        for (int pr = n * PPS; pr < n * PPS + PPS && pr < NPAIR; ++pr) {
          const int q = pr % kGroups, pp = pr / kGroups;
          const int kt = pp >> 3, hh = (pp >> 2) & 1, e = 2 * (pp & 3);
          const float p0 = __builtin_amdgcn_exp2f(fmaf(cur[q][kt][8 * hh + e], a.scale_log2, -m[q]));
          const float p1 = __builtin_amdgcn_exp2f(fmaf(cur[q][kt][8 * hh + e + 1], a.scale_log2, -m[q]));
          part[q][kt] = (pp & 7) ? part[q][kt] + (p0 + p1) : p0 + p1;
          w[q][kt][hh][e >> 1] = pack2<T>(p0, p1);
        }
      }
      if (n < NQK) {
        const int st = n >> 1, kt = n & 1;
#pragma unroll
        for (int q = 0; q < kGroups; ++q)
          nxt[q][kt] = T::mfma32(fr[n % 3], qreg[q][st], st == 0 ? f32x16{} : nxt[q][kt]);
        // S_{it+1} in the ragged last block: keys past the sequence end get -inf before the
        // row max reads them (a rare uniform branch, outside the scheduled slices).
        if (n == NQK - 1 && mask) {
          __builtin_amdgcn_sched_barrier(0);
          mask_tail(nxt, it + 1);
        }
      } else {
        const int i = n - NQK, kt = i / (2 * NDT), hh = (i / NDT) & 1, dt = i % NDT;
#pragma unroll
        for (int q = 0; q < kGroups; ++q) {
          const u32x4 pk = {w[q][kt][hh][0], w[q][kt][hh][1], w[q][kt][hh][2], w[q][kt][hh][3]};
          oacc[q][dt] = T::mfma32(fr[n % 3], pk, oacc[q][dt]);
        }
        if constexpr (kNext) {
          // Row max over MPS pairs of S_{it+1} scores (pair mp: group mp % kGroups).
#pragma unroll
          for (int mp = i * MPS; mp < (i + 1) * MPS; ++mp) {
            const int q = mp % kGroups, j = 2 * (mp / kGroups), kt2 = j >> 4, rr = j & 15;
            mx[q] = fmaxf(fmaxf(mx[q], nxt[q][kt2][rr]), nxt[q][kt2][rr + 1]);  // one v_max3_f32
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int q = 0; q < kGroups; ++q) lsum[q] += part[q][0] + part[q][1];
    if constexpr (MODE == kModeDenseHead) {
      if (it + 1 == kept_end) store_head();
    }
    if constexpr (kNext) {
#pragma unroll
      for (int q = 0; q < kGroups; ++q) update_max(q, mx[q]);
    }
    tile_barrier();
  };

  // True when sub-tile `it` of the list lies in the ragged last block.
  auto ragged_at = [&](int it) {
    const int j = MODE == kModeDense ? (it >> 1) : __builtin_amdgcn_readfirstlane(list[first + (it >> 1)]);
    return ragged && j == a.tb - 1;
  };
  // The d = 64 step.  Its softmax work exceeds its matrix work, so the two are pipelined one
  // sub-tile further apart than above: step `it` computes P_it on the VALU while the matrix core
  // runs S_{it+1} and PV_{it-1}, which do not depend on it, alternately.  Slice n issues one
  // MFMA (with the LDS fragment read four slices before) and its share of the P pairs.  The
  // running max is checked and raised at the end of the step, when O holds the sub-tiles before
  // `it`.  (With P and PV of one sub-tile in one step, as above, the PV half of a step had no
  // VALU work and waited for each fragment.  A refresh at 48 heads x 24,706 tokens 19.66 -> 19.38
  // ms, a sparse call at 2 x 4,096 47.8 -> 46.4 us, and no change at 48 x 45,106, where power
  // bounds both forms; the same bits.)
  // `vt` and `kt_next` are the key tiles of sub-tiles it and it + 2.
  auto step64 = [&](int it, int vt, int kt_next, f32x16 (&cur)[kGroups][2],
                    f32x16 (&nxt)[kGroups][2], u32x4 (&w)[4], u32x4 (&wp)[4],
                    bool mask, auto next_tag, auto pv_tag, auto parity_tag) __attribute__((always_inline)) {
    static_assert(kGroups == 1, "one query group per wave");
    constexpr bool kNext = decltype(next_tag)::value;
    constexpr bool kPV = decltype(pv_tag)::value;
    constexpr bool kOdd = decltype(parity_tag)::value;
    constexpr int half = kOdd ? HALF : 0;
    copy(vrs, vt * G::kTileBytes + half, kOdd ? v_lds1 : v_lds0);   // V_it, read in the next step
    if (it + 2 < nsub) copy(krs, kt_next * G::kTileBytes + half, kOdd ? k_lds1 : k_lds0);
    const char* kl = kOdd ? k_lds0 : k_lds1;   // K_{it+1}
    const char* vl = kOdd ? v_lds0 : v_lds1;   // V_{it-1}
    constexpr int NQK = 2 * NS, NPV = 4 * NDT;
    constexpr int NN = (kNext ? NQK : 0) + (kPV ? NPV : 0);
    // MFMA n: alternately S and PV where there are both.
    auto is_qk = [](int n) { return kNext && (!kPV || n % 2 == 0); };
    auto frag = [&](int n) -> u32x4 {
      const int i = kNext && kPV ? n / 2 : n;
      if (is_qk(n)) return lds_load16(kl, G::k_off(32 * (i & 1) + l32, 2 * (i >> 1) + g));
      return lds_load16(vl, G::vt_off(32 * (i % NDT) + l32, 2 * (i / NDT) + g));
    };
    constexpr int kAhead = 4;
    u32x4 fr[kAhead + 1];
#pragma unroll
    for (int n = 0; n < kAhead; ++n) fr[n] = frag(n);
    float part[2];
    auto pair = [&](int pp) {
      const int kt = pp >> 3, hh = (pp >> 2) & 1, e = 2 * (pp & 3);
      const float p0 = __builtin_amdgcn_exp2f(fmaf(cur[0][kt][8 * hh + e], a.scale_log2, -m[0]));
      const float p1 = __builtin_amdgcn_exp2f(fmaf(cur[0][kt][8 * hh + e + 1], a.scale_log2, -m[0]));
      part[kt] = (pp & 7) ? part[kt] + (p0 + p1) : p0 + p1;
      w[2 * kt + hh][e >> 1] = pack2<T>(p0, p1);
    };
    constexpr int PPS = 16 / NN;  // P pairs per slice
#pragma unroll
    for (int n = 0; n < NN; ++n) {
      if (n + kAhead < NN) fr[(n + kAhead) % (kAhead + 1)] = frag(n + kAhead);
      const u32x4 f = fr[n % (kAhead + 1)];
      const int i = kNext && kPV ? n / 2 : n;
      if (is_qk(n)) {
        const int st = i >> 1, kt = i & 1;
        nxt[0][kt] = T::mfma32(f, qreg[0][st], st == 0 ? f32x16{} : nxt[0][kt]);
      } else {
        oacc[0][i % NDT] = T::mfma32(f, wp[i / NDT], oacc[0][i % NDT]);
      }
#pragma unroll
      for (int pp = n * PPS; pp < (n + 1) * PPS; ++pp) {
        pair(pp);
        // Packed and summed here, not after the branches below (which would keep every P alive).
        if ((pp & 3) == 3) asm volatile("" : "+v"(w[pp >> 2]), "+v"(part[pp >> 3]));
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if (mask) {  // S_{it+1} in the ragged last block (a rare uniform branch)
      mask_tail(nxt, it + 1);
    }
    if constexpr (MODE == kModeDenseHead) {
      if (it == kept_end) store_head();
    }
    // A lane whose probabilities overflow the cap (or are not finite, as when m = -inf) redoes
    // the sub-tile against the raised running max, rescaling O and l first.
    if (__any(!(part[0] + part[1] <= kSumCap))) {
      float mx = -INFINITY;
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int rr = 0; rr < 16; ++rr) mx = __builtin_elementwise_maximum(mx, cur[0][kt][rr]);
      const float mnew = pair_max(mx) * a.scale_log2;
      if (mnew > m[0]) {
        const float alpha = __builtin_amdgcn_exp2f(m[0] - mnew);
        lsum[0] *= alpha;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) oacc[0][dt] *= alpha;
        m[0] = mnew;
      }
#pragma unroll
      for (int pp = 0; pp < 16; ++pp) pair(pp);
    }
    lsum[0] += part[0] + part[1];
    tile_barrier();
  };

  f32x16 sa[kGroups][2], sb[kGroups][2];
  // The walk's first scores and running max.  Every segment of a long row starts from the max that
  // the undivided walk has after its first sub-tile: a later segment takes the scores of that one
  // (pass 0) before those of its own (pass 1).  The probabilities, which are rounded to 16 bits
  // relative to the max, are then the undivided walk's (but where a segment's scores make it raise
  // the max again), and only the order of the fp32 sums is another.  From a max of their own, 9-34%
  // of the long rows' elements came out as the neighbouring value (12 heads x 7,800 tokens; 12 x
  // 4,856 in fp16), now 0.8-7%, in the same time.
#pragma unroll 1
  for (int pass = kSplits && first > 0 ? 0 : 1; pass < 2 && nsub > 0; ++pass) {
    const int j = MODE == kModeDense ? 0 : __builtin_amdgcn_readfirstlane(list[pass == 0 ? 0 : first]);
    copy(krs, j * G::kTileBytes, k_lds0);
    if (pass == 1) {
      if constexpr (D != 64) copy(vrs, image(0), v_lds0);   // (at d = 64 its step copies it)
      if (nsub > 1) copy(krs, image(1), k_lds1);
    }
    tile_barrier();
    qk(k_lds0, sa, l32, g);
    if (ragged && j == a.tb - 1) mask_tail(sa, 0);
#pragma unroll
    for (int q = 0; q < kGroups; ++q) {
      const float pm = pair_max(lane_max(sa[q]));
      if (pm > mraw[q] && (D != 64 || m[q] == -INFINITY)) {
        m[q] = pm * a.scale_log2;
        if constexpr (D != 64) mraw[q] = (m[q] + kRescaleSlack) * inv_scale_log2;
      }
    }
    tile_barrier();  // K slot 0 is copied over next
  }
  using F = std::false_type;
  using Tr = std::true_type;
  if (MODE == kModeDenseHead && kept_end == 0) store_head();
  if constexpr (D == 64) {
    // Steps 0 .. nsub - 1 (nsub is even) and PV of the last sub-tile.  Steps 2 i and 2 i + 1 copy
    // V of walk tile i and K of tile i + 1; each list entry is read a pair of steps early.  A
    // ragged block's sub-tiles are the first two (kept, in the masked modes) or the last two.
    if (nsub >= 2) {
      const int ntile = nsub >> 1;
      auto tile = [&](int i) {
        const int j = min(i, ntile - 1);
        return MODE == kModeDense ? j : __builtin_amdgcn_readfirstlane(list[first + j]);
      };
      u32x4 wa[4], wb[4];
      int j0 = tile(0), j1 = tile(1);
      const bool tail = nsub >= 4 && ragged_at(nsub - 1);
      step64(0, j0, j1, sa, sb, wa, wb, ragged_at(1), Tr{}, F{}, F{});
      for (int it = 1; it + 2 < nsub; it += 2) {
        const int j2 = tile((it + 3) >> 1);
        const bool mask = tail && it + 3 == nsub;
        step64(it, j0, j1, sb, sa, wb, wa, mask, Tr{}, Tr{}, Tr{});
        step64(it + 1, j1, j2, sa, sb, wa, wb, mask, Tr{}, Tr{}, F{});
        j0 = j1;
        j1 = j2;
      }
      step64(nsub - 1, j0, j1, sb, sa, wb, wa, false, F{}, Tr{}, Tr{});
#pragma unroll
      for (int i = 0; i < 4 * NDT; ++i) {
        const u32x4 f = lds_load16(v_lds1, G::vt_off(32 * (i % NDT) + l32, 2 * (i / NDT) + g));
        oacc[0][i % NDT] = T::mfma32(f, wb[i / NDT], oacc[0][i % NDT]);
      }
      if (MODE == kModeDenseHead && kept_end == nsub) store_head();
    }
  } else {
  // Steps go in pairs (even step: S in sa -> sb, odd step: sb -> sa) so each array keeps one
  // role.  Step it computes S of sub-tile it + 1, masked when that sub-tile lies in the ragged
  // last block: in the masked modes a kept ragged block goes first (sub-tiles 0 and 1), and in
  // dense mode, or in dense-head mode when the mask drops it, the ragged block goes last, so
  // only the first and the last two pairs are peeled and the main loop runs unmasked.  The
  // final step has no next sub-tile.
  int it = 0;
  if constexpr (MODE != kModeDense) {
    if (nsub >= 4) {
      step(0, sa, sb, ragged_at(1), Tr{}, F{});
      step(1, sb, sa, ragged_at(2), Tr{}, Tr{});
      it = 2;
    }
  }
  for (; it + 4 < nsub; it += 2) {
    step(it, sa, sb, false, Tr{}, F{});
    step(it + 1, sb, sa, false, Tr{}, Tr{});
  }
  if (nsub - it >= 4) {
    step(it, sa, sb, false, Tr{}, F{});
    step(it + 1, sb, sa, ragged_at(it + 2), Tr{}, Tr{});
    it += 2;
  }
  if (nsub >= 2) {
    step(it, sa, sb, ragged_at(it + 1), Tr{}, F{});
    step(it + 1, sb, sa, false, F{}, Tr{});
  }
  }

  constexpr int kStore = MODE == kModeDenseHead ? kModeDense : MODE;
  const AttnArgs& late = reread();
  bool stores = true;
  float lt[kGroups];
#pragma unroll
  for (int q = 0; q < kGroups; ++q)
    lt[q] = pair_sum(lsum[q]);  // lanes l and l ^ 32 share one row: both valid or not
  if constexpr (kSplits) {
    if (nseg > 1) stores = merge_segments<D>(late, bank * nlong + (qt - a.ds), seg, nseg, &claimed, oacc[0], m[0], lt[0]);
  }
  int lane_row = l32;
  asm volatile("" : "+v"(lane_row));  // the row numbers are computed again, not kept
#pragma unroll
  for (int q = 0; q < kGroups; ++q) {
    const int r = qt * kBlock + wave * kRowsPerWave + 32 * q + lane_row;
    if (r < a.n_tokens && stores)
      store_rows<T, D, kStore>(late, bank, b, h, r, nat[q], g, oacc[q], m[q], lt[q]);
  }
  __syncthreads();  // every wave is done with the LDS slots, the list and `claimed`
  }  // items
}

// Segments of each long row (query blocks ds .. tb-1, dense) of a masked launch whose other
// rows keep about `density` of their blocks.  A long row as one item takes its tb tiles
// however idle the chip is, so it is cut until a segment is no longer than the other items, or
// than half of the work there is for each of the 512 workgroups, and not below 16 tiles (a
// segment's state costs about two tiles to store and combine); and where two segments a row fit
// one round of the 512, not so far that the items need a second.  (Two segments stay also where
// the undivided rows alone fit it: 102 us undivided, 71 with two and 70 with the rule's three at
// 12 banks of 42 blocks, 504, 516 and 528 items.)  Attention kernel, 1 segment -> this rule: 101 ->
// 73 us at 12 banks of 38 blocks (2 segments; 3: 80, 6: 73), 203 -> 178 us at 12 of 61 (3; 6:
// 199), 333 -> 275 us at 8 of 125 (4; 6: 276); no change at 12 of 256 (2).  It depends on the
// layer's sizes only, so that every group of its heads is cut alike.
int attn_split(int64_t banks, int64_t tb, int64_t ds, double density) {
  if (ds >= tb) return 1;
  const double longs = (double)(tb - ds), other = density * (double)tb + longs + 1.0;
  const double share = (double)banks * ((double)ds * other + longs * (double)tb) / 512.0;
  const double segment = std::max(16.0, std::max(other, 0.5 * share));
  int split = (int)std::min<double>(kMaxSplit, std::max(1.0, std::ceil((double)tb / segment)));
  while (split > 2 && banks * (ds + (tb - ds) * split) > 512 && banks * (ds + (tb - ds) * 2) <= 512)
    --split;
  return split;
}

// Workgroups of a persistent launch: two per CU (the attention kernel's occupancy), no
// more than there are items.
static int persistent_grid(int items) {
  int device = 0, cus = 0;
  if (hipGetDevice(&device) != hipSuccess ||
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, device) != hipSuccess ||
      cus < 1)
    cus = 256;
  return items < 2 * cus ? items : 2 * cus;
}

template <class T, int D>
static hipError_t launch_attention(const AttnArgs& a, int mode, hipStream_t s) {
  const bool splits = mode == kModeHead || mode == kModeMerge;
  const int items = a.banks * (a.ds + (a.tb - a.ds) * (splits ? a.split : 1));
  const dim3 grid((unsigned)(a.queue != nullptr ? persistent_grid(items) : items)), block(kThreads);
  switch (mode) {
    case kModeHead: hipLaunchKernelGGL((attention_kernel<T, D, kModeHead>), grid, block, 0, s, a); break;
    case kModeDense: hipLaunchKernelGGL((attention_kernel<T, D, kModeDense>), grid, block, 0, s, a); break;
    case kModeDenseHead: hipLaunchKernelGGL((attention_kernel<T, D, kModeDenseHead>), grid, block, 0, s, a); break;
    default: hipLaunchKernelGGL((attention_kernel<T, D, kModeMerge>), grid, block, 0, s, a); break;
  }
  return hipGetLastError();
}

__global__ __launch_bounds__(256) void zero_words_kernel(unsigned* p, int n) {
  for (int i = threadIdx.x; i < n; i += 256) p[i] = 0u;
}

hipError_t run_zero_words(unsigned* p, int n, hipStream_t s) {
  hipLaunchKernelGGL(zero_words_kernel, dim3(1), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t run_attention(const AttnArgs& a, int dtype, int dim, int mode, hipStream_t s) {
  if (dtype == BF16::code)
    return dim == 128 ? launch_attention<BF16, 128>(a, mode, s) : launch_attention<BF16, 64>(a, mode, s);
  return dim == 128 ? launch_attention<F16, 128>(a, mode, s) : launch_attention<F16, 64>(a, mode, s);
}

}  // namespace recap
