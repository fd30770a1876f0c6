// Chunked prefill with LDS-staged KV tiles (head_dim 128 or 64): part of pkv_attention.hip.
//
// Grid (row block, KV head, sequence).  A workgroup of 4 waves owns 128 consecutive query rows (row
// = j * g + head-in-group, so a block spans a few query positions of every head of the group), 32
// per wave, and walks the tiles of its KV head up to its last row's last visible key.
//
// One wave's tile is 32 query rows x 32 tokens per v_mfma_f32_32x32x16_bf16 chain:
//   S^T[tok, row] = K[tok, :] . Q[row, :]       A = K rows (lane: token l % 32, 8 elements at 8 (l / 32))
//                                               B = Q, in registers for the whole call
//   O^T[d, row] += V^T[d, tok] . P^T[tok, row]  A = V^T by LDS transpose reads, B = the S^T accumulator
// Lane (n = l % 32, hi = l / 32) holds, of S^T, row n's scores of tokens 8 (r / 4) + 4 hi + r % 4 (r <
// 16): a row's statistics live in two lanes, and registers 8 s .. 8 s + 7 packed to bf16 are the PV
// operand of key step s as they stand, provided V^T names its tokens in the same order.
//
// Each stage's K and V rows are copied into LDS once per workgroup (8 buffer loads of 1 KiB each,
// two of K and two of V per wave), through a ring of 4 slots of K and one of 4 of V (3 each in the
// two-wave form), with counted vmcnt waits and one raw barrier per stage.
//
// What bounds it: the matrix pipe at 33 cycles per 32x32x16 product (16 products per stage and wave)
// beside 79 other vector instructions and 24 LDS reads.  The pipe is busy 46% of a launch of 1280
// workgroups; a wave issues 47% of its time, waits for a pipe 34% (the other wave of its SIMD has it)
// and at the barrier and copies 19%.  Power is not the limit yet: a register-only loop of these products
// on random data holds 1.53 GHz on 256 CUs, the launch runs at about 1.95.  A wave issues in order, about
// one instruction per 4.4 cycles, so its iteration over stage t mixes three stages to keep both pipes
// fed, in straight-line code (a taken branch costs 50-100 cycles of instruction fetch; rare work sits out
// of line):
//   phase A: S^T products of stage t + 1, with the first half of stage t's exponentials between them,
//            while stage t - 1's V operands arrive from LDS;
//   phase B: PV products of stage t - 1, with the second half and the next stage's score maxima between
//            them, while stage t + 2's K operands arrive.  Phase B runs at raised priority, which
//            drifts the two waves of a SIMD into opposite phases (4096-token 7B prompt 154 -> 148 us).
// The copies of a stage go out one at a time through both phases (all in phase A: 146 -> 139 us).
// Per call: head_dim 64, 4 prompts of 1000 tokens, 93 -> 35 us (it replaces per-wave tiles held in
// registers); head_dim 128, one 4096-token 7B prompt 136 -> 131 us, 8 x 512 14B chunks onto
// prefixes U{0..4096} 169 -> 160 us, 150 tokens onto 3500 (36 workgroups) 104 -> 70 us.  Captured prompts
// of one to three stages take 0.1 to 0.6 us more than with 16x16x32 products.
namespace pf {

template <int HD_>
struct Geo {
  static_assert(HD_ == 64 || HD_ == 128, "head_dim 64 or 128");
  static constexpr int HD = HD_;
  static constexpr int TT = 128 / HD;           // 32-token sub-tiles per stage
  static constexpr int TOK = 32 * TT;           // tokens per stage
  static constexpr int DT = HD / 32;            // 32-element output tiles
  static constexpr int KK = HD / 16;            // key steps of the S^T product
  static constexpr int ROWB = HD * 2;           // bytes of one head's slice of a token row
  static constexpr int CPR = HD / 8;            // 16-byte chunks of it
  static constexpr int RPC = 64 / CPR;          // rows per 1 KiB copy
  static constexpr int STAGE = TOK * ROWB;      // 8 KiB of K (or V) per stage
  static_assert(STAGE == 8192 && TT * KK == 8 && TT * 2 * DT == 8, "8 copies, 8 + 8 products per stage");
  // 16-byte chunk swizzles of a K and of a V row.  K: 16 rows read at one chunk cover all 64 banks.
  // V: the 4 token rows x 64 bytes of a half wave's transpose read do.
  static __device__ __forceinline__ int swz_k(int r) { return HD == 128 ? (r & 15) : ((r >> 1) & 7); }
  static __device__ __forceinline__ int swz_v(int r) { return HD == 128 ? ((r & 3) << 2) : (((r >> 1) & 1) << 2); }
};

constexpr int kWaves = 4;
constexpr int kRows = 32 * kWaves;   // query rows per workgroup
// Verify's workgroups: two waves, 64 query rows.  Their copies run one stage less ahead, so that three
// workgroups' rings fit a CU's LDS.
constexpr int kVerifyWaves = 2;
constexpr int kVerifyRows = 32 * kVerifyWaves;
constexpr int kVerifyPerCu = 3;

// At most N of this wave's copies may stay in flight (LGKM: and none of its LDS reads).
template <int N, bool LGKM = false>
__device__ __forceinline__ void wait_vm() {
  static_assert(N < 64, "vmcnt immediate");
  __builtin_amdgcn_s_waitcnt((LGKM ? 0x0070 : 0x0F70) | (N & 15) | ((N >> 4) << 14));
}

// The larger of the lane's scores (never NaN unless the inputs are, and then the row is NaN anyway).
__device__ __forceinline__ float max2(float a, float b) { return __builtin_elementwise_maximum(a, b); }

// What a workgroup's result becomes.
enum Dest {
  kDirect,   // the bf16 output rows
  kCascade,  // the shared-prefix pass of a cascade launch: fp16 O / l and the log-sum-exp of one key split
  kSplit,    // one of max_splits key ranges: fp32 O and (m, l) for prefill_merge_kernel
};

// Key ranges.  A call with few row blocks (150 tokens onto 3500 at the 7B shape: 36 items of 115 stages)
// leaves most CUs idle at 0.5 us per stage; cut into ranges it takes 28 us a call instead of 68, the merge
// launch included.  The partials stay fp32.
// Key ranges of an item of n stages in a kSplit launch: `chunk` stages each, at least kMinStages (a
// range pays about two stages' time to start and one to end, and a partial of 66 KB: 3 ranges of 8 are
// as fast as 6 of 4 at 24 items and faster from 44 on).  One range writes its rows directly.
constexpr int kMinStages = 8;
constexpr int kMinVerifyStages = 5;
constexpr int kDeepStages = 12;  // two workgroups per CU from this many stages a range on
struct Ranges {
  int chunk, count;
};
__device__ __forceinline__ Ranges ranges_of(const AttnParams& p, int n) {
  Ranges r;
  r.chunk = max((n + p.max_splits - 1) / p.max_splits, kMinStages);
  r.count = n > 0 ? (n + r.chunk - 1) / r.chunk : 1;
  return r;
}

// Stages that rows up to blk_last of a sequence of L keys see.
template <int TOK>
__device__ __forceinline__ int stages_of(const AttnParams& p, int L, int blk_last) {
  const int t_stop = p.causal ? min(L, L - p.s_q + blk_last / p.g + 1) : L;
  return t_stop > 0 ? (t_stop + TOK - 1) / TOK : 0;
}

__device__ __forceinline__ u32x4 lds_read16(uint32_t addr) {
  return *reinterpret_cast<const __attribute__((address_space(3))) u32x4*>(uintptr_t(addr));
}

// 1 KiB straight into LDS: lane l's 16 bytes from byte voff (per lane) + soff of the buffer of `bytes`
// at `base` (uniform) to dst + 16 l.
__device__ __forceinline__ void copy_1k(const uint16_t* base, int bytes, uint32_t voff, int soff, char* dst) {
  const __amdgpu_buffer_rsrc_t rs =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(uniform_ptr(base)), 0, bytes, 0x00020000);
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rs, (rows::lds_void*)dst, 16, int(voff), soff, 0, 0);
}

// acc plus the two bf16 values of a pair.
__device__ __forceinline__ float add_pair(uint32_t pair, float acc) {
  const bf16x2 ones = {static_cast<__bf16>(1.f), static_cast<__bf16>(1.f)};
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), ones, acc, false);
}

// Two probabilities as bf16 pairs hi + lo: hi truncated, so that lo is not negative, and lo a 2^-23 of p
// too large, so that it is not zero either where p is not: an infinite V stays that infinity under both.
__device__ __forceinline__ uint32_t split_pair(float a, float b, uint32_t& hi) {
  const uint32_t ua = __float_as_uint(a), ub = __float_as_uint(b);
  constexpr float kUp = 1.f + 0x1p-23f;
  hi = __builtin_amdgcn_perm(ub, ua, 0x07060302u);
  return pack_bf16x2(fmaf(a, kUp, -__uint_as_float(ua & 0xFFFF0000u)), fmaf(b, kUp, -__uint_as_float(ub & 0xFFFF0000u)));
}

// Over the two lanes {l, l ^ 32} that hold a row.
__device__ __forceinline__ float sum_halves(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}
__device__ __forceinline__ float max_halves(float v) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return max_raw(__uint_as_float(a[0]), __uint_as_float(a[1]));
}

// Keeps values where they are computed: the first use of a phase's exponentials is an iteration
// away, and the compiler would sink them past the products they are to hide behind.
__device__ __forceinline__ void pin(float& v) { asm volatile("" : "+v"(v)); }
__device__ __forceinline__ void pin(uint32_t& v) { asm volatile("" : "+v"(v)); }

// Verify's ranges.  The stages of all sequences, sequence after sequence, are cut into ranges of one
// length (`chunk`: about lean_grid ranges for each KV head, at least kMinVerifyStages stages each: 4 to 6
// are level), each inside
// one sequence: a ragged batch keeps every workgroup at the same work, whatever the longest sequence.
// Range w of KV head h is workgroup w n_kv + h, so that each XCD's L2 serves few heads (a cached prefix
// that the batch shares is then read once per XCD and head).
constexpr int kVerifyBatch = 64;  // one sequence per lane
struct VerifyPlan {
  int n;  // stages of sequence `lane` (0 past the batch)
  int chunk;
};
template <int TOK>
__device__ __forceinline__ VerifyPlan verify_plan(const AttnParams& p) {
  const int lane = threadIdx.x & 63;
  const int cap = p.max_blocks << p.log2_page;
  VerifyPlan v;
  v.n = 0;
  if (lane < p.batch) {
    const int c = min(max(p.seqlens[lane], 0), cap);  // as seq_lengths clamps it
    v.n = max(stages_of<TOK>(p, min(c + (p.has_new ? p.s_q : 0), cap), p.R - 1), 1);
  }
  const int total = __builtin_amdgcn_readlane(wave_incl_scan(v.n), 63);
  v.chunk = max((total + p.lean_grid - 1) / p.lean_grid, kMinVerifyStages);
  // every sequence's last range may be short: lengthen the ranges until they fit one round
  for (int tries = 0; tries < 16; ++tries) {
    const int ranges = __builtin_amdgcn_readlane(wave_incl_scan((v.n + v.chunk - 1) / v.chunk), 63);
    if (ranges <= max(p.lean_grid, p.batch)) break;
    v.chunk += max(v.chunk / 16, 1);
  }
  return v;
}

}  // namespace pf

// CASCADE form (DEST == kCascade): grid (row blocks of the whole batch's query rows, KV heads, key
// splits); block-table row 0 holds the shared pages; split z covers stages [z chunk, (z + 1) chunk)
// of the k0 shared keys, which every row sees whole; the result is a partial (fp16 O / l and fp32
// log-sum-exp) in workspace slot 2 G + b S + z of each row.
//
// W waves own 32 W rows.  W = 2 (kSplit only) is speculative verify: one row block per (sequence, KV
// head); each range appends the new rows it covers itself, before it copies them; P is a bf16 pair (two
// PV products).
template <int HD, int DEST, int W = pf::kWaves>
__global__ __launch_bounds__(64 * W, 2) void prefill_tile_kernel(const AttnParams p) {
  using G = pf::Geo<HD>;
  constexpr int kRows = 32 * W;
  constexpr int kLead = W == pf::kWaves ? 3 : 2;  // iterations between a copy's issue and its use
  static_assert(kLead == 2 || kLead == 3, "V copies start in iteration -2 or -1");
  constexpr int kRing = kLead + 1;                // slots of the K and of the V ring
  constexpr int kCopies = 8 / W;                  // copies of a K (or V) stage per wave
  constexpr int TT = G::TT, DT = G::DT, KK = G::KK, TOK = G::TOK;
  constexpr bool CASCADE = DEST == pf::kCascade;
  constexpr bool PAIR = W != pf::kWaves;          // P as bf16 hi + lo
  constexpr int NP = PAIR ? 4 * TT : 2 * TT;      // PV operands of a stage: hi (then lo) of each key step
  __shared__ __attribute__((aligned(16))) char lds[2 * kRing * G::STAGE];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int ln = lane & 31;
  const int hi = lane >> 5;
  int b, h, xblk;
  int c, L;
  const int R_all = CASCADE ? p.batch * p.R : p.R;  // query rows of the launch's row space
  int t_first = 0;                                  // first stage of this workgroup's key range
  int n;                                            // its stages
  int split = 0, count = 1, chunk = 0;              // kSplit: which range of the item, of how many, stages each
  if constexpr (CASCADE) {
    xblk = blockIdx.x;
    h = blockIdx.y;
    b = 0;
    c = 0;
    L = p.k0;
  } else {
    const int i = int(blockIdx.x + gridDim.x * (blockIdx.y + gridDim.y * blockIdx.z));
    if constexpr (W != pf::kWaves) {
      // found below
    } else if constexpr (DEST == pf::kSplit) {
      // the ranges of an item are consecutive workgroups: with 8 or 16 of them each XCD's L2 serves
      // the same keys for every row block
      split = i % p.max_splits;
      prefill_item(p, i / p.max_splits, int(gridDim.x) / p.max_splits, b, h, xblk);
    } else {
      prefill_item(p, i, int(gridDim.x), b, h, xblk);
    }
    if constexpr (W != pf::kWaves) {
      xblk = 0;
      h = i % p.n_kv;
      const int w = i / p.n_kv;
      const pf::VerifyPlan v = pf::verify_plan<TOK>(p);
      chunk = v.chunk;
      const int ranges = (v.n + chunk - 1) / chunk;
      const int incl = wave_incl_scan(ranges);
      const uint64_t hit = __ballot(incl > w);
      if (!hit) return;  // fewer ranges than the grid allows for
      b = int(__builtin_ctzll(hit));
      count = __builtin_amdgcn_readlane(ranges, b);
      split = w - (__builtin_amdgcn_readlane(incl, b) - count);
      // for the merge: where the sequence's ranges start, and how many they are
      if (h == 0 && split == 0 && threadIdx.x == 0) {
        p.ws_cnt[2 * b] = w;
        p.ws_cnt[2 * b + 1] = count;
      }
    }
    seq_lengths(p, b, c, L);
  }
  b = __builtin_amdgcn_readfirstlane(b);
  h = __builtin_amdgcn_readfirstlane(h);
  xblk = __builtin_amdgcn_readfirstlane(xblk);
  c = __builtin_amdgcn_readfirstlane(c);
  L = __builtin_amdgcn_readfirstlane(L);
  SeqView sv;
  sv.b = b;
  sv.h = h;
  sv.c = c;
  sv.t_end = L;
  sv.bt = p.block_table + int64_t(b) * p.bt_stride;

  const int blk_row0 = xblk * kRows;
  if (blk_row0 >= R_all) return;
  const int row0 = blk_row0 + wave * 32;
  // the block's last row sees the most keys (rows increase with j)
  const int blk_last = min(blk_row0 + kRows, R_all) - 1;
  if constexpr (CASCADE) {
    if (blockIdx.z == 0 && h == 0) cascade_check_sharing(p, blk_row0 / p.R, blk_last / p.R);
    const int n_shared = p.k0 / TOK;
    const int chunk = (n_shared + int(gridDim.z) - 1) / int(gridDim.z);
    t_first = int(blockIdx.z) * chunk;
    n = max(min(chunk, n_shared - t_first), 0);
  } else {
    n = pf::stages_of<TOK>(p, L, blk_last);
    if constexpr (DEST == pf::kSplit) {
      if constexpr (W == pf::kWaves) {
        const pf::Ranges r = pf::ranges_of(p, n);
        if (split >= r.count) return;
        count = r.count;
        chunk = r.chunk;
      }
      t_first = split * chunk;
      n = min(chunk, n - t_first);
    }
  }

  if constexpr (W != pf::kWaves) {
    // the new rows among this range's keys: stored to the cache, then copied from there like any other
    const int a0 = max(c, t_first * TOK), a1 = min(L, (t_first + n) * TOK);
    if (p.has_new && a0 < a1) {
      append_rows<HD>(p, sv, a0, a1, int(threadIdx.x), 64 * W);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): acknowledged, also of the other wave after the barrier
      raw_barrier();
    }
  }

  // Q rows (key step kk: elements 16 kk + 8 hi .. + 7 of row row0 + ln) and the row's last visible key
  bf16x8 qf[KK];
  int lim = kNoQueryRow;
  // row (and its sequence) of lane index l: real rows, sequence, row in it, query position, query head
  struct LaneRow {
    bool real;
    int b, r, j, hq;
  };
  auto lane_row = [&](int l) {
    const int row = row0 + (l & 31);
    LaneRow x;
    x.real = row < R_all;
    x.b = CASCADE ? row / p.R : b;
    x.r = CASCADE ? row - x.b * p.R : row;
    x.j = x.r / p.g;
    x.hq = h * p.g + x.r - x.j * p.g;
    return x;
  };
  const LaneRow lr = lane_row(lane);
  if (lr.real) {
    const uint16_t* src = p.q + lr.b * p.q_sb + lr.j * p.q_ss + lr.hq * p.q_sh + 8 * hi;
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = __builtin_bit_cast(bf16x8, ld16(src + 16 * kk));
    lim = CASCADE ? p.k0 - 1 : min(p.causal ? L - p.s_q + lr.j : L - 1, L - 1);
  } else {
#pragma unroll
    for (int kk = 0; kk < KK; ++kk) qf[kk] = __builtin_bit_cast(bf16x8, u32x4{0u, 0u, 0u, 0u});
  }
  int lim_min = min_real_limit(0x7fffffff, lim);
#pragma unroll
  for (int off = 1; off < 32; off <<= 1) lim_min = min(lim_min, __shfl_xor(lim_min, off, 64));
  lim_min = __builtin_amdgcn_readfirstlane(lim_min);

  BtWindow btw;
  bt_window_load(p, sv, (t_first * TOK) >> p.log2_page, btw);
  // Q and the window are in registers before any tile copy goes out: the loop's waits never have to
  // account for them
  __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0)

  // ---- tile copies ----
  // Copy i (< 8) of a K or V stage: rows RPC i .. + RPC - 1, lane l -> row + l / CPR, LDS chunk l %
  // CPR <- global chunk (l % CPR) ^ swizzle(row).  Wave w issues copies w, w + W, ...; the K swizzle of
  // copy i's first row only flips chunk bits (V's is the same for every copy), so each lane's offset
  // inside a stage's buffer is one register, i's rows a scalar offset.
  const int row_bytes = p.n_kv * HD * 2;
  const int lr0 = lane / G::CPR;
  const uint32_t vk = uint32_t(lr0 * row_bytes + (((lane % G::CPR) ^ G::swz_k(wave * G::RPC + lr0)) << 4));
  const uint32_t vv = uint32_t(lr0 * row_bytes + (((lane % G::CPR) ^ G::swz_v(lr0)) << 4));
  // Element offset of a stage's rows of head h in the pools, for consecutive stages: one stage on from
  // the last, or the first of the next page.
  const int pmask = (1 << p.log2_page) - 1;
  const int stage_elems = TOK * p.n_kv * HD;
  int64_t off_k = 0;
  int T_k = t_first * TOK;
  bool bad_page = false;
  auto page_start = [&] {
    const int col = T_k >> p.log2_page;
    if (col - btw.col0 >= 64) {
      bt_window_load(p, sv, col, btw);
      __builtin_amdgcn_s_waitcnt(0x0F70);  // here, once per 64 pages: not at every use of the window
    }
    const int pid = __builtin_amdgcn_readlane(btw.ids, col - btw.col0);
    const bool ok = unsigned(pid) < unsigned(p.num_pages);
    bad_page |= !ok && T_k < L;
    off_k = int64_t(ok ? pid : 0) * p.page_stride + int64_t(T_k & pmask) * (p.n_kv * HD) + h * HD;
  };
  char* const ring_k = lds;
  char* const ring_v = lds + kRing * G::STAGE;
  // Iteration t issues the copies of K stage t + kLead + 2 and V stage t + kLead - 1 (from t = -kLead -
  // 2, V from stage 0), kCopies of each per wave.  Those of a stage past the last are issued too, with an
  // empty buffer: they fetch nothing and write zeros to a free slot, and the loop has neither branches nor
  // other counts to wait for.  A stage's page lookup serves its K copies and, three iterations later,
  // its V copies: off1 .. off3 hold the offsets of the stages in between, oldest first.
  int64_t off1 = 0, off2 = 0, off3 = 0;
  int slot_k = 0, slot_v = 0;    // ring slots the next copies go to
  int left_k = n, left_v = n;    // stages left to copy
  auto next_slot = [](int slot) { return slot == (kRing - 1) * G::STAGE ? 0 : slot + G::STAGE; };
  auto next_stage = [&] {
    if (__builtin_expect((T_k & pmask) == 0 && left_k > 0, 0)) page_start();
    off1 = off2;
    off2 = off3;
    off3 = off_k;
    off_k += stage_elems;
    T_k += TOK;
  };
  auto copy_k = [&](int k) {
    const int i = wave + W * k;
    pf::copy_1k(p.k_cache + off3, left_k > 0 ? TOK * row_bytes : 0, vk ^ uint32_t(G::swz_k(W * k * G::RPC) << 4),
                i * G::RPC * row_bytes, ring_k + slot_k + i * 1024);
    if (k == kCopies - 1) {
      slot_k = next_slot(slot_k);
      --left_k;
    }
  };
  // off_v: off1 as it was before this iteration's next_stage()
  auto copy_v = [&](int k, int64_t off_v) {
    const int i = wave + W * k;
    pf::copy_1k(p.v_cache + off_v, left_v > 0 ? TOK * row_bytes : 0, vv, i * G::RPC * row_bytes,
                ring_v + slot_v + i * 1024);
    if (k == kCopies - 1) {
      slot_v = next_slot(slot_v);
      --left_v;
    }
  };

  // ---- operand reads ----
  const uint32_t k_lane = uint32_t(ln * G::ROWB + ((hi ^ G::swz_k(ln)) << 4));
  uint32_t rd_k = lds_addr(ring_k);  // slots the next reads come from
  uint32_t rd_v = lds_addr(ring_v);
  u32x4 kr[TT][KK];
  auto read_k = [&](int i) {  // operand i of the 8, in the order the products use them
    const int kk = i / TT, u = i % TT;
    kr[u][kk] = pf::lds_read16((k_lane ^ uint32_t(kk << 5)) + rd_k + u * 32 * G::ROWB);
  };
  auto next_k = [&] {
    rd_k = rd_k + G::STAGE == lds_addr(ring_k) + kRing * G::STAGE ? lds_addr(ring_k) : rd_k + G::STAGE;
  };
  // Transpose reads (ds_read_b64_tr_b16): in each 16-lane group (g), lane 4 j + c names elements 32 dt
  // + 16 (g & 1) + 4 c .. + 3 of token row 16 s + 4 hi + j (then 8 rows further) and receives its
  // column: element 32 dt + ln of 4 tokens.
  const int vj = (lane & 15) >> 2;
  const uint32_t v_lane = uint32_t((4 * hi + vj) * G::ROWB + (G::swz_v(vj) << 4) + ((lane >> 4) & 1) * 32 + (lane & 3) * 8);
  u32x2 vlo[8], vhi[8];  // [(u * 2 + s) * DT + dt]
  auto read_v_issue = [&](int i) {  // a quarter of the operands: sub-tile i % TT, output tile i / TT
    const int dt = i / TT, u = i % TT;
    constexpr int S1 = 16 * G::ROWB, U1 = 32 * G::ROWB, H1 = 8 * G::ROWB;
    const uint32_t a = (v_lane ^ uint32_t(dt << 6)) + rd_v + (u ? U1 : 0);
    const int at = u * 2 * DT + dt;
    vlo[at] = lds_read_tr16_issue<0>(a);
    vhi[at] = lds_read_tr16_issue<H1>(a);
    vlo[at + DT] = lds_read_tr16_issue<S1>(a);
    vhi[at + DT] = lds_read_tr16_issue<S1 + H1>(a);
  };
  auto next_v = [&] {
    rd_v = rd_v + G::STAGE == lds_addr(ring_v) + kRing * G::STAGE ? lds_addr(ring_v) : rd_v + G::STAGE;
  };

  // ---- state ----
  f32x16 o[DT];
#pragma unroll
  for (int dt = 0; dt < DT; ++dt)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
  float m_run = -INFINITY, neg_m = 0.f, l_run = 0.f, lmax = -INFINITY;

  auto product_qk = [&](f32x16 (&s)[TT], int i) {
    const int kk = i / TT, u = i % TT;
    if (kk == 0)
#pragma unroll
      for (int r = 0; r < 16; ++r) s[u][r] = 0.f;
    s[u] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, kr[u][kk]), qf[kk], s[u], 0, 0, 0);
  };
  auto product_pv = [&](const u32x4 (&pk)[NP], int i) {
    const int ks = i / DT, dt = i % DT;
    const bf16x8 v = __builtin_bit_cast(bf16x8, u32x4{vlo[i][0], vlo[i][1], vhi[i][0], vhi[i][1]});
    o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, __builtin_bit_cast(bf16x8, pk[ks]), o[dt], 0, 0, 0);
    if constexpr (PAIR)
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(v, __builtin_bit_cast(bf16x8, pk[2 * TT + ks]), o[dt], 0, 0, 0);
  };
  // Step i (of 16) of a stage's exponentials: 2 TT scores, rounded to bf16 (the PV operand) and summed
  // as rounded (PAIR: kept as a pair, summed in fp32).  At one score pair per two steps the second
  // exponential waits for the odd step.
  float e_held = 0.f, x_held = 0.f;
  auto exps = [&](const f32x16 (&s)[TT], u32x4 (&pk)[NP], int i) {
    const int pr = TT == 2 ? i : i >> 1;  // score pair
    const int u = pr >> 3, e = 2 * (pr & 7);
    if (TT == 2 || (i & 1) == 0) {
      e_held = fast_exp2(fmaf(s[u][e], p.scale_log2, neg_m));
      x_held = fmaf(s[u][e + 1], p.scale_log2, neg_m);
    }
    if (TT == 2 || (i & 1) == 1) {
      const float e1 = fast_exp2(x_held);
      uint32_t pair;
      if constexpr (PAIR) {
        l_run += e_held + e1;
        uint32_t rest = pf::split_pair(e_held, e1, pair);
        pf::pin(rest);
        pk[2 * TT + (pr >> 2)][pr & 3] = rest;
      } else {
        pair = pack_bf16x2(e_held, e1);
        l_run = pf::add_pair(pair, l_run);
      }
      pf::pin(pair);
      pk[pr >> 2][pr & 3] = pair;
    }
  };
  // step i (of 8) of the next stage's score maximum
  auto max_step = [&](const f32x16 (&s)[TT], float& m, int i) {
#pragma unroll
    for (int k = 2 * TT * i; k < 2 * TT * (i + 1); k += 2)
      m = k == 0 ? pf::max2(s[0][0], s[0][1]) : pf::max2(pf::max2(m, s[k >> 4][k & 15]), s[k >> 4][(k & 15) + 1]);
  };

  // Iteration t on the scores s (stage t) and the probabilities pp (stage t - 1): see the top of the
  // file.  The next scores go to sn (the last iteration's are of nothing and unused), stage t's
  // probabilities to pn.
  auto iterate = [&](int t, f32x16 (&s)[TT], f32x16 (&sn)[TT], const u32x4 (&pp)[NP], u32x4 (&pn)[NP]) {
    // K of stage t + 2 and V of stage t - 1 landed (the last kLead - 1 iterations' copies may be in flight),
    // this wave's own reads done
    pf::wait_vm<2 * kCopies * (kLead - 1), true>();
    raw_barrier();
    const int T0 = (t_first + t) * TOK;
    if (__builtin_expect(T0 + TOK - 1 > lim_min, 0)) {
#pragma unroll
      for (int u = 0; u < TT; ++u)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (T0 + 32 * u + 8 * (r >> 2) + 4 * hi + (r & 3) > lim) s[u][r] = -INFINITY;
#pragma unroll
      for (int i = 0; i < 8; ++i) max_step(s, lmax, i);
    }
    bool rescale = false;
    float alpha = 1.f;
    if (__builtin_expect(__any(lmax * p.scale_log2 > m_run + kRescaleSlack), 0)) {
      rescale = true;
      const float mx = pf::max_halves(lmax) * p.scale_log2;
      const float m_new = mx > m_run + kRescaleSlack ? mx : m_run;
      alpha = m_new == -INFINITY ? 1.f : fast_exp2(m_run - m_new);  // a row that has seen no key keeps -inf
      l_run *= alpha;
      m_run = m_new;
      neg_m = m_new == -INFINITY ? 0.f : -m_new;
    }
    const int64_t off_v = off1;
    next_stage();
    // phase A
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      product_qk(sn, i);
      if (i >= 2 && i < 6) read_v_issue(i - 2);
      exps(s, pn, i);
      if (kCopies == 2 ? i == 1 || i == 6 : (i & 1) == 1) copy_k(kCopies == 2 ? i / 6 : i / 2);
      __builtin_amdgcn_sched_barrier(0);
    }
    next_v();
    pf::pin(l_run);
    // phase B
    __builtin_amdgcn_sched_barrier(0);
    lds_tr_wait(vlo, vhi);
    __builtin_amdgcn_sched_barrier(0);
    float mx = 0.f;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      product_pv(pp, i);
      read_k(i);
      exps(s, pn, 8 + i);
      if (i > 0) max_step(sn, mx, i - 1);
      if (kCopies == 2 ? i == 2 || i == 6 : (i & 1) == 1) copy_v(kCopies == 2 ? (i - 2) / 4 : i / 2, off_v);
      __builtin_amdgcn_sched_barrier(0);
    }
    max_step(sn, mx, 7);
    __builtin_amdgcn_s_setprio(0);
    lmax = mx;
    next_k();
    pf::pin(lmax);
    pf::pin(l_run);
    __builtin_amdgcn_sched_barrier(0);
    if (__builtin_expect(rescale, 0)) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) o[dt] *= alpha;
    }
  };

  if (n > 0) {
    // V of stage -1 reads as zero: iteration 0's PV products add nothing
    rd_v = lds_addr(ring_v) + (kRing - 1) * G::STAGE;
    {
      char* z = ring_v + (kRing - 1) * G::STAGE + threadIdx.x * 16;
#pragma unroll
      for (int i = 0; i < kCopies; ++i) *reinterpret_cast<u32x4*>(z + i * 1024 * W) = u32x4{0u, 0u, 0u, 0u};
    }
    page_start();
    int64_t off_v = 0;
    for (int t = -kLead - 2; t < -1; ++t) {
      off_v = off1;
      next_stage();
#pragma unroll
      for (int k = 0; k < kCopies; ++k) copy_k(k);
    }
    if (kLead == 3)
#pragma unroll
      for (int k = 0; k < kCopies; ++k) copy_v(k, off_v);
    // K of stages 0 and 1 landed: those of K stages 2 .. kLead and of V stages 0 .. kLead - 3 were issued after
    pf::wait_vm<kCopies * (kLead - 1 + kLead - 2)>();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0): the zeroed slot
    raw_barrier();
    // The scores and probabilities alternate between two register sets, so the iterations go in pairs;
    // an odd count does stage 0 by itself.
    f32x16 s0[TT], s1[TT];
    u32x4 p0[NP], p1[NP];
#pragma unroll
    for (int ks = 0; ks < NP; ++ks) p0[ks] = p1[ks] = u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int i = 0; i < 8; ++i) read_k(i);
    next_k();
#pragma unroll
    for (int i = 0; i < 8; ++i) product_qk(s0, i);
#pragma unroll
    for (int i = 0; i < 8; ++i) max_step(s0, lmax, i);
#pragma unroll
    for (int i = 0; i < 8; ++i) read_k(i);
    next_k();
    __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
    raw_barrier();                       // K stage 0 is read: its slot takes iteration -1's copies
    off_v = off1;
    next_stage();
#pragma unroll
    for (int k = 0; k < kCopies; ++k) copy_k(k);
#pragma unroll
    for (int k = 0; k < kCopies; ++k) copy_v(k, off_v);
    int t = 0;
    if (n & 1) {
#pragma unroll
      for (int u = 0; u < TT; ++u) s1[u] = s0[u];
      iterate(0, s1, s0, p0, p1);
      t = 1;
    }
    for (; t < n; t += 2) {
      iterate(t, s0, s1, p1, p0);
      iterate(t + 1, s1, s0, p0, p1);
    }
    {
      // the last stage's V landed for every wave, and no copy outlives the workgroup
      pf::wait_vm<0>();
      raw_barrier();
      // the last stage's PV products; keys past the sequence: P = 0 must not meet a stale NaN
#pragma unroll
      for (int i = 0; i < 4; ++i) read_v_issue(i);
      lds_tr_wait(vlo, vhi);
      const int T0 = (t_first + n - 1) * TOK;
      if (T0 + TOK > L) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int k0 = T0 + 16 * (i / DT) + 4 * hi;
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const int k = k0 + 2 * w;
            vlo[i][w] &= (k < L ? 0x0000FFFFu : 0u) | (k + 1 < L ? 0xFFFF0000u : 0u);
            vhi[i][w] &= (k + 8 < L ? 0x0000FFFFu : 0u) | (k + 9 < L ? 0xFFFF0000u : 0u);
          }
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) product_pv(p1, i);
    }
  }
  if (bad_page && lane == 0) flag_status(p.status, PKV_STATUS_BAD_PAGE);

  const float lsum = pf::sum_halves(l_run);
  const float inv = lsum > 0.f ? 1.f / lsum : 0.f;
  uint32_t l_end = threadIdx.x & 63;
  pf::pin(l_end);  // the row is worked out again: kept, it would hold registers through the loop
  const LaneRow lo = lane_row(int(l_end));
  // o[dt][4 q + r] is element 32 dt + 8 q + 4 hi + r of the lane's row
  if constexpr (CASCADE) {
    const uint32_t lse0 = uint32_t(p.ws_ml - p.ws_o) * 4u;
    const __amdgpu_buffer_rsrc_t rs = ws_rsrc(p);
    bool ovf = false;
    if (lo.real) {
      const int slot = 2 * p.lean_grid + lo.b * p.cascade_splits + int(blockIdx.z);
      const uint32_t wrow = uint32_t((slot * rows::NKV + h) * p.R + lo.r);
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[4];
#pragma unroll
          for (int r = 0; r < 4; ++r) v[r] = o[dt][4 * q + r] * inv;
          ovf = ovf || f16_overflows(v[0], v[1]) || f16_overflows(v[2], v[3]);
          const u32x2 ov = {pack_f16x2(v[0], v[1]), pack_f16x2(v[2], v[3])};
          __builtin_amdgcn_raw_buffer_store_b64(ov, rs, int((wrow * HD + 32 * dt + 8 * q + 4 * hi) * 2u), 0, 0);
        }
      const float lse = lsum > 0.f ? m_run + __builtin_amdgcn_logf(lsum) : -INFINITY;
      if (hi == 0) __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, lse), rs, int(lse0 + wrow * 4u), 0, 0);
    }
    if (__any(ovf) && lane == 0) flag_status(p.status, PKV_STATUS_PARTIAL_RANGE);
    return;
  }
  if constexpr (DEST == pf::kSplit) {
    if (count > 1) {
      if (lo.real) {
        int64_t slot = int64_t(blockIdx.x);
        if constexpr (W == pf::kWaves)
          slot = int64_t((b * p.n_kv + h) * (int(gridDim.x) / p.max_splits) + xblk) * p.max_splits + split;
        const int64_t wrow = slot * kRows + lo.r - blk_row0;
        float* dst = p.ws_o + wrow * HD + 4 * hi;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int q = 0; q < 4; ++q)
            *reinterpret_cast<f32x4*>(dst + 32 * dt + 8 * q) =
                f32x4{o[dt][4 * q], o[dt][4 * q + 1], o[dt][4 * q + 2], o[dt][4 * q + 3]};
        if (hi == 0) *reinterpret_cast<f32x2*>(p.ws_ml + 2 * wrow) = f32x2{m_run, lsum};
      }
      return;
    }
  }
  if (lo.real) {
    uint16_t* dst = p.out + lo.b * p.o_sb + lo.j * p.o_ss + lo.hq * p.o_sh + 4 * hi;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const u32x2 ov = {pack_bf16x2(o[dt][4 * q] * inv, o[dt][4 * q + 1] * inv),
                          pack_bf16x2(o[dt][4 * q + 2] * inv, o[dt][4 * q + 3] * inv)};
        *reinterpret_cast<u32x2*>(dst + 32 * dt + 8 * q) = ov;
      }
  }
}

// Merge of a kSplit launch of ROWS-row blocks: grid (row block x ROWS HD / 1024, KV head, sequence),
// 1024 / HD rows of an item per workgroup, one f32x4 of a row per thread.  Every range's load of a batch
// of 8 goes out before any is used.
template <int HD, int ROWS>
__global__ __launch_bounds__(256) void prefill_merge_kernel(const AttnParams p, int nx) {
  constexpr int TPR = HD / 4, RPW = 256 / TPR, B = 8;
  constexpr int BLOCKS = ROWS / RPW;  // workgroups per item
  const int xblk = int(blockIdx.x) / BLOCKS, h = blockIdx.y, b = blockIdx.z;
  const int r = (int(blockIdx.x) % BLOCKS) * RPW + int(threadIdx.x) / TPR;  // row in the block
  const int blk_row0 = xblk * ROWS;
  const int row = blk_row0 + r;
  int count = 1;
  int64_t w0;           // the first range's row in the workspace, and the rows to the next one's
  int64_t w_step = ROWS;
  if constexpr (ROWS == pf::kVerifyRows) {
    const int first = p.ws_cnt[2 * b];
    count = p.ws_cnt[2 * b + 1];
    w0 = (int64_t(first) * p.n_kv + h) * ROWS + r;
    w_step = int64_t(p.n_kv) * ROWS;
  } else {
    int c, L;
    seq_lengths(p, b, c, L);
    count = pf::ranges_of(p, pf::stages_of<pf::Geo<HD>::TOK>(p, L, min(blk_row0 + ROWS, p.R) - 1)).count;
    w0 = int64_t((b * p.n_kv + h) * nx + xblk) * p.max_splits * ROWS + r;
  }
  if (count <= 1 || row >= p.R) return;
  const int d = (int(threadIdx.x) % TPR) * 4;
  float m = -INFINITY, l = 0.f;
  f32x4 o = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < count; s0 += B) {
    f32x4 po[B];
    f32x2 pm[B];
#pragma unroll
    for (int k = 0; k < B; ++k) {
      const int64_t w = w0 + min(s0 + k, count - 1) * w_step;
      po[k] = *reinterpret_cast<const f32x4*>(p.ws_o + w * HD + d);
      pm[k] = *reinterpret_cast<const f32x2*>(p.ws_ml + 2 * w);
    }
    float m_new = m;
#pragma unroll
    for (int k = 0; k < B; ++k) m_new = fmaxf(m_new, pm[k][0]);
    const float keep = m_new == -INFINITY ? 1.f : fast_exp2(m - m_new);
    l *= keep;
    o *= keep;
#pragma unroll
    for (int k = 0; k < B; ++k) {
      // a range of which the row sees no key has l = 0 and m = -inf
      const float wt = s0 + k < count && pm[k][1] > 0.f ? fast_exp2(pm[k][0] - m_new) : 0.f;
      l += wt * pm[k][1];
      o += wt * po[k];
    }
    m = m_new;
  }
  const int j = row / p.g;
  const float inv = l > 0.f ? 1.f / l : 0.f;
  uint16_t* dst = p.out + b * p.o_sb + j * p.o_ss + (h * p.g + row - j * p.g) * p.o_sh + d;
  *reinterpret_cast<u32x2*>(dst) = u32x2{pack_bf16x2(o[0] * inv, o[1] * inv), pack_bf16x2(o[2] * inv, o[3] * inv)};
}
