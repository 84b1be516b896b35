// Long-prompt prefill tiling of the paged attention (included by paged_attention.hip,
// inside its namespace).
//
// Calls whose longest q window reaches kPfMinQ rows (prompt prefill, long chunks) take a
// tiling built for many rows per sequence: one 256-thread workgroup per (sequence,
// 128-row group, kv head), two workgroups per CU, each wave owning 32 rows (one column
// block of v_mfma_f32_32x32x16).  64-position K and V tiles are staged once per
// workgroup in LDS, double-buffered, and shared by the four waves.  The output is
// normalized in the kernel (no split, no merge launch).  Rows of such a call equal the
// per-row form within floating-point tolerance, not bit for bit (the tile boundaries
// differ).
//
// Schedule.  The tile loop is software-pipelined over the two products: iteration i runs
// S(i+1) = K Q^T next to the exponentials of S(i), then O += V(i) P(i) next to the row
// maximum of S(i+1), so the matrix cores always have independent work while the vector
// unit runs the softmax.  K therefore runs one tile ahead of V: during iteration i the
// direct loads of K(i+2) and V(i+1) are in flight, into the buffers whose tiles were
// last read in iteration i - 1.  The order inside a phase is fixed by scheduling barriers
// (left to itself the compiler moves the exponentials behind the products).
//
// What bounds it: a 128-row tile needs ~1030 cycles of a SIMD's matrix core, ~600 of its
// vector unit and ~1020 of the CU's LDS reads (32 KB a wave: every wave reads the whole K
// and V tile), so the three overlap or add up.  bf16, D = 128, 16 / 4 heads, against the
// unpipelined 16x16x32 form of the same split (graph replays, two boxes): 8 x 2048 prompts 254
// -> 176-179 us (541 -> 770-780 TFLOP/s), 4 x 4096 431 -> 296-306, 1 x 8192 400 -> 292-306
// (687 -> 897-943), D = 96 8 x 2048 271 -> 143-149, fp8 8 x 2048 294 -> 203-210; 6 chunks of up to
// 512 rows in fp8 with per-vector scales behind a prefix, store included, 162 -> 110 (a large
// bf16 matrix product reaches 1360 TFLOP/s here).  The time without overlap went into waits:
// the transpose reads waited for the next tile's loads, the matrix cores for the softmax.
#pragma once

constexpr int kPfWaves = 4;                // waves per workgroup (sharing each staged tile)
constexpr int kPfRows = kPfWaves * 32;     // q rows per workgroup
constexpr int kPfKeys = 64;                // key positions per LDS tile
constexpr int kPfThreads = 64 * kPfWaves;
constexpr int kPfMinQ = 64;                // q window length from which a call takes this path
constexpr float kPfLazy = 8.f;             // log2 headroom before the running max moves

// LDS row width in dims: D = 96 rows take a 128-dim row whose last four 16-byte slots
// (their place moves with the swizzle) are never loaded nor read
template <int D>
constexpr int pf_row_dims() { return D == 96 ? 128 : D; }

template <int D>
struct PrefillLds {
  static constexpr int kRowB = pf_row_dims<D>() * 2;  // bytes per position row (XOR-swizzled slots)
  alignas(16) uint8_t k[2][kPfKeys * kRowB];
  alignas(16) uint8_t v[2][kPfKeys * kRowB];
  alignas(16) float ks[2][kPfKeys];  // per-vector fp8 scales of the tile's positions (SM 2)
  alignas(16) float vs[2][kPfKeys];
};

typedef __attribute__((address_space(3))) void lds_void;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

// v_mfma_f32_32x32x16: A lane (m = lane % 32, h = lane / 32) holds contraction slots
// 8 h .. 8 h + 7, B the same with n; C / D lane holds column n = lane % 32, rows
// 8 (i / 4) + 4 h + i % 4.
template <int QT>
__device__ __forceinline__ f32x16 mfma32(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (QT == RLT_BF16) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a),
                                                  __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  }
}

// 16-byte slot of piece `piece` (8 dims) in row r of a staged tile (an involution).  K rows
// XOR the slot with r mod SLOTS, so the S^T operand reads (16 lanes = 16 rows of one piece
// column) meet distinct bank groups.  V rows XOR it with 4 (r & 3) (16 slots; rows of 8
// slots, two of which span the banks, with 4 ((r >> 1) & 1)): a transpose read's 32 lanes
// take 4 rows x one 64-byte dim tile, and the four rows' tiles then cover the banks once.
template <int SLOTS>
__device__ __forceinline__ int k_slot(int r, int piece) { return piece ^ (r & (SLOTS - 1)); }
template <int SLOTS>
__device__ __forceinline__ int v_slot(int r, int piece) {
  return piece ^ (SLOTS >= 16 ? 4 * (r & 3) : 4 * ((r >> 1) & 1));
}

// Direct global -> LDS load of 16 bytes a lane: lane L's bytes land at `lds` + 16 L.  Written
// in assembly (it has no register result) because the compiler, which cannot tell these
// LDS writes from the buffers read meanwhile, made every transpose read wait for all loads
// in flight, and every K read for all reads before it; the caller waits with wait_loads().
// The s_nop covers a base register written by the vector unit just before (5 wait states)
// and M0's own wait state.  (M0 is a reserved register, which the compiler lets no clobber list
// name.  No other instruction of this kernel reads it; one that did -- the compiler may set it
// once for several of its own -- would need it saved and restored here.)
__device__ __forceinline__ uint32_t lds_offset(const void* p) {
  return (uint32_t)(uintptr_t)(lds_void*)p;
}
__device__ __forceinline__ void load_lds16(const void* base, uint32_t lane_bytes, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, %1"
               :
               : "v"(lane_bytes), "s"(base), "s"(lds)
               : "memory");
}
__device__ __forceinline__ void load_lds16(const void* lane_address, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, off"
               :
               : "v"(lane_address), "s"(lds)
               : "memory");
}
__device__ __forceinline__ void wait_loads() { asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); }

// The other half-wave's value of a 32-row lane pair (lane ^ 32), combined.
__device__ __forceinline__ float half_max(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
}
__device__ __forceinline__ float half_sum(float x) {
  const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(a[0]) + __uint_as_float(a[1]);
}

// Walks the block table one 64-position tile at a time: the (table index, offset) of a
// position advances without a division, and the table entry is read one tile before it
// is needed.
struct TileCursor {
  int idx, off;   // of the tile whose entry `next` holds
  int32_t next;   // its table entry, as read
  __device__ __forceinline__ void start(const AttnParams& P, const int32_t* table, int pos) {
    idx = pos / P.block_size;
    off = pos % P.block_size;
    next = table[min(idx, P.table_width - 1)];
  }
  __device__ __forceinline__ void advance(const AttnParams& P, const int32_t* table, int dq, int dr) {
    idx += dq;
    off += dr;
    if (off >= P.block_size) {
      off -= P.block_size;
      ++idx;
    }
    next = table[min(idx, P.table_width - 1)];
  }
};

// UB: block_size % 16 == 0 (and a token stride that fits 32-bit lane offsets), so each
// 16-position group of a tile lies in one block, whose table entry is wave-uniform.
// KVT: the pool type, QT's own or fp8-e4m3 with scale mode SM (1 per-tensor, 2
// per-vector).  16-bit tiles are staged by direct global -> LDS loads.  FP8 tiles are
// staged through registers: each thread loads 8-code pieces (item e = 256 j + t: LDS slot
// e % SLOTS of row e / SLOTS, holding the piece the swizzle puts there) while the previous
// tile is in use, then widens them to QT (exact for e4m3) into the same swizzled LDS
// layout; the per-tensor key scale folds into the score scale and the value scale into
// the output, per-vector scales multiply each position's score and (for P V only) its
// weight.
template <int QT, int KVT, int D, int SM, bool UB>
__global__ __launch_bounds__(kPfThreads, 2) void rlt_prefill_kernel(AttnParams P) {
  using M = Mfma<QT>;
  using L = PrefillLds<D>;
  constexpr int NQS = D / 16;       // 16-wide contraction slices of S^T
  constexpr int ND = D / 32;        // 32-wide dim tiles of O^T
  constexpr int PIECES = D / 8;     // 16-byte pieces of a position row in the pool
  constexpr int SLOTS = pf_row_dims<D>() / 8;  // 16-byte slots per LDS row (>= PIECES)
  constexpr int ROWS_PER_LD = 64 / SLOTS;      // rows one wave-wide direct load fills
  constexpr int LD = kPfKeys / ROWS_PER_LD / kPfWaves;  // direct loads per wave per tile (K, V each)
  static_assert(LD * ROWS_PER_LD == 16, "a wave's direct loads fill one 16-position group");
  constexpr bool FP8 = KVT != QT;
  static_assert(!FP8 || KVT == RLT_FP8_E4M3, "16-bit pools match q");
  static_assert(FP8 == (SM != 0), "scale modes are for fp8 pools");
  constexpr int FJ = kPfKeys * SLOTS / kPfThreads;  // fp8 LDS slots per thread per tile (K, V each)
  static_assert(FJ * kPfThreads == kPfKeys * SLOTS, "the threads' fp8 slots cover a tile");
  // operand reads in flight ahead of their MFMAs: S^T slices, O^T steps (fp8 tiles leave
  // fewer registers)
  constexpr int kAheadK = FP8 ? 2 : 4;
  constexpr int kAheadV = FP8 ? 2 : 3;
  // fp8 V is loaded with K where the registers hold both (after K's pieces have left theirs, V's
  // latency shows on cold keys: 8 windows of up to 130 rows behind 3000, 16 heads of 64 dims,
  // 80.7 -> 62.3 us; with per-vector scales it took 88.6 -> 93.1)
  constexpr bool kEarlyV = SM == 1 && D <= 64;
  constexpr int NC = FP8 ? FJ : 1;  // 16-position groups a wave loads from per tile
  __shared__ L sh;
  const int t = threadIdx.x, lane = t & 63, l32 = lane & 31, h = lane >> 5;
  const int w = __builtin_amdgcn_readfirstlane(t >> 6);

  // heaviest row-groups (latest positions) first across the whole batch: the
  // row-group index is outermost, then the sequence, then the kv head
  const int64_t id = blockIdx.x;
  const int kvh = (int)(id % P.hkv);
  const int64_t sr = id / P.hkv;
  const int seq = (int)(sr % P.num_seqs);
  const int rg = P.rowgroups - 1 - (int)(sr / P.num_seqs);
  const SeqView sv = seq_view(P, seq);
  const int rows_total = sv.q_len * P.group;
  const int rg_begin = rg * kPfRows;
  if (rg_begin >= rows_total) return;  // uniform over the workgroup
  const int rg_rows = min(kPfRows, rows_total - rg_begin);
  int lo_first, hi_first, lo_last, hi_last;
  group_range(P, sv, rg_begin, rg_rows, lo_first, hi_first, lo_last, hi_last);

  // this lane's row: B operand of S^T = K Q^T
  u32x4 qreg[NQS];
  int row_lo, row_hi;
  // the wave's common visible range: tiles inside [wlo, whi) need no position masks
  // (rows past the group are not stored and do not narrow it)
  int wlo = -(1 << 30), whi = 1 << 30;
  const int local = w * 32 + l32;
  const int rho = rg_begin + local;
  const int qi = rho / P.group;
  const int head = kvh * P.group + rho % P.group;
  if (local < rg_rows) {
    row_range(P, sv, qi, row_lo, row_hi);
    wlo = row_lo;
    whi = row_hi;
    const uint16_t* qp = (const uint16_t*)P.q + (int64_t)(sv.q_begin + qi) * P.q_row_stride +
                         (int64_t)head * P.q_head_stride + h * 8;
#pragma unroll
    for (int s = 0; s < NQS; ++s) qreg[s] = *(const u32x4*)(qp + 16 * s);
  } else {
    row_lo = row_hi = 0;
#pragma unroll
    for (int s = 0; s < NQS; ++s) qreg[s] = u32x4{0, 0, 0, 0};
  }
  for (int off = 16; off >= 1; off >>= 1) {
    wlo = max(wlo, __shfl_xor(wlo, off, RLT_WAVE));
    whi = min(whi, __shfl_xor(whi, off, RLT_WAVE));
  }
  wlo = __builtin_amdgcn_readfirstlane(wlo);
  whi = __builtin_amdgcn_readfirstlane(whi);

  f32x16 oacc[ND];
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int i = 0; i < 16; ++i) oacc[dt][i] = 0.f;
  float m_run = -INFINITY, m_use = 0.f;
  float l_run = 0.f;  // this half-wave's share of the row's weights

  const int kt0 = lo_first / kPfKeys;
  const int kt1 = (hi_last + kPfKeys - 1) / kPfKeys;

  // ---- global -> LDS staging.  Direct loads: wave w's j-th load fills rows 16 w +
  // ROWS_PER_LD j + [0, ROWS_PER_LD); lane L takes row + L / SLOTS and LDS slot L % SLOTS,
  // into which it loads the row's swizzled piece
  const int ld_row = lane / SLOTS;
  const int ld_slot = lane % SLOTS;
  const int64_t k_head = (int64_t)kvh * P.k_head_stride;
  const int64_t v_head = (int64_t)kvh * P.v_head_stride;
  const int32_t* table = P.tables + (int64_t)seq * P.table_stride;
  const int dq = kPfKeys / P.block_size, dr = kPfKeys % P.block_size;
  // block id and offset of position pos: entries outside the pool read block 0
  auto pool_block = [&](int32_t e) { return (e >= 0 && e < P.num_blocks) ? e : 0; };
  // the tile's row whose block the wave's c-th cursor follows: the first of the 16-position
  // group of its c-th access (UB), or, in lane i, the row that access i / ROWS_PER_LD of lanes
  // (i % ROWS_PER_LD) SLOTS .. reads (one lookup per row and wave; a lookup with its divisions
  // per access took 44.3 us where this takes 30.0, 4 prompts of 300-500 rows at block size 8)
  auto cursor_row = [&](int c) {
    const int i = UB ? ROWS_PER_LD * c : lane & 15;
    const int r = FP8 ? i / ROWS_PER_LD * (kPfThreads / SLOTS) + w * ROWS_PER_LD + i % ROWS_PER_LD
                      : 16 * w + i;
    return UB ? r & ~15 : r;
  };
  // blocks and offsets of the K tile loaded last; the cursor holds the next tile's
  constexpr int CUR = UB ? NC : 1;
  TileCursor cur[CUR];
  int kblk[CUR] = {}, koff[CUR] = {};
  // per-vector scales: wave 0 stages the keys' (with the K tile), wave 1 the values'
  TileCursor scur;
  const bool scale_wave = SM == 2 && w < 2;

  uint2 kraw[FP8 ? FJ : 1], vraw[FP8 ? FJ : 1];
  float sraw = 0.f;

  // bytes from a 16-position group's first row to what this lane reads of it.  The swizzle's
  // piece of an fp8 item is the same for every j; a direct load's rows are ROWS_PER_LD
  // apart (the scalar base moves), which changes the piece of K only
  const int lane_r = FP8 ? (t / SLOTS) & 15 : ld_row;
  const int lane_sl = FP8 ? t % SLOTS : ld_slot;
  constexpr int ELT = FP8 ? 1 : 2;  // bytes of a pool element
  const uint32_t k_tok = (uint32_t)P.k_token_stride * ELT, v_tok = (uint32_t)P.v_token_stride * ELT;
  const int v_piece = v_slot<SLOTS>(lane_r, lane_sl);
  const uint32_t v_off = lane_r * v_tok + v_piece * 8 * ELT;

  // the lane's j-th access of K / V: from the 16-position group at (blk, off) (UB) or from
  // the lane's own position there
  auto load_k_piece = [&](int b, int j, int64_t blk, int off) {
    const uint8_t* base = (const uint8_t*)P.k +
                          (blk * P.k_block_stride + k_head + (int64_t)off * P.k_token_stride) * ELT;
    const int pc = k_slot<SLOTS>(lane_r + (FP8 ? 0 : ROWS_PER_LD * j), lane_sl);
    if (UB && !FP8) base += (int64_t)(ROWS_PER_LD * j) * k_tok;
    const uint32_t lane_off = lane_r * k_tok + pc * 8 * ELT;
    // padded rows: lanes whose slot holds a piece past the row load nothing
    if (PIECES == SLOTS || pc < PIECES) {
      if constexpr (FP8) {
        kraw[j] = UB ? *(const uint2*)(base + lane_off) : *(const uint2*)(base + pc * 8);
      } else {
        const uint32_t lds = lds_offset(sh.k[b]) + (16 * w + ROWS_PER_LD * j) * L::kRowB;
        if (UB) load_lds16(base, lane_off, lds);
        else load_lds16(base + pc * 16, lds);
      }
    }
  };
  auto load_v_piece = [&](int b, int j, int64_t blk, int off) {
    const uint8_t* base = (const uint8_t*)P.v +
                          (blk * P.v_block_stride + v_head + (int64_t)off * P.v_token_stride) * ELT;
    static_assert(FP8 || ROWS_PER_LD % 4 == 0, "one V piece per lane");
    const int pc = v_piece;
    if (UB && !FP8) base += (int64_t)(ROWS_PER_LD * j) * v_tok;
    if (PIECES == SLOTS || pc < PIECES) {
      if constexpr (FP8) {
        vraw[j] = UB ? *(const uint2*)(base + v_off) : *(const uint2*)(base + pc * 8);
      } else {
        const uint32_t lds = lds_offset(sh.v[b]) + (16 * w + ROWS_PER_LD * j) * L::kRowB;
        if (UB) load_lds16(base, v_off, lds);
        else load_lds16(base + pc * 16, lds);
      }
    }
  };
  constexpr int NJ = FP8 ? FJ : LD;
  // the cursor's tile becomes the K tile to load, and the next entry is read (before any
  // load of this iteration is in flight: the entry's use would wait for all of them)
  auto next_blocks = [&]() {
#pragma unroll
    for (int c = 0; c < CUR; ++c) {
      kblk[c] = pool_block(UB ? __builtin_amdgcn_readfirstlane(cur[c].next) : cur[c].next);
      koff[c] = cur[c].off;
      cur[c].advance(P, table, dq, dr);
    }
  };
  // block and offset of this lane's j-th access among the wave's
  auto access = [&](const int (&x)[CUR], int j) {
    if (UB) return x[FP8 ? j : 0];
    return __builtin_amdgcn_ds_bpermute(4 * (ROWS_PER_LD * j + lane / SLOTS), x[0]);
  };
  auto load_k = [&](int b) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_k_piece(b, j, access(kblk, j), access(koff, j));
  };
  // V of a tile into buffer b, from the blocks `blks`, `offs` that its K was loaded from
  auto load_v = [&](int b, const int (&blks)[CUR], const int (&offs)[CUR]) {
#pragma unroll
    for (int j = 0; j < NJ; ++j) load_v_piece(b, j, access(blks, j), access(offs, j));
  };
  // the scales of the cursor's tile, read into a register (wave 0 keys, wave 1 values)
  auto load_scale = [&](int tile) {
    const float x = (w == 0 ? P.k_scale : P.v_scale)[pool_block(scur.next) * P.s_block_stride +
                                                     (int64_t)scur.off * P.s_token_stride +
                                                     (int64_t)kvh * P.s_head_stride];
    sraw = tile * kPfKeys + lane < hi_last ? x : 0.f;
    scur.advance(P, table, dq, dr);
  };
  // fp8: the loaded pieces of K / V of `tile`, widened, into buffer b (two 8-byte halves:
  // 16-byte LDS writes of a whole wave conflicted, the counters read 4x an ideal write)
  auto put_k = [&](int b) {
#pragma unroll
    for (int j = 0; j < FJ; ++j) {
      const int e = j * kPfThreads + t;
      const int r = e / SLOTS, sl = e % SLOTS;
      // (pad slots of 96-dim rows are never read: left unwritten)
      if (PIECES == SLOTS || k_slot<SLOTS>(r, sl) < PIECES) {
        const uint2 k0 = fp8x4_to_16<QT>(kraw[j].x), k1 = fp8x4_to_16<QT>(kraw[j].y);
        uint2* kd = (uint2*)(sh.k[b] + r * L::kRowB + sl * 16);
        kd[0] = k0;
        kd[1] = k1;
      }
    }
  };
  auto put_v = [&](int tile, int b) {
#pragma unroll
    for (int j = 0; j < FJ; ++j) {
      const int e = j * kPfThreads + t;
      const int r = e / SLOTS, sl = e % SLOTS;
      if (PIECES == SLOTS || v_slot<SLOTS>(r, sl) < PIECES) {
        uint2 v0 = make_uint2(0, 0), v1 = v0;
        if (tile * kPfKeys + r < hi_last) {
          v0 = fp8x4_to_16<QT>(vraw[j].x);
          v1 = fp8x4_to_16<QT>(vraw[j].y);
        }
        uint2* vd = (uint2*)(sh.v[b] + r * L::kRowB + sl * 16);
        vd[0] = v0;
        vd[1] = v1;
      }
    }
  };
  // After this wave's direct loads of V of `tile` into buffer b landed: its rows past the
  // sequence may hold any bits (NaN included) and are zeroed, since their weight 0 times
  // NaN would not vanish.  Only the tiles that reach past hi_last do work.
  auto zero_tail = [&](int tile, int b) {
    const int base = tile * kPfKeys;
    if (base + kPfKeys > hi_last) {
#pragma unroll
      for (int j = 0; j < LD; ++j) {
        const int r = 16 * w + ROWS_PER_LD * j + ld_row;
        if (base + r >= hi_last)
          *(uint4*)(sh.v[b] + r * L::kRowB + ld_slot * 16) = make_uint4(0, 0, 0, 0);
      }
    }
  };

  // S^T operand reads: row 32 u + l32, piece 2 s + h at slot (2 s) ^ (h ^ (l32 mod SLOTS))
  const int k_lane = l32 * L::kRowB;
  const int k_x = (h ^ (l32 & (SLOTS - 1))) * 16;
  // V^T operand reads (transpose loads): within a 16-lane group, lane i receives element
  // i & 3 of the 8-byte reads of lanes (i >> 2) + 4 k, so lane i reads row (i >> 2) at dims
  // 4 (i & 3) and the group gets 16 dims at 4 positions.  Contraction slots 8 h + j of a
  // 16-position chunk c are positions 16 c + 4 h + j (j < 4) and 16 c + 8 + 4 h + j - 4: the
  // order in which the S^T accumulators hold them.
  const int i4 = (lane >> 2) & 3;
  const int v_lane = (4 * h + i4) * L::kRowB + (2 * ((lane >> 4) & 1) + ((lane >> 1) & 1)) * 16 +
                     (lane & 1) * 8;
  const int v_x = SLOTS >= 16 ? i4 : i4 >> 1;

  float qk_scale = P.qk_scale_log2;
  float v_mul = 1.f;
  if (SM == 1) {
    qk_scale *= P.k_scale[0];
    v_mul = P.v_scale[0];
  }

  // ---- S^T = K Q^T of the tile in buffer b: s[u] holds positions 32 u + 8 (i / 4) + 4 h + i % 4
  auto read_k = [&](u32x4 (&a)[2], int c, int b) {
#pragma unroll
    for (int u = 0; u < 2; ++u)
      a[u] = *(const u32x4*)(sh.k[b] + k_lane + u * 32 * L::kRowB + ((32 * c) ^ k_x));
  };
  // `beside(c)` is work that fills the vector unit during contraction slice c; the
  // operands are read kAheadK slices ahead, and nothing moves across a slice
  auto scores = [&](f32x16 (&s)[2], int b, auto&& beside) {
    u32x4 a[kAheadK + 1][2];
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) s[u][i] = 0.f;
#pragma unroll
    for (int c = 0; c < kAheadK && c < NQS; ++c) read_k(a[c], c, b);
#pragma unroll
    for (int c = 0; c < NQS; ++c) {
      __builtin_amdgcn_sched_barrier(0);
      if (c + kAheadK < NQS) read_k(a[(c + kAheadK) % (kAheadK + 1)], c + kAheadK, b);
#pragma unroll
      for (int u = 0; u < 2; ++u) s[u] = mfma32<QT>(a[c % (kAheadK + 1)][u], qreg[c], s[u]);
      beside(c);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // per-vector key scales and the position mask of the tile's scores, in place
  auto scale_scores = [&](f32x16 (&s)[2], int b) {
    if constexpr (SM == 2) {
#pragma unroll
      for (int u = 0; u < 2; ++u)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const f32x4 x = *(const f32x4*)(sh.ks[b] + 32 * u + 8 * g + 4 * h);
#pragma unroll
          for (int i = 0; i < 4; ++i) s[u][4 * g + i] *= x[i];
        }
    }
  };
  auto mask = [&](f32x16 (&s)[2], int tile) {
    const int base = tile * kPfKeys;
    if (base >= wlo && base + kPfKeys <= whi) return;  // wave-uniform
    const int lo = row_lo - base - 4 * h, hi = row_hi - base - 4 * h;
#pragma unroll
    for (int u = 0; u < 2; ++u)
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int pos = 32 * u + 8 * (i >> 2) + (i & 3);
        s[u][i] = (pos >= lo && pos < hi) ? s[u][i] : -INFINITY;
      }
  };
  // The running max moves only when a tile's max exceeds it by more than kPfLazy (weights
  // stay below 2^kPfLazy), so the accumulators are rarely rescaled; the scale enters as
  // one fma per score (qk_scale > 0: the max of raw scores scales).
  auto max_quad = [&](float& m, const f32x16 (&s)[2], int g) {
    const int i = 4 * (g & 3);
    m = fmaxf(fmaxf(m, s[g >> 2][i]), s[g >> 2][i + 1]);
    m = fmaxf(fmaxf(m, s[g >> 2][i + 2]), s[g >> 2][i + 3]);
  };
  auto move_max = [&](float m) {
    const float mx = half_max(m) * qk_scale;
    const bool grow = mx > m_run + kPfLazy;
    if (__builtin_amdgcn_ballot_w64(grow) != 0) {
      const float m_new = grow ? mx : m_run;
      const float use = m_new == -INFINITY ? 0.f : m_new;
      const float corr = grow ? __builtin_amdgcn_exp2f(m_run - use) : 1.f;
      l_run *= corr;
#pragma unroll
      for (int dt = 0; dt < ND; ++dt) oacc[dt] *= corr;
      m_run = m_new;
      m_use = use;
    }
  };
  // ---- weights of four of the tile's scores (positions 8 g + 4 h + [0, 4)): words 2 g and
  // 2 g + 1 of the P^T operands (chunk g / 2)
  auto weigh_quad = [&](const f32x16 (&s)[2], uint32_t (&p)[16], int g, int b) {
    float x[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      x[i] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[g >> 2][4 * (g & 3) + i], qk_scale, -m_use));
    l_run += (x[0] + x[1]) + (x[2] + x[3]);
    if constexpr (SM == 2) {
      const f32x4 y = *(const f32x4*)(sh.vs[b] + 8 * g + 4 * h);
#pragma unroll
      for (int i = 0; i < 4; ++i) x[i] *= y[i];
    }
    p[2 * g] = M::pack2(x[0], x[1]);
    p[2 * g + 1] = M::pack2(x[2], x[3]);
    // (made here: the compiler would sink them to their use, behind the mask's branch)
    asm volatile("" : "+v"(p[2 * g]), "+v"(p[2 * g + 1]), "+v"(l_run));
  };
  // ---- O^T += V^T P^T of the tile in buffer b, one (chunk, dim tile) a step
  auto read_v = [&](u32x4& a, int n, int b) {
    const int c = n / ND, dt = n % ND;
    const uint8_t* vr = sh.v[b] + v_lane + 16 * c * L::kRowB + 64 * (dt ^ v_x);
    const s16x4 x0 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(lds_void*)vr);
    const s16x4 x1 = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
        (__attribute__((address_space(3))) s16x4*)(lds_void*)(vr + 8 * L::kRowB));
    __builtin_memcpy(&a, &x0, 8);
    __builtin_memcpy((char*)&a + 8, &x1, 8);
  };
  auto accumulate = [&](const uint32_t (&p)[16], int b, auto&& beside) {
    u32x4 a[kAheadV + 1];
#pragma unroll
    for (int n = 0; n < kAheadV; ++n) read_v(a[n], n, b);
#pragma unroll
    for (int n = 0; n < 4 * ND; ++n) {
      const int c = n / ND, dt = n % ND;
      __builtin_amdgcn_sched_barrier(0);
      if (n + kAheadV < 4 * ND) read_v(a[(n + kAheadV) % (kAheadV + 1)], n + kAheadV, b);
      const u32x4 pc = {p[4 * c], p[4 * c + 1], p[4 * c + 2], p[4 * c + 3]};
      oacc[dt] = mfma32<QT>(a[n % (kAheadV + 1)], pc, oacc[dt]);
      beside(n);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // the part of the tile's 8 quads that falls to step i of n
  auto quads = [](int i, int n, auto&& f) {
#pragma unroll
    for (int g = 0; g < 8; ++g)
      if (g >= 8 * i / n && g < 8 * (i + 1) / n) f(g);
  };

  if (kt0 < kt1) {
    // ---- first tiles: K and V of kt0, K of kt0 + 1, the scores of kt0
#pragma unroll
    for (int c = 0; c < CUR; ++c) cur[c].start(P, table, kt0 * kPfKeys + cursor_row(c));
    if (scale_wave) scur.start(P, table, kt0 * kPfKeys + lane);
    next_blocks();
    load_k(0);
    load_v(0, kblk, koff);
    if constexpr (FP8) {
      put_k(0);
      put_v(kt0, 0);
      if (scale_wave) {
        load_scale(kt0);
        (w == 0 ? sh.ks : sh.vs)[0][lane] = sraw;
      }
    }
    if (kt0 + 1 < kt1) {
      next_blocks();
      load_k(1);
      if constexpr (FP8) {
        put_k(1);
        if (scale_wave && w == 0) {
          load_scale(kt0 + 1);
          sh.ks[1][lane] = sraw;
        }
      }
    }
    if constexpr (!FP8) {
      wait_loads();
      zero_tail(kt0, 0);
    }
    __syncthreads();
    f32x16 sa[2], sb[2];
    scores(sa, 0, [](int) {});
    scale_scores(sa, 0);
    mask(sa, kt0);
    float mx = -INFINITY;
    quads(0, 1, [&](int g) { max_quad(mx, sa, g); });
    move_max(mx);
    __syncthreads();  // K buffer 0 is free

    // one tile: `cur_s` are its scores, b its buffers; the next tile's scores go to `next_s`
    auto step = [&](int tile, int b, f32x16 (&cur_s)[2], f32x16 (&next_s)[2]) {
      const bool more = tile + 2 < kt1;
      int vblk[CUR], voff[CUR];
#pragma unroll
      for (int c = 0; c < CUR; ++c) {
        vblk[c] = kblk[c];
        voff[c] = koff[c];
      }
      if (more) next_blocks();
      if constexpr (!FP8) load_v(b ^ 1, vblk, voff);
      if (more) load_k(b);
      if constexpr (kEarlyV) load_v(b ^ 1, vblk, voff);
      if (SM == 2 && (w == 1 || (w == 0 && more))) load_scale(tile + (w == 0 ? 2 : 1));
      uint32_t p[16];
      scores(next_s, b ^ 1, [&](int c) {
        quads(c, NQS, [&](int g) { weigh_quad(cur_s, p, g, b); });
      });
      if constexpr (FP8) {
        // (both buffers are free for the whole iteration)
        if (more) put_k(b);
        if constexpr (!kEarlyV) load_v(b ^ 1, vblk, voff);
      }
      scale_scores(next_s, b ^ 1);
      mask(next_s, tile + 1);
      float mx = -INFINITY;
      accumulate(p, b, [&](int n) {
        quads(n, 4 * ND, [&](int g) { max_quad(mx, next_s, g); });
      });
      move_max(mx);
      if constexpr (FP8) {
        put_v(tile + 1, b ^ 1);
        if (SM == 2 && w == 1) sh.vs[b ^ 1][lane] = sraw;
        if (SM == 2 && w == 0 && more) sh.ks[b][lane] = sraw;
      } else {
        wait_loads();
        zero_tail(tile + 1, b ^ 1);
      }
      __syncthreads();
    };
    auto last = [&](int b, f32x16 (&cur_s)[2]) {
      uint32_t p[16];
      quads(0, 1, [&](int g) { weigh_quad(cur_s, p, g, b); });
      accumulate(p, b, [](int) {});
    };
    // (one loop with one exit: leaving it between the two steps made the compiler copy
    // the accumulators)
    int tile = kt0;
    for (; tile + 2 < kt1; tile += 2) {
      step(tile, 0, sa, sb);
      step(tile + 1, 1, sb, sa);
    }
    if (tile + 1 < kt1) {
      step(tile, 0, sa, sb);
      last(1, sb);
    } else {
      last(0, sa);
    }
  }

  // ---- normalized output: lane holds dims 32 dt + 8 g + 4 h + [0, 4) of its row
  if (local >= rg_rows) return;
  const float inv = v_mul / fmaxf(half_sum(l_run), 1.0e-30f);
  const int64_t off = (int64_t)(sv.q_begin + qi) * P.out_row_stride + (int64_t)head * P.out_head_stride;
  uint16_t* op = (uint16_t*)P.out + off + 4 * h;
  // four dims per 8-byte store where the output's rows allow it
  const bool wide = (((uintptr_t)P.out % 8) | (uintptr_t)(P.out_row_stride % 4) |
                     (uintptr_t)(P.out_head_stride % 4)) == 0;
#pragma unroll
  for (int dt = 0; dt < ND; ++dt)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const f32x16& o = oacc[dt];
      const uint32_t x0 = M::pack2(o[4 * g] * inv, o[4 * g + 1] * inv);
      const uint32_t x1 = M::pack2(o[4 * g + 2] * inv, o[4 * g + 3] * inv);
      uint16_t* d = op + 32 * dt + 8 * g;
      if (wide) {
        *(uint2*)d = make_uint2(x0, x1);
      } else {
        d[0] = (uint16_t)x0;
        d[1] = (uint16_t)(x0 >> 16);
        d[2] = (uint16_t)x1;
        d[3] = (uint16_t)(x1 >> 16);
      }
    }
}
