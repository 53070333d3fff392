// The tiled kernel: many query rows of one KV head (prompt chunks, long verifications, large
// query groups) against K/V tiles shared through LDS.  Included by paged_decode.hip inside its
// anonymous namespace, after the split-grid kernel.

typedef __attribute__((ext_vector_type(16))) float f32x16;

// Waves per workgroup, WR of them over the query rows (32 rows each) and NW / WR over the keys,
// and the keys of one LDS tile.
template <int D>
constexpr int tile_waves() {
  return D == 256 ? 4 : 8;
}
constexpr int tile_keys_of(int64_t head_dim, int wr) { return head_dim == 256 || wr == 2 ? 32 : 64; }

// Largest batch ordered by length (MainShape::longest_first), and cut by its lengths (cut_tiles).
constexpr int kTileSortBatch = 512;
constexpr int kTileCutBatch = 1024;
constexpr int kTileMaxPieces = 32;      // pieces of the longest sequence
constexpr int kTileMinPieceKeys = 128;  // two tiles
constexpr float kTileStartUs = 5.f;     // start and end of a workgroup in the cut's model
// Word of the workspace's status region in which a cut launch leaves its tiles per piece for the
// combine kernel behind it.
constexpr int kTileCutWord = 8;

// One 16-byte LDS segment of a tile row from the 8 elements a lane loaded.
__device__ __forceinline__ u32x4 tile_segment(u32x4 x) { return x; }
__device__ __forceinline__ u32x4 tile_segment(u32x2 x) {
  return u32x4{fp8x2_to_bf16x2<false>(x[0]), fp8x2_to_bf16x2<true>(x[0]),
               fp8x2_to_bf16x2<false>(x[1]), fp8x2_to_bf16x2<true>(x[1])};
}

// The 8 bf16 elements of a new token's row as the cache will hold them: the values themselves, or
// (fp8 caches) the e4m3fn values nearest to x / scale.
template <bool kFp8>
__device__ __forceinline__ u32x4 stored_segment(u32x4 x, float scale) {
  if constexpr (kFp8)
    return tile_segment(
        u32x2{bf16x4_to_fp8x4(x[0], x[1], scale), bf16x4_to_fp8x4(x[2], x[3], scale)});
  return x;
}

// max / sum over the two lanes {l, l^32} that share one query row.
__device__ __forceinline__ float pair_max(float x) {
  auto a = __builtin_amdgcn_permlane32_swap(as_u32(x), as_u32(x), false, false);
  return fmaxf(as_float(a[0]), as_float(a[1]));
}
__device__ __forceinline__ float pair_sum(float x) {
  auto a = __builtin_amdgcn_permlane32_swap(as_u32(x), as_u32(x), false, false);
  return as_float(a[0]) + as_float(a[1]);
}

// Tiles of KB keys that row block [r0, r0 + nrows) of a sequence of `seq` keys sees.
__device__ __forceinline__ int block_tiles(int r0, int nrows, int seq, int kb,
                                           const MainShape& sh) {
  const int top = min(seq, row_key_limit(r0 + nrows - 1, seq, sh));
  return top > 0 ? (top + kb - 1) / kb : 0;
}

// Pieces of a sequence or row block of `tiles` tiles, at most `per` (inv = 1.0 / per) each.
__device__ __forceinline__ int tile_pieces(int tiles, int per, double inv) {
  return max(1, div_floor(tiles + per - 1, inv));
}

// Modelled time (us) of a launch of `count` workgroups over `slots` resident ones, the longest of
// which takes `longest` and all of which take `total`: rounds of the longest, or a list of unequal
// ones that ends at most one workgroup after the mean, whichever is less.
__device__ __forceinline__ float tile_launch_us(float count, float slots_inv, float longest,
                                                float total) {
  const float rounds = ceilf(count * slots_inv - 1e-3f);  // (a full round's product may exceed 1)
  return fminf(rounds * longest, total * slots_inv + longest);
}

// How a batch is cut (MainShape::cut_rows > 0), from its lengths alone and not from the capacity,
// which is the block table's width and often far beyond them: the longest sequence into n
// pieces, every other one into pieces of at most that many tiles, for the n of 1 .. kTileMaxPieces
// whose modelled time is shortest among those with at most cut_rows pieces in the batch and, if
// n > 1, at least kTileMinPieceKeys keys in one.  Grid row y is the batch's y-th piece.
struct TileCut {
  int b;      // sequence, or -1: the batch has no piece y
  int piece;  // of the sequence
  int per;    // tiles per piece
  int len;    // the sequence's seq_lens entry
};

// max / unsigned min over the 64 lanes of a wave (x >= 0), in every lane (cf. wave_inclusive_sum).
#define MX_WAVE_FOLD(OP, ID)                                                                    \
  x = OP(x, (decltype(x))__builtin_amdgcn_update_dpp(ID, (int)x, 0x111, 0xf, 0xf, false));      \
  x = OP(x, (decltype(x))__builtin_amdgcn_update_dpp(ID, (int)x, 0x112, 0xf, 0xf, false));      \
  x = OP(x, (decltype(x))__builtin_amdgcn_update_dpp(ID, (int)x, 0x114, 0xf, 0xf, false));      \
  x = OP(x, (decltype(x))__builtin_amdgcn_update_dpp(ID, (int)x, 0x118, 0xf, 0xf, false));      \
  x = OP(x, (decltype(x))__builtin_amdgcn_update_dpp(ID, (int)x, 0x142, 0xa, 0xf, false));      \
  x = OP(x, (decltype(x))__builtin_amdgcn_update_dpp(ID, (int)x, 0x143, 0xc, 0xf, false));      \
  return (decltype(x))__builtin_amdgcn_readlane((int)x, 63)
__device__ __forceinline__ int wave_max(int x) { MX_WAVE_FOLD(max, 0); }
__device__ __forceinline__ uint32_t wave_min(uint32_t x) { MX_WAVE_FOLD(min, -1); }
#undef MX_WAVE_FOLD

// Close enough to 1.0 / d for div_floor on tile counts (below 2^27): the reciprocal's approximation
// and one Newton step.
__device__ __forceinline__ double piece_inverse(int d) {
  const double r = __builtin_amdgcn_rcp((double)d);
  return r * (2.0 - d * r);
}

// Every thread of the workgroup calls it, for a batch of at most 64 * kEach: lane l of every wave
// holds the lengths of sequences l * kEach on.  The waves count the pieces of the batch for some n
// each (s_count: kTileMaxPieces words of LDS that the caller does not write before its next
// barrier), then every wave models all n, a lane each, and finds y by a prefix sum.
template <int NW, bool kAppend, int kEach>
__device__ __forceinline__ TileCut cut_tiles_of(const int32_t* __restrict__ seq_lens, int y, int kb,
                                                const MainShape& sh, uint32_t* s_count) {
  constexpr int G = kTileMaxPieces / NW;  // candidates per wave
  const int lane = threadIdx.x & 63;
  const int wv = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const int b0 = lane * kEach;
  int len[kEach], tiles[kEach];
#pragma unroll
  for (int i = 0; i < kEach; ++i) len[i] = seq_lens[min(b0 + i, sh.batch - 1)];
  int top = 0, sum = 0;
#pragma unroll
  for (int i = 0; i < kEach; ++i) {
    const int keys = seq_extent_of<kAppend>(len[i], sh, nullptr, false).keys;
    tiles[i] = keys > 0 && b0 + i < sh.batch ? (keys + kb - 1) / kb : 0;
    top = max(top, tiles[i]);
    sum += tiles[i];
  }
  top = wave_max(top);
  const float total = __builtin_amdgcn_readlane(wave_inclusive_sum(sum), 63);
  // Pieces of this lane's sequences, those of sequences in one piece in the low half.
  auto count = [&](int per, double inv) {
    uint32_t c = 0;
#pragma unroll
    for (int i = 0; i < kEach; ++i) {
      const int np = tile_pieces(tiles[i], per, inv);
      if (b0 + i < sh.batch) c += np > 1 ? (uint32_t)np << 16 : 1u;
    }
    return c;
  };
  const int n = lane % kTileMaxPieces + 1;  // this lane's candidate
  int per = max(1, div_floor(top + n - 1, piece_inverse(n)));
  uint32_t c;
  if (sh.batch == 1) {
    const int np = tile_pieces(top, per, piece_inverse(per));
    c = np > 1 ? (uint32_t)np << 16 : 1u;
  } else {
#pragma unroll
    for (int k = 0; k < G; ++k) {
      const int pk = __builtin_amdgcn_readlane(per, wv * G + k);
      const uint32_t sum_k = wave_inclusive_sum((int)count(pk, piece_inverse(pk)));
      if (lane == 63) s_count[wv * G + k] = sum_k;
    }
    __syncthreads();
    c = s_count[n - 1];
  }
  const float cut = c >> 16, pieces = cut + (c & 0xffff);
  const float wgs = gridDim.x;  // per piece
  const float us =
      tile_launch_us(pieces * wgs, sh.cut_slots_inv, per * sh.cut_tile_us + kTileStartUs,
                     (total * sh.cut_tile_us + pieces * kTileStartUs) * wgs) +
      (n > 1 ? cut * sh.cut_merge_us + sh.cut_fixed_us : 0.f);
  const bool ok = n == 1 || (pieces <= sh.cut_rows && top * kb >= n * kTileMinPieceKeys);
  // (Positive floats order as their bits do; n in the low ones, the least of equal times.)
  const uint32_t best =
      wave_min((as_u32(ok ? fmaxf(us, 0.f) : INFINITY) & ~(kTileMaxPieces - 1u)) +
               (uint32_t)(n - 1));
  per = __builtin_amdgcn_readlane(per, best % kTileMaxPieces);
  const double inv = piece_inverse(per);
  const uint32_t mine2 = count(per, inv);
  const int mine = (int)((mine2 >> 16) + (mine2 & 0xffff));
  const int first = wave_inclusive_sum(mine) - mine;
  const uint64_t holds = __builtin_amdgcn_ballot_w64(first <= y && y < first + mine);
  if (holds == 0) return TileCut{-1, 0, per, 0};
  int i0 = 0, piece = y - first, at = len[0];  // (in the lane that holds y)
#pragma unroll
  for (int i = 0; i + 1 < kEach; ++i) {
    const int np = tile_pieces(tiles[i], per, inv);
    if (i0 == i && piece >= np) {
      piece -= np;
      i0 = i + 1;
      at = len[i + 1];
    }
  }
  const int src = __builtin_ctzll(holds);
  return TileCut{__builtin_amdgcn_readlane(b0 + i0, src), __builtin_amdgcn_readlane(piece, src),
                 per, __builtin_amdgcn_readlane(at, src)};
}

// Bound by its chain of dependent steps, which every workgroup of a cut launch goes through before
// its first load of K: 1 to 2 us for up to 64 sequences, so few steps and no unused code in them (a
// loop over the lengths in LDS took 0.5 us more, and 2 more for 256 sequences).
template <int NW, bool kAppend>
__device__ __forceinline__ TileCut cut_tiles(const int32_t* __restrict__ seq_lens, int y, int kb,
                                             const MainShape& sh, uint32_t* s_count) {
  static_assert(kTileCutBatch == 64 * 16, "the widest form holds the largest batch");
  if (sh.batch <= 64) return cut_tiles_of<NW, kAppend, 1>(seq_lens, y, kb, sh, s_count);
  if (sh.batch <= 256) return cut_tiles_of<NW, kAppend, 4>(seq_lens, y, kb, sh, s_count);
  return cut_tiles_of<NW, kAppend, 16>(seq_lens, y, kb, sh, s_count);
}

// Partials of the tiled launch: one fp32 output row and log2-sum-exp per (query row, piece of its
// sequence).  Pieces of a fixed length: num_splits of every row side by side.  Pieces that follow
// the lengths: the batch's pieces one after another, each with its sequence's rows.
struct TileSlots {
  int64_t mul, add;  // slot of (row, piece): row * mul + add + piece * step
  int step;
  __device__ __forceinline__ int64_t at(int64_t row, int piece) const {
    return row * mul + add + (int64_t)piece * step;
  }
};
// `first`: the batch piece that is sequence b's piece 0.
__device__ __forceinline__ TileSlots tile_slots(int first, int b, const MainShape& sh) {
  if (sh.cut_rows == 0) return TileSlots{sh.num_splits, 0, 1};
  const int seq_rows = sh.seqlen_q * sh.num_heads;
  return TileSlots{1, (int64_t)(first - b) * seq_rows, seq_rows};
}

// The merge tree over the pieces of a row block (merge_tree).
template <int D>
struct TileTree {
  const MainShape& sh;
  float* part_o;
  float* part_lse;
  uint32_t* counters;
  uint16_t* out;
  int64_t rbase;  // row_base of the unit
  TileSlots slots;
  int kv;
  int r0;
  int unit;       // (sequence, KV head and row block) index
  __device__ __forceinline__ int64_t at(int hh, int slot) const {
    return slots.at(rbase + row_offset(kv, r0 + hh, sh), slot);
  }
  __device__ __forceinline__ float* o(int hh, int slot) const { return part_o + at(hh, slot) * D; }
  __device__ __forceinline__ float* lse(int hh, int slot) const { return part_lse + at(hh, slot); }
  __device__ __forceinline__ uint32_t* counter(int level, int slot) const {
    return counters + (int64_t)level * kMaxSlots + (int64_t)unit * sh.split_groups +
           slot / kMergeFanIn;
  }
  __device__ __forceinline__ int lse_step() const { return slots.step; }
  __device__ __forceinline__ int o_step() const { return slots.step * D; }
  __device__ __forceinline__ void store(int hh, int d, f32x4 v, float l) const {
    store_row4<D>(out, sh, rbase + row_offset(kv, r0 + hh, sh), d, v, l);
  }
};

// Grid (KV heads * row blocks, batch), or (KV heads * row blocks, cut_rows) where the batch is cut
// into pieces by its lengths (cut_tiles); see plan_tiled for the shape.  A workgroup holds 32*WR
// query rows of one (sequence, KV head) and streams one piece of their keys in tiles of KB.
//
// What bounds it: with many rows per head the work is two matrix products, 4 * D flop per row and
// key, so K and V are read once per 32*WR rows (the streaming kernels: per 16 or 32) and shared
// through LDS.  A 4 096-token prompt (Hq=32, Hkv=8, D=128) takes 154 us as a whole call without an
// append, 892 TFLOP/s, where a large library product reaches 1 240-1 360 on the same card; the
// streaming kernels ran it at 135.  The matrix cores are busy 37 % of the cycles.  Per tile of 64
// keys a wave issues 32 MFMAs (1 024 cycles) and 180 other VALU instructions, LDS serves 8 waves
// x 32 KB at up to 256 bytes per cycle, and two waves per SIMD (200-230 registers at head_dim
// 128, no scratch) cover each other's softmax and waits.
//
//  * QK is S^T = K . Q^T in 32x32x16 MFMAs: the result leaves lane (row r32, half hi) the scores of
//    keys 4*hi + {0..3, 8..11, 16..19, 24..27} of its own query row, so the row maximum is 31
//    in-lane steps (15 in tiles of 32 keys) and one lane swap.
//  * PV is O^T = V^T . P^T with P straight from those registers: the contraction's key order is free,
//    so V^T is read in the order P has (ds_read_b64_tr_b16 transposes 4 keys x 16 dims per 16
//    lanes), and P never moves.  Both operands are rounded exactly as in the streaming kernels.
//  * Tiles are double-buffered: the next tile's global loads are issued before a tile's math and
//    stored to the other LDS buffer after it, with one barrier per tile.
//  * The NW / WR key groups of a workgroup stream alternate tiles of the piece with buffers of their
//    own and merge their states through LDS at the end.
//  * Masked tiles (causal limits, the sequence's end) take selects on the scores; rows past the
//    sequence's end are stored to LDS as zero V.  A wave skips tiles past its rows' last key.
//  * One code path for masked and full tiles: instantiated twice, the compiler hoisted both tiles'
//    operands and spilled (head_dim 128: 276 bytes per lane, 2.3 times slower).

template <int D, int WR, bool kFp8, bool kAppend>
__global__ __launch_bounds__(64 * tile_waves<D>())
__attribute__((amdgpu_waves_per_eu(D == 256 ? 1 : D == 64 && WR == 2 ? 4 : 2)))
void mx_paged_attend_tiled(
    const uint16_t* __restrict__ q, CachePtr<kAppend, CacheElem<kFp8>> kc,
    CachePtr<kAppend, CacheElem<kFp8>> vc, uint16_t* __restrict__ out,
    const int32_t* __restrict__ seq_lens, const int32_t* __restrict__ block_table,
    float* __restrict__ part_o, float* __restrict__ part_lse, uint32_t* __restrict__ counters,
    uint32_t* __restrict__ status, const MainShape sh) {
  constexpr int NW = tile_waves<D>();
  constexpr int WK = NW / WR;             // key groups: each streams every WK-th tile
  constexpr int KB = tile_keys_of(D, WR);
  constexpr int RB = 32 * WR;             // query rows per workgroup
  constexpr int NKB = KB / 32;            // 32-key blocks per tile
  constexpr int SPR = D / 8;              // 8-element segments per token row
  constexpr int RPI = 64 / SPR;           // token rows per load instruction of a wave
  constexpr int RPW = KB / WR;            // token rows per wave (at most one 16-token chunk)
  constexpr int IPW = RPW / RPI;          // load instructions per wave and tile (K, and V)
  constexpr int kTile = KB * 2 * D;       // bytes of one K or V tile
  static_assert(RPW <= kChunk && RPW % RPI == 0 && IPW >= 1, "a wave loads whole rows of a chunk");
  using LoadT = std::conditional_t<kFp8, u32x2, u32x4>;
  __shared__ __attribute__((aligned(16))) char lds[WK * 4 * kTile];  // K and V, two buffers
  __shared__ float s_lse[RB];
  __shared__ int s_last;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int r32 = lane & 31;
  const int hi = lane >> 5;
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wr = wv % WR;  // row wave: rows 32 * wr ..
  const int wk = wv / WR;  // key group
  // KV heads vary fastest, so the row blocks of a head land on the same XCDs; the last rows
  // first: under a causal mask they have the most keys.
  const int kv = blockIdx.x % sh.num_kv_heads;
  const int blk = sh.row_tiles - 1 - (int)blockIdx.x / sh.num_kv_heads;
  int b = blockIdx.y;
  // (Compiled into the 64-row blocks only: in the wider ones the code, even switched off, cost
  // prompts 1 % and head_dim 256 chunks 4 %.)
  if constexpr (WR == 2) {
    if (sh.longest_first) {
      // Workgroups start in grid order: grid row y takes the y-th longest sequence (ties by index),
      // so the last ones to start are the shortest.  Every workgroup ranks the whole batch.
      int* s_len = reinterpret_cast<int*>(lds);
      for (int i = tid; i < kTileSortBatch; i += 64 * NW)
        s_len[i] = i < sh.batch ? key_count(seq_lens, i, sh.appended) : INT_MIN;
      __syncthreads();
      for (int i = tid; i < sh.batch; i += 64 * NW) {
        const int mine = s_len[i];
        int before = 0;
        for (int j = 0; j < sh.batch; j += 4)
  #pragma unroll
          for (int e = 0; e < 4; ++e) {
            const int other = s_len[j + e];
            before += other > mine || (other == mine && j + e < i);
          }
        if (before == (int)blockIdx.y) s_last = i;
      }
      __syncthreads();
      b = __builtin_amdgcn_readfirstlane(s_last);
    }
  }
  const int r0 = blk * RB;
  const int nrows = min(RB, sh.rows - r0);
  int piece = blockIdx.z, per = sh.tokens_per_split / KB, len;
  int first = 0;  // batch piece of the sequence's piece 0
  if (sh.cut_rows > 0) {
    const TileCut cut =
        cut_tiles<NW, kAppend>(seq_lens, b, KB, sh, reinterpret_cast<uint32_t*>(s_lse));
    if (blockIdx.x == 0 && b == 0 && tid == 0) status[kTileCutWord] = cut.per;
    if (cut.b < 0) return;
    piece = cut.piece;
    per = cut.per;
    len = cut.len;
    first = b - piece;
    b = cut.b;
    __syncthreads();  // (s_lse)
  } else {
    len = seq_lens[b];
  }

  const SeqExtent ext = seq_extent_of<kAppend>(len, sh, status,
                                               piece == 0 && blockIdx.x == 0 && tid == 0);
  const int seq = ext.keys;
  const int nt = block_tiles(r0, nrows, seq, KB, sh);
  int np = tile_pieces(nt, per, piece_inverse(per));
  if (sh.cut_rows == 0) np = min(np, sh.num_splits);
  if (piece >= np) return;
  const int64_t rbase = row_base(b, kv, sh);
  if (nt == 0) {
    for (int e = tid; e < nrows * (D / 4); e += 64 * NW)
      store_row4<D>(out, sh, rbase + row_offset(kv, r0 + e / (D / 4), sh), 4 * (e % (D / 4)),
                    f32x4{0.f, 0.f, 0.f, 0.f}, -INFINITY);
    return;
  }
  const int t_lo = __builtin_amdgcn_readfirstlane((int)((int64_t)nt * piece / np));
  const int t_hi = __builtin_amdgcn_readfirstlane((int)((int64_t)nt * (piece + 1) / np));

  // Query operand (B of the QK MFMA): this lane's row, dims 16*i + 8*hi .. +7.
  const int r = r0 + wr * 32 + r32;
  const bool live = r < sh.rows;
  const uint16_t* qp = q + (rbase + row_offset(kv, live ? r : 0, sh)) * D + 8 * hi;
  bf16x8 qop[D / 16];
  // The running max is taken over raw scores, so a negative scale moves its sign into q.
  const float sc = fabsf(sh.scale_log2);
  const uint32_t flip = sh.scale_log2 < 0.f ? 0x80008000u : 0u;
#pragma unroll
  for (int i = 0; i < D / 16; ++i) {
    u32x4 x = {0, 0, 0, 0};
    if (live) x = *reinterpret_cast<const u32x4*>(qp + 16 * i);
    qop[i] = __builtin_bit_cast(bf16x8, x ^ flip);
  }
  const int lim = min(seq, row_key_limit(r, seq, sh));  // keys this lane's row sees
  // Fewest and most keys of the wave's rows.
  const int rw = r0 + wr * 32;
  const int w_lo = __builtin_amdgcn_readfirstlane(min(seq, row_key_limit(rw, seq, sh)));
  const int w_top = __builtin_amdgcn_readfirstlane(
      rw < sh.rows ? min(seq, row_key_limit(rw + 31, seq, sh)) : 0);

  f32x16 o[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i)
#pragma unroll
    for (int j = 0; j < 16; ++j) o[i][j] = 0.f;
  float m = kNoScore;
  float l = 0.f;

  // Tile loads: row wave wr loads rows wr*RPW .. of the tile, one 16-byte (fp8: 8-byte) piece of a
  // row per lane.
  const int32_t* bt_row = block_table + (int64_t)b * sh.max_pages;
  const int c_top = max((ext.cache + kChunk - 1) / kChunk - 1, 0);
  const int chunk_mask = (1 << sh.chunk_shift) - 1;
  const int row_w = wr * RPW;  // first tile row of this wave
  bool bad_page = false;
  auto tile_base = [&](int t) -> int64_t {
    const int c = min(t * (KB / kChunk) + row_w / kChunk, c_top);
    int pid = scalar_load(bt_row + (c >> sh.chunk_shift));
    if (pid < 0 || (sh.num_pages > 0 && pid >= sh.num_pages)) {
      bad_page = true;
      pid = 0;
    }
    return (int64_t)pid * sh.page_stride +
           (int64_t)((c & chunk_mask) * kChunk + row_w % kChunk) * sh.token_stride + kv * D;
  };
  const uint32_t lane_off = (uint32_t)(lane / SPR) * sh.token_stride + 8u * (lane % SPR);
  LoadT kreg[IPW], vreg[IPW];
  const uint16_t* const k_new = sh.k_new;
  const uint16_t* const v_new = sh.v_new;
  auto load_tile = [&](int64_t base, int t) {
    // Fused append (bf16): positions from ext.cache on are the new tokens' rows.  (The branch is
    // uniform and its addresses are per lane.)
    const bool with_new = kAppend && !kFp8 && (t + 1) * KB > ext.cache;
    const int64_t head0 = (int64_t)b * sh.new_tokens * sh.token_stride + kv * D + 8 * (lane % SPR);
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const CacheElem<kFp8>* kp = kc + base + lane_off + i * RPI * sh.token_stride;
      const CacheElem<kFp8>* vp = vc + base + lane_off + i * RPI * sh.token_stride;
      if constexpr (kAppend && !kFp8) {
        if (with_new) {
          const int j = t * KB + row_w + i * RPI + lane / SPR - ext.cache;
          const int64_t at = head0 + (int64_t)min(j, sh.new_tokens - 1) * sh.token_stride;
          if (j >= 0) {
            kp = k_new + at;
            vp = v_new + at;
          }
        }
      }
      kreg[i] = *reinterpret_cast<const LoadT*>(kp);
      vreg[i] = *reinterpret_cast<const LoadT*>(vp);
    }
  };
  // LDS layout: row-major [KB][D] with the 16-byte segments of a row permuted.  K: segment s of
  // row r at s ^ k_swizzle(r), free of conflicts for the 32 rows x 2 segments of an operand
  // read; V: 64-byte groups permuted by the row, free of conflicts for the 4 rows x 64 bytes a
  // transposing read takes.
  auto v_swizzle = [](int row) { return D == 64 ? ((row >> 1) & 1) : (row & 3); };
  auto store_tile = [&](int buf, int t) {
    char* kb = lds + (wk * 2 + buf) * 2 * kTile;
    char* vb = kb + kTile;
    const bool tail = (t + 1) * KB > seq;
#pragma unroll
    for (int i = 0; i < IPW; ++i) {
      const int row = row_w + i * RPI + lane / SPR;
      const int s = lane % SPR;
      u32x4 kx = tile_segment(kreg[i]);
      u32x4 vx = tile_segment(vreg[i]);
      if constexpr (kAppend && kFp8) {
        // (Loaded here: an fp8 tile's load registers do not hold bf16 rows.)
        const int j = t * KB + row - ext.cache;
        if (j >= 0 && j < sh.new_tokens) {
          const int64_t at = ((int64_t)b * sh.new_tokens + j) * sh.token_stride + kv * D + 8 * s;
          kx = stored_segment<kFp8>(*reinterpret_cast<const u32x4*>(k_new + at), sh.k_scale);
          vx = stored_segment<kFp8>(*reinterpret_cast<const u32x4*>(v_new + at), sh.v_scale);
        }
      }
      if (tail && t * KB + row >= seq) vx = u32x4{0, 0, 0, 0};  // unused slots may hold NaN
      *reinterpret_cast<u32x4*>(kb + row * 2 * D + 16 * (s ^ k_swizzle<D>(row))) = kx;
      *reinterpret_cast<u32x4*>(vb + row * 2 * D + 16 * (s ^ (v_swizzle(row) << 2))) = vx;
    }
  };

  int k_off[D / 16];
#pragma unroll
  for (int i = 0; i < D / 16; ++i)
    k_off[i] = r32 * 2 * D + 16 * ((2 * i + hi) ^ k_swizzle<D>(r32));
  int v_off[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    const int vr = 4 * hi + ((lane & 15) >> 2);
    v_off[i] = kTile + vr * 2 * D + 64 * (i ^ v_swizzle(vr)) + 32 * ((lane >> 4) & 1) +
               8 * (lane & 3);
  }

  auto compute = [&](int buf, int t) {
    const char* base = lds + (wk * 2 + buf) * 2 * kTile;
    f32x16 s[NKB];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int j = 0; j < 16; ++j) s[kb][j] = 0.f;
#pragma unroll
    for (int i = 0; i < D / 16; ++i)
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb) {
        const bf16x8 a = __builtin_bit_cast(
            bf16x8, *reinterpret_cast<const u32x4*>(base + k_off[i] + kb * 32 * 2 * D));
        s[kb] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, qop[i], s[kb], 0, 0, 0);
      }
    if ((t + 1) * KB > w_lo) {  // some row of the wave does not see the whole tile
      const int left = lim - t * KB - 4 * hi;  // keys of the tile this lane's row sees
#pragma unroll
      for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
        for (int j = 0; j < 16; ++j)
          if (32 * kb + (j & 3) + 8 * (j >> 2) >= left) s[kb][j] = -INFINITY;
    }
    float cm = s[0][0];
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int j = 0; j < 16; ++j) cm = fmaxf(cm, s[kb][j]);
    cm = pair_max(cm) * sc;
    if (__builtin_amdgcn_ballot_w64(cm > m + kRescaleSlack)) {
      const float mn = fmaxf(m, cm);
      const float alpha = __builtin_amdgcn_exp2f(m - mn);
      m = mn;
      l *= alpha;
#pragma unroll
      for (int i = 0; i < D / 32; ++i) o[i] *= alpha;
    }
    bf16x8 pop[NKB][2];
    float ls[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32x4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float p0 = __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][8 * h + 2 * j], sc, -m));
          const float p1 =
              __builtin_amdgcn_exp2f(__builtin_fmaf(s[kb][8 * h + 2 * j + 1], sc, -m));
          ls[j] += p0 + p1;
          w[j] = pack_bf16x2(p0, p1);
        }
        pop[kb][h] = __builtin_bit_cast(bf16x8, w);
      }
    l += (ls[0] + ls[1]) + (ls[2] + ls[3]);
#pragma unroll
    for (int kb = 0; kb < NKB; ++kb)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < D / 32; ++i) {
          typedef __attribute__((address_space(3))) s16x4* LdsP;
          const char* p = base + v_off[i] + (32 * kb + 16 * h) * 2 * D;
          const s16x4 x = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsP)(p));
          const s16x4 y = __builtin_amdgcn_ds_read_tr16_b64_v4i16((LdsP)(p + 8 * 2 * D));
          const bf16x8 a = __builtin_bit_cast(
              bf16x8, __builtin_shufflevector(x, y, 0, 1, 2, 3, 4, 5, 6, 7));
          o[i] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, pop[kb][h], o[i], 0, 0, 0);
        }
  };

  // Key group wk takes tiles t_lo + wk, + WK, ...; every wave runs the same number of steps (a
  // tile past the piece is loaded, clamped to the sequence, and not computed).
  const int steps = (t_hi - t_lo + WK - 1) / WK;
  int t = t_lo + wk;
  load_tile(tile_base(t), t);
  if constexpr (kAppend) {
    // One workgroup per (sequence, KV head) writes the new tokens to the cache: that of the last row
    // block, whose last row sees every key (so it never returned above).  No slot written is used
    // by this launch (cache rows of a tile are used below ext.cache only).
    if (blk == sh.row_tiles - 1 && piece == 0)
      copy_new_tokens<D, kFp8>(seq_lens, block_table, b, kv, sh, status, tid, 64 * NW);
  }
  int64_t next = tile_base(t + WK);
  store_tile(0, t);
  __syncthreads();
  for (int i = 0; i < steps; ++i, t += WK) {
    const bool more = i + 1 < steps;
    if (more) {
      load_tile(next, t + WK);
      next = tile_base(t + 2 * WK);
    }
    if (t * KB < w_top && (WK == 1 || t < t_hi)) compute(i & 1, t);
    if (more) store_tile((i & 1) ^ 1, t + WK);
    __syncthreads();
  }
  if (bad_page && lane == 0) atomicOr(status, (uint32_t)MX_DEVICE_BAD_PAGE_ID);

  l = pair_sum(l);
  if constexpr (WK > 1) {
    // The key groups' states of a row wave have the same lane layout: groups 1.. leave theirs in
    // LDS (the K/V tiles are dead after the last barrier) and group 0 merges them.
    constexpr int kState = 64 * (D / 2 + 2) * 4;  // bytes of a wave's state
    static_assert((NW - WR) * kState <= (int)sizeof(lds), "merge states fit the tiles' LDS");
    if (wk > 0) {
      float* st = reinterpret_cast<float*>(lds + ((wk - 1) * WR + wr) * kState);
#pragma unroll
      for (int i = 0; i < D / 32; ++i)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<f32x4*>(st + ((i * 4 + g) * 64 + lane) * 4) =
              f32x4{o[i][4 * g], o[i][4 * g + 1], o[i][4 * g + 2], o[i][4 * g + 3]};
      st[32 * D + lane] = m;
      st[32 * D + 64 + lane] = l;
    }
    __syncthreads();
    if (wk == 0) {
      float mx = m;
#pragma unroll
      for (int k = 1; k < WK; ++k)
        mx = fmaxf(mx, reinterpret_cast<const float*>(lds + ((k - 1) * WR + wr) *
                                                                kState)[32 * D + lane]);
      const float a0 = __builtin_amdgcn_exp2f(m - mx);
      l *= a0;
#pragma unroll
      for (int i = 0; i < D / 32; ++i) o[i] *= a0;
      for (int k = 1; k < WK; ++k) {
        const float* st =
            reinterpret_cast<const float*>(lds + ((k - 1) * WR + wr) * kState);
        const float a = __builtin_amdgcn_exp2f(st[32 * D + lane] - mx);
        l += a * st[32 * D + 64 + lane];
#pragma unroll
        for (int i = 0; i < D / 32; ++i)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 x = *reinterpret_cast<const f32x4*>(st + ((i * 4 + g) * 64 + lane) * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) o[i][4 * g + j] += a * x[j];
          }
      }
      m = mx;
    }
  }
  const bool seen = l > 0.f;
  float inv = seen ? 1.0f / l : 0.f;
  if constexpr (kFp8) inv *= sh.v_scale;
  const float lse = seen ? m + log2f(l) : -INFINITY;
  const int64_t row = rbase + row_offset(kv, live ? r : 0, sh);
  const TileSlots slots = tile_slots(first, b, sh);
  const int64_t prow = slots.at(row, piece);
  if (live && wk == 0) {
#pragma unroll
    for (int i = 0; i < D / 32; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int d = 32 * i + 8 * g + 4 * hi;
        const f32x4 v = f32x4{o[i][4 * g], o[i][4 * g + 1], o[i][4 * g + 2], o[i][4 * g + 3]} * inv;
        if (np == 1)
          store_row4<D>(out, sh, row, d, v, lse);
        else if (sh.fused_combine)
          store_partial4(part_o, part_o + prow * D + d, v);
        else
          *reinterpret_cast<f32x4*>(part_o + prow * D + d) = v;
      }
    if (np > 1 && hi == 0) {
      if (sh.fused_combine)
        store_partial1(part_lse + prow, lse);
      else
        part_lse[prow] = lse;
    }
  }
  if (np == 1 || !sh.fused_combine) return;
  const TileTree<D> tree{sh, part_o, part_lse, counters, out, rbase, slots, kv, r0,
                         b * (int)gridDim.x + (int)blockIdx.x};
  merge_tree<D, NW, kMergeFanIn>(tree, piece, np, nrows, s_lse, &s_last);
}
