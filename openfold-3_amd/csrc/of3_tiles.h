// Tiling of the N x N positions of a batch element into tiles of TP (128, or 64) positions for the position-wise passes.
// Plain C++ (no HIP types): the kernels and the host-side test of the scheme compile the same functions.
#pragma once

#if defined(__HIPCC__)
#define OF3_HD __host__ __device__
#else
#define OF3_HD
#endif

namespace of3 {

// The whole TP-wide pieces of every row come first (full_per_row per row), then the remaining N % TP
// columns in pieces of 2^s columns x (TP >> s) consecutive rows, 2^s >= 2^min_shift: one power of two that covers them, or two
// (72 columns: 64 + 8) where that makes fewer tiles.  tail_shift: s of the first piece + 256 * s of the second, 0 if there is
// none.  N = 200 takes 313 tiles of 128 with two and 400 with one.
struct RaggedTiles {
  int full_per_row, tail_shift, per_batch;
};
template <int TP = 128>
OF3_HD inline int tiles_of_columns(int N, int shift) {  // tiles of N rows x 2^shift columns
  const int rows = TP >> shift;
  return (N + rows - 1) / rows;
}
template <int TP = 128>
inline RaggedTiles ragged_tiles(int N, int min_shift = 3) {
  RaggedTiles t;
  t.full_per_row = N / TP;
  const int r = N % TP;
  t.tail_shift = r ? min_shift : TP == 128 ? 7 : 6;
  while ((1 << t.tail_shift) < r) ++t.tail_shift;
  int tail = r ? tiles_of_columns<TP>(N, t.tail_shift) : 0;
  const int s1 = t.tail_shift - 1;
  if (r && s1 >= min_shift) {
    int s2 = min_shift;
    while ((1 << s1) + (1 << s2) < r) ++s2;
    const int two = tiles_of_columns<TP>(N, s1) + tiles_of_columns<TP>(N, s2);
    if (two < tail) tail = two, t.tail_shift = s1 + 256 * s2;
  }
  t.per_batch = N * t.full_per_row + tail;
  return t;
}

// Where a tile lies: batch element, first row, first column, log2 of its width.  Position pos (0..TP - 1) of
// the tile is row i0 + (pos >> shift), column j0 + (pos & ((1 << shift) - 1)).
struct TilePlace {
  int b, i0, j0, shift;
};
// RAGGED = false: whole-row pieces only (full_per_row pieces per row, per_batch = rows * full_per_row).
// keep_rows_inside: the last piece of some ragged columns is moved up so that it ends at row N - 1 (its rows
// all exist, some of them belong to the piece before it as well; needs N >= TP >> tail_shift); otherwise it
// runs past the last row and the caller leaves those positions out.
template <bool RAGGED, int TP = 128>
OF3_HD inline TilePlace tile_place(int tile_id, int N, int full_per_row, int tail_shift, int per_batch,
                                   bool keep_rows_inside) {
  TilePlace t;
  t.b = tile_id / per_batch;
  const int rem = tile_id - t.b * per_batch;
  const int main_tiles = N * full_per_row;
  if (!RAGGED || rem < main_tiles) {
    t.i0 = rem / full_per_row;
    t.j0 = (rem - t.i0 * full_per_row) * TP;
    t.shift = TP == 128 ? 7 : 6;
  } else {
    int at = rem - main_tiles;
    t.shift = tail_shift & 255;
    t.j0 = full_per_row * TP;
    const int first = tiles_of_columns<TP>(N, t.shift);
    if (at >= first) {
      at -= first;
      t.j0 += 1 << t.shift;
      t.shift = tail_shift >> 8;
    }
    const int rows = TP >> t.shift;
    t.i0 = at * rows;
    if (keep_rows_inside && t.i0 + rows > N) t.i0 = N - rows;
  }
  return t;
}

// ---- tiles of TP consecutive positions of the flattened [B][N][N] index space (triattn_out) ------------
// A tile starts at position p0 = TP * tile_id = (b0, i0, j0).  MODE 0: N is a multiple of TP, a tile lies
// inside one row; 1: N >= TP, at most two rows, whose element offsets in the strided view are row0 and row1;
// 2: any N, the general walk.
struct FlatTile {
  int b0, i0, j0;
  long long row0, row1;
};
template <int TP = 128>
OF3_HD inline FlatTile flat_tile(int tile_id, int N, long long stride_b, long long stride_r) {
  FlatTile t;
  const unsigned p0 = (unsigned)tile_id * (unsigned)TP, nn = (unsigned)N * (unsigned)N;
  t.b0 = (int)(p0 / nn);
  const unsigned rem = p0 - (unsigned)t.b0 * nn;
  t.i0 = (int)(rem / (unsigned)N);
  t.j0 = (int)(rem - (unsigned)t.i0 * (unsigned)N);
  const bool last = t.i0 + 1 == N;
  t.row0 = t.b0 * stride_b + t.i0 * stride_r;
  t.row1 = (t.b0 + (last ? 1 : 0)) * stride_b + (last ? 0 : t.i0 + 1) * stride_r;
  return t;
}
// element offset of position d (0..TP - 1) of the tile in the view; the position must exist
template <int MODE>
OF3_HD inline long long flat_offset(const FlatTile& t, int d, int N, long long stride_b, long long stride_r,
                                    long long stride_k) {
  int j = t.j0 + d;
  if (MODE == 0) {
    return t.row0 + j * stride_k;
  } else if (MODE == 1) {
    const bool wrapped = j >= N;
    j -= wrapped ? N : 0;
    return (wrapped ? t.row1 : t.row0) + j * stride_k;
  } else {
    int b = t.b0, i = t.i0;
    while (j >= N) j -= N, ++i;  // at most once when N >= TP
    while (i >= N) i -= N, ++b;
    return b * stride_b + i * stride_r + j * stride_k;
  }
}

// ---- the last round of a persistent pass ----------------------------------------------------------------
// `tiles` tiles of TP = 128 positions on `grid` work-groups: the tiles that are left for a last round of their own, if
// there are no more than half (a quarter) as many as work-groups, go in two (four) pieces of 64 (32) positions each (tiles of 64 in halves only), one
// piece per work-group: that round then takes as long as its piece, not as a tile.  Items 0 .. whole - 1 are
// whole tiles, the rest pieces; whole is a multiple of grid where there are pieces.  256 CUs, 128 channels, us per pass, whole
// tiles / pieces: triangle multiplication in at N = 128 (half a round) 11.2 / 9.0, at 200 (1.37 rounds) 15.8 / 14.5, attention in
// 12.9 / 11.8 and 17.8 / 16.4, attention out at 200 14.0 / 12.0.  From three rounds on the kernels with pieces, which hold
// more registers and address their loads at run time, lose what the last round gains: N = 384 (4.5 rounds) the same, 929 167.7 / 171.4.
struct LastRound {
  int whole, items, piece;
};
template <int TP = 128>
inline LastRound last_round(long tiles, int grid) {
  const int left = (int)(tiles % grid);
  LastRound r = {(int)tiles, (int)tiles, TP};
  if (left == 0 || 2 * left > grid || tiles >= 3L * grid) return r;
  const int split = TP == 128 && 4 * left <= grid ? 4 : 2;
  r.piece = TP / split;
  r.whole = (int)(tiles - left);
  r.items = r.whole + split * left;
  return r;
}

// Positions of a tile of the triangle multiplication's output pass (planes: it reads x, channel by channel) and of the attention's: tiles of
// 64 on work-groups of four waves, or of 128 on eight.  A wave does the same either way; where the smaller work-groups share a CU (two at
// 128 channels, three at 64 in the multiplication's pass) their barriers, three a tile, do not coincide.  128 / 64 positions, us a launch of
// the multiplication's pass at 128 channels: N = 300 24.7 / 22.9, 384 35.0 / 32.0, 451 52.8 / 47.8, 768 118 / 116, 850 157 / 148, 1100 236 / 226, 1700
// 546 / 536; at 64, three templates of 300 30.8 / 25.8, four of 512 95.0 / 86.9.  Of the attention's at 128: N = 300 21.5 / 21.4, 384 31.9 /
// 28.5, 640 79.8 / 75.1, 896 148 / 143, 1280 275 / 269; at 64 its launch does not ask: two work-groups of eight waves share a CU there, 42.4 / 42.7 for two of 512.
// Launches by themselves of the attention's off multiples of 64 between 500 and 740 tokens prefer 128 (540 52.0 / 54.3, 600 61.4 / 64.6, 720 85.9 / 89.3), whole
// passes do not: pair stack 540 963 / 961, 600 1209 / 1201, 720 1741 / 1736, and 257 261 / 255, 580 1173 / 1157, 1000 3702 / 3707.
// Beyond 1536 tokens the attention's lose (1536 401 / 402, 1792 528 / 546, 2048 708 / 742: more rows open in memory at once).  The multiplication's go
// either way there (128 channels 1600 462 / 450, 1700 521 / 522, 1792 564 / 571, others within 1 %; 64 channels 1600 221 / 202, 1700 250 / 240, 1792 263 / 273, 1920 302 / 314)
// and keep to the same line.  x loses at whole multiples of 1024, where the 128-byte pieces of a tile's planes are a power of two apart (929 170 /
// 173, 1024 203 / 211, 2048 779 / 814).
inline int out_tile_positions(int N, bool planes) {
  if (N > 1536) return 128;
  return planes && (N + 127) / 128 % 8 == 0 ? 128 : 64;
}

// ---- the bf16 attention core's work-groups (triattn_flash.hip) --------------------------------------------
constexpr int kFlashRows = 4;
// work-groups to a CU by the queries of their range
constexpr int flash_groups_per_cu(int D, int queries) { return D == 32 ? (queries == 64 ? 4 : queries == 96 ? 3 : 2) : (queries == 128 ? 3 : 4); }
// Queries of a work-group's range, 64, 96 or 128: the form with the least estimated time, its rounds (work-groups over places on the chip)
// times a round's time in that form.  What is left for a last round is dealt to the CUs one by one, so that round takes as long as the CU with the
// most of them, k of its places: `alone` of a round for the first, and the rest of it in equal steps for the others.  Rounds' times and `alone` were
// fitted to whole passes, 238 of them in each form (launches by themselves favour the larger forms: one after another they run at a lower clock): the form taken costs a
// pass 0.06 % (heads of 32) and 0.12 % (16) against the best on average, 1.3 % at most; with a last round in proportion to what is left, 0.42 and 0.19 % on
// average, 3.6 % at most.  us a pass, 64 / 96 / 128 queries (256 CUs): pair stack 257 tokens 239 / 243 / 244, 345 350 / 350 / 356, 453 635 / 620 / 632, 512 764 /
// 760 / 751, 700 1657 / 1606 / 1629, 768 1953 / 1888 / 1886, 969 3571 / 3525 / 3474, two tensors of 221 279 / 287 / 286; templates 3 x 228 546 / 550 /
// 553, 3 x 294 852 / 864 / 853, 4 x 404 2309 / 2241 / 2251, 4 x 503 3600 / 3519 / 3491.
inline int flash_queries(int N, long slices, int D, int cus) {  // slices: batch elements times heads
  struct Form {
    int queries;
    double round, alone;
  };
  const Form forms[2][3] = {{{64, 0.71, 0.24}, {96, 1.08, 0.0}, {128, 1.0, 0.17}}, {{64, 1.1, 0.0}, {96, 1.15, 0.2}, {128, 1.0, 0.45}}};
  auto groups = [&](int queries) { return (long)((N + queries - 1) / queries) * ((N + kFlashRows - 1) / kFlashRows) * slices; };
  // up to three work-groups of 64 queries per CU nothing else has enough of them (heads of 32, N = 128: 6.3 against 8.0 for 128; heads of 16, 1 x 150: 8.7 and
  // 10.0 for 96); beyond four rounds of them, which read every K and V^T tile the most times, they were behind but
  // for three templates of 294 to 316, by 0.1 to 1 % of a pass
  const long small = groups(64), places64 = (long)flash_groups_per_cu(D, 64) * cus;
  if (small <= 3L * cus) return 64;
  int best = 0;
  double least = 0;
  for (const Form& f : forms[D == 32]) {
    if (f.queries == 64 && small > 4 * places64) continue;
    const int per_cu = flash_groups_per_cu(D, f.queries);
    const long places = (long)per_cu * cus, items = groups(f.queries), left = items % places, k = (left + cus - 1) / cus;
    const double t = f.round * ((double)(items / places) + (left ? f.alone + (1 - f.alone) * (double)k / per_cu : 0.0));
    if (!best || t < least) best = f.queries, least = t;
  }
  return best;
}

// Item of a persistent pass -> its tile, its first position in it, how many positions it has (group_bits: log2 of the
// groups of eight).  PART: positions per piece, TP: no pieces.
struct TilePiece {
  int tile, first, count, group_bits;
};
template <int PART, int TP = 128>
OF3_HD inline TilePiece tile_piece(int item, int whole) {
  if (PART == TP || item < whole) return {item, 0, TP, TP == 128 ? 4 : 3};
  const int split = TP / PART, left = item - whole;
  return {whole + left / split, left % split * PART, PART, PART == 64 ? 3 : 2};
}

// ---- order of the attention core's work-groups -----------------------------------------------------------
// Work items of one (batch element, head) are (query range qc < n_qc, row group rg < n_rg).  They are taken in
// blocks of RB row groups x QB query ranges; inside a block the query range runs fastest, then the row group.
struct FlashItem {
  int bh, qc, rg;
};
OF3_HD inline FlashItem flash_item(int logical, int n_qc, int n_rg, int RB, int QB) {
  FlashItem w;
  const int per_bh = n_qc * n_rg;
  w.bh = logical / per_bh;
  const int idx = logical - w.bh * per_bh;
  const int rb = idx / (RB * n_qc);
  const int within = idx - rb * (RB * n_qc);
  const int rows_here = n_rg - rb * RB < RB ? n_rg - rb * RB : RB;  // the last block of row groups may be short
  const int qb = within / (rows_here * QB);
  const int w2 = within - qb * (rows_here * QB);
  const int qw = n_qc - qb * QB < QB ? n_qc - qb * QB : QB;        // and so may the last block of query ranges
  const int rg_local = w2 / qw;
  w.qc = qb * QB + (w2 - rg_local * qw);
  w.rg = rb * RB + rg_local;
  return w;
}

// ---- contraction: rows a direct-to-LDS instruction brings in -------------------------------------------
// A tile's operand rows start at tile_first; an instruction covers the 16 rows from tile_first + rb on.  Rows
// from `token_rows` (the tokens, rounded up to whole 32-blocks) on are padding: such a block takes the last 16
// rows with tokens instead (lines the caches already hold), wherever the tile lies.  Returns the first row.
OF3_HD inline int contract_rows_first(int tile_first, int rb, int token_rows) {
  const int left = token_rows - tile_first;  // may be zero or less for a tile that lies in the padding
  return tile_first + (rb + 16 <= left ? rb : left - 16);
}

}  // namespace of3
