// Host side of the attention kernels: the tables of 64 x 64 tiles of a layout, read along lines of rows and along columns of
// keys, for the kernels that keep no sparse tensor (attention_fwd.hip, attention_bwd.hip: bsp_attention_tables_build) and for
// those that store p (attention_core.hip, attention_long.hip, attention_kv.hip: bsp_attention_stored_tables_build).  A new
// operator pays for both in its first call, whatever that call's masks are, so that calls of the other kind may be captured
// after it.  Host code on a bit per block, both sets: 0.5 ms for a layout of 16 x 64 x 64 blocks of 64 and 6 ms for
// 16 x 256 x 256 blocks of 16, where tensor operations took 1.0 and 11.8 ms for those of the second kind alone.
#include "bsp_common.h"
#include <algorithm>
#include <cstring>
#include <vector>

namespace bsp {
namespace {

// One head of a layout as a bit per block, rows of whole words
struct Bits {
  int rows, cols, words;
  std::vector<uint64_t> w;
  Bits(int r, int c) : rows(r), cols(c), words((c + 63) / 64), w((size_t)r * ((c + 63) / 64), 0) {}
  uint64_t *row(int r) { return w.data() + (size_t)r * words; }
  const uint64_t *row(int r) const { return w.data() + (size_t)r * words; }
  bool at(int r, int c) const { return (row(r)[c >> 6] >> (c & 63)) & 1; }
  void clear() { std::fill(w.begin(), w.end(), 0); }
};

void read_head(const uint8_t *lay, Bits &b) {
  for (int r = 0; r < b.rows; r++, lay += b.cols)
    for (int k = 0; k < b.words; k++) {
      const int n = std::min(64, b.cols - 64 * k);
      uint64_t bits = 0;
      int c = 0;
      for (; c + 8 <= n; c += 8) {                      // eight bytes to eight bits: each byte to 0 or 1, then one multiplication
        uint64_t x;
        std::memcpy(&x, lay + 64 * k + c, 8);
        x |= x >> 4;
        x |= x >> 2;
        x |= x >> 1;
        bits |= (((x & 0x0101010101010101ull) * 0x0102040810204080ull) >> 56) << c;
      }
      for (; c < n; c++) bits |= (uint64_t)(lay[64 * k + c] != 0) << c;
      b.row(r)[k] = bits;
    }
}

template <class F> void each_bit(uint64_t bits, int base, F &&f) {
  for (; bits; bits &= bits - 1) f(base + __builtin_ctzll(bits));
}

// One tile: S indices of blocks on its gathered side, and which of its S x S blocks exist: bit S * (index along the fixed
// side) + slot of the gathered one
struct Tile { int at[4]; unsigned blocks; };

// The tiles of one line, the S rows of bits from `fixed` on: the indices with a bit in any of them, ascending, S a tile (slots
// past the end repeat the tile's first index and hold no block)
void gather(const Bits &b, int fixed, int S, std::vector<Tile> &out) {
  int used = S;
  for (int k = 0; k < b.words; k++) {
    uint64_t any = 0;
    for (int f = 0; f < S; f++) any |= b.row(fixed + f)[k];
    each_bit(any, 64 * k, [&](int i) {
      if (used == S) {
        out.push_back(Tile{{i, i, i, i}, 0});
        used = 0;
      }
      Tile &t = out.back();
      t.at[used] = i;
      for (int f = 0; f < S; f++) t.blocks |= (unsigned)b.at(fixed + f, i) << (S * f + used);
      used++;
    });
  }
}

// positions of the four groups of sixteen that S blocks of 64 / S make up
void positions(const int *at, int S, int32_t *out) {
  const int shift = S == 1 ? 2 : S == 2 ? 1 : 0;        // 4 / S groups a block
  for (int g = 0; g < 4; g++) out[g] = ((at[g >> shift] << shift) + (g & ((1 << shift) - 1))) * 16;
}

// a tile's entry; by_rows: its rows are the fixed side (bit 4 * row group + column group)
void entry(const Tile &t, int S, bool by_rows, int32_t *out) {
  positions(t.at, S, out);
  const int per = 4 / S;
  int bits = 0xFFFF;
  if (t.blocks != (1u << (S * S)) - 1) {
    bits = 0;
    for (int f = 0; f < 4; f++)
      for (int g = 0; g < 4; g++)
        if ((t.blocks >> (S * (f / per) + g / per)) & 1) bits |= 1 << (by_rows ? 4 * f + g : 4 * g + f);
  }
  out[4] = bits;
  out[5] = out[6] = out[7] = 0;
}

// The block-columns of a head in the order in which S of them form a column of tiles.  They should have their blocks in the
// same block-rows: first the long ones (more than four times the median: the global columns of a layout), longest first,
// then the others as they lie (neighbours share their rows in banded layouts).
void column_order(const std::vector<int> &length, int S, std::vector<int> &order) {
  const int C = (int)length.size();
  order.resize(C);
  for (int c = 0; c < C; c++) order[c] = c;
  if (S == 1) return;
  std::vector<int> sorted(length);
  std::nth_element(sorted.begin(), sorted.begin() + (C - 1) / 2, sorted.end());
  const int median = std::max(1, sorted[(C - 1) / 2]);
  auto rank = [&](int c) { return length[c] > 4 * median ? length[c] : 0; };
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return rank(a) > rank(b); });
}

// A head read along its block-columns, in the order in which they form columns of tiles: turned's rows
void turn(const Bits &head, int S, std::vector<int> &length, std::vector<int> &order, std::vector<int> &place, Bits &turned) {
  std::fill(length.begin(), length.end(), 0);
  for (int r = 0; r < head.rows; r++)
    for (int k = 0; k < head.words; k++) each_bit(head.row(r)[k], 64 * k, [&](int c) { length[c]++; });
  column_order(length, S, order);
  for (int c = 0; c < head.cols; c++) place[order[c]] = c;
  turned.clear();
  for (int r = 0; r < head.rows; r++)
    for (int k = 0; k < head.words; k++) each_bit(head.row(r)[k], 64 * k, [&](int c) { turned.row(place[c])[r >> 6] |= (uint64_t)1 << (r & 63); });
}

// Work items: columns of tiles, those that stand out (of more than `part` tiles; 0: more than 16 and than twice the average)
// in parts of near-equal size with a slot each
struct Item { int count, begin, col, slot; };
struct Split { int col, first, parts; };
void cut_columns(const std::vector<int> &size, int64_t part, std::vector<Item> &items, std::vector<Split> &splits, int &n_slots) {
  int64_t total = 0;
  for (int n : size) total += n;
  const int64_t n_cols = (int64_t)size.size();
  if (part <= 0) part = std::max<int64_t>(16, (2 * total + n_cols - 1) / n_cols);
  for (int i = 0, begin = 0; i < (int)n_cols; begin += size[i], i++) {
    const int parts = (int)std::max<int64_t>(1, (size[i] + part - 1) / part), base = size[i] / parts, rem = size[i] % parts;
    if (parts > 1) splits.push_back(Split{i, n_slots, parts});
    for (int k = 0, at = begin; k < parts; k++) {
      const int count = base + (k < rem);
      items.push_back(Item{count, at, i, parts > 1 ? n_slots++ : -1});
      at += count;
    }
  }
}

// The block ids of a head: given, or the positions in the row-major order of the nonzero blocks, from `next` on
struct Ids {
  const int32_t *given;                                 // [R, C] of the head, or NULL
  const Bits &head;
  std::vector<int32_t> start;                           // id of the first block of each word
  Ids(const int32_t *given_, const Bits &head_, int32_t &next) : given(given_), head(head_), start(given_ ? 0 : head_.w.size()) {
    for (size_t i = 0; i < start.size(); i++) {
      start[i] = next;
      next += __builtin_popcountll(head.w[i]);
    }
  }
  int32_t at(int r, int c) const {                      // of a block that exists
    if (given) return given[(size_t)r * head.cols + c];
    const size_t i = (size_t)r * head.words + (c >> 6);
    return start[i] + __builtin_popcountll(head.w[i] & (((uint64_t)1 << (c & 63)) - 1));
  }
};

// the S indices of a tile's gathered side (or of a column's block-columns), the last repeated up to four
void indices(const int *at, int S, int32_t *out) {
  for (int g = 0; g < 4; g++) out[g] = at[std::min(g, S - 1)];
}

}  // namespace
}  // namespace bsp

using namespace bsp;

static int attention_tables_build(const uint8_t *h_layout, int H, int R, int C, int block, int32_t *h_tables,
                                  int64_t cap, bsp_attention_tables *info) {
  if (!h_layout || !info || H <= 0 || R <= 0 || C <= 0 || (cap > 0 && !h_tables)) return BSP_ERR_ARG;
  if (block != 16 && block != 32 && block != 64) return BSP_ERR_UNSUPPORTED;
  const int S = 64 / block;
  if (R % S || C % S) return BSP_ERR_UNSUPPORTED;
  const int lines = R / S, columns = C / S;
  *info = bsp_attention_tables{};
  info->lines = lines;
  info->columns = columns;

  std::vector<Tile> rows, cols;                         // tiles by line of rows, and by column of keys
  std::vector<int> row_size, col_size, order, place(C), length(C);
  std::vector<int> keys;                                // [H * columns][S] block-columns
  keys.reserve((size_t)H * C);
  Bits head(R, C), turned(C, R);                        // turned: rows are the block-columns in the order of the columns of tiles
  for (int h = 0; h < H; h++) {
    read_head(h_layout + (size_t)h * R * C, head);
    for (int l = 0; l < lines; l++) {
      const size_t first = rows.size();
      gather(head, l * S, S, rows);
      row_size.push_back((int)(rows.size() - first));
      info->longest_line = std::max(info->longest_line, row_size.back());
    }
    turn(head, S, length, order, place, turned);
    keys.insert(keys.end(), order.begin(), order.end());
    for (int c = 0; c < columns; c++) {
      const size_t first = cols.size();
      gather(turned, c * S, S, cols);
      col_size.push_back((int)(cols.size() - first));
    }
  }

  std::vector<Item> items;
  std::vector<Split> splits;
  cut_columns(col_size, 0, items, splits, info->n_slots);
  // four heads at a time, the longest items first: their q and do rows stay in L2, and no long item starts last (measured:
  // 261 -> 248 us for the column kernel of the module's default configuration, 134 -> 126 in the headline's)
  std::stable_sort(items.begin(), items.end(), [&](const Item &a, const Item &b) {
    const int ga = a.col / columns / 4, gb = b.col / columns / 4;
    return ga != gb ? ga < gb : a.count > b.count;
  });
  info->n_items = (int)items.size();
  info->n_split = (int)splits.size();

  auto up8 = [](int64_t n) { return (n + 7) / 8 * 8; };
  const int64_t row_first = up8(2 * (int64_t)H * lines), item_first = up8(12 * (int64_t)items.size());
  info->items_offset = row_first + 8 * (int64_t)rows.size();
  info->split_offset = info->items_offset + item_first + 8 * (int64_t)cols.size();
  info->total = info->split_offset + 8 * (int64_t)splits.size();
  if (info->total > cap) return BSP_ERR_CAPACITY;

  int32_t *t = h_tables;
  std::fill(t, t + row_first, 0);
  int64_t at = row_first;
  for (int i = 0; i < H * lines; i++) {
    t[2 * i] = row_size[i];
    t[2 * i + 1] = (int32_t)at;
    at += 8 * (int64_t)row_size[i];
  }
  for (size_t i = 0; i < rows.size(); i++) entry(rows[i], S, true, t + row_first + 8 * (int64_t)i);
  t = h_tables + info->items_offset;
  std::fill(t, t + item_first, 0);
  for (size_t i = 0; i < items.size(); i++) {
    int32_t *e = t + 12 * i;
    e[0] = items[i].count;
    e[1] = (int32_t)(item_first + 8 * (int64_t)items[i].begin);
    e[2] = items[i].col / columns;
    e[3] = items[i].col % columns;
    e[4] = items[i].slot;
    positions(&keys[(size_t)items[i].col * S], S, e + 8);
  }
  for (size_t i = 0; i < cols.size(); i++) entry(cols[i], S, false, t + item_first + 8 * (int64_t)i);
  t = h_tables + info->split_offset;
  for (size_t i = 0; i < splits.size(); i++) {
    int32_t *e = t + 8 * i;
    e[0] = splits[i].col / columns;
    e[1] = splits[i].col % columns;
    e[2] = splits[i].first;
    e[3] = splits[i].parts;
    positions(&keys[(size_t)splits[i].col * S], S, e + 4);
  }
  return BSP_OK;
}
extern "C" int bsp_attention_tables_build(const uint8_t *h_layout, int H, int R, int C, int block, int32_t *h_tables,
                                          int64_t cap, bsp_attention_tables *info) {
  return no_throw([&] { return attention_tables_build(h_layout, H, R, C, block, h_tables, cap, info); });
}

static int attention_stored_tables_build(const uint8_t *h_layout, const int32_t *h_ids, int H, int R, int C, int block, int part,
                                         int32_t *h_tables, int64_t cap, bsp_attention_tables *info) {
  if (!h_layout || !info || H <= 0 || R <= 0 || C <= 0 || part < 0 || (cap > 0 && !h_tables)) return BSP_ERR_ARG;
  if (block != 16 && block != 32 && block != 64) return BSP_ERR_UNSUPPORTED;
  const int S = 64 / block, ints = S == 1 ? 4 : 8 + S * S;   // ints per entry
  if (R % S) return BSP_ERR_UNSUPPORTED;
  const int lines = R / S, columns = C % S ? 0 : C / S;
  *info = bsp_attention_tables{};
  info->lines = lines;
  info->columns = columns;

  std::vector<Tile> rows, cols;
  std::vector<int> row_size, col_size, order, place(C), length(C), keys;
  std::vector<Bits> heads;
  heads.reserve(H);
  Bits turned(C, R);
  for (int h = 0; h < H; h++) {
    heads.emplace_back(R, C);
    Bits &head = heads.back();
    read_head(h_layout + (size_t)h * R * C, head);
    for (int l = 0; l < lines; l++) {
      const size_t first = rows.size();
      gather(head, l * S, S, rows);
      row_size.push_back((int)(rows.size() - first));
      info->longest_line = std::max(info->longest_line, row_size.back());
    }
    if (!columns) continue;
    turn(head, S, length, order, place, turned);
    keys.insert(keys.end(), order.begin(), order.end());
    for (int c = 0; c < columns; c++) {
      const size_t first = cols.size();
      gather(turned, c * S, S, cols);
      col_size.push_back((int)(cols.size() - first));
    }
  }
  std::vector<Item> items;
  std::vector<Split> splits;
  if (columns) cut_columns(col_size, part, items, splits, info->n_slots);
  info->n_items = (int)items.size();
  info->n_split = (int)splits.size();
  const int64_t row_first = 2 * (int64_t)H * lines, item_first = 12 * (int64_t)items.size();
  info->items_offset = row_first + ints * (int64_t)rows.size();
  info->split_offset = info->items_offset + item_first + ints * (int64_t)cols.size();
  info->total = info->split_offset + 8 * (int64_t)splits.size();
  if (info->total > cap) return BSP_ERR_CAPACITY;

  int32_t *t = h_tables;
  int64_t at = row_first;
  for (int i = 0; i < H * lines; i++) {
    t[2 * i] = row_size[i];
    t[2 * i + 1] = (int32_t)at;
    at += ints * (int64_t)row_size[i];
  }
  // The entry of a tile of one view: (id, index of its block on the gathered side, line, head) at blocks of 64, else (number
  // of the tile, 0, line, head, its S gathered indices, the ids as [row][column] of the tile)
  auto put = [&](int32_t *e, int tile, const Tile &x, int line, int h, bool by_rows, auto &&id_of) {
    if (S == 1) {
      e[0] = id_of(0, 0); e[1] = x.at[0]; e[2] = line; e[3] = h;
      return;
    }
    e[0] = tile; e[1] = 0; e[2] = line; e[3] = h;
    indices(x.at, S, e + 4);
    for (int f = 0; f < S; f++)                         // (f along the line or column, g along the gathered side)
      for (int g = 0; g < S; g++) e[8 + (by_rows ? S * f + g : S * g + f)] = (x.blocks >> (S * f + g)) & 1 ? id_of(f, g) : -1;
  };
  int32_t *to_row = t + row_first, *to_col = h_tables + info->items_offset + item_first, next = 0;
  for (int h = 0, row = 0, col = 0; h < H; h++) {
    const Ids ids(h_ids ? h_ids + (size_t)h * R * C : nullptr, heads[h], next);
    for (int l = 0; l < lines; l++)
      for (int k = 0; k < row_size[h * lines + l]; k++, row++, to_row += ints)
        put(to_row, row, rows[row], l, h, true, [&](int f, int g) { return ids.at(l * S + f, rows[row].at[g]); });
    for (int c = 0; c < columns; c++)
      for (int k = 0; k < col_size[h * columns + c]; k++, col++, to_col += ints)
        put(to_col, col, cols[col], c, h, false, [&](int f, int g) { return ids.at(cols[col].at[g], keys[(size_t)h * C + c * S + f]); });
  }
  t = h_tables + info->items_offset;
  for (size_t i = 0; i < items.size(); i++) {
    int32_t *e = t + 12 * i;
    e[0] = items[i].count;
    e[1] = (int32_t)(item_first + ints * (int64_t)items[i].begin);
    e[2] = items[i].col / columns;
    e[3] = items[i].col % columns;
    e[4] = items[i].slot;
    e[5] = e[6] = e[7] = 0;
    indices(&keys[(size_t)items[i].col * S], S, e + 8);
  }
  t = h_tables + info->split_offset;
  for (size_t i = 0; i < splits.size(); i++) {
    int32_t *e = t + 8 * i;
    e[0] = splits[i].col / columns;
    e[1] = splits[i].col % columns;
    e[2] = splits[i].first;
    e[3] = splits[i].parts;
    indices(&keys[(size_t)splits[i].col * S], S, e + 4);
  }
  return BSP_OK;
}
extern "C" int bsp_attention_stored_tables_build(const uint8_t *h_layout, const int32_t *h_ids, int H, int R, int C, int block, int part,
                                                 int32_t *h_tables, int64_t cap, bsp_attention_tables *info) {
  return no_throw([&] { return attention_stored_tables_build(h_layout, h_ids, H, R, C, block, part, h_tables, cap, info); });
}
