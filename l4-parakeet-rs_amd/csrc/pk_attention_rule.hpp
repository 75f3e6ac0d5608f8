// Which kernel a short-form attention call takes, and the rows a tile of the
// tile kernel loads.  constexpr, so that the same functions run in a host test.
#pragma once

namespace pk {

// True for the fp32 tile kernel (a workgroup per 16 queries and head), false
// for one wave per (query, head).  `live` queries have an output, a query
// sees at most `keys` keys.  The wave kernel's time grows with the keys of a
// query and with its workgroups per CU; a tile takes 8-18 us by its window and
// its workgroups run one to a CU, so a last round of them that is nearly empty
// costs a whole one.  Measured, wave / tile us, by live queries and keys:
//   160 keys and up: 160 x 160 13.7 / 13.5, 176 x 176 14.7 / 13.7, 496 x 257 32.8 / 18.7,
//     and in several rounds 520 x 193 24.6 / 20.2, 520 x 161 21.0 / 19.1, 640 x 161 24.2 / 24.8;
//   96 keys and up: last round two thirds full 392 x 97 12.9 / 11.0, 1024 x 129 30.9 / 25.1,
//     4096 x 97 87.0 / 81.4; less 200 x 129 11.6 / 13.1, 520 x 129 17.6 / 18.9;
//   fewer: 384 x 81 10.2 / 10.6, 496 x 33 7.0 / 8.4, 496 x 11 4.7 / 8.0.
constexpr bool short_takes_tile(int live, int keys, int cus) {
    const int tiles = 8 * ((live + 15) / 16);
    const int rounds = (tiles + cus - 1) / cus;
    const bool full = 3 * (long long)tiles >= (3LL * rounds - 1) * cus;
    return keys >= (full ? 96 : (rounds <= 1 ? 160 : 192));
}

// A tile of 16 queries from qb < live loads whole blocks of rows, more than its
// queries see: rows past their last key (or before key 0) are those at the
// ends instead, and queries without an output the last live one.  K and V may
// end there: valid_rows may exceed padded_rows, and the window's right end the rows of K.
constexpr int tile_last_key(int qb, int live, int valid, int right) {
    const int reach = (qb + 15 < live - 1 ? qb + 15 : live - 1) + right;
    return reach < valid - 1 ? reach : valid - 1;
}
constexpr int tile_key_row(int key, int last_key) { return key < 0 ? 0 : (key < last_key ? key : last_key); }
constexpr int tile_query_row(int query, int live) { return query < live - 1 ? query : live - 1; }

}  // namespace pk
