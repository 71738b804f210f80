// Row tiling of the 8-wave attention units (attention.hip): which query rows of
// which heads a unit computes and stores. Plain C++ for the host too, so that
// the ownership of rows is checked without a GPU.
#pragma once
#if defined(__HIPCC__)
#define FA_HD __host__ __device__ __forceinline__
#else
#define FA_HD inline
#endif

#define FA_ROWS 256        // query rows of a unit
#define FA_NO_ROW 0x7fffffff

// Per (batch, kv head) the rows [row0, row0 + 256 * ntile + left) are `ntile`
// whole 256-row tiles of every query head of the group, then the `left` rows
// after them. The left-over rows of up to `hp` heads share one unit (they read
// the same keys), so 1024 + 1 rows cost 4 + 1/4 tiles per head and not 5; hp = 1
// gives every head a left-over unit of its own. Units are numbered whole tiles
// first.
struct FaRows {
    int row0, ntile, left, hp;
};
FA_HD FaRows fa_rows_of(int row0, int rows, int group, bool share) {
    FaRows r = {row0, rows / FA_ROWS, rows % FA_ROWS, 1};
    if (r.left && share) r.hp = FA_ROWS / r.left < group ? FA_ROWS / r.left : group;
    return r;
}
FA_HD int fa_rows_units(const FaRows &r, int batch, int kv_heads, int group) {
    return batch * kv_heads * (r.ntile * group + (r.left ? (group + r.hp - 1) / r.hp : 0));
}

// Unit `lin` of a row tiling: batch, kv head, first row and first query head
// of the group; left: rows per head of a left-over unit, 0 for a whole tile; hp:
// heads that a left-over unit owns (further ones belong to other units).
struct FaUnit {
    int b, hk, qbase, g0, left, hp;
};
FA_HD FaUnit fa_unit(const FaRows &r, int batch, int kv_heads, int group, int lin) {
    const int n_whole_tiles = batch * kv_heads * r.ntile * group;
    FaUnit u;
    int bh;
    if (lin < n_whole_tiles) {   // heads of a group are neighbours: they share K / V^T in L2
        u.g0 = lin % group;
        lin /= group;
        u.qbase = r.row0 + (lin % r.ntile) * FA_ROWS;
        bh = lin / r.ntile;
        u.left = 0;
    } else {
        lin -= n_whole_tiles;
        const int per = (group + r.hp - 1) / r.hp;
        u.g0 = (lin % per) * r.hp;
        u.qbase = r.row0 + r.ntile * FA_ROWS;
        bh = lin / per;
        u.left = r.left;
    }
    u.hp = r.hp;
    u.hk = bh % kv_heads;
    u.b = bh / kv_heads;
    return u;
}

// The i-th causal unit to start, as a number of fa_unit: longest first (a unit of
// causal rows reads the keys up to its last row), so the blocks that start last
// end soonest. Left-over rows, then the whole tiles downwards, each of every head.
FA_HD int fa_longest_first(const FaRows &r, int batch, int kv_heads, int group, int i) {
    const int per_tile = batch * kv_heads * group, n_left = r.left ? batch * kv_heads * ((group + r.hp - 1) / r.hp) : 0;
    if (i < n_left) return per_tile * r.ntile + i;
    i -= n_left;
    const int tile = r.ntile - 1 - i / per_tile, j = i % per_tile;
    return (j / group * r.ntile + tile) * group + j % group;
}

// Query row and head of row i (0..255) of a unit; row = FA_NO_ROW where it has none.
struct FaRowHead {
    int row, head;
};
FA_HD FaRowHead fa_unit_row(const FaUnit &u, int group, int i) {
    const int h0 = u.hk * group + u.g0;
    if (u.left == 0) return FaRowHead{u.qbase + i, h0};
    const int k = i / u.left;
    if (k >= u.hp || u.g0 + k >= group) return FaRowHead{FA_NO_ROW, h0};
    return FaRowHead{u.qbase + i % u.left, h0 + k};
}
