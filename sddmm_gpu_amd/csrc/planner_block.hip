// The row-block launch of the SDDMM planner for gfx950 (MI355X): rows with mostly the same columns, computed as whole
// 32 x 32 tiles on the matrix cores (kernels_block.hip).
#include <hip/hip_runtime.h>
#include <algorithm>
#include <atomic>
#include "plan.hpp"

namespace sddmm {

namespace {

// The distinct columns of a few rows, ascending, and the place of each among them.
class ColumnSet {
public:
    explicit ColumnSet(int64_t n_cols) : bits((size_t)(n_cols / 64 + 1), 0), before((size_t)(n_cols / 64 + 1), 0) {}
    void add(int32_t col)
    {
        uint64_t &w = bits[(size_t)(col >> 6)];
        if (!w) words.push_back(col >> 6);
        w |= (uint64_t)1 << (col & 63);
    }
    int32_t rank()  // to be called before list and place
    {
        std::sort(words.begin(), words.end());
        int32_t n = 0;
        for (int32_t w : words) {
            before[(size_t)w] = n;
            n += __builtin_popcountll(bits[(size_t)w]);
        }
        return n;
    }
    void list(std::vector<int32_t> &cols) const
    {
        for (int32_t w : words)
            for (uint64_t b = bits[(size_t)w]; b; b &= b - 1) cols.push_back(w * 64 + __builtin_ctzll(b));
    }
    int32_t place(int32_t col) const
    {
        return before[(size_t)(col >> 6)] + __builtin_popcountll(bits[(size_t)(col >> 6)] & (((uint64_t)1 << (col & 63)) - 1));
    }
    void clear()
    {
        for (int32_t w : words) bits[(size_t)w] = 0;
        words.clear();
    }

private:
    std::vector<uint64_t> bits;
    std::vector<int32_t> before, words;
};

constexpr int64_t kUnitTiles = 4;   // tiles per unit of a row block that is several

}  // namespace

// Lays S out for the row-block kernels if that pays; *taken: it does.  rows: the rows with nonzeros, ascending.  Rows of
// more than twice the mean (tokens that look at all others) are put into blocks of their own, as they would fill the
// others' with their columns.
// Where the line lies, in cells computed per nonzero; us, row blocks against tiles or walk and the softmax's own passes, at
// K = 32 / 64 / 128.
//   Plans that serve the product as well (attention), softmax + product: 2.5.  Windows of 128 on either side of 16,384 tokens,
//       1.1 cells: 39 / 53 / 75 against 102 / 135 / 227; 1.9 cells (40 % left out): 24 / 35 / 52 against 70 / 82 / 124; 2.5
//       cells: 24 / 34 / 51 against 60 / 71 / 101; of 400, 60,000 tokens, 2.9 cells: 178 / 275 / 397 against 235 / 313 / 338.
//   The SDDMM alone: 1.6, from half a million nonzeros on.  1.1 cells: 15 / 21 / 35 against 24 / 40 / 77; 1.9: 12 / 17 / 24
//       against 12 / 17 / 27; 2.5: 12 / 17 / 24 against 11 / 14 / 24; 400 thousand nonzeros, 1.6 cells: 5.9 / 7.7 / 10.5
//       against 6.9 / 8.0 / 9.9, 200 thousand: 5.6 / 7.4 / 10.1 against 4.8 / 5.6 / 8.3.
int add_blocks(Ctx &c, const std::vector<int32_t> &rows, bool *taken)
{
    *taken = false;
    constexpr int R = kBlockRows;
    const bool product = c.opt.spmm_stream > 0;
    const double most_cells = (product ? 2.5 : 1.6) * (double)c.nnz;
    if (!product && c.nnz < 500000) return SDDMM_OK;
    // (the kernels address W by 32-bit float4 indices, H by 32-bit byte offsets)
    if (!block_supported(c.K) || rows.empty() || c.orig || c.n_rows * (int64_t)(c.K / 4) > (int64_t)UINT32_MAX ||
        c.n_cols * (int64_t)c.K > (int64_t)UINT32_MAX / 4)
        return SDDMM_OK;
    auto len = [&](int32_t r) { return (int64_t)c.row_ptr[r + 1] - c.row_ptr[r]; };
    const int64_t long_row = 2 * (c.nnz / (int64_t)rows.size() + 1);
    auto cells = [&](int64_t cols) { return (cols + R - 1) / R * R * R; };
    {  // a few blocks first: most matrices are nowhere near
        ColumnSet set(c.n_cols);
        const size_t blocks = (rows.size() + R - 1) / R, stride = std::max<size_t>(1, blocks / 16);
        int64_t nnz = 0, computed = 0;
        for (size_t b = stride / 2; b < blocks; b += stride) {
            for (size_t i = b * R; i < std::min(rows.size(), b * R + R); ++i) {
                if (len(rows[i]) > long_row) continue;
                nnz += len(rows[i]);
                for (int32_t p = c.row_ptr[rows[i]]; p < c.row_ptr[rows[i] + 1]; ++p) set.add(c.col_ind[p]);
            }
            computed += cells(set.rank());
            set.clear();
        }
        if ((double)computed * (double)c.nnz > most_cells * (double)nnz) return SDDMM_OK;
    }
    std::vector<int32_t> block_rows;  // padded
    for (int pass = 0; pass < 2; ++pass) {
        for (int32_t r : rows)
            if ((len(r) > long_row) == (pass == 1)) block_rows.push_back(r);
        while (block_rows.size() % R) block_rows.push_back(-1);  // (padded below)
    }
    const int64_t n_blocks = (int64_t)block_rows.size() / R;
    struct Block { std::vector<int32_t> cols; std::vector<uint2> info; };
    std::vector<Block> blocks((size_t)n_blocks);
    std::atomic<bool> twice{false};
    std::atomic<int64_t> n_cells{0};
    parallel_dynamic(n_blocks, 8, [&](int64_t b0, int64_t b1, int) {
        ColumnSet set(c.n_cols);
        for (int64_t b = b0; b < b1; ++b) {
            const int32_t *r = block_rows.data() + b * R;
            Block &B = blocks[(size_t)b];
            for (int i = 0; i < R && r[i] >= 0; ++i)
                for (int32_t p = c.row_ptr[r[i]]; p < c.row_ptr[r[i] + 1]; ++p) set.add(c.col_ind[p]);
            const int64_t n = set.rank();
            if ((double)(n_cells += cells(n)) > most_cells) return;
            set.list(B.cols);
            B.cols.resize((size_t)(cells(n) / R), B.cols.back());
            B.info.assign(B.cols.size(), make_uint2(0u, 0u));
            for (int i = 0; i < R && r[i] >= 0; ++i)
                for (int32_t p = c.row_ptr[r[i]]; p < c.row_ptr[r[i] + 1]; ++p) {
                    const int32_t at = set.place(c.col_ind[p]);
                    uint2 &f = B.info[(size_t)(at / R * R + i)];
                    const uint32_t bit = 1u << (at % R);
                    if (f.x & bit) twice = true;  // (a mask cannot hold an entry that S has twice)
                    if (!f.x) f.y = (uint32_t)p;
                    f.x |= bit;
                }
            set.clear();
        }
    });
    if (twice || (double)n_cells > most_cells) return SDDMM_OK;

    // Few blocks: the one with the most tiles that a workgroup computes alone is what the launches take, and the general
    // path's time grows with the nonzeros instead.  Both in us for softmax + product, fitted to windows of 200 to 4000 tokens.
    // Blocks and general path at K = 32 / 64 / 80 / 128: 559 tokens, 83 on either side, 24 full rows (18 tiles) 20 / 27 / 31 / 38
    // and 19 / 20 / 23 / 23; 1000, 40 (32 tiles) 28 / 38 / 44 / 55 and 19 / 21 / 23 / 27; 334, 167 (11 tiles) 16 / 21 / 23
    // / 30 and 18 / 20 / 22 / 21; 2000, 100 (7 tiles, the full rows in parts) 20 / 24 / 27 / 32 and 36 / 40 / 46 / 46;
    // 2000, 24 (4) 18 / 22 / 23 / 28 and 23 / 25 / 28 / 31.  On 120 other patterns (windows without full rows, one-sided,
    // thinned; dense blocks and triangles; profiles/row_blocks_few.txt) at four ranks what this takes is the faster one or
    // within 5 % of it, but for 10 of 460 cases, at worst 19 % slower (1024 tokens in dense blocks of 64, K = 128: 21.3
    // with blocks, 18.0 without).
    if (product && n_blocks <= c.cus && c.opt.dense_blocks != 2) {
        int64_t most = 0;
        bool parts = false;
        for (const Block &B : blocks) {
            const int64_t n = (int64_t)B.cols.size() / R;
            parts = parts || n > kBlockTiles;
            most = std::max(most, n > kBlockTiles ? kUnitTiles : n);
        }
        const double K = c.K, with = 6.1 + 0.075 * K + (double)most * (0.4 + 0.0064 * K) + (parts ? 3.5 : 0.0);
        const double without = 12.7 + 0.042 * K + 1e-6 * (double)c.nnz * (30.0 + 0.16 * K);
        if (with > without) return SDDMM_OK;
    }

    Launch L;
    L.kind = SDDMM_KERNEL_DENSE_BLOCK;
    L.fn_kind = 6;
    big_vector<int32_t> cols;
    big_vector<uint2> info;
    std::vector<int32_t> first_tile((size_t)n_blocks + 1, 0), empty_rows;
    for (int64_t b = 0; b < n_blocks; ++b) first_tile[(size_t)b + 1] = first_tile[(size_t)b] + (int32_t)(blocks[(size_t)b].cols.size() / R);
    const int64_t n_tiles = first_tile[(size_t)n_blocks];
    cols.resize((size_t)n_tiles * R);
    info.resize((size_t)n_tiles * R);
    parallel_ranges(n_blocks, 16, [&](int64_t b0, int64_t b1, int) {
        for (int64_t b = b0; b < b1; ++b) {
            std::copy(blocks[(size_t)b].cols.begin(), blocks[(size_t)b].cols.end(), cols.begin() + (size_t)first_tile[(size_t)b] * R);
            std::copy(blocks[(size_t)b].info.begin(), blocks[(size_t)b].info.end(), info.begin() + (size_t)first_tile[(size_t)b] * R);
        }
    });
    // Units: the whole row blocks first, an eighth of them, neighbours all, to the workgroups of each die (workgroup b runs
    // on die b % 8): neighbouring blocks use the same rows of H, which are then fetched into one die's L2.  Then the
    // parts of row blocks that are several, small ones, which even out what the compute units have got.
    std::vector<int4> units, parts, sums, long_pieces;
    bool in_pieces = false;
    std::vector<int32_t> whole;
    int64_t records = 0, lds_tiles = 0;
    for (int64_t b = 0; b < n_blocks; ++b) {
        const int32_t t0 = first_tile[(size_t)b], t1 = first_tile[(size_t)b + 1];
        if (t1 - t0 <= kBlockTiles) {
            whole.push_back((int32_t)b);
            lds_tiles = std::max<int64_t>(lds_tiles, t1 - t0);
            continue;
        }
        sums.push_back(make_int4((int)b, (int)records, (int)((t1 - t0 + kUnitTiles - 1) / kUnitTiles), 0));
        for (int64_t t = t0; t < t1; t += kUnitTiles) parts.push_back(make_int4((int)b, (int)t, (int)std::min<int64_t>(t1, t + kUnitTiles), (int)records++));
        for (int i = 0; i < R; ++i)
            if (const int32_t r = block_rows[(size_t)(b * R + i)]; r >= 0) {
                const int n = (int)((len(r) + kLongPiece - 1) / kLongPiece), first = (int)long_pieces.size();
                for (int k = 0; k < n; ++k)
                    long_pieces.push_back(make_int4(c.row_ptr[r] + k * kLongPiece, (int)std::min<int64_t>(kLongPiece, len(r) - (int64_t)k * kLongPiece), first, n));
                in_pieces = in_pieces || n > 1;
            }
    }
    const int64_t nw = (int64_t)whole.size();
    for (int64_t i = 0; i < (nw + 7) / 8; ++i)
        for (int64_t die = 0; die < 8; ++die) {
            const int64_t at = nw * die / 8 + i;
            if (at >= nw * (die + 1) / 8) continue;
            const int32_t b = whole[(size_t)at];
            units.push_back(make_int4(b, first_tile[(size_t)b], first_tile[(size_t)b + 1], -1));
        }
    units.insert(units.end(), parts.begin(), parts.end());
    for (int64_t b = 0; b < n_blocks; ++b)  // a short block's last row again (its info is empty there)
        for (int i = 1; i < R; ++i)
            if (block_rows[(size_t)(b * R + i)] < 0) block_rows[(size_t)(b * R + i)] = block_rows[(size_t)(b * R + i - 1)];
    BlockArgs &a = L.ba;
    int4 *d_units = nullptr, *d_sums = nullptr, *d_long = nullptr;
    int32_t *d_rows = nullptr, *d_cols = nullptr, *d_empty = nullptr;
    uint2 *d_info = nullptr;
    if (int rc = c.up(&d_units, units)) return rc;
    if (int rc = c.up(&d_rows, block_rows)) return rc;
    if (int rc = c.up(&d_cols, cols)) return rc;
    if (int rc = c.up(&d_info, info)) return rc;
    if (int rc = c.up(&d_long, long_pieces)) return rc;
    a.units = d_units; a.rows = d_rows; a.cols = d_cols; a.info = d_info; a.long_pieces = d_long;
    a.n_units = (int32_t)units.size(); a.n_long_pieces = (int32_t)long_pieces.size();
    a.K = c.K; a.nnz = (int32_t)c.nnz;
    if (in_pieces) {
        const size_t bytes = long_pieces.size() * sizeof(float2);
        float2 *d_rec = nullptr;
        HIP_TRY(hipMalloc((void **)&d_rec, bytes));
        c.P->owned.push_back({d_rec, bytes, true});
        c.dev_bytes += (int64_t)bytes;
        a.long_records = d_rec;
        L.part_bytes = (int64_t)bytes;
    }
    if (product) {
        for (int64_t r = 0; r < c.n_rows; ++r)
            if (c.row_ptr[r + 1] == c.row_ptr[r]) empty_rows.push_back((int32_t)r);
        if (int rc = c.up(&d_sums, sums)) return rc;
        if (int rc = c.up(&d_empty, empty_rows)) return rc;
        a.sums = d_sums; a.n_sums = (int32_t)sums.size();
        a.empty_rows = d_empty; a.n_empty = (int32_t)empty_rows.size();
        const size_t bytes = (size_t)records * ((c.K + 31) / 32) * 4096;
        if (bytes) {
            float *d_part = nullptr;
            HIP_TRY(hipMalloc((void **)&d_part, bytes));
            c.P->owned.push_back({d_part, bytes, true});
            c.dev_bytes += (int64_t)bytes;
            a.part = d_part;
        }
        L.sp_on = 3; L.sp_part_bytes = (int64_t)bytes;
        c.P->info.spmm_runs += records * R;
    }
    L.nnz = c.nnz; L.rows = (int64_t)rows.size(); L.positions = n_tiles * R * R;
    // Eight waves per workgroup instead of four where there is a workgroup for every compute unit at most, or room in LDS for one.
    L.fn_nwaves = a.n_units <= c.cus ? 8 : 4;
    L.softmax_waves = lds_tiles > kBlockTilesFew ? 8 : L.fn_nwaves;
    L.grid = a.n_units; L.block = 64 * L.fn_nwaves; L.k_slice = c.K;
    L.lds = (int32_t)(std::max(lds_tiles, std::min<int64_t>(records ? kUnitTiles : 0, kBlockTiles)) * kBlockTileBytes);  // the softmax form's: scores and masks
    if (int rc = resolve_functions(L)) return rc;
    c.P->info.dense_nnz += c.nnz;
    c.P->info.dense_blocks += n_tiles;
    c.P->launches.push_back(L);
    *taken = true;
    return SDDMM_OK;
}

}  // namespace sddmm
