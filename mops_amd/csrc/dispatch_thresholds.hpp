// The problem sizes at which an operation changes kernels, in one place, each
// with the measurement that set it (MI355X, one GPU; whole calls timed on the
// device unless it says otherwise). The kernels' own capacity limits (what a
// layout can hold) stay with the kernels; what is here decides between two
// kernels that could both serve the shape.
#ifndef MOPS_AMD_DISPATCH_THRESHOLDS_HPP
#define MOPS_AMD_DISPATCH_THRESHOLDS_HPP

#include <cstddef>
#include <cstdint>

namespace mops::amd::thresholds {

// ---- HPE (hpe.hip) ---------------------------------------------------------
/// The three families of kernels: a tile of 4 to 16 rows in LDS and the monomials
/// spread over a workgroup of 1024 threads (hpe_tiles.hip), a lane per row
/// (hpe_rows.hip), and a few rows per workgroup of 256 threads (hpe.hip; in the
/// gradients with accumulators in LDS).
enum class HpeKernels { TILES, ROWS, FEW };

/// Forward pass. The tiles pay for filling LDS, a reduction over 256 teams and
/// two barriers per 16 rows (fewer where rows are wide), whatever the length of
/// the table; a lane per row pays a readlane per factor; a few rows per
/// workgroup read the table once for every few rows, from the caches. By
/// `factors` of the table (monomials x order), measured at 1370 points (64 to
/// 100 000 rows, 10 to 2000 features, 30 to 90 000 factors; the rule is on
/// average 1.3 % above the best of the three there, always tiles 30 %), us,
/// tiles / rows / few: 100 000 rows x 10 features, 150 factors, f32 27.5 / 8.0 /
/// 7.7, f64 41.6 / 11.4 / 10.4, 2000 factors f32 34.7 / 24.0 / 62.8, 9000 60.7 /
/// 87.8 / 174; 100 000 x 100, 600: 40.2 / 19.8 / 31.8, f64 66 / 32 / 40; 13 000 x
/// 30, 300: 6.8 / 4.6 / 4.9; 4000 x 250, 600, f64: 16.7 / 7.7 / 5.8; 1000 x 100,
/// 9000: 7.1 / 27.9 / 5.2, 30 000: 10.2 / 80 / 9.7, 90 000: 13.5 / 230 / 21.8.
inline HpeKernels hpe_forward(int64_t rows, int64_t features, int64_t factors, int64_t element_size) {
    const int64_t row_bytes = features * element_size;
    const bool single = element_size == 4;
    const int64_t rows_factors =
        (single ? (rows / 12 < 5000 ? rows / 12 : 5000) : (rows * 3 / 20 < 3000 ? rows * 3 / 20 : 3000)) + 2 * row_bytes;
    if (rows >= 10000 && row_bytes <= (single ? 850 : 2100) && factors <= rows_factors) {
        return HpeKernels::ROWS;
    }
    bool few;
    if (rows < 3000) {
        few = rows * factors <= 30 * 1000 * 1000 && (row_bytes >= 200 || 6 * rows < factors) &&
              (factors >= (single && row_bytes > 2500 ? row_bytes : 2500) || (!single && row_bytes >= 400));
    } else if (single) {
        few = row_bytes >= 300 && row_bytes <= 1000 && factors <= 1000;
    } else {
        const int64_t more = rows >= 5000 ? row_bytes * 5 / 4 : row_bytes * 4 < 7000 ? row_bytes * 4 : 7000;
        few = row_bytes >= 200 && row_bytes <= 10000 && factors <= 1000 + more;
    }
    return few ? HpeKernels::FEW : HpeKernels::TILES;
}

/// Gradients. Tiles and a lane per row turn the table round first (one or two
/// launches in front); the accumulators in LDS of a few rows per workgroup are
/// cleared and added up for every group of rows, which is work per feature, and
/// take an LDS addition per factor. The rule is on average 2 % above the best of
/// the three at 370 points (1000 to 100 000 rows, 10 to 250 features, 30 to 9000
/// factors); tiles from 10^7 factors of all rows on and few rows below are 16 %. us,
/// tiles / rows / few: 1000 rows x 100 features, 8000 factors, f32 18.0 / 27.6 /
/// 11.5; 13 000 x 30, 300: 13.7 / 10.4 / 9.0; 100 000 x 10, 150: 42.5 / 15.2 /
/// 22.6, f64 87 / 17.7 / 25.4, 2000: 48.0 / 40.4 / 113, 9000: 121 / 218 / 497;
/// 40 000 x 100, 300: 30.0 / 31.1 / 42.4, 3000: 42.6 / 55.1 / 159.
inline HpeKernels hpe_vjp(int64_t rows, int64_t features, int64_t factors, int64_t element_size) {
    const bool single = element_size == 4;
    const bool little = rows * factors < 10 * 1000 * 1000;
    if (features > 16 && little && rows * features < 3 * 1000 * 1000) {
        return HpeKernels::FEW;
    }
    const int64_t by_table = features <= 64 ? 3000 - 20 * features : features <= 120 ? 600 : 0;
    const int64_t rows_factors = (rows / 10 < by_table ? rows / 10 : by_table) * (single ? 5 : 8) / 5;
    if (rows >= 8000 + 100 * features && factors <= rows_factors) {
        return HpeKernels::ROWS;
    }
    const bool few = little || (features > 16 && factors < 500 && rows >= 10000 && rows * features < 2500 * 1000);
    return few ? HpeKernels::FEW : HpeKernels::TILES;
}

/// Second order: tiles or few rows (a lane per row has no second-order kernel).
/// us, tiles / few: 100 000 rows x 10 features, 150 factors, f32 102 / 23.3, f64
/// 165 / 26.7, 900: 121 / 77, 200 / 100; 100 000 x 30, 900: 143 / 131, 225 / 157;
/// 100 000 x 100, 300: 123 / 110, 600: 132 / 160; 1000 x 100, 8000, f64 45 / 17.
inline HpeKernels hpe_vjp_vjp(int64_t rows, int64_t features, int64_t factors, int64_t element_size) {
    const bool narrow = element_size == 4 && features <= 16 && rows < 30000;
    const int64_t millions = narrow ? 11 : element_size == 4 ? 16 : 24;
    const bool few = rows * factors < millions * 1000 * 1000 || (!narrow && rows >= 10000 && factors < 1500 - 10 * features);
    return few ? HpeKernels::FEW : HpeKernels::TILES;
}

// ---- SAP (sap_mfma.hip) ----------------------------------------------------
/// Tiles of 16 rows per wavefront of the device from which a launch has as many
/// workgroups as the device holds, each building the dense table once and
/// walking over tiles, instead of a workgroup (and a table build) per 128 rows.
/// nA, nB, nO = 13, 7, 20 over 65 000 to 560 000 rows: the forward pass gains
/// from one tile per wavefront on (200 000 rows, f32: 33.3 -> 30.0 us; f64 at
/// 100 000: 30.0 -> 25.9), the vjp from two (400 000 rows, f32: 88.9 -> 83.5
/// us; with one, 140 000 rows take 41.4 instead of 35.9 us).
constexpr int64_t SAP_FORWARD_WALK_TILES_PER_WAVE = 1;
constexpr int64_t SAP_VJP_WALK_TILES_PER_WAVE = 2;

/// Rows from which a lane per row (sap_rows.hip) takes the vjp, and the forward pass of two pairs; half
/// as many in double where the table fits the scalar cache. vjp, matrix cores / a lane per row, us: nA, nB,
/// nO = 13, 7, 20, 120 000 rows 26.4 / 22.0 (f32), 50.0 / 30.5 (f64), 60 000 rows 16.4 / 19.2, 28.1 / 24.1;
/// 5, 4, 12, 120 000 rows 15.6 / 12.1, 22.9 / 15.0; a million rows of 13, 7, 20: 133 / 83, 272 / 133.
constexpr int32_t SAP_ROWS_VJP = 100000;
/// The same for the forward pass, which the matrix cores pad less: 13, 7, 20 in double, 250 000 rows 39.8 /
/// 42.1, 500 000 64.5 / 58.6, a million 132 / 113; 16, 16, 8: 250 000 48.7 / 41.1, 500 000 86 / 61.
constexpr int32_t SAP_ROWS_FORWARD = 300000;
/// ... and for shapes that the matrix cores do not take (more than 64 columns, a table larger than the LDS).
/// 4, 9, 90 with 1500 entries, forward, 30 000 rows 26.9 / 30.3, 60 000 42.2 / 31.2, 250 000 152 / 60 (f32),
/// vjp 52.9 / 30.2, 81 / 31, 298 / 67; 10, 13, 30 in double, vjp, 30 000 rows 61 / 44, 500 000 823 / 290.
constexpr int32_t SAP_ROWS_BEYOND_MATRIX_CORES = 50000;
constexpr int32_t SAP_ROWS_BEYOND_MATRIX_CORES_VJP = 25000;
/// Bytes of a table that stays in the scalar cache.
constexpr int64_t SAP_ROWS_CACHED_TABLE = 16 * 1024;

// ---- OPSA / OPSAW (opsa.hip) -----------------------------------------------
/// Forward pass: segments are cut every so many positions of the sorted index,
/// and the pieces added by a second launch, when the average segment is twice
/// as long (pooling over whole structures: one wavefront per segment would
/// leave the device idle). 50 rows of 2400 edges: 94 -> 21 us in f32.
constexpr int OPSA_SPLIT_POSITIONS = 256;
/// vjp: columns of A up to which the per-edge kernel keeps a receiver's rows
/// of grad_output as matrix operands in registers (one to four tiles of 16);
/// beyond, the LDS-staged kernels. 60 000 edges, K = L = 48: 34 us against 82
/// (f32), 61 against 150 (f64); K = L = 64: 58 against 140, 107 against 552;
/// K = 56, L = 128: 118 against 507, 177 against 994; OPSAW K = L = 64: 97
/// against 220, 133 against 566.
constexpr int32_t OPSA_VJP_ROWS_IN_REGISTERS = 64;

// ---- the edges of every sender (grad_W of OPSAW and SASAW) -------------------
/// Index reads (edges x workgroups) up to which every workgroup finds its
/// senders' edges by reading the whole sender index; beyond, a counting sort
/// of the edges by sender (at 60 000 edges the sort costs more than the reads:
/// 52 us against 32 for the whole OPSAW vjp).
constexpr size_t SENDER_SCAN_LIMIT = 100u * 1000 * 1000;
/// Edges per sender on average up to which the lists are kept in slots (the
/// index in 4 parts, 32 places per sender and part: a part then holds 12 edges
/// of a sender on average; a sender that overflows is served by a wavefront
/// reading the whole index). OPSAW, 60 000 edges over 2000 senders, L = 32,
/// f32: 33 -> 22 us for the whole vjp.
constexpr int32_t SLOT_MEAN_EDGES = 48;
/// Edges up to which SASAW's gradients with a lane per column are one launch, where every node's workgroup looks
/// through the whole index of senders (three quarters of it for 16 components in float, half in double), with no more
/// nodes and tiles of columns than workgroups at a time. Beyond, an index that is read often or in several rounds, and
/// sums that take the registers of the edges, cost more than a second launch; grad_W alone comes to this first, and
/// its bits are not to depend on what else is wanted. One launch / two, us, whole vjp and grad_W alone, 32 columns. 9
/// components, f32 (768 workgroups): 12 000 edges of 400 nodes 23.0 / 26.6, 16.5 / 17.0; 16 000 of 533 26.2 / 29.6, 19.1 /
/// 18.9; 10 000 of 1000 26.0 / 29.0, 23.9 / 19.1; 24 000 of 800 34.4 / 33.6, 32.7 / 21.2; f64 (512): 16 000 of 250 29.2 / 32.3,
/// 20.9 / 18.7, of 533 34.3 / 38.1, 31.6 / 23.2. 4 components, f32 (1024): 16 000 of 533 15.2 / 20.0, 14.1 / 13.8; 24 000 of 800
/// 19.6 / 22.2, 18.2 / 14.8. 16 components, f32 (512): 12 000 of 400 39.6 / 41.3, 23.8 / 23.4; 16 000 of 250 41.8 / 39.3, 25.3 /
/// 20.9; f64 (two tiles): 5000 of 100 29.3 / 44.1; 16 000 of 250 63.5 / 59.2.
constexpr int32_t COLUMNS_EDGES_AS_THEY_ARE = 16384;
/// Edges per sender on average up to which lists are made by arrival (128 places
/// per sender). SASAW, 1000 nodes x 60 edges, whole vjp 87.6 -> 76.6 us (f32), 143.8
/// -> 115.3 (f64) against the kernels of sasaw_mfma.hip; at 100 per sender the
/// lists overflow (375 against 101 us). OPSAW, f32, whole vjp, by arrival / in-kernel
/// gather at 3000 senders x 60 edges: 44.7 / 74.3 us with senders drawn uniformly,
/// 105 / 95 with one of 300 edges, 304 / 400 with a density that falls along the
/// senders; 1000 x 60: 35.5 / 36.7, 69 / 63, 158 / 228.
constexpr int32_t ARRIVAL_MEAN_EDGES = 64;
/// Nodes from which the lists are made by arrival (one look at every edge, an
/// integer atomic each) rather than in slots (edges x nodes / 16 tests).
/// SASAW f32 vjp at 30 edges per node, by arrival / in slots: 2000 nodes 66.7 /
/// 60.7 us, 3000: 93.8 / 92.8, 4000: 113.7 / 114.0, 6000: 170 / 179, 8000: 233
/// / 255, 20 000: 682 / 820. OPSAW f32 vjp: 2000 senders 27.6 / 22.6, 3000:
/// 33.4 / 29.6, 4000: 37.6 / 39.3, 6000: 48 / 75, 20 000: 156 / 212.
constexpr int32_t ARRIVAL_NODES = 4000;
/// Edges up to which OPSAW lists by arrival; beyond, the counting sort (see
/// opsa.hip).
constexpr int32_t ARRIVAL_EDGES = 500000;

// ---- SASAW (sasaw_columns.hip) ------------------------------------------------
/// Edges from which the forward pass of a shape that fills the matrix cores (16
/// components, at most 16 columns, f32) stays with them: 300 000 edges 65 us
/// against 81; 60 000 edges 31 against 22.
constexpr int32_t COLUMNS_EDGES_AT_16 = 150000;

// ---- SASAW (sasaw_segments.hip) ----------------------------------------------
/// Values of a component index that one launch of the matrix-core kernels
/// covers (l <= 3); larger ranges go in parts, a launch per triple of parts,
/// up to SASAW_MAX_PARTS launches, then the general kernels of sasaw.hip.
/// 13 x 7 x 100 components, 900 entries, 60 000 edges: forward 1373 -> 46 us
/// (f32), 1631 -> 105 us (f64) against the general kernel, vjp 3404 -> 862 and
/// 5282 -> 1248 us.
constexpr int SASAW_INDEX_VALUES = 16;
constexpr int32_t SASAW_MAX_PARTS = 64;
/// Rows of W and of grad_output per launch of the gradient kernel when the
/// ranges go in parts: the kernel with 9 accumulator tiles does a row in less
/// than half the time of the one with 16 (13 x 7 x 100 components, 60 000
/// edges, f32: 16 rows 222 us per launch, 9 rows 60 us). In double also the
/// limit for ONE launch on ranges that would fit 16: the 16-tile kernel spills
/// (16 x 16 x 16 components, 64 columns: 950 us in one launch, 784 in four).
constexpr int32_t SASAW_GRADIENT_PART_ROWS = 9;

} // namespace mops::amd::thresholds

#endif
