// tfs_layout.hpp -- device data layouts of one CRS matrix (host-side build).
//
// The solver keeps the matrix in three row orders, each chosen for the
// memory access pattern of the kernels that use it.  None changes any
// arithmetic: rows keep their entries in the caller's column order, so every
// row sum is formed exactly as the reference forms it.
//
//   S  (SpMV and the Krylov vectors): reverse Cuthill-McKee order of the
//      pattern, so that the x gathers of a wavefront's rows fall in a narrow
//      band (L2-resident) even when the caller numbers cells randomly.
//   L  (factor and forward sweep): rows grouped by level of the lower
//      dependency DAG of the CALLER's numbering (which defines the
//      incomplete factor), ties in S order; only the strictly-lower entries
//      are stored, contiguously, level after level.
//   U  (backward sweep): the L order backwards, strictly-upper entries.  A
//      row's upper dependencies sit at deeper lower levels, so they come
//      first; the backward sweep reads the forward sweep's output in runs.
#pragma once

#include <cstddef>
#include <future>
#include <vector>

namespace tfs {

// f(part, first, last) over [0, n) in kBeside parts, beside one another where there
// are at least `least` of them in all (else in turn).
constexpr int kBeside = 8;
template <typename F>
void in_parts(int n, int least, F f) {
  std::future<void> part[kBeside];
  const std::launch how =
      n < least ? std::launch::deferred : std::launch::async | std::launch::deferred;
  for (int k = 0; k < kBeside; ++k)
    part[k] = std::async(how, f, k, (int)((long long)n * k / kBeside),
                         (int)((long long)n * (k + 1) / kBeside));
  for (std::future<void> &p : part) p.get();
}

struct Segment {
  int l0, l1;  // levels [l0, l1)
  int rows;
  bool small;  // a run of small levels walked by one workgroup
};

struct SweepLayout {
  int nlev = 0;
  std::vector<int> lev_ptr;   // nlev+1 position starts of the levels
  std::vector<int> ptr;       // n+1 offsets of each position's triangle entries
  std::vector<int> col;       // neighbour positions in this layout
  std::vector<int> src;       // index of the entry in the caller's val[]
  std::vector<int> diag_src;  // index of the row's diagonal in val[]
  std::vector<int> orig;      // caller's row number of each position
  std::vector<int> of_orig;   // position of each caller row
  std::vector<Segment> segs;
};

struct Layout {
  int n = 0;
  long long nnz = 0;
  // S layout
  std::vector<int> s_orig, s_of_orig;   // S position <-> caller row
  std::vector<int> s_row, s_col, s_src, s_diag_src;
  std::vector<int> s_rblk;              // SpMV row blocks over S rows
  SweepLayout L, U;
  std::vector<int> l_to_s;  // S position of the row at L position p
  std::vector<int> u_to_l;  // L position of the row at U position q
  std::vector<int> s_to_u;  // U position of the row at S position k
  int bandwidth = 0;        // max |S(i) - S(j)| over entries (diagnostic)
};

// Greedy colouring of the (symmetrised) pattern, vertices visited in index
// order, each taking the smallest colour none of its neighbours has.
// `perm` lists the vertices by colour, index order within a colour (new
// position -> vertex); returns the number of colours.  Rows of one colour
// are independent, so an incomplete factor in this order has one level per
// colour.  With block > 1, runs of `block` consecutive vertices are coloured
// as units (block multi-colouring): a block keeps its internal couplings, in
// order, and an incomplete factor has at most `block` levels per colour.
int colour_order(int n, const int *row, const int *col, std::vector<int> &perm,
                 std::vector<int> *colour = nullptr, int block = 1);

// Algebraic block multi-colour order (Iwashita, Nakashima & Takahashi,
// "Algebraic Block Multi-Color Ordering Method for Parallel Multi-Threaded
// Sparse Triangular Solver in ICCG Method", IPDPS 2012): blocks of at most
// `block` rows grown breadth-first over the symmetrised pattern (seeds in
// index order, a block's rows in the order the search reached them, neighbours
// in ascending index), the block graph coloured greedily in block order, and
// the rows listed by colour, then block, then discovery order.  An incomplete
// factor in this order couples a row only to earlier rows of its own block and
// to rows of blocks of earlier colours: a sweep is one pass per colour whose
// blocks are independent, each block walked in its own (short) level order.
// `perm` maps new position -> vertex; `colour` and `block_of` are per vertex
// (block numbers in growth order).  Returns the number of colours.
int block_colour_order(int n, const int *row, const int *col, int block, std::vector<int> &perm,
                       std::vector<int> *colour = nullptr, std::vector<int> *block_of = nullptr);

// The FP32 sweeps of a brick-ordered copy, one wavefront per unit of bricks of
// one colour (k_brick_sweep): bricks of one colour do not couple, so a unit of
// several has no more levels than one and fuller ones.  A unit's rows are sorted
// by their level inside their brick and cut into steps of at most a
// wavefront's rows of one level, one row per lane; both triangles use the same order.  A
// row's first three entries of a triangle and its factor are one record; the
// rows of a step with more come first and have a second record.
constexpr int kBrickLanes = 64;      // rows of one step
constexpr int kBrickWide = 6;        // entries of a row in one triangle
constexpr int kUnitRows = 4096;      // rows of a unit (one 16^3 brick)
constexpr int kUnitFull = 1024;      // bricks are merged up to this many rows
struct BrickUnit {
  int row0, rows, step0, steps;      // first row, rows, first step, steps
  int lh0, lh, uh0, uh;              // halo entries of the lower / upper triangle
};
struct BrickStep {                   // one step of one triangle
  int x0;                            // its first second record
  unsigned what;                     // first row in the unit, rows, rows with a second record
  int p0() const { return (int)(what & 0xfffu); }
  int rows() const { return (int)(what >> 12 & 0x7fu); }
  int more() const { return (int)(what >> 20); }
};
struct BrickSource { int e[4]; };    // where a record's values come from
struct BrickPlaces { unsigned short at[4]; };
struct BrickTriangle {
  std::vector<BrickStep> step;
  // Per row, then per second record (after all rows' first ones): the byte
  // offsets in the unit's LDS array of floats of its entries' values -- slot 0
  // holds zero (padding), 1 + h halo entry h at the start -- and, fourth in a
  // first record, of its own result.  A slot is used again once the last step
  // that reads its value is over, so the array holds what is live, not the unit.
  std::vector<BrickPlaces> idx;
  // the entries' places in val[] (-1 padding); fourth in a first record the
  // row's place in the copy, for its factor
  std::vector<BrickSource> src;
  std::vector<int> halo;             // S position of each halo entry
};
struct BrickLayout {
  bool ok = false;
  int slots[2] = {0, 0};             // LDS floats of the largest unit, per triangle
  int steps = 0;                     // steps of the largest unit
  std::vector<BrickUnit> unit;       // colour after colour
  std::vector<int> colour0;          // first unit of each colour (ncolours + 1)
  std::vector<int> row, pos;         // copy row and its S position, unit order
  BrickTriangle L, U;
};
// row/col/dia: the copy's CRS (0-based, its own order); blk and colour: the
// block of each row and the colour of each block; s_of: S position of each row.
// Not ok where a coupling does not stay in its block or go between colours in
// the copy's order, or a limit is exceeded.
void build_bricks(int n, const int *row, const int *col, const int *dia,
                  const std::vector<int> &blk, const std::vector<int> &colour,
                  const std::vector<int> &s_of, BrickLayout &out);

// row/col/dia are 0-based, validated (diagonal present, columns ascending).
// identity_s keeps the caller's order as the S order (for a matrix whose rows
// are already in the order its kernels want, e.g. a block multi-colour copy).
// Block multi-colour order for the FP32 inner solves, from the caller's
// numbering: rows grouped by (phi_0 / edge, phi_1 / edge, phi_2 / edge) of the
// monotone potentials of the lower triangle's dependency graph -- phi_c(i) is
// the longest path to i counting the dependencies j -> i (j < i) of class c,
// the classes being the binary orders of the index step i - j merged into
// three groups of about equal entry counts; on a lexicographically numbered
// grid (steps 1, nx, nx ny) they are the cell's coordinates, so the groups are
// edge^3 bricks -- groups larger than `cap` rows split in caller order, and the
// blocks coloured greedily (in order of their first row) so that no two
// adjacent blocks share a colour.  perm lists the rows by (colour, block,
// caller order); bstart (nblocks + 1) gives each block's first position in
// that order and bcolour its colour.  Returns the number of colours.
// row/col/dia: 0-based CRS in the caller's order, columns ascending.
int brick_colour_order(int n, const int *row, const int *col, const int *dia, int edge, int cap,
                       std::vector<int> &perm, std::vector<int> &bstart,
                       std::vector<int> &bcolour);

// Blocks of the two triangular sweeps in the caller's own order (the factor
// the drop-in must apply), one workgroup per block (k_block_sweep): rows
// grouped by their monotone potentials as brick_colour_order groups them
// (kBlockEdge^3 bricks on a lexicographic grid), every block's rows sorted by
// their dependency level inside the block.  A row then depends on earlier
// steps of its own block and on rows of earlier blocks (its halo).
constexpr int kBlockEdge = 8;
constexpr int kBlockRows = 512;      // rows of one block
constexpr int kBlockSteps = 63;      // steps of one block (their starts fit one wavefront)
constexpr int kBlockHalo = 384;      // halo entries of one block (six per lane)
constexpr int kBlockLanes = 64;      // rows of one step
constexpr int kBlockWide = 6;        // entries of a row in one triangle

struct Block {     // one block of one triangle, as the kernel reads it
  int row0, rows;  // its rows in block order (upper triangle: the order backwards)
  int rpad;        // rows rounded up to eight: the stride between entry slots
  int ent0;        // first entry slot: slot k of row p is ent0 + k rpad + p
  int idx0;        // its rows' places begin at idx0 times the places per row
  int halo0, halo; // its halo entries
  int step0, steps;
};

struct BlockTriangle {
  std::vector<Block> blk;
  // per row, 4 (8 for wide rows) places of its entries' values in the block's
  // LDS array, as byte offsets: slot 0 holds zero (the padding), 1 + p a row
  // of the block, 1 + rows + h a halo entry
  std::vector<unsigned short> idx;
  std::vector<int> src;               // entry of the caller's val[], -1 padding
  std::vector<int> halo;              // block-order position of each halo entry
  std::vector<unsigned short> step;   // steps + 1 row starts per block
  int halo_max = 0;
};

struct BlockLayout {
  bool ok = false;                    // the structure suits block sweeps
  int nblk = 0, depth = 0, width = 0; // blocks, depth of their graph, entry slots per row
  int places() const { return width <= 3 ? 4 : 8; }
  std::vector<int> orig, of_orig;     // block-order position <-> caller row
  BlockTriangle L, U;
};

// Builds the blocks if the structure suits them (`out.ok`): structurally
// symmetric, within the limits above, at least kBlockLevels levels deep (a
// random numbering of a hex mesh has 13 to 20, in no blocks worth having) and
// the block graph at least kBlockGain times shallower than the nlev levels.
// Nearly empty blocks (many small systems in a batch, chains, thin boxes) keep the
// chip busy staging them: a sweep then takes kBlockNs + kBlockStepNs per step for
// each block, twice that where rows are wide, and the level-ordered one kLevelNs a
// level and kRowNs a row; blocks are built where they are the cheaper.  us per
// sweep, levels / blocks: 1371 systems of 9^3 42 / 73, 578 of 12^3 54 / 41, 814 of
// 17^3 107 / 187, 64 of 25^3 106 / 46, 256 of 25^3 136 / 165, 62500 chains of 32 rows
// 54 / 1221, 625 of them 36 / 15; nine-point rows, 1388 squares of 12^2 51 / 103,
// 195 of 32^2 137 / 70 (the estimates are within a fifth of all of these).
constexpr int kBlockGain = 4, kBlockLevels = 24;
constexpr double kBlockNs = 2.0, kBlockStepNs = 0.45, kLevelNs = 1400.0, kRowNs = 0.0105;
void build_blocks(int n, const int *row, const int *col, const int *dia,
                  const std::vector<int> &s_of_orig, int nlev, BlockLayout &out);

// Columns of a sliced ELL (64 rows a slice, slot-major) in 16 bits: a slice's
// columns fall in at most kWindows windows of kWindow rows each, a code is 4 bits
// of window and 12 of place in it, two consecutive slots in one word (the first
// in the low half).  Not ok where some slice needs more windows.
constexpr int kWindows = 16, kWindow = 4096;
struct ShortColumns {
  bool ok = false;
  std::vector<int> window;           // kWindows first rows per slice
  std::vector<long long> off;        // words before each slice, and in all
  std::vector<unsigned> code;        // slots 2 q, 2 q + 1 of lane l: off[s] + 64 q + l
};
// off: slots before each slice and in all; col: their columns, none negative.
void short_columns(const std::vector<long long> &off, const std::vector<int> &col,
                   ShortColumns &out);

// Average number of 128-byte lines of x that 64 consecutive rows gather from, over
// up to 256 such groups spread over the matrix.
double gather_lines(int n, const int *row, const int *col);

// `blocks`: build_blocks' result too (null: not built).
void build_layout(int n, const int *row, const int *col, const int *dia, int spmv_rows,
                  int spmv_cap, int small_level, Layout &out, bool identity_s = false,
                  BlockLayout *blocks = nullptr);

// The faces of every cell for the kernels that give a cell one lane: 64 cells a
// slice, slot-major, so that a wavefront's list entries are one contiguous run.
// An entry is 2 s + side (side 0: the cell is the face's first one), a cell's
// entries ascend by face -- the order of the reference's face loops -- and
// entries past kFaceSlots stand in a per-cell tail.
// The cells' order is the caller's or, where that scatters, the order in which
// the face list first names them: face lists follow the mesh's geometry even
// where cells are numbered at random, and face arrays are then read in order
// too.  Reordering pays with a pass in and out, so it has to halve the 128-byte
// lines of a cell field and a face field that a slice touches (on a 96^3 box 42 in
// lexicographic order, 707 in a random one, 42 in its first-named order).
constexpr int kFaceSlots = 32;
constexpr unsigned kNoFace = 0xffffffffu;
struct FaceLists {
  int n = 0;
  bool reordered = false;
  std::vector<int> orig, of;         // position <-> caller's cell, if reordered
  std::vector<long long> off;        // entries before each slice, and in all
  std::vector<unsigned> inc;         // slot j of lane l of slice s: off[s] + 64 j + l
  std::vector<int> tptr;             // n + 1, empty if no cell has a tail
  std::vector<unsigned> tail;
  int at(int c) const { return reordered ? of[(std::size_t)c] : c; }
};
// faces: pairs (c1, c2) in 1..n (base 1) or 0..n-1 (base 0), c1 an interior cell,
// c2 below that range for a boundary face; at most 2^31 entries in all.
// Cells are reordered in meshes of `from` cells and more: in smaller ones the
// fields stay in the caches whatever the order, and the passes in and out cost
// more than they save.  us with the cells reordered / in the caller's order, at
// 64^3, 72^3, 80^3 and 100^3 numbered at random: gradients 118/107, 135/122,
// 152/150, 235/276; pressure step 265/285, 328/377, 392/472, 618/841; momentum
// assembly and residual 110/115, 140/150, 167/187, 303/341 (48^3: 105/94, 220/219,
// 89/85).
constexpr int kReorderGradient = 1 << 19, kReorderAssembly = 1 << 18;
void build_face_lists(int n, long long nf, const int *faces, int base, int from, FaceLists &out);

}  // namespace tfs
