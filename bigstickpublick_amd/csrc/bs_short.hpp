// H x on bases of short neutron rows (bs_short.hip): tables and launches.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "bs_tables.hpp"

namespace bss {

// Longest neutron row: nine 64-column chunks (pf rows of four neutrons have up to 565
// SDs, of five 1,651, which the tile kernel takes).
constexpr int kMaxRow = 576;
constexpr int kMaxChain = 256;           // the same for the ordered shapes
// Shapes below kSplit share a column's sum among waves; the next two (FP32) keep its
// order.
// From kPnOnly on, shapes 1 .. 4 again for the PN part alone, after the PP and NN
// kernels (bs_like.hip).
constexpr int kShapes = 11, kSplit = 5, kPnOnly = 7;
constexpr int kRows[kShapes] = {1, 2, 2, 4, 4, 1, 1, 2, 2, 4, 4};        // proton rows of a workgroup
constexpr int kWaves[kShapes] = {8, 8, 16, 16, 8, 8, 16, 8, 16, 16, 8};  // its waves
constexpr bool ordered(int shape) { return shape >= kSplit && shape < kPnOnly; }
// In FP32 the shapes that share a sum start at this size: below it the ordered ones,
// which a solve takes there, are about as fast (sd 4p4n, 28,503 states: 12.7 us, shared
// 11.2; from it on sd 6p6n, 93,710: 28.0 and 24.3), and H x alone and in a solve are the
// same bits.
constexpr int64_t kSplitDim = 65536;

// A tile of up to R proton rows of a sector (they follow one another in the vector)
struct Tile {
  uint32_t base;    // vector offset of the first row
  uint32_t rows;    // rows | row length << 16
  uint32_t f0;      // first proton SD
  uint32_t nf0;     // first neutron SD of the row
  uint32_t b0, b1;  // PN batches
  uint32_t e0, e1;  // PP union entries
  uint32_t nnE;     // NN slots of a column
  uint32_t nn;      // NN slot 0 of column 0
  uint32_t q0, q1;  // pairs of jumps (R = 1)
};

struct Tab {
  int ntile, xcd;             // tiles; XCD-grouped order
  int ls;                     // staged row length
  int wrows;                  // coefficient rows of a batch, 2 * (largest class + 1)
  int call_spe, like;         // like: SPE, PP and NN too
  const Tile* tile;
  // PN batch: { neutron entry quads of (sector, class), source row length |
  // operators << 16, entries of each 64-column chunk (a byte each; 3 words), 0 } and for each
  // row { source row's offset, coefficient row | negative phase << 31 } (offset
  // kNone: no jump)
  const uint32_t* batch;
  int pairs;                  // most pairs of jumps of a row
  const uint32_t* pair;       // a row's jumps of a class two by two: records as for R = 2
  const uint32_t* quad;       // neutron one-body entries, four of a column together
  const float* W;
  const uint32_t* pp_src;     // PP union: source SD | rows it feeds << 27
  const float* pp32;          // [entry][R]
  const double* pp64;
  const int32_t* nn_src;      // NN, slot-major
  const float* nn32;
  const double* nn64;
  const float* pspe;
  const float* nspe;
};
constexpr uint32_t kNone = 0xffffffffu;

// What build() reads of the engine's tables (host)
struct Host {
  const bs::Tables& t;
  const std::vector<int32_t>& nlen;
  const std::vector<int32_t>& srcsec;
  const std::vector<int32_t>& pcls;
  const std::vector<int32_t>& p1_src;
  const std::vector<int16_t>& p1_meta;
  const std::vector<int64_t>& n1q_base;
  const std::vector<uint8_t>& n1_chunk;
  const std::vector<int64_t>& nn_base;
  const std::vector<int32_t>& nn_emax;
  const std::vector<int32_t>& woff;
  const std::vector<int32_t>& wstride;
  const std::vector<int32_t>& negk;
  const std::vector<int32_t>* tile_f0;  // [R = 1, 2, 4]
  const std::vector<int32_t>* tile_nr;
  const std::vector<int64_t>* tpp_ptr;
};

struct Owner {
  bool ok = false;
  int lmax = 0, ls = 0, wrows = 0;
  int64_t dim = 0;
  int pairs = 0;
  uint32_t* pair = nullptr;
  struct Set {
    int ntile = 0, most = 0;  // tiles; most batches of one
    Tile* tile = nullptr;
    uint32_t* batch = nullptr;
  } set[3];                   // R = 1, 2, 4
  std::vector<void*> mem;
  ~Owner() { release(); }
  bool has(int shape, bool f32) const;  // it can run
  // Shape to take where none has been timed: few rows are shared by more waves (sd
  // 4p4n FP32, 495 rows: two rows to 16 waves 11.2 us, to 8 waves 13.8), many rows
  // want more workgroups on a CU (pf 4p3n, 4,845 rows: 166 against 118 us); the
  // largest bases have the four-row tables alone (16 waves 527, 8 waves 433 us on pf
  // 5p3n); rows of more than 256 columns take the PN part alone if the PP
  // and NN kernels can run (like).  -1: none
  int usual(bool f32, bool like) const;
  void release();
};

// device work goes to `st`, which is waited for
void build(Owner& o, const Host& h, hipStream_t st);

// y (+)= H x by shape 0 .. kShapes - 1; z holds the engine's tables for its R
// (tiles, batches and LDS strides are filled in)
void apply(const Owner& o, int shape, Tab z, const float* x, float* y, int accumulate, hipStream_t st);
void apply(const Owner& o, int shape, Tab z, const double* x, double* y, int accumulate, hipStream_t st);

}  // namespace bss
