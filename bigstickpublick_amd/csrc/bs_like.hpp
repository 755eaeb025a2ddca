// The like-particle (PP and NN) parts of H x on large bases (bs_like.hip):
// tables and launches.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <vector>

#include "bs_tables.hpp"

namespace bsl {

constexpr int kPpRows = 16;  // proton rows of a PP tile
constexpr int kNnRows = 8;   // proton rows of an NN tile

struct Tab {
  int npp, nnn;               // PP work items, NN tiles
  // PP item: tile | first column << 32; its tile's rows and source blocks
  const uint64_t* pitem;
  const int64_t* tsec;        // [tile] vector offset of the sector
  const uint32_t* tbytes;     // [tile] elements of the sector
  const int32_t* tfirst;      // [tile] first row within the sector
  const int32_t* tnr;         // [tile] rows
  const int32_t* tL;          // [tile] row length
  const int32_t* tblk;        // [tile + 1] first block of 16 sources
  const uint32_t* psrc;       // [block][k % 4][k / 4]: source row's offset within the sector
  const float* pA32;          // [block][lane][step]: see k_pp
  const double* pA64;         // [block][step / 2][lane][step % 2]
  const int32_t* trow0;       // [tile] first proton SD
  const int64_t* pp_ptr;      // the entries by proton SD
  const int32_t* pp_src;
  const double* pp_val;
  // NN
  const int32_t* nf0;         // [tile] first proton row
  const int32_t* nnr;         // [tile] rows
  const int32_t* psec;
  const int32_t* pconj;
  const int32_t* nlen;
  const int64_t* pstart;
  // entries of column chunk cc of neutron sector c, source columns below 2048
  // (h = 0) and from 2048 on (h = 1, counted from there): g = nng[(c * 64 + cc) *
  // 2 + h], rows of 64 words (two entries' source columns, each plus one; 0: none)
  // from row g >> 10, (g & 1023) of them (an even number); values [2 row + entry][64]
  const uint32_t* nng;
  const uint32_t* nsrc;
  const float* nval32;
  const double* nval64;
};

struct Owner {
  bool ok[2] = {false, false};  // tables and values of FP32, FP64
  int lmax = 0;
  Tab t{};                      // without the values
  const float *pA32 = nullptr, *nval32 = nullptr;
  const double *pA64 = nullptr, *nval64 = nullptr;
  int ntile = 0;                // PP tiles, their first rows and sources, for the values
  int64_t blocks = 0, nrows = 0;
  const int32_t* usrc = nullptr;
  std::vector<uint32_t> nng;
  std::vector<void*> mem;
  ~Owner() { release(); }
  void release();
};

// What build() reads of the engine's tables (the pointers: on the device)
struct Host {
  const bs::Tables& t;
  const std::vector<int32_t>& nlen_h;
  const int64_t* pstart;
  const int32_t* psec;
  const int32_t* pconj;
  const int32_t* nlen;
  const int64_t* pp_ptr;
  const int32_t* pp_src;
  const double* pp_val;
};

// Tables with the values of one type; the other type's are added by a second call.
// Device work goes to `st`, which is waited for.
void build(Owner& o, const Host& h, bool f32, hipStream_t st);

// y (+)= (H_pp + H_nn) x
void apply(const Owner& o, const float* x, float* y, int accumulate, hipStream_t st);
void apply(const Owner& o, const double* x, double* y, int accumulate, hipStream_t st);

}  // namespace bsl
