// bs_short.hip -- H x on bases of short neutron rows.
//
// On rows of at most a few waves' columns the tile kernel's time is a chain of
// latencies: a batch of jumps is fetched, staged between two barriers and walked
// by the one or two waves that have columns, some 30 times in a row.  Here a
// workgroup's waves share the columns AND the work on a column: all jumps of the
// tile's rows are staged in LDS at once (in as few passes as LDS takes), each
// wave walks its share of the batches, of the PP sources and of the NN slots for
// one 64-column chunk, and the shares are added up in LDS at the end.
//
// Tiles / here, us: sd 4p4n FP64 36.6 / 13.2, sd 5p6n FP64 71 / 26, sd 6p6n FP64 80 / 30,
// pf 3p3n FP32 88 / 33, pf 4p3n FP32 296 / 118, pf 8p3n FP32 9829 / 5549, pf 8p2n FP32
// 6847 (rows) / 1832.  From some hundred columns on PP and NN go to their own kernels
// (bs_like.hip): pf 4p4n FP32 460 / 319 (404 with PP and NN here), FP64 700 / 552, pf 6p4n
// FP32 4037 / 3011.  Columns cut into equal runs over the waves, so that nine chunks
// load 16 waves evenly, gained nothing (pf 6p4n 3037, pf 4p3n FP64 168 -> 207).  On
// small bases the launch (some 5 us) and the chain tile - batch - source rows - walk -
// sum bound it (LDS busy for 6 to 15% of the cycles).  On pf 4p4n LDS is busy for 37%
// (11% conflicts), the vector units issue 0.43 a cycle and CU: the waves wait, one
// workgroup of 16 to a CU, some of their lanes past a row's end.
#include "bs_short.hpp"

#include <algorithm>
#include <cstring>
#include <stdexcept>
#include <string>

namespace bss {
namespace {

#define HIP_OK(expr)                                                                       \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess) throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef uint32_t u4 __attribute__((ext_vector_type(4)));

template <typename V> using cptr = const __attribute__((address_space(4))) V*;
template <typename V> __device__ __forceinline__ cptr<V> cst(const V* p) {
  return (cptr<V>)(uintptr_t)p;
}

template <typename T, int R>
struct alignas(sizeof(T) * R) Row {
  T v[R];
};

template <typename T> __device__ __forceinline__ const T* pick(const float* a, const double* b);
template <> __device__ __forceinline__ const float* pick<float>(const float* a, const double*) { return a; }
template <> __device__ __forceinline__ const double* pick<double>(const float*, const double* b) { return b; }

// A workgroup of NW waves per tile of R rows, S batches staged at a time; CH:
// 64-column chunks of the longest row.  LDS: the tile's own rows [column][R], then
// per batch the source rows [column][R] and the signed coefficients [2 * operator +
// sign][R] (the entry quads hold byte offsets into both).
// (CH 9: launched with waves enough for every chunk, more than 8.)
template <typename T, int R, int WAVES, int CH>
__global__ __launch_bounds__((CH == 9 && WAVES < 10 ? 10 : WAVES) * 64) void k_short(Tab z, int S, const T* __restrict__ x, T* __restrict__ y, int accumulate) {
  extern __shared__ __align__(16) unsigned char smem[];
  using XV = Row<T, R>;
  using WV = Row<float, R>;
  constexpr int BS = 6 + 2 * R;  // words of a batch
  const int NW = CH == 9 ? (int)blockDim.x >> 6 : WAVES;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  // workgroup b runs on XCD b % 8: on bases of many tiles, runs of 32 tiles, which
  // share source rows, each
  const int b = blockIdx.x, ti = z.xcd ? (b >> 8) * 256 + (b & 7) * 32 + (b >> 3 & 31) : b;
  if (ti >= z.ntile) return;
  const cptr<Tile> tp = cst(z.tile) + ti;
  const uint32_t base = tp->base;
  const int nr = tp->rows & 0xffff, L = tp->rows >> 16, f0 = tp->f0;
  const int b0 = tp->b0, b1 = tp->b1;
  const int nc = (L + 63) >> 6, chunk = w % nc, sub = w / nc, nsub = (NW - chunk + nc - 1) / nc;
  const int cl = min(chunk * 64 + lane, L - 1);
  XV* own = reinterpret_cast<XV*>(smem);
  unsigned char* area = smem + (size_t)z.ls * sizeof(XV);
  const uint32_t xbytes = (uint32_t)z.ls * sizeof(XV), bbytes = xbytes + (uint32_t)z.wrows * sizeof(WV);
  T acc[R];
#pragma unroll
  for (int r = 0; r < R; r++) acc[r] = T(0);
  for (int c = tid; z.like && c < L; c += NW * 64) {
    XV v;
#pragma unroll
    for (int r = 0; r < R; r++) v.v[r] = r < nr ? x[base + (uint32_t)(r * L + c)] : T(0);
    own[c] = v;
  }
  int p0 = b0;
  do {
    const int p1 = min(p0 + S, b1);
    if (p0 != b0) __syncthreads();
    // staging, a wave a batch
    for (int i = p0 + w; i < p1; i += NW) {
      const cptr<uint32_t> rec = cst(z.batch) + (size_t)i * BS;
      const int Li = rec[1] & 0xffff, ws = rec[1] >> 16;
      unsigned char* at = area + (uint32_t)(i - p0) * bbytes;
      uint32_t src[R], wr[R];
#pragma unroll
      for (int r = 0; r < R; r++) src[r] = rec[6 + 2 * r], wr[r] = rec[7 + 2 * r];
      XV v[CH];
      WV c[2];
#pragma unroll
      for (int u = 0; u < CH; u++)
#pragma unroll
        for (int r = 0; r < R; r++)
          v[u].v[r] = lane + 64 * u < Li && src[r] != kNone ? x[src[r] + (uint32_t)(lane + 64 * u)] : T(0);
#pragma unroll
      for (int u = 0; u < 2; u++) {
        const int row = lane + 64 * u, op = row >> 1;
#pragma unroll
        for (int r = 0; r < R; r++) {
          const float a = op < ws && src[r] != kNone ? z.W[(wr[r] & 0x7fffffffu) + (uint32_t)op] : 0.0f;
          c[u].v[r] = __uint_as_float(__float_as_uint(a) ^ ((wr[r] & 0x80000000u) ^ ((uint32_t)row << 31)));
        }
      }
#pragma unroll
      for (int u = 0; u < CH; u++)
        if (lane + 64 * u < Li) reinterpret_cast<XV*>(at)[lane + 64 * u] = v[u];
#pragma unroll
      for (int u = 0; u < 2; u++)
        if (lane + 64 * u < 2 * (ws + 1)) reinterpret_cast<WV*>(at + xbytes)[lane + 64 * u] = c[u];
    }
    __syncthreads();
    if (p0 == b0 && z.like) {
      if (z.call_spe && sub == 0) {
        const XV v = own[cl];
#pragma unroll
        for (int r = 0; r < R; r++)
          if (r < nr) acc[r] = fma((T)z.pspe[f0 + r] + (T)z.nspe[tp->nf0 + cl], v.v[r], acc[r]);
      }
      {  // PP: this wave's run of the tile's union of source rows
        constexpr int U = R == 4 ? 4 : 8;
        const int n = tp->e1 - tp->e0, per = (n + nsub - 1) / nsub;
        const int ea = tp->e0 + min(sub * per, n), eb = tp->e0 + min((sub + 1) * per, n);
        const cptr<T> val = cst(pick<T>(z.pp32, z.pp64));
        for (int e = ea; e < eb; e += U) {
          uint32_t m[U];
          T v[U][R], xv[U];
#pragma unroll
          for (int u = 0; u < U; u++) {
            const int i = min(e + u, eb - 1);
            m[u] = cst(z.pp_src)[i];
#pragma unroll
            for (int r = 0; r < R; r++) v[u][r] = val[(size_t)i * R + r];
          }
#pragma unroll
          for (int u = 0; u < U; u++) xv[u] = x[base + (uint32_t)(((int)(m[u] & 0x7ffffffu) - f0) * L + cl)];
#pragma unroll
          for (int u = 0; u < U; u++)
            if (e + u < eb)
#pragma unroll
              for (int r = 0; r < R; r++)
                if (m[u] >> (27 + r) & 1) acc[r] = fma(v[u][r], xv[u], acc[r]);
        }
      }
      {  // NN: its run of the slots
        constexpr int U = 8;
        const int n = tp->nnE, per = (n + nsub - 1) / nsub;
        const int ea = min(sub * per, n), eb = min((sub + 1) * per, n);
        const int32_t* ps = z.nn_src + tp->nn + cl;
        const T* pv = pick<T>(z.nn32, z.nn64) + tp->nn + cl;
        for (int e = ea; e < eb; e += U) {
          int s[U];
          T v[U];
#pragma unroll
          for (int u = 0; u < U; u++) {
            const uint32_t o = (uint32_t)(min(e + u, eb - 1) * L);
            s[u] = ps[o];
            v[u] = pv[o];
          }
#pragma unroll
          for (int u = 0; u < U; u++)
            if (e + u < eb) {
              const XV xv = own[s[u]];
#pragma unroll
              for (int r = 0; r < R; r++) acc[r] = fma(v[u], xv.v[r], acc[r]);
            }
        }
      }
    }
    // PN: its share of the staged batches; a batch's first 12 entries are
    // fetched while the one before is applied
    {
      const int m = max((p1 - p0 - sub + nsub - 1) / nsub, 0);  // (64 at most)
      uint32_t dq = 0, dE = 0;
      if (lane < m) {
        const uint32_t* rec = z.batch + (size_t)(p0 + sub + lane * nsub) * BS;
        dq = rec[0];
        dE = rec[2 + (chunk >> 2)] >> (8 * (chunk & 3)) & 255u;
      }
      const u4* quad = reinterpret_cast<const u4*>(z.quad);
      u4 nx[3] = {};
      auto fetch = [&](int i) {
        const int E = __builtin_amdgcn_readlane(dE, i);
        const uint32_t q = __builtin_amdgcn_readlane(dq, i);
#pragma unroll
        for (int j = 0; j < 3; j++)
          if (4 * j < E) nx[j] = quad[q + (uint32_t)(j * L + cl)];
      };
      if (m > 0) fetch(0);
      for (int i = 0; i < m; i++) {
        const int E = __builtin_amdgcn_readlane(dE, i);
        const uint32_t q = __builtin_amdgcn_readlane(dq, i);
        const unsigned char* xs = area + (uint32_t)(sub + i * nsub) * bbytes;
        const unsigned char* wb = xs + xbytes;
        const u4 cu[3] = {nx[0], nx[1], nx[2]};
        if (i + 1 < m) fetch(i + 1);
        auto apply4 = [&](u4 p) {  // (slots past the column's entries hold a zero coefficient row)
          XV xv[4];
          WV wv[4];
#pragma unroll
          for (int k = 0; k < 4; k++) {
            xv[k] = *reinterpret_cast<const XV*>(xs + (p[k] & 0x1ffffu));
            wv[k] = *reinterpret_cast<const WV*>(wb + (p[k] >> 17));
          }
#pragma unroll
          for (int k = 0; k < 4; k++)
#pragma unroll
            for (int r = 0; r < R; r++) acc[r] = fma((T)wv[k].v[r], xv[k].v[r], acc[r]);
        };
#pragma unroll
        for (int j = 0; j < 3; j++)
          if (4 * j < E) apply4(cu[j]);
        for (int e = 12; e < E; e += 4) apply4(quad[q + (uint32_t)((e >> 2) * L + cl)]);
      }
    }
    p0 += S;
  } while (p0 < b1);
  __syncthreads();
  XV* red = reinterpret_cast<XV*>(smem);
  {
    XV v;
#pragma unroll
    for (int r = 0; r < R; r++) v.v[r] = acc[r];
    red[tid] = v;
  }
  __syncthreads();
  for (int i = tid; i < nr * L; i += NW * 64) {
    const int r = R == 1 ? 0 : i / L, c = i - r * L, ch = c >> 6;
    T s = T(0);
    for (int q = ch; q < NW; q += nc) s += reinterpret_cast<const T*>(red + q * 64 + (c & 63))[r];
    T* o = y + base + (uint32_t)i;
    *o = accumulate ? *o + s : s;
  }
}

// The same sums in the order of the tile kernel's one-row, two-jump shape, to the same
// bits (FP32): a workgroup per row.  A pair of jumps of a class is staged and summed
// over the neutron entries by a wave, apart from the rest; the PP and NN entries are
// fetched by the waves in turn, an item of 16 and the next one each, and added while the
// sum goes from wave to wave through LDS (a turn is 16 products, an LDS write and read
// and a barrier); the pairs' sums come last.  Tiles / here, us: sd 2p2n 17.2 / 8.0, sd
// 4p4n 33.7 / 12.7, sd 4p5n 36.3 / 13.4, pf 2p3n 31.3 / 11.6; sd 6p6n 55.6 / 27.3, where
// k_short takes 23.6.
template <int NW>
__global__ __launch_bounds__(NW * 64) void k_chain(Tab z, const float* __restrict__ x, float* __restrict__ y, int accumulate) {
  extern __shared__ __align__(16) unsigned char smem[];
  using V2 = Row<float, 2>;
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const cptr<Tile> tp = cst(z.tile) + blockIdx.x;
  const uint32_t base = tp->base;
  const int L = tp->rows >> 16, f0 = tp->f0, b0 = tp->q0, nb = tp->q1 - b0;
  const int nc = (L + 63) >> 6, chunk = w % nc, sub = w / nc, nsub = NW / nc;
  const int cl = min(chunk * 64 + lane, L - 1);
  float* sum = reinterpret_cast<float*>(smem);  // [chunk][lane]
  float* own = sum + 256;
  float* pairs = own + z.ls;                    // [pair][column]
  unsigned char* area = reinterpret_cast<unsigned char*>(pairs + (size_t)z.pairs * z.ls);
  const uint32_t xbytes = (uint32_t)z.ls * 8, bbytes = xbytes + (uint32_t)z.wrows * 8;
  const int e0 = tp->e0, npp = tp->e1 - e0, nnn = tp->nnE;
  const int ip = (npp + 15) >> 4, items = ip + ((nnn + 15) >> 4);
  uint32_t r1[16] = {};
  float r2[16] = {};
  // an item's loads: PP source value and coefficient, NN source column and coefficient
  // (places past the last: zeros)
  auto fetch = [&](int i) {
    if (i < ip) {
      const int n = min(16, npp - 16 * i);
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const int e = e0 + 16 * i + min(u, n - 1);
        const float v = cst(z.pp32)[e];
        const float s = x[base + (uint32_t)(((int)(cst(z.pp_src)[e] & 0x7ffffffu) - f0) * L + cl)];
        r1[u] = __float_as_uint(u < n ? s : 0.0f);
        r2[u] = u < n ? v : 0.0f;
      }
    } else if (i < items) {
      const int e1 = 16 * (i - ip), n = min(16, nnn - e1);
#pragma unroll
      for (int u = 0; u < 16; u++) {
        const uint32_t o = (uint32_t)tp->nn + (uint32_t)((e1 + min(u, n - 1)) * L + cl);
        r1[u] = (uint32_t)z.nn_src[o];
        const float v = z.nn32[o];
        r2[u] = u < n ? v : 0.0f;
      }
    }
  };
  const bool walks = sub < nsub;
  if (walks) fetch(sub);
  // this wave's pairs: their entry quads and numbers of entries, the first one's fetched
  const int m = walks ? max((nb - sub + nsub - 1) / nsub, 0) : 0;  // (64 at most)
  uint32_t dq = 0, dE = 0;
  if (lane < m) {
    const uint32_t* rec = z.pair + (size_t)(b0 + sub + lane * nsub) * 10;
    dq = rec[0];
    dE = rec[2] >> (8 * chunk) & 255u;
  }
  const u4* quad = reinterpret_cast<const u4*>(z.quad);
  u4 nx[3] = {};
  auto entries = [&](int i) {
    const int E = __builtin_amdgcn_readlane(dE, i);
    const uint32_t q = __builtin_amdgcn_readlane(dq, i);
#pragma unroll
    for (int j = 0; j < 3; j++)
      if (4 * j < E) nx[j] = quad[q + (uint32_t)(j * L + cl)];
  };
  if (m > 0) entries(0);
  for (int c = tid; c < L; c += NW * 64) own[c] = x[base + (uint32_t)c];
  for (int b = w; b < nb; b += NW) {
    const cptr<uint32_t> rec = cst(z.pair) + (size_t)(b0 + b) * 10;
    const int Li = rec[1] & 0xffff, ws = rec[1] >> 16;
    const uint32_t s0 = rec[6], w0 = rec[7], s1 = rec[8], w1 = rec[9];
    unsigned char* at = area + (uint32_t)b * bbytes;
    V2 v[4], c[2];
#pragma unroll
    for (int u = 0; u < 4; u++) {
      const uint32_t k = (uint32_t)(lane + 64 * u);
      v[u].v[0] = (int)k < Li ? x[s0 + k] : 0.0f;
      v[u].v[1] = (int)k < Li && s1 != kNone ? x[s1 + k] : 0.0f;
    }
#pragma unroll
    for (int u = 0; u < 2; u++) {
      const int row = lane + 64 * u, op = row >> 1;
      const float a0 = op < ws ? z.W[(w0 & 0x7fffffffu) + (uint32_t)op] : 0.0f;
      const float a1 = op < ws && s1 != kNone ? z.W[(w1 & 0x7fffffffu) + (uint32_t)op] : 0.0f;
      c[u].v[0] = __uint_as_float(__float_as_uint(a0) ^ ((w0 & 0x80000000u) ^ ((uint32_t)row << 31)));
      c[u].v[1] = __uint_as_float(__float_as_uint(a1) ^ ((w1 & 0x80000000u) ^ ((uint32_t)row << 31)));
    }
#pragma unroll
    for (int u = 0; u < 4; u++)
      if (lane + 64 * u < Li) reinterpret_cast<V2*>(at)[lane + 64 * u] = v[u];
#pragma unroll
    for (int u = 0; u < 2; u++)
      if (lane + 64 * u < 2 * (ws + 1)) reinterpret_cast<V2*>(at + xbytes)[lane + 64 * u] = c[u];
  }
  __syncthreads();
  for (int i = 0; i < m; i++) {
    const int E = __builtin_amdgcn_readlane(dE, i);
    const uint32_t q = __builtin_amdgcn_readlane(dq, i);
    const int b = sub + i * nsub;
    const unsigned char* xs = area + (uint32_t)b * bbytes;
    const unsigned char* wb = xs + xbytes;
    const u4 cu[3] = {nx[0], nx[1], nx[2]};
    if (i + 1 < m) entries(i + 1);
    float a = 0.0f;
    auto apply4 = [&](u4 p) {  // (slots past the column's entries hold a zero coefficient row)
      V2 xv[4], wv[4];
#pragma unroll
      for (int k = 0; k < 4; k++) {
        xv[k] = *reinterpret_cast<const V2*>(xs + (p[k] & 0x1ffffu));
        wv[k] = *reinterpret_cast<const V2*>(wb + (p[k] >> 17));
      }
#pragma unroll
      for (int k = 0; k < 4; k++) a = fma(wv[k].v[1], xv[k].v[1], fma(wv[k].v[0], xv[k].v[0], a));
    };
#pragma unroll
    for (int j = 0; j < 3; j++)
      if (4 * j < E) apply4(cu[j]);
    for (int e = 12; e < E; e += 4) apply4(quad[q + (uint32_t)((e >> 2) * L + cl)]);
    if (chunk * 64 + lane < L) pairs[b * z.ls + chunk * 64 + lane] = a;
  }
  if (sub == 0)
    sum[chunk * 64 + lane] = z.call_spe ? fma(z.pspe[f0] + z.nspe[tp->nf0 + cl], own[cl], 0.0f) : 0.0f;
  for (int i0 = 0; i0 < items; i0 += nsub) {
    const int i = i0 + sub;
    float a[16], b[16];
#pragma unroll
    for (int u = 0; u < 16; u++) a[u] = b[u] = 0.0f;
    if (walks && i < items) {
      const int n = nnn - 16 * (i - ip);
#pragma unroll
      for (int u = 0; u < 16; u++) {
        a[u] = r2[u];
        if (i < ip) {
          b[u] = __uint_as_float(r1[u]);
        } else {
          const float s = own[r1[u]];
          b[u] = u < n ? s : 0.0f;
        }
      }
      if (i + nsub < items) fetch(i + nsub);
    }
    const int turns = min(nsub, items - i0);
    for (int t = 0; t < turns; t++) {
      if (sub == t) {
        float s = sum[chunk * 64 + lane];
#pragma unroll
        for (int u = 0; u < 16; u++) s = fma(a[u], b[u], s);
        sum[chunk * 64 + lane] = s;
      }
      __syncthreads();
    }
  }
  __syncthreads();
  if (tid < L) {
    float s = sum[tid];
#pragma unroll 8
    for (int p = 0; p < nb; p++) s += pairs[p * z.ls + tid];
    float* o = y + base + (uint32_t)tid;
    *o = accumulate ? *o + s : s;
  }
}

// Tables that go to the device in one allocation and one copy
struct Parcel {
  std::vector<char> bytes;
  std::vector<std::pair<void*, size_t>> at;  // address of a pointer, offset of its table
  template <typename V>
  void add(V** p, const std::vector<V>& v) {
    at.push_back({p, bytes.size()});
    const char* b = reinterpret_cast<const char*>(v.data());
    bytes.insert(bytes.end(), b, b + v.size() * sizeof(V));
    bytes.resize((bytes.size() / 256 + 1) * 256);
  }
  void send(Owner& o, hipStream_t st) {
    void* d = nullptr;
    o.mem.reserve(1);
    HIP_OK(hipMalloc(&d, bytes.size()));
    o.mem.push_back(d);
    HIP_OK(hipMemcpyAsync(d, bytes.data(), bytes.size(), hipMemcpyHostToDevice, st));
    HIP_OK(hipStreamSynchronize(st));
    for (const auto& a : at) {
      void* q = static_cast<char*>(d) + a.second;
      memcpy(a.first, &q, sizeof q);
    }
  }
};

int set_of(int R) { return R == 1 ? 0 : R == 2 ? 1 : 2; }

constexpr size_t kLds = 160 * 1024;
constexpr size_t kManyJumps = (size_t)1 << 20, kMaxJumps = (size_t)1 << 25;

// more LDS than a kernel has without asking
void room(const void* fn, size_t lds) {
  if (lds > 64 * 1024) HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kLds));
}

template <typename T, int SH, int CH>
void launch(const Owner& o, const Tab& z, const T* x, T* y, int accumulate, hipStream_t st) {
  constexpr int R = kRows[SH], NW = kWaves[SH];
  const int ncmax = (o.lmax + 63) / 64, waves = CH < 9 ? NW : NW == 8 ? ncmax : std::min(16, 2 * ncmax);
  const Owner::Set& q = o.set[set_of(R)];
  const size_t own = (size_t)o.ls * R * sizeof(T), batch = own + (size_t)o.wrows * R * sizeof(float);
  // LDS of a workgroup: what leaves room for as many on a CU as there are (32 waves at most)
  const int want = std::max(1, std::min((q.ntile + 255) / 256, CH < 9 ? 32 / NW : NW == 8 ? 2 : 1));
  const int fit = (int)std::max<size_t>(1, (kLds / want - own) / batch);
  const int most = std::max(q.most, 1), pass = (most + std::min(fit, 64) - 1) / std::min(fit, 64);
  const int S = (most + pass - 1) / pass;
  const size_t lds = std::max(own + S * batch, (size_t)waves * 64 * R * sizeof(T));
  room(reinterpret_cast<const void*>(k_short<T, R, NW, CH>), lds);
  hipLaunchKernelGGL((k_short<T, R, NW, CH>), dim3(z.xcd ? (q.ntile + 255) / 256 * 256 : q.ntile), dim3(waves * 64), lds, st, z, S, x, y, accumulate);
  HIP_OK(hipGetLastError());
}

template <typename T, int SH>
void launch_ch(const Owner& o, const Tab& z, const T* x, T* y, int accumulate, hipStream_t st) {
  if (o.lmax <= 64) launch<T, SH, 1>(o, z, x, y, accumulate, st);
  else if (o.lmax <= 128) launch<T, SH, 2>(o, z, x, y, accumulate, st);
  else if (o.lmax > 256) launch<T, SH, 9>(o, z, x, y, accumulate, st);
  else launch<T, SH, 4>(o, z, x, y, accumulate, st);
}

size_t chain_lds(const Owner& o) {
  return (size_t)(256 + o.ls) * 4 + (size_t)o.pairs * (o.ls * 12 + o.wrows * 8);
}

template <int NW>
void launch_chain(const Owner& o, const Tab& z, const float* x, float* y, int accumulate, hipStream_t st) {
  room(reinterpret_cast<const void*>(k_chain<NW>), chain_lds(o));
  hipLaunchKernelGGL(k_chain<NW>, dim3(o.set[0].ntile), dim3(NW * 64), chain_lds(o), st, z, x, y, accumulate);
  HIP_OK(hipGetLastError());
}

template <typename T>
void apply_t(const Owner& o, int shape, Tab z, const T* x, T* y, int accumulate, hipStream_t st) {
  if (!o.has(shape, sizeof(T) == 4)) throw std::runtime_error("short-row tables missing");
  const Owner::Set& q = o.set[set_of(kRows[shape])];
  z.tile = q.tile;
  z.pair = o.pair;
  z.pairs = o.pairs;
  z.batch = q.batch;
  z.ls = o.ls;
  z.wrows = o.wrows;
  z.ntile = q.ntile;
  z.xcd = q.ntile >= 2048;
  z.like = shape < kPnOnly;
  if (shape >= kPnOnly) {
    accumulate = 1;  // after PP and NN
    shape -= kPnOnly - 1;
  }
  switch (shape) {
    case 0: launch_ch<T, 0>(o, z, x, y, accumulate, st); break;
    case 1: launch_ch<T, 1>(o, z, x, y, accumulate, st); break;
    case 2: launch_ch<T, 2>(o, z, x, y, accumulate, st); break;
    case 3: launch_ch<T, 3>(o, z, x, y, accumulate, st); break;
    case 4: launch_ch<T, 4>(o, z, x, y, accumulate, st); break;
    default:
      if constexpr (sizeof(T) == 4) {
        if (shape == 5) launch_chain<8>(o, z, x, y, accumulate, st);
        else launch_chain<16>(o, z, x, y, accumulate, st);
      }
  }
}

}  // namespace

bool Owner::has(int shape, bool f32) const {
  if (!ok || set[set_of(kRows[shape])].ntile == 0) return false;
  if (shape >= kSplit && shape < kPnOnly) return f32 && lmax <= kMaxChain && pairs <= 64 && chain_lds(*this) <= kLds;
  if (shape >= kPnOnly && lmax <= kMaxChain / 2) return false;  // too short to pay
  return !f32 || dim >= kSplitDim;
}

int Owner::usual(bool f32, bool like) const {
  const int q = lmax > kMaxChain && like ? kPnOnly + 2 : !set[0].ntile ? 4 : set[0].ntile <= 2048 ? 2 : 1;
  return has(q, f32) ? q : has(kSplit + 1, f32) ? kSplit + 1 : -1;
}

void Owner::release() {
  for (void* p : mem) (void)hipFree(p);
  mem.clear();
  for (Set& q : set) q = Set{};
  ok = false;
}

void apply(const Owner& o, int shape, Tab z, const float* x, float* y, int accumulate, hipStream_t st) {
  apply_t<float>(o, shape, z, x, y, accumulate, st);
}
void apply(const Owner& o, int shape, Tab z, const double* x, double* y, int accumulate, hipStream_t st) {
  apply_t<double>(o, shape, z, x, y, accumulate, st);
}

void build(Owner& o, const Host& h, hipStream_t st) {
  o.release();
  const bs::Species& P = h.t.sp[0];
  const bs::Species& N = h.t.sp[1];
  const int nd = (int)h.t.delta_of_class.size();
  o.lmax = 0;
  o.dim = h.t.dim;
  o.pairs = 0;
  for (int s = 0; s < P.nsec; s++) o.lmax = std::max(o.lmax, h.nlen[P.conj[s]]);
  // short rows, 32-bit offsets; on bases of many rows the tables of the four-row
  // tiles only (12 bytes a jump)
  if (o.lmax < 1 || o.lmax > kMaxRow || h.t.dim >= (int64_t)1 << 31 || h.p1_src.size() > kMaxJumps) return;
  const int first = h.p1_src.size() > kManyJumps ? 2 : 0;
  int cmax = 0;
  for (int k = 0; k < nd; k++) cmax = std::max(cmax, h.wstride[k]);
  o.wrows = (2 * (cmax + 1) + 3) / 4 * 4;  // (so that a batch's bytes are a multiple of 16)
  if (o.wrows > 128) return;
  o.ls = (o.lmax + 3) / 4 * 4;
  Parcel parcel;
  for (int v = first; v < 3; v++) {
    const int R = 1 << v, BS = 6 + 2 * R;
    std::vector<Tile> tile(h.tile_f0[v].size());
    std::vector<uint32_t> batch;
    std::vector<uint32_t> pair;
    int most = 0;
    for (size_t i = 0; i < tile.size(); i++) {
      const int f0 = h.tile_f0[v][i], nr = h.tile_nr[v][i], sp = P.sdsec[f0], cn = P.conj[sp], L = h.nlen[cn];
      if (L < 1) return;
      Tile& q = tile[i];
      q.base = (uint32_t)P.start[f0];
      q.rows = (uint32_t)nr | (uint32_t)L << 16;
      q.f0 = (uint32_t)f0;
      q.nf0 = (uint32_t)N.secfirst[cn];
      if (h.tpp_ptr[v][i + 1] >= (int64_t)1 << 31 || h.nn_base[cn] + (int64_t)h.nn_emax[cn] * L >= (int64_t)1 << 31) return;
      q.e0 = (uint32_t)h.tpp_ptr[v][i];
      q.e1 = (uint32_t)h.tpp_ptr[v][i + 1];
      q.nnE = (uint32_t)h.nn_emax[cn];
      q.nn = (uint32_t)h.nn_base[cn];
      q.b0 = (uint32_t)(batch.size() / BS);
      q.q0 = (uint32_t)(pair.size() / 10);
      for (int k = 0; k < nd; k++) {
        int nb = 0;
        for (int r = 0; r < nr; r++) {
          const int32_t* c = h.pcls.data() + (size_t)(f0 + r) * (nd + 1) + k;
          nb = std::max(nb, c[1] - c[0]);
        }
        if (!nb) continue;
        const size_t ck = (size_t)cn * nd + h.negk[k];
        const uint8_t* ch = h.n1_chunk.data() + ck * 64;
        uint32_t E[3];
        for (int u = 0; u < 3; u++)
          E[u] = (uint32_t)ch[4 * u] | (uint32_t)ch[4 * u + 1] << 8 | (uint32_t)ch[4 * u + 2] << 16 | (uint32_t)ch[4 * u + 3] << 24;
        if (h.n1q_base[ck] / 4 >= (int64_t)1 << 31) return;
        if (!(E[0] | E[1] | E[2])) continue;  // no neutron jump meets it
        const int Li = h.nlen[P.conj[h.srcsec[(size_t)sp * nd + k]]];
        for (int b = 0; b < nb; b++) {
          batch.push_back((uint32_t)(h.n1q_base[ck] / 4));
          batch.push_back((uint32_t)Li | (uint32_t)h.wstride[k] << 16);
          batch.push_back(E[0]);
          batch.push_back(E[1]);
          batch.push_back(E[2]);
          batch.push_back(0u);
          for (int r = 0; r < R; r++) {
            uint32_t src = kNone, wr = 0;
            if (r < nr) {
              const int32_t* c = h.pcls.data() + (size_t)(f0 + r) * (nd + 1) + k;
              if (c[0] + b < c[1]) {
                const int j = c[0] + b, meta = h.p1_meta[j];
                src = (uint32_t)P.start[h.p1_src[j]];
                wr = (uint32_t)(h.woff[k] + (meta & 0xff) * h.wstride[k]) | (meta >> 8 ? 0x80000000u : 0u);
              }
            }
            batch.push_back(src);
            batch.push_back(wr);
          }
        }
        if (R == 1) {  // the same jumps two by two
          const uint32_t* rec = batch.data() + batch.size() - (size_t)nb * BS;
          for (int b = 0; b < nb; b += 2, rec += 2 * BS) {
            pair.insert(pair.end(), rec, rec + BS);
            pair.push_back(b + 1 < nb ? rec[BS + 6] : kNone);
            pair.push_back(b + 1 < nb ? rec[BS + 7] : 0u);
          }
        }
      }
      q.b1 = (uint32_t)(batch.size() / BS);
      q.q1 = (uint32_t)(pair.size() / 10);
      if (R == 1) o.pairs = std::max(o.pairs, (int)(q.q1 - q.q0));
      most = std::max(most, (int)(q.b1 - q.b0));
    }
    o.set[v].ntile = (int)tile.size();
    o.set[v].most = most;
    parcel.add(&o.set[v].tile, tile);
    parcel.add(&o.set[v].batch, batch);
    if (R == 1) parcel.add(&o.pair, pair);
  }
  parcel.send(o, st);
  o.ok = true;
}

}  // namespace bss
