// bs_like.hip -- proton-proton and neutron-neutron parts of H x on large bases.
#include "bs_like.hpp"
#include "bs_parallel.hpp"

#include <algorithm>
#include <stdexcept>
#include <string>

namespace bsl {
namespace {

#define HIP_OK(expr)                                                                       \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess) throw std::runtime_error(std::string(#expr) + ": " + hipGetErrorString(e_)); \
  } while (0)

typedef float f4 __attribute__((ext_vector_type(4)));
typedef double d4 __attribute__((ext_vector_type(4)));
typedef double d2 __attribute__((ext_vector_type(2)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
// vectors that start on any element
typedef f4 f4u __attribute__((aligned(4)));
typedef d4 d4u __attribute__((aligned(8)));

template <typename V> using cptr = const __attribute__((address_space(4))) V*;
template <typename V> __device__ __forceinline__ cptr<V> cst(const V* p) {
  return (cptr<V>)(uintptr_t)p;
}

// Loads at or beyond `bytes` return zero.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(base), (short)0, (int)bytes, 0x00020000);
}

// PP: Y[16 rows][64 columns] += A[16 rows][sources] X[sources][64 columns] on
// the matrix cores, a wave an item.  The tile's rows share their source rows:
// the union is walked in blocks of 16 (dense coefficients, zeros where a
// source does not feed a row), so a source row is read once per 16 target
// rows.  Lane l takes source k = l / 16 of each of a block's four steps, at
// columns 4 (l % 16) .. + 3 (FP32; FP64: 2 (l % 16), + 1 and 32 further), and
// feeds v_mfma_*_16x16x4 once per column: result register r is row
// 4 (l / 16) + r of the tile (FP64: the matrix rows are permuted for that).
// A zero of the union times an infinity is NaN: a result that is not finite is
// left out and summed over its row's own entries instead (again), so that a
// source that is not finite reaches the rows that H connects it to and no others.
// sets results that are not finite to zero: bit 4 i + u is column u of row i
template <typename V>
__device__ __forceinline__ uint32_t take_out(V (&d)[4]) {
  uint32_t out = 0;
#pragma unroll
  for (int u = 0; u < 4; u++)
#pragma unroll
    for (int i = 0; i < 4; i++)
      if (!isfinite(d[u][i])) {
        out |= 1u << (4 * i + u);
        d[u][i] = 0;
      }
  return out;
}

// yrow[col] += proton SD f's sum over its own entries
template <typename T>
__device__ __forceinline__ void again(const Tab& z, const T* __restrict__ x, T* __restrict__ yrow, int64_t f, int col) {
  T s = T(0);
  for (int64_t e = z.pp_ptr[f]; e < z.pp_ptr[f + 1]; e++)
    s = fma((T)z.pp_val[e], x[z.pstart[z.pp_src[e]] + col], s);
  yrow[col] += s;
}

__global__ __launch_bounds__(256) void k_pp(Tab z, const float* __restrict__ x, float* __restrict__ y) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t it = cst(z.pitem)[blockIdx.x];
  const int t = (int)(uint32_t)it, c0 = (int)(it >> 32) + 64 * w;
  const int L = cst(z.tL)[t];
  if (c0 >= L) return;
  const int li = lane & 15, lk = lane >> 4;
  const int64_t sec = cst(z.tsec)[t];
  const __amdgpu_buffer_rsrc_t r = rsrc(x + sec, cst(z.tbytes)[t] * 4u);
  const int b0 = cst(z.tblk)[t], nb = cst(z.tblk)[t + 1] - b0;
  const u4* ps = reinterpret_cast<const u4*>(z.psrc) + (size_t)b0 * 4 + lk;
  const f4* pa = reinterpret_cast<const f4*>(z.pA32) + (size_t)b0 * 64 + lane;
  // the lane's four columns, moved back into the row at its end (only the
  // columns from c on are stored)
  const int c = c0 + 4 * li, cl = max(min(c, L - 4), 0);
  const uint32_t vo = (uint32_t)cl;
  f4 d[4];
#pragma unroll
  for (int u = 0; u < 4; u++) d[u] = f4{0.0f, 0.0f, 0.0f, 0.0f};
  u4 s = ps[0];
  f4 a = pa[0];
  for (int b = 0; b < nb; b++) {
    f4 xv[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
      if (L >= 4) {
        xv[q] = __builtin_bit_cast(f4, __builtin_amdgcn_raw_buffer_load_b128(r, (s[q] + vo) * 4u, 0, 0));
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++)
          xv[q][u] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (s[q] + (uint32_t)min(u, L - 1)) * 4u, 0, 0));
      }
    }
    const f4 ac = a;
    const int b1 = min(b + 1, nb - 1);
    s = ps[b1 * 4];
    a = pa[b1 * 64];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int u = 0; u < 4; u++) d[u] = __builtin_amdgcn_mfma_f32_16x16x4f32(ac[q], xv[q][u], d[u], 0, 0, 0);
  }
  const int nr = cst(z.tnr)[t], f0 = cst(z.tfirst)[t];
  uint32_t out = take_out(d);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = 4 * lk + i;
    if (row < nr) {
      float* o = y + sec + (int64_t)(f0 + row) * L + cl;
      if (c + 3 < L) {
        f4u v = *reinterpret_cast<const f4u*>(o);
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] += d[u][i];
        *reinterpret_cast<f4u*>(o) = v;
      } else {
#pragma unroll
        for (int u = 0; u < 4; u++)
          if (cl + u >= c && cl + u < L) o[u] += d[u][i];
      }
    }
  }
  for (; out; out &= out - 1) {
    const int q = __builtin_ctz(out), row = 4 * lk + (q >> 2), col = cl + (q & 3);
    if (row < nr && col >= c && col < L)
      again(z, x, y + sec + (int64_t)(f0 + row) * L, (int64_t)z.trow0[t] + row, col);
  }
}

__global__ __launch_bounds__(256) void k_pp(Tab z, const double* __restrict__ x, double* __restrict__ y) {
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const uint64_t it = cst(z.pitem)[blockIdx.x];
  const int t = (int)(uint32_t)it, c0 = (int)(it >> 32) + 64 * w;
  const int L = cst(z.tL)[t];
  if (c0 >= L) return;
  const int li = lane & 15, lk = lane >> 4;
  const int64_t sec = cst(z.tsec)[t];
  const __amdgpu_buffer_rsrc_t r = rsrc(x + sec, cst(z.tbytes)[t] * 8u);
  const int b0 = cst(z.tblk)[t], nb = cst(z.tblk)[t + 1] - b0;
  const u4* ps = reinterpret_cast<const u4*>(z.psrc) + (size_t)b0 * 4 + lk;
  const d2* pa = reinterpret_cast<const d2*>(z.pA64) + (size_t)b0 * 128 + lane;
  int c[2], cl[2];  // the lane's two pairs of columns, moved back into the row at its end
#pragma unroll
  for (int h = 0; h < 2; h++) {
    c[h] = c0 + 2 * li + 32 * h;
    cl[h] = max(min(c[h], L - 2), 0);
  }
  d4 d[4];
#pragma unroll
  for (int u = 0; u < 4; u++) d[u] = d4{0.0, 0.0, 0.0, 0.0};
  u4 s = ps[0];
  d2 a[2] = {pa[0], pa[64]};
  for (int b = 0; b < nb; b++) {
    d2 xv[4][2];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int h = 0; h < 2; h++) {
        if (L >= 2) {
          xv[q][h] = __builtin_bit_cast(d2, __builtin_amdgcn_raw_buffer_load_b128(r, (s[q] + (uint32_t)cl[h]) * 8u, 0, 0));
        } else {
          xv[q][h][0] = xv[q][h][1] = __builtin_bit_cast(double, __builtin_amdgcn_raw_buffer_load_b64(r, s[q] * 8u, 0, 0));
        }
      }
    const d2 ac[2] = {a[0], a[1]};
    const int b1 = min(b + 1, nb - 1);
    s = ps[b1 * 4];
    a[0] = pa[b1 * 128];
    a[1] = pa[b1 * 128 + 64];
#pragma unroll
    for (int q = 0; q < 4; q++)
#pragma unroll
      for (int u = 0; u < 4; u++)
        d[u] = __builtin_amdgcn_mfma_f64_16x16x4f64(ac[q / 2][q % 2], xv[q][u / 2][u % 2], d[u], 0, 0, 0);
  }
  const int nr = cst(z.tnr)[t], f0 = cst(z.tfirst)[t];
  uint32_t out = take_out(d);
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const int row = 4 * lk + i;
    if (row < nr) {
      double* o = y + sec + (int64_t)(f0 + row) * L;
#pragma unroll
      for (int u = 0; u < 4; u++) {
        const int cu = cl[u / 2] + u % 2;
        if (cu >= c[u / 2] && cu < L) o[cu] += d[u][i];
      }
    }
  }
  for (; out; out &= out - 1) {
    const int q = __builtin_ctz(out), row = 4 * lk + (q >> 2), h = q >> 1 & 1;
    const int at = h ? c[1] : c[0], col = (h ? cl[1] : cl[0]) + (q & 1);
    if (row < nr && col >= at && col < L)
      again(z, x, y + sec + (int64_t)(f0 + row) * L, (int64_t)z.trow0[t] + row, col);
  }
}

// NN: a tile of 8 proton rows staged in LDS (16-byte pieces of a column's 8
// values, one array a piece, so that neighbouring columns are neighbours), one
// read of a column's entry (source column, value) serves all of them.  FP64
// stages 2,048 source columns at a time.  Each half of a row has a column of
// zeros before it, which the padding entries name: no padding reads an amplitude.
template <typename T>
__global__ __launch_bounds__(1024) void k_nn(Tab z, const T* __restrict__ x, T* __restrict__ y, int accumulate) {
  constexpr int R = kNnRows, V = 16 / (int)sizeof(T), NA = R / V;  // values a piece, pieces
  constexpr int C = sizeof(T) == 4 ? 4096 : 2048;
  struct alignas(16) Piece { T v[V]; };
  extern __shared__ __align__(16) unsigned char smem[];
  Piece* xs = reinterpret_cast<Piece*>(smem);
  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6), NW = blockDim.x >> 6;
  const int b = blockIdx.x;
  const int t = (b >> 8) * 256 + (b & 7) * 32 + ((b >> 3) & 31);
  if (t >= z.nnn) return;
  const int f0 = cst(z.nf0)[t], nr = cst(z.nnr)[t];
  const int cn = cst(z.pconj)[cst(z.psec)[f0]];
  const int L = cst(z.nlen)[cn], ncc = (L + 63) >> 6;
  // places of staged columns and zeros (stride of the pieces)
  const int cs = sizeof(T) == 4 ? L + 1 + (L > 2048) : min(L, C) + 1;
  const int64_t base = cst(z.pstart)[f0];
  constexpr int Q = 4;  // column chunks of a wave (rows up to 4096 columns)
  for (int h = 0; h < (sizeof(T) == 8 ? 2 : 1); h++) {
    const int h0 = h * C;
    if (h0 >= L) break;
    if (h) __syncthreads();
    if (tid < NA) {
      Piece u;
#pragma unroll
      for (int i = 0; i < V; i++) u.v[i] = T(0);
      xs[tid * cs] = u;
      if (sizeof(T) == 4 && L > 2048) xs[tid * cs + 2049] = u;
    }
    for (int c = tid; c < min(C, L - h0); c += blockDim.x) {
      const int at = c + 1 + (sizeof(T) == 4 && c >= 2048);
#pragma unroll
      for (int p = 0; p < NA; p++) {
        Piece u;
#pragma unroll
        for (int i = 0; i < V; i++) u.v[i] = p * V + i < nr ? x[base + (int64_t)(p * V + i) * L + h0 + c] : T(0);
        xs[p * cs + at] = u;
      }
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; q++) {
      const int cc = w + q * NW;
      if (cc >= ncc) break;
      T a[R];
#pragma unroll
      for (int r = 0; r < R; r++) a[r] = T(0);
      for (int hh = (sizeof(T) == 8 ? h : 0); hh < (sizeof(T) == 8 ? h + 1 : 2); hh++) {
        const uint32_t g = cst(z.nng)[(cn * 64 + cc) * 2 + hh];
        const int np = g & 1023;
        const uint32_t* ps = z.nsrc + (size_t)(g >> 10) * 64 + lane;
        const T* pv;
        if constexpr (sizeof(T) == 4) pv = z.nval32 + (size_t)(g >> 10) * 128 + lane;
        else pv = z.nval64 + (size_t)(g >> 10) * 128 + lane;
        // two rows (four entries) ahead
        uint32_t s0 = 0, s1 = 0;
        T v[4] = {T(0), T(0), T(0), T(0)};
        if (np > 0) {
          s0 = ps[0];
          s1 = ps[64];
#pragma unroll
          for (int i = 0; i < 4; i++) v[i] = pv[i * 64];
        }
        for (int p = 0; p < np; p += 2) {
          const uint32_t c0 = s0, c1 = s1;
          T u[4];
#pragma unroll
          for (int i = 0; i < 4; i++) u[i] = v[i];
          if (p + 2 < np) {
            ps += 128;
            pv += 256;
            s0 = ps[0];
            s1 = ps[64];
#pragma unroll
            for (int i = 0; i < 4; i++) v[i] = pv[i * 64];
          }
          const uint32_t col[4] = {c0 & 0xffffu, c0 >> 16, c1 & 0xffffu, c1 >> 16};
#pragma unroll
          for (int i = 0; i < 4; i++)
#pragma unroll
            for (int k = 0; k < NA; k++) {
              const Piece e = xs[k * cs + (sizeof(T) == 4 ? hh * 2049 : 0) + col[i]];
#pragma unroll
              for (int j = 0; j < V; j++) a[k * V + j] = fma(u[i], e.v[j], a[k * V + j]);
            }
        }
      }
      const int c = cc * 64 + lane;
      if (c < L) {
#pragma unroll
        for (int r = 0; r < R; r++)
          if (r < nr) {
            T* o = y + base + (int64_t)r * L + c;
            *o = accumulate || h ? *o + a[r] : a[r];
          }
      }
    }
  }
}

// A[block][lane][step] of the PP tiles from the merged entries by row
__global__ __launch_bounds__(256) void k_pp_fill(int ntile, const int32_t* row0, const int32_t* tnr, const int32_t* tblk,
                                                 const int32_t* usrc, const int64_t* pp_ptr, const int32_t* pp_src,
                                                 const double* pp_val, float* A32, double* A64) {  // (one of A32, A64)
  const int t = blockIdx.x;
  const int b0 = tblk[t], n = (tblk[t + 1] - b0) * 16;
  const int32_t* u = usrc + (int64_t)b0 * 16;
  for (int r = 0; r < tnr[t]; r++) {
    const int64_t f = row0[t] + r;
    for (int64_t e = pp_ptr[f] + threadIdx.x; e < pp_ptr[f + 1]; e += 256) {
      int lo = 0, hi = n - 1;
      while (lo < hi) {  // first place of the source in the sorted union
        const int m = (lo + hi) / 2;
        if (u[m] < pp_src[e]) lo = m + 1;
        else hi = m;
      }
      const int64_t blk = b0 + lo / 16;
      const int s = lo % 16 / 4, lk = lo % 4;
      if (A32) A32[(blk * 64 + lk * 16 + r) * 4 + s] = (float)pp_val[e];
      // FP64 result register i of lane group g is matrix row g + 4 i
      const int i = r / 4 + 4 * (r % 4);
      if (A64) A64[((blk * 2 + s / 2) * 64 + lk * 16 + i) * 2 + s % 2] = pp_val[e];
    }
  }
}

template <typename V>
V* get(Owner& o, size_t n) {
  void* p = nullptr;
  o.mem.reserve(o.mem.size() + 1);
  HIP_OK(hipMalloc(&p, std::max<size_t>(n, 1) * sizeof(V)));
  o.mem.push_back(p);
  return static_cast<V*>(p);
}
template <typename V>
V* put(Owner& o, const std::vector<V>& v, hipStream_t st) {
  V* p = get<V>(o, v.size());
  if (!v.empty()) {
    HIP_OK(hipMemcpyAsync(p, v.data(), v.size() * sizeof(V), hipMemcpyHostToDevice, st));
    HIP_OK(hipStreamSynchronize(st));
  }
  return p;
}

template <typename T>
void apply_t(const Owner& o, const T* x, T* y, int accumulate, hipStream_t st) {
  if (!o.ok[sizeof(T) == 4 ? 0 : 1]) throw std::runtime_error("like-particle tables missing");
  Tab z = o.t;
  if constexpr (sizeof(T) == 4) z.pA32 = o.pA32, z.nval32 = o.nval32;
  else z.pA64 = o.pA64, z.nval64 = o.nval64;
  constexpr int C = sizeof(T) == 4 ? 4096 : 2048;
  const int nw = std::min(16, (o.lmax + 63) / 64);
  const size_t lds = (size_t)(std::min(o.lmax, C) + 2) * kNnRows * sizeof(T);
  hipLaunchKernelGGL(k_nn<T>, dim3((o.t.nnn + 255) / 256 * 256), dim3(64 * nw), lds, st, z, x, y, accumulate);
  HIP_OK(hipGetLastError());
  if (o.t.npp > 0) {
    k_pp<<<o.t.npp, 256, 0, st>>>(z, x, y);
    HIP_OK(hipGetLastError());
  }
}

}  // namespace

void Owner::release() {
  for (void* p : mem) (void)hipFree(p);
  mem.clear();
  ok[0] = ok[1] = false;
  ntile = 0;
}

void apply(const Owner& o, const float* x, float* y, int accumulate, hipStream_t st) { apply_t<float>(o, x, y, accumulate, st); }
void apply(const Owner& o, const double* x, double* y, int accumulate, hipStream_t st) { apply_t<double>(o, x, y, accumulate, st); }

namespace {

// entries of the neutron columns n0 .. n0 + nl of one half (source columns below 2048 of
// the sector, from 2048 on): [lo, hi) of each, and the most of one
int half_entries(const bs::TwoBody& nn, int64_t sec, int64_t n0, int nl, int h, int64_t* lo, int64_t* hi) {
  int most = 0;
  for (int l = 0; l < nl; l++) {
    const auto b = nn.src.begin() + nn.rowptr[n0 + l], e = nn.src.begin() + nn.rowptr[n0 + l + 1];
    const auto m = std::lower_bound(b, e, (int32_t)(sec + 2048));
    lo[l] = (h ? m : b) - nn.src.begin();
    hi[l] = (h ? e : m) - nn.src.begin();
    most = std::max(most, (int)(hi[l] - lo[l]));
  }
  return most;
}

bool structure(Owner& o, const Host& g, hipStream_t st) {
  const bs::Tables& t = g.t;
  const std::vector<int32_t>& nlen_h = g.nlen_h;
  const bs::Species& P = t.sp[0];
  const bs::Species& N = t.sp[1];
  const int nP = (int)P.mask.size();
  int lmax = 0;
  for (int c : nlen_h) lmax = std::max(lmax, c);
  if (lmax < 1 || lmax > 4096 || t.call_spe || nP < 1) return false;
  // PP tiles: 16 rows of a sector, the union of their sources in blocks of 16
  std::vector<int32_t> row0, tnr, tL, tfirst, tblk(1, 0);
  std::vector<int64_t> tsec;
  std::vector<uint32_t> tbytes;
  for (int s = 0; s < P.nsec; s++) {
    const int L = nlen_h[P.conj[s]];
    const int64_t el = P.seccount[s] * L;
    if (el * 8 >= (int64_t)1 << 31) return false;  // a sector is addressed with 32-bit byte offsets
    for (int64_t f = 0; f < P.seccount[s]; f += kPpRows) {
      row0.push_back((int32_t)(P.secfirst[s] + f));
      tnr.push_back((int32_t)std::min<int64_t>(kPpRows, P.seccount[s] - f));
      tL.push_back(L);
      tfirst.push_back((int32_t)f);
      tsec.push_back(P.start[P.secfirst[s]]);
      tbytes.push_back((uint32_t)el);
    }
  }
  const int nt = (int)row0.size();
  std::vector<std::vector<int32_t>> uni(nt);
  bs::parallel(nt, [&](int i) {
    std::vector<int32_t>& u = uni[i];
    const int64_t a = t.tb[0].rowptr[row0[i]], b = t.tb[0].rowptr[row0[i] + tnr[i]];
    u.assign(t.tb[0].src.begin() + a, t.tb[0].src.begin() + b);
    std::sort(u.begin(), u.end());
    u.erase(std::unique(u.begin(), u.end()), u.end());
    while (!u.empty() && u.size() % 16) u.push_back(u.back());
  });
  std::vector<int32_t> usrc;
  std::vector<uint32_t> psrc;
  for (int i = 0; i < nt; i++) {
    const std::vector<int32_t>& u = uni[i];
    tblk.push_back(tblk.back() + (int)(u.size() / 16));
    usrc.insert(usrc.end(), u.begin(), u.end());
    for (size_t b = 0; b < u.size(); b += 16)
      for (int lk = 0; lk < 4; lk++)
        for (int s = 0; s < 4; s++) psrc.push_back((uint32_t)(P.start[u[b + 4 * s + lk]] - tsec[i]));
  }
  // items of 256 columns: sector after sector, columns after columns, so that
  // the tiles of an XCD's run share their source columns
  std::vector<uint64_t> items;
  for (int i = 0; i < nt;) {
    int j = i;
    while (j < nt && tsec[j] == tsec[i]) j++;
    for (int c = 0; c < tL[i]; c += 256)
      for (int q = i; q < j; q++)
        if (tblk[q + 1] > tblk[q]) items.push_back((uint64_t)q | (uint64_t)c << 32);
    i = j;
  }
  // workgroup b runs on XCD b % 8: runs of 32 consecutive items each
  std::vector<uint64_t> pitem;
  for (size_t b0 = 0; b0 < items.size(); b0 += 256)
    for (size_t b = b0; b < b0 + 256; b++) {
      const size_t i = b0 + (b & 7) * 32 + ((b >> 3) & 31);
      if (i < items.size()) pitem.push_back(items[i]);
    }
  // NN tiles and entries
  std::vector<int32_t> nf0, nnr;
  for (int s = 0; s < P.nsec; s++)
    for (int64_t f = 0; f < P.seccount[s]; f += kNnRows) {
      nf0.push_back((int32_t)(P.secfirst[s] + f));
      nnr.push_back((int32_t)std::min<int64_t>(kNnRows, P.seccount[s] - f));
    }
  std::vector<uint32_t> nng((size_t)N.nsec * 128, 0), nsrc;
  int64_t lo[64], hi[64];
  for (int c = 0; c < N.nsec; c++)
    for (int cc = 0; cc * 64 < nlen_h[c]; cc++)
      for (int h = 0; h < 2; h++) {
        const int nl = std::min(64, nlen_h[c] - cc * 64);
        const int np = (half_entries(t.tb[1], N.secfirst[c], N.secfirst[c] + cc * 64, nl, h, lo, hi) + 3) / 4 * 2;
        if (np > 1023) return false;
        const size_t o0 = nsrc.size() / 64;
        if (o0 >= (1u << 22)) return false;
        nng[((size_t)c * 64 + cc) * 2 + h] = (uint32_t)o0 << 10 | (uint32_t)np;
        // padding entries: value zero at the column of zeros
        nsrc.resize(nsrc.size() + (size_t)np * 64, 0u);
        for (int l = 0; l < nl; l++)
          for (int64_t q = lo[l]; q < hi[l]; q++) {
            const int i = (int)(q - lo[l]);
            const uint32_t sc = (uint32_t)(t.tb[1].src[q] - N.secfirst[c]) - 2048u * h + 1u;
            nsrc[(o0 + i / 2) * 64 + l] |= sc << (16 * (i % 2));
          }
      }
  Tab& d = o.t;
  d = Tab{};
  d.npp = (int)pitem.size();
  d.nnn = (int)nf0.size();
  d.pitem = put(o, pitem, st);
  d.tsec = put(o, tsec, st);
  d.tbytes = put(o, tbytes, st);
  d.tfirst = put(o, tfirst, st);
  d.tnr = put(o, tnr, st);
  d.tL = put(o, tL, st);
  d.tblk = put(o, tblk, st);
  d.psrc = put(o, psrc, st);
  d.nf0 = put(o, nf0, st);
  d.nnr = put(o, nnr, st);
  d.psec = g.psec;
  d.pconj = g.pconj;
  d.nlen = g.nlen;
  d.pstart = g.pstart;
  d.nng = put(o, nng, st);
  d.nsrc = put(o, nsrc, st);
  d.trow0 = put(o, row0, st);
  d.pp_ptr = g.pp_ptr;
  d.pp_src = g.pp_src;
  d.pp_val = g.pp_val;
  o.usrc = put(o, usrc, st);
  o.blocks = tblk.back();
  o.nrows = (int64_t)nsrc.size() / 64;
  o.nng = std::move(nng);
  o.lmax = lmax;
  for (const void* fn : {reinterpret_cast<const void*>(k_nn<float>), reinterpret_cast<const void*>(k_nn<double>)})
    HIP_OK(hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024));
  o.ntile = nt;
  return true;
}

// the PP coefficients and the NN values of one type
template <typename T>
void values(Owner& o, const Host& g, const T** pA, const T** nval, hipStream_t st) {
  const bs::Species& N = g.t.sp[1];
  const size_t na = std::max<size_t>((size_t)o.blocks * 256, 1);
  T* A = get<T>(o, na);
  HIP_OK(hipMemsetAsync(A, 0, na * sizeof(T), st));
  if constexpr (sizeof(T) == 4)
    k_pp_fill<<<o.ntile, 256, 0, st>>>(o.ntile, o.t.trow0, o.t.tnr, o.t.tblk, o.usrc, g.pp_ptr, g.pp_src, g.pp_val, A, nullptr);
  else
    k_pp_fill<<<o.ntile, 256, 0, st>>>(o.ntile, o.t.trow0, o.t.tnr, o.t.tblk, o.usrc, g.pp_ptr, g.pp_src, g.pp_val, nullptr, A);
  HIP_OK(hipGetLastError());
  std::vector<T> v((size_t)o.nrows * 128, T(0));
  int64_t lo[64], hi[64];
  for (int c = 0; c < N.nsec; c++)
    for (int cc = 0; cc * 64 < g.nlen_h[c]; cc++)
      for (int h = 0; h < 2; h++) {
        const int nl = std::min(64, g.nlen_h[c] - cc * 64);
        half_entries(g.t.tb[1], N.secfirst[c], N.secfirst[c] + cc * 64, nl, h, lo, hi);
        T* at = v.data() + (size_t)(o.nng[((size_t)c * 64 + cc) * 2 + h] >> 10) * 128;
        for (int l = 0; l < nl; l++)
          for (int64_t q = lo[l]; q < hi[l]; q++) at[(q - lo[l]) * 64 + l] = (T)g.t.tb[1].val[q];
      }
  *nval = put(o, v, st);  // (waits for k_pp_fill too)
  HIP_OK(hipStreamSynchronize(st));
  *pA = A;
}

}  // namespace

void build(Owner& o, const Host& g, bool f32, hipStream_t st) {
  if (o.ok[f32 ? 0 : 1]) return;
  const size_t had = o.mem.size();
  try {
    if (!o.ntile && !structure(o, g, st)) return;
    if (f32) values<float>(o, g, &o.pA32, &o.nval32, st);
    else values<double>(o, g, &o.pA64, &o.nval64, st);
    o.ok[f32 ? 0 : 1] = true;
  } catch (...) {  // the other type keeps what it has
    (void)hipStreamSynchronize(st);
    for (size_t i = had; i < o.mem.size(); i++) (void)hipFree(o.mem[i]);
    o.mem.resize(had);
    if (!had) o.ntile = 0;
    throw;
  }
}

}  // namespace bsl
