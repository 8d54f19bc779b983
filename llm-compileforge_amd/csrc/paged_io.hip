// Paged-cache row I/O kernels.
//
// paged_write: token i's row goes to slot slots[i] = block * bs + offset of
// a [NB, bs, H, D] cache (the reference's token placement,
// python_runtime/engine/cache_manager.py:139-171 and _kv_cache.py:68-104),
// converted to the cache dtype: e4m3fn codes are e4m3_from_f32(x / scale[h])
// (FP8KVCacheQuantizer's arithmetic, compiler/quantize/fp8_kv_cache.py:89),
// bf16 / fp16 round to nearest even, f32 is exact.  Slots outside
// [0, NB * bs) are skipped.
//
// paged_gather: out[r, s] = the row of token s of table r (block
// tables[r][s / bs], offset s % bs), dequantized (e4m3fn: code * scale[h]);
// a table entry outside [0, NB) gives zeros (the reference gathers a
// request's blocks in table order and leaves positions past its table zero,
// cache_manager.py:173-197).
//
// A thread of the row kernels takes a piece of one (token, head) row: as many
// channels as make 16 bytes of the wider side where rows are contiguous and
// aligned (so a wave's accesses on that side are whole 1 KiB runs), one
// channel in small calls otherwise, and a piece with one side or both moved by
// element in large ones.  Channel-major caches of whole 16-token pieces (the
// native V layout: the tokens of a channel are contiguous) have kernels of
// their own for all but small calls, a thread taking one channel's 16 tokens:
// every access is then a run along the channels or along the tokens.  All are
// bound by latency for a decode step's rows and by bytes for a prompt's.
#include <algorithm>

#include "cf_device.hpp"
#include "cf_host.hpp"
#include "paged_io.hpp"

namespace cf {

namespace {

template <int DT>
__device__ __forceinline__ float load_as_f32(const void* base, int64_t i) {
  using E = Elem<DT>;
  return E::load((const typename E::T*)base + i);
}

template <int DT>
__device__ __forceinline__ void store_from_f32(void* base, int64_t i, float v) {
  using E = Elem<DT>;
  E::store((typename E::T*)base + i, v);
}

// Bytes of an element, and channels per piece of a pair of dtypes.
template <int DT>
constexpr int esize() {
  return (int)sizeof(typename Elem<DT>::T);
}
template <int A, int B>
constexpr int piece_channels() {
  return 16 / (esize<A>() > esize<B>() ? esize<A>() : esize<B>());
}

template <int BYTES>
struct Raw;
template <>
struct Raw<4> {
  using T = uint32_t;
};
template <>
struct Raw<8> {
  using T = uint2;
};
template <>
struct Raw<16> {
  using T = uint4;
};

// N consecutive elements (aligned accesses of 4, 8 or 16 bytes) as f32.
template <int DT, int N>
__device__ __forceinline__ void load_piece(const void* base, int64_t off, float* f) {
  using T = typename Elem<DT>::T;
  constexpr int B = N * esize<DT>(), W = B < 16 ? B : 16;
  using R = typename Raw<W>::T;
  union {
    R raw[B / W];
    T e[N];
  } u;
#pragma unroll
  for (int w = 0; w < B / W; ++w) u.raw[w] = ((const R*)((const T*)base + off))[w];
#pragma unroll
  for (int k = 0; k < N; ++k) f[k] = Elem<DT>::load(&u.e[k]);
}

// One value as DT's bits (e4m3fn: the code of f / scale).
template <int DT>
__device__ __forceinline__ typename Elem<DT>::T encode(float f, const Fp8Quant& qz) {
  typename Elem<DT>::T v;
  if constexpr (DT == kE4M3) v = qz(f);
  else Elem<DT>::store(&v, f);
  return v;
}

template <int DT, int N>
__device__ __forceinline__ void store_piece(void* base, int64_t off, const float* f, const Fp8Quant& qz) {
  using T = typename Elem<DT>::T;
  constexpr int B = N * esize<DT>(), W = B < 16 ? B : 16;
  using R = typename Raw<W>::T;
  union {
    R raw[B / W];
    T e[N];
  } u;
  if constexpr (DT == kE4M3 && N == 16) {
    u.raw[0] = qz.pack16(f);
  } else {
#pragma unroll
    for (int k = 0; k < N; ++k) u.e[k] = encode<DT>(f[k], qz);
  }
#pragma unroll
  for (int w = 0; w < B / W; ++w) ((R*)((T*)base + off))[w] = u.raw[w];
}

// The same at an element stride, where a side's rows are not whole 16-byte runs.
template <int DT, int N>
__device__ __forceinline__ void load_strided(const void* base, int64_t off, int64_t stride, float* f) {
#pragma unroll
  for (int k = 0; k < N; ++k) f[k] = load_as_f32<DT>(base, off + k * stride);
}
template <int DT, int N>
__device__ __forceinline__ void store_strided(void* base, int64_t off, int64_t stride, const float* f,
                                              const Fp8Quant& qz) {
#pragma unroll
  for (int k = 0; k < N; ++k) ((typename Elem<DT>::T*)base)[off + k * stride] = encode<DT>(f[k], qz);
}

template <int ST>
__device__ __forceinline__ int64_t slot_of(const PagedWriteParams& p, int64_t i) {
  return ST == kI64 ? ((const int64_t*)p.slots)[i * p.slot_s] : (int64_t)((const int32_t*)p.slots)[i * p.slot_s];
}

// Workgroups of a launch in a grid of grid_of(): x first, then y.
constexpr int kGridRowBits = 23;
__device__ __forceinline__ int64_t block_index() { return ((int64_t)blockIdx.y << kGridRowBits) | blockIdx.x; }

// One thread per piece of N channels (N == 1: any strides).  VEC: both sides
// move in whole pieces; otherwise the sides that xvec / cvec name.
template <int XT, int ST, int CT, int N, bool VEC>
__global__ __launch_bounds__(256) void paged_write_kernel(PagedWriteParams p, bool xvec, bool cvec) {
  const int np = p.D / N;
  const int64_t u = block_index() * 256 + threadIdx.x;
  const int64_t total = p.T * p.H * np;
  if (u >= total) return;
  int64_t i;
  int h, c;
  if (total <= (int64_t)UINT32_MAX) {  // 32-bit divisions
    const uint32_t v = (uint32_t)u, r = v / (uint32_t)np;
    c = (int)(v - r * (uint32_t)np);
    i = r / (uint32_t)p.H;
    h = (int)(r - (uint32_t)i * (uint32_t)p.H);
  } else {
    c = (int)(u % np), h = (int)((u / np) % p.H);
    i = u / ((int64_t)np * p.H);
  }
  float f[N];
  const int64_t xo = i * p.x_s[0] + h * p.x_s[1] + (int64_t)c * N * p.x_s[2];
  if constexpr (N == 1) f[0] = load_as_f32<XT>(p.x, xo);
  else if (VEC || xvec) load_piece<XT, N>(p.x, xo, f);
  else load_strided<XT, N>(p.x, xo, p.x_s[2], f);
  // (read before the slot is known: one round trip instead of two)
  const float sc = CT == kE4M3 ? p.scale[h * p.sc_s] : 1.0f;
  const int64_t sl = slot_of<ST>(p, i);
  if (sl < 0 || sl >= p.NB * p.bs) return;
  // (32-bit division wherever the slot fits)
  const int64_t blk = (sl >> 32) == 0 ? (int64_t)((uint32_t)sl / (uint32_t)p.bs) : sl / p.bs, off = sl - blk * p.bs;
  const Fp8Quant qz(sc);
  const int64_t co = blk * p.c_s[0] + off * p.c_s[1] + h * p.c_s[2] + (int64_t)c * N * p.c_s[3];
  if constexpr (N == 1) ((typename Elem<CT>::T*)p.cache)[co] = encode<CT>(f[0], qz);
  else if (VEC || cvec) store_piece<CT, N>(p.cache, co, f, qz);
  else store_strided<CT, N>(p.cache, co, p.c_s[3], f, qz);
}

// Channel-major blocks of whole 16-token pieces (token stride 1): a
// workgroup takes 16 new rows of 256 (head, channel)s, a thread one channel.
// Rows are split into runs of consecutive slots inside one piece; the group
// writes the runs that start in it (the last may reach up to 15 rows past
// it), a run of 16 as the piece's whole channel row.  Run boundaries depend
// only on the slots, so every thread of the group writes the same runs.
template <int XT, int ST, int CT>
__global__ __launch_bounds__(256) void paged_write_tile_kernel(PagedWriteParams p, uint32_t chunks) {
  using X = typename Elem<XT>::T;
  using C = typename Elem<CT>::T;
  const uint32_t block = (uint32_t)block_index(), g = block / chunks;
  if ((int64_t)g * 16 >= p.T) return;  // past the last group
  // Rows are read from lanes by their number, so no lane of a wave may leave on
  // its own: lanes past the last channel repeat it (the same bytes to the same
  // place), and only whole waves past it leave.
  const int hd0 = (int)(block - g * chunks) * 256 + (int)threadIdx.x;
  if (hd0 - (int)(threadIdx.x & 63) >= p.H * p.D) return;
  const int hd = min(hd0, p.H * p.D - 1);
  const int h = hd / p.D, d = hd % p.D;
  // lane l: the slot of row g * 16 - 1 + l (-1 outside [0, T))
  const int lane = (int)(threadIdx.x & 63);
  const int64_t r = (int64_t)g * 16 - 1 + lane;
  const int64_t sl = r >= 0 && r < p.T ? slot_of<ST>(p, r) : -1;
  // rows g*16 .. g*16+30 of this channel (clamped to the last row), loaded
  // while the slots are in flight
  const int64_t row0 = (int64_t)g * 16;
  const int last = (int)(p.T - 1 - row0 < 30 ? p.T - 1 - row0 : 30);
  const float sc = CT == kE4M3 ? p.scale[h * p.sc_s] : 1.0f;
  const X* src = (const X*)p.x + row0 * p.x_s[0] + h * p.x_s[1] + (int64_t)d * p.x_s[2];
  X raw[31];
#pragma unroll
  for (int e = 0; e < 31; ++e) raw[e] = src[(int64_t)(e < last ? e : last) * p.x_s[0]];
  const bool valid = sl >= 0 && sl < p.NB * p.bs;
  const int64_t up = __shfl_up(sl, 1, 64);
  const bool cont = valid && lane > 0 && sl == up + 1 && (sl & 15) != 0;
  const uint32_t vm = (uint32_t)__ballot(valid), cm = (uint32_t)__ballot(cont);
  // lane 1 + e <-> row e of the group
  const int64_t blk = p.bs == 16 ? sl >> 4 : sl / p.bs;
  const int64_t dst = valid ? blk * p.c_s[0] + (sl - blk * p.bs) : 0;
  const uint32_t starts = vm & ~cm & 0x1FFFEu;
  if (starts == 0u) return;  // uniform
  const int e0 = __builtin_ctz(starts) - 1;    // first owned row, 0..15
  const int ext = __builtin_ctz(~(cm >> 17));  // rows past the group that continue its last run, <= 15
  const uint32_t own = ((vm & 0x1FFFEu & ~((2u << e0) - 1u)) >> 1) | (((1u << ext) - 1u) << 16);
  C* chan = (C*)p.cache + (int64_t)h * p.c_s[2] + (int64_t)d * p.c_s[3];
  auto dst_of = [&](int e) {  // row e's block and token offset (uniform)
    const uint32_t lo = __builtin_amdgcn_readlane((uint32_t)(uint64_t)dst, e + 1);
    const uint32_t hi = __builtin_amdgcn_readlane((uint32_t)((uint64_t)dst >> 32), e + 1);
    return (int64_t)(((uint64_t)hi << 32) | lo);
  };
  const Fp8Quant qz(sc);
  if ((own >> e0) == 0xFFFFu && ((cm >> (e0 + 2)) & 0x7FFFu) == 0x7FFFu) {
    // 16 rows that fill a block's channel row
    union {
      uint4 q[esize<CT>()];
      C c[16];
    } out;
#pragma unroll
    for (int k = 0; k < 16; ++k) {
      if (e0 == k) {
#pragma unroll
        for (int j = 0; j < 16; ++j) out.c[j] = encode<CT>(Elem<XT>::load(&raw[k + j]), qz);
      }
    }
    uint4* to = (uint4*)(chan + dst_of(e0));
#pragma unroll
    for (int q = 0; q < esize<CT>(); ++q) to[q] = out.q[q];
    return;
  }
#pragma unroll
  for (int e = 0; e < 31; ++e)
    if ((own >> e) & 1u) chan[dst_of(e)] = encode<CT>(Elem<XT>::load(&raw[e]), qz);
}

template <int CT, int OT, int N, bool VEC>
__global__ __launch_bounds__(256) void paged_gather_kernel(PagedGatherParams p, bool cvec, bool ovec) {
  const int np = p.D / N;
  const int64_t u = block_index() * 256 + threadIdx.x;
  const int64_t total = (int64_t)p.R * p.S * p.H * np;
  if (u >= total) return;
  int c, h, s, r;
  if (total <= (int64_t)UINT32_MAX) {
    const uint32_t v = (uint32_t)u, a = v / (uint32_t)np, b = a / (uint32_t)p.H;
    c = (int)(v - a * (uint32_t)np);
    h = (int)(a - b * (uint32_t)p.H);
    r = (int)(b / (uint32_t)p.S);
    s = (int)(b - (uint32_t)r * (uint32_t)p.S);
  } else {
    c = (int)(u % np), h = (int)((u / np) % p.H);
    const int64_t rs = u / ((int64_t)np * p.H);
    s = (int)(rs % p.S), r = (int)(rs / p.S);
  }
  const int jb = s / p.bs;
  int64_t blk = -1;
  if (jb < p.Mb) {
    const int id = p.tables[(int64_t)r * p.t_sr + (int64_t)jb * p.t_sm];
    if (id >= 0 && id < p.NB) blk = id;
  }
  float f[N];
  if (blk >= 0) {
    const int64_t co =
        blk * p.c_s[0] + (int64_t)(s - jb * p.bs) * p.c_s[1] + h * p.c_s[2] + (int64_t)c * N * p.c_s[3];
    if constexpr (N == 1) f[0] = load_as_f32<CT>(p.cache, co);
    else if (VEC || cvec) load_piece<CT, N>(p.cache, co, f);
    else load_strided<CT, N>(p.cache, co, p.c_s[3], f);
    if constexpr (CT == kE4M3) {
      const float sc = p.scale[h * p.sc_s];
#pragma unroll
      for (int e = 0; e < N; ++e) f[e] *= sc;
    }
  } else {
#pragma unroll
    for (int e = 0; e < N; ++e) f[e] = 0.0f;
  }
  const int64_t oo = (int64_t)r * p.o_s[0] + (int64_t)s * p.o_s[1] + h * p.o_s[2] + (int64_t)c * N * p.o_s[3];
  if constexpr (N == 1) store_from_f32<OT>(p.out, oo, f[0]);
  else if (VEC || ovec) store_piece<OT, N>(p.out, oo, f, Fp8Quant(1.0f));
  else store_strided<OT, N>(p.out, oo, p.o_s[3], f, Fp8Quant(1.0f));
}

// Channel-major 16-token pieces into token rows: a thread reads the 16 tokens
// of P adjacent channels of one piece (whole runs along the channels) and
// writes them to the 16 rows, P channels a store (4 bytes: 256-byte runs).
template <int CT, int OT, int P>
__global__ __launch_bounds__(256) void paged_gather_tile_kernel(PagedGatherParams p, int blocks_per_row) {
  using C = typename Elem<CT>::T;
  using O = typename Elem<OT>::T;
  const uint32_t per = (uint32_t)(p.H * p.D / P);
  const int64_t u = block_index() * 256 + threadIdx.x;
  const int64_t total = (int64_t)p.R * blocks_per_row * per;
  if (u >= total) return;
  int64_t rb;
  int r;
  if (total <= (int64_t)UINT32_MAX) {
    rb = (uint32_t)u / per;
    r = (int)((uint32_t)rb / (uint32_t)blocks_per_row);
  } else {
    rb = u / per;
    r = (int)(rb / blocks_per_row);
  }
  const int hd = (int)(u - rb * per) * P;
  const int piece = (int)(rb - (int64_t)r * blocks_per_row), s0 = piece * 16;  // first token
  const int jb = p.bs == 16 ? piece : (int)((uint32_t)s0 / (uint32_t)p.bs);
  const int h = hd / p.D, d = hd - h * p.D;
  int64_t blk = -1;
  if (jb < p.Mb) {
    const int id = p.tables[(int64_t)r * p.t_sr + (int64_t)jb * p.t_sm];
    if (id >= 0 && id < p.NB) blk = id;
  }
  union {
    uint4 q[P][esize<CT>()];
    C c[P][16];
  } in;
  if (blk >= 0) {
    const C* src = (const C*)p.cache + blk * p.c_s[0] + (int64_t)h * p.c_s[2] + (int64_t)d * p.c_s[3] + (s0 - jb * p.bs);
#pragma unroll
    for (int k = 0; k < P; ++k)
#pragma unroll
      for (int q = 0; q < esize<CT>(); ++q) in.q[k][q] = ((const uint4*)(src + k * p.c_s[3]))[q];
  }
  const float sc = CT == kE4M3 ? p.scale[h * p.sc_s] : 1.0f;
  const int ns = min(16, p.S - s0);
  O* out = (O*)p.out + (int64_t)r * p.o_s[0] + (int64_t)s0 * p.o_s[1] + (int64_t)h * p.o_s[2] + d;
#pragma unroll
  for (int t = 0; t < 16; ++t) {
    if (t < ns) {
      O v[P];
#pragma unroll
      for (int k = 0; k < P; ++k) {
        float f = blk >= 0 ? Elem<CT>::load(&in.c[k][t]) : 0.0f;
        if constexpr (CT == kE4M3) f = blk >= 0 ? f * sc : 0.0f;
        Elem<OT>::store(&v[k], f);
      }
      if constexpr (P * sizeof(O) == 4) *(uint32_t*)(out + (int64_t)t * p.o_s[1]) = __builtin_bit_cast(uint32_t, v);
      else out[(int64_t)t * p.o_s[1]] = v[0];
    }
  }
}

// Whether rows at element strides `strides` (and base) start on multiples of
// `bytes` and are contiguous along the channels.
bool rows_aligned(const void* base, const int64_t* strides, int n_outer, int64_t inner, int eb, int bytes) {
  if (inner != 1 || ((uintptr_t)base & (uintptr_t)(bytes - 1))) return false;
  for (int i = 0; i < n_outer; ++i)
    if ((strides[i] * eb) % bytes != 0) return false;
  return true;
}

// Channel-major blocks (the native V layout) of whole 16-token pieces, each
// 16-byte aligned.
bool channel_tiles(const void* base, const int64_t* c_s, int bs, int eb) {
  return bs % 16 == 0 && c_s[1] == 1 && ((uintptr_t)base & 15) == 0 && (c_s[0] * eb) % 16 == 0 &&
         (c_s[2] * eb) % 16 == 0 && (c_s[3] * eb) % 16 == 0;
}

// Workgroups of 256 threads for `threads`, and the grid that holds them: a
// dimension of 2^32 threads or more is launched modulo 2^32, without an error.
int64_t blocks_of(int64_t threads) { return (threads + 255) / 256; }
dim3 grid_of(int64_t blocks) {
  constexpr int64_t row = (int64_t)1 << kGridRowBits;
  return dim3((unsigned)std::min(blocks, row), (unsigned)ceil_div(blocks, row));
}

// Values (rows x channels) from which channel-major blocks are written by whole
// 16-token pieces.  A thread there walks 16 rows, which takes 3.0-3.6 us (4.4-5.4
// into e4m3fn) where runs fill their pieces and 5.5 us where they do not,
// however few they are; a thread per element is done in 2.5 us for a decode
// step, but writes 1 to 4 bytes of every 16 to 64.  By element / by piece, whole
// runs / short ones: 512,000 fp16 values 4.2 / 3.3 / 5.5 us, 768,000 6.8 / 3.7 /
// 5.5 us; into e4m3fn 512,000 values 4.4 / 5.3 us, 768,000 6.3 / 5.4 us.
constexpr int64_t kTileWriteValues = 5 << 17;
// The same for gathers (3.3 us by pieces, 4.7 from e4m3fn): 256,000
// fp32 values 3.2 / 3.4 us, 384,000 3.8 / 3.5 us; e4m3fn 384,000 3.9 / 4.8 us,
// 768,000 5.7 / 4.9 us.
template <int CT>
constexpr int64_t tile_gather_values() {
  return CT == kE4M3 ? 1 << 19 : 1 << 18;
}
// Values from which unit-stride rows that are not 16-byte aligned go by pieces
// as well, loaded or stored by element on the unaligned side (4,000 fp16 rows
// of 8 heads of 128: 15.7 us by element, 8.6 us; 32 rows: 2.3, 2.7 us).
constexpr int64_t kPieceValues = 1 << 18;
// fp32 rows into e4m3fn from this many values on: 16 channels a thread, so that
// a cache row is stored in 16-byte pieces (4,000 rows of 8 heads of 128: 7.1 us
// by 4 channels, 5.2 us by 16; 1,000 rows 3.5, 3.6 us.  16-bit rows gain nothing:
// 6.7 us by 8 channels, 6.6 us by 16).
constexpr int64_t kWholePieceValues = 1 << 21;
// Rows with a channel stride on either side: 16 (gathers: 8) channels a thread
// put several tokens, which such layouts keep side by side, in a wave.  New rows
// with one: 4,000 fp16 rows of 8 heads of 128 15.4 us by element, 7.9 us; 500
// rows into e4m3fn 3.9, 5.9 us.  Caches with one, heads x head_dim below 1,024:
// fp32 rows of 4 heads of 64, 500 of them 3.5, 4.0 us, 1,000 4.8, 4.1, 2,000 7.3,
// 4.2; with 8 heads of 128 a wave holds one token either way.
constexpr int64_t kStridedRowValues = 7 << 17;
constexpr int64_t kStridedCacheValues = 7 << 15;
constexpr int64_t kStridedGatherValues = 5 << 17;

template <int XT, int ST, int CT, int N, bool VEC>
int32_t launch_write_n(const PagedWriteParams& p, hipStream_t stream) {
  const bool xv = VEC || rows_aligned(p.x, p.x_s, 2, p.x_s[2], esize<XT>(), std::min(16, N * esize<XT>()));
  const bool cv = VEC || rows_aligned(p.cache, p.c_s, 3, p.c_s[3], esize<CT>(), std::min(16, N * esize<CT>()));
  const int64_t blocks = blocks_of(p.T * p.H * (p.D / N));
  CF_CHECK(blocks < (int64_t)INT32_MAX, "paged write too large");
  CF_LAUNCH((paged_write_kernel<XT, ST, CT, N, VEC>), grid_of(blocks), dim3(256), 0, stream, p, xv, cv);
  CF_HIP_CHECK(hipGetLastError());
  return CF_OK;
}

template <int XT, int ST, int CT>
int32_t launch_write_t(const PagedWriteParams& p, hipStream_t stream) {
  ProfileScope prof("cf_paged_write", stream);
  const int64_t values = p.T * p.H * p.D;
  if (values >= kTileWriteValues && channel_tiles(p.cache, p.c_s, p.bs, esize<CT>())) {
    const int64_t chunks = blocks_of((int64_t)p.H * p.D), blocks = ceil_div(p.T, 16) * chunks;
    CF_CHECK(blocks < (int64_t)INT32_MAX, "paged write too large");
    CF_LAUNCH((paged_write_tile_kernel<XT, ST, CT>), grid_of(blocks), dim3(256), 0, stream, p, (uint32_t)chunks);
    CF_HIP_CHECK(hipGetLastError());
    return CF_OK;
  }
  auto whole = [&](int n) {  // both sides in aligned pieces of n channels
    return p.D % n == 0 &&
           rows_aligned(p.x, p.x_s, 2, p.x_s[2], esize<XT>(), std::min(16, n * esize<XT>())) &&
           rows_aligned(p.cache, p.c_s, 3, p.c_s[3], esize<CT>(), std::min(16, n * esize<CT>()));
  };
  if constexpr (CT == kE4M3 && XT == kF32) {
    if (values >= kWholePieceValues && whole(16)) return launch_write_n<XT, ST, CT, 16, true>(p, stream);
  }
  constexpr int N = piece_channels<XT, CT>();
  if (whole(N)) return launch_write_n<XT, ST, CT, N, true>(p, stream);
  const bool unit = p.x_s[2] == 1 && p.c_s[3] == 1;
  if (unit && p.D % N == 0 && values >= kPieceValues) return launch_write_n<XT, ST, CT, N, false>(p, stream);
  if (!unit && p.D % 16 == 0 &&
      (p.c_s[3] == 1 ? values >= kStridedRowValues : values >= kStridedCacheValues && (int64_t)p.H * p.D < 1024))
    return launch_write_n<XT, ST, CT, 16, false>(p, stream);
  return launch_write_n<XT, ST, CT, 1, false>(p, stream);
}

template <int XT, int ST>
int32_t launch_write_c(const PagedWriteParams& p, int cache_dt, hipStream_t stream) {
  switch (cache_dt) {
    case kF32: return launch_write_t<XT, ST, kF32>(p, stream);
    case kF16: return launch_write_t<XT, ST, kF16>(p, stream);
    case kBF16: return launch_write_t<XT, ST, kBF16>(p, stream);
    case kE4M3: return launch_write_t<XT, ST, kE4M3>(p, stream);
  }
  set_error("paged write: unsupported cache dtype %d", cache_dt);
  return CF_ERR_UNSUPPORTED;
}

template <int ST>
int32_t launch_write_x(const PagedWriteParams& p, int x_dt, int cache_dt, hipStream_t stream) {
  switch (x_dt) {
    case kF32: return launch_write_c<kF32, ST>(p, cache_dt, stream);
    case kF16: return launch_write_c<kF16, ST>(p, cache_dt, stream);
    case kBF16: return launch_write_c<kBF16, ST>(p, cache_dt, stream);
  }
  set_error("paged write: unsupported row dtype %d", x_dt);
  return CF_ERR_UNSUPPORTED;
}

template <int CT, int OT, int N, bool VEC>
int32_t launch_gather_n(const PagedGatherParams& p, hipStream_t stream) {
  const bool cv = VEC || rows_aligned(p.cache, p.c_s, 3, p.c_s[3], esize<CT>(), std::min(16, N * esize<CT>()));
  const bool ov = VEC || rows_aligned(p.out, p.o_s, 3, p.o_s[3], esize<OT>(), std::min(16, N * esize<OT>()));
  const int64_t blocks = blocks_of((int64_t)p.R * p.S * p.H * (p.D / N));
  CF_CHECK(blocks < (int64_t)INT32_MAX, "paged gather too large");
  CF_LAUNCH((paged_gather_kernel<CT, OT, N, VEC>), grid_of(blocks), dim3(256), 0, stream, p, cv, ov);
  CF_HIP_CHECK(hipGetLastError());
  return CF_OK;
}

template <int CT, int OT>
int32_t launch_gather_t(const PagedGatherParams& p, hipStream_t stream) {
  ProfileScope prof("cf_paged_gather", stream);
  const int64_t values = (int64_t)p.R * p.S * p.H * p.D;
  // Channels per thread of the tile kernel: 4 bytes of output, but one of
  // e4m3fn codes, whose conversion is the thread's time (4,000 rows of 8 heads
  // of 128 to bf16: 7.9 us by two channels, 7.1 by one; 32 rows 6.6, 4.7).
  constexpr int P = esize<OT>() == 4 || CT == kE4M3 ? 1 : 2;
  if (values >= tile_gather_values<CT>() && channel_tiles(p.cache, p.c_s, p.bs, esize<CT>()) && p.D % P == 0 &&
      (int64_t)p.H * p.D < INT32_MAX && rows_aligned(p.out, p.o_s, 3, p.o_s[3], esize<OT>(), P * esize<OT>())) {
    const int64_t bpr = ceil_div(p.S, 16), blocks = blocks_of((int64_t)p.R * bpr * (p.H * p.D / P));
    CF_CHECK(blocks < (int64_t)INT32_MAX, "paged gather too large");
    CF_LAUNCH((paged_gather_tile_kernel<CT, OT, P>), grid_of(blocks), dim3(256), 0, stream, p, (int)bpr);
    CF_HIP_CHECK(hipGetLastError());
    return CF_OK;
  }
  constexpr int N = piece_channels<CT, OT>();
  if (p.D % N == 0 && rows_aligned(p.cache, p.c_s, 3, p.c_s[3], esize<CT>(), N * esize<CT>()) &&
      rows_aligned(p.out, p.o_s, 3, p.o_s[3], esize<OT>(), N * esize<OT>()))
    return launch_gather_n<CT, OT, N, true>(p, stream);
  const bool unit = p.c_s[3] == 1 && p.o_s[3] == 1;
  if (unit && p.D % N == 0 && values >= kPieceValues) return launch_gather_n<CT, OT, N, false>(p, stream);
  if (!unit && p.D % 8 == 0 && values >= kStridedGatherValues) return launch_gather_n<CT, OT, 8, false>(p, stream);
  return launch_gather_n<CT, OT, 1, false>(p, stream);
}

template <int CT>
int32_t launch_gather_o(const PagedGatherParams& p, int out_dt, hipStream_t stream) {
  switch (out_dt) {
    case kF32: return launch_gather_t<CT, kF32>(p, stream);
    case kF16: return launch_gather_t<CT, kF16>(p, stream);
    case kBF16: return launch_gather_t<CT, kBF16>(p, stream);
  }
  set_error("paged gather: unsupported output dtype %d", out_dt);
  return CF_ERR_UNSUPPORTED;
}

}  // namespace

int32_t launch_paged_write(const PagedWriteParams& p, int x_dt, int slot_dt, int cache_dt, hipStream_t stream) {
  if (p.T == 0 || p.H == 0 || p.D == 0) return CF_OK;
  return slot_dt == kI64 ? launch_write_x<kI64>(p, x_dt, cache_dt, stream)
                         : launch_write_x<kI32>(p, x_dt, cache_dt, stream);
}

int32_t launch_paged_gather(const PagedGatherParams& p, int cache_dt, int out_dt, hipStream_t stream) {
  if (p.R == 0 || p.S == 0 || p.H == 0 || p.D == 0) return CF_OK;
  switch (cache_dt) {
    case kF32: return launch_gather_o<kF32>(p, out_dt, stream);
    case kF16: return launch_gather_o<kF16>(p, out_dt, stream);
    case kBF16: return launch_gather_o<kBF16>(p, out_dt, stream);
    case kE4M3: return launch_gather_o<kE4M3>(p, out_dt, stream);
  }
  set_error("paged gather: unsupported cache dtype %d", cache_dt);
  return CF_ERR_UNSUPPORTED;
}

// ---- upload of host-packed tables --------------------------------------------
// Copies n 16-byte words from device-visible pinned host memory into device
// memory: the upload rides the compute queue with the kernels that read it,
// so back-to-back calls hand nothing between the copy engine and the
// compute queue.  Host memory is read once: plain vector loads.
__global__ __launch_bounds__(256) void stage_from_host_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst,
                                                              int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) dst[i] = src[i];
}

int32_t launch_stage_from_host(const void* src_dev_view, void* dst, uint64_t bytes, hipStream_t stream) {
  const int64_t n = (int64_t)(bytes / 16);
  if (n == 0) return CF_OK;
  const int64_t blocks = std::min<int64_t>(ceil_div(n, 256), 64);
  ProfileScope prof("cf_stage_from_host", stream);
  CF_LAUNCH(stage_from_host_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, (const uint4*)src_dev_view,
            (uint4*)dst, n);
  CF_HIP_CHECK(hipGetLastError());
  return CF_OK;
}

}  // namespace cf
