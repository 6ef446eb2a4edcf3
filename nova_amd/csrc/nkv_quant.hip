// Asymmetric int8 quantize / dequantize kernels (token axis and channel axis).
//
// All of them are bound by memory, and small inputs by the latency of one pass: the quantizer of the
// token axis is therefore spread over a workgroup per group (below), and the others take tiles of 16 or
// 64 tokens x 128 channels, 8 channels of one to four rows per thread: 16-byte loads, one 128-element
// row = 256 contiguous bytes per 16 lanes, every load of a thread issued before the first is used.
#include "nkv_common.h"

#include <mutex>
#include <string>

namespace nkv {

static thread_local std::string g_err;

void set_error(const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
}

int fail(int code, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(NKV_ERR_HIP, "%s: launch failed: %s", what, hipGetErrorString(e));
  return NKV_OK;
}

// ---------------------------------------------------------------- element loads

template <int DT>
struct Elem8;

template <>
struct Elem8<NKV_F16> {
  static __device__ __forceinline__ void load(const void* base, int64_t off, float (&v)[8]) {
    uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + off);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = h2f((uint16_t)(w[i] & 0xffffu));
      v[2 * i + 1] = h2f((uint16_t)(w[i] >> 16));
    }
  }
};

template <>
struct Elem8<NKV_BF16> {
  static __device__ __forceinline__ void load(const void* base, int64_t off, float (&v)[8]) {
    uint4 u = *reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(base) + off);
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      v[2 * i] = __uint_as_float(w[i] << 16);
      v[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
    }
  }
};

template <>
struct Elem8<NKV_F32> {
  static __device__ __forceinline__ void load(const void* base, int64_t off, float (&v)[8]) {
    const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(base) + off);
    float4 a = p[0], b = p[1];
    v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
    v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
  }
};

__device__ __forceinline__ uint2 pack_codes8(const float (&x)[8], const float (&mn)[8],
                                             const float (&st)[8], const float (&inv)[8]) {
  float c[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) c[i] = ruler_code_f(x[i], mn[i], st[i], inv[i]);
  return pack_u8x8(c);
}

// How the 256 threads of a workgroup lie over rows of at most 64 channels: as many lanes to a row as it has
// 8-channel units, so that none idles (8 x 32768 rows of 8 channels, fp16: dequantized in 14.2 us with 15 of 16
// lanes idle, 4.9 so). Rows of 72 to 120 channels take the 16 lanes of 128: theirs would start off the cache
// lines (96 channels 15.2 against 18.0 us). mul: tid / lanes == tid * mul >> 16 (lanes <= 16, tid < 256).
struct TileLanes {
  uint32_t lanes, mul, rows;
  explicit TileLanes(int64_t dim)
      : lanes((uint32_t)std::min<int64_t>(16, dim / 8)), mul(65536u / lanes + 1), rows(256u / lanes) {}
  TileLanes() = default;
};

// The dequantizers give a thread one row up to 32768 rows of 128 channels (the latency of more would show: 1600 rows of
// fp16, token axis, 2.8 against 3.5 us), else four (262144 rows: 17.4 against 20.1 us).
// fp32 outputs are bound by their stores and take one row at every size (262144 rows, tok: 26.1 against 27.3 us).
static bool few_rows(int64_t rows, int out_dtype) { return rows <= 32768 || out_dtype == NKV_F32; }

__device__ __forceinline__ uint4 pack_h8(const float (&v)[8]) {
  uint4 r;
  r.x = (uint32_t)f2h(v[0]) | ((uint32_t)f2h(v[1]) << 16);
  r.y = (uint32_t)f2h(v[2]) | ((uint32_t)f2h(v[3]) << 16);
  r.z = (uint32_t)f2h(v[4]) | ((uint32_t)f2h(v[5]) << 16);
  r.w = (uint32_t)f2h(v[6]) | ((uint32_t)f2h(v[7]) << 16);
  return r;
}

// ---------------------------------------------------------------- token-axis quantize
//
// The format the decode path reads (src/nova/kvquant.py:136-149). W waves quantize one (slab, group of
// `gs` tokens, 128-channel chunk): lanes 0..15 of each 16 own 8 consecutive channels, the 4 W rows of
// 16 lanes stride over the group's tokens. Groups of at most 4 W R tokens stay in registers between the
// two passes (R rows per lane), longer ones are read twice. The extremes meet across a wave's four rows
// by lane swaps and across waves in LDS, where one thread per channel makes the ruler.
// Bound by memory at size and by one pass's latency below: 8 heads x 32768 fp16 tokens (100 MB moved)
// in 25 us (4.1 TB/s) against 42 us with one wave per group (128 values per lane, one chain of 2000
// instructions), 2048 tokens in 5.5 us against 12.6 us. One group of 2048 tokens per head: 31 us against 360 us.

struct QuantTokArgs {
  const void* x;
  int64_t x_rs;
  int64_t rows, n, dim, gs, ngroups, nchunks;
  uint8_t* codes;
  int64_t c_rs;
  uint16_t* mins;
  uint16_t* steps;
  int64_t s_rs;
  int64_t items;
  // page destination (paged cache): group gi of slab r goes to page table[first_group + gi], KV
  // head r, tensor `which` (0 K, 1 V) of the page layout [K codes 64 x 128 | V codes | kst | kmn |
  // vst | vmn]; groups whose table entry is outside [0, num_pages) are skipped
  uint8_t* pages;
  const int32_t* table;
  int64_t first_group, num_pages;
  int which;
};

constexpr int64_t PAGE_GROUP_BYTES = 2 * 64 * 128 + 4 * 128 * 2;  // 17408

template <int W>
struct QuantTokSmem {
  float ext[2][W][128];  // per wave: channel minima, maxima
  float rul[3][128];     // min, step, 1 / step
};

// The workgroup's rulers from its waves' channel extremes (lanes 8 cl .. + 7 of each 16): stores the
// `nch` channels' mins and steps, returns each lane's in mn, st, inv. Two barriers; calls may follow one
// another (one writes ext before its first barrier, and rul after it: no third barrier).
template <int W>
__device__ __forceinline__ void meet_rulers(QuantTokSmem<W>& sm, float (&mn)[8], const float (&mx)[8], float (&st)[8],
                                            float (&inv)[8], uint16_t* mins, uint16_t* steps, int nch) {
  const int t = threadIdx.x, lane = t & 63, wave = t >> 6, cl = t & 15;
  if (lane < 16) {
    float4* lo = reinterpret_cast<float4*>(sm.ext[0][wave] + 8 * cl);
    float4* hi = reinterpret_cast<float4*>(sm.ext[1][wave] + 8 * cl);
    lo[0] = make_float4(mn[0], mn[1], mn[2], mn[3]); lo[1] = make_float4(mn[4], mn[5], mn[6], mn[7]);
    hi[0] = make_float4(mx[0], mx[1], mx[2], mx[3]); hi[1] = make_float4(mx[4], mx[5], mx[6], mx[7]);
  }
  __syncthreads();
  if (t < 128) {
    float lo = sm.ext[0][0][t], hi = sm.ext[1][0][t];
#pragma unroll
    for (int w = 1; w < W; ++w) { lo = fminf(lo, sm.ext[0][w][t]); hi = fmaxf(hi, sm.ext[1][w][t]); }
    const float s = ruler_step(lo, hi);
    sm.rul[0][t] = lo;
    sm.rul[1][t] = s;
    sm.rul[2][t] = ruler_inv(s);
    if (t < nch) {
      mins[t] = f2h(lo);
      steps[t] = f2h(s);
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 8; j += 4) {
    const float4 m4 = *reinterpret_cast<const float4*>(sm.rul[0] + 8 * cl + j);
    const float4 s4 = *reinterpret_cast<const float4*>(sm.rul[1] + 8 * cl + j);
    const float4 i4 = *reinterpret_cast<const float4*>(sm.rul[2] + 8 * cl + j);
    mn[j] = m4.x; mn[j + 1] = m4.y; mn[j + 2] = m4.z; mn[j + 3] = m4.w;
    st[j] = s4.x; st[j + 1] = s4.y; st[j + 2] = s4.z; st[j + 3] = s4.w;
    inv[j] = i4.x; inv[j + 1] = i4.y; inv[j + 2] = i4.z; inv[j + 3] = i4.w;
  }
}

// W == 1: four independent items (one per wave) in a workgroup of 256 threads, no LDS. R == 0: the
// group's rows are read in a loop, twice.
template <int DT, int W, int R, bool PAGES = false>
__global__ __launch_bounds__(W == 1 ? 256 : 64 * W) void quant_token_kernel(QuantTokArgs a) {
  __shared__ __attribute__((aligned(16))) QuantTokSmem<W> sm;
  constexpr int RS = 4 * W;            // rows between a lane's rows
  constexpr int C = R > 0 ? R : 1;
  const int lane = threadIdx.x & 63, ti = W == 1 ? lane : (int)threadIdx.x;
  const int cl = ti & 15, rl = ti >> 4;
  const uint32_t items = (uint32_t)a.items, nchunks = (uint32_t)a.nchunks, ngroups = (uint32_t)a.ngroups;
  const uint32_t first = W == 1 ? blockIdx.x * 4 + (threadIdx.x >> 6) : blockIdx.x;
  for (uint32_t item = first; item < items; item += W == 1 ? gridDim.x * 4 : gridDim.x) {
    const uint32_t chunk = item % nchunks, rest = item / nchunks, gi = rest % ngroups, r = rest / ngroups;
    const int64_t ch = (int64_t)chunk * 128 + cl * 8;
    const bool active = ch < a.dim;
    const int64_t t0 = (int64_t)gi * a.gs;
    const int64_t nr = min(a.gs, a.n - t0);
    const int64_t base = r * a.x_rs + t0 * a.dim + ch;

    float mn[8], mx[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) { mn[j] = __builtin_huge_valf(); mx[j] = -__builtin_huge_valf(); }
    float cache[C][8];
    if (active) {
      if constexpr (R > 0) {
#pragma unroll
        for (int i = 0; i < R; ++i)  // (a row past the group repeats its last one: the extremes stay)
          Elem8<DT>::load(a.x, base + min<int64_t>(rl + RS * i, nr - 1) * a.dim, cache[i]);
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
          for (int j = 0; j < 8; ++j) { mn[j] = fminf(mn[j], cache[i][j]); mx[j] = fmaxf(mx[j], cache[i][j]); }
      } else {
#pragma unroll 4
        for (int64_t t = rl; t < nr; t += RS) {
          float v[8];
          Elem8<DT>::load(a.x, base + t * a.dim, v);
#pragma unroll
          for (int j = 0; j < 8; ++j) { mn[j] = fminf(mn[j], v[j]); mx[j] = fmaxf(mx[j], v[j]); }
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      mn[j] = min4rows(mn[j]);
      mx[j] = max4rows(mx[j]);
    }
    uint8_t* codes = a.codes + r * a.c_rs + t0 * a.dim;  // the group's first code row
    uint16_t* mins = a.mins + r * a.s_rs + (int64_t)gi * a.dim;
    uint16_t* steps = a.steps + r * a.s_rs + (int64_t)gi * a.dim;
    if constexpr (PAGES) {
      // token t of the group is row t of its page's code block; the rulers follow the code blocks
      const int32_t page = a.table[a.first_group + gi];
      if (page < 0 || page >= a.num_pages) continue;  // (the whole item agrees)
      uint8_t* pg = a.pages + ((int64_t)page * a.rows + r) * PAGE_GROUP_BYTES;
      codes = pg + a.which * 64 * 128;
      steps = reinterpret_cast<uint16_t*>(pg + 2 * 64 * 128) + a.which * 2 * 128;
      mins = steps + 128;
    }
    float st[8], inv[8];
    if constexpr (W == 1) {
#pragma unroll
      for (int j = 0; j < 8; ++j) { st[j] = ruler_step(mn[j], mx[j]); inv[j] = ruler_inv(st[j]); }
      if (active && rl == 0) {
        *reinterpret_cast<uint4*>(mins + ch) = pack_h8(mn);
        *reinterpret_cast<uint4*>(steps + ch) = pack_h8(st);
      }
    } else {
      meet_rulers<W>(sm, mn, mx, st, inv, mins + (int64_t)chunk * 128, steps + (int64_t)chunk * 128,
                     (int)min<int64_t>(128, a.dim - (int64_t)chunk * 128));
    }
    if (!active) continue;
    if constexpr (R > 0) {
#pragma unroll
      for (int i = 0; i < R; ++i) {
        const int64_t t = rl + RS * i;
        const uint2 c8 = pack_codes8(cache[i], mn, st, inv);
        if (t < nr) *reinterpret_cast<uint2*>(codes + t * a.dim + ch) = c8;
      }
    } else {
#pragma unroll 4
      for (int64_t t = rl; t < nr; t += RS) {
        float v[8];
        Elem8<DT>::load(a.x, base + t * a.dim, v);
        *reinterpret_cast<uint2*>(codes + t * a.dim + ch) = pack_codes8(v, mn, st, inv);
      }
    }
  }
}

template <int DT, int W, int R>
static void launch_quant_token_as(const QuantTokArgs& a, hipStream_t s) {
  const int64_t groups = W == 1 ? cdiv(a.items, 4) : a.items, most = 1 << 20;  // more are taken in turns
  hipLaunchKernelGGL((quant_token_kernel<DT, W, R>), dim3((unsigned)std::min(groups, most)), dim3(W == 1 ? 256 : 64 * W), 0, s, a);
}

// Waves per item, by the tokens of a group that there are (a slab can be shorter than one), and the rows
// that a lane keeps. A few waves per group hide the latency of one pass, but each of a group's waves costs
// the ruler's meeting, so short groups take no more than their rows fill: 16384 fp16 groups of 128 channels
// with one / two / four waves: 8 rows 19.7 / 32 / 44 us, 16 rows 27 / 35 / 45, 32 rows 42 / 39 / 49; few of
// them take four (512 of 16 rows 4.7 / 5.1 / 4.4, one of 32 5.5 / 4.4 / 3.7). 33 to 64 rows: four waves of 4 rows a lane (64 rows 82 us; two of 8 rows the
// same, and 5.7 against 4.5 us alone). Longer groups are read twice, by as many waves as leave each about
// 16 rows: of many groups (fp16, 4096: 65 rows 28.6 / 34 / 65 us with 4 / 8 / 16 waves, 128 rows 52 / 48 / 77,
// 512 groups of 512 rows 36 / 28 / 28), of few the more the rows (one group: 65 rows 5.7 / 4.9 / 5.2 us, 512
// rows 22 / 13 / 10.7). fp32 rows count twice.
template <int DT>
static void launch_quant_token(const QuantTokArgs& a, hipStream_t s) {
  const int64_t gr = std::min(a.gs, a.n), bytes = gr * (DT == NKV_F32 ? 4 : 2);
  if (gr <= 8) return launch_quant_token_as<DT, 1, 2>(a, s);
  if (gr <= 32 && a.items <= 1024) return launch_quant_token_as<DT, 4, 2>(a, s);
  if (gr <= 16) return launch_quant_token_as<DT, 1, 4>(a, s);
  if (gr <= 32) return launch_quant_token_as<DT, 2, 4>(a, s);
  if (gr <= 64) return launch_quant_token_as<DT, 4, 4>(a, s);
  const bool many = a.items >= 512;
  if constexpr (DT != NKV_F32)
    if (many && bytes <= 192) return launch_quant_token_as<DT, 4, 0>(a, s);
  if (many ? bytes <= 768 : gr <= 96) return launch_quant_token_as<DT, 8, 0>(a, s);
  launch_quant_token_as<DT, 16, 0>(a, s);
}

// ---------------------------------------------------------------- a prefill chunk lands in the cache
//
// One workgroup per (KV head, K or V, 64 tokens of the chunk) reads its rows once, from wherever the
// model left them (any token and head stride), and writes what the streaming cache keeps of them: the
// fp16 copy that the chunk's own attention reads, the newest 64 tokens' ring slots and, for a whole group,
// codes and rulers (as quant_token_kernel computes them). 2048 tokens x 8 heads of token-major fp16: one
// launch of 8 us against two copies, two quantizer launches and five small ones for the ring (about
// 37 us on the GPU).
struct LandArgs {
  const uint16_t* src[2];
  int64_t ts[2], hs[2];  // token and head strides
  int64_t n, start, capacity, ngroups_cap;
  int hkv;
  uint16_t* copy[2];     // [hkv][n][128]
  uint8_t* codes[2];     // [hkv][capacity][128]
  uint16_t* mins[2];     // [hkv][ngroups_cap][128]
  uint16_t* steps[2];
  uint16_t* ring[2];     // [hkv][64][128]
};

__global__ __launch_bounds__(256) void land_chunk_kernel(LandArgs a) {
  __shared__ __attribute__((aligned(16))) QuantTokSmem<4> sm;
  const int cl = threadIdx.x & 15, rl = threadIdx.x >> 4;
  const int h = blockIdx.x % a.hkv, which = blockIdx.x / a.hkv & 1;
  const int64_t g = blockIdx.x / (2 * a.hkv), t0 = g * 64;
  const int nr = (int)min<int64_t>(64, a.n - t0);
  const uint16_t* src = a.src[which] + h * a.hs[which] + t0 * a.ts[which] + 8 * cl;
  uint4 raw[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) raw[i] = *reinterpret_cast<const uint4*>(src + min(rl + 16 * i, nr - 1) * a.ts[which]);
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int r = rl + 16 * i;
    if (r >= nr) break;
    *reinterpret_cast<uint4*>(a.copy[which] + (h * a.n + t0 + r) * 128 + 8 * cl) = raw[i];
    if (t0 + r >= a.n - 64)
      *reinterpret_cast<uint4*>(a.ring[which] + ((int64_t)h * 64 + (a.start + t0 + r) % 64) * 128 + 8 * cl) = raw[i];
  }
  if (nr < 64) return;  // (a partial group stays in the ring)
  float v[4][8], mn[8], mx[8], st[8], inv[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) { mn[j] = __builtin_huge_valf(); mx[j] = -__builtin_huge_valf(); }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint32_t w[4] = {raw[i].x, raw[i].y, raw[i].z, raw[i].w};
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[i][j] = h2f((uint16_t)(w[j >> 1] >> (16 * (j & 1))));
      mn[j] = fminf(mn[j], v[i][j]);
      mx[j] = fmaxf(mx[j], v[i][j]);
    }
  }
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    mn[j] = min4rows(mn[j]);
    mx[j] = max4rows(mx[j]);
  }
  const int64_t so = ((int64_t)h * a.ngroups_cap + a.start / 64 + g) * 128;
  meet_rulers<4>(sm, mn, mx, st, inv, a.mins[which] + so, a.steps[which] + so, 128);
  uint8_t* codes = a.codes[which] + ((int64_t)h * a.capacity + a.start + t0 + rl) * 128 + 8 * cl;
#pragma unroll
  for (int i = 0; i < 4; ++i) *reinterpret_cast<uint2*>(codes + 16 * 128 * i) = pack_codes8(v[i], mn, st, inv);
}

// ---------------------------------------------------------------- channel-axis quantize

struct QuantChanArgs {
  const void* x;
  int64_t x_rs;
  int64_t rows, n, dim, gc, ngc;
  uint8_t* codes;
  int64_t c_rs;
  uint16_t* mins;
  uint16_t* steps;
  int64_t s_rs;
  int64_t items;  // rows * n * ngc
  TileLanes tl{};
};

template <int DT>
__device__ __forceinline__ float load1(const void* p, int64_t off) {
  if (DT == NKV_F16) return h2f(static_cast<const uint16_t*>(p)[off]);
  if (DT == NKV_BF16) return bf2f(static_cast<const uint16_t*>(p)[off]);
  return static_cast<const float*>(p)[off];
}

template <int DT>
__global__ __launch_bounds__(256) void quant_channel_kernel(QuantChanArgs a) {
  const int64_t item = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (item >= a.items) return;
  const int64_t g = item % a.ngc;
  const int64_t t = (item / a.ngc) % a.n;
  const int64_t r = item / (a.ngc * a.n);
  const int64_t xo = r * a.x_rs + t * a.dim + g * a.gc;
  float mn = __builtin_huge_valf(), mx = -__builtin_huge_valf();
  for (int64_t j = 0; j < a.gc; ++j) {
    float v = load1<DT>(a.x, xo + j);
    mn = fminf(mn, v);
    mx = fmaxf(mx, v);
  }
  const float st = ruler_step(mn, mx);
  const float inv = ruler_inv(st);
  const int64_t co = r * a.c_rs + t * a.dim + g * a.gc;
  for (int64_t j = 0; j < a.gc; ++j) a.codes[co + j] = (uint8_t)ruler_code_rcp(load1<DT>(a.x, xo + j), mn, st, inv);
  const int64_t so = r * a.s_rs + t * a.ngc + g;
  a.mins[so] = f2h(mn);
  a.steps[so] = f2h(st);
}

// The same for groups of 8, 16, 32, 64 or 128 channels and 16-byte rows: 16 tokens x 128 channels per
// workgroup (more tokens of narrower rows), 8 channels of one token per lane, a group's extremes over its gc / 8 lanes by lane swaps.
// 8 heads x 3001 bf16 tokens, groups of 32 / 64: 4.8 / 4.8 us against 22 / 33 us with a thread per group
// (2-byte loads, one byte per store); 32768 fp16 tokens, groups of 64: 24 against 1390 us. Four tokens per
// thread were slower at every size (2048 tokens: 5.4 against 4.0 us, 32768: 24.2 against 23.7 us).
template <int DT, int L, bool NARROW>  // L: lanes per group; NARROW: fewer than 128 channels (TileLanes)
__global__ __launch_bounds__(256) void quant_channel8_kernel(QuantChanArgs a) {
  const int rl = NARROW ? threadIdx.x * a.tl.mul >> 16 : threadIdx.x >> 4;
  const int cl = threadIdx.x - rl * (NARROW ? a.tl.lanes : 16);
  int64_t ch, t;
  uint32_t r;
  // (the lanes that leave are whole groups: dim is a multiple of gc, and a row's lanes are one of L)
  if constexpr (NARROW) {
    const uint32_t row = blockIdx.x * a.tl.rows + rl;
    if (rl >= (int)a.tl.rows || row >= (uint32_t)(a.rows * a.n)) return;
    r = row / (uint32_t)a.n;
    t = row - r * (uint32_t)a.n;
    ch = cl * 8;
  } else {
    const uint32_t nchunks = (uint32_t)((a.dim + 127) / 128), nblocks = (uint32_t)((a.n + 15) / 16);
    const uint32_t chunk = blockIdx.x % nchunks, rest = blockIdx.x / nchunks, tb = rest % nblocks;
    r = rest / nblocks;
    ch = (int64_t)chunk * 128 + cl * 8;
    t = (int64_t)tb * 16 + rl;
    if (ch >= a.dim || t >= a.n) return;
  }
  float v[8];
  Elem8<DT>::load(a.x, r * a.x_rs + t * a.dim + ch, v);
  float lo = __builtin_huge_valf(), hi = -__builtin_huge_valf();
#pragma unroll
  for (int j = 0; j < 8; ++j) { lo = fminf(lo, v[j]); hi = fmaxf(hi, v[j]); }
#pragma unroll
  for (int o = 1; o < L; o *= 2) { lo = fminf(lo, shfl_xor(lo, o)); hi = fmaxf(hi, shfl_xor(hi, o)); }
  const float st = ruler_step(lo, hi), inv = ruler_inv(st);
  float c[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) c[j] = ruler_code_f(v[j], lo, st, inv);
  *reinterpret_cast<uint2*>(a.codes + r * a.c_rs + t * a.dim + ch) = pack_u8x8(c);
  if (cl % L == 0) {
    const int64_t so = r * a.s_rs + t * a.ngc + ch / a.gc;
    a.mins[so] = f2h(lo);
    a.steps[so] = f2h(st);
  }
}

template <int DT, bool NARROW>
static void launch_quant_channel8(const QuantChanArgs& a, int64_t tiles, hipStream_t s) {
  const dim3 grid((unsigned)tiles), block(256);
  if (a.gc == 8) hipLaunchKernelGGL((quant_channel8_kernel<DT, 1, NARROW>), grid, block, 0, s, a);
  else if (a.gc == 16) hipLaunchKernelGGL((quant_channel8_kernel<DT, 2, NARROW>), grid, block, 0, s, a);
  else if (a.gc == 32) hipLaunchKernelGGL((quant_channel8_kernel<DT, 4, NARROW>), grid, block, 0, s, a);
  else if (a.gc == 64) hipLaunchKernelGGL((quant_channel8_kernel<DT, 8, NARROW>), grid, block, 0, s, a);
  else if constexpr (!NARROW) hipLaunchKernelGGL((quant_channel8_kernel<DT, 16, NARROW>), grid, block, 0, s, a);
}

template <int DT>
static void launch_quant_channel(QuantChanArgs a, bool wide, hipStream_t s) {
  if (wide && (a.gc == 8 || a.gc == 16 || a.gc == 32 || a.gc == 64 || a.gc == 128)) {
    const bool narrow = a.dim <= 64;
    if (narrow) a.tl = TileLanes(a.dim);
    const int64_t tiles = narrow ? cdiv(a.rows * a.n, (int64_t)a.tl.rows) : a.rows * cdiv(a.n, 16) * cdiv(a.dim, 128);
    if (tiles < (1 << 24)) {  // (a grid of at most 2^32 threads)
      if (narrow) launch_quant_channel8<DT, true>(a, tiles, s);
      else launch_quant_channel8<DT, false>(a, tiles, s);
      return;
    }
  }
  hipLaunchKernelGGL(quant_channel_kernel<DT>, dim3((unsigned)cdiv(a.items, 256)), dim3(256), 0, s, a);
}

// ---------------------------------------------------------------- dequantize

struct DequantArgs {
  const uint8_t* codes;
  int64_t c_rs;
  const uint16_t* mins;
  const uint16_t* steps;
  int64_t s_rs;
  int64_t rows, n, dim, group, axis;
  void* out;
  int64_t o_rs;
  int64_t items;  // tiles: rows * ceil(n / rows of a tile) * ceil(dim / 128)
  int vec;        // token axis: the rulers of 8 channels are 16-byte aligned
  TileLanes tl;
};

template <int OT>
__device__ __forceinline__ void store8(void* out, int64_t off, const float (&v)[8]) {
  if (OT == NKV_F16) {
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) + off) = pack_h8(v);
  } else if (OT == NKV_BF16) {
    uint4 r;
    r.x = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
    r.y = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
    r.z = (uint32_t)f2bf(v[4]) | ((uint32_t)f2bf(v[5]) << 16);
    r.w = (uint32_t)f2bf(v[6]) | ((uint32_t)f2bf(v[7]) << 16);
    *reinterpret_cast<uint4*>(static_cast<uint16_t*>(out) + off) = r;
  } else {
    float4* p = reinterpret_cast<float4*>(static_cast<float*>(out) + off);
    p[0] = make_float4(v[0], v[1], v[2], v[3]);
    p[1] = make_float4(v[4], v[5], v[6], v[7]);
  }
}

// 16 R tokens x 128 channels per workgroup (more tokens of narrower rows), R rows of 8 channels per thread. A lane's rulers are loaded
// once per group it meets: token axis 8 steps and 8 mins (two 16-byte loads when `vec`), channel axis one
// pair for its 8 channels when the group is a multiple of 8, else one per channel. 8 heads x 3001 /
// 32768 fp16 tokens, groups of 64: token axis 4.6 / 17.4 us against 8.7 / 64 us, channel axis 4.6 / 20 us
// against 7.9 / 49 us with a ruler load per value and 64-bit divisions.
template <int OT, int R, bool NARROW>
__global__ __launch_bounds__(256) void dequant_kernel(DequantArgs a) {
  const int rl = NARROW ? threadIdx.x * a.tl.mul >> 16 : threadIdx.x >> 4;
  const int cl = threadIdx.x - rl * (NARROW ? a.tl.lanes : 16);
  const uint32_t RR = NARROW ? a.tl.rows : 16;  // rows of a pass
  const bool token = a.axis == NKV_AXIS_TOKEN;
  if (NARROW && rl >= (int)RR) return;
  const uint32_t nchunks = (uint32_t)((a.dim + 127) / 128), nblocks = (uint32_t)((a.n + 16 * R - 1) / (16 * R));
  const uint32_t all = (uint32_t)(a.rows * a.n);  // (NARROW: the slabs' rows as one sequence)
  for (uint32_t tile = blockIdx.x; tile < (uint32_t)a.items; tile += gridDim.x) {
    uint32_t chunk = 0, r = 0;
    int64_t t0;
    if constexpr (NARROW) {
      t0 = (int64_t)tile * RR * R + rl;
    } else {
      const uint32_t rest = tile / nchunks;
      chunk = tile % nchunks;
      r = rest / nblocks;
      t0 = (int64_t)(rest % nblocks) * (16 * R) + rl;
    }
    const int64_t ch = (int64_t)chunk * 128 + cl * 8, last = (NARROW ? (int64_t)all : a.n) - 1;
    if (ch >= a.dim) continue;
    uint2 cw[R];
    [[maybe_unused]] uint32_t slab[R], tok[R];  // NARROW: of each pass's row
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if constexpr (NARROW) {
        const uint32_t row = (uint32_t)min(t0 + RR * i, last);
        slab[i] = row / (uint32_t)a.n;
        tok[i] = row - slab[i] * (uint32_t)a.n;
        cw[i] = *reinterpret_cast<const uint2*>(a.codes + slab[i] * a.c_rs + (int64_t)tok[i] * a.dim + ch);
      } else {
        cw[i] = *reinterpret_cast<const uint2*>(a.codes + r * a.c_rs + min(t0 + 16 * i, last) * a.dim + ch);
      }
    }
    float st[8], mn[8];
    int64_t have = -1;  // the group of st, mn (NARROW: the offset of its rulers)
#pragma unroll
    for (int i = 0; i < R; ++i) {
      if (t0 + RR * i > last) break;
      int64_t t = t0 + RR * i;
      if constexpr (NARROW) {
        r = slab[i];
        t = tok[i];
      }
      if (token) {
        // (32-bit: the tile count bounds n)
        const int64_t gi = (uint32_t)t / (uint32_t)a.group;
        const int64_t so = r * a.s_rs + gi * a.dim + ch, key = NARROW ? so : gi;
        if (key != have) {
          have = key;
          if (a.vec) {
            Elem8<NKV_F16>::load(a.steps, so, st);
            Elem8<NKV_F16>::load(a.mins, so, mn);
          } else {
#pragma unroll
            for (int j = 0; j < 8; ++j) { st[j] = h2f(a.steps[so + j]); mn[j] = h2f(a.mins[so + j]); }
          }
        }
      } else {
        const uint32_t ngc = (uint32_t)(a.dim / a.group);
        const int64_t so = r * a.s_rs + t * ngc;
        if (a.group % 8 == 0) {
          const uint32_t gc = (uint32_t)ch / (uint32_t)a.group;
          const float s1 = h2f(a.steps[so + gc]), m1 = h2f(a.mins[so + gc]);
#pragma unroll
          for (int j = 0; j < 8; ++j) { st[j] = s1; mn[j] = m1; }
        } else {
          // one division, then a ruler per group that the channels meet (with a division and two loads per
          // channel, groups of 4: 8 x 32768 rows of 80 channels 37.9 us, 21.0 so)
          uint32_t gc = (uint32_t)ch / (uint32_t)a.group, left = (gc + 1) * (uint32_t)a.group - (uint32_t)ch;
          float s1 = h2f(a.steps[so + gc]), m1 = h2f(a.mins[so + gc]);
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            if (left == 0) {
              ++gc;
              left = (uint32_t)a.group;
              s1 = h2f(a.steps[so + gc]);
              m1 = h2f(a.mins[so + gc]);
            }
            --left;
            st[j] = s1;
            mn[j] = m1;
          }
        }
      }
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t code = ((j < 4 ? cw[i].x : cw[i].y) >> (8 * (j & 3))) & 0xffu;
        // the product of an 8-bit code and an fp16 step is exact in fp32; one rounding in the add
        v[j] = __fadd_rn(__fmul_rn((float)code, st[j]), mn[j]);
      }
      store8<OT>(a.out, r * a.o_rs + t * a.dim + ch, v);
    }
  }
}

// ---------------------------------------------------------------- per-token symmetric ("tok")

// One (slab, token) row of 128 values per 16-lane row: lane l & 15 quantizes values
// 8 (l & 15) .. + 7 (16-byte loads, 8-byte code stores); a workgroup takes 16 tokens of one slab. The
// absmax is reduced with DPP within the 16-lane row. 8 heads x 8191 / 32768 fp16 tokens: 7.3 / 19.8 us against
// 9.7 / 29 us with an IEEE division per value and 64-bit divisions per thread (four tokens per thread:
// 8.3 / 20.5 us).
struct QuantSymArgs {
  const void* x;
  int64_t x_rs;
  int64_t rows, n;
  uint8_t* codes;
  int64_t c_rs;
  uint16_t* scales;
  int64_t s_rs;
  int64_t items;  // tiles: rows * ceil(n / rows of a tile)
  // page destination (paged cache): token t of slab r is token first_token + t of a sequence,
  // stored in page table[(first_token + t) / 64], KV head r, row (first_token + t) % 64 of
  // tensor `which` (0 K, 1 V) of the page layout [K codes 64 x 128 | V codes | K scales 64 |
  // V scales 64]; tokens whose table entry is outside [0, num_pages) are skipped
  uint8_t* pages;
  const int32_t* table;
  int64_t first_token, num_pages;
  int which;
};

constexpr int64_t PAGE_TOK_BYTES = 2 * 64 * 128 + 2 * 64 * 2;  // 16640

template <int DT, bool PAGES = false>
__global__ __launch_bounds__(256) void quant_sym_kernel(QuantSymArgs a) {
  const int c8 = (threadIdx.x & 15) * 8, rl = threadIdx.x >> 4;
  const uint32_t nblocks = (uint32_t)((a.n + 15) / 16);
  for (uint32_t tile = blockIdx.x; tile < (uint32_t)a.items; tile += gridDim.x) {
    const uint32_t tb = tile % nblocks, r = tile / nblocks;
    const int64_t t = (int64_t)tb * 16 + rl;
    if (t >= a.n) continue;  // (whole 16-lane rows agree)
    float v[8];
    Elem8<DT>::load(a.x, r * a.x_rs + t * 128 + c8, v);
    float scale;
    const uint2 cw = sym_quant8<true>(v, scale);
    uint8_t* code_row = a.codes + r * a.c_rs + t * 128;
    uint16_t* scale_at = a.scales + r * a.s_rs + t;
    if constexpr (PAGES) {
      const int64_t tok = a.first_token + t;
      const int32_t page = a.table[tok / 64];
      if (page < 0 || page >= a.num_pages) continue;
      uint8_t* pg = a.pages + ((int64_t)page * a.rows + r) * PAGE_TOK_BYTES;
      code_row = pg + a.which * 64 * 128 + (tok % 64) * 128;
      scale_at = reinterpret_cast<uint16_t*>(pg + 2 * 64 * 128) + a.which * 64 + tok % 64;
    }
    *reinterpret_cast<uint2*>(code_row + c8) = cw;
    if (c8 == 0) *scale_at = f2h(scale);
  }
}

struct DequantSymArgs {
  const uint8_t* codes;
  int64_t c_rs;
  const uint16_t* scales;
  int64_t s_rs;
  int64_t rows, n;
  void* out;
  int64_t o_rs;
  int64_t items;  // tiles: rows * ceil(n / rows of a tile)
};

template <int OT, int R>
__global__ __launch_bounds__(256) void dequant_sym_kernel(DequantSymArgs a) {
  const int c8 = (threadIdx.x & 15) * 8, rl = threadIdx.x >> 4;
  const uint32_t nblocks = (uint32_t)((a.n + 16 * R - 1) / (16 * R));
  for (uint32_t tile = blockIdx.x; tile < (uint32_t)a.items; tile += gridDim.x) {
    const uint32_t tb = tile % nblocks, r = tile / nblocks;
    const int64_t t0 = (int64_t)tb * (16 * R) + rl;
    uint2 cw[R];
    float sc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t t = min(t0 + 16 * i, a.n - 1);
      cw[i] = *reinterpret_cast<const uint2*>(a.codes + r * a.c_rs + t * 128 + c8);
      sc[i] = h2f(a.scales[r * a.s_rs + t]);
    }
#pragma unroll
    for (int i = 0; i < R; ++i) {
      const int64_t t = t0 + 16 * i;
      if (t >= a.n) break;
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const int code = (int)(int8_t)(((j < 4 ? cw[i].x : cw[i].y) >> (8 * (j & 3))) & 0xffu);
        v[j] = __fmul_rn((float)code, sc[i]);  // exact in fp32; rounded once by the store
      }
      store8<OT>(a.out, r * a.o_rs + t * 128 + c8, v);
    }
  }
}

// ---------------------------------------------------------------- copy (traffic calibration)

__global__ __launch_bounds__(256) void copy16_kernel(const uint4* __restrict__ src,
                                                     uint4* __restrict__ dst, int64_t n16) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  for (; i < n16; i += stride) dst[i] = src[i];
}

// Read-only streaming probe: every lane reads 16-byte words with a grid stride and folds
// them into one XOR checksum per workgroup (written so the loads cannot be elided).
__global__ __launch_bounds__(256) void read_bw_kernel(const uint4* __restrict__ src, int64_t n16,
                                                      uint32_t* __restrict__ sink) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t stride = (int64_t)gridDim.x * blockDim.x;
  uint32_t x = 0;
  for (; i + 3 * stride < n16; i += 4 * stride) {
    const uint4 a = src[i], b = src[i + stride], c = src[i + 2 * stride], d = src[i + 3 * stride];
    x ^= a.x ^ a.y ^ a.z ^ a.w ^ b.x ^ b.y ^ b.z ^ b.w ^ c.x ^ c.y ^ c.z ^ c.w ^ d.x ^ d.y ^ d.z ^ d.w;
  }
  for (; i < n16; i += stride) {
    const uint4 a = src[i];
    x ^= a.x ^ a.y ^ a.z ^ a.w;
  }
  for (int m = 32; m >= 1; m >>= 1) x ^= (uint32_t)__shfl_xor((int)x, m, 64);
  __shared__ uint32_t part[4];
  if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = x;
  __syncthreads();
  if (threadIdx.x == 0) sink[blockIdx.x] = part[0] ^ part[1] ^ part[2] ^ part[3];
}

// One row per thread or four (fp32 outputs always take one: few_rows).
template <int OT, bool NARROW>
static void launch_dequant_as(const DequantArgs& a, bool few, dim3 grid, hipStream_t s) {
  if constexpr (OT != NKV_F32)
    if (!few) {
      hipLaunchKernelGGL((dequant_kernel<OT, 4, NARROW>), grid, dim3(256), 0, s, a);
      return;
    }
  hipLaunchKernelGGL((dequant_kernel<OT, 1, NARROW>), grid, dim3(256), 0, s, a);
}
template <int OT>
static void launch_dequant(const DequantArgs& a, bool narrow, bool few, dim3 grid, hipStream_t s) {
  if (narrow) launch_dequant_as<OT, true>(a, few, grid, s);
  else launch_dequant_as<OT, false>(a, few, grid, s);
}
template <int OT>
static void launch_dequant_sym(const DequantSymArgs& a, bool few, dim3 grid, hipStream_t s) {
  if constexpr (OT != NKV_F32)
    if (!few) {
      hipLaunchKernelGGL((dequant_sym_kernel<OT, 4>), grid, dim3(256), 0, s, a);
      return;
    }
  hipLaunchKernelGGL((dequant_sym_kernel<OT, 1>), grid, dim3(256), 0, s, a);
}

// The kernels that take tiles in turns count them in 32 bits, one stride of the grid (at most 2^22 tiles)
// past the last: below 2^31 that sum does not wrap, and every workgroup leaves its loop.
static int check_items(const char* what, int64_t items) {
  if (items < (int64_t(1) << 31)) return NKV_OK;
  return fail(NKV_ERR_UNSUPPORTED, "%s: %lld tiles (fewer than 2^31)", what, (long long)items);
}

static bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace nkv

using namespace nkv;

extern "C" int nkv_abi_version(void) { return NKV_ABI_VERSION; }

extern "C" const char* nkv_last_error(void) { return g_err.c_str(); }

extern "C" int nkv_quantize_int8(const void* x, int x_dtype, int64_t x_row_stride, int64_t rows,
                                 int64_t n, int64_t dim, int64_t group, int axis, uint8_t* codes,
                                 int64_t codes_row_stride, uint16_t* mins, uint16_t* steps,
                                 int64_t scale_row_stride, void* stream) {
  g_err.clear();
  if (x_dtype != NKV_F16 && x_dtype != NKV_BF16 && x_dtype != NKV_F32)
    return fail(NKV_ERR_INVALID, "quantize: unknown dtype %d", x_dtype);
  if (rows < 0 || n < 0 || dim <= 0 || group < 0)
    return fail(NKV_ERR_INVALID, "quantize: bad sizes rows=%lld n=%lld dim=%lld group=%lld",
                (long long)rows, (long long)n, (long long)dim, (long long)group);
  if (rows == 0 || n == 0) return NKV_OK;
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (axis == NKV_AXIS_TOKEN) {
    const int64_t gs = group ? group : n;
    if (dim % 8) return fail(NKV_ERR_UNSUPPORTED, "quantize: head_dim %lld is not a multiple of 8", (long long)dim);
    const int esz = x_dtype == NKV_F32 ? 4 : 2;
    if (!aligned16(x) || !aligned16(mins) || !aligned16(steps) || (reinterpret_cast<uintptr_t>(codes) & 7u) ||
        (x_row_stride * esz) % 16 || codes_row_stride % 8 || (scale_row_stride * 2) % 16)
      return fail(NKV_ERR_UNSUPPORTED, "quantize: buffers or row strides are not 16-byte aligned");
    QuantTokArgs a{x, x_row_stride, rows, n, dim, gs, cdiv(n, gs), cdiv(dim, 128), codes,
                   codes_row_stride, mins, steps, scale_row_stride, 0};
    a.items = rows * a.ngroups * a.nchunks;
    if (int rc = check_items("quantize", a.items)) return rc;
    if (x_dtype == NKV_F16) launch_quant_token<NKV_F16>(a, s);
    else if (x_dtype == NKV_BF16) launch_quant_token<NKV_BF16>(a, s);
    else launch_quant_token<NKV_F32>(a, s);
    return check_launch("quantize_int8(token)");
  }
  if (axis == NKV_AXIS_CHANNEL) {
    const int64_t gc = group ? group : dim;
    if (dim % gc) return fail(NKV_ERR_INVALID, "head_dim %lld is not divisible by group_size %lld", (long long)dim, (long long)gc);
    // slabs that follow one another are one slab
    if (x_row_stride == n * dim && codes_row_stride == n * dim && scale_row_stride == n * (dim / gc)) {
      n *= rows;
      rows = 1;
    }
    QuantChanArgs a{x, x_row_stride, rows, n, dim, gc, dim / gc, codes, codes_row_stride,
                    mins, steps, scale_row_stride, 0};
    a.items = rows * n * a.ngc;
    const int esz = x_dtype == NKV_F32 ? 4 : 2;
    const bool wide = dim % 8 == 0 && aligned16(x) && (x_row_stride * esz) % 16 == 0 &&
                      (reinterpret_cast<uintptr_t>(codes) & 7u) == 0 && codes_row_stride % 8 == 0;
    if (x_dtype == NKV_F16) launch_quant_channel<NKV_F16>(a, wide, s);
    else if (x_dtype == NKV_BF16) launch_quant_channel<NKV_BF16>(a, wide, s);
    else launch_quant_channel<NKV_F32>(a, wide, s);
    return check_launch("quantize_int8(channel)");
  }
  return fail(NKV_ERR_INVALID, "axis must be channel (0) or token (1), got %d", axis);
}

extern "C" int nkv_paged_quantize_t64(const void* x, int x_dtype, int64_t x_head_stride, int64_t hkv, int64_t n,
                                      int which, uint8_t* pages, const int32_t* table_row, int64_t first_group,
                                      int64_t num_pages, void* stream) {
  g_err.clear();
  if (x_dtype != NKV_F16 && x_dtype != NKV_BF16 && x_dtype != NKV_F32)
    return fail(NKV_ERR_INVALID, "paged_quantize: unknown dtype %d", x_dtype);
  if (hkv <= 0 || n < 0 || n % 64 || first_group < 0 || (which != 0 && which != 1) || num_pages <= 0)
    return fail(NKV_ERR_INVALID, "paged_quantize: bad sizes hkv=%lld n=%lld (whole groups of 64) first_group=%lld "
                "which=%d num_pages=%lld", (long long)hkv, (long long)n, (long long)first_group, which,
                (long long)num_pages);
  if (n == 0) return NKV_OK;
  if (!x || !pages || !table_row) return fail(NKV_ERR_INVALID, "paged_quantize: null pointer argument");
  const int esz = x_dtype == NKV_F32 ? 4 : 2;
  if (!aligned16(x) || !aligned16(pages) || (x_head_stride * esz) % 16 || x_head_stride < n * 128)
    return fail(NKV_ERR_UNSUPPORTED, "paged_quantize: x must be 16-byte aligned with a head stride >= n * 128");
  QuantTokArgs a{x, x_head_stride, hkv, n, 128, 64, n / 64, 1, nullptr, 0, nullptr, nullptr, 0, 0,
                 pages, table_row, first_group, num_pages, which};
  a.items = hkv * a.ngroups;
  if (int rc = check_items("paged_quantize", a.items)) return rc;
  const dim3 grid((unsigned)std::min<int64_t>(a.items, 1 << 20)), block(256);
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (x_dtype == NKV_F16) hipLaunchKernelGGL((quant_token_kernel<NKV_F16, 4, 4, true>), grid, block, 0, s, a);
  else if (x_dtype == NKV_BF16) hipLaunchKernelGGL((quant_token_kernel<NKV_BF16, 4, 4, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((quant_token_kernel<NKV_F32, 4, 4, true>), grid, block, 0, s, a);
  return check_launch("paged_quantize_t64");
}

extern "C" int nkv_prefill_land_t64(const uint16_t* k, const uint16_t* v, int64_t k_token_stride, int64_t k_head_stride,
                                    int64_t v_token_stride, int64_t v_head_stride, int64_t n, int64_t start,
                                    int64_t hkv, int64_t head_dim, int64_t capacity, uint16_t* k16, uint16_t* v16,
                                    uint8_t* kq, uint16_t* kmn, uint16_t* kst, uint8_t* vq, uint16_t* vmn,
                                    uint16_t* vst, uint16_t* tail_k, uint16_t* tail_v, void* stream) {
  g_err.clear();
  if (head_dim != 128) return fail(NKV_ERR_UNSUPPORTED, "prefill_land: head_dim %lld (only 128 is built)", (long long)head_dim);
  if (hkv <= 0 || hkv > (1 << 16) || n <= 0 || n > (1 << 24) || start < 0 || start % 64 || start + n > capacity)
    return fail(NKV_ERR_INVALID, "prefill_land: %lld tokens from %lld (a multiple of 64), hkv=%lld, capacity %lld",
                (long long)n, (long long)start, (long long)hkv, (long long)capacity);
  if (!k || !v || !k16 || !v16 || !kq || !kmn || !kst || !vq || !vmn || !vst || !tail_k || !tail_v)
    return fail(NKV_ERR_INVALID, "prefill_land: null pointer argument");
  const void* al[] = {k, v, k16, v16, kq, kmn, kst, vq, vmn, vst, tail_k, tail_v};
  for (const void* p : al)
    if (!aligned16(p)) return fail(NKV_ERR_UNSUPPORTED, "prefill_land: buffers must be 16-byte aligned");
  if (k_token_stride % 8 || k_head_stride % 8 || v_token_stride % 8 || v_head_stride % 8)
    return fail(NKV_ERR_UNSUPPORTED, "prefill_land: strides must be multiples of 8");
  const int64_t blocks = cdiv(n, 64) * hkv * 2;
  if (blocks >= (1 << 24)) return fail(NKV_ERR_UNSUPPORTED, "prefill_land: %lld tokens of %lld heads", (long long)n, (long long)hkv);
  LandArgs a{{k, v}, {k_token_stride, v_token_stride}, {k_head_stride, v_head_stride}, n, start, capacity,
             cdiv(capacity, 64), (int)hkv, {k16, v16}, {kq, vq}, {kmn, vmn}, {kst, vst}, {tail_k, tail_v}};
  hipLaunchKernelGGL(land_chunk_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), a);
  return check_launch("prefill_land_t64");
}

extern "C" int nkv_dequantize_int8(const uint8_t* codes, int64_t codes_row_stride,
                                   const uint16_t* mins, const uint16_t* steps,
                                   int64_t scale_row_stride, int64_t rows, int64_t n, int64_t dim,
                                   int64_t group, int axis, void* out, int out_dtype,
                                   int64_t out_row_stride, void* stream) {
  g_err.clear();
  if (out_dtype != NKV_F16 && out_dtype != NKV_BF16 && out_dtype != NKV_F32)
    return fail(NKV_ERR_INVALID, "dequantize: unknown dtype %d", out_dtype);
  if (axis != NKV_AXIS_TOKEN && axis != NKV_AXIS_CHANNEL)
    return fail(NKV_ERR_INVALID, "axis must be channel (0) or token (1), got %d", axis);
  if (rows < 0 || n < 0 || dim <= 0 || group < 0) return fail(NKV_ERR_INVALID, "dequantize: bad sizes");
  if (rows == 0 || n == 0) return NKV_OK;
  if (dim % 8) return fail(NKV_ERR_UNSUPPORTED, "dequantize: head_dim %lld is not a multiple of 8", (long long)dim);
  int64_t g = group ? group : (axis == NKV_AXIS_TOKEN ? n : dim);
  if (axis == NKV_AXIS_CHANNEL && dim % g) return fail(NKV_ERR_INVALID, "head_dim is not divisible by group_size");
  const int esz = out_dtype == NKV_F32 ? 4 : 2;
  if ((reinterpret_cast<uintptr_t>(codes) & 7u) || codes_row_stride % 8 || !aligned16(out) ||
      (out_row_stride * esz) % 16)
    return fail(NKV_ERR_UNSUPPORTED, "dequantize: buffers or row strides are not aligned");
  if (axis == NKV_AXIS_TOKEN) g = std::min(g, n);  // (a longer group is the whole slab)
  // slabs that follow one another, each of whole groups, are one slab
  const int64_t rulers = axis == NKV_AXIS_CHANNEL ? n * (dim / g) : n % g ? -1 : n / g * dim;
  if (codes_row_stride == n * dim && out_row_stride == n * dim && scale_row_stride == rulers) {
    n *= rows;
    rows = 1;
  }
  const TileLanes tl(dim);
  const bool narrow = dim <= 64, few = few_rows(rows * n * tl.lanes / 16, out_dtype);
  const int64_t pass = (narrow ? tl.rows : 16) * (few ? 1 : 4);
  DequantArgs a{codes, codes_row_stride, mins, steps, scale_row_stride, rows, n, dim, g, axis,
                out, out_row_stride, narrow ? cdiv(rows * n, pass) : rows * cdiv(n, pass) * cdiv(dim, 128),
                aligned16(mins) && aligned16(steps) && scale_row_stride % 8 == 0, tl};
  if (int rc = check_items("dequantize", a.items)) return rc;
  if (n >= (int64_t(1) << 32) || dim >= (int64_t(1) << 32) || (narrow && rows * n >= (int64_t(1) << 32)))
    return fail(NKV_ERR_UNSUPPORTED, "dequantize: rows=%lld n=%lld dim=%lld", (long long)rows, (long long)n, (long long)dim);
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)std::min<int64_t>(a.items, 1 << 20));
  if (out_dtype == NKV_F16) launch_dequant<NKV_F16>(a, narrow, few, grid, s);
  else if (out_dtype == NKV_BF16) launch_dequant<NKV_BF16>(a, narrow, few, grid, s);
  else launch_dequant<NKV_F32>(a, narrow, few, grid, s);
  return check_launch("dequantize_int8");
}

extern "C" int nkv_quantize_tok(const void* x, int x_dtype, int64_t x_row_stride, int64_t rows, int64_t n,
                                int64_t dim, int8_t* codes, int64_t codes_row_stride, uint16_t* scales,
                                int64_t scale_row_stride, void* stream) {
  g_err.clear();
  if (x_dtype != NKV_F16 && x_dtype != NKV_BF16 && x_dtype != NKV_F32)
    return fail(NKV_ERR_INVALID, "quantize_tok: unknown dtype %d", x_dtype);
  if (rows < 0 || n < 0 || dim <= 0)
    return fail(NKV_ERR_INVALID, "quantize_tok: bad sizes rows=%lld n=%lld dim=%lld", (long long)rows,
                (long long)n, (long long)dim);
  if (dim != 128) return fail(NKV_ERR_UNSUPPORTED, "quantize_tok: head_dim %lld (only 128 is built)", (long long)dim);
  if (rows == 0 || n == 0) return NKV_OK;
  const int esz = x_dtype == NKV_F32 ? 4 : 2;
  if (!x || !codes || !scales || !aligned16(x) || (reinterpret_cast<uintptr_t>(codes) & 7u) ||
      (reinterpret_cast<uintptr_t>(scales) & 1u) || (x_row_stride * esz) % 16 || codes_row_stride % 8)
    return fail(NKV_ERR_UNSUPPORTED, "quantize_tok: buffers or row strides are not aligned");
  if (x_row_stride == n * dim && codes_row_stride == n * dim && scale_row_stride == n) {  // one slab
    n *= rows;
    rows = 1;
  }
  QuantSymArgs a{x, x_row_stride, rows, n, reinterpret_cast<uint8_t*>(codes), codes_row_stride, scales,
                 scale_row_stride, rows * cdiv(n, 16)};
  if (int rc = check_items("quantize_tok", a.items)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)std::min<int64_t>(a.items, 1 << 22)), block(256);
  if (x_dtype == NKV_F16) hipLaunchKernelGGL((quant_sym_kernel<NKV_F16>), grid, block, 0, s, a);
  else if (x_dtype == NKV_BF16) hipLaunchKernelGGL((quant_sym_kernel<NKV_BF16>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((quant_sym_kernel<NKV_F32>), grid, block, 0, s, a);
  return check_launch("quantize_tok");
}

extern "C" int nkv_paged_quantize_tok(const void* x, int x_dtype, int64_t x_head_stride, int64_t hkv, int64_t n,
                                      int which, uint8_t* pages, const int32_t* table_row, int64_t first_token,
                                      int64_t num_pages, void* stream) {
  g_err.clear();
  if (x_dtype != NKV_F16 && x_dtype != NKV_BF16 && x_dtype != NKV_F32)
    return fail(NKV_ERR_INVALID, "paged_quantize_tok: unknown dtype %d", x_dtype);
  if (hkv <= 0 || n < 0 || first_token < 0 || (which != 0 && which != 1) || num_pages <= 0)
    return fail(NKV_ERR_INVALID, "paged_quantize_tok: bad sizes hkv=%lld n=%lld first_token=%lld which=%d "
                "num_pages=%lld", (long long)hkv, (long long)n, (long long)first_token, which, (long long)num_pages);
  if (n == 0) return NKV_OK;
  if (!x || !pages || !table_row) return fail(NKV_ERR_INVALID, "paged_quantize_tok: null pointer argument");
  const int esz = x_dtype == NKV_F32 ? 4 : 2;
  if (!aligned16(x) || !aligned16(pages) || (x_head_stride * esz) % 16 || x_head_stride < n * 128)
    return fail(NKV_ERR_UNSUPPORTED, "paged_quantize_tok: x must be 16-byte aligned with a head stride >= n * 128");
  QuantSymArgs a{x, x_head_stride, hkv, n, nullptr, 0, nullptr, 0, hkv * cdiv(n, 16), pages, table_row, first_token,
                 num_pages, which};
  if (int rc = check_items("paged_quantize_tok", a.items)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)std::min<int64_t>(a.items, 1 << 22)), block(256);
  if (x_dtype == NKV_F16) hipLaunchKernelGGL((quant_sym_kernel<NKV_F16, true>), grid, block, 0, s, a);
  else if (x_dtype == NKV_BF16) hipLaunchKernelGGL((quant_sym_kernel<NKV_BF16, true>), grid, block, 0, s, a);
  else hipLaunchKernelGGL((quant_sym_kernel<NKV_F32, true>), grid, block, 0, s, a);
  return check_launch("paged_quantize_tok");
}

extern "C" int nkv_dequantize_tok(const int8_t* codes, int64_t codes_row_stride, const uint16_t* scales,
                                  int64_t scale_row_stride, int64_t rows, int64_t n, int64_t dim, void* out,
                                  int out_dtype, int64_t out_row_stride, void* stream) {
  g_err.clear();
  if (out_dtype != NKV_F16 && out_dtype != NKV_BF16 && out_dtype != NKV_F32)
    return fail(NKV_ERR_INVALID, "dequantize_tok: unknown dtype %d", out_dtype);
  if (rows < 0 || n < 0 || dim <= 0) return fail(NKV_ERR_INVALID, "dequantize_tok: bad sizes");
  if (dim != 128) return fail(NKV_ERR_UNSUPPORTED, "dequantize_tok: head_dim %lld (only 128 is built)", (long long)dim);
  if (rows == 0 || n == 0) return NKV_OK;
  const int esz = out_dtype == NKV_F32 ? 4 : 2;
  if (!codes || !scales || !out || (reinterpret_cast<uintptr_t>(codes) & 7u) || codes_row_stride % 8 ||
      !aligned16(out) || (out_row_stride * esz) % 16)
    return fail(NKV_ERR_UNSUPPORTED, "dequantize_tok: buffers or row strides are not aligned");
  if (codes_row_stride == n * dim && out_row_stride == n * dim && scale_row_stride == n) {  // one slab
    n *= rows;
    rows = 1;
  }
  const bool few = few_rows(rows * n, out_dtype);
  DequantSymArgs a{reinterpret_cast<const uint8_t*>(codes), codes_row_stride, scales, scale_row_stride, rows, n,
                   out, out_row_stride, rows * cdiv(n, few ? 16 : 64)};
  if (int rc = check_items("dequantize_tok", a.items)) return rc;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)std::min<int64_t>(a.items, 1 << 20));
  if (out_dtype == NKV_F16) launch_dequant_sym<NKV_F16>(a, few, grid, s);
  else if (out_dtype == NKV_BF16) launch_dequant_sym<NKV_BF16>(a, few, grid, s);
  else launch_dequant_sym<NKV_F32>(a, few, grid, s);
  return check_launch("dequantize_tok");
}

extern "C" int nkv_copy_bytes(const void* src, void* dst, int64_t nbytes, void* stream) {
  g_err.clear();
  if (nbytes < 0 || nbytes % 16 || !aligned16(src) || !aligned16(dst))
    return fail(NKV_ERR_INVALID, "copy: nbytes must be a multiple of 16 and buffers 16-byte aligned");
  if (nbytes == 0) return NKV_OK;
  const int64_t n16 = nbytes / 16;
  const unsigned blocks = (unsigned)std::min<int64_t>(cdiv(n16, 256), 2048);
  hipLaunchKernelGGL(copy16_kernel, dim3(blocks), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint4*>(src), static_cast<uint4*>(dst), n16);
  return check_launch("copy_bytes");
}

extern "C" int nkv_read_bw(const void* src, int64_t nbytes, uint32_t* sink, int64_t blocks, void* stream) {
  g_err.clear();
  if (!src || !sink || nbytes <= 0 || nbytes % 16 || !aligned16(src))
    return fail(NKV_ERR_INVALID, "read_bw: nbytes must be a positive multiple of 16 and src 16-byte aligned");
  if (blocks <= 0 || blocks > (1 << 20)) return fail(NKV_ERR_INVALID, "read_bw: blocks must be in [1, 2^20]");
  hipLaunchKernelGGL(read_bw_kernel, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream),
                     static_cast<const uint4*>(src), nbytes / 16, sink);
  return check_launch("read_bw");
}
