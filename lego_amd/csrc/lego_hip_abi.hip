// C-ABI entry points of liblego_hip.so (declared in include/lego_hip.h).
//
// This file is written by hand; the kernels and their launchers are generated from LEGO
// layouts (python -m lego_amd.build) into csrc/generated/ and declared in
// generated/launchers.h.  An entry point validates what the generated code assumes --
// non-null, 16-byte aligned pointers and shapes that divide the tiles -- and enqueues one
// kernel on the caller's stream.  It allocates nothing and never synchronises.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <string.h>

#include <algorithm>
#include <mutex>
#include <new>
#include <vector>

#include "lego_hip.h"
#include "generated/launchers.h"

namespace {

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }
inline bool usable(const void* p) { return p != nullptr && aligned16(p); }
// a tensor base that only has its elements' alignment (a sliced view): the kernels for rows and shapes of any
// length take those, with 16-byte accesses wherever their result has its 16-byte boundaries
inline bool element_aligned(const void* p, unsigned bytes) { return p != nullptr && (reinterpret_cast<uintptr_t>(p) & (bytes - 1u)) == 0; }
inline hipStream_t as_stream(void* s) { return static_cast<hipStream_t>(s); }
inline int ok_or(hipError_t e) { return static_cast<int>(e); }
constexpr int kInvalid = static_cast<int>(hipErrorInvalidValue);

// plain grid-stride copy, one 16-byte vector per lane per step
__global__ void __launch_bounds__(256) lego_copy16_kernel(const uint4* __restrict__ in, uint4* __restrict__ out, size_t n)
{
  const size_t stride = static_cast<size_t>(gridDim.x) * blockDim.x;
  for (size_t i = static_cast<size_t>(blockIdx.x) * blockDim.x + threadIdx.x; i < n; i += stride) out[i] = in[i];
}

// streaming copy: a workgroup owns one contiguous 16 KiB chunk, four non-temporal 16-byte loads
// per lane in flight, then four non-temporal stores
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
__global__ void __launch_bounds__(256) lego_copy16_stream_kernel(const u32x4* __restrict__ in, u32x4* __restrict__ out)
{
  const size_t base = static_cast<size_t>(blockIdx.x) * 1024 + threadIdx.x;
  u32x4 v[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) v[u] = __builtin_nontemporal_load(in + base + u * 256);
#pragma unroll
  for (int u = 0; u < 4; ++u) __builtin_nontemporal_store(v[u], out + base + u * 256);
}

// What the memory delivers to one-directional streams, in the access shape of lego_copy16_stream_kernel (V
// non-temporal 16-byte vectors per lane, a contiguous V*4 KiB chunk per workgroup): a read-only stream whose
// values are folded into one word and compared with a constant (the loads must depend on the data, or the
// compiler drops them; a lane whose words happen to fold to the constant stores one vector into the first 4 KiB
// of `sink`), and a write-only stream of a lane-dependent pattern.
template <int V>
__global__ void __launch_bounds__(256) lego_probe_read_kernel(const u32x4* __restrict__ in, u32x4* __restrict__ sink)
{
  const size_t base = static_cast<size_t>(blockIdx.x) * (256 * V) + threadIdx.x;
  u32x4 v[V];
#pragma unroll
  for (int u = 0; u < V; ++u) v[u] = __builtin_nontemporal_load(in + base + u * 256);
  unsigned acc = 0;
#pragma unroll
  for (int u = 0; u < V; ++u) acc ^= v[u][0] ^ v[u][1] ^ v[u][2] ^ v[u][3];
  if (acc == 0x9e3779b9u) sink[threadIdx.x] = v[0];
}
template <int V>
__global__ void __launch_bounds__(256) lego_probe_write_kernel(u32x4* __restrict__ out)
{
  const size_t base = static_cast<size_t>(blockIdx.x) * (256 * V) + threadIdx.x;
  const u32x4 v = {threadIdx.x, blockIdx.x, 3u, 4u};
#pragma unroll
  for (int u = 0; u < V; ++u) __builtin_nontemporal_store(v, out + base + u * 256);
}
template <int V>
__global__ void __launch_bounds__(256) lego_probe_copy_kernel(const u32x4* __restrict__ in, u32x4* __restrict__ out)
{
  const size_t base = static_cast<size_t>(blockIdx.x) * (256 * V) + threadIdx.x;
  u32x4 v[V];
#pragma unroll
  for (int u = 0; u < V; ++u) v[u] = __builtin_nontemporal_load(in + base + u * 256);
#pragma unroll
  for (int u = 0; u < V; ++u) __builtin_nontemporal_store(v[u], out + base + u * 256);
}

// What the matrix cores sustain when nothing else happens: every wave of a workgroup of four (one per SIMD, 256
// accumulator registers, as in the GEMM kernels) loads sixteen operand fragments once and then issues nothing but
// MFMAs on them, a 128 x 128 block of accumulators per wave.  With random operands this is the rate the socket's
// power limit leaves to a GEMM whose loads, LDS traffic and address arithmetic cost nothing.
typedef _Float16 probe_half8 __attribute__((ext_vector_type(8)));
typedef __bf16 probe_bhalf8 __attribute__((ext_vector_type(8)));
typedef float probe_float16 __attribute__((ext_vector_type(16)));
typedef float probe_float4 __attribute__((ext_vector_type(4)));
// The same with two waves per SIMD (workgroups of eight waves, 128 accumulator registers each, a 128 x 64 block):
// whether a second wave to issue from changes what the pipe sustains.
template <int SHAPE>      // 3: v_mfma_f32_16x16x32_f16 (8 x 4 blocks)  4: v_mfma_f32_32x32x16_f16 (4 x 2 blocks)
__global__ void __launch_bounds__(512) lego_mfma_probe2_kernel(const probe_half8* __restrict__ operands, float* __restrict__ sink, unsigned iters)
{
  const probe_half8* mine = operands + (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x % 256) * 16;
  probe_half8 fa[8], fb[4];
#pragma unroll
  for (int f = 0; f < 8; ++f) fa[f] = mine[f];
#pragma unroll
  for (int f = 0; f < 4; ++f) fb[f] = mine[8 + f];
  float total = 0.0f;
  if (SHAPE == 3) {
    probe_float4 acc[8][4];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) acc[i][j] = probe_float4{0.0f, 0.0f, 0.0f, 0.0f};
    for (unsigned it = 0; it < iters; ++it) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) total += acc[i][j][0] + acc[i][j][1] + acc[i][j][2] + acc[i][j][3];
  } else {
    probe_float16 acc[4][2];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    for (unsigned it = 0; it < iters; ++it) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) total += acc[i][j][r];
  }
  sink[static_cast<size_t>(blockIdx.x) * 512 + threadIdx.x] = total;
}

template <int SHAPE>      // 0: v_mfma_f32_32x32x16_f16 (4 x 4 blocks)  1: v_mfma_f32_16x16x32_f16 (8 x 8 blocks)  2: v_mfma_f32_32x32x16_bf16
__global__ void __launch_bounds__(256) lego_mfma_probe_kernel(const probe_half8* __restrict__ operands, float* __restrict__ sink, unsigned iters)
{
  constexpr int T = SHAPE == 1 ? 8 : 4;
  const probe_half8* mine = operands + (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 16;
  probe_half8 fa[8], fb[8];
#pragma unroll
  for (int f = 0; f < 8; ++f) { fa[f] = mine[f]; fb[f] = mine[8 + f]; }
  float total = 0.0f;
  if (SHAPE == 1) {
    probe_float4 acc[8][8];
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) acc[i][j] = probe_float4{0.0f, 0.0f, 0.0f, 0.0f};
    for (unsigned it = 0; it < iters; ++it) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
#pragma unroll
        for (int j = 0; j < 8; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j) total += acc[i][j][0] + acc[i][j][1] + acc[i][j][2] + acc[i][j][3];
  } else {
    probe_float16 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    for (unsigned it = 0; it < iters; ++it) {
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) {
          if (SHAPE == 0) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fb[j], fa[i], acc[i][j], 0, 0, 0);
          else acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(probe_bhalf8, fb[j]), __builtin_bit_cast(probe_bhalf8, fa[i]), acc[i][j], 0, 0, 0);
        }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) total += acc[i][j][r];
  }
  sink[static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x] = total;
}

// 8-bit operands: v_mfma_f32_32x32x64_f8f6f4 on 4 x 4 blocks, the operands' bits read as OCP e5m2 (shape 5) or e4m3 (6)
typedef int probe_int8 __attribute__((ext_vector_type(8)));
template <int FORMAT>     // 0: e4m3  1: e5m2 (the instruction's format codes)
__global__ void __launch_bounds__(256) lego_mfma_probe_8bit_kernel(const probe_int8* __restrict__ operands, float* __restrict__ sink, unsigned iters)
{
  const probe_int8* mine = operands + (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  probe_int8 fa[4], fb[4];
#pragma unroll
  for (int f = 0; f < 4; ++f) { fa[f] = mine[f]; fb[f] = mine[4 + f]; }
  probe_float16 acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  for (unsigned it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fb[j], fa[i], acc[i][j], FORMAT, FORMAT, 0, 0, 0, 0);
  }
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) total += acc[i][j][r];
  sink[static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x] = total;
}

// The same operands through v_mfma_f32_16x16x128_f8f6f4 on 8 x 8 blocks (shape 7): the fragments of the second four
// block rows and columns are those of the first four with their halves swapped, in registers of their own
__global__ void __launch_bounds__(256) lego_mfma_probe_8bit_16x16_kernel(const probe_int8* __restrict__ operands, float* __restrict__ sink, unsigned iters)
{
  const probe_int8* mine = operands + (static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x) * 8;
  probe_int8 fa[8], fb[8];
#pragma unroll
  for (int f = 0; f < 4; ++f) {
    fa[f] = mine[f];
    fb[f] = mine[4 + f];
    fa[4 + f] = __builtin_shufflevector(fa[f], fa[f], 4, 5, 6, 7, 0, 1, 2, 3);
    fb[4 + f] = __builtin_shufflevector(fb[f], fb[f], 4, 5, 6, 7, 0, 1, 2, 3);
  }
  probe_float4 acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) acc[i][j] = probe_float4{0.0f, 0.0f, 0.0f, 0.0f};
  for (unsigned it = 0; it < iters; ++it) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int j = 0; j < 8; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(fb[j], fa[i], acc[i][j], 1, 1, 0, 0, 0, 0);
  }
  float total = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) total += acc[i][j][r];
  sink[static_cast<size_t>(blockIdx.x) * 256 + threadIdx.x] = total;
}

typedef unsigned u32x4w __attribute__((ext_vector_type(4)));
typedef unsigned u32x4w_any __attribute__((ext_vector_type(4), aligned(1)));     // the same 16 bytes at any byte

// Matrices on their way into, or out of, copies whose rows are whole 16-byte chunks on a 16-byte aligned base: up to kCopies of them
// in one launch, told apart by the running total of workgroups (a launch of its own for each took 2-3 us, more than most of the
// copies themselves).  One lane per 16-byte chunk; a chunk that lies inside the matrix as a whole is one access on either side.
// The list is kernel arguments, and the largest is 3 KB of them, a microsecond of each launch: a single product's copies, and those of a few,
// have lists of their own.  Where a workgroup belongs takes one round of scalar loads of the list's totals, and none of a list of two (640 x
// 1439 x 64, B and the result copied, with one list of 64 searched entry by entry 13.9 us, 13.4).
constexpr int kCopies = 64, kSomeCopies = 12, kFewCopies = 2;
struct Copy {
  const void* from;
  void* to;
  unsigned rows, row_bytes;        // of the matrix as it is
  unsigned rows_to, pitch;         // of the copy: rows beyond `rows` and bytes beyond `row_bytes` are zeros
  unsigned first;                  // workgroup of the launch
};
template <int MAX>
struct Copies {
  unsigned end[MAX];               // workgroups up to and including each one; ~0 past the last
  Copy of[MAX];
};
static_assert(sizeof(Copies<kFewCopies>) <= 128, "what a single product's copies add to a launch");

template <bool PAD, int MAX>
__global__ void __launch_bounds__(256) lego_copies_kernel(const Copies<MAX> copies)
{
  Copy c;      // the same for the whole workgroup
  if constexpr (MAX == 2) {
    c = copies.of[0];
    const Copy& d = copies.of[1];
    if (blockIdx.x >= copies.end[0]) c = d;
  } else {
    int i = 0;
#pragma unroll
    for (int j = 0; j + 1 < MAX; ++j) i += blockIdx.x >= copies.end[j] ? 1 : 0;
    c = copies.of[i];
  }
  const unsigned chunk = (blockIdx.x - c.first) * 256 + threadIdx.x;      // of less than 2^32, as a launch has lanes
  const unsigned per_row = c.pitch / 16, at = chunk % per_row * 16;
  const size_t r = chunk / per_row;
  if (PAD) {
    if (r >= c.rows_to) return;
    u32x4w v = {0u, 0u, 0u, 0u};
    if (r < c.rows && at < c.row_bytes) {
      const size_t offset = r * c.row_bytes + at;
      const uint8_t* p = static_cast<const uint8_t*>(c.from) + offset;
      const unsigned valid = c.row_bytes - at;
      if (offset + 16 <= static_cast<size_t>(c.rows) * c.row_bytes) {      // the matrix has sixteen bytes from here on, this row's or the next one's
        v = *reinterpret_cast<const u32x4w_any*>(p);
#pragma unroll
        for (unsigned e = 0; e < 4; ++e)
          v[e] = valid >= 4 * e + 4 ? v[e] : valid > 4 * e ? v[e] & ((1u << (8 * (valid - 4 * e))) - 1u) : 0u;
      } else {
#pragma unroll
        for (unsigned e = 0; e < 16; ++e)
          if (e < valid) v[e / 4] |= static_cast<uint32_t>(p[e]) << (8 * (e % 4));
      }
    }
    *reinterpret_cast<u32x4w*>(static_cast<uint8_t*>(c.to) + r * c.pitch + at) = v;
  } else {
    if (r >= c.rows || at >= c.row_bytes) return;
    const u32x4w v = *reinterpret_cast<const u32x4w*>(static_cast<const uint8_t*>(c.from) + r * c.pitch + at);
    uint8_t* q = static_cast<uint8_t*>(c.to) + r * c.row_bytes + at;
    if (at + 16 <= c.row_bytes) {
      *reinterpret_cast<u32x4w_any*>(q) = v;
    } else {
#pragma unroll
      for (unsigned e = 0; e < 16; e += 2)       // two-byte elements
        if (at + e < c.row_bytes) *reinterpret_cast<uint16_t*>(q + e) = static_cast<uint16_t>(v[e / 4] >> (8 * (e % 4)));
    }
  }
}

// Collects copies of matrices that lie one after the other in a workspace and enqueues them, kCopies at a time.
class Copier {
 public:
  Copier(bool pad, hipStream_t stream) : pad_(pad), stream_(stream) {}
  // rows x cols elements of `bytes` bytes each, copied to (pad) or from (otherwise) rows of cols_to elements
  void add(const void* from, void* to, long rows, long cols, long rows_to, long cols_to, int bytes)
  {
    if (count_ == kCopies) (void)flush();      // its error is kept
    const unsigned long long chunks = static_cast<unsigned long long>(pad_ ? rows_to : rows) * (cols_to * bytes / 16);
    copies_[count_++] = {from, to, static_cast<unsigned>(rows), static_cast<unsigned>(cols * bytes), static_cast<unsigned>(rows_to),
                            static_cast<unsigned>(cols_to * bytes), workgroups_};
    workgroups_ += static_cast<unsigned>((chunks + 255) / 256);
  }
  hipError_t flush()
  {
    if (count_ == 0) return err_;
    if (count_ <= kFewCopies) launch<kFewCopies>();
    else if (count_ <= kSomeCopies) launch<kSomeCopies>();
    else launch<kCopies>();
    count_ = 0;
    workgroups_ = 0;
    const hipError_t e = hipGetLastError();
    if (err_ == hipSuccess) err_ = e;
    return err_;
  }

 private:
  template <int MAX>
  void launch()
  {
    Copies<MAX> list;
    for (int i = 0; i < MAX; ++i) {
      list.of[i] = copies_[i < count_ ? i : 0];
      list.end[i] = i + 1 < count_ ? copies_[i + 1].first : ~0u;
    }
    if (pad_) hipLaunchKernelGGL((lego_copies_kernel<true, MAX>), dim3(workgroups_), dim3(256), 0, stream_, list);
    else hipLaunchKernelGGL((lego_copies_kernel<false, MAX>), dim3(workgroups_), dim3(256), 0, stream_, list);
  }

  bool pad_;
  hipStream_t stream_;
  Copy copies_[kCopies];
  int count_ = 0;
  unsigned workgroups_ = 0;
  hipError_t err_ = hipSuccess;
};

// Scratch of lego_hip_layernorm_bwd_f16_noalloc: the fp32 dw/db partial rows that the other
// LayerNorm backward entry points take from the caller.  One copy per device, held until the process
// ends.  In host code the array's name is only a handle for hipGetSymbolAddress; kernels and launchers
// receive the device address kept in scratch_ptr[device].
constexpr unsigned long long kScratchBytes = 32ull << 20;
static __device__ __align__(256) float scratch[kScratchBytes / sizeof(float)];
constexpr int kMaxDevices = 64;
float* scratch_ptr[kMaxDevices];
std::mutex scratch_mutex;

// Device address of the current device's scratch array (looked up on the first call per device).
hipError_t scratch_address(float** out)
{
  int dev = -1;
  hipError_t err = hipGetDevice(&dev);
  if (err != hipSuccess) return err;
  if (dev < 0 || dev >= kMaxDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> hold(scratch_mutex);
  if (scratch_ptr[dev] == nullptr) {
    void* p = nullptr;
    err = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return err;
    if (p == nullptr) return hipErrorInvalidSymbol;
    scratch_ptr[dev] = static_cast<float*>(p);
  }
  *out = scratch_ptr[dev];
  return hipSuccess;
}

}  // namespace

extern "C" {

int lego_hip_abi_version(void) { return 1; }

int lego_hip_transpose_f32(const void* in, void* out, int rows, int cols, void* stream)
{
  if (!element_aligned(in, 4) || !element_aligned(out, 4) || in == out) return kInvalid;
  if (rows <= 0 || cols <= 0) return kInvalid;
  if (!aligned16(in) || !aligned16(out))      // a base at any element: the kernels whose vectors sit at any element
    return ok_or(lego_transpose_f32_dispatch_any_base(in, out, rows, cols, as_stream(stream)));
  return ok_or(lego_transpose_f32_dispatch(in, out, rows, cols, as_stream(stream)));
}

int lego_hip_transpose_f16(const void* in, void* out, int rows, int cols, void* stream)
{
  if (!element_aligned(in, 2) || !element_aligned(out, 2) || in == out) return kInvalid;
  if (rows <= 0 || cols <= 0) return kInvalid;
  if (!aligned16(in) || !aligned16(out))
    return ok_or(lego_transpose_f16_dispatch_any_base(in, out, rows, cols, as_stream(stream)));
  return ok_or(lego_transpose_f16_dispatch(in, out, rows, cols, as_stream(stream)));
}

int lego_hip_transpose_f32_tiling(const void* in, void* out, int rows, int cols, int tiling, void* stream)
{
  if (!aligned16(in) || !aligned16(out) || in == out || rows <= 0 || cols <= 0) return kInvalid;
  return ok_or(lego_transpose_f32_tiling(tiling, in, out, rows, cols, as_stream(stream)));
}

int lego_hip_transpose_f16_tiling(const void* in, void* out, int rows, int cols, int tiling, void* stream)
{
  if (!aligned16(in) || !aligned16(out) || in == out || rows <= 0 || cols <= 0) return kInvalid;
  return ok_or(lego_transpose_f16_tiling(tiling, in, out, rows, cols, as_stream(stream)));
}

int lego_hip_softmax_f16_wpr(const void* x, void* y, int M, int N, int waves_per_row, void* stream)
{
  if (!usable(x) || !usable(y)) return kInvalid;
  if (M <= 0 || N <= 0 || N % 8 || N > LEGO_ROWWISE_MAX_N) return kInvalid;
  switch (waves_per_row) {
    case 1:   // rows of at most 16 or 32 vectors: several rows per wave
      return ok_or((N <= 128 ? lego_softmax_f16_l16_launch : N <= 256 ? lego_softmax_f16_l32_launch : lego_softmax_f16_w1_launch)(
          x, y, M, N, as_stream(stream)));
    case 2: return ok_or(lego_softmax_f16_w2_launch(x, y, M, N, as_stream(stream)));
    case 4: return ok_or(lego_softmax_f16_w4_launch(x, y, M, N, as_stream(stream)));
    case 8: return ok_or(lego_softmax_f16_w8_launch(x, y, M, N, as_stream(stream)));
    case 16: return ok_or(lego_softmax_f16_w16_launch(x, y, M, N, as_stream(stream)));
    default: return kInvalid;
  }
}

int lego_hip_softmax_f16(const void* x, void* y, int M, int N, void* stream)
{
  if (!element_aligned(x, 2) || !element_aligned(y, 2) || M <= 0 || N <= 0) return kInvalid;
  if (N > LEGO_ROWWISE_MAX_N) return ok_or(lego_softmax_long_f16_launch(x, y, M, N, as_stream(stream)));   // two passes
  const bool long_row = N > LEGO_ROWWISE_MAX_N_SMALL_TEAMS;
  if (N % 8 || !aligned16(x) || !aligned16(y))   // rows of any length, or at any element
    return ok_or((N <= 128 ? lego_softmax_f16s_l16_launch : N <= 256 ? lego_softmax_f16s_l32_launch
                  : lego_rowwise_f16_wpr(M, N) == 8 ? lego_softmax_f16s_w8_launch
                  : long_row ? lego_softmax_f16s_w16_launch : lego_rowwise_default_wpr(N) == 1 ? lego_softmax_f16s_w1_launch
                                                                                           : lego_softmax_f16s_w4_launch)(
        x, y, M, N, as_stream(stream)));
  return lego_hip_softmax_f16_wpr(x, y, M, N, lego_rowwise_f16_wpr(M, N), stream);
}

int lego_hip_softmax_f32(const void* x, void* y, int M, int N, void* stream)
{
  if (!element_aligned(x, 4) || !element_aligned(y, 4) || M <= 0 || N <= 0) return kInvalid;
  if (N > LEGO_ROWWISE_MAX_N) return ok_or(lego_softmax_long_f32_launch(x, y, M, N, as_stream(stream)));   // two passes
  const bool long_row = N > LEGO_ROWWISE_MAX_N_SMALL_TEAMS;
  if (N % 4 || !aligned16(x) || !aligned16(y))   // rows of any length, or at any element
    return ok_or((N <= 64 ? lego_softmax_f32s_l16_launch : N <= 128 ? lego_softmax_f32s_l32_launch
                  : lego_rowwise_f16_wpr(M, 2 * N) == 8 ? lego_softmax_f32s_w8_launch
                  : long_row ? lego_softmax_f32s_w16_launch : N <= 1024 ? lego_softmax_f32s_w1_launch
                                                                      : lego_softmax_f32s_w4_launch)(x, y, M, N, as_stream(stream)));
  if (N <= 1024)   // rows of at most 16 or 32 vectors: several rows per wave
    return ok_or((N <= 64 ? lego_softmax_f32_l16_launch : N <= 128 ? lego_softmax_f32_l32_launch : lego_softmax_f32_w1_launch)(
        x, y, M, N, as_stream(stream)));
  // eight waves for the rows that take them in the 16-bit types, by their bytes (8192^2: softmax +3 %, LayerNorm +6 %;
  // 16384 x 4096 +6 % and +2 %)
  if (lego_rowwise_f16_wpr(M, 2 * N) == 8) return ok_or(lego_softmax_f32_w8_launch(x, y, M, N, as_stream(stream)));
  return ok_or((long_row ? lego_softmax_f32_w16_launch : lego_softmax_f32_w4_launch)(x, y, M, N, as_stream(stream)));
}

int lego_hip_layernorm_fwd_f16_wpr(const void* x, void* y, const void* w, const void* b,
                                   float* mean, float* rstd, int M, int N, float eps,
                                   int waves_per_row, void* stream)
{
  if (!usable(x) || !usable(y) || !usable(w) || !usable(b) || mean == nullptr || rstd == nullptr) return kInvalid;
  if (M <= 0 || N <= 0 || N % 8 || N > LEGO_ROWWISE_MAX_N || !(eps >= 0.0f)) return kInvalid;
  switch (waves_per_row) {
    case 1:   // rows of at most 16 or 32 vectors: several rows per wave
      return ok_or((N <= 128 ? lego_layernorm_fwd_f16_l16_launch : N <= 256 ? lego_layernorm_fwd_f16_l32_launch
                                                                         : lego_layernorm_fwd_f16_w1_launch)(
          x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
    case 2: return ok_or(lego_layernorm_fwd_f16_w2_launch(x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
    case 4: return ok_or(lego_layernorm_fwd_f16_w4_launch(x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
    case 8: return ok_or(lego_layernorm_fwd_f16_w8_launch(x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
    case 16: return ok_or(lego_layernorm_fwd_f16_w16_launch(x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
    default: return kInvalid;
  }
}

int lego_hip_layernorm_fwd_f16(const void* x, void* y, const void* w, const void* b,
                               float* mean, float* rstd, int M, int N, float eps, void* stream)
{
  if (!element_aligned(x, 2) || !element_aligned(y, 2) || !element_aligned(w, 2) || !element_aligned(b, 2)) return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4)) return kInvalid;
  if (M <= 0 || N <= 0 || N > LEGO_ROWWISE_MAX_N || !(eps >= 0.0f)) return kInvalid;
  const bool long_row = N > LEGO_ROWWISE_MAX_N_SMALL_TEAMS;
  if (N % 8 || !aligned16(x) || !aligned16(y) || !aligned16(w) || !aligned16(b))   // rows of any length, or at any element
    return ok_or((N <= 128 ? lego_layernorm_fwd_f16s_l16_launch : N <= 256 ? lego_layernorm_fwd_f16s_l32_launch
                  : lego_rowwise_f16_wpr(M, N) == 8 ? lego_layernorm_fwd_f16s_w8_launch
                  : long_row ? lego_layernorm_fwd_f16s_w16_launch : lego_rowwise_default_wpr(N) == 1 ? lego_layernorm_fwd_f16s_w1_launch
                                                                                                 : lego_layernorm_fwd_f16s_w4_launch)(
        x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  return lego_hip_layernorm_fwd_f16_wpr(x, y, w, b, mean, rstd, M, N, eps, lego_rowwise_f16_wpr(M, N), stream);
}

int lego_hip_layernorm_fwd_f32(const void* x, void* y, const void* w, const void* b,
                               float* mean, float* rstd, int M, int N, float eps, void* stream)
{
  if (!element_aligned(x, 4) || !element_aligned(y, 4) || !element_aligned(w, 4) || !element_aligned(b, 4)) return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4)) return kInvalid;
  if (M <= 0 || N <= 0 || N > LEGO_ROWWISE_MAX_N || !(eps >= 0.0f)) return kInvalid;
  const bool long_row = N > LEGO_ROWWISE_MAX_N_SMALL_TEAMS;
  if (N % 4 || !aligned16(x) || !aligned16(y) || !aligned16(w) || !aligned16(b))   // rows of any length, or at any element
    return ok_or((N <= 64 ? lego_layernorm_fwd_f32s_l16_launch : N <= 128 ? lego_layernorm_fwd_f32s_l32_launch
                  : lego_rowwise_f16_wpr(M, 2 * N) == 8 ? lego_layernorm_fwd_f32s_w8_launch
                  : long_row ? lego_layernorm_fwd_f32s_w16_launch : N <= 1024 ? lego_layernorm_fwd_f32s_w1_launch
                                                                            : lego_layernorm_fwd_f32s_w4_launch)(
        x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  if (N <= 1024)
    return ok_or((N <= 64 ? lego_layernorm_fwd_f32_l16_launch : N <= 128 ? lego_layernorm_fwd_f32_l32_launch
                                                                      : lego_layernorm_fwd_f32_w1_launch)(
        x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  if (lego_rowwise_f16_wpr(M, 2 * N) == 8)   // as the 16-bit types, by the bytes of a row
    return ok_or(lego_layernorm_fwd_f32_w8_launch(x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  return ok_or((long_row ? lego_layernorm_fwd_f32_w16_launch : lego_layernorm_fwd_f32_w4_launch)(
      x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
}

int lego_hip_softmax_bf16(const void* x, void* y, int M, int N, void* stream)
{
  if (!element_aligned(x, 2) || !element_aligned(y, 2) || M <= 0 || N <= 0) return kInvalid;
  if (N > LEGO_ROWWISE_MAX_N) return ok_or(lego_softmax_long_bf16_launch(x, y, M, N, as_stream(stream)));   // two passes
  const int wpr = lego_rowwise_default_wpr(N);
  if (N % 8 || !aligned16(x) || !aligned16(y))   // rows of any length, or at any element
    return ok_or((N <= 128 ? lego_softmax_bf16s_l16_launch : N <= 256 ? lego_softmax_bf16s_l32_launch
                  : lego_rowwise_f16_wpr(M, N) == 8 ? lego_softmax_bf16s_w8_launch
                  : wpr == 16 ? lego_softmax_bf16s_w16_launch : wpr == 1 ? lego_softmax_bf16s_w1_launch
                                                                       : lego_softmax_bf16s_w4_launch)(x, y, M, N, as_stream(stream)));
  if (N <= 256) return ok_or((N <= 128 ? lego_softmax_bf16_l16_launch : lego_softmax_bf16_l32_launch)(x, y, M, N, as_stream(stream)));
  if (lego_rowwise_f16_wpr(M, N) == 8) return ok_or(lego_softmax_bf16_w8_launch(x, y, M, N, as_stream(stream)));   // as fp16
  return ok_or((wpr == 16 ? lego_softmax_bf16_w16_launch : wpr == 1 ? lego_softmax_bf16_w1_launch
                                                                    : lego_softmax_bf16_w4_launch)(x, y, M, N, as_stream(stream)));
}

int lego_hip_layernorm_fwd_bf16(const void* x, void* y, const void* w, const void* b,
                                float* mean, float* rstd, int M, int N, float eps, void* stream)
{
  if (!element_aligned(x, 2) || !element_aligned(y, 2) || !element_aligned(w, 2) || !element_aligned(b, 2)) return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4)) return kInvalid;
  if (M <= 0 || N <= 0 || N > LEGO_ROWWISE_MAX_N || !(eps >= 0.0f)) return kInvalid;
  const int wpr = lego_rowwise_default_wpr(N);
  if (N % 8 || !aligned16(x) || !aligned16(y) || !aligned16(w) || !aligned16(b))   // rows of any length, or at any element
    return ok_or((N <= 128 ? lego_layernorm_fwd_bf16s_l16_launch : N <= 256 ? lego_layernorm_fwd_bf16s_l32_launch
                  : lego_rowwise_f16_wpr(M, N) == 8 ? lego_layernorm_fwd_bf16s_w8_launch
                  : wpr == 16 ? lego_layernorm_fwd_bf16s_w16_launch : wpr == 1 ? lego_layernorm_fwd_bf16s_w1_launch
                                                                             : lego_layernorm_fwd_bf16s_w4_launch)(
        x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  if (N <= 256)
    return ok_or((N <= 128 ? lego_layernorm_fwd_bf16_l16_launch : lego_layernorm_fwd_bf16_l32_launch)(
        x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  if (lego_rowwise_f16_wpr(M, N) == 8)   // as fp16
    return ok_or(lego_layernorm_fwd_bf16_w8_launch(x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
  return ok_or((wpr == 16 ? lego_layernorm_fwd_bf16_w16_launch : wpr == 1 ? lego_layernorm_fwd_bf16_w1_launch
                                                                          : lego_layernorm_fwd_bf16_w4_launch)(
      x, y, w, b, mean, rstd, M, N, eps, as_stream(stream)));
}

int lego_hip_layernorm_bwd_workspace_bytes(int M, int N, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || N > LEGO_LAYERNORM_BWD_MAX_N) return kInvalid;
  const unsigned long long pitch = (static_cast<unsigned long long>(N) + 7) / 8 * 8;
  *bytes = 2ull * lego_layernorm_bwd_groups(M, N) * pitch * sizeof(float);
  return 0;
}

int lego_hip_layernorm_bwd_f16(const void* dy, const void* x, const void* w, const float* mean,
                               const float* rstd, void* dx, void* dw, void* db, void* workspace,
                               unsigned long long workspace_bytes, int M, int N, void* stream)
{
  unsigned long long need = 0;
  if (lego_hip_layernorm_bwd_workspace_bytes(M, N, &need) != 0) return kInvalid;
  if (!element_aligned(dy, 2) || !element_aligned(x, 2) || !element_aligned(w, 2) || !element_aligned(dx, 2) ||
      !element_aligned(dw, 2) || !element_aligned(db, 2) || !usable(workspace))
    return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4) || workspace_bytes < need) return kInvalid;
  const int any_base = !(aligned16(dy) && aligned16(x) && aligned16(w) && aligned16(dx));
  return ok_or(lego_layernorm_bwd_f16_launch(dy, x, w, mean, rstd, dx, dw, db, static_cast<float*>(workspace), M, N, any_base,
                                             as_stream(stream)));
}

int lego_hip_layernorm_bwd_f16_noalloc(const void* dy, const void* x, const void* w, const float* mean,
                                       const float* rstd, void* dx, void* dw, void* db, int M, int N, void* stream)
{
  unsigned long long need = 0;
  if (lego_hip_layernorm_bwd_workspace_bytes(M, N, &need) != 0) return kInvalid;
  if (need > kScratchBytes) return kInvalid;     // partial rows beyond the built-in scratch
  if (!element_aligned(dy, 2) || !element_aligned(x, 2) || !element_aligned(w, 2) || !element_aligned(dx, 2) ||
      !element_aligned(dw, 2) || !element_aligned(db, 2))
    return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4)) return kInvalid;
  const int any_base = !(aligned16(dy) && aligned16(x) && aligned16(w) && aligned16(dx));
  float* partials = nullptr;
  const hipError_t err = scratch_address(&partials);
  if (err != hipSuccess) return ok_or(err);
  // every partial row that the reduction reads is written by the first stage of the same call, so
  // what an earlier call left in the array needs no clearing
  return ok_or(lego_layernorm_bwd_f16_launch(dy, x, w, mean, rstd, dx, dw, db, partials, M, N, any_base, as_stream(stream)));
}

int lego_hip_layernorm_bwd_f32_workspace_bytes(int M, int N, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || N > LEGO_LAYERNORM_BWD_MAX_N) return kInvalid;
  const unsigned long long pitch = (static_cast<unsigned long long>(N) + 7) / 8 * 8;
  *bytes = 2ull * lego_layernorm_bwd_f32_groups(M, N) * pitch * sizeof(float);
  return 0;
}

int lego_hip_layernorm_bwd_f32(const void* dy, const void* x, const void* w, const float* mean,
                               const float* rstd, void* dx, void* dw, void* db, void* workspace,
                               unsigned long long workspace_bytes, int M, int N, void* stream)
{
  unsigned long long need = 0;
  if (lego_hip_layernorm_bwd_f32_workspace_bytes(M, N, &need) != 0) return kInvalid;
  if (!element_aligned(dy, 4) || !element_aligned(x, 4) || !element_aligned(w, 4) || !element_aligned(dx, 4) ||
      !element_aligned(dw, 4) || !element_aligned(db, 4) || !usable(workspace))
    return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4) || workspace_bytes < need) return kInvalid;
  const int any_base = !(aligned16(dy) && aligned16(x) && aligned16(w) && aligned16(dx));
  return ok_or(lego_layernorm_bwd_f32_launch(dy, x, w, mean, rstd, dx, dw, db, static_cast<float*>(workspace), M, N, any_base,
                                             as_stream(stream)));
}

int lego_hip_layernorm_bwd_bf16_workspace_bytes(int M, int N, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || N > LEGO_LAYERNORM_BWD_MAX_N) return kInvalid;
  const unsigned long long pitch = (static_cast<unsigned long long>(N) + 7) / 8 * 8;
  *bytes = 2ull * lego_layernorm_bwd_bf16_groups(M, N) * pitch * sizeof(float);
  return 0;
}

int lego_hip_layernorm_bwd_bf16(const void* dy, const void* x, const void* w, const float* mean,
                                const float* rstd, void* dx, void* dw, void* db, void* workspace,
                                unsigned long long workspace_bytes, int M, int N, void* stream)
{
  unsigned long long need = 0;
  if (lego_hip_layernorm_bwd_bf16_workspace_bytes(M, N, &need) != 0) return kInvalid;
  if (!element_aligned(dy, 2) || !element_aligned(x, 2) || !element_aligned(w, 2) || !element_aligned(dx, 2) ||
      !element_aligned(dw, 2) || !element_aligned(db, 2) || !usable(workspace))
    return kInvalid;
  if (!element_aligned(mean, 4) || !element_aligned(rstd, 4) || workspace_bytes < need) return kInvalid;
  const int any_base = !(aligned16(dy) && aligned16(x) && aligned16(w) && aligned16(dx));
  return ok_or(lego_layernorm_bwd_bf16_launch(dy, x, w, mean, rstd, dx, dw, db, static_cast<float*>(workspace), M, N, any_base,
                                              as_stream(stream)));
}

namespace {
typedef hipError_t (*gemm_launcher)(const void*, const void*, void*, int, int, int, int, hipStream_t);
struct GemmKernels {
  gemm_launcher big[4];     // 256 x 256 tiles, one workgroup per CU; index 2*trans_a + trans_b
  gemm_launcher small[4];   // 128 x 128 tiles, two workgroups per CU (null: not built for this type)
  gemm_launcher deep[4];    // 128 x 128 tiles on four buffers of LDS, one workgroup per CU
  gemm_launcher sparse[4];  // 256 x 256 tiles on 32x32x16 MFMAs, for launches that leave many CUs idle (null: not built for this type)
};
// Fewer 256 x 256 tiles than this and the 128 x 128 kernel, with four times as many workgroups,
// keeps more of the 256 CUs busy than its higher LDS traffic per flop costs.
constexpr long kSmallTileBelow = 129;
// One round of 256 x 256 tiles that leaves this many CUs or more without a tile runs faster on the 32x32x16 MFMA: away
// from the socket's power limit its fewer LDS reads per flop count for more than the 16x16x32's lower energy per flop
// (fp16, 144 tiles: 0.95 -> 1.02 PFLOP/s at 2304 x 4096 x 4096, 0.75 -> 0.85 at 3072 x 3072 x 1024; 160 tiles 1.05 -> 1.08;
// 176 tiles 1.08 -> 1.09; 192 tiles 1.16 -> 1.14).
constexpr long kSparseRoundBelow = 176;
// Time of a last round in which only `share` of the workgroup slots hold a tile, in units of a full round.  A few busy
// CUs run at the clock that the socket's power limit denies the full chip, so the round is shorter than a full one
// even though each of its tiles takes a CU to itself.
inline double partial_round(double share, double least, double knee)
{
  if (share <= 0.0) return 0.0;
  return share <= knee ? least : least + (share - knee) * (1.0 - least) / (1.0 - knee);
}
// Larger products whose 256 x 256 tiles leave the last round of workgroups mostly empty take the small tile when the
// estimate of its time is the lower one: whole rounds of 256 big or 512 small tiles (the small tile runs at about 0.8
// of the large tile's rate, so a round of it costs 0.625 of a big one) plus the partial last round.  Measured on fp16
// products 4096 deep, time of a round of big tiles by the share of CUs it keeps busy: 0.06-0.5 -> 0.69-0.71, 0.56 ->
// 0.76, 0.69 -> 0.82, 0.81 -> 0.88, 0.94 -> 0.97; of small tiles: 0.13 -> 0.51, 0.5 -> 0.58.  4352 x 4096 x 4096 (272
// tiles): 0.81 big, 0.87 small; 5120 x 4096 (320): 0.95 / 1.00; 4608^3 (324): 0.98 / 1.02; 6144 x 4096 (384, a half
// round left over): 1.13 / 1.04; 5120^3 and 6144^3 stay with the big tile.
inline bool small_tiles_fill_better(int M, int N, long tiles)
{
  if (tiles < kSmallTileBelow) return true;
  const long small = static_cast<long>((M + 127) / 128) * ((N + 127) / 128);
  const double big_time = static_cast<double>(tiles / 256) + partial_round(static_cast<double>(tiles % 256) / 256.0, 0.69, 0.5);
  const double small_time = 0.625 * (static_cast<double>(small / 512) + partial_round(static_cast<double>(small % 512) / 512.0, 0.5, 0.4));
  return small_time < big_time;
}

// Which build a product in whole 16-byte chunks takes: 0 = 256 x 256 tiles on the type's own MFMA, 1 = 128 x 128 tiles,
// 2 = 256 x 256 tiles on the 32x32x16 MFMA (16-bit operands: one round that leaves a third of the CUs idle).
inline int gemm_choice(int M, int N, bool has_small, bool has_sparse)
{
  const long tiles = static_cast<long>((M + LEGO_GEMM_BM - 1) / LEGO_GEMM_BM) * ((N + LEGO_GEMM_BN - 1) / LEGO_GEMM_BN);
  if (has_small && small_tiles_fill_better(M, N, tiles)) return 1;
  return has_sparse && tiles < kSparseRoundBelow ? 2 : 0;
}

// Few rows against a k-major B: columns of C per workgroup of the kernel that reads B once, straight into registers, or 0: tiles.
// A workgroup reads its columns of B and all of A, which tell in rounds of one workgroup per CU: the least of rounds * (columns + 3/4 M), and 4 KB
// of a row for a workgroup's start; wider where that is a thirtieth less (16 / 32 / 64 columns, us, bf16: 1 x 8576 x 6784 32 / 39 / 37, 16 x 8192 x 8192
// 35 / 25 / 46, 16 x 16384 x 8192 68 / 58 / 52; over 2148 drawn products 1.004 of the best of the three).  Tiles / this: 16 x 1024 x 1024 12.0 / 4.6, 16 x 4096 x 4096 15.0 / 10.3, 16 x 8192 x 8192 33.2 / 25.3,
// 16 x 16384 x 4096 33.4 / 27.8, 1 x 5120 x 8192 28.7 / 19.0.  Tiles are better
//   where there is next to nothing to read: K of 256 bytes 4.4 / 5.0, of 384 4.5 / 5.0 (8 x 23040 x 432 of 8 bits 7.3 / 5.2);
//   where K is long beside N: 1024 x 8192 16.0 / 16.8 (and 64 x 8192 14.2 / 16.7);
//   of many columns, where they fill the chip without a split: 16 x 40960 x 8192 174 / 191 (from 2 KB a row on: 12 x 46912 x 544 15.4 / 13.1), 8 x 65536 x 6144 151 / 163;
//   of more than eight rows, for which A is read often: 16 x 2048 x 6144 12.8 / 13.6, 16 x 5120 x 5120 18.1 / 20.7 (5120 x 4096 20.6 / 13.8, and of
//   eight rows all that was drawn), 16 x 8448 x 10240 54 / 64.
// Of 32 rows, which read A twice as often, 8192 x 8192 34.3 / 34.5.
inline int rows_columns(int M, int N, int K, int trans_a, int trans_b, int bytes)
{
  const long k_bytes = static_cast<long>(K) * bytes;
  if (M > 16 || trans_a || !trans_b || N < 1024 || K > 4l * N || k_bytes <= (N <= 8192 ? 384 : 256) || 64 * k_bytes >= (1l << 31) || static_cast<long>(N) * K >= (1l << 31)) return 0;
  if (N > (M > 8 && k_bytes > 2 << 10 ? 36864 : 49152)) return 0;
  if (M > 8 && ((N < 2560 && k_bytes >= 11 << 10) || (N > 4096 && N < 6144 && k_bytes > 8 << 10) || (N > 8192 && N < 12288 && k_bytes > 16 << 10))) return 0;
  int best = 0;
  long least = 0;
  for (const int columns : {16, 32, 64}) {
    const long rounds = ((N + columns - 1) / columns + 255) / 256, cost = rounds * (k_bytes * (4 * columns + 3 * M) + (16 << 10));
    if (best == 0 || 33 * cost < 32 * least) { best = columns; least = cost; }
  }
  return best;
}

// Up to one 128 x 128 tile per CU runs on four buffers of LDS instead of two workgroups of two: what bounds such a launch is how far ahead
// of a workgroup's k-tiles its operands are asked for.  us, two buffers / four, operands from memory (from the caches): e5m2 1000 x
// 2048 x 2048 18.0 / 12.9 (10.4 / 9.1), fp16 2048^3 (256 tiles) 31.4 / 22.7 (25.3 / 20.1), 256 x 4096 x 1024 16.4 / 11.6 (8.6 / 8.5), 64 x 2800 x 128
// 4.2 / 4.0.  Beyond, two workgroups per CU are ahead: 2304 x 2048 x 2048 (288 tiles) 32.5 / 35.3, 4096 x 2048 x 2048 42.6 / 44.5, 2496 x 2944 x 512
// 14.9 / 22.5.  A lane's offset within a tile stays below a descriptor's 2 GiB.
constexpr long kDeepTiles = 256;
inline bool deep_offsets(int M, int N, int K, int bytes) { return 128l * bytes * std::max(M, std::max(N, K)) < (1l << 31); }
inline bool deep_tiles(int M, int N, int K, int bytes)
{
  return static_cast<long>((M + 127) / 128) * ((N + 127) / 128) <= kDeepTiles && deep_offsets(M, N, K, bytes);
}

int gemm_ex(const GemmKernels& k, int element, const void* a, const void* b, void* c, int M, int N, int K,
            int trans_a, int trans_b, int activation, void* stream, int bk = LEGO_GEMM_BK, int chunk = 8)
{
  if (a == nullptr || b == nullptr || c == nullptr || M <= 0 || N <= 0 || K <= 0) return kInvalid;
  if (activation != 0 && activation != 1) return kInvalid;
  // The tiled kernels move 16-byte chunks (`chunk` elements): bases 16-byte aligned and every operand row
  // in whole chunks -- rows of C and of B as given run along N, rows of A as given and of a transposed B
  // along K, rows of a transposed A along M.  Tiles may be ragged in M, N and K.  Everything else -- the
  // reference keeps M, N, K symbolic (matmul_sympy.py:69-70) -- goes to the kernel that reads vectors at any
  // element.
  (void)bk;
  const bool tiled = usable(a) && usable(b) && usable(c) && N % chunk == 0 &&
                     (trans_a ? M % chunk == 0 : K % chunk == 0) && (!trans_b || K % chunk == 0);
  if (!tiled) {
    const uintptr_t in_mask = element <= 1 || element == 4 ? 1u : 0u;       // 2-byte or 1-byte operand elements; C is 2-byte
    if ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b)) & in_mask) return kInvalid;
    if (reinterpret_cast<uintptr_t>(c) & 1u) return kInvalid;
    return ok_or(lego_gemm_any_launch(a, b, c, M, N, K, trans_a ? 1 : 0, trans_b ? 1 : 0, activation, element,
                                      as_stream(stream)));
  }
  if (const int columns = rows_columns(M, N, K, trans_a, trans_b, element == 2 || element == 3 ? 1 : 2))
    return ok_or(lego_gemm_rows_launch(a, b, c, M, N, K, columns, activation, element, as_stream(stream)));
  const int layout = (trans_a ? 2 : 0) + (trans_b ? 1 : 0);
  const int choice = gemm_choice(M, N, k.small[layout] != nullptr, k.sparse[layout] != nullptr);
  const gemm_launcher* by_layout = choice == 1 && deep_tiles(M, N, K, 16 / chunk) ? k.deep : choice == 1 ? k.small : choice == 2 ? k.sparse : k.big;
  return ok_or(by_layout[layout](a, b, c, M, N, K, activation, as_stream(stream)));
}

// Parts along K for a product of few tiles (1: one workgroup per tile does it all): as many as the estimate of the launch's time is least
// for, one round of workgroups of two k-tiles each at least.  In ns, whole 2400 + 420 per k-tile; parts 5200, the second launch in it, 420
// per k-tile of a part, and the sums of every part, 24 for a tile's worth of them and 4 for each workgroup.  Fitted to 90 drawn products of up
// to 128 tiles in each number of parts: the rule takes 1.016 times the best of them with operands from memory, 1.014 from the caches.  us
// from memory (from the caches), whole / parts: fp16 512 x 512 x 512 5.8 / two 6.8, 512 x 512 x 1024 8.4 / four 7.4, 1024^3 9.0 / two 10.6, 1024 x 2048 x 3584
// 35.0 (24.5) / two 29.0 (27.0), 1024 x 1024 x 4096 36.0 (24.8) / three 20.9 (18.4), four 20.7 (19.6), six, more than a round, 26.4 (23.5); 16 x 8192 x 8192
// 54.6 / three 27.7, four 29.0; e5m2 1000 x 2048 x 2048 12.9 / two 15.2, 256 x 2048 x 4096 22.0 / four 12.5; e4m3 1024 x 1024 x 4096 19.6 / three 14.7.
int splitk_parts(int M, int N, int K, int bk)
{
  const long tiles = static_cast<long>((M + 127) / 128) * ((N + 127) / 128), depth = (K + bk - 1) / bk;
  if (tiles > kDeepTiles / 2) return 1;
  // chains of 65537 k-tiles and more, past the reach of a descriptor: two workgroups per CU on two buffers
  if (!deep_offsets(M, N, K, 2 * LEGO_GEMM_BK / bk)) return static_cast<int>(std::min((512 + tiles - 1) / tiles, 64l));
  const long most = std::min(std::min(kDeepTiles / tiles, depth / 2), 64l);
  long best = 1, least = 2400 + 420 * depth;
  for (long parts = 2; parts <= most; ++parts) {
    const long sums = 24l * M * N / (128 * 128) + 4 * tiles;
    const long time = 5200 + parts * sums + 420 * ((depth + parts - 1) / parts);
    if (time < least) { best = parts; least = time; }
  }
  return static_cast<int>(best);
}
// As many of those parts as a launch takes: three quarters where all would put a workgroup on every CU, each reading rows of a k-major operand of up to 64
// rows or columns against a large one from a multiple of 32 k-tiles on: they are then a multiple of 4 KiB apart in every row, and what they ask memory for at a time
// falls on few of its channels.  us from memory (from the caches), 256 workgroups / 192: fp16 24 x 8192 x 8192 with B transposed 39.0 (24.5) / 33.2 (24.5),
// 64 x 8192 x 8192 42.0 (27.5) / 35.0 (27.2), 8192 x 64 x 8192 39.8 (26.3) / 33.2 (26.0), e5m2 24 x 8192 x 16384 38.9 / 33.3; parts of 20 k-tiles, 40 x 8192 x 5120, 22.0 / 23.0, of 16,
// 24 x 4096 x 8192, 17.8 / 18.4, and 128 rows, 128 x 8192 x 16384, 61.6 / 65.2 from the caches, stay whole rounds.
int launched_parts(int parts, int M, int N, int K, int trans_a, int trans_b, int bk)
{
  const long tiles = static_cast<long>((M + 127) / 128) * ((N + 127) / 128), depth = (K + bk - 1) / bk;
  const bool few = (M <= 64 && trans_b) || (N <= 64 && !trans_a);
  return few && parts >= 4 && parts * tiles == kDeepTiles && (depth + parts - 1) / parts % 32 == 0 ? parts - parts / 4 : parts;
}
typedef hipError_t (*splitk_launcher)(const void*, const void*, void*, int, int, int, int, int, float*, hipStream_t);
struct SplitkKernels {
  splitk_launcher deep[4], far[4];      // on four buffers; on two, whose instructions have bases of their own and reach 4 GiB from there: index 2*trans_a + trans_b
  splitk_launcher of(int M, int N, int K, int trans_a, int trans_b, int bytes) const
  {
    return (deep_offsets(M, N, K, bytes) ? deep : far)[(trans_a ? 2 : 0) + (trans_b ? 1 : 0)];
  }
};
#define LEGO_SPLITK(DT) {{lego_gemm_##DT##_nn_t128x128_deep_splitk_launch, lego_gemm_##DT##_nt_t128x128_deep_splitk_launch,  \
                          lego_gemm_##DT##_tn_t128x128_deep_splitk_launch, lego_gemm_##DT##_tt_t128x128_deep_splitk_launch}, \
                         {lego_gemm_##DT##_nn_t128x128_splitk_launch, lego_gemm_##DT##_nt_t128x128_splitk_launch,            \
                          lego_gemm_##DT##_tn_t128x128_splitk_launch, lego_gemm_##DT##_tt_t128x128_splitk_launch}}

// Operand rows that are not whole 16-byte chunks: the tiled kernels run on zero-padded copies (every side a multiple of `chunk`
// elements; the padding adds zeros to the sums) and the result is copied back: two more launches and three more passes over
// the matrices, against the kernel that takes any shape, here when it moved one element per access.  8-bit operands, us by
// elements / on copies: 320 x 1984 x 7959 829 / 35, 2000 x 2000 x 2001 276 / 27, 5000 x 3001 x 136 93 / 32, 6902 x 192 x 296 31 / 28, 1000 x
// 1001 x 264 38 / 14, 16 x 65 x 257 20 / 16, 33 x 100 x 200 16 / 23, 1000 x 1000 x 136 16 / 22: copies from K = 256 on, or from as many 64 x 64 tiles of the
// result as kept it busy for 30 us; of these the rule below sends to that kernel what it now does sooner.
inline bool copies_gain_8bit(int M, int N, int K)
{
  const double tiles = static_cast<double>((M + 63) / 64) * ((N + 63) / 64);
  return K >= 256 || tiles * K >= 150000.0;
}
inline int round_up(int v, int to) { return (v + to - 1) / to * to; }
inline unsigned long long padded_bytes(int M, int N, int K, int chunk, int bytes)
{
  const unsigned long long m = round_up(M, chunk), n = round_up(N, chunk), k = round_up(K, chunk);
  return bytes * (m * k + k * n) + 2ull * m * n;
}
// Whether a product whose rows are not whole 16-byte chunks is better off with the kernel that takes any than on padded copies, one or two
// launches more.  In us: there 3.7 and the longer of one tile's chain of k-tiles and the tiles' work over the chip's CUs; here 9.5, or 8.2 where
// the result is not copied back, and the copies' bytes, read and written, at 2 TB/s.  Over 203 drawn ragged products of all types and layouts the
// rule takes 0.80 of the time on copies, the better of the two each time 0.78.  us direct / on copies, 16 bits: 64 x 852 x 64 4.5 / 10.5, 55 x 512 x 93
// 5.6 / 15.3, 64 x 3594 x 314 6.6 / 10.9, 3039 x 336 x 518 10.8 / 13.0; 6 x 383 x 1688 16.4 / 14.4, 1152 x 5120 x 113 19.2 / 10.5, 1618 x 2024 x 485
// 22.3 / 14.6, 496 x 135 x 3878 24.4 / 18.6.  Those had sides
// of up to 8192; taller ones are bound by memory, 2 TB/s there too, and an A beyond the L2s' 32 MB is read again for every column of tiles: 4194305 x 63 x 63
// 657 / 755, 4194241 x 9 x 130 516 / 789, 1000000 x 63 x 63 137 / 185; 5000000 x 100 x 60 989 / 880, 1000000 x 100 x 60 201 / 196, 100000 x 66 x 200 with B
// transposed 28.4 / 26.2; 20000 x 1001 x 50, whose A stays in the L2s, 29.4 / 32.5.  (7778 x 110 x 2114 with B transposed is 17.3 / 32.0.)
inline bool direct_gains(int M, int N, int K, int trans_a, int trans_b, int chunk, int bytes)
{
  const double tiles = static_cast<double>((M + 63) / 64) * ((N + 63) / 64), depth = (K + 63) / 64;
  const double step = !trans_a && trans_b && K % 8 == 0 ? 0.25 : 0.42;      // both operands k-major: four accesses a lane and k-tile instead of eight
  const double a_bytes = static_cast<double>(bytes) * M * K, reads = a_bytes > 32e6 ? (N + 63) / 64 : 1;
  // A large A in whole chunks is no copy: the product reads it where it is, at 4.5 TB/s, and here its tiles are bound by how often it is read.  us direct / on copies
  // from memory: bf16 6174 x 68 x 5808 with B transposed 41.9 / 31.2, f16 7452 x 277 x 5680 115 / 68, bf16 6831 x 315 x 3176 with A stored row-major first 89 / 61.
  const bool in_place = a_bytes > 32e6 && K % chunk == 0 && !(trans_a && M % chunk);
  const double work = in_place && step < 0.42 ? 0.45 : 0.9 * step;
  const double memory = M > 8192 ? (reads * a_bytes + 2.0 * M * N) / 2e6 : 0.0;
  const double direct = 3.7 + std::max(std::max(step * depth, (1 + work * depth) * tiles / 256), memory);
  const bool back = N % chunk || (trans_a && M % chunk);
  const double results = back ? 0.0 : 2.0 * round_up(M, chunk) * N;
  const double copied = padded_bytes(M, N, K, chunk, bytes) - results - (in_place ? static_cast<double>(bytes) * round_up(M, chunk) * K : 0.0);
  return direct <= (back ? 9.5 : 8.2) + copied / 2e6 + (in_place ? a_bytes / 4.5e6 : 0.0);
}
inline unsigned long long parts_bytes(int M, int N, int parts)
{
  const unsigned long long tiles = static_cast<unsigned long long>((M + 127) / 128) * ((N + 127) / 128);
  return parts > 1 ? parts * tiles * 128ull * 128ull * sizeof(float) : 0ull;
}

// `product(a, b, c, M, N, K, sums)` on padded copies in the workspace, whose part for sums follows them.
extern "C++" template <class Product>
int on_padded_copies(int chunk, int bytes, const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                     void* workspace, void* stream, const Product& product)
{
  const int Mr = round_up(M, chunk), Nr = round_up(N, chunk), Kr = round_up(K, chunk);
  const int Mp = trans_a ? Mr : M;                 // rows of the padded product: a transposed A has rows of M elements
  uint8_t* ap = static_cast<uint8_t*>(workspace);
  uint8_t* bp = ap + static_cast<size_t>(Mr) * Kr * bytes;
  uint8_t* cp = bp + static_cast<size_t>(Kr) * Nr * bytes;
  void* sums = cp + static_cast<size_t>(Mr) * Nr * 2;
  const bool copy_a = Kr != K || Mp != M || !usable(a), copy_b = Kr != K || Nr != N || !usable(b), copy_c = Nr != N || Mp != M || !usable(c);
  Copier pads(true, as_stream(stream));
  if (copy_a) trans_a ? pads.add(a, ap, K, M, Kr, Mr, bytes) : pads.add(a, ap, M, K, M, Kr, bytes);
  if (copy_b) trans_b ? pads.add(b, bp, N, K, Nr, Kr, bytes) : pads.add(b, bp, K, N, Kr, Nr, bytes);
  const hipError_t err = pads.flush();
  if (err != hipSuccess) return ok_or(err);
  const int rc = product(copy_a ? ap : a, copy_b ? bp : b, copy_c ? cp : c, Mp, Nr, Kr, sums);
  if (rc != 0 || !copy_c) return rc;
  Copier back(false, as_stream(stream));
  back.add(cp, c, M, N, M, Nr, 2);
  return ok_or(back.flush());
}

// 8-bit operands: both tile sizes in all four layouts, one MFMA shape.  The rule between the tiles is that of the 16-bit
// operands; us on big / small tiles, e5m2 A*B: 512 x 512 x 2048 19.5 / 8.6, 1000 x 2048 x 2048 22.1 / 13.6 (32 and 128
// workgroups), 2048^3 22.0 / 14.1, 2048 x 4096 x 4096 39.4 / 31.0, 4352 x 4096 x 4096 78.4 / 73.7, 4608^3 88.3 / 84.6.
#define LEGO_GEMM_KERNELS_8BIT(DT)                                                                     \
  {{lego_gemm_##DT##_nn_launch, lego_gemm_##DT##_nt_launch, lego_gemm_##DT##_tn_launch,              \
    lego_gemm_##DT##_tt_launch},                                                                       \
   {lego_gemm_##DT##_nn_t128x128_launch, lego_gemm_##DT##_nt_t128x128_launch,                         \
    lego_gemm_##DT##_tn_t128x128_launch, lego_gemm_##DT##_tt_t128x128_launch},                         \
   {lego_gemm_##DT##_nn_t128x128_deep_launch, lego_gemm_##DT##_nt_t128x128_deep_launch,               \
    lego_gemm_##DT##_tn_t128x128_deep_launch, lego_gemm_##DT##_tt_t128x128_deep_launch},               \
   {nullptr, nullptr, nullptr, nullptr}}
#define LEGO_GEMM_KERNELS(DT)                                                                          \
  {{lego_gemm_##DT##_nn_launch, lego_gemm_##DT##_nt_launch, lego_gemm_##DT##_tn_launch,              \
    lego_gemm_##DT##_tt_launch},                                                                       \
   {lego_gemm_##DT##_nn_t128x128_launch, lego_gemm_##DT##_nt_t128x128_launch,                         \
    lego_gemm_##DT##_tn_t128x128_launch, lego_gemm_##DT##_tt_t128x128_launch},                         \
   {lego_gemm_##DT##_nn_t128x128_deep_launch, lego_gemm_##DT##_nt_t128x128_deep_launch,               \
    lego_gemm_##DT##_tn_t128x128_deep_launch, lego_gemm_##DT##_tt_t128x128_deep_launch},               \
   {lego_gemm_##DT##_nn_m32_launch, lego_gemm_##DT##_nt_m32_launch, lego_gemm_##DT##_tn_m32_launch,  \
    lego_gemm_##DT##_tt_m32_launch}}
}  // namespace

int lego_hip_gemm_f16_ex(const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                         int activation, void* stream)
{
  static const GemmKernels k = LEGO_GEMM_KERNELS(f16);
  return gemm_ex(k, 0, a, b, c, M, N, K, trans_a, trans_b, activation, stream);
}

int lego_hip_gemm_bf16_ex(const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                          int activation, void* stream)
{
  static const GemmKernels k = LEGO_GEMM_KERNELS(bf16);
  return gemm_ex(k, 1, a, b, c, M, N, K, trans_a, trans_b, activation, stream);
}

int lego_hip_gemm_bf16_f16_ex(const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                              int activation, void* stream)
{
  static const GemmKernels k = LEGO_GEMM_KERNELS(bf16h);
  return gemm_ex(k, 4, a, b, c, M, N, K, trans_a, trans_b, activation, stream);
}

namespace {
// Room that a product of this kind uses: for zero-padded copies of both operands and of the result, N or K not being a multiple of 8 (M only
// matters as the row length of a transposed A; that case alone stays with the kernel for any shape), and for its sums, `parts(M, N, K)` of them.
extern "C++" template <class Parts>
unsigned long long room_16bit(int M, int N, int K, const Parts& parts)
{
  unsigned long long copies = 0;
  if (N % 8 || K % 8) {
    copies = padded_bytes(M, N, K, 8, 2);
    M = round_up(M, 8); N = round_up(N, 8); K = round_up(K, 8);     // the product that then runs
  }
  return copies + parts_bytes(M, N, parts(M, N, K));
}
// What the entry points that know no layout ask for where there are no copies: the products they split are those of 32 k-tiles and more, of 8-bit operands those of up to two
// tiles' worth of the result per k-tile.
int stated_parts(int M, int N, int K, int bk)
{
  const long tiles = static_cast<long>((M + 127) / 128) * ((N + 127) / 128), depth = (K + bk - 1) / bk;
  if (tiles > kDeepTiles / 2 || depth < 32 || (bk == LEGO_GEMM_BK_8BIT && static_cast<long>(M) * N > 2 * depth * 128 * 128)) return 1;
  return std::max(2, splitk_parts(M, N, K, bk));
}
}  // namespace

int lego_hip_gemm_workspace_bytes(int M, int N, int K, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || K <= 0) return kInvalid;
  const bool copied = N % 8 || K % 8;
  *bytes = room_16bit(M, N, K, [=](int m, int n, int k) { return (copied ? splitk_parts : stated_parts)(m, n, k, LEGO_GEMM_BK); });
  return 0;
}

int lego_hip_gemm_ex_ws(int element, const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                        int activation, void* workspace, unsigned long long workspace_bytes, void* stream)
{
  static const SplitkKernels f16 = LEGO_SPLITK(f16), bf16 = LEGO_SPLITK(bf16), bf16h = LEGO_SPLITK(bf16h);
  if (element != 0 && element != 1 && element != 4) return kInvalid;
  const SplitkKernels& kernels = element == 0 ? f16 : element == 1 ? bf16 : bf16h;
  const auto whole = [&](const void* aa, const void* bb, void* cc, int m, int n, int k) {
    switch (element) {
      case 0: return lego_hip_gemm_f16_ex(aa, bb, cc, m, n, k, trans_a, trans_b, activation, stream);
      case 1: return lego_hip_gemm_bf16_ex(aa, bb, cc, m, n, k, trans_a, trans_b, activation, stream);
      default: return lego_hip_gemm_bf16_f16_ex(aa, bb, cc, m, n, k, trans_a, trans_b, activation, stream);
    }
  };
  if (M <= 0 || N <= 0 || K <= 0) return kInvalid;
  const unsigned long long need = room_16bit(M, N, K, [](int m, int n, int k) { return splitk_parts(m, n, k, LEGO_GEMM_BK); });
  if (need == 0 || workspace_bytes < need || !usable(workspace)) return whole(a, b, c, M, N, K);
  const bool tiled = usable(a) && usable(b) && usable(c) && N % 8 == 0 && (trans_a ? M % 8 == 0 : K % 8 == 0) &&
                     (!trans_b || K % 8 == 0);
  if (!tiled && N % 8 == 0 && K % 8 == 0) return whole(a, b, c, M, N, K);
  if (a == nullptr || b == nullptr || c == nullptr || (activation != 0 && activation != 1)) return kInvalid;
  if ((reinterpret_cast<uintptr_t>(a) | reinterpret_cast<uintptr_t>(b) | reinterpret_cast<uintptr_t>(c)) & 1u) return kInvalid;
  const auto product = [&](const void* aa, const void* bb, void* cc, int m, int n, int k, void* sums) {
    // as many parts as there is room for: that of a product on copies is asked for with M rounded up, and the estimate of a smaller M
    // may want more of them (130 x 136 x 8200 43, 136 x 136 x 8200 33)
    const int parts = N % 8 || K % 8 ? splitk_parts(round_up(m, 8), n, round_up(k, 8), LEGO_GEMM_BK) : splitk_parts(m, n, k, LEGO_GEMM_BK);
    if (parts < 2 || rows_columns(m, n, k, trans_a, trans_b, 2)) return whole(aa, bb, cc, m, n, k);
    return ok_or(kernels.of(m, n, k, trans_a, trans_b, 2)(aa, bb, cc, m, n, k, activation, launched_parts(parts, m, n, k, trans_a, trans_b, LEGO_GEMM_BK), static_cast<float*>(sums), as_stream(stream)));
  };
  if (tiled) return product(a, b, c, M, N, K, workspace);
  return on_padded_copies(8, 2, a, b, c, M, N, K, trans_a, trans_b, workspace, stream, product);
}

int lego_hip_gemm_fp8_ex(const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                         int activation, int format, void* stream)
{
  static const GemmKernels e4m3 = LEGO_GEMM_KERNELS_8BIT(e4m3);
  static const GemmKernels e5m2 = LEGO_GEMM_KERNELS_8BIT(e5m2);
  if (format != 0 && format != 1) return kInvalid;
  return gemm_ex(format == 0 ? e4m3 : e5m2, format == 0 ? 2 : 3, a, b, c, M, N, K, trans_a, trans_b, activation,
                 stream, LEGO_GEMM_BK_8BIT, 16);
}

// Room for the sums of a split product; none where gemm_ex would not take the tiled kernels in any layout.
int lego_hip_gemm_fp8_workspace_bytes(int M, int N, int K, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || K <= 0) return kInvalid;
  *bytes = parts_bytes(M, N, N % 16 ? 1 : stated_parts(M, N, K, LEGO_GEMM_BK_8BIT));
  return 0;
}

namespace {
const SplitkKernels& fp8_parts(int format)
{
  static const SplitkKernels e4m3 = LEGO_SPLITK(e4m3), e5m2 = LEGO_SPLITK(e5m2);
  return format == 0 ? e4m3 : e5m2;
}
}  // namespace

int lego_hip_gemm_fp8_ex_ws(const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                            int activation, int format, void* workspace, unsigned long long workspace_bytes, void* stream)
{
  if ((format != 0 && format != 1) || M <= 0 || N <= 0 || K <= 0) return kInvalid;
  const bool tiled = usable(a) && usable(b) && usable(c) && N % 16 == 0 && (trans_a ? M % 16 == 0 : K % 16 == 0) &&
                     (!trans_b || K % 16 == 0);
  const int parts = splitk_parts(M, N, K, LEGO_GEMM_BK_8BIT);
  if (parts < 2 || !tiled || !usable(workspace) || workspace_bytes < parts_bytes(M, N, parts) || rows_columns(M, N, K, trans_a, trans_b, 1))
    return lego_hip_gemm_fp8_ex(a, b, c, M, N, K, trans_a, trans_b, activation, format, stream);
  if (activation != 0 && activation != 1) return kInvalid;
  return ok_or(fp8_parts(format).of(M, N, K, trans_a, trans_b, 1)(a, b, c, M, N, K, activation, launched_parts(parts, M, N, K, trans_a, trans_b, LEGO_GEMM_BK_8BIT), static_cast<float*>(workspace), as_stream(stream)));
}

// What is used for operands of one layout, shallow products that gain from parts among them; the kernels for few rows and for any shape take
// some and need no room.
int lego_hip_gemm_layout_workspace_bytes(int M, int N, int K, int trans_a, int trans_b, int element_bytes, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || K <= 0 || (element_bytes != 1 && element_bytes != 2)) return kInvalid;
  const int chunk = 16 / element_bytes;
  *bytes = 0;
  if (N % chunk == 0 && K % chunk == 0 && rows_columns(M, N, K, trans_a, trans_b, element_bytes)) return 0;
  const bool ragged = N % chunk || (trans_a ? M : K) % chunk || (trans_b && K % chunk);
  if (ragged && direct_gains(M, N, K, trans_a, trans_b, chunk, element_bytes)) return 0;
  if (element_bytes == 1 && ragged) return lego_hip_gemm_fp8_padded_bytes(M, N, K, trans_a, trans_b, bytes);
  if (element_bytes == 1) *bytes = parts_bytes(M, N, splitk_parts(M, N, K, LEGO_GEMM_BK_8BIT));
  else *bytes = room_16bit(M, N, K, [](int m, int n, int k) { return splitk_parts(m, n, k, LEGO_GEMM_BK); });
  return 0;
}

// Whether a product whose rows are not whole 16-byte chunks gains from copies that are; room for these and for the sums of their product.
int lego_hip_gemm_fp8_padded_bytes(int M, int N, int K, int trans_a, int trans_b, unsigned long long* bytes)
{
  if (bytes == nullptr || M <= 0 || N <= 0 || K <= 0) return kInvalid;
  const bool tiled = N % 16 == 0 && (trans_a ? M % 16 == 0 : K % 16 == 0) && (!trans_b || K % 16 == 0);
  if (tiled || !copies_gain_8bit(M, N, K)) { *bytes = 0; return 0; }
  const int Mp = trans_a ? round_up(M, 16) : M, Nr = round_up(N, 16), Kr = round_up(K, 16);
  *bytes = padded_bytes(M, N, K, 16, 1) + parts_bytes(Mp, Nr, splitk_parts(Mp, Nr, Kr, LEGO_GEMM_BK_8BIT));
  return 0;
}

int lego_hip_gemm_fp8_padded(const void* a, const void* b, void* c, int M, int N, int K, int trans_a, int trans_b,
                             int activation, int format, void* workspace, unsigned long long workspace_bytes, void* stream)
{
  unsigned long long need = 0;
  if ((format != 0 && format != 1) || lego_hip_gemm_fp8_padded_bytes(M, N, K, trans_a, trans_b, &need) != 0) return kInvalid;
  const auto whole = [&](const void* aa, const void* bb, void* cc, int m, int n, int k) {
    return lego_hip_gemm_fp8_ex(aa, bb, cc, m, n, k, trans_a, trans_b, activation, format, stream);
  };
  if (need == 0 || !usable(workspace) || workspace_bytes < need) return whole(a, b, c, M, N, K);
  if (a == nullptr || b == nullptr || c == nullptr || (activation != 0 && activation != 1)) return kInvalid;
  if (reinterpret_cast<uintptr_t>(c) & 1u) return kInvalid;
  return on_padded_copies(16, 1, a, b, c, M, N, K, trans_a, trans_b, workspace, stream,
                          [&](const void* aa, const void* bb, void* cc, int m, int n, int k, void* sums) {
    const int parts = splitk_parts(m, n, k, LEGO_GEMM_BK_8BIT);
    if (parts < 2 || rows_columns(m, n, k, trans_a, trans_b, 1)) return whole(aa, bb, cc, m, n, k);
    return ok_or(fp8_parts(format).of(m, n, k, trans_a, trans_b, 1)(aa, bb, cc, m, n, k, activation, launched_parts(parts, m, n, k, trans_a, trans_b, LEGO_GEMM_BK_8BIT), static_cast<float*>(sums), as_stream(stream)));
  });
}

int lego_hip_gemm_f16_variant(const void* a, const void* b, void* c, int M, int N, int K, int variant, void* stream)
{
  if (!usable(a) || !usable(b) || !usable(c) || M <= 0 || N <= 0 || K <= 0 || N % 8 || K % 8) return kInvalid;
  if (variant == 0) return ok_or(lego_gemm_f16_nn_launch(a, b, c, M, N, K, 0, as_stream(stream)));
  if (variant == 1) return ok_or(lego_gemm_f16_nn_m32_launch(a, b, c, M, N, K, 0, as_stream(stream)));
  if (variant == 2) return ok_or(lego_gemm_f16_nn_w2x4_launch(a, b, c, M, N, K, 0, as_stream(stream)));
  if (variant == 3) return ok_or(lego_gemm_f16_nn_stamps_launch(a, b, c, M, N, K, 0, as_stream(stream)));
  return kInvalid;
}

int lego_hip_gemm_f16_act(const void* a, const void* b, void* c, int M, int N, int K, int activation, void* stream)
{
  return lego_hip_gemm_f16_ex(a, b, c, M, N, K, 0, 0, activation, stream);
}

int lego_hip_gemm_f16(const void* a, const void* b, void* c, int M, int N, int K, void* stream)
{
  return lego_hip_gemm_f16_ex(a, b, c, M, N, K, 0, 0, 0, stream);
}

namespace {
int stencil(const float* in, float* out, const float* c, int n, int radius, int kind, int bricks, int keep, void* stream)
{
  if (!usable(in) || !usable(out) || c == nullptr || in == out) return kInvalid;
  if (n <= 0 || n % LEGO_STENCIL_BRICK || n > 1024 || radius < 1 || radius > (kind == 1 ? LEGO_STENCIL_STAR_MAX_RADIUS : LEGO_STENCIL_MAX_RADIUS) || 2 * radius >= n)
    return kInvalid;
  return ok_or(lego_stencil_f32_launch(in, out, c, n, radius, kind, bricks ? 1 : 0, keep, as_stream(stream)));
}
}  // namespace

int lego_hip_stencil_f3d_f32(const float* in, float* out, const float* c, int n, int radius, int bricks, void* stream)
{
  return stencil(in, out, c, n, radius, 0, bricks, 1, stream);
}

int lego_hip_stencil_laplacian_f32(const float* in, float* out, const float* c, int n, int radius, int bricks,
                                   void* stream)
{
  return stencil(in, out, c, n, radius, 1, bricks, 1, stream);
}

int lego_hip_stencil_f3d_f32_zeros(const float* in, float* out, const float* c, int n, int radius, int bricks, void* stream)
{
  return stencil(in, out, c, n, radius, 0, bricks, 0, stream);
}

int lego_hip_stencil_laplacian_f32_zeros(const float* in, float* out, const float* c, int n, int radius, int bricks,
                                         void* stream)
{
  return stencil(in, out, c, n, radius, 1, bricks, 0, stream);
}

int lego_hip_stencil_f32_plan(int n, int radius, int star, int bricks, int* plan2)
{
  if (plan2 == nullptr || n <= 0 || n % LEGO_STENCIL_BRICK || n > 1024 || radius < 1 || 2 * radius >= n ||
      radius > (star ? LEGO_STENCIL_STAR_MAX_RADIUS : LEGO_STENCIL_MAX_RADIUS))
    return kInvalid;
  return ok_or(lego_stencil_f32_plan(n, radius, star ? 1 : 0, bricks ? 1 : 0, plan2));
}

int lego_hip_lud_f32(float* m, int n, void* stream)
{
  if (!usable(m)) return kInvalid;
  if (n <= 0 || n % LEGO_LUD_BLOCK || n > 32768) return kInvalid;
  return ok_or(lego_lud_f32_launch(m, n, as_stream(stream)));
}

int lego_hip_lud_f32_plan(int n, int* records, int capacity, int* count)
{
  if (!count || capacity < 0 || (capacity > 0 && !records)) return kInvalid;
  if (n <= 0 || n % LEGO_LUD_BLOCK || n > 32768) return kInvalid;
  return ok_or(lego_lud_f32_plan(n, records, capacity, count));
}

int lego_hip_nw_i32(const int* reference, int* matrix, int n, int penalty, void* stream)
{
  if (!usable(reference) || !usable(matrix)) return kInvalid;
  if (n <= 0 || n % LEGO_NW_TILE || n > 32768) return kInvalid;
  // one workgroup needs no room for handing columns over; a single tile (n = 64) is one launch of the tile kernel, which
  // has no ring to fill and drain: 5.8 us against 8.8
  if (n > LEGO_NW_TILE && lego_nw_i32_strips_words(n) == 0)
    return ok_or(lego_nw_i32_strips_launch(reference, matrix, n, penalty, nullptr, as_stream(stream)));
  return ok_or(lego_nw_i32_launch(reference, matrix, n, penalty, as_stream(stream)));
}

int lego_hip_nw_i32_workspace_bytes(int n, unsigned long long* bytes)
{
  if (bytes == nullptr || n <= 0 || n % LEGO_NW_TILE || n > 32768) return kInvalid;
  *bytes = 8 * lego_nw_i32_strips_words(n);
  return 0;
}

int lego_hip_nw_i32_ws(const int* reference, int* matrix, int n, int penalty, void* workspace, unsigned long long workspace_bytes,
                       void* stream)
{
  unsigned long long need = 0;
  if (!usable(reference) || !usable(matrix) || lego_hip_nw_i32_workspace_bytes(n, &need) != 0) return kInvalid;
  if (need == 0 || !usable(workspace) || workspace_bytes < need) return lego_hip_nw_i32(reference, matrix, n, penalty, stream);
  return ok_or(lego_nw_i32_strips_launch(reference, matrix, n, penalty, static_cast<unsigned long long*>(workspace), as_stream(stream)));
}

namespace {
// Time of a grouped launch: list scheduling of its workgroups, in launch order, on `slots` workgroups
// that run at once (a workgroup goes to the slot that frees up first).  The launch is a sequence of
// batches of count[i] workgroups that take cost[i] each.  The slot loads are kept as a sorted list of
// (load, how many slots) levels, so a batch of equal workgroups costs a few steps.
double grouped_makespan(const long* count, const double* cost, int batches, long slots)
{
  struct Level { double load; long count; };
  Level lv[8 * LEGO_GROUPED_MAX_GROUPS + 8];
  int n = 1;
  lv[0] = {0.0, slots};
  for (int g = 0; g < batches; ++g) {
    long left = count[g];
    const double d = cost[g];
    while (left > 0) {
      // the least loaded level takes workgroups, one per slot; its slots move up by d
      const long take = left < lv[0].count ? left : lv[0].count;
      const double moved = lv[0].load + d;
      lv[0].count -= take;
      left -= take;
      if (lv[0].count == 0) {
        for (int i = 1; i < n; ++i) lv[i - 1] = lv[i];
        --n;
      }
      // insert (moved, take) keeping the list sorted; merge equal loads
      int pos = 0;
      while (pos < n && lv[pos].load < moved) ++pos;
      if (pos < n && lv[pos].load == moved) {
        lv[pos].count += take;
      } else if (n < static_cast<int>(sizeof(lv) / sizeof(lv[0]))) {
        for (int i = n; i > pos; --i) lv[i] = lv[i - 1];
        lv[pos] = {moved, take};
        ++n;
      } else {
        lv[n - 1].count += take;        // out of levels (never with <= 64 groups): fold into the top one
        if (lv[n - 1].load < moved) lv[n - 1].load = moved;
      }
    }
  }
  return lv[n - 1].load;
}

// What a grouped call launches: the kernel on 256 x 256 tiles with the last `split` tiles of its launch
// order as two 128 x 256 halves each (kind 0), or the kernel on 128 x 128 tiles, two workgroups per CU (kind 1) or one (kind 2).
struct GroupedPlan {
  int kind, tiles, split;
  double time;      // the estimate that chose it, in the units below
  int limit;        // k-tiles of a unit where the call is shorter with deep problems in parts, given room for their sums (0: nowhere), ...
  int sums;         // ... and the tiles of those
};

// Costs in units of one k-tile step of a 256 x 256 tile that has its CU to itself (about 1.8 us for
// fp16), measured on MI355X: a tile pays a start-up and an epilogue on top of its steps (31.4 us for
// 16 steps); a 128 x 256 half-tile takes 19.2 us for 16 steps; a 128 x 128 tile sharing its CU with
// another one takes 0.66 of a whole tile of the same depth.  One on four buffers, alone on its CU, takes 0.38 of a step
// per k-tile and two steps beside them: the choice between the two so estimated takes 1.0005 times the better one over 72
// drawn calls of 1 to 16 problems (us, two workgroups per CU / one: 112 x 120 x 2816 and 128 x 184 x 512 30.5 / 19.7; 16 problems, 546 tiles of up to
// 57 k-tiles, 68 / 45; nine of 565 tiles 71 / 52; 13 of 1056 tiles, deep ones among them in every round, 80 / 91; 14 of 762 tiles of up to 12 k-tiles 25.6 / 28.0).
// In parts along K: the same per k-tile and a little more for the sums that a workgroup stores, the second launch, and for each tile of sums its
// way to memory and back; parts where that is less than 0.9 of the best whole launch.  Over 36 drawn calls of 1 to 16 problems this takes 0.94 of
// the whole launches' time, the best of eight limits for each call 0.93, and over 60 others 0.92 (us, whole / parts: five problems of 43 to 8 k-tiles 34.1 / 20.1, six
// 42 / 23, thirteen of 13 GFLOP 48 / 28; without the margin thirteen of 34.7 took 37.7).
constexpr double kPartOverhead = 2.3, kPartLaunch = 2.2, kPartSum = 0.035, kPartGain = 0.9;
constexpr int kPartTiles = 1024;       // partial sums of a call, 64 KiB each
constexpr double kTileOverhead = 1.6, kHalfStep = 0.58, kHalfOverhead = 1.5, kSmallCost = 0.66, kDeepStep = 0.38, kDeepOverhead = 2.0;
// Problems per call.  A launch carries its pointers and sizes as kernel arguments, LEGO_GROUPED_MAX_GROUPS problems
// at most; a call with more is enqueued as several launches (below).
constexpr int kGroupedMaxProblems = 1 << 20;

GroupedPlan grouped_plan_uncached(const int* sizes3, int groups)
{
  GroupedPlan plan;
  int order[LEGO_GROUPED_MAX_GROUPS];       // problems in launch order: decreasing depth, stable
  for (int g = 0; g < groups; ++g) order[g] = g;
  for (int i = 1; i < groups; ++i) {
    const int o = order[i];
    int j = i;
    while (j > 0 && sizes3[3 * order[j - 1] + 2] < sizes3[3 * o + 2]) { order[j] = order[j - 1]; --j; }
    order[j] = o;
  }
  long big[LEGO_GROUPED_MAX_GROUPS], small[LEGO_GROUPED_MAX_GROUPS];
  double depth[LEGO_GROUPED_MAX_GROUPS], small_cost[LEGO_GROUPED_MAX_GROUPS], deep_cost[LEGO_GROUPED_MAX_GROUPS];
  long total = 0;
  bool deep = true;
  for (int s = 0; s < groups; ++s) {
    const int g = order[s];
    const int m = sizes3[3 * g], n = sizes3[3 * g + 1];
    big[s] = static_cast<long>((m + 255) / 256) * ((n + 255) / 256);
    small[s] = static_cast<long>((m + 127) / 128) * ((n + 127) / 128);
    depth[s] = (sizes3[3 * g + 2] + LEGO_GEMM_BK - 1) / LEGO_GEMM_BK;
    small_cost[s] = kSmallCost * (depth[s] + kTileOverhead);
    deep_cost[s] = kDeepStep * depth[s] + kDeepOverhead;
    deep = deep && deep_offsets(m, n, sizes3[3 * g + 2], 2);
    total += big[s];
  }
  const long cus = 256;                 // MI355X
  // 256 x 256 tiles, the last `split` of them as halves: the best split among multiples of 16 tiles
  // up to two rounds of the CUs
  double best = 0.0;
  long best_split = 0;
  const long max_split = total < 2 * cus ? total : 2 * cus;
  for (long split = 0; split <= max_split; split += 16) {
    long count[2 * LEGO_GROUPED_MAX_GROUPS];
    double cost[2 * LEGO_GROUPED_MAX_GROUPS];
    int nb = 0;
    long whole_left = total - split;
    for (int s = 0; s < groups; ++s) {
      const long w = big[s] < whole_left ? big[s] : whole_left;
      whole_left -= w;
      if (w > 0) { count[nb] = w; cost[nb++] = depth[s] + kTileOverhead; }
    }
    whole_left = total - split;
    for (int s = 0; s < groups; ++s) {
      const long w = big[s] < whole_left ? big[s] : whole_left;
      whole_left -= w;
      if (big[s] > w) { count[nb] = 2 * (big[s] - w); cost[nb++] = kHalfStep * depth[s] + kHalfOverhead; }
    }
    const double t = grouped_makespan(count, cost, nb, cus);
    // equal estimates: the larger split (more, shorter workgroups in the last round measured faster)
    if (split == 0 || t <= best) { best = t; best_split = split; }
  }
  const double t_small = grouped_makespan(small, small_cost, groups, 2 * cus);
  const double t_deep = deep ? grouped_makespan(small, deep_cost, groups, cus) : t_small;
  plan.kind = t_deep < t_small && t_deep < best ? 2 : t_small < best ? 1 : 0;
  plan.tiles = static_cast<int>(total);
  plan.split = plan.kind == 0 ? static_cast<int>(best_split) : 0;
  plan.time = plan.kind == 2 ? t_deep : plan.kind == 1 ? t_small : best;
  plan.limit = plan.sums = 0;
  double least = kPartGain * plan.time;
  for (const int limit : {4, 6, 8, 12, 16, 24, 32, 48}) {
    if (!deep || limit >= depth[0]) break;      // the deepest problem is the first
    long count[LEGO_GROUPED_MAX_GROUPS], sums = 0;
    double length[LEGO_GROUPED_MAX_GROUPS], cost[LEGO_GROUPED_MAX_GROUPS];
    for (int s = 0; s < groups; ++s) {
      const long d = static_cast<long>(depth[s]), parts = (d + limit - 1) / limit, per = (d + parts - 1) / parts, used = (d + per - 1) / per;
      if (used > 1) sums += used * small[s];
      const double t = kDeepStep * per + (used > 1 ? kPartOverhead : kDeepOverhead);
      int j = s;
      while (j > 0 && length[j - 1] < per) { length[j] = length[j - 1]; cost[j] = cost[j - 1]; count[j] = count[j - 1]; --j; }
      length[j] = per; cost[j] = t; count[j] = used * small[s];
    }
    if (sums > kPartTiles) continue;
    const double t = grouped_makespan(count, cost, groups, cus) + kPartLaunch + kPartSum * sums;
    if (t < least) { least = t; plan.limit = limit; plan.sums = static_cast<int>(sums); }
  }
  return plan;
}

// The plan is a few hundred list-scheduling steps per candidate split, tens of microseconds of host time in front
// of a launch of about a hundred: a serving loop calls with the same sizes again and again, so the last few plans
// are kept, keyed by the sizes themselves.
GroupedPlan grouped_plan(const int* sizes3, int groups)
{
  struct Kept { int groups; int sizes[3 * LEGO_GROUPED_MAX_GROUPS]; GroupedPlan plan; };
  constexpr int kKept = 8;
  static Kept kept[kKept];
  static int next = 0;
  static std::mutex kept_mutex;
  const size_t bytes = sizeof(int) * 3 * static_cast<size_t>(groups);
  {
    std::lock_guard<std::mutex> hold(kept_mutex);
    for (int i = 0; i < kKept; ++i)
      if (kept[i].groups == groups && memcmp(kept[i].sizes, sizes3, bytes) == 0) return kept[i].plan;
  }
  const GroupedPlan plan = grouped_plan_uncached(sizes3, groups);
  std::lock_guard<std::mutex> hold(kept_mutex);
  Kept& slot = kept[next];
  next = (next + 1) % kKept;
  slot.groups = groups;
  memcpy(slot.sizes, sizes3, bytes);
  slot.plan = plan;
  return plan;
}

// 0: every problem fits the tiled kernels (one launch); 2: the arguments are valid but some problem needs
// the kernel for any shape (N or K not in whole 16-byte chunks, a base that is not 16-byte aligned);
// kInvalid otherwise
int grouped_check(const void* const* a, const void* const* b, void* const* c, const int* sizes3, int groups)
{
  if (a == nullptr || b == nullptr || c == nullptr || sizes3 == nullptr) return kInvalid;
  if (groups <= 0 || groups > kGroupedMaxProblems) return kInvalid;
  int verdict = 0;
  for (int g = 0; g < groups; ++g) {
    const int m = sizes3[3 * g], n = sizes3[3 * g + 1], k = sizes3[3 * g + 2];
    if (a[g] == nullptr || b[g] == nullptr || c[g] == nullptr || m <= 0 || n <= 0 || k <= 0) return kInvalid;
    if ((reinterpret_cast<uintptr_t>(a[g]) | reinterpret_cast<uintptr_t>(b[g]) | reinterpret_cast<uintptr_t>(c[g])) & 1u)
      return kInvalid;
    if (!usable(a[g]) || !usable(b[g]) || !usable(c[g]) || n % 8 || k % 8) verdict = 2;    // M may be anything
  }
  return verdict;
}

// A grouped call with a problem that the one-launch kernels do not take: one launch per problem on the
// same stream, each through the plain GEMM's dispatch (the reference walks its problems in one kernel,
// grouped_gemm.py:61-116, but takes whole tiles only).
int grouped_one_by_one(const void* const* a, const void* const* b, void* const* c, const int* sizes3, int groups,
                       void* stream)
{
  for (int g = 0; g < groups; ++g) {
    const int err = lego_hip_gemm_f16_ex(a[g], b[g], c[g], sizes3[3 * g], sizes3[3 * g + 1], sizes3[3 * g + 2], 0, 0, 0, stream);
    if (err != 0) return err;
  }
  return 0;
}
}  // namespace

namespace {
// More problems than one launch carries (the reference's host function takes any number: its tables live in
// device memory, grouped_gemm.py:120-162): all problems in order of decreasing depth (stable), cut into runs of
// LEGO_GROUPED_MAX_GROUPS, one launch per run on the same stream -- so every launch still starts with its longest
// tiles, and only the last launches hold the shallow problems whose tail rounds are short.
int grouped_in_runs(const void* const* a, const void* const* b, void* const* c, const int* sizes3, int groups, void* stream)
{
  std::vector<int> order(static_cast<size_t>(groups));
  for (int g = 0; g < groups; ++g) order[static_cast<size_t>(g)] = g;
  std::stable_sort(order.begin(), order.end(), [sizes3](int p, int q) { return sizes3[3 * p + 2] > sizes3[3 * q + 2]; });
  const void* ra[LEGO_GROUPED_MAX_GROUPS];
  const void* rb[LEGO_GROUPED_MAX_GROUPS];
  void* rc[LEGO_GROUPED_MAX_GROUPS];
  int rs[3 * LEGO_GROUPED_MAX_GROUPS];
  for (int first = 0; first < groups; first += LEGO_GROUPED_MAX_GROUPS) {
    const int count = groups - first < LEGO_GROUPED_MAX_GROUPS ? groups - first : LEGO_GROUPED_MAX_GROUPS;
    for (int i = 0; i < count; ++i) {
      const int g = order[static_cast<size_t>(first + i)];
      ra[i] = a[g]; rb[i] = b[g]; rc[i] = c[g];
      rs[3 * i] = sizes3[3 * g]; rs[3 * i + 1] = sizes3[3 * g + 1]; rs[3 * i + 2] = sizes3[3 * g + 2];
    }
    const int err = lego_hip_grouped_gemm_f16(ra, rb, rc, rs, count, stream);
    if (err != 0) return err;
  }
  return 0;
}
}  // namespace

int lego_hip_grouped_gemm_f16(const void* const* a, const void* const* b, void* const* c,
                              const int* sizes3, int groups, void* stream)
{
  const int checked = grouped_check(a, b, c, sizes3, groups);
  if (checked == 2) return grouped_one_by_one(a, b, c, sizes3, groups, stream);
  if (checked != 0) return kInvalid;
  if (groups > LEGO_GROUPED_MAX_GROUPS) return grouped_in_runs(a, b, c, sizes3, groups, stream);
  // One launch: on 256 x 256 tiles (one workgroup per CU), the last tiles of the launch order split
  // into halves when whole tiles would leave the last round mostly empty, or on 128 x 128 tiles (four
  // times as many workgroups of a quarter of the work, two per CU) when the big ones leave most CUs
  // idle; whichever the estimate finishes first.  Problems are launched in order of decreasing
  // depth, so the longest tiles start first.  (Splitting the problems over both tile sizes in two
  // launches was measured and never beat the better single launch.)
  const GroupedPlan plan = grouped_plan(sizes3, groups);
  if (plan.kind == 2) return ok_or(lego_grouped_gemm_f16_t128x128_deep_launch(a, b, c, sizes3, groups, as_stream(stream)));
  if (plan.kind == 1) return ok_or(lego_grouped_gemm_f16_t128x128_launch(a, b, c, sizes3, groups, as_stream(stream)));
  if (plan.split == 0) return ok_or(lego_grouped_gemm_f16_launch(a, b, c, sizes3, groups, as_stream(stream)));
  return ok_or(lego_grouped_gemm_f16_split_launch(a, b, c, sizes3, groups, plan.split, as_stream(stream)));
}

// Ragged problems that a single product splits along K: in the grouped launch they are chains of whole depth, apart each is some four
// launches more.  Apart, then, where the launch without them is estimated shorter by more than 20 steps for each and twice what it is of a step of
// the whole chip.  Us with what the host adds, together / apart: 64 x 64 x 4095 beside one of 64^3 31 / 28, beside two 32 / 32 (beside fifteen, which
// the estimate cannot tell, 65 / 74), 512 x 512 x 4095 beside two of 512^3 36 / 34, which stay together, and beside eight 44 / 53; 64 x 64 x 2577 beside eight of
// 1024^3 44 / 52, four of 64 x 64 x 4095 35 / 66.  Over 90 drawn calls with such problems the rule, and all together, take the better of the two.
int lego_hip_grouped_gemm_f16_apart(const int* sizes3, int groups, int* apart) try
{
  if (sizes3 == nullptr || apart == nullptr || groups <= 0 || groups > kGroupedMaxProblems) return kInvalid;
  std::vector<int> order(static_cast<size_t>(groups));
  for (int g = 0; g < groups; ++g) {
    if (sizes3[3 * g] <= 0 || sizes3[3 * g + 1] <= 0 || sizes3[3 * g + 2] <= 0) return kInvalid;
    order[static_cast<size_t>(g)] = g;
    apart[g] = 0;
  }
  std::stable_sort(order.begin(), order.end(), [sizes3](int p, int q) { return sizes3[3 * p + 2] > sizes3[3 * q + 2]; });
  // what the first launch carries: the deepest problems
  const int count = groups < LEGO_GROUPED_MAX_GROUPS ? groups : LEGO_GROUPED_MAX_GROUPS;
  int all[3 * LEGO_GROUPED_MAX_GROUPS], rest[3 * LEGO_GROUPED_MAX_GROUPS], deep[LEGO_GROUPED_MAX_GROUPS], others = 0, deeps = 0;
  double alone = 0.0;
  for (int i = 0; i < count; ++i) {
    const int g = order[static_cast<size_t>(i)], m = sizes3[3 * g], n = sizes3[3 * g + 1], k = sizes3[3 * g + 2];
    const bool ragged = n % 8 || k % 8;
    const int size[3] = {m, ragged ? round_up(n, 8) : n, ragged ? round_up(k, 8) : k};
    memcpy(all + 3 * i, size, sizeof(size));
    if (ragged && k > 31 * LEGO_GEMM_BK) {
      deep[deeps++] = g;
      alone += 20.0 + 2.0 * m * n * k / (256.0 * 256 * 256 * LEGO_GEMM_BK);
    } else {
      memcpy(rest + 3 * others++, size, sizeof(size));
    }
  }
  if (deeps == 0) return 0;
  const double without = others ? grouped_plan(rest, others).time : 0.0;
  if (grouped_plan(all, count).time > without + alone)
    for (int i = 0; i < deeps; ++i) apart[deep[i]] = 1;
  return 0;
} catch (const std::bad_alloc&) {
  return ok_or(hipErrorOutOfMemory);
}

namespace {
// Copies of the ragged problems of a call lie in the workspace together up to this much; what is beyond follows in further runs of the
// same call, copies, launch and way back each, with no problem's own copies cut.  Sixteen products of 4095^3: 1.6 GB at once, 0.5 GB in runs
// of five, whose 1280 tiles are five rounds of the chip.
constexpr unsigned long long kCopyRoom = 512ull << 20;

inline unsigned long long copies_of(const int* size) { return size[1] % 8 || size[2] % 8 ? padded_bytes(size[0], size[1], size[2], 8, 2) : 0ull; }

// `run(problems, count, bytes)` for each run, as the call lists the problems where one run is all, otherwise deepest first.
extern "C++" template <class Run>
int grouped_copy_runs(const int* sizes3, int groups, const Run& run)
{
  unsigned long long total = 0;
  std::vector<int> order(static_cast<size_t>(groups));
  for (int g = 0; g < groups; ++g) {
    order[static_cast<size_t>(g)] = g;
    total += copies_of(sizes3 + 3 * g);
  }
  if (total > kCopyRoom) std::stable_sort(order.begin(), order.end(), [sizes3](int p, int q) { return sizes3[3 * p + 2] > sizes3[3 * q + 2]; });
  for (int first = 0; first < groups;) {
    unsigned long long used = 0;
    int count = 0;
    for (; first + count < groups; ++count) {
      const unsigned long long more = copies_of(sizes3 + 3 * order[static_cast<size_t>(first + count)]);
      if (used != 0 && used + more > kCopyRoom) break;
      used += more;
    }
    const int rc = run(order.data() + first, count, used);
    if (rc != 0) return rc;
    first += count;
  }
  return 0;
}
}  // namespace

// Room for zero-padded copies of the problems whose N or K is no multiple of 8: that of the largest run.
int lego_hip_grouped_gemm_f16_workspace_bytes(const int* sizes3, int groups, unsigned long long* bytes) try
{
  if (sizes3 == nullptr || bytes == nullptr || groups <= 0 || groups > kGroupedMaxProblems) return kInvalid;
  for (int i = 0; i < 3 * groups; ++i)
    if (sizes3[i] <= 0) return kInvalid;
  unsigned long long most = 0;
  grouped_copy_runs(sizes3, groups, [&](const int*, int, unsigned long long used) { most = std::max(most, used); return 0; });
  *bytes = most;
  return 0;
} catch (const std::bad_alloc&) {
  return ok_or(hipErrorOutOfMemory);
}

namespace {
constexpr unsigned long long kSumBytes = 128 * 128 * sizeof(float);
// The launch of a call in parts, its problems on whole chunks: as the plan for their sizes has it.  One launch's problems, in one run of copies.
inline GroupedPlan parts_plan(const int* sizes3, int groups, unsigned long long copies)
{
  GroupedPlan none{};
  if (groups > LEGO_GROUPED_MAX_GROUPS || copies > kCopyRoom) return none;
  int sizes[3 * LEGO_GROUPED_MAX_GROUPS];
  for (int g = 0; g < groups; ++g) {
    const int m = sizes3[3 * g], n = sizes3[3 * g + 1], k = sizes3[3 * g + 2];
    const bool ragged = n % 8 || k % 8;
    const int size[3] = {m, ragged ? round_up(n, 8) : n, ragged ? round_up(k, 8) : k};
    memcpy(sizes + 3 * g, size, sizeof(size));
  }
  return grouped_plan(sizes, groups);
}
inline unsigned long long all_copies(const int* sizes3, int groups)
{
  unsigned long long total = 0;
  for (int g = 0; g < groups; ++g) total += copies_of(sizes3 + 3 * g);
  return total;
}
}  // namespace

int lego_hip_grouped_gemm_f16_room(const int* sizes3, int groups, unsigned long long* bytes, int* limit)
{
  if (limit == nullptr) return kInvalid;
  const int rc = lego_hip_grouped_gemm_f16_workspace_bytes(sizes3, groups, bytes);
  if (rc != 0) return rc;
  const GroupedPlan plan = parts_plan(sizes3, groups, all_copies(sizes3, groups));
  *limit = plan.limit;
  *bytes += plan.sums * kSumBytes;
  return 0;
}

int lego_hip_grouped_gemm_f16_ws(const void* const* a, const void* const* b, void* const* c, const int* sizes3, int groups,
                                 void* workspace, unsigned long long workspace_bytes, void* stream) try
{
  const int checked = grouped_check(a, b, c, sizes3, groups);
  unsigned long long need = 0;
  // the products, their copies in the first `used` bytes of the workspace: with deep ones in parts where there is room for the sums
  const auto products = [&](const void* const* aa, const void* const* bb, void* const* cc, const int* sizes, int count, unsigned long long used) {
    if (count == groups && used <= workspace_bytes && usable(workspace) && grouped_check(aa, bb, cc, sizes, count) == 0) {
      const GroupedPlan plan = parts_plan(sizes, count, used);
      if (plan.limit && workspace_bytes - used >= plan.sums * kSumBytes)
        return ok_or(lego_grouped_gemm_f16_t128x128_deep_parts_launch(aa, bb, cc, sizes, count, plan.limit,
                                                                      reinterpret_cast<float*>(static_cast<uint8_t*>(workspace) + used), as_stream(stream)));
    }
    return lego_hip_grouped_gemm_f16(aa, bb, cc, sizes, count, stream);
  };
  if (checked == 0) return products(a, b, c, sizes3, groups, 0);
  if (checked != 2 || lego_hip_grouped_gemm_f16_workspace_bytes(sizes3, groups, &need) != 0 || need == 0 || workspace_bytes < need || !usable(workspace))
    return lego_hip_grouped_gemm_f16(a, b, c, sizes3, groups, stream);
  std::vector<const void*> aa, bb;
  std::vector<void*> cc;
  std::vector<int> sizes, copied;
  return grouped_copy_runs(sizes3, groups, [&](const int* problems, int count, unsigned long long used) {
    aa.clear(); bb.clear(); cc.clear(); sizes.clear(); copied.clear();
    Copier pads(true, as_stream(stream)), back(false, as_stream(stream));
    uint8_t* at = static_cast<uint8_t*>(workspace);
    for (int i = 0; i < count; ++i) {
      const int g = problems[i], m = sizes3[3 * g], n = sizes3[3 * g + 1], k = sizes3[3 * g + 2];
      const bool ragged = n % 8 || k % 8;
      const int mr = round_up(m, 8), nr = ragged ? round_up(n, 8) : n, kr = ragged ? round_up(k, 8) : k;
      aa.push_back(a[g]); bb.push_back(b[g]); cc.push_back(c[g]);
      sizes.insert(sizes.end(), {m, nr, kr});
      if (!ragged) continue;
      uint8_t *ap = at, *bp = ap + 2 * static_cast<size_t>(mr) * kr, *cp = bp + 2 * static_cast<size_t>(kr) * nr;
      at = cp + 2 * static_cast<size_t>(mr) * nr;
      if (kr != k || !usable(a[g])) { pads.add(a[g], ap, m, k, m, kr, 2); aa[i] = ap; }
      if (kr != k || nr != n || !usable(b[g])) { pads.add(b[g], bp, k, n, kr, nr, 2); bb[i] = bp; }
      if (nr != n || !usable(c[g])) { cc[i] = cp; copied.push_back(i); }
    }
    const hipError_t err = pads.flush();
    if (err != hipSuccess) return ok_or(err);
    const int rc = products(aa.data(), bb.data(), cc.data(), sizes.data(), count, used);
    if (rc != 0) return rc;
    for (const int i : copied) back.add(cc[i], c[problems[i]], sizes[3 * i], sizes3[3 * problems[i] + 1], sizes[3 * i], sizes[3 * i + 1], 2);
    return ok_or(back.flush());
  });
} catch (const std::bad_alloc&) {
  return ok_or(hipErrorOutOfMemory);
}

int lego_hip_rows_f16_plan(int M, int N, int* waves_per_row)
{
  if (waves_per_row == nullptr || M <= 0 || N <= 0 || N % 8 != 0 || N > LEGO_ROWWISE_MAX_N) return kInvalid;
  *waves_per_row = lego_rowwise_f16_wpr(M, N);
  return 0;
}

int lego_hip_gemm_plan(int M, int N, int K, int* plan2)
{
  if (plan2 == nullptr || M <= 0 || N <= 0 || K <= 0) return kInvalid;
  const int choice = gemm_choice(M, N, true, true);
  plan2[0] = choice == 1 ? 128 : 256;
  plan2[1] = choice == 0 ? 16 : 32;
  return 0;
}

int lego_hip_gemm_parts_plan(int M, int N, int K, int element_bytes, int* plan2)
{
  if (plan2 == nullptr || M <= 0 || N <= 0 || K <= 0 || (element_bytes != 1 && element_bytes != 2)) return kInvalid;
  plan2[0] = deep_offsets(M, N, K, element_bytes) ? splitk_parts(M, N, K, element_bytes == 1 ? LEGO_GEMM_BK_8BIT : LEGO_GEMM_BK) : 1;
  plan2[1] = plan2[0] > 1 || deep_tiles(M, N, K, element_bytes) ? 4 : 2;
  return 0;
}

int lego_hip_gemm_rows_plan(int M, int N, int K, int trans_a, int trans_b, int element_bytes, int* columns)
{
  if (columns == nullptr || M <= 0 || N <= 0 || K <= 0 || (element_bytes != 1 && element_bytes != 2)) return kInvalid;
  *columns = rows_columns(M, N, K, trans_a, trans_b, element_bytes);
  return 0;
}

int lego_hip_grouped_gemm_f16_plan(const int* sizes3, int groups, int* plan3)
{
  if (sizes3 == nullptr || plan3 == nullptr || groups <= 0 || groups > LEGO_GROUPED_MAX_GROUPS) return kInvalid;
  for (int g = 0; g < groups; ++g)
    if (sizes3[3 * g] <= 0 || sizes3[3 * g + 1] <= 0 || sizes3[3 * g + 2] <= 0) return kInvalid;
  const GroupedPlan plan = grouped_plan(sizes3, groups);
  plan3[0] = plan.kind == 0 ? 256 : 128;
  plan3[1] = plan.tiles;
  plan3[2] = plan.split;
  return 0;
}

int lego_hip_grouped_gemm_f16_split(const void* const* a, const void* const* b, void* const* c,
                                    const int* sizes3, int groups, int split_tiles, void* stream)
{
  if (groups > LEGO_GROUPED_MAX_GROUPS || grouped_check(a, b, c, sizes3, groups) != 0) return kInvalid;     // one launch of tiled problems only
  if (split_tiles < 0)
    return ok_or(lego_grouped_gemm_f16_t128x128_launch(a, b, c, sizes3, groups, as_stream(stream)));
  return ok_or(lego_grouped_gemm_f16_split_launch(a, b, c, sizes3, groups, split_tiles, as_stream(stream)));
}

int lego_hip_grouped_gemm_f16_stamps(const void* const* a, const void* const* b, void* const* c,
                                     const int* sizes3, int groups, void* stream)
{
  if (groups > LEGO_GROUPED_MAX_GROUPS || grouped_check(a, b, c, sizes3, groups) != 0) return kInvalid;
  const GroupedPlan plan = grouped_plan(sizes3, groups);
  if (plan.kind != 0) return kInvalid;        // the measurement build exists for the 256 x 256 tiles only
  if (plan.split == 0) return ok_or(lego_grouped_gemm_f16_stamps_launch(a, b, c, sizes3, groups, as_stream(stream)));
  return ok_or(lego_grouped_gemm_f16_stamps_split_launch(a, b, c, sizes3, groups, plan.split, as_stream(stream)));
}

int lego_hip_gemm_stamps_read(unsigned long long* host, int workgroups)
{
  if (host == nullptr) return kInvalid;
  return ok_or(lego_gemm_stamps_read(host, workgroups));
}

int lego_hip_copy16(const void* in, void* out, unsigned long long bytes, void* stream)
{
  if (!usable(in) || !usable(out) || bytes == 0 || bytes % 16) return kInvalid;
  const size_t n = bytes / 16;
  const unsigned grid = static_cast<unsigned>(n / 256 < 256 * 32 ? (n + 255) / 256 : 256 * 32);
  hipLaunchKernelGGL(lego_copy16_kernel, dim3(grid), dim3(256), 0, as_stream(stream),
                     static_cast<const uint4*>(in), static_cast<uint4*>(out), n);
  return ok_or(hipGetLastError());
}

int lego_hip_copy16_stream(const void* in, void* out, unsigned long long bytes, void* stream)
{
  if (!usable(in) || !usable(out) || bytes == 0 || bytes % 16384 || bytes / 16384 > 0x7fffffffull) return kInvalid;
  hipLaunchKernelGGL(lego_copy16_stream_kernel, dim3(static_cast<unsigned>(bytes / 16384)), dim3(256), 0,
                     as_stream(stream), static_cast<const u32x4*>(in), static_cast<u32x4*>(out));
  return ok_or(hipGetLastError());
}

int lego_hip_hbm_probe(const void* in, void* out, unsigned long long bytes, int mode, int vectors_per_lane, void* stream)
{
  if (!usable(in) || !usable(out) || in == out) return kInvalid;
  if (mode < 0 || mode > 2 || (vectors_per_lane != 1 && vectors_per_lane != 4)) return kInvalid;
  const unsigned long long chunk = 4096ull * vectors_per_lane;
  if (bytes == 0 || bytes % chunk || bytes / chunk > 0x7fffffffull) return kInvalid;
  const dim3 grid(static_cast<unsigned>(bytes / chunk)), block(256);
  const u32x4* src = static_cast<const u32x4*>(in);
  u32x4* dst = static_cast<u32x4*>(out);
  hipStream_t s = as_stream(stream);
  if (vectors_per_lane == 1) {
    if (mode == 0) hipLaunchKernelGGL(lego_probe_read_kernel<1>, grid, block, 0, s, src, dst);
    else if (mode == 1) hipLaunchKernelGGL(lego_probe_write_kernel<1>, grid, block, 0, s, dst);
    else hipLaunchKernelGGL(lego_probe_copy_kernel<1>, grid, block, 0, s, src, dst);
  } else {
    if (mode == 0) hipLaunchKernelGGL(lego_probe_read_kernel<4>, grid, block, 0, s, src, dst);
    else if (mode == 1) hipLaunchKernelGGL(lego_probe_write_kernel<4>, grid, block, 0, s, dst);
    else hipLaunchKernelGGL(lego_probe_copy_kernel<4>, grid, block, 0, s, src, dst);
  }
  return ok_or(hipGetLastError());
}

int lego_hip_mfma_probe(const void* operands, float* sink, int shape, int iters, int workgroups, void* stream)
{
  if (!usable(operands) || !usable(sink) || shape < 0 || shape > 7 || iters <= 0 || workgroups <= 0) return kInvalid;
  const dim3 grid(static_cast<unsigned>(workgroups)), block(256);
  const probe_half8* src = static_cast<const probe_half8*>(operands);
  hipStream_t s = as_stream(stream);
  if (shape == 5) hipLaunchKernelGGL(lego_mfma_probe_8bit_kernel<1>, grid, block, 0, s, static_cast<const probe_int8*>(operands), sink, static_cast<unsigned>(iters));
  else if (shape == 6) hipLaunchKernelGGL(lego_mfma_probe_8bit_kernel<0>, grid, block, 0, s, static_cast<const probe_int8*>(operands), sink, static_cast<unsigned>(iters));
  else if (shape == 7) hipLaunchKernelGGL(lego_mfma_probe_8bit_16x16_kernel, grid, block, 0, s, static_cast<const probe_int8*>(operands), sink, static_cast<unsigned>(iters));
  else if (shape == 3) hipLaunchKernelGGL(lego_mfma_probe2_kernel<3>, grid, dim3(512), 0, s, src, sink, static_cast<unsigned>(iters));
  else if (shape == 4) hipLaunchKernelGGL(lego_mfma_probe2_kernel<4>, grid, dim3(512), 0, s, src, sink, static_cast<unsigned>(iters));
  else if (shape == 0) hipLaunchKernelGGL(lego_mfma_probe_kernel<0>, grid, block, 0, s, src, sink, static_cast<unsigned>(iters));
  else if (shape == 1) hipLaunchKernelGGL(lego_mfma_probe_kernel<1>, grid, block, 0, s, src, sink, static_cast<unsigned>(iters));
  else hipLaunchKernelGGL(lego_mfma_probe_kernel<2>, grid, block, 0, s, src, sink, static_cast<unsigned>(iters));
  return ok_or(hipGetLastError());
}

}  // extern "C"
