// The merged projections of the LoRA-adapted layer for gfx950: W' = round(W + s A B) for up to
// kMaxMerge projections in one launch (the reference's _merge, src/tjev/model/lora.py:284-295: A and
// B rounded to the compute dtype, their product accumulated in fp32, one rounding of the sum).
//
// Bound by memory: W is read and W' written once in bf16 (2560 x 8192: 84 MB), the adapters are
// small. A workgroup of 4 waves owns 128 columns and 128 rows: B's columns are rounded into LDS
// once ([column][rank], so a fragment is one 16-byte read), each wave then takes two strips of 16
// rows, the second's inputs loaded while the first is computed. The product is accumulated
// transposed (B^T's fragment as the MFMA's first operand), with the columns of a pair of tiles
// interleaved so that a lane holds 8 consecutive columns of its row: W and W' move as 16-byte
// pieces, 64 contiguous bytes per row and instruction. Measured at the 4B layer (qkv, z, b and a
// of 2560 inputs, rank 64, in one launch): 37 us, 3.4 TB/s, against 134 us for the four GEMMs
// with their copies; out_proj (4096 x 2560) 14 us against 34; 256 rows per workgroup 37 and 16 us.
#include <hip/hip_runtime.h>

#include <string>

#include "../../include/tjev_gdn.h"
#include "gdn_device.h"
#include "gdn_launch.h"

namespace gdn {
namespace {

constexpr int kMaxMerge = TJEV_GDN_MAX_MERGE;
constexpr int kCols = 128, kRows = 128, kThreads = 256;

struct MergeArgs {
  tjev_gdn_merge p[kMaxMerge];
  unsigned first[kMaxMerge];  // the projection's first workgroup
  int n;
};

template <int KS>
__global__ __launch_bounds__(kThreads) void k_lora_merge(MergeArgs M) {
  constexpr int R = 32 * KS, LD = R + 8;
  __shared__ __align__(16) uint16_t sb[kCols * LD];  // B^T, rounded: [column][rank]
  GDN_POISON_LDS(sb);
  int d = 0;
  for (int i = 1; i < M.n; ++i)
    if (blockIdx.x >= M.first[i]) d = i;
  const tjev_gdn_merge P = M.p[d];
  const unsigned id = blockIdx.x - M.first[d], tiles = (unsigned)(P.out + kCols - 1) / kCols;
  const int c0 = (int)(id % tiles) * kCols;
  const long row0 = (long)(id / tiles) * kRows;
  const int tid = threadIdx.x, l = lane(), r = l & 15, g = l >> 4;
  const float* B = P.b;
  auto stage = [&]() {
    for (int idx = tid; idx < R / 2 * (kCols / 4); idx += kThreads) {  // 4 columns of a pair of B's rows
      const int k = 2 * (idx / (kCols / 4)), c = 4 * (idx % (kCols / 4));
      float4 x = make_float4(0.f, 0.f, 0.f, 0.f), y = x;
      if (c0 + c < P.out) {  // out is a multiple of 8
        x = *reinterpret_cast<const float4*>(B + (size_t)k * P.out + c0 + c);
        y = *reinterpret_cast<const float4*>(B + (size_t)(k + 1) * P.out + c0 + c);
      }
      uint32_t* s = reinterpret_cast<uint32_t*>(sb + c * LD + k);
      s[0] = pack2(x.x, y.x);
      s[LD / 2] = pack2(x.y, y.y);
      s[LD] = pack2(x.z, y.z);
      s[3 * LD / 2] = pack2(x.w, y.w);
    }
  };
  // the lane's column within a pair of tiles when it feeds B: tile t covers 8 (r / 4) + 4 t + r % 4
  const uint16_t* bp = sb + (8 * (r >> 2) + (r & 3)) * LD + 8 * g;
  // a strip's inputs, held while the strip before it is computed (the first strip's: while B is
  // staged)
  struct Strip {
    uint4 w[kCols / 32];
    float a[KS][8];
  };
  auto fetch = [&](Strip& x, int it) {
    const long i = row0 + 16 * (4 * it + wave()) + r, row = i < P.in ? i : P.in - 1;
    const uint16_t* w = static_cast<const uint16_t*>(P.w) + (size_t)row * P.out;
#pragma unroll
    for (int p = 0; p < kCols / 32; ++p) {  // columns past the last: the row's first ones (not stored)
      const int c = c0 + 32 * p + 8 * g;
      x.w[p] = *reinterpret_cast<const uint4*>(w + (c < P.out ? c : 0));
    }
#pragma unroll
    for (int s = 0; s < KS; ++s) ld8(P.a + (size_t)row * R + 32 * s + 8 * g, x.a[s]);
  };
  Strip cur, next;
  fetch(cur, 0);
  stage();
  __syncthreads();
#pragma unroll
  for (int it = 0; it < kRows / 64; ++it) {
    const long i0 = row0 + 16 * (4 * it + wave());
    if (i0 >= P.in) break;
    if (it + 1 < kRows / 64) fetch(next, it + 1);
    Frag<P_BF16> fa[KS];
#pragma unroll
    for (int s = 0; s < KS; ++s) fa[s] = make_frag<P_BF16>(cur.a[s]);
    uint16_t* o = static_cast<uint16_t*>(P.merged) + (size_t)(i0 + r) * P.out + c0 + 8 * g;
#pragma unroll
    for (int p = 0; p < kCols / 32; ++p) {
      f32x4 acc[2];
      zero(acc);
#pragma unroll
      for (int s = 0; s < KS; ++s)
#pragma unroll
        for (int t = 0; t < 2; ++t) {
          const bf16x8 fb = *reinterpret_cast<const bf16x8*>(bp + (32 * p + 4 * t) * LD + 32 * s);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb, fa[s].hi, acc[t], 0, 0, 0);
        }
      const uint32_t x[4] = {cur.w[p].x, cur.w[p].y, cur.w[p].z, cur.w[p].w};
      float v[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float we = __uint_as_float(e % 2 ? x[e / 2] & 0xffff0000u : x[e / 2] << 16);
        v[e] = fmaf(P.scale, acc[e / 4][e % 4], we);
      }
      if (i0 + r < P.in && c0 + 32 * p + 8 * g < P.out) st8_io(o + 32 * p, v);
    }
    if (it + 1 < kRows / 64) cur = next;
  }
}

}  // namespace
}  // namespace gdn

extern "C" int tjev_gdn_lora_merge(const tjev_gdn_merge* m, int n, void* stream) {
  auto fail = [](int status, const std::string& msg) { return gdn::fail(status, msg.c_str()); };
  if (!m) return fail(TJEV_GDN_EINVAL, "null tensor argument");
  if (n < 1 || n > gdn::kMaxMerge)
    return fail(TJEV_GDN_EINVAL, "1 to " + std::to_string(gdn::kMaxMerge) + " projections per call");
  gdn::MergeArgs M{};
  M.n = n;
  unsigned long blocks = 0;
  for (int i = 0; i < n; ++i) {
    const tjev_gdn_merge& p = m[i];
    if (p.in <= 0 || p.out <= 0 || p.rank <= 0) return fail(TJEV_GDN_EINVAL, "a projection's sizes must be positive");
    if (p.out % 8 || p.rank % 32 || p.rank > 128 || p.rank != m[0].rank)
      return fail(TJEV_GDN_EUNSUPPORTED, "merged projections: outputs in multiples of 8, one rank of 32, 64, 96 or 128");
    if (!p.w || !p.a || !p.b || !p.merged) return fail(TJEV_GDN_EINVAL, "null tensor argument");
    for (const void* q : {p.w, (const void*)p.a, (const void*)p.b, (const void*)p.merged})
      if (reinterpret_cast<uintptr_t>(q) % 16) return fail(TJEV_GDN_EINVAL, "tensors must be 16-byte aligned");
    M.p[i] = p;
    M.first[i] = (unsigned)blocks;
    blocks += (unsigned long)((p.out + gdn::kCols - 1) / gdn::kCols) * ((p.in + gdn::kRows - 1) / gdn::kRows);
    if (blocks * gdn::kThreads >= (1ul << 32)) return fail(TJEV_GDN_EUNSUPPORTED, "projections too large for one launch");
  }
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid((unsigned)blocks), block(gdn::kThreads);
  switch (m[0].rank / 32) {
    case 1: hipLaunchKernelGGL((gdn::k_lora_merge<1>), grid, block, 0, st, M); break;
    case 2: hipLaunchKernelGGL((gdn::k_lora_merge<2>), grid, block, 0, st, M); break;
    case 3: hipLaunchKernelGGL((gdn::k_lora_merge<3>), grid, block, 0, st, M); break;
    default: hipLaunchKernelGGL((gdn::k_lora_merge<4>), grid, block, 0, st, M); break;
  }
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(TJEV_GDN_EHIP, std::string("HIP launch failed: ") + hipGetErrorString(e));
  return 0;
}
