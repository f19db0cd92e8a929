// A contiguous v_fp8 cache -- k BF16 (B,KV,T,D), E4M3FN codes (B,KV,T,D), fp32 scales (B,KV,T), the
// layout the reference's cache dict holds (specdec/engine/model_self.py:778-800) and its op takes
// (specdec/kernels/ops.py:67-76) -- written into pages for sdv_paged_attention.
//
// One wavefront writes one page (16 tokens of one KV head); pages are numbered in the order of
// their addresses, so a workgroup's four wavefronts write consecutive memory.  K moves in 16-byte
// pieces whose lanes hold consecutive tokens of one 8-dimension chunk, the page's order (the reads
// are 64-byte runs of 16 rows).  V codes are transposed four tokens by four dimensions in
// registers (v_perm_b32).  Bound by its one pass over memory and, at the few MB of a decode step's
// layer, by the launch: 5 x 4097 verify (12/2/128) took eight elementwise launches of 38 us in
// all before and 4.4 us as this one.
#include "sdv_internal.h"

namespace sdv {

struct PackArgs {
  const uint16_t* k;
  const uint8_t* v;
  const float* s;
  uint16_t* k_pages;
  uint8_t* v_pages;
  float* v_scales;
  int32_t* block_table;
  int KV, T, nbps;  // nbps: blocks per sequence
  int n_pages;
};

constexpr int kPackWaves = 4;

template <int D>
__global__ __launch_bounds__(64 * kPackWaves) void pack_kernel(PackArgs a) {
  const int lane = threadIdx.x & (kWave - 1);
  const int page = __builtin_amdgcn_readfirstlane((int)blockIdx.x * kPackWaves + (int)(threadIdx.x / kWave));
  if (page >= a.n_pages) return;
  const int blk = page / a.KV, kvh = page - blk * a.KV, b = blk / a.nbps, j = blk - b * a.nbps;
  const int64_t row0 = ((int64_t)b * a.KV + kvh) * a.T;
  const int t0 = j * kBlock;  // the page's first token; tokens past T - 1 become K 0, code 0, scale 1

  uint4 kw[D / 32];
#pragma unroll
  for (int i = 0; i < D / 32; ++i) {
    const int p = i * kWave + lane, t = t0 + (p & 15);
    kw[i] = load_stream16(a.k + (row0 + min(t, a.T - 1)) * D + (p >> 4) * 8);
    if (t >= a.T) kw[i] = make_uint4(0, 0, 0, 0);
  }
  // lane (dq, tg): dimensions 64h + 4dq .. +3 of tokens 4tg .. +3
  const int tg = lane & 3, dq = lane >> 2;
  uint32_t r[D / 64][4];
#pragma unroll
  for (int h = 0; h < D / 64; ++h)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int t = t0 + 4 * tg + i;
      r[h][i] = *reinterpret_cast<const uint32_t*>(a.v + (row0 + min(t, a.T - 1)) * D + 64 * h + 4 * dq);
      if (t >= a.T) r[h][i] = 0;
    }
  float sc = 1.0f;
  if (lane < kBlock && t0 + lane < a.T) sc = a.s[row0 + t0 + lane];

  uint4* kd = reinterpret_cast<uint4*>(a.k_pages + (int64_t)page * (kBlock * D));
#pragma unroll
  for (int i = 0; i < D / 32; ++i) kd[i * kWave + lane] = kw[i];
  uint8_t* vd = a.v_pages + (int64_t)page * (D * kBlock) + 4 * tg;
#pragma unroll
  for (int h = 0; h < D / 64; ++h) {
    const uint32_t lo01 = __builtin_amdgcn_perm(r[h][1], r[h][0], 0x05010400u), hi01 = __builtin_amdgcn_perm(r[h][1], r[h][0], 0x07030602u);
    const uint32_t lo23 = __builtin_amdgcn_perm(r[h][3], r[h][2], 0x05010400u), hi23 = __builtin_amdgcn_perm(r[h][3], r[h][2], 0x07030602u);
    const uint32_t o[4] = {__builtin_amdgcn_perm(lo23, lo01, 0x05040100u), __builtin_amdgcn_perm(lo23, lo01, 0x07060302u),
                           __builtin_amdgcn_perm(hi23, hi01, 0x05040100u), __builtin_amdgcn_perm(hi23, hi01, 0x07060302u)};
#pragma unroll
    for (int c = 0; c < 4; ++c) *reinterpret_cast<uint32_t*>(vd + (64 * h + 4 * dq + c) * kBlock) = o[c];
  }
  if (lane < kBlock) a.v_scales[(int64_t)page * kBlock + lane] = sc;
  if (lane == 0 && kvh == 0) a.block_table[blk] = blk;
}

}  // namespace sdv

using namespace sdv;

extern "C" int sdv_pack_contiguous(const void* k, const void* v_codes, const float* v_scales, int32_t batch,
                                   int32_t kv_heads, int32_t seq_len, int32_t head_dim, void* k_pages, void* v_pages,
                                   float* page_scales, int32_t* block_table, void* stream) {
  if (!k || !v_codes || !v_scales || !k_pages || !v_pages || !page_scales || !block_table) return SDV_ERR_NULL;
  if (batch <= 0 || kv_heads <= 0 || seq_len <= 0 || seq_len > INT32_MAX - kBlock) return SDV_ERR_SHAPE;
  if (head_dim != 64 && head_dim != 128) return SDV_ERR_UNSUPPORTED;
  const int64_t nbps = (seq_len + kBlock - 1) / kBlock, pages = batch * nbps;
  if (pages > INT32_MAX / kv_heads) return SDV_ERR_SHAPE;
  if (!aligned(k, 16) || !aligned(v_codes, 4) || !aligned(v_scales, 4) || !aligned(k_pages, 16) || !aligned(v_pages, 4) ||
      !aligned(page_scales, 4) || !aligned(block_table, 4))
    return SDV_ERR_ALIGN;
  PackArgs a;
  a.k = static_cast<const uint16_t*>(k);
  a.v = static_cast<const uint8_t*>(v_codes);
  a.s = v_scales;
  a.k_pages = static_cast<uint16_t*>(k_pages);
  a.v_pages = static_cast<uint8_t*>(v_pages);
  a.v_scales = page_scales;
  a.block_table = block_table;
  a.KV = kv_heads;
  a.T = seq_len;
  a.nbps = (int)nbps;
  a.n_pages = (int)(pages * kv_heads);
  const dim3 grid((unsigned)((a.n_pages + (int64_t)kPackWaves - 1) / kPackWaves)), block(kWave * kPackWaves);
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (head_dim == 128)
    hipLaunchKernelGGL(pack_kernel<128>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(pack_kernel<64>, grid, block, 0, st, a);
  return hipGetLastError() == hipSuccess ? SDV_OK : SDV_ERR_HIP;
}
