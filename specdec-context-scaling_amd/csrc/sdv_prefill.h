// Prefill rows: shapes with more query rows than one row-tile group holds (R = G*S > 64: prefill
// and chunked-prefill blocks, model_self.py:471-504, 637-648) in two passes and a launch that
// sums the parts of pass 2.
// Included by sdv_attn.hip, which defines AttnArgs, the synchronisation area and the helpers.
//
//   pass 1  S^T = K Q^T on MFMA, scores rounded to BF16 as the eager path does, offset-causal
//           mask, online (max, sum) per row.  Also dequantizes V once, in the lane order of pass
//           2's MFMA operand.
//   pass 2  recomputes the scores, forms p = bf16(exp(s - M) / L) from pass 1's statistics and
//           accumulates O^T = V_hat^T P^T on MFMA; a third launch sums its parts.
//
// Rows are token-major (row r: token r / G, head r % G), so the rows of a group of 256 see nearly
// the same keys.  Row r sees keys j <= T - S + r / G (the eager mask); a row that sees no key
// outputs 0.
//
// A workgroup of 8 wavefronts takes a row group of 256 rows, 32 per wavefront, and streams stages
// of 64 keys.  All products are v_mfma_f32_32x32x16_bf16: the K page is the A operand as it lies
// in memory (lane (g, m): token m % 16 of block m / 16, dimensions 8g..8g+7 of the 16-dimension
// step), the rows the B operand, and a lane's result (row n, tokens 8j + 4g + i of two blocks) is
// the B operand of the p.V product with those tokens as its k-slots.
//
// Split of the work: the stages of all row groups, in order (layer, KV head, sequence, row
// group), are cut into equal contiguous ranges, one per workgroup, as many workgroups as the
// device holds.  A range covers the end of one row group, whole ones, and the start of another;
// a row group cut by a range's end is a segment per range, whose statistics (pass 1) or fp32
// outputs (pass 2, summed by a third launch) are merged in range order.  Parts of a row group
// per workgroup instead leave the longest part to set the end: 2048 x 8192 has 96 row groups of
// 97 to 128 stages, 42 stages per CU in equal ranges and 64 in parts of two.
//
// Short contexts (kPfShortStages) hold too few stages to share: what they cost is starts, merges and
// launches.  There a workgroup of four wavefronts takes a whole row group of 128 rows, workgroups
// of their own dequantize V beside pass 1, and no parts are left to sum.  80 x 80 of 12/2/128 28.3 ->
// 16.0 us, 300 x 300 32.8 -> 23.1, 28 layers of 512 x 512 95 -> 78; 14/2/64 21.8 -> 12.8, 25.2 -> 16.7,
// 70 -> 53.
//
// What bounds it: both passes keep the VALU and the matrix cores busy together.  A score costs
// about 29 VALU cycles per lane in either pass (two roundings, a multiply, an FMA, v_exp_f32 at
// half rate, and a sum or half a conversion), an MFMA 32 cycles per 16 scores of a lane; per
// unit of 32 keys pass 2 has 512 and about 460 cycles of the two, and the clock falls to 1.8-1.9
// GHz under them.  Per stage of 64 keys and two wavefronts per SIMD: 3,285 cycles in pass 2
// (head_dim 128; MFMA 2,048).  Measured, both passes, of one KV pair's 2048 rows x 8192 keys
// (12/2/128, 14/2/64), 777 x 5000 (14/2/64), 2048 x 2048 and 300 x 5000 (12/2/128), before (16x16
// MFMAs, a row group's rows of one head, parts per row group) and now:
//   233 -> 175, 152 -> 120, 83 -> 50, 77 -> 57, 74 -> 50 us.
// What it took: one wave's LDS operand reads run across the stage barrier (three buffers, waits
// counted by hand: 92 -> 80 us of pass 2's loop), the parts' sum in its own launch (the last part
// to finish summing 470 KB alone held the end up by 29 us), q.k^T, scores and p.V of three units
// in flight (the compiler's own order: 150 us for pass 2).
#pragma once

namespace sdv {

constexpr int kPfWaves = 8;                    // wavefronts per workgroup
constexpr int kPfRows = 32 * kPfWaves;         // rows of a row group
constexpr int kPfShortWaves = 4;               // the same where the contexts are short
constexpr int kPfShortRows = 32 * kPfShortWaves;
constexpr int kPfStage = 64;                   // keys per stage: two units of 32
constexpr int kPfIds = 2048;                   // page ids staged in LDS at a time (a multiple of 4)
constexpr int kPfShortIds = 256;
typedef float f32x16 __attribute__((ext_vector_type(16)));

// One workgroup per CU, two wavefronts per SIMD: pass 2 for head_dim 128 needs the registers (64
// accumulators per lane), and with two workgroups per CU the others were no faster over long
// ranges (pass 1 of 2048 x 8192 76 us either way) and paid twice the starts (2048 x 2048 28.9
// against 22.2 us).
constexpr int kPfWorkgroups = 256;
// Fewest stages of a workgroup's range (150 x 400 of 14/2/64: 30 us with 6, 27 with 4, 24.7 with 3)
constexpr int kPfMinStages = 3;
// Stages that starting a row group costs, about (777 x 5000 of 14/2/64: 61 us with 2, 58 with 4, 56
// with 6; 100 x 16000 of 12/2/128 76, 75, 68)
constexpr int kPfSegStages = 6;

// Most stages of a row group of a short call that has n row groups of 128 rows: few leave ranges with
// few parts to merge, many leave them with more starts.  Short against ranges, us: 12/2/128 16 x 300
// (n = 2, 5 stages) 21.6, 25.8 and x 420 26.3, 25.4; 80 x 510 (8, 8) 29.8, 31.6 and x 540 31.8, 31.2; two
// of 300 x 600 (60, 10) 34.2, 37.9 and x 768 38.4, 39.1.  14/2/64 16 x 540 (2, 9) 21.4, 21.6 and x 600
// 22.8, 21.3; 80 x 660 (10, 11) 24.8, 25.6 and x 720 26.2, 25.3; 300 x 768 (34, 12) 26.5, 26.6 and x 900
// 29.3, 27.1.
__host__ __device__ constexpr int pf_short_stages(int D, int64_t n) {
  return D == 128 ? (n < 4 ? 6 : n < 32 ? 8 : 10) : (n < 4 ? 9 : n < 32 ? 11 : 12);
}
// Workgroups that dequantize V beside pass 1's in a short call, at most.  By the row groups' own
// workgroups after their stages: 11 x 300 of 12/2/128 27.6 -> 21.7 us, 80 x 80 17.3 -> 16.1.
constexpr int kPfShortVWorkgroups = 512;

// Stages of row group i of `rows` rows (of S tokens x G heads) over T keys; at least one, so that a row group
// that sees nothing still has a workgroup to write its zeros.
__host__ __device__ inline int pf_stages(int i, int rows, int S, int G, int T) {
  const int last = min(S - 1, (rows * (i + 1) - 1) / G);
  return max(1, (T - S + last + kPfStage) / kPfStage);
}

// A workgroup's position in the stage order.
struct PfPos {
  int lk, f;         // layer * KV + KV head; sequence * n_row_groups + row group
  int wt;            // its weight: stages and the cost of its start
  int start;         // its first stage in the whole order
};

// Inclusive sum over the lanes of a wavefront (DPP row shifts and row broadcasts).
__device__ __forceinline__ int wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xF, 0xF, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xA, 0xF, false);  // lane 15 of rows 0, 2 to rows 1, 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xC, 0xF, false);  // lane 31 to the upper half
  return v;
}

// Bound of pass 1's sums of exponentials in the fully visible stages, whose exponents are taken
// against an earlier maximum: a stage that would bring a lane's sum to this much goes through the
// online update instead.  The two lanes of a row and its segments (at most 64) can then be added
// without overflow, and a sum that a merge scales by a factor below the smallest normal fp32
// number was worth less than 2^-66 of the row's.  Tested once per stage, for which the first unit's
// products are kept: a test per unit cost pass 1 of head_dim 64 6% (2048 x 16000, both passes 217 us
// without a bound, 225 with a test per unit, 216 with one per stage).  The updates cost 2-5% at scores
// of N(0, 45^2) and N(0, 80^2), where repeating a segment whose sum overflowed cost 40%.
constexpr float kPfSumBound = 0x1p60f;

// bf16(x) as fp32: the pair conversion with a zero low half leaves the value in place.
__device__ __forceinline__ float rnd(float x) { return __builtin_bit_cast(float, pack_bf16x2(0.0f, x)); }

// Pass 2's row groups that several ranges cut: (first workgroup, segments) of every row group,
// at the end of the sync area's partials, and the part slots, in the workspace and then in the
// rest of the partials (which carry nothing from one call to the next).  Segment k of a row group
// belongs to workgroup w0 + k; its slot is dense over the segments (each next one is of the next
// workgroup, the next row group or both) or one of two per workgroup (a range cuts at most the
// row group it begins in and the one it ends in).
constexpr int kPfMaxGroups = 1 << 14;
constexpr size_t kPfDescBytes = (size_t)kPfMaxGroups * 8;
__device__ __forceinline__ int2* pf_desc(const AttnArgs& a) {
  return reinterpret_cast<int2*>(reinterpret_cast<char*>(sync_parts(a)) + kSyncPartBytes - kPfDescBytes);
}
__device__ __forceinline__ float4* pf_slot(const AttnArgs& a, int D, int w0, int k, int rgi) {
  const int id = a.pf_dense ? w0 + k + rgi : 2 * (w0 + k) + (k == 0 ? 1 : 0);
  const int64_t n = kPfRows * D / 4;  // float4s of a slot
  return id < a.pf_slots ? reinterpret_cast<float4*>(a.partial) + id * n
                         : reinterpret_cast<float4*>(sync_parts(a)) + (id - a.pf_slots) * n;
}

// W wavefronts per workgroup: kPfWaves, or kPfShortWaves for short calls, which hold two LDS buffers
// instead of three (a second barrier per stage) so that two workgroups fit a CU: 64 sequences of
// 300 x 300 (12/2/128) 133 -> 93 us, one sequence the same either way.
template <int D, bool OUT, int W>
__global__ __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(2)))
void prefill_kernel(AttnArgs a, int layers) {
  constexpr bool SHORT = W == kPfShortWaves;
  constexpr int NTHR = 64 * W, ROWS = 32 * W;
  constexpr int NB = SHORT ? 2 : 3, IDS = SHORT ? kPfShortIds : kPfIds;
  static_assert(IDS % NTHR == 0 && IDS % 4 == 0, "the threads share the page ids evenly, whole stages of them");
  constexpr int KS = D / 16;        // MFMA steps of one q.k^T product over the head dimension
  constexpr int DT = D / 32;        // 32-dimension output tiles
  constexpr int CU = D / 16;        // 1 KiB chunks of one unit's K (and of its V)
  constexpr int PU = CU / 2;        // chunks per page block
  constexpr int NK = 2 * CU, NC = OUT ? 2 * NK : NK, CPW = NC / W;
  static_assert(CPW * W == NC && NK % W == 0, "the wavefronts share the chunks evenly");
  __shared__ uint4 ring[NB][NC * 64];
  __shared__ int lpb[IDS];
  __shared__ int s_scan[W], s_rest[W], s_pos[2], s_bad;
  const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, g = lane >> 5, n = lane & 31;
  const int nrg = a.pf_nrg, nf = a.B * nrg, LK = layers * a.KV;

  // a row group's weight in the order: its stages and, before them, the cost of its start
  auto weight_of = [&](int f) { return kPfSegStages + pf_stages(f % nrg, ROWS, a.S, a.G, seq_len_of(a, f / nrg)); };

  int window = 0;  // page-id windows staged so far
  if (tid == 0) s_bad = 0;
  // ---- this workgroup's range of stages
  PfPos pos;
  int u = 0, uend = 0;       // current stage and end of the range
  int per1 = 0, per2 = 0;    // stages per workgroup of the two passes (0: whole row groups)
  if (SHORT || (OUT ? a.pf_w2 : a.pf_w1) == 0) {  // a row group per workgroup, the longest (last) ones first
    const int i = (int)blockIdx.x;
    pos.lk = i % LK;
    pos.f = max(nf - 1 - i / LK, 0);
    pos.wt = weight_of(pos.f);
    pos.start = 0;
    u = 0;
    uend = !SHORT || i < nf * LK ? pos.wt : 0;  // the workgroups past them dequantize V
  } else {
    // weights of the row groups of one (layer, KV head): each wavefront scans up to 64 of them in
    // its lanes, more are scanned NTHR at a time by the workgroup; `lo` of this thread's row
    // group, `first` of those scanned so far, and the sum C of all
    const bool few = nf <= kWave;
    const int f0 = few ? lane : tid;
    int v = f0 < nf ? weight_of(f0) : 0, inc = wave_scan(v);
    int lo = inc - v, first = __builtin_amdgcn_readlane(inc, 63), C = first;
    if (!few) {  // workgroup-uniform
      if (lane == 63) s_scan[wave] = inc;
      int rest = 0;
      for (int f = NTHR + tid; f < nf; f += NTHR) rest += weight_of(f);
      rest = wave_scan(rest);
      if (lane == 63) s_rest[wave] = rest;
      __syncthreads();
      first = C = 0;
#pragma unroll
      for (int i = 0; i < W; ++i) {
        lo += i < wave ? s_scan[i] : 0;
        first += s_scan[i];
        C += s_scan[i] + s_rest[i];
      }
    }
    const int U = C * LK;  // the host sends calls of 2^30 stages or more to whole row groups
    per1 = a.pf_w1 ? max((U + a.pf_w1 - 1) / a.pf_w1, a.pf_min1) : 0;
    per2 = max((U + a.pf_w2 - 1) / a.pf_w2, a.pf_min2);
    // Consecutive ranges on one XCD (workgroup i runs on XCD i mod 8), so that an XCD's L2 holds
    // the K and V of few KV heads -- where those of all do not fit its 4 MiB (BF16 K and
    // dequantized V, 4 bytes a dimension).  Where they fit, ranges in launch order are faster
    // (777 x 5000 of 14/2/64 53 against 50 us, 2048 x 2048 of 12/2/128 60 against 57; 1500 x 12000 of
    // 14/2/64, 6 MiB: 133 against 135).
    const int nw = (int)gridDim.x, q8 = nw >> 3, r8 = nw & 7, xcd = (int)blockIdx.x & 7;
    const bool large = (int64_t)LK * a.B * a.max_seq_len * (4 * D) > (4 << 20);
    const int w = large ? xcd * q8 + min(xcd, r8) + ((int)blockIdx.x >> 3) : (int)blockIdx.x;
    const int per = OUT ? per2 : per1;
    u = min(w * per, U);
    uend = min(u + per, U);
    if (u < uend) {  // workgroup-uniform
      pos.lk = u / C;
      const int rem = u - pos.lk * C;
      if (few) {
        pos.f = __popcll(__ballot(lane < nf && inc <= rem));
        pos.start = pos.lk * C + __builtin_amdgcn_readlane(lo, pos.f);
      } else {
        for (int base = 0;;) {
          if (rem >= lo && rem < lo + v) {
            s_pos[0] = base + tid;
            s_pos[1] = lo;
          }
          if (rem < first) break;  // workgroup-uniform
          base += NTHR;
          v = base + tid < nf ? weight_of(base + tid) : 0;
          inc = wave_scan(v);
          __syncthreads();
          if (lane == 63) s_scan[wave] = inc;
          __syncthreads();
          lo = first + inc - v;
#pragma unroll
          for (int i = 0; i < W; ++i) {
            lo += i < wave ? s_scan[i] : 0;
            first += s_scan[i];
          }
        }
        __syncthreads();
        pos.f = __builtin_amdgcn_readfirstlane(s_pos[0]);
        pos.start = pos.lk * C + __builtin_amdgcn_readfirstlane(s_pos[1]);
      }
      pos.wt = __builtin_amdgcn_readfirstlane(weight_of(pos.f));
    }
  }

  constexpr float kUnit = D == 64 ? 0.125f : 1.0f;
  constexpr float kExpCoef = kLog2e * kUnit;
  const float csc = a.inv_sqrt_d;
  // eager score of x in units of kUnit: bf16(bf16(x) * RN(1/sqrt(D))); for head_dim 64 the factor
  // 1/8 is exact and goes into the max and the exponent's coefficient, bit for bit the same
  auto eager = [&](float x) { return D == 64 ? rnd(x) : rnd(rnd(x) * csc); };

  const unsigned kofs = (unsigned)((n >> 4) * (PU * 1024) + g * 256 + (n & 15) * 16);

  while (u < uend) {  // one segment; workgroup-uniform
    const int slo = max(u - pos.start - kPfSegStages, 0), shi = min(uend - pos.start, pos.wt) - kPfSegStages;
    const int next = pos.start + pos.wt;  // the next row group's
    if (slo >= shi) {                     // the range ends within the row group's start
      u = next;
      break;
    }
    const int layer = pos.lk / a.KV, kvh = pos.lk - layer * a.KV, b = pos.f / nrg, rg = pos.f - b * nrg;
    const int zb = layer * a.B + b, grp = zb * a.KV + kvh;
    const int T = seq_len_of(a, b);
    const int nbk = (T + kBlock - 1) / kBlock;
    const int* btrow = a.block_table + (int64_t)b * a.max_blocks;
    const uint16_t* klayer = a.k_pages + layer * a.k_ls + (int64_t)kvh * (kBlock * D);
    const int64_t kpage = (int64_t)a.KV * (kBlock * D);
    // segments of this row group in the two passes: workgroups w0 .. w0 + nseg - 1
    const int s0 = pos.start + kPfSegStages;  // its first stage's place in the order
    const int w0a = per1 ? s0 / per1 : 0, nseg1 = per1 ? (next - 1) / per1 - w0a + 1 : 1;
    const int w0b = per2 ? s0 / per2 : 0, nseg2 = per2 ? (next - 1) / per2 - w0b + 1 : 1;
    const int seg = OUT ? (per2 ? (s0 + slo) / per2 - w0b : 0) : (per1 ? (s0 + slo) / per1 - w0a : 0);

    // this lane's row (of a wavefront without rows, or past the last, row R - 1: loaded, never
    // stored)
    const int r = rg * ROWS + wave * 32 + n;
    const bool rv = r < a.R;
    const int rc = min(r, a.R - 1), si = rc / a.G, hl = rc - si * a.G;
    const int lim = rv ? min(T - 1, T - a.S + si) : -1;
    const int64_t qofs = layer * a.q_ls + b * a.q_sb + (int64_t)(kvh * a.G + hl) * a.q_sh + si * a.q_ss;
    bf16x8 qop[KS];
#pragma unroll
    for (int kk = 0; kk < KS; ++kk) qop[kk] = load_bf16x8(a.q + qofs + kk * 16 + g * 8);
    float2* st = a.stats + ((int64_t)grp * a.R + rc) * a.pf_split;
    // pass 2: the row's statistics of pass 1's segments, lane g's every other one; eight of each
    // lane are loaded ahead
    float2 sv[8];
    if constexpr (OUT) {
#pragma unroll
      for (int i = 0; i < 8; ++i) sv[i] = st[min(2 * i + g, nseg1 - 1)];
    }
    // page ids of a window of the segment's blocks, to LDS
    auto stage_ids = [&](int wlo) {
      const int blk0 = 4 * wlo, nids = 4 * min(IDS / 4, shi - wlo);
      int id[IDS / NTHR];
#pragma unroll
      for (int i = 0; i < IDS / NTHR; ++i) id[i] = i * NTHR + tid < nids ? btrow[max(0, min(blk0 + i * NTHR + tid, nbk - 1))] : -1;
      ++window;
      __syncthreads();  // the ids before these are no longer read
#pragma unroll
      for (int i = 0; i < IDS / NTHR; ++i) {
        const int j = i * NTHR + tid;
        if (j < nids) {
          const bool in = blk0 + j < nbk, ok = in && id[i] >= 0 && id[i] < a.num_blocks;
          if (in && !ok) s_bad = window;
          lpb[j] = ok ? id[i] : -1;
        }
      }
      __syncthreads();
    };
    stage_ids(slo);
    float nml = 0.0f;  // pass 2: -M log2 e - log2 L
    if constexpr (OUT) {
      float m = -INFINITY, l = 0.0f;
      for (int k = 0;; k += 16) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          if (k + 2 * i + g < nseg1) merge_fast(m, l, sv[i].x, sv[i].y);
        if (k + 16 >= nseg1) break;
#pragma unroll
        for (int i = 0; i < 8; ++i) sv[i] = st[min(k + 16 + 2 * i + g, nseg1 - 1)];
      }
      merge_lanes<32>(m, l);
      // p = exp(s - M) / L as one exp2: 2^(s log2 e - M log2 e - log2 L) (v_log_f32 is within
      // 1 ulp; 1 <= L < 2^67, kPfSumBound for each of two lanes and at most 64 segments, so its
      // rounding moves p by less than 5e-6 relative, far below its BF16 step)
      if (l > 0.0f) nml = -m * kLog2e - __builtin_amdgcn_logf(l);
    }
    // the keys every row of the wavefront sees whole, in units (scalar)
    int kmin = rv ? lim : INT_MAX;
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) kmin = min(kmin, __shfl_xor(kmin, off));
    const bool active = rg * ROWS + wave * 32 < a.R;  // the wavefront has rows
    const uint64_t rows = __ballot(rv);                  // the lanes that stand for one
    const int ufull = __builtin_amdgcn_readfirstlane(kmin == INT_MAX ? 0 : (kmin + 1) >> 5);

    f32x16 acc[OUT ? DT : 1];
    float m_run = -INFINITY, l_run = 0.0f;  // pass 1
    if constexpr (OUT) {
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) acc[dt] = (f32x16)0.0f;
    }
    for (int wlo = slo; wlo < shi; wlo += IDS / 4) {  // page-id windows; workgroup-uniform
      const int nit = min(IDS / 4, shi - wlo);           // stages in the window
      if (wlo > slo) stage_ids(wlo);
      const bool bad = __builtin_amdgcn_readfirstlane(s_bad) == window;  // an invalid id in the window
      // units of the window (32 keys): x = 0 .. 2 nit - 1, the first at key 32 * ux0
      const int ux0 = 2 * wlo, nx = 2 * nit;
      const uint4* vh_grp = a.vhat + (int64_t)grp * a.vh_stages * (DT * 128) + lane;
      // The loop multiplies q.k^T one unit ahead of the scores and p.V one unit behind them:
      // buffer s holds K of units 2s + 1, 2s + 2 and V of units 2s - 1, 2s.  Past the window's
      // ends the nearest unit is loaded; its products are not used, or meet p = 0.
      int id[NK / W];   // page ids of the next fetch
      uint4 stg[CPW];   // this wavefront's chunks of the next stage
      auto next_ids = [&](int s) {
#pragma unroll
        for (int j = 0; j < NK / W; ++j) {
          const int c = j * W + wave, x = min(max(2 * s + 1 + c / CU, 0), nx - 1);
          id[j] = lpb[2 * x + (c % CU) / PU];
        }
      };
      auto fetch1 = [&](int s, int j) {  // chunk j * W + wave of stage s
        const int c = j * W + wave;
        if (j < NK / W) {
          const int64_t pg = max(__builtin_amdgcn_readfirstlane(id[j]), 0);
          // cached, unlike the other kernels' K: every row group reads it again (2048 x 8192 of
          // 12/2/128 183 us with the streaming hint, 175 without)
          return *reinterpret_cast<const uint4*>(klayer + pg * kpage + (c % PU) * 512 + lane * 8);
        }
        const int cc = c - NK, x = min(max(2 * s - 1 + cc / CU, 0), nx - 1);
        const int blk = min(2 * (ux0 + x) + (cc % CU) / PU, 2 * a.vh_stages - 1);
        return vh_grp[(int64_t)blk * (DT * 64) + (cc % PU) * 64];
      };
      auto stash1 = [&](uint4* buf, int j) { buf[(j * W + wave) * 64 + lane] = stg[j]; };
      auto publish = [&]() {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
      };
      // The wavefront's iterations: those of fully visible stages, then those that need the mask
      // (pass 1: the first stage too, whose maximum the fast ones start from).
      const int nfast = !active || bad ? 0 : min(nit, max(0, (ufull - ux0) >> 1));

      // One iteration is 2 units x NM steps.  A step issues one MFMA -- q.k^T of the next unit,
      // and in pass 2 p.V of the one before in turn -- reads the LDS operand of the step kAhead
      // later and works on 16 / NM scores of this unit.  The three do not depend on each other,
      // and the scheduling barriers hold the order: an MFMA takes 32 cycles of the matrix unit, a
      // score about as many of the VALU.  The first steps also write a chunk each of the next
      // stage, whose loads went out an iteration ago, to the third buffer, and send the loads of
      // the stage after it; the iteration's one barrier, at the end of the first unit, publishes
      // the stage, so that the operand reads run on across iterations.  With two buffers the next
      // stage's is the last one's: a barrier at the start, when every wavefront's products of it
      // have gone out.
      constexpr int NM = OUT ? KS + 2 * DT : KS, SPM = 16 / NM, kAhead = OUT ? 4 : 2;
      constexpr int MS = (CPW + 1) & ~1;  // the steps that write and load chunks
      static_assert(CPW <= NM / 2, "kLater operand reads lie between the chunk writes and the barrier");
      constexpr int kLater = NM - MS < NM / 2 ? NM - MS : NM / 2;
      static_assert(KS == 2 * DT && NM * SPM == 16, "q.k^T and p.V steps alternate");
      uint4 *cur = ring[0], *nxt = ring[1], *third = ring[NB - 1];
      auto rotate = [&]() {
        uint4* const t = cur;
        cur = nxt;
        nxt = NB == 2 ? t : third;
        third = t;
      };
      auto operand = [&](const uint4* sb, int m) {  // step m: of unit m / NM, k step or tile i
        const int un = m / NM, i = OUT ? (m % NM) / 2 : m % NM;
        const char* kb = reinterpret_cast<const char*>(sb) + kofs;
        return OUT && (m & 1) ? __builtin_bit_cast(bf16x8, sb[(NK + un * CU + i) * 64 + lane])
                              : *reinterpret_cast<const bf16x8*>(kb + un * (CU * 1024) + i * 512);
      };
      bf16x8 op[kAhead];
      f32x16 sc;        // products of the unit whose scores come next
      uint32_t pw[8];   // p of the unit whose p.V product comes next: two MFMA operands
      auto pop = [&](int h) {
        return __builtin_bit_cast(bf16x8, make_uint4(pw[4 * h], pw[4 * h + 1], pw[4 * h + 2], pw[4 * h + 3]));
      };
      // Pass 1's online (max, sum) per lane of a unit's scores y: the running sum rescaled by
      // exp2((m_old - m_new) log2 e), which is exactly 1 while the max stays (the one-FMA form
      // exp2(m_old log2 e - RN(m_new log2 e)) is off by the product's rounding on every update, and
      // L drifted by ~1e-5 at T = 8192: rel-L2 7e-4 against eager).
      auto online = [&](float (&y)[16]) {
#pragma clang fp contract(off)
        float mt = -INFINITY;
#pragma unroll
        for (int w = 0; w < 16; w += 2) mt = max3f(mt, y[w], y[w + 1]);
        mt *= kUnit;
        if (mt != -INFINITY) {
          const float mn = fmaxf(m_run, mt);
          const float f = __builtin_amdgcn_exp2f((m_run - mn) * kLog2e), nm = -mn * kLog2e;
#pragma unroll
          for (int w = 0; w < 16; ++w) y[w] = __builtin_amdgcn_exp2f(__builtin_fmaf(y[w], kExpCoef, nm));
#pragma unroll
          for (int w = 4; w < 16; ++w) y[w & 3] = y[w & 3] + y[w];
          l_run = l_run * f + ((y[0] + y[1]) + (y[2] + y[3]));
          m_run = mn;
        }
      };
      auto body = [&](int it, bool mask) {
        if constexpr (NB == 2) {
          __builtin_amdgcn_sched_barrier(0);
          asm volatile("" ::: "memory");
          __builtin_amdgcn_s_barrier();
          asm volatile("" ::: "memory");
          __builtin_amdgcn_sched_barrier(0);
        }
        next_ids(it + 2);
        f32x16 sn = (f32x16)0.0f;
        uint32_t pn[8];
        float last = 0.0f, l_next = 0.0f;
        const float nm = OUT ? nml : -m_run * kLog2e;
        float y[16];
        f32x16 first;  // pass 1: the first unit's products, should the sum leave its bound
#pragma unroll
        for (int m = 0; m < 2 * NM; ++m) {
          const int un = m / NM, mm = m % NM, i = OUT ? mm / 2 : mm;
          if (OUT && (m & 1))
            acc[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[m % kAhead], pop(i / DT), acc[i % DT], 0, 0, 0);
          else
            sn = __builtin_amdgcn_mfma_f32_32x32x16_bf16(op[m % kAhead], qop[i], mm == 0 ? (f32x16)0.0f : sn, 0, 0, 0);
          op[m % kAhead] = m + kAhead < 2 * NM ? operand(cur, m + kAhead) : operand(nxt, m + kAhead - 2 * NM);
          // lane (g, n), score e: key 8 (e / 4) + 4 g + e % 4 of the unit
          int limb[2];
          if (mask) {
#pragma unroll
            for (int h = 0; h < 2; ++h) limb[h] = lpb[2 * (2 * it + un) + h] >= 0 ? lim - 32 * (ux0 + 2 * it + un) - 4 * g : -1;
          }
#pragma unroll
          for (int e = mm * SPM; e < (mm + 1) * SPM; ++e) {
            float v = eager(sc[e]);
            if (mask) v = 8 * (e >> 2) + (e & 3) <= limb[e >> 3] ? v : -INFINITY;
            if (!OUT && mask) {
              y[e] = v;
              continue;
            }
            const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(v, kExpCoef, nm));
            if (OUT) {
              if (e & 1)
                pn[e / 2] = pack_bf16x2(last, p);
              else
                last = p;
            } else {
              y[e & 3] = e < 4 ? p : y[e & 3] + p;
            }
          }
          if (m < CPW) {
            stash1(nxt, m);
            stg[m] = fetch1(it + 2, m);
          }
          if (SPM > 1 || (m & 1)) __builtin_amdgcn_sched_barrier(0);
          if (m == MS - 1) asm volatile("" ::: "memory");
          if (m == NM - 1) {
            // LDS operations of a wavefront complete in order: with at most kLater outstanding, all
            // issued after the writes (the operand reads of steps MS .. NM - 1), the writes are done
            asm volatile("" ::: "memory");
            __builtin_amdgcn_s_waitcnt(0xC07F | (kLater << 8));
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            __builtin_amdgcn_sched_barrier(0);
          }
          if (mm == NM - 1) {
            if constexpr (OUT) {
#pragma unroll
              for (int w = 0; w < 8; ++w) pw[w] = pn[w];
            } else {
#pragma clang fp contract(off)
              if (mask) {
                online(y);
              } else {
                const float sum = (un == 0 ? l_run : l_next) + ((y[0] + y[1]) + (y[2] + y[3]));
                if (un == 0) {
                  l_next = sum;
                  first = sc;
                } else if (__ballot(!(sum < kPfSumBound)) & rows) {  // scalar
#pragma unroll
                  for (int w = 0; w < 16; ++w) y[w] = eager(first[w]);
                  online(y);
#pragma unroll
                  for (int w = 0; w < 16; ++w) y[w] = eager(sc[w]);
                  online(y);
                } else {
                  l_run = sum;
                }
              }
            }
            sc = sn;
          }
        }
        rotate();
      };

      // stage 0 and unit 0's K (slot 1 of stage -1), loaded together
      uint4 stg0[NK / W];
      next_ids(-1);
#pragma unroll
      for (int j = 0; j < NK / W; ++j) stg0[j] = fetch1(-1, j);
      next_ids(0);
#pragma unroll
      for (int j = 0; j < CPW; ++j) stg[j] = fetch1(0, j);
      next_ids(1);
#pragma unroll
      for (int j = 0; j < NK / W; ++j) third[(j * W + wave) * 64 + lane] = stg0[j];
#pragma unroll
      for (int j = 0; j < CPW; ++j) {
        stash1(cur, j);
        stg[j] = fetch1(1, j);
      }
      publish();
      {
        const char* kb = reinterpret_cast<const char*>(third) + CU * 1024 + kofs;
        sc = (f32x16)0.0f;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk)
          sc = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8*>(kb + kk * 512), qop[kk], sc, 0, 0, 0);
#pragma unroll
        for (int w = 0; w < 8; ++w) pw[w] = 0;
#pragma unroll
        for (int m = 0; m < kAhead; ++m) op[m] = operand(cur, m);
      }
      int it = 0;
      if (!OUT && active) body(it++, true);
      for (; it < nfast; ++it) body(it, false);
      if (active) {
        for (; it < nit; ++it) body(it, true);
      } else {  // a wavefront without rows loads its share
        for (; it < nit; ++it) {
          if constexpr (NB == 2) publish();
          next_ids(it + 2);
#pragma unroll
          for (int j = 0; j < CPW; ++j) {
            stash1(nxt, j);
            stg[j] = fetch1(it + 2, j);
          }
          publish();
          rotate();
        }
      }
      if constexpr (OUT) {  // the last unit's p.V
        if (active) {
#pragma unroll
          for (int i = 0; i < 2 * DT; ++i)
            acc[i % DT] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(operand(cur, 2 * i + 1), pop(i / DT), acc[i % DT], 0, 0, 0);
        }
      }
    }

    if constexpr (!OUT) {
      // (max, sum) of each row over its two lanes
      merge_lanes<32>(m_run, l_run);
      if (g == 0 && rv) st[seg] = make_float2(m_run, l_run);
    } else {
      const int rgi = pos.lk * nf + pos.f;
      if (seg == 0 && tid == 0 && per2) pf_desc(a)[rgi] = make_int2(w0b, nseg2);
      if (nseg2 > 1) {  // workgroup-uniform: this segment's fp32 part, in lane order
        float4* slot = pf_slot(a, D, w0b, seg, rgi) + wave * (DT * 4 * 64) + lane;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            slot[(dt * 4 + j) * 64] = make_float4(acc[dt][4 * j], acc[dt][4 * j + 1], acc[dt][4 * j + 2], acc[dt][4 * j + 3]);
      } else if (rv) {
        uint16_t* op = a.out + qofs + 4 * g;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
          for (int j = 0; j < 4; ++j)
            *reinterpret_cast<uint2*>(op + dt * 32 + 8 * j) =
                make_uint2(pack_bf16x2(acc[dt][4 * j], acc[dt][4 * j + 1]), pack_bf16x2(acc[dt][4 * j + 2], acc[dt][4 * j + 3]));
      }
    }

    // the next row group of the range
    if constexpr (SHORT) break;
    u = next;
    if (u < uend) {
      pos.start = next;
      if (++pos.f == nf) {
        pos.f = 0;
        ++pos.lk;
      }
      pos.wt = weight_of(pos.f);
    }
  }

  if constexpr (!OUT) {
    // Pass 2's V operand, a page block per wavefront: bf16(fp32(code) * scale), per 32-dimension
    // tile 64 lanes x 16 bytes (lane (g, m): dimension 32 dt + m, tokens 4g..4g+3 and
    // 8+4g..8+4g+3).  Codes and scales of tokens that are not in the sequence (past T, invalid or
    // absent blocks) become 0, so that no NaN pattern of an unwritten slot reaches the MFMA; up
    // to the end of the last stage every block is written, an empty sequence's one stage too.
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const int nbmax = 2 * a.vh_stages;
    const int64_t items = (int64_t)LK * a.B * nbmax;
    const int first = SHORT ? nf * LK : 0, wg = (int)blockIdx.x - first, wgs = (int)gridDim.x - first;
    if (wg < 0) return;
    for (int64_t i = (int64_t)wg * W + wave; i < items; i += (int64_t)wgs * W) {
      const int z = (int)(i / nbmax), blk = (int)(i - (int64_t)z * nbmax);
      const int zb = z / a.KV, kvh = z - zb * a.KV, layer = zb / a.B, b = zb - layer * a.B;
      const int T = seq_len_of(a, b), nbk = (T + kBlock - 1) / kBlock;
      if (blk >= max((nbk + 3) & ~3, kPfStage / kBlock)) continue;
      int pb = blk < nbk ? a.block_table[(int64_t)b * a.max_blocks + blk] : -1;
      if (pb >= a.num_blocks) pb = -1;
      const int64_t pg = max(pb, 0);
      const uint8_t* vp = a.v_pages + layer * a.v_ls + (pg * a.KV + kvh) * (D * kBlock);
      const float* sp = a.v_scales + layer * a.s_ls + (pg * a.KV + kvh) * kBlock;
      uint32_t w[DT][2];
      float4 sc[2];
#pragma unroll
      for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int h = 0; h < 2; ++h) w[dt][h] = *reinterpret_cast<const uint32_t*>(vp + (dt * 32 + n) * kBlock + 8 * h + 4 * g);
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        sc[h] = *reinterpret_cast<const float4*>(sp + 8 * h + 4 * g);
        const int nv = pb >= 0 ? min(max(T - (blk * kBlock + 8 * h + 4 * g), 0), 4) : 0;
        const uint32_t mask = nv >= 4 ? 0xFFFFFFFFu : (1u << (8 * nv)) - 1u;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) w[dt][h] &= mask;
        sc[h].x = nv > 0 ? sc[h].x : 0.0f;
        sc[h].y = nv > 1 ? sc[h].y : 0.0f;
        sc[h].z = nv > 2 ? sc[h].z : 0.0f;
        sc[h].w = nv > 3 ? sc[h].w : 0.0f;
      }
      uint4* dst = a.vhat + ((int64_t)z * nbmax + blk) * (DT * 64) + lane;
#pragma unroll
      for (int dt = 0; dt < DT; ++dt) {
        uint32_t o[4];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const f32x2 f01 = __builtin_amdgcn_cvt_pk_f32_fp8(w[dt][h], false);
          const f32x2 f23 = __builtin_amdgcn_cvt_pk_f32_fp8(w[dt][h], true);
          o[2 * h] = pack_bf16x2(f01.x * sc[h].x, f01.y * sc[h].y);
          o[2 * h + 1] = pack_bf16x2(f23.x * sc[h].z, f23.y * sc[h].w);
        }
        dst[dt * 64] = make_uint4(o[0], o[1], o[2], o[3]);
      }
    }
  }
}

// Sums the parts of the row groups that several ranges cut, in range order, and writes BF16.  A
// workgroup takes the 32 rows of one wavefront's slot share; a thread 8 dimensions of a row (the
// 16-byte pieces of lanes n and n + 32) per step.
template <int D>
__global__ __launch_bounds__(256) void prefill_reduce_kernel(AttnArgs a) {
  constexpr int DT = D / 32;
  const int rgi = (int)blockIdx.x / kPfWaves, wave = (int)blockIdx.x % kPfWaves;
  const int2 d = pf_desc(a)[rgi];
  if (d.y <= 1) return;
  const int nf = a.B * a.pf_nrg, lk = rgi / nf, f = rgi - lk * nf;
  const int layer = lk / a.KV, kvh = lk - layer * a.KV, b = f / a.pf_nrg, rg = f - b * a.pf_nrg;
  const int n = threadIdx.x & 31, r = rg * kPfRows + wave * 32 + n;
  if (r >= a.R) return;
  const int si = r / a.G, hl = r - si * a.G;
  uint16_t* op = a.out + layer * a.q_ls + b * a.q_sb + (int64_t)(kvh * a.G + hl) * a.q_sh + si * a.q_ss;
  constexpr int P = DT * 4 / 8;  // pieces per thread: of the row's DT x 4, every eighth
  float4 sum[P][2];
#pragma unroll
  for (int i = 0; i < P; ++i) sum[i][0] = sum[i][1] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int k0 = 0; k0 < d.y; k0 += 4) {
    float4 v[4][P][2];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const float4* slot = pf_slot(a, D, d.x, min(k0 + k, d.y - 1), rgi) + wave * (DT * 4 * 64) + n;
#pragma unroll
      for (int i = 0; i < P; ++i)
#pragma unroll
        for (int h = 0; h < 2; ++h) v[k][i][h] = slot[(i * 8 + (threadIdx.x >> 5)) * 64 + 32 * h];
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (k0 + k < d.y) {
#pragma unroll
        for (int i = 0; i < P; ++i)
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            sum[i][h].x += v[k][i][h].x;
            sum[i][h].y += v[k][i][h].y;
            sum[i][h].z += v[k][i][h].z;
            sum[i][h].w += v[k][i][h].w;
          }
      }
  }
#pragma unroll
  for (int i = 0; i < P; ++i) {
    const float4 x = sum[i][0], y = sum[i][1];
    *reinterpret_cast<uint4*>(op + (i * 8 + (threadIdx.x >> 5)) * 8) =
        make_uint4(pack_bf16x2(x.x, x.y), pack_bf16x2(x.z, x.w), pack_bf16x2(y.x, y.y), pack_bf16x2(y.z, y.w));
  }
}

}  // namespace sdv
