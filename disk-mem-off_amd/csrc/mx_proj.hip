// Projections of short inputs (at most MX_PROJ_MAX_TOKENS tokens): y_s[T, N_s] =
// a[T, K] W_s[N_s, K]^T for up to MX_GEMM_MAX_SEG row-major fp16 or per-row int8 weight
// matrices that share the fp16 activation a (linear_t, offload_runtime/executors/
// _common.py:101-103, of the attention blocks' decode batches).
//
// Bound by the weight stream.  A block owns 16 NB output columns; its 4 waves split the
// reduction (and, for products of few columns, up to MX_PROJ_MAX_SLICES grid slices split
// it further), so a block reads whole weight rows at once and a wave issues up to 16 KiB of
// weight pieces before it waits for the first.  The single-group form of the expert
// kernels, which ran these products before, walks the whole reduction per wave with a few
// pieces in flight, on 16 blocks in all for a 2048-column projection of 17 and more tokens.
// The activation rows come from L2, in two register sets; each of their fragment loads
// touches 16 cache lines for 64 bytes apiece, which is what bounds 17 and more tokens, so
// there two column tiles share them (NB = 2).
// Measured (rocprofv3, distinct weights per call, hidden 2048): qkvz + ba of 20,512 rows, one
// token 24.8 -> 18.9 us (4.4 TB/s), 24 tokens 63.8 -> 27.9 us (NB = 1: 32.9); the 2048-row
// output projection of 4096 columns, one token 13.1 -> 6.1 us, 24 tokens 58.1 -> 7.5 us.
// Slower: the nontemporal hint the expert kernels use (20.2 us; it drops lines whose other
// half is still to be read in this row-major form), 8 waves per block (24 tokens 29.7 us),
// NB = 4 (33.7 us), NB = 2 for one token (20.6 us).
//
// Operands as in the expert kernels: lane 16 q + j holds 16 bytes of weight row n0 + j and
// of activation row j at the same reduction columns; the weights are the MFMA's A operand,
// so lane (j, q) ends with columns n0 + 4 q .. + 3 of token j.
#include "mx_common.h"
#include "mx_internal.h"

namespace {

#define PJ_OOB 0x80000000u  // any offset >= this is outside every descriptor built here

__device__ __forceinline__ __amdgpu_buffer_rsrc_t pj_rsrc(const void* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc((void*)base, (short)0, (int)bytes, 0x00020000);
}

struct ProjArgs {
  MxProjSeg seg[MX_GEMM_MAX_SEG];
  int unit0[MX_GEMM_MAX_SEG + 1];  // first 16 NB-column unit of each segment, then the total
  int nseg, T, K;
  const half_t* a;
};

template <int WF, int MT, int UB, int NB>
__global__ __launch_bounds__(256) void k_proj(const ProjArgs p) {
  constexpr int EPL = WF == MX_DT_I8 ? 16 : 8;  // columns per 16-byte weight piece
  constexpr int ESZ = WF == MX_DT_I8 ? 1 : 2;
  constexpr int KC = 4 * EPL;         // columns per chunk (one piece per lane)
  constexpr int AV = EPL / 8;         // activation pieces per chunk
  constexpr int UA = 8 / (MT * AV);   // chunks per activation set
  constexpr int NA = UB / UA;
  static_assert(UB % UA == 0, "whole activation sets");

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int j = lane & 15, q = lane >> 4;
  int s = 0;
#pragma unroll
  for (int i = 1; i < MX_GEMM_MAX_SEG; ++i)
    if (i < p.nseg && (int)blockIdx.x >= p.unit0[i]) s = i;
  const MxProjSeg sg = p.seg[s];
  const int n0 = ((int)blockIdx.x - p.unit0[s]) * 16 * NB;
  const int K = p.K, T = p.T;

  const __amdgpu_buffer_rsrc_t rw = pj_rsrc(sg.w, (uint32_t)sg.n * (uint32_t)K * ESZ);
  const __amdgpu_buffer_rsrc_t ra = pj_rsrc(p.a, (uint32_t)T * (uint32_t)K * 2);
  uint32_t woff[NB];
#pragma unroll
  for (int f = 0; f < NB; ++f)
    woff[f] = n0 + 16 * f + j < sg.n
                  ? (uint32_t)(n0 + 16 * f + j) * (uint32_t)K * ESZ + (uint32_t)(q * 16)
                  : PJ_OOB;
  uint32_t aoff[MT];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi)
    aoff[mi] = 16 * mi + j < T ? (uint32_t)(16 * mi + j) * (uint32_t)K * 2 + (uint32_t)(q * EPL * 2)
                               : PJ_OOB;

  // This wave's chunks [cb, ce) of the ceil(K / KC).
  const int nch = (K + KC - 1) / KC;
  const int parts = 4 * (int)gridDim.y;
  const int cw = (nch + parts - 1) / parts;
  const int cb = min(nch, ((int)blockIdx.y * 4 + wave) * cw), ce = min(nch, cb + cw);

  half_t sc[NB][4];  // row scales of the lane's columns, requested ahead of the weights
  if constexpr (WF == MX_DT_I8) {
#pragma unroll
    for (int f = 0; f < NB; ++f)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        sc[f][i] = ((const half_t*)sg.scale)[min(n0 + 16 * f + 4 * q + i, sg.n - 1)];
  }

  float4_t acc[MT][NB];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi)
#pragma unroll
    for (int f = 0; f < NB; ++f) acc[mi][f] = (float4_t){0.f, 0.f, 0.f, 0.f};

  // Whether the lane's piece of chunk c is inside the wave's range and the row.
  auto in = [&](int c) { return c < ce && c * KC + q * EPL < K; };
  for (int c0 = cb; c0 < ce; c0 += UB) {
    int4_t b[UB][NB], a[2][UA][MT][AV];
#pragma unroll
    for (int u = 0; u < UB; ++u)
#pragma unroll
      for (int f = 0; f < NB; ++f)
        b[u][f] = __builtin_amdgcn_raw_buffer_load_b128(
            rw, in(c0 + u) ? woff[f] + (uint32_t)((c0 + u) * KC * ESZ) : PJ_OOB, 0, 0);
    auto load_a = [&](int set, int4_t (&d)[UA][MT][AV]) {
#pragma unroll
      for (int u = 0; u < UA; ++u) {
        const int c = c0 + set * UA + u;
        const bool ok = in(c);
#pragma unroll
        for (int mi = 0; mi < MT; ++mi)
#pragma unroll
          for (int v = 0; v < AV; ++v)
            d[u][mi][v] = __builtin_amdgcn_raw_buffer_load_b128(
                ra, ok ? aoff[mi] + (uint32_t)(c * KC * 2 + 16 * v) : PJ_OOB, 0, 0);
      }
    };
    load_a(0, a[0]);
    // Without the scheduling barriers the compiler trades the loads in flight for registers.
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int set = 0; set < NA; ++set) {
      if (set + 1 < NA) load_a(set + 1, a[(set + 1) & 1]);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int u = 0; u < UA; ++u) {
#pragma unroll
        for (int f = 0; f < NB; ++f) {
          const int4_t w = b[set * UA + u][f];
          half8_t wf[AV];
          if constexpr (WF == MX_DT_I8)
            mx_i8_to_f16(w, wf[0], wf[1]);
          else
            wf[0] = __builtin_bit_cast(half8_t, w);
#pragma unroll
          for (int mi = 0; mi < MT; ++mi)
#pragma unroll
            for (int v = 0; v < AV; ++v)
              acc[mi][f] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                  wf[v], __builtin_bit_cast(half8_t, a[set & 1][u][mi][v]), acc[mi][f], 0, 0, 0);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
  }

  // The waves' partial tiles, added in wave order; tile i (token tile i / NB, column tile
  // i % NB) is finished by wave i % 4.
  constexpr int NT = MT * NB;
  __shared__ float4_t red[4][NT][64];
#pragma unroll
  for (int i = 0; i < NT; ++i) red[wave][i][lane] = acc[i / NB][i % NB];
  __syncthreads();
#pragma unroll
  for (int i0 = 0; i0 < NT; i0 += 4) {
    const int i = i0 + wave;
    if (i >= NT) return;
    float4_t r = red[0][i][lane];
#pragma unroll
    for (int w = 1; w < 4; ++w) r += red[w][i][lane];
    const int f = i % NB, n = n0 + 16 * f + 4 * q, t = 16 * (i / NB) + j;
    if (t >= T) continue;
    if constexpr (WF == MX_DT_I8) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        half_t v = sc[0][e];
#pragma unroll
        for (int g = 1; g < NB; ++g) v = f == g ? sc[g][e] : v;
        r[e] *= (float)v;
      }
    }
    float* y = sg.y + ((size_t)blockIdx.y * T + t) * sg.ldy;
    if (n + 3 < sg.n && (sg.ldy & 3) == 0) {
      *(float4_t*)(y + n) = r;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < sg.n) y[n + e] = r[e];
    }
  }
}

template <int WF, int MT, int NB>
void launch_mt(const ProjArgs& p, dim3 grid, int cw, hipStream_t s) {
  // 8 chunks per set of loads where they are a wave's whole range or come NB = 2 wide.
  if (WF == MX_DT_I8 || cw <= 8 || NB > 1)
    hipLaunchKernelGGL((k_proj<WF, MT, 8, NB>), grid, dim3(256), 0, s, p);
  else
    hipLaunchKernelGGL((k_proj<WF, MT, 16, NB>), grid, dim3(256), 0, s, p);
}

template <int WF>
void launch_wf(const ProjArgs& p, dim3 grid, int cw, hipStream_t s) {
  if (p.T <= 16)
    launch_mt<WF, 1, 1>(p, grid, cw, s);
  else if (p.T <= 32)
    launch_mt<WF, 2, 2>(p, grid, cw, s);
  else
    launch_mt<WF, 4, 2>(p, grid, cw, s);
}

// Column tiles per block: two where the activation loads bound (see the top).
int nb_of(int T) { return T <= 16 ? 1 : 2; }

int chunk_cols(int wdt) { return wdt == MX_DT_I8 ? 64 : 32; }

}  // namespace

bool mx_proj_ok(int wdt, int T, int K) {
  return T <= MX_PROJ_MAX_TOKENS &&
         ((wdt == MX_DT_F16 && K % 8 == 0) || (wdt == MX_DT_I8 && K % 16 == 0));
}

int mx_proj_slices(int wdt, int N, int K) {
  // Up to 512 16-column units, while a wave keeps at least four chunks of its reduction: two
  // blocks per CU up to 16 tokens, one of two units above.
  const int units = mx_ceil_div(N, 16), nch = mx_ceil_div(K, chunk_cols(wdt));
  int s = 1;
  while (s < MX_PROJ_MAX_SLICES && units * s < 512 && nch >= 4 * 4 * 2 * s) s *= 2;
  return s;
}

int mx_proj(int wdt, const void* a, int T, int K, const MxProjSeg* segs, int nseg, int slices,
            hipStream_t s) {
  if (!mx_proj_ok(wdt, T, K)) return MX_ERR_UNSUPPORTED;
  if (T <= 0 || K <= 0 || !a || !segs || nseg < 1 || nseg > MX_GEMM_MAX_SEG || slices < 1 ||
      slices > MX_PROJ_MAX_SLICES || (slices > 1 && (nseg != 1 || segs[0].ldy != segs[0].n)))
    return MX_ERR_INVALID;
  if (!mx_aligned16(a)) return MX_ERR_ALIGNMENT;
  ProjArgs p = {};
  int units = 0;
  for (int i = 0; i < nseg; ++i) {
    if (!segs[i].w || !segs[i].y || segs[i].n <= 0 || (wdt == MX_DT_I8 && !segs[i].scale))
      return MX_ERR_INVALID;
    if ((long)segs[i].n * K * (wdt == MX_DT_I8 ? 1 : 2) >= (1l << 31)) return MX_ERR_UNSUPPORTED;
    if (!mx_aligned16(segs[i].w) || !mx_aligned16(segs[i].y)) return MX_ERR_ALIGNMENT;
    p.seg[i] = segs[i];
    p.unit0[i] = units;
    units += mx_ceil_div(segs[i].n, 16 * nb_of(T));
  }
  if ((long)T * K * 2 >= (1l << 31)) return MX_ERR_UNSUPPORTED;
  p.unit0[nseg] = units;
  p.nseg = nseg;
  p.T = T;
  p.K = K;
  p.a = (const half_t*)a;
  const int cw = mx_ceil_div(mx_ceil_div(K, chunk_cols(wdt)), 4 * slices);
  mx_clear_error();
  if (wdt == MX_DT_I8)
    launch_wf<MX_DT_I8>(p, dim3(units, slices), cw, s);
  else
    launch_wf<MX_DT_F16>(p, dim3(units, slices), cw, s);
  return mx_launch_status();
}
