// Dense projections of the attention blocks: y[T, N] = a[T, K] W^T on the single-group
// down-projection kernels of the MoE experts (fp32 weights, and reduction lengths that the
// others do not take), and the projection that ends an attention block, on whichever of
// mx_proj (short inputs), mx_gemm (long ones) and those kernels runs it.
#include "mx_common.h"
#include "mx_internal.h"

namespace {

__global__ __launch_bounds__(256) void k_dense_setup(int T, int m_blk, int n_mt,
                                                     MxDenseEntries ents, int n_ent,
                                                     MxExpertPtrs* __restrict__ entries,
                                                     int* __restrict__ tabs,
                                                     int* __restrict__ mt_group,
                                                     int* __restrict__ mt_row0,
                                                     float* __restrict__ ones) {
  const int i = blockIdx.x * 256 + threadIdx.x;
  if (i < n_ent) entries[i] = ents.e[i];
  if (i == 0) {
    tabs[0] = 0;  // g_expert
    tabs[1] = 0;  // g_start
    tabs[2] = T;  // g_count
    tabs[3] = n_mt;
  }
  if (i < n_mt) {
    mt_group[i] = 0;
    mt_row0[i] = i * m_blk;
  }
  if (i < T) ones[i] = 1.f;
}

// out = x + y, or + the slices of y (n floats each) in slice order; y then receives their sum
// where it is wanted.
template <bool SLICED>
__global__ __launch_bounds__(256) void k_residual(const float* x, float* y, long n4, int slices,
                                                  bool keep, float* out) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const float4_t a = ((const float4_t*)x)[i];
  float4_t b = ((const float4_t*)y)[i];
  if constexpr (SLICED) {
    float4_t e[MX_GEMM_MAX_SLICES - 1];
#pragma unroll
    for (int s = 1; s < MX_GEMM_MAX_SLICES; ++s)
      if (s < slices) e[s - 1] = ((const float4_t*)y)[i + s * n4];
#pragma unroll
    for (int s = 1; s < MX_GEMM_MAX_SLICES; ++s)
      if (s < slices) b += e[s - 1];
    if (keep) ((float4_t*)y)[i] = b;
  }
  ((float4_t*)out)[i] = a + b;
}

static_assert(MX_PROJ_MAX_SLICES <= MX_GEMM_MAX_SLICES, "k_residual adds either's slices");

// Up to here the product goes through y whatever its slices.
#define MX_OUT_Y_TOKENS 64

// Whether the whole product is left in y (the header's view): always for int8 weights, and
// for fp16 ones up to MX_OUT_Y_TOKENS tokens.
bool keep_product(int wdt, int T) { return wdt == MX_DT_I8 || T <= MX_OUT_Y_TOKENS; }

// Reduction slices of an output projection.
int out_slices(int wdt, int T, int N, int K) {
  if (mx_use_proj(wdt, T, K, N)) return mx_proj_slices(wdt, N, K);
  if (mx_dense_on_gemm(wdt, T, K, N)) return mx_gemm_slice_count(wdt, T, N, K);
  return 1;
}

}  // namespace

size_t mx_out_rows(int T, int N) {
  // At least slices x T for every path's slice count, and never less for fewer tokens (a
  // workspace sized for a batch serves the shorter ones).  mx_proj doubles its slices while
  // ceil(N / 16) times half of them is below 512, so N < 16384 / slices: with T <= 64 that is
  // slices x T < 2^20 / N rows (and at most 256), inside `most`, about 2^22 / N.  The GEMM keeps
  // slices times its 128 x 128 tiles within MX_GEMM_SLICE_BLOCKS.
  const size_t most = (size_t)128 * MX_GEMM_SLICE_BLOCKS / mx_ceil_div(N, 128);
  const size_t want = (size_t)MX_GEMM_MAX_SLICES * T;
  const size_t rows = want < most ? want : most;
  return rows > (size_t)T ? rows : (size_t)T;
}

int mx_out_project(const MxDenseWork& dw, int ent, int wdt, const void* w, const void* scale,
                   int T, int N, int K, const void* a, float* y, const float* x, float* out,
                   hipStream_t s) {
  const int slices = out_slices(wdt, T, N, K);
  if (mx_use_proj(wdt, T, K, N)) {
    const MxProjSeg g{w, scale, y, N, N};
    return mx_proj(wdt, a, T, K, &g, 1, slices, s);
  }
  if (mx_dense_on_gemm(wdt, T, K, N)) {
    if (slices > 1 || T <= MX_OUT_Y_TOKENS) {
      const MxGemmSeg g{w, y, N, N, nullptr, nullptr, scale};
      return mx_gemm_slices(wdt, a, T, K, &g, slices, s);
    }
    if (!x || !out) return MX_ERR_INVALID;
    const MxGemmSeg g{w, out, N, N, nullptr, x, scale, keep_product(wdt, T) ? y : nullptr};
    return mx_gemm(wdt, a, T, K, &g, 1, s);
  }
  return mx_project(dw, ent, wdt, T, N, K, a, y, s);
}

int mx_out_residual(int wdt, int T, int N, int K, float* y, const float* x, float* out,
                    hipStream_t s) {
  const int slices = out_slices(wdt, T, N, K);
  const bool gemm = !mx_use_proj(wdt, T, K, N) && mx_dense_on_gemm(wdt, T, K, N);
  if (gemm && slices == 1 && T > MX_OUT_Y_TOKENS) return MX_OK;  // added in the GEMM's epilogue
  const long n4 = (long)T * N / 4;
  const dim3 grid((unsigned)((n4 + 255) / 256));
  mx_clear_error();
  if (slices > 1)
    hipLaunchKernelGGL(k_residual<true>, grid, dim3(256), 0, s, x, y, n4, slices,
                       keep_product(wdt, T), out);
  else
    hipLaunchKernelGGL(k_residual<false>, grid, dim3(256), 0, s, x, y, n4, 1, false, out);
  return mx_launch_status();
}

size_t mx_dense_work_bytes(int T, int weight_dtype, int n_ent) {
  const int Tn = T > 0 ? T : 1;
  const int m_blk = mx_m_blk_for(Tn, weight_dtype);
  const size_t n_mt = (size_t)mx_ceil_div(Tn, m_blk);
  return mx_align_up((size_t)n_ent * sizeof(MxExpertPtrs), 256) + 256 +
         2 * mx_align_up(n_mt * 4, 256) + mx_align_up((size_t)Tn * 4, 256);
}

void mx_dense_work_carve(char* base, int T, int weight_dtype, int n_ent, MxDenseWork* w) {
  const int Tn = T > 0 ? T : 1;
  w->m_blk = mx_m_blk_for(Tn, weight_dtype);
  w->n_mt = mx_ceil_div(Tn, w->m_blk);
  w->n_ent = n_ent;
  char* p = base;
  w->entries = (MxExpertPtrs*)p;
  p += mx_align_up((size_t)n_ent * sizeof(MxExpertPtrs), 256);
  w->tabs = (int*)p;
  p += 256;
  w->mt_group = (int*)p;
  p += mx_align_up((size_t)w->n_mt * 4, 256);
  w->mt_row0 = (int*)p;
  p += mx_align_up((size_t)w->n_mt * 4, 256);
  w->ones = (float*)p;
}

int mx_dense_setup(const MxDenseWork& w, const MxDenseEntries& ents, int T, hipStream_t s) {
  if (w.n_ent > MX_DENSE_MAX_ENT) return MX_ERR_INVALID;
  int nth = T > w.n_mt ? T : w.n_mt;
  if (w.n_ent > nth) nth = w.n_ent;
  mx_clear_error();
  hipLaunchKernelGGL(k_dense_setup, dim3(mx_ceil_div(nth, 256)), dim3(256), 0, s, T, w.m_blk,
                     w.n_mt, ents, w.n_ent, w.entries, w.tabs, w.mt_group, w.mt_row0, w.ones);
  return mx_launch_status();
}

int mx_project(const MxDenseWork& w, int ent, int wdt, int T, int N, int K, const void* a,
               float* y, hipStream_t s) {
  if (ent < 0 || ent >= w.n_ent) return MX_ERR_INVALID;
  const MxDenseTables tab{w.tabs + 0, w.tabs + 1, w.tabs + 2, w.mt_group, w.mt_row0,
                          w.tabs + 3, w.ones, w.m_blk};
  return mx_dense_linear(wdt, 0, w.entries + ent, tab, T, N, K, a, y, s);
}
