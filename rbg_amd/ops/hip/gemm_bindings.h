// Binding of the decode-shape GEMM, for every extension that links
// skinny_gemm.hip.
#pragma once
#include <torch/extension.h>
#include <ATen/hip/HIPContext.h>

#include <hip/hip_runtime.h>

#include <algorithm>

extern "C" {
void launch_skinny_gemm(void*, void*, const void*, const void*, int, int,
                        int, int, int, int, hipStream_t);
void launch_reduce_splits(void*, const void*, int, long, hipStream_t);
}

inline hipStream_t gemm_stream() {
  return at::hip::getCurrentHIPStream().stream();
}

// Which kernel a shape takes: waves per workgroup (0: the kernel of a few
// rows) and the parts that K is split into.
struct SkinnyPlan {
  int waves, splits;
};

inline SkinnyPlan pick_skinny(int M, int N, int K) {
  // a few rows, where K is whole turns of that kernel (8 waves x 4 chunks of 64
  // in flight; in a part of one it loads the last chunk again, with K = 2560 8
  // times for 5 chunks), or short, where that costs less than a reduction (2048 x
  // 5632, 1 row: 9.0 us against 9.7, 4 rows 10.1 against 10.0).
  if ((M <= 4 && K % 2048 == 0) || (M <= 2 && K <= 8192 && N <= 12288))
    return {0, 1};
  // One round of workgroups, the last of 1.5 or 2.5 is lost (10240 x 8192, 64 rows:
  // 3 parts = 240 workgroups 38 us, 4 parts 48, 6 parts 40).  Of those the form in
  // which a CU has the least to read, as it reads about as fast with four waves as with
  // eight, and between nearly equal ones that with fewer parts, which are written and
  // read again.  Of all forms at 774 shapes of 5 to 128 rows, 1024 to 10240 columns and
  // 1024 to 25600 k, the parts' reader at 4 TB/s, it takes 0.6% more than the best one;
  // up to three workgroups of four waves on a CU took 8% (7 rows: 4096 x 12288 19.0, 4
  // parts 18.3; 6144 x 4096 10.9, 11.0; 32 rows of 8192 x 2048 1.35 of the best).
  SkinnyPlan best{8, 1};
  float least = 1e30f;
  for (int waves = M <= 32 ? 4 : 8; waves <= 8; waves += 4)
    for (int splits : {1, 2, 3, 4, 5, 6, 8, 10, 12, 16}) {
      if (splits > std::max(1, K / 256) ||
          (N + 16 * waves - 1) / (16 * waves) * splits > 256)
        break;
      const float t = (K / 128 + splits - 1) / splits * waves +
                      splits * (1.f + 0.02f * M);
      if (t < least) {
        least = t;
        best = {waves, splits};
      }
    }
  return best;
}

// The same for a product whose parts a launch of its own adds up, which a few
// long parts repay and many short ones do not: the form with the least time by
// a model of it in us, fitted to all forms at 5083 shapes of 1 to 256 rows, 1024
// to 128256 columns and 512 to 28672 k with cold weights.  Its choices take 0.7%
// longer than the fastest form on average; pick_skinny's take 5.4% (8 rows, 1024
// x 512: two parts 5.6, one 4.2 us; 128 rows, 10240 x 1024: 19.9 and 17.9).
inline SkinnyPlan pick_summed(int M, int N, int K) {
  // a few rows: where one round of workgroups covers N, or K is whole turns of
  // that kernel (1 row, 4096 x 1536: 5.2 us against 7.3 of the other forms; 5120
  // x 2048 7.8 against 9.0, 5120 x 2560 13.1 against 11.0)
  if (M <= 4 && K >= 1024 &&
      (N <= 4096 ? K <= 3 * N
                 : (N <= 8192 && K < 2048) || (K % 2048 == 0 && K <= 8192)))
    return {0, 1};
  const int tiles = (M + 15) / 16;
  SkinnyPlan best{8, 1};
  float least = 1e30f;
  for (int waves = M <= 32 ? 4 : 8; waves <= 8; waves += 4)
    for (int splits : {1, 2, 3, 4, 5, 6, 8, 12, 16}) {
      if (splits > std::max(1, K / 256)) break;
      const int groups = (N + 16 * waves - 1) / (16 * waves) * splits;
      const int chunks = (K / 128 + splits - 1) / splits;
      float t;
      if (waves == 4)   // two on a CU share its bandwidth
        t = (groups + 511) / 512 * chunks *
            std::max(0.67f, std::min(2, (groups + 255) / 256) *
                                (0.46f + 0.088f * tiles));
      else
        t = (groups + 255) / 256 * (0.69f + chunks * (0.63f + 0.16f * tiles));
      if (splits > 1) t += 3.57f + 1.83e-6f * splits * M * N;
      t *= 1.f + 0.0084f * (splits - 1);
      if (t < least) {
        least = t;
        best = {waves, splits};
      }
    }
  return best;
}

inline bool skinny_gemm_supported(int64_t M, int64_t N, int64_t K) {
  return M >= 1 && M <= 256 && (N % 32) == 0 && (K % 256) == 0;
}

inline void check_skinny(const torch::Tensor& a, const torch::Tensor& w) {
  for (const auto& t : {a, w})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                t.is_contiguous() && t.dim() == 2,
                "operands must be contiguous bf16 matrices on GPU");
  TORCH_CHECK(w.size(1) == a.size(1), "K mismatch");
  TORCH_CHECK(skinny_gemm_supported(a.size(0), w.size(0), a.size(1)),
              "unsupported skinny shape");
}

// wide: the result, rounded to bf16 all the same, in f32
inline torch::Tensor skinny_gemm(torch::Tensor a, torch::Tensor w,
                                 int64_t force_splits = 0, bool wide = false) {
  check_skinny(a, w);
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0);
  SkinnyPlan plan = pick_summed((int)M, (int)N, (int)K);
  if (force_splits > 0 && K % (force_splits * 256) == 0)
    plan = {plan.waves ? plan.waves : 8, (int)force_splits};
  const bool direct = wide && plan.splits == 1;
  auto c = torch::empty(
      {M, N}, direct ? a.options().dtype(torch::kFloat32) : a.options());
  torch::Tensor ws;
  void* wsp = direct ? c.data_ptr() : nullptr;
  if (plan.splits > 1) {
    ws = torch::empty({plan.splits, M, N}, a.options().dtype(torch::kFloat32));
    wsp = ws.data_ptr();
  }
  launch_skinny_gemm(direct ? nullptr : c.data_ptr(), wsp, a.data_ptr(), w.data_ptr(), (int)M,
                     (int)N, (int)K, plan.waves, plan.splits, 0,
                     gemm_stream());
  if (plan.splits > 1)
    launch_reduce_splits(c.data_ptr(), wsp, plan.splits, (long)(M * N),
                         gemm_stream());
  return wide && !direct ? c.to(torch::kFloat32) : c;
}
