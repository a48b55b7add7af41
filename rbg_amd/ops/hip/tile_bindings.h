// Forms of the GEMM of prompts (tile_gemm.hip): which tiles, how many parts.
#pragma once
#include <torch/extension.h>

#include <hip/hip_runtime.h>

#include <algorithm>

#include "gemm_bindings.h"

extern "C" int launch_tile_gemm(void*, const void*, const void*, int, int, int,
                                int, int, int, int, int, int, int, hipStream_t);

enum TileEnd { TILE_PLAIN, TILE_PARTS, TILE_GLU };

// A tile of 32 wm rows and 32 wn rows of W and the time of a launch in us: fixed
// + rounds * (round + stages * (step + busy * share of workgroups with work)) +
// write * MB of the result.  Fitted to 1600 to 4900 launches of each form, 65 to 4096
// rows, 1024 to 65536 columns, 1024 to 28672 k with cold weights (half of them within 4
// to 10%).  A stage takes longer where more CUs are busy, as the chip lowers its clock.
// The numbers of rows lie so that few are lost: 300 are two tiles of 160, not of 192 or
// 256.  Choices by this, with the reader of the result, take 1.4% more than the best
// form of 2800 shapes with its best parts; the first six forms' best takes 2.6% more.
struct TileForm {
  int wm, wn, fill;             // fill: fewest stages of an item
  bool sums, glu;               // candidates for plain products, or with silu
  float fixed, round, step, busy, write;
};

constexpr TileForm TILE_FORMS[] = {
    {8, 8, 2, true, true, 5.33f, 5.04f, 0.741f, 0.644f, 0.018f},
    {6, 8, 2, true, true, 8.28f, 0.52f, 0.768f, 0.431f, 0.037f},
    {8, 6, 2, true, false, 5.59f, 1.94f, 0.661f, 0.428f, 0.088f},
    {6, 6, 3, true, false, 7.41f, 0.00f, 0.495f, 0.381f, 0.120f},
    {8, 4, 3, true, true, 4.66f, 1.35f, 0.529f, 0.270f, 0.098f},
    {4, 4, 4, true, true, 5.45f, 0.00f, 0.349f, 0.204f, 0.096f},
    {2, 4, 6, false, true, 5.19f, 0.00f, 0.214f, 0.224f, 0.000f},
    {2, 8, 4, false, false, 0.f, 0.f, 0.f, 0.f, 0.f},
    {7, 8, 2, true, true, 7.22f, 2.78f, 0.745f, 0.529f, 0.019f},
    {5, 8, 3, true, true, 7.79f, 0.60f, 0.630f, 0.334f, 0.084f},
    {5, 4, 4, true, true, 5.70f, 0.00f, 0.373f, 0.260f, 0.091f},
    {3, 4, 5, true, true, 4.82f, 0.00f, 0.360f, 0.116f, 0.133f},
    {4, 2, 6, true, false, 5.13f, 0.00f, 0.210f, 0.151f, 0.100f},
};

// Of gate/up of up to 64 rows, which ops._tile_few names: rings of W 6 and 4 stages
// deep.  Tiles of 128 rows of W while the chip has a CU for each, then of 256 (us,
// 64 rows, 128 / 256: 28672 x 4096 43.6 / 57.7, 40960 x 4096 78 / 68).
constexpr const TileForm* TILE_FEW = TILE_FORMS + 6;

struct TilePlan {
  float time;                   // us
  const TileForm* form;
  int parts;
  const TileForm* rest;         // of the columns from `to` on; null: none
  int to;
};

// `cols` of the result, which for GLU are half of W's rows
inline float tile_time(const TileForm& f, int M, int cols, int K, int end,
                       int parts) {
  const int wide = end == TILE_GLU ? 16 * f.wn : 32 * f.wn;
  const long items = (long)((M + 32 * f.wm - 1) / (32 * f.wm)) *
                     ((cols + wide - 1) / wide) * parts;
  const long rounds = ((items + 7) / 8 + 31) / 32;
  const float stages = K / 64.f / parts;
  const float share = items / (256.f * rounds);
  const float mb = 1e-6f * M * cols * (end == TILE_PARTS ? 4.f * parts : 2.f);
  return f.fixed +
         rounds * (f.round + stages * (f.step + f.busy * share)) + f.write * mb;
}

inline bool tile_takes(const TileForm& f, int K, int end) {
  return (end == TILE_GLU ? f.glu : f.sums) && K / 64 >= f.fill;
}

inline TilePlan pick_tile(int M, int N, int K, int end) {
  const int cols = end == TILE_GLU ? N / 2 : N;
  TilePlan best{1e30f, nullptr, 1, nullptr, cols};
  auto consider = [&](const TilePlan& p) {
    if (p.time < best.time) best = p;
  };
  for (const TileForm& f : TILE_FORMS) {
    if (!tile_takes(f, K, end)) continue;
    consider({tile_time(f, M, cols, K, end, 1), &f, 1, nullptr, cols});
    // whole rounds of these tiles, and others for the columns that are left:
    // 2048 x 28672 x 4096 is 3.5 rounds, whose half takes as long as a whole
    const int wide = end == TILE_GLU ? 16 * f.wn : 32 * f.wn;
    const int down = (M + 32 * f.wm - 1) / (32 * f.wm);
    const long items = (long)down * ((cols + wide - 1) / wide);
    const int to = (int)(items / 256 * 256 / down * wide);
    if (to > 0 && to < cols && f.wm == 8 && f.wn == 8)
      for (const TileForm& r : TILE_FORMS) {
        if (!tile_takes(r, K, end)) continue;
        consider({tile_time(f, M, to, K, end, 1) +
                      tile_time(r, M, cols - to, K, end, 1),
                  &f, 1, &r, to});
      }
  }
  return best;
}

// Parts of K whose f32 sums a reader adds up, where that is faster with what it reads
// more than bf16, at 4 TB/s.  A k below 4736 of more than 256 rows stays whole: it
// stands in for a rounded product of the library, and is rounded as that is.  In parts
// it would be sooner (us with the norm, library / whole / parts: 4096 x 4096, 288 rows
// 29.4 / 28 / 24.4, 384 rows 29.6 / 33 / 27.2; 6144 x 4096, 384 rows 42 / 41 / 35), and
// ops._tile leaves the library the sizes at which the whole tiles are the slower ones.
inline TilePlan pick_tile_parts(int M, int N, int K) {
  TilePlan best = pick_tile(M, N, K, TILE_PLAIN);
  if (M > 256 && K < 4736) return best;
  // Where both are within 10% the reader gets the f32 sums, not a rounded product.  Of
  // results up to 5.25 M the model has parts of a long k too slow (whole / parts, us:
  // 288 x 10240 x 5120 59.0 / 53.4, 384 65.0 / 56.9; 800 x 6144 x 5120 67.9 / 61.6; of 82
  // sizes that this line and the one above split 0.91 of the time, 974 x 4416 x 4800
  // 49.9 / 55.8), not of larger ones (704 x 10240 x 8192 112 / 115, 768 112 / 119) nor
  // of a short k (88 x 12096 x 1024 14.9 / 16.1).
  float least = best.time;
  if (K >= 3584 && (long)M * N <= 5250000) least *= 1.1f;
  for (const TileForm& f : TILE_FORMS)
    for (int parts : {2, 3, 4, 5, 6, 8, 10, 12}) {
      const int tiles =
          ((M + 32 * f.wm - 1) / (32 * f.wm)) * ((N + 32 * f.wn - 1) / (32 * f.wn));
      // one round, which also bounds the sums (67 MB); a second of few stages costs 4 to
      // 5 us, which the above does not know (2048 x 2048, 190 rows in 320: 17, in 192: 13)
      if (tiles * parts > 256 || !tile_takes(f, K / parts, TILE_PARTS)) break;
      const float time = tile_time(f, M, N, K, TILE_PARTS, parts) +
                         (4 * parts - 2) * 2.5e-7f * M * N;
      if (time < least) {
        least = time;
        best = {time, &f, parts, nullptr, N};
      }
    }
  return best;
}

// The parts of tile_parts, for tests.
inline int64_t tile_split(int64_t M, int64_t N, int64_t K) {
  TORCH_CHECK(M >= 1 && N >= 64 && K >= 256 && M < (1 << 24) && N < (1 << 24) &&
              K < (1 << 24), "sizes");
  return pick_tile_parts((int)M, (int)N, (int)K).parts;
}

inline void check_tile(const torch::Tensor& a, const torch::Tensor& w) {
  for (const auto& t : {a, w})
    TORCH_CHECK(t.is_cuda() && t.scalar_type() == torch::kBFloat16 &&
                t.is_contiguous() && t.dim() == 2 &&
                (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0,
                "operands must be contiguous, aligned bf16 matrices on GPU");
  const int64_t M = a.size(0), K = a.size(1), N = w.size(0);
  TORCH_CHECK(w.size(1) == K, "K mismatch");
  // offsets within a tile's rows and W's halves are 32 bits, tiles' numbers too
  TORCH_CHECK(M >= 1 && N >= 64 && N % 64 == 0 && K >= 256 && K % 64 == 0 &&
              M < (1 << 24) && (N / 2 + 256) * K < (1ll << 31) &&
              ((M + 127) / 128) * ((N + 127) / 128) < (1 << 24),
              "unsupported shape");
}

inline void launch_tile_plan(const TilePlan& p, void* out, const torch::Tensor& a,
                             const torch::Tensor& w, int end) {
  const int M = a.size(0), K = a.size(1), N = w.size(0);
  const int cols = end == TILE_GLU ? N / 2 : N;
  // Workgroups begin at different k where the weights are the bound and rows of
  // A fit an L2: all rows are K apart, and in step they ask the same channels
  // (128 rows, 28672 x 4096: 57 -> 53 us).  In step they share rows of A and W,
  // which many rows need.
  const int turn = M <= 256;
  auto go = [&](const TileForm* f, int from, int to) {
    TORCH_CHECK(launch_tile_gemm(out, a.data_ptr(), w.data_ptr(), M, N, K, end,
                                 f->wm, f->wn, from, to, p.parts, turn,
                                 gemm_stream()), "no such tile");
  };
  go(p.form, 0, p.to);
  if (p.rest) go(p.rest, p.to, cols);
}

// silu(a Wg^T) * (a Wu^T), w = [Wg; Wu].
inline torch::Tensor tile_swiglu(torch::Tensor a, torch::Tensor w) {
  check_tile(a, w);
  auto c = torch::empty({a.size(0), w.size(0) / 2}, a.options());
  const TileForm* few = TILE_FEW + (w.size(0) > 32768);
  const bool takes = a.size(0) <= 64 && a.size(1) / 64 >= few->fill;
  launch_tile_plan(
      takes ? TilePlan{0.f, few, 1, nullptr, (int)(w.size(0) / 2)}
            : pick_tile(a.size(0), w.size(0), a.size(1), TILE_GLU),
      c.data_ptr(), a, w, TILE_GLU);
  return c;
}

// a W^T in bf16, or where K is split its parts' sums, f32 [parts, M, N].
inline torch::Tensor tile_parts(torch::Tensor a, torch::Tensor w) {
  check_tile(a, w);
  const int64_t M = a.size(0), N = w.size(0);
  const TilePlan p = pick_tile_parts(M, N, a.size(1));
  const bool split = p.parts > 1;
  auto c = split ? torch::empty({p.parts, M, N},
                                a.options().dtype(torch::kFloat32))
                 : torch::empty({M, N}, a.options());
  launch_tile_plan(p, c.data_ptr(), a, w, split ? TILE_PARTS : TILE_PLAIN);
  return c;
}

// a W^T in f32.
inline torch::Tensor tile_f32(torch::Tensor a, torch::Tensor w) {
  check_tile(a, w);
  const int M = a.size(0), N = w.size(0), K = a.size(1);
  auto c = torch::empty({M, N}, a.options().dtype(torch::kFloat32));
  TilePlan best{1e30f, nullptr, 1, nullptr, N};
  for (const TileForm& f : TILE_FORMS) {
    const float time = tile_time(f, M, N, K, TILE_PARTS, 1);
    if (tile_takes(f, K, TILE_PARTS) && time < best.time) best = {time, &f, 1, nullptr, N};
  }
  launch_tile_plan(best, c.data_ptr(), a, w, TILE_PARTS);
  return c;
}

// One form of the above, for tests: its number, the parts, and for a second form the
// column that it begins at.
inline torch::Tensor tile_form(torch::Tensor a, torch::Tensor w, int64_t end,
                               int64_t form, int64_t parts, int64_t rest,
                               int64_t to) {
  check_tile(a, w);
  const int64_t M = a.size(0), N = w.size(0), K = a.size(1);
  const int64_t cols = end == TILE_GLU ? N / 2 : N;
  const int64_t forms = sizeof(TILE_FORMS) / sizeof(TILE_FORMS[0]);
  TORCH_CHECK(form >= 0 && form < forms, "form");
  const TileForm* f = TILE_FORMS + form;
  TORCH_CHECK(end >= 0 && end <= TILE_GLU &&
              rest < forms && parts >= 1 && (parts == 1 || end == TILE_PARTS) &&
              K / 64 / parts >= f->fill &&
              (rest < 0 || (to > 0 && to < cols && to % 32 == 0 &&
                            K / 64 / parts >= TILE_FORMS[rest].fill)), "form");
  auto c = end == TILE_PARTS
               ? torch::empty({parts, M, N}, a.options().dtype(torch::kFloat32))
               : torch::empty({M, cols}, a.options());
  launch_tile_plan({0.f, f, (int)parts,
                    rest < 0 ? nullptr : TILE_FORMS + rest,
                    (int)(rest < 0 ? cols : to)},
                   c.data_ptr(), a, w, (int)end);
  return c;
}
