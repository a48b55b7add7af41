// GEMM of prompts and large decode batches, C[M,N] = A[M,K] x W[N,K]^T, bf16
// in, f32 accumulators: bf16 out, f32 sums of the parts of a split K, or
// silu(A Wg^T) * (A Wu^T) where W's halves are a gate and an up matrix.
//
// Bound: the matrix cores' power.  8192 x 8192 x 4096 takes 372 us (1478
// TFLOP/s, the library 353) at 1.7 GHz, the products alone, without loads, 288;
// on 8 CUs, at 2.4 GHz, a tile of 256 x 256 takes 1.1 us per 64 k of which the
// products are 0.85.  4 waves of 128 x 128 share a tile, a workgroup to a CU:
//  * Rows come straight to LDS, 128 bytes of each, whole lines: half lines cost
//    half of L2's rate (loads alone 303 us, with whole lines 196).  A's ring is
//    one stage longer than W's, so that all 160 KB are in use.
//  * Half a stage is 64 products of 16x16x32 with the next half's fragments
//    read and later stages asked for between them, one at a time, pinned there;
//    what stands between is hidden, what stands in a row is not.  One barrier a
//    stage.  (32x32x16 moves the accumulators twice as often: 415 us.)
//  * Nothing but two pointers changes from stage to stage: with conditions and
//    addresses of the next tile in the loop it took 390 us.
//  * A workgroup goes from tile to tile without draining its loads.
//  * Stores bring whole lines of a row, four rows each: a CU stores the 16 bytes of a
//    lane in a cycle, whatever they are beside, so lanes along the rows of A took 3.4 us
//    for a tile of 256 x 256 in bf16, 6.6 of f32 sums and 3.8 behind silu, of which 1.9,
//    1.9 and 3.2 are left (128 x 128 0.8 and 1.7, now 0.5).  In all 8192 x 28672 x 4096
//    with silu 1318 -> 1258 us, 2048 rows 361 -> 342; in parts 128 x 4096 x 4096 14.8 ->
//    13.5, 256 x 4096 x 4096 22.1 -> 19.8; 1500 x 4096 x 4096 52.7 -> 51.5.
// It gains on the library by what the library does not do: silu in the product
// (8192 x 28672 x 4096 with silu 1327 us, the library and silu_mul 1463, both on a card
// that is slower than that of the figures above; 2048 rows 371 / 412), parts of a long k
// (2048 x 4096 x 14336 201 / 244 with the norm that adds them up), and tiles by the
// shape.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "mfma_util.h"

namespace {

enum TileEnd { TILE_PLAIN, TILE_PARTS, TILE_GLU };

// 16 bytes per lane from base + off to 16 * lane past the wave's LDS address.
// Not the compiler's builtin: it would wait for the data before any LDS read.
DEV_INLINE void tg_load(const uint32_t off, const void* base,
                        const uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\t"
               "global_load_lds_dwordx4 %0, %1"
               :: "v"(off), "s"(base), "s"(lds) : "memory", "m0");
}

// By a reciprocal: a division's ten instructions for 128 values a lane took 3% of a
// product of 4096 k.  Its error against 64 bits is the same to 8 digits (0.00165792,
// 8192 x 28672 x 4096; ten other shapes).  Of a quarter of the divisor, which is a
// normal number for any finite exponential, as is its reciprocal: those of gates
// below -87.3 came out as 0 (0.3% more time, the others the same).
DEV_INLINE float tg_silu(float g) {
  return 0.25f * g *
         __builtin_amdgcn_rcpf(__builtin_fmaf(0.25f, __expf(-g), 0.25f));
}

template <class F, int... I>
DEV_INLINE void tg_each_of(F f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
// f of 0 .. N - 1 as constants: arrays that they index stay in registers
template <int N, class F>
DEV_INLINE void tg_each(F f) {
  tg_each_of(f, std::make_integer_sequence<int, N>());
}

// A lane's values in one store, at a multiple of their size.
template <int N, class T>
DEV_INLINE void tg_put(const T (&v)[N], char* to) {
  __builtin_memcpy(__builtin_assume_aligned(to, sizeof(v)), v, sizeof(v));
}

// Is k the place of the q-th of n things spread over [0, to)?  Not the first:
// products go first after a barrier.
constexpr bool tg_due(int q, int n, int to, int k) {
  return ((q + 1) * to + n - 1) / n - 1 == k;
}

struct TileMap {
  int rows, cols, items;        // tiles down and across; times parts
  int parts, group;             // tiles of `group` rows of tiles go column by
                                // column: what runs at a time shares rows
  int from, to;                 // columns of the result
  int turn;                     // workgroups begin at different k
};

// Tiles of 32 WM rows and 32 WN rows of W, NA and NW stages of 64 k in LDS.
template <int WM, int WN, int NA, int NW, int END>
__global__ __launch_bounds__(256, 1) void tile_gemm_kernel(
    const __hip_bfloat16* __restrict__ a,   // [M, K]
    const __hip_bfloat16* __restrict__ w,   // [N, K]
    void* __restrict__ out,                 // [M, N], GLU: [M, N / 2], PARTS:
                                            // f32 [parts, M, N]
    const int M, const int N, const int K, const TileMap map) {
  // columns beside one another in as many fragments of W, a lane's for one store: 16
  // lanes have 64 to 256 bytes of a row
  constexpr int NEAR = END == TILE_GLU ? WN / 2 : WN % 4 == 0 ? 4 : 2;
  static_assert(WN % 2 == 0 && (END != TILE_GLU || WN % 4 == 0 && WN <= 8),
                "fragments in groups");
  constexpr int BM = 32 * WM, BN = 32 * WN, AB = BM * 128, WB = BN * 128;
  constexpr int COLS = END == TILE_GLU ? BN / 2 : BN;
  constexpr int S = WM * WN, READS = WM + WN;
  constexpr int FILL = std::max(NA - 1, NW);      // fewest stages of an item
  // loads younger than those of the next stage when it has to be there
  constexpr int FLY = std::min((NA - 2) * (WM + WN),
                               (NW - 1) * WM + (NW - 2) * WN);
  extern __shared__ __align__(16) char tg_lds[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)tg_lds;
  // workgroup i runs on XCD i % 8: each takes an eighth of the tiles, in order
  const int xcd = blockIdx.x & 7, per = (gridDim.x + 7 - xcd) >> 3;
  const int hi = (int)((long)map.items * (xcd + 1) / 8);
  int item = (int)((long)map.items * xcd / 8) + (blockIdx.x >> 3);
  if (item >= hi) return;
  const int last = item + (hi - 1 - item) / per * per;

  struct Tile { int m0, n0, c0, n, part; };
  const int tiles = map.rows * map.cols;
  auto locate = [&](int it) {
    Tile t;
    t.part = it / tiles;
    const int r = it - t.part * tiles, full = map.group * map.cols;
    const int g = r / full, in = r - g * full;
    const int rows = min(map.group, map.rows - g * map.group);
    t.m0 = (g * map.group + in % rows) * BM;
    t.n0 = map.from + in / rows * COLS;
    const int stages = K / 64;
    t.c0 = stages * t.part / map.parts;
    t.n = stages * (t.part + 1) / map.parts - t.c0;
    return t;
  };
  // what is loaded, ahead of what is used.  A load brings 8 rows; the piece of
  // 16 bytes at place p of row r is p ^ (r / 2 % 8): no bank conflicts.
  const int piece = ((lane & 7) ^ ((wave & 1) * 4 + (lane >> 4))) * 16;
  int a_item = item, a_n, w_item = item, w_n;
  const char *ab, *wb;
  uint32_t ao[WM], wo[WN];
  auto a_rows = [&]() {
    const Tile t = locate(a_item);
    a_n = t.n;
    ab = (const char*)(a + (size_t)t.m0 * K + t.c0 * 64);
#pragma unroll
    for (int c = 0; c < WM; ++c)
      ao[c] = (uint32_t)min((c * 4 + wave) * 8 + (lane >> 3), M - 1 - t.m0) *
                  (uint32_t)(K * 2) + piece;
  };
  auto w_rows = [&]() {
    const Tile t = locate(w_item);
    w_n = t.n;
    wb = (const char*)(w + (size_t)t.n0 * K + t.c0 * 64);
#pragma unroll
    for (int c = 0; c < WN; ++c) {
      // row r of the tile's W: fragment j of its wave has columns NEAR r + j % NEAR
      const int r = (c * 4 + wave) * 8 + (lane >> 3);
      const int j = r / 16 % WN, at = r / (16 * WN) * WN;
      int n = (at + j / NEAR * NEAR) * 16 + r % 16 * NEAR + j % NEAR;
      if (END == TILE_GLU)        // the gate's fragments, then the up matrix's
        n = min(at * 8 + r % 16 * NEAR + j % NEAR, map.to - 1 - t.n0) +
            j / NEAR * (N / 2);
      else
        n = min(n, map.to - 1 - t.n0);
      wo[c] = (uint32_t)n * (uint32_t)(K * 2) + piece;
    }
  };
  // A turn: from there to the end, then from the beginning.  Past the last item
  // that one is loaded again, to no use.
  auto turn = [&](int n) {
    return map.turn
        ? min(((int)(blockIdx.x >> 3) * 5 + xcd * 3) % n, n - FILL) : 0;
  };
  a_rows();
  w_rows();
  int a_turn = turn(a_n), w_turn = turn(w_n);
  int a_left = a_n - a_turn, w_left = w_n - w_turn;
  ab += a_turn * 128;
  wb += w_turn * 128;
#define TG_A_ON(steps)                                                     \
  if ((a_left -= (steps)) == 0) {                                          \
    const bool again = a_turn > 0;                                         \
    if (!again) {                                                           \
      a_item = min(a_item + per, last);                                    \
      a_rows();                                                            \
    }                                                                      \
    const int t_ = again ? 0 : turn(a_n);                                  \
    ab += (again ? -a_n : t_) * 128;                                       \
    a_left = again ? a_turn : a_n - t_;                                    \
    a_turn = t_;                                                           \
  }
#define TG_W_ON(steps)                                                     \
  if ((w_left -= (steps)) == 0) {                                          \
    const bool again = w_turn > 0;                                         \
    if (!again) {                                                           \
      w_item = min(w_item + per, last);                                    \
      w_rows();                                                            \
    }                                                                      \
    const int t_ = again ? 0 : turn(w_n);                                  \
    wb += (again ? -w_n : t_) * 128;                                       \
    w_left = again ? w_turn : w_n - t_;                                    \
    w_turn = t_;                                                           \
  }
  const uint32_t al = lds0 + wave * 1024, wl = lds0 + NA * AB + wave * 1024;
#pragma unroll
  for (int s = 0; s < FILL; ++s) {
    if (s < NA - 1) {
#pragma unroll
      for (int c = 0; c < WM; ++c)
        tg_load(ao[c], ab + s * 128, al + s * AB + c * 4096);
    }
    if (s < NW) {
#pragma unroll
      for (int c = 0; c < WN; ++c)
        tg_load(wo[c], wb + s * 128, wl + s * WB + c * 4096);
    }
  }
  ab += (NA - 1) * 128;
  wb += NW * 128;
  TG_A_ON(NA - 1)
  TG_W_ON(NW)

  const int g = lane >> 4;
  int af[2], wf[2];             // a fragment of half h: 32 k of 16 rows
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int at = (lane & 15) * 128 + ((4 * h + g) ^ ((lane >> 1) & 7)) * 16;
    af[h] = wm * WM * 2048 + at;
    wf[h] = NA * AB + wn * WN * 2048 + at;
  }
  mf_bf8 fa[2][WM], fw[2][WN];
  f32x4 acc[WM][WN];
  int a_at = 0, w_at = 0;       // the stage in use
  auto read = [&](auto h, auto q) {
    if constexpr (q < WN)
      fw[h][q] = frag8((const __hip_bfloat16*)(tg_lds + w_at + wf[h] +
                                               q * 2048));
    else
      fa[h][q - WN] = frag8((const __hip_bfloat16*)(tg_lds + a_at + af[h] +
                                                    (q - WN) * 2048));
  };
  constexpr std::integral_constant<int, 0> H0{};
  constexpr std::integral_constant<int, 1> H1{};
  // one half's products, with R reads and L loads between them
  constexpr int PLACES = S - S / 6;
  auto half = [&](auto h, auto loads, auto load, auto next) {
    constexpr int L = decltype(loads)::value, T = READS + L;
    constexpr int H = decltype(h)::value;
    tg_each<S>([&](auto kk) {
      constexpr int k = decltype(kk)::value;
      acc[k / WN][k % WN] = mfma_bf16_k32(fa[H][k / WN], fw[H][k % WN],
                                          acc[k / WN][k % WN]);
      __builtin_amdgcn_sched_barrier(0);
      tg_each<T>([&](auto qq) {
        constexpr int q = decltype(qq)::value;
        if constexpr (tg_due(q, T, PLACES, k)) {
          constexpr int l = q * L / T;
          if constexpr (l != (q + 1) * L / T)
            load(l);
          else
            read(std::integral_constant<int, 1 - H>(),
                 std::integral_constant<int, q - l>());
        }
      });
      if constexpr (k == PLACES) next();
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier"
               :: "n"((NA - 2) * WM + (NW - 1) * WN) : "memory");
  tg_each<READS>([&](auto q) { read(H0, q); });
  uint32_t a_to = al + (NA - 1) * AB;
  for (; item < hi; item += per) {
    const Tile t = locate(item);
    int left = t.n;
#pragma unroll
    for (int f = 0; f < WM; ++f)
#pragma unroll
      for (int j = 0; j < WN; ++j) acc[f][j] = {0.f, 0.f, 0.f, 0.f};
    while (left > 0) {
      const int run = min(left, min(a_left, w_left));
      uint32_t w_to = 0;
      int a_new = 0, w_new = 0;
      for (int s = 0; s < run; ++s) {
        half(H0, std::integral_constant<int, WM>(),
             [&](int l) { tg_load(ao[l], ab, a_to + l * 4096); },
             [&]() {
               ab += 128;
               a_to = al + a_at;
               w_to = wl + w_at;
               a_new = a_at == (NA - 1) * AB ? 0 : a_at + AB;
               w_new = w_at == (NW - 1) * WB ? 0 : w_at + WB;
             });
        // this stage is read, the next is there
        asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier"
                     :: "n"(FLY) : "memory");
        a_at = a_new;
        w_at = w_new;
        half(H1, std::integral_constant<int, WN>(),
             [&](int l) { tg_load(wo[l], wb, w_to + l * 4096); },
             [&]() { wb += 128; });
      }
      left -= run;
      TG_A_ON(run)
      TG_W_ON(run)
    }

    // lane l: rows 4g.. of a fragment of A, row l & 15 of W's
    constexpr int STEP = END == TILE_GLU ? WN : NEAR;
    constexpr uint32_t ES = END == TILE_PARTS ? 4 : 2;
    const uint32_t pitch = (END == TILE_GLU ? N / 2 : N) * ES;
    const int m = t.m0 + wm * WM * 16, n = t.n0 + wn * (COLS / 2);
    tg_each<WN / STEP>([&](auto jj) {
      constexpr int j = decltype(jj)::value * STEP;
      const int col = j * 16 + (lane & 15) * NEAR;
      if (n + col >= map.to) return;
      uint32_t at[4];
#pragma unroll
      for (int q = 0; q < 4; ++q) at[q] = (g * 4 + q) * pitch + col * ES;
      char* to = (char*)out + ((size_t)t.part * M + m) * pitch + n * ES;
      tg_each<WM>([&](auto ff) {
        constexpr int f = decltype(ff)::value;
        const int left = M - m - f * 16;
        __builtin_amdgcn_sched_barrier(0);
        if (left <= 0) return;
        if (left < 16) {        // rows past the last are that one once more
#pragma unroll
          for (int q = 0; q < 4; ++q)
            at[q] = min(g * 4 + q, left - 1) * pitch + col * ES;
        }
#pragma unroll
        for (int i = 0; i < STEP; ++i) asm volatile("" : "+a"(acc[f][j + i]));
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          float v[NEAR];
          __hip_bfloat16 o[NEAR];
#pragma unroll
          for (int i = 0; i < NEAR; ++i) {
            v[i] = acc[f][j + i][q];
            if constexpr (END == TILE_GLU)
              v[i] = tg_silu(v[i]) * acc[f][j + NEAR + i][q];
            o[i] = f2bf(v[i]);
          }
          if constexpr (END == TILE_PARTS)
            tg_put(v, to + at[q]);
          else
            tg_put(o, to + at[q]);
        }
        to += 16 * (size_t)pitch;
      });
    });
  }
#undef TG_A_ON
#undef TG_W_ON
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // LDS is in use until then
}

template <int WM, int WN, int NA, int NW, int END>
void launch_tile(void* out, const void* a, const void* w, int M, int N, int K,
                 int from, int to, int parts, int turn, hipStream_t stream) {
  constexpr int lds = (NA * WM + NW * WN) * 32 * 128;
  static_assert(lds <= 160 * 1024, "LDS of a CU");
  (void)hipFuncSetAttribute(
      (const void*)tile_gemm_kernel<WM, WN, NA, NW, END>,
      hipFuncAttributeMaxDynamicSharedMemorySize, lds);
  constexpr int COLS = END == TILE_GLU ? 16 * WN : 32 * WN;
  TileMap map;
  map.rows = (M + 32 * WM - 1) / (32 * WM);
  map.cols = (to - from + COLS - 1) / COLS;
  map.parts = parts;
  map.items = map.rows * map.cols * parts;
  map.group = 8;
  map.from = from;
  map.to = to;
  map.turn = turn;
  const int grid = std::min(256, (map.items + 7) / 8 * 8);
  tile_gemm_kernel<WM, WN, NA, NW, END><<<dim3(grid), dim3(256), lds, stream>>>(
      (const __hip_bfloat16*)a, (const __hip_bfloat16*)w, out, M, N, K, map);
}

}  // namespace

// Columns [from, to) of the result; wm and wn choose the tile.  0: no such form.
extern "C" int launch_tile_gemm(void* out, const void* a, const void* w, int M,
                                int N, int K, int end, int wm, int wn, int from,
                                int to, int parts, int turn,
                                hipStream_t stream) {
#define TG_GO(WM, WN, NA, NW, END)                                         \
  if (wm == WM && wn == WN && end == END) {                                \
    launch_tile<WM, WN, NA, NW, END>(out, a, w, M, N, K, from, to, parts,  \
                                     turn, stream);                        \
    return 1;                                                              \
  }
#define TG_ENDS(WM, WN, NA, NW)                                            \
  TG_GO(WM, WN, NA, NW, TILE_PLAIN)                                        \
  TG_GO(WM, WN, NA, NW, TILE_PARTS)                                        \
  TG_GO(WM, WN, NA, NW, TILE_GLU)
  TG_ENDS(8, 8, 3, 2)
  TG_ENDS(7, 8, 3, 2)
  TG_ENDS(6, 8, 3, 2)
  TG_ENDS(5, 8, 3, 3)
  TG_GO(8, 6, 3, 2, TILE_PLAIN)
  TG_GO(8, 6, 3, 2, TILE_PARTS)
  TG_GO(6, 6, 3, 3, TILE_PLAIN)
  TG_GO(6, 6, 3, 3, TILE_PARTS)
  TG_ENDS(8, 4, 3, 3)
  TG_ENDS(5, 4, 4, 4)
  TG_ENDS(4, 4, 5, 4)
  TG_ENDS(3, 4, 6, 5)
  TG_GO(4, 2, 7, 6, TILE_PLAIN)
  TG_GO(4, 2, 7, 6, TILE_PARTS)
  TG_GO(2, 4, 6, 6, TILE_GLU)
  TG_GO(2, 8, 4, 4, TILE_GLU)
#undef TG_ENDS
#undef TG_GO
  return 0;
}
