// The workgroups of prompt attention, found on the host once for all layers of a step.
//
// Before a prompt's first kernels the GPU waits for this, and a short prompt is bound
// by its host: numpy's twenty calls, each of a few numbers, and their copy to the GPU
// took 55 us of the 431 of 37 rows in six layers; that prompt 447 -> 397 us.
// ops/__init__.py has the same steps for a device that is not a GPU.
#pragma once
#include <stdint.h>

#include <algorithm>
#include <functional>
#include <numeric>
#include <queue>
#include <vector>

struct PrefillWork {
  std::vector<int32_t> blocks, lens, items, joins;    // of 4, 1, 4 and 3 numbers
  int64_t parts = 0;
};

// Blocks of so many tiles, most first, as shares of the CUs (ops/__init__.py
// _cut_prefill has the reasons and figures); false where whole blocks are as good.
inline bool cut_prefill(const std::vector<int64_t>& tiles, int64_t kv_heads,
                        PrefillWork* to) {
  const int64_t cus = std::max<int64_t>(1, 256 / kv_heads), n = tiles.size();
  if (n == 0 || n > 4 * cus) return false;
  const int64_t work = std::accumulate(tiles.begin(), tiles.end(), (int64_t)0);
  const int64_t share = std::max<int64_t>((work + cus - 1) / cus, 4);
  const double part_time = kv_heads * 0.026, tile_time = n <= cus ? 1.2 : 1.0;
  int64_t above = 0;
  for (const int64_t t : tiles) above += t > share;
  const double least = tile_time * share + 5 + part_time * 2 * above;
  double whole = 1.2 * tiles[0];
  using Heap = std::priority_queue<int64_t, std::vector<int64_t>,
                                   std::greater<int64_t>>;
  if (n > cus) {
    Heap load(std::greater<int64_t>(),
              std::vector<int64_t>(tiles.begin(), tiles.begin() + cus));
    int64_t most = tiles[0];
    for (int64_t i = cus; i < n; ++i) {
      const int64_t sum = load.top() + tiles[i];
      load.pop();
      load.push(sum);
      most = std::max(most, sum);
    }
    whole = std::max(whole, (double)most);
  }
  if (least > 0.95 * whole) return false;
  std::vector<int64_t> cut;
  std::priority_queue<int64_t> rooms;
  for (int64_t i = 0; i < cus; ++i) rooms.push(share);
  std::vector<int32_t> items, joins;
  int64_t parts = 0, longest = 0;
  const auto put = [&](int64_t b, int64_t from, int64_t end, int64_t part) {
    for (const int64_t x : {b, from, end, part}) items.push_back((int32_t)x);
    longest = std::max(longest, end - from);
  };
  for (int64_t b = 0; b < n; ++b) {
    if (tiles[b] > rooms.top()) {
      cut.push_back(b);
      continue;
    }
    const int64_t left = rooms.top() - tiles[b];
    rooms.pop();
    rooms.push(left);
    put(b, 0, tiles[b], -1);
  }
  std::vector<int64_t> room(cus);                     // the most last
  for (int64_t i = cus - 1; i >= 0; --i) {
    room[i] = rooms.top();
    rooms.pop();
  }
  const int64_t over = std::max<int64_t>(2, share / 8);
  for (const int64_t b : cut) {
    const int64_t first = parts;
    for (int64_t done = 0; done < tiles[b];) {
      int64_t take = tiles[b] - done;
      if (!room.empty() && take > room.back() + over) take = room.back();
      if (!room.empty()) {
        room.back() -= take;
        if (room.back() <= over) {
          room.pop_back();
          if (!room.empty() && room.back() <= over) room.clear();
        }
      }
      put(b, done, done + take, parts++);
      done += take;
    }
    if (parts == first + 1) {       // whole after all
      items.back() = -1;
      parts = first;
    } else {
      for (const int64_t x : {b, first, parts - first})
        joins.push_back((int32_t)x);
    }
  }
  const double cost =
      std::max(1.2 * longest, tile_time * share) + 5 + part_time * parts;
  if (joins.empty() || cost > 0.95 * whole) return false;
  to->items = std::move(items);
  to->joins = std::move(joins);
  to->parts = parts;
  return true;
}

// Most work first; where all run at once the second half the other way round
// (ops/__init__.py _turn_round).
inline void turn_round(std::vector<int64_t>* order, int64_t kv_heads) {
  const int64_t n = order->size(), half = 256 / kv_heads;
  if (n * kv_heads <= 512 && half < n)
    std::reverse(order->begin() + half, order->end());
}

// cu, cu_k: where a sequence's query and key rows begin; `tokens` of a block, 0 for
// more heads a key head than a block has rows, which has no plan.
inline PrefillWork plan_prefill(const std::vector<int64_t>& cu,
                                const std::vector<int64_t>& cu_k, int64_t tokens,
                                int64_t kv_heads) {
  struct Block { int64_t seq, nth, past, need; };
  std::vector<Block> all;
  for (size_t s = 0; s + 1 < cu.size(); ++s) {
    const int64_t rows = cu[s + 1] - cu[s], keys = cu_k[s + 1] - cu_k[s];
    for (int64_t i = 0; tokens && i * tokens < rows; ++i)
      all.push_back({(int64_t)s, i, keys - rows,
                     std::min(keys - rows + (i + 1) * tokens, keys)});
  }
  std::stable_sort(all.begin(), all.end(),
                   [](const Block& a, const Block& b) { return a.need > b.need; });
  std::vector<int64_t> tiles, order(all.size());
  for (const Block& b : all)
    tiles.push_back(b.need > 0 ? (b.need + 63) / 64 : 0);
  std::iota(order.begin(), order.end(), 0);
  PrefillWork work;
  if (cut_prefill(tiles, kv_heads, &work)) {
    const std::vector<int32_t> by_block = work.items;
    std::vector<int64_t> turn(by_block.size() / 4);
    std::iota(turn.begin(), turn.end(), 0);
    const auto length = [&](int64_t i) {
      return by_block[i * 4 + 2] - by_block[i * 4 + 1];
    };
    std::stable_sort(turn.begin(), turn.end(),
                     [&](int64_t a, int64_t b) { return length(a) > length(b); });
    turn_round(&turn, kv_heads);
    for (size_t i = 0; i < turn.size(); ++i)
      std::copy_n(&by_block[turn[i] * 4], 4, &work.items[i * 4]);
  } else {
    turn_round(&order, kv_heads);
  }
  for (const int64_t i : order) {
    const Block& b = all[i];
    for (const int64_t x : {cu[b.seq], b.nth, cu_k[b.seq], b.past})
      work.blocks.push_back((int32_t)x);
    work.lens.push_back((int32_t)(cu_k[b.seq + 1] - cu_k[b.seq]));
  }
  return work;
}
