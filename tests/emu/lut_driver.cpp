// The cell table against a binary search over the range starts: keys at and
// beside every start, past the ends of every table and random ones, for start
// lists that fill the level-2 and level-3 tables, run out of them or have none.
#pragma GCC optimize("no-thread-jumps", "no-tree-dominator-opts", "no-tree-vrp", "no-tree-ch", "no-split-paths", \
                     "no-unswitch-loops", "no-split-loops", "no-tree-pre", "no-tree-loop-distribution", "no-ipa-cp")
#include "hip/hip_runtime.h"
#include <algorithm>
#include <atomic>
#include <random>
#include <vector>
#include "select_kernels.hpp"
using namespace ggms;

template <class F> void launch(F&& f) {
  blockDim = dim3(1024);
  g_bar.reset(1024);
  std::vector<std::thread> th;
  for (uint32_t t = 0; t < 1024; ++t) th.emplace_back([&, t] { threadIdx = dim3(t); f(t); g_bar.exit_thread(); });
  for (auto& t : th) t.join();
}

// clusters of `per` starts within 2^spread keys, spread evenly over the window
template <class K> int run(const char* name, uint32_t clusters, uint32_t per, uint32_t spread, bool win, uint64_t seed) {
  using G = LutGeom<K>;
  std::mt19937_64 rng(seed);
  const uint32_t wsh = win ? G::S1 - 8 : G::S1;
  const K wbase = win ? (K)((K)0x5 << (G::KB - 4)) : (K)0;
  const K width = wsh >= G::S1 ? KeyMax<K>::v : (K)(((K)G::L1CELLS << wsh) - 1);
  std::vector<K> starts{0, wbase, KeyMax<K>::v, (K)(wbase + width)};
  for (uint32_t c = 0; c < clusters; ++c) {
    const K at = c + 1 == clusters && !win ? (K)(KeyMax<K>::v - ((K)1 << spread) + 1)
                                           : (K)(wbase + width / clusters * c + (K)rng() % 1000);
    for (uint32_t i = 0; i < per; ++i) starts.push_back((K)(at + ((K)rng() & (((K)1 << spread) - 1))));
  }
  std::sort(starts.begin(), starts.end());
  starts.erase(std::unique(starts.begin(), starts.end()), starts.end());
  const uint32_t R = (uint32_t)starts.size();
  std::vector<uint64_t> lut_mem(G::kEntries + 2);
  std::vector<uint64_t> params(Pass0Map<K>::param_bytes(R) / 8 + 2);
  Pass0Map<K> mp;
  mp.lut = reinterpret_cast<K*>(((uintptr_t)lut_mem.data() + 15) & ~(uintptr_t)15);
  mp.set_params(reinterpret_cast<unsigned char*>(params.data()), R);
  for (uint32_t r = 0; r < R; ++r) {
    MapParam<K> q{};  // bucket = range
    q.lo = starts[r];
    q.base = r;
    q.mult = 1;
    q.sh = sizeof(K) == 8 ? 32 : 0;
    mp.store_param(r, q);
  }
  mp.wbase = wbase;
  mp.wsh = wsh;
  mp.wmax = width;
  auto of = [&](K k) { return (uint32_t)(std::upper_bound(starts.begin(), starts.end(), k) - starts.begin()) - 1; };
  mp.r_below = wbase ? of((K)(wbase - 1)) : 0;
  mp.r_above = (K)(wbase + width) < KeyMax<K>::v ? of((K)(wbase + width + 1)) : R - 1;
  std::vector<uint32_t> l2(1024);
  launch([&](uint32_t t) { l2[t] = build_lut<K>(starts.data(), R, mp.lut, wbase, wsh); });
  std::vector<K> keys{0, KeyMax<K>::v};
  for (K s : starts)
    for (int d = -2; d <= 2; ++d) keys.push_back((K)(s + (K)d));
  for (K s : starts)
    for (int i = 0; i < 8; ++i) keys.push_back((K)(s + ((K)rng() & (((K)2 << (rng() % (spread + 2))) - 1))));
  while (keys.size() < 20000 || keys.size() % 4096) keys.push_back((K)rng());
  std::atomic<uint32_t> bad{0};
  launch([&](uint32_t t) {
    for (size_t i = 0; i < keys.size(); i += 4096) {
      K k[4];
      uint32_t b[4];
      for (int j = 0; j < 4; ++j) k[j] = keys[i + t * 4 + j];
      if (win) mp.template buckets<4, true>(k, b);
      else mp.template buckets<4, false>(k, b);
      const uint32_t one = win ? mp.template range_of<true>(k[0]) : mp.template range_of<false>(k[0]);
      for (int j = 0; j < 4; ++j) bad += b[j] != of(k[j]);
      bad += one != of(k[0]);
    }
  });
  uint32_t deep = 0, search = 0;
  for (uint32_t i = 0; i < G::L1CELLS + l2[0] * 64; ++i)
    if ((mp.lut[i] & G::FLAG) && !(mp.lut[i] & G::TABLE)) ((mp.lut[i] & G::DEEP) ? deep : search) += 1;
  for (uint32_t t = 1; t < 1024; ++t) bad += l2[t] != l2[0];
  printf("%s: R %u tables %u level-3 %u search %u bad %u %s\n", name, R, l2[0], deep, search, bad.load(),
         bad.load() ? "FAILED" : "ok");
  return bad.load() ? 1 : 0;
}

template <class K> int all(const char* t) {
  int rc = 0;
  constexpr uint32_t s2 = LutGeom<K>::S2;
  printf("%s\n", t);
  rc |= run<K>("no cluster", 1, 1, 4, false, 1);
  rc |= run<K>("narrow clusters", 5, 17, s2 - 4, false, 2);
  rc |= run<K>("as wide as a sub-cell", 6, 40, s2, false, 3);
  rc |= run<K>("neighbouring keys", 4, 30, 6, false, 4);
  rc |= run<K>("out of tables", 60, 12, s2 - 2, false, 5);
  rc |= run<K>("few starts each", 19, 2, s2 - 5, false, 6);
  rc |= run<K>("windowed", 5, 17, s2 - 10, true, 7);
  rc |= run<K>("windowed, out of tables", 50, 9, s2 - 9, true, 8);
  return rc;
}

int main() { return all<uint32_t>("u32") | all<uint64_t>("u64"); }
