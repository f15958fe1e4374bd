// k_plan_reg against k_plan: the same histogram, ranges and ks through both;
// every table, control block and answer has to agree (the k lists and the
// finish order up to the order inside a segment and a size class).
// One copy of every wave operation: the emulation tells the operations of a
// wave apart by their call sites, which these passes would duplicate.
#pragma GCC optimize("no-thread-jumps", "no-tree-dominator-opts", "no-tree-vrp", "no-tree-ch", "no-split-paths", \
                     "no-unswitch-loops", "no-split-loops", "no-tree-pre", "no-tree-loop-distribution", "no-ipa-cp")
#include "hip/hip_runtime.h"
#include <algorithm>
#include <random>
#include <vector>
#include "select_kernels.hpp"
using namespace ggms;

template <class T> struct Tables {
  using K = typename KeyTraits<T>::K;
  std::vector<uint32_t> totals, k_rank, k_state, k_aux, slot_dst, slot_bucket, act_bucket, act_cls, act_cnt, act_dst,
      act_slot, small_start, small_len, small_kstart, small_order, klist, wg, grp_cursor, grp_start;
  std::vector<uint16_t> slot_of_bucket;
  std::vector<K> act_klo, act_khi, small_klo, small_khi;
  std::vector<Range<K>> ranges, next_ranges;
  std::vector<MapParam<K>> next_params;
  std::vector<uint64_t> rank_words;
  std::vector<T> out;
  PassCtl ctl{}, ctl_next{}, mirror[2]{};
  uint32_t seq = 0, nan = 0;
};

template <class F> void launch(size_t lds, F&& f) {
  std::vector<unsigned char> mem(lds + 16, 0xA5);
  g_dyn_smem = reinterpret_cast<unsigned char*>((reinterpret_cast<uintptr_t>(mem.data()) + 15) & ~(uintptr_t)15);
  blockDim = dim3(1024);
  g_bar.reset(1024);
  std::vector<std::thread> th;
  for (uint32_t t = 0; t < 1024; ++t) th.emplace_back([&, t] { threadIdx = dim3(t); f(); g_bar.exit_thread(); });
  for (auto& t : th) t.join();
}

struct Form {
  uint32_t B, R, nk, fin_cap, finish_cap;
  bool merge, force, groups, mirror, dead;
};

template <class T, uint32_t KPT> int run(const char* name, const Form& f, uint64_t seed) {
  using K = typename KeyTraits<T>::K;
  std::mt19937_64 rng(seed);
  Tables<T> in;
  // ranges: a partition of the key space, some one key wide
  std::vector<K> starts{0};
  while (starts.size() < f.R) {
    K v = (K)rng();
    starts.push_back(v);
    if (rng() % 4 == 0 && v != KeyMax<K>::v) starts.push_back((K)(v + 1));
  }
  std::sort(starts.begin(), starts.end());
  starts.erase(std::unique(starts.begin(), starts.end()), starts.end());
  const uint32_t R = (uint32_t)starts.size();
  uint32_t B = 0;
  for (uint32_t r = 0; r < R; ++r) {
    Range<K> g{};
    g.lo = starts[r];
    g.hi = r + 1 < R ? (K)(starts[r + 1] - 1) : KeyMax<K>::v;
    make_map<K>(g, std::max<uint32_t>(1, f.B / R + (uint32_t)(rng() % 3)));
    g.base = B;
    B += g.nb;
    in.ranges.push_back(g);
  }
  const uint32_t Bm = (B + 64 + 7) / 8 * 8, Rm = std::max(Bm, f.nk) + 64;
  in.totals.assign(Bm, 0xDEADu);  // room past B holds garbage
  uint64_t n = 0;
  for (uint32_t b = 0; b < B; ++b) {
    uint32_t c = rng() % 3 == 0 ? 0u : (uint32_t)(rng() % 40);
    if (rng() % 50 == 0) c = (uint32_t)(rng() % 60000);
    in.totals[b] = c;
    n += c;
  }
  if (n == 0) in.totals[0] = (uint32_t)(n = 1);
  in.ctl.n = (uint32_t)n;
  in.ctl.R = R;
  in.ctl.B = B;
  in.ctl.tile = 64;
  in.ctl.G = 1;
  in.ctl.append = 5;
  in.ctl.nan_lo_bucket = f.merge ? 0u : kNone32;
  in.ctl.nan_hi_bucket = f.merge ? B - 1 : kNone32;
  in.k_rank.resize(f.nk);
  in.k_state.resize(f.nk);
  for (uint32_t k = 0; k < f.nk; ++k) {
    in.k_rank[k] = 1 + (uint32_t)(rng() % n);
    if (k && rng() % 5 == 0) in.k_rank[k] = in.k_rank[rng() % k];
    in.k_state[k] = f.dead && rng() % 3 == 0 ? (uint32_t)(rng() % 2 ? kDone : kSmall) : (uint32_t)kLive;
  }
  in.k_aux.assign(f.nk, 77);
  auto fill = [&](auto& v, size_t m) { v.resize(m); memset((void*)v.data(), 0x5A, m * sizeof(v[0])); };
  fill(in.slot_dst, Rm); fill(in.slot_bucket, Rm); fill(in.act_bucket, Rm); fill(in.act_cls, Rm); fill(in.act_cnt, Rm);
  fill(in.act_dst, Rm); fill(in.act_slot, Rm); fill(in.small_start, Rm); fill(in.small_len, Rm); fill(in.small_kstart, Rm);
  fill(in.small_order, Rm); fill(in.klist, f.nk); fill(in.wg, 600); fill(in.grp_cursor, 300); fill(in.grp_start, 300);
  fill(in.slot_of_bucket, Bm); fill(in.act_klo, Rm); fill(in.act_khi, Rm); fill(in.small_klo, Rm); fill(in.small_khi, Rm);
  fill(in.next_ranges, Rm); fill(in.next_params, Rm); fill(in.rank_words, rank_word_count(Bm)); fill(in.out, f.nk);
  Tables<T> x = in, y = in;
  auto args = [&](Tables<T>& v) {
    PlanArgs<K> a{};
    a.totals = v.totals.data(); a.ranges = v.ranges.data(); a.ctl = &v.ctl; a.ctl_next = &v.ctl_next;
    a.next_ranges = v.next_ranges.data(); a.nk = f.nk; a.k_rank = v.k_rank.data(); a.k_state = v.k_state.data();
    a.k_aux = v.k_aux.data(); a.slot_of_bucket = v.slot_of_bucket.data(); a.slot_dst = v.slot_dst.data();
    a.slot_bucket = v.slot_bucket.data(); a.act_bucket = v.act_bucket.data(); a.act_cls = v.act_cls.data();
    a.act_cnt = v.act_cnt.data(); a.act_dst = v.act_dst.data(); a.act_slot = v.act_slot.data();
    a.act_klo = v.act_klo.data(); a.act_khi = v.act_khi.data(); a.small_start = v.small_start.data();
    a.small_len = v.small_len.data(); a.small_klo = v.small_klo.data(); a.small_khi = v.small_khi.data();
    a.small_kstart = v.small_kstart.data(); a.small_order = v.small_order.data(); a.klist = v.klist.data();
    a.wg_first_next = v.wg.data(); a.out = v.out.data(); a.fin_cap = f.fin_cap; a.finish_cap = f.finish_cap;
    a.B_req = 14336; a.B_cap = 16384; a.G_max = 512; a.min_tile = 4096; a.force_finish = f.force; a.merge_small = f.merge;
    a.next_params = f.merge ? v.next_params.data() : nullptr;
    a.rank_words = f.merge ? v.rank_words.data() : nullptr;
    a.mirror = f.mirror ? v.mirror : nullptr; a.mirror_seq = &v.seq; a.seq = 9;
    a.nan_out = f.merge ? &v.nan : nullptr;
    a.grp_cursor = f.groups ? v.grp_cursor.data() : nullptr;
    a.grp_start = f.groups ? v.grp_start.data() : nullptr;
    return a;
  };
  PlanArgs<K> ax = args(x), ay = args(y);
  const size_t lds0 = (size_t)B * 8 + (size_t)rank_word_count(B) * 8 + ((size_t)std::min(f.nk, B) + 1) * 4;
  ax.lds_words = (uint32_t)(lds0 / 4);
  launch(lds0, [&] { k_plan<T>(ax); });
  const uint32_t Bb = B + (uint32_t)(rng() % 9), Rb = R + (uint32_t)(rng() % 3);  // bounds, as the host passes them
  launch(plan_reg_lds_bytes(Bb, Rb, KPT), [&] { k_plan_reg<T, KPT>(ay, Bb, Rb); });

  int bad = 0;
  auto same = [&](const char* what, const auto& p, const auto& q, size_t m) {
    if (m && memcmp(p.data(), q.data(), m * sizeof(p[0]))) { printf("  %s differs\n", what); bad++; }
  };
  if (memcmp(&x.ctl, &y.ctl, sizeof(PassCtl)) || memcmp(&x.ctl_next, &y.ctl_next, sizeof(PassCtl))) { printf("  control blocks differ\n"); bad++; }
  if (memcmp(x.mirror, y.mirror, sizeof(x.mirror)) || x.seq != y.seq || x.nan != y.nan) { printf("  mirror differs\n"); bad++; }
  const uint32_t Ub = x.ctl.U_big, Us = x.ctl.U_small, slots = Ub + Us;
  same("slot_of_bucket", x.slot_of_bucket, y.slot_of_bucket, B);
  same("slot_dst", x.slot_dst, y.slot_dst, slots);
  same("slot_bucket", x.slot_bucket, y.slot_bucket, slots);
  same("small_start", x.small_start, y.small_start, Us);
  same("small_len", x.small_len, y.small_len, Us);
  same("small_klo", x.small_klo, y.small_klo, Us);
  same("small_khi", x.small_khi, y.small_khi, Us);
  same("small_kstart", x.small_kstart, y.small_kstart, Us + 1);
  same("out", x.out, y.out, f.nk);
  for (uint32_t k = 0; k < f.nk; ++k)  // the rank of an answered k is not read again
    if (x.k_state[k] != kDone && x.k_rank[k] != y.k_rank[k]) { printf("  rank of k %u differs\n", k); bad++; break; }
  same("k_state", x.k_state, y.k_state, f.nk);
  same("wg_first", x.wg, y.wg, x.ctl_next.G);
  if (f.merge) { same("rank_words", x.rank_words, y.rank_words, rank_word_count(B)); }
  for (uint32_t j = 0; j < Ub; ++j) {
    const auto &p = x.next_ranges[j], &q = y.next_ranges[j];
    if (p.lo != q.lo || p.hi != q.hi || p.base != q.base || p.nb != q.nb || p.sh != q.sh || p.mult != q.mult ||
        p.seg_start != q.seg_start || p.seg_end != q.seg_end) { printf("  next range %u differs\n", j); bad++; break; }
    if (f.merge) {
      const auto &a = x.next_params[j], &b = y.next_params[j];
      if (a.lo != b.lo || a.base != b.base || a.mult != b.mult || a.sh != b.sh) { printf("  next param %u differs\n", j); bad++; break; }
    }
  }
  if (f.groups) {
    const uint32_t ng = (slots + kGroupSlots - 1) / kGroupSlots;
    same("grp_start", x.grp_start, y.grp_start, ng + 1);
    same("grp_cursor", x.grp_cursor, y.grp_cursor, ng);
  }
  for (uint32_t j = 0; j < Us && !bad; ++j) {
    const uint32_t q0 = x.small_kstart[j], q1 = x.small_kstart[j + 1];
    std::vector<uint32_t> p(x.klist.begin() + q0, x.klist.begin() + q1), q(y.klist.begin() + q0, y.klist.begin() + q1);
    std::sort(p.begin(), p.end());
    std::sort(q.begin(), q.end());
    if (p != q) { printf("  k list of segment %u differs\n", j); bad++; }
  }
  auto bin = [&](uint32_t j) {
    return order_bin<K>(x.small_len[j], x.small_klo[j], x.small_khi[j], f.fin_cap, x.small_kstart[j + 1] - x.small_kstart[j],
                        Us >= kFinishWaveMinSegs);
  };
  std::vector<uint32_t> po, qo;
  for (uint32_t j = 0; j < Us && !bad; ++j) {
    if (y.small_order[j] >= Us || bin(x.small_order[j]) != bin(y.small_order[j])) { printf("  finish order %u differs\n", j); bad++; }
    po.push_back(x.small_order[j]);
    qo.push_back(y.small_order[j]);
  }
  std::sort(po.begin(), po.end());
  std::sort(qo.begin(), qo.end());
  if (po != qo) { printf("  finish order is no permutation\n"); bad++; }
  printf("%s KPT %u: B %u R %u nk %u: U %u big %u small %u %s\n", name, KPT, B, R, f.nk, x.ctl.U, Ub, Us, bad ? "FAIL" : "ok");
  return bad ? 1 : 0;
}

int main() {
  int bad = 0;
  //                       B      R    nk    fin    finish  merge  force  groups mirror dead
  const Form merged{14336, 20, 1001, 32768, 32768, true, false, false, true, false};
  const Form seg{14336, 20, 1001, 4096, 4096, false, false, true, true, false};
  bad += run<float, 1>("merged", merged, 1);
  bad += run<double, 1>("merged f64", merged, 2);
  bad += run<float, 1>("segmented", seg, 3);
  bad += run<double, 8>("segmented f64", {16384, 130, 8192, 16384, 16384, false, false, true, true, false}, 4);
  bad += run<float, 8>("many ks", {16384, 130, 8192, 32768, 32768, false, false, true, true, false}, 5);
  bad += run<float, 8>("merged many", {14336, 17, 3500, 32768, 32768, true, false, false, false, false}, 6);
  bad += run<float, 8>("later pass", {16000, 3000, 8001, 4096, 4096, false, false, false, true, true}, 7);
  bad += run<float, 8>("last pass", {9000, 300, 1025, 4096, 4096, false, true, false, true, true}, 8);
  bad += run<uint32_t, 1>("few buckets", {16, 3, 1024, 500, 500, false, false, true, true, false}, 9);
  bad += run<int32_t, 1>("one k", {2, 1, 1, 32768, 32768, true, false, false, true, false}, 10);
  bad += run<float, 1>("no live ks", {1000, 5, 40, 64, 64, false, false, true, true, true}, 11);
  bad += run<float, 1>("most ranges", {20000, 1000, 1024, 64, 64, false, false, true, true, false}, 12);
  return bad;
}
