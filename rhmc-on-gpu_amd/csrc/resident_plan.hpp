// resident_plan.hpp -- how the systems of a one-launch solve (resident.hpp) are
// laid over a device's workgroups, where its power iterations stop, and the
// share of the device that each takes.  Host code without a device call.
#pragma once

#include <algorithm>
#include <condition_variable>
#include <mutex>
#include <vector>

namespace rhmc {

constexpr int kResMaxMembers = 22;  // members a launch's argument table holds (ResGroup)

// a lattice of a solve: half sites, right-hand sides, whether each
// right-hand side's vectors are whole cache lines
struct ResidentLattice {
  long Vh;
  int nrhs;
  bool whole_lines;
};

// One launch of k_bms_resident: the lattices of a solve that share it
// (indices), the right-hand sides per member, threads per workgroup, each
// lattice's sites per lane and workgroups per member.
struct ResidentLaunch {
  int nr = 1, threads = 512, sites_max = 1;
  std::vector<int> lat, sites, nwg;
  int members = 0;
  unsigned total = 0;  // workgroups
};

// workgroups of a lattice's member, rounded up to the 8 XCDs
inline unsigned resident_wgs(long Vh, int threads, int sites, int &nwg) {
  const long per = (long)(threads / 4) * sites;
  nwg = (int)((Vh + per - 1) / per);
  return (unsigned)((nwg + 7) / 8 * 8);
}

// The launches of a solve over one or several lattices; empty where the
// launches per iteration are used.  Measured per iteration (us, one launch
// against the two tuned launches; FP64, FP32):
//   8^3x4 1 to 8 systems  7.9 / 18,     7.5 / 18
//   12^4  1               8.0 / 18,     7.0 / 17
//   12^4  8 (4 a member) 19.9 / 28,    14.2 / 20
//   16^4  1              12.0 / 22,     9.3 / 16
//   16^4  2 (2 a member) 16.8 / 25,    12.5 / 18
//   16^4  4 (4 a member) 25.4 / 28,    17.5 / 28
//   16^4  8 (8 a member) 46   / 43,    32   / 28   (not taken)
//   24^3x8 1 (two sites) 24.8 / 28,    17.7 / 19
// The rule: the fewest systems per member (1, 2 or 4), then the smaller
// workgroups, for which there is at most one workgroup per CU (16^4 with one
// system: 14.5 us with 512 workgroups of 256 lanes).  One system on a lattice
// too large for that may take two sites per lane (two systems of 16^4 that
// way: 26 us).  Several lattices that do not fit that way
// share the CUs as far as registers allow (the largest with two sites per
// lane), else they run as up to three launches.
// No launch has more than kResMaxMembers members (a member takes at least 8
// workgroups, so the CUs alone would admit 32).  cus: compute units;
// per_cu(): workgroups of 512 lanes with two sites per lane that one holds.
template <typename PerCu>
std::vector<ResidentLaunch> resident_pack(const std::vector<ResidentLattice> &ls, unsigned cus, PerCu &&per_cu) {
  const int n = (int)ls.size();
  int nvec = 0;
  bool split = true;
  for (const ResidentLattice &q : ls) {
    nvec = std::max(nvec, q.nrhs);
    split = split && q.whole_lines;
  }
  auto all = [&](int nr, int threads, int sites) {
    ResidentLaunch r;
    r.nr = nr;
    r.threads = threads;
    r.sites_max = sites;
    r.sites.assign(n, sites);
    r.nwg.resize(n);
    for (int l = 0; l < n; l++) {
      const int m = (ls[l].nrhs + nr - 1) / nr;
      r.members += m;
      r.lat.push_back(l);
      r.total += resident_wgs(ls[l].Vh, threads, sites, r.nwg[l]) * m;
    }
    if (r.members > kResMaxMembers || (!split && nr < nvec)) r.total = ~0u;
    return r;
  };
  for (int nr = 1; nr <= 4; nr *= 2)
    for (int threads = 256; threads <= 512; threads *= 2)
      if (const ResidentLaunch r = all(nr, threads, 1); r.total <= cus) return {r};
  if (n == 1) {
    if (nvec == 1)
      if (const ResidentLaunch r = all(1, 512, 2); r.total <= cus) return {r};
    return {};
  }
  // several lattices, one system per member: as many workgroups as the CUs
  // hold, the largest lattices with two sites per lane until they fit
  ResidentLaunch r = all(1, 512, 1);
  if (r.total != ~0u) {
    const unsigned room = cus * (unsigned)per_cu();
    r.sites_max = 2;
    while (r.total > room) {
      int big = -1;
      for (int l = 0; l < n; l++)
        if (r.sites[l] == 1 && (big < 0 || ls[l].Vh > ls[big].Vh)) big = l;
      if (big < 0) break;
      r.total -= (unsigned)((r.nwg[big] + 7) / 8 * 8) * ls[big].nrhs;
      r.sites[big] = 2;
      r.total += resident_wgs(ls[big].Vh, 512, 2, r.nwg[big]) * ls[big].nrhs;
    }
    if (r.total <= room) return {r};
  }
  // in turn: the largest first, each into the first launch with room for it
  std::vector<int> order(n);
  for (int l = 0; l < n; l++) order[l] = l;
  std::stable_sort(order.begin(), order.end(), [&](int a, int b) { return ls[a].Vh > ls[b].Vh; });
  std::vector<ResidentLaunch> out;
  for (const int l : order) {
    int nwg = 0;
    const unsigned t = resident_wgs(ls[l].Vh, 512, 1, nwg) * (unsigned)ls[l].nrhs;
    if (t > cus || !split || ls[l].nrhs > kResMaxMembers) return {};
    size_t q = 0;
    while (q < out.size() && (out[q].total + t > cus || out[q].members + ls[l].nrhs > kResMaxMembers)) q++;
    if (q == out.size()) out.emplace_back();
    out[q].lat.push_back(l);
    out[q].sites.push_back(1);
    out[q].nwg.push_back(nwg);
    out[q].members += ls[l].nrhs;
    out[q].total += t;
  }
  return out.size() <= 3 ? out : std::vector<ResidentLaunch>();
}

// The result of a launch of power iterations i0, i0+1, ...: it ran `ran` of
// them, the last of which met the test or not.  The kernel is the judge (what
// it did not run was not written); the host adds the largest number of
// iterations.  Returns the iteration that gives the result, 0 to go on; q:
// its place in the launch, from 1.
inline int power_stop(int i0, int ran, bool met, int most, int &q) {
  q = std::min(ran, most - i0 + 1);
  return met || i0 + ran > most ? i0 + q - 1 : 0;
}

// Workgroups of the one-launch solves in flight on a device, as a share of
// its compute units: solves of several handles (threads) run at the same
// time only while all their workgroups fit, at most one per CU, so that
// every grid is resident as a whole.  Shares are given in the order in which
// they were asked for: one of the whole device would else wait for as long as
// smaller ones overlap.
class ResidentShare {
 public:
  ResidentShare(int device, double share) : d_(device < 0 || device >= kDevices ? 0 : device), s_(share) {
    Slots &t = slots();
    std::unique_lock<std::mutex> l(t.m);
    const unsigned long turn = t.asked[d_]++;
    t.cv.wait(l, [&] { return t.given[d_] == turn && t.used[d_] + s_ <= 1.0 + 1e-9; });
    t.used[d_] += s_;
    t.given[d_]++;
    l.unlock();
    t.cv.notify_all();  // the next in turn may fit beside it
  }
  ~ResidentShare() {
    Slots &t = slots();
    {
      std::lock_guard<std::mutex> l(t.m);
      t.used[d_] -= s_;
    }
    t.cv.notify_all();
  }
  ResidentShare(const ResidentShare &) = delete;
  ResidentShare &operator=(const ResidentShare &) = delete;

 private:
  static constexpr int kDevices = 64;
  struct Slots {
    std::mutex m;
    std::condition_variable cv;
    double used[kDevices] = {};
    unsigned long asked[kDevices] = {}, given[kDevices] = {};
  };
  static Slots &slots() {
    static Slots t;
    return t;
  }
  int d_;
  double s_;
};

}  // namespace rhmc
