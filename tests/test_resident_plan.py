"""The host rule that lays the systems of a one-launch solve over the
device's workgroups (csrc/resident_plan.hpp), compiled with g++."""
import ctypes as C
import itertools
import os
import subprocess

import pytest

ROOT = os.path.abspath(os.path.join(os.path.dirname(__file__), ".."))

SHIM = r"""
#include "resident_plan.hpp"
#include <atomic>
#include <chrono>
#include <thread>
using namespace rhmc;
// two threads that take a tenth each over and over, never both without it for
// long: how often they did before a third got the whole, at most limit
extern "C" int turns(int limit) {
  std::atomic<int> n{0};
  std::atomic<bool> waiting{false}, got{false};
  auto small = [&](int ms) {
    while (!got && n < limit) {
      ResidentShare s(0, 0.1);
      if (waiting) n++;
      std::this_thread::sleep_for(std::chrono::milliseconds(ms));
    }
  };
  std::thread a(small, 3), b(small, 4);
  std::this_thread::sleep_for(std::chrono::milliseconds(20));
  std::thread c([&] {
    waiting = true;
    ResidentShare s(0, 1.0);
    got = true;
  });
  a.join(); b.join(); c.join();
  return n;
}
// out: launches, then of each nr, threads, members, total, lattices, and of each lattice index, sites, nwg
extern "C" int plan(int n, const long *vh, const int *nrhs, int whole, int cus, int per_cu, int *out) {
  std::vector<ResidentLattice> ls;
  for (int l = 0; l < n; l++) ls.push_back({vh[l], nrhs[l], whole != 0});
  int *o = out;
  const std::vector<ResidentLaunch> p = resident_pack(ls, (unsigned)cus, [&] { return per_cu; });
  *o++ = (int)p.size();
  for (const ResidentLaunch &r : p) {
    *o++ = r.nr; *o++ = r.threads; *o++ = r.members; *o++ = (int)r.total; *o++ = (int)r.lat.size();
    for (size_t q = 0; q < r.lat.size(); q++) { *o++ = r.lat[q]; *o++ = r.sites[q]; *o++ = r.nwg[q]; }
  }
  return (int)(o - out);
}
// the iteration that gives the result (0: go on); its place in the launch to *q
extern "C" int stop(int i0, int ran, int met, int most, int *q) { return power_stop(i0, ran, met != 0, most, *q); }
extern "C" int max_members() { return kResMaxMembers; }
"""


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    src, so = d / "shim.cpp", d / "shim.so"
    src.write_text(SHIM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-pthread", "-shared", "-fPIC", "-I",
                    os.path.join(ROOT, "rhmc-on-gpu_amd", "csrc"), str(src), "-o", str(so)], check=True)
    return C.CDLL(str(so))


def plan(lib, lats, whole=True, cus=256, per_cu=2):
    """[(nr, threads, members, total, [(lattice, sites, nwg), ...]), ...]"""
    n = len(lats)
    out = (C.c_int * 4096)()
    lib.plan(n, (C.c_long * n)(*[v for v, _ in lats]), (C.c_int * n)(*[r for _, r in lats]), int(whole), cus, per_cu,
             out)
    it = iter(out)
    res = []
    for _ in range(next(it)):
        nr, threads, members, total, k = (next(it) for _ in range(5))
        res.append((nr, threads, members, total, [(next(it), next(it), next(it)) for _ in range(k)]))
    return res


def check(lib, lats, whole, cus, per_cu):
    p = plan(lib, lats, whole, cus, per_cu)
    if not p:
        return 0
    assert len(p) <= 3
    assert sorted(q[0] for r in p for q in r[4]) == list(range(len(lats)))
    for nr, threads, members, total, ls in p:
        assert nr in (1, 2, 4) and threads in (256, 512)
        wgs = got = 0
        for l, sites, nwg in ls:
            vh, nrhs = lats[l]
            assert sites == 1 or (sites == 2 and nr == 1 and threads == 512)
            assert (nwg - 1) * (threads // 4) * sites < vh <= nwg * (threads // 4) * sites
            m = -(-nrhs // nr)
            got += m
            wgs += m * (-(-nwg // 8) * 8)
        assert members == got and total == wgs
        assert members <= lib.max_members()
        # more workgroups than CUs only in the form of which a CU holds per_cu
        assert total <= (cus * max(1, per_cu) if nr == 1 and threads == 512 and len(p) == 1 else cus)
        assert whole or all(lats[l][1] <= nr for l, _, _ in ls)
    return len(p)


SIZES = [4 ** 4 // 2, 6 ** 4 // 2, 8 ** 3 * 4 // 2, 12 ** 4 // 2, 16 ** 4 // 2, 24 ** 3 * 8 // 2]


@pytest.mark.parametrize("cus,per_cu", [(256, 2), (256, 1), (304, 2), (64, 2), (32, 0), (8, 2)])
def test_plan_places_every_lattice_and_bounds_the_members(lib, cus, per_cu):
    """Equal lattices and pairs of sizes, 1 to 16 lattices (the most of a
    lockstep solve), 1 to 32 right-hand sides each: every lattice is in one
    launch, no launch has more members than its table or more workgroups than
    the device holds at once."""
    planned = 0
    for n, whole in itertools.product(range(1, 17), (True, False)):
        for a, b in itertools.combinations_with_replacement(SIZES, 2):
            for ra, rb in itertools.product((1, 2, 3, 5, 8, 23, 32), repeat=2):
                lats = [(a, ra) if l < (n + 1) // 2 else (b, rb) for l in range(n)]
                planned += check(lib, lats, whole, cus, per_cu) > 0
    assert planned > 0


def test_plan_of_many_small_systems(lib):
    """Groups that fill up a launch's member table before its CUs: twelve
    lattices of 8^3x4 with 8 systems each, sixteen with 5, one 16^4 with one
    and three 8^3x4 with 8."""
    small, big = 8 ** 3 * 4 // 2, 16 ** 4 // 2
    for lats in ([(small, 8)] * 12, [(small, 5)] * 12, [(small, 5)] * 16, [(big, 1)] + [(small, 8)] * 3):
        check(lib, lats, True, 256, 2)


# (first iteration, iterations run, met) of launches of 64, at most 20000: (iteration of the result or 0, its place)
@pytest.mark.parametrize("i0,ran,met,result,place", [
    (1, 1, 1, 1, 1), (1, 10, 1, 10, 10), (1, 64, 1, 64, 64), (1, 64, 0, 0, None), (65, 3, 1, 67, 3),
    (19905, 64, 0, 0, None), (19969, 64, 0, 20000, 32), (19969, 32, 1, 20000, 32), (19969, 31, 1, 19999, 31),
    (19969, 33, 1, 20000, 32), (19969, 64, 1, 20000, 32)])
def test_power_iterations_stop_where_the_kernel_did(lib, i0, ran, met, result, place):
    """A launch that ended early is the end whatever the host would make of
    the norms (what it did not run holds nothing); the iterations past the
    largest number are not used."""
    q = C.c_int()
    assert lib.stop(i0, ran, met, 20000, C.byref(q)) == result
    if result:
        assert q.value == place


def test_whole_device_gets_its_turn(lib):
    """A solve that needs every compute unit comes before those that ask for
    theirs after it: at most the share that each of two other threads was about
    to take when it began to wait."""
    assert lib.turns(200) <= 4
