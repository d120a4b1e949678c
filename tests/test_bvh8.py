"""The 8-wide collapse on the CPU: bvh.cpp compiled with a small driver that walks the
nodes.  Every triangle lies in one leaf, every child box holds its triangles'
vertices (in exact arithmetic), slots are either interior, a leaf of at most four or
unused, and a scene that cannot be encoded has no 8-wide nodes but a 4-wide tree."""
import os
import shutil
import subprocess

import numpy as np
import pytest

import cudapt_amd as ca
from cudapt_amd import scenes

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "cudapt_amd", "csrc")

DRIVER = r'''
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <string>
#include "cpt_internal.h"
using namespace cpt;
#define NEED(c) do { if (!(c)) { std::printf("failed: %s (node %u)\n", #c, at); std::exit(1); } } while (0)
static BvhHost b;
static std::vector<float> pos;
static std::vector<int> seen;
static double half(uint16_t h) {
  const int e = h >> 10, m = h & 0x3FF;
  return e ? std::ldexp(m + 1024.0, e - 25) : std::ldexp((double)m, -24);
}
struct Box { double lo[3], hi[3]; };
// the triangles below node `at` lie in every box on the way to it
static u32 walk(u32 at, std::vector<Box>& path, u32 depth) {
  NEED(at < b.nodes8.size());
  NEED(depth <= b.depth8);
  const Node8& n = b.nodes8[at];
  u32 next = n.child, tri = n.tri, total = 0;
  for (int s = 0; s < 8; s++) {
    const u32 leaf = n.valid >> (4 * s) & 15u;
    const bool inner = n.exps >> (24 + s) & 1u;
    NEED(!(inner && leaf));
    NEED(leaf == 0 || leaf == 1 || leaf == 3 || leaf == 7 || leaf == 15);
    Box x;
    for (int a = 0; a < 3; a++) {
      const double ext = std::ldexp(1.0, (int)(n.exps >> (8 * a) & 255u) - 127);
      NEED(n.h[a][0][s] <= 0x3C00 && n.h[a][1][s] <= 0x3C00);
      x.lo[a] = (double)n.o[a] + half(n.h[a][0][s]) * ext;
      x.hi[a] = (double)n.o[a] + half(n.h[a][1][s]) * ext;
      NEED(std::fabs(x.lo[a]) <= b.qmag && std::fabs(x.hi[a]) <= b.qmag);
    }
    if (!inner && !leaf) { NEED(n.h[0][0][s] > n.h[0][1][s]); continue; }
    path.push_back(x);
    if (inner) total += walk(next++, path, depth + 1);
    for (u32 m = leaf; m; m &= m - 1, tri++, total++) {
      NEED(tri < b.order8.size());
      const u32 o = b.dreorder[b.order8[tri]];
      seen[o]++;
      for (const Box& q : path)
        for (int k = 0; k < 9; k++) {
          const double v = pos[o * 9 + k];
          NEED(q.lo[k % 3] <= v && v <= q.hi[k % 3]);
        }
    }
    path.pop_back();
  }
  return total;
}
int main(int argc, char** argv) {
  std::FILE* f = std::fopen(argv[1], "rb");
  float v;
  while (std::fread(&v, 4, 1, f) == 1) pos.push_back(v);
  const u32 nt = (u32)pos.size() / 9, leaf = (u32)std::atoi(argv[2]), at = 0;
  std::vector<u32> idx(nt * 3);
  for (u32 i = 0; i < nt * 3; i++) idx[i] = i;
  NEED(build_bvh_device(pos.data(), idx.data(), nt, b));
  collapse_bvh4(pos.data(), idx.data(), b, leaf);
  if (!collapse_bvh8(b, leaf)) { std::printf("refused\n"); return 0; }
  NEED(!b.nodes4.empty());
  if (b.nodes8.empty()) { NEED(b.order8.empty()); std::printf("none\n"); return 0; }
  seen.assign(nt, 0);
  std::vector<Box> path;
  NEED(walk(0, path, 1) == nt && b.order8.size() == nt);
  for (int s : seen) NEED(s == 1);
  std::printf("ok %zu %u\n", b.nodes8.size(), b.depth8);
}
'''


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not found")
    d = tmp_path_factory.mktemp("bvh8")
    (d / "d.cpp").write_text(DRIVER)
    r = subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-I", CSRC, str(d / "d.cpp"),
                        os.path.join(CSRC, "bvh.cpp"), "-o", str(d / "d")], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr

    def run(tri, leaf):
        np.ascontiguousarray(tri, np.float32).tofile(str(d / "t.bin"))
        r = subprocess.run([str(d / "d"), str(d / "t.bin"), str(leaf)], capture_output=True, text=True, timeout=60)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.strip()
    return run


def _mesh(kind):
    g = np.random.default_rng(3)
    if kind in ("cornell", "grid"):
        sc = scenes.cornell() if kind == "cornell" else scenes.sphere_grid(grid=8)
        return np.asarray(sc["pos"])[np.asarray(sc["idx"])]
    if kind == "one":
        return g.uniform(-1, 1, (1, 3, 3))
    if kind == "coincident":
        return np.repeat(g.uniform(-1, 1, (1, 3, 3)), 200, 0)
    if kind == "chain":                              # every split takes one triangle off
        return g.uniform(-1, 1, (100, 3, 3)) * 2.0 ** -np.arange(100)[:, None, None]
    n, scale, at = {"nine": (9, 1, 0), "points": (50, 0, 0), "tiny": (500, 1e-38, 0), "offset": (500, 1e-3, 4096),
                    "large": (300, 8e37, 0)}[kind]
    c = g.uniform(-1, 1, (n, 1, 3)) * max(scale, 1e-30)
    return at + c + g.uniform(-0.1, 0.1, (n, 3, 3)) * scale


@pytest.mark.parametrize("leaf", [1, 2, 4, 64])
@pytest.mark.parametrize("kind", ["cornell", "grid", "one", "nine", "coincident", "chain", "points", "tiny", "offset",
                                  "large"])
def test_nodes_hold_every_triangle_once(walk, kind, leaf):
    # "large" is 1.76e38 wide, past the largest extent of 2^127
    assert walk(_mesh(kind), leaf).split()[0] == ("none" if kind == "large" else "ok")


# vertices that 8-wide nodes cannot encode leave the scene to the FP32 layout; one at minus infinity is refused
@pytest.mark.parametrize("value,says", [(1.6e38, "ok"), (1.8e38, "none"), (3e38, "none"), (-3e38, "none"),
                                        (np.inf, "none"), (-np.inf, "refused")])
@pytest.mark.parametrize("n", [1, 20])
def test_far_vertices(walk, value, says, n):
    t = np.random.default_rng(0).uniform(-1, 1, (n, 3, 3)).astype(np.float32)
    t[0, 0, 0] = value
    assert walk(t, 2).split()[0] == says
    with np.errstate(all="ignore"):
        sc = scenes.mesh_scene(t.reshape(-1, 3), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))
    if says == "refused":
        with pytest.raises(Exception, match="minus infinity"):
            ca.Scene(sc, upload=False)
    else:
        ca.Scene(sc, upload=False)
