// Host check of the lane-group marcher (march.h: march_probe, group_plan)
// against march_trip, launch by launch: every ray of a pixel subsample is
// marched with random sample budgets per launch both ways, a group's lanes one
// after the other; sample start times, the bin where each launch stops,
// whether the ray lives on, and the bins passed must be equal.  Reads
// <dir>/scene.bin, rm.bin (the fvc_scene_info and fvc_raymarch_info records)
// and occ.bin (uint8 [nlvl][128][128][128]).
// Usage: march_group_check <dir> <pixel stride> <lanes>.  Exits 1 on any mismatch.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "../frustumvolumecaching_amd/csrc/march.h"

using namespace fvc;

static std::vector<uint8_t> read_file(const std::string& p) {
  std::vector<uint8_t> v;
  FILE* f = std::fopen(p.c_str(), "rb");
  if (!f) std::exit(2);
  std::fseek(f, 0, SEEK_END);
  v.resize((size_t)std::ftell(f));
  std::fseek(f, 0, SEEK_SET);
  if (std::fread(v.data(), 1, v.size(), f) != v.size()) std::exit(2);
  std::fclose(f);
  return v;
}

// march_group (render_common.h) with the lanes of one group in a loop
static bool march_group_host(int G, const MarchGrid& g, const uint32_t* coarse, MarchRay& r, int n_steps,
                             std::vector<float>& t0s, int& bins) {
  int cnt = 0;
  bool alive = true;
  while (cnt < n_steps) {
    uint32_t occ = 0, past = 0;
    float t0[16], top = -1.0f;
    for (int k = 0; k < G; k++) {
      float hi;
      const int res = march_probe(g, coarse, r, r.j + k, t0[k], hi);
      if (res == PROBE_SAMPLE) occ |= 1u << k;
      if (res == PROBE_PAST) past |= 1u << k;
      top = hi > top ? hi : top;
    }
    const GroupPlan p = group_plan(G, occ, past, n_steps - cnt);
    for (int k = 0; k < G; k++)
      if ((p.samples >> k) & 1u) { t0s.push_back(t0[k]); cnt++; }
    bins += p.bins;
    r.j += p.bins;
    if (p.ended) { alive = false; bins++; break; }
    if (p.full) break;
    if (top > 0.0f) bins += table_jump(g.tab, r.row, r.m, r.j, r.t1, top);
  }
  r.t1 = g.tab.t[r.row.base + r.j];
  return alive;
}

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const std::string dir = argv[1];
  const int stride = std::atoi(argv[2]), G = std::atoi(argv[3]);
  const std::vector<uint8_t> scb = read_file(dir + "/scene.bin"), rmb = read_file(dir + "/rm.bin");
  const std::vector<uint8_t> occ = read_file(dir + "/occ.bin");
  fvc_scene_info sc;
  fvc_raymarch_info rm;
  if (scb.size() != sizeof(sc) || rmb.size() != sizeof(rm)) return 2;
  std::memcpy(&sc, scb.data(), sizeof(sc));
  std::memcpy(&rm, rmb.data(), sizeof(rm));
  const int nlvl = sc.grid_nlvl, V = 128 * 128 * 128;
  if (occ.size() != (size_t)nlvl * V) return 2;
  std::vector<uint64_t> bf((size_t)nlvl * V / 64, 0);
  for (int l = 0; l < nlvl; l++)
    for (int x = 0; x < 128; x++)
      for (int y = 0; y < 128; y++)
        for (int z = 0; z < 128; z++)
          if (occ[(size_t)l * V + ((size_t)x * 128 + y) * 128 + z]) {
            const uint64_t bit = (uint64_t)l * V + morton3d(x, y, z);
            bf[bit >> 6] |= 1ull << (bit & 63);
          }
  const std::vector<uint32_t> coarse = build_coarse(occ.data(), nlvl);
  MarchGrid g;
  g.occ = occ_params(sc);
  g.st = rm.stepsize_info;
  const fvc_stepsize_info& s = g.st;
  const V3 from = cvt(sc.aabb_from), to = cvt(sc.aabb_to), eye = translation(rm.cam_info.cam2world);
  float need = 0.0f;
  for (int c = 0; c < 8; c++) {
    const V3 q = {(c & 1) ? to.x : from.x, (c & 2) ? to.y : from.y, (c & 4) ? to.z : from.z};
    const V3 v = q - eye;
    need = std::max(need, std::sqrt(dot3(v, v)));
  }
  need = std::min(need, s.far_);
  std::vector<float> tt;
  std::vector<int> off;
  const int rows = build_step_rows(s, need * 1.02f + 4.0f * s.dt_max, tt, off);
  g.tab = step_view(s);
  g.tab.t = tt.data();
  g.tab.off = off.data();
  g.tab.n_rows = rows;
  g.bf64 = bf.data();
  const int W = rm.cam_info.res_x, H = rm.cam_info.res_y;
  long long n_rays = 0, n_samples = 0, n_launches = 0, bad = 0, unusable = 0;
  uint32_t rnd = 12345u;
  for (int y = 0; y < H; y += stride)
    for (int x = 0; x < W; x += stride) {
      const Ray ray = gen_ray(rm.cam_info, (float)x + 0.5f, (float)y + 0.5f);
      float t0, t1;
      if (!ray_aabb(ray, from, to, t0, t1)) continue;
      const float mf = std::round(step_from_t(s, std::max(t0, s.near_)) - s.near_i);
      MarchRay a;
      a.o = ray.o;
      a.d = ray.d;
      a.slab = ray_slab(ray.o, ray.d);
      a.far_ = std::min(t1, s.far_);
      a.m = (int)mf;
      a.j = 0;
      a.t1 = t_from_step(s, mf + s.near_i);
      a.sk = no_skip();
      a.row = step_row(g.tab, a.m);
      MarchRay b = a;
      n_rays++;
      if (!group_usable(g, b)) { unusable++; continue; }
      bool alive = true, same = true;
      while (alive && same) {
        rnd = rnd * 1664525u + 1013904223u;
        const int budget = 1 + (int)((rnd >> 16) & 63u);
        // a launch starts without a skip interval
        a.sk = no_skip();
        std::vector<float> sa, sb;
        int ba = 0, bb = 0;
        bool alive_a = true;
        while ((int)sa.size() < budget) {
          float ts;
          const int res = march_trip(g, coarse.data(), a, ts, ba);
          if (res == TRIP_END) { alive_a = false; break; }
          if (res == TRIP_SAMPLE) sa.push_back(ts);
        }
        const bool alive_b = march_group_host(G, g, coarse.data(), b, budget, sb, bb);
        n_launches++;
        n_samples += (long long)sa.size();
        same = alive_a == alive_b && sa.size() == sb.size() && ba == bb &&
               std::memcmp(sa.data(), sb.data(), sa.size() * sizeof(float)) == 0 &&
               (!alive_a || (a.j == b.j && a.t1 == b.t1));
        alive = alive_a;
      }
      if (!same) {
        if (bad < 5) std::printf("mismatch at pixel (%d, %d)\n", x, y);
        bad++;
      }
    }
  std::printf("%lld rays, %lld samples, %lld launches, %lld rays without a usable row, %lld mismatching rays\n", n_rays,
              n_samples, n_launches, unusable, bad);
  return bad != 0 || n_samples == 0 || unusable == n_rays;
}
