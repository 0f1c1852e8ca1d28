// Checks of a single layer tree (tree.hip) against the runtime and kernel
// stand-ins of this folder.  Usage: emu_tree CHECK; a failed check is named and
// ends with status 2.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "../../include/gcomcot_hip.h"
#include "comcot_consts.h"
#include "tree.h"

using namespace gc;

namespace {

[[noreturn]] void die(const char *m) {
  std::fprintf(stderr, "%s\n", m);
  std::exit(2);
}
void ok(bool c, const char *m) {
  if (!c) die(m);
}

void add_root(Tree &T, int laycord, int laygov, int nx, int ny) {
  const int corners[4] = {1, nx, 1, ny};
  const std::vector<float> h((size_t)nx * ny, 100.0f), z((size_t)nx * ny, 0.0f);
  if (tree_create_layer(T, nullptr, 1, -1, 1, laycord, laygov, 1, 1, corners, 0, 0.013f, 1.0f, 1.0f, 1.0f,
                        nx, ny, h.data(), z.data()) ||
      tree_upload_coef(T.layers[1], std::vector<float>((size_t)kNumCoef * ny, 0.0f)))
    die("layer 1");
}

// A tuned layer whose launches cannot march, because MAX_AMP's maximum is kept
// or a sponge set, takes the tuner's best tile; as soon as they can again, its
// tuned form.
void tuned_fallback() {
  Tree T;
  add_root(T, 0, 1, 70, 60);
  LayerRec &R = T.layers[1];
  T.variant = 2;
  auto step = [&] {
    ok(tree_enqueue_root_step(T, nullptr) == 0, "root step");
    return emu_last_variant();
  };
  ok(step() == 2, "an untuned layer's variant");
  R.variant = 8;
  R.tile_variant = 3;
  ok(step() == 8, "a tuned layer's variant");
  T.raw_max = 1;
  ok(step() == 3, "the best tile where the maximum is kept");
  T.raw_max = 0;
  ok(step() == 8, "the tuned variant again");
  tree_free(T);

  add_root(T, 0, 0, 70, 60);
  T.blocking = 2;
  auto two = [&] {
    ok(tree_step2_eligible(T), "two steps per launch");
    ok(tree_enqueue_root_steps2(T, nullptr) == 0, "two root steps");
    return emu_last_step2() + 1;
  };
  ok(two() == 2, "an untuned layer's mode");
  T.layers[1].blocking = 1;
  T.layers[1].tile_blocking = 5;
  ok(blocking_mode(T) == 1, "a tuned layer's mode");
  T.raw_max = 1;
  ok(two() == 5, "the best two-step tile where the maximum is kept");
  T.layers[1].tile_blocking = 0;
  ok(!tree_step2_eligible(T), "one step per launch where that was the fastest without marching");
  tree_free(T);
}

int add_child(Tree &T, int id, int parent, int laygov, int R, int rt, const int *c) {
  const int nx = (c[1] - c[0] + 1) * R + 1, ny = (c[3] - c[2] + 1) * R + 1;
  const std::vector<float> h((size_t)nx * ny, 50.0f), z((size_t)nx * ny, 0.0f);
  return tree_create_layer(T, nullptr, id, parent, T.layers[parent].level + 1, 1, laygov, R, rt, c, 0, 0.013f,
                           1.0f, 1.0f, 1.0f, nx, ny, h.data(), z.data()) ||
         tree_upload_coef(T.layers[id], std::vector<float>((size_t)kNumCoef * ny, 0.0f));
}

// Every sub-step of a nest finds its boundary fluxes made, whatever JNQ makes
// ahead, JNZ takes along or the root's march runs beside: REL_TIMEs on every
// remainder and beyond the slots, two children, and a child of a child.
void substeps() {
  for (int rt = 1; rt <= 21; ++rt)
    for (int form = 0; form < 3; ++form) {  // one child; two; one with a child of its own
      Tree T;
      add_root(T, 0, form == 2 ? 1 : 0, 60, 50);
      const int a[4] = {6, 13, 7, 15}, b[4] = {20, 30, 9, 18}, g[4] = {5, 12, 4, 11};
      const int rt2 = (rt + 3) % 7 + 1;
      ok(add_child(T, 2, 1, rt % 2, 3, rt, a) == 0, "layer 2");
      if (form == 1) ok(add_child(T, 3, 1, 1, 2, rt2, b) == 0, "layer 3");
      if (form == 2) ok(add_child(T, 3, 2, 1, 2, rt2, g) == 0, "layer 3");
      const int steps = 5;
      for (int k = 1; k <= steps; ++k) ok(tree_enqueue_root_step(T, nullptr, k < steps) == 0, "root step");
      const int want[4] = {0, steps, steps * rt, form == 2 ? steps * rt * rt2 : steps * rt2};
      for (int id = 1; id <= (form ? 3 : 2); ++id) {
        const LayerRec &L = T.layers[id];
        for (size_t c = 0; c < L.nxy(); ++c)
          ok(L.z[L.cur][c] == want[id] && L.m[L.cur][c] == want[id] && L.n[L.cur][c] == want[id], "step count");
      }
      tree_free(T);
    }
}

// Device memory that the layers report is what they allocate: in a tree, and
// through the batch engine's entries, whose footprint of a layer is exact with
// its REL_TIME and a bound without.
void footprint() {
  const int kind[][3] = {{0, 0, 1}, {0, 1, 1}, {1, 0, 1}, {1, 1, 1}, {0, 1, 2}, {1, 1, 4}, {0, 0, 5}, {1, 0, 21}};
  for (const auto &k : kind) {
    int lc = k[0], lg = k[1], rt = k[2], one = 1, two = 2, root = -1, cart = 1, nx = 77, ny = 60, R = 3;
    int corners[4] = {1, nx, 1, ny}, foot[4] = {8, 30, 9, 25}, fs = 0;
    int cnx = 23 * R + 1, cny = 17 * R + 1, sid = 0;
    float fc = 0.013f, dt = 1.0f, d = 1.0f;
    long long steps = 1, live = emu_live_bytes();
    std::vector<float> h(100 * 100, 50.0f), z(100 * 100, 0.0f), coef(10 * 100, 0.0f);
    ok(gcomcot_batch_new_scenario_(&steps, &sid) == 0, "scenario");
    ok(gcomcot_batch_add_layer_(&sid, &one, &root, &lc, &lg, &one, &one, corners, &fs, &fc, &dt, &d, &d,
                                coef.data(), h.data(), z.data(), &nx, &ny) == 0, "layer 1");
    long long want = gcomcot_layer_footprint_ex_(&nx, &ny, &lc, &lg, &one);
    ok(want <= gcomcot_layer_footprint_(&nx, &ny, &lg), "the bound of layer 1");
    if (rt > 1) {
      ok(gcomcot_batch_add_layer_(&sid, &two, &one, &cart, &lg, &R, &rt, foot, &fs, &fc, &dt, &d, &d, nullptr,
                                  h.data(), z.data(), &cnx, &cny) == 0, "layer 2");
      const long long child = gcomcot_layer_footprint_ex_(&cnx, &cny, &cart, &lg, &rt);
      ok(child <= gcomcot_layer_footprint_(&cnx, &cny, &lg), "the bound of layer 2");
      want += child;
    }
    ok(gcomcot_batch_device_bytes_(&sid) == want, "the scenario's bytes and its layers' footprints");
    // beside its layers a scenario holds its two step counters
    ok(emu_live_bytes() - live == want + 2 * (long long)sizeof(int), "the bytes allocated");
    ok(gcomcot_batch_remove_(&sid) == 0 && emu_live_bytes() == live, "removal");
  }
  ok(gcomcot_batch_reset_() == 0, "reset");
}

}  // namespace

int main(int argc, char **argv) {
  const char *check = argc > 1 ? argv[1] : "";
  if (!std::strcmp(check, "tuned-fallback")) tuned_fallback();
  else if (!std::strcmp(check, "footprint")) footprint();
  else if (!std::strcmp(check, "substeps")) substeps();
  else die("no such check");
  if (emu_live_bytes() != 0) die("device memory leaked");
  std::printf("%s passed\n", check);
}
