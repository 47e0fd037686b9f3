// The step's field-map lookups (MapField, MapFieldF) on the host, one lane:
// for axes that multiply by reciprocals and axes that divide, with and
// without the cell-major copy.  Every lookup equals gridField bit for bit
// (the FP32 one the same lookup without the lane's cell copy); with a cell-major map a
// lookup leaves the cell's record in the lane's copy, and one in the same
// cell reads that copy, not the map.
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>
#include <vector>

#include "../../acts_amd/csrc/kf_field_host.hpp"
#include "../../acts_amd/csrc/kf_mixed.hpp"

using namespace kf;

namespace {

int failures = 0;
void expect(bool ok, const char* what, const char* map) {
  if (ok) return;
  ++failures;
  std::printf("FAILED %s: %s\n", map, what);
}

// Cell records of a padded point array (fieldCellsKernel).
template <typename T>
std::vector<T> cellRecords(const DevField& F, const std::vector<T>& v, int stride) {
  const int64_t sy = F.nb[2] + 1, sx = static_cast<int64_t>(F.nb[1] + 1) * sy;
  std::vector<T> out(static_cast<size_t>(stride) * F.nb[0] * F.nb[1] * F.nb[2] + 64, T(0));
  size_t at = 0;
  for (int x = 0; x < F.nb[0]; ++x)
    for (int y = 0; y < F.nb[1]; ++y)
      for (int z = 0; z < F.nb[2]; ++z, at += stride)
        for (int i = 0; i < 4; ++i)
          for (int k = 0; k < 6; ++k)
            out[at + 6 * i + k] = v[3 * ((x + (i >> 1)) * sx + (y + (i & 1)) * sy + z) + k];
  return out;
}

bool same(double a, double b) { return std::memcmp(&a, &b, sizeof a) == 0; }
bool same(float a, float b) { return std::memcmp(&a, &b, sizeof a) == 0; }
template <typename V>
bool same3(const V& a, const V& b) {
  return same(a.x, b.x) && same(a.y, b.y) && same(a.z, b.z);
}

template <typename T>
T* aligned(std::vector<T>& v) {
  auto p = reinterpret_cast<uintptr_t>(v.data());
  return reinterpret_cast<T*>((p + 127) / 128 * 128);
}

// One lane's lookups: Field is MapField or MapFieldF, Value V3 or F3.
template <typename Field, typename Value, typename T>
void check(DevField& F, T* cells, size_t cellValues, CellCache cache, T* copy, const char* map,
           const std::vector<Value>& points) {
  const Field cached{F, cache}, plain{F, CellCache{nullptr, nullptr, nullptr}};
  cache.idx[0] = -1;
  bool equal = true, filled = true, kept = true;
  const std::vector<T> record(cells, cells + cellValues);
  for (const Value& p : points) {
    Value want, got, again;
    const bool in = plain(p, want);
    equal = equal && cached(p, got) == in && (!in || same3(got, want));
    if (!in) continue;
    filled = filled && cache.idx[0] >= 0;
    if (cache.idx[0] < 0) continue;
    const size_t stride = sizeof(T) == 8 ? kCellDoubles : kCellFloats;
    for (int j = 0; j < kCellValues; ++j)
      filled = filled && same(copy[j * kCellCacheStride], record[stride * cache.idx[0] + j]);
    // the map gone: the lane's copy serves the cell
    T* rec = cells + stride * cache.idx[0];
    for (int j = 0; j < kCellValues; ++j) rec[j] = std::numeric_limits<T>::quiet_NaN();
    cached(p, again);
    kept = kept && same3(again, want);
    for (int j = 0; j < kCellValues; ++j) rec[j] = record[stride * cache.idx[0] + j];
  }
  expect(equal, "a lookup with the cell copy gives another field", map);
  expect(filled, "a lookup does not leave its cell in the lane's copy", map);
  expect(kept, "a lookup in the same cell reads the map again", map);
}

void run(const char* name, const int32_t n[3], const double lo[3], const double hi[3],
         bool reciprocals) {
  std::mt19937_64 rng(7);
  std::uniform_real_distribution<double> u(-1, 1);
  std::vector<double> values(static_cast<size_t>(3) * n[0] * n[1] * n[2]);
  for (double& v : values) v = u(rng);
  acts_kf_field in{};
  in.kind = ACTS_KF_FIELD_GRID_XYZ;
  for (int a = 0; a < 3; ++a) {
    in.n[a] = n[a];
    in.point_min[a] = lo[a];
    in.point_max[a] = hi[a];
  }
  in.values = values.data();
  DevField F{};
  std::vector<double> padded;
  if (!buildGridField(in, F, padded)) std::abort();
  expect((F.recip != 0) == reciprocals, "not the kind of axes meant", name);
  for (int a = 0; a < 3; ++a) {
    F.minF[a] = static_cast<float>(F.min[a]);
    F.widthF[a] = static_cast<float>(F.width[a]);
    F.upperF[a] = static_cast<float>(F.upper[a]);
    F.rwF[a] = 1.0f / F.widthF[a];
  }
  std::vector<V3> points;
  std::vector<F3> pointsF;
  for (int i = 0; i < 4000; ++i) {
    double x[3];
    for (int a = 0; a < 3; ++a) {
      // inside, on the cells' edges, and some outside
      x[a] = 0.5 * (lo[a] + hi[a]) + 0.53 * (hi[a] - lo[a]) * u(rng);
      if (i % 3 == 0) x[a] = F.min[a] + std::floor((x[a] - F.min[a]) / F.width[a]) * F.width[a];
    }
    points.push_back(mk(x[0], x[1], x[2]));
    pointsF.push_back(mkf(static_cast<float>(x[0]), static_cast<float>(x[1]),
                          static_cast<float>(x[2])));
  }
  points.push_back(mk(std::nan(""), lo[1], lo[2]));
  points.push_back(mk(HUGE_VAL, lo[1], lo[2]));

  int32_t idx[kCellCacheStride];
  std::vector<double> copy(kCellValues * kCellCacheStride);
  std::vector<float> copyF(kCellValues * kCellCacheStride);
  std::vector<double> cells0 = cellRecords(F, padded, kCellDoubles);
  double* cells = aligned(cells0);
  {
    const std::vector<double> c = cellRecords(F, padded, kCellDoubles);
    std::copy(c.begin(), c.end() - 64, cells);
  }
  // point arrays: no copy to keep, the same field
  F.v = padded.data();
  F.cells = nullptr;
  bool equal = true;
  for (const V3& p : points) {
    V3 a, b;
    const bool in1 = MapField{F, CellCache{nullptr, nullptr, nullptr}}(p, a);
    equal = equal && in1 == (gridField(F, p, b) == 0) && (!in1 || same3(a, b));
  }
  expect(equal, "point arrays: another field than gridField's", name);
  F.cells = cells;
  equal = true;
  for (const V3& p : points) {
    V3 a, b;
    const bool in1 = MapField{F, CellCache{nullptr, nullptr, nullptr}}(p, a);
    equal = equal && in1 == (gridField(F, p, b) == 0) && (!in1 || same3(a, b));
  }
  expect(equal, "cell records: another field than gridField's", name);
  const size_t nCells = static_cast<size_t>(F.nb[0]) * F.nb[1] * F.nb[2];
  check<MapField, V3, double>(F, cells, nCells * kCellDoubles,
                              CellCache{copy.data(), nullptr, idx}, copy.data(), name, points);

  std::vector<float> paddedF(padded.begin(), padded.end());
  std::vector<float> cellsF0 = cellRecords(F, paddedF, kCellFloats);
  float* cellsF = aligned(cellsF0);
  {
    const std::vector<float> c = cellRecords(F, paddedF, kCellFloats);
    std::copy(c.begin(), c.end() - 64, cellsF);
  }
  F.cellsF = cellsF;
  for (int recipF = 0; recipF < 2; ++recipF) {
    F.recipF = recipF;
    check<MapFieldF, F3, float>(F, cellsF, nCells * kCellFloats,
                                CellCache{nullptr, copyF.data(), idx}, copyF.data(),
                                recipF ? "FP32, reciprocals" : "FP32, divisions", pointsF);
  }
}

}  // namespace

int main() {
  const double lo[3] = {-2000, -2000, -2800}, hi[3] = {2000, 2000, 2800};
  const int32_t even[3] = {11, 11, 15}, odd[3] = {57, 57, 8};
  run("reciprocals", even, lo, hi, true);
  run("divisions", odd, lo, hi, false);
  if (failures == 0) std::printf("ok\n");
  return failures ? 1 : 0;
}
