// Prints the records that a random ray meets (OctreeFlat::ray_records) of a raw float32 triangle file.
//   ray_records_probe FILE SPLIT DEPTH
#include <cstdio>
#include <cstdlib>
#include <vector>
#include "dr_octree_build.h"

int main(int argc, char **argv) {
  if (argc != 4) return 2;
  FILE *f = std::fopen(argv[1], "rb");
  if (!f) return 2;
  std::vector<float> t;
  float v;
  while (std::fread(&v, 4, 1, f) == 1) t.push_back(v);
  std::fclose(f);
  dr::OctreeHost h;
  dr::OctreeFlat flat;
  if (dr::build_octree(t.data(), (int)(t.size() / 9), std::atoi(argv[2]), std::atoi(argv[3]), 4, h) != 0) return 3;
  if (dr::flatten_octree(h, flat) != 0) return 4;
  std::printf("%.17g\n", flat.ray_records);
  return 0;
}
