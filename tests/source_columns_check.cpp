/*
 * Goes through every index the one-pass sources (kd_src_fused2) form on a 2-D
 * mesh and prints the number of updated cells and of faults.
 *
 *   source_columns_check NX NY ENERGY
 *     ENERGY 1: one row more is updated, as the adiabatic sources do
 *
 * A lane evaluates the stress of its cell i in the rows r0-1 .. r1 of its
 * block of rows, which reads the cells i, i-1 and i+1 (around the ring) in the
 * rows one below to one above.  Faults: a cell outside the ring, an element outside
 * the array of (NY + 6) NX, a cell updated more or less than once, an updated cell
 * whose neighbouring lanes do not hold the neighbouring cells.
 */
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "../fargo3d_amd/csrc/hip/f3d_columns.h"

int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const int nx = atoi(argv[1]), ny = atoi(argv[2]), ngh = 3, end = ngh + ny + atoi(argv[3]);
  long faults = 0, cells = 0;
  std::vector<int> times(nx, 0);
  for (int wave = 0; wave < (nx + kSrcCols - 1) / kSrcCols; wave++)
    for (int lane = 0; lane < 64; lane++) {
      const int is = src_position(wave, lane), i = src_cell(is, nx);
      faults += i < 0 || i >= nx;
      const int around[] = {i > 0 ? i - 1 : nx - 1, i, i < nx - 1 ? i + 1 : 0};
      for (int row = ngh - 1; row <= end; row++)
        for (int r = row - 1; r <= row + 1; r++)
          for (int c : around) {
            const long l = c + (long)r * nx;
            faults += l < 0 || l >= (long)(ny + 2 * ngh) * nx;
          }
      if (!src_updates(is, lane, nx)) continue;
      cells++;
      if (i >= 0 && i < nx) times[i]++;
      faults += src_cell(src_position(wave, lane - 1), nx) != around[0];
      faults += src_cell(src_position(wave, lane + 1), nx) != around[2];
    }
  for (int t : times) faults += t != 1;
  printf("%ld %ld\n", cells, faults);
  return 0;
}
