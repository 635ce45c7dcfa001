// Host-only check of the passes' tiles along bounded and periodic rows
// (sg_internal.h): every point belongs to exactly one tile of one launch, the
// closure rows to edge tiles, and a grid whose tiles fit the chip at once
// takes one launch.
#include <cstdio>
#include <vector>

#include "sg_internal.h"

using namespace sg;

int main() {
  int bad = 0, split = 0, whole = 0;
  for (int ns : {2, 3, 4, 9, 16, 18})
    for (int bounded : {0, 1})
      for (int nx = 11; nx <= 200; nx++)
        for (int ny : {11, 33, 128})
          for (int nz : {11, 64, 200}) {
            Params P{};
            P.nx = nx; P.ny = ny; P.nz = nz; P.ns = ns;
            P.bnd[0] = bounded;
            P.xsplit = pass_split(P);
            std::vector<int> owner(nx, 0);
            for (int xp : {0, 1, 2}) {
              if (bounded ? xp == 0 : xp != 0) continue;
              for (int b = 0; b < pass_xtiles(P, xp); b++)
                for (int i = pass_x0(P, xp, b), q = 0; q < 16; q++, i++) {
                  if (i >= (xp == 1 ? nx - PASS_EW : nx)) continue;   // outside this tile
                  owner[i]++;
                  if (xp == 1 && (i < PASS_EW || i >= nx - PASS_EW)) bad++;
                }
            }
            for (int i = 0; i < nx; i++) bad += owner[i] != 1;
            const long tiles = (long)((nx + 15) / 16) * ((ny + 15) / 16) * nz;
            if (bounded && tiles <= 256 && pass_xtiles(P, 1) != 0) bad++;   // fits at one block a CU
            if (bounded && nx >= 32 && tiles > 1024 && !P.xsplit) bad++;    // fits nowhere
            (P.xsplit ? split : whole)++;
          }
  printf("%s split %d whole %d\n", bad || !split || !whole ? "FAILED" : "ok", split, whole);
  return bad || !split || !whole;
}
