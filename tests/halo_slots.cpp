// Host check of the slots from which the fused MD step reads a staged block's
// x3-neighbours (halo_slots, halo_site in su3_dev.h): for every site of every
// block -- the last one partly filled included -- the site staged in slot sp
// (sm) must be the site's forward (backward) neighbour along x3, and every
// staged site must lie on the lattice.  Exit status 0 when all agree.
#include "../mesh_amd/csrc/su3_dev.h"
#include <cstdio>

using namespace mesh_dev;

int main()
{
	long bad = 0, count = 0;
	for (int L3 = 2; L3 <= 140; ++L3)
		for (int rows : {1, 2, 3, 4, 7, 16, 30})
		{
			const long V = (long)L3 * rows;
			for (long b0 = 0; b0 < V; b0 += 64)
			{
				const int n = V - b0 < 64 ? (int)(V - b0) : 64;
				long site[68];
				for (int s = 0; s < 64; ++s)
					site[s] = -1;
				for (int l = 0; l < n; ++l)
					site[block_slot(l)] = b0 + l;
				for (int h = 0; h < 4; ++h)
				{
					site[64 + h] = halo_site(L3, FastDiv(L3), b0, n, h);
					bad += site[64 + h] < 0 || site[64 + h] >= V;
				}
				for (int l = 0; l < n; ++l, ++count)
				{
					const long x = b0 + l, row = x / L3 * L3;
					const int c3 = (int)(x - row);
					const LaneSlots at = halo_slots(L3, n, l, c3);
					if (site[at.me] != x || site[at.sp] != row + (c3 + 1) % L3 ||
					    site[at.sm] != row + (c3 + L3 - 1) % L3)
					{
						if (bad < 5)
							std::printf("L3 %d rows %d x %ld\n", L3, rows, x);
						++bad;
					}
				}
			}
		}
	std::printf("%ld sites, %ld wrong\n", count, bad);
	return bad != 0;
}
