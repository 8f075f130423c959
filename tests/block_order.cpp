// Host check of the stencil kernels' block orders (ordered_block_of in
// mesh_internal.h): over even and odd extents, row-block lengths, orders and
// tiles, the launch indices must reach every block exactly once.  Exit status
// 0 when all do.
#include "../mesh_amd/csrc/mesh_internal.h"
#include <cstdio>

int main()
{
	long bad = 0, count = 0;
	for (int l0 : {2, 3, 4, 7, 8, 9, 16, 18, 20, 36, 40})
		for (int l1 : {2, 3, 4, 15, 16, 44})
			for (int l2 : {2, 5, 8, 16, 20, 25, 36})
				for (int l3 : {2, 3, 8, 16, 20, 22, 32, 64, 100})
					for (int order = 0; order <= 4; ++order)
						for (int tile : {0, 1, 2, 4, 8})
							for (int sbk : {64, 128, 256})
							{
								mesh_dev::Geo g{};
								g.nd = 4;
								g.L[0] = l0, g.L[1] = l1, g.L[2] = l2, g.L[3] = l3;
								const long V = (long)l0 * l1 * l2 * l3;
								const int nb = (int)((V + sbk - 1) / sbk), grid = order ? (nb + 7) / 8 * 8 : nb;
								std::vector<char> seen(nb, 0);
								for (int b = 0; b < grid; ++b)
								{
									const int o = mesh_dev::ordered_block_of(g, nb, sbk, order | (tile << 4), b);
									if (o >= nb || (o >= 0 && seen[o]++))
										++bad;
								}
								for (char c : seen)
									bad += c != 1;
								++count;
							}
	std::printf("%ld orders, %ld wrong\n", count, bad);
	return bad != 0;
}
