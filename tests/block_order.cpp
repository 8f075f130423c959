// Host check of the stencil kernels' block orders (block_order in
// mesh_internal.h): over even and odd extents, row-block lengths, orders and
// tiles, the launch indices must reach every block exactly once; and of the
// division by multiplication they use (FastDiv in su3_dev.h).  Exit status 0 when
// all do.
#include "../mesh_amd/csrc/mesh_internal.h"
#include <cstdio>

int main()
{
	long bad = 0, count = 0;
	for (uint32_t i = 1; i < 4000; ++i)
		for (uint32_t d : {i, i * 7919u, (1u << 26) - i, 0x7fffffffu - i})
		{
			const mesh_dev::FastDiv by(d);
			for (uint64_t m : {0ull, 1ull, 2ull, 1ull << 13, 0x7fffffffull / d})
				for (int64_t n : {(int64_t)(m * d) - 1, (int64_t)(m * d), (int64_t)(m * d) + 1, (int64_t)0x7fffffff - i})
					if (n >= 0 && n <= 0x7fffffff)
						bad += by((uint32_t)n) != (uint32_t)n / d;
		}
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
								const mesh_dev::BlockOrder ord = mesh_dev::block_order(g, nb, sbk, order | (tile << 4));
								std::vector<char> seen(nb, 0);
								for (int b = 0; b < grid; ++b)
								{
									const int o = ord.at(b);
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
