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
								for (mesh_dev::Walk walk : {mesh_dev::Walk{}, mesh_dev::Walk{9, 2, true}})
								{
									if (tile > 1 && walk.cache) // tiles and walks do not meet
										continue;
									const mesh_dev::BlockOrder ord = mesh_dev::block_order(g, nb, sbk, order | (tile << 4), walk);
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
							}
	// the walks of the SU(3) kernels where no slab order is: 'c' order 2, 'm' memory
	// order, 's' slices side by side, of the fused step FP64 and FP32 and of Delta H
	struct
	{
		int L[4];
		const char *walks;
	} const routes[] = {{{18, 16, 16, 16}, "cmcm"}, {{18, 8, 32, 32}, "cmcm"}, {{6, 32, 32, 32}, "cmcm"},
	                    {{10, 64, 32, 32}, "cmcs"}, {{18, 32, 32, 32}, "smcs"}, {{30, 32, 32, 32}, "smms"},
	                    {{22, 16, 16, 64}, "mmmm"}, {{18, 24, 24, 24}, "mmmm"}, {{30, 32, 32, 16}, "cmmm"},
	                    {{26, 26, 26, 26}, "mmms"}, {{18, 36, 36, 36}, "smms"},
	                    {{22, 22, 22, 22}, "mmmm"}, {{28, 28, 28, 28}, "smms"}, {{36, 36, 36, 36}, "ssms"},
	                    {{18, 15, 20, 22}, "mmmm"}};
	for (auto const &r : routes)
	{
		mesh_dev::Geo g{};
		g.nd = 4;
		long V = 1;
		for (int i = 0; i < 4; ++i)
			V *= g.L[i] = r.L[i];
		for (int k = 0; k < 4; ++k)
		{
			const bool dh = k >= 2, f64 = k % 2 == 0;
			const int sbk = dh ? 128 : 64;
			const mesh_dev::BlockOrder o = mesh_dev::block_order(
			    g, (int)((V + sbk - 1) / sbk), sbk, 3 | (4 << 4), dh ? mesh_dev::delta_h_walk(g, f64) : mesh_dev::fused_walk(g, f64));
			const char walk = o.kind == mesh_dev::BlockOrder::CACHE ? 'c' : (o.S ? 's' : 'm');
			if (walk != r.walks[k])
			{
				std::printf("%dx%dx%dx%d kernel %d: %c\n", r.L[0], r.L[1], r.L[2], r.L[3], k, walk);
				++bad;
			}
		}
	}
	std::printf("%ld orders, %ld wrong\n", count, bad);
	return bad != 0;
}
