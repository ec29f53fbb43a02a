// Host checks of the sizes of the random-candidate kernels' group memory
// (kernel_table.h), compiled with g++ by tests/test_table_sizes.py.
#include <cstdio>
#include <initializer_list>

#include "kernel_table.h"

int main()
{
	for (int rb : {S2TC_RB_FEW, S2TC_RB_MANY})
		for (int pbw_max = 1; pbw_max <= 14; ++pbw_max) {
			const int ints = normal_row_ints(pbw_max, rb);
			for (int pbw = 1; pbw <= pbw_max; ++pbw) {
				const int t = normal_table_ints(pbw, ints);
				// within the memory that there is, and for a block of few candidates
				// as if its class had no larger ones
				if (t < 0 || t > ints || (rb == S2TC_RB_FEW && t != normal_row_ints(pbw, rb))) {
					printf("tables: %d of %d row blocks, %d in registers: %d of %d ints\n", pbw, pbw_max, rb, t, ints);
					return 1;
				}
				if (pbw <= 2 && t != 0) {
					printf("tables for %d row blocks\n", pbw);
					return 1;
				}
			}
			if (rb == S2TC_RB_MANY && pbw_max >= 5 && normal_table_ints(pbw_max, ints) != ints) {
				printf("one image, %d row blocks: %d of %d ints\n", pbw_max, normal_table_ints(pbw_max, ints), ints);
				return 1;
			}
		}
	// three row blocks in registers only where most of a class's pair work wants them
	const auto work = [](int pbw, int textures) { return 4096.0 * textures * pbw * pbw; };
	const struct {
		int few, nfew, nmany;
		bool many;
	} classes[] = {{3, 0, 40, true}, {2, 40, 1, false}, {2, 40, 10, false}, {4, 40, 1, false}, {3, 4, 40, true}};
	for (const auto &c : classes) {
		const double m = work(5, c.nmany), all = m + work(c.few, c.nfew);
		if (class_many(m, all, 5, 1 << 20, 256) != c.many || class_many(m, all, 5, 100, 256) ||
		    class_many(m, all, 9, 1 << 20, 256)) {
			printf("class of %d textures with %d row blocks and %d with 5\n", c.nfew, c.few, c.nmany);
			return 1;
		}
	}
	// more workgroups than eight to a CU of the device, however many it has
	if (normal_many(5, 8 * 256, 256) || !normal_many(5, 8 * 256 + 1, 256) || normal_many(5, 256, 32) ||
	    !normal_many(5, 257, 32)) {
		printf("workgroups per CU\n");
		return 1;
	}
	printf("ok\n");
	return 0;
}
