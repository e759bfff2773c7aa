// GroupWalk (parallel-rdp_amd/csrc/rdp_groups.hpp) over rounds given as text lines
// "passes scratch upscaled": prints "begins base passes" for each, where its
// scratch begins and the passes of its group so far.
#include <stdio.h>
#include <stdlib.h>

#include "../parallel-rdp_amd/csrc/rdp_groups.hpp"

int main(int argc, char **argv)
{
	rdp_mi::GroupWalk w;
	w.own = argc > 1 && atoi(argv[1]);
	unsigned passes, upscaled;
	unsigned long long scratch;
	while (scanf("%u %llu %u", &passes, &scratch, &upscaled) == 3) {
		const bool begins = w.next(passes, (size_t)scratch, upscaled != 0);
		printf("%d %zu %u\n", (int)begins, w.scratch, w.passes);
		w.scratch += (size_t)scratch;
	}
	return 0;
}
