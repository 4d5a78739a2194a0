/*
Cells per march of a pass over `blocks` blocks of lines with nd cells each,
at most `most`, when `resident` blocks run on a CU at once: a march of km
cells costs about km + 1.5 faces, and the blocks run in
ceil(blocks * chunks / (256 * resident)) rounds, so a fixed km leaves CUs
idle in the last round or altogether.  FP64 HLLD step, 32-cell marches ->
this rule: 128^3 545 -> 412 us, 192^3 1493 -> 1387 us; 256^3 3210 (32 cells)
against 3230 (29; there VALU issue is the bound whatever the rounds).
At most `most` candidates, the distinct march lengths: a loop over the
number of chunks took 0.5 ms of every step's launch on a line of 131072 cells.
*/
#pragma once
#include <algorithm>

namespace pamhd_dev {

inline int march_cells(unsigned blocks, int nd, int resident, int most)
{
	const long long slots = 256ll * resident;
	int best = 1;
	double best_cost = 1e300;
	for (int km = std::min(most, nd); km >= 1; km--) {
		const int chunks = (nd + km - 1) / km;
		km = (nd + chunks - 1) / chunks;   /* the shortest with as many chunks */
		const double cost = (double)((blocks * (long long)chunks + slots - 1) / slots) * (km + 1.5);
		if (cost < best_cost) {
			best_cost = cost;
			best = km;
		}
	}
	return best;
}

} // namespace pamhd_dev
