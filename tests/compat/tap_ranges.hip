/* Host program: every load of tap_product.hpp's kernels over small problems, by the offsets that they form. Prints how many it looked at. */
#include "tap_product.hpp"

#include <cstdio>

using namespace cattle_hip;
using namespace cattle_hip::tap_product;

namespace {

long loads = 0, taken = 0, refused = 0;

bool in_range(const char* what, unsigned lane, unsigned wave, unsigned bytes, bool wanted, unsigned want, const GatherGeom& g, int channel, int t) {
	++loads;
	const bool ok = wave <= bytes && (lane == OUTSIDE ? !wanted : wanted && lane < OUTSIDE && lane + wave == want && lane + wave + 4 <= bytes);
	if (!ok)
		std::printf("%s: lane %u wave %u of %u bytes: %d x %d x %d, %d samples, output %d x %d, steps %d %d from %d %d, channel %d tap %d\n", what, lane, wave,
				bytes, g.LH, g.LW, g.LC, g.NS, g.OA, g.OB, g.RA, g.RB, g.PA, g.PB, channel, t);
	return ok;
}

/* what share_of_product does for a wavefront's channels, for all rows */
bool check(const GatherGeom& g) {
	if (!addressable(g)) {
		++refused;
		return true;
	}
	++taken;
	const StepGeom G = step_geom(g);
	const int pairs = (g.LC + 1) / 2, plane = g.NS * g.LH * g.LW;
	bool ok = true;
	for (int i = 0; i < pairs; ++i)
		for (int t = 0; t < TAPS; ++t)
			for (int lk = 0; lk < 2; ++lk) {
				const int first = 0, channel = 2 * i + lk;
				const bool exists = channel < g.LC;
				for (int f = 0; f < tiles_of(g.F) * TL; f += TL - 1)
					ok &= in_range("weights", exists ? wt_lane(g, f, lk) : OUTSIDE, wt_first(g, first) + wt_tap(g, t) + (unsigned) i * 8u * (unsigned) (TAPS * g.ldw), G.wt_bytes, exists,
							4u * (unsigned) ((channel * TAPS + t) * g.ldw + f), g, channel, t);
				for (int b = 0; b < g.OB; ++b)
					for (int a = 0; a < g.OA; ++a)
						for (int n = 0; n < g.N; ++n) {
							const bool inside = exists && row_inside(g, a, t % 3) && column_inside(g, b, t / 3);
							const int ya = a + g.PA + t % 3 * g.RA, yb = b + g.PB + t / 3 * g.RB;
							ok &= in_range("source", inside ? src_lane(g, plane, (unsigned) n, (unsigned) a, (unsigned) b, lk) : OUTSIDE,
									src_first(g, plane, G.before, first) + src_tap(g, t) + (unsigned) i * 8u * (unsigned) plane, G.src_bytes, inside,
									G.before + 4u * (unsigned) (n + g.NS * (ya + g.LH * yb) + plane * channel), g, channel, t);
						}
			}
	return ok;
}

GatherGeom geom(int N, int NS, int LH, int LW, int LC, int F, int OA, int OB, int RA, int RB, int PA, int PB) {
	GatherGeom g = {};
	g.N = N; g.NS = NS; g.LH = LH; g.LW = LW; g.LC = LC; g.OA = OA; g.OB = OB;
	g.R = g.S = 3; g.SA = g.SB = g.DA = g.DB = 1;
	g.RA = RA; g.RB = RB; g.PA = PA; g.PB = PB;
	g.M = N * OA * OB; g.K = 9 * LC; g.F = F; g.ldw = (F + 127) / 128 * 128;
	return g;
}

} /* namespace */

int main() {
	bool ok = true;
	for (int H = 1; H <= 5; ++H)
		for (int W = 1; W <= 5; ++W)
			for (int C : { 1, 2, 3, 4, 5, 6, 8 })
				for (int pv = 0; pv <= 4; ++pv)
					for (int ph = 0; ph <= 4; ++ph)
						for (int dv = 0; dv <= 2; ++dv)
							for (int dh = 0; dh <= 2; ++dh) {
								const int OH = H + 2 * pv - 2 * (dv + 1), OW = W + 2 * ph - 2 * (dh + 1);
								if (OH < 1 || OW < 1)
									continue;
								/* a forward product and an input gradient of a layer; the first samples of a longer sequence */
								ok &= check(geom(2, 2, H, W, C, 40, OH, OW, dv + 1, dh + 1, -pv, -ph));
								ok &= check(geom(2, 3, OH, OW, C, 9, H, W, -(dv + 1), -(dh + 1), pv, ph));
							}
	/* sides of one that are refused, and their neighbours that are not */
	ok &= !addressable(geom(4, 4, 9, 1, 1, 16, 9, 1, 1, 1, -1, -1)) && !addressable(geom(4, 4, 1, 1, 5, 16, 1, 1, 1, 1, -1, -1));
	ok &= addressable(geom(4, 4, 9, 1, 2, 16, 9, 1, 1, 1, -1, -1)) && addressable(geom(4, 4, 9, 2, 3, 16, 9, 2, 1, 1, -1, -1)) &&
			addressable(geom(4, 4, 1, 9, 1, 16, 1, 9, 1, 1, -1, -1));
	std::printf("%ld loads of %ld problems, %ld refused: %s\n", loads, taken, refused, ok ? "all in range" : "FAILED");
	return ok ? 0 : 1;
}
