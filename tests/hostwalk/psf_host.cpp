// Host build of the two forms of a projection-space PSF weight (psfWeight,
// psfWeightTab) for CPU tests.
#include "yrtmi_rays.hpp"

#include <vector>

using namespace yrtmi;

extern "C" {

// n footprints [x0, x1] under a row of K taps ks apart: out[2 i] psfWeight,
// out[2 i + 1] psfWeightTab.
void hw_psf(const float* taps, int K, float ks, int64_t n, const float* x0, const float* x1,
            float* out)
{
	DPsf P{};
	P.numS = 1;
	P.K = K;
	P.kSpacing = ks;
	P.rks = rcpNearest(ks);
	std::vector<float> row(psfRowTaps(K), 0.f);
	std::copy(taps, taps + K, row.begin() + 2);
	std::vector<double> cum(K + 2);
	psfPrefixSums(taps, 1, K, ks, cum.data());
	std::vector<float4> tab(psfSegments(K));
	for (int e = 0; e < psfSegments(K); e++)
		psfSegment(row.data(), cum.data(), K, e, &tab[e]);
	for (int64_t i = 0; i < n; i++)
	{
		out[2 * i] = psfWeight(P, row.data(), cum.data(), x0[i], x1[i]);
		out[2 * i + 1] = psfWeightTab(P, tab.data(), x0[i], x1[i]);
	}
}

}  // extern "C"
