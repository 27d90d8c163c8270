// pathtracer.hip - the megakernel path tracer for gfx950
// (MegakernelPathTracer, src/render/megakernel/device.cu:50-195).
//
// One lane runs one pixel's samples from the camera ray to the end of each
// path: closest hit, emission with its MIS weight, Russian roulette from the
// first vertex on, a light sample on smooth surfaces (power heuristic,
// src/render/sampling.h:8-28), then the BSDF sample.  Pixels are taken in 8 x
// 8-pixel tiles, so a wave's primary rays are coherent.  No media: rays ignore
// medium interfaces, as in the reference, and meshes without material are
// rejected by the host.
//
// A lane has one ray in flight, its path's closest ray or its shadow ray, and a
// wave's rays advance together (traverseSteps) until fewer than refillLanes of
// 64 still do; the others shade, go on with their next ray, sample or pixel.
// Lanes that ran a tile's pixels to the end of the tile's longest path, each
// wave waiting for its slowest ray at every bounce, took 968 us for a 960x540
// frame of a 328 K-triangle field; this took 827 us (1 lane: 837, 4: 821, 16:
// 856), and takes 808 us with the triangle records.  Waves wait for memory 62 %
// of their time, and 23 % of the lanes are in use per vector instruction.
#include "pathtracer.h"

namespace krr {

// evalMIS(1, p0, 1, p1) with MIS_POWER_HEURISTIC (sampling.h:20-28).
KRR_DEV float misPower(float p0, float p1) {
	const float q0 = p0 * p0, q1 = p1 * p1;
	return q0 / (q0 + q1);
}

KRR_DEV bool finiteWeight(float w) { return !(__builtin_isnan(w) || __builtin_isinf(w)); }

// The path of a lane between two of its rays.
struct PtPath {
	f3 thp, L, ctxP;
	float pdf;
	int bsdfType, depth;
};

// The path's vertex for the closest hit h of the ray (o, d), in the order of
// device.cu:52-122.  next: the path goes on with the ray (no, nd); shadow: its
// light sample contributes `contrib` when nothing occludes (so, sd) up to 1.
// The shadow ray is traced before the path's next vertex, so the radiance is
// added in the reference's order.  TEX = false: the scene has no textures,
// image-lit infinite lights or alpha tests.
template <bool TEX>
KRR_DEV void pathVertex(const PtArgs &A, const TravState &h, const f3 &d, Pcg &rng, PtPath &p, bool &next, f3 &no, f3 &nd, bool &shadow, f3 &so,
						f3 &sd, f3 &contrib) {
	const DevScene &sc = A.sc;
	const int nL	   = sc.nLights;
	const float selPdf = 1.f / (float) (nL > 0 ? nL : 1);
	next = shadow = false;
	if (h.prim < 0) { // handleMiss (device.cu:67-79)
		for (int li = 0; li < nL; li++) {
			const DevLight Lr = sc.lights[li];
			if (Lr.type != 1) continue;
			float w = 1.f;
			if (A.nee && p.depth > 0 && !(p.bsdfType & BSDF_SPECULAR)) {
				w = misPower(p.pdf, kInv4Pi * selPdf);
				if (!finiteWeight(w)) w = 1.f;
			}
			p.L = p.L + p.thp * w * infiniteLi<TEX>(Lr, d);
		}
		return;
	}
	SurfaceInteraction intr;
	surfaceAt<TEX>(sc, h.prim, h.b1, h.b2, d, -1, intr);
	if (intr.light >= 0) { // handleHit (device.cu:52-65)
		const DevLight Lr = sc.lights[intr.light];
		const f3 Le		  = areaLightL<TEX>(Lr, intr.n, intr.wo, intr.u, intr.v);
		float w			  = 1.f;
		if (A.nee && p.depth > 0) {
			const float lightPdf = lightPdfLi(sc, intr.light, intr.p, intr.n, p.ctxP) * selPdf;
			if (!(p.bsdfType & BSDF_SPECULAR)) w = misPower(p.pdf, lightPdf);
			if (!finiteWeight(w)) w = 1.f;
		}
		p.L = p.L + Le * w * p.thp;
	}
	if (p.depth == A.maxDepth || (A.rr < 1.f && rng.get1D() > A.rr)) return;
	p.thp				  = p.thp / A.rr;
	const DevMaterial mat = materialAt<TEX>(sc, intr);
	BSDF bsdf;
	bsdf.setup(mat);
	const f3 woL = intr.toLocal(intr.wo);
	if (A.nee && (bsdfTypeOf(mat.type, mat.roughness) & BSDF_SMOOTH) && nL > 0) { // evalDirect (device.cu:101-106)
		const float ul		 = rng.get1D();
		const int li		 = min((int) (uint32_t) (ul * (float) nL), nL - 1);
		const float u0		 = rng.get1D(), u1 = rng.get1D();
		const LightSample ls = sampleLi<TEX>(sc, li, u0, u1, intr.p);
		const f3 wiL		 = intr.toLocal(normalize(ls.p - intr.p));
		const float lightPdf = selPdf * ls.pdf;
		if (lightPdf != 0.f) {
			const float bp = bsdf.pdf(woL, wiL);
			const f3 bv	   = bsdf.f(woL, wiL) * fabsf(wiL.z);
			const float w  = misPower(lightPdf, bp);
			if (finiteWeight(w) && bv.any()) {
				const f3 to	= offsetRayOrigin(ls.p, ls.n, intr.p - ls.p);
				so			= offsetRayOrigin(intr.p, intr.n, to - intr.p);
				sd			= to - so;
				contrib		= p.thp * bv * w / lightPdf * ls.L;
				shadow		= true;
			}
		}
	}
	// generateScatterRay (device.cu:108-122)
	const BSDFSample bs = bsdf.sample(woL, rng);
	if (bs.pdf == 0.f || !bs.f.any()) return;
	const f3 wiW = intr.toWorld(bs.wi);
	p.bsdfType	 = bs.flags;
	no			 = offsetRayOrigin(intr.p, intr.n, wiW);
	nd			 = wiW;
	p.ctxP		 = intr.p;
	p.pdf		 = bs.pdf;
	p.thp		 = p.thp * (bs.f * fabsf(bs.wi.z) / bs.pdf);
	p.depth++;
	next = p.thp.any();
}

// FIXED: each wave's places are given shares (WorkShare without a counter),
// taken up half a wave at a time; else a counter's, as lanes end.
template <bool TEX, bool FIXED> __global__ void __launch_bounds__(256) k_path_tracer(PtArgs A) {
	extern __shared__ int ldsStack[];
	const LaneStack stack = laneStack(A.bvh, ldsStack, A.ovf);
	uint32_t nClosest = 0, nShadow = 0, nv = 0, nt = 0;
	bool exhausted = false, active = false, going = false, shadowRay = false, next = false;
	int left = 0, x = 0, y = 0; // samples of the pixel (x, y) still to start
	Pcg rng{0, 0};
	PtPath p;
	f3 color, o, d, no, nd, contrib; // the ray in flight, and while it is a shadow ray the path's next one
	TravState ts;
	const int places = A.nTiles * 64;
	WorkShare share	 = FIXED ? firstShare(A.fetchLanes, places) : WorkShare{};
	while (true) {
		if (!exhausted) {
			const bool need = !active && left == 0 && laneId() < A.fetchLanes;
			int i;
			if constexpr (!FIXED) {
				i = wavePush(A.work, need);
				if (__ballot(need && i >= places)) exhausted = true;
			} else {
				i = -1;
				if (2 * __popcll(__ballot(need)) >= A.fetchLanes) {
					i		  = takePlace(share, need, nullptr, A.fetchLanes, places);
					exhausted = share.empty();
				}
			}
			if (need && (!FIXED || i >= 0) && i < places) {
				const int tile = i >> 6;
				x = (tile % A.tilesX) * 8 + (i & 7);
				y = (tile / A.tilesX) * 8 + ((i >> 3) & 7);
				if (x < A.W && y < A.H) { // else a place of the tile outside the image: take another
					left  = A.spp;
					color = f3();
					rng.setSeed((uint64_t) interleave32((uint32_t) x, (uint32_t) y), (uint64_t) A.sampleIndex);
				}
			}
		}
		if (!active && left > 0) {
			left--;
			const RayItem cr = cameraRay(A.cam, A.W, A.H, x, y, rng);
			(void) rng.get1D(); // SampledWavelengths::sampleUniform
			o		  = cr.o;
			d		  = cr.d;
			p		  = PtPath{f3(1.f), f3(), f3(), 0.f, BSDF_UNSET, 0};
			active	  = true;
			going	  = true;
			shadowRay = false;
			travInit(ts, A.bvh, __builtin_inff());
			nClosest++;
		}
		const int nActive = __popcll(__ballot(active));
		if (nActive == 0) {
			if (exhausted) break;
			continue; // every place taken was outside the image
		}
		// every active lane has a ray in flight, and the threshold is at most
		// their number: each round finishes at least one ray
		const bool drain   = exhausted && __ballot(left > 0) == 0;
		const int minLanes = drain ? 1 : max(1, (nActive * A.refillLanes) >> 6);
		traverseSteps<false, TEX>(A.bvh, o, d, shadowRay, going, ts, stack, minLanes, nv, nt, nullptr, 0, kDefaultLeafShare);
		if (!active || going) continue;
		if (shadowRay) {
			if (ts.prim < 0) p.L = p.L + contrib;
		} else {
			bool shadow;
			f3 so, sd;
			pathVertex<TEX>(A, ts, d, rng, p, next, no, nd, shadow, so, sd, contrib);
			if (shadow) {
				nShadow++;
				o		  = so;
				d		  = sd;
				shadowRay = true;
				going	  = true;
				travInit(ts, A.bvh, 1.f);
				continue;
			}
		}
		if (next) {
			o		  = no;
			d		  = nd;
			shadowRay = false;
			going	  = true;
			travInit(ts, A.bvh, __builtin_inff());
			nClosest++;
			continue;
		}
		active = false;
		color  = color + p.L;
		if (left == 0) {
			const float inv = (float) A.spp;
			A.film[(size_t) (A.H - 1 - y) * A.W + x] = make_float4(color.x / inv, color.y / inv, color.z / inv, 1.f);
		}
	}
	waveAddU64(&A.rays[0], nClosest);
	waveAddU64(&A.rays[1], nShadow);
}

__global__ void k_path_tracer_clear(unsigned long long *rays, int *work) {
	if (threadIdx.x < 2) rays[threadIdx.x] = 0ull;
	if (threadIdx.x == 2) *work = 0;
}

template <class F> static void withPathTracer(bool textured, bool fixed, F &&f) {
	if (textured) fixed ? f(k_path_tracer<true, true>) : f(k_path_tracer<true, false>);
	else fixed ? f(k_path_tracer<false, true>) : f(k_path_tracer<false, false>);
}

hipError_t launchPathTracer(const PtArgs &a, int grid, int tb, size_t lds, hipStream_t st) {
	hipLaunchKernelGGL(k_path_tracer_clear, dim3(1), dim3(64), 0, st, a.rays, a.work);
	withPathTracer(a.textured, a.fixedShares, [&](auto k) { hipLaunchKernelGGL(k, dim3(grid), dim3(tb), lds, st, a); });
	return hipGetLastError();
}

int pathTracerBlocksPerCU(int tb, size_t lds, bool textured, bool fixedShares) {
	int nb		 = 0;
	hipError_t e = hipSuccess;
	withPathTracer(textured, fixedShares, [&](auto k) { e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k, tb, lds); });
	if (e != hipSuccess || nb < 1) nb = 1;
	return nb;
}

} // namespace krr
