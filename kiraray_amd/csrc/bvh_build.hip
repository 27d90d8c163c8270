// bvh_build.hip - binned-SAH BVH builder on the GPU, producing the 4-wide
// layout of bvh.h (the layout the traversal kernels read).
//
// Same algorithm and decisions as the host builder (bvh.cpp; binned SAH
// after Wald, IEEE RT 2007): per node the centroids are binned into 16 bins
// per axis, the split with the lowest cost nodeCost + (A_L N_L + A_R N_R) / A
// is taken (first minimum in axis-major, bin-minor order), a node of at most
// maxLeafSize triangles becomes a leaf when that is cheaper, a node whose
// centroids coincide is split at the middle (or kept as a leaf of <= 8).
// The float arithmetic is the host's, operation for operation, so both build
// the same binary tree except where the host's unstable partition order
// reaches a middle split.
//
// GPU organisation:
//  * large nodes (> kSmall references) are processed level by level, all
//    nodes of a level together: bounds, bins (LDS per block, merged with
//    integer atomics on order-preserving float encodings), split choice, a
//    stable partition between two reference buffers (places from the blocks'
//    bin counts) that also takes the children's bounds, and the next level's list
//    made on the device.  Two passes over the references per level, bound by
//    the latency of gathered boxes and by atomics on few addresses: 13 levels of a
//    328 K-triangle build 0.94 ms, 1.30 ms with bounds and counts in two more
//    passes and blocks of 2,048 references;
//  * every node of at most kSmall references roots a subtree that one block
//    builds alone in LDS, level by level, a node per wave;
//  * the binary tree is collapsed into 4-wide nodes level by level (open the
//    child with the largest surface area until four children), nodes of a
//    level numbered by block sums and a scan, children of a node contiguous;
//  * leaf triangles are stored in reference order, so a binary leaf
//    [first, first + count) is directly its triangle range.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdint>
#include <cstring>
#include <limits>
#include <type_traits>
#include <vector>

#include "bvh.h"
#include "bvh_build.h"

namespace krr {
namespace bvhdev {

constexpr int NB	   = 16;   // SAH bins per axis (the host builder's default)
constexpr int kSmall   = 1024; // nodes of at most this many references are built by one block
// References and threads per block in the level-synchronous phase: its passes
// wait for gathered boxes, and a level of 328 K references in blocks of 2,048 and
// 256 threads is less than one wave per SIMD.  2,048 with 1,024 threads, a
// build and two traces 4.48 against 4.43 ms.
constexpr int kChunk   = 1024;
constexpr int kThreads = 512;

// Order-preserving float <-> int map: a < b (floats) <=> ordF(a) < ordF(b).
__host__ __device__ inline int ordF(float f) {
	int i;
	std::memcpy(&i, &f, 4);
	return i >= 0 ? i : i ^ 0x7fffffff;
}
__host__ __device__ inline float unordF(int i) {
	int j = i >= 0 ? i : i ^ 0x7fffffff;
	float f;
	std::memcpy(&f, &j, 4);
	return f;
}

struct Box {
	float lo[3], hi[3];
	__host__ __device__ void reset() {
		for (int a = 0; a < 3; a++) {
			lo[a] = __builtin_inff();
			hi[a] = -__builtin_inff();
		}
	}
	__host__ __device__ void grow(const Box &b) {
		for (int a = 0; a < 3; a++) {
			lo[a] = fminf(lo[a], b.lo[a]);
			hi[a] = fmaxf(hi[a], b.hi[a]);
		}
	}
	// the host builder's Box::area, operation for operation
	__host__ __device__ float area() const {
		float e0 = hi[0] - lo[0], e1 = hi[1] - lo[1], e2 = hi[2] - lo[2];
		if (!(e0 >= 0) || !(e1 >= 0) || !(e2 >= 0)) return 0.f;
		return 2.f * (e0 * e1 + e1 * e2 + e2 * e0);
	}
};

// Bins of one node: per axis and bin the reference count and the union of
// the primitive boxes, as order-preserving ints.
struct Bins {
	int cnt[3][NB];
	int lo[3][NB][3];
	int hi[3][NB][3];
};

__device__ inline void binsReset(Bins &b, int t, int nt) {
	int *p = &b.cnt[0][0];
	for (int i = t; i < (int) (sizeof(Bins) / 4); i += nt) {
		const int k = i - 3 * NB; // lo block, then hi block
		p[i]		= i < 3 * NB ? 0 : (k < 3 * NB * 3 ? ordF(__builtin_inff()) : ordF(-__builtin_inff()));
	}
}

__device__ inline int binOf(float c, float lo, float scale) { return min(NB - 1, (int) ((c - lo) * scale)); }

struct Split {
	int axis, bin; // axis < 0: no binned split
	float cost;
};

// v combined over 16 lanes (a DPP row) by f, the result in each of them; over
// the wave when wide.
template <class F> __device__ inline float rowReduce(float v, F f, bool wide) {
	auto dpp = [&](auto ctrl) { return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), ctrl.value, 0xf, 0xf, true)); };
	v = f(v, dpp(std::integral_constant<int, 0xB1>{}));	 // lanes xor 1 (quad_perm 1 0 3 2)
	v = f(v, dpp(std::integral_constant<int, 0x4E>{}));	 // lanes xor 2 (quad_perm 2 3 0 1)
	v = f(v, dpp(std::integral_constant<int, 0x141>{})); // row_half_mirror
	v = f(v, dpp(std::integral_constant<int, 0x140>{})); // row_mirror
	if (wide) {
		v = f(v, __shfl_xor(v, 16));
		v = f(v, __shfl_xor(v, 32));
	}
	return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

// Inclusive scan over the 16 lanes of a row, from lane 0 up (CTRL0 0x110,
// row_shr) or from lane 15 down (0x100, row_shl); lanes without a source take
// the identity.
template <int CTRL0, class F> __device__ inline int rowScan(int v, int identity, F f) {
	v = f(v, __builtin_amdgcn_update_dpp(identity, v, CTRL0 + 1, 0xf, 0xf, false));
	v = f(v, __builtin_amdgcn_update_dpp(identity, v, CTRL0 + 2, 0xf, 0xf, false));
	v = f(v, __builtin_amdgcn_update_dpp(identity, v, CTRL0 + 4, 0xf, 0xf, false));
	v = f(v, __builtin_amdgcn_update_dpp(identity, v, CTRL0 + 8, 0xf, 0xf, false));
	return v;
}
template <int CTRL0> __device__ inline Box rowScanBox(Box b) {
	auto lo = [](int x, int y) { return __float_as_int(fminf(__int_as_float(x), __int_as_float(y))); };
	auto hi = [](int x, int y) { return __float_as_int(fmaxf(__int_as_float(x), __int_as_float(y))); };
	for (int a = 0; a < 3; a++) {
		b.lo[a] = __int_as_float(rowScan<CTRL0>(__float_as_int(b.lo[a]), __float_as_int(__builtin_inff()), lo));
		b.hi[a] = __int_as_float(rowScan<CTRL0>(__float_as_int(b.hi[a]), __float_as_int(-__builtin_inff()), hi));
	}
	return b;
}

// SAH over a node's bins exactly as the host builder (bvh.cpp
// Builder2::build), one wave per node: lane 16 a + k of the first 48 holds bin k
// of axis a (its box and count), prefix and suffix boxes over the 16 bins are
// DPP scans within a row of 16 lanes, and each lane prices the split after its
// bin; the first minimum in axis-major, bin-minor order wins.  mine: the lane
// holds a bin of an axis the centroids extend along.  Minima, maxima and counts
// are exact in any order.  nPre: references up to the lane's bin.
__device__ inline Split waveSplit(const Box &own, int cnt, bool mine, float pA, float nodeCost, int &nPre) {
	const int bin = __lane_id() & 15;
	auto add	  = [](int x, int y) { return x + y; };
	const Box pre = rowScanBox<0x110>(own);
	Box suf		  = rowScanBox<0x100>(own);
	nPre		  = rowScan<0x110>(cnt, 0, add);
	int nSuf	  = rowScan<0x100>(cnt, 0, add);
	// lane k takes the suffix from bin k + 1
	for (int a = 0; a < 3; a++) {
		suf.lo[a] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(suf.lo[a]), 0x101, 0xf, 0xf, true));
		suf.hi[a] = __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(suf.hi[a]), 0x101, 0xf, 0xf, true));
	}
	nSuf	   = __builtin_amdgcn_update_dpp(0, nSuf, 0x101, 0xf, 0xf, true);
	float cost = __builtin_inff();
	if (mine && bin < NB - 1 && nPre != 0 && nSuf != 0) cost = nodeCost + (pre.area() * nPre + suf.area() * nSuf) / fmaxf(pA, 1e-30f);
	if (!(cost < __builtin_inff())) cost = __builtin_inff(); // not a number: never the minimum
	const float best = rowReduce(cost, [](float x, float y) { return fminf(x, y); }, true);
	if (!(best < __builtin_inff())) return Split{-1, -1, __builtin_inff()};
	const int w = __ffsll((unsigned long long) __ballot(cost == best)) - 1;
	return Split{w >> 4, w & 15, best};
}

// Decision for a node of `count` references: 0 split (binned), 1 leaf,
// 2 split at the middle (bvh.cpp, after the SAH loop).
__device__ inline int decide(const Split &s, int count, int maxLeaf) {
	if (count <= maxLeaf && (s.axis < 0 || (float) count <= s.cost)) return 1;
	if (s.axis >= 0) return 0;
	return count <= 8 ? 1 : 2;
}

struct Prims {
	const float4 *lo, *hi; // primitive boxes (w unused)
};

__device__ inline void primBox(const Prims &P, int p, Box &b, float c[3]) {
	const float4 l = P.lo[p], h = P.hi[p];
	b.lo[0] = l.x, b.lo[1] = l.y, b.lo[2] = l.z;
	b.hi[0] = h.x, b.hi[1] = h.y, b.hi[2] = h.z;
	for (int a = 0; a < 3; a++) c[a] = 0.5f * (b.lo[a] + b.hi[a]);
}

// Binary node: lo.w = left child, hi.w = right child (as int bits), range =
// {first, count}; count > 0 marks a leaf.
struct Nodes2 {
	float4 *lo, *hi;
	int2 *range;
};

__device__ inline void writeNode(const Nodes2 &N, int i, const Box &b, int left, int right, int first, int count) {
	N.lo[i]	   = make_float4(b.lo[0], b.lo[1], b.lo[2], __int_as_float(left));
	N.hi[i]	   = make_float4(b.hi[0], b.hi[1], b.hi[2], __int_as_float(right));
	N.range[i] = make_int2(first, count);
}

// ------------------------------------------------------------ primitives

__global__ void k_prim_boxes(const float *pos, const int *idx, int n, float4 *lo, float4 *hi, int *refs) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	float l[3] = {__builtin_inff(), __builtin_inff(), __builtin_inff()}, h[3] = {-__builtin_inff(), -__builtin_inff(), -__builtin_inff()};
	for (int v = 0; v < 3; v++) {
		const int vi = idx[3 * (size_t) i + v];
		for (int a = 0; a < 3; a++) {
			const float x = pos[3 * (size_t) vi + a];
			l[a]		  = fminf(l[a], x);
			h[a]		  = fmaxf(h[a], x);
		}
	}
	lo[i]	= make_float4(l[0], l[1], l[2], 0.f);
	hi[i]	= make_float4(h[0], h[1], h[2], 0.f);
	refs[i] = i;
}

// ------------------------------------------------- large nodes, per level

// Per node of the level: first, count, binary node index; bounds and bins
// accumulated by the blocks of the node.
struct Level {
	const int *first, *count, *node;
	int *box;  // 6 ints per node: lo xyz, hi xyz (ordered)
	int *cbox; // centroid bounds, same layout
	Bins *bins;
	int *decision, *axis, *bin; // split per node
	int *nLeft;					// left references per node
	int *blockNode;				// node of each block
	int *blockStart;			// first reference of each block
	int *blockCnt;				// the axes' bin counts of each block's references
	int *childBox;				// per node 24 ints: bounds and centroid bounds of the left child, then the right
	const int *blockBegin;		// first block of each node (n + 1 entries)
	int *blockOff;				// left references of the node before each block (nodes of many blocks: k_level_offsets)
};

// One of the two node lists that the levels alternate between.
struct LevelList {
	int *first, *count, *node, *blockBegin, *box, *cbox;
};

// What the host reads between levels, and the running totals.
struct LevelCtl {
	int nodes, blocks;	 // of the next level
	int most;			 // blocks of its largest node, if more than kThreads
	int small, nextNode; // subtrees handed to k_small, binary nodes numbered so far
	int bad;			 // a split left a side empty
};

// Empty bounds, as ordered ints: entry e of a box is one of lo xyz, hi xyz.
__device__ inline int emptyBound(int e) { return e % 6 < 3 ? ordF(__builtin_inff()) : ordF(-__builtin_inff()); }

// Bins, child bounds and blocks of each node of the level.
__global__ void k_level_reset(Level L, int nNodes) {
	const int t = blockIdx.x;
	if (t >= nNodes) return;
	for (int e = threadIdx.x; e < 24; e += blockDim.x) L.childBox[24 * t + e] = emptyBound(e);
	binsReset(L.bins[t], threadIdx.x, blockDim.x);
	for (int b = L.blockBegin[t] + (int) threadIdx.x; b < L.blockBegin[t + 1]; b += blockDim.x) {
		L.blockNode[b]	= t;
		L.blockStart[b] = L.first[t] + (b - L.blockBegin[t]) * kChunk;
	}
}

__device__ inline float waveMin(float v) {
	for (int o = 32; o > 0; o >>= 1) v = fminf(v, __shfl_xor(v, o));
	return v;
}
__device__ inline float waveMax(float v) {
	for (int o = 32; o > 0; o >>= 1) v = fmaxf(v, __shfl_xor(v, o));
	return v;
}

// A wave's bounds and centroid bounds into twelve ordered ints.
__device__ inline void mergeBounds(int *to, const Box &box, const Box &cen) {
#pragma unroll
	for (int a = 0; a < 3; a++) {
		const float v[4] = {waveMin(box.lo[a]), waveMax(box.hi[a]), waveMin(cen.lo[a]), waveMax(cen.hi[a])};
		if (__lane_id() == 0) {
			atomicMin(&to[a], ordF(v[0]));
			atomicMax(&to[3 + a], ordF(v[1]));
			atomicMin(&to[6 + a], ordF(v[2]));
			atomicMax(&to[9 + a], ordF(v[3]));
		}
	}
}

__device__ inline void growCentroid(Box &cen, const float c[3]) {
	for (int a = 0; a < 3; a++) {
		cen.lo[a] = fminf(cen.lo[a], c[a]);
		cen.hi[a] = fmaxf(cen.hi[a], c[a]);
	}
}

// Bounds of the root (a child's come from the scatter of its parent), by few
// blocks: their atomics meet at twelve addresses.
constexpr int kRootBlocks = 128;
__global__ void __launch_bounds__(kThreads) k_root_bounds(Prims P, int n, int *box, int *cbox) {
	__shared__ int bounds[12];
	if (threadIdx.x < 12) bounds[threadIdx.x] = emptyBound(threadIdx.x);
	__syncthreads();
	Box bb, cb;
	bb.reset();
	cb.reset();
	for (int i = blockIdx.x * kThreads + (int) threadIdx.x; i < n; i += gridDim.x * kThreads) {
		Box pb;
		float c[3];
		primBox(P, i, pb, c);
		bb.grow(pb);
		growCentroid(cb, c);
	}
	mergeBounds(bounds, bb, cb);
	__syncthreads();
	const int e = threadIdx.x;
	if (e < 12) {
		int *to = e < 6 ? box + e : cbox + e - 6;
		if (e % 6 < 3) atomicMin(to, bounds[e]);
		else atomicMax(to, bounds[e]);
	}
}

__device__ inline Box loadBox(const int *p) {
	Box b;
	for (int a = 0; a < 3; a++) {
		b.lo[a] = unordF(p[a]);
		b.hi[a] = unordF(p[3 + a]);
	}
	return b;
}

__global__ void __launch_bounds__(kThreads) k_level_bins(Level L, Prims P, const int *refs) {
	__shared__ Bins sb;
	const int b = blockIdx.x, t = L.blockNode[b];
	binsReset(sb, threadIdx.x, kThreads);
	__syncthreads();
	const Box cb  = loadBox(L.cbox + 6 * t);
	const int end = min(L.blockStart[b] + kChunk, L.first[t] + L.count[t]);
	float scale[3];
	for (int a = 0; a < 3; a++) {
		const float ext = cb.hi[a] - cb.lo[a];
		scale[a]		= ext > 0 ? NB / ext : 0.f;
	}
	for (int i = L.blockStart[b] + (int) threadIdx.x; i < end; i += kThreads) {
		Box pb;
		float c[3];
		primBox(P, refs[i], pb, c);
		for (int a = 0; a < 3; a++) {
			if (!(scale[a] > 0)) continue;
			const int k = binOf(c[a], cb.lo[a], scale[a]);
			atomicAdd(&sb.cnt[a][k], 1);
			for (int e = 0; e < 3; e++) {
				atomicMin(&sb.lo[a][k][e], ordF(pb.lo[e]));
				atomicMax(&sb.hi[a][k][e], ordF(pb.hi[e]));
			}
		}
	}
	__syncthreads();
	Bins &g = L.bins[t];
	for (int i = threadIdx.x; i < 3 * NB; i += kThreads) {
		const int a = i / NB, k = i % NB;
		L.blockCnt[(size_t) b * 3 * NB + i] = sb.cnt[a][k];
		if (sb.cnt[a][k] == 0) continue;
		atomicAdd(&g.cnt[a][k], sb.cnt[a][k]);
		for (int e = 0; e < 3; e++) {
			atomicMin(&g.lo[a][k][e], sb.lo[a][k][e]);
			atomicMax(&g.hi[a][k][e], sb.hi[a][k][e]);
		}
	}
}

__global__ void __launch_bounds__(64) k_level_split(Level L, int nNodes, float nodeCost, int maxLeaf) {
	const int t = blockIdx.x, lane = threadIdx.x;
	if (t >= nNodes) return;
	const Box bb = loadBox(L.box + 6 * t), cb = loadBox(L.cbox + 6 * t);
	const int axis = min(lane >> 4, 2), k = lane & 15;
	Box own;
	own.reset();
	int cnt			= 0;
	const bool mine = lane < 48 && cb.hi[axis] - cb.lo[axis] > 0;
	if (mine) {
		const Bins &b = L.bins[t];
		cnt			  = b.cnt[axis][k];
		for (int e = 0; e < 3; e++) {
			own.lo[e] = unordF(b.lo[axis][k][e]);
			own.hi[e] = unordF(b.hi[axis][k][e]);
		}
	}
	int nPre;
	const Split s = waveSplit(own, cnt, mine, bb.area(), nodeCost, nPre);
	const int d	  = decide(s, L.count[t], maxLeaf);
	const int nl  = d == 0 ? __builtin_amdgcn_readlane(nPre, s.axis * 16 + s.bin) : L.count[t] / 2;
	if (lane == 0) {
		L.decision[t] = d;
		L.axis[t]	  = s.axis;
		L.bin[t]	  = s.bin;
		L.nLeft[t]	  = nl;
	}
}

__device__ inline bool goesLeft(const Level &L, int t, const Box &cb, float scale, int pos, float c) {
	if (L.decision[t] != 0) return pos < L.first[t] + L.count[t] / 2;
	return binOf(c, cb.lo[L.axis[t]], scale) <= L.bin[t];
}

__device__ inline float splitScale(const Level &L, int t, const Box &cb) {
	const int a = L.axis[t] < 0 ? 0 : L.axis[t];
	const float ext = cb.hi[a] - cb.lo[a];
	return ext > 0 ? NB / ext : 0.f;
}

// Left references of block e of node t.
__device__ inline int blockLefts(const Level &L, int t, int e) {
	if (L.decision[t] != 0) {
		const int size = min(kChunk, L.first[t] + L.count[t] - L.blockStart[e]);
		return min(max(L.first[t] + L.count[t] / 2 - L.blockStart[e], 0), size);
	}
	const int *cnt = L.blockCnt + (size_t) e * 3 * NB + L.axis[t] * NB;
	int n		   = 0;
	for (int k = 0; k <= L.bin[t]; k++) n += cnt[k];
	return n;
}

// Nodes of at most kThreads blocks have their earlier blocks' left references
// counted by each block of the scatter, one row per thread (a launch less).
// Those of larger nodes are added up once: counted by each block, the work
// grows with the square of the node.  Root's scatter 4.24 ms for 16.8 M triangles
// that way, 0.72 ms and 0.10 ms for the sums this way; 4.2 M 0.32 against 0.19 and
// 0.02 ms; 1.05 M 0.06 ms both.
__device__ inline bool offsetsListed(const Level &L, int t) { return L.blockBegin[t + 1] - L.blockBegin[t] > kThreads; }

__global__ void __launch_bounds__(1024) k_level_offsets(Level L) {
	const int t = blockIdx.x;
	if (!offsetsListed(L, t)) return;
	__shared__ int part[16];
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, end = L.blockBegin[t + 1];
	int carry = 0; // of the blocks before base
	for (int base = L.blockBegin[t]; base < end; base += 1024) {
		const int e	  = base + (int) threadIdx.x;
		const int own = e < end ? blockLefts(L, t, e) : 0;
		int incl	  = own;
		for (int o = 1; o < 64; o <<= 1) {
			const int u = __shfl_up(incl, o);
			if (lane >= o) incl += u;
		}
		if (lane == 63) part[wave] = incl;
		__syncthreads();
		int before = carry;
		for (int w = 0; w < 16; w++) {
			if (w < wave) before += part[w];
			carry += part[w];
		}
		if (e < end) L.blockOff[e] = before + incl - own;
		__syncthreads();
	}
}

// Stable partition: thread j of the block owns the references [per j, per j + per)
// of the block's chunk, in order.  The bounds of a child that is a large node
// itself are taken on the way.
__global__ void __launch_bounds__(kThreads) k_level_scatter(Level L, Prims P, const int *refs, int *tmp) {
	constexpr int per = kChunk / kThreads, waves = kThreads / 64;
	__shared__ int lefts[waves], earlier[waves], bounds[24];
	const int b = blockIdx.x, t = L.blockNode[b], lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const Box cb	  = loadBox(L.cbox + 6 * t);
	const float scale = splitScale(L, t, cb);
	const int ax	  = L.axis[t] < 0 ? 0 : L.axis[t];
	const int first = L.first[t], end = min(L.blockStart[b] + kChunk, first + L.count[t]);
	const int i0 = L.blockStart[b] + (int) threadIdx.x * per;
	if (threadIdx.x < 24) bounds[threadIdx.x] = emptyBound(threadIdx.x);
	int r[per];
	bool left[per];
	Box box[2], cen[2];
#pragma unroll
	for (int k = 0; k < 2; k++) {
		box[k].reset();
		cen[k].reset();
	}
#pragma unroll
	for (int k = 0; k < per; k++) {
		const int i = i0 + k;
		r[k]		= i < end ? refs[i] : -1;
		left[k]		= false;
		if (i < end) {
			Box pb;
			float c[3];
			primBox(P, r[k], pb, c);
			left[k] = goesLeft(L, t, cb, scale, i, c[ax]);
#pragma unroll
			for (int side = 0; side < 2; side++) {
				if (left[k] != (side == 0)) continue;
				box[side].grow(pb);
				growCentroid(cen[side], c);
			}
		}
	}
	// left references of the node's earlier blocks, of the block's earlier waves
	// and of the wave's earlier lanes
	int before		  = 0;
	const bool listed = offsetsListed(L, t);
	if (!listed && L.blockBegin[t] + (int) threadIdx.x < b) before = blockLefts(L, t, L.blockBegin[t] + (int) threadIdx.x);
	for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
	int leftBefore = 0, waveLefts = 0;
#pragma unroll
	for (int k = 0; k < per; k++) {
		const uint64_t m = __ballot(left[k]);
		leftBefore += __popcll(m & ((1ull << lane) - 1));
		waveLefts += __popcll(m);
	}
	if (lane == 0) {
		earlier[wave] = before;
		lefts[wave]	  = waveLefts;
	}
	__syncthreads();
	before = listed ? L.blockOff[b] : 0;
	for (int w = 0; w < waves; w++) {
		before += earlier[w];
		if (w < wave) leftBefore += lefts[w];
	}
	const int blockBefore = i0 - L.blockStart[b]; // references of earlier threads of this block
	int lp = first + before + leftBefore;
	int rp = first + L.nLeft[t] + (L.blockStart[b] - first - before) + (blockBefore - leftBefore);
#pragma unroll
	for (int k = 0; k < per; k++) {
		if (i0 + k >= end) break;
		if (left[k]) tmp[lp++] = r[k];
		else tmp[rp++] = r[k];
	}
	const int sizes[2] = {L.nLeft[t], L.count[t] - L.nLeft[t]};
#pragma unroll
	for (int side = 0; side < 2; side++) {
		if (sizes[side] <= kSmall) continue;
		mergeBounds(bounds + 12 * side, box[side], cen[side]);
	}
	__syncthreads();
	const int e = threadIdx.x;
	if (e < 24 && sizes[e / 12] > kSmall) {
		if (e % 6 < 3) atomicMin(&L.childBox[24 * t + e], bounds[e]);
		else atomicMax(&L.childBox[24 * t + e], bounds[e]);
	}
}

struct SmallTask {
	int node, first, count, nodeBase; // descendants take nodeBase, nodeBase + 1, ...
	int buf;						  // which of the two reference buffers holds the range
};

__global__ void k_level_init(LevelList list, SmallTask *small, LevelCtl *ctl, int n) {
	const bool large = n > kSmall;
	list.first[0]	 = 0;
	list.count[0]	 = n;
	list.node[0]	 = 0;
	list.blockBegin[0] = 0;
	for (int e = 0; e < 6; e++) list.box[e] = list.cbox[e] = emptyBound(e); // k_root_bounds fills them
	list.blockBegin[1] = (n + kChunk - 1) / kChunk;
	small[0]		 = SmallTask{0, 0, n, 1, 0};
	const int blocks = (n + kChunk - 1) / kChunk;
	*ctl			 = LevelCtl{large ? 1 : 0, blocks, blocks, large ? 0 : 1, large ? 1 : 2 * n - 1, 0};
}

// Binary nodes of the level, the next level's list and the subtrees that are
// small now (their references are in buffer `buf`), in the nodes' order: one
// block, 1024 nodes at a time, places by a scan.
__global__ void __launch_bounds__(1024) k_level_next(Level L, int nNodes, LevelList next, SmallTask *small, int buf, Nodes2 N, LevelCtl *ctl) {
	__shared__ int4 part[16];
	__shared__ int most;
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const int node0 = ctl->nextNode, small0 = ctl->small;
	if (threadIdx.x == 0) most = 0; // the loop's first barrier lies before its other uses
	int4 carry		= make_int4(0, 0, 0, 0); // large children, their blocks, small children, their descendants
	for (int base = 0; base < nNodes; base += 1024) {
		const int t	 = base + (int) threadIdx.x;
		const bool v = t < nNodes;
		int f[2] = {0, 0}, c[2] = {0, 0};
		int4 own = make_int4(0, 0, 0, 0);
		if (v) {
			f[0] = L.first[t];
			c[0] = L.nLeft[t];
			f[1] = f[0] + c[0];
			c[1] = L.count[t] - c[0];
			if (c[0] <= 0 || c[1] <= 0) ctl->bad = 1;
			writeNode(N, L.node[t], loadBox(L.box + 6 * t), node0 + 2 * t, node0 + 2 * t + 1, 0, 0);
			for (int k = 0; k < 2; k++) {
				if (c[k] > kSmall) own.x++, own.y += (c[k] + kChunk - 1) / kChunk;
				else own.z++, own.w += 2 * max(c[k], 1) - 2;
			}
		}
		int4 incl = own;
		for (int o = 1; o < 64; o <<= 1) {
			const int x = __shfl_up(incl.x, o), y = __shfl_up(incl.y, o), z = __shfl_up(incl.z, o), w = __shfl_up(incl.w, o);
			if (lane >= o) incl.x += x, incl.y += y, incl.z += z, incl.w += w;
		}
		if (lane == 63) part[wave] = incl;
		__syncthreads();
		int4 at = carry;
		for (int w = 0; w < 16; w++) {
			const int4 p = part[w];
			if (w < wave) at.x += p.x, at.y += p.y, at.z += p.z, at.w += p.w;
			carry.x += p.x, carry.y += p.y, carry.z += p.z, carry.w += p.w;
		}
		at.x += incl.x - own.x, at.y += incl.y - own.y, at.z += incl.z - own.z, at.w += incl.w - own.w;
		for (int k = 0; k < 2 && v; k++) {
			const int node = node0 + 2 * t + k;
			if (c[k] > kSmall) {
				next.first[at.x]	  = f[k];
				next.count[at.x]	  = c[k];
				next.node[at.x]		  = node;
				next.blockBegin[at.x] = at.y;
				for (int e = 0; e < 6; e++) {
					next.box[6 * at.x + e]	= L.childBox[24 * t + 12 * k + e];
					next.cbox[6 * at.x + e] = L.childBox[24 * t + 12 * k + 6 + e];
				}
				at.x++;
				at.y += (c[k] + kChunk - 1) / kChunk;
				if (c[k] > kThreads * kChunk) atomicMax(&most, (c[k] + kChunk - 1) / kChunk);
			} else {
				small[small0 + at.z] = SmallTask{node, f[k], c[k], node0 + 2 * nNodes + at.w, buf};
				at.z++;
				at.w += 2 * max(c[k], 1) - 2;
			}
		}
		__syncthreads();
	}
	if (threadIdx.x == 0) {
		next.blockBegin[carry.x] = carry.y;
		ctl->nodes				 = carry.x;
		ctl->blocks				 = carry.y;
		ctl->most				 = most;
		ctl->small				 = small0 + carry.z;
		ctl->nextNode			 = node0 + 2 * nNodes + carry.w;
	}
}

// -------------------------------------------- small subtrees, one per block

// One block builds the subtree of one task level by level, each wave taking
// nodes of the level in turn; references (as local indices), primitive boxes
// and the node lists stay in LDS (44 KB).
//
// A subtree of 1,024 triangles has about 1,000 nodes, most of two or three
// references, and a node's chain of passes is what bounds it: latency, not
// bandwidth.  So a node's work is spread over the lanes instead of repeated by
// each: lane (axis, bin) of 48 walks the node's references (broadcast LDS
// reads) and keeps its own bin's box and count, prefix and suffix boxes over the
// 16 bins are DPP scans within a row of 16 lanes, and each lane prices the split
// after its bin.  Minima, maxima and counts are exact in any order and the
// areas and costs are the host builder's expressions, so the tree is the same.
// One wave per subtree, with LDS atomics for the bins and every lane going
// through all 45 splits, took 14.9 ms for the 504 subtrees of 328 K triangles;
// this takes 1.23 ms, and is bound by vector issue (about 900 instructions a
// node).
constexpr int kSmallThreads = 512;

__global__ void __launch_bounds__(kSmallThreads) k_small(const SmallTask *tasks, int nTasks, Prims P, const int *refs1, int *refs, Nodes2 N, float nodeCost, int maxLeaf) {
	__shared__ float4 sLo[kSmall], sHi[kSmall]; // boxes of the task's primitives, in the order of the references at the start
	__shared__ uint16_t sRef[kSmall], sTmp[kSmall];
	__shared__ int2 sList[2][kSmall / 2]; // nodes of a level with at least two references: {node, first << 11 | count}
	__shared__ int sCount[2], sNodes;
	const int ti = blockIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	constexpr int waves = kSmallThreads / 64;
	if (ti >= nTasks) return;
	const SmallTask tk = tasks[ti];
	auto sBox = [&](int r) {
		const float4 l = sLo[r], h = sHi[r];
		Box b;
		b.lo[0] = l.x, b.lo[1] = l.y, b.lo[2] = l.z;
		b.hi[0] = h.x, b.hi[1] = h.y, b.hi[2] = h.z;
		return b;
	};
	for (int i = threadIdx.x; i < tk.count; i += kSmallThreads) {
		const int r = (tk.buf ? refs1 : refs)[tk.first + i];
		float4 l = P.lo[r];
		l.w	   = __int_as_float(r); // the reference travels with its box
		sLo[i] = l;
		sHi[i] = P.hi[r];
		sRef[i] = (uint16_t) i;
	}
	if (threadIdx.x == 0) {
		sList[0][0] = make_int2(tk.node, tk.count);
		sCount[0]	= 1;
		sNodes		= 0;
	}
	__syncthreads();
	if (tk.count < 2) { // a single reference is a leaf, as in the loop below
		if (threadIdx.x == 0 && tk.count == 1) {
			writeNode(N, tk.node, sBox(0), -1, -1, tk.first, 1);
			refs[tk.first] = __float_as_int(sLo[0].w);
		}
		return;
	}
	const int axis = min(lane >> 4, 2), bin = lane & 15;
	const bool binLane = lane < 48, ax0 = axis == 0, ax1 = axis == 1;
	// each level has fewer references per node than the one above, so there are
	// at most tk.count levels
	for (int cur = 0;; cur ^= 1) {
		const int nLevel = sCount[cur];
		if (nLevel == 0) break;
		__syncthreads();
		if (threadIdx.x == 0) sCount[cur ^ 1] = 0;
		__syncthreads();
		for (int q = wave; q < nLevel; q += waves) {
			const int2 e	= sList[cur][q];
			const int node	= __builtin_amdgcn_readfirstlane(e.x);
			const int first = __builtin_amdgcn_readfirstlane(e.y) >> 11, count = __builtin_amdgcn_readfirstlane(e.y) & 2047;
			// bounds and centroid bounds
			Box bb, cb;
			bb.reset();
			cb.reset();
			for (int i = first + lane; i < first + count; i += 64) {
				const Box pb = sBox(sRef[i]);
				bb.grow(pb);
				for (int a = 0; a < 3; a++) {
					const float c = 0.5f * (pb.lo[a] + pb.hi[a]);
					cb.lo[a]	  = fminf(cb.lo[a], c);
					cb.hi[a]	  = fmaxf(cb.hi[a], c);
				}
			}
			const bool wide = count > 16;
			auto mn = [](float x, float y) { return fminf(x, y); };
			auto mx = [](float x, float y) { return fmaxf(x, y); };
			for (int a = 0; a < 3; a++) {
				bb.lo[a] = rowReduce(bb.lo[a], mn, wide);
				bb.hi[a] = rowReduce(bb.hi[a], mx, wide);
				cb.lo[a] = rowReduce(cb.lo[a], mn, wide);
				cb.hi[a] = rowReduce(cb.hi[a], mx, wide);
			}
			// this lane's bin
			const float cLo = ax0 ? cb.lo[0] : (ax1 ? cb.lo[1] : cb.lo[2]), cHi = ax0 ? cb.hi[0] : (ax1 ? cb.hi[1] : cb.hi[2]);
			const float ext = cHi - cLo, scale = ext > 0 ? NB / ext : 0.f;
			const bool mine = binLane && scale > 0;
			Box own;
			own.reset();
			int cnt = 0;
#pragma unroll 4
			for (int i = first; i < first + count; i++) {
				const int r	   = sRef[i];
				const float4 l = sLo[r], h = sHi[r];
				const float c = 0.5f * ((ax0 ? l.x : (ax1 ? l.y : l.z)) + (ax0 ? h.x : (ax1 ? h.y : h.z)));
				if (mine && binOf(c, cLo, scale) == bin) {
					own.lo[0] = fminf(own.lo[0], l.x), own.lo[1] = fminf(own.lo[1], l.y), own.lo[2] = fminf(own.lo[2], l.z);
					own.hi[0] = fmaxf(own.hi[0], h.x), own.hi[1] = fmaxf(own.hi[1], h.y), own.hi[2] = fmaxf(own.hi[2], h.z);
					cnt++;
				}
			}
			int nPre;
			const Split s = waveSplit(own, cnt, mine, bb.area(), nodeCost, nPre);
			const int d = decide(s, count, maxLeaf);
			if (d == 1) {
				if (lane == 0) writeNode(N, node, bb, -1, -1, tk.first + first, count);
				continue;
			}
			// stable partition; the left count from the bins (binned split) or half
			int nLeft = count / 2;
			if (d == 0) {
				nLeft = __builtin_amdgcn_readlane(nPre, s.axis * 16 + s.bin);
				const float sLoA = s.axis == 0 ? cb.lo[0] : (s.axis == 1 ? cb.lo[1] : cb.lo[2]), sHiA = s.axis == 0 ? cb.hi[0] : (s.axis == 1 ? cb.hi[1] : cb.hi[2]);
				const float sScale = NB / (sHiA - sLoA);
				int nl = 0, nr = 0;
				uint16_t *dst = count <= 64 ? sRef : sTmp; // a node of one pass is read whole before it is written
				for (int base = first; base < first + count; base += 64) {
					const int i	 = base + lane;
					const bool v = i < first + count;
					int r		 = 0;
					bool left	 = false;
					if (v) {
						r				= sRef[i];
						const float4 l = sLo[r], h = sHi[r];
						const float c = 0.5f * (s.axis == 0 ? l.x + h.x : (s.axis == 1 ? l.y + h.y : l.z + h.z));
						left		  = binOf(c, sLoA, sScale) <= s.bin;
					}
					const uint64_t lm = __ballot(v && left), rm = __ballot(v && !left);
					const uint64_t below = lane == 0 ? 0ull : (~0ull >> (64 - lane));
					const int slot = left ? first + nl + __popcll(lm & below) : first + nLeft + nr + __popcll(rm & below);
					if (v && slot < first + count) dst[slot] = (uint16_t) r; // always in range: nl ends equal to nLeft
					nl += __popcll(lm);
					nr += __popcll(rm);
				}
				if (count > 64) {
					__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
					for (int i = first + lane; i < first + count; i += 64) sRef[i] = sTmp[i];
				}
			}
			__builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); // other lanes' sRef entries are read from here on
			// children: two or more references go to the next level's list, a
			// single one is a leaf.  A side is never empty (binned splits skip
			// empty sides, middle splits halve at least 9 references).
			if (lane == 0) {
				const int l = tk.nodeBase + 2 * atomicAdd(&sNodes, 1);
				writeNode(N, node, bb, l, l + 1, 0, 0);
				for (int k = 0; k < 2; k++) {
					const int f = k ? first + nLeft : first, c = k ? count - nLeft : nLeft;
					if (c > 1) sList[cur ^ 1][atomicAdd(&sCount[cur ^ 1], 1)] = make_int2(l + k, (f << 11) | c);
					else writeNode(N, l + k, sBox(sRef[f]), -1, -1, tk.first + f, 1);
				}
			}
		}
		__syncthreads();
	}
	for (int i = threadIdx.x; i < tk.count; i += kSmallThreads) refs[tk.first + i] = __float_as_int(sLo[sRef[i]].w);
}

// ------------------------------------------------------------- collapse

__device__ inline void padBox(float &lo, float &hi) {
	const float pad = (fabsf(lo) + fabsf(hi) + (hi - lo)) * 9.5367431640625e-07f; // 2^-20, as the host builder
	lo -= pad;
	hi += pad;
}

__device__ inline float nodeArea(const Nodes2 &N, int i) {
	const float4 l = N.lo[i], h = N.hi[i];
	Box b;
	b.lo[0] = l.x, b.lo[1] = l.y, b.lo[2] = l.z;
	b.hi[0] = h.x, b.hi[1] = h.y, b.hi[2] = h.z;
	return b.area();
}

// Children of the 4-wide node made from binary node b: open the inner child
// with the largest area (first maximum) until four children or only leaves.
__device__ int collapseKids(const Nodes2 &N, int b, int kids[4]) {
	int nk = 0;
	if (N.range[b].y > 0) {
		kids[nk++] = b;
		return nk;
	}
	kids[nk++] = __float_as_int(N.lo[b].w);
	kids[nk++] = __float_as_int(N.hi[b].w);
	while (nk < 4) {
		int best = -1;
		float ba = -1.f;
		for (int k = 0; k < nk; k++) {
			if (N.range[kids[k]].y > 0) continue;
			const float a = nodeArea(N, kids[k]);
			if (a > ba) {
				ba	 = a;
				best = k;
			}
		}
		if (best < 0) break;
		const int c = kids[best];
		kids[best]	= __float_as_int(N.lo[c].w);
		kids[nk++]	= __float_as_int(N.hi[c].w);
	}
	return nk;
}

// Inner children of each node of the level, summed per block of 256.
__global__ void __launch_bounds__(256) k_collapse_count(Nodes2 N, const int *level, int n, int *blockSum) {
	__shared__ int part[4];
	const int i = blockIdx.x * 256 + threadIdx.x;
	int c		= 0;
	if (i < n) {
		int kids[4];
		const int nk = collapseKids(N, level[i], kids);
		for (int k = 0; k < nk; k++) c += N.range[kids[k]].y > 0 ? 0 : 1;
	}
	for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
	if (__lane_id() == 0) part[threadIdx.x / 64] = c;
	__syncthreads();
	if (threadIdx.x == 0) blockSum[blockIdx.x] = part[0] + part[1] + part[2] + part[3];
}

// The level's 4-wide nodes; the inner children's places in the next level are
// the sum of the earlier blocks' counts and a scan within the block.  (The sums
// are few: 256 nodes a block; with the counts scanned by a launch of its own the
// emissions of 16.8 M triangles took 1.24 ms as well.)
__global__ void __launch_bounds__(256) k_collapse_emit(Nodes2 N, const int *level, int n, int levelBase, const int *blockSum, int nextBase,
													   int *nextLevel, Bvh4Node *out, int *total) {
	__shared__ int earlier[4], part[4];
	const int i = blockIdx.x * 256 + threadIdx.x, lane = threadIdx.x & 63, wave = threadIdx.x / 64;
	int before = 0;
	for (int e = (int) threadIdx.x; e < (int) blockIdx.x; e += 256) before += blockSum[e];
	for (int o = 32; o > 0; o >>= 1) before += __shfl_xor(before, o);
	int kids[4];
	const int nk = i < n ? collapseKids(N, level[i], kids) : 0;
	int own		 = 0;
	for (int k = 0; k < nk; k++) own += N.range[kids[k]].y > 0 ? 0 : 1;
	int incl = own;
	for (int o = 1; o < 64; o <<= 1) {
		const int u = __shfl_up(incl, o);
		if (lane >= o) incl += u;
	}
	if (lane == 0) earlier[wave] = before;
	if (lane == 63) part[wave] = incl;
	__syncthreads();
	int off = earlier[0] + earlier[1] + earlier[2] + earlier[3] + incl - own;
	for (int w = 0; w < wave; w++) off += part[w];
	if (i == n - 1) *total = off + own;
	if (i >= n) return;
	Bvh4Node node;
	for (int c = 0; c < 4; c++) {
		node.lox[c] = node.loy[c] = node.loz[c] = __builtin_inff();
		node.hix[c] = node.hiy[c] = node.hiz[c] = -__builtin_inff();
		node.child[c] = -1;
		node.pad[c]	  = 0;
	}
	int j = 0;
	for (int c = 0; c < nk; c++) {
		const int k	   = kids[c];
		const float4 l = N.lo[k], h = N.hi[k];
		float lx = l.x, hx = h.x, ly = l.y, hy = h.y, lz = l.z, hz = h.z;
		padBox(lx, hx);
		padBox(ly, hy);
		padBox(lz, hz);
		node.lox[c] = lx;
		node.hix[c] = hx;
		node.loy[c] = ly;
		node.hiy[c] = hy;
		node.loz[c] = lz;
		node.hiz[c] = hz;
		const int2 r = N.range[k];
		if (r.y > 0) node.child[c] = ~(r.x * 8 + (r.y - 1));
		else {
			const int slot	= off + j++;
			node.child[c]	= nextBase + slot;
			nextLevel[slot] = k;
		}
	}
	out[levelBase + i] = node;
}

__global__ void k_leaf_tris(const float *pos, const int *idx, const unsigned char *nullFlag, const int *refs, int n, LeafTri *tris) {
	const int i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= n) return;
	const int p = refs[i];
	LeafTri t;
	for (int a = 0; a < 3; a++) {
		t.v0[a] = pos[3 * (size_t) idx[3 * (size_t) p] + a];
		t.v1[a] = pos[3 * (size_t) idx[3 * (size_t) p + 1] + a];
		t.v2[a] = pos[3 * (size_t) idx[3 * (size_t) p + 2] + a];
	}
	t.prim	= p;
	t.flags = nullFlag ? (int32_t) (nullFlag[p] & (kLeafNull | kLeafAlpha)) : 0;
	t.pad	= 0;
	tris[i] = t;
}

// ------------------------------------------------------------------ host

struct Buf {
	void *p = nullptr;
	~Buf() {
		if (p) (void) hipFree(p);
	}
	hipError_t alloc(size_t bytes) {
		if (p) (void) hipFree(p);
		p = nullptr;
		return hipMalloc(&p, std::max<size_t>(bytes, 16));
	}
	template <class T> T *as() const { return reinterpret_cast<T *>(p); }
};

#define BVHD_HIP(x)                                                                                                                        \
	do {                                                                                                                                   \
		hipError_t e_ = (x);                                                                                                               \
		if (e_ != hipSuccess) {                                                                                                            \
			err = std::string(#x) + ": " + hipGetErrorString(e_);                                                                          \
			return -1;                                                                                                                     \
		}                                                                                                                                  \
	} while (0)

// Every temporary of a build in one allocation: sizes are added up first (null
// base), then taken again from the block.
struct Arena {
	char *base	= nullptr;
	size_t used = 0;
	template <class T> T *take(size_t count) {
		used		= (used + 255) / 256 * 256;
		T *p		= reinterpret_cast<T *>(base + used);
		used	   += count * sizeof(T);
		return p;
	}
};

} // namespace bvhdev

using namespace bvhdev;

int buildBvh4Device(const float *pos, int64_t nVerts, const int32_t *idx, int64_t nTris, const uint8_t *nullFlag, const BvhBuildOptions &opt,
					DeviceBvh &out, std::string &err) {
	const auto t0 = std::chrono::steady_clock::now();
	out			  = DeviceBvh{};
	if (nTris <= 0 || nTris > (int64_t) 0x0fffffff) {
		err = "device BVH build needs 1 .. 2^28 triangles";
		return -1;
	}
	const int n		  = (int) nTris;
	const int maxLeaf = std::max(1, std::min(8, opt.maxLeafSize));
	const float cost  = std::max(0.f, opt.nodeCost);
	hipStream_t st	  = nullptr;
	BVHD_HIP(hipStreamCreateWithFlags(&st, hipStreamNonBlocking));
	struct StreamGuard {
		hipStream_t s;
		~StreamGuard() { (void) hipStreamDestroy(s); }
	} guard{st};
	// at most one large node per kSmall + 1 references of a level, and a block
	// per kChunk references or part of them
	const size_t maxT = (size_t) n / (kSmall + 1) + 1, maxB = (size_t) n / kChunk + maxT + 1, maxNodes2 = 2 * (size_t) n;
	float *dPos;
	int *dIdx, *refs[2];
	unsigned char *dNull;
	float4 *pLo, *pHi, *nLo, *nHi;
	int2 *nRange;
	LevelList list[2];
	Level L;
	SmallTask *small;
	LevelCtl *ctl;
	int *total;
	auto layout = [&](Arena &m) {
		dPos   = m.take<float>((size_t) nVerts * 3);
		dIdx   = m.take<int>((size_t) n * 3);
		dNull  = m.take<unsigned char>((size_t) n);
		pLo	   = m.take<float4>((size_t) n);
		pHi	   = m.take<float4>((size_t) n);
		nLo	   = m.take<float4>(maxNodes2);
		nHi	   = m.take<float4>(maxNodes2);
		nRange = m.take<int2>(maxNodes2);
		for (int k = 0; k < 2; k++) {
			refs[k] = m.take<int>((size_t) n);
			list[k] = LevelList{m.take<int>(maxT), m.take<int>(maxT), m.take<int>(maxT), m.take<int>(maxT + 1), m.take<int>(6 * maxT), m.take<int>(6 * maxT)};
		}
		L		   = Level{};
		L.childBox = m.take<int>(24 * maxT);
		L.bins	   = m.take<Bins>(maxT);
		L.decision = m.take<int>(maxT);
		L.axis	   = m.take<int>(maxT);
		L.bin	   = m.take<int>(maxT);
		L.nLeft	   = m.take<int>(maxT);
		L.blockNode	 = m.take<int>(maxB);
		L.blockStart = m.take<int>(maxB);
		L.blockCnt	 = m.take<int>(3 * NB * maxB);
		L.blockOff	 = m.take<int>(maxB);
		small		 = m.take<SmallTask>((size_t) n);
		ctl			 = m.take<LevelCtl>(1);
		total		 = m.take<int>(1);
	};
	Arena size, arena;
	layout(size);
	Buf block;
	BVHD_HIP(block.alloc(size.used));
	arena.base = block.as<char>();
	layout(arena);
	BVHD_HIP(hipMemcpyAsync(dPos, pos, (size_t) nVerts * 3 * sizeof(float), hipMemcpyHostToDevice, st));
	BVHD_HIP(hipMemcpyAsync(dIdx, idx, (size_t) n * 3 * sizeof(int), hipMemcpyHostToDevice, st));
	if (nullFlag) BVHD_HIP(hipMemcpyAsync(dNull, nullFlag, (size_t) n, hipMemcpyHostToDevice, st));
	else BVHD_HIP(hipMemsetAsync(dNull, 0, (size_t) n, st));
	BVHD_HIP(hipStreamSynchronize(st));
	const auto tUp = std::chrono::steady_clock::now();
	const Prims P{pLo, pHi};
	const Nodes2 N{nLo, nHi, nRange};
	hipLaunchKernelGGL(k_prim_boxes, dim3((n + 255) / 256), dim3(256), 0, st, dPos, dIdx, n, pLo, pHi, refs[0]);
	hipLaunchKernelGGL(k_level_init, dim3(1), dim3(1), 0, st, list[0], small, ctl, n);

	if (n > kSmall)
		hipLaunchKernelGGL(k_root_bounds, dim3(std::min(kRootBlocks, (n + kThreads - 1) / kThreads)), dim3(kThreads), 0, st, P, n, list[0].box, list[0].cbox);
	BVHD_HIP(hipGetLastError());

	// ---- large nodes, level by level: the lists stay on the device, the host
	// reads the next level's size (uploading the lists and allocating their
	// buffers anew per level took 6 of the 8.4 ms of a 328 K-triangle build)
	LevelCtl c{};
	BVHD_HIP(hipMemcpyAsync(&c, ctl, sizeof(c), hipMemcpyDeviceToHost, st));
	BVHD_HIP(hipStreamSynchronize(st));
	int levels = 0, cur = 0;
	while (c.nodes > 0) {
		const int T = c.nodes, B = c.blocks;
		// guards against a malformed level; a split always leaves fewer references a node
		if ((size_t) T > maxT || (size_t) B > maxB || levels > n) {
			err = "device BVH build: malformed level";
			return -1;
		}
		L.first		 = list[cur].first;
		L.count		 = list[cur].count;
		L.node		 = list[cur].node;
		L.blockBegin = list[cur].blockBegin;
		L.box		 = list[cur].box;
		L.cbox		 = list[cur].cbox;
		const int *in = refs[levels & 1];
		int *to		  = refs[(levels & 1) ^ 1];
		hipLaunchKernelGGL(k_level_reset, dim3(T), dim3(256), 0, st, L, T);
		hipLaunchKernelGGL(k_level_bins, dim3(B), dim3(kThreads), 0, st, L, P, in);
		hipLaunchKernelGGL(k_level_split, dim3(T), dim3(64), 0, st, L, T, cost, maxLeaf);
		if (c.most > kThreads) hipLaunchKernelGGL(k_level_offsets, dim3(T), dim3(1024), 0, st, L);
		hipLaunchKernelGGL(k_level_scatter, dim3(B), dim3(kThreads), 0, st, L, P, in, to);
		hipLaunchKernelGGL(k_level_next, dim3(1), dim3(1024), 0, st, L, T, list[cur ^ 1], small, (levels & 1) ^ 1, N, ctl);
		BVHD_HIP(hipGetLastError());
		BVHD_HIP(hipMemcpyAsync(&c, ctl, sizeof(c), hipMemcpyDeviceToHost, st));
		BVHD_HIP(hipStreamSynchronize(st));
		if (c.bad) {
			err = "device BVH build: empty side in a large-node split";
			return -1;
		}
		cur ^= 1;
		levels++;
	}
	const auto tLarge = std::chrono::steady_clock::now();
	// ---- small subtrees, one block each; descendants numbered per subtree
	if ((size_t) c.nextNode > maxNodes2 || c.small > n) {
		err = "device BVH build: node count overflow";
		return -1;
	}
	if (c.small > 0) {
		hipLaunchKernelGGL(k_small, dim3((unsigned) c.small), dim3(kSmallThreads), 0, st, small, c.small, P, refs[1], refs[0], N, cost, maxLeaf);
		BVHD_HIP(hipGetLastError());
		BVHD_HIP(hipStreamSynchronize(st));
	}
	const auto tSmall = std::chrono::steady_clock::now();
	// ---- collapse to 4-wide nodes, level by level; the level lists and block
	// sums take the place of the primitive boxes and the second references
	Buf nodes4, tris;
	int *lvl[2]	  = {reinterpret_cast<int *>(pLo), reinterpret_cast<int *>(pHi)};
	int *blockSum = refs[1];
	// at most one 4-wide node per inner binary node, plus the root
	const size_t cap4 = (size_t) c.nextNode / 2 + 1;
	BVHD_HIP(nodes4.alloc(cap4 * sizeof(Bvh4Node)));
	const int zero = 0;
	BVHD_HIP(hipMemcpyAsync(lvl[0], &zero, sizeof(int), hipMemcpyHostToDevice, st));
	int levelN = 1, levelBase = 0, depth = 0;
	cur = 0;
	while (levelN > 0) {
		depth++;
		// a well-formed tree never trips these; they keep a malformed one from
		// writing past the node array or looping
		if (depth > 64 || (size_t) levelBase + (size_t) levelN > cap4 || levelN > n) {
			err = "device BVH build: malformed tree in the 4-wide collapse";
			return -1;
		}
		const unsigned g   = (unsigned) ((levelN + 255) / 256);
		const int nextBase = levelBase + levelN;
		hipLaunchKernelGGL(k_collapse_count, dim3(g), dim3(256), 0, st, N, (const int *) lvl[cur], levelN, blockSum);
		hipLaunchKernelGGL(k_collapse_emit, dim3(g), dim3(256), 0, st, N, (const int *) lvl[cur], levelN, levelBase, (const int *) blockSum, nextBase,
						   lvl[cur ^ 1], nodes4.as<Bvh4Node>(), total);
		BVHD_HIP(hipGetLastError());
		int nextN = 0;
		BVHD_HIP(hipMemcpyAsync(&nextN, total, sizeof(int), hipMemcpyDeviceToHost, st));
		BVHD_HIP(hipStreamSynchronize(st));
		levelBase = nextBase;
		levelN	  = nextN;
		cur ^= 1;
	}
	BVHD_HIP(tris.alloc((size_t) n * sizeof(LeafTri)));
	hipLaunchKernelGGL(k_leaf_tris, dim3((n + 255) / 256), dim3(256), 0, st, (const float *) dPos, (const int *) dIdx, (const unsigned char *) dNull,
					   (const int *) refs[0], n, tris.as<LeafTri>());
	BVHD_HIP(hipGetLastError());
	BVHD_HIP(hipStreamSynchronize(st));
	out.nodes	   = nodes4.p;
	out.tris	   = tris.p;
	nodes4.p	   = nullptr;
	tris.p		   = nullptr;
	out.nNodes	   = levelBase;
	out.nTris	   = n;
	out.nBinary	   = c.nextNode;
	out.maxDepth   = depth;
	out.largeLevels = levels;
	out.smallTrees = c.small;
	const auto t1  = std::chrono::steady_clock::now();
	out.seconds	   = std::chrono::duration<double>(t1 - t0).count();
	out.buildSeconds = std::chrono::duration<double>(t1 - tUp).count();
	out.largeSeconds = std::chrono::duration<double>(tLarge - tUp).count();
	out.smallSeconds = std::chrono::duration<double>(tSmall - tLarge).count();
	out.collapseSeconds = std::chrono::duration<double>(t1 - tSmall).count();
	return 0;
}

} // namespace krr
