// gfx950 kernels of the baking hot path and the DeviceScene that owns their
// device-resident data.  See device.h for the stage contracts.
//
// Query semantics (all order independent, hence equal to the reference's
// tree walks):
//  * distance(p): min(2, min over shadow triangles of PointTriangleDistance)
//    (lighter.cpp:150-188);
//  * closest(A,B): min over triangles of the segment hit parameter on A->B
//    shrunk by 0.001 at both ends, 2 when nothing is hit (lighter.cpp:254-289);
//  * occluded(A,B): some triangle hit with r < 1 on the same shrunk segment
//    (lighter.cpp:112-147).
#include <hip/hip_runtime.h>
#include <mutex>
#include <stdlib.h>

#include <math.h>
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <chrono>
#include <set>
#include <stdexcept>
#include <string>
#include <thread>
#include <vector>

#include "bvh.h"
#include "device.h"
#include "geom.h"
#include "normals.h"

namespace lgx {

#define HIPCHECK(x)                                                                                          \
	do {                                                                                                     \
		hipError_t e_ = (x);                                                                                 \
		if (e_ != hipSuccess)                                                                                \
			throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e_) + " at " __FILE__ ":" + \
			                         std::to_string(__LINE__) + ": " #x);                                    \
	} while (0)

constexpr int kStackSize = 96; // >= 3 x (wide BVH depth) + 1, checked at build
constexpr int kBlock = 256;
constexpr int kNumCounters = 6;
constexpr uint32_t kSkipBits = 0xFFFFFFFFu; // weight of a texel the reference skips
constexpr uint32_t kSampleBits = 26;
constexpr uint32_t kSampleMask = (1u << kSampleBits) - 1;

struct View {
	const WideNode* __restrict__ nodes;
	const DistTri* __restrict__ dtri;
	const RayTri* __restrict__ rtri;
	int has_tris;
	// scene box grown by the distance-query radius plus a safety margin:
	// outside it every distance query returns exactly 2
	float xlo[3], xhi[3];
	// entry grid: cell (ix, iy, iz) of size 1 / ginv from glo; its entry node
	// is nodes[gbase + (iz * gn[1] + iy) * gn[0] + ix]; gbase = 0: no grid
	float glo[3], ginv;
	int gn[3];
	int32_t gbase;
	// the same cells again from gfine on, each a cut for the cell grown by
	// kGridFineReach only, for distance queries of radius <= 1 (0: none)
	int32_t gfine;
};

// The entry grid.  Every query of the kernels here that is local (a distance
// query of radius <= kGridReach, a segment no longer than kGridReach) can
// only be answered by triangles that meet the ball of that radius around
// its point (the segment's start).  Each cell of a uniform grid over the
// scene holds a virtual wide node (after the tree's nodes) whose children
// are a cut of the tree: at most four subtrees such that every triangle
// meeting the cell grown by kGridReach (plus a rounding margin) lies in one
// of them.  A second node per cell (from gfine on) is the same cut for the
// cell grown by kGridFineReach only, for distance queries of radius <= 1:
// a smaller region, a deeper cut.  A local query starts at its cell's node
// instead of the root, so it skips the levels above the cut and still
// meets every triangle that can change its answer; its result is the same
// minimum.
constexpr float kGridReach = kPenumbraSize;
constexpr float kGridFineReach = kPenumbraStep; // 1 m: the radius of many march queries
constexpr uint32_t kGridCells = 1u << 22; // cells at most (two nodes of 128 bytes each, 1 GB)
constexpr float kGridMinCell = 1.0f;      // metres: finer cells gain nothing against the 2 m reach

// entry node of a query at p (the root outside the grid); fine: the query's
// radius is at most kGridFineReach
__device__ __forceinline__ int32_t entry_node(const View& V, f3 p, bool fine = false)
{
	if (!V.gbase)
		return 0;
	const float fx = (p.x - V.glo[0]) * V.ginv, fy = (p.y - V.glo[1]) * V.ginv, fz = (p.z - V.glo[2]) * V.ginv;
	if (!(fx >= 0.0f && fy >= 0.0f && fz >= 0.0f && fx < (float)V.gn[0] && fy < (float)V.gn[1] &&
	      fz < (float)V.gn[2]))
		return 0;
	const int ix = min((int)fx, V.gn[0] - 1), iy = min((int)fy, V.gn[1] - 1), iz = min((int)fz, V.gn[2] - 1);
	return (fine && V.gfine ? V.gfine : V.gbase) + (iz * V.gn[1] + iy) * V.gn[0] + ix;
}

// ---------------------------------------------------------------------------
// transcendental helpers: evaluated in double and rounded once, which is the
// correctly rounded value except in vanishingly rare ties
// ---------------------------------------------------------------------------
__device__ __forceinline__ float pow_r(float x, float y)
{
	if (y == 1.0f)
		return x;
	return (float)pow((double)x, (double)y);
}
__device__ __forceinline__ float acos_r(float x) { return (float)acos((double)x); }

struct WNode {
	float4 lx, ly, lz, hx, hy, hz; // the four children's boxes, one plane per float4
	int4 c;                        // their references
};

__device__ __forceinline__ WNode load_node(const WideNode* nodes, int32_t i)
{
	const float4* q = reinterpret_cast<const float4*>(nodes + i);
	WNode n;
	n.lx = q[0];
	n.ly = q[1];
	n.lz = q[2];
	n.hx = q[3];
	n.hy = q[4];
	n.hz = q[5];
	n.c = reinterpret_cast<const int4*>(q)[6];
	return n;
}

// ascending order of (key, reference) pairs
__device__ __forceinline__ void cswap(float& ka, int32_t& ra, float& kb, int32_t& rb)
{
	const bool sw = kb < ka;
	const float k = sw ? kb : ka;
	kb = sw ? ka : kb;
	ka = k;
	const int32_t r = sw ? rb : ra;
	rb = sw ? ra : rb;
	ra = r;
}

__device__ __forceinline__ void sort4(float (&k)[4], int32_t (&r)[4])
{
	cswap(k[0], r[0], k[1], r[1]);
	cswap(k[2], r[2], k[3], r[3]);
	cswap(k[0], r[0], k[2], r[2]);
	cswap(k[1], r[1], k[3], r[3]);
	cswap(k[1], r[1], k[2], r[2]);
}

__device__ __forceinline__ float box_d2(f3 p, float lx, float ly, float lz, float hx, float hy, float hz)
{
	float dx = fmaxf(fmaxf(lx - p.x, p.x - hx), 0.0f);
	float dy = fmaxf(fmaxf(ly - p.y, p.y - hy), 0.0f);
	float dz = fmaxf(fmaxf(lz - p.z, p.z - hz), 0.0f);
	return dx * dx + dy * dy + dz * dz;
}

__device__ __forceinline__ DistTri load_dtri(const DistTri* t, uint32_t i)
{
	const float4* q = reinterpret_cast<const float4*>(t + i);
	DistTri r;
	float4* o = reinterpret_cast<float4*>(&r);
#pragma unroll
	for (int k = 0; k < 10; ++k)
		o[k] = q[k];
	return r;
}

__device__ __forceinline__ RayTri load_rtri(const RayTri* t, uint32_t i)
{
	const float4* q = reinterpret_cast<const float4*>(t + i);
	RayTri r;
	float4* o = reinterpret_cast<float4*>(&r);
#pragma unroll
	for (int k = 0; k < 4; ++k)
		o[k] = q[k];
	return r;
}

typedef float v4f __attribute__((ext_vector_type(4)));

// True when the triangle cannot lower the distance bound `best`: the box of
// its three vertices (DistTri quads 4-6, qa..qc) lies farther than best +
// margin.
// The distance the reference's formula returns is the distance to a point of
// the triangle (a vertex, a point of an edge line inside the edge's span, or
// the projection into the face), up to rounding in its region tests of a few
// ulps of the coordinates, so it is never below the box distance minus that;
// the margin (1e-5 of the coordinates' magnitude, hundreds of ulps) covers
// it, and a skipped triangle could only have returned a value >= best, which
// leaves the minimum unchanged.
__device__ __forceinline__ bool tri_box_beyond_q(f3 p, v4f qa, v4f qb, v4f qc, float best)
{
	// vertices (qa.w, qb.x, qb.y), (qb.z, qb.w, qc.x), (qc.y, qc.z, qc.w)
	float lx = fminf(fminf(qa.w, qb.z), qc.y), hx = fmaxf(fmaxf(qa.w, qb.z), qc.y);
	float ly = fminf(fminf(qb.x, qb.w), qc.z), hy = fmaxf(fmaxf(qb.x, qb.w), qc.z);
	float lz = fminf(fminf(qb.y, qc.x), qc.w), hz = fmaxf(fmaxf(qb.y, qc.x), qc.w);
	float lim = best + 1e-5f * (1.0f + fabsf(p.x) + fabsf(p.y) + fabsf(p.z));
	return box_d2(p, lx, ly, lz, hx, hy, hz) > lim * lim;
}

// Traversal stacks.  The traversals below are nearest-first: at an inner
// node they descend into the nearest child and push the other (at most
// three) children that are still within reach, so the stack holds at most
// three entries per level of the current path and 3 x the BVH's depth + 1
// bounds it.
// Entry = node reference + key (squared box distance, or the segment's entry
// parameter); a popped entry is skipped when its key exceeds the current
// bound.
struct PrivStack { // per-lane arrays (private segment)
	int32_t ref[kStackSize];
	float key[kStackSize];
	__device__ __forceinline__ void put(int i, int32_t r, float k)
	{
		ref[i] = r;
		key[i] = k;
	}
	__device__ __forceinline__ int32_t r(int i) const { return ref[i]; }
	__device__ __forceinline__ float k(int i) const { return key[i]; }
};

// A column of LDS per lane: references [level][lane] as int32, keys as FP16
// rounded toward zero.  Keys are non-negative, so the stored key never
// exceeds the true one and skipping stays conservative: at worst a node is
// visited that the exact key would have skipped, which changes no result.
__device__ __forceinline__ _Float16 f16_down(float x)
{
	_Float16 h = (_Float16)x;
	if ((float)h > x) {
		uint16_t b;
		memcpy(&b, &h, 2);
		b = (uint16_t)(b - 1); // x >= 0 and h > x imply h > 0
		memcpy(&h, &b, 2);
	}
	return h;
}

// The first kLdsLevels levels in LDS, deeper ones (rare: only a path that
// pushed at more than kLdsLevels of its levels) in a per-lane array.
constexpr int kLdsLevels = 12;

// LDS-qualified element types: through a generic pointer the stack would be
// accessed with FLAT instructions, which count against both the vector-memory
// and the LDS wait counters (every node fetch would then wait for the stack's
// stores and vice versa)
typedef __attribute__((address_space(3))) int32_t lds_int32_t;
typedef __attribute__((address_space(3))) _Float16 lds_half_t;

struct LdsStack {
	lds_int32_t* ref; // &refs[0][lane]
	lds_half_t* key;  // &keys[0][lane]
	int32_t oref[kStackSize - kLdsLevels];
	float okey[kStackSize - kLdsLevels];
	__device__ __forceinline__ void put(int i, int32_t r, float k)
	{
		if (i < kLdsLevels) {
			ref[i * kBlock] = r;
			key[i * kBlock] = f16_down(k);
		} else {
			oref[i - kLdsLevels] = r;
			okey[i - kLdsLevels] = k;
		}
	}
	__device__ __forceinline__ int32_t r(int i) const { return i < kLdsLevels ? ref[i * kBlock] : oref[i - kLdsLevels]; }
	__device__ __forceinline__ float k(int i) const
	{
		return i < kLdsLevels ? (float)key[i * kBlock] : okey[i - kLdsLevels];
	}
};

// The calling lane's LDS stack in the kernel's dynamic LDS (kBlock x depth
// int32 references, then kBlock x depth FP16 keys).
__device__ __forceinline__ LdsStack lds_stack_of_lane(unsigned char* lds, int depth)
{
	LdsStack st;
	st.ref = (lds_int32_t*)(reinterpret_cast<int32_t*>(lds) + threadIdx.x);
	st.key = (lds_half_t*)(reinterpret_cast<_Float16*>(lds + 4 * (size_t)kBlock * depth) + threadIdx.x);
	return st;
}

// Nearest-first traversal for the distance query: min(radius, distance to the
// nearest triangle closer than radius).
template <bool COUNT, class Stack>
__device__ float q_distance(const View& V, f3 p, float radius, unsigned long long* cnt, Stack& st)
{
	float best = radius;
	if (!V.has_tris)
		return best;
	int sp = 0;
	int32_t ref = radius <= kGridReach ? entry_node(V, p, radius <= kGridFineReach) : 0;
	unsigned nn = 0, nt = 0, ncull = 0;
	for (;;) {
		if (ref >= 0) {
			WNode n = load_node(V.nodes, ref);
			nn++;
			float d[4] = {box_d2(p, n.lx.x, n.ly.x, n.lz.x, n.hx.x, n.hy.x, n.hz.x),
			              box_d2(p, n.lx.y, n.ly.y, n.lz.y, n.hx.y, n.hy.y, n.hz.y),
			              box_d2(p, n.lx.z, n.ly.z, n.lz.z, n.hx.z, n.hy.z, n.hz.z),
			              box_d2(p, n.lx.w, n.ly.w, n.lz.w, n.hx.w, n.hy.w, n.hz.w)};
			int32_t r[4] = {n.c.x, n.c.y, n.c.z, n.c.w};
			sort4(d, r);
			float lim = best * best;
			if (d[0] <= lim) {
				// farthest first, so that the nearer ones pop first
				if (d[3] <= lim)
					st.put(sp++, r[3], d[3]);
				if (d[2] <= lim)
					st.put(sp++, r[2], d[2]);
				if (d[1] <= lim)
					st.put(sp++, r[1], d[1]);
				ref = r[0];
				continue;
			}
		} else {
			uint32_t f = leaf_first(ref), c = leaf_count(ref);
			for (uint32_t i = 0; i < c; ++i) {
				// the plane, tangents and vertices (quads 0-6) in one round
				// trip with the box pre-test's vertices; the edge normals
				// (quads 7-9) only where the vertex regions do not decide.
				// The empty asm takes the seven quads as register operands
				// here, so the compiler issues their loads together instead
				// of moving quads 0-3 behind the pre-test's branch (a second
				// round trip to memory for almost every triangle).
				const v4f* q = reinterpret_cast<const v4f*>(V.dtri + f + i);
				const v4f q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3], q4 = q[4], q5 = q[5], q6 = q[6];
				asm volatile("" ::"v"(q0), "v"(q1), "v"(q2), "v"(q3), "v"(q4), "v"(q5), "v"(q6));
				if (tri_box_beyond_q(p, q4, q5, q6, best)) {
					ncull++;
					continue;
				}
				DistTri T;
				v4f* o = reinterpret_cast<v4f*>(&T);
				o[0] = q0;
				o[1] = q1;
				o[2] = q2;
				o[3] = q3;
				o[4] = q4;
				o[5] = q5;
				o[6] = q6;
				o[7] = q[7];
				o[8] = q[8];
				o[9] = q[9];
				float d = dist_tri_pre(p, T);
				nt++;
				if (d < best)
					best = d;
			}
		}
		// pop the next entry still within reach
		bool found = false;
		while (sp > 0) {
			--sp;
			if (st.k(sp) <= best * best) {
				ref = st.r(sp);
				found = true;
				break;
			}
		}
		if (!found)
			break;
	}
	if (COUNT) {
		atomicAdd(cnt + 0, (unsigned long long)nn);
		atomicAdd(cnt + 1, (unsigned long long)nt);
		atomicAdd(cnt + 5, (unsigned long long)ncull);
		atomicAdd(cnt + 3, 1ull);
	}
	return best;
}

template <bool COUNT>
__device__ __forceinline__ float q_distance(const View& V, f3 p, float radius, unsigned long long* cnt)
{
	PrivStack st;
	return q_distance<COUNT>(V, p, radius, cnt, st);
}

struct Seg {
	f3 o, dir, inv;
};

__device__ __forceinline__ Seg make_seg(f3 A, f3 B)
{
	f3 dn = normalized(B - A);
	f3 mA = A + dn * kSmall;
	f3 mB = B - dn * kSmall;
	Seg s;
	s.o = mA;
	s.dir = mB - mA;
	float ex = fabsf(s.dir.x) > 1e-30f ? s.dir.x : copysignf(1e-30f, s.dir.x);
	float ey = fabsf(s.dir.y) > 1e-30f ? s.dir.y : copysignf(1e-30f, s.dir.y);
	float ez = fabsf(s.dir.z) > 1e-30f ? s.dir.z : copysignf(1e-30f, s.dir.z);
	s.inv = mk3(1.0f / ex, 1.0f / ey, 1.0f / ez);
	return s;
}

// entry parameter of the segment into a box, or +inf when [0, tlim] misses it
__device__ __forceinline__ float slab(const Seg& s, float lx, float ly, float lz, float hx, float hy, float hz,
                                      float tlim)
{
	float tx0 = (lx - s.o.x) * s.inv.x, tx1 = (hx - s.o.x) * s.inv.x;
	float ty0 = (ly - s.o.y) * s.inv.y, ty1 = (hy - s.o.y) * s.inv.y;
	float tz0 = (lz - s.o.z) * s.inv.z, tz1 = (hz - s.o.z) * s.inv.z;
	float tn = fmaxf(fmaxf(fminf(tx0, tx1), fminf(ty0, ty1)), fmaxf(fminf(tz0, tz1), 0.0f));
	float tf = fminf(fminf(fmaxf(tx0, tx1), fmaxf(ty0, ty1)), fminf(fmaxf(tz0, tz1), tlim));
	return tn <= tf ? tn : INFINITY;
}

// ANY = true: returns 0 on the first hit with r < 1 (occlusion), else 2.
// start >= 0: the walk starts at that node, which the caller took from the
// entry grid at A for a segment of at most kGridReach; -1: at A's cell for
// such a segment, else at the root.
template <bool ANY, bool COUNT, class Stack>
__device__ float q_segment(const View& V, f3 A, f3 B, unsigned long long* cnt, Stack& st, int32_t start = -1)
{
	float best = 2.0f;
	if (!V.has_tris)
		return best;
	Seg s = make_seg(A, B);
	int sp = 0;
	const f3 AB = B - A;
	int32_t ref = start >= 0 ? start : dot(AB, AB) <= kGridReach * kGridReach ? entry_node(V, A) : 0;
	unsigned nn = 0, nt = 0;
	for (;;) {
		if (ref >= 0) {
			WNode n = load_node(V.nodes, ref);
			nn++;
			float tl = fminf(best, 1.0f);
			float t[4] = {slab(s, n.lx.x, n.ly.x, n.lz.x, n.hx.x, n.hy.x, n.hz.x, tl),
			              slab(s, n.lx.y, n.ly.y, n.lz.y, n.hx.y, n.hy.y, n.hz.y, tl),
			              slab(s, n.lx.z, n.ly.z, n.lz.z, n.hx.z, n.hy.z, n.hz.z, tl),
			              slab(s, n.lx.w, n.ly.w, n.lz.w, n.hx.w, n.hy.w, n.hz.w, tl)};
			int32_t r[4] = {n.c.x, n.c.y, n.c.z, n.c.w};
			sort4(t, r);
			if (t[0] != INFINITY) {
				if (t[3] != INFINITY)
					st.put(sp++, r[3], t[3]);
				if (t[2] != INFINITY)
					st.put(sp++, r[2], t[2]);
				if (t[1] != INFINITY)
					st.put(sp++, r[1], t[1]);
				ref = r[0];
				continue;
			}
		} else {
			uint32_t f = leaf_first(ref), c = leaf_count(ref);
			nt += c;
			bool done = false;
			for (uint32_t i = 0; i < c; ++i) {
				RayTri T = load_rtri(V.rtri, f + i);
				float r = seg_tri_pre(s.o, s.dir, T);
				if (r < best)
					best = r;
				if (ANY && best < 1.0f) {
					done = true;
					break;
				}
			}
			if (done)
				break;
		}
		bool found = false;
		while (sp > 0) {
			--sp;
			if (st.k(sp) <= fminf(best, 1.0f)) {
				ref = st.r(sp);
				found = true;
				break;
			}
		}
		if (!found)
			break;
	}
	if (COUNT) {
		atomicAdd(cnt + 0, (unsigned long long)nn);
		atomicAdd(cnt + 1, (unsigned long long)nt);
		atomicAdd(cnt + 3, 1ull);
	}
	return best;
}

template <bool ANY, bool COUNT>
__device__ __forceinline__ float q_segment(const View& V, f3 A, f3 B, unsigned long long* cnt)
{
	PrivStack st;
	return q_segment<ANY, COUNT>(V, A, B, cnt, st);
}

// Exit parameter of the ray from + rd*t from the grown scene box, padded so
// that points beyond it are certainly outside; -inf if the ray misses it.
__device__ __forceinline__ float box_exit(const View& V, f3 from, f3 rd)
{
	float lo[3] = {V.xlo[0], V.xlo[1], V.xlo[2]}, hi[3] = {V.xhi[0], V.xhi[1], V.xhi[2]};
	float o[3] = {from.x, from.y, from.z}, d[3] = {rd.x, rd.y, rd.z};
	float tn = -INFINITY, tf = INFINITY;
#pragma unroll
	for (int a = 0; a < 3; ++a) {
		if (d[a] != 0.0f) {
			float t0 = (lo[a] - o[a]) / d[a], t1 = (hi[a] - o[a]) / d[a];
			tn = fmaxf(tn, fminf(t0, t1));
			tf = fminf(tf, fmaxf(t0, t1));
		} else if (o[a] < lo[a] || o[a] > hi[a]) {
			return -INFINITY;
		}
	}
	if (tn > tf)
		return -INFINITY;
	return tf * 1.0001f + 0.01f;
}

// CalcInvShadowFactor (lighter.cpp:190-207) as a resumable state machine, one
// distance query per step.  Two shortcuts leave the result unchanged:
//  * once the march has left the grown scene box every remaining step sees
//    h = 2 and, for k >= 0, cannot lower res (2 / min(t*k, 2) >= 1 >= res),
//    so the march stops there;
//  * the distance to the scene is 1-Lipschitz, so the next query's search
//    radius starts at min(2, h + step + margin) instead of 2: every
//    triangle closer than that is still found, hence the same minimum;
//  * for k >= 0 a step's distance h matters only below
//    need = max(1, res m (1 + 2^-20)), m = min(t k, 2): at or beyond it the
//    step is min(h, 1) = 1 and h / m >= res after rounding (the factor
//    1 + 2^-20 is far above the two roundings of res m and h / m), so res
//    keeps its value.  The query radius is therefore min(2, Lipschitz bound,
//    need); when it was set by need and nothing lies closer, the step is 1,
//    res is unchanged and the next Lipschitz bound is unknown (2).
// A march whose t no longer advances (t + step == t, where the reference
// would loop forever) ends with the current factor.
struct March {
	f3 from, rd;
	float t, maxt, k, res, t_out, radius;
	uint32_t steps;
};

__device__ __forceinline__ void march_init(March& M, const View& V, f3 from, f3 to, float k)
{
	M.from = from;
	M.rd = normalized(to - from);
	M.t = 0.001f;
	M.maxt = length(to - from);
	M.k = k;
	M.res = 1.0f;
	M.t_out = (k >= 0.0f) ? box_exit(V, from, M.rd) : INFINITY;
	M.radius = kPenumbraSize;
	M.steps = 0;
}

// margin of the next search radius: covers the rounding of the computed
// distances (a few ulps of the coordinates) and of the march position
__device__ __forceinline__ float lipschitz_margin(f3 p)
{
	return 1e-4f + 1e-5f * fmaxf(fmaxf(fabsf(p.x), fabsf(p.y)), fabsf(p.z));
}

// Advances one step; returns true when the march is over (result in M.res).
// dist(p, R): min(R, distance of p to the nearest triangle).
template <class Dist>
__device__ __forceinline__ bool march_step(March& M, Dist&& dist)
{
	if (!(M.t < M.maxt) || M.t > M.t_out)
		return true;
	f3 p = M.from + M.rd * M.t;
	const float m = tmin(M.t * M.k, kPenumbraSize);
	const float lowers = M.k >= 0.0f ? M.res * m * (1.0f + 0x1p-20f) : INFINITY; // only h below it lowers res
	const float need = M.k >= 0.0f ? fmaxf(kPenumbraStep, lowers) : kPenumbraSize;
	const float R = fminf(M.radius, need);
	float h = dist(p, R);
	M.steps++;
	if (need < M.radius && h >= R) {
		// nothing closer than need (>= 1): step 1, res unchanged
		float tn = M.t + kPenumbraStep;
		if (tn == M.t)
			return true;
		M.radius = kPenumbraSize;
		M.t = tn;
		return false;
	}
	if (h < 0.001f) {
		M.res = 0.0f;
		return true;
	}
	if (!(h >= lowers))
		M.res = tmin(M.res, h / m);
	float st = tmin(h, kPenumbraStep);
	float tn = M.t + st;
	if (tn == M.t)
		return true;
	M.radius = fminf(h + st + lipschitz_margin(p), kPenumbraSize);
	M.t = tn;
	return false;
}

// ---------------------------------------------------------------------------
// Reference-shaped traversal counts (measurement only).  The byte count a
// roofline fraction is stated on must not depend on this build's own tree,
// so it is taken on a plain binary SAH tree (16 bins, at most 4 triangles
// per leaf) with the reference's query semantics: every march step of
// CalcInvShadowFactor (lighter.cpp:190-207) is a fresh distance query of
// radius MAX_PENUMBRA_SIZE (no exit test, no Lipschitz or need bound), the
// nearer child is visited first and the radius shrinks with every triangle
// distance found.  A node visit is one box tested (32 bytes of node in the
// reference layout), a triangle test one point-triangle distance (36 bytes
// of vertices).  The march's factor is compared with the product's, bit for
// bit, as a by-product.
// ---------------------------------------------------------------------------
struct CanonView {
	const BvhNode* __restrict__ nodes;
	const DistTri* __restrict__ dtri;
	float lo[3], hi[3]; // the root's box, padded as the builder pads node boxes
};

// The builder's outward padding of a box (bvh.cpp), for the root's box.
inline void canon_root_box(const BinaryBvh& b, float lo[3], float hi[3])
{
	const float l[3] = {b.lo.x, b.lo.y, b.lo.z}, h[3] = {b.hi.x, b.hi.y, b.hi.z};
	for (int a = 0; a < 3; ++a) {
		const float m = 1e-5f * std::max(fabsf(l[a]), fabsf(h[a])) + 1e-6f;
		lo[a] = l[a] - m;
		hi[a] = h[a] + m;
	}
}
constexpr int kCanonStack = 64; // >= the binary tree's depth, checked at build

__device__ float canon_distance(const CanonView& C, f3 p, unsigned long long& nvis, unsigned long long& ntri)
{
	float best = kPenumbraSize;
	nvis++; // the root's box
	if (box_d2(p, C.lo[0], C.lo[1], C.lo[2], C.hi[0], C.hi[1], C.hi[2]) > best * best)
		return best;
	int32_t st[kCanonStack];
	float sk[kCanonStack];
	int sp = 0;
	int32_t ref = 0;
	for (;;) {
		if (ref >= 0) {
			const BvhNode n = C.nodes[ref];
			float da = box_d2(p, n.lo0x, n.lo0y, n.lo0z, n.hi0x, n.hi0y, n.hi0z);
			float db = box_d2(p, n.lo1x, n.lo1y, n.lo1z, n.hi1x, n.hi1y, n.hi1z);
			int32_t a = n.c0, b = n.c1;
			nvis += 2;
			if (db < da) {
				float t = da;
				da = db;
				db = t;
				int32_t u = a;
				a = b;
				b = u;
			}
			const float lim = best * best;
			if (da <= lim) {
				if (db <= lim) {
					st[sp] = b;
					sk[sp] = db;
					sp++;
				}
				ref = a;
				continue;
			}
		} else {
			const uint32_t f = leaf_first(ref), c = leaf_count(ref);
			for (uint32_t i = 0; i < c; ++i) {
				const float d = dist_tri_pre(p, load_dtri(C.dtri, f + i));
				ntri++;
				if (d < best)
					best = d;
			}
		}
		bool found = false;
		while (sp > 0) {
			--sp;
			if (sk[sp] <= best * best) {
				ref = st[sp];
				found = true;
				break;
			}
		}
		if (!found)
			break;
	}
	return best;
}

// One lane per entry of the last direct-light run's march list.  out:
// node visits, triangle tests, distance queries, factors that differ from
// the product's (vis).
__global__ __launch_bounds__(kBlock) void k_march_canon(CanonView C, View V, const float* __restrict__ pos,
                                                        const float* __restrict__ nrm,
                                                        const DevLight* __restrict__ lights,
                                                        const uint32_t* __restrict__ items,
                                                        const uint32_t* __restrict__ mlist, uint32_t nmarch,
                                                        const float* __restrict__ vis, unsigned long long* out)
{
	const uint32_t idx = blockIdx.x * kBlock + threadIdx.x;
	if (idx >= nmarch)
		return;
	const uint32_t k = mlist[idx];
	const uint32_t code = items[k];
	const DevLight& L = lights[code >> kSampleBits];
	const uint32_t s = code & kSampleMask;
	const f3 SP = ld3(pos + 3 * s), SN = ld3(nrm + 3 * s);
	const f3 to = (L.type == 3) ? SP + ld3(L.dir) * L.range : ld3(L.pos);
	March M;
	march_init(M, V, SP + SN * kShadowOffset, to, L.radius);
	unsigned long long nv = 0, nt = 0, nq = 0;
	float res = 1.0f;
	for (float t = M.t; t < M.maxt;) {
		const float h = canon_distance(C, M.from + M.rd * t, nv, nt);
		nq++;
		if (h < 0.001f) {
			res = 0.0f;
			break;
		}
		res = tmin(res, h / tmin(t * M.k, kPenumbraSize));
		const float tn = t + tmin(h, kPenumbraStep);
		if (tn == t)
			break;
		t = tn;
	}
	atomicAdd(out + 0, nv);
	atomicAdd(out + 1, nt);
	atomicAdd(out + 2, nq);
	if (vis && __float_as_uint(res) != __float_as_uint(vis[k]))
		atomicAdd(out + 3, 1ull);
}

// ---------------------------------------------------------------------------
// direct light
// ---------------------------------------------------------------------------
// Shading gate of each (light, texel) item (Job_LMRender_*_Inner up to the
// shadow march, lighter.cpp:485-553, 586): items with a zero shading factor
// get their final weight here; the others are appended to the march list
// with the factor the shadow term multiplies.  A block takes kGateRounds x
// kBlock consecutive items, collects its marches in LDS, sorts them by
// (light, Morton code of the texel position) and appends them with one
// atomic (one per wave on a single counter serialised in L2).  Items come in
// atlas order, rows of texels; after the sort a wave's 64 marches start from
// a compact patch of space towards one light, so their traversals overlap
// (-9 % march time on the terrain workload).  Only the order in which
// marches are taken changes, not any result.
constexpr int kGateRounds = 8;
constexpr size_t kAOChunk = size_t(1) << 20; // texels per AO launch when progress is followed
constexpr uint32_t kMarchBatch = 64; // march-list positions a wave claims at a time
static_assert(kMarchBatch >= 64, "a refill of all 64 lanes must fit in one claim");

__device__ __forceinline__ bool gate_item(const float* __restrict__ pos, const float* __restrict__ nrm,
                                          const DevLight* __restrict__ lights, const uint32_t* __restrict__ items,
                                          uint32_t k, float* __restrict__ gate, float* __restrict__ wout,
                                          float* __restrict__ vout)
{
	bool march = false;
	{
		uint32_t code = items[k];
		const DevLight& L = lights[code >> kSampleBits];
		uint32_t s = code & kSampleMask;
		f3 SP = ld3(pos + 3 * s), SN = ld3(nrm + 3 * s);
		float w = __uint_as_float(kSkipBits), g = 0.0f;
		if (L.type == 3) {
			float fn = tmax(0.0f, dot(ld3(L.dir), SN));
			if (fn > 0) {
				march = true;
				g = fn;
			} else {
				w = fn; // +-0 times a finite non-negative shadow factor
			}
		} else if (L.type == 1 || L.type == 2) {
			f3 s2l = ld3(L.pos) - SP;
			float dist = length(s2l);
			if (dist)
				s2l = s2l / dist;
			float fd = pow_r(1 - tmin(1.0f, dist / L.range), L.power);
			float fn = tmax(0.0f, dot(s2l, SN));
			float gt;
			if (L.type == 2) {
				float ang = acos_r(tmin(1.0f, dot(s2l, -ld3(L.dir))));
				float fdir = tmax(0.0f, tmin(1.0f, (ang - L.spot_out_rad) / L.spot_diff));
				fdir = pow_r(fdir, L.spot_curve);
				gt = fd * fn * fdir;
			} else {
				gt = fd * fn;
			}
			if (!(gt <= 0)) {
				march = true;
				g = gt;
			}
		}
		if (march) {
			gate[k] = g;
		} else {
			wout[k] = w;
			if (vout)
				vout[k] = 1.0f;
		}
	}
	return march;
}

__global__ __launch_bounds__(kBlock) void k_direct_gate(const float* __restrict__ pos, const float* __restrict__ nrm,
                                                        const DevLight* __restrict__ lights,
                                                        const uint32_t* __restrict__ items, uint32_t nitems,
                                                        float* __restrict__ gate, float* __restrict__ wout,
                                                        float* __restrict__ vout, uint32_t* __restrict__ mlist,
                                                        uint32_t* __restrict__ mcount, const uint32_t* __restrict__ skey)
{
	__shared__ uint32_t list[kGateRounds * kBlock];
	__shared__ uint32_t keys[kGateRounds * kBlock];
	__shared__ uint32_t n, base, l0;
	const uint64_t k0 = (uint64_t)blockIdx.x * (kGateRounds * kBlock);
	if (threadIdx.x == 0) {
		n = 0;
		l0 = items[k0] >> kSampleBits;
	}
	__syncthreads();
	const int lane = threadIdx.x & 63;
	for (int r = 0; r < kGateRounds; ++r) {
		const uint64_t k = k0 + (uint64_t)r * kBlock + threadIdx.x;
		const bool march = k < nitems && gate_item(pos, nrm, lights, items, (uint32_t)k, gate, wout, vout);
		const uint64_t m = __ballot(march);
		uint32_t wbase = 0;
		if (lane == 0 && m)
			wbase = atomicAdd(&n, (uint32_t)__popcll(m)); // LDS atomic, one per wave
		wbase = (uint32_t)__shfl((int)wbase, 0);
		if (march) {
			const uint32_t slot = wbase + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
			const uint32_t code = items[k];
			const uint32_t dl = min((code >> kSampleBits) - l0, 2u); // keys stay below the padding 0xFFFFFFFF
			list[slot] = (uint32_t)k;
			keys[slot] = (dl << 30) | skey[code & kSampleMask];
		}
	}
	__syncthreads();
	// sort the block's marches by (light, Morton code of the texel)
	uint32_t N = 1;
	while (N < n)
		N <<= 1;
	for (uint32_t i = n + threadIdx.x; i < N; i += kBlock)
		keys[i] = 0xFFFFFFFFu;
	for (uint32_t size = 2; size <= N; size <<= 1)
		for (uint32_t stride = size >> 1; stride > 0; stride >>= 1) {
			__syncthreads();
			for (uint32_t i = threadIdx.x; i < N / 2; i += kBlock) {
				const uint32_t lo = 2 * stride * (i / stride) + (i & (stride - 1)), hi = lo + stride;
				const bool up = (lo & size) == 0;
				const uint32_t a = keys[lo], b = keys[hi];
				if ((a > b) == up) {
					keys[lo] = b;
					keys[hi] = a;
					const uint32_t t = list[lo];
					list[lo] = list[hi];
					list[hi] = t;
				}
			}
		}
	__syncthreads();
	if (threadIdx.x == 0)
		base = n ? atomicAdd(mcount, n) : 0u;
	__syncthreads();
	for (uint32_t i = threadIdx.x; i < n; i += kBlock)
		mlist[base + i] = list[i];
}

// Where a march kernel's marches come from and where their results go.
struct DirectSrc { // the marches of the direct light: work items, neighbours in order
	static constexpr uint32_t kWaveMax = 3u << 15;
	const float* __restrict__ pos;
	const float* __restrict__ nrm;
	const DevLight* __restrict__ lights;
	const uint32_t* __restrict__ items;
	const uint32_t* __restrict__ mlist;
	const float* __restrict__ gate;
	float* __restrict__ wout;
	float* __restrict__ vout;
	__device__ __forceinline__ uint32_t key(uint32_t idx) const { return mlist[idx]; }
	__device__ __forceinline__ void init(March& M, const View& V, uint32_t k) const
	{
		const uint32_t code = items[k];
		const DevLight& L = lights[code >> kSampleBits];
		const uint32_t s = code & kSampleMask;
		const f3 SP = ld3(pos + 3 * s), SN = ld3(nrm + 3 * s);
		const f3 to = (L.type == 3) ? SP + ld3(L.dir) * L.range : ld3(L.pos);
		march_init(M, V, SP + SN * kShadowOffset, to, L.radius);
	}
	__device__ __forceinline__ void finish(const March& M, uint32_t k) const
	{
		// weight = (shading factor) * shadow factor, in the reference's order
		wout[k] = gate[k] * M.res;
		if (vout)
			vout[k] = M.res;
	}
};

struct QuerySrc { // the marches of lgx_QueryShadow, in the caller's order: lanes of a wave far apart
	// whole calls with waves and on lanes, ms: 100,003 scattered in a city 1.21
	// and 2.01, in a terrain 1.79 and 1.91; 131,001: 1.51 and 1.94, 2.25 and
	// 1.86
	static constexpr uint32_t kWaveMax = 1u << 17;
	const float* __restrict__ from;
	const float* __restrict__ to;
	const float* __restrict__ k;
	float* __restrict__ out;
	uint32_t* __restrict__ steps;
	__device__ __forceinline__ uint32_t key(uint32_t idx) const { return idx; }
	__device__ __forceinline__ void init(March& M, const View& V, uint32_t i) const
	{
		march_init(M, V, ld3(from + 3 * (size_t)i), ld3(to + 3 * (size_t)i), k[i]);
	}
	__device__ __forceinline__ void finish(const March& M, uint32_t i) const
	{
		out[i] = M.res;
		steps[i] = M.steps;
	}
};

// A march in progress, handed from the lane that began it to k_march_wave:
// what march_init does not give again.
struct LongMarch {
	uint32_t key;
	float t, res, radius;
	uint32_t steps;
};
// Words of a march's control block (zeroed before the launches).
constexpr int kMarchCursor = 0, kMarchAbort = 1, kMarchLong = 2, kMarchWords = 3;
// Marches that can be handed over (20 bytes each, 10 MiB); a lane keeps the
// rest and asks no more.  As many as the lanes of a launch, and more than any
// measured one hands over (107,000 of a city's 1.6 M): with a full list it is
// the first to get there, not the longest, that went to waves (156,588 over
// a list of 131,072: 18.2 ms instead of 12.0).
constexpr uint32_t kLongCap = 1u << 19;
constexpr int kFewLong = 48;

// Persistent shadow-march kernel: every lane pulls a new march from the list
// as soon as its current one ends (one atomic per wave per refill), so the
// very uneven march lengths do not idle the wave.  Every wave leaves once the
// list is exhausted and its lanes' marches have ended.  ctl (optional, host
// memory): the claims of positions 0, 64 x kMarchBatch, .. post the
// position to ctl[1] (progress) and, when ctl[0] is set, raise the device
// flag next[kMarchAbort]; a wave that finds it set at a claim leaves at once
// (abort), so every wave stops within one claim of the first such post.  (A variant that
// interleaves single traversal actions of all lanes in one loop measured
// 37% slower on the terrain workload.)
// A march of limit steps or more, or of tail steps once the list is empty
// (looked at every 16 steps), goes to the list of long marches (lng), which
// k_march_wave finishes with a wave for each: a lane takes about 4.5 us for a
// step, so one march of 1,791 steps along a wall kept a launch of 161,236
// marches (mean 28 steps) running for 8.1 ms.  A wave of which more than
// kFewLong lanes march long keeps them: its lanes are all at work and mostly
// on the same nodes (a plane under a grazing sun, 260,100 marches of
// thousands of steps each: 285 ms handed over, 102 kept; 500,001 grazing
// queries in a room 2.78 and 2.46 ms).  With 16 in place of 48 the waves that
// hold several of a city's long marches keep them too long (2.07 M marches
// 13.5 ms instead of 11.1; 32: 11.1, and a terrain of 1.29 M 7.9 instead of
// 7.5).
// The traversal stack's first levels live in LDS (dynamic, kBlock * depth * 6
// bytes: an int32 reference and an FP16 key per level and lane), depth =
// min(kLdsLevels, levels of the BVH plus margin).
template <bool COUNT, class Src>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_march(View V, Src src, uint32_t nmarch, uint32_t* __restrict__ next,
                                                  unsigned long long* cnt, int depth, uint32_t* ctl, uint32_t limit,
                                                  uint32_t tail, LongMarch* __restrict__ lng)
{
	extern __shared__ __align__(16) unsigned char lds_stack[];
	LdsStack st = lds_stack_of_lane(lds_stack, depth);
	bool active = false, done = false;
	uint32_t k = 0;
	March M;
	// the wave's reservation [rbeg, rend) of march-list positions: refills
	// take from it and claim kMarchBatch more with one atomic when it runs
	// short, so a wave keeps working on neighbouring items (one texel region
	// and light) and the list counter sees one atomic per kMarchBatch marches
	const int lane = threadIdx.x & 63;
	uint32_t rbeg = 0, rend = 0;
	for (;;) {
		bool need = !active && !done;
		const uint64_t nm = __ballot(need);
		if (nm) {
			const uint32_t cnt_need = (uint32_t)__popcll(nm);
			const uint32_t rank = (uint32_t)__popcll(nm & ((1ull << lane) - 1ull));
			const uint32_t avail = rend - rbeg;
			uint32_t idx;
			if (avail >= cnt_need) {
				idx = rbeg + rank;
				rbeg += cnt_need;
			} else {
				uint32_t nb = 0, stop = 0;
				if (lane == 0) {
					// every claim reads the device abort flag (an L2
					// access in flight together with the claim's atomic);
					// one claim in 64 also makes the host round trip:
					// progress out, the host's abort flag in, passed on to
					// the device's (a host round trip at every claim cost 3 %)
					if (ctl)
						stop = __hip_atomic_load(next + kMarchAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					nb = atomicAdd(next + kMarchCursor, kMarchBatch);
					if (ctl && ((nb / kMarchBatch) & 63u) == 0) {
						__hip_atomic_store(ctl + 1, nb, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
						if (__hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))
							__hip_atomic_store(next + kMarchAbort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
					}
				}
				nb = (uint32_t)__shfl((int)nb, 0);
				if (__shfl((int)stop, 0))
					break; // aborted: the wave leaves its marches unfinished
				idx = rank < avail ? rbeg + rank : nb + (rank - avail);
				rbeg = nb + (cnt_need - avail);
				rend = nb + kMarchBatch;
			}
			if (need) {
				if (idx < nmarch) {
					k = src.key(idx);
					src.init(M, V, k);
					active = true;
				} else {
					done = true;
				}
			}
			if (__any(done))
				limit = tail; // the list is empty: what is left is the launch's tail
		}
		if (__all(done))
			break;
		// as it will be after the step
		const bool few = !COUNT && __popcll(__ballot(active && M.steps + 1 >= limit)) <= kFewLong;
		if (active) {
			if (march_step(M, [&](f3 p, float R) { return q_distance<COUNT>(V, p, R, cnt, st); })) {
				src.finish(M, k);
				if (COUNT) {
					atomicAdd(cnt + 2, (unsigned long long)M.steps);
					atomicAdd(cnt + 4, 1ull);
				}
				active = false;
			} else if (few && M.steps >= limit && (M.steps & 15u) == 0) {
				const uint32_t at = atomicAdd(next + kMarchLong, 1u);
				if (at < kLongCap) {
					lng[at] = LongMarch{k, M.t, M.res, M.radius, M.steps};
					active = false;
				} else {
					limit = tail = UINT32_MAX;
				}
			}
		}
	}
}

// ---------------------------------------------------------------------------
// One wave per march: the long marches of k_march, and every march of a
// launch too small to fill the chip's lanes.  A march is a chain of distance
// queries, each a walk of dependent node and triangle fetches (about 4.5 us
// a step on one lane whatever the other lanes do), and it is long where it
// creeps along a surface: its steps and search radii are then centimetres,
// so the next dozens of queries are answered by the same few triangles.  The
// wave therefore gathers every triangle whose leaf box lies within `rad` of
// the point at hand (rad = reach x the query's radius, 2 m at most), one
// triangle per lane in registers, and answers each query R at p by the
// lanes' distances and a wave minimum while the ball of R around p stays
// inside the gathered ball.  The gathered set holds every triangle nearer
// than R, and the distances are dist_tri_pre's, so the minimum is the walk's,
// bit for bit.  Where one triangle's face is the nearest by a margin (its
// region tests, the second nearest triangle and the gathered ball give how
// far the march can go before that can change; every distance is 1-Lipschitz
// and lipschitz_margin covers the rounding, as for the search radii above),
// the steps up to there take only that plane's distance, the value
// dist_tri_pre returns for a face, and no reduction.  The march moves along a
// unit direction, so these balls are intervals of t.
// reach doubles (to 64) after a gather of few triangles and
// halves after one that did not fit the 64 lanes; where even the query's own
// ball holds more, the query takes the ordinary walk.  It is bound by the
// issue of one wave's serial chain: about 0.4 us a step (0.9 us without the
// face intervals and with a claim per march), where a lane's walk takes 4.5.
// A city's 161,236 marches (longest 1,791 steps): 8.1 ms on lanes alone,
// 1.52 + 0.57 ms with the long ones here; 64 probes in a room: 1,000 -> 210 us.
// ---------------------------------------------------------------------------
constexpr float kFaceNear = 0.25f; // steps shorter than this try the face interval
constexpr int kGatherQueue = 256; // node references in flight per wave (a power of two)

__device__ __forceinline__ float lane_value(float v, int lane)
{
	return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// minimum over the 64 lanes (all active), the same on every lane
__device__ __forceinline__ float wave_min(float v)
{
	const int inf = __float_as_int(INFINITY);
	v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(v), 0x111, 0xf, 0xf, false))); // row_shr:1
	v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(v), 0x112, 0xf, 0xf, false))); // row_shr:2
	v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(v), 0x114, 0xf, 0xf, false))); // row_shr:4
	v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(v), 0x118, 0xf, 0xf, false))); // row_shr:8
	v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(v), 0x142, 0xa, 0xf, false))); // row_bcast:15
	v = fminf(v, __int_as_float(__builtin_amdgcn_update_dpp(inf, __float_as_int(v), 0x143, 0xc, 0xf, false))); // row_bcast:31
	return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ void wave_lds_sync()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
	__builtin_amdgcn_wave_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Triangles whose leaf box lies within D (<= kGridReach) of p into tri[0..63];
// their number, or -1 when more than 64 (or more nodes than the queue holds)
// lie there.  Sixteen nodes at a time, a lane per child.
__device__ __forceinline__ int wave_gather(const View& V, f3 p, float D, uint32_t* queue, uint32_t* tri)
{
	const int lane = threadIdx.x & 63;
	const uint64_t below = (1ull << lane) - 1ull;
	const float D2 = D * D;
	if (lane == 0)
		queue[0] = (uint32_t)entry_node(V, p, D <= kGridFineReach);
	wave_lds_sync();
	uint32_t head = 0, end = 1;
	int n = 0;
	while (head != end) {
		const uint32_t take = min(end - head, 16u);
		bool hit = false;
		int32_t c = 0;
		if ((uint32_t)lane < 4 * take) {
			const uint32_t node = queue[(head + (uint32_t)(lane >> 2)) & (kGatherQueue - 1)];
			const float* q = reinterpret_cast<const float*>(V.nodes + node) + (lane & 3);
			c = reinterpret_cast<const int32_t*>(q)[24];
			hit = box_d2(p, q[0], q[4], q[8], q[12], q[16], q[20]) <= D2;
		}
		head += take;
		const uint64_t inner = __ballot(hit && c >= 0);
		const uint64_t one = __ballot(hit && c < 0), two = __ballot(hit && c < 0 && leaf_count(c) > 1);
		const int nt = __popcll(one) + __popcll(two), nn = __popcll(inner);
		if (n + nt > 64 || end - head + (uint32_t)nn > (uint32_t)kGatherQueue)
			return -1;
		if (hit && c >= 0)
			queue[(end + (uint32_t)__popcll(inner & below)) & (kGatherQueue - 1)] = (uint32_t)c;
		if (hit && c < 0) {
			const int at = n + __popcll(one & below) + __popcll(two & below);
			tri[at] = leaf_first(c);
			if (leaf_count(c) > 1)
				tri[at + 1] = leaf_first(c) + 1;
		}
		end += (uint32_t)nn;
		n += nt;
		wave_lds_sync();
	}
	return n;
}
static_assert(kLeafMax <= 2, "wave_gather takes leaves of at most two triangles");

// dist_tri_pre without branches: the lanes' triangles lie in different
// regions, so its branches would run one after another, a square root each;
// here the regions select one operand.  The same operations give the value.
__device__ __forceinline__ float dist_tri_select(f3 p, const DistTri& T)
{
	const float pd = fabsf(dot(mk3(T.nx, T.ny, T.nz), p) - T.nd);
	const float t0p = dot(mk3(T.a0x, T.a0y, T.a0z), p);
	const float t1p = dot(mk3(T.a1x, T.a1y, T.a1z), p);
	const float t2p = dot(mk3(T.a2x, T.a2y, T.a2z), p);
	const bool v0 = T.t0min >= t0p & T.t2max <= t2p;
	const bool v1 = T.t1min >= t1p & T.t0max <= t0p;
	const bool v2 = T.t2min >= t2p & T.t1max <= t1p;
	const float ptd0 = dot(mk3(T.e0x, T.e0y, T.e0z), p) - T.e0d;
	const float ptd1 = dot(mk3(T.e1x, T.e1y, T.e1z), p) - T.e1d;
	const float ptd2 = dot(mk3(T.e2x, T.e2y, T.e2z), p) - T.e2d;
	const bool e0 = ptd0 >= 0 & t0p >= T.t0min & t0p <= T.t0max;
	const bool e1 = ptd1 >= 0 & t1p >= T.t1min & t1p <= T.t1max;
	const bool e2 = ptd2 >= 0 & t2p >= T.t2min & t2p <= T.t2max;
	// values before the selects: a select between members of a reference
	// becomes one between addresses and puts the triangle into scratch memory
	const float ax = T.v0x, ay = T.v0y, az = T.v0z, bx = T.v1x, by = T.v1y, bz = T.v1z;
	const float cx = T.v2x, cy = T.v2y, cz = T.v2z;
	const f3 V = mk3(v0 ? ax : v1 ? bx : cx, v0 ? ay : v1 ? by : cy, v0 ? az : v1 ? bz : cz);
	const float pe = e0 ? ptd0 : e1 ? ptd1 : ptd2;
	const bool vert = v0 | v1 | v2;
	const float q = vert ? lensq(p - V) : pd * pd + pe * pe;
	return (vert | e0 | e1 | e2) ? sqrtf(q) : pd;
}

// How far p can move, up to rounding, with every region test of dist_tri_pre
// still choosing the face (the plane's distance); <= 0 in another region.
// A vertex region takes both of its inequalities, an edge region is ruled
// out by lying inside that edge.
__device__ __forceinline__ float face_slack(f3 p, const DistTri& T)
{
	const float t0p = dot(mk3(T.a0x, T.a0y, T.a0z), p);
	const float t1p = dot(mk3(T.a1x, T.a1y, T.a1z), p);
	const float t2p = dot(mk3(T.a2x, T.a2y, T.a2z), p);
	const float ptd0 = dot(mk3(T.e0x, T.e0y, T.e0z), p) - T.e0d;
	const float ptd1 = dot(mk3(T.e1x, T.e1y, T.e1z), p) - T.e1d;
	const float ptd2 = dot(mk3(T.e2x, T.e2y, T.e2z), p) - T.e2d;
	const float v0 = fmaxf(t0p - T.t0min, T.t2max - t2p), v1 = fmaxf(t1p - T.t1min, T.t0max - t0p);
	const float v2 = fmaxf(t2p - T.t2min, T.t1max - t1p);
	return fminf(fminf(fminf(v0, v1), v2), -fmaxf(fmaxf(ptd0, ptd1), ptd2));
}

// march_step's steps up to t = face, the distance that of the plane (n, d);
// leaves the step that would end the march or step by its need to it.
__device__ __forceinline__ void face_steps(March& M, f3 n, float d, float face)
{
	const float last = fminf(face, M.t_out);
	while (M.t < M.maxt && M.t <= last) {
		const f3 p = M.from + M.rd * M.t;
		const float m = tmin(M.t * M.k, kPenumbraSize);
		const float lowers = M.k >= 0.0f ? M.res * m * (1.0f + 0x1p-20f) : INFINITY;
		const float need = M.k >= 0.0f ? fmaxf(kPenumbraStep, lowers) : kPenumbraSize;
		const float R = fminf(M.radius, need);
		const float h = fminf(R, fabsf(dot(n, p) - d));
		const float st = tmin(h, kPenumbraStep);
		const float tn = M.t + st;
		if ((need < M.radius && h >= R) || h < 0.001f || tn == M.t)
			break;
		M.steps++;
		if (!(h >= lowers))
			M.res = tmin(M.res, h / m);
		M.radius = fminf(h + st + lipschitz_margin(p), kPenumbraSize);
		M.t = tn;
	}
}

template <class Src>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(4, 8))) void k_march_wave(View V, Src src, uint32_t nfresh,
                                                       const LongMarch* __restrict__ lng, uint32_t* next,
                                                       uint32_t* ctl, int depth)
{
	extern __shared__ __align__(16) unsigned char lds_stack[];
	__shared__ uint32_t queues[kBlock / 64][kGatherQueue], tris[kBlock / 64][64];
	LdsStack st = lds_stack_of_lane(lds_stack, depth);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	uint32_t* queue = queues[wave];
	uint32_t* tri = tris[wave];
	const uint32_t n = lng ? (uint32_t)__builtin_amdgcn_readfirstlane((int)min(next[kMarchLong], kLongCap)) : nfresh;
	// a fixed stride over the list: a claim per march on one counter would
	// take longer than most marches here
	const uint32_t w0 = (uint32_t)__builtin_amdgcn_readfirstlane((int)(blockIdx.x * (kBlock / 64) + wave));
	for (uint32_t idx = w0; idx < n; idx += gridDim.x * (kBlock / 64)) {
		// as k_march's claims: every march first reads the device's abort flag,
		// one wave in 64 also the host's and posts the marches begun (64 for
		// each of its own, a lane one; when they come from lng, all of them
		// are).  The decision is the wave's: its lanes march together.
		if (ctl) {
			if ((w0 & 63u) == 0) {
				if (!lng) {
					const uint32_t begun = (uint32_t)__builtin_amdgcn_readfirstlane((int)atomicAdd(next + kMarchCursor, 1u));
					__hip_atomic_store(ctl + 1, begun, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
				}
				if (__hip_atomic_load(ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM))
					__hip_atomic_store(next + kMarchAbort, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
			}
			if (__builtin_amdgcn_readfirstlane(
			        (int)__hip_atomic_load(next + kMarchAbort, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)))
				break;
		}
		March M;
		const uint32_t k = lng ? lng[idx].key : src.key(idx);
		src.init(M, V, k);
		if (lng) {
			M.t = lng[idx].t;
			M.res = lng[idx].res;
			M.radius = lng[idx].radius;
			M.steps = lng[idx].steps;
		}
		DistTri T = {};
		float room = -1.0f;  // the gathered ball serves queries with t + R + margin <= room
		float face = -1.0f;  // up to this t the nearest triangle's plane gives the distance
		f3 fn = mk3(0, 0, 0);
		float fd = 0.0f, reach = 8.0f;
		int have = 0, walks = 0, plain = 0;
		auto dist = [&](f3 p, float R) {
			if (!V.has_tris)
				return R;
			if (M.t <= face)
				return fminf(R, fabsf(dot(fn, p) - fd));
			const float margin = lipschitz_margin(p);
			if (!(M.t + R + margin <= room)) {
				room = -1.0f;
				bool walk = walks > 0; // a crowded place: some ordinary walks before the next try
				walks -= walk;
				float D = 0.0f;
				while (!walk) {
					D = fminf(R * reach, kGridReach);
					have = wave_gather(V, p, D, queue, tri);
					if (have >= 0)
						break;
					walk = !(D > R);
					reach = fmaxf(0.5f * reach, 1.0f);
					walks = walk ? 4 : 0;
				}
				if (walk)
					return q_distance<false>(V, p, R, nullptr, st);
				if (have <= 24)
					reach = fminf(2.0f * reach, 64.0f);
				room = M.t + D;
				if (lane < have)
					T = load_dtri(V.dtri, tri[lane]);
			}
			const float t = dist_tri_select(p, T);
			const float d = lane < have && t < R ? t : R;
			const float h = wave_min(d);
			if (--plain < 0 && h < kFaceNear && h < R) {
				// creeping along a surface: the distance stays that of the
				// nearest triangle's plane while its region tests, the other
				// gathered triangles and the gathered ball leave room
				const int w = __ffsll((unsigned long long)__ballot(lane < have && t == h)) - 1;
				const float in = lane_value(face_slack(p, T), w);
				const float other = wave_min(lane < have && lane != w ? t : INFINITY);
				const float slack = fminf(in, 0.5f * fminf(other - h, room - M.t - h)) - margin;
				plain = 2;
				if (slack > 2.0f * h) {
					face = M.t + slack;
					fn = mk3(lane_value(T.nx, w), lane_value(T.ny, w), lane_value(T.nz, w));
					fd = lane_value(T.nd, w);
					plain = 0;
				}
			}
			return h;
		};
		do {
			face_steps(M, fn, fd, face);
		} while (!march_step(M, dist));
		// every lane, the same values: a branch on the lane here lets the
		// compiler send the others into the next march by themselves
		src.finish(M, k);
	}
}

// lightmap[s] += color * w for the items of one light (no sample repeats
// within a light, so no two lanes touch the same texel).
__global__ __launch_bounds__(kBlock) void k_accumulate(const uint32_t* __restrict__ items,
                                                       const float* __restrict__ w, uint32_t begin, uint32_t end,
                                                       float cr, float cg, float cb, float* __restrict__ lm)
{
	uint32_t k = begin + blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= end)
		return;
	float wk = w[k];
	if (__float_as_uint(wk) == kSkipBits)
		return;
	uint32_t s = items[k] & kSampleMask;
	f3 c = mk3(cr, cg, cb);
	f3 v = ld3(lm + 3 * s) + c * wk;
	st3(lm + 3 * s, v);
}

// ---------------------------------------------------------------------------
// Reverse mode of the accumulation above: the lightmap gains color_l * w
// per item (lighter.cpp:505-513), so dL/dcolor_l[c] = sum over light l's
// items of w * lam[s][c], lam = dL/dlightmap per sample.  One launch, grid
// (kGradBlocks, lights); each block writes FP64 partial sums, reduced in a
// fixed order on the host.
// ---------------------------------------------------------------------------
constexpr int kGradBlocks = 256; // blocks per light

__global__ __launch_bounds__(kBlock) void k_color_grad(const uint32_t* __restrict__ items,
                                                       const float* __restrict__ w,
                                                       const uint32_t* __restrict__ light_off,
                                                       const double* __restrict__ lam, double* __restrict__ part)
{
	const uint32_t l = blockIdx.y;
	const uint32_t begin = light_off[l], end = light_off[l + 1];
	double a0 = 0, a1 = 0, a2 = 0;
	for (uint32_t k = begin + blockIdx.x * kBlock + threadIdx.x; k < end; k += kGradBlocks * kBlock) {
		float wk = w[k];
		if (__float_as_uint(wk) == kSkipBits)
			continue;
		uint32_t s = items[k] & kSampleMask;
		a0 += (double)wk * lam[3 * (uint64_t)s];
		a1 += (double)wk * lam[3 * (uint64_t)s + 1];
		a2 += (double)wk * lam[3 * (uint64_t)s + 2];
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) {
		a0 += __shfl_xor(a0, o);
		a1 += __shfl_xor(a1, o);
		a2 += __shfl_xor(a2, o);
	}
	__shared__ double red[kBlock / 64][3];
	const int wave = threadIdx.x >> 6;
	if ((threadIdx.x & 63) == 0) {
		red[wave][0] = a0;
		red[wave][1] = a1;
		red[wave][2] = a2;
	}
	__syncthreads();
	if (threadIdx.x < 3) {
		double t = 0;
		for (int q = 0; q < kBlock / 64; ++q)
			t += red[q][threadIdx.x];
		part[3 * ((uint64_t)l * kGradBlocks + blockIdx.x) + threadIdx.x] = t;
	}
}

// ---------------------------------------------------------------------------
// ambient occlusion (lighter.cpp:799-841)
// ---------------------------------------------------------------------------
// a value that every lane of the wave holds, kept in a scalar register
__device__ __forceinline__ float wave_uniform(float x)
{
	return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// ---------------------------------------------------------------------------
// One walk for a wave's 64 segments: the wave goes to every node that any of
// them meets, so a node's and a triangle's data are the same on every lane
// (scalar loads), nothing is sorted per lane and the stack is one list of
// references in LDS.  A segment that would have passed a node by takes its
// children's tests too; whether it is hit at all does not depend on that.
// (For the rays of ambient occlusion, which part in all directions, it lost:
// 64 rays a texel on a terrain 5.26 ms against 3.95 with a walk per lane.)
// ---------------------------------------------------------------------------
typedef __attribute__((address_space(4))) const v4f const_v4f; // read-only for the kernel: scalar loads
typedef int32_t v4i __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(4))) const v4i const_v4i;


// The children of node ref that live lanes meet within tlim: the one that
// most meet is returned, the others go onto the stack; kNoNode for none.
constexpr int32_t kNoNode = INT32_MIN;
__device__ __forceinline__ int32_t wave_children(const View& V, int32_t ref, const Seg& s, float tlim, uint64_t alive,
                                                 uint32_t* stack, uint32_t& sp)
{
	const_v4f* q = (const_v4f*)(uintptr_t)(V.nodes + ref);
	const v4f lx = q[0], ly = q[1], lz = q[2], hx = q[3], hy = q[4], hz = q[5];
	const v4i c = *(const_v4i*)(uintptr_t)(V.nodes[ref].child);
	const float t[4] = {slab(s, lx.x, ly.x, lz.x, hx.x, hy.x, hz.x, tlim), slab(s, lx.y, ly.y, lz.y, hx.y, hy.y, hz.y, tlim),
	                    slab(s, lx.z, ly.z, lz.z, hx.z, hy.z, hz.z, tlim), slab(s, lx.w, ly.w, lz.w, hx.w, hy.w, hz.w, tlim)};
	int32_t go = kNoNode;
	uint64_t most = 0;
#pragma unroll
	for (int k = 0; k < 4; ++k) {
		const uint64_t m = __ballot(t[k] != INFINITY) & alive;
		if (!m)
			continue;
		const bool first = !most || __popcll(m) > __popcll(most);
		if (most)
			stack[sp++] = (uint32_t)(first ? go : c[k]);
		if (first) {
			go = c[k];
			most = m;
		}
	}
	return __builtin_amdgcn_readfirstlane(go);
}

__device__ __forceinline__ float wave_leaf_tri(const View& V, uint32_t f, const Seg& s)
{
	const_v4f* q = (const_v4f*)(uintptr_t)(V.rtri + f);
	const v4f q0 = q[0], q1 = q[1], q2 = q[2], q3 = q[3];
	const RayTri T{q0.x, q0.y, q0.z, q0.w, q1.x, q1.y, q1.z, q1.w, q2.x, q2.y, q2.z, q2.w, q3.x, q3.y, q3.z, q3.w};
	return seg_tri_pre(s.o, s.dir, T);
}

// lanes whose segment P -> Q hits a triangle with r < 1; A: an end that all
// live segments share
__device__ __forceinline__ uint64_t wave_occluded(const View& V, f3 A, f3 P, f3 Q, bool live, uint32_t* stack)
{
	uint64_t alive = __ballot(live), hit = 0;
	if (!V.has_tris || !alive)
		return 0;
	const Seg s = make_seg(P, Q);
	// segments of at most kGridReach from A start at its cell
	const f3 d = Q - P;
	int32_t ref = __any(live && !(dot(d, d) <= kGridReach * kGridReach)) ? 0 : entry_node(V, A);
	ref = __builtin_amdgcn_readfirstlane(ref);
	uint32_t sp = 0;
	for (;;) {
		if (ref >= 0) {
			ref = wave_children(V, ref, s, 1.0f, alive, stack, sp);
			if (ref != kNoNode)
				continue;
		} else {
			const uint32_t f = leaf_first(ref), c = leaf_count(ref);
			for (uint32_t i = 0; i < c; ++i) {
				const uint64_t h = __ballot(wave_leaf_tri(V, f + i, s) < 1.0f) & alive;
				hit |= h;
				alive &= ~h;
			}
			if (!alive)
				break;
		}
		if (sp == 0)
			break;
		wave_lds_sync();
		ref = __builtin_amdgcn_readfirstlane((int)stack[--sp]);
	}
	return hit;
}

struct AOParams {
	int n;
	float distance, multiplier, falloff, effect;
	float color[3];
};

// sum plus the terms of the lanes in `of`, in ray order; only the rays that
// hit something: the others would add zero to a sum that is not negative.
__device__ __forceinline__ float add_terms(float sum, float term, uint64_t of)
{
	for (uint64_t h = __ballot(term != 0.0f) & of; h; h &= h - 1)
		sum += lane_value(term, __ffsll((unsigned long long)h) - 1);
	return sum;
}

// the texel's factor from the sum of its rays' terms, and its colour
__device__ __forceinline__ void ao_blend(uint32_t s, float ao, const AOParams& P, float* __restrict__ lm,
                                         float* __restrict__ fac_out)
{
	ao /= P.n;
	ao = tmin(ao * P.multiplier, 1.0f);
	if (P.falloff)
		ao = pow_r(ao, P.falloff);
	if (fac_out)
		fac_out[s] = ao;
	f3 out = ld3(lm + 3 * s);
	f3 col = mk3(P.color[0], P.color[1], P.color[2]);
	if (P.effect >= 0) {
		out = out * (1 - ao * (1 - P.effect)) + col * ao;
	} else {
		out = lerp3(out, lerp3(col, col * out, -P.effect), ao);
	}
	st3(lm + 3 * s, out);
}

// One wave per texel, one lane per ray (rays beyond 64 in further rounds of
// the wave): the rays of a texel start together and stay coherent, and a
// small scene still fills the GPU.  The rays' terms are then added in ray
// order, the reference's summation order, so the sum is the same.
template <bool COUNT>
// at most 80 VGPRs (6 waves per SIMD instead of 5): -3 % on the terrain's
// 191 M rays; 8 waves spill and lose
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_ao(View V, const float* __restrict__ pos, const float* __restrict__ nrm,
                                               const float* __restrict__ randoff, const float2* __restrict__ side,
                                               AOParams P, uint32_t s0, uint32_t S, float* __restrict__ lm,
                                               unsigned long long* cnt, int depth, float* __restrict__ fac_out)
{
	extern __shared__ __align__(16) unsigned char lds_stack[];
	LdsStack st = lds_stack_of_lane(lds_stack, depth);
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	// The wave's texel is uniform, so its normal, ray origin and rotation
	// offset stay in scalar registers across the traversals: in vector
	// registers they pushed the kernel past its 80-register budget, and the
	// spills wrote about 1.5 KB per wave to scratch memory.
	const uint32_t s = __builtin_amdgcn_readfirstlane(s0 + blockIdx.x * (kBlock / 64) + wave); // texels [s0, S)
	if (s >= S)
		return; // whole waves: no barrier below
	const f3 SP = ld3(pos + 3 * s), SNv = ld3(nrm + 3 * s);
	const f3 SN = mk3(wave_uniform(SNv.x), wave_uniform(SNv.y), wave_uniform(SNv.z));
	const f3 ov = SP + SN * (kSmall * 2);
	const f3 origin = mk3(wave_uniform(ov.x), wave_uniform(ov.y), wave_uniform(ov.z));
	const float ro = wave_uniform(randoff[s]);
	// The rays (at most P.distance <= kGridReach long) start at the origin's
	// entry-grid cell; its node is fetched here, before the directions are
	// computed, so that the fetch overlaps that arithmetic (taken at the
	// first walk's start instead, it was one exposed miss per texel and
	// cost more than the levels it skips).
	const int32_t start = P.distance <= kGridReach ? entry_node(V, origin) : 0;
	const uint32_t touch = reinterpret_cast<const uint32_t*>(V.nodes + start)[lane & 31];
	float ao = 0;
	for (int i0 = 0; i0 < P.n; i0 += 64) {
		const int i = i0 + lane;
		float term = 0.0f;
		if (i < P.n) {
			float angle = (i + ro) * kGoldenAngle;
			double sa, ca;
			sincos((double)angle, &sa, &ca);
			float2 sd = side[i];
			f3 d = spiral_dir(SN, sd.x, sd.y, (float)ca, (float)sa) * P.distance;
			asm volatile("" ::"v"(touch));
			const float hit = q_segment<false, COUNT>(V, origin, origin + d, cnt, st, start);
			if (hit < 1.0f)
				term = 1.0f - hit; // a miss adds nothing (ao + 0 = ao)
		}
		ao = add_terms(ao, term, ~0ull);
	}
	if (lane != 0)
		return;
	ao_blend(s, ao, P, lm, fac_out);
}

// The same for at most 32 rays: T <= 64 / n texels per wave, lane q n + i the
// i-th ray of its q-th texel.  Bound by the walks' instruction issue as k_ao is
// (0.28 VALU instructions per SIMD-cycle, 82 % L2 hits); a wave per texel left
// 47 lanes idle at 17 rays (a city's 700,001 texels 1.97 ms; packed 0.90).
// Above 32 rays no second texel fits.
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(6, 8))) void k_ao_packed(
    View V, const float* __restrict__ pos, const float* __restrict__ nrm, const float* __restrict__ randoff,
    const float2* __restrict__ side, AOParams P, uint32_t T, uint32_t s0, uint32_t S, float* __restrict__ lm,
    int depth, float* __restrict__ fac_out)
{
	extern __shared__ __align__(16) unsigned char lds_stack[];
	LdsStack st = lds_stack_of_lane(lds_stack, depth);
	const uint32_t lane = threadIdx.x & 63, n = (uint32_t)P.n;
	const uint32_t q = lane / n, i = lane - q * n;
	const uint32_t s = s0 + (blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6)) * T + q;
	const bool in = q < T && s < S;
	float term = 0.0f;
	if (in) {
		const f3 SN = ld3(nrm + 3 * (size_t)s), origin = ld3(pos + 3 * (size_t)s) + SN * (kSmall * 2);
		const float angle = (i + randoff[s]) * kGoldenAngle;
		double sa, ca;
		sincos((double)angle, &sa, &ca);
		const float2 sd = side[i];
		const f3 d = spiral_dir(SN, sd.x, sd.y, (float)ca, (float)sa) * P.distance;
		const int32_t start = P.distance <= kGridReach ? entry_node(V, origin) : 0;
		const float hit = q_segment<false, false>(V, origin, origin + d, nullptr, st, start);
		if (hit < 1.0f)
			term = 1.0f - hit;
	}
	float ao = 0.0f;
	for (uint32_t t = 0; t < T; ++t) {
		const float a = add_terms(0.0f, term, ((n < 64 ? 1ull << n : 0ull) - 1ull) << (t * n));
		ao = q == t ? a : ao;
	}
	if (in && i == 0)
		ao_blend(s, ao, P, lm, fac_out);
}

// Closest hit of DistanceTestBBT (lighter.cpp:254-289) on the binary tree
// with the canonical semantics: nearest child first by entry parameter, the
// segment's far end shrinking to the closest hit found.  Counts as
// canon_distance does.
// ANY = true: any hit, the walk ending at the first hit with r < 1 (the
// reference's VisibilityTest, lighter.cpp:112-147).
template <bool ANY>
__device__ float canon_segment(const CanonView& C, const RayTri* __restrict__ rtri, f3 A, f3 B,
                               unsigned long long& nvis, unsigned long long& ntri)
{
	float best = 2.0f;
	const Seg s = make_seg(A, B);
	nvis++; // the root's box
	if (slab(s, C.lo[0], C.lo[1], C.lo[2], C.hi[0], C.hi[1], C.hi[2], 1.0f) == INFINITY)
		return best;
	int32_t st[kCanonStack];
	float sk[kCanonStack];
	int sp = 0;
	int32_t ref = 0;
	for (;;) {
		if (ref >= 0) {
			const BvhNode n = C.nodes[ref];
			const float tl = fminf(best, 1.0f);
			float ta = slab(s, n.lo0x, n.lo0y, n.lo0z, n.hi0x, n.hi0y, n.hi0z, tl);
			float tb = slab(s, n.lo1x, n.lo1y, n.lo1z, n.hi1x, n.hi1y, n.hi1z, tl);
			int32_t a = n.c0, b = n.c1;
			nvis += 2;
			if (tb < ta) {
				float t = ta;
				ta = tb;
				tb = t;
				int32_t u = a;
				a = b;
				b = u;
			}
			if (ta != INFINITY) {
				if (tb != INFINITY) {
					st[sp] = b;
					sk[sp] = tb;
					sp++;
				}
				ref = a;
				continue;
			}
		} else {
			const uint32_t f = leaf_first(ref), c = leaf_count(ref);
			for (uint32_t i = 0; i < c; ++i) {
				const float r = seg_tri_pre(s.o, s.dir, load_rtri(rtri, f + i));
				ntri++;
				if (r < best)
					best = r;
				if (ANY && best < 1.0f)
					return best;
			}
		}
		bool found = false;
		while (sp > 0) {
			--sp;
			if (sk[sp] <= fminf(best, 1.0f)) {
				ref = st[sp];
				found = true;
				break;
			}
		}
		if (!found)
			break;
	}
	return best;
}

// The AO factor of every texel (Job_AORender_Inner, lighter.cpp:812-831)
// with the rays traced by canon_segment: one wave per texel, one lane per
// ray, the terms added in ray order, as k_ao does.  out: node visits,
// triangle tests, rays.
__global__ __launch_bounds__(kBlock) void k_ao_canon(CanonView C, const RayTri* __restrict__ rtri,
                                                     const float* __restrict__ pos, const float* __restrict__ nrm,
                                                     const float* __restrict__ randoff,
                                                     const float2* __restrict__ side, AOParams P, uint32_t S,
                                                     float* __restrict__ fac_out, unsigned long long* out)
{
	const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const uint32_t s = blockIdx.x * (kBlock / 64) + wave;
	if (s >= S)
		return;
	f3 SP = ld3(pos + 3 * s), SN = ld3(nrm + 3 * s);
	f3 origin = SP + SN * (kSmall * 2);
	float ro = randoff[s];
	float ao = 0;
	unsigned long long nv = 0, nt = 0, nr = 0;
	for (int i0 = 0; i0 < P.n; i0 += 64) {
		const int i = i0 + lane;
		float term = 0.0f;
		if (i < P.n) {
			float angle = (i + ro) * kGoldenAngle;
			double sa, ca;
			sincos((double)angle, &sa, &ca);
			float2 sd = side[i];
			f3 d = spiral_dir(SN, sd.x, sd.y, (float)ca, (float)sa) * P.distance;
			float hit = canon_segment<false>(C, rtri, origin, origin + d, nv, nt);
			nr++;
			if (hit < 1.0f)
				term = 1.0f - hit;
		}
		const int m = P.n - i0 < 64 ? P.n - i0 : 64;
		for (int k = 0; k < m; ++k)
			ao += __shfl(term, k);
	}
	atomicAdd(out + 0, nv);
	atomicAdd(out + 1, nt);
	atomicAdd(out + 2, nr);
	if (lane != 0)
		return;
	ao /= P.n;
	ao = tmin(ao * P.multiplier, 1.0f);
	if (P.falloff)
		ao = pow_r(ao, P.falloff);
	fac_out[s] = ao;
}

// The occlusion test of every candidate pair of the last link search
// (Int_RDGenLinks, lighter.cpp:751) with the canonical any-hit walk; out:
// node visits, triangle tests, pairs whose link bit differs from the
// product's.
__global__ __launch_bounds__(kBlock) void k_link_canon(CanonView C, const RayTri* __restrict__ rtri,
                                                       const float* __restrict__ pos,
                                                       const uint2* __restrict__ cand, uint64_t ncand,
                                                       const uint8_t* __restrict__ linked_by_product,
                                                       unsigned long long* out)
{
	const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= ncand)
		return;
	const uint2 c = cand[k];
	unsigned long long nv = 0, nt = 0;
	const bool occluded = canon_segment<true>(C, rtri, ld3(pos + 3 * c.x), ld3(pos + 3 * c.y), nv, nt) < 1.0f;
	const bool linked = linked_by_product[k] != 0;
	atomicAdd(out + 0, nv);
	atomicAdd(out + 1, nt);
	if (occluded != linked)
		atomicAdd(out + 2, 1ull);
}

// ---------------------------------------------------------------------------
// point-query kernels (tests, timing)
// ---------------------------------------------------------------------------
__global__ void k_q_distance(View V, const float* p, uint32_t n, float* out)
{
	uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = q_distance<false>(V, ld3(p + 3 * i), kPenumbraSize, nullptr);
}

__global__ void k_q_closest(View V, const float* a, const float* b, uint32_t n, float* out)
{
	uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = q_segment<false, false>(V, ld3(a + 3 * i), ld3(b + 3 * i), nullptr);
}

__global__ void k_q_occluded(View V, const float* a, const float* b, uint32_t n, uint8_t* out)
{
	uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = q_segment<true, false>(V, ld3(a + 3 * i), ld3(b + 3 * i), nullptr) < 1.0f ? 1 : 0;
}

// ---------------------------------------------------------------------------
// radiosity links (lighter.cpp:728-759)
// ---------------------------------------------------------------------------
// Form factor of the pair (i < j) exactly as the reference evaluates it, or
// -1 when the pair fails the geometric thresholds (NaN inputs fail neither
// comparison, as in the reference, and give a NaN factor).
__device__ __forceinline__ float pair_factor(f3 ap, f3 an, f3 bp, f3 bn)
{
	f3 d = bp - ap;
	float da = dot(an, d);
	float db = dot(bn, -d);
	if (da <= kSmall || db <= kSmall)
		return -1.0f;
	float l2 = lensq(d);
	float f = da * db / (l2 * l2 * kPiF);
	if (f < kSmall)
		return -1.0f;
	return f;
}

constexpr int kPairChunk = 256;

// Pass 0 counts, pass 1 writes: candidates of row i in columns
// [c*kPairChunk, +kPairChunk) restricted to j > i, in ascending j.
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void k_pairs(const float* __restrict__ pos, const float* __restrict__ nrm,
                                                  uint32_t N, uint32_t nchunks, uint32_t* __restrict__ counts,
                                                  const uint64_t* __restrict__ offsets, uint2* __restrict__ cand)
{
	uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	uint32_t c = blockIdx.y;
	if (i >= N)
		return;
	uint32_t j0 = c * kPairChunk, j1 = min(N, j0 + kPairChunk);
	if (j0 <= i)
		j0 = i + 1;
	uint32_t n = 0;
	uint64_t base = WRITE ? offsets[(uint64_t)i * nchunks + c] : 0;
	if (j0 < j1) {
		f3 ap = ld3(pos + 3 * i), an = ld3(nrm + 3 * i);
		for (uint32_t j = j0; j < j1; ++j) {
			float f = pair_factor(ap, an, ld3(pos + 3 * j), ld3(nrm + 3 * j));
			if (!(f < 0.0f)) { // -1: failed; NaN passes, as in the reference's comparisons
				if (WRITE)
					cand[base + n] = make_uint2(i, j);
				n++;
			}
		}
	}
	if (!WRITE)
		counts[(uint64_t)i * nchunks + c] = n;
}

// ---------------------------------------------------------------------------
// The link search over clusters of 64 patches.  Patches are binned by the
// dominant axis of their normal and a cell of their position, so a cluster
// (and each quarter of it) is a compact patch of one kind of surface; its box
// and the range of its normals bound every factor between two clusters, and
// only pairs of clusters with quarters that could hold a pair of kSmall or
// more are looked at.  One wave takes a pair of clusters and tests its pairs
// of patches with the arithmetic of the all-pairs search (pair_factor; it
// gives the same bits from either end, since the differences and dot
// products only change sign) into a 64 x 64 bit matrix; the occlusion tests
// take 64 of its pairs at a time, which start and end at neighbouring
// patches, and leave the links' bits in it.  No candidate is stored, and the
// CSR's counts and cursors take one atomic per patch and cluster pair
// instead of one per link.
// ---------------------------------------------------------------------------
constexpr uint32_t kCl = 64;        // patches per cluster, and clusters per super-cluster
constexpr uint32_t kNoPatch = ~0u;  // padding of the last cluster

struct ClBox {
	float lo[3], hi[3];   // positions
	float nlo[3], nhi[3]; // normals
};

// Bins of the patches: the dominant axis and sign of the normal, then the
// cell of a uniform grid along a Morton curve (in x-major order the 64
// patches of a cluster lay in a row of cells, 119 m long in a city).
struct PatchBins {
	float lo[3], inv;  // 1 / cell width
	uint32_t bits[3];  // 2^bits cells per axis
};

__global__ void k_patch_bins(const float* __restrict__ pos, const float* __restrict__ nrm, uint32_t N, PatchBins G,
                             uint32_t* __restrict__ bin, uint32_t* __restrict__ count)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= N)
		return;
	const f3 p = ld3(pos + 3 * (size_t)i), n = ld3(nrm + 3 * (size_t)i);
	const float ax = fabsf(n.x), ay = fabsf(n.y), az = fabsf(n.z);
	const uint32_t side = ax >= ay && ax >= az ? (n.x < 0 ? 0u : 1u) : ay >= az ? (n.y < 0 ? 2u : 3u) : (n.z < 0 ? 4u : 5u);
	const float q[3] = {(p.x - G.lo[0]) * G.inv, (p.y - G.lo[1]) * G.inv, (p.z - G.lo[2]) * G.inv};
	uint32_t c[3], k = side, bits = max(max(G.bits[0], G.bits[1]), G.bits[2]);
	for (int a = 0; a < 3; ++a)
		c[a] = min((1u << G.bits[a]) - 1, (uint32_t)q[a]); // p >= lo: q >= 0
	while (bits--)
		for (int a = 2; a >= 0; --a)
			if (bits < G.bits[a])
				k = k << 1 | (c[a] >> bits & 1u);
	bin[i] = k;
	atomicAdd(count + k, 1u);
}

// The patches in bin order (any order within a bin: it only decides which
// patches share a cluster), padded to whole clusters: position and index,
// normal.  count serves as the bins' cursors, counted down to zero.
__global__ void k_patch_place(const float* __restrict__ pos, const float* __restrict__ nrm, uint32_t N, uint32_t Npad,
                              const uint32_t* __restrict__ bin, const uint64_t* __restrict__ start,
                              uint32_t* __restrict__ count, float4* __restrict__ sp, float4* __restrict__ sn)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= Npad)
		return;
	uint64_t t = i;
	float4 a = make_float4(0, 0, 0, __uint_as_float(kNoPatch)), b = make_float4(0, 0, 0, 0);
	if (i < N) {
		const uint32_t k = bin[i];
		t = start[k] + (atomicSub(count + k, 1u) - 1u);
		const f3 p = ld3(pos + 3 * (size_t)i), n = ld3(nrm + 3 * (size_t)i);
		a = make_float4(p.x, p.y, p.z, __uint_as_float(i));
		b = make_float4(n.x, n.y, n.z, 0.0f);
	}
	sp[t] = a;
	sn[t] = b;
}

// the union over the lane's group of G lanes
template <int G>
__device__ __forceinline__ void group_box(ClBox& b)
{
	for (int o = G / 2; o > 0; o >>= 1)
		for (int a = 0; a < 3; ++a) {
			b.lo[a] = fminf(b.lo[a], __shfl_xor(b.lo[a], o));
			b.hi[a] = fmaxf(b.hi[a], __shfl_xor(b.hi[a], o));
			b.nlo[a] = fminf(b.nlo[a], __shfl_xor(b.nlo[a], o));
			b.nhi[a] = fmaxf(b.nhi[a], __shfl_xor(b.nhi[a], o));
		}
}

__device__ __forceinline__ ClBox empty_box()
{
	ClBox b;
	for (int a = 0; a < 3; ++a) {
		b.lo[a] = b.nlo[a] = INFINITY;
		b.hi[a] = b.nhi[a] = -INFINITY;
	}
	return b;
}

// one wave per cluster: its bounds and those of its quarters (16 patches)
__global__ __launch_bounds__(kBlock) void k_cluster_boxes(const float4* __restrict__ sp, const float4* __restrict__ sn,
                                                          uint32_t nc, ClBox* __restrict__ box, ClBox* __restrict__ quart)
{
	const uint32_t c = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if (c >= nc)
		return;
	ClBox b = empty_box();
	const float4 p = sp[(size_t)c * kCl + lane], n = sn[(size_t)c * kCl + lane];
	if (__float_as_uint(p.w) != kNoPatch) {
		b.lo[0] = b.hi[0] = p.x, b.lo[1] = b.hi[1] = p.y, b.lo[2] = b.hi[2] = p.z;
		b.nlo[0] = b.nhi[0] = n.x, b.nlo[1] = b.nhi[1] = n.y, b.nlo[2] = b.nhi[2] = n.z;
	}
	group_box<16>(b);
	if ((lane & 15) == 0)
		quart[4 * (size_t)c + (lane >> 4)] = b;
	group_box<64>(b);
	if (lane == 0)
		box[c] = b;
}

// one wave per super-cluster: the bounds of its 64 clusters
__global__ __launch_bounds__(kBlock) void k_super_boxes(const ClBox* __restrict__ box, uint32_t nc, uint32_t ns,
                                                        ClBox* __restrict__ sup)
{
	const uint32_t s = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if (s >= ns)
		return;
	const size_t c = (size_t)s * kCl + lane;
	ClBox b = c < nc ? box[c] : empty_box();
	group_box<64>(b);
	if (lane == 0)
		sup[s] = b;
}

// False when no patch of A and patch of B can pass pair_factor.  With d
// from A to B in [dlo, dhi], dA = nA . d and dB = -nB . d are at most the
// interval products' sums; both have to exceed kSmall, and f = dA dB / (pi
// l^4) has to reach it with l at least the boxes' distance; dA <= |nA| l and
// dB <= |nB| l give three more bounds.  The margins (4e-6 of the terms'
// magnitude, 1e-3 of f) are tens of times the rounding of pair_factor and of
// these bounds.  Distances of 1e9 and more, whose powers might overflow in
// pair_factor, are left to it.
__device__ __forceinline__ bool may_link(const ClBox& A, const ClBox& B)
{
	float da = 0, db = 0, l2 = 0, ext = 0, na = 0, nb = 0, na2 = 0, nb2 = 0;
#pragma unroll
	for (int a = 0; a < 3; ++a) {
		const float dlo = B.lo[a] - A.hi[a], dhi = B.hi[a] - A.lo[a];
		da += fmaxf(fmaxf(A.nlo[a] * dlo, A.nlo[a] * dhi), fmaxf(A.nhi[a] * dlo, A.nhi[a] * dhi));
		db += fmaxf(fmaxf(-B.nlo[a] * dlo, -B.nlo[a] * dhi), fmaxf(-B.nhi[a] * dlo, -B.nhi[a] * dhi));
		const float gap = fmaxf(fmaxf(dlo, -dhi), 0.0f);
		l2 += gap * gap;
		ext += fmaxf(fabsf(dlo), fabsf(dhi));
		const float ma = fmaxf(fabsf(A.nlo[a]), fabsf(A.nhi[a])), mb = fmaxf(fabsf(B.nlo[a]), fabsf(B.nhi[a]));
		na += ma;
		nb += mb;
		na2 += ma * ma;
		nb2 += mb * mb;
	}
	da += 4e-6f * ext * na;
	db += 4e-6f * ext * nb;
	if (da <= kSmall || db <= kSmall)
		return false;
	if (l2 > 0.0f && l2 < 1e18f) {
		const float l = sqrtf(l2), lim = kSmall * kPiF * 0.999f;
		na2 = sqrtf(na2) * 1.0001f;
		nb2 = sqrtf(nb2) * 1.0001f;
		if (da * db < lim * l2 * l2 || da * nb2 < lim * l2 * l || db * na2 < lim * l2 * l || na2 * nb2 < lim * l2)
			return false;
	}
	return true;
}

// One wave per cluster a: its partners b >= a, super-clusters first, then
// clusters, then the 16 pairs of quarters (four partners at a time).  Pass 0
// counts, pass 1 writes the pair and the quarters that may link (bit 4 qa +
// qb) of the clusters from a0 to a1 - 1, whose first is the pair base.
template <bool WRITE>
__global__ __launch_bounds__(kBlock) void k_cluster_pairs(const ClBox* __restrict__ box, const ClBox* __restrict__ quart,
                                                          uint32_t nc, const ClBox* __restrict__ sup, uint32_t ns,
                                                          uint32_t a0, uint32_t a1, uint32_t* __restrict__ count,
                                                          const uint64_t* __restrict__ offs, uint64_t base,
                                                          uint2* __restrict__ out, uint16_t* __restrict__ quarters)
{
	const uint32_t a = a0 + blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
	if (a >= a1)
		return;
	const ClBox A = box[a], Aq = quart[4 * (size_t)a + ((lane >> 2) & 3)];
	uint64_t at = WRITE ? offs[a] - base : 0;
	for (uint32_t s0 = a / kCl; s0 < ns; s0 += 64) {
		uint64_t m = __ballot(s0 + lane < ns && may_link(A, sup[min(s0 + lane, ns - 1)]));
		while (m) {
			const uint32_t b0 = (s0 + (uint32_t)__ffsll((unsigned long long)m) - 1u) * kCl, b = b0 + lane;
			m &= m - 1;
			uint64_t k = __ballot(b >= a && b < nc && may_link(A, box[min(b, nc - 1)]));
			while (k) {
				// the next four partners, one per 16 lanes
				uint32_t mine = 64;
				for (uint32_t g = 0; g < 4 && k; ++g) {
					if (lane >> 4 == g)
						mine = (uint32_t)__ffsll((unsigned long long)k) - 1u;
					k &= k - 1;
				}
				const bool ok = mine < 64 && may_link(Aq, quart[4 * (size_t)(b0 + (mine & 63)) + (lane & 3)]);
				const uint64_t q = __ballot(ok);
				for (uint32_t g = 0; g < 4; ++g) {
					const uint32_t bits = (uint32_t)(q >> (16 * g)) & 0xffffu;
					if (!bits)
						continue;
					if (WRITE && lane == 16 * g) {
						out[at] = make_uint2(a, b0 + mine);
						quarters[at] = (uint16_t)bits;
					}
					++at;
				}
			}
		}
	}
	if (!WRITE && lane == 0)
		count[a] = (uint32_t)at;
}

struct PairWork {
	const float4* __restrict__ sp;
	const float4* __restrict__ sn;
	const uint2* __restrict__ pairs;
	uint32_t npairs;
};

// One wave per cluster pair: the bit matrix of the pairs that pass
// pair_factor (row: a patch of the first cluster) and their number.  A lane
// keeps its patch of the second cluster; the first cluster's patches are
// uniform.  Bound by instruction issue, about 30 a pair of patches (0.23-0.27
// VALU and 0.09 scalar instructions per SIMD-cycle, 11-14 % of the wave-cycles
// waiting).
__global__ __launch_bounds__(kBlock) void k_cluster_masks(PairWork W, const uint16_t* __restrict__ quarters,
                                                          uint64_t* __restrict__ mask, uint32_t* __restrict__ ncand)
{
	const uint32_t lane = threadIdx.x & 63;
	const uint32_t p = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
	if (p >= W.npairs)
		return;
	const uint2 ab = W.pairs[p];
	const uint32_t qm = (uint32_t)__builtin_amdgcn_readfirstlane((int)quarters[p]);
	const size_t a0 = (size_t)ab.x * kCl;
	const float4 jp = W.sp[(size_t)ab.y * kCl + lane], jn = W.sn[(size_t)ab.y * kCl + lane];
	const f3 bp = mk3(jp.x, jp.y, jp.z), bn = mk3(jn.x, jn.y, jn.z);
	const bool jok = __float_as_uint(jp.w) != kNoPatch;
	const uint32_t from = ab.x == ab.y ? lane : kCl; // within a cluster: rows above the diagonal
	uint64_t row = 0;
	uint32_t n = 0;
	for (uint32_t q = 0; q < 4; ++q) {
		const uint32_t g = (qm >> (4 * q)) & 15u;
		if (!g)
			continue;
		const bool in = jok && (g >> (lane >> 4) & 1u);
		for (uint32_t i = 16 * q; i < 16 * q + 16; ++i) {
			const float4 ip = W.sp[a0 + i], in_ = W.sn[a0 + i];
			const bool ok = in && i < from && __float_as_uint(ip.w) != kNoPatch &&
			                !(pair_factor(mk3(ip.x, ip.y, ip.z), mk3(in_.x, in_.y, in_.z), bp, bn) < 0.0f);
			const uint64_t m = __ballot(ok);
			row = lane == i ? m : row;
			n += (uint32_t)__popcll(m);
		}
	}
	if (lane == 0)
		ncand[p] = n;
	if (n)
		mask[(size_t)p * kCl + lane] = row;
}

// The pairs that hold candidates, in order: their places before compaction
// (of[], where their masks are) and the first of each cluster (first[p] -
// base before).
__global__ void k_cluster_flags(const uint32_t* __restrict__ ncand, uint64_t n, uint32_t* __restrict__ flag)
{
	const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (p <= n)
		flag[p] = p < n && ncand[p] ? 1u : 0u;
}

__global__ void k_cluster_compact(uint64_t n, const uint64_t* __restrict__ at, uint32_t nc,
                                  const uint64_t* __restrict__ first, uint64_t base, const uint2* __restrict__ pairs,
                                  uint2* __restrict__ pairs2, uint32_t* __restrict__ of, uint64_t* __restrict__ first2)
{
	const uint64_t p = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (p < n && at[p + 1] != at[p]) {
		pairs2[at[p]] = pairs[p];
		of[at[p]] = (uint32_t)p;
	}
	if (p <= nc)
		first2[p] = at[first[p] - base];
}

// The occlusion tests, one wave per patch i of a cluster: its candidates in
// the cluster's partners, 64 partners at a time, through a queue in LDS into
// batches of 64.  A pair links when the segment between the patches hits a
// shadow caster (VisibilityTest returns the any-hit query's hit,
// lighter.cpp:137-147, and Int_RDGenLinks keeps the pair when it is true,
// lighter.cpp:751-752), the lower index as its start.  A batch's segments
// share one end, and the other ends go along the clusters' Morton order, so
// their walks take much the same nodes (batches per cluster pair, some seven
// patches of the first cluster in each, took 19.3 ms instead of 16.4 on a
// city of 440,003 patches with 139 M candidates).  Bound by the walks'
// instruction issue (0.33 VALU and 0.14-0.15 scalar instructions per
// SIMD-cycle; 95 % of the fetches hit the L2).  A city's whole search, kernels: 50 ms with a uniform
// grid's candidate list (30.1 ms of pair tests, made twice; 12.6 ms of
// occlusion tests on the list), 26 ms so (pair tests 2.4 ms); a room's 20 ->
// 12 ms.
// Where the patches are too few to fill the chip's waves, 2^split waves take a
// patch, each a run of its cluster's partners, until there are kLinkWaves
// (whole searches: a terrain of 3,001 patches 1.27 -> 0.70 ms, of 12,001 3.77
// -> 2.60, a room of 6,001 1.43 -> 1.10; up to twice as many gained a terrain
// of 32,768 6.24 -> 5.72 and lost a city of 32,768 2.05 -> 2.26).
// a0: the cluster that first[0] is of.
// mask: the candidates' bits in, the links' out.  cand, linked (optional): the
// candidates and whether each linked, a wave's from its candoff on.
// The walk is one for the wave (wave_occluded).  Against a walk per lane: a room's
// 12.7 -> 8.8 ms (25 G segments/s), a city's 16.4 -> 14.5 ms.
constexpr uint32_t kLinkWaves = 32768, kLinkSplitMax = 4;
struct LinkWave {
	uint32_t stack[kStackSize];
	uint32_t row[128]; // the candidates of 64 partners, from when they are queued on the links among them
	uint16_t queue[128];
};
__global__ __launch_bounds__(kBlock) void k_cluster_links(
    View V, PairWork W, uint32_t a0, const uint64_t* __restrict__ first, const uint32_t* __restrict__ of,
    uint32_t split, uint64_t* __restrict__ mask, const uint64_t* __restrict__ candoff, uint2* __restrict__ cand,
    uint8_t* __restrict__ linked)
{
	__shared__ LinkWave waves[kBlock / 64];
	constexpr uint32_t per = kCl / (kBlock / 64); // blocks per cluster
	const uint32_t lane = threadIdx.x & 63;
	const uint32_t wave = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
	const uint32_t a = (blockIdx.x / per) >> split, part = (blockIdx.x / per) & ((1u << split) - 1u);
	const uint32_t i = blockIdx.x % per * (kBlock / 64) + wave;
	const float4 A = W.sp[(size_t)(a0 + a) * kCl + i];
	const uint32_t ia = __float_as_uint(A.w);
	if (ia == kNoPatch)
		return; // the whole wave; no block barrier below
	LinkWave& L = waves[wave];
	const uint64_t begin = first[a], partners = first[a + 1] - begin;
	const uint64_t end = begin + (partners * (part + 1) >> split);
	uint64_t at = cand ? candoff[blockIdx.x * (kBlock / 64) + wave] : 0;
	for (uint64_t p0 = begin + (partners * part >> split); p0 < end; p0 += 64) {
		uint64_t parts;
		{
			const uint64_t m = p0 + lane < end ? mask[(size_t)of[p0 + lane] * kCl + i] : 0;
			L.row[2 * lane] = (uint32_t)m;
			L.row[2 * lane + 1] = (uint32_t)(m >> 32);
			parts = __ballot(m != 0);
		}
		if (!parts)
			continue;
		wave_lds_sync();
		uint32_t qn = 0;
		for (;;) {
			while (qn < 64 && parts) { // partners into the queue until it holds 64 candidates
				const uint32_t q = (uint32_t)__ffsll((unsigned long long)parts) - 1u;
				parts &= parts - 1;
				const uint64_t m = (uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)L.row[2 * q + 1]) << 32 |
				                   (uint32_t)__builtin_amdgcn_readfirstlane((int)L.row[2 * q]);
				if (m >> lane & 1ull)
					L.queue[qn + __popcll(m & ((1ull << lane) - 1ull))] = (uint16_t)(q << 6 | lane);
				L.row[2 * q] = L.row[2 * q + 1] = 0u;
				qn += (uint32_t)__popcll(m);
			}
			if (!qn)
				break;
			wave_lds_sync();
			const uint32_t n = min(qn, 64u);
			const uint32_t e0 = L.queue[min(lane, n - 1)];
			const float4 B = W.sp[(size_t)W.pairs[p0 + (e0 >> 6)].y * kCl + (e0 & 63u)];
			const bool up = ia < __float_as_uint(B.w);
			const f3 P = mk3(up ? A.x : B.x, up ? A.y : B.y, up ? A.z : B.z);
			const f3 Q = mk3(up ? B.x : A.x, up ? B.y : A.y, up ? B.z : A.z);
			const bool l = wave_occluded(V, mk3(A.x, A.y, A.z), P, Q, lane < n, L.stack) >> lane & 1ull;
			wave_lds_sync();
			if (l) {
				const uint32_t e = L.queue[lane];
				atomicOr(&L.row[e >> 5], 1u << (e & 31u));
			}
			if (cand) {
				if (lane < n) {
					const uint32_t e = L.queue[lane];
					const uint32_t ib = __float_as_uint(W.sp[(size_t)W.pairs[p0 + (e >> 6)].y * kCl + (e & 63u)].w);
					cand[at + lane] = make_uint2(min(ia, ib), max(ia, ib));
					linked[at + lane] = l ? 1 : 0;
				}
				at += n;
			}
			const uint16_t rest = L.queue[64 + lane];
			wave_lds_sync();
			if (lane + 64 < qn)
				L.queue[lane] = rest;
			wave_lds_sync();
			qn -= n;
		}
		if (p0 + lane < end)
			mask[(size_t)of[p0 + lane] * kCl + i] = (uint64_t)L.row[2 * lane + 1] << 32 | L.row[2 * lane];
		wave_lds_sync();
	}
}

// The candidates of each of k_cluster_links' waves (measurement only): an
// atomic on one cursor per batch doubled the search of a room of 32,768
// patches with 215 M of them (22 -> 44 ms).
__global__ __launch_bounds__(kBlock) void k_cluster_wave_candidates(const uint64_t* __restrict__ first,
                                                                    const uint32_t* __restrict__ of, uint32_t split,
                                                                    const uint64_t* __restrict__ mask,
                                                                    uint32_t* __restrict__ count)
{
	constexpr uint32_t per = kCl / (kBlock / 64);
	const uint32_t lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
	const uint32_t a = (blockIdx.x / per) >> split, part = (blockIdx.x / per) & ((1u << split) - 1u);
	const uint32_t i = blockIdx.x % per * (kBlock / 64) + wave;
	const uint64_t begin = first[a], partners = first[a + 1] - begin;
	const uint64_t end = begin + (partners * (part + 1) >> split);
	uint32_t n = 0;
	for (uint64_t p = begin + (partners * part >> split) + lane; p < end; p += 64)
		n += (uint32_t)__popcll(mask[(size_t)of[p] * kCl + i]);
	for (int o = 32; o > 0; o >>= 1)
		n += (uint32_t)__shfl_xor((int)n, o);
	if (lane == 0)
		count[blockIdx.x * (kBlock / 64) + wave] = n;
}

// One wave per cluster pair: its links per patch of both clusters.
__global__ __launch_bounds__(kBlock) void k_cluster_degrees(PairWork W, const uint32_t* __restrict__ of,
                                                            const uint64_t* __restrict__ mask,
                                                            uint32_t* __restrict__ deg)
{
	const uint32_t lane = threadIdx.x & 63;
	const uint32_t p = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
	if (p >= W.npairs)
		return;
	const uint2 ab = W.pairs[p];
	const uint64_t row = mask[(size_t)of[p] * kCl + lane];
	if (!__any(row != 0))
		return;
	uint32_t col = 0;
	for (uint32_t j = 0; j < kCl; ++j) {
		const uint32_t c = (uint32_t)__popcll(__ballot((row >> j) & 1ull));
		col = lane == j ? c : col;
	}
	if (row)
		atomicAdd(deg + __float_as_uint(W.sp[(size_t)ab.x * kCl + lane].w), (uint32_t)__popcll(row));
	if (col)
		atomicAdd(deg + __float_as_uint(W.sp[(size_t)ab.y * kCl + lane].w), col);
}

// One wave per cluster pair that holds links: its links into both patches'
// rows (any order; the row sort orders them).  fill starts at zero.
__global__ __launch_bounds__(kBlock) void k_cluster_fill(PairWork W, const uint32_t* __restrict__ of,
                                                         const uint64_t* __restrict__ mask,
                                                         const uint64_t* __restrict__ rowptr,
                                                         uint32_t* __restrict__ fill, uint32_t* __restrict__ colx)
{
	const uint32_t lane = threadIdx.x & 63;
	const uint32_t p = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
	if (p >= W.npairs)
		return;
	const uint2 ab = W.pairs[p];
	const uint32_t ia = __float_as_uint(W.sp[(size_t)ab.x * kCl + lane].w), ib = __float_as_uint(W.sp[(size_t)ab.y * kCl + lane].w);
	const uint64_t row = mask[(size_t)of[p] * kCl + lane], below = (1ull << lane) - 1ull;
	if (!__any(row != 0))
		return;
	uint64_t at = row ? rowptr[ia] + atomicAdd(fill + ia, (uint32_t)__popcll(row)) : 0;
	for (uint32_t i = 0; i < kCl; ++i) {
		const uint64_t r = __shfl(row, (int)i), o = __shfl(at, (int)i);
		if (r >> lane & 1ull)
			colx[o + __popcll(r & below)] = ib;
	}
	uint64_t col = 0;
	for (uint32_t j = 0; j < kCl; ++j) {
		const uint64_t c = __ballot((row >> j) & 1ull);
		col = lane == j ? c : col;
	}
	at = col ? rowptr[ib] + atomicAdd(fill + ib, (uint32_t)__popcll(col)) : 0;
	for (uint32_t j = 0; j < kCl; ++j) {
		const uint64_t c = __shfl(col, (int)j), o = __shfl(at, (int)j);
		if (c >> lane & 1ull)
			colx[o + __popcll(c & below)] = ia;
	}
}

// The occlusion test of each candidate: the pair links when the segment
// between the patches hits a shadow caster (VisibilityTest returns the
// any-hit query's hit, lighter.cpp:137-147, and Int_RDGenLinks keeps the
// pair when it is true, lighter.cpp:751-752).  Each link (i, j > i) also
// counts toward row j's links below the diagonal; the candidates of one row
// are contiguous, so the lanes of a wave add to different rows.
__global__ __launch_bounds__(kBlock) void k_link_test(View V, const float* __restrict__ pos,
                                                      const uint2* __restrict__ cand, uint64_t ncand,
                                                      uint8_t* __restrict__ linked, uint32_t* __restrict__ lower,
                                                      int depth)
{
	extern __shared__ __align__(16) unsigned char lds_stack[];
	LdsStack st = lds_stack_of_lane(lds_stack, depth);
	const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= ncand)
		return;
	const uint2 c = cand[k];
	const bool l = q_segment<true, false>(V, ld3(pos + 3 * c.x), ld3(pos + 3 * c.y), nullptr, st) < 1.0f;
	linked[k] = l ? 1 : 0;
	if (l)
		atomicAdd(lower + c.y, 1u);
}

// Links of row i above the diagonal: its own linked candidates, one wave
// per row.  With colx null, their count goes to upper[i]; otherwise they
// are written after the row's lower part, in candidate order.
__global__ __launch_bounds__(kBlock) void k_link_upper(uint32_t N, const uint64_t* __restrict__ coff,
                                                       const uint2* __restrict__ cand,
                                                       const uint8_t* __restrict__ linked,
                                                       uint32_t* __restrict__ upper,
                                                       const uint64_t* __restrict__ rowptr,
                                                       const uint32_t* __restrict__ lower, uint32_t* __restrict__ colx)
{
	const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
	const int lane = threadIdx.x & 63;
	if (i >= N)
		return; // the whole wave
	const uint64_t e = coff[i + 1];
	uint64_t at = colx ? rowptr[i] + lower[i] : 0;
	for (uint64_t k0 = coff[i]; k0 < e; k0 += 64) {
		const uint64_t k = k0 + lane;
		const bool l = k < e && linked[k];
		const uint64_t m = __ballot(l);
		if (colx && l)
			colx[at + __popcll(m & ((1ull << lane) - 1ull))] = cand[k].y;
		at += __popcll(m);
	}
	if (!colx && lane == 0)
		upper[i] = (uint32_t)at;
}

// Links of row j below the diagonal: every linked candidate (i, j) puts i
// into row j's lower part (any order; the row sort orders it)
__global__ void k_link_lower(const uint2* __restrict__ cand, const uint8_t* __restrict__ linked, uint64_t ncand,
                             const uint64_t* __restrict__ rowptr, uint32_t* __restrict__ lfill,
                             uint32_t* __restrict__ colx)
{
	const uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (k >= ncand || !linked[k])
		return;
	const uint2 c = cand[k];
	colx[rowptr[c.y] + atomicAdd(lfill + c.y, 1u)] = c.x;
}

__global__ void k_row_sum(uint32_t N, const uint32_t* __restrict__ a, const uint32_t* __restrict__ b,
                          uint32_t* __restrict__ out)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i < N)
		out[i] = a[i] + b[i];
}

// factor of every link (columns ascending within a row), one wave per row;
// the reference evaluates each pair with the lower index as A
__global__ __launch_bounds__(kBlock) void k_link_factors(uint32_t N, const uint64_t* __restrict__ rowptr,
                                                         const uint32_t* __restrict__ col,
                                                         const float* __restrict__ pos,
                                                         const float* __restrict__ nrm, float* __restrict__ val)
{
	const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
	const int lane = threadIdx.x & 63;
	if (i >= N)
		return;
	const f3 ip = ld3(pos + 3 * i), in_ = ld3(nrm + 3 * i);
	const uint64_t e = rowptr[i + 1];
	for (uint64_t o = rowptr[i] + lane; o < e; o += 64) {
		const uint32_t j = col[o];
		const f3 jp = ld3(pos + 3 * j), jn = ld3(nrm + 3 * j);
		val[o] = (i < j) ? pair_factor(ip, in_, jp, jn) : pair_factor(jp, jn, ip, in_);
	}
}

// first candidate of every row from the all-pairs search's per-(row, chunk)
// offsets
__global__ void k_row_first(uint32_t N, uint32_t nchunks, const uint64_t* __restrict__ offs, uint64_t total,
                            uint64_t* __restrict__ coff)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i <= N)
		coff[i] = i < N ? offs[(uint64_t)i * nchunks] : total;
}

__global__ void k_u64_to_u32(const uint64_t* __restrict__ in, uint64_t n, uint32_t* __restrict__ out)
{
	const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
	if (i < n)
		out[i] = (uint32_t)in[i];
}

// One bounce of Int_RDBounce (lighter.cpp:767-797) as a gather over the
// symmetric links: in_i = sum_j ((out_j * diffuse_j) * area_j) * f_ij.  The
// factor-free part x_j = (out_j * diffuse_j) * area_j is formed once per
// patch (the same products in the same order as the reference's per-link
// expression); one wave per row then sums x_j * f_ij over the row's links,
// lane l taking links l, l + 64, .., and the lanes' partial sums meet in a
// fixed butterfly (deterministic, and rows of thousands of links read
// their columns and factors in coalesced runs).
__global__ void k_bounce_prep(uint32_t N, const float* __restrict__ out, const float* __restrict__ diffuse,
                              const float* __restrict__ area, float4* __restrict__ x)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= N)
		return;
	const f3 v = (ld3(out + 3 * i) * ld3(diffuse + 3 * i)) * area[i];
	x[i] = make_float4(v.x, v.y, v.z, 0.0f);
}

__global__ __launch_bounds__(kBlock) void k_bounce_rows(uint32_t N, const uint64_t* __restrict__ rowptr,
                                                        const uint32_t* __restrict__ col,
                                                        const float* __restrict__ val, const float4* __restrict__ x,
                                                        float* __restrict__ in, float* __restrict__ total)
{
	const uint32_t i = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6);
	const int lane = threadIdx.x & 63;
	if (i >= N)
		return; // the whole wave
	float a0 = 0.0f, a1 = 0.0f, a2 = 0.0f;
	const uint64_t e = rowptr[i + 1];
	for (uint64_t k = rowptr[i] + lane; k < e; k += 64) {
		const float4 v = x[col[k]];
		const float f = val[k];
		a0 += v.x * f;
		a1 += v.y * f;
		a2 += v.z * f;
	}
#pragma unroll
	for (int o = 32; o > 0; o >>= 1) {
		a0 += __shfl_xor(a0, o);
		a1 += __shfl_xor(a1, o);
		a2 += __shfl_xor(a2, o);
	}
	if (lane == 0) {
		const f3 acc = mk3(a0, a1, a2);
		st3(in + 3 * i, acc);
		st3(total + 3 * i, ld3(total + 3 * i) + acc);
	}
}

// ---------------------------------------------------------------------------
// exclusive scan of u32 counts into u64 offsets (three-phase)
// ---------------------------------------------------------------------------
__global__ void k_scan_blocks(const uint32_t* __restrict__ in, uint64_t n, uint64_t* __restrict__ out,
                              uint64_t* __restrict__ block_sums)
{
	__shared__ uint64_t sh[kBlock];
	constexpr int kPer = 16;
	uint64_t base = (uint64_t)blockIdx.x * kBlock * kPer + (uint64_t)threadIdx.x * kPer;
	uint64_t local[kPer];
	uint64_t s = 0;
	for (int k = 0; k < kPer; ++k) {
		uint64_t idx = base + k;
		local[k] = s;
		s += (idx < n) ? in[idx] : 0;
	}
	sh[threadIdx.x] = s;
	__syncthreads();
	for (int off = 1; off < kBlock; off <<= 1) {
		uint64_t v = threadIdx.x >= (unsigned)off ? sh[threadIdx.x - off] : 0;
		__syncthreads();
		sh[threadIdx.x] += v;
		__syncthreads();
	}
	uint64_t excl = sh[threadIdx.x] - s;
	for (int k = 0; k < kPer; ++k) {
		uint64_t idx = base + k;
		if (idx < n)
			out[idx] = excl + local[k];
	}
	if (threadIdx.x == kBlock - 1)
		block_sums[blockIdx.x] = sh[threadIdx.x];
}

// one block: each thread's run of block sums, the runs' scan, the runs again
__global__ __launch_bounds__(kBlock) void k_scan_sums(uint64_t* sums, uint32_t nb, uint64_t* total)
{
	__shared__ uint64_t sh[kBlock];
	const uint32_t per = (nb + kBlock - 1) / kBlock, b0 = min(nb, threadIdx.x * per), b1 = min(nb, b0 + per);
	uint64_t s = 0;
	for (uint32_t b = b0; b < b1; ++b)
		s += sums[b];
	sh[threadIdx.x] = s;
	__syncthreads();
	for (int off = 1; off < kBlock; off <<= 1) {
		const uint64_t v = threadIdx.x >= (unsigned)off ? sh[threadIdx.x - off] : 0;
		__syncthreads();
		sh[threadIdx.x] += v;
		__syncthreads();
	}
	uint64_t run = sh[threadIdx.x] - s;
	for (uint32_t b = b0; b < b1; ++b) {
		const uint64_t v = sums[b];
		sums[b] = run;
		run += v;
	}
	if (threadIdx.x == kBlock - 1)
		*total = run;
}

__global__ void k_scan_add(uint64_t* out, uint64_t n, const uint64_t* sums)
{
	constexpr int kPer = 16;
	uint64_t base = (uint64_t)blockIdx.x * kBlock * kPer + (uint64_t)threadIdx.x * kPer;
	uint64_t add = sums[blockIdx.x];
	for (int k = 0; k < kPer; ++k)
		if (base + k < n)
			out[base + k] += add;
}

// ===========================================================================
// host side
// ===========================================================================
static inline unsigned grid_for(uint64_t n) { return (unsigned)((n + kBlock - 1) / kBlock); }
static inline unsigned gridn_waves(uint64_t n) { return (unsigned)((n + kBlock / 64 - 1) / (kBlock / 64)); }

// The HIP runtime draws from (or reseeds) the C library's random generator
// while it initialises (the stream, memory and code-object set-up behind the
// process's first device scene).  A bake replays that generator's sequence
// for the AO rotation offsets, one draw per texel as the reference's randf()
// makes them (lighter.cpp:819, lighter_int.hpp:271), so the runtime is
// initialised once per process, on the first GPU request, with a private
// generator state switched in; the caller's sequence is left where it was.
namespace {
struct PrivateRandState {
	char buf[128];
	char* saved;
	PrivateRandState() { saved = initstate(0x4C54u, buf, sizeof(buf)); }
	~PrivateRandState() { setstate(saved); }
};
} // namespace

__global__ void k_warm(uint32_t* p)
{
	p[threadIdx.x] = threadIdx.x;
}

// A stream, device and pinned memory and one kernel launch: the runtime's
// one-time set-up, best effort (errors surface again in the calls that need
// the runtime).
static void init_runtime_once()
{
	hipStream_t s = nullptr;
	if (hipStreamCreate(&s) != hipSuccess)
		return;
	void* d = nullptr;
	if (hipMalloc(&d, 256) == hipSuccess) {
		k_warm<<<1, 64, 0, s>>>((uint32_t*)d);
		(void)hipStreamSynchronize(s);
		(void)hipFree(d);
	}
	void* h = nullptr;
	if (hipHostMalloc(&h, 256, hipHostMallocDefault) == hipSuccess)
		(void)hipHostFree(h);
	(void)hipStreamDestroy(s);
}

void require_gpu()
{
	static std::once_flag once;
	std::call_once(once, [] {
		PrivateRandState private_rand;
		int n = 0;
		if (hipGetDeviceCount(&n) == hipSuccess && n > 0)
			init_runtime_once();
		(void)hipGetLastError();
	});
	int n = 0;
	hipError_t e = hipGetDeviceCount(&n);
	if (e != hipSuccess || n == 0)
		throw std::runtime_error("liblighter_amd: no HIP device available (the bake stages run only on the GPU)");
}

std::string device_name()
{
	hipDeviceProp_t p;
	if (hipGetDeviceProperties(&p, 0) != hipSuccess)
		return "unknown";
	return std::string(p.name) + " " + p.gcnArchName;
}

template <class T> static T* dalloc(size_t n) { return (T*)device_alloc(n * sizeof(T)); }

template <class T> static void dfree(T*& p)
{
	if (p)
		(void)hipFree((void*)p);
	p = nullptr;
}

// a device array owned for one scope
template <class T> struct DevArray {
	T* p = nullptr;
	explicit DevArray(size_t n) : p(dalloc<T>(n)) {}
	DevArray(const DevArray&) = delete;
	DevArray& operator=(const DevArray&) = delete;
	~DevArray() { dfree(p); }
};

// Allocating and freeing large blocks costs more than the work on them: the
// links of a city's 440,003 patches took 31 ms in a new device scene and 60
// to 130 ms in later passes, which also freed the last one's blocks; 29 ms in
// all passes with the blocks kept.  A room's 32,768 patches: 14.7 -> 12.9 ms;
// 100,003 probe points: 2.44 -> 2.26 ms.
constexpr size_t kSpareMax = size_t(8) << 30;

// Every scene's spare blocks.  Blocks that a call holds are not among them,
// and hipFree waits for the work on those it frees, so any thread may give
// back another scene's.
static std::mutex g_spares_mu;
static std::set<SpareBlocks*>& spares()
{
	static std::set<SpareBlocks*>& all = *new std::set<SpareBlocks*>; // outlives any scene
	return all;
}

SpareBlocks::SpareBlocks()
{
	std::lock_guard<std::mutex> g(g_spares_mu);
	spares().insert(this);
}

SpareBlocks::~SpareBlocks()
{
	{
		std::lock_guard<std::mutex> g(g_spares_mu);
		spares().erase(this);
	}
	release();
}

void* device_alloc(size_t bytes)
{
	void* p = nullptr;
	bytes = std::max<size_t>(bytes, 1);
	if (hipMalloc(&p, bytes) == hipSuccess)
		return p;
	(void)hipGetLastError();
	{
		std::lock_guard<std::mutex> g(g_spares_mu);
		for (SpareBlocks* s : spares())
			s->release();
	}
	const hipError_t e = hipMalloc(&p, bytes);
	if (e != hipSuccess) {
		(void)hipGetLastError();
		throw std::runtime_error(std::string("HIP error ") + hipGetErrorString(e) + ": allocating " +
		                         std::to_string(bytes) + " bytes of device memory");
	}
	return p;
}

void* SpareBlocks::take(size_t bytes, size_t* cap)
{
	bytes = (std::max<size_t>(bytes, 1) + 4095) & ~size_t(4095);
	{
		std::lock_guard<std::mutex> g(mu_);
		auto it = spare_.lower_bound(bytes);
		if (it != spare_.end() && it->first / 2 <= bytes) {
			void* p = it->second;
			*cap = it->first;
			total_ -= it->first;
			spare_.erase(it);
			return p;
		}
	}
	void* p = device_alloc(bytes);
	*cap = bytes;
	return p;
}

void SpareBlocks::give(void* p, size_t cap)
{
	if (!p)
		return;
	{
		std::lock_guard<std::mutex> g(mu_);
		if (total_ + cap <= kSpareMax) {
			spare_.emplace(cap, p);
			total_ += cap;
			return;
		}
	}
	(void)hipFree(p);
}

void SpareBlocks::release()
{
	std::lock_guard<std::mutex> g(mu_);
	for (auto& e : spare_)
		(void)hipFree(e.second);
	spare_.clear();
	total_ = 0;
}

// ---------------------------------------------------------------------------
// Scratch of the allocation-free direct-light pass (run_direct_noalloc): the
// buffers run_direct allocates (per-item shading factor, the march list, the
// march count and control words, the traversal counters, the lights and their
// item ranges, the list of long marches) carved out of one file-scope device
// array.  Each GPU holds its own copy for the life of the process; every call
// on a GPU uses that copy, so calls that overlap on one GPU race.
// ---------------------------------------------------------------------------
constexpr size_t kNoAllocGateOff = 0;                                          // float per item
constexpr size_t kNoAllocListOff = kNoAllocGateOff + 4 * kNoAllocMaxItems;      // uint32 per item
constexpr size_t kNoAllocHeadOff = kNoAllocListOff + 4 * kNoAllocMaxItems;      // march count, control words, bad-item flag
constexpr size_t kNoAllocCntOff = kNoAllocHeadOff + 256;                        // traversal counters
constexpr size_t kNoAllocLightOff = kNoAllocCntOff + 256;                       // 64 lights
constexpr size_t kNoAllocOffOff = kNoAllocLightOff + 64 * sizeof(DevLight);     // 65 item offsets
constexpr size_t kNoAllocLongOff = kNoAllocOffOff + 512;                        // long marches
constexpr size_t kNoAllocBytes = kNoAllocLongOff + kLongCap * sizeof(LongMarch);
static_assert(kNumCounters * 8 <= 256, "counters fit their slot");
static_assert(kNoAllocLightOff % 256 == 0 && kNoAllocOffOff % 256 == 0, "aligned slots");

static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];

// Device address of `scratch` on the current GPU, looked up once per device
// (the array's name is only a host-side stand-in for it).
static void* noalloc_scratch()
{
	static std::mutex mu;
	static void* addr[kMaxDevices] = {};
	int dev = 0;
	HIPCHECK(hipGetDevice(&dev));
	if (dev < 0 || dev >= kMaxDevices)
		throw std::runtime_error("device ordinal beyond the supported " + std::to_string(kMaxDevices));
	std::lock_guard<std::mutex> g(mu);
	if (!addr[dev]) {
		PrivateRandState private_rand; // the lookup may set up the device's code object
		void* p = nullptr;
		const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
		if (e != hipSuccess || !p)
			throw std::runtime_error(std::string("hipGetSymbolAddress(scratch) failed: ") + hipGetErrorString(e));
		addr[dev] = p;
	}
	return addr[dev];
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t n, uint32_t v)
{
	for (uint32_t i = threadIdx.x; i < n; i += blockDim.x)
		p[i] = v;
}

// Sets *bad when an item names a light other than its segment's or a sample
// beyond the device's samples (the kernels index samples by the items).
__global__ void k_check_items(const uint32_t* __restrict__ items, uint32_t nitems, const uint32_t* __restrict__ off,
                              uint32_t nlights, uint32_t nsamples, uint32_t* bad)
{
	const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
	if (i >= nitems)
		return;
	const uint32_t code = items[i], l = code >> kSampleBits;
	if (l >= nlights || i < off[l] || i >= off[l + 1] || (code & kSampleMask) >= nsamples)
		atomicOr(bad, 1u);
}

DeviceScene::DeviceScene()
{
	require_gpu();
	hipStream_t s;
	HIPCHECK(hipStreamCreate(&s));
	stream_ = s;
	d_counters_ = dalloc<unsigned long long>(kNumCounters);
	d_mcount_ = dalloc<uint32_t>(1 + kMarchWords + 6); // + the samples' bounds
	d_scratch_ = noalloc_scratch();
	// the march's abort flag and progress word: pinned, coherent host memory
	// the kernel reads and writes while it runs
	HIPCHECK(hipHostMalloc((void**)&ctl_host_, 2 * sizeof(uint32_t), hipHostMallocMapped | hipHostMallocCoherent));
	ctl_host_[0] = ctl_host_[1] = 0u;
	HIPCHECK(hipHostGetDevicePointer((void**)&ctl_dev_, ctl_host_, 0));
}

// Blocks of the persistent march kernel: as many as can be resident at once.
// LDS stack levels of the traversal kernels (march, AO, link visibility): a
// leaf at depth d has at most d entries below it on the stack; at most
// kLdsLevels levels (18 KB per block) live in LDS
int DeviceScene::march_stack_depth() const { return std::min(kLdsLevels, 3 * bvh_depth_ + 1); }

size_t DeviceScene::march_lds_bytes() const { return (size_t)kBlock * march_stack_depth() * 6; }

unsigned DeviceScene::persistent_blocks()
{
	if (!persist_blocks_) { // calls that overlap may both find it so: they store the same value
		int dev = 0, per_cu = 0;
		hipDeviceProp_t p;
		HIPCHECK(hipGetDevice(&dev));
		HIPCHECK(hipGetDeviceProperties(&p, dev));
		HIPCHECK(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_march<false, DirectSrc>, kBlock,
		                                                      march_lds_bytes()));
		persist_blocks_ = (unsigned)std::max(1, per_cu) * (unsigned)p.multiProcessorCount;
	}
	return persist_blocks_;
}

// Launches the marches of src (nmarch of them) on the stream; next: the
// control words, zeroed on the stream but for an abort flag, and lng: the
// list of long marches, both the launch's own while it runs (neither is
// touched at up to Src::kWaveMax marches that cannot be stopped).  Up to
// Src::kWaveMax marches take a wave each from the start: that few leave a
// lane's marches waiting on the slowest walk of its wave, about 16 us a step
// (128,001 items of a room, 87,091 marches: 1,156 us with waves, 1,198 us on
// lanes; 8,001 items: 250 us and 1,100 us).  More keep the lanes busy, and
// only marches that would hold the launch up go to waves: while the list
// lasts, those longer than what a lane marches in all (kShareSteps steps for
// each march that falls to it), as beside shorter ones it has other work; at
// the end, those of kTailSteps steps.  A pass in ms, by the first limit (the
// rule's choice in brackets, "-" for none) and without hand-over:
//   marches                  64    96    128   192   -     none
//   terrain 1.29 M  [79]    7.36  7.41  7.65  7.49  7.75
//   city    1.60 M  [98]    8.43  8.09  8.16  8.11  8.08
//   city    2.07 M [126]   12.0  11.2  11.2  11.1  11.2   19.3
//   terrain 3.80 M [232]   18.4  17.1  16.7  16.4  16.5   19.9
// kTailSteps, with no first limit: city of 2.07 M 16 steps 15.0, 32 12.1, 64
// 11.3, 128 11.0; a room of 161,931 items 0.83 (32), 1.12 (64), 1.48 (128),
// 1.77 (none); 500,001 grazing queries in a terrain 7.2, 5.3, 5.5, 6.0.
// With counters every march stays on its lane, whose walk the counters are
// stated on.
constexpr uint32_t kShareSteps = 24, kTailSteps = 64;
template <class Src>
static void launch_marches(const View& V, const Src& src, uint32_t nmarch, uint32_t* next, LongMarch* lng,
                           unsigned long long* cnt, bool counting, int depth, size_t lds, unsigned blocks, uint32_t* ctl,
                           hipStream_t s)
{
	constexpr unsigned per = kBlock / 64;
	if (counting) {
		k_march<true><<<blocks, kBlock, lds, s>>>(V, src, nmarch, next, cnt, depth, ctl, UINT32_MAX, UINT32_MAX, nullptr);
	} else if (nmarch <= Src::kWaveMax) {
		k_march_wave<<<std::min((nmarch + per - 1) / per, blocks), kBlock, lds, s>>>(V, src, nmarch, nullptr, next, ctl,
		                                                                              depth);
	} else {
		const uint64_t share = (uint64_t)kShareSteps * nmarch / (blocks * kBlock);
		k_march<false><<<blocks, kBlock, lds, s>>>(V, src, nmarch, next, cnt, depth, ctl,
		                                           (uint32_t)std::max<uint64_t>(kTailSteps, share), kTailSteps, lng);
		HIPCHECK(hipGetLastError());
		k_march_wave<<<blocks, kBlock, lds, s>>>(V, src, 0, lng, next, ctl, depth);
	}
	HIPCHECK(hipGetLastError());
}

DeviceScene::~DeviceScene()
{
	free_all();
	dfree(d_counters_);
	dfree(d_mcount_);
	if (stream_)
		(void)hipStreamDestroy((hipStream_t)stream_);
	if (ctl_host_)
		(void)hipHostFree(ctl_host_);
}

void DeviceScene::free_all()
{
	nm_clear();
	dfree(d_cand_);
	dfree(d_clinked_);
	ncand_ = 0;
	dfree(d_nodes_);
	dfree(d_dtri_);
	dfree(d_rtri_);
	dfree(d_pos_);
	dfree(d_nrm_);
	dfree(d_skey_);
	dfree(d_ao_);
	dfree(d_side_);
	dfree(d_lm_);
	dfree(d_w_);
	dfree(d_vis_);
	dfree(d_items_);
	dfree(d_lights_);
	dfree(d_gate_);
	dfree(d_mlist_);
	dfree(rad.pos);
	dfree(rad.nrm);
	dfree(rad.rowptr);
	dfree(rad.rowptr64);
	dfree(rad.col);
	dfree(rad.val);
	dfree(rad.diffuse);
	dfree(rad.area);
	dfree(rad.total);
	dfree(rad.out);
	dfree(rad.in);
	dfree(rad.x);
}

static View make_view(void* nodes, void* dtri, void* rtri, size_t ntri, const float* lo, const float* hi,
                      const GridSpec& G, int32_t gbase, int32_t gfine)
{
	View v;
	v.gfine = gfine;
	for (int a = 0; a < 3; ++a) {
		v.glo[a] = G.lo[a];
		v.gn[a] = G.n[a];
	}
	v.ginv = 1.0f / G.g;
	v.gbase = gbase;
	v.nodes = (const WideNode*)nodes;
	v.dtri = (const DistTri*)dtri;
	v.rtri = (const RayTri*)rtri;
	v.has_tris = ntri > 0;
	for (int a = 0; a < 3; ++a) {
		float m = kPenumbraSize * 1.001f + 0.01f + 1e-4f * fmaxf(fabsf(lo[a]), fabsf(hi[a]));
		v.xlo[a] = lo[a] - m;
		v.xhi[a] = hi[a] + m;
	}
	return v;
}

// The triangles' precomputed forms in leaf order (make_dist_tri and
// make_ray_tri, the host's functions, on the device).
__global__ __launch_bounds__(kBlock) void k_tri_forms(const float* __restrict__ tris,
                                                      const uint32_t* __restrict__ order, size_t n,
                                                      DistTri* __restrict__ dt, RayTri* __restrict__ rt)
{
	const size_t i = (size_t)blockIdx.x * kBlock + threadIdx.x;
	if (i >= n)
		return;
	const float* p = tris + 9 * (size_t)order[i];
	const f3 a = ld3(p), c = ld3(p + 3), e = ld3(p + 6);
	dt[i] = make_dist_tri(a, c, e);
	rt[i] = make_ray_tri(a, c, e);
}

__device__ __forceinline__ bool box_meets(const float* lo, const float* hi, float lx, float ly, float lz, float hx,
                                          float hy, float hz)
{
	return lx <= hi[0] && hx >= lo[0] && ly <= hi[1] && hy >= lo[1] && lz <= hi[2] && hz >= lo[2];
}

// One lane per grid cell: its virtual node.  Starting from the root's
// children that meet the cell's region (the cell grown by pad), the largest
// inner node of the set is replaced by its children that meet the region
// while the set stays within four nodes; a node whose children would not
// fit stays.  Children that miss the region hold no triangle meeting it (a
// node's box holds its subtree's triangles; boxes with a NaN bound hold only
// triangles whose distances are NaN, which lower no minimum).
__global__ __launch_bounds__(256) void k_entry_cells(const WideNode* __restrict__ nodes, GridSpec G,
                                                     WideNode* __restrict__ cells)
{
	const uint32_t c = blockIdx.x * 256 + threadIdx.x;
	const uint32_t total = (uint32_t)G.n[0] * G.n[1] * G.n[2];
	if (c >= total)
		return;
	const int ix = (int)(c % (uint32_t)G.n[0]), iy = (int)((c / (uint32_t)G.n[0]) % (uint32_t)G.n[1]),
	          iz = (int)(c / ((uint32_t)G.n[0] * G.n[1]));
	const int ic[3] = {ix, iy, iz};
	float rlo[3], rhi[3];
	for (int a = 0; a < 3; ++a) {
		rlo[a] = G.lo[a] + (float)ic[a] * G.g - G.pad;
		rhi[a] = G.lo[a] + (float)(ic[a] + 1) * G.g + G.pad;
	}
	float blo[4][3], bhi[4][3];
	int32_t ref[4];
	bool open[4];
	int k = 0;
	{
		const WideNode& r = nodes[0];
		for (int j = 0; j < 4; ++j)
			if (box_meets(rlo, rhi, r.lox[j], r.loy[j], r.loz[j], r.hix[j], r.hiy[j], r.hiz[j])) {
				blo[k][0] = r.lox[j]; blo[k][1] = r.loy[j]; blo[k][2] = r.loz[j];
				bhi[k][0] = r.hix[j]; bhi[k][1] = r.hiy[j]; bhi[k][2] = r.hiz[j];
				ref[k] = r.child[j];
				open[k] = r.child[j] >= 0;
				++k;
			}
	}
	for (;;) {
		int e = -1;
		float area = -1.0f;
		for (int i = 0; i < k; ++i) {
			if (!open[i])
				continue;
			const float dx = bhi[i][0] - blo[i][0], dy = bhi[i][1] - blo[i][1], dz = bhi[i][2] - blo[i][2];
			const float s2 = dx * dy + dy * dz + dz * dx;
			if (e < 0 || s2 > area) {
				e = i;
				area = s2;
			}
		}
		if (e < 0)
			break;
		const WideNode& n = nodes[ref[e]];
		int take[4], m = 0;
		for (int j = 0; j < 4; ++j)
			if (box_meets(rlo, rhi, n.lox[j], n.loy[j], n.loz[j], n.hix[j], n.hiy[j], n.hiz[j]))
				take[m++] = j;
		if (k - 1 + m > 4) {
			open[e] = false;
			continue;
		}
		// entry e is replaced by the last entry, then the children appended
		--k;
		for (int a = 0; a < 3; ++a) {
			blo[e][a] = blo[k][a];
			bhi[e][a] = bhi[k][a];
		}
		ref[e] = ref[k];
		open[e] = open[k];
		for (int t = 0; t < m; ++t) {
			const int j = take[t];
			blo[k][0] = n.lox[j]; blo[k][1] = n.loy[j]; blo[k][2] = n.loz[j];
			bhi[k][0] = n.hix[j]; bhi[k][1] = n.hiy[j]; bhi[k][2] = n.hiz[j];
			ref[k] = n.child[j];
			open[k] = n.child[j] >= 0;
			++k;
		}
	}
	WideNode w;
	for (int j = 0; j < 4; ++j) {
		const bool use = j < k;
		w.lox[j] = use ? blo[j][0] : kFarBox;
		w.loy[j] = use ? blo[j][1] : kFarBox;
		w.loz[j] = use ? blo[j][2] : kFarBox;
		w.hix[j] = use ? bhi[j][0] : kFarBox;
		w.hiy[j] = use ? bhi[j][1] : kFarBox;
		w.hiz[j] = use ? bhi[j][2] : kFarBox;
		w.child[j] = use ? ref[j] : leaf_ref(0, 1);
		w.pad[j] = 0;
	}
	cells[c] = w;
}

// Sizes the entry grid over the scene box grown by kGridReach: cubic cells
// of at least kGridMinCell, at most kGridCells of them; false when the box
// is not finite.
static bool grid_spec(const float lo[3], const float hi[3], GridSpec& G)
{
	double e[3], vol = 1.0, mx = 0.0;
	for (int a = 0; a < 3; ++a) {
		if (!std::isfinite(lo[a]) || !std::isfinite(hi[a]) || !(hi[a] >= lo[a]))
			return false;
		G.lo[a] = (float)((double)lo[a] - kGridReach);
		e[a] = (double)hi[a] - lo[a] + 2.0 * kGridReach;
		vol *= e[a];
		mx = std::max(mx, std::max(fabs((double)lo[a]), fabs((double)hi[a])));
	}
	double g = std::max((double)kGridMinCell, std::cbrt(vol / kGridCells));
	for (int it = 0; it < 64; ++it) {
		double cells = 1.0;
		for (int a = 0; a < 3; ++a)
			cells *= std::max(1.0, std::ceil(e[a] / g));
		if (cells <= kGridCells)
			break;
		g *= 1.05;
	}
	for (int a = 0; a < 3; ++a)
		G.n[a] = (int)std::max(1.0, std::ceil(e[a] / g));
	if ((double)G.n[0] * G.n[1] * G.n[2] > kGridCells)
		return false;
	G.g = (float)g;
	// rounding of the cell index and of the region's bounds: a query point
	// lies within 1e-3 of a cell plus 1e-5 of the coordinates' magnitude of
	// its cell; distances within the same relative bound of the radius
	G.pad = kGridReach * (1.0f + 1e-4f) + 1e-3f * G.g + 1e-5f * (float)mx + 1e-3f;
	return true;
}

void DeviceScene::set_triangles(const float* tris, size_t ntri)
{
	dfree(d_nodes_);
	dfree(d_dtri_);
	dfree(d_rtri_);
	ntri_ = ntri;
	times.bvh_ms = 0;
	if (ntri == 0) {
		nnodes_ = 0;
		return;
	}
	if (ntri >= (1u << 27))
		throw std::runtime_error("too many triangles for the leaf encoding");
	hipStream_t s = (hipStream_t)stream_;
	// triangles up, the tree built on the device (the host build's tree,
	// bvh_gpu.hip), the triangle forms made there in leaf order
	DevArray<float> d_tris(9 * ntri);
	DevArray<uint32_t> d_order(ntri);
	HIPCHECK(hipMemcpyAsync(d_tris.p, tris, 36 * ntri, hipMemcpyHostToDevice, s));
	double kms = 0;
	BvhBuild b = build_bvh_gpu(d_tris.p, ntri, d_order.p, stream_, &kms);
	times.bvh_ms = kms;
	if (3 * b.depth + 1 > kStackSize)
		throw std::runtime_error("BVH deeper than the traversal stack");
	bvh_depth_ = b.depth;
	persist_blocks_ = 0; // the march kernel's LDS stack follows the depth
	nnodes_ = b.nodes.size();
	lo_[0] = b.lo.x; lo_[1] = b.lo.y; lo_[2] = b.lo.z;
	hi_[0] = b.hi.x; hi_[1] = b.hi.y; hi_[2] = b.hi.z;
	GridSpec G{};
	const bool grid = grid_spec(lo_, hi_, G) && nnodes_ + (size_t)G.n[0] * G.n[1] * G.n[2] < (size_t)INT32_MAX;
	const size_t ncells = grid ? (size_t)G.n[0] * G.n[1] * G.n[2] : 0;
	const bool fine = grid && nnodes_ + 2 * ncells < (size_t)INT32_MAX;
	d_nodes_ = dalloc<WideNode>(nnodes_ + (fine ? 2 : 1) * ncells);
	d_dtri_ = dalloc<DistTri>(ntri);
	d_rtri_ = dalloc<RayTri>(ntri);
	HIPCHECK(hipMemcpyAsync(d_nodes_, b.nodes.data(), sizeof(WideNode) * nnodes_, hipMemcpyHostToDevice, s));
	k_tri_forms<<<grid_for(ntri), kBlock, 0, s>>>(d_tris.p, d_order.p, ntri, (DistTri*)d_dtri_, (RayTri*)d_rtri_);
	HIPCHECK(hipGetLastError());
	grid_ = G;
	grid_base_ = 0;
	if (grid) {
		k_entry_cells<<<(unsigned)((ncells + 255) / 256), 256, 0, s>>>((const WideNode*)d_nodes_, G,
		                                                               (WideNode*)d_nodes_ + nnodes_);
		HIPCHECK(hipGetLastError());
		grid_base_ = (int32_t)nnodes_;
	}
	grid_fine_ = 0;
	if (fine) {
		GridSpec F = G;
		F.pad = G.pad - kGridReach * (1.0f + 1e-4f) + kGridFineReach * (1.0f + 1e-4f);
		k_entry_cells<<<(unsigned)((ncells + 255) / 256), 256, 0, s>>>((const WideNode*)d_nodes_, F,
		                                                               (WideNode*)d_nodes_ + nnodes_ + ncells);
		HIPCHECK(hipGetLastError());
		grid_fine_ = (int32_t)(nnodes_ + ncells);
	}
	HIPCHECK(hipStreamSynchronize(s));
}

// Order-preserving key of a float that is not NaN, and back.
__host__ __device__ __forceinline__ uint32_t order_key(float f)
{
	uint32_t u;
	memcpy(&u, &f, 4);
	return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__host__ __device__ __forceinline__ float order_value(uint32_t k)
{
	const uint32_t u = (k & 0x80000000u) ? (k & 0x7fffffffu) : ~k;
	float f;
	memcpy(&f, &u, 4);
	return f;
}

// Bounds of n positions as keys: minima into b[0..2], maxima into b[3..5]
// (NaN coordinates take no part).
__global__ __launch_bounds__(kBlock) void k_sample_bounds(const float* __restrict__ pos, uint32_t n,
                                                          uint32_t* __restrict__ b)
{
	float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
	for (uint32_t i = blockIdx.x * kBlock + threadIdx.x; i < n; i += gridDim.x * kBlock)
		for (int a = 0; a < 3; ++a) {
			const float p = pos[3 * (size_t)i + a];
			lo[a] = fminf(lo[a], p);
			hi[a] = fmaxf(hi[a], p);
		}
	for (int o = 32; o > 0; o >>= 1)
		for (int a = 0; a < 3; ++a) {
			lo[a] = fminf(lo[a], __shfl_xor(lo[a], o));
			hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], o));
		}
	if ((threadIdx.x & 63) == 0)
		for (int a = 0; a < 3; ++a) {
			atomicMin(b + a, order_key(lo[a]));
			atomicMax(b + 3 + a, order_key(hi[a]));
		}
}

__global__ void k_fill_bounds(uint32_t* b) { b[threadIdx.x] = threadIdx.x < 3 ? 0xffffffffu : 0u; }

// 30-bit Morton code of each texel position over the samples' box, in cubic
// cells: the march order.  A pass over the positions each, at the copies'
// end (computed on the host and with all arrays allocated anew, setting
// 700,001 samples and 64 occlusion rays for each took 6.9 ms; 4.25 so).
__global__ __launch_bounds__(kBlock) void k_sample_keys(const float* __restrict__ pos, uint32_t n,
                                                        const uint32_t* __restrict__ b, uint32_t* __restrict__ key)
{
	const uint32_t i = blockIdx.x * kBlock + threadIdx.x;
	if (i >= n)
		return;
	float mn[3], ext = -INFINITY;
	for (int a = 0; a < 3; ++a) {
		mn[a] = order_value(b[a]);
		ext = fmaxf(ext, order_value(b[3 + a]) - mn[a]);
	}
	const float q = ext > 0.0f ? 1023.0f / ext : 0.0f;
	uint32_t c = 0;
	for (int a = 0; a < 3; ++a) {
		const float f = (pos[3 * (size_t)i + a] - mn[a]) * q;
		uint32_t v = f > 0.0f ? (uint32_t)fminf(f, 1023.0f) : 0u;
		v = (v | (v << 16)) & 0x030000ffu;
		v = (v | (v << 8)) & 0x0300f00fu;
		v = (v | (v << 4)) & 0x030c30c3u;
		v = (v | (v << 2)) & 0x09249249u;
		c |= v << a;
	}
	key[i] = c;
}

void DeviceScene::set_samples(const float* pos, const float* nrm, size_t n)
{
	if (n > kSampleMask)
		throw std::runtime_error("too many samples for the work-item encoding");
	hipStream_t s = (hipStream_t)stream_;
	nsamples_ = 0;
	// the arrays are kept for sample sets of much the same size
	if (!d_pos_ || n > samples_cap_ || n < samples_cap_ / 4) {
		dfree(d_pos_);
		dfree(d_nrm_);
		dfree(d_lm_);
		dfree(d_skey_);
		samples_cap_ = 0;
		d_pos_ = dalloc<float>(3 * n);
		d_nrm_ = dalloc<float>(3 * n);
		d_lm_ = dalloc<float>(3 * n);
		d_skey_ = dalloc<uint32_t>(n);
		samples_cap_ = n;
	}
	if (n) {
		HIPCHECK(hipMemcpyAsync(d_pos_, pos, 12 * n, hipMemcpyHostToDevice, s));
		HIPCHECK(hipMemcpyAsync(d_nrm_, nrm, 12 * n, hipMemcpyHostToDevice, s));
		HIPCHECK(hipMemsetAsync(d_lm_, 0, 12 * n, s));
		uint32_t* b = d_mcount_ + 1 + kMarchWords;
		k_fill_bounds<<<1, 6, 0, s>>>(b);
		k_sample_bounds<<<std::min(grid_for(n), 1024u), kBlock, 0, s>>>(d_pos_, (uint32_t)n, b);
		k_sample_keys<<<grid_for(n), kBlock, 0, s>>>(d_pos_, (uint32_t)n, b, d_skey_);
		HIPCHECK(hipGetLastError());
	}
	HIPCHECK(hipStreamSynchronize(s));
	nsamples_ = n;
}

void DeviceScene::set_lightmap(const float* rgb)
{
	if (nsamples_)
		HIPCHECK(hipMemcpy(d_lm_, rgb, 12 * nsamples_, hipMemcpyHostToDevice));
}

void DeviceScene::get_lightmap(float* rgb) const
{
	if (nsamples_)
		HIPCHECK(hipMemcpy(rgb, d_lm_, 12 * nsamples_, hipMemcpyDeviceToHost));
}

struct EventTimer {
	hipEvent_t a, b;
	hipStream_t s;
	explicit EventTimer(hipStream_t st) : s(st)
	{
		HIPCHECK(hipEventCreate(&a));
		HIPCHECK(hipEventCreate(&b));
		HIPCHECK(hipEventRecord(a, s));
	}
	double stop()
	{
		HIPCHECK(hipEventRecord(b, s));
		HIPCHECK(hipEventSynchronize(b));
		float ms = 0;
		HIPCHECK(hipEventElapsedTime(&ms, a, b));
		return ms;
	}
	~EventTimer()
	{
		(void)hipEventDestroy(a);
		(void)hipEventDestroy(b);
	}
};

void DeviceScene::set_direct_work(const std::vector<DevLight>& lights, const std::vector<uint32_t>& items,
                                  const std::vector<uint32_t>& light_off, bool keep_weights)
{
	hipStream_t s = (hipStream_t)stream_;
	if (lights.size() > 64)
		throw std::runtime_error("direct_light: at most 64 lights per batch");
	if (light_off.size() != lights.size() + 1 || light_off.back() != items.size() || light_off[0] != 0)
		throw std::runtime_error("direct_light: light offsets do not match the work items");
	// every item must name its segment's light and a sample on the device
	for (size_t l = 0; l < lights.size(); ++l) {
		if (light_off[l + 1] < light_off[l])
			throw std::runtime_error("direct_light: light offsets must not decrease");
		for (uint32_t k = light_off[l]; k < light_off[l + 1]; ++k)
			if ((items[k] >> kSampleBits) != l || (items[k] & kSampleMask) >= nsamples_)
				throw std::runtime_error("direct_light: work item " + std::to_string(k) +
				                         " names another light or a sample beyond the device's samples");
	}
	dfree(d_w_);
	dfree(d_vis_);
	dfree(d_items_);
	dfree(d_lights_);
	dfree(d_gate_);
	dfree(d_mlist_);
	nitems_ = items.size();
	d_w_ = dalloc<float>(nitems_);
	if (keep_weights)
		d_vis_ = dalloc<float>(nitems_);
	d_gate_ = dalloc<float>(nitems_);
	d_mlist_ = dalloc<uint32_t>(nitems_);
	d_items_ = dalloc<uint32_t>(nitems_);
	d_lights_ = dalloc<DevLight>(lights.size());
	HIPCHECK(hipMemcpyAsync(d_items_, items.data(), 4 * nitems_, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_lights_, lights.data(), sizeof(DevLight) * lights.size(), hipMemcpyHostToDevice, s));
	HIPCHECK(hipStreamSynchronize(s));
	h_lights_ = lights;
	h_light_off_ = light_off;
}

// While the march kernel runs: progress to keep_going (the fraction of the
// march list claimed) every millisecond, and the abort flag raised when it
// returns false.  True when the march was aborted (also when the device's
// abort request was set before the launch: the kernel then leaves at once).
bool DeviceScene::wait_march(uint32_t nmarch, const std::function<bool(float)>& keep_going)
{
	if (abort_requested_)
		return true;
	if (!keep_going)
		return false;
	hipStream_t s = (hipStream_t)stream_;
	volatile uint32_t* ctl = ctl_host_;
	bool stop = false;
	float done = 0.0f; // posts of different waves may arrive in another order
	for (;;) {
		const hipError_t e = hipStreamQuery(s);
		if (e == hipSuccess)
			break;
		if (e != hipErrorNotReady)
			HIPCHECK(e);
		if (!stop) {
			done = std::max(done, std::min(1.0f, (float)ctl[1] / (float)nmarch));
			if (!keep_going(done)) {
				stop = true;
				ctl[0] = 1u;
			}
		}
		std::this_thread::sleep_for(std::chrono::milliseconds(1));
	}
	return stop;
}

bool DeviceScene::run_direct(const std::function<bool(float)>& keep_going)
{
	hipStream_t s = (hipStream_t)stream_;
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	bool aborted = false;
	ctl_host_[0] = 0u; // read by the kernel after the launch below
	ctl_host_[1] = 0u;
	HIPCHECK(hipMemsetAsync(d_counters_, 0, kNumCounters * sizeof(unsigned long long), s));
	EventTimer all(s);
	if (nitems_) {
		HIPCHECK(hipMemsetAsync(d_mcount_, 0, (1 + kMarchWords) * sizeof(uint32_t), s));
		// the device abort flag starts raised under request_abort: every wave
		// then leaves at its first claim, before any march
		if (abort_requested_)
			HIPCHECK(hipMemsetAsync(d_mcount_ + 1 + kMarchAbort, 1, sizeof(uint32_t), s));
		k_direct_gate<<<(unsigned)((nitems_ + kGateRounds * kBlock - 1) / (kGateRounds * kBlock)), kBlock, 0, s>>>(
		    d_pos_, d_nrm_, d_lights_, d_items_, (uint32_t)nitems_, d_gate_, d_w_, d_vis_, d_mlist_, d_mcount_, d_skey_);
		HIPCHECK(hipGetLastError());
		uint32_t nmarch = 0;
		HIPCHECK(hipMemcpyAsync(&nmarch, d_mcount_, 4, hipMemcpyDeviceToHost, s));
		HIPCHECK(hipStreamSynchronize(s));
		nmarch_ = nmarch;
		Scratch<LongMarch> lng(spare_, nmarch > DirectSrc::kWaveMax ? kLongCap : 0);
		EventTimer tm(s);
		if (nmarch) {
			// the abort and progress path only for runs that can be stopped
			// (it costs up to 2 % of the march on the city block)
			uint32_t* ctl = (keep_going || abort_requested_) ? ctl_dev_ : nullptr;
			const DirectSrc src{d_pos_, d_nrm_, d_lights_, d_items_, d_mlist_, d_gate_, d_w_, d_vis_};
			launch_marches(V, src, nmarch, d_mcount_ + 1, lng.p, d_counters_, count_queries, march_stack_depth(),
			               march_lds_bytes(), persistent_blocks(), ctl, s);
			aborted = wait_march(nmarch, keep_going);
		}
		times.direct_march_ms = tm.stop();
	}
	if (aborted) { // the lightmap keeps its colours
		times.direct_ms = all.stop();
		read_counters();
		return false;
	}
	for (size_t l = 0; l < h_lights_.size(); ++l) {
		uint32_t b = h_light_off_[l], e = h_light_off_[l + 1];
		if (e > b) {
			k_accumulate<<<grid_for(e - b), kBlock, 0, s>>>(d_items_, d_w_, b, e, h_lights_[l].color[0],
			                                                h_lights_[l].color[1], h_lights_[l].color[2], d_lm_);
			HIPCHECK(hipGetLastError());
		}
	}
	times.direct_ms = all.stop();
	read_counters();
	return true;
}

// [p, p + bytes) must lie inside one device allocation of the current GPU.
static void check_device_range(const void* p, size_t bytes, const char* what)
{
	hipDeviceptr_t base = nullptr;
	size_t size = 0;
	const hipError_t e = hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p);
	if (e != hipSuccess)
		(void)hipGetLastError(); // the failed lookup must not surface as a later launch's error
	if (e != hipSuccess || !base || (const char*)p + bytes > (const char*)base + size)
		throw std::runtime_error(std::string("direct_light_noalloc: ") + what +
		                         " is not a device buffer of the current GPU large enough for the work items");
}

void DeviceScene::run_direct_noalloc(const DevLight* lights, int nlights, const uint32_t* d_items, size_t nitems,
                                     const uint32_t* light_off, float* d_w, float* d_vis)
{
	if (nitems > kNoAllocMaxItems)
		throw std::runtime_error("direct_light_noalloc: " + std::to_string(nitems) +
		                         " work items exceed the scratch's maximum of " + std::to_string(kNoAllocMaxItems));
	if (nlights < 0 || nlights > 64)
		throw std::runtime_error("direct_light_noalloc: 0..64 lights per call");
	if (light_off[0] != 0 || light_off[nlights] != nitems)
		throw std::runtime_error("direct_light_noalloc: light offsets do not match the work items");
	for (int l = 0; l < nlights; ++l)
		if (light_off[l + 1] < light_off[l])
			throw std::runtime_error("direct_light_noalloc: light offsets must not decrease");
	if (nitems == 0)
		return;
	if (!nsamples_)
		throw std::runtime_error("direct_light_noalloc: the device holds no samples");
	check_device_range(d_items, 4 * nitems, "the work-item array");
	check_device_range(d_w, 4 * nitems, "the weight array");
	if (d_vis)
		check_device_range(d_vis, 4 * nitems, "the shadow-factor array");
	hipStream_t s = (hipStream_t)stream_;
	char* sc = (char*)d_scratch_;
	float* gate = (float*)(sc + kNoAllocGateOff);
	uint32_t* mlist = (uint32_t*)(sc + kNoAllocListOff);
	uint32_t* head = (uint32_t*)(sc + kNoAllocHeadOff); // [0] march count, [1..] the march's words, [kBad] bad item
	constexpr int kBad = 1 + kMarchWords;
	unsigned long long* cnt = (unsigned long long*)(sc + kNoAllocCntOff);
	DevLight* dl = (DevLight*)(sc + kNoAllocLightOff);
	uint32_t* doff = (uint32_t*)(sc + kNoAllocOffOff);
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	if (nlights)
		HIPCHECK(hipMemcpyAsync(dl, lights, sizeof(DevLight) * nlights, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(doff, light_off, 4 * (size_t)(nlights + 1), hipMemcpyHostToDevice, s));
	// counters and flags start at zero (the array keeps the last call's contents)
	k_fill_u32<<<1, 64, 0, s>>>(head, 2 + kMarchWords, 0u);
	k_fill_u32<<<1, 64, 0, s>>>((uint32_t*)cnt, 2 * kNumCounters, 0u);
	k_check_items<<<grid_for(nitems), kBlock, 0, s>>>(d_items, (uint32_t)nitems, doff, (uint32_t)nlights,
	                                                  (uint32_t)nsamples_, head + kBad);
	HIPCHECK(hipGetLastError());
	uint32_t h[kBad + 1] = {};
	HIPCHECK(hipMemcpyAsync(h, head, sizeof(h), hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	if (h[kBad])
		throw std::runtime_error("direct_light_noalloc: a work item names another light or a sample beyond the "
		                         "device's samples");
	k_direct_gate<<<(unsigned)((nitems + kGateRounds * kBlock - 1) / (kGateRounds * kBlock)), kBlock, 0, s>>>(
	    d_pos_, d_nrm_, dl, d_items, (uint32_t)nitems, gate, d_w, d_vis, mlist, head, d_skey_);
	HIPCHECK(hipGetLastError());
	HIPCHECK(hipMemcpyAsync(h, head, 4, hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	const uint32_t nmarch = h[0];
	if (nmarch) {
		const DirectSrc src{d_pos_, d_nrm_, dl, d_items, mlist, gate, d_w, d_vis};
		launch_marches(V, src, nmarch, head + 1, (LongMarch*)(sc + kNoAllocLongOff), cnt, false, march_stack_depth(), march_lds_bytes(),
		               persistent_blocks(), nullptr, s);
	}
	for (int l = 0; l < nlights; ++l) {
		const uint32_t b = light_off[l], e = light_off[l + 1];
		if (e > b) {
			k_accumulate<<<grid_for(e - b), kBlock, 0, s>>>(d_items, d_w, b, e, lights[l].color[0], lights[l].color[1],
			                                                lights[l].color[2], d_lm_);
			HIPCHECK(hipGetLastError());
		}
	}
	HIPCHECK(hipStreamSynchronize(s));
}

void DeviceScene::reference_counts(const float* tris, size_t ntri, uint64_t out[5])
{
	for (int i = 0; i < 5; ++i)
		out[i] = 0;
	if (ntri != ntri_)
		throw std::runtime_error("reference_counts: the triangles must be those of the device scene");
	if (!d_vis_)
		throw std::runtime_error("reference_counts: run the direct light with kept weights first");
	if (nmarch_ == 0 || ntri == 0)
		return;
	BinaryBvh b = build_bvh_binary(tris, ntri, 16, 4);
	if (b.depth > kCanonStack)
		throw std::runtime_error("reference_counts: binary tree deeper than the counting stack");
	std::vector<DistTri> dt(ntri);
	for (size_t i = 0; i < ntri; ++i) {
		const float* p = tris + 9 * (size_t)b.order[i];
		dt[i] = make_dist_tri(ld3(p), ld3(p + 3), ld3(p + 6));
	}
	BvhNode* d_nodes = dalloc<BvhNode>(b.nodes.size());
	DistTri* d_dt = dalloc<DistTri>(ntri);
	unsigned long long* d_out = dalloc<unsigned long long>(4);
	struct Free {
		BvhNode*& a;
		DistTri*& b;
		unsigned long long*& c;
		~Free()
		{
			dfree(a);
			dfree(b);
			dfree(c);
		}
	} fr{d_nodes, d_dt, d_out};
	hipStream_t s = (hipStream_t)stream_;
	HIPCHECK(hipMemcpyAsync(d_nodes, b.nodes.data(), b.nodes.size() * sizeof(BvhNode), hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_dt, dt.data(), ntri * sizeof(DistTri), hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemsetAsync(d_out, 0, 4 * sizeof(unsigned long long), s));
	CanonView C;
	C.nodes = d_nodes;
	C.dtri = d_dt;
	canon_root_box(b, C.lo, C.hi);
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	k_march_canon<<<grid_for(nmarch_), kBlock, 0, s>>>(C, V, d_pos_, d_nrm_, d_lights_, d_items_, d_mlist_, nmarch_,
	                                                   d_vis_, d_out);
	HIPCHECK(hipGetLastError());
	unsigned long long h[4];
	HIPCHECK(hipMemcpyAsync(h, d_out, sizeof(h), hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	for (int i = 0; i < 4; ++i)
		out[i] = h[i];
	out[4] = nmarch_;
}

void DeviceScene::reference_counts_ao(const float* tris, size_t ntri, const float* randoff, int num_samples,
                                      float distance, float multiplier, float falloff, uint64_t out[5])
{
	for (int i = 0; i < 5; ++i)
		out[i] = 0;
	if (ntri != ntri_)
		throw std::runtime_error("reference_counts_ao: the triangles must be those of the device scene");
	if (nsamples_ == 0 || num_samples <= 0 || ntri == 0)
		return;
	BinaryBvh b = build_bvh_binary(tris, ntri, 16, 4);
	if (b.depth > kCanonStack)
		throw std::runtime_error("reference_counts_ao: binary tree deeper than the counting stack");
	std::vector<RayTri> rt(ntri);
	for (size_t i = 0; i < ntri; ++i) {
		const float* p = tris + 9 * (size_t)b.order[i];
		rt[i] = make_ray_tri(ld3(p), ld3(p + 3), ld3(p + 6));
	}
	std::vector<float2> side(num_samples);
	for (int i = 0; i < num_samples; ++i) {
		float q = (i + 0.5f) / num_samples;
		float cs = sqrtf(q);
		side[i] = make_float2(cs, sinf(acosf(cs)));
	}
	hipStream_t s = (hipStream_t)stream_;
	BvhNode* d_nodes = dalloc<BvhNode>(b.nodes.size());
	RayTri* d_rt = dalloc<RayTri>(ntri);
	float2* d_side = dalloc<float2>(num_samples);
	float* d_ro = dalloc<float>(nsamples_);
	float* d_fp = dalloc<float>(nsamples_);
	float* d_fc = dalloc<float>(nsamples_);
	float* d_lm_keep = dalloc<float>(3 * nsamples_);
	unsigned long long* d_out = dalloc<unsigned long long>(4);
	struct Free {
		std::vector<void*> p;
		~Free()
		{
			for (void* q : p)
				if (q)
					(void)hipFree(q);
		}
	} fr{{d_nodes, d_rt, d_side, d_ro, d_fp, d_fc, d_lm_keep, d_out}};
	HIPCHECK(hipMemcpyAsync(d_nodes, b.nodes.data(), b.nodes.size() * sizeof(BvhNode), hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_rt, rt.data(), ntri * sizeof(RayTri), hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_side, side.data(), sizeof(float2) * num_samples, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_ro, randoff, 4 * nsamples_, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemsetAsync(d_out, 0, 4 * sizeof(unsigned long long), s));
	// the product's factors, with the lightmap put back afterwards
	HIPCHECK(hipMemcpyAsync(d_lm_keep, d_lm_, 12 * nsamples_, hipMemcpyDeviceToDevice, s));
	const float black[3] = {0, 0, 0};
	const bool counting = count_queries;
	count_queries = false;
	const StageTimes keep_times = times;
	ambient_occlusion(randoff, num_samples, distance, multiplier, falloff, 0.0f, black, d_fp);
	count_queries = counting;
	times = keep_times;
	HIPCHECK(hipMemcpyAsync(d_lm_, d_lm_keep, 12 * nsamples_, hipMemcpyDeviceToDevice, s));
	AOParams P;
	P.n = num_samples;
	P.distance = distance;
	P.multiplier = multiplier;
	P.falloff = falloff;
	P.effect = 0.0f;
	P.color[0] = P.color[1] = P.color[2] = 0.0f;
	CanonView C;
	C.nodes = d_nodes;
	C.dtri = nullptr;
	canon_root_box(b, C.lo, C.hi);
	const unsigned grid = (unsigned)((nsamples_ + kBlock / 64 - 1) / (kBlock / 64));
	k_ao_canon<<<grid, kBlock, 0, s>>>(C, d_rt, d_pos_, d_nrm_, d_ro, d_side, P, (uint32_t)nsamples_, d_fc, d_out);
	HIPCHECK(hipGetLastError());
	unsigned long long h[4];
	HIPCHECK(hipMemcpyAsync(h, d_out, sizeof(h), hipMemcpyDeviceToHost, s));
	std::vector<float> fp(nsamples_), fc(nsamples_);
	HIPCHECK(hipMemcpyAsync(fp.data(), d_fp, 4 * nsamples_, hipMemcpyDeviceToHost, s));
	HIPCHECK(hipMemcpyAsync(fc.data(), d_fc, 4 * nsamples_, hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	uint64_t differ = 0;
	for (size_t i = 0; i < nsamples_; ++i)
		differ += memcmp(&fp[i], &fc[i], 4) != 0;
	out[0] = h[0];
	out[1] = h[1];
	out[2] = h[2];
	out[3] = differ;
	out[4] = nsamples_;
}

void DeviceScene::reference_counts_links(const float* tris, size_t ntri, uint64_t out[5])
{
	for (int i = 0; i < 5; ++i)
		out[i] = 0;
	if (ntri != ntri_)
		throw std::runtime_error("reference_counts_links: the triangles must be those of the device scene");
	if (!d_cand_)
		throw std::runtime_error("reference_counts_links: run the link search with counting on first");
	if (ncand_ == 0 || ntri == 0)
		return;
	BinaryBvh b = build_bvh_binary(tris, ntri, 16, 4);
	if (b.depth > kCanonStack)
		throw std::runtime_error("reference_counts_links: binary tree deeper than the counting stack");
	std::vector<RayTri> rt(ntri);
	for (size_t i = 0; i < ntri; ++i) {
		const float* p = tris + 9 * (size_t)b.order[i];
		rt[i] = make_ray_tri(ld3(p), ld3(p + 3), ld3(p + 6));
	}
	hipStream_t s = (hipStream_t)stream_;
	BvhNode* d_nodes = dalloc<BvhNode>(b.nodes.size());
	RayTri* d_rt = dalloc<RayTri>(ntri);
	unsigned long long* d_out = dalloc<unsigned long long>(3);
	struct Free {
		std::vector<void*> p;
		~Free()
		{
			for (void* q : p)
				if (q)
					(void)hipFree(q);
		}
	} fr{{d_nodes, d_rt, d_out}};
	HIPCHECK(hipMemcpyAsync(d_nodes, b.nodes.data(), b.nodes.size() * sizeof(BvhNode), hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_rt, rt.data(), ntri * sizeof(RayTri), hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemsetAsync(d_out, 0, 3 * sizeof(unsigned long long), s));
	CanonView C;
	C.nodes = d_nodes;
	C.dtri = nullptr;
	canon_root_box(b, C.lo, C.hi);
	k_link_canon<<<grid_for(ncand_), kBlock, 0, s>>>(C, d_rt, rad.pos, (const uint2*)d_cand_, ncand_,
	                                                 (const uint8_t*)d_clinked_, d_out);
	HIPCHECK(hipGetLastError());
	unsigned long long h[3];
	HIPCHECK(hipMemcpyAsync(h, d_out, sizeof(h), hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	out[0] = h[0];
	out[1] = h[1];
	out[2] = ncand_;
	out[3] = h[2];
	out[4] = rad.nnz / 2;
}

void DeviceScene::read_counters()
{
	if (!count_queries)
		return;
	unsigned long long c[kNumCounters];
	HIPCHECK(hipMemcpy(c, d_counters_, sizeof(c), hipMemcpyDeviceToHost));
	counters.nodes = c[0];
	counters.tris = c[1];
	counters.steps = c[2];
	counters.queries = c[3];
	counters.marches = c[4];
	counters.pretests = c[5];
}

bool DeviceScene::direct_light(const std::vector<DevLight>& lights, const std::vector<uint32_t>& items,
                               const std::vector<uint32_t>& light_off, bool keep_weights,
                               const std::function<bool(float)>& keep_going)
{
	set_direct_work(lights, items, light_off, keep_weights);
	return run_direct(keep_going);
}

// ---------------------------------------------------------------------------
// Normal-map data on the GPU (lighter.cpp:505-513, 959-1030): one lane per
// sample walks the kept lights in order twice, as the host restatement
// walks its contribution list: first the sum of the scaled sample normal
// and the contributions and their count, then, against the mean, the
// min-dot product (normals.h serves both sides).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_nm_data(const float* __restrict__ pos, const float* __restrict__ nrm,
                                                    uint32_t n, const uint32_t* __restrict__ inst_off, int ninst,
                                                    const DevLight* __restrict__ lights, int nl,
                                                    const int32_t* __restrict__ first,
                                                    const float* const* __restrict__ visp, float ab,
                                                    float* __restrict__ out)
{
	const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
	if (s >= n)
		return;
	int lo = 0, hi = ninst - 1; // the sample's instance: last with inst_off <= s
	while (lo < hi) {
		const int mid = (lo + hi + 1) >> 1;
		if (inst_off[mid] <= s)
			lo = mid;
		else
			hi = mid - 1;
	}
	const int inst = lo;
	const uint32_t within = s - inst_off[inst];
	const f3 SP = ld3(pos + 3 * (size_t)s), SN = ld3(nrm + 3 * (size_t)s);
	f3 sum = SN * ab;
	int count = 1;
	for (int l = 0; l < nl; ++l) {
		const int32_t f = first[(size_t)l * ninst + inst];
		f3 c;
		if (f >= 0 && nm_contrib(lights[l], SP, SN, visp[l][(uint32_t)f + within], &c)) {
			sum += c;
			++count;
		}
	}
	const f3 mean = sum / (float)count;
	float md = 1.0f;
	for (int l = 0; l < nl; ++l) {
		const int32_t f = first[(size_t)l * ninst + inst];
		f3 c;
		if (f >= 0 && nm_contrib(lights[l], SP, SN, visp[l][(uint32_t)f + within], &c))
			md *= nm_mindot_factor(mean, c);
	}
	const f3 N = normalized(mean);
	out[4 * (size_t)s + 0] = N.x;
	out[4 * (size_t)s + 1] = N.y;
	out[4 * (size_t)s + 2] = N.z;
	out[4 * (size_t)s + 3] = md;
}

void DeviceScene::nm_clear()
{
	for (float*& p : nm_vis_)
		dfree(p);
	nm_vis_.clear();
	nm_lights_.clear();
	nm_first_.clear();
	nm_light_batch_.clear();
	nm_batch_items_.clear();
	nm_ninst_ = 0;
}

void DeviceScene::nm_keep_batch(const std::vector<DevLight>& lights, const std::vector<int32_t>& first_item,
                                size_t ninst)
{
	if (!d_vis_)
		throw std::runtime_error("nm_keep_batch: the direct-light run kept no shadow factors");
	if (first_item.size() != lights.size() * ninst || (nm_ninst_ && nm_ninst_ != ninst))
		throw std::runtime_error("nm_keep_batch: item table does not match the lights and instances");
	for (int32_t f : first_item)
		if (f >= 0 && (size_t)f >= nitems_)
			throw std::runtime_error("nm_keep_batch: item offset beyond the run's items");
	nm_ninst_ = ninst;
	float* v = dalloc<float>(nitems_);
	hipStream_t s = (hipStream_t)stream_;
	HIPCHECK(hipMemcpyAsync(v, d_vis_, 4 * std::max<size_t>(nitems_, 1), hipMemcpyDeviceToDevice, s));
	HIPCHECK(hipStreamSynchronize(s));
	nm_vis_.push_back(v);
	nm_batch_items_.push_back(nitems_);
	for (size_t l = 0; l < lights.size(); ++l) {
		nm_lights_.push_back(lights[l]);
		nm_light_batch_.push_back((uint32_t)(nm_vis_.size() - 1));
	}
	nm_first_.insert(nm_first_.end(), first_item.begin(), first_item.end());
}

void DeviceScene::nm_compute(const std::vector<uint32_t>& inst_off, float ambient_bright, float* out4)
{
	const size_t ni = inst_off.size() - 1;
	if (inst_off.size() < 2 || ni != nm_ninst_ || inst_off.back() != nsamples_)
		throw std::runtime_error("nm_compute: instance offsets do not match the kept batches or the samples");
	// every kept item must lie inside its batch: first + instance size <= items
	const int nl = (int)nm_lights_.size();
	for (int l = 0; l < nl; ++l)
		for (size_t i = 0; i < ni; ++i) {
			const int32_t f = nm_first_[(size_t)l * ni + i];
			if (f >= 0 && (size_t)f + (inst_off[i + 1] - inst_off[i]) > nm_batch_items_[nm_light_batch_[l]])
				throw std::runtime_error("nm_compute: an instance's items run past its batch");
		}
	hipStream_t s = (hipStream_t)stream_;
	std::vector<const float*> visp(nl);
	for (int l = 0; l < nl; ++l)
		visp[l] = nm_vis_[nm_light_batch_[l]];
	DevArray<uint32_t> d_off(inst_off.size());
	DevArray<DevLight> d_l(std::max(nl, 1));
	DevArray<int32_t> d_first(std::max<size_t>(nm_first_.size(), 1));
	DevArray<const float*> d_visp(std::max(nl, 1));
	DevArray<float> d_out(4 * std::max<size_t>(nsamples_, 1));
	HIPCHECK(hipMemcpyAsync(d_off.p, inst_off.data(), 4 * inst_off.size(), hipMemcpyHostToDevice, s));
	if (nl) {
		HIPCHECK(hipMemcpyAsync(d_l.p, nm_lights_.data(), sizeof(DevLight) * nl, hipMemcpyHostToDevice, s));
		HIPCHECK(hipMemcpyAsync(d_first.p, nm_first_.data(), 4 * nm_first_.size(), hipMemcpyHostToDevice, s));
		HIPCHECK(hipMemcpyAsync(d_visp.p, visp.data(), sizeof(float*) * nl, hipMemcpyHostToDevice, s));
	}
	if (nsamples_) {
		k_nm_data<<<grid_for(nsamples_), kBlock, 0, s>>>(d_pos_, d_nrm_, (uint32_t)nsamples_, d_off.p, (int)ni, d_l.p,
		                                                 nl, d_first.p, d_visp.p, ambient_bright, d_out.p);
		HIPCHECK(hipGetLastError());
		HIPCHECK(hipMemcpyAsync(out4, d_out.p, 16 * nsamples_, hipMemcpyDeviceToHost, s));
	}
	HIPCHECK(hipStreamSynchronize(s));
}

void DeviceScene::direct_grad(const double* lam3, double* dcolor3)
{
	hipStream_t s = (hipStream_t)stream_;
	const size_t L = h_lights_.size();
	if (!d_w_ && nitems_)
		throw std::runtime_error("direct_grad: no direct-light work on the device");
	double* dlam = dalloc<double>(3 * std::max<size_t>(nsamples_, 1));
	double* dpart = dalloc<double>(3 * kGradBlocks * std::max<size_t>(L, 1));
	HIPCHECK(hipMemcpyAsync(dlam, lam3, 24 * nsamples_, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemsetAsync(dpart, 0, 24 * kGradBlocks * std::max<size_t>(L, 1), s));
	uint32_t* doff = dalloc<uint32_t>(L + 1);
	HIPCHECK(hipMemcpyAsync(doff, h_light_off_.data(), 4 * (L + 1), hipMemcpyHostToDevice, s));
	EventTimer tm(s);
	if (L) {
		k_color_grad<<<dim3(kGradBlocks, (unsigned)L), kBlock, 0, s>>>(d_items_, d_w_, doff, dlam, dpart);
		HIPCHECK(hipGetLastError());
	}
	times.grad_ms = tm.stop();
	std::vector<double> hp(3 * kGradBlocks * L);
	if (L)
		HIPCHECK(hipMemcpy(hp.data(), dpart, 8 * hp.size(), hipMemcpyDeviceToHost));
	dfree(dlam);
	dfree(dpart);
	dfree(doff);
	for (size_t l = 0; l < L; ++l)
		for (int c = 0; c < 3; ++c) {
			double t = 0;
			for (int b = 0; b < kGradBlocks; ++b)
				t += hp[3 * (kGradBlocks * l + b) + c];
			dcolor3[3 * l + c] = t;
		}
}

void DeviceScene::get_weights(float* out, size_t n) const
{
	if (n > nitems_)
		throw std::runtime_error("get_weights: more than available");
	if (n)
		HIPCHECK(hipMemcpy(out, d_w_, 4 * n, hipMemcpyDeviceToHost));
}

void DeviceScene::get_vis(float* out, size_t n) const
{
	if (!d_vis_ || n > nitems_)
		throw std::runtime_error("get_vis: shadow factors were not kept");
	if (n)
		HIPCHECK(hipMemcpy(out, d_vis_, 4 * n, hipMemcpyDeviceToHost));
}

void DeviceScene::ambient_occlusion(const float* randoff, int num_samples, float distance, float multiplier,
                                    float falloff, float effect, const float* color, float* fac_out,
                                    const std::function<bool(float)>& between)
{
	hipStream_t s = (hipStream_t)stream_;
	if (nsamples_ == 0 || num_samples <= 0)
		return;
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	// (i + 0.5) / n, its square root and sin(acos(.)) depend only on (i, n):
	// evaluated here with the C library the reference uses
	std::vector<float2> side(num_samples);
	for (int i = 0; i < num_samples; ++i) {
		float q = (i + 0.5f) / num_samples;
		float cs = sqrtf(q);
		side[i] = make_float2(cs, sinf(acosf(cs)));
	}
	if (nsamples_ > ao_cap_ || nsamples_ < ao_cap_ / 4) {
		dfree(d_ao_);
		ao_cap_ = 0;
		d_ao_ = dalloc<float>(nsamples_);
		ao_cap_ = nsamples_;
	}
	if ((size_t)num_samples > side_cap_) {
		dfree(d_side_);
		side_cap_ = 0;
		d_side_ = dalloc<float2>(num_samples);
		side_cap_ = num_samples;
	}
	float2* d_side = (float2*)d_side_;
	float* d_ro = d_ao_;
	HIPCHECK(hipMemcpyAsync(d_side, side.data(), sizeof(float2) * num_samples, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemcpyAsync(d_ro, randoff, 4 * nsamples_, hipMemcpyHostToDevice, s));
	HIPCHECK(hipMemsetAsync(d_counters_, 0, kNumCounters * sizeof(unsigned long long), s));
	AOParams P;
	P.n = num_samples;
	P.distance = distance;
	P.multiplier = multiplier;
	P.falloff = falloff;
	P.effect = effect;
	P.color[0] = color[0];
	P.color[1] = color[1];
	P.color[2] = color[2];
	// one launch, or, when the caller follows progress, chunks of texels
	// with the caller asked between them whether to go on
	const size_t chunk = between ? kAOChunk : nsamples_;
	const size_t resident = (size_t)persistent_blocks() * (kBlock / 64);
	EventTimer tm(s);
	for (size_t b = 0; b < nsamples_; b += chunk) {
		const size_t e = std::min(nsamples_, b + chunk);
		const unsigned ao_grid = (unsigned)((e - b + kBlock / 64 - 1) / (kBlock / 64)); // a wave per texel
		// Texels per wave: three for each texel per wave that fits the chip
		// (6,144), since waves that would fit find the chip idle.  One ray
		// of 2,001 texels in a city: 64 to a wave 56 us, one 40; 17 rays of
		// 6,001 texels in a terrain: three 69 us, one 80; over 301 .. 300,001
		// texels and 1 .. 32 rays twice and four times as many were 0.3 and
		// 1 % slower in the mean.
		const size_t T = std::min<size_t>(64 / num_samples, (3 * (e - b) + resident - 1) / resident);
		if (!count_queries && T > 1) {
			const size_t per = (size_t)(kBlock / 64) * T; // texels per block
			k_ao_packed<<<(unsigned)((e - b + per - 1) / per), kBlock, march_lds_bytes(), s>>>(
			    V, d_pos_, d_nrm_, d_ro, d_side, P, (uint32_t)T, (uint32_t)b, (uint32_t)e, d_lm_, march_stack_depth(),
			    fac_out);
		} else if (count_queries)
			k_ao<true><<<ao_grid, kBlock, march_lds_bytes(), s>>>(V, d_pos_, d_nrm_, d_ro, d_side, P, (uint32_t)b,
			                                                      (uint32_t)e, d_lm_, d_counters_,
			                                                      march_stack_depth(), fac_out);
		else
			k_ao<false><<<ao_grid, kBlock, march_lds_bytes(), s>>>(V, d_pos_, d_nrm_, d_ro, d_side, P, (uint32_t)b,
			                                                       (uint32_t)e, d_lm_, d_counters_,
			                                                       march_stack_depth(), fac_out);
		HIPCHECK(hipGetLastError());
		if (between) {
			HIPCHECK(hipStreamSynchronize(s));
			if (!between((float)e / (float)nsamples_))
				break;
		}
	}
	times.ao_ms = tm.stop();
	read_counters();
}

// ---------------------------------------------------------------------------
void DeviceScene::query_distance(const float* pts, size_t n, float* out)
{
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	Scratch<float> pp(spare_, 3 * n), po(spare_, n);
	float *dp = pp.p, *dout = po.p;
	HIPCHECK(hipMemcpy(dp, pts, 12 * n, hipMemcpyHostToDevice));
	k_q_distance<<<grid_for(n), kBlock, 0, (hipStream_t)stream_>>>(V, dp, (uint32_t)n, dout);
	HIPCHECK(hipGetLastError());
	HIPCHECK(hipStreamSynchronize((hipStream_t)stream_));
	HIPCHECK(hipMemcpy(out, dout, 4 * n, hipMemcpyDeviceToHost));
}

void DeviceScene::query_shadow(const float* from, const float* to, const float* k, size_t n, float* out,
                               uint32_t* steps)
{
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	Scratch<float> pa(spare_, 3 * n), pb(spare_, 3 * n), pk(spare_, n), po(spare_, n);
	Scratch<uint32_t> ps(spare_, n);
	float *da = pa.p, *db = pb.p, *dk = pk.p, *dout = po.p;
	uint32_t* dst = ps.p;
	HIPCHECK(hipMemcpy(da, from, 12 * n, hipMemcpyHostToDevice));
	HIPCHECK(hipMemcpy(db, to, 12 * n, hipMemcpyHostToDevice));
	HIPCHECK(hipMemcpy(dk, k, 4 * n, hipMemcpyHostToDevice));
	hipStream_t s = (hipStream_t)stream_;
	const size_t chunk = size_t(1) << 30; // the list cursor is 32-bit
	// control words and list of this call's own: other calls on this device
	// scene may overlap it, and k_march's claims and hand-overs are theirs
	const bool lanes = n > QuerySrc::kWaveMax;
	Scratch<uint32_t> words(spare_, lanes ? kMarchWords : 0);
	Scratch<LongMarch> lng(spare_, lanes ? kLongCap : 0);
	size_t b = 0;
	do {
		const uint32_t m = (uint32_t)std::min(n - b, chunk);
		if (lanes)
			k_fill_u32<<<1, 64, 0, s>>>(words.p, kMarchWords, 0u);
		const QuerySrc src{da + 3 * b, db + 3 * b, dk + b, dout + b, dst + b};
		launch_marches(V, src, m, words.p, lng.p, nullptr, false, march_stack_depth(), march_lds_bytes(),
		               persistent_blocks(), nullptr, s);
		b += m;
	} while (b < n);
	HIPCHECK(hipStreamSynchronize((hipStream_t)stream_));
	HIPCHECK(hipMemcpy(out, dout, 4 * n, hipMemcpyDeviceToHost));
	if (steps)
		HIPCHECK(hipMemcpy(steps, dst, 4 * n, hipMemcpyDeviceToHost));
}

void DeviceScene::query_closest(const float* a, const float* b, size_t n, float* out)
{
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	Scratch<float> pa(spare_, 3 * n), pb(spare_, 3 * n), po(spare_, n);
	float *da = pa.p, *db = pb.p, *dout = po.p;
	HIPCHECK(hipMemcpy(da, a, 12 * n, hipMemcpyHostToDevice));
	HIPCHECK(hipMemcpy(db, b, 12 * n, hipMemcpyHostToDevice));
	k_q_closest<<<grid_for(n), kBlock, 0, (hipStream_t)stream_>>>(V, da, db, (uint32_t)n, dout);
	HIPCHECK(hipGetLastError());
	HIPCHECK(hipStreamSynchronize((hipStream_t)stream_));
	HIPCHECK(hipMemcpy(out, dout, 4 * n, hipMemcpyDeviceToHost));
}

void DeviceScene::query_occluded(const float* a, const float* b, size_t n, uint8_t* out)
{
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	Scratch<float> pa(spare_, 3 * n), pb(spare_, 3 * n);
	Scratch<uint8_t> po(spare_, n);
	float *da = pa.p, *db = pb.p;
	uint8_t* dout = po.p;
	HIPCHECK(hipMemcpy(da, a, 12 * n, hipMemcpyHostToDevice));
	HIPCHECK(hipMemcpy(db, b, 12 * n, hipMemcpyHostToDevice));
	k_q_occluded<<<grid_for(n), kBlock, 0, (hipStream_t)stream_>>>(V, da, db, (uint32_t)n, dout);
	HIPCHECK(hipGetLastError());
	HIPCHECK(hipStreamSynchronize((hipStream_t)stream_));
	HIPCHECK(hipMemcpy(out, dout, n, hipMemcpyDeviceToHost));
}

// ---------------------------------------------------------------------------
// radiosity
// ---------------------------------------------------------------------------
static void scan_u32_to_u64(const uint32_t* d_in, uint64_t n, uint64_t* d_out, uint64_t* h_total, hipStream_t s)
{
	constexpr uint64_t per_block = (uint64_t)kBlock * 16;
	uint32_t nb = (uint32_t)((n + per_block - 1) / per_block);
	if (nb == 0) {
		*h_total = 0;
		return;
	}
	uint64_t* sums = dalloc<uint64_t>(nb + 1);
	k_scan_blocks<<<nb, kBlock, 0, s>>>(d_in, n, d_out, sums);
	k_scan_sums<<<1, kBlock, 0, s>>>(sums, nb, sums + nb);
	k_scan_add<<<nb, kBlock, 0, s>>>(d_out, n, sums);
	HIPCHECK(hipGetLastError());
	HIPCHECK(hipMemcpyAsync(h_total, sums + nb, 8, hipMemcpyDeviceToHost, s));
	HIPCHECK(hipStreamSynchronize(s));
	dfree(sums);
}

void DeviceScene::rad_set_patches(const float* pos, const float* nrm, size_t n)
{
	dfree(rad.pos);
	dfree(rad.nrm);
	npatches = n;
	rad.pos = dalloc<float>(3 * n);
	rad.nrm = dalloc<float>(3 * n);
	if (n) {
		HIPCHECK(hipMemcpy(rad.pos, pos, 12 * n, hipMemcpyHostToDevice));
		HIPCHECK(hipMemcpy(rad.nrm, nrm, 12 * n, hipMemcpyHostToDevice));
	}
	// bounds and the longest normal, for the grid of the link search
	links_lo_[0] = links_lo_[1] = links_lo_[2] = INFINITY;
	links_hi_[0] = links_hi_[1] = links_hi_[2] = -INFINITY;
	links_nmax2_ = 0.0;
	links_finite_ = true;
	for (size_t i = 0; i < n; ++i) {
		double l2 = 0.0;
		for (int a = 0; a < 3; ++a) {
			const float p = pos[3 * i + a], q = nrm[3 * i + a];
			if (!std::isfinite(p) || !std::isfinite(q))
				links_finite_ = false;
			links_lo_[a] = std::min(links_lo_[a], p);
			links_hi_[a] = std::max(links_hi_[a], p);
			l2 += (double)q * q;
		}
		links_nmax2_ = std::max(links_nmax2_, l2);
	}
}

// All pairs (i, j > i) that pass the factor thresholds, in chunks of
// kPairChunk columns per row (the reference's loop, lighter.cpp:728-749).
void* DeviceScene::link_candidates_all(uint64_t& ncand, uint64_t* coff)
{
	hipStream_t s = (hipStream_t)stream_;
	const uint32_t N = (uint32_t)npatches;
	if (npatches > kMaxAllPairsPatches)
		throw std::runtime_error("radiosity: the all-pairs link search takes at most " +
		                         std::to_string(kMaxAllPairsPatches) + " patches (" + std::to_string(npatches) +
		                         (links_finite_ ? " given)" : " given; positions or normals are not finite)"));
	const uint32_t nchunks = (N + kPairChunk - 1) / kPairChunk;
	const uint64_t ncounts = (uint64_t)N * nchunks;
	DevArray<uint32_t> counts(ncounts);
	DevArray<uint64_t> offs(ncounts);
	const dim3 g(grid_for(N), nchunks);
	k_pairs<false><<<g, kBlock, 0, s>>>(rad.pos, rad.nrm, N, nchunks, counts.p, nullptr, nullptr);
	HIPCHECK(hipGetLastError());
	scan_u32_to_u64(counts.p, ncounts, offs.p, &ncand, s);
	uint2* cand = dalloc<uint2>(ncand);
	k_pairs<true><<<g, kBlock, 0, s>>>(rad.pos, rad.nrm, N, nchunks, nullptr, offs.p, cand);
	k_row_first<<<grid_for((uint64_t)N + 1), kBlock, 0, s>>>(N, nchunks, offs.p, ncand, coff);
	HIPCHECK(hipGetLastError());
	HIPCHECK(hipStreamSynchronize(s));
	return cand;
}

// Most pairs of clusters and clusters of one run of the search: launches of a
// wave for each pair and of 16 blocks for each cluster stay below 2^32
// threads.
constexpr uint64_t kLinkRunPairs = (1ull << 26) - 4096;
constexpr uint32_t kLinkRunClusters = 1u << 19;

// The links over clusters of patches: degrees, CSR offsets and columns (in
// any order within a row).  Returns the entries; colx: the columns.
uint64_t DeviceScene::links_by_clusters(uint32_t** colx, size_t* cap)
{
	hipStream_t s = (hipStream_t)stream_;
	const uint32_t N = (uint32_t)npatches;
	const uint32_t nc = (N + kCl - 1) / kCl, ns = (nc + kCl - 1) / kCl, Npad = nc * kCl;
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	Scratch<float4> sp(spare_, Npad), sn(spare_, Npad);
	{
		// cells of a sixteenth of the longest linking distance (l^2 <= |nA| |nB|
		// / (pi kSmall): 17.8 m for unit normals), 2^24 bins at most; sized in
		// double, which a large extent does not overflow
		double w = std::sqrt(links_nmax2_ / (M_PI * (double)kSmall)) / 16, cells;
		for (int a = 0; a < 3; ++a)
			w = std::max(w, ((double)links_hi_[a] - links_lo_[a]) * 1e-6);
		w = std::max(w, 1e-30);
		PatchBins G;
		for (;; w *= 1.26) {
			cells = 6;
			for (int a = 0; a < 3; ++a) {
				const double n = std::floor(((double)links_hi_[a] - links_lo_[a]) / w) + 1;
				for (G.bits[a] = 0; std::ldexp(1.0, (int)G.bits[a]) < n; ++G.bits[a]) {
				}
				cells *= std::ldexp(1.0, (int)G.bits[a]);
			}
			if (cells <= (double)(1u << 24))
				break;
		}
		for (int a = 0; a < 3; ++a)
			G.lo[a] = links_lo_[a];
		G.inv = (float)(1.0 / w);
		const size_t nb = (size_t)cells;
		Scratch<uint32_t> bin(spare_, N), count(spare_, nb + 1);
		Scratch<uint64_t> start(spare_, nb + 1);
		HIPCHECK(hipMemsetAsync(count.p, 0, 4 * (nb + 1), s));
		k_patch_bins<<<grid_for(N), kBlock, 0, s>>>(rad.pos, rad.nrm, N, G, bin.p, count.p);
		HIPCHECK(hipGetLastError());
		uint64_t total = 0;
		scan_u32_to_u64(count.p, nb + 1, start.p, &total, s);
		k_patch_place<<<grid_for(Npad), kBlock, 0, s>>>(rad.pos, rad.nrm, N, Npad, bin.p, start.p, count.p, sp.p, sn.p);
		HIPCHECK(hipGetLastError());
		HIPCHECK(hipStreamSynchronize(s)); // before bin .. start go
	}
	Scratch<ClBox> box(spare_, nc), quart(spare_, 4 * (size_t)nc), sup(spare_, ns);
	Scratch<uint32_t> count(spare_, (uint64_t)nc + 1);
	Scratch<uint64_t> coff(spare_, (uint64_t)nc + 1);
	k_cluster_boxes<<<gridn_waves(nc), kBlock, 0, s>>>(sp.p, sn.p, nc, box.p, quart.p);
	k_super_boxes<<<gridn_waves(ns), kBlock, 0, s>>>(box.p, nc, ns, sup.p);
	HIPCHECK(hipMemsetAsync(count.p + nc, 0, 4, s));
	k_cluster_pairs<false><<<gridn_waves(nc), kBlock, 0, s>>>(box.p, quart.p, nc, sup.p, ns, 0, nc, count.p, nullptr, 0,
	                                                          nullptr, nullptr);
	HIPCHECK(hipGetLastError());
	uint64_t npairs = 0;
	scan_u32_to_u64(count.p, (uint64_t)nc + 1, coff.p, &npairs, s);
	// The pairs of clusters in runs of consecutive first clusters, as many as
	// a launch's 2^32 threads and a quarter of the free memory take (some 550
	// bytes each): one run but for the largest scenes.  With several, each is
	// gone through twice, for the degrees and for the columns.
	struct Run {
		uint32_t a0, a1;
		uint64_t base, n; // first pair, pairs
	};
	std::vector<Run> runs;
	uint64_t limit = std::min(links_run_pairs, kLinkRunPairs);
	if (npairs > (1u << 22)) {
		size_t free_bytes = 0, total_bytes = 0;
		HIPCHECK(hipMemGetInfo(&free_bytes, &total_bytes));
		limit = std::min<uint64_t>(limit, std::max<uint64_t>(free_bytes / 4 / 550, 1u << 20));
	}
	if (npairs <= limit && nc <= kLinkRunClusters) {
		runs.push_back(Run{0, nc, 0, npairs});
	} else {
		std::vector<uint64_t> off((size_t)nc + 1);
		HIPCHECK(hipMemcpyAsync(off.data(), coff.p, 8 * off.size(), hipMemcpyDeviceToHost, s));
		HIPCHECK(hipStreamSynchronize(s));
		for (uint32_t a = 0; a < nc;) {
			uint32_t e = a + 1; // a cluster has fewer than 2^26 partners
			while (e < nc && off[e + 1] - off[a] <= limit && e - a < kLinkRunClusters)
				++e;
			runs.push_back(Run{a, e, off[a], off[e] - off[a]});
			a = e;
		}
	}
	uint64_t most = 0;
	uint32_t most_clusters = 0;
	for (const Run& r : runs) {
		most = std::max(most, r.n);
		most_clusters = std::max(most_clusters, r.a1 - r.a0);
	}
	Scratch<uint2> pairs(spare_, most), pairs2(spare_, most);
	Scratch<uint16_t> quarters(spare_, most);
	Scratch<uint64_t> mask(spare_, most * kCl);
	Scratch<uint32_t> ncand(spare_, most + 1), of(spare_, most), deg(spare_, (uint64_t)N + 1);
	Scratch<uint64_t> first2(spare_, (uint64_t)most_clusters + 1);
	HIPCHECK(hipMemsetAsync(deg.p, 0, 4 * ((size_t)N + 1), s));
	uint32_t split = 0;
	while (split < kLinkSplitMax && ((uint64_t)Npad << split) < kLinkWaves)
		++split;
	std::vector<uint64_t> run_cand(runs.size(), 0); // candidates of the runs before (counting)
	// The pairs of run q that hold candidates, their masks the links'.  With
	// count, its number of candidates joins ncand_; with keep, they are
	// written to d_cand_ and d_clinked_, which a single run allocates.
	auto search = [&](size_t q, bool count, bool keep) {
		const Run& r = runs[q];
		PairWork F{sp.p, sn.p, pairs2.p, 0};
		if (!r.n)
			return F;
		k_cluster_pairs<true><<<gridn_waves(r.a1 - r.a0), kBlock, 0, s>>>(box.p, quart.p, nc, sup.p, ns, r.a0, r.a1,
		                                                                  nullptr, coff.p, r.base, pairs.p, quarters.p);
		HIPCHECK(hipGetLastError());
		const PairWork W{sp.p, sn.p, pairs.p, (uint32_t)r.n};
		k_cluster_masks<<<gridn_waves(r.n), kBlock, 0, s>>>(W, quarters.p, mask.p, ncand.p);
		HIPCHECK(hipGetLastError());
		Scratch<uint64_t> at(spare_, r.n + 1);
		Scratch<uint32_t> flag(spare_, r.n + 1);
		k_cluster_flags<<<grid_for(r.n + 1), kBlock, 0, s>>>(ncand.p, r.n, flag.p);
		HIPCHECK(hipGetLastError());
		uint64_t nfull = 0;
		scan_u32_to_u64(flag.p, r.n + 1, at.p, &nfull, s);
		F.npairs = (uint32_t)nfull;
		const uint32_t ncl = r.a1 - r.a0;
		k_cluster_compact<<<grid_for(std::max<uint64_t>(r.n, (uint64_t)ncl + 1)), kBlock, 0, s>>>(
		    r.n, at.p, ncl, coff.p + r.a0, r.base, pairs.p, pairs2.p, of.p, first2.p);
		HIPCHECK(hipGetLastError());
		if (nfull) {
			const uint32_t blocks = ncl * (kCl / (kBlock / 64)) << split;
			const uint64_t nwaves = (uint64_t)blocks * (kBlock / 64);
			Scratch<uint32_t> wcount(spare_, count || keep ? nwaves + 1 : 0);
			Scratch<uint64_t> woff(spare_, count || keep ? nwaves + 1 : 0);
			if (count || keep) {
				uint64_t n = 0;
				k_cluster_wave_candidates<<<blocks, kBlock, 0, s>>>(first2.p, of.p, split, mask.p, wcount.p);
				HIPCHECK(hipGetLastError());
				HIPCHECK(hipMemsetAsync(wcount.p + nwaves, 0, 4, s));
				scan_u32_to_u64(wcount.p, nwaves + 1, woff.p, &n, s);
				if (count) {
					run_cand[q] = ncand_;
					ncand_ += n;
				}
				if (keep && count) {
					d_cand_ = dalloc<uint2>(ncand_);
					d_clinked_ = dalloc<uint8_t>(ncand_);
				}
			}
			k_cluster_links<<<blocks, kBlock, 0, s>>>(V, F, r.a0, first2.p, of.p, split, mask.p, woff.p,
			                                          keep ? (uint2*)d_cand_ + run_cand[q] : nullptr,
			                                          keep ? (uint8_t*)d_clinked_ + run_cand[q] : nullptr);
			HIPCHECK(hipGetLastError());
			HIPCHECK(hipStreamSynchronize(s)); // before at .. woff go
		}
		return F;
	};
	const bool one = runs.size() == 1;
	PairWork F{sp.p, sn.p, pairs2.p, 0};
	for (size_t q = 0; q < runs.size(); ++q) {
		F = search(q, count_queries, count_queries && one);
		if (F.npairs) {
			k_cluster_degrees<<<gridn_waves(F.npairs), kBlock, 0, s>>>(F, of.p, mask.p, deg.p);
			HIPCHECK(hipGetLastError());
		}
	}
	uint64_t nnz = 0;
	scan_u32_to_u64(deg.p, (uint64_t)N + 1, rad.rowptr64, &nnz, s);
	*colx = (uint32_t*)spare_.take(4 * nnz, cap);
	const bool keep = count_queries && !one && ncand_;
	if (keep) {
		d_cand_ = dalloc<uint2>(ncand_);
		d_clinked_ = dalloc<uint8_t>(ncand_);
	}
	if (nnz || keep) {
		HIPCHECK(hipMemsetAsync(deg.p, 0, 4 * ((size_t)N + 1), s)); // the rows' cursors
		for (size_t q = 0; q < runs.size(); ++q) {
			if (!one)
				F = search(q, false, keep);
			if (F.npairs && nnz) {
				k_cluster_fill<<<gridn_waves(F.npairs), kBlock, 0, s>>>(F, of.p, mask.p, rad.rowptr64, deg.p, *colx);
				HIPCHECK(hipGetLastError());
			}
		}
	}
	HIPCHECK(hipStreamSynchronize(s)); // before the arrays here go
	return nnz;
}

// The same from all pairs, as the reference enumerates them: candidates, an
// occlusion test of each, links per row below the diagonal (atomics from the
// other end) and above it (the row's own candidates).
uint64_t DeviceScene::links_by_all_pairs(uint32_t** colx, size_t* cap)
{
	hipStream_t s = (hipStream_t)stream_;
	const uint32_t N = (uint32_t)npatches;
	View V = make_view(d_nodes_, d_dtri_, d_rtri_, ntri_, lo_, hi_, grid_, use_grid_ ? grid_base_ : 0, use_grid_ ? grid_fine_ : 0);
	DevArray<uint64_t> coff((uint64_t)N + 1); // first candidate of each row
	uint64_t ncand = 0;
	uint2* cand = (uint2*)link_candidates_all(ncand, coff.p);
	d_cand_ = cand;
	uint8_t* linked = dalloc<uint8_t>(ncand);
	d_clinked_ = linked;
	DevArray<uint32_t> lower((uint64_t)N + 1), upper((uint64_t)N + 1), cnt((uint64_t)N + 1);
	HIPCHECK(hipMemsetAsync(lower.p, 0, 4 * ((size_t)N + 1), s));
	HIPCHECK(hipMemsetAsync(cnt.p, 0, 4 * ((size_t)N + 1), s));
	if (ncand) {
		k_link_test<<<grid_for(ncand), kBlock, march_lds_bytes(), s>>>(V, rad.pos, cand, ncand, linked, lower.p,
		                                                               march_stack_depth());
		HIPCHECK(hipGetLastError());
	}
	k_link_upper<<<gridn_waves(N), kBlock, 0, s>>>(N, coff.p, cand, linked, upper.p, nullptr, nullptr, nullptr);
	k_row_sum<<<grid_for(N), kBlock, 0, s>>>(N, upper.p, lower.p, cnt.p);
	HIPCHECK(hipGetLastError());
	uint64_t nnz = 0;
	scan_u32_to_u64(cnt.p, (uint64_t)N + 1, rad.rowptr64, &nnz, s);
	*colx = (uint32_t*)spare_.take(4 * nnz, cap);
	if (nnz) {
		k_link_upper<<<gridn_waves(N), kBlock, 0, s>>>(N, coff.p, cand, linked, nullptr, rad.rowptr64, lower.p, *colx);
		HIPCHECK(hipMemsetAsync(upper.p, 0, 4 * ((size_t)N + 1), s)); // the lower parts' fill counters
		k_link_lower<<<grid_for(ncand), kBlock, 0, s>>>(cand, linked, ncand, rad.rowptr64, upper.p, *colx);
		HIPCHECK(hipGetLastError());
	}
	HIPCHECK(hipStreamSynchronize(s)); // before the arrays here go
	if (count_queries) { // the candidates are kept for reference_counts_links
		ncand_ = ncand;
	} else {
		dfree(d_cand_);
		dfree(d_clinked_);
	}
	return nnz;
}

// Up to so many patches the pairs are fewer than the clusters' launches and
// waits are worth (ms, all pairs and clusters: 2 patches 0.18 and 0.28; 3,001
// scattered in a city 0.49 and 0.85, in a row of a terrain 0.69 and 0.70, in
// a room 0.76 and 0.73; 6,001 0.48 and 0.95, 1.10 and 1.15, 1.33 and 1.10;
// 8,001 in a room 2.24 and 1.43).
constexpr uint32_t kAllPairsBelow = 6144;

size_t DeviceScene::rad_links()
{
	hipStream_t s = (hipStream_t)stream_;
	const uint32_t N = (uint32_t)npatches;
	dfree(rad.rowptr);
	dfree(rad.rowptr64);
	spare_.give(rad.col, col_cap_);
	rad.col = nullptr;
	spare_.give(rad.val, val_cap_);
	rad.val = nullptr;
	dfree(d_cand_);
	dfree(d_clinked_);
	ncand_ = 0;
	rad.nnz = 0;
	rad.rowptr64 = dalloc<uint64_t>((uint64_t)N + 1);
	EventTimer tm(s);
	uint32_t* colx = nullptr;
	size_t colx_cap = 0;
	struct Free {
		SpareBlocks& b;
		uint32_t*& p;
		size_t& cap;
		~Free() { b.give(p, cap); }
	} fr{spare_, colx, colx_cap};
	// symmetric CSR, columns ascending within a row; 32-bit row offsets too
	// while they fit (the solver forms take those)
	uint64_t nnz = 0;
	if (N > 1) {
		const bool all = links_mode == 1 || (links_mode == 0 && N <= kAllPairsBelow) || !links_finite_;
		nnz = all ? links_by_all_pairs(&colx, &colx_cap) : links_by_clusters(&colx, &colx_cap);
	} else {
		HIPCHECK(hipMemsetAsync(rad.rowptr64, 0, 8 * ((size_t)N + 1), s));
	}
	if (nnz < (1ull << 32)) {
		rad.rowptr = dalloc<uint32_t>((uint64_t)N + 1);
		k_u64_to_u32<<<grid_for((uint64_t)N + 1), kBlock, 0, s>>>(rad.rowptr64, (uint64_t)N + 1, rad.rowptr);
		HIPCHECK(hipGetLastError());
	}
	rad.nnz = nnz;
	rad.col = (uint32_t*)spare_.take(4 * nnz, &col_cap_);
	rad.val = (float*)spare_.take(4 * nnz, &val_cap_);
	if (nnz) {
		int bits = 1;
		while (bits < 32 && (1ull << bits) < N)
			++bits;
		sort_row_columns(colx, rad.col, nnz, N, rad.rowptr64, bits, spare_, s);
		k_link_factors<<<gridn_waves(N), kBlock, 0, s>>>(N, rad.rowptr64, rad.col, rad.pos, rad.nrm, rad.val);
		HIPCHECK(hipGetLastError());
	}
	HIPCHECK(hipStreamSynchronize(s)); // before colx goes
	times.links_ms = tm.stop();
	nlinks_ = nnz / 2;
	return nlinks_;
}

void DeviceScene::rad_get_csr(std::vector<uint32_t>& rowptr, std::vector<uint32_t>& col,
                              std::vector<float>& val) const
{
	if (!rad.rowptr)
		throw std::runtime_error("radiosity: the link CSR holds " + std::to_string(rad.nnz) +
		                         " entries; reading it takes fewer than 2^32");
	rowptr.resize(npatches + 1);
	col.resize(rad.nnz);
	val.resize(rad.nnz);
	HIPCHECK(hipMemcpy(rowptr.data(), rad.rowptr, 4 * (npatches + 1), hipMemcpyDeviceToHost));
	if (rad.nnz) {
		HIPCHECK(hipMemcpy(col.data(), rad.col, 4 * rad.nnz, hipMemcpyDeviceToHost));
		HIPCHECK(hipMemcpy(val.data(), rad.val, 4 * rad.nnz, hipMemcpyDeviceToHost));
	}
}

void DeviceScene::rad_get_links(uint32_t* rowmap, uint32_t* other, float* factor) const
{
	std::vector<uint32_t> rp, col;
	std::vector<float> val;
	rad_get_csr(rp, col, val);
	uint32_t o = 0;
	for (size_t i = 0; i < npatches; ++i) {
		rowmap[2 * i] = o;
		uint32_t c = 0;
		for (uint32_t k = rp[i]; k < rp[i + 1]; ++k) {
			if (col[k] > i) {
				other[o] = col[k];
				factor[o] = val[k];
				o++;
				c++;
			}
		}
		rowmap[2 * i + 1] = c;
	}
}

void DeviceScene::rad_set_colors(const float* diffuse3, const float* emit3, const float* area)
{
	size_t n = npatches;
	dfree(rad.diffuse);
	dfree(rad.area);
	dfree(rad.total);
	dfree(rad.out);
	dfree(rad.in);
	dfree(rad.x);
	rad.diffuse = dalloc<float>(3 * n);
	rad.area = dalloc<float>(n);
	rad.total = dalloc<float>(3 * n);
	rad.out = dalloc<float>(3 * n);
	rad.in = dalloc<float>(3 * n);
	rad.x = dalloc<float>(4 * n);
	if (n) {
		HIPCHECK(hipMemcpy(rad.diffuse, diffuse3, 12 * n, hipMemcpyHostToDevice));
		HIPCHECK(hipMemcpy(rad.area, area, 4 * n, hipMemcpyHostToDevice));
		HIPCHECK(hipMemcpy(rad.total, emit3, 12 * n, hipMemcpyHostToDevice));
		HIPCHECK(hipMemcpy(rad.out, emit3, 12 * n, hipMemcpyHostToDevice));
	}
}

void DeviceScene::rad_bounce(int count)
{
	hipStream_t s = (hipStream_t)stream_;
	uint32_t N = (uint32_t)npatches;
	EventTimer tm(s);
	for (int b = 0; b < count && N; ++b) {
		k_bounce_prep<<<grid_for(N), kBlock, 0, s>>>(N, rad.out, rad.diffuse, rad.area, (float4*)rad.x);
		k_bounce_rows<<<gridn_waves(N), kBlock, 0, s>>>(N, rad.rowptr64, rad.col, rad.val, (const float4*)rad.x,
		                                                 rad.in, rad.total);
		HIPCHECK(hipGetLastError());
		std::swap(rad.out, rad.in);
	}
	times.bounce_ms = tm.stop();
}

void DeviceScene::rad_get_total(float* out3) const
{
	if (npatches)
		HIPCHECK(hipMemcpy(out3, rad.total, 12 * npatches, hipMemcpyDeviceToHost));
}

} // namespace lgx
