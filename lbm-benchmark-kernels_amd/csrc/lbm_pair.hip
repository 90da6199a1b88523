// lbm_pair.hip -- an even and an odd AA step of one lattice in one launch.
//
// The even step of the AA pattern is local to a node and the odd step reads
// the neighbours' results of it, so both can be done while a window of three
// x planes is held on chip: the PDFs then pass through memory once per two
// steps instead of twice.  A block owns a tile of TY x TZ cells of the y-z
// plane and sweeps it along a segment of x.  For each plane it
//   * collides the tile and a halo of one cell (even step; the halo is
//     computed by the neighbouring tiles as well),
//   * passes the values that travel to other cells of the tile through LDS,
//   * collides the tile's cells of the plane before (odd step) and stores
//     each value where the odd step would: slot d of the neighbour x + c_d,
//     or the cell's own slot inv(d) when that neighbour is solid
//     (src/BenchKernelD3Q19ListAaPv.c:755-845).
// A launch reads one PDF array and writes the other, since a tile's halo
// belongs to other tiles.  Every slot of a fluid cell is written by exactly
// one node.  Each node's arithmetic is that of the separate kernels: the
// same trt_collide on the same operands, the even step's results rounded to
// the storage type in between, so results are the same bits.
//
// Values of direction d travel to plane x + c_x,d.  While plane p is
// collided, the odd step works on plane q = p - 1 and needs the c_x < 0
// values of plane p, the c_x = 0 values of plane p - 1 and the c_x > 0 values
// of plane p - 2.  The thread that computed them holds the older ones in
// registers until then, so that LDS keeps 18 values per cell and parity; two
// parities make one barrier per plane enough.
//
// What bounds it (MI355X), and the two launches' time -> this one's per pair:
// * large lattices: HBM.  256^3 list FP64 moves 4.67 GB (13 % over the PDFs
//   once in and out: halos, lines shared with solid cells) at 4.07 TB/s, 1.50
//   -> 1.15 ms; aa-soa FP64 5.62 GB at 4.5 TB/s, 1.81 -> 1.24 ms, FP32 2.76 GB
//   at 4.45 TB/s, 0.94 -> 0.62 ms; 19 streams updated in place reach 4.7 TB/s.
// * FP16, and FP32 up to about 100^3: vector issue, 566 and 484 instructions
//   per lane and plane (470 and 394 of them arithmetic) at four wavefronts per
//   SIMD: pipe 129x83x110 FP16 52.2 -> 39.4 us.
// * FP64 up to about 100^3: loads of the halos and the lead planes, 1.8 to 2
//   times the cells' own with segments of a few planes: 64^3 29.6 -> 21.4 us.
// * 24^3 to 40^3: the latency of map, PDFs and stores in turn: 6 to 8 us
//   against 8 to 14 us.
#include "lbm_pair.h"

#include <math.h>
#include <stdio.h>
#include <mutex>

namespace lbm {

constexpr int kIndexOf(int d)    // LDS array of direction d: c_x < 0, = 0, > 0
{
	int n = cx(d) < 0 ? 0 : cx(d) == 0 ? 5 : 13;
	for (int e = 0; e < d; ++e) n += cx(e) == cx(d);
	return n;
}
constexpr int kAgeOf(int d) { return kIndexOf(d) - 13; }   // of a c_x > 0 direction

// ------------------------------------------------------- memory accesses
// Buffer accesses: an offset past the end of the window reads 0 and writes
// nothing, which takes the place of branches around solid cells and around
// the lanes of the halo.
typedef int v4i __attribute__((ext_vector_type(4)));
__device__ double raw_load_f64(v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.load.f64");
__device__ float raw_load_f32(v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.load.f32");
__device__ int raw_load_i32(v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.load.i32");
__device__ short raw_load_i16(v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.load.i16");
__device__ void raw_store_f64(double, v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.store.f64");
__device__ void raw_store_f32(float, v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.store.f32");
__device__ void raw_store_i16(short, v4i, int, int, int) __asm("llvm.amdgcn.raw.buffer.store.i16");

__device__ __forceinline__ void get(double & x, v4i r, uint32_t off) { x = raw_load_f64(r, (int)off, 0, 0); }
__device__ __forceinline__ void get(float & x, v4i r, uint32_t off) { x = raw_load_f32(r, (int)off, 0, 0); }
__device__ __forceinline__ void get(uint16_t & x, v4i r, uint32_t off) { x = (uint16_t)raw_load_i16(r, (int)off, 0, 0); }
__device__ __forceinline__ void put(double x, v4i r, uint32_t off) { raw_store_f64(x, r, (int)off, 0, 0); }
__device__ __forceinline__ void put(float x, v4i r, uint32_t off) { raw_store_f32(x, r, (int)off, 0, 0); }
__device__ __forceinline__ void put(uint16_t x, v4i r, uint32_t off) { raw_store_i16((short)x, r, (int)off, 0, 0); }

constexpr uint32_t kWindowBytes = 0xfffffff0u;

// A window of kWindowBytes into an array, moved from plane to plane.  The
// empty asm keeps the four words in place: otherwise the compiler holds 38
// bases in scalar registers and spills them.
struct Window {
	v4i r;
	__device__ __forceinline__ explicit Window(const void * p)
	{
		const uint64_t a = (uint64_t)p;
		r = v4i{(int)(uint32_t)a, (int)(uint32_t)(a >> 32), (int)kWindowBytes, 0x00020000};
		asm volatile("" : "+s"(r));
	}
	__device__ __forceinline__ void move(uint32_t bytes)
	{
		const uint64_t a = (((uint64_t)(uint32_t)r.y << 32) | (uint32_t)r.x) + bytes;
		r.x = (int)(uint32_t)a;
		r.y = (int)(uint32_t)(a >> 32);
		asm volatile("" : "+s"(r));
	}
};

// Barrier for LDS alone: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_barrier()
{
	__builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
	__builtin_amdgcn_s_barrier();
	__builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// The body-force increment of direction d (3 w_d c_x,d F; none where c_x = 0).
template <class R>
struct PairForce {
	R axis, diagonal;
	__device__ __forceinline__ R add(R f, int d) const
	{
		const R a = cy(d) != 0 || cz(d) != 0 ? diagonal : axis;
		return cx(d) > 0 ? f + a : cx(d) < 0 ? f - a : f;
	}
};

struct PairGrid {
	int X, Y, Z, py, pz;
	int y0, y1, z0, z1;          // the tiles cover y0 <= y < y1, z0 <= z < z1
	int nTy, nTz, seg, nSeg;
	uint32_t perXcd;             // tiles per XCD
	uint32_t planeBytes;
};

// LDS of a block: offsets of the cells of four planes (then empty ones, for
// lanes without a cell), and 18 values per cell of two parities.
template <class R, int TY, int TZ>
struct PairTile {
	static constexpr int W = TZ + 2, P = (TY + 2) * W, E = W + 1;
	static constexpr int kIdBytes = ((4 * P + 2 * E + 1) * 4 + 7) / 8 * 8;
	static constexpr size_t kLds = kIdBytes + sizeof(R) * 2 * 18 * P;
};

template <class Codec, int TY, int TZ, int NT, int WAVES, bool EL, bool OL, bool FS>
__global__ __launch_bounds__(NT, WAVES) void k_pair(const typename Codec::S * __restrict__ src,
                                                    typename Codec::S * __restrict__ dst, Codec cod,
                                                    const uint32_t * __restrict__ map, PairGrid g,
                                                    TrtC<typename Codec::R> k, PairForce<typename Codec::R> ft)
{
	using S = typename Codec::S;
	using R = typename Codec::R;
	using Tile = PairTile<R, TY, TZ>;
	constexpr int W = Tile::W, P = Tile::P, E = Tile::E;
	constexpr uint32_t kNone = 0u - (uint32_t)sizeof(S);    // offset of no cell: past every window
	static_assert(P <= NT, "one thread per cell of the tile and its halo");
	extern __shared__ char smem[];
	uint32_t * ids = reinterpret_cast<uint32_t *>(smem);
	R * val = reinterpret_cast<R *>(smem + Tile::kIdBytes);

	// consecutive blocks go to the 8 XCDs in turn: each XCD takes consecutive
	// tiles, so that the halos of tiles running side by side meet in its L2
	const uint32_t tile = (blockIdx.x & 7u) * g.perXcd + (blockIdx.x >> 3);
	if (tile >= (uint32_t)(g.nTy * g.nTz * g.nSeg)) return;
	const int tz = (int)(tile % (uint32_t)g.nTz), ty = (int)(tile / (uint32_t)g.nTz % (uint32_t)g.nTy);
	const int sg = (int)(tile / (uint32_t)(g.nTz * g.nTy));
	const int x0 = sg * g.seg, x1 = min(g.X, x0 + g.seg);

	// this thread's cell of the tile (threads past the last cell repeat it)
	const int t = min((int)threadIdx.x, P - 1);
	const int row = t / W, col = t % W;
	int y = g.y0 + ty * TY + row - 1, z = g.z0 + tz * TZ + col - 1;
	bool ok = y <= g.y1 && z <= g.z1;
	const bool inner = row >= 1 && row <= TY && col >= 1 && col <= TZ && y < g.y1 && z < g.z1;
	if (y < 0 || y >= g.Y) { if (g.py) y = y < 0 ? g.Y - 1 : 0; else ok = false; }
	if (z < 0 || z >= g.Z) { if (g.pz) z = z < 0 ? g.Z - 1 : 0; else ok = false; }
	const uint32_t cellOff = ok ? ((uint32_t)y * (uint32_t)g.Z + (uint32_t)z) * 4u : 0xfffffffcu;
	const uint32_t mapPlane = (uint32_t)g.Y * (uint32_t)g.Z * 4u;
	Window mapWin(reinterpret_cast<const char *>(map) + (size_t)x0 * mapPlane);     // plane x0 - 1
	auto next_id = [&](int plane) __attribute__((always_inline)) -> uint32_t {     // planes x0 - 1, x0, ... in turn
		const uint32_t id = (uint32_t)raw_load_i32(mapWin.r, (int)(plane <= x1 ? cellOff : 0xfffffffcu), 0, 0);
		mapWin.move(mapPlane);
		return id;
	};
	auto offset_of = [&](uint32_t id) __attribute__((always_inline)) -> uint32_t {
		return id * (uint32_t)sizeof(S) - (uint32_t)sizeof(S);
	};
	for (int i = (int)threadIdx.x; i < 2 * E + 1; i += NT) ids[4 * P + i] = kNone;

	S raw[19], raw1[19];         // values of the next plane (of plane x0), in flight
	R ga[19], gb[19], old[5];    // even-step results of planes p and p - 1 in turn, c_x > 0 ones of p - 2
	uint32_t offCur = offset_of(next_id(x0 - 1)), offPrev = kNone;
	uint32_t offNext = offset_of(next_id(x0)), idNext = next_id(x0 + 1);

	auto load = [&](S (&to)[19], uint32_t off) __attribute__((always_inline)) {
		Window w(src);
#pragma unroll
		for (int d = 0; d < 19; ++d) {
			if (d) w.move(g.planeBytes);
			get(to[d], w.r, off);
		}
	};
	// Even step of plane p.  FP16: the results as decoded values, which
	// measured 2-3 % faster on dense lattices than 16-bit ones decoded when read.
	auto even_part = [&](int p, R (&cur)[19], const S (&from)[19]) __attribute__((always_inline)) {
#pragma unroll
		for (int d = 0; d < 19; ++d) {
			cur[d] = cod.dec(from[d]);
			if (EL) cur[d] = ft.add(cur[d], d);
		}
		trt_collide(cur, k);
		if constexpr (sizeof(S) != sizeof(R)) {
#pragma unroll
			for (int d = 0; d < 19; ++d) cur[d] = cod.dec(cod.enc(cur[d]));
		}
		ids[(p & 3) * P + t] = offCur;
	};
	// The values that leave a cell into LDS.
	auto pass_on = [&](int p, const R (&cur)[19], const R (&prev)[19]) __attribute__((always_inline)) {
		R * v = val + (p & 1) * 18 * P + t;
#pragma unroll
		for (int d = 0; d < 18; ++d)
			v[kIndexOf(d) * P] = cx(d) < 0 ? cur[d] : cx(d) == 0 ? prev[d] : old[cx(d) > 0 ? kAgeOf(d) : 0];
	};
	// Odd step of plane q = p - 1.
	const int from = (inner ? t : E) - E;
	auto odd_part = [&](int p, const R (&prev)[19]) __attribute__((always_inline)) {
		const bool act = inner && offPrev != kNone;
		const uint32_t own = act ? offPrev : kNone;
		const uint32_t * n0 = ids + (act ? ((p - 2) & 3) * P + t - E : 4 * P);   // plane q - 1
		const uint32_t * n1 = ids + (act ? ((p - 1) & 3) * P + t - E : 4 * P);   // plane q
		const uint32_t * n2 = ids + (act ? (p & 3) * P + t - E : 4 * P);         // plane q + 1
		const R * v = val + (p & 1) * 18 * P + from;
		uint32_t nb[18];         // offset of the cell x - c_d, where direction d comes from and inv(d) goes
		R in[18];
		R f[19];
#pragma unroll
		for (int d = 0; d < 18; ++d) {
			const int at = E - cy(d) * W - cz(d);
			nb[d] = (cx(d) > 0 ? n0 : cx(d) == 0 ? n1 : n2)[at];
			in[d] = v[kIndexOf(d) * P + at];
			asm("" : "+v"(in[d]));       // read without a branch on nb[d]
		}
#pragma unroll
		for (int d = 0; d < 18; ++d) {
			f[d] = nb[d] != kNone ? in[d] : prev[inv_dir(d)];
			if (OL) f[d] = ft.add(f[d], d);
		}
		f[dC] = prev[dC];
		trt_collide(f, k);
		// opposite directions share a window that spans both their planes
		Window w(dst);
		int at = 0;
#pragma unroll
		for (int d = 0; d < 18; ++d) {
			const int e = inv_dir(d);
			if (e < d) continue;
			if (d != at) w.move((uint32_t)(d - at) * g.planeBytes);
			at = d;
			const uint32_t apart = (uint32_t)(e - d) * g.planeBytes;
			const bool fd = nb[e] != kNone, fe = nb[d] != kNone;
			R vd = f[d], ve = f[e];
			if (FS) {
				vd = fd ? ft.add(vd, d) : ft.add(vd, e);
				ve = fe ? ft.add(ve, e) : ft.add(ve, d);
			}
			put(cod.enc(vd), w.r, fd ? nb[e] : __builtin_elementwise_add_sat(own, apart));
			put(cod.enc(ve), w.r, fe ? nb[d] + apart : own);
		}
		w.move((uint32_t)(dC - at) * g.planeBytes);
		put(cod.enc(f[dC]), w.r, own);
	};
	// the c_x > 0 values of the plane before last, and the next plane
	auto advance = [&](const R (&prev)[19]) __attribute__((always_inline)) {
#pragma unroll
		for (int d = 0; d < 18; ++d)
			if (cx(d) > 0) old[cx(d) > 0 ? kAgeOf(d) : 0] = prev[d];
		offPrev = offCur;
		offCur = offNext;
	};

	// Planes x0 - 1 and x0: even part only, both loads in flight at once (with
	// short segments the latency of one is a tenth of the launch).
	load(raw, offCur);
	load(raw1, offNext);
	even_part(x0 - 1, ga, raw);
	offPrev = offCur;
	offCur = offNext;
	offNext = offset_of(idNext);
	load(raw, offNext);
	idNext = next_id(x0 + 2);
	even_part(x0, gb, raw1);
	advance(ga);
	auto step = [&](int p, R (&cur)[19], const R (&prev)[19]) __attribute__((always_inline)) {
		even_part(p, cur, raw);
		pass_on(p, cur, prev);
		offNext = p < x1 ? offset_of(idNext) : kNone;
		lds_barrier();
		load(raw, offNext);
		idNext = next_id(p + 2);
		odd_part(p, prev);
		advance(prev);
	};
	// as many stores (of no cell) as a step issues: the loop's first wait for
	// the loads may then count on them as all later ones do
	{
		Window w(dst);
#pragma unroll
		for (int d = 0; d < 19; ++d) put(S(0), w.r, kNone);
	}
	int p = x0 + 1;
	for (;;) {
		step(p, ga, gb);
		if (++p > x1) break;
		step(p, gb, ga);
		if (++p > x1) break;
	}
}

// ------------------------------------------------------------ launch shapes
// Tile shapes (cells in y and z, threads).  A block holds its tile's state in
// registers and LDS: at most 512 cells with halo in FP64, 1024 in the narrow
// types.  Rows of 32 cells and more keep whole lines in a row's accesses;
// 256^3 FP64 1.20 ms with 13 x 32, 1.33 with 10 x 40, 1.27 with 8 x 48, 1.35
// with 17 x 24.  The other shapes fit ragged planes (18 x 48, 28 x 32: measured
// on one, pipe 129x83x110 FP16, 39.5 against 40.7 us and more), small ones
// (5 x 32: 24^3 7.0 against 9.2 us) and large narrow ones (13 x 64).
constexpr int kShapes = 5;
constexpr int kTileY[kShapes] = {13, 13, 5, 18, 28}, kTileZ[kShapes] = {32, 64, 32, 48, 32};
constexpr int kTileThreads[kShapes] = {512, 1024, 256, 1024, 1024};

// Estimated time of a launch, per storage type and tile shape, in a unit of
// its own.  A block takes base + perBlock * (blocks on its CU) per plane, the
// two halo planes of a segment together as many as `lead`; blocksPerCU fit on
// a CU (registers, LDS; 0: shape not used).  Moving the values of a cell, the
// tile's halo included, takes `cell`.  More blocks than fit run in rounds, of
// which the last counts as full with the weight 1 - spread.  The constants
// were chosen for the least average loss over 44 lattices of 24^3 to 256^3
// (channels, pipes, blocks, porous media; up to 30 shapes and segment lengths
// each): the plan takes on average 0.5 %, at most 5 %, longer than the best.
// Per pair: aa-soa 64^3 FP32 17.3 -> 13.9 us against the smallest number of
// planes in turn, porous 96^3 FP32 37.1 -> 33.0 us.
// The list kernel's even and odd launch cost splitLaunch + splitNode * nodes in
// the same unit: they skip solid cells, a tile's lanes do not.
struct TypeCost { double start, lead, cell, spread, splitLaunch, splitNode; };
struct ShapeCost { int blocksPerCU; double base, perBlock; };
constexpr TypeCost kTypeCost[3] = {{2.6, 1.1, 2.6e-5, 0.2, 10.0, 7.5e-5},
                                     {0.8, 1.0, 0.7e-5, 0.6, 4.0, 2.1e-5},
                                     {0.8, 0.7, 1.5e-5, 0.65, 5.2, 2.3e-5}};
constexpr ShapeCost kShapeCost[3][kShapes] = {
	{{1, 2.66, 0}, {0, 0, 0}, {2, 1.1, 0.72}, {0, 0, 0}, {0, 0, 0}},
	{{2, 0.63, 0.71}, {1, 1.8, 0}, {4, 0.62, 0.34}, {1, 2.05, 0}, {1, 2.1, 0}},
	{{2, 0.67, 1.7}, {1, 3.5, 0}, {4, 0.7, 0.8}, {1, 3.5, 0}, {1, 3.95, 0}},
};

size_t pair_map_cells(const PairPlan & p) { return (size_t)(p.X + 2) * p.Y * p.Z; }

// Whether the first (end 0) or last plane of cells along an axis holds fluid.
static bool face_fluid(const LatticeDesc * ld, int axis, int end)
{
	const int X = ld->Dims[0], Y = ld->Dims[1], Z = ld->Dims[2];
	const int n[3] = {X, Y, Z};
	const int v = axis == 0 ? 1 : 0, u = 3 - axis - v;   // inner loop along x
	for (int i = 0; i < n[u]; ++i)
		for (int j = 0; j < n[v]; ++j) {
			int c[3];
			c[axis] = end ? n[axis] - 1 : 0;
			c[u] = i;
			c[v] = j;
			if (ld->Lattice[((size_t)c[2] * Y + c[1]) * X + c[0]] != LBM_CELL_OBSTACLE) return true;
		}
	return false;
}

// Tile shape and segment length with the least estimated time: that of the
// blocks a CU runs one after the other or that of moving the values, whichever
// is longer (with a smooth change between them).  Returns that time.
static double pair_shape(PairPlan * p, int nCU)
{
	const TypeCost & c = kTypeCost[p->prec];
	double best = 0.0;
	for (int s = 0; s < kShapes; ++s) {
		const ShapeCost & w = kShapeCost[p->prec][s];
		if (w.blocksPerCU == 0) continue;
		const int nTy = (p->y1 - p->y0 + kTileY[s] - 1) / kTileY[s], nTz = (p->z1 - p->z0 + kTileZ[s] - 1) / kTileZ[s];
		// the distinct segment lengths, each with the smallest n that gives it:
		// about 2 sqrt(X) of them, a long lattice has far more n
		for (int n = 1, seg; n <= p->X; n = seg > 1 ? (p->X + seg - 2) / (seg - 1) : p->X + 1) {
			seg = (p->X + n - 1) / n;
			const double blocks = (double)nTy * nTz * n, r = blocks / ((double)w.blocksPerCU * nCU);
			const double rounds = r <= 1.0 ? 1.0 : c.spread * r + (1.0 - c.spread) * ceil(r);
			const double idle = r <= 1.0 ? 1.0 : rounds / r;
			const double onCU = fmin(w.blocksPerCU, ceil(blocks / nCU));
			const double planes = seg + c.lead;
			const double inTurn = rounds * planes * (w.base + w.perBlock * onCU);
			const double moved = blocks * planes * (kTileY[s] + 1) * (kTileZ[s] + 1) * c.cell * idle * idle;
			const double t = c.start + cbrt(inTurn * inTurn * inTurn + moved * moved * moved);
			if (best == 0.0 || t < best) {
				best = t;
				p->shape = s;
				p->seg = seg;
				p->nSeg = n;
				p->nTy = nTy;
				p->nTz = nTz;
			}
		}
	}
	return best;
}

void pair_plan(PairPlan * p, const Common & common, const LatticeDesc * ld, uint64_t plane, bool openFaces)
{
	const KernelArgs & a = common.args;
	const int nCU = common.nCU;
	*p = PairPlan();
	p->device = common.device;
	const int periodic[3] = {ld->PeriodicX, ld->PeriodicY, ld->PeriodicZ};
	p->X = ld->Dims[0]; p->Y = ld->Dims[1]; p->Z = ld->Dims[2];
	p->py = periodic[1]; p->pz = periodic[2];
	p->prec = a.prec;
	p->f16Shift = a.f16Shift;
	const uint64_t elem = p->prec == PREC_FP64 ? 8 : p->prec == PREC_FP32S ? 4 : 2;
	if (a.twoStep == 0 || (a.twoStep < 0 && a.splitOption) || ld->nFluid == 0 || !ld->Lattice) return;
	// Slots of solid cells (and of a z row's ends) leave lines that a tile
	// writes in part, which costs more than the two copies of a call: aa-soa
	// channel, per pair, 256^3 FP64 1.63 -> 1.24 ms, 144^3 FP32 174 -> 129 us;
	// equal below 64^3.  Planes of the dense arrays begin 128 B behind a
	// multiple of 16 KiB, so that equal cells of the planes lie in different
	// cache channels.
	p->useDense = plane == 0;
	if (p->useDense) {
		const uint64_t page = 16384 / elem;
		plane = ((uint64_t)ld->nFluid + page - 1) / page * page + 128 / elem;
	}
	p->plane = plane;
	// opposite directions lie up to six planes apart and share a window; the
	// map's offsets within a plane of cells are 32-bit too
	if (7 * plane * elem > kWindowBytes || (uint64_t)p->Y * p->Z * 4 > kWindowBytes) return;
	const bool any = periodic[0] || periodic[1] || periodic[2];
	bool fluid[3][2];
	for (int i = 0; i < 3; ++i)
		for (int end = 0; end < 2; ++end) {
			fluid[i][end] = face_fluid(ld, i, end);
			if (!periodic[i] && !(openFaces && !any) && fluid[i][end]) return;
		}
	// tiles begin behind a solid face: with walls on the z faces the loads of
	// a row (tile and halo) then begin on a line of the full array
	p->y0 = fluid[1][0] ? 0 : 1;
	p->y1 = p->Y - (fluid[1][1] ? 0 : 1);
	p->z0 = fluid[2][0] ? 0 : 1;
	p->z1 = p->Z - (fluid[2][1] ? 0 : 1);
	if (p->y1 <= p->y0 || p->z1 <= p->z0) return;
	// Speed-up over the list kernel's two launches, porous media and channels:
	// FP64 1.14-1.43 below 64^3 and 1.05-1.3 above at a fluid fraction of 0.65
	// and more, 0.79-1.15 below that; FP32 1.2-1.58, 1.0-1.3 and 0.91-1.01; FP16
	// 1.04-1.68 below 64^3, above it 0.71-1.07 and only for dense lattices that
	// the tiles cover well 1.05 (128^3) to 1.21 (256^3).  The comparison below
	// takes most that gain more than 5 % and, of 160 lattices, one that loses
	// more than 3 % (FP64 176x134x188 at 0.53, 0.96).  aa-soa's launches visit
	// every cell: 1.04-2.5 in all types, also at 0.55.
	// Where the separate launches' array fits well into the 256 MiB last-level
	// cache and two arrays hardly do, the launch reads more from memory than they
	// do.  Porous media of 102 to 187 MiB, two launches' time over one's: where
	// the estimates are within a factor of 1.45, FP64 0.86-1.14 and FP32 0.81-1.1
	// (once 1.37, 126x96x139 at 104 MiB), further apart FP64 0.97-1.2 and FP32
	// 0.98-1.14.  So what is taken loses 3 % at most, and twelve refused ones would
	// have gained 5 % on average.  From 188 MiB on 1.03-1.29 in both types.  One
	// lattice at other addresses varied by 0.94-1.12 (FP64 133x129x75, 172 MiB).
	double t = pair_shape(p, nCU > 0 ? nCU : 256);
	const TypeCost & c = kTypeCost[p->prec];
	const double bytes = 19.0 * (double)elem * ld->nFluid, cache = 256.0 * (1 << 20);
	if (bytes > 0.4 * cache && bytes < 0.73 * cache) t *= 1.45;
	if (a.twoStep < 0 && !p->useDense && t > c.splitLaunch + c.splitNode * ld->nFluid) return;
	p->use = true;
}

void pair_report(const PairPlan & p)
{
	if (p.use)
		printf("# two-step launch:       tiles of %d x %d cells (y, z), %d segments of %d planes\n", kTileY[p.shape],
		       kTileZ[p.shape], p.nSeg, p.seg);
}

void pair_tile(const PairPlan & p, int * y, int * z)
{
	*y = kTileY[p.shape];
	*z = kTileZ[p.shape];
}

static size_t aligned(size_t n) { return (n + 4095) / 4096 * 4096; }
static size_t pdf_bytes(const PairPlan & p)
{
	return aligned((p.prec == PREC_FP64 ? 8 : p.prec == PREC_FP32S ? 4 : 2) * (size_t)19 * p.plane);
}
static size_t row_bytes(const PairPlan & p)
{
	return p.useDense ? aligned(sizeof(uint32_t) * ((size_t)p.X * p.Y + 1)) : 0;
}

// Plans that hold arrays, linked through `next`, and their `busy` marks.  The
// arrays are the library's own choice: an allocation that a lattice cannot do
// without takes them back from lattices that are not being stepped.
static std::mutex g_lock;
static PairPlan * g_held = nullptr;

PairUse::PairUse(PairPlan * plan) : p(plan)
{
	if (!p) return;
	std::lock_guard<std::mutex> hold(g_lock);
	p->busy = true;
}

PairUse::~PairUse()
{
	if (!p) return;
	std::lock_guard<std::mutex> hold(g_lock);
	p->busy = false;
}

size_t pair_bytes(const PairPlan & p)
{
	return (p.useDense ? 2 : 1) * pdf_bytes(p) + aligned(sizeof(uint32_t) * pair_map_cells(p)) + row_bytes(p);
}

bool pair_alloc(PairPlan * p)
{
	if (p->block) return true;
	const size_t pdf = pdf_bytes(*p), need = pair_bytes(*p);
	size_t free = 0, total = 0;
	int current = 0;
	void * block = nullptr, * own = nullptr;
	bool ok = hipGetDevice(&current) == hipSuccess && (current == p->device || hipSetDevice(p->device) == hipSuccess);
	ok = ok && hipMemGetInfo(&free, &total) == hipSuccess && need <= free / 2;
	ok = ok && hipMalloc(&block, need - (p->useDense ? 0 : pdf)) == hipSuccess;
	ok = ok && (p->useDense || hipMalloc(&own, pdf) == hipSuccess);
	if (current != p->device) (void)hipSetDevice(current);
	if (!ok) {
		(void)hipFree(block);
		(void)hipGetLastError();
		return false;
	}
	char * at = (char *)block;
	if (p->useDense) {
		p->other = at;
		at += pdf;
		p->dense = at;
		at += pdf;
		p->rows = (uint32_t *)at;
		at += row_bytes(*p);
	} else {
		p->other = own;
	}
	p->map = (uint32_t *)at;
	++p->generation;
	std::lock_guard<std::mutex> hold(g_lock);
	p->block = block;
	p->next = g_held;
	g_held = p;
	return true;
}

// With g_lock held.
static size_t release_locked(PairPlan * p)
{
	if (!p->block) return 0;
	PairPlan ** at = &g_held;
	while (*at != p) at = &(*at)->next;
	*at = p->next;
	p->next = nullptr;
	(void)hipFree(p->block);
	if (!p->useDense) (void)hipFree(p->other);
	p->block = nullptr;
	p->map = nullptr;
	p->other = nullptr;
	p->dense = nullptr;
	p->rows = nullptr;
	p->current = false;
	return pair_bytes(*p);
}

void pair_release(PairPlan * p)
{
	std::lock_guard<std::mutex> hold(g_lock);
	(void)release_locked(p);
}

size_t pair_reclaim(PairPlan * p)
{
	std::lock_guard<std::mutex> hold(g_lock);
	return p->busy ? 0 : release_locked(p);
}

size_t pair_reclaim_device(int device)
{
	std::lock_guard<std::mutex> hold(g_lock);
	size_t freed = 0;
	for (PairPlan * p = g_held, * next; p; p = next) {
		next = p->next;
		if (!p->busy && p->device == device) freed += release_locked(p);
	}
	return freed;
}

size_t pair_held(const PairPlan * p)
{
	std::lock_guard<std::mutex> hold(g_lock);
	return p->block ? pair_bytes(*p) : 0;
}

void pair_free(PairPlan * p)
{
	pair_release(p);
	p->use = false;
}

template <class Codec, int SHAPE>
static void launch_shape(const PairPlan & p, const void * src, void * dst, Codec cod, const TrtConsts & k0,
                         const ForceTerms & f0, bool el, bool ol, bool fs, hipStream_t stream)
{
	using S = typename Codec::S;
	using R = typename Codec::R;
	constexpr int TY = kTileY[SHAPE], TZ = kTileZ[SHAPE], NT = kTileThreads[SHAPE];
	constexpr int WAVES = sizeof(S) == 8 ? 2 : 4;
	const uint32_t tiles = (uint32_t)(p.nTy * p.nTz * p.nSeg);
	const PairGrid g = {p.X, p.Y, p.Z, p.py, p.pz, p.y0, p.y1, p.z0, p.z1, p.nTy, p.nTz, p.seg, p.nSeg, (tiles + 7) / 8,
	                    (uint32_t)(p.plane * sizeof(S))};
	const TrtC<R> k = trt_cast<R>(k0);
	const PairForce<R> ft = {(R)f0.f[dE], (R)f0.f[dNE]};
	const dim3 grid(8 * g.perXcd), block(NT);
	const size_t lds = PairTile<R, TY, TZ>::kLds;
	const S * s = (const S *)src;
	S * d = (S *)dst;
	if (!ol)           k_pair<Codec, TY, TZ, NT, WAVES, false, false, false><<<grid, block, lds, stream>>>(s, d, cod, p.map, g, k, ft);
	else if (el && fs) k_pair<Codec, TY, TZ, NT, WAVES, true, true, true><<<grid, block, lds, stream>>>(s, d, cod, p.map, g, k, ft);
	else if (el)       k_pair<Codec, TY, TZ, NT, WAVES, true, true, false><<<grid, block, lds, stream>>>(s, d, cod, p.map, g, k, ft);
	else if (fs)       k_pair<Codec, TY, TZ, NT, WAVES, false, true, true><<<grid, block, lds, stream>>>(s, d, cod, p.map, g, k, ft);
	else               k_pair<Codec, TY, TZ, NT, WAVES, false, true, false><<<grid, block, lds, stream>>>(s, d, cod, p.map, g, k, ft);
}

template <class Codec>
static void launch_codec(const PairPlan & p, const void * src, void * dst, Codec cod, const TrtConsts & k,
                         const ForceTerms & f, bool el, bool ol, bool fs, hipStream_t stream)
{
	if constexpr (sizeof(typename Codec::S) < 8) {
		switch (p.shape) {
			case 1: launch_shape<Codec, 1>(p, src, dst, cod, k, f, el, ol, fs, stream); return;
			case 3: launch_shape<Codec, 3>(p, src, dst, cod, k, f, el, ol, fs, stream); return;
			case 4: launch_shape<Codec, 4>(p, src, dst, cod, k, f, el, ol, fs, stream); return;
		}
	}
	if (p.shape == 2) launch_shape<Codec, 2>(p, src, dst, cod, k, f, el, ol, fs, stream);
	else launch_shape<Codec, 0>(p, src, dst, cod, k, f, el, ol, fs, stream);
}

void pair_launch(const PairPlan & p, const void * src, void * dst, const TrtConsts & k, const ForceTerms & f, bool el,
                 bool ol, bool fs, hipStream_t stream)
{
	const float s16 = (float)(1 << p.f16Shift);
	switch (p.prec) {
		case PREC_FP32S: launch_codec(p, src, dst, CodecF32{}, k, f, el, ol, fs, stream); break;
		case PREC_FP16S: launch_codec(p, src, dst, CodecF16{s16, 1.0f / s16}, k, f, el, ol, fs, stream); break;
		default: launch_codec(p, src, dst, CodecF64{}, k, f, el, ol, fs, stream);
	}
}

// Device memory that the library cannot do without.
hipError_t device_alloc(void ** p, size_t bytes)
{
	hipError_t e = hipMalloc(p, bytes);
	int device = 0;
	if (e == hipErrorOutOfMemory && hipGetDevice(&device) == hipSuccess && pair_reclaim_device(device) > 0) {
		(void)hipGetLastError();
		e = hipMalloc(p, bytes);
	}
	return e;
}

}  // namespace lbm
