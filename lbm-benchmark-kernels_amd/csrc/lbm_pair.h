// lbm_pair.h -- two time steps (an even and an odd step) in one launch, for a
// single list-aa-pv-soa or aa-soa lattice; see lbm_pair.hip.
#pragma once

#include "lbm_device.h"
#include "lbm_runtime.h"

namespace lbm {

// The launch plan of a lattice and what it owns on the device.  `map` holds,
// z fastest, for every cell of the box and one ghost plane at either end of x
// (its periodic image, or solid) the cell's index within a direction plane
// plus one, 0 for solid cells.  A launch reads one PDF array and writes
// another, `other`; the first is the kernel's own or, where that holds slots
// of solid cells between the fluid ones (aa-soa), `dense`, which holds the
// fluid cells' values alone.
struct PairPlan {
	bool use = false;
	int X = 0, Y = 0, Z = 0, py = 0, pz = 0;
	int y0 = 0, y1 = 0, z0 = 0, z1 = 0;   // range the tiles cover (solid faces left out)
	int prec = 0, f16Shift = 0;
	int device = 0;              // the lattice's, whatever the calling thread's current one is
	uint64_t plane = 0;          // values per direction plane of the arrays stepped
	int shape = 0;               // tile shape, see lbm_pair.hip
	int seg = 0, nSeg = 0, nTy = 0, nTz = 0;
	void * block = nullptr;      // the allocation of map, rows, dense and dense's other
	uint32_t * map = nullptr;
	void * other = nullptr;      // without dense an allocation of its own: it changes places with the kernel's array
	void * dense = nullptr;
	uint32_t * rows = nullptr;   // scratch of the dense map: one word per z row and their sum
	bool useDense = false;       // the arrays stepped are dense and other
	bool current = false;        // dense holds the kernel's present state
	int launches = 0;            // of the last Kernel() call
	unsigned generation = 0;     // counts pair_alloc's allocations: a graph captured with other arrays is stale
	// arrays that no Kernel() call is using can be given back, see pair_reclaim
	bool busy = false;
	PairPlan * next = nullptr;
};

// Decides whether the lattice is stepped in pairs (-two-step) and sets the
// launch shape; allocates nothing.  openFaces: fluid cells on a non-periodic
// face bounce there whatever the other axes are (the list kernel without any
// periodic axis); otherwise such a lattice is left to the separate kernels.
// plane: values per direction plane of the kernel's own array, or 0 to step
// dense ones.
void pair_plan(PairPlan * p, const Common & c, const LatticeDesc * ld, uint64_t plane, bool openFaces);

// Words of `map`.
size_t pair_map_cells(const PairPlan & p);
// Device memory of all the arrays.
size_t pair_bytes(const PairPlan & p);
// Cells of a tile in y and z.
void pair_tile(const PairPlan & p, int * y, int * z);

// Held by a Kernel() call that may step in pairs, from before it looks at the
// arrays until it returns.
struct PairUse {
	PairPlan * p;
	explicit PairUse(PairPlan * plan);
	~PairUse();
	PairUse(const PairUse &) = delete;
};

// Allocates the arrays unless the plan has them.  False where they would take
// more than half of the device's free memory: the call goes on with the
// separate kernels, and a later one asks again.
bool pair_alloc(PairPlan * p);
// Frees the arrays; the plan stays, and the next pair_alloc takes them again.
// Between Kernel() calls they hold nothing that is not in the kernel's own
// array too, or of use to the next call.
void pair_release(PairPlan * p);
// The arrays of one lattice, or of all lattices of a device, given back
// unless a Kernel() call is using them; the bytes freed.
size_t pair_reclaim(PairPlan * p);
size_t pair_reclaim_device(int device);
// Bytes the arrays hold at present.
size_t pair_held(const PairPlan * p);
// The same, and the lattice is stepped by the separate kernels from now on.
void pair_free(PairPlan * p);

// The launch shape, as a line of Init's report.
void pair_report(const PairPlan & p);

// One launch: both steps from src into dst.  evenLoad / oddLoad / oddStore:
// where the body-force increment is added, as in the two kernels.
void pair_launch(const PairPlan & p, const void * src, void * dst, const TrtConsts & k, const ForceTerms & f,
                 bool evenLoad, bool oddLoad, bool oddStore, hipStream_t stream);

}  // namespace lbm
