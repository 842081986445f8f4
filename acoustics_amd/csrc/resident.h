// resident.h -- scenes small enough to stay on the chip for a block of steps.
//
// One step of a small grid moves little data but costs a launch, a cold start
// of every workgroup and a trip of the whole state through memory.  A resident
// launch instead keeps a scene's state in registers and LDS for up to AMP_ROWS
// steps: each workgroup owns a box of cells, and per step the workgroups
// exchange only the pressures on the faces of their boxes.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <memory>
#include <string>
#include <vector>

#include "kernels.h"

namespace fdtd {

// Cells of one class form up to 27 boxes (the products of the three segments
// of each axis: damped, plain, damped); each is cut into tiles of at most
// RES_COLUMNS columns along x.
enum : int { RES_THREADS = 256, RES_COLUMNS = 256 };

struct ResBox {
    int32_t lo[3], len[3];      // cells
    int32_t size[3], count[3];  // tile edge (the last tile of an axis may be smaller) and tiles per axis
    int32_t first;              // its first tile
    int32_t damped;             // bit d: axis d is damped
    int32_t slab;               // PML slab that stores its state (-1: no damped axis)
    int32_t swap;               // its tiles' columns run along y
};

// A tile in its own frame: columns along its first axis, x, or y with swap (the
// second axis is then x).  A class damped along x is thin there: along y it gives
// longer columns and fewer tiles.
struct ResTile {
    int32_t i0, j0, k0, bx, by, bz;
    int32_t swap;
    int32_t pitch;              // LDS words from one row of columns (along z) to the next
    int32_t damped, slab;       // (axes of the grid)
    uint32_t word0;             // its first word in the exchange buffer and in the route table
    int32_t words;              // faces' cells: x low, x high, y low, y high, z low, z high (one more word follows)
    int32_t tb, te;             // listener terms
    int32_t rb, re;             // object-adjacent records
    int32_t src, skip;          // meets a pressure source's box; holds object cells
};

// where the own cell next to a face word is sent, and the LDS places of that
// cell (low half) and of the halo cell received for the word (high half)
struct ResRoute {
    uint32_t to;                // word of the neighbour's buffer
    uint32_t lds;
};

// device block of one resident scene
struct ResScene {
    const SceneDev *S;
    const ResTile *tiles;
    const ResBox *boxes;
    ResRoute *route;
    unsigned long long *words;  // [2][nwords] pressure bits, and above them the tag of the step
    const int32_t *recs;        // records by tile
    const TermRef *terms;
    uint32_t nwords;
    int32_t ntiles, nboxes, pad;
};

// a workgroup's tile (null: padding)
struct ResItem {
    const ResScene *scene;
    int32_t tile, pad;
};

// Tile shapes: cells per column by number of damped axes, and the LDS words
// of a column (its cells, the high halo after them, the low halo last).
struct ResShape {
    int plain, one, more;
    int column_words, lds_words;  // of one buffer
    int buffers;                // of pressures
    int max_words, max_recs;    // face words and records a tile may hold
};
enum : int { RES_FINE = 0, RES_COARSE = 1, RES_LARGE = 2, RES_SHAPES = 3 };
ResShape resident_shape(int shape);

struct SceneSetup;
struct DeviceScene;

// Tiles of a scene (host).
struct ResPlan {
    int shape = RES_FINE;
    std::vector<ResBox> boxes;
    std::vector<ResTile> tiles;
    std::vector<int32_t> recs;
    std::vector<int32_t> order; // tiles in the order of their dispatch
    std::vector<TermRef> terms;
    uint32_t nwords = 0;
    int tile_of(int i, int j, int k) const;
};

// Why a scene cannot run resident, or null.  Which scenes can: the collocated
// scheme with static rasterized objects, and the staggered scheme, with
// pressure sources and the merged state.  Everything else keeps the step kernels.
const char *resident_refusal(const SceneSetup &S);
// Cuts the scene for a shape; false when a tile would exceed what the kernel
// holds per workgroup.
bool resident_plan(const DeviceScene &D, int shape, ResPlan &out);

// Host check of a scene's cut (an error text, or empty): every cell, record
// and listener term in exactly one tile of its class, every tile within what
// a workgroup holds.
std::string resident_check(const DeviceScene &D, int shape);

// A scene's tables and exchange buffers on the device.
struct ResidentScene {
    ResPlan plan;
    char *mem = nullptr;
    size_t bytes = 0;
    ResScene *dev = nullptr;
    // Plans the scene and places its tables (stream-ordered; returns with the
    // copies done).  False, with nothing held, when the scene or the device
    // does not take it: the step kernels then run it.
    // max_bytes bounds its device memory.
    bool build(const DeviceScene &D, hipStream_t st, size_t max_bytes = SIZE_MAX);
    void release();
};

// Steps from which a launch beats the step kernels: it loads and stores the whole
// state, once for each time its workgroups fill the device (`rounds`).  us per
// block, launched resident and by step kernels: 64^3 18 + 2 a step and 6.5 a step;
// 128^3 40 + 4 and 13; 144x144x144 45 + 8 and 14, and four of them in a batch 250 +
// 38 and 47; eight of 64^3 45 + 6 and 20.
inline int resident_least(int shape, int rounds) { return shape == RES_LARGE ? 8 * rounds : 4; }

// The launches of a set of resident scenes.
struct ResidentProgram {
    ResItem *items = nullptr;   // device
    int n = 0, shape = RES_FINE;
    int room = 0;               // workgroups of the shape that the device holds
    uint32_t tag = 1;
    int *trouble = nullptr;     // pinned host memory: see launch_resident
    int wait_limit = 0;
    bool callers_stream = false;   // the stream may be captured between launches
    // Scenes of one shape.  They are listed so that their workgroups fill the
    // device side by side; a scene's start at a multiple of eight and follow
    // each other within an XCD.
    fdtd_status upload(const std::vector<const ResidentScene *> &scenes, hipStream_t st);
    fdtd_status enqueue(hipStream_t st, int nsteps);
    bool gave_up() const { return trouble && *trouble != 0; }
    int least() const { return n > 0 ? resident_least(shape, (n + room - 1) / room) : 0; }
    void release();
};

// Step that a scene's clock is at; one that gave up gets its target back and its
// gate shut, for the step kernels to go on from there (the stream idle).
fdtd_status resident_reopen(const SceneDev &dev, long long *step);

// After a wait for a stream: what had been launched on it when resident_seq was
// called, before the wait, runs no more.
uint64_t resident_seq();
void resident_idle(hipStream_t st, uint64_t seq);

// Call before a stream that had resident launches goes away, with it idle.
void resident_forget_stream(hipStream_t st);

// Workgroups of a shape that the device holds at once (0: none).
int resident_capacity(int shape);
hipError_t launch_resident_routes(const ResScene *scene, int ntiles, int shape, hipStream_t s);
// Runs each listed scene up to nsteps steps from its clock.  tag: a number
// that grows by at least nsteps + 1 from launch to launch over the same
// buffers.  wait_limit bounds the wait for the scene's other workgroups to be
// dispatched; past it the scene gives the block up untouched, and every
// later one, and `trouble` (host memory) becomes 1.  A later wait that does not end sets it to 2.
// done: an event that the launch's end completes.
hipError_t launch_resident(int shape, const ResItem *items, int n, int nsteps, uint32_t tag, int wait_limit,
                           int *trouble, hipStream_t s, hipEvent_t done);

}  // namespace fdtd
