// psv_resident.h -- launch parameters of the resident time loop: many steps of a
// shot in one cooperative launch, its wavefields held in registers.
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>

#include "psv_step.h"

namespace psv {

// Velocity halo of a tile.  Two half-steps reach four cells, but not in one direction: where the
// staggered difference of one half reaches two cells the other's reaches one.
constexpr int kResHalo = 3;
constexpr int kResOwnX = 64 - 2 * kResHalo;    // columns a tile owns between two others

// One workgroup's tile: it owns the cells [z0, z1) x [x0, x1) and holds the region
// that starts at (zr, xr): kResHalo more cells on every side that has a neighbour.
struct ResTile {
    int z0, z1, x0, x1;
    int zr, xr;
    int edge;    // the region meets a CPML strip, the free surface or the grid's frame
    int row0;    // rows of all waves of the tiles before this one
    int xs, xe;  // columns of the launch: it has no tiles outside
    int shadow;  // computed for its neighbours only, writes nothing
    int pad;
};

// A grid with more tiles than CUs runs as strips of columns, some steps at a time: without
// neighbours the outer kResHalo columns of a strip go wrong every step, so a strip has more columns
// of tiles on each side that are computed and thrown away, each kStripCells wide, which lasts for
// kStripSteps steps.
constexpr int kStripSteps = kResOwnX / kResHalo;
constexpr int kStripCells = kStripSteps * kResHalo;
constexpr int kStripColumns = 4;  // at most

// The state's arrays in the order vx, vz, sxx, szx, szz, mvxx, mvzx, msxxx, mszxx, mvzz, mvxz,
// mszzz, mszxz.
constexpr int kStateArrays = 13;

// Point sources and receivers of a (slot, tile, wave): layers of at most one entry per
// lane, in the order they act; head: row | comp << 8 | receiver << 16; id: signal row or
// receiver of the lane (-1: none).
struct ResPoints {
    const int* off;   // [(slot * ntile + tile) * waves + wave] into head
    const int* head;
    const int* id;    // [layer][64]
};

// What a launch runs: the forward and adjoint steps (kForward, kAdjoint), and for the exact
// gradient a forward segment that writes its derivative terms and the transposed steps that
// read them back.
enum { kReplay = 2, kReverse = 3 };

template <typename T>
struct ResidentParams {
    StepParams<T> p;         // fields, model and tables of the launch's first slot
    const ResTile* tiles;
    int ntile;
    int it0, it1;            // steps [it0, it1), each slot up to its own nt
    ResPoints pts;
    size_t tf_stride;        // elements from one stored time to the next
    // velocity exchange: per slot two generations of [nzt][xpitch] cells for the rims' rows and
    // [nxt][zpitch] for their columns, every 32 bits of a value a 64-bit word with a tag
    unsigned long long* exch;
    size_t exch_slot;        // words per slot
    int xpitch, zpitch;
    unsigned tag;            // tag of the launch's first step
    int* aborted;            // host memory: set when a wait ran out
    int kdiv;                // some CPML K differs from 1
    T* out[kStateArrays];    // the state after the steps: p's own arrays, or another set where
                             // strips still have to read the state before them
    // replay and reverse: five values per cell, [step - it0][slot][row of a wave][5][64 lanes],
    // and the reverse steps' gradients (lam, mu, mu_zx, rho_zp, rho_xp)
    T* terms;                // (of step terms_it0)
    size_t terms_step, terms_slot;
    int terms_it0;
    T* g5[5];
};

// The tile shapes (ResShape) of each type: X(index, waves, rows, rows_edge, us, forward, adjoint).
// 12 waves have 168 registers each and 8 have 256, which hold about 9 rows of FP32 and 6 of the
// 8-byte types.
#define PSV_RESIDENT_F32(X)                                                                      \
    X(0, 8, 2, 2, 2.9, 2.9, 2.9) X(1, 8, 3, 2, 3.3, 3.3, 3.3) X(2, 12, 3, 2, 3.5, 3.5, 3.5)       \
    X(3, 12, 4, 3, 4.0, 4.0, 4.0) X(4, 12, 5, 4, 4.7, 4.6, 4.8) X(5, 12, 6, 4, 5.2, 5.1, 5.3)     \
    X(6, 12, 7, 5, 6.0, 5.9, 6.2) X(7, 12, 8, 5, 7.0, 6.8, 7.4) X(8, 12, 9, 5, 7.6, 7.2, 8.8)
#define PSV_RESIDENT_F64(X)                                                                      \
    X(0, 8, 2, 2, 3.4, 3.4, 3.4) X(1, 8, 3, 2, 4.4, 4.4, 4.6) X(2, 12, 3, 2, 5.0, 5.0, 5.2)       \
    X(3, 8, 4, 3, 5.3, 5.3, 5.5) X(4, 8, 6, 4, 7.3, 7.2, 7.4) X(5, 8, 9, 5, 16.5, 11.0, 20.0)
#define PSV_RESIDENT_F32X2(X)                                                                    \
    X(0, 8, 2, 2, 9.0, 9.0, 9.0) X(1, 8, 3, 2, 13.7, 13.7, 13.7) X(2, 12, 2, 2, 14.2, 14.2, 14.2) \
    X(3, 8, 4, 3, 17.2, 17.2, 17.2)

// Tile shapes a launch can take: waves of a workgroup, stacked in z, and rows per wave of
// the interior and of the edge tiles; us: what a step takes (forward and adjoint mean, order
// 4, one MI355X, a grid that fills the launch), for the choice among them; forward, adjoint: the two
// apart, for the choice of the split step instead.
struct ResShape {
    int waves, rows, rows_edge;
    double us, forward, adjoint;
};

// The shapes built for a type (sizeof(T) bytes per value), smallest first; returns their
// number (0: the type has no resident loop).
template <typename T>
int resident_shapes(const ResShape** out);

// The kernel of an order, mode and shape and its workgroup size (null: not built): forward and
// adjoint, replay and reverse.
template <typename T>
const void* resident_kernel(int order, int mode, int shape, int* threads);
template <typename T>
const void* resident_kernel_discrete(int order, int mode, int shape, int* threads);

// Workgroups of one launch that are resident together on the current device.
template <typename T>
hipError_t resident_capacity(int order, int mode, int shape, int* workgroups);

// nslots * ntile workgroups; hipErrorInvalidValue for an order, mode or shape not built.
template <typename T>
hipError_t launch_resident(const ResidentParams<T>& a, int order, int mode, int shape, hipStream_t s);

}  // namespace psv
