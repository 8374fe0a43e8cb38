// resident.hpp -- solver iterations that stay on the chip (gfx950).
//
// A mesh whose solver fields fit the chip is cut into one tile per workgroup
// (at most one workgroup per compute unit), every cell's fields stay in
// registers and its face coefficients in LDS for many iterations, and one
// launch runs the iterations to the caller's stopping test.  Between launches of the separate kernels an
// iteration of a small or middling mesh waits for launches, reduction passes
// and the host; here it waits for two exchanges among the workgroups.
//
// Tiles: bands of at most 62 columns (one lane per column, one halo lane on
// each side), RES_WAVES waves stacked in y, at most S block-Jacobi strips of 4
// rows per wave (the tile's strips spread evenly over its waves).  The halo
// lanes and the rows above and below a wave carry their own copies of what the
// stencil reads, advanced with the same expressions as the neighbour's, so an
// exchange never waits for a scalar.
//
// Exchange: every 8-byte word holds 32 bits of data and a 32-bit tag, written
// and read with relaxed device-scope atomics; a word whose tag matches is
// complete, so no fences or counters are needed and one exchange costs one
// store-to-load latency across the chip.  Words alternate between two slots: a
// workgroup writes a slot again only after every reader has posted a later
// word that follows its read.
//
// Reductions are compensated (double-double) like everywhere in the engine;
// every workgroup merges all partials in the same order, so all hold the same
// bits and take the same branch.
#pragma once
#include <hip/hip_runtime.h>

#include "engine_device.hpp"

namespace tea {
namespace res {

constexpr int RES_WAVES = 8;        // two per SIMD, 256 registers each
constexpr int RES_BLOCK = RES_WAVES * WAVE;
constexpr int RES_OUT_X = WAVE - 2;
constexpr int RES_MAX_WG = 256;
constexpr int RES_HISTORY = 1024;   // iterations per launch at most

// Words of the exchange buffers (all zero before the first launch).
constexpr int RED_COPIES = 8;
constexpr size_t RED_WORDS = 2 * (size_t)RED_COPIES * 8 * RES_MAX_WG;   // [slot][copy][word][workgroup]
constexpr int FACE_WORDS = 32;      // a column face of a wave: 16 rows in FP64, 32 in FP32
constexpr size_t COL_WORDS = 2 * (size_t)RES_MAX_WG * 2 * RES_WAVES * FACE_WORDS;   // [slot][workgroup][side][wave][word]
constexpr size_t ROW_WORDS = 2 * (size_t)RES_MAX_WG * 2 * 2 * 64; // [slot][workgroup][side][word][lane]
constexpr size_t EXCHANGE_WORDS = RED_WORDS + COL_WORDS + ROW_WORDS + 16;

typedef unsigned long long word_t;
enum : unsigned { VERDICT_NONE = 0, VERDICT_GO = 1, VERDICT_ABORT = 2 };   // whether all workgroups are resident

struct Exchange {
    word_t *red, *col, *row;
    double *history;        // device memory: the values of a run's iterations as they come
    unsigned *ctl;          // arrived, verdict, left
    unsigned tag;           // tags of this launch start above it
};

struct Tiles {
    Ext e;
    long pitch;
    int ow;                 // columns per band
    int nbx, nby;           // bands, tiles per band
    int ts;                 // strips per tile
    int s;                  // strips per wave
};

// Chooses the tiles of an nx x ny interior for at most max_wg workgroups;
// false when the mesh does not fit.
bool plan_tiles(Tiles &t, int nx, int ny, int h, long pitch, int bits, int max_wg);

// When the iterations end (besides the count): the caller's own tests, formed
// with its expressions.
struct Stop {
    double error_below;     // sqrt|rrn| < error_below
    int switch_after;       // from this iteration of the launch on (1-based) ...
    double switch_error;    // ... sqrt|rrn| <= switch_error
    // residual replacement due: drop = sqrt|q / q_ref| < delta or
    // sqrt|rr_ref| * drop < target (with have_q 0 the first q is the reference)
    int reliable, have_q;
    double q_ref, rr_ref, delta, target;
};

template <typename T> struct Fields {
    T *u, *p, *r, *z;
    const T *Kx, *Ky;
    T *rstore, *sd, *rtemp, *utemp;   // PPCG
    const T *z_in;                    // PPCG: z as the run finds it
    const T *u0;                      // Chebyshev
    T *w;
};

// What a run leaves for the host (host-visible memory), before the history.
struct Outcome {
    int iterations;         // done; -1: not every workgroup was resident, nothing was changed; -2: an exchange timed out
    int at_ur;              // PPCG: the last iteration ended at its replacement test, before its inner steps
    double rrn_end;         // PPCG: (r - rstore).z of the latest end
};

// CG iterations ([p = z + beta p], w = A p, u, r, z, r.z) with the values of
// the separate kernels.  history: p.w and r.z of each.
template <typename T>
hipError_t launch_cg(const Tiles &t, int prec, const Fields<T> &f, const Exchange &x, int with_p, double beta,
                     double rro, const Stop &stop, int max_its, double *history, Outcome *out, hipStream_t stream);

// PPCG outer iterations (begin, ur, `steps` inner steps with the coefficients
// coef[0 .. steps) and coef[coef_stride ...], end) with the values of the
// separate kernels.  from_inner: the first one starts at its inner steps, from
// r (rro: its r.z), and is not counted.  history: p.w, r.z, ur's r.z and the
// end's r.z of each.
template <typename T>
hipError_t launch_ppcg(const Tiles &t, int prec, const Fields<T> &f, const Exchange &x, int from_inner, int with_p,
                       double beta, double rro, double theta, const double *coef, int coef_stride, int steps,
                       const Stop &stop, int max_its, double *history, Outcome *out, hipStream_t stream);

// Chebyshev iterations n, n + 1, ... of the caller's loop (coef as above, from
// the first one's): in those with n >= check_from and n % 10 == 0 the caller's
// error becomes r.r, and after each its square root is taken; the run ends when
// that is below `target`.  history: r.r of each (0 where it is not formed).
template <typename T>
hipError_t launch_cheby(const Tiles &t, int prec, const Fields<T> &f, const Exchange &x, const double *coef,
                        int coef_stride, int n, int check_from, double error, double target, int max_its,
                        double *history, Outcome *out, hipStream_t stream);

}  // namespace res
}  // namespace tea
