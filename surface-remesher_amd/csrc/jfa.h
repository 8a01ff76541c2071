// jfa.h -- launcher of the JFA pass kernel (jfa.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "cvt_types.h"

namespace cvt {

// Launch shape of a JFA pass for one grid: the quad kernel (4 pixels per
// lane, persistent workgroups over runs or bands of rows) when W % 4 == 0
// (quad), and on the steps that take runs at other widths from 9 up (ragged),
// with the site table in a static LDS array of lds_entries float2 (16, 40 or
// 160 KB) when it fits, or, for larger tables, lds_entries = -20480: the
// first 20478 entries and a zero entry in LDS, the rest gathered from global
// memory;
// otherwise one pixel per lane.  tail_entries: the array (16 or 40 KB) that
// launch_jfa_tail stages the table in, at any width; 0 when it is larger.
// runs_mask < 0 (JFA_AUTO): runs where every wave of the launch gets one (on
// ragged plans from 1.5 per CU), bands of rows (one pixel per lane) elsewhere; otherwise bit k set = runs at step 2^k, clear =
// bands (the labels do not depend on it).
enum { JFA_AUTO = -1 };
struct JfaPlan {
    bool quad = false, ragged = false, lds = false;
    int grid = 0, threads = 0, table_f4 = 0, lds_entries = 0, tail_entries = 0;
    size_t lds_bytes = 0;
    int runs_mask = JFA_AUTO, blocks_per_cu = 0;
};
// blocks_per_cu > 0 replaces the built-in grid (four 256-thread workgroups
// per CU for tables of up to 5120 entries, one 1024-thread workgroup per CU
// above); runs_mask as in JfaPlan.
JfaPlan plan_jfa(int W, int H, int capS, int runs_mask = JFA_AUTO, int blocks_per_cu = 0);
// the steps 2^k that take runs under this plan (bit k)
int jfa_runs_mask(const JfaPlan &p, int W, int H);

// One JFA pass over a W x H map of byte-offset labels (8 * site index, `none`
// for no site): out(p) = best of the 9 labels at p + step * {-1, 0, 1}^2.
// If clear is non-null it is reset to `none`: with nclear > 0 in the quad kernel
// only where it can hold entries, the seed pixels q of sites [0, nclear)
// (rstep == 0) or q + rstep * {-1, 0, 1}^2 (rstep > 0); otherwise pixel by
// pixel.  The site table must hold capS + 1 entries rounded up to an even
// count.
// A non-null `stop` makes the pass write nothing while *stop is set (it is
// read with the pass's first loads).
void launch_jfa_pass(hipStream_t st, const JfaPlan &plan, const uint32_t *in, uint32_t *out,
                     const float2 *sites, int W, int H, int step, uint32_t *clear, uint32_t none,
                     int nclear = 0, int rstep = 0, const int *stop = nullptr);

// The last passes (five: steps 8, 4, 2, 1, 1; or the last three or four of
// them) fused into one launch over 32 x 32 tiles with a halo staged in LDS,
// for plans whose site table fits a 16 or 40 KB array and JFAs of eight passes
// or more: how many such a JFA takes with `done` passes run
// by launch_jfa_lattice (0: none), and the launch: out = those passes applied
// to `in`, bit for bit.  With a non-null clear that map is reset to `none` at
// the seed pixels of sites [0, nclear).  `stop` as in launch_jfa_pass.
int jfa_tail_passes(const JfaPlan &plan, int passes, int done);
void launch_jfa_tail(hipStream_t st, const JfaPlan &plan, int passes, const uint32_t *in,
                     uint32_t *out, const float2 *sites, int W, int H, uint32_t *clear,
                     uint32_t none, int nclear, const int *stop = nullptr);

// The first passes of a JFA in one launch over residue classes
// (jfa_lattice.hip): how many a map of W x H pixels and S sites takes that way
// (0: none), and the launch, which reads the seed map and writes the map after
// those passes to `out`, every pixel of it.  The seed map is left as it is.
// stop, blockpart, dstate and fa as in launch_jfa_seed_pass.
int jfa_lattice_passes(int W, int H, int S);
void launch_jfa_lattice(hipStream_t st, const uint32_t *seed, uint32_t *out,
                        const float2 *sites, int W, int H, uint32_t none,
                        const int *stop = nullptr, const double *blockpart = nullptr,
                        int *dstate = nullptr, const FinalArgs *fa = nullptr);

// The first pass from a seed map (labels only at the seed pixels of sites
// [0, S), none elsewhere), computed from the seeds into a map `out` that
// holds none everywhere: the same output as launch_jfa_pass with in = seed.
// Only the receivers q + step * {-1, 0, 1}^2 of the seed pixels q are
// written.  With a non-null fa, one more workgroup runs the previous site
// update's deferred finalize (cvt_finalize.h) if one is pending in dstate.
void launch_jfa_seed_pass(hipStream_t st, const uint32_t *seed, uint32_t *out,
                          const float2 *sites, int S, int W, int H, int step,
                          const int *stop = nullptr, const double *blockpart = nullptr,
                          int *dstate = nullptr, const FinalArgs *fa = nullptr);

// A patch of a batch, as the batched kernels see it.  Maps are concatenated
// (pix_off), site tables too (site_off; entry site_off + cap is the patch's
// sentinel, so `none` = 8 * (site_off + cap)); labels are byte offsets into
// the concatenated table.
struct BatchPatch {
    int W, H;
    long pix_off;
    int site_off, cap, S;      // table base, capacity (sentinel index), live sites
    int passes, first_step;    // JFA schedule
    int tile, tiles_x, tiles_y, tile_off;   // moment tiles
    int blk_off, nblk;         // update blocks [blk_off, blk_off + nblk)
    float rho_scale;           // 2^-k
    int done;                  // passes run by the lattice launch (0: none)
    int lat_off;               // its first workgroup of that launch
    int pad;
};
// a workgroup's share of a JFA pass: part b of the nb parts of one patch,
// either its rows [y0, y1) (bands) or the b-th share of the pass's runs
struct BatchUnit {
    int patch, y0, y1, b, nb, pad[3];
};

// Pass `pass` (0 .. pmax-1) of the batched JFA over all units; lds_bytes = 0
// gathers sites from global memory, otherwise every patch's table (at most
// lds_bytes) is staged in LDS.  One launch per step class in `modes` (bit 0:
// step >= 4, bit 1: step 1, bit 2: step 2); a unit runs in the launch of its
// patch's class.
// A patch whose first `done` passes run on residue classes
// (launch_jfa_batch_lattice, before every batched pass) reads `first` in its
// pass `done`, which resets the seed map at its seed pixels.  Any other patch
// of three passes or more starts with a scatter of its seeds into `first`
// (launch_jfa_batch_seeds, at the batched pass where its own pass 0 falls; its
// units skip that pass), reads `first` in its pass 1, which resets the seed
// map at its seed pixels, and resets `first` at the seeds' receivers in pass
// 2: its part of `first` holds its `none` between JFAs, as every patch's part
// of the seed map does.
void launch_jfa_batch(hipStream_t st, const BatchPatch *patches, const BatchUnit *units, int nunits,
                      uint32_t *seed, uint32_t *first, uint32_t *lab0, uint32_t *lab1,
                      const float2 *sites, int pass, int pmax, size_t lds_bytes, unsigned modes);
// site_patch[i]: the patch owning site slot i of the concatenated table (-1
// for padding and sentinels)
void launch_jfa_batch_seeds(hipStream_t st, const BatchPatch *patches, const int *site_patch,
                            int total_sites, const uint32_t *seed, uint32_t *first,
                            const float2 *sites, int pass, int pmax);

// The passes on residue classes of every patch with done > 0: workgroups
// [lat_off, lat_off + jfa_batch_lattice_groups) are the patch's, group_patch
// names the patch of each.  jfa_batch_lattice_passes: the `done` of a patch.
int jfa_batch_lattice_passes(int W, int H, int S);
int jfa_batch_lattice_groups(int W, int H);
void launch_jfa_batch_lattice(hipStream_t st, const BatchPatch *patches, const int *group_patch,
                              int groups, const uint32_t *seed, uint32_t *first,
                              const float2 *sites);

}  // namespace cvt
