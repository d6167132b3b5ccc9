/* Shared host/device definitions for the SES engine. */
#ifndef QS_COMMON_H
#define QS_COMMON_H

#include <math.h>
#include <stdint.h>

#define QS_PROBE 1.4f         /* probe radius, Angstrom (Kernels.cu:26) */
#define QS_EPS 0.001f         /* weld / outside tolerance (Kernels.cu:27) */
#define QS_EMPTY (2147483647 - 1) /* empty-cell marker in cell ranges (Kernels.cu:25) */

/* voxel labels written by field pass 1 */
#define QS_OUT 0   /* no atom within r + probe: field = probe      */
#define QS_SHELL 1 /* within r + probe of an atom, inside none      */
#define QS_IN 2    /* within r - dx of some atom: field = -dx       */

/* One SES grid: neighbour grid and SES grid share the origin (CudaSurf.cu:564-574). */
struct QsGrid {
    float ox, oy, oz; /* origin */
    float dx;         /* SES voxel size */
    float dxn;        /* neighbour-cell size = probe + max radius */
    int g;            /* SES grid points per axis */
    int gn;           /* neighbour cells per axis */
    int r;            /* pass-2 half window = ceil(probe / dx) */
    int lim;          /* cubes (i,j,k) with i,j,k < lim are polygonised */
};

/* Field pass 2: bit n is set when a window minimum of squared integer norm n can only be
   attained by offsets of norm n (no longer offset is within rounding of it), n < 256. */
struct QsNormFlags {
    uint64_t w[4];
};

/* Field pass 2: the shell voxels whose values a mesh can read, by their window minimum n of squared
   integer norms.  A vertex reads the two ends of an edge whose signs differ, so a voxel is read only
   if a neighbour one step away has the other sign (or is zero).  The distance to the nearest
   outside voxel changes by at most one voxel per step: n <= lo is positive with only positive
   neighbours, n >= hi is negative with only negative ones, and only lo < n < hi is evaluated and
   stored; the signs of the others follow from n.  The window (r voxels along each axis) limits n to
   offsets within it: a negative voxel next to a voxel whose nearest outside voxel lies r steps along
   an axis may see it no longer.  That takes a non-negative value at norm r^2, so a probe of r whole
   voxels (`edge`): then far voxels (n >= hi, or none in reach) with an outside voxel r + 1 steps away
   along an axis are stored too.  `all`: every shell voxel with n > lo is stored.  With lo = -1 that is
   the whole field.  Normals read the neighbours of those two ends too, so with lo a step further from
   the probe radius (a voxel that near to the outside has only positive ones within two steps) they
   have what they read; above it there is no bound within the window that leaves much out. */
struct QsBand {
    int lo, hi;
    int edge, all;
};

/* One molecule of a batch: its grid and where its rows live in the concatenated arrays. */
struct QsMol {
    QsGrid G;
    uint32_t atom_off, n_atoms; /* atoms (input order and cell order) */
    uint32_t cell_off, W;       /* first neighbour cell; 64-voxel words per grid row */
    uint64_t word_off;          /* first row word (bit masks, slot masks, counts) */
    uint64_t vox_off;           /* first voxel (field, cube records) */
    uint32_t vert_off, n_vert;  /* vertices (set after counting) */
    uint32_t tri_off, n_tri;    /* triangles (set after counting) */
    int rows_per_wave;          /* field pass 1, row kernel: rows per wavefront */
    int slab_rows;              /* field pass 1, slab kernel: y rows per block */
    /* x planes each stage produces (the whole grid, [0, g), unless the grid runs in x-slabs):
       field pass 1 labels [p1_lo, p1_hi), field pass 2 evaluates [p2_lo, p2_hi), the
       marching-cubes count covers grid points [mc_lo, mc_hi), and cubes with origin
       x < cube_hi are polygonised.  word_off and vox_off address global plane x, so a slab
       whose arrays start at plane p1_lo has offsets that wrap below zero. */
    int p1_lo, p1_hi, p2_lo, p2_hi, mc_lo, mc_hi, cube_hi;
    /* first of the molecule's field-pass-2 tile flags (in pass-2 tile order; ~0: none kept) */
    uint32_t tile_off;
};

/* Coarse indexes of prefix arrays: coarse[k] = the segment that holds item k << shift, with
   shift QS_COARSE_BLOCKS for block prefixes and QS_COARSE_ITEMS for row-word and vertex
   prefixes. */
#define QS_COARSE_BLOCKS 6
#define QS_COARSE_ITEMS 12

/* A launch over a batch: block b belongs to molecule mid[j] (or j) where
   bpre[j] <= b < bpre[j+1]; coarse indexes bpre. */
struct QsBatch {
    const QsMol *mols;
    const uint32_t *bpre;
    const uint32_t *coarse;
    const int *mid;
    int n;
};

/* Field pass 1: the bounds of its closed forms, for the kernel and for host checks of them. */
#ifdef __HIPCC__
#define QS_HD __host__ __device__ __forceinline__
#else
#define QS_HD inline
#endif

/* How far a float predicate's interval end may lie from its closed form along an axis of origin o
   (|o| + g dx bounds the coordinates), in voxels: qs_interval_eps0 + qs_interval_eps1 * ss for a
   threshold ss (see qs_closed_interval) */
QS_HD float qs_interval_eps0(float o, int g, float dx, float inv_dx) { return 1.2e-7f * inv_dx * (fabsf(o) + 6.0f * (float)g * dx + 4.0f); }
QS_HD float qs_interval_eps1(float inv_dx) { return 9.6e-7f * inv_dx; }

/* margin of the rows an atom reaches, each of which is tested exactly: the bound above along y, and the
   root of 4 u ss for a half-width near zero (sqrt(ss) = r + probe at most) */
QS_HD float qs_row_margin(float o, int g, float dx, float inv_dx) { return qs_interval_eps0(o, g, dx, inv_dx) + 1.0e-3f; }
QS_HD float qs_row_margin_r(float inv_dx) { return 6.0e-4f * inv_dx; }
QS_HD int qs_row_lo(float yc, float h, float ym) { return (int)ceilf(yc - h - ym); }
QS_HD int qs_row_hi(float yc, float h, float ym) { return (int)floorf(yc + h + ym); }

/* The z-interval of an atom in a row (all z of [zlo, zhi] with fl(S + fl(e(z)^2)) < ss) from its closed
   form, zc -+ h in voxel units (h2 = ss - S, h = root / dx, root within an ulp of sqrt(h2)), without
   evaluating the predicate.  The predicate's roundings move a boundary by at most
   u (A + g dx + 5/2 H + ss / 2H) / dx voxels and the closed form is off by at most u (4 g dx + 5 H) / dx
   (u = 2^-24, A the largest |z| of the grid, H = sqrt(h2) <= (1 + ss) / 2), so an end that is farther
   than eps = 2 u (A + 5 g dx + 4 + 8 ss) / dx from every grid point is decided by its side of it; the
   bound takes H >= 1/8.  False: an end is nearer than that, or H is smaller (a few intervals in a
   thousand). */
QS_HD bool qs_closed_interval(float root, float h2, float zc, float inv_dx, float eps, int zlo, int zhi, int &L, int &R)
{
    const float h = root * inv_dx;
    const float lo = zc - h, hi = zc + h;
    const int l = (int)ceilf(lo), r = (int)floorf(hi);
    L = l > zlo ? l : zlo;
    R = r < zhi ? r : zhi;
    const float d = fminf(fabsf(lo - rintf(lo)), fabsf(hi - rintf(hi)));
    return d > eps && h2 > 0.015625f;
}

#endif
