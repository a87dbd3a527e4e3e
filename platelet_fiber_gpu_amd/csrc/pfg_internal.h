/*
 * pfg_internal.h -- device-side state of a pfg_handle and the launchers each
 * translation unit provides.  Not part of the C ABI.
 */
#ifndef PFG_INTERNAL_H
#define PFG_INTERNAL_H

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <vector>

#include "../../include/pfg.h"
#include "pfg_lattice.h"

namespace pfg {

/* Steps captured per chunk graph (even: a chunk ends on the copy of f it
 * started from). */
constexpr int GRAPH_CHUNK = 8;

/* IB work units: at most IB_CHUNK consecutive markers of one body, staged
 * in LDS; when their stencils span at most IB_BOX_CELLS lattice nodes the
 * chunk is summed node by node. */
constexpr int SCAN_SPAN = 8192; /* bins per block of the bin-count scan */
/* When the cell lists leave the elements out (only the fibrin ligand search
 * reads them), their bins are COARSE_BINS bins of the full grid along each
 * axis: a scan over 64 times fewer bins for a few more candidates. */
constexpr int COARSE_BINS = 4;
constexpr int IB_CHUNK_MIN = 16, IB_CHUNK = 128; /* markers of a chunk */
/* Chunks to have before they are made longer: two per CU.  A longer chunk
 * adds fewer of its nodes to the lattice twice; us per step with 2048 and
 * 512: 16625 markers 82 and 77, 31200 148 and 137, 62400 211 and 187, 25344 in
 * 24 lattices 186 and 175 (256 chunks: within 3 us of 512). */
constexpr int IB_CHUNKS_MIN = 512;
/* workgroups of the tile-gather spreading launch (each takes listed tiles in
 * turn) */
constexpr int SPREAD_TILE_GRID = 4096;
constexpr int IB_BOX_CELLS = 1024;
/* Markers listed for direct spreading per workgroup: their atomics follow
 * one another in two wavefronts, so that few markers go IB_DIRECT at a time
 * (625 scattered fibrin nodes among 1009 chunks: the launch takes 24 us, 60
 * with IB_CHUNK, whose five workgroups were the last to end); many fill
 * IB_DIRECT_GROUPS workgroups first, up to IB_CHUNK each (20000 nodes: 157 us
 * with IB_CHUNK, 167 with 16, whose idle lanes and staging cost more than
 * the shorter chain gives). */
constexpr int IB_DIRECT = 16, IB_DIRECT_GROUPS = 128;
/* Body spreading (spreading form 4): the chunks of a compact body (a
 * platelet of at most BODY_MAX_MARKERS markers, its stencils at most
 * BODY_BOX_DIM nodes along each axis) write their LDS sums to a scratch box
 * each; a workgroup per body adds its chunks' boxes over the body's box
 * (at most BODY_BOX_TILES tiles for the tile claims, at most
 * BODY_MAX_CHUNKS chunks) */
constexpr int BODY_MAX_MARKERS = 4096;
constexpr int BODY_BOX_DIM = 256;
constexpr int BODY_BOX_TILES = 1024;
constexpr int BODY_MAX_CHUNKS = 256;
/* Force pass by body: a workgroup per body of at most FB_MAX markers keeps
 * their positions and a cell list of at most FB_BINS bins in LDS for the
 * Morse pairs (which act within a body only) */
constexpr int FB_MAX = 1024;
constexpr int FB_BINS = 2048;
/* its neighbour lists: at most FB_NBR_MAX partners per element within the
 * cutoff plus a skin of FB_SKIN cutoffs */
constexpr int FB_NBR_MAX = 64;
constexpr float FB_SKIN = 0.25f;
/* Force pass with a wavefront per marker: its platelet's elements are taken
 * 64 at a time (a run of the index order), and runs whose bounding box is
 * beyond the Morse cutoff are skipped; a lane tests a box, so a platelet has
 * at most 64 runs */
constexpr int MORSE_RUN = 64, MORSE_RUNS_MAX = 64;
/* lanes of the per-body workgroups (force pass, second spreading pass) */
constexpr int BODY_THREADS = 1024;
/* Markers in chunks from which spreading is staged through LDS by default: when
 * the force launch could spread as well, and when spreading is a launch of its
 * own anyway.  us per step, direct / staged, on 160x96x96 FP32: fused 1536
 * markers 60.5 / 62.8, 2048 62.0 / 64.4, 3000 66.9 / 62.6, 6000 77 / 66; own
 * launch 1024 62.0 / 62.7, 1536 65.2 / 63.6, 2048 67.7 / 65.3.  Scattered
 * markers do not count: nothing of them is staged, and they take a wavefront
 * each in the direct form (fibrin nodes alone, 160^3 FP16: 3000 118 / 134,
 * 10 000 162 / 211, 30 000 265 / 302, 60 000 257 / 291; 30 000 beside 2000
 * elements 180 / 212; 100 000 in 256^3 605 / 616, 600 000 in 448^3 3591 / 3529). */
constexpr int IB_STAGED_MIN = 2560, IB_STAGED_MIN_ALONE = 1280;
/* ... and from which it goes by body when the model has compact platelets. */
constexpr int SPREAD_BODY_MIN = 1 << 20;
/* Marker count from which the forces take 4 lanes per marker in bin order, or
 * the pass by body where it applies (below it, a wavefront per marker).  us
 * per step, wavefront / by body: 31 200 markers 187 / 224, 46 800 246 / 259,
 * 83 200 442 / 441, 156 000 497 / 477.  Platelets of 5000 elements, too long
 * for the runs, wavefront / 4 lanes: 40 000 markers 157 / 195, 60 000 216 / 233.
 * Without platelets a marker has a few links and no Morse partners for its
 * lanes: clots of 34 000 fibrin nodes 122 / 113, 50 000 146 / 133, 64 000
 * 173 / 157 (below, few wavefronts are left: the same to 5 %). */
constexpr int FORCES_SORTED_MIN = 65536, FORCES_SORTED_MIN_FIBRIN = 32768;
/* Marker count from which the force pass by body is taken without being asked
 * for (where the library does not take a wavefront per marker), and
 * pfg_download_cells leaves the elements of such models out. */
constexpr int BY_BODY_MIN = 32768;
/* Receptor count up to which the cell-list/bond launch resolves the bonds
 * itself (its last workgroup takes them all). */
constexpr int RESOLVE_IN_GATHER_MAX = 2048;
/* Marker count below which the counting launch adds the scan's span totals
 * (above it the counting wavefronts meet on few spans and a reduction
 * launch is cheaper). */
constexpr int SPAN_COUNT_MAX = 32768;
/* Both copies of the populations together, up to which the LB update stores
 * through the caches, and up to which each XCD takes a contiguous range of
 * blocks by default (so do single lattices from LB_LARGE_CELLS up); the
 * figures are at the launcher in lb.hip. */
constexpr int64_t LB_CACHED_MAX_BYTES = (int64_t)320 << 20;
constexpr int64_t LB_XCD_MAX_BYTES = (int64_t)256 << 20;
constexpr int64_t LB_LARGE_CELLS = (int64_t)1 << 27;
/* Kind of a block of 64 cells: no solid cell and no solid upstream
 * neighbour, some, or solid cells only. */
constexpr int BLOCK_FLUID = 0, BLOCK_MIXED = 1, BLOCK_SOLID = 2;
/* Cell lists a handle holds: the empty ones of the load, none (a step that
 * reads no list keeps none), those of the markers other than elements on the
 * coarse grid (a step's own have bin_scatter, which the bonds read, but not
 * its order in bin_items), those of every marker. */
enum { LISTS_AS_LOADED, LISTS_NONE, LISTS_COARSE_UNORDERED, LISTS_COARSE, LISTS_FULL };
/* Device counters of a handle (Markers::counters). */
constexpr int N_COUNTERS = 16;
/* Morse pairs whose distance lies within this of the cutoff are counted: a
 * rounding difference can switch them. */
constexpr float MORSE_EPS_R = 1e-4f;

/* Everything the fused LB kernel needs, passed by value. */
struct LBArgs {
  const void *fin;        /* post-collision state of the previous step      */
  void *fout;             /* post-collision state of this step              */
  float *aux;             /* [3][plane]: IB force in, zeroed once read      */
  float4 *vel;            /* per cell (ux, uy, uz, 0): IB velocity out       */
  int64_t plane;          /* stride between the components of aux            */
  const int32_t *tile_stamp; /* per tile: the last step that spread into it */
  const uint8_t *solid;   /* nullptr when there are no solid cells          */
  const uint32_t *bbmask; /* per cell: bit d = upstream of d is solid,
                             bit 31 = cell is solid; nullptr without flags  */
  const int32_t *block_kind; /* per block of 64 cells: BLOCK_FLUID, ...;
                             nullptr without flags                          */
  const int64_t *halt;    /* nonzero *halt: leave the lattice unchanged
                             (run halted at detach); nullptr: never          */
  const int32_t *row_stamp; /* per block of 64 cells: the last step whose IB
                             stencils touch the block                        */
  const int64_t *step;    /* the current step (device counter)              */
  int nx, ny, nz;
  uint32_t ncell;         /* cells of the lattice                             */
  float inv_nx, inv_ny;   /* 1 / nx, 1 / ny                                   */
  int64_t block0;         /* first workgroup of this lattice in a batched
                             launch                                          */
  int tnx, tny;           /* tiles per axis                                   */
  int periodic[3];
  int wall_moves;         /* some wall_term is not zero                       */
  float omega;            /* 1/tau                                           */
  float guo;              /* 1 - 1/(2 tau)                                   */
  float g[3];             /* body force                                      */
  float scale, inv_scale; /* FP16 deviation scale                            */
  /* collision constants for the three weight classes (rest, axis, diagonal),
   * in storage units: ws = w * scale, gB = 9 guo ws, gD = 3 guo ws */
  float keep;             /* 1 - omega                                       */
  float om15, om45, om3, guo3; /* 1.5 omega, 4.5 omega, 3 omega, 3 guo        */
  float ws[3], gB[3], gD[3];
  /* 6 w_d (c_d . u_wall) for [axis][0 lower, 1 upper][d] */
  float wall_term[3][2][Q];
  int zvel;               /* z faces are Zou/He velocity faces                */
  int xcd_rows;           /* 1: each XCD takes a contiguous range of rows     */
  float zvel_u[2][3];     /* their velocities (z = 0, z = nz-1)               */
};

/* Lattice side of the IB coupling for one lattice of a batch (a handle
 * with one lattice has one). */
struct MLat {
  float *aux;             /* the lattice's cells of the [3][plane] force      */
  const float4 *vel;      /* the lattice's cells of the velocity field        */
  int32_t *tile_stamp;    /* the lattice's tiles                              */
  uint64_t *tile_owner;   /* the lattice's tiles (body spreading claims)       */
  int tnx, tny, tnz;
  int nx, ny, nz;
  int periodic[3];
  int nb[3];              /* cell-list bins per axis                          */
  int bin0;               /* first global bin of the lattice                  */
  int nbc[3];             /* coarse bins per axis (lists without elements)    */
  int binc0;              /* first global coarse bin of the lattice           */
  int64_t tile0;          /* first global tile of the lattice                 */
  int32_t *row_stamp;     /* the lattice's blocks of 64 cells (nullptr: unused) */
  /* counter-RNG key of the lattice's own draws (bonds, noise): its seed and
   * lattice-local receptor and marker indices, so that a lattice of a batch
   * draws what it draws in a handle of its own */
  uint64_t seed;
  int32_t rec0;           /* first receptor of the lattice                    */
  int32_t marker0;        /* first marker of the lattice                      */
};

/* Tile-gather spreading: a marker's first stencil node (w = 1: IB-coupled),
 * its kernel weights along x, y, z and its force, per cell-list slot. */
struct SpreadRec {
  int4 o;
  float4 wx, wy, wz, f;
};

/* Marker-side device arrays. */
struct Markers {
  int n = 0;
  int32_t *minst = nullptr;      /* lattice of each marker (batches only)    */
  float *x = nullptr, *y = nullptr, *z = nullptr;
  float4 *pos4 = nullptr;        /* x, y, z, Morse tag per marker, this step */
  float *vx = nullptr, *vy = nullptr, *vz = nullptr;
  float *fx = nullptr, *fy = nullptr, *fz = nullptr;
  /* PFG_SEM_BBK: the fluid velocity interpolated at each marker (the
   * element's own velocity stays in vx, vy, vz) */
  float4 *uib = nullptr;
  int32_t *kind = nullptr, *body = nullptr;
  /* platelets */
  int n_plt = 0;
  int32_t *plt_elem_start = nullptr, *plt_tri_start = nullptr;
  int n_tri = 0;
  int32_t *tri = nullptr;        /* 3*n_tri */
  double *tri_S0 = nullptr, *tri_S = nullptr, *tri_V = nullptr;
  /* per (triangle, vertex slot) 3t+s: area gradient -(L_s x n)/2 and the
   * local area strain (S - S0)/S0; per triangle: (x1-x0) x (x2-x0), the
   * volume gradient at any of its vertices (written each step) */
  float4 *tri_g = nullptr, *tri_a2 = nullptr;
  double *plt_S0 = nullptr, *plt_V0 = nullptr, *plt_S = nullptr, *plt_V = nullptr;
  int32_t *plt_lowest = nullptr; /* lowest element per platelet             */
  /* CSR marker -> incident triangles (value = 3 * triangle + vertex slot) */
  int32_t *m2t_start = nullptr, *m2t = nullptr;
  /* membrane bending: triangles as 6-node elements (3 vertices, 3 edge
   * midpoints), ordered vertex rings, node normals and mean curvature */
  int bend = 0;                  /* the chain runs each step                 */
  int n_tedges = 0;              /* edges of the triangles (midpoint nodes)  */
  int32_t *tri_edge = nullptr;   /* 3 per triangle: edges v0v1, v0v2, v1v2   */
  int32_t *edge_tri = nullptr;   /* 2 per edge: 3 * triangle + slot, or -1   */
  int32_t *ring_start = nullptr, *ring = nullptr; /* empty ring: open vertex */
  double *vn = nullptr, *en = nullptr; /* unit normals of vertices, edges     */
  double *tri_n = nullptr;       /* unit normals of the triangles            */
  double *km = nullptr;          /* mean curvature per vertex                */
  /* CSR marker -> mesh-edge partners with rest length */
  int n_edges = 0;
  int32_t *m2e_start = nullptr, *m2e_nbr = nullptr;
  float *m2e_l0 = nullptr;
  /* receptors */
  int n_rec = 0;
  int32_t *rec_tri = nullptr;
  float *rec_r1 = nullptr, *rec_r2 = nullptr;
  int32_t *rec_bond = nullptr;   /* ligand id or -1                          */
  int32_t *rec_cand = nullptr;   /* candidate ligand this step or -1         */
  int32_t *rec_release = nullptr;/* 1 if the bond ruptures this step         */
  float *rec_force = nullptr;    /* 3*n_rec force on the receptor            */
  float *rec_w = nullptr;        /* 3*n_rec share of that force per vertex   */
  int32_t *m2r_start = nullptr, *m2r = nullptr; /* marker -> (receptor*3+slot) */
  /* ligands */
  int n_wall_lig = 0;
  int fibrin_lig = 0;
  int n_lig = 0;                 /* n_wall_lig + n (fibrin node ids)         */
  float *lig_x = nullptr, *lig_y = nullptr, *lig_z = nullptr;
  int32_t *lig_owner = nullptr;  /* receptor or -1                           */
  int32_t *lig_claim = nullptr;  /* lowest claiming receptor or INT_MAX      */
  /* static ligands binned on the cell-list grid: lg_start[nbins+1] */
  int32_t *lg_start = nullptr, *lg_items = nullptr;
  float4 *lg_pos = nullptr;       /* per lg_items slot: x, y, z, ligand index */
  float4 *rec_pos = nullptr;      /* receptor positions of this step, lattice
                                     index in .w (int bits)                   */
  /* fibrin links, CSR marker -> (partner, rest length) */
  int n_links = 0;
  int32_t *m2l_start = nullptr, *m2l_nbr = nullptr;
  float *m2l_l0 = nullptr;
  /* cell list */
  int nb[3] = {1, 1, 1};
  int64_t nbins = 0;
  int64_t nbinsc = 0, scan_blocks_c = 0; /* the coarse grid                  */
  int32_t *bin_count = nullptr, *bin_start = nullptr, *bin_items = nullptr,
          *marker_bin = nullptr, *marker_slot = nullptr;
  int32_t *bin_scatter = nullptr; /* items in scatter (atomic slot) order    */
  float4 *sorted_pos = nullptr;   /* per bin_items slot: x, y, z, Morse tag  */
  int32_t *scan_partials = nullptr; /* sums of SCAN_SPAN bins */
  int64_t scan_blocks = 0;
  /* IB chunks: chunk k holds the markers chunk_items[chunk_start[k] ..
   * chunk_start[k+1]-1], at most IB_CHUNK markers of one body (a platelet,
   * or the markers outside platelets) of one lattice that lay close together
   * at load time; the n_direct markers chunk_items[chunk_start[n_chunks] ..]
   * were too far apart and are spread directly */
  int n_chunks = 0, n_direct = 0;
  int n_chunk_items = 0;         /* markers in the chunks (the direct list follows) */
  int32_t *chunk_start = nullptr;
  int32_t *chunk_items = nullptr;
  /* per chunk the marker whose periodic image places its stencils: the
   * first marker of its platelet (body spreading), else its own first */
  int32_t *chunk_ref = nullptr;
  /* tile-gather spreading: the tiles this step's stencils meet, listed once
   * each (global tile index); tile_count[0] tiles listed, [1] workgroups of
   * the gather launch done (the last one empties the list).  Usable when
   * every periodic axis is at least twice the tile's extent along it */
  int32_t *tile_list = nullptr;
  int32_t *tile_count = nullptr;
  /* body spreading: bodies (compact platelets: body_range[4g .. 4g+3] =
   * their markers m0..m1-1 and chunks c0..c1-1; every marker of a body is
   * in one of its chunks), chunk_body (the body of each chunk, -1: none),
   * the chunks' scratch boxes (chunk_sum: 6 x IB_BOX_CELLS floats per chunk;
   * chunk_info: the box's first node and extents per chunk, extent 0: not
   * written this step), and the chunks and direct list of every marker
   * outside the bodies (the chunk lists' format); per tile of all
   * lattices, the step and the body that claimed it alone this step
   * (OWNER_SHARED: more than one contributor), written by the force launch
   * and read by spreading */
  int n_bodies = 0;
  int32_t *body_range = nullptr;
  int32_t *chunk_body = nullptr;
  float *chunk_sum = nullptr;
  int4 *chunk_info = nullptr;
  int n_rchunks = 0, n_rdirect = 0, n_ritems = 0;
  int32_t *rchunk_start = nullptr, *rchunk_items = nullptr;
  uint64_t *tile_owner = nullptr;
  int32_t *body_spread = nullptr;   /* per body: the last step it spread in  */
  int32_t *body_fallback = nullptr; /* per body: the last step one of its
                                       chunks spread with atomics            */
  /* force pass by body: bodies of at most FB_MAX markers (marker ranges
   * fbody_range[2g], fbody_range[2g+1]) when every body's elements form one
   * run of indices, and every other marker (frest_items) */
  int n_fbodies = 0, n_frest = 0;
  int fb_all_elements = 0;       /* every element is in one of those bodies  */
  int32_t *fbody_range = nullptr, *frest_items = nullptr;
  /* per marker: the positions of its body's last list build (NaN: build),
   * its list length and its partners (body-local indices, partner q of
   * marker i at fb_nbr[q * n + i]) */
  float4 *fb_ref = nullptr;
  int16_t *fb_nlen = nullptr;
  int16_t *fb_nbr = nullptr;
  int32_t *fb_done = nullptr;    /* per body: the step whose forces the build
                                    kernel summed (its lists overflowed)     */
  /* runs of MORSE_RUN elements of a platelet: per run its markers
   * [run_range[2r], run_range[2r+1]) and this step's bounding box; per marker
   * the first run of its platelet and their number (0: not an element).
   * n_runs = 0 when some platelet's elements are no single run of indices,
   * or too many */
  int n_runs = 0;
  int32_t *run_range = nullptr;
  float4 *run_lo = nullptr, *run_hi = nullptr;
  int2 *marker_runs = nullptr;
  SpreadRec *spread_rec = nullptr; /* per cell-list slot: the marker's record */
  int tile_gather_ok = 0;
  /* platelet-platelet contact: per platelet pair (lo * n_plt + hi) the best
   * proposal (distance bits << 32 | element of the lower platelet), and the
   * pairs proposed this step */
  uint64_t *contact_slot = nullptr;
  int32_t *contact_list = nullptr;
  /* counters (N_COUNTERS): [0] total bonds, [1] detached, [2] near-threshold
   * lo, [3] hi, [4] events lo, [5] events hi, [6] the step index recorded by
   * the first launch of the step, [7] platelet pairs in contact this step,
   * [8] Morse pair visits within MORSE_EPS_R of the cutoff, [9] contact
   * candidates beyond the per-element platelet slots */
  int64_t *counters = nullptr;
  int32_t *ticket = nullptr;      /* workgroups of the gather launch done       */
  int64_t *detach_step = nullptr;
  int64_t *d_step = nullptr;
};

/* Host-side description of one lattice of a handle. */
struct Inst {
  pfg_params p{};          /* lattice and fluid fields apply per lattice     */
  int64_t N = 0;           /* cells                                          */
  int64_t cell0 = 0;       /* first cell in the concatenated cell fields     */
  int64_t fblk0 = 0;       /* first block in the population arrays            */
  int64_t nfblk = 0;       /* its blocks of 64 cells                          */
  int tnx = 0, tny = 0, tnz = 0;
  int64_t ntiles = 0, tile0 = 0;
  int nb[3] = {1, 1, 1};
  int64_t nbins = 0, bin0 = 0;
  int nbc[3] = {1, 1, 1};
  int64_t nbinsc = 0, binc0 = 0;
  int64_t lb_blocks = 0, lb_block0 = 0; /* workgroups in the batched LB launch */
  int32_t rec0 = 0, marker0 = 0;  /* first receptor and marker of the lattice */
};

}  // namespace pfg

struct pfg_handle {
  pfg_params p{};
  int device = 0;
  hipStream_t stream = nullptr;
  int64_t N = 0, plane = 0;
  int esize = 4;
  /* populations, blocked: direction d of cell i = x + nx*(y + ny*z) at
   * ((i/64)*19 + d)*64 + i%64 */
  void *f[2] = {nullptr, nullptr};
  int cur = 0;
  /* IB coupling fields: spreading adds the force of a step into aux and
   * stamps the 4x4x4 tiles it touches with the step; the LB update reads
   * the force of stamped tiles, zeroes it there for the next step and
   * writes the velocity the interpolation reads into vel.  The force is
   * kept as three planes, so the three atomic adds of a node go to three
   * cache lines (atomics to one line are serialised); the velocity is one
   * float4 per cell, so a gather of a node reads one line */
  float *aux = nullptr;
  float4 *vel = nullptr;
  int32_t *tile_stamp = nullptr;
  int tnx = 0, tny = 0, tnz = 0;
  int64_t ntiles = 0;
  uint8_t *solid = nullptr;
  uint32_t *bbmask = nullptr;  /* per-cell bounce mask built from solid        */
  int32_t *block_kind = nullptr; /* per block of 64 cells, from the masks      */
  double *red = nullptr;       /* reduction partials                        */
  int64_t red_blocks = 0;
  int lb_cpt = 1;              /* LB launch: cells (blocks in a row) per lane */
  int lb_xcd_rows = 0;         /* LB launch: contiguous rows per XCD        */
  pfg::Markers m;
  bool model_loaded = false;
  bool in_step = false;        /* launches of a whole step (not of a stage)     */
  /* what the last steps or CELLS stage left of the positions in pos4: which
   * cell lists, and whether the runs' boxes */
  int lists_kept = pfg::LISTS_AS_LOADED;
  bool boxes_kept = false;
  bool fluid_only = false;
  bool halt_on_detach = false; /* steps after the detach test fired change nothing */
  int ib_staging = 0;          /* spreading: 0 auto, 1 LDS-staged chunks, 2 direct */
  int forces_lanes = 0;        /* lanes per marker in the forces: 0 auto, 1, 4, 16, 64 */
  int forces_body = 0;         /* force pass by body: 0 auto, 1 on, 2 off     */
  /* LB rows away from IB stencils update on stream2 while the marker
   * pipeline runs; the rows the stencils touch update after spreading.  Off
   * by default: on MI355X the LB launch saturates HBM and the CU slots, and
   * the latency-bound marker kernels slow down as much as they overlap. */
  bool overlap = false;
  hipStream_t stream2 = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  int32_t *row_stamp = nullptr;    /* per block of every lattice            */
  int64_t h_step = 0;
  /* lattices: one, or a batch stepped together */
  int K = 1;
  std::vector<pfg::Inst> inst;
  pfg::LBArgs *d_lbargs[2] = {nullptr, nullptr}; /* per starting copy of f, [K] */
  int32_t *lb_block_inst = nullptr;              /* batched LB: lattice per block */
  int64_t lb_blocks = 0;
  /* batched LB: 1 = one persistent launch of resident workgroups taking the
   * table's tasks from a work queue (lb_queue: next task, workgroups done) */
  int lb_persistent = 0;
  uint32_t *lb_queue = nullptr; /* LB_QUEUES range counters, then the done count */
  pfg::MLat *d_lats = nullptr;                   /* [K] */
  int64_t *d_tile0 = nullptr;                    /* [K+1] first tile per lattice */
  std::vector<int32_t> marker0;                  /* [K+1] first marker per lattice */
  bool use_graph = true;
  /* [starting copy of f][0: one step, 1: GRAPH_CHUNK steps] */
  hipGraphExec_t graphs[2][2] = {{nullptr, nullptr}, {nullptr, nullptr}};
  bool graph_valid = false;
  size_t dev_bytes = 0;
};

namespace pfg {

/* lb.hip; k selects a lattice of the handle */
void make_lb_args(const pfg_handle *h, int k, int cur, LBArgs *a);
/* the block order a handle starts with (pfg_set_lb_xcd_rows) */
int lb_default_xcd_rows(const pfg_handle *h);
hipError_t launch_lb(pfg_handle *h);
/* part 1: blocks no IB stencil touches this step (on stream s); part 2: the
 * blocks they touch, with the IB force (then the copies of f alternate) */
hipError_t launch_lb_part(pfg_handle *h, int part, hipStream_t s);
hipError_t launch_bbmask(pfg_handle *h, int k);
/* per_z: the inputs hold one value per z-plane of lattice k */
hipError_t launch_init_eq(pfg_handle *h, int k, const float *rho, const float *ux,
                          const float *uy, const float *uz, bool per_z = false);
hipError_t launch_convert_f(pfg_handle *h, float *f_out_or_null,
                            const float *f_in_or_null);
hipError_t launch_conservation(pfg_handle *h, int k, double out[4]);
/* persistent batched LB launch: ranges (one per XCD) and blocks per grab */
constexpr int LB_QUEUES = 8;
constexpr int LB_QUEUE_GRAB = 16;
/* pfg_download_fields_noalloc: staging in a fixed device array of
 * FIELDS_SCRATCH_FLOATS floats per device (no allocation) */
constexpr int64_t FIELDS_SCRATCH_FLOATS = PFG_FIELDS_SCRATCH_FLOATS;
constexpr int FIELDS_SCRATCH_MAX_DEVICES = 64;
/* the array's device address on `device` (looked up on the first call) */
hipError_t fields_scratch_setup(int device, float **out_or_null);
/* rho, ux, uy, uz of a single lattice to host (any may be NULL), window of
 * whole z-planes at a time through the fixed array */
hipError_t download_fields_noalloc(pfg_handle *h, float *const host[4]);

/* rho, ux, uy, uz of the cells [lo, hi) of lattice k, into windows of hi - lo
 * values (nullptr: not wanted); solid cells read 0 */
hipError_t launch_lb_fields_window(pfg_handle *h, int k, uint32_t lo, uint32_t hi,
                                   float *const win[4]);

/* frames.hip: to host arrays through pinned memory.  hipErrorOutOfMemory: no
 * pinned buffer could be had, nothing was written. */
struct Piece {
  void *dst;        /* host                  */
  const void *src;  /* device                */
  size_t bytes;     /* a multiple of 4; 0: skipped */
};
hipError_t fetch_pieces(pfg_handle *h, const Piece *pieces, int n);
hipError_t fetch_fields(pfg_handle *h, int k, float *const host[4]);
/* the counters, the detach step and the step index, after the work enqueued
 * so far */
hipError_t fetch_report(pfg_handle *h, int64_t out[N_COUNTERS + 2]);
/* every handle holds a reference; the last one frees the pinned buffers */
void frames_ref();
void frames_unref();

/* markers.hip: fused marker-side launches, each with the roles it runs */
void fill_mlat(const pfg_handle *h, int k, MLat *L);
hipError_t launch_begin(pfg_handle *h, bool clear, bool count, bool geometry = false);
/* the cell lists and run boxes of the positions the last step started from */
hipError_t launch_cells_again(pfg_handle *h);
/* the bending chain's normals and curvature, after the triangle terms */
hipError_t launch_bend(pfg_handle *h);
hipError_t launch_scan(pfg_handle *h);
hipError_t launch_place(pfg_handle *h, bool scatter, bool geometry);
/* resolved != nullptr: resolve the bonds in the same launch when there are
 * few receptors (*resolved says whether it did) */
hipError_t launch_gather(pfg_handle *h, bool sort, bool sums, bool decide,
                         bool *resolved = nullptr);
hipError_t launch_resolve(pfg_handle *h);
/* spread = true: the force pass also spreads (only when forces_can_spread) */
hipError_t launch_forces(pfg_handle *h, bool spread = false, bool sums = false);
/* whether the cell lists that pfg_download_cells gives hold the elements (else
 * only the other markers) */
bool bin_elements(const pfg_handle *h);
/* whether a step's own lists do, whether a step needs lists at all, and
 * whether its platelet sums can go with the force launch */
bool step_bin_elements(const pfg_handle *h);
bool step_lists(const pfg_handle *h);
/* whether stage s reads cell lists or run boxes */
bool stage_reads_lists(const pfg_handle *h, int s);
/* whether a step writes the runs' boxes */
bool by_runs(const pfg_handle *h);
bool sums_with_forces(const pfg_handle *h);
bool forces_can_spread(const pfg_handle *h);
hipError_t launch_spread(pfg_handle *h);
hipError_t launch_move(pfg_handle *h, bool interp, bool update);

}  // namespace pfg

#endif
