// step_args.h -- argument blocks of the time-step kernels.  One block per
// box: passed by value for a single box, or gathered into per-case tables in
// device memory when one grid advances several boxes (ensemble engine).
#pragma once
#include "internal.h"

namespace mfc {

struct ForceArgs {
  const double* gcur;   // forcing table of the current step (may be null)
  const double* gmac;   // forcing table captured by the last macrovar (may be null)
  const double* phx;    // (cos,sin)(2 pi m / nx)
  double bfx, bfy, bfz; // uniform body force
};

// Arguments of the collide kernel (fluid.hip).
struct CollideArgs {
  const void* A;
  void* B;
  const uint32_t* mask;
  Grid g;
  CollideConsts k;
  ForceArgs fa;
  double* rho;
  const double *ux, *uy, *uz;
  int arr;   // batched launches: conserved moments from the arrays (else recomputed)
};

struct PGeom {
  int nx, ny, nz, walls_y;
  double rad, radp2, r2;
  // (r + 1.5)^2: a node farther than r + 1.5 from the centre is neither
  // solid nor has a link, since every lattice vector is shorter than 1.5
  // (the margin over sqrt(2) dwarfs any rounding of the squared distances)
  double rlink2;
  // z planes per segment (Particles::slab)
  int slab;
  FastDiv dseg;   // division by the segments per particle
};

struct FillArgs {
  const double *ypglbp, *wp, *wpp, *omgp, *omgpp;
  const int32_t* isn_old;
  const uint32_t *mask_new, *mask_old;
  const uint32_t* sol_old;    // solid lists of the previous map build
  const int32_t* sol_cnt_old;
  int seg_cap;
  double rad, rho0, ww0, ww1, ww2;
  int32_t* status;
};

// Boundary links: segment b's are the cnt[b] entries from b * cap on.
struct LinkSlots {
  uint32_t* node;
  uint8_t* dir;
  double* alpha;
  int32_t* cnt;
  int cap;
};

// Contact links (node solid for another sphere) of the current build.
struct ContactArgs {
  LinkSlots lk;
  const uint32_t* mask;
  uint64_t* ct_list;    // (particle << 40) | link
  int32_t* ct_count;    // cleared by the links scan
  int64_t ct_cap;
  FastDiv dseg;
};

// Uniform cell grid of the particle pair searches (lubrication, overlap
// check): cells at least as wide as the longest pair range, at most
// kCellCap particles each.  cnt == nullptr: all pairs are searched.
struct CellArgs {
  int32_t* cnt;
  int32_t* list;   // kCellCap slots per cell
  int ncx, ncy, ncz;
};

struct LubArgs {
  CellArgs cells;
  double mingap, fpc, stf0, stf1;
  double mingap_w, stf0_w, stf1_w;   // sphere-wall lubrication (walls_y)
  double* flubp;
};

struct MoveArgs {
  double *yp, *ypglb, *ypglbp, *wp, *wpp, *omgp, *omgpp, *fHIp, *flubp, *torqp, *forcep, *forcepp,
      *torqpp, *dwdt, *domgdt, *thetap;
  double volp, rhog, amp, aip;
  double bfx, bfy, bfz;   // fluid body force (acts on the displaced volume)
  double pfx, pfy, pfz;   // force per unit sphere volume on the spheres only
};

struct ScanArgs {
  const double* ypglb;
  int np;
  int nseg;
  int seg_cap;
  PGeom G;
  int32_t* isn;
  uint32_t* mask;
  uint32_t* sol_list;
  int32_t* sol_cnt;
  LinkSlots lk;
  int32_t* ct_count;
  int ovl;
  int istep;
  int32_t* status;
  CellArgs cells;
};

// Arguments of the bounce-back grid (nlub lubrication blocks, the link
// segments, the map-clearing blocks and those of the pair-search cells) and of
// its pre-pass grid (nct blocks for the contact links).
struct BounceArgs {
  void* A;
  const void* old;              // the field before the collide, if the other buffer holds it
  Grid g;
  PGeom G;
  const uint32_t* mask;
  int nseg;
  LinkSlots lk;
  double2* lk_out;              // (f9, ff1) of the contact links
  const uint64_t* ct_list;      // contact links: (particle << 40) | link
  const int32_t* ct_count;
  int64_t ct_cap;
  const double* ypglb;
  const double* wp;
  const double* omgp;
  double ww1;
  double ww2;
  double* seg_ft;
  int32_t* status;
  int nsegs;
  int np;
  int split;                    // bounce-back work units per segment (seg_ft has nsegs * split)
  int nct;                      // contact blocks of the pre-pass grid
  int ref_order;                // contact links in the reference's in-place order (one block)
  OrderEntry* ord;              // its table (ord_cap entries) and the current owner map
  int64_t ord_cap;
  const int32_t* isn;
  int nlub;                     // lubrication blocks (fused step, else 0)
  LubArgs lub;
  int seg_cap;                  // map clearing (clr_* of map buffer map_cur ^ 1)
  const uint32_t* clr_list;
  const int32_t* clr_cnt;
  int32_t* clr_isn;
  uint32_t* clr_mask;
  int nclr;                     // blocks of the map clearing, then of the cells'
  int ncell;                    // pair-search cells to clear (0: none)
  int32_t* clr_cells;
};

struct MoveKArgs {
  MoveArgs m;
  int np;
  int first;
  int wrap;
  PGeom G;
  int32_t* status;
  const double* seg_ft;   // non-null: fHIp / torqp are first summed from the segments
  int nseg;
  CellArgs cells;         // cnt non-null: (cleared) cells to enter the new centres in
};

// Arguments of the refill grid: nfill blocks of beads_filling (segments of the
// previous build), then nct blocks listing contact links.
struct FillKArgs {
  void* A;
  Grid g;
  FillArgs fa;
  ContactArgs ct;
  int nfill, nct;
};

// ---- argument builders (fluid.hip, particles.hip) ----
CollideArgs collide_args(Ctx& c);
ScanArgs scan_args(Ctx& c, int target, int ovl, int istep);
size_t scan_lds(const Ctx& c);   // dynamic LDS of the links scan
// bb_blocks: the bounce-back grid; pre_blocks: the pre-pass grid
BounceArgs bounce_args(Ctx& c, bool fused, int nct, int* bb_blocks, int* pre_blocks);
MoveKArgs move_args(Ctx& c, int first, int wrap, bool from_seg, int* blocks);
FillKArgs fill_args(Ctx& c, bool refill, bool contacts, int* blocks);

// ---- launches over several boxes: t = device table of the stage's argument
// blocks (one per box), off = device block offsets (nc + 1), `blocks` = off[nc]
enum Stage { SG_CONTACT, SG_BOUNCE, SG_MOVE, SG_SCAN, SG_FILL };
hipError_t launch_batched(Stage st, int prec, int walls, const void* t, const int* off, int nc,
                          int blocks, size_t lds, hipStream_t s);
// arr_any: some member's CollideArgs::arr is set
hipError_t launch_batched_collide(int prec, int walls, int bs, int remap, const void* t, const int* off,
                                  int nc, int blocks, bool arr_any, bool ntl, hipStream_t s);
size_t stage_arg_bytes(Stage st);

}  // namespace mfc
