// Device-side data layout and kernel launchers of the ARAP path (gfx950).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>

namespace md {

struct alignas(16) f4 { float x, y, z, w; };
struct alignas(32) d4 { double x, y, z, w; };

template <typename T> struct V4T;
template <> struct V4T<float> { using type = f4; };
template <> struct V4T<double> { using type = d4; };

// Per-supernode record of the block LDL^T sweeps (see Factor in md_analysis.h).
// Pointers of the device records below are in the global address space in the device pass of
// the kernels' file (md_kernels.hip defines MD_KERNELS_DEVICE), so the kernels' loads and stores
// are global (not flat) instructions: they wait on the vector memory counter alone, in issue
// order, instead of on the LDS counter as well. Host code sees plain pointers of the same size.
#if defined(__HIP_DEVICE_COMPILE__) && defined(MD_KERNELS_DEVICE)
#define MD_G __attribute__((address_space(1)))
#else
#define MD_G
#endif

struct SnDev {
    int c0, w, noff, roff;     // columns [c0, c0+w), off rows offrows[roff .. roff+noff)
    int kc, kr, uk, dstride;   // partial counts of u_s / x_s, update slots per front position,
                               //   the parent's front size (stride of u_s's partials in its slots)
    long long pc_off, pr_off;  // column-major G_s, row-major [Dinv_s; G_s]
    long long ubase, xoff;     // first update slot of the front / partial solution entries
};

// One level tile of a sweep: the supernode's record and the tile origin, so a tile is one load.
struct TileDev {
    SnDev s;
    int a, b, pad0, pad1;      // forward (r0, q0); backward (q0, p0)
};

// Device view of one mesh. All pointers are device pointers into the mesh's arena.
// Internal vertex ids: [0, nf) free vertices in solve order, [nf, n) constrained ones.
struct MeshDev {
    int n, nf, nslices, ns;
    int nslices_free;           // slices covering internal ids [0, nf)
    int F;
    long long slots;            // 64 * slice_ptr[nslices]
    const MD_G int *slice_ptr;  // nslices + 1 (64-wide slot columns)
    const MD_G int *sell_col;   // slots: neighbour internal id (self = padding)
    MD_G float *a32;            // 3 planes of slots: w_ij (p_i - p_j), FP32
    MD_G double *a64;           // 3 planes of slots, FP64
    MD_G double *w64;           // slots: cotan weight w_ij
    const MD_G int *tri;        // 3F internal ids
    MD_G double *fe_val;        // 3F half-cotangents (face edge 3f+k)
    const MD_G int *slot_fe_ptr; // slots + 1
    const MD_G int *slot_fe;    // face-edge ids feeding each slot, face order
    MD_G d4 *p;                 // rest positions (internal order)
    MD_G d4 *pp;                // current positions p'
    MD_G void *quat;            // rotations as quaternions (x, y, z, w=scalar): f4 or d4
    MD_G void *r, *z;           // residual and forward result (V4 of the solve type), nf each
    MD_G void *upart, *xpart;   // update slots of the level fronts / partial solutions (V4)
    const MD_G long long *udst; // per off-row entry of a level supernode or subtree root: its
                                //   update slot in the parent's front (partial cb: + cb * dstride)
    const MD_G int4 *rowinfo;   // per row: (first partial, stride, count, 0)
    const MD_G int4 *xloc;      // per off row entry: rowinfo of that row
    const MD_G void *pc, *pr;   // panels (float or double), forward and backward layouts
    const MD_G TileDev *ftile, *btile; // level tiles, level by level (bases in the launch tables)
    // bottom subtrees, one workgroup each (layouts in md_analysis.h, Factor)
    const MD_G int4 *sub;       // (first record, end record, height table offset, heights)
    const MD_G int *sub_h;      // first record of each (subtree, height), + a terminal per subtree
    const MD_G int4 *snode;     // supernode records, four int4 each (SubNode)
    const MD_G int2 *scp;       // forward positions: first two child update entries (LDS), overflow
    const MD_G int *sfc;        // -1-terminated overflow lists of child update entries
    const MD_G int2 *sbo;       // backward off-row sources
    int nsub;                   // bottom subtrees (their rows' x is added to p' by k_sub_bwd)
    const MD_G int4 *srow;      // two per subtree: (first row, rows, first forward position,
                                //   positions), (first backward off row, off rows, 0, 0)
    const MD_G int *sfi;        // per free row of a subtree: its forward position in LDS
    int nlrows;                 // rows of level-swept supernodes, increasing
    const MD_G int *lrows;      //   (their residual: extra blocks of k_sub_fwd; x summed from the
                                //   partials and added to p': extra blocks of k_sub_bwd)
    MD_G double *energy_part;   // one partial sum per 256 vertices
    // Jacobi-PCG alternative to the triangular sweeps (solve type vectors, nf entries)
    MD_G float *w32;            // slots: cotan weights in FP32
    MD_G void *diag;            // nf: L_ii = sum_j w_ij (solve type scalar)
    MD_G void *cg_x, *cg_p;     // correction, direction (V4)
    MD_G void *cg_v;            // 5 vectors (V4): r (second buffer; the first is r), w and s (two each)
    MD_G void *cg_part;         // 4 nblk + 5 (V4): partials of (r, u) and (w, u) for two parities,
                                //   then (gamma, alpha) for two parities and the first gamma
    int nblk_free;              // 256-vertex blocks covering [0, nf)
    double pcg_tol2;            // stop (freeze) when r.z <= tol^2 * (r.z)_0, per coordinate
};

// Device numeric factorization (multifrontal, FP64): per supernode record (stored by height, so a
// workgroup's is one load) and the buffers.
struct FacDev {
    int c0, w, noff, roff;          // columns, off rows (offrows[roff ..], rel[roff ..])
    int cb, ce, m, pad;             // children FacArgs::child[cb .. ce), m = w + noff
    long long poff, soff, toff, uoff;  // the front's first w columns (m x w), their second workspace
                                       // (off rows, noff x w; pivot rows, w x w), update matrix (noff x
                                       // noff); all column-major
    long long pc_off, pr_off;       // solve-precision panels of the sweeps
};

// A child as its parent's assembly reads it: rows, their map in rel, update matrix.
struct FacChild {
    int noff, roff;
    long long uoff;
};

// Words of the factorization that start at zero: partial maxima of |L_ii| (256 bytes apart: atomics on
// one line follow one another), then the flag.
constexpr int kFacMaxima = 8, kFacMaxStride = 32, kFacWords = kFacMaxima * kFacMaxStride + 1;
struct FacArgs {
    const MD_G FacDev *sn;          // by height
    const MD_G FacChild *child;
    const MD_G int *offrows, *rel;
    const MD_G int *slice_ptr, *sell_col;
    const MD_G double *w64;         // cotan weights over the one-ring slots
    int nf;
    MD_G double *P, *S, *T, *U, *diag;
    MD_G unsigned long long *amax;  // max |L_ii| as the bits of a non-negative double, in kFacMaxima parts
    MD_G int *flag;                 // 1: a pivot block is not positive definite; 2: structure
    MD_G void *pc, *pr;             // the sweeps' panels (float or double), written in the solve
    int solve64;                    //   precision (1: double)
    unsigned long long *stamp;      // clock at the first height (may be null)
};

// A set of meshes processed by one launch. Block b belongs to mesh k where
// prefix[k] <= b < prefix[k+1]; `meshes` and `prefix` are device arrays.
struct LaunchSet {
    const MD_G MeshDev *meshes;
    const MD_G int *prefix;
    int nactive;
    const MD_G int *bmesh;      // optional: mesh of every block (static batches), else a binary search
    const MD_G int *tbase;      // per mesh: first tile of the launch's level (level sweeps), else 0
    const MD_G TileDev *tiles;  // one-mesh level launches: the level's first tile (else null)
};

// Launchers (grid = total blocks of the launch, from the host-side prefix table).
void launch_cotan_face(hipStream_t s, LaunchSet L, int blocks);
// One mesh, a block per slice; diag, amax: L_ii of the free vertices and their maxima (may be null).
void launch_cotan_slot(hipStream_t s, LaunchSet L, int blocks, double *diag, unsigned long long *amax);
void launch_local(hipStream_t s, LaunchSet L, int blocks, bool fp64);
void launch_residual(hipStream_t s, LaunchSet L, int blocks, bool fp64);
void launch_fwd(hipStream_t s, LaunchSet L, int blocks, int level, bool fp64);
void launch_bwd(hipStream_t s, LaunchSet L, int blocks, int level, bool fp64);
// Bottom-subtree sweeps, one workgroup per subtree: LDS for the largest subtree's supernode records,
// heights, forward positions, backward vector entries and backward off rows. block: kSubBlock threads
// where the launch's subtrees are at most kSubFew (at most four workgroups per CU, so their chain
// counts), else fewer: 64 forward with the residual (its registers allow three wavefronts per
// SIMD), 128 forward without it and backward. Measured, 64 / 128 / 256 threads: 91 subtrees (FP32) 17.2 /
// 12.5 / 11.1 us forward with the residual, 18.8 / 12.4 / 10.2 backward; 612 (FP32) 18.7 / 14.2 / 15.1 and
// 20.8 / 14.8 / 12.2; 2,825 (FP64) 40 / 42 / 63 and 38 / 31 / 34; a batch's 7,413 (FP32, without the
// residual) 38 / 34 / 47 and 57 / 59 / 80.
// Launches over several meshes are split by LDS class (subtree_classes), since every workgroup of a launch
// gets the LDS of its largest subtree. The smallest class, whose subtrees are a supernode or two, takes 64
// threads where they are many (45 meshes of 5k to 164k vertices all at budget 128: 0.75 -> 0.68 ms per
// iteration).
// fused: the launch also forms the residual (one-mesh plans; blocks past the subtrees take
// the level rows), else k_residual ran before it.
struct SubLds {
    int block, nodes, heights, fwd, bwd, off;
};
constexpr int kSubBlock = 256;
// Level rows per workgroup of the fused launch, past the subtrees (its threads).
inline int sub_rows_fused(const SubLds &D) { return D.block == kSubBlock ? kSubBlock : 64; }
void launch_sub_fwd(hipStream_t s, LaunchSet L, int blocks, const SubLds &D, bool fused, bool fp64);
void launch_sub_bwd(hipStream_t s, LaunchSet L, int blocks, const SubLds &D, bool fp64);
void launch_energy(hipStream_t s, LaunchSet L, int blocks, bool fp64);
// A target of a served request: the device address of its vertex's p' entry and the position.
struct alignas(16) TargetEntry {
    unsigned long long addr;
    double x, y, z;
};
// *entry.addr = (x, y, z) for k entries (targets of several meshes in one launch).
void launch_scatter_entries(hipStream_t s, const TargetEntry *e, int k);
void launch_normals(hipStream_t s, LaunchSet Lf, int blocks_face, LaunchSet Ls, int blocks_slice, double *fn, d4 *out,
                    double *packed = nullptr, const int *orig = nullptr);
void launch_pcg_diag(hipStream_t s, LaunchSet L, int blocks, bool fp64);
// Jacobi-PCG in the Chronopoulos-Gear form: one launch per CG iteration (step i).
void launch_pcg_init(hipStream_t s, LaunchSet L, int blocks, bool fp64);
void launch_pcg_step(hipStream_t s, LaunchSet L, int blocks, int step, bool fp64);
void launch_pcg_apply(hipStream_t s, LaunchSet L, int blocks, bool fp64);
// Device numeric factorization: diagonal and its maximum, then per height (the `count`
// supernodes from sn[h0]) the front assembly and the block sweeps, whose last step writes D^{-1} and G
// to the solve-precision panels.
// The assembly of a height of `count` fronts of at most mm rows, at most `no` of them off rows, with
// at most `maps` = children x rows of one front: `per` workgroups per front, each `cols` columns by one
// of rch ranges of rlen rows. 64 columns, halved down to 4 (one quad for the four wavefronts) while
// the height has fewer than 4,096 workgroups: the top heights' few fronts take the largest children.
// ninv LDS entries hold the inverted row maps (as many children at a time as fit, at most 32 KB),
// nrows the front's row list.
constexpr int kAsmInv = 8192, kAsmRows = 4096, kAsmWorkgroups = 4096;
struct FacAssembly {
    int per, cols, rch, rlen, ninv, nrows;
};
inline FacAssembly fac_assembly(int count, int mm, int no, long long maps) {
    FacAssembly a;
    a.rlen = std::min(mm, kAsmInv);
    a.rch = (mm + a.rlen - 1) / a.rlen;
    a.cols = 64;
    while (a.cols > 4 && (long long)count * ((mm + a.cols - 1) / a.cols) < kAsmWorkgroups) a.cols /= 2;
    a.per = (mm + a.cols - 1) / a.cols * a.rch;
    a.ninv = (int)std::max<long long>(a.rlen, std::min<long long>(kAsmInv, maps));
    a.nrows = std::min(kAsmRows, no);
    return a;
}
// One height: assembly, then the block sweeps of its fronts, nb launches (column blocks of 64 in the
// widest pivot block) of `tiles` workgroups per front (lower 64 x 64 tiles of the largest, pivot rows
// and off rows each rounded up).
void launch_fac_height(hipStream_t s, const FacArgs &A, int h0, int count, int nb, const FacAssembly &as, int tiles);
// Fronts of m <= mm <= kFacSmallFront rows: every step of launch_fac_height for one front in one
// workgroup, without the FP64 panel workspace: of one wavefront on heights of more than kSmallManyFronts
// fronts of up to 48 rows (6,616: 50 us, with two 53; 1,380: 20 and 23), of two on heights of more than
// kSmallManyWide with larger ones (1,137: 36 us, with one 49; 685: 25, with four 33), else of four.
constexpr int kFacSmallFront = 64;
constexpr int kSmallManyFronts = 1024, kSmallManyWide = 512;
void launch_fac_small(hipStream_t s, const FacArgs &A, int h0, int count, int mm);
// Whether a height's `small` such fronts of `all` leave its general launches for the fused one: when
// they are all of it, or at least 512 and the larger part (the 164k icosphere's second and third
// heights took 116 and 114 us split, 140 and 152 together; a smaller share only adds a launch).
inline bool fac_split_small(int small, int all) { return small == all || (small >= 512 && 2 * small >= all); }
// Internal-order vectors (positions, normals) to packed xyz in original order (internal: internal
// id per original id); stamp: clock at the start (may be null).
void launch_pack_xyz(hipStream_t s, const d4 *v, const int *internal, int n, double *dst, unsigned long long *stamp);
// The packed positions of `count` meshes, n vertices in blocks of kBlock threads from `block` each.
struct PackEntry {
    const MD_G d4 *x;
    const MD_G int *internal;
    MD_G double *dst;
    int n, block;
};
void launch_pack_results(hipStream_t s, const PackEntry *e, int count, int blocks);
// Packed xyz to internal order (p and/or pp; pp takes the targets tgt, internal order, for the
// constrained ids [nf, n), and comes with identity rotations in quat).
struct UnpackArgs {
    const double *xyz;
    const int *internal;
    int n, nf;
    const double *tgt;
    d4 *p, *pp;
    void *quat;
    unsigned long long *clear, *stamp;
};
void launch_unpack_xyz(hipStream_t s, const UnpackArgs &a, bool fp64);
// Clock and *flag (may be null) to pinned host memory; nothing without a stamp.
void launch_publish(hipStream_t s, unsigned long long *stamp, const int *flag, int *out);

// Per-GPU device workspace of the non-allocating entry points (a static device array of
// kScratchBytes): its address on the current device, from hipGetSymbolAddress. Call once per
// device with that device current and use only the returned address in host code.
constexpr size_t kScratchBytes = size_t(64) << 20;
hipError_t scratch_address(void **ptr);
// Plain copy of n16 16-byte elements (counter calibration, copy bandwidth).
void launch_copy_probe(hipStream_t s, const void *src, void *dst, long long n16);

// Threads per block and work per block of each kernel (used for the prefix tables).
constexpr int kBlock = 256;
constexpr int kSlicesPerBlock = kBlock / 64;  // one 64-vertex slice per wavefront

}  // namespace md
