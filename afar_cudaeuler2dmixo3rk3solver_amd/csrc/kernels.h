// Device pointer bundle and kernel launchers of the AFAR stage pipeline.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

namespace afar {

constexpr int kCflBlocks = 1024;
constexpr int kCflGroup = 32, kCflGroups = kCflBlocks / kCflGroup;  // blocks that share a ticket counter
constexpr int kMaxSten = 20;  // largest stencil (the reference's limit, basicCUDAsolver.cpp:393-397)

template <typename R> struct VT;
template <> struct VT<double> {
    using v4 = double4;
    using v2 = double2;
};
template <> struct VT<float> {
    using v4 = float4;
    using v2 = float2;
};

// How a kernel's tiles are dealt to its blocks (xcd_tile): n tiles in 2^mlog
// chunks, chunk j the tiles [j n / 2^mlog, (j + 1) n / 2^mlog), per the largest
// chunk, magic = ceil(2^32 / per) or 0 for per = 1 (i / per without a division,
// exact while i * per < 2^32).
struct TileMap {
    int n, per, mlog;
    unsigned magic;
};

// Everything a kernel reads or writes, passed by value.  Cell arrays hold nc
// real cells followed (where noted) by nb boundary pseudo-cells.  A kernel
// waits for each 64-byte line of its arguments in turn, so the fields lie by
// use: the counts fill the first line, the second and the start of the third
// are the update's, the next the BVD's, the reconstruction's and the flux's
// (back to back on 20k quads: update 4.9 us with its fields spread over five
// lines, 4.4 so; BVD 4.1, 3.9; float flux with the CFL bound 7.0, 6.7).
template <typename R>
struct DevPtrs {
    using v4 = typename VT<R>::v4;
    using v2 = typename VT<R>::v2;
    int nc, nf, nb, maxC;
    TileMap map;               // of the kernel that is launched (set by the launchers)
    int stenW;                 // ids per row of sten, a multiple of 8
    int hfix, hcap;            // halo ids per row, capacity of the LDS halo (the dummy member follows it)
    int rbfRow;                // elements of a row of coefficients
    int lds_sten_off;          // byte offset of the stencil ids in the reconstruction kernels' LDS
    int lds_m_off;             // byte offset of the tile's least-squares weights (four-lane kernel)
    int lds_bvd_sten_off;      // byte offset of the stencil ids in the BVD kernel's LDS
    int16_t boundaryFirstOrder;  // extension: first-order faces in cells with a boundary face
    int16_t storeFlat;         // the reconstruction stores what fflat lets it leave out, too

    v4* W;                     // nc+nb primitive p, Ux, Uy, T
    const int32_t* slot_face;  // sliced ELL, +-(face+1), slices of whole tiles
    const uint8_t* ccnt;       // nc compact stencil size
    const uint8_t* scnt;       // nc stencil size
    double4* U;                // nc conserved rho, rhoUx, rhoUy, rhoE
    double4* Uold;             // nc
    const double* vol;         // nc
    const int32_t* cinst;      // nc instance of each cell, or nullptr (see ninst)

    double4* flux;             // nf + nb face fluxes (FP32-mixed face-centre path: boundary faces only)
    float4* flux32;            // FP32-mixed face-centre path: the nf internal faces' fluxes as computed,
                               // in float (exact); else null
    int8_t* smooth;            // nc+nb smoothness flag (shockIndicator[2c])
    int8_t* tlim;              // nc: BJ(raw T limiter) < VALID_LIM_FACTOR (the BVD test's limiter condition)
    R* tTVD;                   // sliced ELL, the BVD test's limited linear temperature on the cell's face,
                               // Tc + BJ(raw T limiter) * (grad T . d), formed by the reconstruction
    R* fvT;                    // 2*nf face temperatures (see fv)
    const uint16_t* sten;      // one row per cell: LDS-local stencil ids, then the dummy member's
    const int32_t* halo;       // ntiles rows of hfix ids

    const int32_t* more_ptr;   // ntiles+1, ids of the longer lists past their row
    const int32_t* halo_more;
    int8_t* ftype;             // nc final reconstruction type (shockIndicator[2c+1])
    v4* lim;                   // nc limiters p, Ux, Uy, T, then one entry of ones
    // nf pairs (own, nei), face-centre path: that side's cell is flat, so its
    // face state is W + grad . d and its limiters 1; the face pass forms both,
    // the BVD the temperatures it needs, and the reconstruction stores neither
    // (storeFlat: it stores them too).  Written only where a cell's branch
    // changed.
    uint8_t* fflat;
    // nc: grad p; grad T; (dUx/dx, dUx/dy); (dUy/dx, dUy/dy)
    v2 *gp, *gT, *gu;

    v2* gv;
    uint8_t* flat_prev;        // nc: the cell took the flat branch at the last reconstruction (what fflat is of)
    // FP64 four-lane reconstruction: the slot geometry and least-squares
    // weights are formed from these instead of read from slot_d, slot_dr, lsq
    const double2* fcen;       // nf+nb face centres
    const double2* cen;        // nc+nb cell and pseudo-cell centres
    const double2* fshift;     // nf periodic shift of the neighbour centre, or null when every shift is zero
    // 2*nf reconstructed face values [2f + side].  FP64: one array per
    // variable (fvp, fvu, fvv, fvT; fv null).  FP32-mixed: (p, Ux, Uy, T)
    // records in fv and the temperatures again in fvT (fvp, fvu, fvv null):
    // 4-byte scattered stores into four arrays measured slower than one
    // 16-byte record.  The BVD test reads fvT alone.
    R *fvp, *fvu, *fvv;

    v4* fv;
    const int2* fcell;         // nf own, nei
    // Faces.  The CFL bound needs Sf, magSf and fcfl in double in either
    // precision; the FP64 face-centre flux forms the face's offsets from both
    // cell centres from cen, fcen, fshift; FP32-mixed reads its own records.
    const double2* fsf;        // nf Sf
    const double* fmag;        // nf magSf
    const double2* fcfl;       // nf distance of the cell centres, the owner's share of it
    const float4* fsf32;       // FP32-mixed: nf (Sfx, Sfy, magSf, 0) rounded to float; else null
    const float4* foff32;      // FP32-mixed: nf (dxo, dyo, dxn, dyn) rounded to float; else null
    double* dt_part;           // partial minima: kCflBlocks, or two per tile of the flux pass, if more

    const R* rbf;              // RBF coefficients: maxC rows per slice (DevLayout::rbf_at)
    const v2* slot_d;          // sliced ELL, face centre - cell centre, in the kernels' precision
    v2* lsq;                   // sliced ELL, least-squares weights
    R* slot_dr;                // sliced ELL, |slot_e| in the kernels' precision (written by K3)
    const double2* slot_e;     // sliced ELL, compact neighbour - cell centre (K3 only)
    const int32_t* bcell;      // nb
    const uint8_t* blabel;     // nb
    const double4* bgeo;       // nb (Sfx, Sfy, magSf, 0)
    const double4* bval;       // nb fixed values of label 6
    int maxS, ntiles;
    // extension (faceQuadrature): flux at ngp points per internal face
    int ngp;                   // 0: face centre only (reference)
    double gpw[4];             // point weights, sum 1
    const R* rbf_gp;           // RBF coefficients at the points: ngp * maxC rows per slice
    const v4* fgd;             // ngp*nf: point - owner centre (x, y), point - neighbour centre (z, w),
                               // in the kernels' precision
    v4* fvg;                   // ngp*2*nf reconstructed states at the points, [(g*nf + f)*2 + side]
    double* dt;                // device time step of each instance (ninst)
    unsigned int* dt_count;    // tickets of the CFL pass: kCflGroups + 1 counters 128 bytes apart
    // Batches: ninst independent meshes stored one after the other (cells,
    // internal faces, boundary faces each contiguous per instance).  Each has
    // its own CFL time step.  A single mesh is ninst = 1 with cinst = nullptr.
    int ninst;
    const int32_t* finst_off;  // ninst+1 first internal face of each instance
    // Device clock of each instance: tctl[4i] = t, tctl[4i+1] = end time,
    // tctl[4i+2] = steps taken.  The device time step is clipped to land on
    // the end time; once there, steps leave the state unchanged (time step 0).
    double* tctl;
    double* res_part;          // partial sums of the residual norm (one per 256 cells), then their sum
};

template <typename R> void launch_lsq(const DevPtrs<R>& p, hipStream_t s);
// host_dt (optional): pinned host memory that receives the time step too.
template <typename R>
void launch_cfl(const DevPtrs<R>& p, double Rg, double Cv, double CFL, double* host_dt, hipStream_t s);
// lanes: 1 = one thread per cell (any mesh), 4 = four threads per cell (meshes
// whose cells have at most four faces).
template <typename R> void launch_reconstruct(const DevPtrs<R>& p, int tile, size_t lds, hipStream_t s, int lanes);
template <typename R> void launch_bvd(const DevPtrs<R>& p, int tile, size_t lds, hipStream_t s);
template <typename R> void launch_flux(const DevPtrs<R>& p, double Rg, double Cv, hipStream_t s);
// Flux pass that also reduces the CFL bound of the current state (the state
// the step starts from) to per-block minima in p.dt_part; launch_dt_reduce
// then stores their minimum in *p.dt.
template <typename R> void launch_flux_dt(const DevPtrs<R>& p, double Rg, double Cv, double CFL, hipStream_t s);
// Tiles of the flux pass that reduces the CFL bound (256 faces each, two partials a tile).
int flux_tiles(int nf, int nb);
template <typename R> void launch_dt_reduce(const DevPtrs<R>& p, hipStream_t s);
// Sum over cells of (density residual / volume)^2 from the current fluxes
// into *out (device); res_part needs residual_blocks(nc) entries.
int residual_blocks(int nc);
template <typename R> void launch_residual_norm(const DevPtrs<R>& p, double* out, hipStream_t s);
template <typename R>
void launch_update(const DevPtrs<R>& p, double Rg, double gamma, double dt, const double* dt_ptr, double b1, double b2,
                   double b3, int last, hipStream_t s);
// Output in another cell order: rows idx[0..n) of the conserved state src, and
// of the primitive state (as doubles) with the types or (pairs) the smoothness
// flag and type of each.
void launch_gather_state(const double4* src, const int32_t* idx, double4* dst, int n, hipStream_t s);
template <typename R>
void launch_gather_fields(const DevPtrs<R>& p, const int32_t* idx, double4* W, int8_t* flags, int pairs, int n,
                          hipStream_t s);
// FP64 at the face centre: stores the face states and limiters that the last
// reconstruction left out (DevPtrs::fflat).  U: the conserved state that it
// started from, or null if that is W; dt_ptr: the device time steps of the step
// that followed (0: none was taken), or null.
void launch_store_flat(const DevPtrs<double>& p, const double4* U, const double* dt_ptr, double Rg, double gamma,
                       hipStream_t s);
// Raises each reconstruction kernel's dynamic-LDS limit to lds minus its static LDS.
template <typename R> hipError_t set_lds_limits(size_t lds);
void launch_math_selftest(const double* x, double* out, int n, hipStream_t s);
void launch_math_selftest_f32(const float* x, float* out, int n, hipStream_t s);
// The CFL time step over the caller's device arrays in the reference's layout
// (FD, CELL, FACE, neighbour, optional FSHIFT) into *deltaT (device memory),
// on stream s; allocates nothing (its partial minima are a static device array).
void adjust_time_step_noalloc(const double* FD, const double* CELL, const double* FACE, const int32_t* neighbour,
                              const double* FSHIFT, int nf, double R, double Cv, double CFL, double* deltaT,
                              hipStream_t s);

}  // namespace afar
