// atx_device.h -- compiled-lattice format shared by the host compiler
// (atx_host.cpp) and the tracking kernels (atx_kernel.hip).
//
// A lattice is compiled into an array of fixed 64-byte element headers plus
// one pool of doubles holding every element-constant value. Everything that
// depends only on element parameters, the ring energy or the ring length is
// evaluated once on the host in FP64 with the C library (the same values the
// reference integrators compute inside their particle loops: KickAngle
// folding, Forest-Ruth slice lengths, irho, edge tan(), elegant fringe
// matrices, rad_const = RAD_CONST*gamma^3, RF nv/2*pi*f/(h/f - T0)). The
// kernel reads headers and pool through uniform (scalar) loads: every lane of
// a workgroup walks the same element sequence.
#pragma once

#include <stdint.h>

namespace atx {

// XCDs of the device: the hardware deals the workgroups of a launch to them
// in turn (workgroup i to XCD i mod kXcds), and each has its own L2.
constexpr int kXcds = 8;

// Dispatch kinds of the kernel switch (one per in-scope pass method).
enum Kind : int32_t {
  K_IDENTITY = 0,
  K_DRIFT = 1,
  K_STR = 2,      // StrMPoleSymplectic4Pass
  K_BND = 3,      // BndMPoleSymplectic4Pass
  K_STRRAD = 4,   // StrMPoleSymplectic4RadPass
  K_BNDRAD = 5,   // BndMPoleSymplectic4RadPass
  K_THIN = 6,     // ThinMPolePass
  K_RF = 7,       // RFCavityPass
  K_CORR = 8,     // CorrectorPass
  K_APERTURE = 9, // AperturePass
  K_CAVITY = 10,      // CavityPass
  K_EXDRIFT = 11,     // ExactDriftPass
  K_EXMPOLE = 12,     // ExactMultipolePass
  K_EXMPOLERAD = 13   // ExactMultipoleRadPass
};

// Header flags.
enum : uint32_t {
  F_EDGEB_IN = 1u << 20,   // FringeInt1 > 0 and FullGap > 0 (diff_bend_fringe.c:36-44)
  F_EDGEB_OUT = 1u << 21,  // FringeInt2 > 0 and FullGap > 0
  F_T1 = 1u << 0,
  F_R1 = 1u << 1,
  F_R2 = 1u << 2,
  F_T2 = 1u << 3,
  F_RAP = 1u << 4,
  F_EAP = 1u << 5,
  F_SCALE = 1u << 6,      // FieldScaling != 1
  F_THICK = 1u << 7,      // RF / corrector with non-zero length
  F_RFKICK = 1u << 8,     // RF with nv != 0
  F_LEAN = 1u << 9,       // thick multipole without FieldScaling, quadrupole fringes, edges with
                          // a tangent per particle and op table
};

// Edge-focusing modes (vertical term fy) chosen on the host from
// FringeBendEntrance/Exit and whether the fringe correction is zero.
enum EdgeMode : int32_t {
  E_CONST = 0,   // fy = irho*tan(edge)                         (element constant)
  E_DIVP = 1,    // fy = (irho*tan(edge)) / (1+dp)               non-rad method 2, corr = 0
  E_MULPN = 2,   // fy = (irho*tan(edge)) * pn                   rad method 2, psi = 0
  E_TAN1 = 3,    // fy = irho*tan(edge - corr/(1+dp))            non-rad method 1/legacy
  E_TAN2 = 4,    // fy = irho*tan(edge - corr/(1+dp))/(1+dp)     non-rad method 2
  E_TAN3 = 5,    // fy = irho*tan(edge - corr +- px/(1+dp))      non-rad method 3
  E_RTAN1 = 6,   // fy = irho*tan(edge - psi*pn)                 rad method 1/legacy
  E_RTAN2 = 7,   // fy = irho*tan(edge - psi*pn)*pn              rad method 2
  E_RTAN3 = 8    // fy = irho*tan(edge - psi +- px*pn)           rad method 3
};

// Quadrupole-fringe modes.
enum QuadFringe : int32_t { Q_NONE = 0, Q_LEE = 1, Q_ELEGANT = 2 };

// Scalar-block slots (pool[h.sc + S_*]).
enum Slot : int32_t {
  S_L1 = 0, S_L2 = 1, S_K1 = 2, S_K2 = 3,   // Forest-Ruth drift/kick lengths
  S_IRHO = 4,
  S_SCALE = 5, S_INVSCALE = 6,
  S_B2 = 7,                                 // PolynomB[1] for the quad fringes
  S_FX_IN = 8, S_FY_IN = 9, S_FX_OUT = 10, S_FY_OUT = 11,
  S_EDGE_IN = 12, S_CORR_IN = 13, S_EDGE_OUT = 14, S_CORR_OUT = 15,
  S_RADC = 16,
  S_BAX = 17, S_BAY = 18,
  S_RK1 = 19, S_RK2 = 20,                   // S_RADC * S_K1, S_RADC * S_K2 (fast build)
  S_ELEN = 21,                              // Length (exact multipoles)
  S_DIFC = 22,                              // DIF_CONST * gamma^5 (diffusion matrices)
  S_NSCALAR = 23,
  S_NSHORT = 8,                             // of elements that are no multipoles
  // RF cavity
  S_RF_HALF = 0, S_RF_NV = 1, S_RF_TWOPIF = 2, S_RF_LAG = 3, S_RF_PHILAG = 4, S_RF_HFT0 = 5,
  // corrector
  S_C_XK = 0, S_C_YK = 1, S_C_LEN = 2, S_C_Q0 = 3,  // S_C_Q0 = xk*xk/3 + yk*yk/3
  // drift
  S_D_LEN = 0
};

struct DevElem {
  int32_t kind;
  uint32_t flags;
  int32_t order;      // MaxOrder
  int32_t nslice;     // NumIntSteps
  int32_t sc;         // pool offset of the scalar block
  int32_t poly;       // pool offset of A[0..order], then B[0..order]
  int32_t t1, r1;     // pool offsets (valid when the flag is set)
  int32_t r2, t2;
  int32_t rap, eap;   // RApertures (4) / Limits (4); EApertures (2)
  int32_t edge;       // EdgeMode at entrance | (EdgeMode at exit << 8)
  int32_t ops;        // pool offset of the slice op table (integrators other than 4), -1: none
  int32_t fringe;     // QuadFringe at entrance | (QuadFringe at exit << 8)
  int32_t fq;         // pool offset of the elegant fringe matrices: in-P, in-M, out-M, out-P (8 each)
};

// Slice op table of a non-default integrator: pool[ops] = number of ops,
// then (code, length) pairs with code 0 = drift of that length, 1 = kick.
static_assert(sizeof(DevElem) == 64, "DevElem must stay 64 bytes (dword fields: scalar loads)");

// The tracking kernel's program of a lattice: one record per element that
// does work, holding the markers and the plain drift before it, so that a
// record costs one round of scalar loads and one dispatch. Elements of a
// record, in order: markers (IdentityPass without attributes), a plain drift
// (flag OPF_DRIFT), the element of `op` (other than OP_NONE); `last` is the
// index of the last of them. The constants an op needs are in the record
// itself, at fixed offsets, so that no address depends on an earlier load. A
// terminal record follows the last one, whole like the others: the kernel reads
// a record's head and a word of each of its next two lines (up to byte 132) one
// record ahead.
enum OpKind : int32_t {
  OP_NONE = 0,      // no element after the markers and the drift
  OP_GENERIC = 1,   // the element by its DevElem header
  OP_APERTURE = 2,  // AperturePass: c[0..3] = limits
  OP_CORR = 3,      // CorrectorPass: c[OC_*]
  // thick multipoles with all coefficients (of order 0: as of order 1): c[OM_*]
  OP_STR1 = 4,
  OP_STR2 = 5,
  OP_STR3 = 6,
  OP_BND1 = 7,
  OP_STRRAD1 = 8,
  OP_BNDRAD1 = 9,
  // ThinMPolePass: c[OT_*], c[OM_POLY...]
  OP_THIN2 = 10,
  OP_THIN3 = 11,
  // those of any order up to 3 with few coefficients that are not zero: one B only (L, its
  // index), B[2], B[0] and A[0] (D), none (0)
  OP_STR1L = 12,
  OP_STR2L = 13,
  OP_STR2D = 14,
  OP_STR3L = 15,
  OP_BND1L = 16,
  OP_BND0 = 17,
  OP_STRRAD1L = 18,
  OP_BNDRAD1L = 19,
  OP_BNDRAD0 = 20,
  OP_STRRAD2 = 21,
  OP_STRRAD3 = 22,
  OP_BND2 = 23,
  OP_BND3 = 24,
  OP_BNDRAD2 = 25,
  OP_BNDRAD3 = 26,
  OP_MARK = 27,     // IdentityPass with apertures
  OP_DRIFT = 28,    // DriftPass with apertures: c[0] = length
};
// The strict build evaluates all coefficients: its kinds, in the highest byte of
// `op`, are the four kinds of multipole plus MaxOrder. OP_NONE to OP_CORR keep
// their numbers.
enum StrictKind : int32_t {
  SK_THIN2 = 4,
  SK_THIN3 = 5,
  SK_MARK = 6,
  SK_DRIFT = 7,
  SK_STR = 8,
  SK_BND = 12,
  SK_STRRAD = 16,
  SK_BNDRAD = 20,
};
enum : int32_t {
  OPF_DRIFT = 1 << 8,  // a plain drift of length `len` before the element
  OPF_THICK = 2 << 8,  // corrector of non-zero length
  OPF_XF = 4 << 8,     // misaligned by transverse shifts and rolls: c[OM_XF...]
  OPF_ENDS = 8 << 8,   // a bend's edges by its header (not of constant strength, or with
                       // quadrupole fringes)
  OPF_MPOLE = 16 << 8, // a thick multipole
  OPF_RAD = 32 << 8,   // a radiating one
  OPF_R1 = 64 << 8,    // misaligned with a roll at the entry, at the exit
  OPF_R2 = 128 << 8,
  OPF_FRINGE = 1 << 16,  // a straight magnet's quadrupole fringes, by the header
  OPF_HXF = 2 << 16,     // misaligned otherwise: by the header
  OPF_RAP = 4 << 16,     // rectangular aperture at entry and exit: c[OM_RAP...]
  OPF_EAP = 8 << 16,     // elliptical one: c[OM_EAP...]
  OPF_SCALE = 16 << 16,  // FieldScaling: c[OM_SCALE...]
  OPF_FULL = 32 << 16,   // rare, run by the kernel's full loop only (fast build, strict build)
  OPF_FULL_STRICT = 64 << 16,
  OPF_AROUND = OPF_XF | OPF_HXF | OPF_RAP | OPF_EAP | OPF_SCALE | OPF_FRINGE,
};
constexpr int kStrictShift = 24;
// constants of OP_CORR, the thin and the thick multipoles
enum OpSlot : int32_t {
  OC_XK = 0, OC_YK = 1, OC_LEN = 2, OC_Q0 = 3,
  OT_BAX = 0, OT_BAY = 1,
  OM_L1 = 0, OM_L2 = 1, OM_K1 = 2, OM_K2 = 3, OM_IRHO = 4, OM_RADC = 5, OM_RK1 = 6, OM_RK2 = 7,
  OM_POLY = 8,  // A[0..order], then B[0..order] (of order 0: as of order 1)
  OM_FX_IN = 12, OM_FY_IN = 13, OM_FX_OUT = 14, OM_FY_OUT = 15,  // bends
  // entry: x, px, y, py shifts, then cos and sin of the roll; exit: cos, sin, shifts
  OM_XF = 16,
  OM_INV = 28,    // cos and sin of the inverse rolls (adjoint): entry, exit
  OM_POLY2 = 32,  // A and B of bends of order 2 and 3, in the place of OM_POLY
  OM_RAP = 40, OM_EAP = 44,
  OM_SCALE = 46,  // FieldScaling and its reciprocal
  OM_ZERO = 48,   // strict build: zeros that an OPF_XF adds to delta and ct at entry, exit
};
constexpr int kOpConsts = 60;  // 52 and padding
struct LatOp {
  int32_t op;      // OpKind | OPF_* | StrictKind << kStrictShift
  int32_t last;    // index of the record's last element
  double len;      // the drift's length
  int32_t first;   // index of its first element (the next record's: one past its last)
  int32_t nslice;  // at least 1 (thick multipoles)
  double lead;     // their highest coefficient that is not zero (B)
  double c[kOpConsts];
};
// Four lines of the L2: with 448 bytes, where every other record starts in the middle
// of one, a turn of the large ring takes 1.92 ms instead of 1.88 (24,001 particles).
static_assert(sizeof(LatOp) == 512, "LatOp: four 128-byte lines");

// One tracked lattice instance inside a launch. A single-lattice call has one
// instance; batched error realisations have one per lattice.
struct Instance {
  const DevElem* elems;
  const double* pool;
  const LatOp* ops;         // program records
  const int32_t* opof;      // record of each element
  const int32_t* slots;     // 2*(nelem/32+1): a bit per element with a copy, first turn then later turns
  double* r;                // particle state, updated in place
  double* rout;             // refpt copies (6, N, R, T) F-order
  uint8_t* lost_flag;
  uint32_t* lost_turn;
  uint32_t* lost_elem;
  double* lost_coord;       // (6, N) F-order
  int64_t pstride;          // distance between particles in r (6: (6,N) F-order; 1: SoA)
  int64_t cstride;          // distance between coordinates in r (1: F-order; N: SoA)
  int32_t nelem;
  int32_t npart;
  int32_t nturns;
  int32_t turn0;
  int32_t start_elem;
  int32_t end_elem;
  int32_t n_first;          // copies made on the first turn
  int32_t n_std;            // copies made on each later turn
  int32_t block_begin;      // first workgroup of this instance
  int32_t losses;           // 1: record the loss map (at.c checkiflost); 0: setlost only;
                            // 2: as 1, continuing the map of an earlier call
  int32_t elempass;         // 1: single element pass, no loss check (at.c at_elempass)
  int32_t full;             // the lattice has records with OPF_FULL (OPF_FULL_STRICT)
  // Repacked launches: lanes take particles idx[0..*nlive) instead of
  // 0..npart (both written by repack_kernel); NULL for plain launches.
  const int32_t* idx;
  const int32_t* nlive;
};

// Per-element data of the adjoint kernel: gradient slot (-1: none) and
// PolynomB index of the differentiated coefficient; pool offsets of the
// inverse misalignment matrices.
struct AdjElem {
  int32_t slot;
  int32_t coeff;
  int32_t r1inv;
  int32_t r2inv;
};

// The same of a record's element, beside the record.
struct AdjRec {
  int32_t slot;
  int32_t coeff;
};

// Diffusion matrices (one lane per element): B of each radiating element
// from its entrance orbit.
struct DiffArgs {
  const DevElem* elems;
  const double* pool;
  const double* orbits;  // (6, nelem): orbit at the entrance of each element
  double* bdiff;         // nelem x 36, column-major 6x6 per element
  int32_t nelem;
  int32_t row_major;     // [i][j] at j+6i
};

// Element matrices by central differences (one wave per element).
struct ElemMatArgs {
  const DevElem* elems;
  const double* pool;
  const LatOp* ops;
  const int32_t* opof;
  const double* orbits;  // (6, nelem): orbit at the entrance of each element
  double* m66;           // nelem x 36, column-major 6x6 per element
  double step;
  int32_t nelem;
  int32_t row_major;     // [i][j] at j+6i
};

// One block of turns of the adjoint sweep (gridDim.y indexes the items).
struct AdjItem {
  const double* states;  // (nturns+1) blocks of (6, N): turn-start states, then the end state
  double* lam;           // (6, N) adjoint of the end state in, of the start state out
  double* grad;          // accumulated dL/dPolynomB[coeff] per slot; NULL: not accumulated
  int32_t npart;
  int32_t nturns;
  int32_t turn0;         // turn counter of the first turn of the block
  int32_t pad;
};

struct AdjArgs {
  const DevElem* elems;
  const double* pool;
  const AdjElem* adj;
  const LatOp* ops;
  const AdjRec* recs;
  const AdjItem* items;
  int32_t nops;
  int32_t nitems;
};

}  // namespace atx
