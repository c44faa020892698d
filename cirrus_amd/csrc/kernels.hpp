// HIP kernels of the MGPCG path for gfx950 (device code, included by mgpcg.hip).
//
// Layout in HBM (structure of arrays, one problem or many in one pool):
//   channel c of tile t, cell (i,j,k):  ch[c][t*512 + (i<<6 | j<<3 | k)]  (FP32)
//   cell types:                        ctype[t*512 + ...]                (u8)
//   worklists:                          arrays of 128-byte TileRec (one per tile
//                                       and phase), so a workgroup finds its
//                                       tile, neighbours and children in one
//                                       scalar load
//   per-problem scalars:                ProbState
// Execution: one 64-lane wavefront per 8^3 tile.  Lane l = (i,j) = (l>>3, l&7)
// owns the k-pencil of 8 cells at offsets l*8..l*8+7 (32 contiguous bytes), so a
// wavefront reads or writes a whole channel of a tile as 2 KB of coalesced
// 16-byte accesses.  Neighbours in k are in the lane's registers; neighbours in
// i and j come from an LDS copy of the pencils plus a one-pencil halo ring
// loaded from the face-neighbour tiles; the two k-halo cells are read straight
// into registers.
//
// Floating-point operations are written out in the reference's order with
// explicit fmaf where the reference's compiler fuses a multiply-add, and the
// library is compiled with -ffp-contract=off, so every kernel reproduces the
// CPU transcription bit for bit.  FP64 dot products use one fixed summation
// order (per lane over its 8 cells, a xor-butterfly across the wavefront, then
// per problem over the tile partials the same way).
#pragma once
#include <hip/hip_runtime.h>
#include <type_traits>
#include <stdint.h>

namespace cg {

enum : uint8_t { T_LEAF = 1, T_NONLEAF = 2, T_GHOST = 4 };
enum : uint8_t { C_DIR = 1, C_INT = 2, C_NEU = 4 };
typedef __bf16 bf16;
typedef _Float16 f16;

struct alignas(16) TileRec {
  int32_t nbr[6];     // same-level face neighbours x-,y-,z-,x+,y+,z+ (-1: none)
  int32_t parent;     // -1 on level 0
  int32_t prob;       // problem index in the pool
  int32_t leaf_slot;  // LEAF: slot of its dot partial; -1 otherwise
  int32_t gslot;      // GHOST: slot in the 64-value ghost buffer; LEAF with ghost children: the slot of the
                      // first of them, where its GhostKids entry is; -1 otherwise
  int32_t self;       // the tile's index
  float h;            // cell size of the tile's level
  uint32_t meta;      // level | type << 8 | octant << 16 | has_gchild << 24 | all_interior << 25 |
                      // inert_candidate << 26 | all_open << 27 | uniform << 28
  uint32_t ntypes;    // type of face neighbour f in bits 4f..4f+3 (0: none), std_face f in bit 24 + f
  float bc[7];        // face coefficients of the smoothing view (subtree at the
                      // tile's own level): faces x-,y-,z-,x+,y+,z+, then inside
  int32_t nbr_parent[6];  // parent tile of face neighbour f (-1: no neighbour or level 0)
  int32_t pad0;
  double rdiag;       // 1 / D, D = the sweep's diagonal of a cell whose six faces have the inside coefficient
  int32_t pad1[2];
};
static_assert(sizeof(TileRec) == 128, "TileRec is 128 bytes");
// The ghost children of a LEAF tile by octant (-1: none): tile and ghost slot.
struct alignas(16) GhostKids {
  int32_t tile[8];
  int32_t slot[8];
};
// Fields packed in dwords so that a workgroup fetches them with scalar loads.
__host__ __device__ __forceinline__ int tr_level(const TileRec& T) { return int(T.meta & 0xff); }
__host__ __device__ __forceinline__ uint8_t tr_type(const TileRec& T) { return uint8_t((T.meta >> 8) & 0xff); }
__host__ __device__ __forceinline__ int tr_octant(const TileRec& T) { return int((T.meta >> 16) & 0xff); }
__host__ __device__ __forceinline__ bool tr_has_gchild(const TileRec& T) { return ((T.meta >> 24) & 1) != 0; }
// every one of the tile's 512 cells is INTERIOR (its cell types need not be read)
__host__ __device__ __forceinline__ bool tr_all_int(const TileRec& T) { return ((T.meta >> 25) & 1) != 0; }
// a LEAF tile without ghost children and without an INTERIOR cell: when its
// right-hand side is zero as well (decided per solve), every CG iteration
// leaves each of its values as it found them (see k_cg_init)
__host__ __device__ __forceinline__ bool tr_inert_cand(const TileRec& T) { return ((T.meta >> 26) & 1) != 0; }
// every cell INTERIOR and no face cut by a NEUMANN cell: each face mask byte is
// M_OPEN_INT (the masks need not be read); of a LEAF or NONLEAF tile also: every
// cell's diagonal is finite and not 0
__host__ __device__ __forceinline__ bool tr_all_open(const TileRec& T) { return ((T.meta >> 27) & 1) != 0; }
// every face of the tile has the inside coefficient: with all_open every cell's
// diagonal is D (rdiag)
__host__ __device__ __forceinline__ bool tr_uniform(const TileRec& T) { return ((T.meta >> 28) & 1) != 0; }
// every face neighbour is missing, a GHOST tile, or all_open and uniform (so the
// diagonal of its cells is D)
__host__ __device__ __forceinline__ bool tr_std_faces(const TileRec& T) { return ((T.ntypes >> 24) & 0x3f) == 0x3f; }
__host__ __device__ __forceinline__ uint8_t tr_ntype(const TileRec& T, int f) { return uint8_t((T.ntypes >> (4 * f)) & 0xf); }

struct alignas(16) ProbState {
  double gamma, gamma_old, alpha, beta;
  double bb, thr, rr, pAp;
  double mean, tol2;
  double thr_abs;   // floor of the stop threshold (|r|^2 < max(tol2 |b|^2, thr_abs)); 0: none
  double tol_abs2;  // FIN_IRBB: thr_abs = tol_abs2 * |b_outer|^2
  double bb_b;      // |b_outer|^2 of an FP64 refinement (the outer right-hand side)
  int32_t iter, done, converged, max_iters;
  uint32_t counter;
  int32_t leaf_begin, leaf_count, pure_neumann;
  int32_t check_stride;  // test convergence after iterations k*check_stride; <= 0: never
  int32_t scale_exp;     // float16 storage: the right-hand side is solved scaled by 2^scale_exp
};

// Channel pointers passed to every kernel by value.
struct Ctx {
  const uint8_t* ctype;
  const uint8_t* fmask;  // per cell: bit e (faces x-, x+, y-, y+, z-, z+) set if the face is not cut by a
                         // NEUMANN cell on either side, bit 6 set on INTERIOR cells (see k_face_mask)
  const uint32_t* fsplit;  // the same masks by colour: per tile [colour][lane], byte m = cell k = 2m + p
                           // of the lane's pencil, p = (colour + i + j) & 1 (k_face_mask)
  float* x;      // pressure / CG x
  float* r;      // rhs b, then residual r
  float* p;      // CG direction
  float* ap;     // A p
  float* z;      // preconditioned residual (V-cycle x)
  float* rhsv;   // V-cycle rhs: r on LEAF tiles (plus ghost sums), restricted residual on NONLEAF
  float* zb;     // damped-Jacobi ping-pong buffer; RB-GS down-sweep values
  bf16* zh;      // z, rhsv and zb stored as bfloat16 (mixed-precision form; null until used)
  bf16* rhsvh;
  bf16* zbh;
  f16* zf;       // the same buffers holding float16 values (one storage type per solve)
  f16* rhsvf;
  f16* zbf;
  float* gsum;   // 64 per ghost: 2x2x2 sums of the ghost rows of A p
  ProbState* ps;
  int32_t* progress;  // per problem 2 * iterations + done, in host memory, which the host polls (null: nobody does)
  const int32_t* pmap;  // finalize workgroup -> problem (null: identity)
  double* part;  // per-leaf-slot dot partials
  double* part2; // second partial stream (mean counts)
  const float* diag;  // per cell, colour-split order: the V-cycle colour sweep's diagonal D (k_diag)
  const TileRec* tiles;  // every tile's record by tile index (null where the handle has none)
  const GhostKids* kids;  // ghost children of LEAF tiles, by TileRec::gslot
  uint8_t* inert = nullptr;  // per tile: 1 while the current solve leaves the tile untouched (k_cg_init)
};

// The V-cycle vectors of the storage type V.
template <class V> __device__ __forceinline__ V* vc_z(const Ctx& c);
template <class V> __device__ __forceinline__ V* vc_rhs(const Ctx& c);
template <> __device__ __forceinline__ float* vc_z<float>(const Ctx& c) { return c.z; }
template <> __device__ __forceinline__ bf16* vc_z<bf16>(const Ctx& c) { return c.zh; }
template <> __device__ __forceinline__ float* vc_rhs<float>(const Ctx& c) { return c.rhsv; }
template <> __device__ __forceinline__ bf16* vc_rhs<bf16>(const Ctx& c) { return c.rhsvh; }
template <> __device__ __forceinline__ f16* vc_z<f16>(const Ctx& c) { return c.zf; }
template <> __device__ __forceinline__ f16* vc_rhs<f16>(const Ctx& c) { return c.rhsvf; }
template <class V> __device__ __forceinline__ V* vc_zb(const Ctx& c);
template <> __device__ __forceinline__ float* vc_zb<float>(const Ctx& c) { return c.zb; }
template <> __device__ __forceinline__ bf16* vc_zb<bf16>(const Ctx& c) { return c.zbh; }
template <> __device__ __forceinline__ f16* vc_zb<f16>(const Ctx& c) { return c.zbf; }

// ---------------------------------------------------------------------------
// small helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

__host__ __device__ __forceinline__ uint8_t subtree_type(uint8_t type, int level, int sl) {
  return (level == sl && type == T_NONLEAF) ? T_LEAF : type;
}
// Face coefficient before the NEUMANN cut (GMGSolver.cu:26-39): 1/h^2 on
// LEAF-LEAF faces, (2/3)/h^2 on LEAF-GHOST faces, 0 otherwise.
__host__ __device__ __forceinline__ float base_coeff(uint8_t t0, uint8_t t1, float cll, float clg) {
  bool both = (t0 & T_LEAF) && (t1 & T_LEAF);
  bool lg = ((t0 & T_LEAF) && (t1 & T_GHOST)) || ((t0 & T_GHOST) && (t1 & T_LEAF));
  return both ? cll : (lg ? clg : 0.f);
}
__device__ __forceinline__ uint8_t ct_at(uint64_t w, int k) { return uint8_t(w >> (8 * k)); }

__device__ __forceinline__ void load8(const float* __restrict__ p, float v[8]) {
  float4 a = reinterpret_cast<const float4*>(p)[0];
  float4 b = reinterpret_cast<const float4*>(p)[1];
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
// The same past the caches, for an array that is used once an iteration: x, which
// k_cg_update_p reads and writes while its p is about to be read by the operator.
// Refined 45,054-tile scene 45.5 -> 45.2 ms a solve, 24 problems 19.34 -> 19.16, 7
// problems 6.51 -> 6.41, 256 problems 216.2 -> 215.7.  (r too: a gain on the larger
// two, none on the others.)
typedef float Quad __attribute__((ext_vector_type(4)));
__device__ __forceinline__ void load8_once(const float* __restrict__ p, float v[8]) {
  const Quad* q = reinterpret_cast<const Quad*>(p);
  const Quad a = __builtin_nontemporal_load(q), b = __builtin_nontemporal_load(q + 1);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    v[k] = a[k];
    v[4 + k] = b[k];
  }
}
__device__ __forceinline__ void store8_once(float* __restrict__ p, const float v[8]) {
  Quad* q = reinterpret_cast<Quad*>(p);
  __builtin_nontemporal_store(Quad{v[0], v[1], v[2], v[3]}, q);
  __builtin_nontemporal_store(Quad{v[4], v[5], v[6], v[7]}, q + 1);
}
__device__ __forceinline__ void store8(float* __restrict__ p, const float v[8]) {
  reinterpret_cast<float4*>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
  reinterpret_cast<float4*>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
// V-cycle vectors may be stored as bfloat16 (8-bit significand, the FP32
// exponent range) and are always computed on in FP32: a stored value widens
// exactly, and every store rounds to nearest even (v_cvt_pk_bf16_f32).  One
// pencil of 8 values is then one 16-byte access.
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float to_f(float v) { return v; }
__device__ __forceinline__ float to_f(bf16 v) { return float(v); }
template <class V> __device__ __forceinline__ V from_f(float v);
template <> __device__ __forceinline__ float from_f<float>(float v) { return v; }
template <> __device__ __forceinline__ bf16 from_f<bf16>(float v) { return bf16(v); }
// the value a store of v to V-typed memory leaves (identity for FP32)
template <class V> __device__ __forceinline__ float vround(float v) { return to_f(from_f<V>(v)); }
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ uint32_t bf_pack(float a, float b) { return __builtin_bit_cast(uint32_t, bf16x2{bf16(a), bf16(b)}); }
__device__ __forceinline__ void load8(const bf16* __restrict__ p, float v[8]) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  v[0] = bf_lo(q.x); v[1] = bf_hi(q.x); v[2] = bf_lo(q.y); v[3] = bf_hi(q.y);
  v[4] = bf_lo(q.z); v[5] = bf_hi(q.z); v[6] = bf_lo(q.w); v[7] = bf_hi(q.w);
}
__device__ __forceinline__ void store8(bf16* __restrict__ p, const float v[8]) {
  *reinterpret_cast<uint4*>(p) = make_uint4(bf_pack(v[0], v[1]), bf_pack(v[2], v[3]), bf_pack(v[4], v[5]), bf_pack(v[6], v[7]));
}
// a pencil as two float4 (k 0..3, 4..7)
__device__ __forceinline__ void load_pencil(const float* __restrict__ p, float4& a, float4& b) {
  const float4* q = reinterpret_cast<const float4*>(p);
  a = q[0];
  b = q[1];
}
__device__ __forceinline__ void load_pencil(const bf16* __restrict__ p, float4& a, float4& b) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  a = make_float4(bf_lo(q.x), bf_hi(q.x), bf_lo(q.y), bf_hi(q.y));
  b = make_float4(bf_lo(q.z), bf_hi(q.z), bf_lo(q.w), bf_hi(q.w));
}
__device__ __forceinline__ void store_pencil(float* __restrict__ p, float4 a, float4 b) {
  float4* q = reinterpret_cast<float4*>(p);
  q[0] = a;
  q[1] = b;
}
__device__ __forceinline__ void store_pencil(bf16* __restrict__ p, float4 a, float4 b) {
  *reinterpret_cast<uint4*>(p) = make_uint4(bf_pack(a.x, a.y), bf_pack(a.z, a.w), bf_pack(b.x, b.y), bf_pack(b.z, b.w));
}
// four consecutive values (a parent quad)
__device__ __forceinline__ float4 load4(const float* __restrict__ p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ float4 load4(const bf16* __restrict__ p) {
  const uint2 q = *reinterpret_cast<const uint2*>(p);
  return make_float4(bf_lo(q.x), bf_hi(q.x), bf_lo(q.y), bf_hi(q.y));
}
__device__ __forceinline__ void store4(float* __restrict__ p, float4 a) { *reinterpret_cast<float4*>(p) = a; }
__device__ __forceinline__ void store4(bf16* __restrict__ p, float4 a) {
  *reinterpret_cast<uint2*>(p) = make_uint2(bf_pack(a.x, a.y), bf_pack(a.z, a.w));
}

// two consecutive values
__device__ __forceinline__ float2 load2(const float* __restrict__ p) { return *reinterpret_cast<const float2*>(p); }
__device__ __forceinline__ float2 load2(const bf16* __restrict__ p) {
  const uint32_t q = *reinterpret_cast<const uint32_t*>(p);
  return make_float2(bf_lo(q), bf_hi(q));
}
__device__ __forceinline__ void store2(float* __restrict__ p, float2 a) { *reinterpret_cast<float2*>(p) = a; }
__device__ __forceinline__ void store2(bf16* __restrict__ p, float2 a) { *reinterpret_cast<uint32_t*>(p) = bf_pack(a.x, a.y); }

// Or as float16 (11-bit significand, largest finite value 65504): a store
// clamps to +-65504 and rounds to nearest even (v_cvt_f16_f32); a solve in this
// storage scales its right-hand side by a power of two (k_finalize FIN_SCALE)
// so that the values sit well inside that range.
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float to_f(f16 v) { return float(v); }
template <> __device__ __forceinline__ f16 from_f<f16>(float v) {
  v = v > 65504.f ? 65504.f : (v < -65504.f ? -65504.f : v);
  return f16(v);
}
__device__ __forceinline__ float h_lo(uint32_t w) { return float(__builtin_bit_cast(f16, uint16_t(w & 0xffffu))); }
__device__ __forceinline__ float h_hi(uint32_t w) { return float(__builtin_bit_cast(f16, uint16_t(w >> 16))); }
__device__ __forceinline__ uint32_t h_pack(float a, float b) {
  return __builtin_bit_cast(uint32_t, f16x2{from_f<f16>(a), from_f<f16>(b)});
}
__device__ __forceinline__ void load8(const f16* __restrict__ p, float v[8]) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  v[0] = h_lo(q.x); v[1] = h_hi(q.x); v[2] = h_lo(q.y); v[3] = h_hi(q.y);
  v[4] = h_lo(q.z); v[5] = h_hi(q.z); v[6] = h_lo(q.w); v[7] = h_hi(q.w);
}
__device__ __forceinline__ void store8(f16* __restrict__ p, const float v[8]) {
  *reinterpret_cast<uint4*>(p) = make_uint4(h_pack(v[0], v[1]), h_pack(v[2], v[3]), h_pack(v[4], v[5]), h_pack(v[6], v[7]));
}
__device__ __forceinline__ void load_pencil(const f16* __restrict__ p, float4& a, float4& b) {
  const uint4 q = *reinterpret_cast<const uint4*>(p);
  a = make_float4(h_lo(q.x), h_hi(q.x), h_lo(q.y), h_hi(q.y));
  b = make_float4(h_lo(q.z), h_hi(q.z), h_lo(q.w), h_hi(q.w));
}
__device__ __forceinline__ void store_pencil(f16* __restrict__ p, float4 a, float4 b) {
  *reinterpret_cast<uint4*>(p) = make_uint4(h_pack(a.x, a.y), h_pack(a.z, a.w), h_pack(b.x, b.y), h_pack(b.z, b.w));
}
__device__ __forceinline__ float4 load4(const f16* __restrict__ p) {
  const uint2 q = *reinterpret_cast<const uint2*>(p);
  return make_float4(h_lo(q.x), h_hi(q.x), h_lo(q.y), h_hi(q.y));
}
__device__ __forceinline__ void store4(f16* __restrict__ p, float4 a) {
  *reinterpret_cast<uint2*>(p) = make_uint2(h_pack(a.x, a.y), h_pack(a.z, a.w));
}
__device__ __forceinline__ float2 load2(const f16* __restrict__ p) {
  const uint32_t q = *reinterpret_cast<const uint32_t*>(p);
  return make_float2(h_lo(q), h_hi(q));
}
__device__ __forceinline__ void store2(f16* __restrict__ p, float2 a) { *reinterpret_cast<uint32_t*>(p) = h_pack(a.x, a.y); }

__device__ __forceinline__ uint64_t load_ct8(const uint8_t* __restrict__ p) {
  return *reinterpret_cast<const uint64_t*>(p);
}
// The lane's 8 cell types, or eight INTERIOR bytes without a load when the
// record says every cell of the tile is INTERIOR.
__device__ __forceinline__ uint64_t tile_ct8(const TileRec& T, const uint8_t* __restrict__ p) {
  return tr_all_int(T) ? 0x0101010101010101ull * C_INT : load_ct8(p);
}

// A wavefront-uniform value (keeps record fields in scalar registers).
__device__ __forceinline__ int uni(int v) { return __builtin_amdgcn_readfirstlane(v); }
// v[g] for a lane-dependent g in 0..3, as register selects
// One of four values by g in 0..3 (two selects on g's bits: no branches).
__device__ __forceinline__ int pick4(int g, int a, int b, int c, int d) {
  const int lo = (g & 1) ? b : a;
  const int hi = (g & 1) ? d : c;
  return (g & 2) ? hi : lo;
}

// The quotient a / d, correctly rounded, from rd = 1/d in FP64 (within 2^-51
// of it): the product's relative error is below 2^-50, and a quotient of two
// 24-bit significands lies at least 2^-49 (relative) from every rounding
// boundary of FP32, so the conversion rounds to the same value.  Below 2^-126,
// where FP32 has fewer bits, a quotient can lie on a boundary, a multiple of
// 2^-150 (else it is at least 2^-48 away from one): where the product is within
// 2^-49 of such a multiple, that is the quotient (div_again, run for subnormal
// results; a result of 0 is right as it is).  4 issue slots and one for the test
// against 15.5 for the FP32 division on gfx950.
__device__ __forceinline__ float div_by(float a, double rd) { return float(double(a) * rd); }
__device__ __forceinline__ bool subnormal(float q) { return __builtin_amdgcn_classf(q, 0x90); }
__device__ __forceinline__ float div_again(float q, float a, double rd) {
  constexpr double kToGrid = 0x1.8p-98;  // adding it leaves a multiple of 2^-150
  const double v = double(a) * rd, t = (v + kToGrid) - kToGrid;
  return subnormal(q) && __builtin_fabs(v - t) <= __builtin_fabs(v) * 0x1p-49 ? float(t) : q;
}
__device__ __forceinline__ float div_by_checked(float a, double rd) {
  float q = div_by(a, rd);
  if (__builtin_expect(subnormal(q), 0)) q = div_again(q, a, rd);
  return q;
}
// The same without a test, where a branch is on the critical path: the product
// rounded to 50 bits is still on its side of every boundary that it is not on, and
// is the quotient where that has 25 bits (rd within 2^-52 of 1/d: the product is at
// most 3 units of its last place off, and 4 go to the next multiple of 8).  Rounded
// as an integer, which leaves an infinite product infinite and NaN NaN.
__device__ __forceinline__ float div_by_rounded(float a, double rd) {
  const uint64_t v = __builtin_bit_cast(uint64_t, double(a) * rd);
  return float(__builtin_bit_cast(double, (v + 4) & ~uint64_t(7)));
}
// Four quotients with one test for all.
__device__ __forceinline__ void div4_by(const float a[4], double r0, double r1, double r2, double r3, float q[4]) {
  q[0] = div_by(a[0], r0);
  q[1] = div_by(a[1], r1);
  q[2] = div_by(a[2], r2);
  q[3] = div_by(a[3], r3);
  if (__builtin_expect(int(subnormal(q[0])) | int(subnormal(q[1])) | int(subnormal(q[2])) | int(subnormal(q[3])), 0)) {
    q[0] = div_again(q[0], a[0], r0);
    q[1] = div_again(q[1], a[1], r1);
    q[2] = div_again(q[2], a[2], r2);
    q[3] = div_again(q[3], a[3], r3);
  }
}
// 1/d in FP64 for d != 0: the FP32 reciprocal and two Newton steps (a divisor
// beyond the range where that reciprocal is a normal number: the division).  NaN for
// an infinite d: it comes of infinite coefficients, whose row is infinite or NaN, and
// so is the quotient NaN, not 0.
__device__ __forceinline__ double recip64(float d) {
  const double dd = double(d);
  const float a = __builtin_fabsf(d);
  if (!(a >= 0x1p-100f && a <= 0x1p100f)) return a == __builtin_inff() ? __builtin_nan("") : 1.0 / dd;
  double y = double(__builtin_amdgcn_rcpf(d));
  y = __builtin_fma(__builtin_fma(-dd, y, 1.0), y, y);
  return __builtin_fma(__builtin_fma(-dd, y, 1.0), y, y);
}

// Wavefront sum of a double in the fixed xor-butterfly order (masks 32..1);
// every lane ends with the same bits.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int m = 32; m >= 1; m >>= 1) v = v + __shfl_xor(v, m, 64);
  return v;
}

// Block -> worklist position.  Consecutive workgroups go round-robin to the 8
// XCDs; giving each XCD a contiguous (Morton-ordered) run of tiles keeps the
// face halos of a tile in the L2 of the XCD that reads them.
// n: the launch's work items (its grid, rounded up to a multiple of 8 with the
// swizzle).
__device__ __forceinline__ int work_index(int xcd_swizzle, int n) {
  const int b = blockIdx.x;
  const int per = (n + 7) >> 3;
  return xcd_swizzle ? (b & 7) * per + (b >> 3) : b;
}

// Each tile is worked by exactly one wavefront with its own LDS region, so
// staging only needs ordering inside the wavefront.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ---------------------------------------------------------------------------
// Kernel flags
// ---------------------------------------------------------------------------
enum : int {
  F_ZERO_X = 1,      // X is implicitly zero (first sweep)
  F_GHOST_ZERO = 2,  // ghost X is zero (V-cycle downstroke)
  F_VCYCLE = 4,      // V-cycle mode: rhs from rhsv; restriction into rhsv (ghosts +=)
  F_SWIZZLE = 16,    // XCD-aware tile order
  F_CHECK_DONE = 32, // skip tiles of converged problems
  F_DOT_RZ = 64,     // last colour pass of a level's up-sweep: also the r.z partial of each LEAF tile
  F_INERT = 128,     // a CG iteration's launch: tiles the solve's init found inert are skipped
};

// A problem's done flag, loaded with the tile's data (without F_CHECK_DONE the face
// masks stand in as a readable address) and tested once that is here: tested by a
// load of its own it cost every kernel of the iteration another memory round trip
// (adaptive 256^3 problem: the operator 6.73 -> 6.42 us, the residual update 5.19 ->
// 4.77, restriction from 3,232 tiles 4.40 -> 4.20; large pools within 1 %).
__device__ __forceinline__ uint32_t done_load(const Ctx& c, const TileRec& T, int flags) {
  return *((flags & F_CHECK_DONE) ? reinterpret_cast<const uint32_t*>(&c.ps[T.prob].done)
                                  : reinterpret_cast<const uint32_t*>(c.fmask));
}
__device__ __forceinline__ bool done_test(uint32_t word, int flags) {
  __asm__("" : "+v"(word));
  return (flags & F_CHECK_DONE) && word;
}
// A problem's state as one load of the wavefront (word `lane` of it), its fields
// taken from the lanes once they are needed: the load goes out with the partials'.
__device__ __forceinline__ uint32_t state_word(const ProbState* ps) {
  constexpr int kWords = int(sizeof(ProbState) / 4);
  static_assert(kWords <= 64, "one word a lane");
  return reinterpret_cast<const uint32_t*>(ps)[min(lane_id(), kWords - 1)];
}
__device__ __forceinline__ ProbState state_of(uint32_t word) {
  union {
    uint32_t w[sizeof(ProbState) / 4];
    ProbState s;
  } u;
  __asm__("" : "+v"(word));
#pragma unroll
  for (int i = 0; i < int(sizeof(ProbState) / 4); i++) u.w[i] = uint32_t(__builtin_amdgcn_readlane(int(word), i));
  return u.s;
}


__device__ __forceinline__ void unpack8(float4 a, float4 b, float v[8]) {
  v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w; v[4] = b.x; v[5] = b.y; v[6] = b.z; v[7] = b.w;
}
// Cells of one parity of a k-pencil held as two float4 (k 0..3, 4..7).
__device__ __forceinline__ float4 even4(float4 a, float4 b) { return make_float4(a.x, a.z, b.x, b.z); }
__device__ __forceinline__ float4 odd4(float4 a, float4 b) { return make_float4(a.y, a.w, b.y, b.w); }
__device__ __forceinline__ float4 sel4(bool p, float4 if_false, float4 if_true) {
  return make_float4(p ? if_true.x : if_false.x, p ? if_true.y : if_false.y, p ? if_true.z : if_false.z,
                     p ? if_true.w : if_false.w);
}
__device__ __forceinline__ float comp4(float4 v, int m) { return m == 0 ? v.x : (m == 1 ? v.y : (m == 2 ? v.z : v.w)); }

// ---------------------------------------------------------------------------
// Colour-split layout of the V-cycle arrays (z on every level, its rhs and the
// down-sweep scratch).  Within a tile the 256 cells of colour 0 ((i+j+k) even)
// come first, then the 256 of colour 1; lane l = (i,j) keeps its four cells of
// each colour at [colour*256 + l*4, +4) in k order.  A red-black colour pass
// then reads the updated colour's rhs and writes its x as contiguous halves,
// and a neighbour's other-colour quad lines up component by component with the
// lane's own updated quad.  Channels seen by the caller and the CG vectors keep
// the natural order.
// ---------------------------------------------------------------------------
__host__ __device__ __forceinline__ int split_cell(int i, int j, int k) {
  return (((i + j + k) & 1) << 8) | (((i << 3) | j) << 2) | (k >> 1);
}
__host__ __device__ __forceinline__ int split_index(int cell) { return split_cell(cell >> 6, (cell >> 3) & 7, cell & 7); }
// colour of the even-k cells of pencil pl = (i,j)
__device__ __forceinline__ int even_colour(int pl) { return ((pl >> 3) + pl) & 1; }
// pencil pl of a tile (tile = the tile's first value) as natural float4 halves
template <class V>
__device__ __forceinline__ void load_pencil_split(const V* __restrict__ tile, int pl, float4& a, float4& b) {
  const bool q0 = even_colour(pl);
  const float4 h0 = load4(tile + pl * 4), h1 = load4(tile + 256 + pl * 4);
  const float4 E = sel4(q0, h0, h1), O = sel4(q0, h1, h0);
  a = make_float4(E.x, O.x, E.y, O.y);
  b = make_float4(E.z, O.z, E.w, O.w);
}
template <class V>
__device__ __forceinline__ void store_pencil_split(V* __restrict__ tile, int pl, float4 a, float4 b) {
  const bool q0 = even_colour(pl);
  const float4 E = even4(a, b), O = odd4(a, b);
  store4(tile + pl * 4, sel4(q0, E, O));
  store4(tile + 256 + pl * 4, sel4(q0, O, E));
}
template <class V>
__device__ __forceinline__ void load8_split(const V* __restrict__ tile, int pl, float v[8]) {
  float4 a, b;
  load_pencil_split(tile, pl, a, b);
  unpack8(a, b, v);
}
template <class V>
__device__ __forceinline__ void store8_split(V* __restrict__ tile, int pl, const float v[8]) {
  store_pencil_split(tile, pl, make_float4(v[0], v[1], v[2], v[3]), make_float4(v[4], v[5], v[6], v[7]));
}
// natural cells (i,j,K0..K0+3) of pencil pl, K0 in {0, 4}
template <class V>
__device__ __forceinline__ float4 load_quad_split(const V* __restrict__ tile, int pl, int K0) {
  const bool q0 = even_colour(pl);
  const float2 h0 = load2(tile + pl * 4 + (K0 >> 1)), h1 = load2(tile + 256 + pl * 4 + (K0 >> 1));
  const float2 E = q0 ? h1 : h0, O = q0 ? h0 : h1;
  return make_float4(E.x, O.x, E.y, O.y);
}
template <class V>
__device__ __forceinline__ void store_quad_split(V* __restrict__ tile, int pl, int K0, float4 v) {
  const bool q0 = even_colour(pl);
  const float2 E = make_float2(v.x, v.z), O = make_float2(v.y, v.w);
  store2(tile + pl * 4 + (K0 >> 1), q0 ? O : E);
  store2(tile + 256 + pl * 4 + (K0 >> 1), q0 ? E : O);
}

// Raw loads: a quad or a single value of V-typed storage as loaded (FP32
// values, or the bits of 16-bit ones), widened to FP32 only after every load of
// a tile has been issued; a widening inside the branch that loads a value would
// make that branch wait for its load.  hold() puts an empty asm the compiler
// cannot see through on the raw bits, so that it cannot move the widening up.
// A device array of zeros as large as one tile of FP64 values: loads of values
// that are 0 by definition read it (L2-resident) instead of being skipped.
// Nothing writes it; it is not declared const so that it sits in global
// memory like the arrays it stands in for (one kind of load for both).
__device__ __align__(16) float kZeroPage[1024] = {};
template <class V> __device__ __forceinline__ const V* zero_page() { return reinterpret_cast<const V*>(kZeroPage); }
// The face masks of a tile whose masks are all M_OPEN_INT (tr_all_open), in
// both layouts (512 cell bytes; 128 colour-split words), read in place of the
// tile's own: a load that stays in the caches instead of one from HBM.
#define CG_R8(x) x, x, x, x, x, x, x, x
__device__ __align__(16) uint32_t kOpenPage[128] = {CG_R8(CG_R8(0x7f7f7f7fu)), CG_R8(CG_R8(0x7f7f7f7fu))};
#undef CG_R8
__device__ __forceinline__ const uint8_t* own_masks(const Ctx& c, const TileRec& T) {
  return tr_all_open(T) ? reinterpret_cast<const uint8_t*>(kOpenPage) : c.fmask + size_t(T.self) * 512;
}
__device__ __forceinline__ const uint32_t* own_split_masks(const Ctx& c, const TileRec& T) {
  return tr_all_open(T) ? kOpenPage : c.fsplit + size_t(T.self) * 128;
}

template <class V> struct RawV;
template <> struct RawV<float> { typedef float4 Q; typedef float S; typedef float2 S2; };
template <> struct RawV<bf16> { typedef uint2 Q; typedef uint32_t S; typedef uint32_t S2; };
template <> struct RawV<f16> { typedef uint2 Q; typedef uint32_t S; typedef uint32_t S2; };
// a pair of consecutive values
__device__ __forceinline__ float2 load2_raw(const float* p) { return *reinterpret_cast<const float2*>(p); }
__device__ __forceinline__ uint32_t load2_raw(const bf16* p) { return *reinterpret_cast<const uint32_t*>(p); }
__device__ __forceinline__ uint32_t load2_raw(const f16* p) { return *reinterpret_cast<const uint32_t*>(p); }
template <class V> __device__ __forceinline__ float2 pair_f(typename RawV<V>::S2 v);
template <> __device__ __forceinline__ float2 pair_f<float>(float2 v) { return v; }
template <> __device__ __forceinline__ float2 pair_f<bf16>(uint32_t v) { return make_float2(bf_lo(v), bf_hi(v)); }
template <> __device__ __forceinline__ float2 pair_f<f16>(uint32_t v) { return make_float2(h_lo(v), h_hi(v)); }
__device__ __forceinline__ float4 load_q_raw(const float* p) { return *reinterpret_cast<const float4*>(p); }
__device__ __forceinline__ uint2 load_q_raw(const bf16* p) { return *reinterpret_cast<const uint2*>(p); }
__device__ __forceinline__ uint2 load_q_raw(const f16* p) { return *reinterpret_cast<const uint2*>(p); }
__device__ __forceinline__ float load_s_raw(const float* p) { return *p; }
__device__ __forceinline__ uint32_t load_s_raw(const bf16* p) { return *reinterpret_cast<const uint16_t*>(p); }
__device__ __forceinline__ uint32_t load_s_raw(const f16* p) { return *reinterpret_cast<const uint16_t*>(p); }
template <class V> __device__ __forceinline__ float4 quad_f(typename RawV<V>::Q q);
template <> __device__ __forceinline__ float4 quad_f<float>(float4 q) { return q; }
template <> __device__ __forceinline__ float4 quad_f<bf16>(uint2 q) { return make_float4(bf_lo(q.x), bf_hi(q.x), bf_lo(q.y), bf_hi(q.y)); }
template <> __device__ __forceinline__ float4 quad_f<f16>(uint2 q) { return make_float4(h_lo(q.x), h_hi(q.x), h_lo(q.y), h_hi(q.y)); }
template <class V> __device__ __forceinline__ float single_f(typename RawV<V>::S v);
template <> __device__ __forceinline__ float single_f<float>(float v) { return v; }
template <> __device__ __forceinline__ float single_f<bf16>(uint32_t v) { return bf_lo(v); }
template <> __device__ __forceinline__ float single_f<f16>(uint32_t v) { return h_lo(v); }
__device__ __forceinline__ void hold(float4&) {}
__device__ __forceinline__ void hold(float&) {}
// the same for an FP32 value whose later select must not pull its wait forward
__device__ __forceinline__ void hold_f(float& v) { __asm__("" : "+v"(v)); }
__device__ __forceinline__ void hold8(float v[8]) {
#pragma unroll
  for (int k = 0; k < 8; k++) hold_f(v[k]);
}
__device__ __forceinline__ void hold(uint2& q) { __asm__("" : "+v"(q.x), "+v"(q.y)); }
__device__ __forceinline__ void hold(uint32_t& v) { __asm__("" : "+v"(v)); }

// Raw loads of a colour-split pencil (both colour halves' quads), widened and
// put in natural order only after every load of the tile is out.
template <class V> struct RawPencil { typename RawV<V>::Q h0, h1; };
template <class V>
__device__ __forceinline__ RawPencil<V> load_pencil_split_raw(const V* __restrict__ tile, int pl) {
  RawPencil<V> r;
  r.h0 = load_q_raw(tile + pl * 4);
  r.h1 = load_q_raw(tile + 256 + pl * 4);
  return r;
}
// load_pencil_split's arrangement of the raw halves
template <class V>
__device__ __forceinline__ void pencil_split_f(const RawPencil<V>& r, int pl, float4& a, float4& b) {
  const bool q0 = even_colour(pl);
  const float4 h0 = quad_f<V>(r.h0), h1 = quad_f<V>(r.h1);
  const float4 E = sel4(q0, h0, h1), O = sel4(q0, h1, h0);
  a = make_float4(E.x, O.x, E.y, O.y);
  b = make_float4(E.z, O.z, E.w, O.w);
}
// hold for every storage type (FP32 values too: their rearrangement must not
// pull the wait forward either)
__device__ __forceinline__ void hold_all(float4& q) {
  hold_f(q.x);
  hold_f(q.y);
  hold_f(q.z);
  hold_f(q.w);
}
__device__ __forceinline__ void hold_all(uint2& q) { hold(q); }
__device__ __forceinline__ void hold_all(float& v) { hold_f(v); }
__device__ __forceinline__ void hold_all(uint32_t& v) { hold(v); }
__device__ __forceinline__ void hold_all(float2& v) {
  hold_f(v.x);
  hold_f(v.y);
}
template <class V> __device__ __forceinline__ void hold_all(RawPencil<V>& r) {
  hold_all(r.h0);
  hold_all(r.h1);
}

// ---------------------------------------------------------------------------
// Tile + halo staging
// ---------------------------------------------------------------------------
struct TileLDS {
  float4 xs[2][100];   // pencils (i,j), i,j in -1..8, index (i+1)*10 + (j+1); [0]: k 0..3, [1]: k 4..7
};

// Face-mask bits of a cell (Ctx::fmask).
enum : int { M_INT = 64 };
// A cell with all six faces uncut and INTERIOR.
constexpr uint32_t M_OPEN_INT = 0x7fu;

// The masks of a pencil's four colour cells k = p, 2+p, 4+p, 6+p (byte m = cell
// 2m + p) from its eight (byte k = cell k).
__device__ __forceinline__ uint32_t quad_mask(uint64_t m, bool p) {
  const uint64_t s = p ? (m >> 8) : m;
  return uint32_t(s & 0xffu) | uint32_t((s >> 8) & 0xff00u) | uint32_t((s >> 16) & 0xff0000u) |
         uint32_t((s >> 24) & 0xff000000u);
}

struct Stencil {
  float own[8];
  uint64_t m;          // own face masks, one byte per cell
  float xkm, xkp;      // k-halo values (z- neighbour cell (i,j,7), z+ neighbour cell (i,j,0))
  float b_int, b_f[6]; // base coefficients: inside the tile and across face f
  float h;
  bool open;           // tr_all_open
};
__device__ __forceinline__ void stencil_coeffs(const TileRec& T, const float bcv[7], Stencil& S) {
  S.h = T.h;
  S.open = tr_all_open(T);
  S.b_int = bcv[6];
  for (int f = 0; f < 6; f++) S.b_f[f] = bcv[f];
}

// Stage tile T's X values (zeros where the flags say so) and face masks.
//   zero_all:   treat X as 0 everywhere (first sweep from a zero guess)
//   ghost_zero: treat X of GHOST tiles as 0 (downstroke of the V-cycle)
//   bcv:        the 7 face coefficients of the view (faces x-..z+, inside)
// X holds active tiles, XG ghost tiles (they differ only for the damped-Jacobi
// ping-pong, where ghost values stay in the primary buffer).  SPLIT: X and XG
// are V-cycle arrays in the colour-split layout (the staged pencils are in
// natural order either way).
template <class V>
struct StageRaw {
  RawPencil<V> own, halo;
  typename RawV<V>::S km, kp;
  uint64_t m;
};
// A pencil's raw loads in either layout: colour-split (SPLIT, both halves'
// quads) or natural (cells 0..3 and 4..7).
template <bool SPLIT, class V>
__device__ __forceinline__ RawPencil<V> load_pencil_any_raw(const V* __restrict__ tile, int pl) {
  if (SPLIT) return load_pencil_split_raw(tile, pl);
  RawPencil<V> r;
  r.h0 = load_q_raw(tile + pl * 8);
  r.h1 = load_q_raw(tile + pl * 8 + 4);
  return r;
}
template <bool SPLIT, class V>
__device__ __forceinline__ void pencil_any_f(const RawPencil<V>& r, int pl, float4& a, float4& b) {
  if (SPLIT) {
    pencil_split_f(r, pl, a, b);
  } else {
    a = quad_f<V>(r.h0);
    b = quad_f<V>(r.h1);
  }
}
// The halo ring's lanes: lane g*8 + t (g < 4) fetches one neighbour pencil
//   g = 0: x- (pencil (7,t) of nbr 0), 1: x+ ((0,t) of nbr 3), 2: y- ((t,7) of nbr 1), 3: y+ ((t,0) of nbr 4)
// into LDS slot ring_dst (pencil index (i+1)*10 + (j+1) of the 10x10 frame).
__device__ __forceinline__ int ring_face(int g) { return pick4(g, 0, 3, 1, 4); }
__device__ __forceinline__ int ring_src(int g, int t) { return pick4(g, 56 + t, t, t * 8 + 7, t * 8); }
__device__ __forceinline__ int ring_dst(int g, int t) { return pick4(g, t + 1, 91 + t, (t + 1) * 10, (t + 1) * 10 + 9); }

// The loads of stage_tile, as raw bits: the own pencil, the face masks, the
// halo pencil of lanes 0..31 and the two k halos.  Every load is
// unconditional: a value that counts as 0 (a zero guess, outside the grid, a
// ghost in the down-sweep, lanes 32..63 of the ring) is read from the zero
// page, so no load sits in a branch whose merge would make the wavefront wait.
template <bool SPLIT, class V>
__device__ __forceinline__ StageRaw<V> stage_issue(const Ctx& c, const TileRec& T, const V* __restrict__ X,
                                                   const V* __restrict__ XG, bool zero_all, bool ghost_zero) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const bool own_ghost = tr_type(T) == T_GHOST;
  const V* zp = zero_page<V>();
  StageRaw<V> r;
  const bool own_zero = zero_all || (ghost_zero && own_ghost);
  r.own = load_pencil_any_raw<SPLIT>(own_zero ? zp : (own_ghost ? XG : X) + size_t(T.self) * 512, lane);
  r.m = load_ct8(own_masks(c, T) + lane * 8);
  {
    const int g = (lane >> 3) & 3, t = lane & 7;
    const int f = ring_face(g);
    const int n = pick4(g, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
    const bool gh = tr_ntype(T, f) == T_GHOST;
    // else x = 0 (outside the grid: GMGSolver.cu:120-122)
    const bool ok = lane < 32 && n >= 0 && !(zero_all || (ghost_zero && gh));
    r.halo = load_pencil_any_raw<SPLIT>(ok ? (gh ? XG : X) + size_t(n) * 512 : zp, ok ? ring_src(g, t) : 0);
  }
  // k halos: cell (i,j,7) of the z- neighbour, (i,j,0) of the z+ neighbour
  const int o7 = SPLIT ? split_cell(i, j, 7) : lane * 8 + 7, o0 = SPLIT ? split_cell(i, j, 0) : lane * 8;
  const int nm = T.nbr[2], np = T.nbr[5];
  const bool ghm = tr_ntype(T, 2) == T_GHOST, ghp = tr_ntype(T, 5) == T_GHOST;
  const bool okm = nm >= 0 && !(zero_all || (ghost_zero && ghm));
  const bool okp = np >= 0 && !(zero_all || (ghost_zero && ghp));
  r.km = load_s_raw(okm ? (ghm ? XG : X) + size_t(nm) * 512 + o7 : zp);
  r.kp = load_s_raw(okp ? (ghp ? XG : X) + size_t(np) * 512 + o0 : zp);
  return r;
}
// The rest of stage_tile: one wait, then the values into LDS and the stencil.
template <bool SPLIT, class V>
__device__ __forceinline__ void stage_commit(StageRaw<V>& r, const TileRec& T, const float bcv[7], TileLDS& L,
                                             Stencil& S) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  hold_all(r.own);
  hold_all(r.halo);
  hold_all(r.km);
  hold_all(r.kp);
  float4 a, b;
  pencil_any_f<SPLIT>(r.own, lane, a, b);
  S.own[0] = a.x; S.own[1] = a.y; S.own[2] = a.z; S.own[3] = a.w;
  S.own[4] = b.x; S.own[5] = b.y; S.own[6] = b.z; S.own[7] = b.w;
  S.m = r.m;
  const int pc = (i + 1) * 10 + (j + 1);
  L.xs[0][pc] = a;
  L.xs[1][pc] = b;
  if (lane < 32) {
    const int g = lane >> 3, t = lane & 7;
    float4 v0, v1;
    pencil_any_f<SPLIT>(r.halo, ring_src(g, t), v0, v1);
    L.xs[0][ring_dst(g, t)] = v0;
    L.xs[1][ring_dst(g, t)] = v1;
  }
  S.xkm = single_f<V>(r.km);
  S.xkp = single_f<V>(r.kp);
  stencil_coeffs(T, bcv, S);
}

// Stage tile T's X values (zeros where the flags say so) and face masks.
//   zero_all:   treat X as 0 everywhere (first sweep from a zero guess)
//   ghost_zero: treat X of GHOST tiles as 0 (downstroke of the V-cycle)
//   bcv:        the 7 face coefficients of the view (faces x-..z+, inside)
// X holds active tiles, XG ghost tiles (they differ only for the damped-Jacobi
// ping-pong, where ghost values stay in the primary buffer).  SPLIT: X and XG
// are V-cycle arrays in the colour-split layout (the staged pencils are in
// natural order either way).
template <bool SPLIT, class V>
__device__ __forceinline__ void stage_tile(const Ctx& c, const TileRec& T, const V* __restrict__ X,
                                           const V* __restrict__ XG, bool zero_all, bool ghost_zero,
                                           const float bcv[7], TileLDS& L, Stencil& S) {
  StageRaw<V> r = stage_issue<SPLIT>(c, T, X, XG, zero_all, ghost_zero);
  stage_commit<SPLIT>(r, T, bcv, L, S);
}

// The CG operator's staging, where p is not stored on GHOST tiles: a GHOST
// cell's value is its parent cell's if that cell is INTERIOR, else 0 (the
// copy into ghost tiles the reference makes before the operator,
// PoissonGrid.cu:585-605), read from the parent (a LEAF tile one level up)
// wherever the tile itself or a face neighbour in its halo is a GHOST.  FP32,
// natural layout; every load unconditional as in stage_issue.
struct StagePG {
  float4 own0, own1, halo0, halo1;
  uint32_t own_ct, halo_ct, km_ct, kp_ct;
  float km, kp;
  uint64_t m;
  bool halo_gh;  // the lane's ring pencil is a GHOST's (from its parent)
};
// Cell of `parent` that holds cell (i, j, 2 k4 .. 2 k4 + 1) of its child with
// octant o (the pencil's four parent cells start at k4 = 0).
__device__ __forceinline__ size_t pg_cell(int parent, int o, int i, int j, int k4) {
  return size_t(parent) * 512 +
         size_t((((o & 1) * 4 + (i >> 1)) * 8 + (((o >> 1) & 1) * 4 + (j >> 1))) * 8 + ((o >> 2) & 1) * 4 + k4);
}
__device__ __forceinline__ StagePG stage_issue_pg(const Ctx& c, const TileRec& T, const float* __restrict__ X) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const bool own_ghost = tr_type(T) == T_GHOST;
  const int oct = tr_octant(T);
  const float* zp = zero_page<float>();
  const uint32_t* zw = reinterpret_cast<const uint32_t*>(kZeroPage);
  StagePG r;
  // own pencil, or its four parent cells and their types
  const size_t po = pg_cell(own_ghost ? T.parent : 0, oct, i, j, 0);
  const float* own = own_ghost ? X + po : X + size_t(T.self) * 512 + lane * 8;
  r.own0 = *reinterpret_cast<const float4*>(own);
  r.own1 = *reinterpret_cast<const float4*>(own_ghost ? zp : own + 4);
  r.own_ct = *(own_ghost ? reinterpret_cast<const uint32_t*>(c.ctype + po) : zw);
  r.m = load_ct8(own_masks(c, T) + lane * 8);
  {  // ring: lanes 0..31, one neighbour pencil each (x = 0 outside the grid)
    const int g = (lane >> 3) & 3, t = lane & 7;
    const int f = ring_face(g);
    const int n = pick4(g, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
    const int npar = pick4(g, uni(T.nbr_parent[0]), uni(T.nbr_parent[3]), uni(T.nbr_parent[1]), uni(T.nbr_parent[4]));
    const bool ok = lane < 32 && n >= 0;
    const bool gh = ok && tr_ntype(T, f) == T_GHOST;
    const int sp = ring_src(g, t);                        // the neighbour's pencil si * 8 + sj
    const int no = oct ^ (g < 2 ? 1 : 2);                 // its octant: across x or y
    const size_t pn = pg_cell(gh ? npar : 0, no, sp >> 3, sp & 7, 0);
    const float* h = !ok ? zp : (gh ? X + pn : X + size_t(n) * 512 + sp * 8);
    r.halo0 = *reinterpret_cast<const float4*>(h);
    r.halo1 = *reinterpret_cast<const float4*>((ok && !gh) ? h + 4 : zp);
    r.halo_ct = *(gh ? reinterpret_cast<const uint32_t*>(c.ctype + pn) : zw);
    r.halo_gh = gh;
  }
  // k halos: cell (i,j,7) of the z- neighbour, (i,j,0) of the z+ neighbour
  const int nm = T.nbr[2], np = T.nbr[5];
  const bool ghm = nm >= 0 && tr_ntype(T, 2) == T_GHOST, ghp = np >= 0 && tr_ntype(T, 5) == T_GHOST;
  const size_t pm = pg_cell(ghm ? T.nbr_parent[2] : 0, oct ^ 4, i, j, 3);
  const size_t pp = pg_cell(ghp ? T.nbr_parent[5] : 0, oct ^ 4, i, j, 0);
  r.km = *(nm < 0 ? zp : (ghm ? X + pm : X + size_t(nm) * 512 + lane * 8 + 7));
  r.kp = *(np < 0 ? zp : (ghp ? X + pp : X + size_t(np) * 512 + lane * 8));
  r.km_ct = *(ghm ? c.ctype + pm : reinterpret_cast<const uint8_t*>(zw));
  r.kp_ct = *(ghp ? c.ctype + pp : reinterpret_cast<const uint8_t*>(zw));
  return r;
}
// A ghost pencil from its four parent cells: cells 2m and 2m + 1 take parent
// value m if that cell is INTERIOR, else 0.
__device__ __forceinline__ void pg_expand(float4 q, uint32_t ct, float4& a, float4& b) {
  const float v0 = (ct & C_INT) ? q.x : 0.f, v1 = ((ct >> 8) & C_INT) ? q.y : 0.f;
  const float v2 = ((ct >> 16) & C_INT) ? q.z : 0.f, v3 = ((ct >> 24) & C_INT) ? q.w : 0.f;
  a = make_float4(v0, v0, v1, v1);
  b = make_float4(v2, v2, v3, v3);
}
__device__ __forceinline__ void stage_commit_pg(StagePG& r, const TileRec& T, const float bcv[7], TileLDS& L,
                                                Stencil& S) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  hold_all(r.own0);
  hold_all(r.own1);
  hold_all(r.halo0);
  hold_all(r.halo1);
  hold_all(r.km);
  hold_all(r.kp);
  hold_all(r.own_ct);
  hold_all(r.halo_ct);
  hold_all(r.km_ct);
  hold_all(r.kp_ct);
  float4 a = r.own0, b = r.own1;
  if (tr_type(T) == T_GHOST) pg_expand(r.own0, r.own_ct, a, b);
  S.own[0] = a.x; S.own[1] = a.y; S.own[2] = a.z; S.own[3] = a.w;
  S.own[4] = b.x; S.own[5] = b.y; S.own[6] = b.z; S.own[7] = b.w;
  S.m = r.m;
  const int pc = (i + 1) * 10 + (j + 1);
  L.xs[0][pc] = a;
  L.xs[1][pc] = b;
  if (lane < 32) {
    const int g = lane >> 3, t = lane & 7;
    float4 v0 = r.halo0, v1 = r.halo1;
    if (r.halo_gh) pg_expand(r.halo0, r.halo_ct, v0, v1);
    L.xs[0][ring_dst(g, t)] = v0;
    L.xs[1][ring_dst(g, t)] = v1;
  }
  const bool ghm = T.nbr[2] >= 0 && tr_ntype(T, 2) == T_GHOST, ghp = T.nbr[5] >= 0 && tr_ntype(T, 5) == T_GHOST;
  S.xkm = (ghm && !(r.km_ct & C_INT)) ? 0.f : r.km;
  S.xkp = (ghp && !(r.kp_ct & C_INT)) ? 0.f : r.kp;
  stencil_coeffs(T, bcv, S);
}

// Face coefficients of tile T seen with the subtree view at level sl
// (GMGSolver.cu:26-39): 1/h^2 and (2/h/3)/h as the reference forms them; an
// absent neighbour counts as the tile's own type (GMGSolver.cu:118-122).
__host__ __device__ __forceinline__ void view_coeffs(const TileRec& T, int sl, float bcv[7]) {
  const float ooh = 1.0f / T.h;
  const float cll = ooh * ooh;
  const float clg = ((2.0f * ooh) / 3.0f) * ooh;
  const uint8_t to = subtree_type(tr_type(T), tr_level(T), sl);
  bcv[6] = base_coeff(to, to, cll, clg);
  for (int f = 0; f < 6; f++) {
    const uint8_t tn = (T.nbr[f] < 0) ? to : subtree_type(tr_ntype(T, f), tr_level(T), sl);
    bcv[f] = base_coeff(to, tn, cll, clg);
  }
}


// The 7-point row of one cell: faces visited in the reference's order x-, x+,
// y-, y+, z-, z+ (GMGSolver.cu:62-73); returns A x and D (times h^3, 0 off
// INTERIOR cells).
// The NEUMANN cuts and the INTERIOR test come from the cell's face mask m: a
// NEUMANN cell on either side of a face cuts it (coefficient 0).
// BITS (the colour sweeps' four cells): bit e of m as all ones or zero (one
// bitfield extract), so that the coefficient or +0 comes from one AND rather
// than a compare and a select; the empty asm keeps the compiler from turning
// the AND back into a select.  The same value either way; the eight-cell
// operator rows keep the select, which needs fewer registers there.
template <bool BITS = false>
__device__ __forceinline__ void cell_row_m(float x0, uint32_t m, const float xn[6], const float bc[6], float h, float& ax,
                                           float& dg) {
  float s = 0.f, d = 0.f;
#pragma unroll
  for (int e = 0; e < 6; e++) {
    float cf;
    if (BITS) {
      uint32_t open = uint32_t(int32_t(m << (31 - e)) >> 31);
      __asm__("" : "+v"(open));
      cf = __uint_as_float(__float_as_uint(bc[e]) & open);
    } else {
      cf = (m & (1u << e)) ? bc[e] : 0.f;
    }
    s = __builtin_fmaf(cf, x0 - xn[e], s);
    d = d + cf;
  }
  const bool in = m & M_INT;
  ax = in ? ((s * h) * h) * h : 0.f;
  dg = in ? ((d * h) * h) * h : 0.f;
}

// The four i/j-neighbour pencils of a lane (values and cell types).
struct NbrPencils {
  float4 im0, im1, ip0, ip1, jm0, jm1, jp0, jp1;
};
__device__ __forceinline__ NbrPencils lds_nbrs(const TileLDS& L) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const int pc = (i + 1) * 10 + (j + 1);
  NbrPencils N;
  N.im0 = L.xs[0][pc - 10]; N.im1 = L.xs[1][pc - 10];
  N.ip0 = L.xs[0][pc + 10]; N.ip1 = L.xs[1][pc + 10];
  N.jm0 = L.xs[0][pc - 1];  N.jm1 = L.xs[1][pc - 1];
  N.jp0 = L.xs[0][pc + 1];  N.jp1 = L.xs[1][pc + 1];
  return N;
}

// A x (and its diagonal) on all 8 cells of the lane, its i/j neighbours read from
// the staged pencils.  Open tiles take the short rows, one half of the pencil at a
// time (both at once need more registers than eight wavefronts a SIMD leave, and
// HBM-bound passes need those wavefronts).  The apply of the refined 45,054-tile
// scene 61 -> 55 us, of the 256-problem pool 1089 -> 1060 us (5.9 TB/s).
template <bool WANT_AX, bool WANT_D>
__device__ __forceinline__ void apply_pencil(const TileLDS& L, const Stencil& S, float ax[8], float dg[8]) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const float bim = (i == 0) ? S.b_f[0] : S.b_int;
  const float bip = (i == 7) ? S.b_f[3] : S.b_int;
  const float bjm = (j == 0) ? S.b_f[1] : S.b_int;
  const float bjp = (j == 7) ? S.b_f[4] : S.b_int;
  if (WANT_AX && !WANT_D && S.open) {
    // every cell INTERIOR, no face cut: the base coefficients as they are
    // (cell_row_m's sums; 13 or 15 operations a cell instead of about 30), one
    // half of the pencil at a time
    const int pc = (i + 1) * 10 + (j + 1);
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const float4 im = L.xs[h][pc - 10], ip = L.xs[h][pc + 10], jm = L.xs[h][pc - 1], jp = L.xs[h][pc + 1];
#pragma unroll
      for (int m = 0; m < 4; m++) {
        const int k = 4 * h + m;
        const float x0 = S.own[k];
        float s = 0.f;
        s = __builtin_fmaf(bim, x0 - comp4(im, m), s);
        s = __builtin_fmaf(bip, x0 - comp4(ip, m), s);
        s = __builtin_fmaf(bjm, x0 - comp4(jm, m), s);
        s = __builtin_fmaf(bjp, x0 - comp4(jp, m), s);
        s = __builtin_fmaf((k == 0) ? S.b_f[2] : S.b_int, x0 - ((k == 0) ? S.xkm : S.own[k - 1]), s);
        s = __builtin_fmaf((k == 7) ? S.b_f[5] : S.b_int, x0 - ((k == 7) ? S.xkp : S.own[k + 1]), s);
        ax[k] = ((s * S.h) * S.h) * S.h;
      }
    }
    return;
  }
  const NbrPencils N = lds_nbrs(L);
  float xim[8], xip[8], xjm[8], xjp[8];
  unpack8(N.im0, N.im1, xim);
  unpack8(N.ip0, N.ip1, xip);
  unpack8(N.jm0, N.jm1, xjm);
  unpack8(N.jp0, N.jp1, xjp);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const float xn[6] = {xim[k], xip[k], xjm[k], xjp[k], (k == 0) ? S.xkm : S.own[k - 1], (k == 7) ? S.xkp : S.own[k + 1]};
    const float bc[6] = {bim, bip, bjm, bjp, (k == 0) ? S.b_f[2] : S.b_int, (k == 7) ? S.b_f[5] : S.b_int};
    float a, d;
    cell_row_m(S.own[k], ct_at(S.m, k), xn, bc, S.h, a, d);
    if (WANT_AX) ax[k] = a;
    if (WANT_D) dg[k] = d;
  }
}

// What a colour update needs of its tile besides values: the face coefficients
// and sizes, and what the record says of the tile.
struct GsCoef {
  const float* bc;  // faces x-..z+, inside
  float h;
  double rd;
  bool open, uniform;
};
__device__ __forceinline__ GsCoef gs_coef(const TileRec& T) {
  return GsCoef{T.bc, T.h, T.rdiag, tr_all_open(T), tr_uniform(T)};
}
// 1/D of a lane's open cells: those inside the pencil (mid) and at its ends
// k = 0 (lo) and k = 7 (hi), the sums formed as cell_row_m forms them (an open
// tile's are finite and not 0).
struct OpenDiag {
  double mid, lo, hi;
};
__device__ __forceinline__ OpenDiag open_diag(const GsCoef& G, float bim, float bip, float bjm, float bjp) {
  if (G.uniform) return OpenDiag{G.rd, G.rd, G.rd};
  const float bi = G.bc[6], d4 = (((0.f + bim) + bip) + bjm) + bjp;
  auto inv = [&](float d) { return recip64(((d * G.h) * G.h) * G.h); };
  return OpenDiag{inv((d4 + bi) + bi), inv((d4 + G.bc[2]) + bi), inv((d4 + bi) + G.bc[5])};
}

// The four updated cells of a red-black colour pass, in split-layout quads:
// cell k = 2m + p of lane (i,j) (p = (color+i+j)&1) with value X0.m, rhs B.m,
// i/j neighbours XIM..XJP (component m: the neighbours' other-colour quads line
// up with the lane's updated quad), the lane's other-colour quad XO and the
// k-halo value xk (cell (i,j,-1) when p = 0, (i,j,8) when p = 1).
// ZERO: every x is 0 (the first pass), so A x = 0.
// A tile whose record says all_open (every cell INTERIOR, no face cut: two thirds
// of the batched workload's) needs no masks, and D takes at most three values a
// lane, one where no face neighbour is a GHOST: its quotients are products with
// the 64-bit 1/D (div_by).  About 200 vector operations a tile instead of 290;
// the other tiles take the general rows and the FP32 division.  The colour pass
// of the 360,472-tile level of a 256-problem pool, in FP32: 319 -> 300 us; on a
// level of 64 tiles, where a pass is one chain of waits: 2.61 -> 2.48 us.
template <bool ZERO = false>
__device__ __forceinline__ float4 gs_quad(float4 X0, float4 XO, float4 XIM, float4 XIP, float4 XJM, float4 XJP,
                                          float xk, float4 B, uint32_t mq, const GsCoef& G, int i, int j, bool p) {
  // k-1 and k+1 neighbours of cell 2m+p
  const float4 XKM = sel4(p, make_float4(xk, XO.x, XO.y, XO.z), XO);
  const float4 XKP = sel4(p, XO, make_float4(XO.y, XO.z, XO.w, xk));
  const float bi = G.bc[6];
  const float bim = (i == 0) ? G.bc[0] : bi;
  const float bip = (i == 7) ? G.bc[3] : bi;
  const float bjm = (j == 0) ? G.bc[1] : bi;
  const float bjp = (j == 7) ? G.bc[4] : bi;
  float nv[4];
  if (G.open) {
    const OpenDiag D = open_diag(G, bim, bip, bjm, bjp);
    const double dlo = p ? D.mid : D.lo, dhi = p ? D.hi : D.mid;  // of m = 0 and m = 3
    const float bkm = p ? bi : G.bc[2], bkp = p ? G.bc[5] : bi;   // of m = 0 (k - 1) and m = 3 (k + 1)
    float res[4], q[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const float x0 = comp4(X0, m);
      float s = 0.f;
      if (!ZERO) {
        s = __builtin_fmaf(bim, x0 - comp4(XIM, m), s);
        s = __builtin_fmaf(bip, x0 - comp4(XIP, m), s);
        s = __builtin_fmaf(bjm, x0 - comp4(XJM, m), s);
        s = __builtin_fmaf(bjp, x0 - comp4(XJP, m), s);
        s = __builtin_fmaf(m == 0 ? bkm : bi, x0 - comp4(XKM, m), s);
        s = __builtin_fmaf(m == 3 ? bkp : bi, x0 - comp4(XKP, m), s);
      }
      res[m] = comp4(B, m) - (ZERO ? 0.f : ((s * G.h) * G.h) * G.h);
    }
    div4_by(res, dlo, D.mid, D.mid, dhi, q);
    return make_float4(X0.x + q[0], X0.y + q[1], X0.z + q[2], X0.w + q[3]);
  }
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const uint32_t mb = mq >> (8 * m);  // bits 0..6 used
    const float bkm = (!p && m == 0) ? G.bc[2] : bi;
    const float bkp = (p && m == 3) ? G.bc[5] : bi;
    const float x0 = comp4(X0, m);
    const float xn[6] = {comp4(XIM, m), comp4(XIP, m), comp4(XJM, m), comp4(XJP, m), comp4(XKM, m), comp4(XKP, m)};
    const float bc[6] = {bim, bip, bjm, bjp, bkm, bkp};
    float ax, dg;
    cell_row_m<true>(x0, mb, xn, bc, G.h, ax, dg);
    float delta = 0.f;
    if ((mb & M_INT) && dg != 0.f) delta = (comp4(B, m) - (ZERO ? 0.f : ax)) / dg;
    nv[m] = x0 + delta;
  }
  return make_float4(nv[0], nv[1], nv[2], nv[3]);
}

// ---------------------------------------------------------------------------
// Per-tile bodies (one wavefront each)
// ---------------------------------------------------------------------------

struct GsLDS {
  float4 xo[100];  // other-colour quads of the tile's pencils and of the halo ring, index (i+1)*10 + (j+1)
};

// Red-black Gauss-Seidel colour sweep of a LEAF|NONLEAF tile (GMGSolver.cu:216-269)
// on the colour-split arrays: reads the tile's two x halves, the updated
// colour's rhs half and the neighbours' other-colour quads; writes the updated
// colour's half (and, from an implicit zero guess, zeros to the other half).
// An INTERIOR cell with D == 0 is left unchanged.
// The sweep is split into its loads (gs_issue: every global load of the tile,
// as raw bits into registers; gs_convert: to FP32), and the rest (gs_stage:
// the other-colour quads into LDS; gs_finish: the update and its stores), so
// that a wavefront issues every load of its tile (or tiles) before it waits
// on any.  A 16-bit value widens with one shift or conversion; done inside the
// branch that loads it, that would make the branch wait for its load, so the
// raw bits are held (an empty asm the compiler cannot see through) until all
// loads are out.
struct GsIn {
  float4 xc, xo, B, halo;
  float4 r0, r1;  // with F_DOT_RZ on a LEAF tile: r of the lane's pencil, cells 0..3 and 4..7
  uint32_t mask;  // the face masks of the lane's four cells of the pass's colour
  float xk;       // k halo: cell (i,j,7) of the z- neighbour (p = 0) or (i,j,0) of the z+ one (p = 1)
  int32_t done;   // the problem's done flag, loaded with the tile's data (used with F_CHECK_DONE only)
};
template <class V>
struct GsRaw {
  typename RawV<V>::Q xc, xo, B, halo;
  typename RawV<V>::S xk;
  float4 r0, r1;
  uint32_t mask;
  int32_t done;
};
// DOT: the pass carries F_DOT_RZ (a separate instance, so that the other
// passes keep their register count).
template <class V, bool DOT = false>
__device__ __forceinline__ GsRaw<V> gs_issue(const Ctx& c, const TileRec& T, const V* X, const V* F, int color,
                                             int flags) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const bool zero_all = flags & F_ZERO_X, ghost_zero = flags & F_GHOST_ZERO;
  const int hc = color << 8, ho = (color ^ 1) << 8;
  // Every load below is unconditional: a value that is 0 by definition (x from
  // a zero guess, outside the grid, a ghost in the down-sweep, the halo of
  // lanes 32..63) is read from the zero page instead of skipped, so no load
  // sits in a branch whose merge would make the wavefront wait for it.
  const V* zp = zero_page<V>();
  const V* tile = zero_all ? zp : X + size_t(T.self) * 512;
  GsRaw<V> g;
  // one unconditional scalar load issued with the others, tested after the LDS
  // stage; without F_CHECK_DONE the face masks stand in as a readable address
  const int32_t* dp = (flags & F_CHECK_DONE) ? &c.ps[T.prob].done : reinterpret_cast<const int32_t*>(c.fmask);
  g.done = *dp;
  g.xc = load_q_raw(tile + hc + lane * 4);
  g.xo = load_q_raw(tile + ho + lane * 4);
  g.mask = own_split_masks(c, T)[color * 64 + lane];
  if (DOT) {
    // r of the lane's pencil on LEAF tiles (zeros otherwise)
    const float* rp = tr_type(T) == T_LEAF ? c.r + size_t(T.self) * 512 : zero_page<float>();
    const float4* r4 = reinterpret_cast<const float4*>(rp + lane * 8);
    g.r0 = r4[0];
    g.r1 = r4[1];
  }
  const V* src = (flags & F_VCYCLE) ? vc_rhs<V>(c) : F;
  g.B = load_q_raw(src + size_t(T.self) * 512 + hc + lane * 4);
  // halo ring: lanes 0..31 fetch the other-colour quad of one neighbour pencil
  //   q = 0: x- (pencil (7,t) of nbr 0), 1: x+ ((0,t) of nbr 3), 2: y- ((t,7) of nbr 1), 3: y+ ((t,0) of nbr 4)
  // x = 0 outside the grid (GMGSolver.cu:120-122)
  {
    const int q = (lane >> 3) & 3, t = lane & 7;
    const int f = pick4(q, 0, 3, 1, 4);
    const int n = pick4(q, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
    const int src_pl = pick4(q, 56 + t, t, t * 8 + 7, t * 8);
    const bool gh = tr_ntype(T, f) == T_GHOST;
    const bool ok = lane < 32 && n >= 0 && !(zero_all || (ghost_zero && gh));
    g.halo = load_q_raw(ok ? X + size_t(n) * 512 + ho + src_pl * 4 : zp);
  }
  // k halo, the one that the lane's cells of this colour reach (colour ho either way)
  {
    const bool p = ((color + i + j) & 1) != 0;
    const int n = p ? uni(T.nbr[5]) : uni(T.nbr[2]);
    const bool ok = n >= 0 && !(zero_all || (ghost_zero && tr_ntype(T, p ? 5 : 2) == T_GHOST));
    g.xk = load_s_raw(ok ? X + size_t(n) * 512 + ho + lane * 4 + (p ? 0 : 3) : zp);
  }
  return g;
}
template <class V>
__device__ __forceinline__ GsIn gs_convert(GsRaw<V>& r) {
  hold(r.xc);
  hold(r.xo);
  hold(r.B);
  hold(r.halo);
  hold(r.xk);
  GsIn g;
  g.xc = quad_f<V>(r.xc);
  g.xo = quad_f<V>(r.xo);
  g.B = quad_f<V>(r.B);
  g.halo = quad_f<V>(r.halo);
  g.xk = single_f<V>(r.xk);
  g.r0 = r.r0;
  g.r1 = r.r1;
  g.mask = r.mask;
  g.done = r.done;
  return g;
}
template <class V, bool DOT = false>
__device__ __forceinline__ GsIn gs_load(const Ctx& c, const TileRec& T, const V* X, const V* F, int color, int flags) {
  GsRaw<V> r = gs_issue<V, DOT>(c, T, X, F, color, flags);
  return gs_convert<V>(r);
}
__device__ __forceinline__ void gs_stage(const GsIn& g, GsLDS& L) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  L.xo[(i + 1) * 10 + (j + 1)] = g.xo;
  if (lane < 32) {
    const int q = lane >> 3, t = lane & 7;
    const int dst = (q == 0) ? (t + 1) : (q == 1) ? (91 + t) : (q == 2) ? ((t + 1) * 10) : ((t + 1) * 10 + 9);
    L.xo[dst] = g.halo;
  }
}
// after gs_stage and a wave_sync
template <class V, bool DOT = false>
__device__ __forceinline__ void gs_finish(const Ctx& c, const TileRec& T, V* X, int color, int flags, const GsIn& g,
                                          const GsLDS& L) {
  if ((flags & F_CHECK_DONE) && g.done) return;
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const int hc = color << 8, ho = (color ^ 1) << 8;
  V* tile = X + size_t(T.self) * 512;
  const int pc = (i + 1) * 10 + (j + 1);
  const bool p = ((color + i + j) & 1) != 0;
  const float4 nv = gs_quad(g.xc, g.xo, L.xo[pc - 10], L.xo[pc + 10], L.xo[pc - 1], L.xo[pc + 1], g.xk, g.B, g.mask,
                            gs_coef(T), i, j, p);
  store4(tile + hc + lane * 4, nv);
  if (flags & F_ZERO_X) store4(tile + ho + lane * 4, make_float4(0.f, 0.f, 0.f, 0.f));  // the zero guess of the other colour
  if (DOT && tr_type(T) == T_LEAF) {
    // this pass leaves the tile's z final: the updated colour as just stored,
    // the other colour as loaded; r.z over the lane's pencil in cell order,
    // as k_cg_dot_rz sums it
    const float zc[4] = {vround<V>(nv.x), vround<V>(nv.y), vround<V>(nv.z), vround<V>(nv.w)};
    const float zo[4] = {g.xo.x, g.xo.y, g.xo.z, g.xo.w};
    const float rv[8] = {g.r0.x, g.r0.y, g.r0.z, g.r0.w, g.r1.x, g.r1.y, g.r1.z, g.r1.w};
    double a = 0.0;
#pragma unroll
    for (int k = 0; k < 8; k++) {
      const float z = ((k & 1) == int(p)) ? zc[k >> 1] : zo[k >> 1];
      a += double(rv[k]) * double(z);
    }
    a = wave_sum(a);
    if (lane == 0) c.part[T.leaf_slot] = a;
  }
}
template <class V, bool DOT>
__device__ __forceinline__ void tile_gs(const Ctx& c, const TileRec& T, int level, V* X, const V* F, int color,
                                        int flags, GsLDS& L) {
  const GsIn g = gs_load<V, DOT>(c, T, X, F, color, flags);
  gs_stage(g, L);
  wave_sync();
  gs_finish<V, DOT>(c, T, X, color, flags, g, L);
}

// stage_tile on the V-cycle arrays plus the tile's rhs b (natural order; 0 with
// zero_b), the rhs loaded with the stage's loads, ahead of the one wait.
template <class V>
__device__ __forceinline__ void stage_with_rhs(const Ctx& c, const TileRec& T, const V* X, const V* XG, const V* F,
                                               int flags, bool zero_b, TileLDS& L, Stencil& S, float b[8]) {
  const V* src = zero_b ? zero_page<V>() : ((flags & F_VCYCLE) ? vc_rhs<V>(c) : F) + size_t(T.self) * 512;
  StageRaw<V> r = stage_issue<true>(c, T, X, XG, flags & F_ZERO_X, flags & F_GHOST_ZERO);
  RawPencil<V> rb = load_pencil_split_raw(src, lane_id());
  hold_all(rb);
  stage_commit<true>(r, T, T.bc, L, S);
  float4 ba, bb;
  pencil_split_f(rb, lane_id(), ba, bb);
  b[0] = ba.x; b[1] = ba.y; b[2] = ba.z; b[3] = ba.w;
  b[4] = bb.x; b[5] = bb.y; b[6] = bb.z; b[7] = bb.w;
}

// Damped-Jacobi sweep (the update of GMGSolver.cu:508-525 with the level's
// operator): Y = X + omega (b - A X) / D on INTERIOR cells, 0 where D == 0.
template <class V>
__device__ __forceinline__ void tile_jacobi(const Ctx& c, const TileRec& T, int level, const V* X, const V* XG,
                                            V* Y, const V* F, float omega, int flags, TileLDS& L) {
  Stencil S;
  float b[8];
  const uint32_t dn = done_load(c, T, flags);
  stage_with_rhs(c, T, X, XG, F, flags, false, L, S, b);
  if (done_test(dn, flags)) return;
  wave_sync();
  float ax[8], dg[8], out[8];
  if (S.open) {  // as gs_quad's open tiles: no masks, quotients as products with 1/D
    apply_pencil<true, false>(L, S, ax, dg);
    const int i = lane_id() >> 3, j = lane_id() & 7;
    const OpenDiag D = open_diag(gs_coef(T), i == 0 ? T.bc[0] : T.bc[6], i == 7 ? T.bc[3] : T.bc[6],
                                 j == 0 ? T.bc[1] : T.bc[6], j == 7 ? T.bc[4] : T.bc[6]);
    float res[8], q[8];
#pragma unroll
    for (int k = 0; k < 8; k++) res[k] = omega * (b[k] - ax[k]);
    div4_by(res, D.lo, D.mid, D.mid, D.mid, q);
    div4_by(res + 4, D.mid, D.mid, D.mid, D.hi, q + 4);
#pragma unroll
    for (int k = 0; k < 8; k++) out[k] = S.own[k] + q[k];
    store8_split(Y + size_t(T.self) * 512, lane_id(), out);
    return;
  }
  apply_pencil<true, true>(L, S, ax, dg);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    out[k] = S.own[k];
    if (ct_at(S.m, k) & M_INT) {
      float res = b[k] - ax[k];
      out[k] = (dg[k] == 0.f) ? 0.f : S.own[k] + (omega * res) / dg[k];
    }
  }
  store8_split(Y + size_t(T.self) * 512, lane_id(), out);
}

// 2x2x2 sums of a tile's values staged in LDS, in the reference's (ii, jj, kk)
// order (GMGSolver.cu:319-328): lane q = (a,b,c) = (q>>4, (q>>2)&3, q&3) returns
// the sum of fine cells (2a+ii, 2b+jj, 2c+kk).
__device__ __forceinline__ float octet_sum(const float* Ls, int q) {
  int a = q >> 4, bq = (q >> 2) & 3, cq = q & 3;
  float s = 0.f;
  for (int ii = 0; ii < 2; ii++)
    for (int jj = 0; jj < 2; jj++)
      for (int kk = 0; kk < 2; kk++) s += Ls[((2 * a + ii) * 8 + (2 * bq + jj)) * 8 + 2 * cq + kk];
  return s;
}
__device__ __forceinline__ size_t parent_cell(const TileRec& T, int q) {
  int a = q >> 4, bq = (q >> 2) & 3, cq = q & 3;
  const int oct = tr_octant(T), ox = oct & 1, oy = (oct >> 1) & 1, oz = (oct >> 2) & 1;
  return size_t(T.parent) * 512 + ((ox * 4 + a) << 6) + ((oy * 4 + bq) << 3) + (oz * 4 + cq);
}
// the same parent cell in the colour-split layout
__device__ __forceinline__ size_t parent_cell_split(const TileRec& T, int q) {
  int a = q >> 4, bq = (q >> 2) & 3, cq = q & 3;
  const int oct = tr_octant(T), ox = oct & 1, oy = (oct >> 1) & 1, oz = (oct >> 2) & 1;
  return size_t(T.parent) * 512 + split_cell(ox * 4 + a, oy * 4 + bq, oz * 4 + cq);
}

// Residual and restriction of one tile of `level` to level-1
// (GMGSolver.cu:284-339).  Output channel CO (rhsv in V-cycle mode): the
// parent cell = sum * one_over_alpha, or += sum for a GHOST fine tile (whose
// LEAF parent's rhs already holds r).  In V-cycle mode a ghost's rhs is 0.
template <class V>
__device__ __forceinline__ void tile_restrict(const Ctx& c, const TileRec& T, int level, const V* X, const V* F,
                                              V* CO, float one_over_alpha, int flags, TileLDS& L, float* res) {
  Stencil S;
  const int lane = lane_id();
  float b[8];
  const uint32_t dn = done_load(c, T, flags);
  stage_with_rhs<V>(c, T, X, X, F, flags, (flags & F_VCYCLE) && tr_type(T) == T_GHOST, L, S, b);
  if (done_test(dn, flags)) return;
  wave_sync();
  float ax[8], dg[8];
  apply_pencil<true, false>(L, S, ax, dg);
  for (int k = 0; k < 8; k++) res[lane * 8 + k] = b[k] - ax[k];
  wave_sync();
  float s = octet_sum(res, lane);
  const bool ghost = tr_type(T) == T_GHOST;
  V* out = (flags & F_VCYCLE) ? vc_rhs<V>(c) : CO;
  size_t pcell = parent_cell_split(T, lane);
  if (ghost) out[pcell] = from_f<V>(to_f(out[pcell]) + s);
  else out[pcell] = from_f<V>(s * one_over_alpha);
}

// Prolongation and update of one tile of `level` (GMGSolver.cu:345-376):
// ghosts take the parent value, others add prolong_coeff * parent value, on
// INTERIOR cells; other cells become 0.  Ghost results go to XG (the primary
// buffer) and active tiles to XO (a Jacobi ping-pong target).
template <class V>
__device__ __forceinline__ void tile_prolong(const Ctx& c, const TileRec& T, int level, const V* XC, const V* XF,
                                             V* XO, V* XG, float pcoef, int flags) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const int oct = tr_octant(T), ox = oct & 1, oy = (oct >> 1) & 1, oz = (oct >> 2) & 1;
  const uint32_t dn = done_load(c, T, flags);
  const float4 pv = load_quad_split(XC + size_t(T.parent) * 512, (ox * 4 + (i >> 1)) * 8 + (oy * 4 + (j >> 1)), oz * 4);
  const float cz[4] = {pv.x, pv.y, pv.z, pv.w};
  const uint64_t ct = load_ct8(c.ctype + base);
  const bool ghost = tr_type(T) == T_GHOST;
  float fx[8];
  if (ghost || (flags & F_ZERO_X)) { for (int k = 0; k < 8; k++) fx[k] = 0.f; }
  else load8_split(XF + size_t(T.self) * 512, lane, fx);
  hold8(fx);
  if (done_test(dn, flags)) return;
  float out[8];
  if (ghost) {
    for (int k = 0; k < 8; k++) out[k] = (ct_at(ct, k) & C_INT) ? cz[k >> 1] : 0.f;
    store8_split(XG + size_t(T.self) * 512, lane, out);
  } else {
    for (int k = 0; k < 8; k++) out[k] = (ct_at(ct, k) & C_INT) ? __builtin_fmaf(pcoef, cz[k >> 1], fx[k]) : 0.f;
    store8_split(XO + size_t(T.self) * 512, lane, out);
  }
}

// ---------------------------------------------------------------------------
// One-tile-per-workgroup kernels over a worklist
// ---------------------------------------------------------------------------
// A tile's record, fetched by two scalar loads that nothing else waits behind: the held
// words keep the compiler from splitting the fetch into pieces that it would
// load, wait for and test one after another.  A wavefront's cost on a small
// level is its chain of memory round trips: with the launch's n and flags
// preloaded (the kernels' first arguments) the record's fetch is the first, the
// tile's loads the second.  k_gs_color on 64 tiles 2.90 -> 2.57 us a launch, on
// the 360,472-tile level of the 256-problem pool in bfloat16 187 -> 178 us; the
// adaptive 256^3 solve 5.18 -> 4.87 ms, the pool 242 -> 231 ms.
typedef int32_t RecWords __attribute__((ext_vector_type(16), aligned(16)));
__device__ __forceinline__ TileRec unpack_rec(RecWords a, RecWords b) {
  TileRec T;
  for (int f = 0; f < 6; f++) T.nbr[f] = a[f];
  T.parent = a[6];
  T.prob = a[7];
  T.leaf_slot = a[8];
  T.gslot = a[9];
  T.self = a[10];
  T.h = __int_as_float(a[11]);
  T.meta = uint32_t(a[12]);
  T.ntypes = uint32_t(a[13]);
  T.bc[0] = __int_as_float(a[14]);
  T.bc[1] = __int_as_float(a[15]);
  for (int f = 2; f < 7; f++) T.bc[f] = __int_as_float(b[f - 2]);
  for (int f = 0; f < 6; f++) T.nbr_parent[f] = b[5 + f];
  T.rdiag = __hiloint2double(b[13], b[12]);
  return T;
}
__device__ __forceinline__ TileRec load_rec(const TileRec* __restrict__ list, int w) {
  const RecWords* r = reinterpret_cast<const RecWords*>(list + w);
  RecWords a = r[0], b = r[1];
  __asm__ volatile("" : "+s"(a), "+s"(b));
  return unpack_rec(a, b);
}
// The same with one pointer of each 64 bytes of the kernel's Ctx argument
// fetched alongside, so that the pointers the loads need are in the scalar
// cache when the record arrives.
__device__ __forceinline__ TileRec load_rec(const TileRec* __restrict__ list, int w, const Ctx& c) {
  const RecWords* r = reinterpret_cast<const RecWords*>(list + w);
  RecWords a = r[0], b = r[1];
  __asm__ volatile("" : "+s"(a), "+s"(b) : "s"(c.fmask), "s"(c.zh), "s"(c.ps));
  return unpack_rec(a, b);
}
#define TILE_KERNEL_PROLOGUE                                                           \
  const int w = work_index(flags & F_SWIZZLE, n);                                      \
  if (w >= n) return;                                                                  \
  const TileRec T = load_rec(list, w);
#define TILE_KERNEL_PROLOGUE_C                                                         \
  const int w = work_index(flags & F_SWIZZLE, n);                                      \
  if (w >= n) return;                                                                  \
  const TileRec T = load_rec(list, w, c);
// In a CG iteration's launch, a tile that k_cg_init found inert exits: the
// launch would write the values its arrays already hold.
#define SKIP_INERT \
  if ((flags & F_INERT) && tr_inert_cand(T) && c.inert[T.self]) return;

template <class V, bool DOT = false>
__global__ __launch_bounds__(64) void k_gs_color(const TileRec* __restrict__ list, int n, int flags, int level, V* X,
                                                 const V* F, int color, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  __shared__ GsLDS L;
  tile_gs<V, DOT>(c, T, level, X, F, color, flags, L);
}
// A colour sweep that writes the tile's whole result (the updated colour and
// the other colour as read) to Y and leaves X as it was, so that the next
// launch may read Y while it writes X.
template <class V>
__global__ __launch_bounds__(64) void k_gs_color_to(const TileRec* __restrict__ list, int n, int flags, const V* X,
                                                    V* Y, int color, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  __shared__ GsLDS L;
  const GsIn g = gs_load<V, false>(c, T, X, static_cast<const V*>(nullptr), color, flags);
  gs_stage(g, L);
  wave_sync();
  if ((flags & F_CHECK_DONE) && g.done) return;
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const int pc = (i + 1) * 10 + (j + 1);
  const bool p = ((color + i + j) & 1) != 0;
  const float4 nv = gs_quad(g.xc, g.xo, L.xo[pc - 10], L.xo[pc + 10], L.xo[pc - 1], L.xo[pc + 1], g.xk, g.B, g.mask,
                            gs_coef(T), i, j, p);
  V* tile = Y + size_t(T.self) * 512;
  store4(tile + (color << 8) + lane * 4, nv);
  store4(tile + ((color ^ 1) << 8) + lane * 4, g.xo);
}
// The same colour sweep with four wavefronts per workgroup, one tile each
// (tiles 4b .. 4b+3 of the list in workgroup b): a quarter of the workgroups
// to dispatch for the same tiles.
template <class V, bool DOT = false>
__global__ __launch_bounds__(256) void k_gs_color4(const TileRec* __restrict__ list, int n, int flags, int level,
                                                   V* X, const V* F, int color, Ctx c) {
  const int wave = threadIdx.x >> 6;
  const int w = work_index(flags & F_SWIZZLE, (n + 3) / 4) * 4 + wave;
  __shared__ GsLDS L[4];
  if (w >= n) return;  // whole wavefronts leave; the others synchronise within their wavefront only
  const TileRec T = list[w];
  tile_gs<V, DOT>(c, T, level, X, F, color, flags, L[wave]);
}
// The same colour sweep with a tile block of two: wavefront w works tiles 2w
// and 2w+1 of the list, loads of both in flight together.  Every tile's
// update is the one above (tiles of a colour pass are independent).
template <class V, bool DOT = false>
__global__ __launch_bounds__(64) void k_gs_color2(const TileRec* __restrict__ list, int n, int flags, int level, V* X,
                                                  const V* F, int color, Ctx c) {
  const int w = work_index(flags & F_SWIZZLE, (n + 1) / 2);
  const int t0 = 2 * w;
  if (t0 >= n) return;
  const bool two = t0 + 1 < n;
  const TileRec T0 = list[t0];
  const TileRec T1 = list[two ? t0 + 1 : t0];
  __shared__ GsLDS L[2];
  GsRaw<V> r0 = gs_issue<V, DOT>(c, T0, X, F, color, flags);
  GsRaw<V> r1{};  // unused without a second tile (no copy of r0, which would wait for its loads)
  if (two) r1 = gs_issue<V, DOT>(c, T1, X, F, color, flags);
  const GsIn g0 = gs_convert<V>(r0);
  const GsIn g1 = gs_convert<V>(r1);
  gs_stage(g0, L[0]);
  if (two) gs_stage(g1, L[1]);
  wave_sync();
  gs_finish<V, DOT>(c, T0, X, color, flags, g0, L[0]);
  if (two) gs_finish<V, DOT>(c, T1, X, color, flags, g1, L[1]);
}
// The same colour sweep with each wavefront walking its share of the list:
// while it updates one tile, the loads of its next tile are already out (a
// straight-line loop; after its last tile a wavefront loads that tile once
// more and drops it), so a wavefront's memory latency overlaps its own work
// instead of needing more wavefronts.  With F_SWIZZLE, the workgroups of XCD x
// (b % 8) walk the x-th eighth of the list (neighbouring tiles, one L2).  The
// grid is sized to the wavefronts the device holds at once.  Every tile's
// update is the one above.
template <class V, bool DOT = false>
__global__ __launch_bounds__(64) void k_gs_color_loop(const TileRec* __restrict__ list, int n, int flags, int level,
                                                      V* X, const V* F, int color, Ctx c) {
  __shared__ GsLDS L;
  const int b = blockIdx.x, nb = gridDim.x;
  int t, end, stride;
  if (flags & F_SWIZZLE) {
    const int per = (n + 7) >> 3, x = b & 7;
    t = x * per + (b >> 3);
    end = min(n, (x + 1) * per);
    stride = nb >> 3;  // nb is a multiple of 8
  } else {
    t = b;
    end = n;
    stride = nb;
  }
  if (t >= end) return;
  TileRec T = list[t];
  GsRaw<V> r = gs_issue<V, DOT>(c, T, X, F, color, flags);
  while (true) {
    const int tn = t + stride < end ? t + stride : t;
    const TileRec Tn = list[tn];
    GsRaw<V> rn = gs_issue<V, DOT>(c, Tn, X, F, color, flags);  // the next tile's loads
    const GsIn g = gs_convert<V>(r);
    gs_stage(g, L);
    wave_sync();
    gs_finish<V, DOT>(c, T, X, color, flags, g, L);
    if (tn == t) break;
    wave_sync();  // the LDS is staged again for the next tile
    t = tn;
    T = Tn;
    r = rn;
  }
}
// The colour sweep's diagonal of every cell of a tile (the D of gs_quad: the
// same coefficient choice and the same operations, in the colour-split order),
// for the fused first iteration below.  Fixed by the face masks and the tile's
// coefficients, so formed once when the problem is built.
__global__ __launch_bounds__(64) void k_diag(Ctx c, const TileRec* __restrict__ list, int n, float* __restrict__ D) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const uint64_t mask = load_ct8(c.fmask + size_t(T.self) * 512 + lane * 8);
  const float bi = T.bc[6];
  const float bim = (i == 0) ? T.bc[0] : bi;
  const float bip = (i == 7) ? T.bc[3] : bi;
  const float bjm = (j == 0) ? T.bc[1] : bi;
  const float bjp = (j == 7) ? T.bc[4] : bi;
  const float xn[6] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int col = 0; col < 2; col++) {
    const bool p = ((col + i + j) & 1) != 0;
    const int sh = p ? 8 : 0;
    float d[4];
#pragma unroll
    for (int m = 0; m < 4; m++) {
      const uint32_t mb = (m < 2 ? uint32_t(mask) : uint32_t(mask >> 32)) >> (16 * (m & 1) + sh);
      const float bkm = (!p && m == 0) ? T.bc[2] : bi;
      const float bkp = (p && m == 3) ? T.bc[5] : bi;
      const float bc[6] = {bim, bip, bjm, bjp, bkm, bkp};
      float ax;
      cell_row_m<true>(0.f, mb, xn, bc, T.h, ax, d[m]);
    }
    *reinterpret_cast<float4*>(D + size_t(T.self) * 512 + (col << 8) + lane * 4) = make_float4(d[0], d[1], d[2], d[3]);
  }
}

// The value a colour-0 cell holds after the first pass from the zero guess:
// 0 + (b - A 0) / D on INTERIOR cells with D != 0 (A 0 = +0), 0 elsewhere
// (D is 0 off INTERIOR cells), as stored in V.
template <class V>
__device__ __forceinline__ float first_red(float b, float d) {
  const float delta = (d != 0.f) ? (b - 0.f) / d : 0.f;
  return vround<V>(0.f + delta);
}

// The first red-black iteration of a down-sweep level from the zero guess in
// one launch: both colour passes of GMGSolver.cu:216-269 (colour 0 from x = 0,
// the other colour written 0; then colour 1).  After the first pass a colour-0
// cell depends on its own rhs and diagonal only, so the colour-0 values of the
// halo are formed from the neighbours' rhs and diagonals and the second pass
// needs no grid-wide wait.  Every value is the one the two passes give.
// Where every face neighbour's diagonals are the record's D (tr_std_faces: most
// tiles) the halo's diagonals are not read (their loads go to the zero page) and
// its five quotients are products with 1/D: 256 problems in bfloat16, the level of
// 360,472 tiles as two passes 222.1 ms a solve, as this one launch 216.6.
template <class V>
__global__ __launch_bounds__(64) void k_gs_first(const TileRec* __restrict__ list, int n, int flags, V* X, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  __shared__ GsLDS L;
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const bool ghost_zero = flags & F_GHOST_ZERO;
  const bool std_faces = tr_std_faces(T);
  const V* R = vc_rhs<V>(c);
  const V* zp = zero_page<V>();
  const float* zf = zero_page<float>();
  // ---- loads, all issued before the first wait
  const int32_t* dp = (flags & F_CHECK_DONE) ? &c.ps[T.prob].done : reinterpret_cast<const int32_t*>(c.fmask);
  const int32_t done = *dp;
  const uint32_t* masks = own_split_masks(c, T);
  const uint32_t mq0 = masks[lane], mq1 = masks[64 + lane];
  typename RawV<V>::Q rb0 = load_q_raw(R + size_t(T.self) * 512 + lane * 4);        // colour-0 rhs quad
  typename RawV<V>::Q rb1 = load_q_raw(R + size_t(T.self) * 512 + 256 + lane * 4);  // colour-1 rhs quad
  // halo ring of the colour-1 pass: lanes 0..31, the colour-0 quad of one
  // neighbour pencil; x = 0 outside the grid and on ghosts in the down-sweep
  // (rhs and diagonal from the zero page)
  const int q = (lane >> 3) & 3, t = lane & 7, f = ring_face(q);
  const int nb = pick4(q, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
  const int src = ring_src(q, t) * 4;
  const bool hok = lane < 32 && nb >= 0 && !(ghost_zero && tr_ntype(T, f) == T_GHOST);
  typename RawV<V>::Q hb = load_q_raw(hok ? R + size_t(nb) * 512 + src : zp);
  float4 hd = *reinterpret_cast<const float4*>(hok && !std_faces ? c.diag + size_t(nb) * 512 + src : zf);
  // k halo of the colour-1 pass: cell (i,j,7) of the z- neighbour (i + j odd) or
  // (i,j,0) of the z+ one (i + j even), a colour-0 cell either way
  const bool p0 = ((i + j) & 1) != 0, p1 = !p0;
  const int nz = p1 ? uni(T.nbr[5]) : uni(T.nbr[2]);
  const bool kok = nz >= 0 && !(ghost_zero && tr_ntype(T, p1 ? 5 : 2) == T_GHOST);
  const int kcell = lane * 4 + (p1 ? 0 : 3);
  typename RawV<V>::S kb = load_s_raw(kok ? R + size_t(nz) * 512 + kcell : zp);
  float kd = *(kok && !std_faces ? c.diag + size_t(nz) * 512 + kcell : zf);
  hold(rb0);
  hold(rb1);
  hold(hb);
  hold_f(hd.x);
  hold_f(hd.y);
  hold_f(hd.z);
  hold_f(hd.w);
  hold(kb);
  hold_f(kd);
  // ---- pass 1: the tile's colour-0 cells from x = 0 (gs_quad as the colour-0 pass runs it)
  const GsCoef G = gs_coef(T);
  const float4 z4 = make_float4(0.f, 0.f, 0.f, 0.f);
  const float4 n0 = gs_quad<true>(z4, z4, z4, z4, z4, z4, 0.f, quad_f<V>(rb0), mq0, G, i, j, p0);
  const float4 xr = make_float4(vround<V>(n0.x), vround<V>(n0.y), vround<V>(n0.z), vround<V>(n0.w));
  // the halo's colour-0 values as that pass leaves them (a value that counts as
  // 0 has rhs 0)
  const float4 hbf = quad_f<V>(hb);
  const float bk = single_f<V>(kb);
  float4 hv;
  float xk;
  if (std_faces) {
    const double rd = T.rdiag;
    const float hb4[4] = {hbf.x - 0.f, hbf.y - 0.f, hbf.z - 0.f, hbf.w - 0.f};
    float q4[4];
    div4_by(hb4, rd, rd, rd, rd, q4);
    hv = make_float4(vround<V>(0.f + q4[0]), vround<V>(0.f + q4[1]), vround<V>(0.f + q4[2]), vround<V>(0.f + q4[3]));
    xk = vround<V>(0.f + div_by_checked(bk - 0.f, rd));
  } else {
    hv = make_float4(first_red<V>(hbf.x, hd.x), first_red<V>(hbf.y, hd.y), first_red<V>(hbf.z, hd.z),
                     first_red<V>(hbf.w, hd.w));
    xk = first_red<V>(bk, kd);
  }
  L.xo[(i + 1) * 10 + (j + 1)] = xr;
  if (lane < 32) L.xo[ring_dst(q, t)] = hv;
  wave_sync();
  if ((flags & F_CHECK_DONE) && done) return;
  // ---- pass 2: colour 1, its own values 0 before the update
  const int pc = (i + 1) * 10 + (j + 1);
  const float4 n1 = gs_quad(z4, xr, L.xo[pc - 10], L.xo[pc + 10], L.xo[pc - 1], L.xo[pc + 1], xk, quad_f<V>(rb1), mq1,
                            G, i, j, p1);
  V* tile = X + size_t(T.self) * 512;
  store4(tile + lane * 4, xr);
  store4(tile + 256 + lane * 4, n1);
}

#include "gs_pair.hpp"

template <class V> struct RawQuadS { typename RawV<V>::S2 h0, h1; };
template <class V>
__device__ __forceinline__ RawQuadS<V> load_quad_split_raw(const V* __restrict__ tile, int pl, int K0) {
  RawQuadS<V> r;
  r.h0 = load2_raw(tile + pl * 4 + (K0 >> 1));
  r.h1 = load2_raw(tile + 256 + pl * 4 + (K0 >> 1));
  return r;
}
// load_quad_split's arrangement of the raw pairs
template <class V>
__device__ __forceinline__ float4 quad_split_f(const RawQuadS<V>& r, int pl) {
  const bool q0 = even_colour(pl);
  const float2 h0 = pair_f<V>(r.h0), h1 = pair_f<V>(r.h1);
  const float2 E = q0 ? h1 : h0, O = q0 ? h0 : h1;
  return make_float4(E.x, O.x, E.y, O.y);
}
// The prolongated values of a pencil's four cells of one colour (split quad): x +
// pcoef * parent on INTERIOR cells of active tiles, the parent value on those of
// GHOST tiles, 0 elsewhere, rounded as a store to V-typed memory would leave
// them.  Cells k = 2 e and 2 e + 1 have parent cell e, so a quad of either colour
// lines up with the parent quad; m: the quad's face masks (their INTERIOR bits).
template <class V>
__device__ __forceinline__ float4 prolong_quad(float4 x, float4 pq, uint32_t m, bool ghost, float pcoef) {
  auto one = [&](float xv, float pv, int e) {
    return ((m >> (8 * e)) & M_INT) ? vround<V>(ghost ? pv : __builtin_fmaf(pcoef, pv, xv)) : 0.f;
  };
  return make_float4(one(x.x, pq.x, 0), one(x.y, pq.y, 1), one(x.z, pq.z, 2), one(x.w, pq.w, 3));
}

// Prolongation fused into the first colour pass of the up-sweep on a level
// (GMGSolver.cu:345-376 then :216-269): every value the pass reads -- the tile's
// cells and the other-colour halo -- is formed on the fly as the prolongation
// would leave it, so no separate launch is needed.  XD holds the down-sweep
// values, XO receives the level's result; GHOST tiles in the list only store
// their prolongated values.
// Every load is issued before the first wait (what does not exist comes from the
// zero page), and the pass works on colour-split quads throughout: of a
// neighbour pencil only the four cells the update reads are formed, of the two k
// halos the one the lane's cells reach, and only the updated colour's rhs is read
// (2.5 s + t + s/8 bytes a cell, s the stored size, instead of 3 s + t + s/8).
// The 532,926-tile level of the 256-problem pool in FP32 769 -> 649 us, in
// bfloat16 469 -> 366; the refined 45,054-tile scene's in bfloat16 34.3 -> 26.2;
// a level of 64 tiles 3.72 -> 2.85.
template <class V>
__global__ __launch_bounds__(64) void k_gs_prolong(const TileRec* __restrict__ list, int n, int flags, const V* XD, V* XO,
                                                   float pcoef, int color, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  __shared__ GsLDS L;
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const int oct = tr_octant(T);
  const bool own_ghost = tr_type(T) == T_GHOST;
  const V* zp = zero_page<V>();
  const uint32_t* zw = reinterpret_cast<const uint32_t*>(kZeroPage);
  const int hc = color << 8, ho = hc ^ 256;
  const bool p = ((color + i + j) & 1) != 0;
  // the parent pencil of pencil (a,b) of a child in octant o
  auto parent_pencil = [](int o, int a, int b) { return ((o & 1) * 4 + (a >> 1)) * 8 + ((o >> 1) & 1) * 4 + (b >> 1); };
  const int32_t* dp = (flags & F_CHECK_DONE) ? &c.ps[T.prob].done : reinterpret_cast<const int32_t*>(c.fmask);
  const int32_t done = *dp;
  const uint32_t* masks = own_split_masks(c, T);
  const uint32_t mc = masks[(hc >> 2) + lane], mo = masks[(ho >> 2) + lane];
  const int ppl = parent_pencil(oct, i, j);
  RawQuadS<V> rpq = load_quad_split_raw(XO + size_t(T.parent) * 512, ppl, ((oct >> 2) & 1) * 4);
  const V* xd = own_ghost ? zp : XD + size_t(T.self) * 512;
  typename RawV<V>::Q rxc = load_q_raw(xd + hc + lane * 4);
  typename RawV<V>::Q rxo = load_q_raw(xd + ho + lane * 4);
  typename RawV<V>::Q rB = load_q_raw((own_ghost ? zp : vc_rhs<V>(c) + size_t(T.self) * 512) + hc + lane * 4);
  // halo ring of lanes 0..31 (x = 0 outside the grid: a missing neighbour's zero
  // masks make every value 0)
  const int g = (lane >> 3) & 3, t = lane & 7, f = ring_face(g);
  const int hn = pick4(g, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
  const int pn = pick4(g, uni(T.nbr_parent[0]), uni(T.nbr_parent[3]), uni(T.nbr_parent[1]), uni(T.nbr_parent[4]));
  const int hpl = ring_src(g, t), noct = oct ^ (g < 2 ? 1 : 2);
  const int hppl = parent_pencil(noct, hpl >> 3, hpl & 7);
  const bool hgh = tr_ntype(T, f) == T_GHOST;
  const bool hok = !own_ghost && lane < 32 && hn >= 0;
  uint32_t hm = *(hok ? c.fsplit + size_t(hn) * 128 + (ho >> 2) + hpl : zw);
  typename RawV<V>::Q rh = load_q_raw(hok && !hgh ? XD + size_t(hn) * 512 + ho + hpl * 4 : zp);
  RawQuadS<V> rhpq = load_quad_split_raw(hok ? XO + size_t(pn) * 512 : zp, hppl, ((noct >> 2) & 1) * 4);
  // k halo: cell (i,j,7) of the z- neighbour (p = 0) or (i,j,0) of the z+ one
  const int kn = p ? uni(T.nbr[5]) : uni(T.nbr[2]), kpn = p ? uni(T.nbr_parent[5]) : uni(T.nbr_parent[2]);
  const bool kgh = tr_ntype(T, p ? 5 : 2) == T_GHOST;
  const bool kok = !own_ghost && kn >= 0;
  const int kcell = ho + lane * 4 + (p ? 0 : 3);
  const int kpl = parent_pencil(oct ^ 4, i, j);
  const int kpcell = split_cell(kpl >> 3, kpl & 7, (((oct ^ 4) >> 2) & 1) * 4 + (p ? 0 : 3));
  uint32_t km = *(kok ? reinterpret_cast<const uint8_t*>(c.fsplit) + size_t(kn) * 512 + kcell
                      : reinterpret_cast<const uint8_t*>(zw));
  typename RawV<V>::S rkp = load_s_raw(kok ? XO + size_t(kpn) * 512 + kpcell : zp);
  typename RawV<V>::S rkx = load_s_raw(kok && !kgh ? XD + size_t(kn) * 512 + kcell : zp);
  hold_all(rpq.h0);
  hold_all(rpq.h1);
  hold_all(rxc);
  hold_all(rxo);
  hold_all(rB);
  hold_all(rh);
  hold_all(rhpq.h0);
  hold_all(rhpq.h1);
  hold_all(hm);
  hold_all(km);
  hold_all(rkp);
  hold_all(rkx);
  if ((flags & F_CHECK_DONE) && done) return;
  const float4 pq = quad_split_f(rpq, ppl);
  const float4 vc = prolong_quad<V>(quad_f<V>(rxc), pq, mc, own_ghost, pcoef);
  const float4 vo = prolong_quad<V>(quad_f<V>(rxo), pq, mo, own_ghost, pcoef);
  V* tile = XO + size_t(T.self) * 512;
  store4(tile + ho + lane * 4, vo);
  if (own_ghost) {
    store4(tile + hc + lane * 4, vc);
    return;
  }
  L.xo[(i + 1) * 10 + (j + 1)] = vo;
  if (lane < 32)
    L.xo[ring_dst(g, t)] = prolong_quad<V>(quad_f<V>(rh), quad_split_f(rhpq, hppl), hm, hgh, pcoef);
  const float kp = single_f<V>(rkp);
  const float xk = (km & M_INT) ? vround<V>(kgh ? kp : __builtin_fmaf(pcoef, kp, single_f<V>(rkx))) : 0.f;
  wave_sync();
  const int pc = (i + 1) * 10 + (j + 1);
  store4(tile + hc + lane * 4, gs_quad(vc, vo, L.xo[pc - 10], L.xo[pc + 10], L.xo[pc - 1], L.xo[pc + 1], xk, quad_f<V>(rB),
                                       mc, gs_coef(T), i, j, p));
}
template <class V>
__global__ __launch_bounds__(64) void k_jacobi(const TileRec* __restrict__ list, int n, int flags, int level,
                                               const V* X, const V* XG, V* Y, const V* F, float omega, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  __shared__ TileLDS L;
  tile_jacobi(c, T, level, X, XG, Y, F, omega, flags, L);
}
template <class V>
__global__ __launch_bounds__(64) void k_restrict(const TileRec* __restrict__ list, int n, int flags, int level,
                                                 const V* X, const V* F, V* CO, float one_over_alpha, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  __shared__ TileLDS L;
  __shared__ float res[512];
  tile_restrict<V>(c, T, level, X, F, CO, one_over_alpha, flags, L, res);
}
template <class V>
__global__ __launch_bounds__(64) void k_prolong(const TileRec* __restrict__ list, int n, int flags, int level,
                                                const V* XC, const V* XF, V* XO, V* XG, float pcoef, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  tile_prolong(c, T, level, XC, XF, XO, XG, pcoef, flags);
}

// ---------------------------------------------------------------------------
// Coarse levels 0..C (C <= 1) of the V-cycle (smoothing, restriction, the bottom
// solve on level 0, prolongation) for one problem in one workgroup, every tile
// of those levels resident in LDS.  The host takes level 0 in when it has at most
// CL_ROOTS tiles, level 1 when it is the eight children of one of them and holds
// no GHOST tile (a third level would have 64 tiles); one launch then replaces the
// ~10 launches per level a grid-wide phase each would need.  The per-cell
// arithmetic is the tile kernels' (GMGSolver.cu:216-376, bottom :432-433).
// ---------------------------------------------------------------------------
constexpr int CL_MAX_LEVELS = 2;
constexpr int CL_ROOTS = 8;                        // tiles on level 0 at most (slots 0 ..)
constexpr int CL_CHILDREN = 8;                     // tiles on level 1 (slots CL_ROOTS ..)
constexpr int CL_SLOTS = CL_ROOTS + CL_CHILDREN;
constexpr int CL_THREADS = 1024;
constexpr int CL_CPT = 8 * 256 / CL_THREADS;       // cells of one colour of a level per thread
constexpr int CL_ZERO = CL_SLOTS * 512;            // LDS index of a cell that stays 0
struct alignas(16) CoarseSlot {
  int32_t tile;      // tile index
  int32_t nbr[6];    // slot of the same-level face neighbour (x-,y-,z-,x+,y+,z+), -1: none
  int32_t parent;    // slot of the parent, -1 on level 0
  int32_t octant;
  float h;
  float bc;          // face coefficient of the slot's level (every face: no GHOST tile, GMGSolver.cu:26-39)
  int32_t pad;
};
static_assert(sizeof(CoarseSlot) == 48, "CoarseSlot is 48 bytes");
struct alignas(16) CoarsePlan {
  int32_t prob;      // problem index in the pool
  int32_t n0, n1;    // tiles on level 0, tiles on level 1 (0: not taken in; CL_CHILDREN)
  int32_t pad;
  CoarseSlot slots[CL_SLOTS];  // level 0 from 0, level 1 from CL_ROOTS
};
struct VCycleArgs {
  int nu, coarsest, smoother;
  float omega, ooa, pcoef;
};
// Colour-split like the V-cycle arrays (slot * 512 + colour * 256 + pencil * 4 +
// k / 2): consecutive threads work consecutive words, and so do their six
// neighbour reads.
struct CoarseLDS {
  float z[CL_ZERO + 4];         // V-cycle x of every slot, then CL_ZERO = 0
  float t[CL_CHILDREN * 512];   // level 1: residuals (restriction) or new values (damped Jacobi)
  float b0[CL_ROOTS * 512];     // V-cycle rhs of level 0
};

// One cell of a level: LDS byte addresses of its six neighbours (faces x-, x+,
// y-, y+, z-, z+; CL_ZERO outside the grid, the cell itself across a face cut by
// a NEUMANN cell, so that its term is c * 0), the reciprocal of its diagonal (0:
// the cell is not updated) and its rhs.  Prepared once per launch and kept in
// registers.
struct CoarseCell {
  uint32_t nb[3];   // two 16-bit addresses each
  double rd;
  float b;
};
__device__ __forceinline__ float& cl_at(CoarseLDS& M, uint32_t byte) {
  return *reinterpret_cast<float*>(reinterpret_cast<char*>(M.z) + byte);
}
// cell r (pencil * 4 + k / 2) of colour col of slot s, with face mask m and diagonal d
__device__ __forceinline__ void cl_prep(const CoarseSlot& S, int s, int col, int r, uint32_t m, float d, CoarseCell& P) {
  const int i = r >> 5, j = (r >> 2) & 7, e = r & 3;
  const bool p = ((col + i + j) & 1) != 0;  // the cell is k = 2 e + p
  const int oth = ((col ^ 1) << 8) + r;     // the other colour's cell of the same pencil and e
  const int own = s * 512 + (col << 8) + r, base = s * 512 + oth;
  auto at = [&](int q, int cell) { return q < 0 ? CL_ZERO : q * 512 + cell; };
  int nb[6];
  nb[0] = i > 0 ? base - 32 : at(S.nbr[0], oth + 224);
  nb[1] = i < 7 ? base + 32 : at(S.nbr[3], oth - 224);
  nb[2] = j > 0 ? base - 4 : at(S.nbr[1], oth + 28);
  nb[3] = j < 7 ? base + 4 : at(S.nbr[4], oth - 28);
  nb[4] = p ? base : (e > 0 ? base - 1 : at(S.nbr[2], oth + 3));
  nb[5] = p ? (e < 3 ? base + 1 : at(S.nbr[5], oth - 3)) : base;
#pragma unroll
  for (int f = 0; f < 6; f++) nb[f] = 4 * (((m >> f) & 1) ? nb[f] : own);
#pragma unroll
  for (int f = 0; f < 3; f++) P.nb[f] = uint32_t(nb[2 * f]) | (uint32_t(nb[2 * f + 1]) << 16);
  P.rd = d != 0.f ? recip64(d) : 0.0;  // D is 0 off INTERIOR cells
}
// b - A x of a prepared cell with value x0 (cell_row_m's operations; a cut face
// adds c * 0).
__device__ __forceinline__ float cl_residual(CoarseLDS& M, const CoarseCell& P, float x0, bool in, float cf, float h) {
  float xn[6];
#pragma unroll
  for (int f = 0; f < 3; f++) {
    xn[2 * f] = cl_at(M, P.nb[f] & 0xffffu);
    xn[2 * f + 1] = cl_at(M, P.nb[f] >> 16);
  }
  float sum = 0.f;
#pragma unroll
  for (int f = 0; f < 6; f++) sum = __builtin_fmaf(cf, x0 - xn[f], sum);
  return P.b - (in ? ((sum * h) * h) * h : 0.f);
}
// The cells of one level that a thread works: cell (tid & 255) of each colour of
// its slots (tid >> 8) + 4 m (one slot per wavefront and m).
struct CoarseCells {
  CoarseCell P[2][CL_CPT];  // [colour][m]
  uint32_t in;              // bit 2 * m + colour: INTERIOR
  uint32_t own;             // LDS byte address of colour 0, m = 0 (+ CL_COL for colour 1, + CL_M per m)
  int n;                    // m < n exist (level 1: all)
  float h, cf;
};
constexpr uint32_t CL_COL = 1024, CL_M = 8192;
// The loads of a level's cells (a slot that does not exist reads slot 0's tile)
struct CoarseRaw {
  uint32_t mask[2][CL_CPT];
  float d[2][CL_CPT], b[2][CL_CPT];
};
template <class V>
__device__ __forceinline__ void cl_issue(const Ctx& c, const CoarsePlan& cp, int first, int n, CoarseRaw& R) {
  const int q0 = uni(int(threadIdx.x) >> 8), r = threadIdx.x & 255;
#pragma unroll
  for (int m = 0; m < CL_CPT; m++) {
    const size_t tile = size_t(cp.slots[q0 + 4 * m < n ? first + q0 + 4 * m : 0].tile) * 512;
#pragma unroll
    for (int col = 0; col < 2; col++) {
      R.mask[col][m] = reinterpret_cast<const uint8_t*>(c.fsplit)[tile + col * 256 + r];
      R.d[col][m] = c.diag[tile + col * 256 + r];
      R.b[col][m] = to_f(vc_rhs<V>(c)[tile + col * 256 + r]);
    }
  }
}
__device__ __forceinline__ void cl_commit(const CoarsePlan& cp, int first, int n, const CoarseRaw& R, CoarseLDS& M,
                                          CoarseCells& L) {
  const int q0 = uni(int(threadIdx.x) >> 8), r = threadIdx.x & 255;
  L.own = uint32_t(4 * ((first + q0) * 512 + r));
  L.n = n > q0 ? (n - q0 + 3) >> 2 : 0;
  L.h = cp.slots[n ? first : 0].h;
  L.cf = cp.slots[n ? first : 0].bc;
  L.in = 0;
#pragma unroll
  for (int m = 0; m < CL_CPT; m++)
    if (m < L.n) {
      const int s = first + q0 + 4 * m;
#pragma unroll
      for (int col = 0; col < 2; col++) {
        L.P[col][m].b = R.b[col][m];
        L.in |= uint32_t((R.mask[col][m] & M_INT) != 0) << (2 * m + col);
        cl_prep(cp.slots[s], s, col, r, R.mask[col][m], R.d[col][m], L.P[col][m]);
        cl_at(M, L.own + m * CL_M + col * CL_COL) = 0.f;
      }
    }
}
// f(m, byte address) for each of the thread's cells of colour col; FULL: every
// m exists (level 1), so the cells' latencies overlap
template <bool FULL, class F>
__device__ __forceinline__ void cl_each(const CoarseCells& L, int col, F f) {
#pragma unroll
  for (int m = 0; m < CL_CPT; m++)
    if (FULL || m < L.n) f(m, L.own + m * CL_M + col * CL_COL);
}
// one red-black colour pass
template <class V, bool FULL>
__device__ __forceinline__ void cl_gs(CoarseLDS& M, const CoarseCells& L, int col) {
  float nv[CL_CPT];
  cl_each<FULL>(L, col, [&](int m, uint32_t at) {
    const CoarseCell& Q = L.P[col][m];
    const float x0 = cl_at(M, at);
    const float res = cl_residual(M, Q, x0, true, L.cf, L.h);  // used on INTERIOR cells only
    nv[m] = vround<V>(x0 + (Q.rd != 0.0 ? div_by_rounded(res, Q.rd) : 0.f));
  });
  cl_each<FULL>(L, col, [&](int m, uint32_t at) { cl_at(M, at) = nv[m]; });
  __syncthreads();
}

// The V-cycle of the resident levels on prepared cells: z from 0, the rhs in the
// cells of the finest level (and in M.b0 where level 0 has more than level 1
// restricts to).  Leaves z in M.z; ends with a barrier if it did anything.
template <class V>
__device__ __forceinline__ void cl_vcycle(CoarseLDS& M, const CoarsePlan& cp, int n1, CoarseCells& L0, CoarseCells& L1,
                                          const VCycleArgs& v) {
  const int tid = threadIdx.x;
  constexpr uint32_t T0 = CL_ROOTS * 512;  // M.t starts at level 1's first cell
  // one damped-Jacobi sweep of level 1
  auto jacobi1 = [&]() {
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<true>(L1, col, [&](int m, uint32_t at) {
        const CoarseCell& Q = L1.P[col][m];
        const bool in = (L1.in >> (2 * m + col)) & 1;
        const float x0 = cl_at(M, at);
        const float res = cl_residual(M, Q, x0, in, L1.cf, L1.h);
        M.t[(at >> 2) - T0] = in ? (Q.rd != 0.0 ? x0 + div_by_rounded(v.omega * res, Q.rd) : 0.f) : x0;
      });
    __syncthreads();
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<true>(L1, col, [&](int, uint32_t at) { cl_at(M, at) = vround<V>(M.t[(at >> 2) - T0]); });
    __syncthreads();
  };
  const int it0 = v.coarsest / 2;
  if (n1) {
    for (int it = 0; it < v.nu; it++) {
      if (v.smoother != 0) jacobi1();
      else { cl_gs<V, true>(M, L1, 0); cl_gs<V, true>(M, L1, 1); }
    }
    // residuals of level 1, then their 2x2x2 sums into the rhs of level 0, in the
    // reference's (ii, jj, kk) order (GMGSolver.cu:319-328)
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<true>(L1, col, [&](int m, uint32_t at) {
        M.t[(at >> 2) - T0] =
            cl_residual(M, L1.P[col][m], cl_at(M, at), (L1.in >> (2 * m + col)) & 1, L1.cf, L1.h);
      });
    __syncthreads();
    if (tid < CL_CHILDREN * 64) {
      const int q = uni(tid >> 6), lq = tid & 63;
      const CoarseSlot& S = cp.slots[CL_ROOTS + q];
      const int a = lq >> 4, bq = (lq >> 2) & 3, cq = lq & 3;
      float sum = 0.f;
#pragma unroll
      for (int o = 0; o < 8; o++)
        sum += M.t[q * 512 + split_cell(2 * a + (o >> 2), 2 * bq + ((o >> 1) & 1), 2 * cq + (o & 1))];
      const int ox = S.octant & 1, oy = (S.octant >> 1) & 1, oz = (S.octant >> 2) & 1;
      M.b0[S.parent * 512 + split_cell(ox * 4 + a, oy * 4 + bq, oz * 4 + cq)] = vround<V>(sum * v.ooa);
    }
    __syncthreads();
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<false>(L0, col, [&](int m, uint32_t at) { L0.P[col][m].b = M.b0[at >> 2]; });
  }
  for (int it = 0; it < it0; it++) { cl_gs<V, false>(M, L0, 0); cl_gs<V, false>(M, L0, 1); }
  for (int it = 0; it < it0; it++) { cl_gs<V, false>(M, L0, 1); cl_gs<V, false>(M, L0, 0); }
  if (n1) {
    const int q0 = uni(tid >> 8), r = tid & 255;
    // prolongation: x += pcoef * parent on INTERIOR cells, 0 elsewhere (the two
    // cells of a pair k = 2 e, 2 e + 1 have one parent cell)
    const int i = r >> 5, j = (r >> 2) & 7, e = r & 3;
    cl_each<true>(L1, 0, [&](int m, uint32_t at) {
      const CoarseSlot& S = cp.slots[CL_ROOTS + q0 + 4 * m];
      const int pi = (S.octant & 1) * 4 + (i >> 1), pj = ((S.octant >> 1) & 1) * 4 + (j >> 1);
      const float cz = M.z[S.parent * 512 + split_cell(pi, pj, ((S.octant >> 2) & 1) * 4 + e)];
#pragma unroll
      for (int col = 0; col < 2; col++) {
        float& z = cl_at(M, at + col * CL_COL);
        z = ((L1.in >> (2 * m + col)) & 1) ? vround<V>(__builtin_fmaf(v.pcoef, cz, z)) : 0.f;
      }
    });
    __syncthreads();
    for (int it = 0; it < v.nu; it++) {
      if (v.smoother != 0) jacobi1();
      else { cl_gs<V, true>(M, L1, 1); cl_gs<V, true>(M, L1, 0); }
    }
  }
}

// Latency bound on one CU (a scalar round trip for the plan, one for the cells,
// then about 30 passes with a barrier each), so what counts is the length of a
// pass: the rows are prepared once and kept for the down- and the up-sweep,
// neighbours are read without bank conflicts, and the division is a product with
// the prepared reciprocal.  Nine tiles, two sweeps per level, ten bottom
// iterations: 21.4 -> 13.5 us; six roots alone: 14.2 -> 10.2 us.  (Sixteen tiles
// on level 1 were measured too: 27 us, no better than that level's grid-wide
// launches.)
template <class V>
__global__ __launch_bounds__(CL_THREADS) void k_coarse_lds(const CoarsePlan* __restrict__ plans, int flags, V* Z,
                                                           VCycleArgs v, Ctx c) {
  __shared__ CoarseLDS M;
  const int tid = threadIdx.x;
  const CoarsePlan& cp = plans[blockIdx.x];
  const int n0 = cp.n0, n1 = cp.n1;
  CoarseCells L0, L1;
  {
    const int32_t done = (flags & F_CHECK_DONE) ? c.ps[cp.prob].done : 0;
    CoarseRaw R0, R1;
    cl_issue<V>(c, cp, CL_ROOTS, n1, R1);
    cl_issue<V>(c, cp, 0, n0, R0);
    if (done) return;
    if (tid < 4) M.z[CL_ZERO + tid] = 0.f;
    cl_commit(cp, CL_ROOTS, n1, R1, M, L1);
    cl_commit(cp, 0, n0, R0, M, L0);
  }
#pragma unroll
  for (int col = 0; col < 2; col++) cl_each<false>(L0, col, [&](int m, uint32_t at) { M.b0[at >> 2] = L0.P[col][m].b; });
  __syncthreads();
  cl_vcycle<V>(M, cp, n1, L0, L1, v);
  const int q0 = uni(tid >> 8), r = tid & 255;
  if (n1) {
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<true>(L1, col, [&](int m, uint32_t at) {
        Z[size_t(cp.slots[CL_ROOTS + q0 + 4 * m].tile) * 512 + col * 256 + r] = from_f<V>(cl_at(M, at));
      });
  }
#pragma unroll
  for (int col = 0; col < 2; col++)
    cl_each<false>(L0, col, [&](int m, uint32_t at) {
      Z[size_t(cp.slots[q0 + 4 * m].tile) * 512 + col * 256 + r] = from_f<V>(cl_at(M, at));
    });
}

// Empty kernel, for measuring the launch floor.
__global__ void k_empty(int* p) {
  if (p && threadIdx.x == 1024) *p = 0;
}

// ---------------------------------------------------------------------------
// CG kernels (rotated loop: V-cycle, gamma/beta, p, A p + alpha, x/r + check).
// Kernels write per-tile FP64 partials; k_finalize reduces them per problem.
// ---------------------------------------------------------------------------
// Per solve, for a candidate tile (LEAF, no ghost child, no INTERIOR cell,
// tr_inert_cand): it is inert when its initial residual is +0 in every cell.
// The residual then stays +0 (A p is 0 off INTERIOR cells), and so does every
// value the iterations would write there: the smoothers and the prolongation
// leave 0 on cells that are not INTERIOR, the residual and the restriction of
// zeros are 0, the operator writes 0, every dot partial is 0 (the slot holds
// the +0 written below) and x keeps its value (the updates are masked).  So
// its V-cycle vectors, A p and its octant block of the parent's V-cycle rhs
// (which only its restriction writes) are set to those values here, and the
// iteration kernels skip it (SKIP_INERT).
template <class V>
__device__ __forceinline__ void mark_inert(const Ctx& c, const TileRec& T, int lane, const float rv[8]) {
  bool zero = true;
  for (int k = 0; k < 8; k++) zero = zero && __float_as_uint(rv[k]) == 0u;
  const bool inert = __all(zero);
  if (lane == 0) c.inert[T.self] = inert ? 1 : 0;
  if (!inert) return;
  const float z8[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  store8(c.ap + size_t(T.self) * 512 + lane * 8, z8);
  store8_split(vc_z<V>(c) + size_t(T.self) * 512, lane, z8);
  store8_split(vc_zb<V>(c) + size_t(T.self) * 512, lane, z8);
  if (T.parent >= 0) vc_rhs<V>(c)[parent_cell_split(T, lane)] = from_f<V>(0.f);
}

// Init: x = 0, p = 0 on LEAF tiles, V-cycle rhs = b; partials of |b|^2
// (GMGSolver.cu:537-555).
template <class V>
__global__ __launch_bounds__(64) void k_cg_init(const TileRec* __restrict__ list, int n, int flags, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  store8(c.x + base, zero);
  store8(c.p + base, zero);
  float rv[8];
  load8(c.r + base, rv);
  store8_split(vc_rhs<V>(c) + size_t(T.self) * 512, lane, rv);
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(rv[k]) * double(rv[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
  if (c.inert && tr_inert_cand(T)) mark_inert<V>(c, T, lane, rv);
}

// Warm-started init: r = b - A x0 on LEAF tiles (A x0 in AP, formed by the
// operator kernels), p = 0, V-cycle rhs = r; partials of |b|^2, against which
// the tolerance is measured.
template <class V>
__global__ __launch_bounds__(64) void k_cg_init_warm(const TileRec* __restrict__ list, int n, int flags,
                                                     const float* __restrict__ B, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float bv[8], av[8], rv[8];
  load8(B + base, bv);
  load8(c.ap + base, av);
  for (int k = 0; k < 8; k++) rv[k] = bv[k] - av[k];
  float zero[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  store8(c.p + base, zero);
  store8(c.r + base, rv);
  store8_split(vc_rhs<V>(c) + size_t(T.self) * 512, lane, rv);
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(bv[k]) * double(bv[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
  if (c.inert && tr_inert_cand(T)) mark_inert<V>(c, T, lane, rv);
}

// Pool build on the device: out[k] = tiles[ids[k]] (the worklists, records
// copied as 16-byte words), and the cell types permuted from the caller's tile
// order (src, tile t at t*512) to the canonical order (tile i from src tile
// ext[i]).
__global__ __launch_bounds__(256) void k_gather_tiles(const TileRec* __restrict__ tiles, const int32_t* __restrict__ ids,
                                                      int64_t n, TileRec* __restrict__ out) {
  constexpr int W = sizeof(TileRec) / 16;
  const int64_t words = n * W;
  for (int64_t k = int64_t(blockIdx.x) * blockDim.x + threadIdx.x; k < words; k += int64_t(gridDim.x) * blockDim.x) {
    const int64_t r = k / W, w = k - r * W;
    reinterpret_cast<int4*>(out + r)[w] = reinterpret_cast<const int4*>(tiles + ids[r])[w];
  }
}
__global__ __launch_bounds__(64) void k_permute_ctype(const uint8_t* __restrict__ src, const int32_t* __restrict__ ext,
                                                      int n, uint8_t* __restrict__ dst) {
  const int i = blockIdx.x;
  if (i >= n) return;
  const uint64_t* s8 = reinterpret_cast<const uint64_t*>(src + size_t(ext[i]) * 512);
  uint64_t* d8 = reinterpret_cast<uint64_t*>(dst + size_t(i) * 512);
  d8[threadIdx.x] = s8[threadIdx.x];
}
// A float channel between the caller's tile order and the canonical order:
// to_canonical: dst tile i = src tile ext[i]; otherwise dst tile ext[i] = src
// tile i.  One wavefront per tile, 32 bytes per lane.
__global__ __launch_bounds__(64) void k_permute_channel(const float* __restrict__ src, const int32_t* __restrict__ ext,
                                                        int n, float* __restrict__ dst, int to_canonical) {
  const int i = blockIdx.x;
  if (i >= n) return;
  const size_t e = size_t(ext[i]) * 512, c = size_t(i) * 512;
  const float4* s4 = reinterpret_cast<const float4*>(src + (to_canonical ? e : c)) + 2 * threadIdx.x;
  float4* d4 = reinterpret_cast<float4*>(dst + (to_canonical ? c : e)) + 2 * threadIdx.x;
  const float4 a = s4[0], b = s4[1];
  d4[0] = a;
  d4[1] = b;
}

// Face masks of every cell of the listed tiles (Ctx::fmask): bit e of cell c is
// set when face e (x-, x+, y-, y+, z-, z+) is not cut, i.e. neither c nor its
// neighbour across e is NEUMANN (GMGSolver.cu:26-39; a neighbour outside the
// grid is DIRICHLET, GMGSolver.cu:120-122); bit 6 when c is INTERIOR.  Cell
// types do not change during a solve, so the masks are formed once.
__global__ __launch_bounds__(64) void k_face_mask(const uint8_t* __restrict__ ctype, uint8_t* __restrict__ fmask,
                                                  uint32_t* __restrict__ fsplit, const TileRec* __restrict__ list, int n) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  __shared__ uint64_t cs[100];
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const uint64_t own = load_ct8(ctype + base);
  const int pc = (i + 1) * 10 + (j + 1);
  cs[pc] = own;
  const uint64_t dir = 0x0101010101010101ull;
  if (lane < 32) {
    const int g = lane >> 3, t = lane & 7;
    const int nb = pick4(g, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
    const int src = (g == 0) ? (56 + t) : (g == 1) ? t : (g == 2) ? (t * 8 + 7) : (t * 8);
    const int dst = (g == 0) ? (t + 1) : (g == 1) ? (91 + t) : (g == 2) ? ((t + 1) * 10) : ((t + 1) * 10 + 9);
    cs[dst] = nb < 0 ? dir : load_ct8(ctype + size_t(nb) * 512 + src * 8);
  }
  const uint8_t ckm = T.nbr[2] < 0 ? uint8_t(C_DIR) : ctype[size_t(T.nbr[2]) * 512 + lane * 8 + 7];
  const uint8_t ckp = T.nbr[5] < 0 ? uint8_t(C_DIR) : ctype[size_t(T.nbr[5]) * 512 + lane * 8];
  wave_sync();
  const uint64_t cim = cs[pc - 10], cip = cs[pc + 10], cjm = cs[pc - 1], cjp = cs[pc + 1];
  uint64_t out = 0;
  for (int k = 0; k < 8; k++) {
    const uint8_t c0 = ct_at(own, k);
    const uint8_t cn[6] = {ct_at(cim, k), ct_at(cip, k), ct_at(cjm, k), ct_at(cjp, k), k == 0 ? ckm : ct_at(own, k - 1),
                           k == 7 ? ckp : ct_at(own, k + 1)};
    uint32_t m = (c0 & C_INT) ? uint32_t(M_INT) : 0u;
    for (int e = 0; e < 6; e++)
      if (!((c0 | cn[e]) & C_NEU)) m |= 1u << e;
    out |= uint64_t(m) << (8 * k);
  }
  *reinterpret_cast<uint64_t*>(fmask + base) = out;
  const bool p0 = ((i + j) & 1) != 0;  // colour 0 holds the cells k = 2m + p0
  fsplit[size_t(T.self) * 128 + lane] = quad_mask(out, p0);
  fsplit[size_t(T.self) * 128 + 64 + lane] = quad_mask(out, !p0);
}

// Seeded update of a right-hand side, for a synthetic client of the serving
// loop: b = rho * b + sigma * u on INTERIOR cells of the listed (LEAF) tiles,
// u uniform on [-sqrt(3), sqrt(3)] (unit variance) from a counter hash of
// (seed, tile, cell).
__device__ __forceinline__ uint32_t hash32(uint64_t x) {
  x ^= x >> 33;
  x *= 0xff51afd7ed558ccdull;
  x ^= x >> 33;
  x *= 0xc4ceb9fe1a85ec53ull;
  x ^= x >> 33;
  return uint32_t(x);
}
__global__ __launch_bounds__(64) void k_perturb_rhs(Ctx c, const TileRec* __restrict__ list, int n, float* __restrict__ B,
                                                    float rho, float sigma, uint64_t seed) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float b[8];
  load8(B + base, b);
  const uint64_t ct = load_ct8(c.ctype + base);
  for (int k = 0; k < 8; k++) {
    if (!(ct_at(ct, k) & C_INT)) continue;
    const uint32_t h = hash32(seed * 0x9e3779b97f4a7c15ull + uint64_t(base + k));
    const float u = (float(h) * 2.3283064365386963e-10f * 2.0f - 1.0f) * 1.7320508075688772f;
    b[k] = rho * b[k] + sigma * u;
  }
  store8(B + base, b);
}

// Staged problem states to their slots: src[i] -> ps[map[i]], i < n (one
// workgroup per state).
__global__ __launch_bounds__(64) void k_ps_scatter(ProbState* __restrict__ ps, const ProbState* __restrict__ src,
                                                   const int32_t* __restrict__ map, int n) {
  static_assert(sizeof(ProbState) % 16 == 0, "ProbState is copied in 16-byte words");
  constexpr int W = sizeof(ProbState) / 16;
  const int i = blockIdx.x;
  if (i >= n) return;
  const int4* from = reinterpret_cast<const int4*>(src + i);
  int4* to = reinterpret_cast<int4*>(ps + map[i]);
  for (int k = threadIdx.x; k < W; k += blockDim.x) to[k] = from[k];
}

// Copy runs of tile records into an assembled worklist: run q copies
// counts[q] records from srcs[q] to dst + offs[q] (grid-stride over records).
__global__ __launch_bounds__(256) void k_gather_recs(const TileRec* const* __restrict__ srcs, const int32_t* __restrict__ offs,
                                                     const int32_t* __restrict__ counts, int nruns, TileRec* __restrict__ dst) {
  constexpr int W = sizeof(TileRec) / 16;
  for (int q = blockIdx.y; q < nruns; q += gridDim.y) {
    const int4* src = reinterpret_cast<const int4*>(srcs[q]);
    int4* out = reinterpret_cast<int4*>(dst + offs[q]);
    const int words = counts[q] * W;
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < words; k += gridDim.x * blockDim.x) out[k] = src[k];
  }
}

// partials of gamma = r.z over LEAF tiles (GMGSolver.cu:634)
template <class V>
__global__ __launch_bounds__(64) void k_cg_dot_rz(const TileRec* __restrict__ list, int n, int flags, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float rv[8], zv[8];
  const uint32_t dn = done_load(c, T, flags);
  load8(c.r + base, rv);
  load8_split(vc_z<V>(c) + size_t(T.self) * 512, lane, zv);
  hold8(rv);  // or the loads would move behind the test
  hold8(zv);
  if (done_test(dn, flags)) return;
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(rv[k]) * double(zv[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
}

// The previous iteration's x += alpha p (deferred from k_cg_update_xr, which
// then reads neither x nor p; the same fma on the same values, one iteration
// later, and k_cg_finish_x applies the last one), then p = z + beta p on
// INTERIOR cells of LEAF tiles (GMGSolver.cu:587-609 and 642-653).  The ghost
// children's p (the parent's INTERIOR values, PoissonGrid.cu:585-605) is not
// stored: the operator reads it from here (k_apply<true>).
template <class V>
__global__ __launch_bounds__(64) void k_cg_update_p(const TileRec* __restrict__ list, int n, int flags, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float pv[8], zv[8], xv[8];
  const uint32_t word = state_word(c.ps + T.prob);
  load8(c.p + base, pv);
  load8_split(vc_z<V>(c) + size_t(T.self) * 512, lane, zv);
  load8_once(c.x + base, xv);
  const uint64_t ct = tile_ct8(T, c.ctype + base);
  const ProbState ps = state_of(word);
  if ((flags & F_CHECK_DONE) && ps.done) return;
  const float beta = float(ps.beta);
  const float alpha = float(ps.alpha);
  const bool upd_x = ps.iter > 0;  // an earlier iteration left its x update pending
  for (int k = 0; k < 8; k++)
    if (ct_at(ct, k) & C_INT) {
      if (upd_x) xv[k] = __builtin_fmaf(alpha, pv[k], xv[k]);
      pv[k] = __builtin_fmaf(beta, pv[k], zv[k]);
    }
  if (upd_x) store8_once(c.x + base, xv);
  store8(c.p + base, pv);
}

// A p on LEAF and GHOST tiles with the subtree view sl.  In CG mode (dot=1)
// LEAF tiles write A p and, when they have no ghost children, their p.Ap
// partial; GHOST tiles write the 2x2x2 sums of their rows for the parent
// (AccumulateToParents128 with all cell types, PoissonGrid.cu:664-710).  In
// channel mode (dot=0) every listed tile writes its rows to AX.
// PG (the CG iteration's operator on p): GHOST values from their parents
// (stage_issue_pg), as p is not copied into ghost tiles.
template <bool PG = false>
__global__ __launch_bounds__(64) void k_apply(const TileRec* __restrict__ list, int n, int flags,
                                              const float* __restrict__ X, float* __restrict__ AX, int sl, int diag,
                                              int dot, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  __shared__ TileLDS L;
  __shared__ float gl[512];
  Stencil S;
  float bcv[7];
  if (PG) {
    // the view of LEAF and GHOST tiles with no subtree level, from the record's
    // (its level's): the same but for NONLEAF neighbours, which count there as LEAF
    for (int f = 0; f < 6; f++) bcv[f] = tr_ntype(T, f) == T_NONLEAF ? 0.f : T.bc[f];
    bcv[6] = T.bc[6];
  } else {
    view_coeffs(T, sl, bcv);
  }
  const uint32_t dn = done_load(c, T, flags);
  if (PG) {
    StagePG r = stage_issue_pg(c, T, X);
    stage_commit_pg(r, T, bcv, L, S);
  } else {
    stage_tile<false>(c, T, X, X, false, false, bcv, L, S);
  }
  if (done_test(dn, flags)) return;
  wave_sync();
  float ax[8], dg[8];
  if (diag) apply_pencil<false, true>(L, S, dg, ax);
  else apply_pencil<true, false>(L, S, ax, dg);
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  if (tr_type(T) == T_GHOST && dot) {
    const uint64_t ct = load_ct8(c.ctype + base);
    for (int k = 0; k < 8; k++) gl[lane * 8 + k] = (ct_at(ct, k) & (C_INT | C_DIR | C_NEU)) ? ax[k] : 0.f;
    wave_sync();
    c.gsum[size_t(T.gslot) * 64 + lane] = octet_sum(gl, lane);
    return;
  }
  store8(AX + base, ax);
  if (!dot || tr_type(T) != T_LEAF || tr_has_gchild(T)) return;
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(S.own[k]) * double(ax[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
}

// LEAF tiles with ghost children: A p += ghost row sums (the += of
// AccumulateToParents128), then the p.Ap partial (GMGSolver.cu:580).
__global__ __launch_bounds__(64) void k_ghost_gather(const TileRec* __restrict__ list, int n, int flags, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float av[8], pv[8];
  const uint32_t dn = done_load(c, T, flags);
  load8(c.ap + base, av);
  load8(c.p + base, pv);
  float4 e[2];
  int gs[2];
  for (int h = 0; h < 2; h++) {
    gs[h] = c.kids[T.gslot].slot[(i >> 2) | ((j >> 2) << 1) | (h << 2)];
    if (gs[h] >= 0) e[h] = *reinterpret_cast<const float4*>(c.gsum + size_t(gs[h]) * 64 + (i & 3) * 16 + (j & 3) * 4);
  }
  if (done_test(dn, flags)) return;
  for (int h = 0; h < 2; h++) {
    if (gs[h] < 0) continue;
    av[4 * h + 0] = av[4 * h + 0] + e[h].x;
    av[4 * h + 1] = av[4 * h + 1] + e[h].y;
    av[4 * h + 2] = av[4 * h + 2] + e[h].z;
    av[4 * h + 3] = av[4 * h + 3] + e[h].w;
  }
  store8(c.ap + base, av);
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(pv[k]) * double(av[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
}

// r -= alpha A p on INTERIOR cells of LEAF tiles (GMGSolver.cu:587-609); r is
// also the next V-cycle's rhs; partials of |r|^2.  The iteration's x += alpha p
// is left to the next k_cg_update_p (or k_cg_finish_x).
template <class V>
__global__ __launch_bounds__(64) void k_cg_update_xr(const TileRec* __restrict__ list, int n, int flags, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float rv[8], av[8];
  const uint32_t word = state_word(c.ps + T.prob);
  load8(c.r + base, rv);
  load8(c.ap + base, av);
  const uint64_t ct = tile_ct8(T, c.ctype + base);
  const ProbState ps = state_of(word);
  if ((flags & F_CHECK_DONE) && ps.done) return;
  const float alpha = float(ps.alpha);
  for (int k = 0; k < 8; k++)
    if (ct_at(ct, k) & C_INT) rv[k] = __builtin_fmaf(-alpha, av[k], rv[k]);
  store8(c.r + base, rv);
  store8_split(vc_rhs<V>(c) + size_t(T.self) * 512, lane, rv);
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(rv[k]) * double(rv[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
}

// The last iteration's pending x += alpha p on INTERIOR cells of LEAF tiles,
// once after a problem's iterations end (every problem of the list, done or
// not; none when no iteration ran).
__global__ __launch_bounds__(64) void k_cg_finish_x(const TileRec* __restrict__ list, int n, int flags, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  SKIP_INERT
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float pv[8], xv[8];
  load8(c.p + base, pv);
  load8(c.x + base, xv);
  const uint64_t ct = tile_ct8(T, c.ctype + base);
  const ProbState& ps = c.ps[T.prob];
  if (ps.iter <= 0) return;
  const float alpha = float(ps.alpha);
  for (int k = 0; k < 8; k++)
    if (ct_at(ct, k) & C_INT) xv[k] = __builtin_fmaf(alpha, pv[k], xv[k]);
  store8(c.x + base, xv);
}

// Sum of a problem's per-tile partials in the fixed order (lane q of the first
// wavefront adds partials q, q + 64, ... in sequence, then the butterfly), by a
// workgroup of NT threads.  The sequence is a chain of count / 64 dependent
// additions, so what can be saved is the wait for the data:
// NT = FIN_WAVE: one wavefront, each lane loading its own sequence, FIN_ROWS
//   values in flight while the FIN_ROWS before them are added; no LDS, no barrier.
// NT = FIN_BLOCK: the whole workgroup loads a chunk into LDS while the first
//   wavefront adds the chunk before it.
// Addresses are clamped into the range; what lies beyond it adds -0.0, which
// leaves every sum as it is.
constexpr int FIN_WAVE = 64;
constexpr int FIN_BLOCK = 1024;
constexpr int FIN_ROWS = 32;
constexpr int FIN_CHUNK = 16384;
constexpr int FIN_PER_THREAD = FIN_CHUNK / FIN_BLOCK;
constexpr int FIN_GROUP = 16;
template <int NT>
__device__ __forceinline__ double block_sum_partials(const double* __restrict__ part, int begin, int count) {
  const int tid = threadIdx.x;
  const double* src = part + begin;
  double a = 0.0;
  if constexpr (NT == FIN_WAVE) {
    auto fetch = [&](int r0, double (&v)[FIN_ROWS]) {
#pragma unroll
      for (int u = 0; u < FIN_ROWS; u++) v[u] = src[min((r0 + u) * 64 + tid, count - 1)];
    };
    double v[FIN_ROWS], w[FIN_ROWS];
    const int rows = (count + 63) >> 6;
    fetch(0, v);
    for (int r0 = 0; r0 < rows; r0 += FIN_ROWS) {
      if (r0 + FIN_ROWS < rows) fetch(r0 + FIN_ROWS, w);
#pragma unroll
      for (int u = 0; u < FIN_ROWS; u++) a += (r0 + u) * 64 + tid < count ? v[u] : -0.0;
#pragma unroll
      for (int u = 0; u < FIN_ROWS; u++) v[u] = w[u];
    }
    return wave_sum(a);
  } else {
    __shared__ double lds[FIN_CHUNK];
    double v[FIN_PER_THREAD];
    auto fetch = [&](int c0) {
#pragma unroll
      for (int u = 0; u < FIN_PER_THREAD; u++) v[u] = src[min(c0 + tid + u * NT, count - 1)];
    };
    fetch(0);
    for (int c0 = 0; c0 < count; c0 += FIN_CHUNK) {
      __syncthreads();  // the previous chunk's sums are done with lds
#pragma unroll
      for (int u = 0; u < FIN_PER_THREAD; u++) lds[tid + u * NT] = c0 + tid + u * NT < count ? v[u] : -0.0;
      __syncthreads();
      if (c0 + FIN_CHUNK < count) fetch(c0 + FIN_CHUNK);
      if (tid < 64) {
        // lane tid continues its sequence tid, tid + 64, ... across chunks (FIN_CHUNK is a multiple of 64 FIN_GROUP)
        const int rows = (min(FIN_CHUNK, count - c0) + 63) >> 6;
        double w[FIN_GROUP], x[FIN_GROUP];
#pragma unroll
        for (int u = 0; u < FIN_GROUP; u++) w[u] = lds[tid + u * 64];
        for (int g0 = 0; g0 < rows; g0 += FIN_GROUP) {
          const int g1 = g0 + FIN_GROUP < rows ? g0 + FIN_GROUP : 0;
#pragma unroll
          for (int u = 0; u < FIN_GROUP; u++) x[u] = lds[tid + (g1 + u) * 64];
#pragma unroll
          for (int u = 0; u < FIN_GROUP; u++) a += w[u];
#pragma unroll
          for (int u = 0; u < FIN_GROUP; u++) w[u] = x[u];
        }
      }
    }
    if (tid < 64) a = wave_sum(a);
    return a;
  }
}
// Per-problem finalisation of a reduction over the LEAF-tile partials.
enum : int { FIN_BB = 0, FIN_RZ = 1, FIN_PAP = 2, FIN_RR = 3, FIN_MEAN = 4, FIN_IRBB = 5, FIN_SCALE = 6 };
// range_count >= 0: the launch's one problem has its partials at range_begin ..
// range_begin + range_count - 1 (its leaf range), given by the host so that
// their loads go out with the problem state's rather than after it.
__device__ __forceinline__ void report_progress(int32_t* progress, int iters, int done) {
  if (progress) __hip_atomic_store(progress + blockIdx.x, 2 * iters + done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <int NT>
__global__ __launch_bounds__(NT) void k_finalize(int mode, int flags, int range_begin, int range_count,
                                                 const double* part, ProbState* states, const int32_t* pmap,
                                                 const double* part2, int32_t* progress) {
  ProbState* ps = states + (pmap ? pmap[blockIdx.x] : int(blockIdx.x));
  const uint32_t word = state_word(ps);
  const bool given = range_count >= 0;
  int begin = range_begin, count = range_count;
  if (!given) {
    const ProbState st = state_of(word);
    if (mode != FIN_BB && (flags & F_CHECK_DONE) && st.done) return;
    if (mode == FIN_MEAN && !st.pure_neumann) return;
    begin = st.leaf_begin;
    count = st.leaf_count;
  }
  const double s = block_sum_partials<NT>(part, begin, count);
  const ProbState st = state_of(word);
  if (given) {  // the same tests, after the sum (whose value is then dropped)
    if (mode != FIN_BB && (flags & F_CHECK_DONE) && st.done) return;
    if (mode == FIN_MEAN && !st.pure_neumann) return;
  }
  double q = 0.0;
  if (mode == FIN_MEAN) q = block_sum_partials<NT>(part2, begin, count);
  if (threadIdx.x != 0) return;
  switch (mode) {
    case FIN_BB: {  // GMGSolver.cu:542-554
      ps->bb = s;
      ps->rr = s;
      double thr = st.tol2 * s;
      thr = thr > st.thr_abs ? thr : st.thr_abs;
      const int done = (s == 0.0 || st.max_iters <= 0) ? 1 : 0;
      ps->thr = thr > 2.2250738585072014e-308 ? thr : 2.2250738585072014e-308;
      ps->iter = 0;
      ps->converged = (s == 0.0) ? 1 : 0;
      ps->done = done;
      ps->gamma = 0.0;
      report_progress(progress, 0, done);
      break;
    }
    case FIN_RZ:  // gamma_old = gamma; gamma = r.z; beta = gamma / gamma_old (GMGSolver.cu:629-638)
      ps->gamma_old = st.gamma;
      ps->gamma = s;
      ps->beta = (st.iter == 0) ? 0.0 : s / st.gamma;
      break;
    case FIN_PAP:  // alpha = gamma / p.Ap (GMGSolver.cu:580-582)
      ps->pAp = s;
      ps->alpha = st.gamma / s;
      break;
    case FIN_RR: {  // GMGSolver.cu:611-619 (checked every sync_stride iterations)
      ps->rr = s;
      const int it = st.iter + 1, cs = st.check_stride;
      const bool converged = cs > 0 && it % cs == 0 && s < st.thr;
      const int done = (converged || it >= st.max_iters) ? 1 : st.done;
      ps->iter = it;
      if (converged) ps->converged = 1;
      ps->done = done;
      report_progress(progress, it, done);
      break;
    }
    case FIN_MEAN:
      ps->mean = s / q;
      break;
    case FIN_IRBB:  // |b|^2 of an FP64 refinement's right-hand side and the inner solves' threshold floor
      ps->bb_b = s;
      ps->thr_abs = st.tol_abs2 * s;
      break;
    case FIN_SCALE: {  // float16 storage: the right-hand side's scale 2^k, from |b|^2 / cells = 2^e f,
                       // f in [1, 2): k = -floor(e/2) - 4 (root mean square near 2^-4)
      int k = 0;
      if (s > 0.0) {
        const int e = ilogb(s / (512.0 * double(st.leaf_count)));
        const int half = (e >= 0) ? e / 2 : -((-e + 1) / 2);
        k = min(120, max(-120, -half - 4));
      }
      ps->scale_exp = k;
      ps->thr_abs = ldexp(st.thr_abs, 2 * k);
      break;
    }
  }
}

// ---------------------------------------------------------------------------
// CG of a problem whose every level is LDS-resident: up to `iters` iterations in
// one launch of one workgroup.  Launch by launch such an iteration was one of this
// kernel's V-cycles and seven launches of 2.2 to 3.7 us for eight tiles of vector
// work each.  Here r, p, A p and z stay in LDS (colour-split, so that the rows are
// those of the V-cycle), x in registers, and an iteration is the V-cycle's passes
// and seven barriers: the vector part's cells are the threads' own cells of the
// finest level, and for a tile's dot partial one wavefront reads its pencils and
// adds them in the order of the per-tile kernels.  One 16^3 box (9 tiles, two
// sweeps a level), 19 iterations: 790 -> 360 us a solve, 10 us of it an iteration,
// bound by the V-cycle's chain of some forty passes with a barrier each.
// ---------------------------------------------------------------------------
// Tile partials: a row for each of the iteration's sums.  Every wavefront reads a row
// behind the barrier that follows its writing, and it is written again an iteration
// later, with the barriers of the other sums between.  (A row for two sums would need
// a barrier of its own: |r|^2 is the last sum that an iteration reads and the mean's
// two are the first that the next one writes, with none between.)
enum : int { SM_MEAN = 0, SM_COUNT, SM_RZ, SM_PAP, SM_RR, SM_SUMS };
struct SmallLDS {
  float p[CL_ZERO + 4];        // in v.z's layout, so that a cell's neighbour addresses serve both
  CoarseLDS v;                 // v.t: A p outside the V-cycle
  float r[CL_CHILDREN * 512];  // from the finest level's first slot
  double part[SM_SUMS][CL_CHILDREN];
  ProbState out;               // the state to leave (thread 0's)
};
// A tile's sum over the 64 pencils (lanes) of f(cell values of the pencil in order).
__device__ __forceinline__ void sm_pencil(const float* a, float o[8]) {  // a: the tile's colour-split cells
  float4 q0, q1;
  load_pencil_split(a, lane_id(), q0, q1);
  o[0] = q0.x; o[1] = q0.y; o[2] = q0.z; o[3] = q0.w;
  o[4] = q1.x; o[5] = q1.y; o[6] = q1.z; o[7] = q1.w;
}
__device__ __forceinline__ double sm_dot(const float* a, const float* b) {
  float x[8], y[8];
  sm_pencil(a, x);
  sm_pencil(b, y);
  double s = 0.0;
#pragma unroll
  for (int k = 0; k < 8; k++) s += double(x[k]) * double(y[k]);
  return wave_sum(s);
}
// The sum of n <= 64 partials as block_sum_partials forms it (every wavefront).
__device__ __forceinline__ double sm_total(const double* part, int n) {
  const int lane = lane_id();
  return wave_sum(0.0 + (lane < n ? part[lane < n ? lane : 0] : -0.0));
}
// KIDS: the problem's LEAF tiles are the children of its one root; else its roots.
template <class V, bool KIDS>
__device__ __forceinline__ void sm_solve(SmallLDS& S, const CoarsePlan& cp, int iters, int flags, V* Z, const VCycleArgs& v,
                                         const Ctx& c) {
  CoarseLDS& M = S.v;
  const int tid = threadIdx.x, wave = uni(tid >> 6), q0 = uni(tid >> 8), r = tid & 255;
  constexpr int first = KIDS ? CL_ROOTS : 0;
  const int n = KIDS ? CL_CHILDREN : cp.n0;  // LEAF tiles
  ProbState* ps = c.ps + cp.prob;
  const ProbState st = state_of(state_word(ps));
  if ((flags & F_CHECK_DONE) && st.done) return;
  CoarseCells L0, L1;
  {
    CoarseRaw R0, R1;
    if (KIDS) cl_issue<V>(c, cp, CL_ROOTS, CL_CHILDREN, R1);
    cl_issue<V>(c, cp, 0, cp.n0, R0);
    if (KIDS) cl_commit(cp, CL_ROOTS, CL_CHILDREN, R1, M, L1);
    cl_commit(cp, 0, cp.n0, R0, M, L0);
  }
  if (tid < 4) M.z[CL_ZERO + tid] = S.p[CL_ZERO + tid] = 0.f;
  CoarseCells& L = KIDS ? L1 : L0;
  auto p_at = [&](uint32_t byte) -> float& { return *reinterpret_cast<float*>(reinterpret_cast<char*>(S.p) + byte); };
  // natural cell index (in its tile) of the thread's cell of colour col
  auto nat = [&](int col) {
    const int i = r >> 5, j = (r >> 2) & 7;
    return (i << 6) + (j << 3) + 2 * (r & 3) + ((col + i + j) & 1);
  };
  float x[2][CL_CPT];
  auto tile_of = [&](int m) { return size_t(cp.slots[first + q0 + 4 * m].tile) * 512; };
  auto leaf_at = [&](uint32_t at) { return (at >> 2) - first * 512; };  // index into S.r, M.t
#pragma unroll
  for (int col = 0; col < 2; col++)
    cl_each<KIDS>(L, col, [&](int m, uint32_t at) {
      const size_t g = tile_of(m) + nat(col);
      x[col][m] = c.x[g];
      S.r[leaf_at(at)] = c.r[g];
      p_at(at) = c.p[g];
    });
  __syncthreads();
  auto interior = [&](int col, int m) { return ((L.in >> (2 * m + col)) & 1) != 0; };
  double gamma = st.gamma, alpha = st.alpha;
  int it = st.iter, done = st.done;
  if (tid == 0) S.out = st;
  for (int k = 0; k < iters && !done; k++) {
    if (st.pure_neumann) {  // k_mean, FIN_MEAN, k_subtract_mean
      if (wave < n) {
        float w[8];
        sm_pencil(S.r + wave * 512, w);
        const uint64_t ct = load_ct8(c.ctype + size_t(cp.slots[first + wave].tile) * 512 + lane_id() * 8);
        double a = 0.0, q = 0.0;
#pragma unroll
        for (int e = 0; e < 8; e++) { a += double(w[e]); q += (ct_at(ct, e) & C_INT) ? 1.0 : 0.0; }
        a = wave_sum(a);
        q = wave_sum(q);
        if (lane_id() == 0) { S.part[SM_MEAN][wave] = a; S.part[SM_COUNT][wave] = q; }
      }
      __syncthreads();
      const double mean = sm_total(S.part[SM_MEAN], n) / sm_total(S.part[SM_COUNT], n);
      if (tid == 0) S.out.mean = mean;
#pragma unroll
      for (int col = 0; col < 2; col++)
        cl_each<KIDS>(L, col, [&](int m, uint32_t at) {
          if (interior(col, m)) S.r[leaf_at(at)] = float(double(S.r[leaf_at(at)]) - mean);
        });
    }
    // z = M^-1 r
#pragma unroll
    for (int col = 0; col < 2; col++) {
      cl_each<false>(L0, col, [&](int, uint32_t at) { cl_at(M, at) = 0.f; });
      if (KIDS) cl_each<true>(L1, col, [&](int, uint32_t at) { cl_at(M, at) = 0.f; });
      cl_each<KIDS>(L, col, [&](int m, uint32_t at) { L.P[col][m].b = vround<V>(S.r[leaf_at(at)]); });
    }
    __syncthreads();
    cl_vcycle<V>(M, cp, KIDS ? CL_CHILDREN : 0, L0, L1, v);
    // gamma = r.z, beta
    if (wave < n) {
      const double a = sm_dot(S.r + wave * 512, M.z + (first + wave) * 512);
      if (lane_id() == 0) S.part[SM_RZ][wave] = a;
    }
    __syncthreads();
    const double gamma_old = gamma;
    gamma = sm_total(S.part[SM_RZ], n);
    const double beta = it == 0 ? 0.0 : gamma / gamma_old;
    if (tid == 0) {
      S.out.gamma_old = gamma_old;
      S.out.beta = beta;
    }
    // the last iteration's x, p = z + beta p
    const float fb = float(beta), fa = float(alpha);
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<KIDS>(L, col, [&](int m, uint32_t at) {
        if (!interior(col, m)) return;
        float& p = p_at(at);
        if (it > 0) x[col][m] = __builtin_fmaf(fa, p, x[col][m]);
        p = __builtin_fmaf(fb, p, cl_at(M, at));
      });
    __syncthreads();
    // A p
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<KIDS>(L, col, [&](int m, uint32_t at) {
        const CoarseCell& Q = L.P[col][m];
        const float p = p_at(at);
        float sum = 0.f;
#pragma unroll
        for (int f = 0; f < 3; f++) {
          sum = __builtin_fmaf(L.cf, p - p_at(Q.nb[f] & 0xffffu), sum);
          sum = __builtin_fmaf(L.cf, p - p_at(Q.nb[f] >> 16), sum);
        }
        M.t[leaf_at(at)] = interior(col, m) ? ((sum * L.h) * L.h) * L.h : 0.f;
      });
    __syncthreads();
    if (wave < n) {
      const double a = sm_dot(S.p + (first + wave) * 512, M.t + wave * 512);
      if (lane_id() == 0) S.part[SM_PAP][wave] = a;
    }
    __syncthreads();
    const double pap = sm_total(S.part[SM_PAP], n);
    if (tid == 0) S.out.pAp = pap;
    alpha = gamma / pap;
    const float na = -float(alpha);
#pragma unroll
    for (int col = 0; col < 2; col++)
      cl_each<KIDS>(L, col, [&](int m, uint32_t at) {
        if (interior(col, m)) S.r[leaf_at(at)] = __builtin_fmaf(na, M.t[leaf_at(at)], S.r[leaf_at(at)]);
      });
    __syncthreads();
    if (wave < n) {
      const double a = sm_dot(S.r + wave * 512, S.r + wave * 512);
      if (lane_id() == 0) S.part[SM_RR][wave] = a;
    }
    __syncthreads();
    const double rr = sm_total(S.part[SM_RR], n);
    it++;
    const int cs = st.check_stride;
    const bool converged = cs > 0 && it % cs == 0 && rr < st.thr;
    if (converged || it >= st.max_iters) done = 1;
    if (tid == 0) {
      S.out.rr = rr;
      if (converged) S.out.converged = 1;
    }
  }
  // back to memory, as the launches of the last iteration would leave it
#pragma unroll
  for (int col = 0; col < 2; col++) {
    cl_each<KIDS>(L, col, [&](int m, uint32_t at) {
      const size_t g = tile_of(m) + nat(col);
      c.x[g] = x[col][m];
      c.p[g] = p_at(at);
      c.r[g] = S.r[leaf_at(at)];
      c.ap[g] = M.t[leaf_at(at)];
      vc_rhs<V>(c)[tile_of(m) + col * 256 + r] = from_f<V>(S.r[leaf_at(at)]);
      Z[tile_of(m) + col * 256 + r] = from_f<V>(cl_at(M, at));
    });
    if (KIDS)
      cl_each<false>(L0, col, [&](int m, uint32_t at) {
        Z[size_t(cp.slots[q0 + 4 * m].tile) * 512 + col * 256 + r] = from_f<V>(cl_at(M, at));
      });
  }
  if (tid != 0) return;
  S.out.gamma = gamma;
  S.out.alpha = alpha;
  S.out.iter = it;
  S.out.done = done;
  *ps = S.out;
  if (c.progress) __hip_atomic_store(c.progress + cp.prob, 2 * it + done, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}
template <class V>
__global__ __launch_bounds__(CL_THREADS) void k_cg_small(const CoarsePlan* __restrict__ plans, int iters, int flags, V* Z,
                                                         VCycleArgs v, Ctx c) {
  __shared__ SmallLDS S;
  const CoarsePlan& cp = plans[blockIdx.x];
  if (cp.n1) sm_solve<V, true>(S, cp, iters, flags, Z, v, c);
  else sm_solve<V, false>(S, cp, iters, flags, Z, v, c);
}

// Pure-Neumann re-centring (MeanAsync + ReCenterLeafVoxels,
// PoissonGrid.cu:231-325, PoissonSolver.cu:356-368): mean of r over all cells
// of LEAF tiles divided by the INTERIOR count, subtracted on INTERIOR cells.
__global__ __launch_bounds__(64) void k_mean(const TileRec* __restrict__ list, int n, int flags,
                                             const float* __restrict__ X, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const uint32_t word = state_word(c.ps + T.prob);
  float v[8];
  load8(X + base, v);
  const uint64_t ct = load_ct8(c.ctype + base);
  hold8(v);
  const ProbState ps = state_of(word);
  if (((flags & F_CHECK_DONE) && ps.done) || !ps.pure_neumann) return;
  double a = 0.0, q = 0.0;
  for (int k = 0; k < 8; k++) { a += double(v[k]); q += (ct_at(ct, k) & C_INT) ? 1.0 : 0.0; }
  a = wave_sum(a);
  q = wave_sum(q);
  if (lane == 0) { c.part[T.leaf_slot] = a; c.part2[T.leaf_slot] = q; }
}
template <class V>
__global__ __launch_bounds__(64) void k_subtract_mean(const TileRec* __restrict__ list, int n, int flags,
                                                      float* __restrict__ X, int write_rhsv, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  const uint32_t word = state_word(c.ps + T.prob);
  float v[8];
  load8(X + base, v);
  const uint64_t ct = load_ct8(c.ctype + base);
  hold8(v);
  const ProbState ps = state_of(word);
  if (((flags & F_CHECK_DONE) && ps.done) || !ps.pure_neumann) return;
  const double mean = ps.mean;
  for (int k = 0; k < 8; k++) if (ct_at(ct, k) & C_INT) v[k] = float(double(v[k]) - mean);
  store8(X + base, v);
  if (write_rhsv) store8_split(vc_rhs<V>(c) + size_t(T.self) * 512, lane_id(), v);
}

// ---------------------------------------------------------------------------
// Channel-level kernels for the operator API
// ---------------------------------------------------------------------------
// Ghost x from the parent's INTERIOR value (PoissonGrid.cu:585-605).
__global__ __launch_bounds__(64) void k_propagate_ghosts(Ctx c, const TileRec* __restrict__ list, int n,
                                                         const float* __restrict__ XC, float* __restrict__ XF) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const int oct = tr_octant(T), ox = oct & 1, oy = (oct >> 1) & 1, oz = (oct >> 2) & 1;
  const size_t pb = size_t(T.parent) * 512 + ((ox * 4 + (i >> 1)) << 6) + ((oy * 4 + (j >> 1)) << 3) + oz * 4;
  const float4 pv = *reinterpret_cast<const float4*>(XC + pb);
  const uint32_t pc = *reinterpret_cast<const uint32_t*>(c.ctype + pb);
  const float cv[4] = {pv.x, pv.y, pv.z, pv.w};
  const uint64_t ct = load_ct8(c.ctype + base);
  float out[8];
  for (int k = 0; k < 8; k++) {
    bool pin = uint8_t(pc >> (8 * (k >> 1))) & C_INT;
    out[k] = ((ct_at(ct, k) & C_INT) && pin) ? cv[k >> 1] : 0.f;
  }
  store8(XF + base, out);
}
// Ghost rows summed into the parent channel (AccumulateToParents128 with
// coefficient 1, additive, all cell types; PoissonGrid.cu:664-719).
__global__ __launch_bounds__(64) void k_accumulate_ghosts(Ctx c, const TileRec* __restrict__ list, int n, float* __restrict__ AX) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  __shared__ float gl[512];
  float v[8];
  load8(AX + base, v);
  const uint64_t ct = load_ct8(c.ctype + base);
  for (int k = 0; k < 8; k++) gl[lane * 8 + k] = (ct_at(ct, k) & (C_INT | C_DIR | C_NEU)) ? v[k] : 0.f;
  wave_sync();
  float s = octet_sum(gl, lane);
  size_t pcell = parent_cell(T, lane);
  AX[pcell] = AX[pcell] + s * 1.0f;
}
// Per-tile dot partials over all cells of the listed tiles, then one total.
// FP64 sum of a[c] * b[c] over the 512 cells of one tile: each lane over its
// pencil in cell order, then the xor butterfly across the wavefront.
__device__ __forceinline__ double tile_dot(const float* __restrict__ A, const float* __restrict__ Bv, int tile) {
  const size_t base = size_t(tile) * 512 + lane_id() * 8;
  float a[8], b[8];
  load8(A + base, a);
  load8(Bv + base, b);
  double s = 0.0;
  for (int k = 0; k < 8; k++) s += double(a[k]) * double(b[k]);
  return wave_sum(s);
}
__global__ __launch_bounds__(64) void k_dot_tiles(const TileRec* __restrict__ list, int n, const float* __restrict__ A,
                                                  const float* __restrict__ Bv, double* __restrict__ part) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const double s = tile_dot(A, Bv, T.self);
  if (lane_id() == 0) part[w] = s;
}
// The indices i < n (ascending) of the tiles whose type is in `types`, written
// to sel[0 ..); one workgroup of SEL_THREADS walks the records in chunks, each
// chunk's ranks from wavefront ballots and a scan of the wavefront counts.
constexpr int SEL_THREADS = 1024;
__global__ __launch_bounds__(SEL_THREADS) void k_select_tiles(const TileRec* __restrict__ tiles, int n, int types,
                                                              int32_t* __restrict__ sel) {
  __shared__ int wcount[SEL_THREADS / 64];
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  int base = 0;
  for (int c0 = 0; c0 < n; c0 += SEL_THREADS) {
    const int i = c0 + tid;
    const bool take = i < n && (tr_type(tiles[i]) & types) != 0;
    const uint64_t bal = __ballot(take);
    const int below = __popcll(bal & ((uint64_t(1) << lane) - 1));
    if (lane == 0) wcount[wave] = __popcll(bal);
    __syncthreads();
    int before = 0, total = 0;
    for (int v = 0; v < SEL_THREADS / 64; v++) {
      before += v < wave ? wcount[v] : 0;
      total += wcount[v];
    }
    if (take) sel[base + before + below] = i;
    base += total;
    __syncthreads();  // wcount is rewritten by the next chunk
  }
}
// Tile partials of the selected tiles: partial q of tile sel[q] (q < count).
__global__ __launch_bounds__(64) void k_dot_selected(const int32_t* __restrict__ sel, int count, const float* __restrict__ A,
                                                     const float* __restrict__ Bv, double* __restrict__ part) {
  const int q = blockIdx.x;
  if (q >= count) return;
  const double s = tile_dot(A, Bv, sel[q]);
  if (lane_id() == 0) part[q] = s;
}
template <int NT>
__global__ __launch_bounds__(NT) void k_sum_partials(const double* __restrict__ part, int n, double* __restrict__ out) {
  const double s = block_sum_partials<NT>(part, 0, n);
  if (threadIdx.x == 0) *out = s;
}
// Copy whole tiles of a list from one channel to another.
__global__ __launch_bounds__(64) void k_copy_tiles(const TileRec* __restrict__ list, int n, const float* __restrict__ src,
                                                   float* __restrict__ dst) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float v[8];
  load8(src + base, v);
  store8(dst + base, v);
}
// Natural <-> colour-split order of whole tiles (channels handed to the
// operator API are natural; the V-cycle kernels work on split arrays).
__global__ __launch_bounds__(64) void k_to_split(const TileRec* __restrict__ list, int n, const float* __restrict__ src,
                                                 float* __restrict__ dst) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  float v[8];
  load8(src + size_t(T.self) * 512 + lane_id() * 8, v);
  store8_split(dst + size_t(T.self) * 512, lane_id(), v);
}
__global__ __launch_bounds__(64) void k_from_split(const TileRec* __restrict__ list, int n, const float* __restrict__ src,
                                                   float* __restrict__ dst) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  float v[8];
  load8_split(src + size_t(T.self) * 512, lane_id(), v);
  store8(dst + size_t(T.self) * 512 + lane_id() * 8, v);
}
// ---------------------------------------------------------------------------
// AMGSolver (AMGSolver.cu): stored coefficients and their V-cycle, natural
// cell order, FP32.  Coefficient arrays: off[a] = the cell's minus-face entry
// along axis a, diag; cell types of the AMG hierarchy in amgct (NONLEAF cells
// retyped by the coarsening, the others as given).
// ---------------------------------------------------------------------------
struct AmgC {
  float* off[3];
  float* diag;
  uint8_t* ct;
};
// AMGSolver.cu:17-36
__device__ __forceinline__ float amg_coeff(float h, uint8_t t0, uint8_t t1, uint8_t c0, uint8_t c1) {
  const int both = (t0 & T_LEAF) && (t1 & T_LEAF);
  const int lg = ((t0 & T_LEAF) && (t1 & T_GHOST)) || ((t0 & T_GHOST) && (t1 & T_LEAF));
  const float odh = (1.f / h) * float(both) + (1.f / (1.5f * h)) * float(lg);
  const int hn = (c0 & C_NEU) || (c1 & C_NEU);
  return hn ? 0.f : odh / h;
}
// face neighbour tile f (x-,y-,z-,x+,y+,z+) of T: index (-1: none) and type
__device__ __forceinline__ int amg_nbr(const TileRec& T, int f) { return uni(T.nbr[f]); }

// Step 1 of CoarsenTypesAndAMGCoeffs (AMGSolver.cu:118-131): a GHOST cell takes
// its parent cell's type (a GHOST tile's parent always exists).
__global__ __launch_bounds__(64) void k_amg_ghost_types(const TileRec* __restrict__ list, int n,
                                                        const uint8_t* __restrict__ ctype, uint8_t* __restrict__ amgct) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const int o = tr_octant(T);
  const size_t pb = size_t(T.parent) * 512 + (((o & 1) * 4 + (i >> 1)) * 8 + (((o >> 1) & 1) * 4 + (j >> 1))) * 8 +
                    ((o >> 2) & 1) * 4;
  for (int k = 0; k < 8; k++) amgct[size_t(T.self) * 512 + lane * 8 + k] = ctype[pb + (k >> 1)];
}

// CalculateAMGCoefficients (AMGSolver.cu:40-107) on LEAF|GHOST tiles: lane
// (i,j) owns cells k = 0..7; neighbour cell types from the own tile or the
// face neighbour (none: DIRICHLET cell, the tile's own type).
__global__ __launch_bounds__(64) void k_amg_coeffs(const TileRec* __restrict__ list, int n, AmgC A) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t tb = size_t(T.self) * 512;
  const uint8_t t0 = tr_type(T);
  const float h = T.h;
  const uint8_t* ctype = A.ct;
  const uint64_t own = load_ct8(ctype + tb + lane * 8);
  // the four in-plane neighbour pencils' cell types and tile types
  uint64_t nct[4];
  uint8_t ntt[4];
  const int pi[4] = {i - 1, i + 1, i, i};
  const int pj[4] = {j, j, j - 1, j + 1};
  const int pf[4] = {0, 3, 1, 4};
  for (int q = 0; q < 4; q++) {
    const bool inside = pi[q] >= 0 && pi[q] < 8 && pj[q] >= 0 && pj[q] < 8;
    if (inside) { nct[q] = load_ct8(ctype + tb + (pi[q] * 8 + pj[q]) * 8); ntt[q] = t0; continue; }
    const int nb = amg_nbr(T, pf[q]);
    if (nb < 0) { nct[q] = 0x0101010101010101ull; ntt[q] = t0; continue; }  // DIRICHLET, own type
    nct[q] = load_ct8(ctype + size_t(nb) * 512 + (((pi[q] + 8) & 7) * 8 + ((pj[q] + 8) & 7)) * 8);
    ntt[q] = tr_ntype(T, pf[q]);
  }
  uint8_t kmc = C_DIR, kpc = C_DIR, kmt = t0, kpt = t0;
  {
    const int nb = amg_nbr(T, 2);
    if (nb >= 0) { kmc = ctype[size_t(nb) * 512 + lane * 8 + 7]; kmt = tr_ntype(T, 2); }
    const int np = amg_nbr(T, 5);
    if (np >= 0) { kpc = ctype[size_t(np) * 512 + lane * 8]; kpt = tr_ntype(T, 5); }
  }
  float out[4][8];
  for (int k = 0; k < 8; k++) {
    const uint8_t c0 = ct_at(own, k);
    const uint8_t c1s[6] = {ct_at(nct[0], k), ct_at(nct[1], k), ct_at(nct[2], k), ct_at(nct[3], k),
                            k > 0 ? ct_at(own, k - 1) : kmc, k < 7 ? ct_at(own, k + 1) : kpc};
    const uint8_t t1s[6] = {ntt[0], ntt[1], ntt[2], ntt[3], k > 0 ? t0 : kmt, k < 7 ? t0 : kpt};
    float diag = 0.f, off[3] = {0.f, 0.f, 0.f};
    for (int e = 0; e < 6; e++) {  // x-, x+, y-, y+, z-, z+
      const float coeff = ((amg_coeff(h, t0, t1s[e], c0, c1s[e]) * h) * h) * h;
      if ((e & 1) == 0 && c1s[e] == C_INT) off[e >> 1] = -coeff;
      diag = diag + coeff;
    }
    const bool in = c0 == C_INT;
    for (int a = 0; a < 3; a++) out[a][k] = in ? off[a] : 0.f;
    out[3][k] = in ? diag : 0.f;
  }
  for (int a = 0; a < 3; a++) store8(A.off[a] + tb + lane * 8, out[a]);
  store8(A.diag + tb + lane * 8, out[3]);
}

// Step 3 of CoarsenTypesAndAMGCoeffs (AMGSolver.cu:137-207) from the child
// side: the tiles of one level (children) each fill the 4x4x4 cells of their
// parent's octant, lane = parent cell.  LEAF|NONLEAF children: the NONLEAF
// parent's cell type and the Galerkin sums times one_over_alpha; GHOST
// children: the sums added to the LEAF parent's own coefficients.  Sums in the
// reference's order (children ci, cj, ck lexicographic).
__global__ __launch_bounds__(64) void k_amg_coarsen(const TileRec* __restrict__ list, int n, AmgC A, float alpha) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id();
  const int qi = lane >> 4, qj = (lane >> 2) & 3, qk = lane & 3;
  const size_t tb = size_t(T.self) * 512;
  float cod[3][8];
  float dsum = 0.f;
  int interior = 0;
  for (int ci = 0; ci < 2; ci++)
    for (int cj = 0; cj < 2; cj++)
      for (int ck = 0; ck < 2; ck++) {
        const int q = (ci * 2 + cj) * 2 + ck;
        const size_t cc = tb + ((2 * qi + ci) * 8 + (2 * qj + cj)) * 8 + (2 * qk + ck);
        dsum = dsum + A.diag[cc];
        interior += A.ct[cc] == C_INT;
        for (int a = 0; a < 3; a++) cod[a][q] = A.off[a][cc];
      }
  float offs[3] = {0.f, 0.f, 0.f};
  for (int ci = 0; ci < 2; ci++)
    for (int cj = 0; cj < 2; cj++)
      for (int ck = 0; ck < 2; ck++) {
        const int q = (ci * 2 + cj) * 2 + ck;
        if (ci == 0) offs[0] = offs[0] + cod[0][q];
        if (ci == 1) dsum = dsum + 2.f * cod[0][q];
        if (cj == 0) offs[1] = offs[1] + cod[1][q];
        if (cj == 1) dsum = dsum + 2.f * cod[1][q];
        if (ck == 0) offs[2] = offs[2] + cod[2][q];
        if (ck == 1) dsum = dsum + 2.f * cod[2][q];
      }
  const int o = tr_octant(T);
  const size_t pc = size_t(T.parent) * 512 + (((o & 1) * 4 + qi) * 8 + (((o >> 1) & 1) * 4 + qj)) * 8 + (((o >> 2) & 1) * 4 + qk);
  if (tr_type(T) == T_GHOST) {
    for (int a = 0; a < 3; a++) A.off[a][pc] = A.off[a][pc] + offs[a];
    A.diag[pc] = A.diag[pc] + dsum;
  } else {
    A.ct[pc] = interior > 0 ? C_INT : C_DIR;
    for (int a = 0; a < 3; a++) A.off[a][pc] = offs[a] * alpha;
    A.diag[pc] = dsum * alpha;
  }
}

// VCycleAMG's first step (AMGSolver.cu:616-628): x = 0, rhs = f (0 on GHOST tiles).
__global__ __launch_bounds__(64) void k_amg_init(const TileRec* __restrict__ list, int n, float* __restrict__ X,
                                                 const float* __restrict__ F, float* __restrict__ RHS, int flags) {
  TILE_KERNEL_PROLOGUE
  const size_t b = size_t(T.self) * 512 + lane_id() * 8;
  float v[8], z[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  if (tr_type(T) == T_GHOST) store8(RHS + b, z);
  else { load8(F + b, v); store8(RHS + b, v); }
  store8(X + b, z);
}

// A x with the stored coefficients for the lane's 8 cells (negativeLapSameLevel,
// AMGSolver.cu:232-250): x0 d + sum over x-, x+, y-, y+, z-, z+ of the face's
// entry times the neighbour's x, the plus faces' entries read from the plus
// neighbour's minus-face entry (0 where there is no neighbour tile: every load is
// unconditional, from the zero page there, and all are out before the first use;
// as branches, and with the uses between them, they were several round trips in
// turn).  A sweep's colour on 64 tiles 3.08 -> 2.62 us, on 2,048 tiles 5.86 -> 5.24.
__device__ __forceinline__ void amg_rows(const TileRec& T, const float* __restrict__ X, const AmgC& A, float x0[8],
                                         float ax[8], float dg[8]) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t tb = size_t(T.self) * 512 + lane * 8;
  const float* zp = zero_page<float>();
  float xs[4][8], os[2][8];  // x of the x-, x+, y-, y+ pencils; off_x of x+, off_y of y+
  auto pencil = [&](int nb, bool inside, int pl, size_t& at) {  // false: outside the grid
    at = size_t(inside ? int(T.self) : nb) * 512 + (pl & 63) * 8;
    return inside || nb >= 0;
  };
  load8(X + tb, x0);
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const bool x = q < 2, plus = q & 1;
    const bool inside = plus ? (x ? i : j) < 7 : (x ? i : j) > 0;
    const int pl = x ? lane + (plus ? 8 : -8) : (inside ? lane + (plus ? 1 : -1) : lane + (plus ? -7 : 7));
    size_t at;
    const bool ok = pencil(amg_nbr(T, (plus ? 3 : 0) + (x ? 0 : 1)), inside, pl, at);
    load8(ok ? X + at : zp, xs[q]);
    if (plus) load8(ok ? A.off[x ? 0 : 1] + at : zp, os[x ? 0 : 1]);
  }
  float ox[8], oy[8], oz[8];
  load8(A.off[0] + tb, ox);
  load8(A.off[1] + tb, oy);
  load8(A.off[2] + tb, oz);
  load8(A.diag + tb, dg);
  const int nm = amg_nbr(T, 2), np = amg_nbr(T, 5);
  const float xkm = *(nm >= 0 ? X + size_t(nm) * 512 + lane * 8 + 7 : zp);
  const float xkp = *(np >= 0 ? X + size_t(np) * 512 + lane * 8 : zp);
  float ozp = *(np >= 0 ? A.off[2] + size_t(np) * 512 + lane * 8 : zp);
  // all of it in flight before the first use
  hold8(x0);
#pragma unroll
  for (int q = 0; q < 4; q++) hold8(xs[q]);
  hold8(os[0]);
  hold8(os[1]);
  hold8(ox);
  hold8(oy);
  hold8(oz);
  hold8(dg);
  hold_f(ozp);
#pragma unroll
  for (int k = 0; k < 8; k++) {
    float sum = x0[k] * dg[k];
    sum = __builtin_fmaf(ox[k], xs[0][k], sum);
    sum = __builtin_fmaf(os[0][k], xs[1][k], sum);
    sum = __builtin_fmaf(oy[k], xs[2][k], sum);
    sum = __builtin_fmaf(os[1][k], xs[3][k], sum);
    sum = __builtin_fmaf(oz[k], k > 0 ? x0[k - 1] : xkm, sum);
    sum = __builtin_fmaf(k < 7 ? oz[k + 1] : ozp, k < 7 ? x0[k + 1] : xkp, sum);
    ax[k] = sum;
  }
}

// One colour of GaussSeidelAMG (AMGSolver.cu:540-578) on LEAF|NONLEAF tiles
// (D = 0 leaves the cell unchanged, as in the GMG smoother).
__global__ __launch_bounds__(64) void k_amg_gs(const TileRec* __restrict__ list, int n, int flags,
                                               float* __restrict__ X, const float* __restrict__ RHS, AmgC A,
                                               int color, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id();
  const size_t b = size_t(T.self) * 512 + lane * 8;
  float rhs[8], x0[8], ax[8], dg[8];
  load8(RHS + b, rhs);
  const uint64_t ct = load_ct8(A.ct + b);
  const uint32_t dn = done_load(c, T, flags);
  amg_rows(T, X, A, x0, ax, dg);
  if (done_test(dn, flags)) return;
  wave_sync();  // every lane has read its neighbours before any lane writes
  const bool odd = even_colour(lane) != color;  // of the pencil's cells the even or the odd ones
#pragma unroll
  for (int m = 0; m < 4; m++) {
    const float d = odd ? dg[2 * m + 1] : dg[2 * m];
    const float res = odd ? rhs[2 * m + 1] - ax[2 * m + 1] : rhs[2 * m] - ax[2 * m];
    const float delta = ((odd ? ct_at(ct, 2 * m + 1) : ct_at(ct, 2 * m)) & C_INT) ? (d != 0.f ? res / d : 0.f) : 0.f;
    x0[2 * m] = odd ? x0[2 * m] : x0[2 * m] + delta;
    x0[2 * m + 1] = odd ? x0[2 * m + 1] + delta : x0[2 * m + 1];
  }
  store8(X + b, x0);
}

// The residual of VCycleAMG (AMGSolver.cu:638-642), rhs - A x on INTERIOR cells
// and 0 elsewhere, on every tile of a level, and its restriction
// (PoissonSolver.cu:292-316): LEAF and NONLEAF tiles fill their parent's octant,
// rhs = the sum over the 8 children (x fastest) of their residuals times
// one_over_alpha; a GHOST tile's residual goes to TMP, for its LEAF parent
// (k_amg_leaf_rhs).
__global__ __launch_bounds__(64) void k_amg_residual(const TileRec* __restrict__ list, int n, int flags,
                                                     const float* __restrict__ X, float* __restrict__ RHS,
                                                     float* __restrict__ TMP, float alpha, AmgC A, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  __shared__ float R[512];
  const int lane = lane_id();
  const size_t b = size_t(T.self) * 512 + lane * 8;
  float x0[8], ax[8], dg[8], rhs[8];
  load8(RHS + b, rhs);
  const uint64_t ct = load_ct8(A.ct + b);
  const uint32_t dn = done_load(c, T, flags);
  amg_rows(T, X, A, x0, ax, dg);
  if (done_test(dn, flags)) return;
  float out[8];
#pragma unroll
  for (int k = 0; k < 8; k++) out[k] = (ct_at(ct, k) == C_INT) ? rhs[k] - ax[k] : 0.f;
  if (tr_type(T) == T_GHOST) {
    store8(TMP + b, out);
    return;
  }
  store8(R + lane * 8, out);
  wave_sync();
  const int qi = lane >> 4, qj = (lane >> 2) & 3, qk = lane & 3;
  float sum = 0.f;
#pragma unroll
  for (int s = 0; s < 8; s++) sum = sum + R[((2 * qi + (s & 1)) * 8 + (2 * qj + ((s >> 1) & 1))) * 8 + (2 * qk + (s >> 2))];
  const int o = tr_octant(T);
  RHS[size_t(T.parent) * 512 + (((o & 1) * 4 + qi) * 8 + (((o >> 1) & 1) * 4 + qj)) * 8 + (((o >> 2) & 1) * 4 + qk)] =
      sum * alpha;
}

// VCycleAMG's rhs on the LEAF tiles of the coarser level that have GHOST children
// (AMGSolver.cu:652-656): f plus the 8-cell sums of their residuals
// (AccumulateToParents, PoissonGrid.cu:721-755).  The other LEAF tiles keep the f
// and the GHOST tiles the 0 of k_amg_init.
__global__ __launch_bounds__(64) void k_amg_leaf_rhs(const TileRec* __restrict__ list, int n, int flags,
                                                     const float* __restrict__ TMP, const float* __restrict__ F,
                                                     float* __restrict__ RHS, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const uint32_t dn = done_load(c, T, flags);
  const GhostKids& kids = c.kids[T.gslot];
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t b = size_t(T.self) * 512 + lane * 8;
  float out[8];
  load8(F + b, out);
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const int g = kids.tile[(i >> 2) | ((j >> 2) << 1) | (h << 2)];  // the ghost child of octant (i, j, h)
    // the child's four pencils under this one, cells 0..7 each
    const float* src = g >= 0 ? TMP + size_t(g) * 512 + ((i & 3) * 16 + (j & 3) * 2) * 8 : zero_page<float>();
    const int di = g >= 0 ? 64 : 0, dj = g >= 0 ? 8 : 0;
    float v[4][8];
#pragma unroll
    for (int q = 0; q < 4; q++) load8(src + (q & 1) * di + (q >> 1) * dj, v[q]);
#pragma unroll
    for (int k = 0; k < 4; k++) {
      float sum = 0.f;
#pragma unroll
      for (int cid = 0; cid < 8; cid++) sum = sum + v[cid & 3][2 * k + (cid >> 2)];
      out[4 * h + k] = __builtin_fmaf(sum, 1.f, out[4 * h + k]);
    }
  }
  if (done_test(dn, flags)) return;
  store8(RHS + b, out);
}

// z of the LEAF tiles into the CG's colour-split array, with the r.z partials that
// k_cg_dot_rz forms.
__global__ __launch_bounds__(64) void k_amg_finish(const TileRec* __restrict__ list, int n, int flags,
                                                   const float* __restrict__ X, float* __restrict__ Z, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id();
  const size_t b = size_t(T.self) * 512 + lane * 8;
  float z[8], r[8];
  const uint32_t dn = done_load(c, T, flags);
  load8(X + b, z);
  load8(c.r + b, r);
  hold8(z);
  hold8(r);
  if (done_test(dn, flags)) return;
  store8_split(Z + size_t(T.self) * 512, lane, z);
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(r[k]) * double(z[k]);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
}

// ProlongateAndUpdate128 (GMGSolver.cu:345-380) on the AMG hierarchy, natural
// order: GHOST x = parent x on INTERIOR cells, others x += pcoef parent x on
// INTERIOR cells, 0 elsewhere.
__global__ __launch_bounds__(64) void k_amg_prolong(const TileRec* __restrict__ list, int n, int flags,
                                                    float* __restrict__ X, AmgC A, float pcoef, Ctx c) {
  TILE_KERNEL_PROLOGUE_C
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t b = size_t(T.self) * 512 + lane * 8;
  float x[8];
  const uint32_t dn = done_load(c, T, flags);
  load8(X + b, x);
  const uint64_t ct = load_ct8(A.ct + b);
  const int o = tr_octant(T);
  const size_t pb = size_t(T.parent) * 512 + (((o & 1) * 4 + (i >> 1)) * 8 + (((o >> 1) & 1) * 4 + (j >> 1))) * 8 +
                    ((o >> 2) & 1) * 4;
  float px[4];
  for (int q = 0; q < 4; q++) px[q] = X[pb + q];
  for (int q = 0; q < 4; q++) hold_f(px[q]);
  hold8(x);
  if (done_test(dn, flags)) return;
  const bool ghost = tr_type(T) == T_GHOST;
  for (int k = 0; k < 8; k++) {
    const bool in = ct_at(ct, k) & C_INT;
    const float cx = px[k >> 1];
    x[k] = in ? (ghost ? cx : __builtin_fmaf(pcoef, cx, x[k])) : 0.f;
  }
  store8(X + b, x);
}

// ---------------------------------------------------------------------------
// The coarse levels 0..C (C <= 1) of VCycleAMG for one problem in one workgroup,
// on the plan of k_coarse_lds and in its LDS layout: the sweeps, residual,
// restriction and prolongation of the kernels above, cell by cell in their
// order (AMGSolver.cu:540-715).  The rows are the stored coefficients: own entry
// across a minus face, the plus neighbour's entry across a plus face (0 without
// a neighbour), the diagonal.  With nine tiles, two sweeps and ten bottom
// iterations it takes the place of 32 launches of 2-4 us, each bound by launch
// and memory latency (the AMG solve on the 128^3 coarse/fine plane 8.2 -> 6.5 ms).
// ---------------------------------------------------------------------------
struct AmgCell {
  uint32_t nb[3];  // LDS byte addresses of the six neighbours' x (CL_ZERO: none)
  float cf[6];     // entries across x-, x+, y-, y+, z-, z+
  float dg, b;
  double rd;       // 1 / dg (0: not updated)
};
struct AmgCells {
  AmgCell P[2][CL_CPT];  // as CoarseCells
  uint32_t in, in1;      // bit 2 * m + colour: type has the INTERIOR bit; type is INTERIOR
  uint32_t own;
  int n;
};
// natural index of cell r (pencil * 4 + k / 2) of colour col
__device__ __forceinline__ int cl_natural(int col, int r) {
  return ((r >> 2) << 3) + 2 * (r & 3) + ((col + (r >> 5) + (r >> 2)) & 1);
}
__device__ __forceinline__ void amg_cells(const CoarsePlan& cp, int first, int n, const AmgC& A,
                                          const float* __restrict__ RHS, AmgCells& L) {
  const int q0 = uni(int(threadIdx.x) >> 8), r = threadIdx.x & 255;
  const int i = r >> 5, j = (r >> 2) & 7;
  L.own = uint32_t(4 * ((first + q0) * 512 + r));
  L.n = n > q0 ? (n - q0 + 3) >> 2 : 0;
  L.in = L.in1 = 0;
#pragma unroll
  for (int m = 0; m < CL_CPT; m++)
    if (m < L.n) {
      const int s = first + q0 + 4 * m;
      const CoarseSlot& S = cp.slots[s];
      const size_t tb = size_t(S.tile) * 512;
#pragma unroll
      for (int col = 0; col < 2; col++) {
        AmgCell& P = L.P[col][m];
        const int cc = cl_natural(col, r), k = cc & 7;
        const bool inside[6] = {i > 0, i < 7, j > 0, j < 7, k > 0, k < 7};
        const int step[6] = {-64, 64, -8, 8, -1, 1};
        const int face[6] = {0, 3, 1, 4, 2, 5};
        uint32_t at[6];
#pragma unroll
        for (int e = 0; e < 6; e++) {
          const int q = inside[e] ? s : S.nbr[face[e]];
          const int nc = inside[e] ? cc + step[e] : cc - 7 * step[e];
          at[e] = 4u * uint32_t(q < 0 ? CL_ZERO : q * 512 + split_index(nc));
          if ((e & 1) == 0) P.cf[e] = A.off[e >> 1][tb + cc];
          else P.cf[e] = q < 0 ? 0.f : A.off[e >> 1][size_t(cp.slots[q].tile) * 512 + nc];
        }
#pragma unroll
        for (int e = 0; e < 3; e++) P.nb[e] = at[2 * e] | (at[2 * e + 1] << 16);
        P.dg = A.diag[tb + cc];
        P.b = RHS[tb + cc];
        const uint8_t ct = A.ct[tb + cc];
        L.in |= uint32_t((ct & C_INT) != 0) << (2 * m + col);
        L.in1 |= uint32_t(ct == C_INT) << (2 * m + col);
        P.rd = ((ct & C_INT) && P.dg != 0.f) ? recip64(P.dg) : 0.0;
      }
    }
}
// rhs - A x of a cell with value x0 (amg_rows' order)
__device__ __forceinline__ float amg_cell_residual(CoarseLDS& M, const AmgCell& P, float x0) {
  float xn[6];
#pragma unroll
  for (int f = 0; f < 3; f++) {
    xn[2 * f] = cl_at(M, P.nb[f] & 0xffffu);
    xn[2 * f + 1] = cl_at(M, P.nb[f] >> 16);
  }
  float sum = x0 * P.dg;
#pragma unroll
  for (int f = 0; f < 6; f++) sum = __builtin_fmaf(P.cf[f], xn[f], sum);
  return P.b - sum;
}
template <class F>
__device__ __forceinline__ void amg_each(const AmgCells& L, int col, F f) {
#pragma unroll
  for (int m = 0; m < CL_CPT; m++)
    if (m < L.n) f(m, L.own + m * CL_M + col * CL_COL);
}
__device__ __forceinline__ void amg_cl_gs(CoarseLDS& M, const AmgCells& L, int col) {
  amg_each(L, col, [&](int m, uint32_t at) {
    const AmgCell& Q = L.P[col][m];
    const float x0 = cl_at(M, at);
    const float res = amg_cell_residual(M, Q, x0);
    cl_at(M, at) = x0 + (Q.rd != 0.0 ? div_by_rounded(res, Q.rd) : 0.f);
  });
  __syncthreads();
}
__global__ __launch_bounds__(CL_THREADS) void k_amg_coarse(const CoarsePlan* __restrict__ plans, int flags,
                                                           float* __restrict__ X, const float* __restrict__ RHS, int nu,
                                                           int coarsest, float alpha, float pcoef, AmgC A, Ctx c) {
  __shared__ CoarseLDS M;
  const int tid = threadIdx.x;
  const CoarsePlan& cp = plans[blockIdx.x];
  const int n0 = cp.n0, n1 = cp.n1;
  if ((flags & F_CHECK_DONE) && c.ps[cp.prob].done) return;
  for (int q = tid; q < CL_ZERO + 4; q += CL_THREADS) M.z[q] = 0.f;
  AmgCells L;
  const int q0 = uni(tid >> 8), r = tid & 255;
  constexpr uint32_t T0 = CL_ROOTS * 512;
  if (n1) {
    amg_cells(cp, CL_ROOTS, n1, A, RHS, L);
    __syncthreads();
    for (int it = 0; it < nu; it++) { amg_cl_gs(M, L, 0); amg_cl_gs(M, L, 1); }
    // residuals on INTERIOR cells (0 elsewhere), then their sums (x fastest)
#pragma unroll
    for (int col = 0; col < 2; col++)
      amg_each(L, col, [&](int m, uint32_t at) {
        const float res = amg_cell_residual(M, L.P[col][m], cl_at(M, at));
        M.t[(at >> 2) - T0] = ((L.in1 >> (2 * m + col)) & 1) ? res : 0.f;
      });
    __syncthreads();
    if (tid < CL_CHILDREN * 64) {
      const int q = uni(tid >> 6), lq = tid & 63;
      const CoarseSlot& S = cp.slots[CL_ROOTS + q];
      const int a = lq >> 4, bq = (lq >> 2) & 3, cq = lq & 3;
      float sum = 0.f;
#pragma unroll
      for (int o = 0; o < 8; o++)  // a cell that is not INTERIOR holds 0 in t
        sum = sum + M.t[q * 512 + split_cell(2 * a + (o & 1), 2 * bq + ((o >> 1) & 1), 2 * cq + (o >> 2))];
      M.b0[S.parent * 512 + split_cell((S.octant & 1) * 4 + a, ((S.octant >> 1) & 1) * 4 + bq,
                                       ((S.octant >> 2) & 1) * 4 + cq)] = sum * alpha;
    }
    __syncthreads();
  }
  amg_cells(cp, 0, n0, A, RHS, L);
  if (n1) {
    // a root with children takes the restricted rhs (a LEAF root keeps its own)
    const int refined = cp.slots[CL_ROOTS].parent;
#pragma unroll
    for (int col = 0; col < 2; col++)
      amg_each(L, col, [&](int m, uint32_t at) {
        if (q0 + 4 * m == refined) L.P[col][m].b = M.b0[at >> 2];
      });
  }
  __syncthreads();
  for (int it = 0; it < coarsest / 2; it++) { amg_cl_gs(M, L, 0); amg_cl_gs(M, L, 1); }
  for (int it = 0; it < coarsest / 2; it++) { amg_cl_gs(M, L, 1); amg_cl_gs(M, L, 0); }
  auto store = [&](int first) {
#pragma unroll
    for (int col = 0; col < 2; col++)
      amg_each(L, col, [&](int m, uint32_t at) {
        X[size_t(cp.slots[first + q0 + 4 * m].tile) * 512 + cl_natural(col, r)] = cl_at(M, at);
      });
  };
  store(0);
  if (n1) {
    // the level's rows again (kept over the bottom solve they would not fit the registers)
    amg_cells(cp, CL_ROOTS, n1, A, RHS, L);
    const int i = r >> 5, j = (r >> 2) & 7, e = r & 3;
    amg_each(L, 0, [&](int m, uint32_t at) {
      const CoarseSlot& S = cp.slots[CL_ROOTS + q0 + 4 * m];
      const int pi = (S.octant & 1) * 4 + (i >> 1), pj = ((S.octant >> 1) & 1) * 4 + (j >> 1);
      const float cz = M.z[S.parent * 512 + split_cell(pi, pj, ((S.octant >> 2) & 1) * 4 + e)];
#pragma unroll
      for (int col = 0; col < 2; col++) {
        float& z = cl_at(M, at + col * CL_COL);
        z = ((L.in >> (2 * m + col)) & 1) ? __builtin_fmaf(pcoef, cz, z) : 0.f;
      }
    });
    __syncthreads();
    for (int it = 0; it < nu; it++) { amg_cl_gs(M, L, 1); amg_cl_gs(M, L, 0); }
    store(CL_ROOTS);
  }
}

// Fill whole tiles of a list with a value.
template <class V = float>
__global__ __launch_bounds__(64) void k_fill_tiles(const TileRec* __restrict__ list, int n, V* __restrict__ dst, float val) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float v[8] = {val, val, val, val, val, val, val, val};
  store8(dst + base, v);
}
// dampedJacobiSolve pieces (GMGSolver.cu:479-525) on LEAF tiles:
// R = B - R on INTERIOR cells; then X += omega R / D (X = 0 where D == 0).
__global__ __launch_bounds__(64) void k_leaf_residual(Ctx c, const TileRec* __restrict__ list, int n,
                                                      const float* __restrict__ B, float* __restrict__ R) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float b[8], r[8];
  load8(B + base, b);
  load8(R + base, r);
  const uint64_t ct = load_ct8(c.ctype + base);
  for (int k = 0; k < 8; k++) if (ct_at(ct, k) & C_INT) r[k] = b[k] - r[k];
  store8(R + base, r);
}
__global__ __launch_bounds__(64) void k_leaf_jacobi_update(Ctx c, const TileRec* __restrict__ list, int n, float* __restrict__ X,
                                                           const float* __restrict__ R, const float* __restrict__ D, float omega) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float x[8], r[8], d[8];
  load8(X + base, x);
  load8(R + base, r);
  load8(D + base, d);
  const uint64_t ct = load_ct8(c.ctype + base);
  for (int k = 0; k < 8; k++)
    if (ct_at(ct, k) & C_INT) x[k] = (d[k] == 0.f) ? 0.f : x[k] + (omega * r[k]) / d[k];
  store8(X + base, x);
}

// ---------------------------------------------------------------------------
// Mixed-precision form: the FP64 outer loop of the iterative refinement (no
// reference counterpart).  x64 and the residual r64 are FP64 arrays beside the
// FP32 channels; the operator is FullNegativeLaplacian (GMGSolver.cu:203-213)
// evaluated in FP64 with the reference's per-face order, so the CPU
// transcription in FP64 gives the same bits.  Each inner solve is the FP32
// MGPCG on the FP32-rounded residual; its x is added to x64.
// ---------------------------------------------------------------------------
__device__ __forceinline__ void load8d(const double* __restrict__ p, double v[8]) {
  const double2* q = reinterpret_cast<const double2*>(p);
#pragma unroll
  for (int h = 0; h < 4; h++) {
    const double2 t = q[h];
    v[2 * h] = t.x;
    v[2 * h + 1] = t.y;
  }
}
__device__ __forceinline__ void store8d(double* __restrict__ p, const double v[8]) {
  double2* q = reinterpret_cast<double2*>(p);
#pragma unroll
  for (int h = 0; h < 4; h++) q[h] = make_double2(v[2 * h], v[2 * h + 1]);
}
// Face coefficient before the NEUMANN cut in FP64 (GMGSolver.cu:26-39).
__device__ __forceinline__ double base_coeff64(uint8_t t0, uint8_t t1, double ooh) {
  const bool both = (t0 & T_LEAF) && (t1 & T_LEAF);
  const bool lg = ((t0 & T_LEAF) && (t1 & T_GHOST)) || ((t0 & T_GHOST) && (t1 & T_LEAF));
  return both ? ooh * ooh : (lg ? ((2.0 * ooh) / 3.0) * ooh : 0.0);
}

// Ghost x64 from the parent's INTERIOR value (PoissonGrid.cu:585-605).
__global__ __launch_bounds__(64) void k_propagate_ghosts64(Ctx c, const TileRec* __restrict__ list, int n, double* __restrict__ X) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const int oct = tr_octant(T), ox = oct & 1, oy = (oct >> 1) & 1, oz = (oct >> 2) & 1;
  const size_t pb = size_t(T.parent) * 512 + ((ox * 4 + (i >> 1)) << 6) + ((oy * 4 + (j >> 1)) << 3) + oz * 4;
  const double2 p0 = reinterpret_cast<const double2*>(X + pb)[0], p1 = reinterpret_cast<const double2*>(X + pb)[1];
  const double cv[4] = {p0.x, p0.y, p1.x, p1.y};
  const uint32_t pc = *reinterpret_cast<const uint32_t*>(c.ctype + pb);
  const uint64_t ct = load_ct8(c.ctype + base);
  double out[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const bool pin = uint8_t(pc >> (8 * (k >> 1))) & C_INT;
    out[k] = ((ct_at(ct, k) & C_INT) && pin) ? cv[k >> 1] : 0.0;
  }
  store8d(X + base, out);
}

// A x64 on every cell of the listed LEAF and GHOST tiles with their own types
// (NegativeLaplacianSameLevel128 with no subtree view, GMGSolver.cu:145-200),
// in FP64.  Neighbour pencils are read straight from memory (this runs once per
// refinement step, not per CG iteration).
__global__ __launch_bounds__(64) void k_apply64(Ctx c, const TileRec* __restrict__ list, int n, const double* __restrict__ X,
                                                double* __restrict__ AX) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  // the tile's pencils and its halo ring, index (i+1)*10 + (j+1), cells 0..7
  __shared__ double xs[100][8];
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t self = size_t(T.self) * 512;
  const size_t base = self + lane * 8;
  const double h = double(T.h);
  const double ooh = 1.0 / h;
  const uint8_t to = tr_type(T);
  const double* zp = zero_page<double>();
  // ---- loads, none in a branch: own pencil, one ring pencil (lanes 0..31;
  // x = 0 outside the grid), the two k halos, the face masks
  double own[8], ring[8];
  load8d(X + base, own);
  const int g = (lane >> 3) & 3, t = lane & 7;
  const int rn = pick4(g, uni(T.nbr[0]), uni(T.nbr[3]), uni(T.nbr[1]), uni(T.nbr[4]));
  const bool rok = lane < 32 && rn >= 0;
  load8d(rok ? X + size_t(rn) * 512 + ring_src(g, t) * 8 : zp, ring);
  const double xkm = *(T.nbr[2] >= 0 ? X + size_t(T.nbr[2]) * 512 + lane * 8 + 7 : zp);
  const double xkp = *(T.nbr[5] >= 0 ? X + size_t(T.nbr[5]) * 512 + lane * 8 : zp);
  const uint64_t m = load_ct8(own_masks(c, T) + lane * 8);
  double bf[6];
#pragma unroll
  for (int f = 0; f < 6; f++) bf[f] = base_coeff64(to, T.nbr[f] < 0 ? to : tr_ntype(T, f), ooh);
  const double bint = base_coeff64(to, to, ooh);
  const int pc = (i + 1) * 10 + (j + 1);
#pragma unroll
  for (int k = 0; k < 8; k++) xs[pc][k] = own[k];
  if (lane < 32) {
#pragma unroll
    for (int k = 0; k < 8; k++) xs[ring_dst(g, t)][k] = ring[k];
  }
  wave_sync();
  const double bim = (i == 0) ? bf[0] : bint, bip = (i == 7) ? bf[3] : bint;
  const double bjm = (j == 0) ? bf[1] : bint, bjp = (j == 7) ? bf[4] : bint;
  double out[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    const double xn[6] = {xs[pc - 10][k], xs[pc + 10][k], xs[pc - 1][k], xs[pc + 1][k], k == 0 ? xkm : own[k - 1],
                          k == 7 ? xkp : own[k + 1]};
    const double bc[6] = {bim, bip, bjm, bjp, k == 0 ? bf[2] : bint, k == 7 ? bf[5] : bint};
    const uint32_t mk = ct_at(m, k);
    double sum = 0.0;
#pragma unroll
    for (int e = 0; e < 6; e++) sum = __builtin_fma((mk & (1u << e)) ? bc[e] : 0.0, own[k] - xn[e], sum);
    out[k] = (mk & M_INT) ? ((sum * h) * h) * h : 0.0;
  }
  store8d(AX + base, out);
}

// Ghost rows of A x64 summed into the parent (AccumulateToParents128 with
// coefficient 1, additive, all cell types; PoissonGrid.cu:664-719).
__global__ __launch_bounds__(64) void k_accumulate_ghosts64(Ctx c, const TileRec* __restrict__ list, int n, double* __restrict__ AX) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  __shared__ double gl[512];
  double v[8];
  load8d(AX + base, v);
  const uint64_t ct = load_ct8(c.ctype + base);
  for (int k = 0; k < 8; k++) gl[lane * 8 + k] = (ct_at(ct, k) & (C_INT | C_DIR | C_NEU)) ? v[k] : 0.0;
  wave_sync();
  const int a = lane >> 4, bq = (lane >> 2) & 3, cq = lane & 3;
  double sum = 0.0;
  for (int ii = 0; ii < 2; ii++)
    for (int jj = 0; jj < 2; jj++)
      for (int kk = 0; kk < 2; kk++) sum += gl[((2 * a + ii) * 8 + (2 * bq + jj)) * 8 + 2 * cq + kk];
  const size_t pcell = parent_cell(T, lane);
  AX[pcell] = AX[pcell] + sum * 1.0;
}

// |b|^2 partials of the LEAF tiles (per leaf slot).
__global__ __launch_bounds__(64) void k_ir_norm(Ctx c, const TileRec* __restrict__ list, int n, const float* __restrict__ B) {
  const int flags = F_SWIZZLE;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float b[8];
  load8(B + base, b);
  double a = 0.0;
  for (int k = 0; k < 8; k++) a += double(b[k]) * double(b[k]);
  a = wave_sum(a);
  if (lane_id() == 0) c.part[T.leaf_slot] = a;
}
// X *= 2^(sign * scale_exp) on every cell of the LEAF tiles (exact: a power of two).
__global__ __launch_bounds__(64) void k_scale_leaf(Ctx c, const TileRec* __restrict__ list, int n, float* __restrict__ X,
                                                   int sign) {
  const int flags = F_SWIZZLE;
  TILE_KERNEL_PROLOGUE
  const float f = ldexpf(1.f, sign * c.ps[T.prob].scale_exp);
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float v[8];
  load8(X + base, v);
  for (int k = 0; k < 8; k++) v[k] = v[k] * f;
  store8(X + base, v);
}
// r64 = b - A x64 on every cell of the LEAF tiles (R holds A x64 on entry).
//   mode 0: the next inner solve's rhs r = float(r64), partials of |r64|^2;
//   mode 1 (pure Neumann, before re-centring): partials of sum r64 and of the
//           INTERIOR count (MeanAsync, PoissonGrid.cu:231-325);
//   mode 2: partials of |r64|^2 only (a check of a finished solve).
__global__ __launch_bounds__(64) void k_ir_residual(Ctx c, const TileRec* __restrict__ list, int n, const float* __restrict__ B,
                                                    double* __restrict__ R, int mode) {
  const int flags = F_SWIZZLE;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  float b[8];
  double r[8];
  load8(B + base, b);
  load8d(R + base, r);
  for (int k = 0; k < 8; k++) r[k] = double(b[k]) - r[k];
  store8d(R + base, r);
  double a = 0.0, q = 0.0;
  if (mode == 0) {
    float rf[8];
    for (int k = 0; k < 8; k++) { rf[k] = float(r[k]); a += r[k] * r[k]; }
    store8(c.r + base, rf);
  } else if (mode == 2) {
    for (int k = 0; k < 8; k++) a += r[k] * r[k];
  } else {
    const uint64_t ct = load_ct8(c.ctype + base);
    for (int k = 0; k < 8; k++) { a += r[k]; q += (ct_at(ct, k) & C_INT) ? 1.0 : 0.0; }
    q = wave_sum(q);
  }
  a = wave_sum(a);
  if (lane == 0) {
    c.part[T.leaf_slot] = a;
    if (mode == 1) c.part2[T.leaf_slot] = q;
  }
}
// Pure Neumann: r64 -= mean on INTERIOR cells (ReCenterLeafVoxels,
// PoissonSolver.cu:356-368, in FP64), then as k_ir_residual mode 0.
__global__ __launch_bounds__(64) void k_ir_recenter(Ctx c, const TileRec* __restrict__ list, int n, double* __restrict__ R,
                                                    int write_r) {
  const int flags = F_SWIZZLE;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id();
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const double mean = c.ps[T.prob].mean;
  double r[8];
  load8d(R + base, r);
  const uint64_t ct = load_ct8(c.ctype + base);
  for (int k = 0; k < 8; k++) if (ct_at(ct, k) & C_INT) r[k] = r[k] - mean;
  store8d(R + base, r);
  float rf[8];
  double a = 0.0;
  for (int k = 0; k < 8; k++) { rf[k] = float(r[k]); a += r[k] * r[k]; }
  if (write_r) store8(c.r + base, rf);
  a = wave_sum(a);
  if (lane == 0) c.part[T.leaf_slot] = a;
}
// x64 = x on LEAF tiles (the FP32 pressure of a finished solve, to be checked).
__global__ __launch_bounds__(64) void k_ir_load_x(Ctx c, const TileRec* __restrict__ list, int n, const float* __restrict__ X,
                                                  double* __restrict__ X64) {
  const int flags = F_SWIZZLE;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  float xf[8];
  double xd[8];
  load8(X + base, xf);
  for (int k = 0; k < 8; k++) xd[k] = double(xf[k]);
  store8d(X64 + base, xd);
}
// x64 += x (the inner solve's correction) on LEAF tiles; finish: x = float(x64).
__global__ __launch_bounds__(64) void k_ir_accumulate(Ctx c, const TileRec* __restrict__ list, int n, double* __restrict__ X64,
                                                      int finish) {
  const int flags = F_SWIZZLE;
  TILE_KERNEL_PROLOGUE
  const size_t base = size_t(T.self) * 512 + lane_id() * 8;
  double xd[8];
  float xf[8];
  load8d(X64 + base, xd);
  if (finish) {
    for (int k = 0; k < 8; k++) xf[k] = float(xd[k]);
    store8(c.x + base, xf);
    return;
  }
  load8(c.x + base, xf);
  for (int k = 0; k < 8; k++) xd[k] = xd[k] + double(xf[k]);
  store8d(X64 + base, xd);
}
// Per problem q (workgroup -> problem through pmap, else the identity): its
// |r64|^2 (the leaf-slot partials) and |b|^2 (ProbState::bb_b) into
// out[2q], out[2q + 1].
template <int NT>
__global__ __launch_bounds__(NT) void k_ir_verdict(Ctx c, double* __restrict__ out) {
  const int q = c.pmap ? c.pmap[blockIdx.x] : int(blockIdx.x);
  const ProbState* ps = c.ps + q;
  const double s = block_sum_partials<NT>(c.part, ps->leaf_begin, ps->leaf_count);
  if (threadIdx.x == 0) {
    out[2 * q] = s;
    out[2 * q + 1] = ps->bb_b;
  }
}
// Per-problem totals of the leaf-slot partials, in the fixed order.
template <int NT>
__global__ __launch_bounds__(NT) void k_prob_sums(Ctx c, double* __restrict__ out) {
  const ProbState* ps = c.ps + blockIdx.x;
  const double s = block_sum_partials<NT>(c.part, ps->leaf_begin, ps->leaf_count);
  if (threadIdx.x == 0) out[blockIdx.x] = s;
}

// ---------------------------------------------------------------------------
// The projection around the solve (FluidEuler::project, FluidEuler.h:581-612):
// face velocities u, v, w (one value per cell: its minus face, natural
// layout), their divergence as the right-hand side, and the pressure gradient
// added back.  One wavefront per tile, lane = pencil; neighbour pencils are
// read straight from memory (these run once per projection).
// ---------------------------------------------------------------------------
struct Vel {
  float* u[3];
};
__device__ __forceinline__ void load8c(const uint8_t* __restrict__ p, uint8_t v[8]) {
  const uint64_t w = load_ct8(p);
#pragma unroll
  for (int k = 0; k < 8; k++) v[k] = ct_at(w, k);
}

// Ghost velocities from the parents (PropagateToChildren with cell types
// INTERIOR|DIRICHLET|NEUMANN, PoissonGrid.cu:635-661): a typed ghost cell takes
// its parent cell's value (0 if the parent cell is untyped).
__global__ __launch_bounds__(64) void k_propagate_vel(Ctx c, const TileRec* __restrict__ list, int n, Vel U) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const int oct = tr_octant(T), ox = oct & 1, oy = (oct >> 1) & 1, oz = (oct >> 2) & 1;
  const size_t pb = size_t(T.parent) * 512 + ((ox * 4 + (i >> 1)) << 6) + ((oy * 4 + (j >> 1)) << 3) + oz * 4;
  const uint32_t pc = *reinterpret_cast<const uint32_t*>(c.ctype + pb);
  const uint64_t ct = load_ct8(c.ctype + base);
  const uint8_t mask = C_INT | C_DIR | C_NEU;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    const float4 pv = load4(U.u[a] + pb);
    const float cv[4] = {pv.x, pv.y, pv.z, pv.w};
    float v[8];
    load8(U.u[a] + base, v);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      if (!(ct_at(ct, k) & mask)) continue;
      const bool pin = uint8_t(pc >> (8 * (k >> 1))) & mask;
      v[k] = pin ? cv[k >> 1] : 0.f;
    }
    store8(U.u[a] + base, v);
  }
}

// Does a face between tiles of types t0 (the cell's) and t1 count?  LEAF-LEAF,
// LEAF-GHOST, GHOST-LEAF (PoissonSolver.cu:113-119).
__device__ __forceinline__ bool flux_face(uint8_t t0, uint8_t t1) {
  return (t0 == T_LEAF && (t1 == T_LEAF || t1 == T_GHOST)) || (t0 == T_GHOST && t1 == T_LEAF);
}

// VelocityVolumeDivergenceOnLeafs (PoissonSolver.cu:66-137) on LEAF|GHOST
// tiles: INTERIOR cells sum u h^2 over their counted faces in the order x-,
// x+, y-, y+, z-, z+ (-u of the own minus face, +u of the plus neighbour's,
// 0 outside the grid, where the neighbour counts as the tile's own type); the
// other cells get 0.
__global__ __launch_bounds__(64) void k_divergence(Ctx c, const TileRec* __restrict__ list, int n, Vel U,
                                                   float* __restrict__ DIV) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t self = size_t(T.self) * 512;
  const size_t base = self + lane * 8;
  const uint8_t t0 = tr_type(T);
  const float h = T.h;
  float own[3][8];
#pragma unroll
  for (int a = 0; a < 3; a++) load8(U.u[a] + base, own[a]);
  // plus neighbours: u of pencil (i+1,j), v of pencil (i,j+1), w of cell (i,j,k+1)
  float up[8], vp[8], wkp = 0.f;
  uint8_t tx = t0, ty = t0, tz = t0;  // tile types across the plus faces on the tile boundary
  {
    const int nx = T.nbr[3], ny = T.nbr[4], nz = T.nbr[5];
    if (i < 7) load8(U.u[0] + base + 64, up);
    else if (nx >= 0) load8(U.u[0] + size_t(nx) * 512 + j * 8, up);
    else for (int k = 0; k < 8; k++) up[k] = 0.f;
    if (j < 7) load8(U.u[1] + base + 8, vp);
    else if (ny >= 0) load8(U.u[1] + size_t(ny) * 512 + i * 64, vp);
    else for (int k = 0; k < 8; k++) vp[k] = 0.f;
    if (nz >= 0) wkp = U.u[2][size_t(nz) * 512 + lane * 8];
    if (i == 7 && nx >= 0) tx = tr_ntype(T, 3);
    if (j == 7 && ny >= 0) ty = tr_ntype(T, 4);
    if (nz >= 0) tz = tr_ntype(T, 5);
  }
  // tile types across the minus faces on the tile boundary
  const uint8_t sx = (i == 0 && T.nbr[0] >= 0) ? tr_ntype(T, 0) : t0;
  const uint8_t sy = (j == 0 && T.nbr[1] >= 0) ? tr_ntype(T, 1) : t0;
  const uint8_t sz = (T.nbr[2] >= 0) ? tr_ntype(T, 2) : t0;
  const uint64_t ct = load_ct8(c.ctype + base);
  float out[8];
#pragma unroll
  for (int k = 0; k < 8; k++) {
    float sum = 0.f;
    if (ct_at(ct, k) & C_INT) {
      const float fu[6] = {-own[0][k], up[k], -own[1][k], vp[k], -own[2][k], k < 7 ? own[2][k + 1] : wkp};
      const uint8_t ft[6] = {sx, tx, sy, ty, k == 0 ? sz : t0, k == 7 ? tz : t0};
#pragma unroll
      for (int e = 0; e < 6; e++)
        if (flux_face(t0, ft[e])) sum = __builtin_fmaf(fu[e] * h, h, sum);
    }
    out[k] = sum;
  }
  store8(DIV + base, out);
}

// AccumulateToParents(ch, ch, -1, LEAF, SUBTREE, mask, coeff, additive)
// (PoissonGrid.cu:721-755) on LEAF tiles: each cell whose type is in mask adds
// coeff times the sum, in child order (x fastest), of its 8 children (cells of
// its ghost child tile) whose type is in mask.
__device__ __forceinline__ void tile_accumulate_children(const Ctx& c, const TileRec& T, float* __restrict__ X,
                                                         uint8_t mask, float coeff) {
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t base = size_t(T.self) * 512 + lane * 8;
  const uint64_t ct = load_ct8(c.ctype + base);
  float x[8];
  load8(X + base, x);
  // ghost children of the pencil's two octants (k 0..3, k 4..7)
  const int o0 = (i >> 2) | ((j >> 2) << 1);
  int g[2] = {-1, -1};
  if (tr_has_gchild(T)) {
    g[0] = c.kids[T.gslot].tile[o0];
    g[1] = c.kids[T.gslot].tile[4 + o0];
  }
  float fv[2][2][2][8];  // [oz][ii][jj][fine k]
  uint8_t fc[2][2][2][8];
#pragma unroll
  for (int oz = 0; oz < 2; oz++)
#pragma unroll
    for (int ii = 0; ii < 2; ii++)
#pragma unroll
      for (int jj = 0; jj < 2; jj++) {
        const int fi = 2 * (i & 3) + ii, fj = 2 * (j & 3) + jj;
        if (g[oz] >= 0) {
          const size_t fb = size_t(g[oz]) * 512 + (fi * 8 + fj) * 8;
          load8(X + fb, fv[oz][ii][jj]);
          load8c(c.ctype + fb, fc[oz][ii][jj]);
        } else {
#pragma unroll
          for (int k = 0; k < 8; k++) { fv[oz][ii][jj][k] = 0.f; fc[oz][ii][jj][k] = 0; }
        }
      }
#pragma unroll
  for (int k = 0; k < 8; k++) {
    if (!(ct_at(ct, k) & mask)) continue;
    const int oz = k >> 2, kl = 2 * (k & 3);
    float sum = 0.f;
#pragma unroll
    for (int cid = 0; cid < 8; cid++) {
      const int ii = cid & 1, jj = (cid >> 1) & 1, kk = (cid >> 2) & 1;
      if (fc[oz][ii][jj][kl + kk] & mask) sum += fv[oz][ii][jj][kl + kk];
    }
    x[k] = x[k] + sum * coeff;
  }
  store8(X + base, x);
}
__global__ __launch_bounds__(64) void k_accumulate_children(Ctx c, const TileRec* __restrict__ list, int n,
                                                            float* __restrict__ X, uint8_t mask, float coeff) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE_C
  tile_accumulate_children(c, T, X, mask, coeff);
}
// The same for the three face-velocity channels in one launch (one after the
// other inside each wavefront).
__global__ __launch_bounds__(64) void k_accumulate_children_vel(Ctx c, const TileRec* __restrict__ list, int n, Vel U,
                                                                uint8_t mask, float coeff) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE_C
  for (int a = 0; a < 3; a++) tile_accumulate_children(c, T, U.u[a], mask, coeff);
}

// AddGradientToFaceCenters (PoissonSolver.cu:144-204) on LEAF|GHOST tiles
// (ghost p already taken from the parents): ghost velocities start at 0; each
// cell's minus face of each axis gets u += (p1 - p0) / dh with p1, p0 the
// INTERIOR values (0 elsewhere) of the cell and its minus neighbour (0 outside
// the grid, where the neighbour counts as the tile's own type and the cell's
// own cell type), dh = h across LEAF-LEAF faces and 1.5 h across LEAF-GHOST /
// GHOST-LEAF faces, no update across other faces or where either cell is NEUMANN.
__global__ __launch_bounds__(64) void k_gradient(Ctx c, const TileRec* __restrict__ list, int n, const float* __restrict__ P,
                                                 Vel U) {
  const int flags = 0;
  TILE_KERNEL_PROLOGUE
  const int lane = lane_id(), i = lane >> 3, j = lane & 7;
  const size_t self = size_t(T.self) * 512;
  const size_t base = self + lane * 8;
  const uint8_t t0 = tr_type(T);
  const float h = T.h;
  const float dh_lg = float(1.5 * double(h));
  uint8_t c0[8];
  float p1[8];
  load8c(c.ctype + base, c0);
  load8(P + base, p1);
  // minus neighbours: pencil (i-1,j), pencil (i,j-1), cell (i,j,-1)
  float px[8], py[8], pz = 0.f;
  uint8_t cx[8], cy[8], cz = 0;
  bool ex = false, ey = false, ez = false;  // outside the grid
  {
    const int nx = T.nbr[0], ny = T.nbr[1], nz = T.nbr[2];
    if (i > 0) { load8(P + base - 64, px); load8c(c.ctype + base - 64, cx); }
    else if (nx >= 0) { load8(P + size_t(nx) * 512 + (56 + j) * 8, px); load8c(c.ctype + size_t(nx) * 512 + (56 + j) * 8, cx); }
    else ex = true;
    if (j > 0) { load8(P + base - 8, py); load8c(c.ctype + base - 8, cy); }
    else if (ny >= 0) { load8(P + size_t(ny) * 512 + (i * 8 + 7) * 8, py); load8c(c.ctype + size_t(ny) * 512 + (i * 8 + 7) * 8, cy); }
    else ey = true;
    if (nz >= 0) { pz = P[size_t(nz) * 512 + lane * 8 + 7]; cz = c.ctype[size_t(nz) * 512 + lane * 8 + 7]; }
    else ez = true;
  }
  const uint8_t sx = (i == 0 && T.nbr[0] >= 0) ? tr_ntype(T, 0) : t0;
  const uint8_t sy = (j == 0 && T.nbr[1] >= 0) ? tr_ntype(T, 1) : t0;
  const uint8_t sz = (T.nbr[2] >= 0) ? tr_ntype(T, 2) : t0;
#pragma unroll
  for (int a = 0; a < 3; a++) {
    float u[8];
    if (t0 == T_GHOST) { for (int k = 0; k < 8; k++) u[k] = 0.f; }
    else load8(U.u[a] + base, u);
#pragma unroll
    for (int k = 0; k < 8; k++) {
      bool outside;
      uint8_t nt, nc;
      float pn;
      if (a == 0) { outside = (i == 0) && ex; nt = sx; nc = outside ? c0[k] : cx[k]; pn = outside ? 0.f : px[k]; }
      else if (a == 1) { outside = (j == 0) && ey; nt = sy; nc = outside ? c0[k] : cy[k]; pn = outside ? 0.f : py[k]; }
      else if (k > 0) { outside = false; nt = t0; nc = c0[k - 1]; pn = p1[k - 1]; }
      else { outside = ez; nt = sz; nc = outside ? c0[0] : cz; pn = outside ? 0.f : pz; }
      const float pa = (c0[k] & C_INT) ? p1[k] : 0.f;
      const float pb = (nc & C_INT) ? pn : 0.f;
      const bool ll = (t0 & T_LEAF) && (nt & T_LEAF);
      const bool lg = ((t0 & T_LEAF) && (nt & T_GHOST)) || ((t0 & T_GHOST) && (nt & T_LEAF));
      if (!(ll || lg) || (c0[k] & C_NEU) || (nc & C_NEU)) continue;
      u[k] = u[k] + (pa - pb) / (ll ? h : dh_lg);
    }
    store8(U.u[a] + base, u);
  }
}

}  // namespace cg
