// xf_kernels.h -- device-side types of the gfx950 FDTD engine.
//
// Layout in HBM.  All field components share one padded node grid of
// (nx+1) x (ny+1) x pz values (3-D; z fastest, pz = nz+1 rounded up to a
// 128-byte multiple) or (nx+1) x py values (2-D TMz; y fastest), so one
// linear index addresses Ex..Hz of the same (i, j, k) and every wave64 load
// is a contiguous, aligned row segment.  Yee coefficients are compressed to
// a per-cell uint8/uint16 index into a per-pass table of 9 values (the three
// (self, curl_a, curl_b) triples of the pass), which replaces the 18 dense
// per-cell arrays of the reference (fdtd_coefficient.cuh:149-167).
#ifndef XF_KERNELS_H_
#define XF_KERNELS_H_

#include <hip/hip_bf16.h>
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <limits.h>
#include <stdint.h>

#include "../../include/xfdtd_hip.h"

namespace xf {

constexpr int kMaxPml = 6;
constexpr int kMaxTfsfJobs = 12;

// Every device buffer of the engine is global memory.  A pointer read from
// memory (a batch's per-grid descriptors) is not known to the compiler to
// be global, so it would be accessed with flat instructions; a flat load
// counts on the LDS/scalar counter as well, and every wait for a scalar load
// then also waits for the field loads in flight.  gp() states the address
// space, so such accesses become global loads and stores.
template <typename T>
__device__ __forceinline__ __attribute__((address_space(1))) T* gp(T* p) {
  return (__attribute__((address_space(1))) T*)p;
}

// Storage <-> compute conversion.  FP64 and FP32 store what they compute;
// bf16 stores value * scale (scale per E/H) and computes in float.
template <typename S>
struct Store;
// ld_nt / st_nt are the non-temporal forms, used for the streams a pass
// reads once and rewrites (the updated component itself), so they do not
// displace the neighbour rows other waves still need from L2.
template <>
struct Store<double> {
  using C = double;
  static __device__ __forceinline__ C ld(const double* p, int64_t i, C) { return gp(p)[i]; }
  static __device__ __forceinline__ void st(double* p, int64_t i, C v, C) { gp(p)[i] = v; }
  static __device__ __forceinline__ C ld_nt(const double* p, int64_t i, C) {
    return __builtin_nontemporal_load(gp(p) + i);
  }
  static __device__ __forceinline__ void st_nt(double* p, int64_t i, C v, C) {
    __builtin_nontemporal_store(v, gp(p) + i);
  }
};
template <>
struct Store<float> {
  using C = float;
  static __device__ __forceinline__ C ld(const float* p, int64_t i, C) { return gp(p)[i]; }
  static __device__ __forceinline__ void st(float* p, int64_t i, C v, C) { gp(p)[i] = v; }
  static __device__ __forceinline__ C ld_nt(const float* p, int64_t i, C) {
    return __builtin_nontemporal_load(gp(p) + i);
  }
  static __device__ __forceinline__ void st_nt(float* p, int64_t i, C v, C) {
    __builtin_nontemporal_store(v, gp(p) + i);
  }
};
template <>
struct Store<__hip_bfloat16> {
  using C = float;
  static __device__ __forceinline__ C ld(const __hip_bfloat16* p, int64_t i, C inv) {
    return (float)gp(reinterpret_cast<const __bf16*>(p))[i] * inv;
  }
  static __device__ __forceinline__ void st(__hip_bfloat16* p, int64_t i, C v, C scale) {
    p[i] = __float2bfloat16(v * scale);  // generic store: a global-space one costs a register
  }
  // the streaming slots use plain accesses: non-temporal 16-bit loads and
  // stores measured slower at 536^3 (59.9 against 61.9 Gcells/s)
  static __device__ __forceinline__ C ld_nt(const __hip_bfloat16* p, int64_t i, C inv) {
    return ld(p, i, inv);
  }
  static __device__ __forceinline__ void st_nt(__hip_bfloat16* p, int64_t i, C v, C scale) {
    st(p, i, v, scale);
  }
};

template <>
struct Store<__half> {
  using C = float;
  static __device__ __forceinline__ C ld(const __half* p, int64_t i, C inv) {
    return (float)gp(reinterpret_cast<const _Float16*>(p))[i] * inv;
  }
  static __device__ __forceinline__ void st(__half* p, int64_t i, C v, C scale) {
    p[i] = __float2half(v * scale);  // generic store: a global-space one costs a register
  }
  // plain accesses in the streaming slots, as for bf16 (non-temporal 16-bit
  // accesses measured slower: 57.9 against 59.9 Gcells/s at 536^3)
  static __device__ __forceinline__ C ld_nt(const __half* p, int64_t i, C inv) { return ld(p, i, inv); }
  static __device__ __forceinline__ void st_nt(__half* p, int64_t i, C v, C scale) { st(p, i, v, scale); }
};

// Compensated bf16 storage: a value y is kept as hi = bf16(y) (round to
// nearest even) and the residual y - hi, which is exact in float and at most
// half a bf16 ulp, quantised to an int8 in steps of 2^-15 of hi's power of
// two.  hi + q 2^(e-15) has at most 16 significant bits and is rebuilt
// exactly in float, so a stored value carries about 16 bits of mantissa in
// 3 bytes.  Values sit in blocks of 64: 64 bf16 words (128 B), then 64
// residual bytes (64 B), so a wave's 64 consecutive values are two
// contiguous segments.  The tag type is never dereferenced.
struct Bf16c {
  unsigned char b[3];
};

__host__ __device__ __forceinline__ void bf16c_encode(float y, uint16_t& h, int8_t& l) {
  const uint32_t yb = __builtin_bit_cast(uint32_t, y);
  const uint32_t hb = (yb + 0x7fffu + ((yb >> 16) & 1u)) & 0xffff0000u;
  h = static_cast<uint16_t>(hb >> 16);
  const float hi = __builtin_bit_cast(float, hb);
  const float p2 = __builtin_bit_cast(float, hb & 0x7f800000u);
  float q = 0.0f;
  if (p2 != 0.0f) q = rintf((y - hi) * 32768.0f / p2);
  q = fminf(fmaxf(q, -127.0f), 127.0f);
  l = static_cast<int8_t>(static_cast<int>(q));
}

__host__ __device__ __forceinline__ float bf16c_decode(uint16_t h, int8_t l) {
  const uint32_t hb = static_cast<uint32_t>(h) << 16;
  const float hi = __builtin_bit_cast(float, hb);
  const float p2 = __builtin_bit_cast(float, hb & 0x7f800000u);
  return hi + static_cast<float>(l) * (p2 * (1.0f / 32768.0f));
}

// Byte offsets are formed in 32 bits from the element index (the host keeps
// 3 x values below 2^32), so every access is a wave-uniform base plus a
// 32-bit lane offset: value i of block i / 64, lane l = i % 64, has its bf16
// word at 3 (i - l) + 2 l = 3 i - l and its residual at 3 i - 2 l + 128.
template <>
struct Store<Bf16c> {
  using C = float;
  static __device__ __forceinline__ uint64_t off_hi(int64_t i) {
    const uint32_t u = (uint32_t)i;
    return (uint64_t)(3u * u - (u & 63u));
  }
  static __device__ __forceinline__ uint64_t off_lo(int64_t i) {
    const uint32_t u = (uint32_t)i;
    return (uint64_t)(3u * u - 2u * (u & 63u) + 128u);
  }
  static __device__ __forceinline__ const unsigned char* bytes(const Bf16c* p) {
    return reinterpret_cast<const unsigned char*>(p);
  }
  static __device__ __forceinline__ unsigned char* bytes(Bf16c* p) { return reinterpret_cast<unsigned char*>(p); }
  static __device__ __forceinline__ C ld(const Bf16c* p, int64_t i, C inv) {
    return bf16c_decode(*gp(reinterpret_cast<const uint16_t*>(bytes(p) + off_hi(i))),
                        *gp(reinterpret_cast<const int8_t*>(bytes(p) + off_lo(i)))) *
           inv;
  }
  static __device__ __forceinline__ void st(Bf16c* p, int64_t i, C v, C scale) {
    uint16_t h;
    int8_t r;
    bf16c_encode(v * scale, h, r);
    *gp(reinterpret_cast<uint16_t*>(bytes(p) + off_hi(i))) = h;
    *gp(reinterpret_cast<int8_t*>(bytes(p) + off_lo(i))) = r;
  }
  static __device__ __forceinline__ C ld_nt(const Bf16c* p, int64_t i, C inv) {
    return bf16c_decode(__builtin_nontemporal_load(gp(reinterpret_cast<const uint16_t*>(bytes(p) + off_hi(i)))),
                        __builtin_nontemporal_load(gp(reinterpret_cast<const int8_t*>(bytes(p) + off_lo(i))))) *
           inv;
  }
  static __device__ __forceinline__ void st_nt(Bf16c* p, int64_t i, C v, C scale) {
    uint16_t h;
    int8_t r;
    bf16c_encode(v * scale, h, r);
    __builtin_nontemporal_store(h, gp(reinterpret_cast<uint16_t*>(bytes(p) + off_hi(i))));
    __builtin_nontemporal_store(r, gp(reinterpret_cast<int8_t*>(bytes(p) + off_lo(i))));
  }
};

// Loads and stores at a small unsigned element offset from a wave-uniform
// base pointer: the offset is zero-extended from 32 bits, which lets the
// compiler address with the SGPR base + 32-bit VGPR offset form of the
// global instructions (no per-lane 64-bit address arithmetic).
template <typename S>
__device__ __forceinline__ typename Store<S>::C ld32(const S* p, uint32_t i, typename Store<S>::C inv) {
  return Store<S>::ld(p, (int64_t)(uint64_t)i, inv);
}
template <typename S>
__device__ __forceinline__ typename Store<S>::C ld32_nt(const S* p, uint32_t i, typename Store<S>::C inv) {
  return Store<S>::ld_nt(p, (int64_t)(uint64_t)i, inv);
}
template <typename S>
__device__ __forceinline__ void st32(S* p, uint32_t i, typename Store<S>::C v, typename Store<S>::C scale) {
  Store<S>::st(p, (int64_t)(uint64_t)i, v, scale);
}
template <typename S>
__device__ __forceinline__ void st32_nt(S* p, uint32_t i, typename Store<S>::C v, typename Store<S>::C scale) {
  Store<S>::st_nt(p, (int64_t)(uint64_t)i, v, scale);
}

template <typename S>
struct Fields {
  S* e[3];
  S* h[3];
};

template <typename C>
struct Scales {
  C inv_e, inv_h;  // stored -> physical
  C s_e, s_h;      // physical -> stored
};

struct Dims {
  int nx, ny, nz;  // cells
  int64_t sx, sy;  // strides of i and j (k stride is 1 in 3-D; unused in 2-D)
};

// Work decomposition of the 3-D marching kernels: a 1-D grid of nkb * njb *
// nch blocks; block (kb, jb, ch) owns k in [64 kb, 64 kb + 64), j in
// [ty jb, ty jb + ty) and marches i through [chunk ch, chunk (ch + 1)).
// With xcd != 0 the hardware block id is remapped so that each of the 8 XCDs
// (which receive hardware ids round-robin) owns a contiguous run of
// logical tiles (k fastest, then j), keeping the j/k halo rows of
// neighbouring tiles in the same XCD's L2.
struct Tiling {
  int nkb, njb, nch;
  int chunk;
  int xcd;
};

__device__ __forceinline__ void tile_coords(const Tiling& T, int& kb, int& jb, int& ch) {
  const int nblk = T.nkb * T.njb * T.nch;
  int id = blockIdx.x;
  if (T.xcd) {
    const int q = nblk / 8, r = nblk % 8;
    const int x = id % 8, n = id / 8;
    id = x * q + min(x, r) + n;
  }
  kb = id % T.nkb;
  id /= T.nkb;
  jb = id % T.njb;
  ch = id / T.njb;
}

// One PML face for one pass (E or H).  Component A is E_A/H_A of the face's
// (a, b, c) frame, B is E_B/H_B (pml_corrector.cu:50-270).
template <typename C>
struct PmlFace {
  int axis;
  int c0, c1;          // corrected nodes along the main axis
  int a0, a1, b0, b1;  // lateral task (extended by one per component)
  int gstart, nstart, off_c;
  const C* ca;
  const C* cb;
  C* psi_a;
  const C* cpsi_a;
  C* psi_b;
  const C* cpsi_b;
  int64_t sa1, sa2, sb1, sb2;  // shape[1], shape[2] of the two psi arrays
  int ta, tb;  // the coefficient (0..8) of a node's table row equal to every
               // c_psi value of psi_a / psi_b, or -1 (read the c_psi array)
};

template <typename C>
struct PmlPass {
  int n;
  PmlFace<C> f[kMaxPml];
};

// The z faces of a pass applied at the end of each Yee tile (at most two,
// in registration order), or n = 0.
template <typename C>
struct PmlZTail {
  int n;
  PmlFace<C> f[2];
};

// A pass's coefficient table and per-node ids (uint8, or uint16 when wide),
// for the CPML corrections that take c_psi from the node's row
// (PmlFace::ta / tb).
template <typename C>
struct RowRef {
  const C* tab;
  const void* ids;
  int wide;
};

// The z faces of a pass as node boxes (k fastest) for k_pml_z: face q
// covers i in [i0, i0 + ni), j in [j0, j0 + nj), k in [k0, k0 + nk), its
// nodes numbered from start[q]; start[n] is the total.
struct PmlZBox {
  int n;
  int i0[2], j0[2], k0[2];
  int nj[2], nk[2];
  int64_t start[3];
};

// Dense per-cell coefficients of one pass: array 3 c + m holds coefficient
// m (self, curl a, curl b) of component c at every cell, in the padded
// layout of the fields (the reference's per-field coefficient arrays,
// fdtd_coefficient.cuh:149-167).  Used when a scene's coefficient rows are
// too many to deduplicate into a table; a[0] == nullptr means table mode.
template <typename C>
struct Dense9 {
  const C* a[9];
};

// A z = const TF/SF correction left to the Yee tiles (XF_TILE_TFSF_ZTAIL):
// the written nodes at k that no other face of the same component also
// writes, [i0, i1) x [j0, j1); the incident value is taken at kinc (k, or
// the node beyond the face on its negative side).
template <typename C>
struct TfsfZJob {
  int comp, dual;
  int k, kinc;
  int i0, i1, j0, j1;
  C coef;
};

// The z = const TF/SF corrections of a pass applied after each tile's
// march, with what the incident interpolation needs (field names as in
// TfsfPass, so tfsf_inc reads either).
template <typename C>
struct TfsfZTail {
  int n;
  int t_arg;
  const int* t_dev;
  TfsfZJob<C> z[4];
  const C* proj_int[3];
  const C* proj_half[3];
  const C* inc;
  int64_t n_aux;
  int g[3];
  C tr[3];
};

// Everything one 3-D Yee pass (H or E) of one grid needs: the kernels take
// it as a kernel argument (one grid) or from an array in device memory
// (a batch of grids, one launch).
template <typename S>
struct YeePass {
  using C = typename Store<S>::C;
  Fields<S> f;
  const void* ids;              // uint8_t or uint16_t per cell (padded layout)
  const C* tab;                 // 9 coefficients per id
  int ntab;
  const unsigned char* eflag;   // E pass: table rows left to the ADE kernel
  const C* dense[9];            // dense coefficients (padded layout), or null
  Dims d;
  Scales<C> sc;
  int nkb, njb, chunk, nch;     // tiling of this grid
  PmlPass<C> pml;
  PmlZTail<C> zt;               // z faces applied after each tile's march
  TfsfZTail<C> tz;              // z = const TF/SF faces, likewise (n = 0: none)
};

// A TFSF face correction of one component (one reference launch of
// __tFSFcorrect, tfsf_corrector.cu:148-153) as a written-cell box.
template <typename C>
struct TfsfJob {
  int comp, face;
  int o[3], n[3];  // written box origin and extent
  int64_t start;   // first flat thread index of the job
  C coef;          // c{a|b}{axis} * coefficient_flag
  int edge_axis;   // -1: a thread per written node; else only the nodes at
                   // the two ends of this axis (the rest is a TfsfZJob's)
};

template <typename C>
struct TfsfPass {
  int njob;
  int is_e;
  TfsfJob<C> job[kMaxTfsfJobs];
  int64_t total;
  const C* proj_int[3];
  const C* proj_half[3];
  const C* inc;  // e_inc for the H pass, h_inc for the E pass
  int64_t n_aux;
  int g[3];  // total_task start
  C tr[3];   // transform_e (H pass) or transform_h (E pass)
};

struct NfFace {
  int o[3], n[3];
  int64_t start;  // first flat thread index
  int64_t off;    // offset of the face in a frequency block (cells)
};

struct NfPass {
  NfFace face[6];
  int64_t total;     // surface cells over the 6 faces
  int64_t block;     // cells of one frequency block (sum of face sizes)
  int nfreq;
  int64_t nt;
  double2* cur;      // [freq][face cells][4] -> laid out [freq][face][comp][cell]
  const double2* te; // [freq][nt]
  const double2* th;
};

// NF2FF time domain (one box).  A face's surface cells are cut into tiles
// of NT_TILE x NT_TILE cells over its two tangential axes (u < v in x, y, z
// order); one block per tile sums the tile's contributions per time bin
// (k_nftd_tile), one wave per bin then adds the tiles' partial sums in a
// fixed order (k_nftd_reduce).
constexpr int NT_TILE = 16;
constexpr int NT_MAXSPAN = 256;  // time bins one tile may touch in a step (LDS: 52 KiB)

struct NtFace {
  int o[3];         // task origin
  int nu, nv;       // extents along the tangential axes u < v
  int tu, tv;       // tiles along u and v
  int blk0;         // first tile of the face
  int bins;         // bin slots of the face's reduce (>= bins touched in a step)
  int rblk0, nrblk; // the face's reduce blocks
  int64_t prev_off; // first prev value of the face: [ea, eb, ha, hb][n_a][n_b]
  int nb;           // extent along b (prev row length)
  double rd_min, rd_max;  // range of r . r_unit over the face's cells
};

struct NtPass {
  NtFace face[6];
  int nblk, nrblk;
  int maxspan;      // bins of one tile's partial
  int64_t n_pot;
  double u[3];
  double dmax_e, dmax_h, c_dt;
  const double* e_node[3];
  const double* h_node[3];
  const double* e_size[3];
  double* pot;      // [face][wa, wb, ua, ub][n_pot]
  double* prev;     // per face at prev_off
  double* part;     // [tile][wa, wb, ua, ub][maxspan]
  int* hdr;         // [tile][bmin_e, span_e, bmin_h, span_h]
};

// Point sources: node index (padded layout) and component of each; the
// values are a [source][step] table of doubles.
struct PointDev {
  int n;
  int64_t nt;
  const int* comp;
  const int64_t* idx;
  const double* value;
};

// A movie monitor's box and its frame buffer (doubles, frames x box).
struct MovieDev {
  int field;           // 0..2 E, 3..5 H
  int o[3], n[3];      // box origin and extent
  int64_t interval, frames, box;
  double* data;
};

// The learned layer (xf_learned_boundary): the faces in the mask, in face
// order, with their column ranges; columns are numbered face by face,
// component E_a then E_b, then a-index, then b-index.
struct LbFace {
  int f, c, a, b, positive;
  int tr;              // y faces: threads walk a (= z) fastest and the device
                       // history is stored [b][a], so both stream along z
  int64_t hist_off;    // first history value of the face
  int64_t na1, nb1;    // n_a + 1, n_b + 1 (history plane)
  int64_t start[2];    // first column of E_a, E_b
  int p1[2], q1[2];    // last a-, b-index of E_a, E_b (first is inset)
};

// The MLP weights as the matrix-core predictor's per-lane operands, built
// on the host from the fp16 weights.  For lane l of a wave, g = l / 32:
// a1 holds W1[l % 32][8g + j] (zero for inputs 12..15); a2[p] holds
// W2[l % 32][16p + 8(j / 4) + 4g + j % 4], the hidden unit the layer-1
// result row of that k-slot carries; c1, c2 and w3 hold b1, b2 and w3 of
// unit 8(i / 4) + 4g + i % 4, the row of accumulator element i.
struct LbPack {
  uint16_t a1[64][8];     // fp16 bits
  uint16_t a2[2][64][8];  // fp16 bits
  float c1[16][64];
  float c2[16][64];
  float w3[16][64];
  float b3;
};

struct LbDev {
  int mode, faces, inset, nface;
  float mur_k;
  const LbPack* pack;  // APPLY: the weights as MFMA operands
  float* hist;
  float* rec;          // RECORD: [slot][column][13]
  int rec_every;
  int64_t rec_slots;
  int64_t total;       // columns
  int n[3];
  LbFace face[6];
  // APPLY: the columns whose layer-0 node lies on two faces (edges), for the
  // edge phase and their history roll; the other columns roll their history
  // in the matrix-core phase
  const uint32_t* edge;
  int64_t n_edge;
};

// One grid's TFSF pass, NF2FF box, point sources or learned layer inside a
// batch of grids: the batched kernels read these from device memory, one per
// grid (or box).
template <typename S>
struct TfsfItem {
  using C = typename Store<S>::C;
  Fields<S> f;
  Scales<C> sc;
  Dims d;
  TfsfPass<C> P;
};

template <typename S>
struct NfItem {
  using C = typename Store<S>::C;
  Fields<S> f;
  Scales<C> sc;
  Dims d;
  NfPass P;
};

template <typename S>
struct PmlZItem {
  using C = typename Store<S>::C;
  Fields<S> f;
  Scales<C> sc;
  Dims d;
  PmlPass<C> P;  // the z faces
  PmlZBox B;
  RowRef<C> R;
};

template <typename S>
struct PointItem {
  using C = typename Store<S>::C;
  Fields<S> f;
  Scales<C> sc;
  PointDev P;
};

template <typename S>
struct LbItem {
  using C = typename Store<S>::C;
  Fields<S> f;
  Scales<C> sc;
  Dims d;
  LbDev L;
};

// One step of one grid in a single pass over memory (k_step3): both passes'
// tables, CPML faces and TF/SF jobs, and the two sets of fields and H-pass
// psi it goes between.  In device memory, one per grid and direction.
constexpr int kStep3Rows = 6;       // j-rows a block owns
constexpr int kStep3MaxRows = 256;  // coefficient rows (pairs of E and H rows) the block's table holds (one-byte ids)
constexpr int kStep3AdeRows = 64;   // ... with dispersive media, whose rows are a 64-bit mask
constexpr int kStep3MaxChunk = 32;  // planes a block marches through at most
constexpr int kStep3Proj = 72;      // projections of one axis a block holds: its 64 lanes (or 33 planes, or rows) and 2 a side
constexpr int kStep3Inc = 192;      // incident values of one table row a block holds
constexpr int kStep3ZJobs = 4;      // TF/SF jobs of z faces a block works out before it marches, a pass

// What a plane's correction by a CPML face of one pass takes, in one scalar
// load.  psi of node (i, j, k) is step3_psi_offset bytes past the biased
// pointer (pml_face's layouts for all three axes); psi_a corrects the planes
// [lo, hi_a), psi_b [lo, hi_b).
typedef int step3_i16 __attribute__((vector_size(64)));
template <typename C>
struct alignas(64) Step3Face {
  const C* a;  // psi_a, psi_b read
  const C* b;
  C* oa;  // ... and written (the H pass: the other set's)
  C* ob;
  uint32_t plane_a, plane_b;  // bytes
  int row_a, row_b;           // values
  int lo, hi_a, hi_b;
  int t_ab;  // PmlFace::ta and tb, a byte each (0xff: none)
  // (a second line) c_psi, indexed like psi, where it is no table row; PmlFace's
  // ranges; a profile value is at node + off
  const C* cpa;
  const C* cpb;
  int axis, c0, c1, a0, a1, b0, b1, off;
  const C* ca;
  const C* cb;
};

// A TF/SF job: its box, and where the projections of a node that its
// incident value takes are among the block's (kStep3Proj per axis and grid).
template <typename C>
struct alignas(64) Step3Job {
  int lo[3], hi[3];
  int at[3];
  int comp;
  int axis;
  C coef, tr;
};

// Where psi of node (i, j, k) lies, in bytes from the pointer of a face whose
// planes begin at lo.  In 32 bits (step3_face_fits), so the planes count from
// lo: i planes of a far x face are the grid's size, 2^32 bytes from 813^3 in
// FP64 on.
template <typename C>
__host__ __device__ __forceinline__ uint32_t step3_psi_offset(int i, int j, int k, int lo, int row, uint32_t plane) {
#ifdef __HIP_DEVICE_COMPILE__
  const uint32_t rows = __umul24(j, row);
#else
  const uint32_t rows = ((uint32_t)j & 0xffffffu) * ((uint32_t)row & 0xffffffu);
#endif
  return (rows + (uint32_t)k) * (uint32_t)sizeof(C) + (uint32_t)(i - lo) * plane;
}

// step3_face, step3_job: from the two-pass kernels' descriptors.
template <typename C>
Step3Face<C> step3_face(const PmlFace<C>& F, bool is_e, C* oa, C* ob) {
  Step3Face<C> D{};
  const int64_t sa = F.sa1 * F.sa2, sb = F.sb1 * F.sb2;
  // planes: the main range of an x face; else the lateral range that holds i,
  // which one of the two psi takes closed and the other half-open
  D.lo = F.axis == 0 ? F.c0 : F.axis == 1 ? F.b0 : F.a0;
  const int64_t ka = F.nstart * (F.axis == 0 ? sa : F.axis == 1 ? F.sa2 : 1) - D.lo * sa;
  const int64_t kb = F.nstart * (F.axis == 0 ? sb : F.axis == 1 ? F.sb2 : 1) - D.lo * sb;
  D.a = F.psi_a - ka;
  D.b = F.psi_b - kb;
  D.oa = oa - ka;
  D.ob = ob - kb;
  D.cpa = F.cpsi_a - ka;
  D.cpb = F.cpsi_b - kb;
  D.plane_a = static_cast<uint32_t>(sa * sizeof(C));
  D.plane_b = static_cast<uint32_t>(sb * sizeof(C));
  D.row_a = static_cast<int>(F.sa2);
  D.row_b = static_cast<int>(F.sb2);
  D.t_ab = (F.ta & 0xff) | (F.tb & 0xff) << 8;
  D.axis = F.axis;
  D.c0 = F.c0;
  D.c1 = F.c1;
  D.a0 = F.a0;
  D.a1 = F.a1;
  D.b0 = F.b0;
  D.b1 = F.b1;
  D.off = F.off_c - F.gstart;
  D.ca = F.ca;
  D.cb = F.cb;
  const int hi = F.axis == 0 ? F.c1 : F.axis == 1 ? F.b1 : F.a1;
  const bool a_closed = (F.axis == 1) == is_e;
  D.hi_a = F.axis == 0 ? hi : a_closed ? hi + 1 : hi;
  D.hi_b = F.axis == 0 ? hi : a_closed ? hi : hi + 1;
  return D;
}
// Whether 32 bits (24 for a row's length and number) hold the offset of every
// node that the face corrects.
template <typename C>
bool step3_face_fits(const Step3Face<C>& D) {
  const int64_t j = D.axis == 0 ? D.a1 : D.axis == 1 ? D.c1 - 1 : D.b1;
  const int64_t k = D.axis == 0 ? D.b1 : D.axis == 1 ? D.a1 : D.c1 - 1;
  const int64_t i = (D.hi_a > D.hi_b ? D.hi_a : D.hi_b) - 1 - D.lo;
  for (int q = 0; q < 2; ++q) {
    const int64_t row = q ? D.row_b : D.row_a, plane = q ? D.plane_b : D.plane_a;
    if (row >= (1 << 24) || j >= (1 << 24)) return false;
    if ((j * row + k) * static_cast<int64_t>(sizeof(C)) + i * plane >= (int64_t(1) << 32)) return false;
  }
  return true;
}
template <typename C>
Step3Job<C> step3_job(const TfsfJob<C>& J, const TfsfPass<C>& T) {
  Step3Job<C> D{};
  const bool is_e = T.is_e != 0;
  const int axis = J.face >> 1, a = axis == 2 ? 0 : axis + 1;
  const int dual = J.comp == a ? (a == 2 ? 0 : a + 1) : a;
  const int back = (J.face & 1) ? 0 : is_e ? -1 : 1;
  for (int d = 0; d < 3; ++d) {
    D.lo[d] = J.o[d];
    D.hi[d] = J.o[d] + J.n[d];
    // incident E (H pass) is on the half grid along its own axis only,
    // incident H across it
    const int half = (dual == d) != is_e ? 1 : 0;
    D.at[d] = (2 * d + half) * kStep3Proj + 2 + (axis == d ? back : 0);
  }
  D.comp = J.comp;
  D.axis = axis;
  D.coef = J.coef;
  D.tr = T.tr[dual];
  return D;
}

template <typename S>
struct Step3Pass {
  using C = typename Store<S>::C;
  const S* e[3];
  const S* h[3];
  S* eo[3];
  S* ho[3];
  const uint8_t* ids;    // per node (padded layout): row of tab, 0 where the node is no cell
  const C* tab;          // 18 coefficients a row: the E pass's nine, the H pass's nine
  int ntab;
  int ade;               // rows of dmask are left to the ADE kernel
  uint64_t dmask;
  Dims d;
  Scales<C> sc;
  int nkb, njb, nch, chunk;
  int n_face;
  Step3Face<C> face[2][kMaxPml];  // of the H and the E pass, by axis, then by place
  int n_job[2];                   // TF/SF jobs of the H and the E pass
  Step3Job<C> job[2][kMaxTfsfJobs];
  const C* proj_int[3];
  const C* proj_half[3];
  int g[3];
  const C* inc[2];  // e_inc and h_inc, and their row lengths
  int64_t n_aux[2];
  int n_proj[3];         // lengths of the projection arrays
};

// Launches k_step3 over `blocks` blocks: grid g owns the blocks
// [block_start[g], block_start[g + 1]).  lds: bytes of the largest table.
template <typename S>
hipError_t step3_launch(const Step3Pass<S>* passes, const int* block_start, int n, int blocks, bool pml, size_t lds,
                        int t_arg, const int* t_dev, hipStream_t stream);

// Blocks of k_step3 one CU holds at a time.
template <typename S>
int step3_blocks_per_cu(bool pml, size_t lds);

// Faces of the pass whose corrected box the column (j, k) can meet for some
// i in [i0, i1): a superset of what pml_face accepts (lateral ranges taken
// with their one-node extension).  Worked out once per tile, it lets the
// interior columns skip the CPML code of every plane.
template <typename C>
__device__ __forceinline__ unsigned pml_mask(const PmlPass<C>& P, int i0, int i1, int j, int k) {
  unsigned bits = 0;
  for (int q = 0; q < P.n; ++q) {
    const PmlFace<C>& F = P.f[q];
    bool hit;
    if (F.axis == 0)  // c = i, a = j, b = k
      hit = F.c0 < i1 && F.c1 > i0 && j >= F.a0 && j <= F.a1 && k >= F.b0 && k <= F.b1;
    else if (F.axis == 1)  // c = j, a = k, b = i
      hit = j >= F.c0 && j < F.c1 && k >= F.a0 && k <= F.a1 && F.b0 < i1 && F.b1 >= i0;
    else  // c = k, a = i, b = j
      hit = k >= F.c0 && k < F.c1 && F.a0 < i1 && F.a1 >= i0 && j >= F.b0 && j <= F.b1;
    if (hit) bits |= 1u << q;
  }
  return bits;
}

// exInc..hzInc (tfsf_corrector.cu:18-130): interpolated 1-D incident value.
// P is a TfsfPass or a TfsfZTail (the same field names).
template <template <typename> class Pass, typename C>
__device__ __forceinline__ C tfsf_inc(const Pass<C>& P, bool inc_is_e, int comp, int t,
                                      int i, int j, int k) {
  const int li = i - P.g[0], lj = j - P.g[1], lk = k - P.g[2];
  C proj;
  if (inc_is_e) {
    if (comp == 0)
      proj = gp(P.proj_half[0])[li + 1] + gp(P.proj_int[1])[lj] + gp(P.proj_int[2])[lk];
    else if (comp == 1)
      proj = gp(P.proj_int[0])[li] + gp(P.proj_half[1])[lj + 1] + gp(P.proj_int[2])[lk];
    else
      proj = gp(P.proj_int[0])[li] + gp(P.proj_int[1])[lj] + gp(P.proj_half[2])[lk + 1];
  } else {
    if (comp == 0)
      proj = gp(P.proj_int[0])[li] + gp(P.proj_half[1])[lj + 1] + gp(P.proj_half[2])[lk + 1] - (C)0.5;
    else if (comp == 1)
      proj = gp(P.proj_half[0])[li + 1] + gp(P.proj_int[1])[lj] + gp(P.proj_half[2])[lk + 1] - (C)0.5;
    else
      proj = gp(P.proj_half[0])[li + 1] + gp(P.proj_half[1])[lj + 1] + gp(P.proj_int[2])[lk] - (C)0.5;
  }
  const uint64_t index = (uint64_t)proj;
  const C weight = proj - (C)index;
  const __attribute__((address_space(1))) C* row = gp(P.inc) + (int64_t)t * P.n_aux;
  return P.tr[comp] * ((1 - weight) * row[index] + weight * row[index + 1]);
}

}  // namespace xf

#endif  // XF_KERNELS_H_
