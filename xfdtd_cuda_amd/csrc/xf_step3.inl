// xf_step3.inl -- one 3-D time step, H then E, in one pass over memory.
//
// k_yee_h3 and k_yee_e3 stream the six components twice a step: 18 values
// moved per cell.  k_step3 reads E(t), H(t-1/2) once and writes E(t+1),
// H(t+1/2) once, 12 values a cell, into a second set of field buffers; the
// engine swaps the two sets after the launch.  It also applies the CPML
// corrections of both passes and (no ADE media) their TF/SF corrections, so
// a step is this launch and the monitors.
//
// Decomposition.  A block of RY + 2 waves owns 64 k by RY rows of j and
// marches i through `chunk` planes.  E(t+1) of a node needs H(t+1/2) at
// j - 1, k - 1 and i - 1: wave 0 computes H on the row below the tile, the
// last wave computes H on the column before it (lanes 0..31) and fetches E
// on the column behind it (lanes 32..63), and i - 1 is carried in registers
// (computed once more at a chunk's first plane).  Nothing a block reads is
// written by the launch, so blocks are independent: the old fields and the
// H pass's old psi stay as they were (its new psi go to a second set too;
// the E pass's psi belong to one thread each and are updated in place).
// The row behind the tile comes straight to LDS (global_load_lds), loads
// run a plane ahead of their use, in two register sets that take turns, and
// one barrier a plane orders the LDS exchange.
//
// Bound: HBM, half reads and half writes over twelve arrays.  536^3 FP64
// without CPML takes 3.0 ms for 15.1 GB, 5.0 TB/s, where a plain copy of six
// such arrays into six others reaches 5.4 TB/s and the two-pass kernels take
// 3.9 ms; with CPML, TF/SF and the surface sums 3.77 ms a step (two passes:
// 4.73 ms).  By the counters the latter is 14.5 GB read past the L2s for 8.9
// that a step needs, since blocks that share halo rows and columns run on
// different XCDs, and 8.1 GB written: 22.7 GB at 94 % of the rate of a copy of
// one array.  A block that CPML or a TF/SF face crosses is bound by its waves'
// chains of dependent scalar, LDS and psi accesses instead, two blocks a CU
// to hide them (127 VGPRs in FP64, 96 in FP32), and by the scalars themselves:
// all 106 SGPRs are in use and some 60 more values live in vector lanes, read
// back lane by lane, beside a face's descriptor loaded at every plane.  156^3
// FP64 takes 161 us a step (two passes: 191), 253^3 FP32 423 (417), FP16 430
// (480); where the two passes are faster they run (Engine::step3_pays).  Tiles
// of 6 to 14 rows and 9 to 54 planes a chunk measured within 3 % of each other;
// loads two planes ahead
// gained FP64 nothing and cost FP32 its third block a CU (443 -> 497 us on
// 320^3 without CPML); other block orders (contiguous ranges per XCD, the
// grid's end tiles first) lose 3 to 15 %, because neighbours in j, which read
// each other's halo rows, no longer run together.
//
// Arithmetic and its order per node are those of the two-pass kernels:
// Yee update, CPML faces in registration order, storage rounding, TF/SF
// jobs in order, storage rounding.

typedef int step3_i2 __attribute__((ext_vector_type(2)));
typedef unsigned step3_u2 __attribute__((ext_vector_type(2)));

// lane l gets lane l + 1's value (shl) or lane l - 1's (shr); the end lane
// keeps its own
__device__ __forceinline__ int step3_shl(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x130, 0xf, 0xf, false); }
__device__ __forceinline__ int step3_shr(int x) { return __builtin_amdgcn_update_dpp(x, x, 0x138, 0xf, 0xf, false); }
__device__ __forceinline__ float step3_shl(float v) {
  return __builtin_bit_cast(float, step3_shl(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float step3_shr(float v) {
  return __builtin_bit_cast(float, step3_shr(__builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double step3_shl(double v) {
  step3_i2 b = __builtin_bit_cast(step3_i2, v);
  b.x = step3_shl(b.x);
  b.y = step3_shl(b.y);
  return __builtin_bit_cast(double, b);
}
__device__ __forceinline__ double step3_shr(double v) {
  step3_i2 b = __builtin_bit_cast(step3_i2, v);
  b.x = step3_shr(b.x);
  b.y = step3_shr(b.y);
  return __builtin_bit_cast(double, b);
}

// What a store and a load of v give back (identity for FP64 and FP32).
template <typename S>
__device__ __forceinline__ typename Store<S>::C step3_rt(typename Store<S>::C v, typename Store<S>::C scale,
                                                         typename Store<S>::C inv) {
  if constexpr (__is_same(S, __hip_bfloat16))
    return __bfloat162float(__float2bfloat16(v * scale)) * inv;
  else if constexpr (__is_same(S, __half))
    return __half2float(__float2half(v * scale)) * inv;
  else if constexpr (__is_same(S, Bf16c)) {
    uint16_t h;
    int8_t r;
    bf16c_encode(v * scale, h, r);
    return bf16c_decode(h, r) * inv;
  } else
    return v;
}

// Value `lane` of a 64-value row segment staged in LDS as it is stored.
template <typename S>
__device__ __forceinline__ typename Store<S>::C step3_lds(const unsigned char* row, int lane,
                                                          typename Store<S>::C inv) {
  if constexpr (__is_same(S, Bf16c))
    return bf16c_decode(reinterpret_cast<const uint16_t*>(row)[lane], reinterpret_cast<const int8_t*>(row + 128)[lane]) *
           inv;
  else if constexpr (__is_same(S, __hip_bfloat16))
    return (float)reinterpret_cast<const __bf16*>(row)[lane] * inv;
  else if constexpr (__is_same(S, __half))
    return (float)reinterpret_cast<const _Float16*>(row)[lane] * inv;
  else
    return reinterpret_cast<const S*>(row)[lane];
}

// 16 bytes a lane from global memory to LDS at lds + 16 * lane, with no
// register in between.  Counts on vmcnt like a load, in order; the compiler
// does not see it, so the one wave that issues it waits for it itself (the
// loads it issues after it and uses a plane before are enough).  m0 cannot be
// named as clobbered: the compiler reserves it and writes it right before each
// use of its own.
__device__ __forceinline__ void step3_dma16(const unsigned char* g, unsigned lds) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %0, off" ::"v"(g), "s"(lds) : "memory");
}

// Stores v (already scaled) at byte offset o of p, non-temporal; offsets from
// 2^31 on are dropped.
template <typename S>
__device__ __forceinline__ void step3_store(S* p, uint32_t o, typename Store<S>::C v) {
  const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc(p, 0, 0x7fffffff, 0x00027000);
  constexpr int NT = 2;
  if constexpr (sizeof(S) == 8)
    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(step3_u2, v), r, o, 0, NT);
  else if constexpr (__is_same(S, float))
    __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), r, o, 0, NT);
  else if constexpr (__is_same(S, __half))
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, __float2half(v)), r, o, 0, NT);
  else if constexpr (__is_same(S, __hip_bfloat16))
    __builtin_amdgcn_raw_buffer_store_b16(__builtin_bit_cast(uint16_t, __float2bfloat16(v)), r, o, 0, NT);
}

// Whether psi_a / psi_b of face F correct the node (pml_face's ranges, the
// axis at run time).
template <bool ISE, typename C>
__device__ __forceinline__ void step3_in(const Step3Face<C>& F, int i, int j, int k, bool& in_a, bool& in_b) {
  const int ax = F.axis;
  const int a = ax == 0 ? j : ax == 1 ? k : i;
  const int b = ax == 0 ? k : ax == 1 ? i : j;
  const int c = ax == 0 ? i : ax == 1 ? j : k;
  const bool in_c = c >= F.c0 && c < F.c1;
  const bool half_a = a >= F.a0 && a < F.a1 && b >= F.b0 && b <= F.b1;
  const bool half_b = a >= F.a0 && a <= F.a1 && b >= F.b0 && b < F.b1;
  in_a = in_c && (ISE ? half_a : half_b);
  in_b = in_c && (ISE ? half_b : half_a);
}

// psi read a plane ahead: two values for the y and the z face that a wave
// meets, and for the x face where C is 32 bits.
template <typename C>
struct Step3Psi {
  C a[3], b[3];
};

template <typename C>
struct Step3V {
  C x, y, z;
};

template <typename S, bool PML>
__global__ void __launch_bounds__(64 * (kStep3Rows + 2), 4)
    k_step3(const Step3Pass<S>* __restrict__ passes, const int* __restrict__ block_start, int n_pass, int t_arg,
            const int* __restrict__ t_dev) {
  using C = typename Store<S>::C;
  using V3 = Step3V<C>;
  constexpr int RY = kStep3Rows;
  constexpr int RB = 64 * (int)sizeof(S);  // bytes of a 64-value row segment
  constexpr int CPR = RB / 16;
  // profile values of the block's planes (from i0 - 1), rows (from j0 - 1) and columns (from k0 - 1)
  constexpr int kProfRow = kStep3MaxChunk + 1, kProfCol = kProfRow + RY + 2, kProf = kProfCol + 65;
  extern __shared__ __align__(16) unsigned char step3_smem[];
  __shared__ C sE[2][2][RY + 1][64], sH[2][2][RY + 1][64];
  __shared__ __align__(16) unsigned char sJ[4][2][RB];
  __shared__ C cE[2][RY + 2][2], cF[2][RY + 2][2], cH[2][RY + 2][2];
  __shared__ C sP[6 * kStep3Proj], sI[2][kStep3Inc], sZ[2][kStep3ZJobs][RY + 1][kStep3MaxChunk + 1];
  __shared__ C sPr[PML ? 2 : 1][2][PML ? kProf : 1];
  int inc0 = 0;
  C* const tab = reinterpret_cast<C*>(step3_smem);
  int g = 0;
  if (n_pass > 1) {
    int lo = 0, hi = n_pass - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (block_start[mid] <= (int)blockIdx.x)
        lo = mid;
      else
        hi = mid - 1;
    }
    g = lo;
  }
  const Step3Pass<S>& P = passes[g];
  const int nx = P.d.nx, ny = P.d.ny, nz = P.d.nz;
  const int64_t sx = P.d.sx, sy = P.d.sy;
  const C inv_e = P.sc.inv_e, inv_h = P.sc.inv_h, s_e = P.sc.s_e, s_h = P.sc.s_h;
  const int t = t_dev ? *t_dev : t_arg;
  for (int q = threadIdx.x; q < 18 * P.ntab; q += blockDim.x) tab[q] = gp(P.tab)[q];

  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  int id = (int)blockIdx.x - block_start[g];
  const int kb = id % P.nkb;
  id /= P.nkb;
  const int jb = id % P.njb, ch = id / P.njb;
  const bool col = w == RY + 1, last = w == RY;
  const int k0 = kb * 64, j0 = jb * RY;
  const bool behind = col && lane >= 32;  // the column behind the tile: E only
  const int row = col ? (behind ? min(lane - 32, RY) : min(lane + 1, RY + 1)) : w;
  const int j = j0 - 1 + row;
  const int k = col ? (behind ? k0 + 64 : k0 - 1) : k0 + lane;
  const bool inside = j >= 0 && j <= ny && k >= 0 && k <= nz;
  const bool own = !col && w >= 1 && inside;
  const bool hnode = inside && !behind && row <= RY;  // this lane forms the node's H
  const bool hmain = hnode && j < ny && k < nz;
  const bool mx = own && hmain && j > 0 && k > 0, my = own && hmain && k > 0, mz = own && hmain && j > 0;
  const int i0 = ch * P.chunk, i1 = min(i0 + P.chunk, nx + 1);
  const int jlow = max(j0 - 1, 0);
  const int64_t jof = (int64_t)jlow * sy;
  const uint32_t vo = (uint32_t)((min(max(j, 0), ny) - jlow) * (int)sy + min(max(k, 0), nz));
  // a halo wave's unused component is read from a line it reads anyway
  const S* const fe0 = P.e[0];
  const S* const fe1 = P.e[1];
  const S* const fe2 = P.e[2];
  const S* const fh0 = P.h[0];
  const S* const fh1 = w == 0 ? P.h[0] : P.h[1];
  const S* const fh2 = col ? P.h[0] : P.h[2];
  const uint8_t* const ids = P.ids;
  // Uniform offset of plane i (the last one repeated past the end), opaque so
  // that it stays a scalar added to the scalar bases.
  auto plane = [&](int i) -> int64_t {
    int64_t b = (int64_t)__builtin_amdgcn_readfirstlane(min(i, nx)) * sx + jof;
    asm volatile("" : "+s"(b));
    return b;
  };
  // A lane's value of a row whose base is uniform: a 32-bit byte offset, so
  // that the address is the base in scalars and one register.
  constexpr bool BYTES = !__is_same(S, Bf16c);
  const uint32_t vb = BYTES ? vo * (uint32_t)sizeof(S) : vo;
  auto ld = [&](const S* p, C inv) __attribute__((always_inline)) {
    asm("" : "+s"(p));
    if constexpr (BYTES)
      return Store<S>::ld(reinterpret_cast<const S*>(reinterpret_cast<const unsigned char*>(p) + vb), 0, inv);
    else
      return Store<S>::ld(p, vb, inv);
  };
  // Every wave makes its six stores a plane, buffer stores whose offset is
  // out of range where the lane owns no node (the hardware drops them): the
  // number of memory operations after a load is then known, and its wait
  // leaves them in flight.  Behind a branch they may not have been issued,
  // and each plane waited for the stores of the one before.
  auto st = [&](S* p, C v, C scale) __attribute__((always_inline)) {
    asm("" : "+s"(p));
    if constexpr (BYTES)
      step3_store<S>(p, own ? vb : 0xffffffffu, sizeof(S) < 4 ? v * scale : v);
    else if (own)
      Store<S>::st_nt(p, vb, v, scale);
  };
  auto load_e = [&](V3& v, int i) {
    const int64_t b = plane(i);
    v.x = ld(fe0 + b, inv_e);
    v.y = ld(fe1 + b, inv_e);
    v.z = ld(fe2 + b, inv_e);
  };
  auto load_h = [&](V3& v, int& d, int i) {
    const int64_t b = plane(i);
    v.x = ld(fh0 + b, inv_h);
    v.y = ld(fh1 + b, inv_h);
    v.z = ld(fh2 + b, inv_h);
    const uint8_t* p = ids + b;
    asm("" : "+s"(p));
    d = (int)gp(p)[BYTES ? vb / (uint32_t)sizeof(S) : vb];
  };
  // The row behind the tile (E_x, E_z at j0 + RY), by its last row's wave.
  const uint32_t jbyte = (uint32_t)(min(j0 + RY, ny) - jlow) * (uint32_t)sy * (uint32_t)sizeof(S) +
                         (uint32_t)min(k0 * (int)sizeof(S) + (lane % CPR) * 16, (int)sy * (int)sizeof(S) - 16);
  const unsigned jlds = (unsigned)(uintptr_t)(__attribute__((address_space(3))) unsigned char*)&sJ[0][0][0];
  auto dma_row = [&](int i) {
    if (last && lane < 2 * CPR)
      step3_dma16(reinterpret_cast<const unsigned char*>((lane < CPR ? fe0 : fe2) + plane(i)) + jbyte,
                  jlds + (unsigned)(i & 3) * (2 * RB));
  };

  // The CPML faces and TF/SF jobs this wave's nodes can meet, one box test a
  // lane: bits 0..11 the H pass's jobs, 12..23 the E pass's, 24..29 the H
  // pass's faces, 30..35 the E pass's (a superset; the nodes test again).
  unsigned th_set, te_set, fh_set, fe_set, z_set;
  int job = 0;   // of lane q < 24: planes (from i0 - 1) of job q, its component, axis and row of sZ
  unsigned bits = 0;  // of a node: psi_a and psi_b of each H and E face, then the rows of sZ, that correct it
  {
    bool meet = false, meet_block = false, z_job = false;
    int comp = 0, p0 = 0, p1 = 0;
    if (lane < 24) {
      const int pass = lane < 12 ? 0 : 1, q = lane - 12 * pass;
      if (q < P.n_job[pass]) {
        const Step3Job<C>& J = P.job[pass][q];
        const bool planes = J.lo[0] < i1 && J.hi[0] > i0 - 1;
        meet_block = planes && J.lo[1] < j0 + RY && J.hi[1] > j0 - 1 && J.lo[2] < k0 + 64 && J.hi[2] > k0 - 1;
        meet = planes && (col ? J.lo[1] < j0 + RY && J.hi[1] > j0 && J.lo[2] < k0 && J.hi[2] > k0 - 1
                              : J.lo[1] <= j0 - 1 + w && J.hi[1] > j0 - 1 + w && J.lo[2] < k0 + 64 && J.hi[2] > k0);
        comp = J.comp;
        p0 = min(max(J.lo[0] - i0 + 1, 0), kStep3MaxChunk + 1);
        p1 = min(max(J.hi[0] - i0 + 1, 0), kStep3MaxChunk + 1);
        z_job = meet_block && J.axis == 2 && J.hi[2] == J.lo[2] + 1;
      }
    } else if (PML && lane < 36) {
      const int pass = lane < 30 ? 0 : 1, q = pass ? lane - 30 : lane - 24;
      if (q < P.n_face) {
        const Step3Face<C>& F = P.face[pass][q];
        const int ja = col ? j0 : j0 - 1 + w, jz = col ? j0 + RY - 1 : ja;
        const int ka = col ? k0 - 1 : k0, kz = col ? ka : k0 + 63;
        if (F.axis == 0)
          meet = F.c0 < i1 && F.c1 > i0 - 1 && jz >= F.a0 && ja <= F.a1 && kz >= F.b0 && ka <= F.b1;
        else if (F.axis == 1)
          meet = jz >= F.c0 && ja < F.c1 && kz >= F.a0 && ka <= F.a1;
        else
          meet = kz >= F.c0 && ka < F.c1 && jz >= F.b0 && ja <= F.b1;
      }
    }
    const uint64_t met = __ballot(meet);
    const bool e_wave = !col && w >= 1;
    th_set = (unsigned)met & 0xfffu;
    te_set = e_wave ? (unsigned)(met >> 12) & 0xfffu : 0u;
    fh_set = (unsigned)(met >> 24) & 0x3fu;
    fe_set = e_wave ? (unsigned)(met >> 30) & 0x3fu : 0u;
    // a z face's jobs are worked out before the march (sZ), the first
    // kStep3ZJobs of each pass that the block meets
    z_set = (unsigned)__ballot(z_job);
    const int first = lane < 12 ? 0 : 12;
    const int slot = __builtin_popcount(z_set >> first & ((1u << (max(lane - first, 0) & 31)) - 1u));
    z_set = (unsigned)__ballot(z_job && slot < kStep3ZJobs);
    job = p0 | p1 << 6 | comp << 12 | (z_job && slot < kStep3ZJobs ? slot : kStep3ZJobs) << 14;
    // The incident field near the block in LDS: the projections of its planes,
    // rows and columns (one node more on each side) and the two table rows of
    // this step over the projections they add up to.
    if (__ballot(meet_block)) {
      for (int q = threadIdx.x; q < 6 * kStep3Proj; q += blockDim.x) {
        const int d = q / (2 * kStep3Proj), half = q / kStep3Proj & 1, e = q % kStep3Proj;
        const int from = (d == 0 ? i0 : d == 1 ? j0 : k0) - 2;
        const int at = min(max(from + e - P.g[d] + half, 0), P.n_proj[d] - 1);
        sP[q] = half ? gp(P.proj_half[d])[at] : gp(P.proj_int[d])[at];
      }
      __syncthreads();
      const int end[3] = {i1 - i0 + 2, RY + 2, 66};  // last entry a node of the block takes
      C low = 0;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        const C* const pi = sP + 2 * d * kStep3Proj;
        low += min(min(pi[0], pi[end[d]]), min(pi[kStep3Proj], pi[kStep3Proj + end[d]]));
      }
      inc0 = max((int)low - 2, 0);
      for (int q = threadIdx.x; q < 2 * kStep3Inc; q += blockDim.x) {
        const bool is_h = q >= kStep3Inc;
        const int64_t n_aux = P.n_aux[is_h];
        const int64_t at = min((int64_t)inc0 + (is_h ? q - kStep3Inc : q), n_aux - 1);
        sI[is_h ? 1 : 0][is_h ? q - kStep3Inc : q] = gp(P.inc[is_h])[(int64_t)t * n_aux + at];
      }
    }
  }
  using False = std::integral_constant<bool, false>;
  using True = std::integral_constant<bool, true>;
  // The TF/SF correction of a job at a node (tfsf_inc's sum, from LDS).
  auto incident = [&](auto ise, const Step3Job<C>& J, int pi, int pj, int pk) __attribute__((always_inline)) {
    constexpr bool ISE = decltype(ise)::value;
    C proj = sP[J.at[0] + pi - i0] + sP[J.at[1] + pj - j0] + sP[J.at[2] + pk - k0];
    if (ISE) proj = proj - (C)0.5;
    const int index = (int)proj;  // 0 or more, and below the table's end
    const C weight = proj - (C)index;
    const int at = min(max(index - inc0, 0), kStep3Inc - 2);
    const C* const line = sI[ISE ? 1 : 0] + at;
    const C inc = J.tr * ((1 - weight) * line[0] + weight * line[1]);
    return inc * J.coef;
  };
  auto prepare = [&](auto ise) __attribute__((always_inline)) {
    constexpr bool ISE = decltype(ise)::value;
    for (unsigned m = z_set >> (ISE ? 12 : 0) & 0xfffu; m; m &= m - 1) {
      const int q = __builtin_ctz(m);
      const Step3Job<C> J = P.job[ISE][q];
      const int slot = __builtin_amdgcn_readlane(job, q + (ISE ? 12 : 0)) >> 14;
      const int pi = i0 - 1 + lane, pj = j0 - 1 + w;
      if (w <= RY && pi < i1 && pi >= J.lo[0] && pi < J.hi[0] && pj >= J.lo[1] && pj < J.hi[1])
        sZ[ISE][slot][w][lane] = incident(ise, J, pi, pj, J.lo[2]);
      if ((ISE ? own : hnode) && k == J.lo[2] && j >= J.lo[1] && j < J.hi[1])
        bits |= 1u << (4 * kMaxPml + (ISE ? kStep3ZJobs : 0) + slot);
    }
  };
  if (z_set) {
    __syncthreads();
    prepare(False{});
    prepare(True{});
  }
  // The TF/SF corrections of a node, in job order.  With 32-bit C the first
  // two x and y jobs of a plane (the two components of one face) are worked
  // out together, so that their chains of three LDS reads overlap; in 64 bits
  // that takes registers that are not there (10 spilled, 166 -> 190 us a step
  // of a 148^3 grid).
  constexpr bool PAIR = sizeof(C) < 8;
  const unsigned z_rows = PAIR ? (unsigned)__ballot(job >> 14 < kStep3ZJobs) : 0;
  auto inject = [&](auto ise, unsigned set, int i, bool mine, V3& v) __attribute__((always_inline)) {
    constexpr bool ISE = decltype(ise)::value;
    constexpr int L0 = ISE ? 12 : 0;
    const int at = i - i0 + 1;
    auto mine_of = [&](const Step3Job<C>& J) __attribute__((always_inline)) {
      return mine && j >= J.lo[1] && j < J.hi[1] && k >= J.lo[2] && k < J.hi[2];
    };
    int q1 = -1, q2 = -1;
    C add1 = 0, add2 = 0;
    bool take1 = false, take2 = false;
    if constexpr (PAIR) {
      set &= (unsigned)__ballot(at >= (job & 63) && at < (job >> 6 & 63)) >> L0;
      const unsigned sum = set & ~(z_rows >> L0);
      if (sum) {
        q1 = __builtin_ctz(sum);
        q2 = sum & (sum - 1) ? __builtin_ctz(sum & (sum - 1)) : q1;
        const Step3Job<C> J1 = P.job[ISE][q1], J2 = P.job[ISE][q2];
        add1 = incident(ise, J1, i, j, k);
        add2 = incident(ise, J2, i, j, k);
        take1 = mine_of(J1);
        take2 = mine_of(J2);
      }
    }
    for (unsigned m = set; m; m &= m - 1) {
      const int q = __builtin_ctz(m);
      const int u = __builtin_amdgcn_readlane(job, q + L0);
      const int slot = u >> 14, comp = u >> 12 & 3;
      if (!PAIR && (at < (u & 63) || at >= (u >> 6 & 63))) continue;
      C add = PAIR && q == q1 ? add1 : add2;
      bool take = PAIR && q == q1 ? take1 : take2;
      if (slot < kStep3ZJobs) {
        take = bits >> (4 * kMaxPml + (ISE ? kStep3ZJobs : 0) + slot) & 1;
        if (take) add = sZ[ISE][slot][row][at];
      } else if (!PAIR || (q != q1 && q != q2)) {
        const Step3Job<C> J = P.job[ISE][q];
        take = mine_of(J);
        if (take) add = incident(ise, J, i, j, k);
      }
      if (take) {
        if (comp == 0)
          v.x += add;
        else if (comp == 1)
          v.y += add;
        else
          v.z += add;
      }
    }
  };

  // CPML.  A node meets at most one face across each axis, and a wave one x
  // face a plane, one y face and one z face, or in a grid of few k two (the
  // host sees to that): x0, x1, y, z, z1 from bit 0 on, four bits each, 15
  // for none.  x1 takes over a plane before its first.
  const bool fh_any = PML && fh_set != 0, fe_any = PML && fe_set != 0;
  unsigned h_faces = 0xfffff, e_faces = 0xfffff;
  int h_turn = INT_MAX, e_turn = INT_MAX;
  Step3Psi<C> sh, se;
  // psi_a, psi_b of face q at plane i: the correction with the values held
  // from the plane before (HELD 1; 0: read here and not written; 2: read
  // here), the differences da, db and the sums added to xa, xb; then, HELD 1,
  // psi of plane i + 1.  FIRST: only psi of plane i.
  auto face = [&](auto ise, auto first, auto held, int q, int prof, int i, C& va, C& vb, const C* rowp, C da, C db, C& xa,
                  C& xb) __attribute__((always_inline)) {
    constexpr bool ISE = decltype(ise)::value, FIRST = decltype(first)::value;
    constexpr int HELD = decltype(held)::value;
    if (q == 15) return;
    step3_i16 u = *reinterpret_cast<const step3_i16*>(&P.face[ISE][q]);
    asm volatile("" : "+s"(u));  // one load, one wait
    const int lo = u[12], hi_a = u[13], hi_b = u[14];
    const unsigned f = bits >> (2 * kMaxPml * ISE + 2 * q);
    const uint32_t oa = step3_psi_offset<C>(i, j, k, lo, u[10], (uint32_t)u[8]);
    const uint32_t ob = step3_psi_offset<C>(i, j, k, lo, u[11], (uint32_t)u[9]);
    auto val = [&](int n, uint32_t o) __attribute__((always_inline)) {
      return gp(reinterpret_cast<C*>(((uint64_t)(uint32_t)u[n] | (uint64_t)(uint32_t)u[n + 1] << 32) + o));
    };
    // c_psi: a coefficient of the node's row, or (seldom) its array, whose load
    // is waited for where it is made and not where the two ways meet
    auto c_psi = [&](int t, const C* array, uint32_t o) __attribute__((always_inline)) {
      if (t != 0xff) return rowp[t];
      C c = *gp(reinterpret_cast<const C*>((uint64_t)array + o));
      asm volatile("" : "+v"(c));
      return c;
    };
    if (!FIRST && i >= lo && i < max(hi_a, hi_b)) {
      const bool on_a = (f & (i < hi_a ? 1u : 0u)) != 0, on_b = (f & (i < hi_b ? 2u : 0u)) != 0;
      const C ca = sPr[ISE][0][prof], cb = sPr[ISE][1][prof];
      const bool write = HELD != 0 && (ISE || (!col && w >= 1));
      if (on_a) {
        if (HELD != 1) va = *val(0, oa);
        va = cb * va + ca * da;
        if (write) *val(4, oa) = va;
        xa += c_psi(u[15] & 0xff, P.face[ISE][q].cpa, oa) * va;
      }
      if (on_b) {
        if (HELD != 1) vb = *val(2, ob);
        vb = cb * vb + ca * db;
        if (write) *val(6, ob) = vb;
        xb += c_psi(u[15] >> 8, P.face[ISE][q].cpb, ob) * vb;
      }
    }
    if constexpr (FIRST || HELD == 1) {
      const int n = FIRST ? i : i + 1;
      if ((f & (n >= lo && n < hi_a ? 1u : 0u)) != 0) va = *val(0, oa + (FIRST ? 0u : (uint32_t)u[8]));
      if ((f & (n >= lo && n < hi_b ? 2u : 0u)) != 0) vb = *val(2, ob + (FIRST ? 0u : (uint32_t)u[9]));
    }
  };
  // The CPML corrections of a node, in registration order: x, y, z faces.
  // d0..d2: the curl differences along x, y, z that psi_a and psi_b of a face
  // across that axis take.
  auto correct = [&](auto ise, auto first, auto held, unsigned set, int turn, int i, Step3Psi<C>& s, const C* rowp, C d0a,
                     C d0b, C d1a, C d1b, C d2a, C d2b, V3& v) __attribute__((always_inline)) {
    constexpr bool FIRST = decltype(first)::value;
    constexpr int HELD = decltype(held)::value;
    const int n = FIRST || HELD == 0 ? i : i + 1;
    using In = std::integral_constant<int, HELD == 0 ? 0 : 2>;
    const int qx = (n >= turn ? set >> 4 : set) & 15;
    if constexpr (sizeof(C) < 8)
      face(ise, first, held, qx, i - i0 + 1, i, s.a[2], s.b[2], rowp, d0a, d0b, v.y, v.z);
    else if constexpr (!FIRST) {  // no registers left to read ahead into, and few planes
      C va, vb;
      face(ise, first, In{}, qx, i - i0 + 1, i, va, vb, rowp, d0a, d0b, v.y, v.z);
    }
    face(ise, first, held, set >> 8 & 15, kProfRow + row, i, s.a[0], s.b[0], rowp, d1a, d1b, v.z, v.x);
    face(ise, first, held, set >> 12 & 15, kProfCol + k - k0 + 1, i, s.a[1], s.b[1], rowp, d2a, d2b, v.x, v.y);
    if constexpr (!FIRST) {
      C va, vb;
      face(ise, first, In{}, set >> 16 & 15, kProfCol + k - k0 + 1, i, va, vb, rowp,
           d2a, d2b, v.x, v.y);
    }
  };
  using Skip = std::integral_constant<int, 0>;
  using Held = std::integral_constant<int, 1>;
  if constexpr (PML) {
    auto mark = [&](auto ise, unsigned set, bool mine, unsigned& slots, int& turn) __attribute__((always_inline)) {
      constexpr bool ISE = decltype(ise)::value;
      for (unsigned m = set; m; m &= m - 1) {
        const int q = __builtin_ctz(m);
        const Step3Face<C>& F = P.face[ISE][q];
        bool in_a, in_b;  // at a plane that the face covers
        step3_in<ISE, C>(F, F.lo, j, k, in_a, in_b);
        bits |= (mine && in_a ? 1u : 0u) << (2 * kMaxPml * ISE + 2 * q) | (mine && in_b ? 2u : 0u) << (2 * kMaxPml * ISE + 2 * q);
        int at = F.axis == 0 ? 0 : F.axis == 1 ? 8 : 12;
        if (F.axis != 1 && (slots >> at & 15) != 15) {
          at += 4;
          if (F.axis == 0) turn = F.lo;
        }
        slots = (slots & ~(15u << at)) | (unsigned)q << at;
      }
    };
    mark(False{}, fh_set, hnode, h_faces, h_turn);
    mark(True{}, fe_set, own, e_faces, e_turn);
    // the profiles of the faces that the block meets
    for (int n = 0; n < 2 * P.n_face; ++n) {
      const int pass = n >= P.n_face;
      const Step3Face<C>& F = P.face[pass][pass ? n - P.n_face : n];
      const int ax = F.axis, first = (ax == 0 ? i0 : ax == 1 ? j0 : k0) - 1, len = ax == 0 ? i1 - i0 + 1 : ax == 1 ? RY + 2 : 65;
      const int c = first + (int)threadIdx.x;
      if (F.c0 < first + len && F.c1 > first && (int)threadIdx.x < len && c >= F.c0 && c < F.c1) {
        const int e = (ax == 0 ? 0 : ax == 1 ? kProfRow : kProfCol) + (int)threadIdx.x;
        sPr[pass][0][e] = gp(F.ca)[c + F.off];
        sPr[pass][1][e] = gp(F.cb)[c + F.off];
      }
    }
  }

  V3 X0, X1, Y;
  int dn;
  dma_row(i0);
  dma_row(i0 + 1);
  load_e(X0, i0);
  load_h(Y, dn, i0);
  load_e(X1, i0 + 1);
  __syncthreads();  // the table is in LDS

  // H_y and H_z of the plane before the chunk, for its first E plane
  C hym = 0, hzm = 0;
  if (!col && w >= 1 && i0 > 0) {  // wave-uniform: inject reads other lanes
    const int i = i0 - 1;
    const int64_t b = plane(i), bn = plane(i0);
    const int64_t o_j = j < ny ? sy : 0;
    const int o_k = k < nz ? 1 : 0;
    V3 e, n, h;
    int d;
    load_e(e, i);
    load_h(h, d, i);
    n.y = ld(fe1 + bn, inv_e);
    n.z = ld(fe2 + bn, inv_e);
    const C xk = Store<S>::ld(fe0 + b, vo + o_k, inv_e), yk = Store<S>::ld(fe1 + b, vo + o_k, inv_e);
    const C xj = Store<S>::ld(fe0 + b + o_j, vo, inv_e), zj = Store<S>::ld(fe2 + b + o_j, vo, inv_e);
    const C* r = tab + 18 * d + 9;
    if (hmain) {
      h.y = r[3] * h.y + r[4] * (n.z - e.z) + r[5] * (xk - e.x);
      h.z = r[6] * h.z + r[7] * (xj - e.x) + r[8] * (n.y - e.y);
    }
    if constexpr (PML)
      if (fh_any)
        correct(False{}, False{}, Skip{}, h_faces, h_turn, i, sh, r, n.z - e.z, n.y - e.y, xj - e.x, zj - e.z, yk - e.y, xk - e.x, h);
    h.y = step3_rt<S>(h.y, s_h, inv_h);
    h.z = step3_rt<S>(h.z, s_h, inv_h);
    if (th_set) {
      inject(False{}, th_set, i, own, h);
      h.y = step3_rt<S>(h.y, s_h, inv_h);
      h.z = step3_rt<S>(h.z, s_h, inv_h);
    }
    hym = h.y;
    hzm = h.z;
  }
  if constexpr (PML) {
    V3 none{0, 0, 0};
    if (fh_any) correct(False{}, True{}, Skip{}, h_faces, h_turn, i0, sh, tab, 0, 0, 0, 0, 0, 0, none);
    if (fe_any) correct(True{}, True{}, Skip{}, e_faces, e_turn, i0, se, tab, 0, 0, 0, 0, 0, 0, none);
  }

  auto stage = [&](int p, const V3& e) {
    if (!col) {
      sE[p][0][w][lane] = e.x;
      sE[p][1][w][lane] = e.z;
      if (lane == 0) {
        cE[p][w][0] = e.x;
        cE[p][w][1] = e.y;
      }
    } else if (lane >= 32 && lane <= 32 + RY) {
      cF[p][row][0] = e.x;
      cF[p][row][1] = e.y;
    }
  };
  stage(i0 & 1, X0);
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the prologue's rows are in LDS
  __syncthreads();

  // Plane i: XE holds E(i), XN E(i + 1), YH H(i) and its row id; their
  // registers take the loads of planes i + 2 and i + 1.
  auto body = [&](int i, V3& XE, const V3& XN, V3& YH, int& YD) __attribute__((always_inline)) {
    const int pa = i & 1, pb = pa ^ 1;
    const V3 e = XE;
    dma_row(i + 2);
    load_e(XE, i + 2);
    C xj, zj, xk, yk;
    if (!col) {
      if (last) {
        xj = step3_lds<S>(sJ[i & 3][0], lane, inv_e);
        zj = step3_lds<S>(sJ[i & 3][1], lane, inv_e);
      } else {
        xj = sE[pa][0][w + 1][lane];
        zj = sE[pa][1][w + 1][lane];
      }
      xk = step3_shl(e.x);
      yk = step3_shl(e.y);
      const C fx = cF[pa][w][0], fy = cF[pa][w][1];
      if (lane == 63) {
        xk = fx;
        yk = fy;
      }
    } else {
      const int r = min(row, RY);
      xj = step3_shl(e.x);
      zj = step3_shl(e.z);
      xk = cE[pa][r][0];
      yk = cE[pa][r][1];
    }
    const C* const r = tab + 18 * YD;
    const C* const rh = r + 9;
    V3 h = YH;
    {
      const V3 u{rh[0] * h.x + rh[1] * (yk - e.y) + rh[2] * (zj - e.z),
                 rh[3] * h.y + rh[4] * (XN.z - e.z) + rh[5] * (xk - e.x),
                 rh[6] * h.z + rh[7] * (xj - e.x) + rh[8] * (XN.y - e.y)};
      if (hmain && i < nx) h = u;
    }
    const int de = YD;
    load_h(YH, YD, i + 1);
    if constexpr (PML)
      if (fh_any)
        correct(False{}, False{}, Held{}, h_faces, h_turn, i, sh, rh, XN.z - e.z, XN.y - e.y, xj - e.x, zj - e.z, yk - e.y, xk - e.x, h);
    if constexpr (sizeof(S) < 4) h = V3{step3_rt<S>(h.x, s_h, inv_h), step3_rt<S>(h.y, s_h, inv_h), step3_rt<S>(h.z, s_h, inv_h)};
    if (th_set) {
      inject(False{}, th_set, i, hnode, h);
      if constexpr (sizeof(S) < 4)
        h = V3{step3_rt<S>(h.x, s_h, inv_h), step3_rt<S>(h.y, s_h, inv_h), step3_rt<S>(h.z, s_h, inv_h)};
    }
    if (!col) {
      sH[pa][0][w][lane] = h.x;
      sH[pa][1][w][lane] = h.z;
    } else if (lane < RY) {
      cH[pa][lane + 1][0] = h.x;
      cH[pa][lane + 1][1] = h.y;
    }
    stage(pb, XN);
    __syncthreads();
    V3 v = e;
    if (!col && w >= 1) {
      C hxk = step3_shr(h.x), hyk = step3_shr(h.y);
      const C gx = cH[pa][w][0], gy = cH[pa][w][1];
      if (lane == 0) {
        hxk = gx;
        hyk = gy;
      }
      const C hxj = sH[pa][0][w - 1][lane], hzj = sH[pa][1][w - 1][lane];
      const C* const re = tab + 18 * de;
      bool up = i < nx;
      if (P.ade) up = up && !((P.dmask >> de) & 1);
      const V3 u{re[0] * e.x + re[1] * (h.y - hyk) + re[2] * (h.z - hzj),
                 re[3] * e.y + re[4] * (h.z - hzm) + re[5] * (h.x - hxk),
                 re[6] * e.z + re[7] * (h.x - hxj) + re[8] * (h.y - hym)};
      v = V3{mx && up ? u.x : e.x, my && up && i > 0 ? u.y : e.y, mz && up && i > 0 ? u.z : e.z};
      if constexpr (PML)
        if (fe_any)
          correct(True{}, False{}, Held{}, e_faces, e_turn, i, se, re, h.z - hzm, h.y - hym, h.x - hxj, h.z - hzj, h.y - hyk, h.x - hxk, v);
      if (te_set) {
        if constexpr (sizeof(S) < 4)
          v = V3{step3_rt<S>(v.x, s_e, inv_e), step3_rt<S>(v.y, s_e, inv_e), step3_rt<S>(v.z, s_e, inv_e)};
        inject(True{}, te_set, i, own, v);
      }
      hym = h.y;
      hzm = h.z;
    }
    const int64_t b = plane(i);
    st(P.ho[0] + b, h.x, s_h);
    st(P.ho[1] + b, h.y, s_h);
    st(P.ho[2] + b, h.z, s_h);
    st(P.eo[0] + b, v.x, s_e);
    st(P.eo[1] + b, v.y, s_e);
    st(P.eo[2] + b, v.z, s_e);
  };
  // registers by turns, without copies at the loop's end (which would wait for
  // the loads in flight)
  for (int i = i0;;) {
    body(i, X0, X1, Y, dn);
    if (++i >= i1) break;
    body(i, X1, X0, Y, dn);
    if (++i >= i1) break;
  }
}
