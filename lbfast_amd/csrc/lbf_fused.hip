// lbf_fused.hip -- fused stream+collide from moments for gfx950.
//
// Replaces fused_LB_kernel (lb_cuda_fused_module.f90:426-750) and, in the
// "inline" variant used by lbf_step, also the moments stage
// (lb_cuda_moments_module.f90:19-341), the phase-field update
// (lb_cuda_update_phi_module.f90:19-104) and the near-wall regularised
// bounce-back (lb_cuda_boundary_module.f90:19-216), so that one launch reads
// the state once and writes the new state once.
//
// Arithmetic.  The reference rebuilds 27 post-collision populations as
//   f*_l = feq_l + (1-omega) fneq_l + F_l/2
// with feq/fneq the second-order terms plus, under HIGHORDER, Minv_mrt(k,l)
// times the monomials E_k and polynomials N_k (k = 10..26, fused:641-702).
// Every term is a Hermite coefficient times Minv_mrt(k,l) = w_l H_k(c_l)/b_k,
// and for D3Q27 the basis is the tensor product of the 1-D basis
// {1, c, c^2-1/3} (vars_module.f90:522-664), so
//   f*_{pqr} = sum_{abc} g_a(p) g_b(q) g_c(r) A_{abc},
//   A_0 = P, A_i = u_i + a_i/2, A_ij = u_i u_j + (1-omega) Pn_ij + (u_i a_j + u_j a_i)/2,
//   A_k = E_k + (1-omega) N_k (k >= 10)
// (a = force/rho_phi; Guo forcing of fused:705-706 is exactly the order-1/2
// Hermite part).  D3Q19 is not a tensor product; its 19 populations are built
// directly from the order <= 2 coefficients.
//
// Streaming + moments.  out_m(x) = sum_l M_ml f*_l(x - c_l) separates by
// axis too, and the axes' operators (reconstruct over a, shift, contract with
// 1, c, c^2 - 1/3) commute, so they run axis by axis on the coefficients and
// the populations as a whole are never formed.  A block owns a 64-wide x
// segment (one wave per y row, lanes = x) of TY output rows plus one halo row
// on each side, and marches z.  For each source plane it:
//   x: reconstructs the 9 lines (b, c), shifts the p = +-1 values one lane
//      (DPP) and contracts over p; the two x-halo nodes of every row are
//      computed by one extra wave, which forms only the side it hands over
//      (through LDS);
//   y: reconstructs the 9 lines (d, c), exchanges the q = +-1 values with the
//      neighbouring rows through LDS (halo rows form one side only) and
//      contracts over q;
//   z: reconstructs the 6 lines (d, e) that are left and adds r = -1/0/+1 into
//      15 per-lane sums in flight; the lowest plane is complete and is stored.
// Every node of the block's (x,y) footprint is collided once per plane; the
// recomputation is only the two y-halo rows, the x-halo wave and the two
// z-halo planes of the march.
//
// Phase-field inputs (two-component, inline variant).  Without internal
// obstacles and with float phase-field storage the block also streams a phi
// tile with a 2-node halo and forms grad phi and lap phi of every collided
// node from the separable partial sums of three planes (part3 / grad_lap,
// the arithmetic of the prep kernel), so the prep only stores div theta.
// With obstacles, PHI_int_boundary (lb_cuda_boundary_module.f90:218-459)
// rewrites phi on solid nodes after compute_norm and before the moments
// stage, so the gradients come from the prep's output instead.
//
// What bounds it: arithmetic and scalar issue, and HBM where the domain is
// large.  Measured at 512^3 before and after the axis-by-axis order (27% fewer
// vector instructions a launch), the 16-byte row transfers, the compiled-in
// switches (std_switches), one buffer resource per set (scalar instructions
// of the plane loop 661 -> 367) and streaming stores (stream_stores): two
// components FP32 3.81 -> 3.18 ms (15.0 GB of compulsory state at 4.7 TB/s, as
// much as a plain copy moves; 19 GB with the excess reads), FP16S 3.15 -> 2.57
// ms, one component 2.76 -> 2.20 ms.
// Registers decide the variants: a spill inside the plane loop makes the compiler
// wait for every transfer in flight (FP16S 2.57 -> 3.70 ms, 32 bytes of spills).
// One remains, in the general D3Q27 HIGHORDER two-component variant of 32 bits
// with 13 rows: a column offset of the phi tile, reloaded in tiles at the x faces.
// Forming it each plane instead was 1-3% slower (scalar spills 22 -> 29 and more).
//
// Periodicity: indices wrap in-kernel (the reference's intpbc halo copies,
// mpi_module.f90:2820-2918).  isfluid and the solid neighbours of near-wall
// nodes come as one word per node of a copy with the reference's 1-node halo
// (periodic image or 1, LBFAST.f90:258-328).
#include "lbf_common.h"
#include "lbf_kernels.h"
#include "lbf_physics.h"

namespace lbf {

// The kernels of one storage precision; each is compiled in a translation
// unit of its own (LBF_FUSED_PREC), the dispatch in one without it.
template <int PREC>
hipError_t fused_prec(const FusedArgs& a, bool inline_moments, hipStream_t s);
template <int PREC>
hipError_t fused_batch_prec(const FusedBatchEntry* tab, int ndom, int total, int lat, bool ho, bool two, bool std, int ty,
                            hipStream_t s);
template <int TY>
__host__ __device__ inline int fused_tiles(const FusedArgs& a) {
  return ((a.dp.nx + 63) / 64) * ((a.dp.ny + TY - 1) / TY) * ((a.dp.nz + a.tz - 1) / a.tz);
}

#ifdef LBF_FUSED_PREC

// Whole-wave lane shifts through DPP (wave_shr:1 / wave_shl:1, a VALU
// operand modifier, no LDS round trip).  With bound_ctrl off, the lane whose
// source lies outside the wave (lane 0 for shr, lane 63 for shl) keeps `fill`.
__device__ __forceinline__ int dpp_shr1(int fill, int v) { return __builtin_amdgcn_update_dpp(fill, v, 0x138, 0xF, 0xF, false); }
__device__ __forceinline__ int dpp_shl1(int fill, int v) { return __builtin_amdgcn_update_dpp(fill, v, 0x130, 0xF, 0xF, false); }
__device__ __forceinline__ float shift_from_lower(float v, float fill) {  // lane L receives lane L-1
  return __builtin_bit_cast(float, dpp_shr1(__builtin_bit_cast(int, fill), __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ float shift_from_upper(float v, float fill) {  // lane L receives lane L+1
  return __builtin_bit_cast(float, dpp_shl1(__builtin_bit_cast(int, fill), __builtin_bit_cast(int, v)));
}
__device__ __forceinline__ double shift_from_lower(double v, double fill) {
  const int2 t = __builtin_bit_cast(int2, v), u = __builtin_bit_cast(int2, fill);
  return __builtin_bit_cast(double, make_int2(dpp_shr1(u.x, t.x), dpp_shr1(u.y, t.y)));
}
__device__ __forceinline__ double shift_from_upper(double v, double fill) {
  const int2 t = __builtin_bit_cast(int2, v), u = __builtin_bit_cast(int2, fill);
  return __builtin_bit_cast(double, make_int2(dpp_shl1(u.x, t.x), dpp_shl1(u.y, t.y)));
}
// Encoded inputs of one node for one source plane.
template <int PREC>
struct RawNode {
  typename Codec<PREC>::T m[10];
  typename Codec<PREC>::T uo[3];
  typename Aux<PREC>::T phi;
  typename Aux<PREC>::T g[5];  // inline: grad phi (3), lap phi, div theta n; stage path: forces (3)
};

// A wave's LDS slots of the prefetched inputs, in bytes from its base: 64
// values of each moment, of u_old (U), of the g set (G: the prep's output or the
// forces; with the gradient formed inside, GI, only div theta) and of phi
// (which comes from the block's phi tile under GI).
template <int PREC, bool TWO, bool INLINE, bool GI>
struct Slots {
  static constexpr int SB = 64 * sizeof(typename Codec<PREC>::T), SA = 64 * sizeof(typename Aux<PREC>::T);
  static constexpr int NU = INLINE && TWO ? 3 : 0, NG = !INLINE ? 3 : !TWO ? 0 : GI ? 1 : 5, NP = TWO && !GI ? 1 : 0;
  static constexpr int U = 10 * SB, G = U + NU * SB, PHI = G + NG * SA, BYTES = (PHI + NP * SA + 255) / 256 * 256;
};

// Per-lane byte offsets of one node inside a z plane of each input buffer,
// and the planes' sizes in bytes: the 10-field moment set, the 3-field
// u_old set, the g set (prep output, 5 fields, or forces, 3 fields) and the
// single phase field.  Field sets are row-interleaved, so a set's field f is
// the same lane offset from a plane base shifted by f*sx elements.
struct FOff {
  uint32_t m, u, g, p;
  uint32_t pm, pu, pg, pp;
  // where the lane's transfers of dma_raw start in the moment, u_old and g sets
  // and in phi.  Row waves (rows != 0, wave-uniform) fetch whole field rows, 16
  // bytes a lane (the lane's node + row_off); the x-halo wave a dword a lane:
  // the aligned dword of its node, or of 64-bit values one of its node's two
  int rows;
  uint32_t lm, lu, lg, lp;
};

// A wave's 64-node row segments of a set move two (64-bit values), four (32) or
// eight (16) fields to a transfer: lane l fetches 16 bytes of field l / G at
// element E (l % G), G lanes to a 64-value row.  Lanes past a short row read
// on into the row's end and the next field; those nodes are never used, and
// every buffer is padded past its last plane.  The transfers were bound by
// their number, not their bytes: with a dword a lane the row waves of a block
// issued 14 a plane (one per field), with 16 bytes 5.
template <class V>
__device__ __forceinline__ uint32_t row_off(int sx) {
  constexpr uint32_t E = 16 / sizeof(V), G = 64 / E;
  const uint32_t l = threadIdx.x & 63;
  return ((l / G) * (uint32_t)sx + (l % G) * E - l) * (uint32_t)sizeof(V);
}
// the NF fields of a set at one plane into the wave's LDS from byte OFF on
template <class V, uint32_t OFF, int NF, int W = 0>
__device__ __forceinline__ void dma_rows(const V* plane0, uint32_t voff, int sx, uint32_t lds0) {
  constexpr int G = 64 * sizeof(V) / 16, PER = 64 / G;  // lanes per row, rows per transfer
  const Rsrc r = mkrsrc(plane0, 0xFFFFFFFFu);
  const uint32_t soff = (uint32_t)(W * PER * sizeof(V)) * (uint32_t)sx;
  if constexpr (NF >= (W + 1) * PER) {
    dma_quad<OFF + 1024u * W>(r, voff, soff, lds0);
    if constexpr (NF > (W + 1) * PER) dma_rows<V, OFF, NF, W + 1>(plane0, voff, sx, lds0);
  } else {
    if ((int)(threadIdx.x & 63) < (NF - W * PER) * G) dma_quad<OFF + 1024u * W>(r, voff, soff, lds0);
  }
}
// the x-halo wave's: at most 32 nodes, a slot of 64 values to a field
template <class V, uint32_t OFF, int NF, int F = 0>
__device__ __forceinline__ void dma_nodes(Rsrc r, uint32_t voff, int sx, uint32_t lds0) {
  dma_dword<OFF + 64u * (uint32_t)sizeof(V) * F>(r, voff, lds0, (uint32_t)(F * sizeof(V)) * (uint32_t)sx);
  if constexpr (F + 1 < NF) dma_nodes<V, OFF, NF, F + 1>(r, voff, sx, lds0);
}

// Direct loads of one plane's inputs (used when the inputs are not prefetched).
// fs = sx, the field stride of the sets.
template <int PREC, bool TWO, bool INLINE>
__device__ __forceinline__ void load_raw(RawNode<PREC>& r, const FusedArgs& a, int zw, size_t fs, const FOff& o) {
  typedef typename Codec<PREC>::T T;
  typedef typename Aux<PREC>::T TA;
  constexpr int GF = INLINE ? 5 : 3;
  const DevParams& dp = a.dp;
  const size_t rows = (size_t)zw * dp.ny;
  const T* S = (const T*)a.min + rows * 10 * fs;
#pragma unroll
  for (int f = 0; f < 10; ++f) r.m[f] = fld(S, fs, f, o.pm, o.m);
  if constexpr (TWO) r.phi = fld((const TA*)a.phin + rows * dp.nx, fs, 0, o.pp, o.p);
  if constexpr (!INLINE) {
    const TA* fr = (const TA*)a.frc + rows * GF * fs;
#pragma unroll
    for (int f = 0; f < 3; ++f) r.g[f] = fld(fr, fs, f, o.pg, o.g);
  } else if constexpr (TWO) {
    const TA* pr = (const TA*)a.pre + rows * GF * fs;
#pragma unroll
    for (int f = 0; f < 5; ++f) r.g[f] = fld(pr, fs, f, o.pg, o.g);
    if (dp.dens) {
      const T* uo = (const T*)a.uin + rows * 3 * fs;
#pragma unroll
      for (int f = 0; f < 3; ++f) r.uo[f] = fld(uo, fs, f, o.pu, o.u);
    }
  }
}

// LDS-DMA prefetch of one plane's inputs into this wave's slots.  The x-halo
// wave moves the aligned dword that holds a 16-bit element (the half is picked
// when read back; sx is even, so every 16-bit field row starts on a dword and
// the u_old offsets share that parity).
template <int PREC, bool TWO, bool INLINE, bool GI>
__device__ __forceinline__ void dma_raw(const FusedArgs& a, int zw, const FOff& o, bool dens, uint32_t lds0) {
  typedef Slots<PREC, TWO, INLINE, GI> SL;
  typedef typename Codec<PREC>::T T;
  typedef typename Aux<PREC>::T TA;
  const int sx = a.dp.sx;
  const T* S = plane_at((const T*)a.min, o.pm, zw);
  const T* uo = plane_at((const T*)a.uin, o.pu, zw);
  const TA* g = plane_at((const TA*)(INLINE ? a.pre : a.frc), o.pg, zw);
  if constexpr (GI) g += 4 * (size_t)sx;
  const TA* ph = plane_at((const TA*)a.phin, o.pp, zw);
  // slot offsets are immediates: only the wave's LDS base stays live
  if constexpr (GI) dma_dword<(uint32_t)SL::G>(mkrsrc(g, o.pg), o.g, lds0);
  if (o.rows) {
    dma_rows<T, 0u, 10>(S, o.lm, sx, lds0);
    if constexpr (!GI && SL::NG > 0) dma_rows<TA, (uint32_t)SL::G, SL::NG>(g, o.lg, sx, lds0);
    if constexpr (SL::NP > 0) dma_rows<TA, (uint32_t)SL::PHI, 1>(ph, o.lp, sx, lds0);
    if constexpr (SL::NU > 0) {
      if (dens) dma_rows<T, (uint32_t)SL::U, 3>(uo, o.lu, sx, lds0);
    }
  } else {
    const int l = threadIdx.x & 63;
    if (l < (sizeof(T) == 8 ? 64 : 32)) {
      dma_nodes<T, 0u, 10>(mkrsrc(S, o.pm), o.lm, sx, lds0);
      if constexpr (SL::NU > 0) {
        if (dens) dma_nodes<T, (uint32_t)SL::U, 3>(mkrsrc(uo, o.pu), o.lu, sx, lds0);
      }
    }
    if (l < (sizeof(TA) == 8 ? 64 : 32)) {
      if constexpr (!GI && SL::NG > 0) dma_nodes<TA, (uint32_t)SL::G, SL::NG>(mkrsrc(g, o.pg), o.lg, sx, lds0);
      if constexpr (SL::NP > 0) dma_nodes<TA, (uint32_t)SL::PHI, 1>(mkrsrc(ph, o.pp), o.lp, sx, lds0);
    }
  }
}

template <int PREC, bool TWO, bool INLINE, bool GI>
__device__ __forceinline__ void lds_raw(RawNode<PREC>& r, const char* slot, int lane, bool dens, uint32_t bT, bool rows) {
  typedef Slots<PREC, TWO, INLINE, GI> SL;
  typedef typename Codec<PREC>::T T;
  typedef typename Aux<PREC>::T TA;
  // a 16-bit element of the x-halo wave is half (bT & 2) of its lane's dword
  const char* at = slot + (sizeof(T) == 2 && !rows ? (uint32_t)lane * 4u + (bT & 2u) : (uint32_t)lane * (uint32_t)sizeof(T));
  const char* aa = slot + (uint32_t)lane * (uint32_t)sizeof(TA);
#pragma unroll
  for (int f = 0; f < 10; ++f) r.m[f] = *(const T*)(at + f * SL::SB);
  if (SL::NU > 0 && dens) {
#pragma unroll
    for (int f = 0; f < 3; ++f) r.uo[f] = *(const T*)(at + SL::U + f * SL::SB);
  }
  if constexpr (SL::NP > 0) r.phi = *(const TA*)(aa + SL::PHI);
  if constexpr (GI) {
    r.g[4] = *(const TA*)(aa + SL::G);
  } else {
#pragma unroll
    for (int f = 0; f < SL::NG; ++f) r.g[f] = *(const TA*)(aa + SL::G + f * SL::SA);
  }
}

// ---------------------------------------------------------------------------
// PF: the next plane's inputs stream into LDS (dma_raw) while the current
// plane is collided and streamed.  All stores of an iteration are issued
// before that DMA, so the wait at the top of the next iteration (which the
// shared load/store counter makes a wait for everything) finds the older
// stores long done.  The completed output plane is therefore stored at the
// top of the following iteration.
// Prefetching instances.  In 64-bit arithmetic the completed plane, held for one
// iteration, spills beside the rest unless a lane has 256 registers: blocks of 5
// rows (8 waves), whose slots also fit the 160 KB beside the y exchange.
template <int PREC, int TY>
constexpr bool fused_prefetch() { return sizeof(typename Codec<PREC>::R) == 4 || TY == 5; }

// One block: tile `tile` (x fastest, then y, then z chunks) of the domain `a`.
// OB: the domain has internal obstacles (node words, solid nodes, the
// near-wall closures); without them that code is compiled out.
// A node next to the wall of a non-periodic axis (coordinate 1 or n-2): a
// superset of the first fluid layers of the open faces.
__device__ __forceinline__ bool open_layer(const DevParams& dp, int x, int y, int z) {
  return (!dp.pbc[0] && (x == 1 || x == dp.nx - 2)) || (!dp.pbc[1] && (y == 1 || y == dp.ny - 2)) ||
         (!dp.pbc[2] && (z == 1 || z == dp.nz - 2));
}

// One population f of velocity (p, q, r) added to the ten closure moments.
template <class R>
__device__ __forceinline__ void add_closure(R (&l)[10], int p, int q, int r, R f) {
  const R cssq = (R)(1.0 / 3.0);
  l[0] += f;
  l[1] += f * (R)p; l[2] += f * (R)q; l[3] += f * (R)r;
  l[4] += f * ((R)(p * p) - cssq); l[5] += f * ((R)(q * q) - cssq); l[6] += f * ((R)(r * r) - cssq);
  l[7] += f * (R)(p * q); l[8] += f * (R)(p * r); l[9] += f * (R)(q * r);
}
// The closure moments of a node of the source plane, put into the z sums of
// its own plane: line k of zn (which becomes za, or part of zb) takes what
// enters that line's difference or only sum, lbs[0..2] what its r = 0 value
// still needs, and lbs[3] the rest of Pi_zz.
template <class R>
__device__ __forceinline__ void closure_to_z(const R (&l)[10], R (&zn)[6], R (&lbs)[4]) {
  zn[0] += l[3]; lbs[0] = l[0] - l[3];
  zn[1] += l[9]; lbs[1] = l[2] - l[9];
  zn[2] += l[8]; lbs[2] = l[1] - l[8];
  zn[3] += (R)3 * l[4]; zn[4] += (R)3 * l[5]; zn[5] += l[7];
  lbs[3] = l[6] - ((R)(2.0 / 3.0) * l[3] - (R)(1.0 / 3.0) * lbs[0]);
}
// One of the three values of recon3, side p = -1, 0 or +1 (uniform over the
// wave), with the same roundings.
template <class R>
__device__ __forceinline__ R recon_one(R A0, R A1, R A2, int p, bool h1, bool h2) {
  const R t = recon_side(A0, A2, h2);
  return p == 0 ? A0 - (R)2 * t : (h1 ? t + (R)p * A1 : t);
}
// Population (p, q, r) from the Hermite coefficients of hermite27.
template <bool HO, class R>
__device__ __forceinline__ R population27(const R (&A)[27], int p, int q, int r) {
  R C[3];
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    R B[3];
#pragma unroll
    for (int b = 0; b < 3; ++b)
      B[b] = HO || b + c <= 2 ? recon_one(A[3 * b + 9 * c], A[1 + 3 * b + 9 * c], A[2 + 3 * b + 9 * c], p,
                                          HO || b + c <= 1, HO || b + c == 0)
                              : (R)0;
    C[c] = recon_one(B[0], B[1], B[2], q, HO || c <= 1, HO || c == 0);
  }
  return recon_one(C[0], C[1], C[2], r, true, true);
}

// OPEN: open faces (with OB and the inline moments stage only): the kernel
// also hands over the post-moments state of the wall-adjacent nodes
template <int LAT, bool HO, int PREC, bool TWO, bool INLINE, int TY, bool OB, bool STD, bool OPEN = false>
__device__ __forceinline__ void fused_body(const FusedArgs& a, int tile) {
  typedef Codec<PREC> C;
  typedef typename C::R R;
  typedef typename C::T T;
  typedef typename Aux<PREC>::T TA;
  constexpr int NW = TY + 2;  // row waves (TY output rows + 2 halo rows)
  // GI: grad phi and lap phi formed here from a phi tile
  constexpr bool GI = TWO && INLINE && fused_grad_inline(PREC, OB);
  typedef Slots<PREC, TWO, INLINE, GI> SL;
  constexpr bool PF = fused_prefetch<PREC, TY>();
  // GI phi tile: rows y0-2 .. y0+TY+1 (tile row r holds y0-2+r), columns
  // x0-2 .. x0+65 (column c holds x0-2+c), both wrapped; a ring of four z
  // planes streamed by LDS DMA three planes ahead of the plane collided
  constexpr int GR = TY + 4, GC = 68;

  __shared__ R sUP[NW][9][64];
  __shared__ R sDN[NW][9][64];
  __shared__ R sHX[NW][2][9];
  __shared__ __align__(16) char sPF[PF ? NW + 1 : 1][PF ? SL::BYTES : 16];
  __shared__ float sPH[GI ? 4 : 1][GI ? GR : 1][GI ? GC : 1];

  const DevParams& dp = a.dp;
  const Phys<R>& ph = dp.ph<R>();
  const bool dens = STD ? TWO : dp.dens != 0;
  const int nx = dp.nx, ny = dp.ny, nz = dp.nz;
  const size_t nxny = (size_t)nx * ny;
  const bool bb = OB && dp.bb != 0;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int ntx = (nx + 63) / 64, nty = (ny + TY - 1) / TY;
  const int tx = tile % ntx, ty = (tile / ntx) % nty, tzi = tile / (ntx * nty);
  const int x0 = tx * 64;
  const int XW = min(64, nx - x0);
  const int y0 = ty * TY;
  const int z0 = tzi * a.tz;
  const int zend = min(z0 + a.tz, nz);
  const bool halo_wave = (wave == NW);

  int w, xs, side = 0;
  bool active = true;
  if (!halo_wave) {
    w = wave;
    xs = x0 + lane;
  } else {
    w = lane >> 1;
    side = lane & 1;
    active = lane < 2 * NW;
    if (!active) w = 0;
    xs = side ? x0 + XW : x0 - 1;
  }
  const int ys = y0 - 1 + w;
  // row waves: w == wave (wave-uniform); the halo wave's lanes map to (row, side)
  const bool out_row = !halo_wave && wave >= 1 && wave <= TY && y0 - 1 + wave < ny;
  const bool out_node = out_row && lane < XW;
  // row waves: lanes past a short row stay unwrapped (never stored)
  const int xw = PF && !halo_wave ? xs : ((xs % nx) + nx) % nx;
  const int yw = ((ys % ny) + ny) % ny;  // ys may exceed 2ny when ny < TY
  constexpr int GF = INLINE ? 5 : 3;     // fields of the g set: prep output or forces
  const int sx = dp.sx;
  const uint32_t srow = (uint32_t)sx * (uint32_t)yw;
  FOff off;
  off.m = ((uint32_t)xw + 10u * srow) * (uint32_t)sizeof(T);
  off.u = ((uint32_t)xw + 3u * srow) * (uint32_t)sizeof(T);
  off.rows = halo_wave ? 0 : 1;
  off.g = ((uint32_t)xw + (uint32_t)GF * srow) * (uint32_t)sizeof(TA);
  off.p = ((uint32_t)xw + (uint32_t)nx * (uint32_t)yw) * (uint32_t)sizeof(TA);
  // (a dword of 64-bit values in the x-halo wave: lane l serves node l / 2)
  auto node_at = [&](uint32_t o, size_t size) -> uint32_t {
    return size == 8 ? (uint32_t)__shfl((int)o, lane >> 1) + 4u * (lane & 1) : o & ~3u;
  };
  off.lm = off.rows ? off.m + row_off<T>(sx) : node_at(off.m, sizeof(T));
  off.lu = off.rows ? off.u + row_off<T>(sx) : node_at(off.u, sizeof(T));
  off.lg = off.rows ? off.g + row_off<TA>(sx) : node_at(off.g, sizeof(TA));
  off.lp = off.rows ? off.p + row_off<TA>(0) : node_at(off.p, sizeof(TA));
  const uint32_t splane = (uint32_t)sx * (uint32_t)ny;
  off.pm = ((10u * splane * (uint32_t)sizeof(T)) + 3u) & ~3u;
  off.pu = ((3u * splane * (uint32_t)sizeof(T)) + 3u) & ~3u;
  off.pg = (uint32_t)GF * splane * (uint32_t)sizeof(TA);
  off.pp = (uint32_t)(nxny * sizeof(TA));
  // node words with halo: per-lane in-plane offset, per-plane uniform base
  const uint32_t bI = 4u * ((uint32_t)(clampi(xs, -1, nx) + 1) + (uint32_t)(nx + 2) * (uint32_t)(clampi(ys, -1, ny) + 1));
  const uint32_t pbI = 4u * (uint32_t)(nx + 2) * (uint32_t)(ny + 2);
  auto word_load = [&](int z) -> uint32_t {
    return __builtin_amdgcn_raw_buffer_load_b32(mkrsrc(plane_at(a.words, pbI, clampi(z, -1, nz) + 1), pbI), bI, 0, 0);
  };

  T* Sout = (T*)a.mout;
  // 16-bit codecs: per-node seed of the stochastic rounding
  // and of the step: without a step term a node whose sibling field is
  // constant (e.g. exactly 0 in a planar flow) would draw the same threshold
  // every step, which makes its rounding deterministic and biased
  uint32_t nseed = 0u;
  if constexpr (C::dev) {
    const uint32_t step = a.seed + (a.seedp ? *a.seedp : 0u);
    nseed = mix32((uint32_t)xw * 0x9E3779B9u ^ (uint32_t)(yw + 1) * 0x85EBCA6Bu ^ mix32(step * 0x632BE5ABu + 0x1B873593u));
  }

  // z sums in flight.  The six lines (d, e) that outlive the x and y
  // contractions -- 0: (0,0), 1: (0,1), 2: (1,0), 3: (2,0), 4: (0,2), 5: (1,1) --
  // each give a source plane s the values r = -1, 0, +1.  zn: r = +1 of the last
  // source plane (it streams to the plane above); za, zb: r = +1 from below and
  // r = 0 of the plane that the next source plane completes, added up where
  // only their sum is needed (lines 3..5).  15 values instead of three planes of
  // ten accumulators, and no moves of whole accumulator planes.
  R zn[6], za[3], zb[6], oc[10];
#pragma unroll
  for (int k = 0; k < 6; ++k) { zn[k] = 0; zb[k] = 0; }
  za[0] = za[1] = za[2] = 0;
  R zbz = 0;  // the closure's share of the pending plane's Pi_zz (OB)
  auto store_oc = [&](int zo) {
    Mom<R> o;
    o.P = oc[0]; o.u = oc[1]; o.v = oc[2]; o.w = oc[3];
    o.xx = oc[4]; o.yy = oc[5]; o.zz = oc[6]; o.xy = oc[7]; o.xz = oc[8]; o.yz = oc[9];
    store_mom_b<PREC>(plane_at(Sout, off.pm, zo), (size_t)sx, off.pm, off.m, o, dp, nseed ^ (uint32_t)zo * 0xC2B2AE35u, a.nt != 0);
  };

  const R third = (R)(1.0 / 3.0);

  uint32_t lds0 = 0;
  uint32_t word_next = NODE_FLUID;
  if constexpr (PF) {
    lds0 = lds_addr((float*)&sPF[wave][0]);
    dma_raw<PREC, TWO, INLINE, GI>(a, wrapg(z0 - 1, nz), off, dens, lds0);
    if constexpr (OB) word_next = word_load(z0 - 1);
  }

  // ---- GI: phi tile stream and the per-node partial sums ------------------------
  // Wave v streams tile row v (v = 0 .. TY+2; the x-halo wave is v = NW), wave
  // 0 also row TY+3: 64 lanes to columns 2..65 and lanes 0-1 to columns 0-1
  // and 66-67.  Plane p lands in slot p & 3.  Iteration zsrc reads plane
  // zsrc+1 (issued in iteration zsrc-2, waited for at the top of zsrc-1 and
  // published by that iteration's barriers) and streams plane zsrc+3 into the
  // slot of plane zsrc-1, which every wave finished reading in iteration
  // zsrc-2.
  uint32_t ph_row1 = 0, ph_row2 = 0, ph_xm = 0, ph_xh = 0;
  const uint32_t lds_ph = GI ? lds_addr(&sPH[0][0][0]) : 0u;
  auto modn = [](int i, int n) { return ((i % n) + n) % n; };
  if constexpr (GI) {
    ph_row1 = __builtin_amdgcn_readfirstlane((uint32_t)modn(y0 - 2 + wave, ny) * (uint32_t)nx * 4u);
    ph_row2 = __builtin_amdgcn_readfirstlane((uint32_t)modn(y0 - 2 + GR - 1, ny) * (uint32_t)nx * 4u);
    ph_xm = (uint32_t)modn(x0 + lane, nx) * 4u;
    // halo columns: lanes 0-1 the left pair, lanes 2-3 the right
    ph_xh = (uint32_t)modn((lane & 2) ? x0 + 62 + (lane & 3) : x0 - 2 + (lane & 1), nx) * 4u;
  }
  // Away from the x faces (no wrap inside the tile's columns) the tile is one
  // run of 17 GR 16-byte pieces, a lane each.
  const bool ph_quad = GI && x0 >= 2 && x0 + 66 <= nx;
  if (ph_quad) {
    const int L = min((int)threadIdx.x, GR * (GC / 4) - 1);
    ph_xm = ((uint32_t)modn(y0 - 2 + L / (GC / 4), ny) * (uint32_t)nx + (uint32_t)(x0 - 2 + 4 * (L % (GC / 4)))) * 4u;
  }
  auto dma_phi = [&](int z) {
    if (ph_quad) {
      if ((int)threadIdx.x < GR * (GC / 4)) {
        const Rsrc rq = mkrsrc(plane_at((const float*)a.phin, off.pp, modn(z, nz)), off.pp);
        dma_quad<0u>(rq, ph_xm, 0u,
                     lds_ph + (uint32_t)(z & 3) * (uint32_t)(GR * GC * 4) + (uint32_t)wave * 1024u);
      }
      return;
    }
    const Rsrc rs = mkrsrc(plane_at((const float*)a.phin, off.pp, modn(z, nz)), off.pp);
    const uint32_t base = lds_ph + (uint32_t)(z & 3) * (uint32_t)(GR * GC * 4);
    const uint32_t r1 = base + (uint32_t)wave * (uint32_t)(GC * 4);
    dma_dword<8u>(rs, ph_row1 + ph_xm, r1);
    if (lane < 2) dma_dword<0u>(rs, ph_row1 + ph_xh, r1);
    if ((lane & ~1) == 2) dma_dword<64u * 4u>(rs, ph_row1 + ph_xh, r1);
    if (wave == 0) {
      const uint32_t r2 = base + (uint32_t)(GR - 1) * (uint32_t)(GC * 4);
      dma_dword<8u>(rs, ph_row2 + ph_xm, r2);
      if (lane < 2) dma_dword<0u>(rs, ph_row2 + ph_xh, r2);
      if ((lane & ~1) == 2) dma_dword<64u * 4u>(rs, ph_row2 + ph_xh, r2);
    }
  };
  // this lane's node sits at tile row w + 1, column pc
  const int pc = halo_wave ? (side ? XW + 2 : 1) : lane + 2;
  auto phi_part = [&](int z) -> Part3<R> {
    const int sl = z & 3;
    R v[3][3];
#pragma unroll
    for (int bb = 0; bb < 3; ++bb)
#pragma unroll
      for (int aa = 0; aa < 3; ++aa) v[bb][aa] = (R)sPH[sl][w + bb][pc - 1 + aa];
    return part3(v);
  };
  Part3<R> gpm{}, gp0{};  // partials of planes zsrc-1 and zsrc (gp0.c: phi at the node)
  if constexpr (GI) {
    dma_phi(z0 - 2);
    dma_phi(z0 - 1);
    dma_phi(z0);
    dma_phi(z0 + 1);
    dma_wait_all();
    __syncthreads();
    gpm = phi_part(z0 - 2);
    gp0 = phi_part(z0 - 1);
    __syncthreads();  // the slots of planes z0-2 and z0-1 are refilled in the first iterations
  }

  for (int zsrc = z0 - 1; zsrc <= zend; ++zsrc) {
    const int zw = wrapg(zsrc, nz);
    const bool own_plane = zsrc >= z0 && zsrc < zend;
    RawNode<PREC> cur;
    uint32_t word = NODE_FLUID;
    if constexpr (PF) {
      dma_wait_all();
      // 16-bit storage: waves between this wait and the next plane's DMA
      // issue (store, decode, moments stage) run at raised priority, ahead of
      // waves in the collision, so the transfers start sooner (fused kernel
      // 3.92 -> 3.43 ms FP16S at 512^3; no gain for FP32)
      if constexpr (sizeof(T) == 2) __builtin_amdgcn_s_setprio(2);
      if constexpr (OB) {
        word = word_next;
        asm volatile("" : "+v"(word));  // consume the prefetched word before this iteration's stores
      }
      // the plane completed by the previous iteration
      if (out_row && lane < XW && zsrc - 2 >= z0) store_oc(zsrc - 2);
      lds_raw<PREC, TWO, INLINE, GI>(cur, sPF[wave], lane, dens, off.m, off.rows != 0);
      if constexpr (GI) {
        // the prep's fields 0-3 (prep_body_z, stored at storage precision)
        const Part3<R> gpp = phi_part(zsrc + 1);
        R gx, gy, gz, lap;
        grad_lap(gpm, gp0, gpp, gx, gy, gz, lap);
        R mg, im;
        grad_norm(gx * gx + gy * gy + gz * gz, mg, im);
        const R mgs = (R)(TA)mg;
        cur.g[0] = (TA)((R)(TA)(gx * im) * mgs);
        cur.g[1] = (TA)((R)(TA)(gy * im) * mgs);
        cur.g[2] = (TA)((R)(TA)(gz * im) * mgs);
        cur.g[3] = (TA)lap;
        cur.phi = (TA)gp0.c;
        gpm = gp0;
        gp0 = gpp;
      }
    } else {
      if constexpr (OB) word = word_load(zsrc);
      load_raw<PREC, TWO, INLINE>(cur, a, zw, (size_t)sx, off);
    }

    // ---- 1. decode + (inline) moments stage + collision ---------------------
    // f: D3Q27 the Hermite coefficients A[a + 3b + 9c] (hermite27), D3Q19 the
    // populations
    R f[27];
    R lbs[4] = {0, 0, 0, 0};  // near-wall closure: what zn cannot take (below)
    {
      NodeIn<R> in;
      Mom<R> m;
      m.P = C::dec(cur.m[0], iscl<PREC>(dp, 0)); m.u = C::dec(cur.m[1], iscl<PREC>(dp, 1));
      m.v = C::dec(cur.m[2], iscl<PREC>(dp, 2)); m.w = C::dec(cur.m[3], iscl<PREC>(dp, 3));
      m.xx = C::dec(cur.m[4], iscl<PREC>(dp, 4)); m.yy = C::dec(cur.m[5], iscl<PREC>(dp, 5));
      m.zz = C::dec(cur.m[6], iscl<PREC>(dp, 6)); m.xy = C::dec(cur.m[7], iscl<PREC>(dp, 7));
      m.xz = C::dec(cur.m[8], iscl<PREC>(dp, 8)); m.yz = C::dec(cur.m[9], iscl<PREC>(dp, 9));
      if constexpr (C::dev) {
        // second moments: stored deviation + u u (one mixed FMA each)
        m.xx = C::decpi(cur.m[4], iscl<PREC>(dp, 4), m.u * m.u);
        m.yy = C::decpi(cur.m[5], iscl<PREC>(dp, 5), m.v * m.v);
        m.zz = C::decpi(cur.m[6], iscl<PREC>(dp, 6), m.w * m.w);
        m.xy = C::decpi(cur.m[7], iscl<PREC>(dp, 7), m.u * m.v);
        m.xz = C::decpi(cur.m[8], iscl<PREC>(dp, 8), m.u * m.w);
        m.yz = C::decpi(cur.m[9], iscl<PREC>(dp, 9), m.v * m.w);
      }
      R phl = 0, Fx, Fy, Fz;
      const bool solid = OB && !(word & NODE_FLUID), wall = OB && (word & NODE_WALL);
      if constexpr (TWO) phl = (R)cur.phi;
      const NodeRates<R> nr = node_rates<TWO, R, STD>(dp, phl);
      const R rinv = nr.irho;
      if constexpr (!INLINE) {
        Fx = (R)cur.g[0] * rinv;
        Fy = (R)cur.g[1] * rinv;
        Fz = (R)cur.g[2] * rinv;
      } else {
        R gfx = 0, gfy = 0, gfz = 0, lap = 0, dvt = 0, uox = 0, uoy = 0, uoz = 0;
        if constexpr (TWO) {
          gfx = (R)cur.g[0];
          gfy = (R)cur.g[1];
          gfz = (R)cur.g[2];
          lap = (R)cur.g[3];
          dvt = (R)cur.g[4];
          if (dens) {
            uox = C::dec(cur.uo[0], iscl<PREC>(dp, 1));
            uoy = C::dec(cur.uo[1], iscl<PREC>(dp, 2));
            uoz = C::dec(cur.uo[2], iscl<PREC>(dp, 3));
          }
        }
        R tFx, tFy, tFz;
        moments_stage<TWO, R, STD>(dp, nr, phl, gfx, gfy, gfz, lap, dvt, uox, uoy, uoz, m, tFx, tFy, tFz);
        // the reference stores S and the forces at storage precision between
        // the moments and fused kernels
        m.u = C::round(m.u); m.v = C::round(m.v); m.w = C::round(m.w);
        m.xx = C::round(m.xx); m.yy = C::round(m.yy); m.zz = C::round(m.zz);
        m.xy = C::round(m.xy); m.xz = C::round(m.xz); m.yz = C::round(m.yz);
        tFx = C::round(tFx); tFy = C::round(tFy); tFz = C::round(tFz);
        Fx = tFx * rinv; Fy = tFy * rinv; Fz = tFz * rinv;
        if (out_node && own_plane && !solid) {
          if constexpr (OPEN) {
            if (wall && open_layer(dp, xs, ys, zsrc)) {
              // open faces: the post-moments state of a first-layer node,
              // which the open-face correction reads after this launch (the
              // stage sequence reads it from S)
              store_mom_b<PREC>(plane_at((T*)a.sopen, off.pm, zw), (size_t)sx, off.pm, off.m, m, dp, 0u, false);
            }
          }
          if constexpr (TWO) {
            if (dens) {
              T e[3] = {C::enc(m.u, scl<PREC>(dp, 1)), C::enc(m.v, scl<PREC>(dp, 2)), C::enc(m.w, scl<PREC>(dp, 3))};
              if constexpr (C::dev) {
                const uint32_t st = (nseed ^ (uint32_t)zw * 0x27D4EB2Fu) & C::RBITS;
                const float xu = m.u * scl<PREC>(dp, 1), xv = m.v * scl<PREC>(dp, 2), xw_ = m.w * scl<PREC>(dp, 3);
                e[0] = C::srx(xu, (__float_as_uint(xv) & C::RBITS) ^ st);
                e[1] = C::srx(xv, (__float_as_uint(xw_) & C::RBITS) ^ st);
                e[2] = C::srx(xw_, (__float_as_uint(xu) & C::RBITS) ^ st);
              }
              store_fields(plane_at((T*)a.uout, off.pu, zw), off.pu, (uint32_t)(sx * sizeof(T)), off.u, e, a.nt != 0);
            }
            // update_phi (update_phi:88-93), u after the moments stage
            const R t = -ph.sharp_c * dvt;
            const R po = phl - m.u * (R)0.5 * (gfx) - m.v * (R)0.5 * (gfy) - m.w * (R)0.5 * (gfz) +
                         ph.tau_diff * lap + t;
            const TA pv[1] = {(TA)po};
            store_fields(plane_at((TA*)a.phiout, off.pp, zw), off.pp, 0u, off.p, pv, a.nt != 0);
          }
          if (OB && !bb && wall) {
            // LB_int_boundary (boundary:117-212) on the post-moments state: the
            // directions that some lane of the wave needs, one at a time
            R lbc[10];
            const R cssq = (R)(1.0 / 3.0);
            const R pxx = m.xx - m.u * m.u, pyy = m.yy - m.v * m.v, pzz = m.zz - m.w * m.w;
            const R pxy = m.xy - m.u * m.v, pxz = m.xz - m.u * m.w, pyz = m.yz - m.v * m.w;
            const R om1 = (R)4.5 * ((R)1 - relax_rate<TWO, R, STD>(dp, nr, pxx, pyy, pzz, pxy, pxz, pyz));
#pragma unroll
            for (int q = 0; q < 10; ++q) lbc[q] = 0;
#pragma unroll
            for (int c = 0; c < 27; ++c) {
              const int p = c % 3 - 1, q = (c / 3) % 3 - 1, r = c / 9 - 1;
              if (c == 13 || !present<LAT>(p, q, r)) continue;
              const bool hit = word & (1u << c);
              if (__ballot(hit) == 0) continue;
              const R qn = ((R)(p * p) - cssq) * pxx + ((R)(q * q) - cssq) * pyy + ((R)(r * r) - cssq) * pzz +
                           (R)(2 * p * q) * pxy + (R)(2 * p * r) * pxz + (R)(2 * q * r) * pyz;
              const R fp = (R)weight<LAT>(p, q, r) * (m.P + om1 * qn);
              add_closure<R>(lbc, p, q, r, hit ? fp : (R)0);
            }
            closure_to_z<R>(lbc, zn, lbs);
          }
        }
      }
      if (solid) {
        m.P = m.u = m.v = m.w = m.xx = m.yy = m.zz = m.xy = m.xz = m.yz = 0;
        Fx = Fy = Fz = 0;
      }
      in.P = m.P; in.u = m.u; in.v = m.v; in.w = m.w;
      in.xx = m.xx - m.u * m.u; in.yy = m.yy - m.v * m.v; in.zz = m.zz - m.w * m.w;
      in.xy = m.xy - m.u * m.v; in.xz = m.xz - m.u * m.w; in.yz = m.yz - m.v * m.w;
      in.ax = Fx; in.ay = Fy; in.az = Fz;
      in.om = relax_rate<TWO, R, STD>(dp, nr, in.xx, in.yy, in.zz, in.xy, in.xz, in.yz);
      if constexpr (PF) {
        // every store of this iteration is issued: stream the next plane in
        lds_wait_all();
        if (zsrc < zend) {
          if (!halo_wave) dma_raw<PREC, TWO, INLINE, GI>(a, wrapg(zsrc + 1, nz), off, dens, lds0);
          if constexpr (OB) word_next = word_load(zsrc + 1);
        }
        if (GI && zsrc + 3 <= zend + 1) dma_phi(zsrc + 3);
        if constexpr (sizeof(T) == 2) __builtin_amdgcn_s_setprio(0);
      }
      if constexpr (LAT == 27) hermite27<HO, R>(in, f);
      else collide<LAT, HO, R>(in, f);
      if (bb && wall && out_node && own_plane) {
        // BOUNCE_BACK (fused_LB_kernel_bb, fused:364-382): a population whose
        // upstream node is solid is replaced by this node's own opposite
        // post-collision population.  The solid node's pushed population is
        // exactly zero (its moments and force are zeroed), so the pull below
        // adds zero and the replacement is this correction.  D3Q27 forms the
        // opposite population from the coefficients, one direction at a time
        // (a loop, not 26 copies: the populations all at once would not fit
        // the registers beside the coefficients).
        R lbc[10];
#pragma unroll
        for (int q = 0; q < 10; ++q) lbc[q] = 0;
        if constexpr (LAT == 27) {
#pragma unroll 1
          for (int c = 0; c < 27; ++c) {
            const bool hit = word & (1u << c);
            if (c == 13 || __ballot(hit) == 0) continue;
            const int p = c % 3 - 1, q = (c / 3) % 3 - 1, r = c / 9 - 1;
            add_closure<R>(lbc, p, q, r, hit ? population27<HO, R>(f, -p, -q, -r) : (R)0);
          }
        } else {
#pragma unroll
          for (int c = 0; c < 27; ++c) {
            const int p = c % 3 - 1, q = (c / 3) % 3 - 1, r = c / 9 - 1;
            if (c == 13 || !present<LAT>(p, q, r)) continue;
            add_closure<R>(lbc, p, q, r, word & (1u << c) ? f[cidx(-p, -q, -r)] : (R)0);
          }
        }
        closure_to_z<R>(lbc, zn, lbs);
      }
    }

    // ---- 2. x: reconstruct over a (D3Q27); the halo's slices through LDS ------------
    // Axis by axis: a line (b, c) of Hermite coefficients (D3Q19: (q, r) of
    // populations) becomes its three x populations, which shift one lane and
    // contract to the moment index d before the next axis is reconstructed.
    // The axes' operators commute, so this is the full reconstruction followed
    // by the full contraction with fewer lines left on the later axes (6
    // instead of 9 in z), and a halo node stops at the one slice that it hands
    // over: the x-halo wave forms 9 of its 27 populations, the halo rows 9
    // partial sums.
    if (halo_wave) {
      // the left halo (side 0) streams +x into lane 0, the right -x into lane XW-1
      if constexpr (LAT == 27) {
        const R sg = side ? (R)-1 : (R)1;
#pragma unroll
        for (int j = 0; j < 9; ++j) {
          const int b = j % 3, c = j / 3;
          R t = 0;
          if (HO || b + c <= 2) t = recon_side(f[3 * j], f[3 * j + 2], HO || b + c == 0);
          if (HO || b + c <= 1) t = t + sg * f[3 * j + 1];
          if (active) sHX[w][side][j] = t;
        }
      } else if (active) {
        // the two sides are separate branches with constant register indices:
        // a select between the sides' values is turned by the compiler into a
        // lane-variable index and expanded into a 27-way compare chain
        if (side == 0) {
#pragma unroll
          for (int j = 0; j < 9; ++j) sHX[w][0][j] = f[3 * j + 2];
        } else {
#pragma unroll
          for (int j = 0; j < 9; ++j) sHX[w][1][j] = f[3 * j];
        }
      }
    } else if constexpr (LAT == 27) {
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const int b = j % 3, c = j / 3;
        if (!HO && b + c > 2) continue;
        R fm, f0, fp;
        recon3(f[3 * j], f[3 * j + 1], f[3 * j + 2], fm, f0, fp, HO || b + c <= 1, HO || b + c == 0);
        f[3 * j] = fm; f[3 * j + 1] = f0; f[3 * j + 2] = fp;
      }
    }
    if constexpr (PF) {
      // The x-halo wave's next-plane inputs (14 scattered dwords per lane)
      // are issued here, after its collision, instead of with the row
      // waves' transfers: the issue points of a block's waves spread over
      // the iteration (fused kernel 3.91 -> 3.82 ms FP32, 3.37 -> 3.22 ms
      // FP16S at 512^3).  Its slots were read at the top of the iteration.
      if (halo_wave && zsrc < zend) {
        lds_wait_all();
        dma_raw<PREC, TWO, INLINE, GI>(a, wrapg(zsrc + 1, nz), off, dens, lds0);
      }
    }
    __syncthreads();

    R G0[9];  // q = 0 partial sums kept in registers: [d][c]
    if (!halo_wave) {
      // ---- 3. x: shift by one lane, contract over p ---------------------------
      // the x-halo values enter as DPP fill operands, read by every lane
      // from one LDS address (a broadcast).  d = 2 is carried as 3 (c^2 - 1/3)
      // = 2, -1, 2 (one multiply-add, one rounding); the factor 1/3 follows
      // when the plane is complete.
      if (XW < 64 && lane == XW) {
        // a short row's right halo enters below lane 63: put it where lane
        // XW - 1 fetches from
#pragma unroll
        for (int j = 0; j < 9; ++j) f[3 * j] = sHX[wave][1][j];
      }
      R G[3][9];  // [d][line]
#pragma unroll
      for (int j = 0; j < 9; ++j) {
        const int b = j % 3, c = j / 3;  // D3Q19: q + 1, r + 1
        const bool any = LAT == 27 ? (HO || b + c <= 2) : true;
        const bool sides = LAT == 27 ? any : present<LAT>(1, b - 1, c - 1);
        R fm_in = 0, fp_in = 0;
        if (sides) {
          fp_in = shift_from_lower(f[3 * j + 2], sHX[wave][0][j]);
          fm_in = shift_from_upper(f[3 * j], sHX[wave][1][j]);
        }
        if (!any) {
          G[0][j] = G[1][j] = G[2][j] = 0;
        } else if (!sides) {
          G[0][j] = f[3 * j + 1]; G[1][j] = 0; G[2][j] = -f[3 * j + 1];
        } else {
          const R sp = fp_in + fm_in;
          G[0][j] = f[3 * j + 1] + sp;
          G[1][j] = fp_in - fm_in;
          G[2][j] = (R)2 * sp - f[3 * j + 1];
        }
      }
      // ---- 4a. y: hand the q = +-1 partial sums to the neighbouring rows ------
      R T0[9], T1[9];
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int c = 0; c < 3; ++c) {
          const int k = d * 3 + c, j = 3 * c;
          if constexpr (LAT == 27) {
            T0[k] = recon_side(G[d][j], G[d][j + 2], HO || c == 0);
            T1[k] = HO || c <= 1 ? G[d][j + 1] : (R)0;
            G0[k] = G[d][j] - (R)2 * T0[k];
          } else {
            T0[k] = G[d][j + 2]; T1[k] = G[d][j];
            G0[k] = G[d][j + 1];
          }
        }
      if (wave < NW - 1) {
#pragma unroll
        for (int k = 0; k < 9; ++k) sUP[wave][k][lane] = LAT == 27 ? T0[k] + T1[k] : T0[k];
      }
      if (wave > 0) {
#pragma unroll
        for (int k = 0; k < 9; ++k) sDN[wave][k][lane] = LAT == 27 ? T0[k] - T1[k] : T1[k];
      }
    }
    __syncthreads();

    if (out_row) {
      // ---- 4b. y: contract over q ------------------------------------------------
      // H[k][c] of the six lines (d, e); e = 2 tripled as d = 2 above
      R H[6][3];
#pragma unroll
      for (int c = 0; c < 3; ++c) {
        {
          const R gp = sUP[wave - 1][c][lane], gm = sDN[wave + 1][c][lane], sp = gp + gm;
          H[0][c] = G0[c] + sp;
          H[1][c] = gp - gm;
          H[4][c] = (R)2 * sp - G0[c];
        }
        {
          const R gp = sUP[wave - 1][3 + c][lane], gm = sDN[wave + 1][3 + c][lane];
          H[2][c] = G0[3 + c] + (gp + gm);
          H[5][c] = gp - gm;
        }
        H[3][c] = G0[6 + c] + (sUP[wave - 1][6 + c][lane] + sDN[wave + 1][6 + c][lane]);
      }
      // ---- 5. z: r = -1 completes plane zsrc-1, r = 0 and +1 stay in flight --------
      // outputs: 0 P(000) 1 u(100) 2 v(010) 3 w(001) 4 xx(200) 5 yy(020) 6 zz(002)
      //          7 xy(110) 8 xz(101) 9 yz(011)
      R hm[6], h0[6], hp[6];
#pragma unroll
      for (int k = 0; k < 6; ++k) {
        if constexpr (LAT == 27) recon3(H[k][0], H[k][1], H[k][2], hm[k], h0[k], hp[k]);
        else { hm[k] = H[k][0]; h0[k] = H[k][1]; hp[k] = H[k][2]; }
      }
      {
        const R sp = za[0] + hm[0];
        oc[0] = zb[0] + sp; oc[3] = za[0] - hm[0]; oc[6] = ((R)2 * sp - zb[0]) * third;
        oc[2] = zb[1] + (za[1] + hm[1]); oc[9] = za[1] - hm[1];
        oc[1] = zb[2] + (za[2] + hm[2]); oc[8] = za[2] - hm[2];
        oc[4] = (zb[3] + hm[3]) * third; oc[5] = (zb[4] + hm[4]) * third; oc[7] = zb[5] + hm[5];
      }
      if constexpr (OB) {
        oc[6] += zbz;
        zbz = lbs[3];
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        za[k] = zn[k];
        zb[k] = h0[k];
        if constexpr (OB) zb[k] += lbs[k];
      }
#pragma unroll
      for (int k = 3; k < 6; ++k) zb[k] = zn[k] + h0[k];
#pragma unroll
      for (int k = 0; k < 6; ++k) zn[k] = hp[k];
      // ---- 6. plane zsrc-1 is complete (stored here, or by the next iteration) --
      if constexpr (!PF) {
        const int zo = zsrc - 1;
        if (lane < XW && zo >= z0 && zo < zend) store_oc(zo);
      }
    }
  }
  if constexpr (PF) {
    if (out_row && lane < XW) store_oc(zend - 1);
  }
}

// One domain per launch: 1-D grid, XCD-aware tile order.
template <int LAT, bool HO, int PREC, bool TWO, bool INLINE, int TY, bool OB, bool STD, bool OPEN>
__global__ void __launch_bounds__((TY + 3) * 64) fused_kernel(FusedArgs a) {
  fused_body<LAT, HO, PREC, TWO, INLINE, TY, OB, STD, OPEN>(a, xcd_tile(blockIdx.x, fused_tiles<TY>(a)));
}

// Many domains per launch: the grid covers every domain's tiles in table
// order (domain-major); a block finds its domain by binary search over the
// tile offsets, then runs the same body on that domain's arguments.
template <int LAT, bool HO, int PREC, bool TWO, int TY, bool STD>
__global__ void __launch_bounds__((TY + 3) * 64)
    fused_kernel_batch(const FusedBatchEntry* __restrict__ tab, int ndom, int total) {
  const int g = xcd_tile(blockIdx.x, total);
  int lo = 0, hi = ndom - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (tab[mid].tile0 <= g) lo = mid; else hi = mid - 1;
  }
  fused_body<LAT, HO, PREC, TWO, true, TY, false, STD>(tab[lo].a, g - tab[lo].tile0);  // batches hold no obstacles
}

// ---------------------------------------------------------------------------
template <int LAT, bool HO, int PREC, bool TWO, bool INLINE, int TY, bool STD>
static hipError_t launch_std(const FusedArgs& a, hipStream_t s) {
  dim3 grid(fused_tiles<TY>(a));
  dim3 block((TY + 3) * 64);
  // open faces reach the fast path with obstacles and 32/64-bit storage only
  constexpr bool open_ok = INLINE && prec_base(PREC) <= PREC_MIXED;
  if (a.dp.obst) {
    if constexpr (open_ok) {
      if (a.sopen) {
        hipLaunchKernelGGL((fused_kernel<LAT, HO, PREC, TWO, INLINE, TY, true, STD, true>), grid, block, 0, s, a);
        return hipGetLastError();
      }
    }
    hipLaunchKernelGGL((fused_kernel<LAT, HO, PREC, TWO, INLINE, TY, true, STD, false>), grid, block, 0, s, a);
  } else {
    hipLaunchKernelGGL((fused_kernel<LAT, HO, PREC, TWO, INLINE, TY, false, STD, false>), grid, block, 0, s, a);
  }
  return hipGetLastError();
}

template <int LAT, bool HO, int PREC, bool TWO, bool INLINE, int TY>
static hipError_t launch_t(const FusedArgs& a, hipStream_t s) {
  // the stage path's kernel has few switches left in it
  if constexpr (INLINE) {
    if (std_switches(a.dp)) return launch_std<LAT, HO, PREC, TWO, INLINE, TY, true>(a, s);
  }
  return launch_std<LAT, HO, PREC, TWO, INLINE, TY, false>(a, s);
}

template <int PREC, bool TWO, bool INLINE, int TY>
static hipError_t launch_lat(const FusedArgs& a, hipStream_t s) {
  if (a.dp.lattice == 19) return launch_t<19, false, PREC, TWO, INLINE, TY>(a, s);
  if (a.dp.highorder) return launch_t<27, true, PREC, TWO, INLINE, TY>(a, s);
  return launch_t<27, false, PREC, TWO, INLINE, TY>(a, s);
}

template <int PREC, bool INLINE, int TY>
static hipError_t launch_two(const FusedArgs& a, hipStream_t s) {
  if (a.dp.twocomp) return launch_lat<PREC, true, INLINE, TY>(a, s);
  return launch_lat<PREC, false, INLINE, TY>(a, s);
}

template <int PREC, bool INLINE>
static hipError_t launch_ty(const FusedArgs& a, hipStream_t s) {
  switch (a.ty) {
    case 5:
      if constexpr (PREC == PREC_FP64 || PREC == PREC_MIXED) return launch_two<PREC, INLINE, 5>(a, s);
      else return hipErrorInvalidValue;
    case 8: return launch_two<PREC, INLINE, 8>(a, s);
    case 13: return launch_two<PREC, INLINE, 13>(a, s);
    default: return hipErrorInvalidValue;
  }
}

template <int PREC, bool TWO, int TY, bool STD>
static hipError_t batch_lat(const FusedBatchEntry* tab, int ndom, int total, int lat, bool ho, hipStream_t s) {
  dim3 grid(total), block((TY + 3) * 64);
  if (lat == 19) hipLaunchKernelGGL((fused_kernel_batch<19, false, PREC, TWO, TY, STD>), grid, block, 0, s, tab, ndom, total);
  else if (ho) hipLaunchKernelGGL((fused_kernel_batch<27, true, PREC, TWO, TY, STD>), grid, block, 0, s, tab, ndom, total);
  else hipLaunchKernelGGL((fused_kernel_batch<27, false, PREC, TWO, TY, STD>), grid, block, 0, s, tab, ndom, total);
  return hipGetLastError();
}

template <int PREC, bool TWO, int TY>
static hipError_t batch_std(const FusedBatchEntry* tab, int ndom, int total, int lat, bool ho, bool std, hipStream_t s) {
  return std ? batch_lat<PREC, TWO, TY, true>(tab, ndom, total, lat, ho, s)
             : batch_lat<PREC, TWO, TY, false>(tab, ndom, total, lat, ho, s);
}

template <int PREC, bool TWO>
static hipError_t batch_ty(const FusedBatchEntry* tab, int ndom, int total, int lat, bool ho, bool std, int ty, hipStream_t s) {
  if constexpr (PREC == PREC_FP64 || PREC == PREC_MIXED) {
    if (ty == 5) return batch_std<PREC, TWO, 5>(tab, ndom, total, lat, ho, std, s);
  }
  if (ty == 8) return batch_std<PREC, TWO, 8>(tab, ndom, total, lat, ho, std, s);
  if (ty == 13) return batch_std<PREC, TWO, 13>(tab, ndom, total, lat, ho, std, s);
  return hipErrorInvalidValue;
}

template <int PREC>
hipError_t fused_batch_prec(const FusedBatchEntry* tab, int ndom, int total, int lat, bool ho, bool two, bool std, int ty,
                            hipStream_t s) {
  if (!two) return batch_ty<PREC, false>(tab, ndom, total, lat, ho, std, ty, s);
  // two components in FP64 are not batched (lbf_batch_create)
  if constexpr (PREC != PREC_FP64) return batch_ty<PREC, true>(tab, ndom, total, lat, ho, std, ty, s);
  else return hipErrorInvalidValue;
}

template <int PREC>
hipError_t fused_prec(const FusedArgs& a, bool inline_moments, hipStream_t s) {
  if (inline_moments) return launch_ty<PREC, true>(a, s);
  // the stage path stores 32 or 64 bits
  if constexpr (PREC <= PREC_MIXED) return launch_ty<PREC, false>(a, s);
  else return hipErrorInvalidValue;
}

template hipError_t fused_prec<LBF_FUSED_PREC>(const FusedArgs&, bool, hipStream_t);
template hipError_t fused_batch_prec<LBF_FUSED_PREC>(const FusedBatchEntry*, int, int, int, bool, bool, bool, int,
                                                         hipStream_t);

#else  // the dispatch

int fused_tile_count(const FusedArgs& a) {
  switch (a.ty) {
    case 5: return fused_tiles<5>(a);
    case 8: return fused_tiles<8>(a);
    case 13: return fused_tiles<13>(a);
  }
  return -1;
}

hipError_t launch_fused_batch(const FusedBatchEntry* dev_tab, int ndom, int total_tiles, int prec, int lattice,
                              bool highorder, bool two, bool std, int ty, hipStream_t s) {
  switch (prec) {
    case PREC_FP16S | PREC_DEFSCALE:
      return fused_batch_prec<PREC_FP16S | PREC_DEFSCALE>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
    case PREC_BF16S | PREC_DEFSCALE:
      return fused_batch_prec<PREC_BF16S | PREC_DEFSCALE>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
    case PREC_FP64: return fused_batch_prec<PREC_FP64>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
    case PREC_FP32: return fused_batch_prec<PREC_FP32>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
    case PREC_MIXED: return fused_batch_prec<PREC_MIXED>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
    case PREC_FP16S: return fused_batch_prec<PREC_FP16S>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
    case PREC_BF16S: return fused_batch_prec<PREC_BF16S>(dev_tab, ndom, total_tiles, lattice, highorder, two, std, ty, s);
  }
  return hipErrorInvalidValue;
}

bool default_scales(const DevParams& dp) {
  for (int i = 0; i < 10; ++i)
    if (dp.scale[i] != def_scale(i)) return false;
  return true;
}

hipError_t launch_fused(const FusedArgs& a, int prec, bool inline_moments, hipStream_t s) {
  if ((prec == PREC_FP16S || prec == PREC_BF16S) && default_scales(a.dp)) prec |= PREC_DEFSCALE;
  switch (prec) {
    case PREC_FP64: return fused_prec<PREC_FP64>(a, inline_moments, s);
    case PREC_FP32: return fused_prec<PREC_FP32>(a, inline_moments, s);
    case PREC_MIXED: return fused_prec<PREC_MIXED>(a, inline_moments, s);
    case PREC_FP16S: return fused_prec<PREC_FP16S>(a, inline_moments, s);
    case PREC_BF16S: return fused_prec<PREC_BF16S>(a, inline_moments, s);
    case PREC_FP16S | PREC_DEFSCALE: return fused_prec<PREC_FP16S | PREC_DEFSCALE>(a, inline_moments, s);
    case PREC_BF16S | PREC_DEFSCALE: return fused_prec<PREC_BF16S | PREC_DEFSCALE>(a, inline_moments, s);
  }
  return hipErrorInvalidValue;
}

#endif

}  // namespace lbf
