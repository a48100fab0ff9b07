// fused_mixed.hip -- the fused (T) kernel on 16x16 MFMA tiles: the d1/d2
// contractions in FP64 or in reduced precision; the denominators, their
// division, the singles term and every energy sum in FP64.
//
//   TCE_T_FP64    v_mfma_f64_16x16x4_f64, FP64 operands and accumulation
//                 (the default FP64 kernel of 8-wide tilings); its D layout
//                 puts row i in lane group i%4, register i/4, so its X rows
//                 are ordered 4r + L' (the roles of the two fields swapped)
//   TCE_T_FP32    v_mfma_f32_16x16x4_f32, FP32 operands and accumulation
//   TCE_T_BF16X3  v_mfma_f32_16x16x32_bf16, each operand x split into
//                 hi = bf16(x), lo = bf16(x - hi); per product hi*hi + hi*lo
//                 + lo*hi (3 terms), FP32 accumulation
//   TCE_T_BF16X6  the same MFMA, x = hi + mid + lo (three bf16, 24 bits);
//                 per product the 6 terms down to 2^-24 relative (hi*hi,
//                 hi*mid, mid*hi, hi*lo, mid*mid, lo*hi), FP32 accumulation;
//                 two LDS chunk buffers (three parts of 24 KB per chunk)
//
// Work item as fused_wg.hip: one task x an 8x8x8 particle box x a 4x4x4 hole
// box; a wave owns one 4x4x4 particle cube of the box by the hole box, 4096 t3
// elements in 16 quads of accumulators per lane.  A workgroup is 8 waves on
// the whole item (split BF16) or 4 waves on one half of it along particle c
// (FP64, FP32), two workgroups to a CU: while one waits at a chunk barrier, for
// its first loads or in its epilogue, the other has the matrix cores.  With 8
// waves in step, an FP64 item spent a quarter (no=40/nv=160) to two thirds
// (short contraction ranges) of its time outside the MFMAs.  Half an item loads
// 1.5 times the bytes per flop (8 to 10 of the L2's 64 bytes per clock and CU at
// the FP64 rate); at the BF16 rate they would be most of that bandwidth.
//
// MFMA lane layout (16x16, probed on the device): A[i][k] at lane i+16(k/E),
// B[k][j] at lane j+16(k/E) (E = k values per lane: 1 for f32, 8 for bf16),
// D[i][j] at lane j+16(i/4), register i%4.  Every d1/d2 contraction is
// X(L, r, s; e) * Y(p1, p2, h; e): lone particle L with the hole pair (r, s)
// on one operand, the particle pair (p1, p2) with the lone hole h on the
// other.  With L fixed, row i = 4L' + r and col j = 4p1' + p2', so
//   lane = 4 p1' + p2' + 16 L', accumulator quad (s, h), component r.
// The lane keeps element (i, j, k) of its hole box at q[4j + k][i].  Lone
// hole j (r = i, s = k) and k (r = i, s = j) find their MFMA quads there; for
// lone hole i (r = j, s = k) the quads of each k are transposed in registers
// (q[4i + k][j]), after which its quads lie as those of lone hole j, so both
// run the same chunk loop.  Changing L (a -> b -> c) is one lane permutation.
// Passes: L = a, b, c x lone hole j, i, k x {d2, d1}; the d2 and d1 chunks of
// one (L, h) form one chunk sequence.
//
// Work that the symmetry of t3 makes redundant is not done.  With equal hole
// boxes, P_h(i,j,k) (the passes of lone hole h) obey P_i = -P_j(i <-> j) for
// I == J and P_k = -P_j(j <-> k) for J == K, so one of the two is left out
// and the sum is antisymmetrised in registers; the third is antisymmetric by
// itself, so only its pairs r < s (quads s >= 1) are formed.  With I == J ==
// K the passes of lone hole k alone give the four distinct elements.  Equal
// particle boxes save the passes of one lone particle (two when all are
// equal) the same way, with the exchange of the waves' accumulators through
// LDS at the end.  Of 18 pass pairs, a box with equal I, J runs 12, one with
// equal I, J, K 6.  Quads past a ragged edge of the hole boxes and waves
// whose particle cube lies past the edge issue no MFMA, and rows no quad
// needs are not loaded.
//
// Operands stream through LDS in chunks of KC contraction values (8 f64, 16
// f32 or 32 bf16 = four 16-byte quads per row): direct global->LDS loads
// (global_load_lds_dwordx4) fetch chunk j + NBUF - 1 while the waves run
// chunk j; the workgroup waits for its own loads of chunk j+1 and
// synchronises once per chunk.  The loads run ahead of the passes: a Loader
// walks the item's chunk sequence by itself.
//
// Code size: the passes are loops over L and the lone hole, not unrolled, so
// the FP64 energy kernel is 51 KB of instructions.  With all 18 passes
// unrolled it was 84 KB, more than the 64 KB instruction cache two CUs share,
// and every item ran from L2.
//
// Together (ms before / after): no=40/nv=160 FP64 635 / 460, no=21/nv=160 in
// ragged tiles 149 / 79, no=26/nv=114 in spin-labelled ragged tiles 17.7 /
// 5.6, no=40/nv=320 in 2 spins x 4 irreps (tiles of 5 holes) 446 / 186,
// bf16x6 no=40/nv=200 530 / 450.
//
// LDS layout of one buffer part (hi or lo; quads, kq = quad 0..3 of a row):
//   X  [4 s][8 L slots][4 r][4 kq ^ x_swz]         512 quads
//   Y  [4 h][8 p1 slots][8 p2 slots][4 kq ^ y_swz] 1024 quads
// Fragment reads (16 lanes of one kq: 4 row/col slots x 4 inner indices)
// touch 16 distinct 4-bank groups; each load instruction writes 64
// consecutive quads and 4 consecutive lanes read one 64-byte row segment.
#include <type_traits>

#include "fused.h"
#include "handover.h"

namespace tce_t {
namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef double d4 __attribute__((ext_vector_type(4)));
typedef double dv2 __attribute__((ext_vector_type(2)));

template <int PREC>
struct Prec;
template <>
struct Prec<TCE_T_FP64> {
  static constexpr int KC = 8;     // contraction values per chunk
  static constexpr int NPART = 1;  // operand parts
  static constexpr int ES = 8;     // bytes per element
  static constexpr int NW = 4;     // waves of a workgroup
  // LDS chunk buffers (24 KB each), chunks loaded NBUF - 1 ahead
  static constexpr int NBUF = 3;
  typedef double acc;
  typedef d4 quad;
};
template <>
struct Prec<TCE_T_FP32> {
  static constexpr int KC = 16;
  static constexpr int NPART = 1;
  static constexpr int ES = 4;
  static constexpr int NW = 4;
  static constexpr int NBUF = 3;
  typedef float acc;
  typedef f4 quad;
};
template <>
struct Prec<TCE_T_BF16X3> {
  static constexpr int KC = 32;
  static constexpr int NPART = 2;  // hi, lo
  static constexpr int ES = 2;
  static constexpr int NW = 8;
  static constexpr int NBUF = 3;
  typedef float acc;
  typedef f4 quad;
};
template <>
struct Prec<TCE_T_BF16X6> {
  static constexpr int KC = 32;
  static constexpr int NPART = 3;  // hi, mid, lo
  static constexpr int ES = 2;
  static constexpr int NW = 8;
  static constexpr int NBUF = 2;   // 3 x 72 KB do not fit the 160 KB of LDS
  typedef float acc;
  typedef f4 quad;
};

constexpr int X_QUADS = 512, Y_QUADS = 1024, PART_QUADS = X_QUADS + Y_QUADS;

// Epilogue staging (doubles), overlaying the chunk buffers after the last
// chunk:
//   S   [hole pair t: (j,k) (i,k) (i,j)][16 pairs u*4+v]
//       [particle pair s: (b,c) (a,c) (a,b)][8 x 8 slots]           9216
//   T1  [particle box a b c][hole box i j k][8 slots][4 holes]        288
constexpr int EPI_S = 3 * 16 * 3 * 64;
constexpr int EPI_T1 = 9 * 32;
constexpr int EPI_QUADS = (EPI_S + EPI_T1) / 2;

template <int PREC>
constexpr int buf_quads() {
  return Prec<PREC>::NPART * PART_QUADS;
}
template <int PREC>
constexpr int lds_quads() {
  constexpr int nb = Prec<PREC>::NBUF;
  return nb * buf_quads<PREC>() > EPI_QUADS ? nb * buf_quads<PREC>() : EPI_QUADS;
}

// Tables the kernel only reads (segments, arguments, tasks), in the constant
// address space: loads from it at uniform addresses are scalar loads, which
// do not wait on (or drain) the chunk loads in flight.
template <class T>
using cptr = const __attribute__((address_space(4))) T *;

// Values the compiler cannot know to be the same in every lane.
__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ long uniform(long x) {
  const unsigned lo = (unsigned)uniform((int)x), hi = (unsigned)uniform((int)(x >> 32));
  return (long)(((unsigned long)hi << 32) | lo);
}

// The lane index again, as a value the compiler cannot see through: what is
// computed from it is computed here and not kept in registers across the item
// loop.  (Kept, it was spilled, and the waits of the reloads drain the chunk
// loads in flight.)
__device__ __forceinline__ int again(int lane) {
  asm volatile("" : "+v"(lane));
  return lane;
}

// Hole box of an item: global hole o + min(b0 + u, rm), u = 0..3; n valid.
struct HoleBox {
  int o, b0, rm, n;
};
__device__ __forceinline__ int hole(const HoleBox &h, int u) { return h.o + min(h.b0 + u, h.rm); }
// Particle range of the workgroup's box: global index g0 + min(slot, sm), slot =
// 0..7 (0..3 of c in a half item); wave bit `bit` holds the wave's cube
// coordinate along it.
struct PRange {
  int g0, sm, bit;
};
__device__ __forceinline__ int particle(const PRange &p, int slot) { return p.g0 + min(slot, p.sm); }
struct ItemGeo {
  HoleBox I, J, K;
  PRange a, b, c;
  int heq;  // EQ_IJ, EQ_JK of the item
  // Whether the pair (u, w) of hole boxes t (0: (j,k), 1: (i,k), 2: (i,j)) has
  // elements that count: inside the boxes, and u < w when the two are one box
  // (the rest follow by antisymmetry, distinct() of them alike).  The epilogue
  // of an item with I == J == K forms 4 elements of a particle triple, not 64:
  // no=8/nv=32 153 us before, 134 after; no=40/nv=160 472 and 462 ms.
  __device__ __forceinline__ bool pair(int t, int u, int w) const {
    const int n1 = t == 0 ? J.n : I.n, n2 = t == 2 ? J.n : K.n;
    const int m = t == 0 ? EQ_JK : (t == 2 ? EQ_IJ : EQ_IJ | EQ_JK);
    return u < n1 && w < n2 && !((heq & m) == m && u >= w);
  }
  __device__ __forceinline__ double distinct() const {
    return heq == 0 ? 1.0 : (heq == (EQ_IJ | EQ_JK) ? 6.0 : 2.0);
  }
};
// Chosen field by field: a choice between the structs themselves would put G
// in scratch memory.
__device__ __forceinline__ HoleBox hole_box(const ItemGeo &G, int t) {
  auto pick = [t](int x, int y, int z) { return t == 0 ? x : (t == 1 ? y : z); };
  return HoleBox{pick(G.I.o, G.J.o, G.K.o), pick(G.I.b0, G.J.b0, G.K.b0),
                 pick(G.I.rm, G.J.rm, G.K.rm), pick(G.I.n, G.J.n, G.K.n)};
}
__device__ __forceinline__ PRange prange(const ItemGeo &G, int t) {
  auto pick = [t](int x, int y, int z) { return t == 0 ? x : (t == 1 ? y : z); };
  return PRange{pick(G.a.g0, G.b.g0, G.c.g0), pick(G.a.sm, G.b.sm, G.c.sm),
                pick(G.a.bit, G.b.bit, G.c.bit)};
}
// Slots of the second particle p2 of the pair beside lone particle L.
template <int PREC>
__device__ __forceinline__ int p2_slots(int L) {
  return Prec<PREC>::NW == 4 && L != 2 ? 4 : 8;
}
// A wave's cube coordinate along a particle range.
__device__ __forceinline__ int cube(int wave, const PRange &p) { return (wave >> p.bit) & 1; }

// Which passes an item runs.  hact / lact: bit h / L set when the passes of
// lone hole h / lone particle L run; s0 of lone hole h: 1 when the hole pair
// beside it is one box (its passes form the pairs r < s only).
struct ItemPlan {
  int eq;          // the item's equal boxes
  int hact, lact;
  __device__ __forceinline__ int s0(int h) const {
    return (h == 2 && (eq & EQ_IJ)) || (h == 0 && (eq & EQ_JK)) ? 1 : 0;
  }
};
// half: a half item holds one c half, whose exchange with a or b needs the
// other, so three equal particle boxes run as two there (the host's one-box
// tasks put a pair of equal boxes on a and b).
__device__ __forceinline__ ItemPlan item_plan(int eq, bool half) {
  ItemPlan P;
  if (half && (eq & EQ_AB)) eq &= ~EQ_BC;
  P.eq = eq;
  const bool ij = eq & EQ_IJ, jk = eq & EQ_JK, ab = eq & EQ_AB, bc = eq & EQ_BC;  // bc: all three
  P.hact = ij ? (jk ? 4 : 6) : (jk ? 3 : 7);  // k | j, k | i, j | all
  P.lact = ab ? (bc ? 4 : 6) : 7;             // c | b, c | all
  return P;
}

// Quad swizzles of the operand rows: LDS position k of a row holds the row's
// global quad k ^ swz, for both the loads (which write each row linearly)
// and the fragment reads.  Measured with gfx950's SQ_LDS_BANK_CONFLICT over
// every swizzle that is linear in the row bits: a ds_read_b128 whose 16
// lanes of one kq read rows (slot or p1 from lane bits 2-3, r or p2 from
// bits 0-1) is conflict-free with s(row) = -(slot & 3) mod 4 (FP32 and bf16
// X reads, every Y read), while (slot & 3) ^ (r & 2) took two passes (4
// conflict cycles per read).  The FP64 X reads put slot on lane bits 0-1 and
// r on bits 2-3, for which (slot & 3) ^ (r & 2) is conflict-free.
template <int PREC>
__device__ __forceinline__ int x_swz(int slot, int r) {
  return PREC == TCE_T_FP64 ? (slot & 3) ^ (r & 2) : (4 - (slot & 3)) & 3;
}
__device__ __forceinline__ int y_swz(int p1) { return (4 - (p1 & 3)) & 3; }

// Direct global->LDS load of 16 bytes per lane: lane l writes LDS bytes
// [m0 + 16 l, m0 + 16 l + 16) from base + off.  Issued by inline assembly so
// that the compiler does not tie later LDS reads of other buffers to it; the
// kernel waits for these loads itself (vmcnt) before the barrier that publishes
// a buffer.  Scalar base and LDS address: a load takes no VALU instruction.
__device__ __forceinline__ void lds_load16(const char *base, unsigned off, unsigned lds_byte) {
  asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds_byte), "v"(off),
               "s"(base)
               : "memory");
}
// s_waitcnt vmcnt(N) with the other counters left alone (gfx9 encoding).
template <int N>
__device__ __forceinline__ void wait_vm() {
  __builtin_amdgcn_s_waitcnt((N & 15) | ((N >> 4) << 14) | (7 << 4) | (15 << 8));
}
// The same for a uniform n in 0..6 (a wave's loads of one chunk; 6 terms: up to
// 9, waited for in full).
__device__ __forceinline__ void wait_vm_n(int n) {
  switch (n) {
    case 6: wait_vm<6>(); break;
    case 5: wait_vm<5>(); break;
    case 4: wait_vm<4>(); break;
    case 3: wait_vm<3>(); break;
    case 2: wait_vm<2>(); break;
    case 1: wait_vm<1>(); break;
    default: wait_vm<0>();
  }
}
__device__ __forceinline__ void block_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// Chunks [c0, c0 + n) that cover contraction range p of a task (fused.h,
// MIXED_PASS): every operand outside it is zero.
template <int PREC>
__device__ __forceinline__ int2 chunks_of(cptr<TaskDev> T, int p) {
  constexpr int KC = Prec<PREC>::KC;
  const unsigned x = T->x[p];
  const int x0 = (int)(x & 0xffffu), x1 = (int)(x >> 16);
  const int c0 = x0 / KC;
  return make_int2(c0, x1 > x0 ? (x1 + KC - 1) / KC - c0 : 0);
}

// The loads of an item's chunk sequence: segments p = 6 L + 2 {j, i, k} +
// {d2, d1} of MIXED_PASS with act's bit set, in order.  A wave loads the X
// blocks of s-index g (64 quads, 4 L slots each) and the Y blocks of h-index g
// (64 quads, 16 particle pairs each), per operand part: with 8 waves g = wave
// >> 1 and the waves of a pair take half of the L slots and p1 slots each, with
// 4 waves g = wave.  Blocks whose rows no quad of the pass reads are skipped
// (nl = loads per chunk of this wave).
template <int PREC>
struct Loader {
  using Pr = Prec<PREC>;
  static constexpr bool HALF = Pr::NW == 4;
  static constexpr int NX = HALF ? 2 : 1, NY = HALF ? 4 : 2;
  // The lane's rows relative to the first one of the box (bytes; 32 bits hold
  // them in any tensor that fits the memory: three occupied indices of X,
  // eight virtual ones of Y) and the tensors at that row and the next chunk.
  unsigned xo[NX], yo[NY];
  const char *xb[Pr::NPART], *yb[Pr::NPART];
  unsigned act;
  int p, left;  // segment (-1: none yet) and its chunks not yet loaded
  unsigned on;  // bits 0..: X blocks loaded; bits 8..: Y blocks
  int nl;
  int no, nv;         // extents of the job
  unsigned rowe, rowm;  // bytes of a d2 and a d1 row

  __device__ __forceinline__ void init(cptr<MixedArgs> A) {
    p = -1;
    left = 0;
    no = A->f.no, nv = A->f.nv;
    rowe = (unsigned)(A->Ek * Pr::ES), rowm = (unsigned)(A->Mk * Pr::ES);
  }
  __device__ __forceinline__ void next_segment(cptr<MixedArgs> A, cptr<TaskDev> T,
                                               const ItemGeo &G, const ItemPlan &P, int wave,
                                               int lane_) {
    constexpr int QB = 16;  // bytes per quad
    const int lane = again(lane_);
    p = __builtin_ctz(act & (~0u << (p + 1)));
    const int L = p / 6, hi = (p >> 1) % 3, kind = p & 1;
    const int h = hi == 0 ? 1 : (hi == 1 ? 0 : 2);
    const HoleBox R = hole_box(G, h == 0 ? 1 : 0), S = hole_box(G, h == 2 ? 1 : 2),
                  H = hole_box(G, h);
    const PRange PL = prange(G, L), P1 = prange(G, L == 0 ? 1 : 0), P2 = prange(G, L == 2 ? 1 : 2);
    const int2 ch = chunks_of<PREC>(T, p);
    left = ch.y;
    const unsigned row = kind ? rowm : rowe;
    const int g = HALF ? wave : wave >> 1;
    const int r0 = hole(R, 0), hs = hole(S, g), hy = hole(H, g);
    const unsigned k0 = (unsigned)(ch.x * Pr::KC * Pr::ES);
    const long x0 = (long)(unsigned)((r0 * no + hs) * nv + PL.g0) * row + k0,
               y0 = (long)(unsigned)((hy * nv + P1.g0) * nv + P2.g0) * row + k0;
#pragma unroll
    for (int part = 0; part < Pr::NPART; ++part) {
      xb[part] = (const char *)(kind ? A->x1[part] : A->x2[part]) + x0;
      yb[part] = (const char *)(kind ? A->y1[part] : A->y2[part]) + y0;
    }
    on = 0;
    nl = 0;
    const int xr = (lane >> 2) & 3, kq = lane & 3;
    const unsigned xrow = (unsigned)((hole(R, xr) - r0) * no * nv);
#pragma unroll
    for (int u = 0; u < NX; ++u) {
      const int first = HALF ? 4 * u : 4 * (wave & 1), slot = first + (lane >> 4);
      if (g >= P.s0(h) && g < S.n && first <= PL.sm) on |= 1u << u, nl += Pr::NPART;
      xo[u] = (xrow + min(slot, PL.sm)) * row + (unsigned)(QB * (kq ^ x_swz<PREC>(slot, xr)));
    }
    const bool wide = p2_slots<PREC>(L) == 8;  // rows of 8 p2 slots: 2 p1 slots to a block
    const int p2 = min(wide ? (lane >> 2) & 7 : (lane >> 2) & 3, P2.sm);
#pragma unroll
    for (int t = 0; t < NY; ++t) {
      const int first = HALF ? (wide ? 2 * t : 4 * t) : 4 * (wave & 1) + 2 * t;
      const int s1 = first + (wide ? lane >> 5 : lane >> 4);
      if (g < H.n && first <= P1.sm && (wide || t < 2)) on |= 256u << t, nl += Pr::NPART;
      yo[t] = (unsigned)(min(s1, P1.sm) * nv + p2) * row + (unsigned)(QB * (kq ^ y_swz(s1)));
    }
  }
  // The loads of the next chunk into the buffer at LDS byte `base`; returns
  // their number.  (Spread over the chunk's MFMAs, one block after each row of
  // quads, they ran 1 to 2% slower than together.)
  __device__ __forceinline__ int load(cptr<MixedArgs> A, cptr<TaskDev> T, const ItemGeo &G,
                                      const ItemPlan &P, unsigned base, int wave, int lane) {
    if (left == 0) next_segment(A, T, G, P, wave, lane);
#pragma unroll
    for (int part = 0; part < Pr::NPART; ++part) {
      const unsigned b = base + part * PART_QUADS * 16u;
#pragma unroll
      for (int u = 0; u < NX; ++u)
        if (on >> u & 1) lds_load16(xb[part], xo[u], b + (NX * wave + u) * 1024u);
#pragma unroll
      for (int t = 0; t < NY; ++t)
        if (on >> (8 + t) & 1)
          lds_load16(yb[part], yo[t], b + X_QUADS * 16u + (NY * wave + t) * 1024u);
      xb[part] += Pr::KC * Pr::ES;
      yb[part] += Pr::KC * Pr::ES;
    }
    --left;
    return nl;
  }
};

// Operand fragments of one chunk in registers: X quads s = 0..3 and Y quads
// h = 0..3 of this lane, per part.
template <int PREC>
struct Frag {
  typedef bf8 vec;
  vec x[Prec<PREC>::NPART][4], y[Prec<PREC>::NPART][4];
};
template <>
struct Frag<TCE_T_FP64> {
  typedef dv2 vec;
  vec x[1][4], y[1][4];
};
template <>
struct Frag<TCE_T_FP32> {
  typedef f4 vec;
  vec x[1][4], y[1][4];
};

// X quad s (offset xa for s = 0, s adds 128 quads) and Y quad h (offset yb
// for h = 0, h adds 256) of the chunk in buffer cb.
template <int PREC>
__device__ __forceinline__ void read_x(Frag<PREC> &F, const f4 *cb, int xa, int s) {
#pragma unroll
  for (int part = 0; part < Prec<PREC>::NPART; ++part)
    F.x[part][s] =
        reinterpret_cast<const typename Frag<PREC>::vec *>(cb)[part * PART_QUADS + xa + 128 * s];
}
template <int PREC>
__device__ __forceinline__ void read_y(Frag<PREC> &F, const f4 *cb, int yb, int h) {
#pragma unroll
  for (int part = 0; part < Prec<PREC>::NPART; ++part)
    F.y[part][h] = reinterpret_cast<const typename Frag<PREC>::vec *>(
        cb)[part * PART_QUADS + X_QUADS + yb + 256 * h];
}

// Accumulator quad of MFMA quad (s, h): lone hole k (KP) has s = j, h = k;
// lone hole j, and i on the transposed quads, s = k, h = j or i.
template <bool KP>
__device__ __forceinline__ constexpr int qi(int s, int h) {
  return KP ? 4 * s + h : 4 * h + s;
}

// Term t of the MFMAs of one quad: 2 halves of the chunk (FP64), 4 quarters
// (FP32), or the 3 / 6 products of the split operands, smallest first
// (lo*hi, hi*lo, hi*hi; lo*hi, hi*lo, mid*mid, mid*hi, hi*mid, hi*hi).
template <int PREC>
constexpr int terms() {
  return PREC == TCE_T_FP64 ? 2 : (PREC == TCE_T_FP32 ? 4 : (PREC == TCE_T_BF16X3 ? 3 : 6));
}
template <int PREC>
__device__ __forceinline__ typename Prec<PREC>::quad mma(const Frag<PREC> &F, int s, int h, int t,
                                                         typename Prec<PREC>::quad c) {
  if constexpr (PREC == TCE_T_FP64) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(F.x[0][s][t], F.y[0][h][t], c, 0, 0, 0);
  } else if constexpr (PREC == TCE_T_FP32) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(F.x[0][s][t], F.y[0][h][t], c, 0, 0, 0);
  } else if constexpr (PREC == TCE_T_BF16X3) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(F.x[t == 0 ? 1 : 0][s], F.y[t == 1 ? 1 : 0][h],
                                                   c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(
        F.x[t == 0 ? 2 : ((t == 2 || t == 3) ? 1 : 0)][s],
        F.y[t == 1 ? 2 : ((t == 2 || t == 4) ? 1 : 0)][h], c, 0, 0, 0);
  }
}

// This lane's fragment offsets for lone particle L: X quad (s = 0), Y quad
// (h = 0).  X row (lane & 15) = 4L' + r (L' = hi, r = lo), quad kq.  The f64
// MFMA writes row i to lane group i % 4, register i / 4 (the f32 and bf16
// ones to group i / 4, register i % 4), so for FP64 the rows are ordered 4r +
// L' instead: either way the result lands at lane 16L' + col, component r.
// Y col (lane & 15) = 4p1' + p2' (p1' = hi, p2' = lo).
template <int PREC>
__device__ __forceinline__ int2 frag_offsets(const ItemGeo &G, int L, int wave, int lane) {
  const int kq = lane >> 4, hi = (lane & 15) >> 2, lo = lane & 3;
  const int xL = PREC == TCE_T_FP64 ? lo : hi, xr = PREC == TCE_T_FP64 ? hi : lo;
  const int slot = 4 * cube(wave, prange(G, L)) + xL;
  const int p1s = 4 * cube(wave, prange(G, L == 0 ? 1 : 0)) + hi,
            p2s = 4 * cube(wave, prange(G, L == 2 ? 1 : 2)) + lo;
  return make_int2((slot * 4 + xr) * 4 + (kq ^ x_swz<PREC>(slot, xr)),
                   (p1s * p2_slots<PREC>(L) + p2s) * 4 + (kq ^ y_swz(p1s)));
}

__device__ __forceinline__ float bperm(float v, int src) {
  return __int_as_float(__builtin_amdgcn_ds_bpermute(src << 2, __float_as_int(v)));
}
__device__ __forceinline__ double bperm(double v, int src) { return perm_lane(v, src); }

template <class Q>
__device__ __forceinline__ void permute_lanes(Q (&q)[16], int src) {
#pragma unroll
  for (int n = 0; n < 16; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) q[n][r] = bperm(q[n][r], src);
}
template <class Q>
__device__ __forceinline__ void negate(Q (&q)[16]) {
#pragma unroll
  for (int n = 0; n < 16; ++n) q[n] = -q[n];
}
// q[4j + k][i] <-> q[4i + k][j]
template <class Q>
__device__ __forceinline__ void transpose_ij(Q (&q)[16]) {
#pragma unroll
  for (int k = 0; k < 4; ++k)
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < i; ++j) {
        const auto t = q[4 * j + k][i];
        q[4 * j + k][i] = q[4 * i + k][j];
        q[4 * i + k][j] = t;
      }
}
// Scales every accumulator, or (PAIR) those of the pairs (r, s), r and s >= 1:
// q[4 s + .][r] (KP) or q[. + s][r].
template <bool PAIR, bool KP, class Q, class T>
__device__ __forceinline__ void scale(Q (&q)[16], T f) {
#pragma unroll
  for (int n = 0; n < 16; ++n) {
    if (PAIR && (KP ? n >> 2 : n & 3) == 0) continue;
#pragma unroll
    for (int r = PAIR ? 1 : 0; r < 4; ++r) q[n][r] *= f;
  }
}

// What the chunk loops carry along.
template <int PREC>
struct Stream {
  Loader<PREC> ld;
  int todo;   // chunks of the item not yet loaded
  int ready;  // chunks not yet contracted
  int buf;    // buffer of the next chunk to contract
};

// The chunks of one (L, h): X quads s0..s1-1 and Y quads 0..h1-1 (none in a
// wave whose cube is past the edge, s1 = 0).  Per chunk j the fragments are
// read and the MFMAs run, with the loads of chunk j+NBUF-1 (into the buffer
// freed by the last barrier) issued among them; then this thread's loads of
// chunk j+1 complete and the barrier publishes it.  With two buffers (6 terms)
// chunk j+2 goes into this chunk's buffer after the barrier, with the whole
// of chunk j+1 to land.
template <int PREC, bool KP>
__device__ __forceinline__ void chunk_loop(typename Prec<PREC>::quad (&q)[16], const f4 *lds,
                                           unsigned lds_base, cptr<MixedArgs> A, cptr<TaskDev> T,
                                           const ItemGeo &G, const ItemPlan &P, int wave, int lane,
                                           int L, int nch, int s0, int s1, int h1,
                                           Stream<PREC> &st) {
  using Pr = Prec<PREC>;
  constexpr int NB = Pr::NBUF, AH = NB - 1;
  const int2 o = frag_offsets<PREC>(G, L, wave, again(lane));
#pragma unroll 1
  for (int c = 0; c < nch; ++c) {
    Frag<PREC> f;
    const f4 *cb = lds + st.buf * buf_quads<PREC>();
    int nl = 0;
    const int nb = st.buf + AH < NB ? st.buf + AH : st.buf + AH - NB;
    const unsigned nbase = lds_base + (unsigned)nb * (buf_quads<PREC>() * 16u);
    const bool more = st.todo > 0;
    // the MFMAs of X quad s with Y quads 0..h1-1; all four term by term, so that
    // dependent MFMAs on one quad are 4 instructions apart
    auto quad = [&](int s, int h) {
#pragma unroll
      for (int t = 0; t < terms<PREC>(); ++t)
        q[qi<KP>(s, h)] = mma<PREC>(f, s, h, t, q[qi<KP>(s, h)]);
    };
    // The masks are nested, so that a short row leaves at its first absent quad
    // and a full one takes one branch: tested quad by quad, the 16 tests of a
    // chunk made no=40/nv=160 484 ms instead of 472, and 201 instead of 189 in
    // tiles of 5 holes (no=40/nv=320 in irreps, one quad to a row in most items).
    auto row = [&](int s) {
      if (h1 == 4) {
#pragma unroll
        for (int t = 0; t < terms<PREC>(); ++t)
#pragma unroll
          for (int h = 0; h < 4; ++h) q[qi<KP>(s, h)] = mma<PREC>(f, s, h, t, q[qi<KP>(s, h)]);
      } else {
        quad(s, 0);
        if (h1 > 1) {
          quad(s, 1);
          if (h1 > 2) quad(s, 2);
        }
      }
    };
    if (s1 > 0) {
#pragma unroll
      for (int h = 0; h < 4; ++h) read_y<PREC>(f, cb, o.y, h);
#pragma unroll
      for (int s = 0; s < 4; ++s) read_x<PREC>(f, cb, o.x, s);
      if (s0 == 0) row(0);
      if (s1 > 1) row(1);
    }
    if (NB >= 3 && more) {
      nl = st.ld.load(A, T, G, P, nbase, wave, lane);
      --st.todo;
    }
    if (s1 > 2) {
      row(2);
      if (s1 > 3) row(3);
    }
    // chunk j+1 landed once at most the loads of the later ones are pending
    if constexpr (NB == 3) wait_vm_n(nl);
    else wait_vm<0>();
    block_barrier();
    if constexpr (NB == 2) {
      if (more) {
        st.ld.load(A, T, G, P, lds_base + (unsigned)st.buf * (buf_quads<PREC>() * 16u), wave, lane);
        --st.todo;
      }
    }
    st.buf = st.buf + 1 < NB ? st.buf + 1 : 0;
  }
}

// Subtracts the partner elements from the accumulators: q - q(a <-> b), or with
// three equal boxes q - q(a <-> c) - q(b <-> c).  Through LDS in rounds of 64 KB.
// A half item has equal boxes a and b only.  Layout c: lane = 4a' + b' + 16c'.
template <int PREC>
__device__ __forceinline__ void exchange_particles(typename Prec<PREC>::quad (&q)[16], f4 *lds,
                                                   const ItemGeo &G, int eq, int wave, int lane_) {
  const int lane = again(lane_);
  constexpr int U = sizeof(typename Prec<PREC>::quad) / 16;  // 16-byte units per quad
  constexpr int NQ = 64 / Prec<PREC>::NW / U;                 // quads per round
  const int a = (lane & 15) >> 2, b = lane & 3, c = lane >> 4;
  const int ca = cube(wave, G.a), cb = cube(wave, G.b), cc = cube(wave, G.c);
  auto from = [&](int x, int y, int z) { return (x << G.a.bit) | (y << G.b.bit) | (z << G.c.bit); };
  const bool all = eq & EQ_BC;
  int w1, l1, w2 = 0, l2 = 0;
  if (all) {
    w1 = from(ca, cc, cb), l1 = 4 * a + c + 16 * b;
    w2 = from(cc, cb, ca), l2 = 4 * c + b + 16 * a;
  } else {
    w1 = from(cb, ca, cc), l1 = 4 * b + a + 16 * c;
  }
#pragma unroll
  for (int r0 = 0; r0 < 16; r0 += NQ) {
#pragma unroll
    for (int n = 0; n < NQ; ++n) {
      const f4 *v = reinterpret_cast<const f4 *>(&q[r0 + n]);
#pragma unroll
      for (int u = 0; u < U; ++u) lds[((wave * NQ + n) * U + u) * 64 + lane] = v[u];
    }
    __syncthreads();
    auto take = [&](int w, int l) {
#pragma unroll
      for (int n = 0; n < NQ; ++n) {
        f4 v[U];
#pragma unroll
        for (int u = 0; u < U; ++u) v[u] = lds[((w * NQ + n) * U + u) * 64 + l];
        q[r0 + n] -= *reinterpret_cast<const typename Prec<PREC>::quad *>(v);
      }
    };
    take(w1, l1);
    if (all) take(w2, l2);
    __syncthreads();
  }
}

// The same for equal hole boxes, in registers (q[4j + k][i]).  All equal: the
// accumulators hold the lone-hole-k passes of the pairs i < j, and t(i < j <
// k) = P(i,j;k) - P(i,k;j) + P(j,k;i).
template <class Q>
__device__ __forceinline__ void exchange_holes(Q (&q)[16], int eq) {
  if ((eq & EQ_IJ) && (eq & EQ_JK)) {
    auto e = [&](int i, int j, int k) { return q[4 * j + k][i]; };
    const auto t012 = e(0, 1, 2) - e(0, 2, 1) + e(1, 2, 0), t013 = e(0, 1, 3) - e(0, 3, 1) + e(1, 3, 0),
               t023 = e(0, 2, 3) - e(0, 3, 2) + e(2, 3, 0), t123 = e(1, 2, 3) - e(1, 3, 2) + e(2, 3, 1);
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int k = 0; k < 4; ++k) {
          const int m = 6 - i - j - k;  // the index left out
          const auto t = m == 3 ? t012 : (m == 2 ? t013 : (m == 1 ? t023 : t123));
          const bool odd = ((i > j) + (i > k) + (j > k)) & 1;
          q[4 * j + k][i] = (i == j || j == k || i == k) ? 0 : (odd ? -t : t);
        }
  } else if (eq & EQ_IJ) {
#pragma unroll
    for (int k = 0; k < 4; ++k)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[4 * i + k][i] = 0;
#pragma unroll
        for (int j = i + 1; j < 4; ++j) {
          const auto t = q[4 * j + k][i] - q[4 * i + k][j];
          q[4 * j + k][i] = t;
          q[4 * i + k][j] = -t;
        }
      }
  } else if (eq & EQ_JK) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      q[5 * j] = Q{0, 0, 0, 0};
#pragma unroll
      for (int k = j + 1; k < 4; ++k) {
        const Q t = q[4 * j + k] - q[4 * k + j];
        q[4 * j + k] = t;
        q[4 * k + j] = -t;
      }
    }
  }
}

// The t3 doubles of one item: lane 4a' + b' + 16c', element (i, j, k) of the
// hole box at q[4j + k][i].  Ends with the chunk buffers free and no load in
// flight.
template <int PREC>
__device__ __forceinline__ void contract(typename Prec<PREC>::quad (&q)[16], f4 *lds,
                                         unsigned lds_base, cptr<MixedArgs> A, cptr<TaskDev> T,
                                         const ItemGeo &G, const ItemPlan &P, int wave, int lane) {
  using Pr = Prec<PREC>;
  using acc = typename Pr::acc;
#pragma unroll
  for (int n = 0; n < 16; ++n) q[n] = typename Pr::quad{0, 0, 0, 0};
  Stream<PREC> st;
  st.ld.act = 0;
  st.todo = 0;
#pragma unroll
  for (int p = 0; p < 18; ++p) {
    const int n = chunks_of<PREC>(T, p).y;
    const bool on = (P.lact >> MIXED_PASS[p].L & 1) && (P.hact >> MIXED_PASS[p].h & 1) && n > 0;
    st.ld.act |= on ? 1u << p : 0u;
    st.todo += on ? n : 0;
  }
  st.ld.init(A);
  st.buf = 0;
  {  // the first two chunks; the first one landed
    int last = 0;
#pragma unroll 1
    for (int k = 0; k < 2; ++k) {
      last = 0;
      if (st.todo > 0) {
        last = st.ld.load(A, T, G, P, lds_base + (unsigned)k * (buf_quads<PREC>() * 16u), wave, lane);
        --st.todo;
      }
    }
    wait_vm_n(last);
    block_barrier();
  }
  const bool live = 4 * cube(wave, G.a) <= G.a.sm && 4 * cube(wave, G.b) <= G.b.sm &&
                    4 * cube(wave, G.c) <= G.c.sm;
  const bool all_h = (P.eq & EQ_IJ) && (P.eq & EQ_JK);
  int lay = -1;      // lone particle of the lane layout
  bool neg = false;  // the accumulators hold -t3
  auto run = [&](auto kp, int L, int h, int hi_) {
    constexpr bool KP = decltype(kp)::value;
    const int p = 6 * L + 2 * hi_;
    const int nch = ((st.ld.act >> p & 1) ? chunks_of<PREC>(T, p).y : 0) +
                    ((st.ld.act >> (p + 1) & 1) ? chunks_of<PREC>(T, p + 1).y : 0);
    if (nch == 0) return;
    const bool minus = MIXED_MINUS >> (3 * L + hi_) & 1;
    if (minus != neg) negate(q), neg = minus;
    const int s0 = P.s0(h), s1 = live ? hole_box(G, h == 2 ? 1 : 2).n : 0, h1 = hole_box(G, h).n;
    const bool pair = s0 && !all_h;
    if (pair) scale<true, KP>(q, (acc)2);
    chunk_loop<PREC, KP>(q, lds, lds_base, A, T, G, P, wave, lane, L, nch, s0, s1, h1, st);
    if (pair) scale<true, KP>(q, (acc)0.5);
  };
#pragma unroll 1
  for (int L = 0; L < 3; ++L) {
    if (!(P.lact >> L & 1)) continue;
    if (lay >= 0) {
      // a -> b: lane (4b'+c') + 16a' -> (4a'+c') + 16b'; b -> c: (4a'+c') +
      // 16b' -> (4a'+b') + 16c'
      const int ln = again(lane), kq = ln >> 4, hi = (ln & 15) >> 2, lo = ln & 3;
      const int src = L == 1 ? 4 * kq + lo + 16 * hi : 4 * hi + kq + 16 * lo;
      permute_lanes(q, src);
    }
    // the passes of a lone particle beside a pair of equal boxes count half:
    // the exchange at the end adds their image (three equal boxes: c alone runs,
    // and counts whole)
    const bool half = (P.eq & EQ_BC) ? (L == 0) : ((P.eq & EQ_AB) && L == 2);
    if (half) scale<false, false>(q, (acc)2);
    // lone hole j, then i on the transposed quads
    const bool do_i = P.hact & 1;
#pragma unroll 1
    for (int hh = 0; hh < 2; ++hh) {
      if (P.hact >> (1 - hh) & 1) run(std::false_type(), L, 1 - hh, hh);
      if (do_i) transpose_ij(q);
    }
    if (P.hact & 4) run(std::true_type(), L, 2, 2);
    if (half) scale<false, false>(q, (acc)0.5);
    lay = L;
  }
  if (neg) negate(q);
  if (P.eq & (EQ_IJ | EQ_JK)) exchange_holes(q, P.eq);
  if (P.eq & (EQ_AB | EQ_BC)) exchange_particles<PREC>(q, lds, G, P.eq, wave, lane);
}

// Stage the item's singles operands into LDS (FP64, as fused_wg.hip): 64 S
// values of one hole pair per wave and load; the pairs past a ragged edge of
// the hole boxes are left out.
// Of the pairs (h, h') and (p, p') of an item: S[h][h'][p][p'] with rows of ld
// elements, and T1 with element (p, h) at p * ldp + h * ldh.
template <int NW>
__device__ __forceinline__ void stage_epilogue(double *e, gptr<const double> S, int ld,
                                               gptr<const double> T1, int ldp, int ldh, int no,
                                               int nv, int wave, int lane_, const ItemGeo &G) {
  const int lane = again(lane_);
  // step 0, 1, 2: particle pair (b,c), (a,c), (a,b), 8 x 8 slots; a half item:
  // (b,c) and (a,c) with 4 c slots in one step, then (a,b)
  constexpr int STEPS = NW == 4 ? 2 : 3, R = 48 / NW;
#pragma unroll
  for (int step = 0; step < STEPS; ++step) {
    const bool both = NW == 4 && step == 0;
    const int sp = both ? lane >> 5 : (NW == 4 ? 2 : step);
    const int p1 = both ? (lane >> 2) & 7 : lane >> 3, p2 = both ? lane & 3 : lane & 7;
    const int ga = particle(G.a, p1), gb = particle(G.b, p1);
    const int g1 = sp == 0 ? gb : ga, g2 = particle(prange(G, step == STEPS - 1 ? 1 : 2), p2);
    double v[R];
    // wave w: hole pairs tp = w, w + NW, ..
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int tp = wave + NW * r, t = (NW * r) >> 4, u = (tp >> 2) & 3, w = tp & 3;
      const HoleBox H1 = hole_box(G, t == 0 ? 1 : 0), H2 = hole_box(G, t == 2 ? 1 : 2);
      v[r] = 0.0;
      if (G.pair(t, u, w))
        v[r] = S[(unsigned long)(unsigned)((hole(H1, u) * no + hole(H2, w)) * nv + g1) * ld + g2];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) e[((wave + NW * r) * 3 + sp) * 64 + p1 * 8 + p2] = v[r];
  }
  for (int x = wave * 64 + lane; x < EPI_T1; x += 64 * NW) {
    const int u = x & 3, slot = (x >> 2) & 7, pt = (x >> 5) / 3, ht = (x >> 5) % 3;
    const int p = pt == 0 ? particle(G.a, slot)
                          : (pt == 1 ? particle(G.b, slot) : particle(G.c, slot));
    const int h = ht == 0 ? hole(G.I, u) : (ht == 1 ? hole(G.J, u) : hole(G.K, u));
    e[EPI_S + x] = T1[p * ldp + h * ldh];
  }
}
// The singles operands of a job.
template <int NW>
__device__ __forceinline__ void stage_singles(double *e, cptr<FusedArgs> A, int wave, int lane,
                                              const ItemGeo &G) {
  stage_epilogue<NW>(e, (gptr<const double>)A->S, A->nv, (gptr<const double>)A->T1, A->no, 1, A->no,
                     A->nv, wave, lane, G);
}

// A lane's place in its item: particle slots in the box (sa, sb, sc), local
// particle indices in the task's tiles (la, lb, lc), first hole of the box in
// the tiles (i0, j0, k0).
struct Place {
  int sa, sb, sc, la, lb, lc, i0, j0, k0;
};
__device__ __forceinline__ bool inside(cptr<TaskDev> T, const Place &p) {
  return p.la < T->r4 && p.lb < T->r5 && p.lc < T->r6;
}
// D of the lane's elements: eh[0][i] + eh[1][j] + eh[2][k] + d0.
struct Denominator {
  double d0, eh[3][4];
};
__device__ __forceinline__ Denominator denominator(cptr<FusedArgs> A, const ItemGeo &G,
                                                   const Place &p) {
  const gptr<const double> evl = (gptr<const double>)A->evl;
  const int no = A->no;
  Denominator D;
  D.d0 = -(evl[no + particle(G.a, p.sa)] + evl[no + particle(G.b, p.sb)] +
           evl[no + particle(G.c, p.sc)]);
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    D.eh[0][u] = evl[hole(G.I, u)];
    D.eh[1][u] = evl[hole(G.J, u)];
    D.eh[2][u] = evl[hole(G.K, u)];
  }
  return D;
}

// Between the parts of an epilogue: no instruction moves across, so that the
// arrays of one part are dead before those of the next are live.
__device__ __forceinline__ void phase() { __builtin_amdgcn_sched_barrier(0); }

// v[r] = f(i, j, k, r), r = 16 i + 4 j + k, over the lane's elements, 0 in the
// hole pairs (j, k) without an element that counts.
template <class F>
__device__ __forceinline__ void each_element(const ItemGeo &G, double (&v)[64], F &&f) {
#pragma unroll
  for (int jj = 0; jj < 4; ++jj)
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
#pragma unroll
      for (int ii = 0; ii < 4; ++ii) v[16 * ii + 4 * jj + kk] = 0.0;
      if (G.pair(0, jj, kk))
#pragma unroll
        for (int ii = 0; ii < 4; ++ii)
          v[16 * ii + 4 * jj + kk] = f(ii, jj, kk, 16 * ii + 4 * jj + kk);
    }
}

// Between the two halves of an item the wave's left-hand values wait in its
// slot of a spill buffer, element r = 16 i + 4 j + k of the lane at [r * 64 +
// lane]; CR: the doubles so, as FP32 where the accumulators are (their exact
// values), the singles behind them.  A slot belongs to a workgroup, not to an
// item: 64 MB for 256 workgroups, CR 128 MB in FP64 and 96 MB in the other modes.
// One slot per item of a window of up to 16 GB, written by a launch over the
// left-hand job and read by one over the right-hand job, cost the allocation of
// the window on each call (45 to 300 ms for the call at no=20/nv=80, 53 ms at
// no=16/nv=72, of which the kernels took 45 and 7.7 ms) and two passes over it
// in HBM.
// What the slots cost is not their own time but the operands they push out of
// the caches: with 64-bit doubles a CR item's bf16x3 contractions at no=40/nv=160
// took 258k clocks a side, 186k without the slot accesses (the FP64 mode's, 742k,
// change by 1%), with FP32 doubles they take 193k.  CR before / now (two launches
// over a window), s: bf16x3 no=40/nv=160 0.351 / 0.276 (0.333), no=40/nv=320 4.19 /
// 3.37 (3.60); bf16x6 0.486 / 0.422 (0.509) and 6.19 / 5.47 (5.97).  Accesses marked
// as streaming: 2% faster there, 1 to 2% slower at no=16/nv=72 in FP64 and FP32.
// The CR doubles' type in the slot, and the singles' place behind them.
template <class Q>
using slot_t = std::conditional_t<sizeof(Q) == 16, float, double>;
template <class T>
constexpr int singles_at() {
  return 64 * 64 * (int)sizeof(T) / 8;
}

// each_element with the element's value x in the slot: v[r] = f(i, j, k, x),
// read 16 at a time (one wait each, not one per hole pair).
template <class F>
__device__ __forceinline__ void each_element_with(const ItemGeo &G, gptr<const double> in, int lane,
                                                  double (&v)[64], F &&f) {
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    double x[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      v[16 * (n >> 2) + 4 * jj + (n & 3)] = 0.0;
      x[n] = in[(16 * (n >> 2) + 4 * jj + (n & 3)) * 64 + lane];
    }
    if (jj < G.J.n)
#pragma unroll
      for (int n = 0; n < 16; ++n)
        if (G.pair(0, jj, n & 3)) v[16 * (n >> 2) + 4 * jj + (n & 3)] = f(n >> 2, jj, n & 3, x[n]);
    phase();
  }
}

// f(r, factor of the singles product of element r) over the 9 singles
// products of the lane's elements, r = 16 i + 4 j + k, from the staged
// operands; hole pairs without an element that counts are skipped.
template <class F>
__device__ __forceinline__ void each_single(const double *e, const ItemGeo &G, const Place &p,
                                            F &&f) {
  const int sa = again(p.sa), sb = again(p.sb), sc = again(p.sc);
  const int obc = 0 * 64 + sb * 8 + sc, oac = 1 * 64 + sa * 8 + sc, oab = 2 * 64 + sa * 8 + sb;
  const double *t1 = e + EPI_S;
#pragma unroll
  for (int t = 0; t < 3; ++t) {
    double ta[4], tb[4], tc[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      ta[u] = t1[((0 * 3 + t) * 8 + sa) * 4 + u];
      tb[u] = t1[((1 * 3 + t) * 8 + sb) * 4 + u];
      tc[u] = t1[((2 * 3 + t) * 8 + sc) * 4 + u];
    }
    const double sg = t == 1 ? -1.0 : 1.0;
#pragma unroll
    for (int u = 0; u < 4; ++u)
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        if (!G.pair(t, u, w)) continue;
        const double *sp = e + (t * 16 + u * 4 + w) * 192;
        const double sbc = sg * sp[obc], sac = sg * sp[oac], sab = sg * sp[oab];
#pragma unroll
        for (int m = 0; m < 4; ++m) {
          const int r = t == 0 ? m * 16 + u * 4 + w : (t == 1 ? u * 16 + m * 4 + w : u * 16 + w * 4 + m);
          f(r, ta[m] * sbc - tb[m] * sac + tc[m] * sab);
        }
      }
  }
}

// FP64 energy of one wave's elements: den = d * factor / (e_h1 + e_h2 + e_h3
// - e_p4 - e_p5 - e_p6), E[T] += den * d, E(T) += den * (d + s) with the 9
// singles products (ccsd_t_dot.F:107 and the s1 table, as fused_wg.hip).
template <class Q>
__device__ __forceinline__ void energy(const Q (&q)[16], const double *e, cptr<FusedArgs> A,
                                       cptr<TaskDev> T, const Place &p, const ItemGeo &G,
                                       double &e4, double &e5) {
  e4 = 0.0;
  e5 = 0.0;
  if (!inside(T, p)) return;
  const Denominator D = denominator(A, G, p);
  const double factor = T->factor * G.distinct();
  double den[64];
  each_element(G, den, [&](int ii, int jj, int kk, int) {
    const double d = (double)q[4 * jj + kk][ii];
    const double dn = d * factor / (D.eh[0][ii] + D.eh[1][jj] + D.eh[2][kk] + D.d0);
    const bool ok = G.pair(2, ii, jj);
    e4 += ok ? dn * d : 0.0;
    return ok ? dn : 0.0;
  });
  double x = 0.0;
  each_single(e, G, p, [&](int r, double s) { x += den[r] * s; });
  e5 = e4 + x;
}

// Tile export: the task's doubles d and singles s (the products of the
// energy's singles term, without the denominator), element (a, b, c, i, j, k)
// of the task at ((((a r5 + b) r6 + c) r1 + i) r2 + j) r3 + k, i.e. the
// reference's triplesx(h3,h2,h1,p6,p5,p4); doubles at A.partials, singles
// n = |tile| doubles after them.  One task per launch (A.tasks[0]).
__device__ __forceinline__ void singles_products(const double *e, const ItemGeo &G, const Place &p,
                                                 double (&sv)[64]) {
#pragma unroll
  for (int r = 0; r < 64; ++r) sv[r] = 0.0;
  each_single(e, G, p, [&](int r, double s) { sv[r] += s; });
}

template <class Q>
__device__ __forceinline__ void store_tiles(const Q (&q)[16], const double *e, cptr<FusedArgs> A,
                                            cptr<TaskDev> T, const Place &p, const ItemGeo &G) {
  if (!inside(T, p)) return;
  const int r1 = T->r1, r2 = T->r2, r3 = T->r3, r5 = T->r5, r6 = T->r6;
  const long n = (long)r1 * r2 * r3 * T->r4 * r5 * r6;
  const gptr<double> td = (gptr<double>)A->partials, ts = td + n;
  const long base = (((long)p.la * r5 + p.lb) * r6 + p.lc) * r1;
  auto put = [&](gptr<double> to, auto &&value) {
#pragma unroll
    for (int ii = 0; ii < 4; ++ii)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj)
#pragma unroll
        for (int kk = 0; kk < 4; ++kk)
          if (ii < G.I.n && jj < G.J.n && kk < G.K.n)
            to[((base + p.i0 + ii) * r2 + p.j0 + jj) * r3 + p.k0 + kk] = value(ii, jj, kk);
  };
  put(td, [&](int i, int j, int k) { return (double)q[4 * j + k][i]; });
  double sv[64];
  singles_products(e, G, p, sv);
  put(ts, [&](int i, int j, int k) { return sv[16 * i + 4 * j + k]; });
}

// Epilogues of the item loop: each item's energy partials, one task's t3
// tiles (store_tiles), or the Lambda- and CR-CCSD(T) sums (lambda.hip), whose
// items run the left-hand job's contractions, then the right-hand job's.
enum { EPI_ENERGY = 0, EPI_TILES = 1, EPI_LAMBDA = 2, EPI_CR = 3 };
constexpr bool pair_epilogue(int epi) { return epi == EPI_LAMBDA || epi == EPI_CR; }

// Left-hand half of a Lambda item: the y3 doubles, i.e. the accumulators plus
// the Fock term P(c/ab) P(k/ij) y(a b i j) f(k c).  Written out, that term is
// the singles term with f(h p) for t1(p h) and y(p p' h h') for S: its operands
// are staged and summed as those (`fock`; y from the job's dense T2e, T2e[h][h'][p][p']).
// Elements outside the task are written too (the right-hand half skips them).
template <class Q>
__device__ __forceinline__ void lambda_left(const Q (&q)[16], const double *e, bool fock,
                                            const Place &p, const ItemGeo &G, gptr<double> out,
                                            int lane) {
  double yd[64];
#pragma unroll
  for (int r = 0; r < 64; ++r) yd[r] = (double)q[r & 15][r >> 4];
  if (fock) each_single(e, G, p, [&](int r, double s) { yd[r] += s; });
#pragma unroll
  for (int r = 0; r < 64; ++r) out[r * 64 + lane] = yd[r];
}

// Left-hand half of a CR item: the t3 doubles and singles.
template <class Q>
__device__ __forceinline__ void cr_left(const Q (&q)[16], const double *e, const Place &p,
                                        const ItemGeo &G, gptr<double> out, int lane) {
#pragma unroll
  for (int r = 0; r < 64; ++r) ((gptr<slot_t<Q>>)out)[r * 64 + lane] = q[r & 15][r >> 4];
  phase();
  double sv[64];
  singles_products(e, G, p, sv);
#pragma unroll
  for (int r = 0; r < 64; ++r) out[singles_at<slot_t<Q>>() + r * 64 + lane] = sv[r];
}

// Right-hand half of a Lambda item: den = t3d * factor / D as in energy(), e1
// += den * yd, e2 += den * (yd + ys) with the left-hand doubles yd of the same
// elements and the left-hand singles ys formed here from the staged operands
// of the left-hand job.
template <class Q>
__device__ __forceinline__ void lambda_right(const Q (&q)[16], const double *e, cptr<FusedArgs> A,
                                             cptr<TaskDev> T, const Place &p, const ItemGeo &G,
                                             gptr<const double> in, int lane, double &e1,
                                             double &e2) {
  e1 = 0.0;
  e2 = 0.0;
  if (!inside(T, p)) return;
  const Denominator D = denominator(A, G, p);
  const double factor = T->factor * G.distinct();
  double den[64];
  each_element_with(G, in, lane, den, [&](int ii, int jj, int kk, double yd) {
    const double dn = (double)q[4 * jj + kk][ii] * factor /
                      (D.eh[0][ii] + D.eh[1][jj] + D.eh[2][kk] + D.d0);
    const bool ok = G.pair(2, ii, jj);
    e1 += ok ? dn * yd : 0.0;
    return ok ? dn : 0.0;
  });
  phase();
  double x = 0.0;
  each_single(e, G, p, [&](int r, double s) { x += den[r] * s; });
  e2 = e1 + x;
}

// Right-hand half of a CR item (cr_ccsd_t.F:150-205): with w = factor / D, the
// right-hand job's doubles r (the moment) and singles q (the denominator
// tile) against the left-hand t3 doubles td and singles ts of the same
// elements: s0 += w r td, s1 += w r (td + ts), s2 += w q td, s3 += w q (td +
// ts).
template <class Q>
__device__ __forceinline__ void cr_right(const Q (&q)[16], const double *e, cptr<FusedArgs> A,
                                         cptr<TaskDev> T, const Place &p, const ItemGeo &G,
                                         gptr<const double> in, int lane, double (&s)[4]) {
  s[0] = s[1] = s[2] = s[3] = 0.0;
  if (!inside(T, p)) return;
  const Denominator D = denominator(A, G, p);
  const double factor = T->factor * G.distinct();
  double d0 = D.d0;
  auto weight = [&](int ii, int jj, int kk) {
    const double w = factor / (D.eh[0][ii] + D.eh[1][jj] + D.eh[2][kk] + d0);
    return G.pair(2, ii, jj) ? w : 0.0;
  };
  // 32-bit accumulators leave room for the 64 singles products: one pass over the
  // slot and 64 divisions instead of two and 192 (no=40/nv=160, bf16x6 566 / 484
  // ms, bf16x3 430 / 353, FP32 634 / 577).
  if constexpr (sizeof(q[0][0]) == 4) {
    const gptr<const slot_t<Q>> in1 = (gptr<const slot_t<Q>>)in;
    const gptr<const double> in2 = in + singles_at<slot_t<Q>>();
    double sv[64];
    singles_products(e, G, p, sv);
    phase();
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
      for (int i0 = 0; i0 < 4; i0 += 2) {
        double td[8], ts[8];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const int r = 16 * (i0 + (n >> 2)) + 4 * jj + (n & 3);
          td[n] = in1[r * 64 + lane];
          ts[n] = in2[r * 64 + lane];
        }
        if (jj < G.J.n)
#pragma unroll
          for (int n = 0; n < 8; ++n)
            if (G.pair(0, jj, n & 3)) {
              const int ii = i0 + (n >> 2);
              const double w = weight(ii, jj, n & 3);
              const double r = (double)q[4 * jj + (n & 3)][ii] * w;
              const double x = sv[16 * ii + 4 * jj + (n & 3)] * w;
              s[0] += r * td[n];
              s[1] += r * ts[n];
              s[2] += x * td[n];
              s[3] += x * ts[n];
            }
        phase();
      }
    s[1] += s[0];
    s[3] += s[2];
    return;
  }
  // the accumulators are read out first, then one 64-value array is live at a
  // time (both together do not fit the registers; a third division is cheaper)
  const gptr<const double> ins = in + singles_at<slot_t<Q>>();
#pragma unroll
  for (int jj = 0; jj < 4; ++jj) {
    double td[16], ts[16];
#pragma unroll
    for (int n = 0; n < 16; ++n) {
      td[n] = in[(16 * (n >> 2) + 4 * jj + (n & 3)) * 64 + lane];
      ts[n] = ins[(16 * (n >> 2) + 4 * jj + (n & 3)) * 64 + lane];
    }
    if (jj < G.J.n)
#pragma unroll
      for (int n = 0; n < 16; ++n)
        if (G.pair(0, jj, n & 3)) {
          const double rd = (double)q[4 * jj + (n & 3)][n >> 2] * weight(n >> 2, jj, n & 3);
          s[0] += rd * td[n];
          s[1] += rd * ts[n];
        }
  }
  s[1] += s[0];
  phase();
#pragma unroll 1
  for (int half = 0; half < 2; ++half) {
    double v[64];
    asm volatile("" : "+v"(d0));  // the 64 weights anew, not kept from the loop above
    each_element_with(G, half ? ins : in, lane, v, [&](int ii, int jj, int kk, double t) {
      return weight(ii, jj, kk) * t;
    });
    phase();
    each_single(e, G, p, [&](int r, double x) { s[3] += v[r] * x; });
    if (!half) s[2] = s[3];
  }
}

// The item loop, with the epilogue EPI.
template <int PREC, int EPI>
__global__ void __launch_bounds__(64 * Prec<PREC>::NW, 2) fused_triples_mixed(const MixedSegment *segments, int nseg,
                                                           long nglobal,
                                                           unsigned long long *sched) {
  __shared__ f4 lds[lds_quads<PREC>()];
  __shared__ NextItem next_item;  // dynamic schedule: the workgroup's next item
  using Pr = Prec<PREC>;
  constexpr int NW = Pr::NW;
  constexpr bool HALF = NW == 4;  // the launch's indices are half items
  if (HALF) nglobal *= 2;
  const int tid = threadIdx.x, wave = uniform(tid >> 6), lane = tid & 63;
  const unsigned lds_base =
      (unsigned)uniform((int)(unsigned long)(__attribute__((address_space(3))) f4 *)lds);
  const cptr<MixedSegment> segs = (cptr<MixedSegment>)segments;
  // Persistent loop over the launch's items: the dynamic schedule of sched_item
  // when `sched` is given, else a static round-robin.  The item is uniform
  // across the workgroup, so its waves (4 or 8) reach the same barriers; an
  // empty half has only the one at the item's end.
  const bool dyn = sched != nullptr;
  // log2 of the slice width; a launch of fewer than eight slices takes narrower
  // ones, so that every XCD has items of its own
  int sh = (dyn ? (int)sched[9] : 0) + (HALF ? 1 : 0);
  while (sh > 0 && (8l << sh) > nglobal) --sh;
  unsigned queue = blockIdx.x & 7u;  // thread 0: the queue it draws from
  unsigned long long ticket = 0;
  long g = 0;
  if (dyn) {
    if (tid == 0)
      next_item.put(-1, sched_item(sched, queue, atomicAdd(&sched[queue], 1ull), nglobal, sh));
    __syncthreads();
    g = uniform(next_item.get(-1));
  }
  int seg = 0;  // segment of the workgroup's current item
  for (long r = 0;; ++r) {
    if (dyn) {
      if (g < 0) break;
    } else {
      if (r * (long)gridDim.x >= nglobal) break;
      g = round_item(r, blockIdx.x, gridDim.x, nseg > 1);
      if (g >= nglobal) continue;  // last round: uniform per workgroup
    }
    const long gi = HALF ? g >> 1 : g;
    const int c4 = HALF ? 4 * (int)(g & 1) : 0;  // first c slot of a half item
    seg = next_segment(segs, nseg, seg, gi);
    const long item = segs[seg].item0 + (gi - segs[seg].g0);
    const cptr<MixedArgs> M = (cptr<MixedArgs>)segs[seg].args;
    const cptr<FusedArgs> A = &M->f;
    const cptr<TaskDev> tasks = (cptr<TaskDev>)A->tasks;
    const cptr<TaskDev> T = tasks + find_task(tasks, A->ntasks, item);
    // boxes of a multi-box task (reference tiling, tile export): hole boxes
    // outermost, particle c fastest.  (Sub-tile and orbital tables have one
    // box per task and order their tasks themselves.)
    long box = item - T->item0;
    const int bc = box % T->nb6; box /= T->nb6;
    const int bb = box % T->nb5; box /= T->nb5;
    const int ba = box % T->nb4; box /= T->nb4;
    const int bk = box % T->nb3; box /= T->nb3;
    const int bj = box % T->nb2; box /= T->nb2;
    const int bi = (int)box;
    ItemGeo G;
    auto hbox = [](int o, int b, int r) { return HoleBox{o, 4 * b, r - 1, min(4, r - 4 * b)}; };
    G.I = hbox(T->oh1, bi, T->r1);
    G.J = hbox(T->oh2, bj, T->r2);
    G.K = hbox(T->oh3, bk, T->r3);
    auto prng = [](int o, int r, int n) { return PRange{o, min(n - 1, r - 1), 0}; };
    // The item's equal boxes: of the same tile, and of the same place in it
    // where the tiles hold several (reference tiling).  Told per task, they served
    // one-box tasks only; reference-tiled no=24/nv=120 in tiles of 12 and 40 then
    // and now: FP64 184 / 144 ms, FP32 119 / 93, bf16x3 47.1 / 39.2, bf16x6 68 / 56.
    int eq = 0;
    if (EPI != EPI_TILES || !T->full) {  // (read by every kernel, the flag cost 2% of no=40/nv=160)
      eq = (T->oh1 == T->oh2 && bi == bj ? EQ_IJ : 0) | (T->oh2 == T->oh3 && bj == bk ? EQ_JK : 0);
      if (T->op4 == T->op5 && ba == bb) eq |= EQ_AB | (T->op5 == T->op6 && bb == bc ? EQ_BC : 0);
    }
    G.heq = eq & (EQ_IJ | EQ_JK);
    G.a = prng(T->op4 + 8 * ba, T->r4 - 8 * ba, 8);
    G.b = prng(T->op5 + 8 * bb, T->r5 - 8 * bb, 8);
    G.c = prng(T->op6 + 8 * bc + c4, T->r6 - 8 * bc - c4, HALF ? 4 : 8);
    {
      // wave bits of the cube coordinates: the ranges with two cubes take the
      // low bits, so the waves with work spread over the four SIMDs (wave w
      // runs on SIMD w % 4)
      const bool wa = G.a.sm >= 4, wb = G.b.sm >= 4, wc = G.c.sm >= 4;
      if (HALF) {
        G.b.bit = wb || !wa ? 0 : 1;
        G.a.bit = 1 - G.b.bit;
        G.c.bit = 2;  // one cube
      } else {
        const int nw = (wa ? 1 : 0) + (wb ? 1 : 0) + (wc ? 1 : 0);
        G.c.bit = wc ? 0 : nw;
        G.b.bit = wb ? (wc ? 1 : 0) : nw + (wc ? 0 : 1);
        G.a.bit = wa ? (wc ? 1 : 0) + (wb ? 1 : 0) : nw + (wc ? 0 : 1) + (wb ? 0 : 1);
      }
    }
    const ItemPlan P = item_plan(eq, HALF);
    const long part = item * 8 + c4 + wave;  // the wave's partial

    double *epi = reinterpret_cast<double *>(lds);
    Place p;  // layout c: lane = 4a' + b' + 16c'
    {
      const int ln = again(lane);
      p.sa = 4 * cube(wave, G.a) + ((ln & 15) >> 2);
      p.sb = 4 * cube(wave, G.b) + (ln & 3);
      p.sc = 4 * cube(wave, G.c) + (ln >> 4);
      p.la = 8 * ba + p.sa, p.lb = 8 * bb + p.sb, p.lc = 8 * bc + c4 + p.sc;
      p.i0 = 4 * bi, p.j0 = 4 * bj, p.k0 = 4 * bk;
    }
    const gptr<double> partials = (gptr<double>)A->partials;
    const gptr<double> den = (gptr<double>)M->cr_den;
    const bool empty = HALF && G.c.sm < 0;  // a half past the edge: no element
    // The next item's ticket is drawn before this one's epilogue and read at its
    // end.  Drawn at the start of the item, the first workgroups of a launch
    // with fewer items than workgroups took two items each (no=8/nv=32, 160
    // half items: 134 us, now 104), and the last round of a longer one was less
    // even (CR no=16/nv=72 4.76 / 4.61 ms, Lambda no=20/nv=80 15.3 / 15.2).
    // (The order of the tests here and below is the faster one of each kernel, all
    // of which sit at the register limit: `dyn` first, no=40/nv=160 460 ms and a
    // tile export of no=24/nv=96 1.30 ms; `dyn` second, 465 and 1.17 ms.)
    if (EPI == EPI_TILES ? empty && dyn && tid == 0 : dyn && empty && tid == 0)
      ticket = atomicAdd(&sched[queue], 1ull);
    if (empty && EPI != EPI_TILES && lane == 0) {
      partials[2 * part] = partials[2 * part + 1] = 0.0;
      if (EPI == EPI_CR) den[2 * part] = den[2 * part + 1] = 0.0;
    }
    // one half, or the left-hand and the right-hand half of a pair's item (the
    // jobs have the same tasks)
#pragma unroll 1
    for (int side = empty ? 2 : (pair_epilogue(EPI) ? 0 : 1); side < 2; ++side) {
      const cptr<MixedArgs> ML = (cptr<MixedArgs>)M->left;
      const cptr<MixedArgs> MS = side ? M : ML;
      typename Pr::quad q[16];
      contract<PREC>(q, lds, lds_base, MS, T, G, P, wave, lane);
      // Epilogue: the chunk buffers are free.
      if (EPI == EPI_TILES ? side == 1 && dyn && tid == 0 : dyn && side == 1 && tid == 0)
        ticket = atomicAdd(&sched[queue], 1ull);
      const long slot = ((long)blockIdx.x * NW + wave) *
                        pair_wave_doubles(EPI == EPI_CR, PREC != TCE_T_FP64);
      const gptr<double> spill = (gptr<double>)M->spill + slot;
      const bool fock = EPI == EPI_LAMBDA && side == 0 && ML->lam_f != nullptr;
      if (fock)
        stage_epilogue<NW>(epi, (gptr<const double>)ML->f.T2e, ML->f.Ep,
                           (gptr<const double>)ML->lam_f, 1, A->nv, A->no, A->nv, wave, lane, G);
      else if (EPI != EPI_LAMBDA || side)
        stage_singles<NW>(epi, EPI == EPI_LAMBDA ? &ML->f : &MS->f, wave, lane, G);
      __syncthreads();
      if constexpr (EPI == EPI_TILES) {
        store_tiles(q, epi, A, T, p, G);
      } else if constexpr (EPI == EPI_ENERGY) {
        double e4, e5;
        energy(q, epi, A, T, p, G, e4, e5);
        wave_sum(e4, e5);
        if (lane == 0) {
          partials[2 * part] = e4;
          partials[2 * part + 1] = e5;
        }
      } else if (side == 0) {
        if constexpr (EPI == EPI_LAMBDA) lambda_left(q, epi, fock, p, G, spill, again(lane));
        else cr_left(q, epi, p, G, spill, again(lane));
        __syncthreads();  // the right-hand half's first loads overwrite the staged data
      } else if constexpr (EPI == EPI_LAMBDA) {
        double e1, e2;
        lambda_right(q, epi, A, T, p, G, spill, again(lane), e1, e2);
        wave_sum(e1, e2);
        if (lane == 0) {
          partials[2 * part] = e1;
          partials[2 * part + 1] = e2;
        }
      } else {
        double cs[4];
        cr_right(q, epi, A, T, p, G, spill, again(lane), cs);
        wave_sum(cs[0], cs[1]);
        wave_sum(cs[2], cs[3]);
        if (lane == 0) {
          partials[2 * part] = cs[0];
          partials[2 * part + 1] = cs[1];
          den[2 * part] = cs[2];
          den[2 * part + 1] = cs[3];
        }
      }
    }
    if (dyn && tid == 0) next_item.put(r, sched_item(sched, queue, ticket, nglobal, sh));
    __syncthreads();  // the next item's first loads overwrite the staged data
    if (dyn) g = uniform(next_item.get(r));
  }
  if (dyn && tid == 0) sched_leave(sched);
}

}  // namespace

// grid: workgroups of 8 waves, at most one per CU (halves: twice as many of 4
// waves).  The contraction extents of every job in the table must be multiples of
// the precision's chunk (8 FP64 / 16 FP32 / 32 bf16 values); the job layer
// pads them.
template <int PREC, int EPI>
static void launch_one(const MixedSegment *segs, int nseg, long total, int grid, hipStream_t s,
                       unsigned long long *sched) {
  constexpr int NW = Prec<PREC>::NW;
  hipLaunchKernelGGL(HIP_KERNEL_NAME(fused_triples_mixed<PREC, EPI>), dim3((unsigned)grid * 8 / NW),
                     dim3(64 * NW), 0, s, segs, nseg, total, sched);
}
template <int EPI>
static int launch_prec(const MixedSegment *segs, int nseg, long total, int precision, int grid,
                       hipStream_t s, unsigned long long *q) {
  if (precision == TCE_T_FP64)
    launch_one<TCE_T_FP64, EPI>(segs, nseg, total, grid, s, q);
  else if (precision == TCE_T_FP32)
    launch_one<TCE_T_FP32, EPI>(segs, nseg, total, grid, s, q);
  else if (precision == TCE_T_BF16X3)
    launch_one<TCE_T_BF16X3, EPI>(segs, nseg, total, grid, s, q);
  else if (precision == TCE_T_BF16X6)
    launch_one<TCE_T_BF16X6, EPI>(segs, nseg, total, grid, s, q);
  else
    return -1;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_fused_mixed(const MixedSegment *segs, int nseg, long total, int precision, int grid,
                       hipStream_t s, unsigned long long *sched) {
  return launch_prec<EPI_ENERGY>(segs, nseg, total, precision, grid, s, sched);
}

int launch_fused_tiles(const MixedSegment *segs, long total, int precision, int grid,
                       hipStream_t s, unsigned long long *sched) {
  return launch_prec<EPI_TILES>(segs, 1, total, precision, grid, s, sched);
}

int launch_fused_pair(const MixedSegment *segs, long total, int precision, int grid, hipStream_t s,
                      unsigned long long *sched, bool cr) {
  return cr ? launch_prec<EPI_CR>(segs, 1, total, precision, grid, s, sched)
            : launch_prec<EPI_LAMBDA>(segs, 1, total, precision, grid, s, sched);
}

}  // namespace tce_t
