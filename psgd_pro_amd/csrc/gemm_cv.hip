// MFMA products of fp32- or bf16-stored operands in any layout (k-contiguous, m/n-contiguous, or a matrix held in its
// upper triangle), of any size and alignment: every contraction of the fp32 precision, and those of the bf16 precision
// whose operands are not already k-contiguous bf16.
//
// The operands are read as stored, converted in registers and staged in LDS as k-contiguous bf16, so that all of them
// run on the bf16 MFMA (2.5 PFLOP/s dense; the fp32 MFMA does 0.157):
//   bf16 precision: each value rounded to bfloat16 (round to nearest even), one product.
//   fp32 precision: each value times 2^16, x, split exactly into three bfloat16 planes, x = h + m + l with h = bf16(x),
//     m = bf16(x - h), l = bf16(x - h - m) (8 + 8 + 8 significant bits; both differences are exact), and the six
//     products h h', h m', m h', m m', h l', l h' accumulated in fp32. The three dropped ones are below 2^-23 |x x'|
//     together in the worst case and about 2^-27 with either sign on random values, under the 2^-24 of the
//     accumulation itself. The factor, taken out of the sums again, changes no rounding, and with it the split is exact
//     down to the least subnormal: bfloat16 ends at 2^-133 (the MFMA keeps its subnormals), so that below 2^-110 an
//     unscaled l, and then m, lose their bits (operands near 1e-36: error 2.6e-5).
// The k loop accumulates blocks of k and folds each block into a second accumulator set: one fp32 chain over all of K
// carries several times the rounding error of blocked summation.
//
// Rounding. Measured on gfx950: the bf16 MFMA aligns the 8 products of a lane to the largest of them and truncates each
// toward zero there at 24 bits (1 + 2^-25 and 1 - 2^-25 give 1); the lane groups' sums and C are then added to the nearest,
// but for what a much larger C leaves of them (below). fp32 sums must not pay for that:
//   64- and 32-row tiles: h h' enters an MFMA with C = 0 and is added to the block by a VALU add, and the five small
//     products have accumulators of their own, so nothing small is aligned to a large sum. Relative error (Frobenius, k
//     1024 normals) 7.4e-8; one fp32 MFMA chain folded every 128 k: 2.1e-7.
//   The diagonal tile of a Gram product X^T X or X X^T, at the k of its own rows: for X near a multiple of the identity (a
//     preconditioner factor) one square outweighs the other 7 of its lane, whose truncation then always lowers the
//     diagonal (by up to 2e-7 of it, which the norm bound of the next product sees doubled): there a row's
//     own k is left out of A's planes and added to the sum by one fp32 multiply-add (mean below 1e-8). Gram products of
//     factors keep to these tiles.
//   128 x 256 tiles: registers for one accumulator set per block only, with all six products on top of it. Bits of a
//     small product below the last of a large C are dropped downward (mean error of 3072^3 -5e-8 of the results' rms), so
//     every other block is computed negated and subtracted (mean below 1e-10). Longer blocks cost roundings inside them,
//     more blocks cost roundings of the whole sum, which matter for operands of one sign: blocks of 64 k up to k 1280, of
//     128 above. Errors of 64, of 128 and of fp32 MFMA chains of 128, in 1e-8: random signs, k 1024 14.7, 18.3, 21.1, k 3072
//     17.9, 19.7, 22.3; one sign, k 1280 7.2, 6.9, 7.4, k 1536 7.13, 6.6, 7.06, k 3072 9.5, 7.4, 7.6.
// Infinities, NaNs, values from 2^112 on and sums from 2^96 on leave non-finite sums: a workgroup whose accumulators are
// not all finite repeats its tile with fp32 MFMAs (mma_f32), whose results are IEEE's.
//
// What bounds it. fp32, 128 x 256: a 32-k stage is 3072 MFMA cycles per SIMD pair of waves against about 180 VALU
// instructions of address, split and store per converting wave, 72 KB of LDS writes and 144 KB of fragment reads: two
// groups of four waves a half step apart, so that one converts while the other multiplies (a single group left the matrix
// cores idle during every conversion). 3072^3: 671 us on the fp32 MFMA kernel this replaces, now 437; two at once 1065,
// now 683; 4096^3 1188, now 663. 64 x 64: latency and occupancy; k split over two wave groups while a launch has at most
// a tile per CU (1024^3: 86 us, now 24; symmetric 2304 x 768 from its triangle: 287, now 118; 1001 x 770 x 770, unaligned
// rows: 148, now 22). Beyond, 64-tiles in groups of four waves; 128 x 256 tiles once they fill half the chip.
// bf16 precision from fp32 or transposed operands: 3 to 8 times faster than reading them into bf16 LDS tiles element by
// element (1531^3 36 us, 4096^3 255).
#include <type_traits>

#include "gemm_cv.h"

namespace psgdk {

namespace {

typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
// four consecutive floats at any 4-byte aligned address (one 16-byte access: the hardware needs dword alignment only)
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));

#define INL __attribute__((always_inline))

constexpr int NT = 256;      // threads that stage one operand tile together
constexpr int KS32 = 32;     // k of one LDS slice (a plane row of 64 bytes)
constexpr float kSplitScale = 65536.f;  // lifts fp32's last bit, 2^-149, to bfloat16's, 2^-133

__device__ __forceinline__ uint32_t cvt2(float lo, float hi) {  // two values to bfloat16, round to nearest even
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2_t{lo, hi}, bf16x2_t));
}
__device__ __forceinline__ float lo_f32(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float hi_f32(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// Byte offset of the 16-byte piece c (0..3: k 8c .. 8c + 7) of row `row` in one 32-k plane: 64-byte rows, the piece XORed
// with bits 2-3 of the row, which puts the 16 rows of a fragment read (one piece each) on 16 distinct bank groups. Rows
// 16 apart, and rows within a group of 4, differ by a constant, so one address register serves all of an operand's reads
// and one all of its stores (the transposing store's rows 4 i + j, fixed j, meet in 4 bank groups: 8 cycles instead of 4
// for its 512 bytes, which the LDS has to spare; XORing more row bits avoided that and cost 24 registers of addresses).
__device__ __forceinline__ int cv_slot(int row, int c) { return row * 64 + ((c ^ ((row >> 2) & 3)) << 4); }

enum How : int { H_KC = 0, H_MC = 1, H_ELEM = 2, H_ZERO = 3 };

__device__ __forceinline__ f32x4_t ld_f32x4(__amdgpu_buffer_rsrc_t rs, int off) {
  return __builtin_bit_cast(f32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, off, 0, 0));
}
__device__ __forceinline__ f32x4_t ld_bf16x4(__amdgpu_buffer_rsrc_t rs, int off) {
  const uint2 u = __builtin_bit_cast(uint2, __builtin_amdgcn_raw_buffer_load_b64(rs, off, 0, 0));
  return f32x4_t{lo_f32(u.x), hi_f32(u.x), lo_f32(u.y), hi_f32(u.y)};
}

// Element (mn, k) of an operand, zero past rows or K; a SYM element below the diagonal is the stored (k, mn) times the
// sign (zero for sign 0), and the diagonal of a skew matrix is zero. Branch-free: the offset is selected first, the load
// is unconditional (element 0 for one that is not read), and the value is selected after it.
template <typename T>
__device__ __forceinline__ float ld_elem(const void* __restrict__ p, const CvOperand& o, int mn, int k, int rows, int K) {
  const bool sym = o.mode == SYM, low = sym & (mn > k), up = (o.mode == KC) | (sym & (mn < k));
  const bool none = (mn >= rows) | (k >= K) | (low & (o.sign == 0)) | (sym & (mn == k) & (o.sign < 0));
  const long long off = none ? 0 : (long long)(up ? mn : k) * o.ld + (up ? k : mn);
  const float v = to_f32<T>(reinterpret_cast<const T*>(p)[off]);
  return none ? 0.f : (low & (o.sign < 0)) ? -v : v;
}

// One operand's tile of ROWS x (32 KS) in registers, as fp32, staged by 256 threads. H_KC / H_ELEM: thread t holds the
// 4-k chunks of k 4 (t % KV) of rows t / KV + i (256 / KV). H_MC: the 4 x 4 block of rows 4 (t % RB) .. and k
// 4 (t / RB) .., one register quad per k, transposed on the way to LDS (a wave reads whole 4 ROWS-byte runs).
// MODE KC or MC: rows in that layout, fp32 or (BF) bf16, whose loads no branch surrounds (registers that meet at the end of a branch
// are copied there, and the copy waits for the load) and whose addresses are one register plus constants: with every
// chunk's offsets and bounds checks computed apart, a tile's staging took 430 VALU instructions, 180 of them the
// conversion. MODE SYM: any operand, its layout and storage known at run time.
template <int ROWS, int KS, int MODE, bool BF>
struct CvTile {
  static constexpr bool ANY = MODE == SYM;
  static constexpr int KV = 8 * KS;        // chunks per row
  static constexpr int NC = ROWS * KV / NT;  // chunks per thread
  static constexpr int RS = NT / KV;       // rows between them
  static constexpr int RB = ROWS / 4, BLK = RB * KV;  // blocks per row of blocks, blocks
  static constexpr int NR = ANY || MODE == MC ? (NC > 4 ? NC : 4) : NC;
  static_assert(ROWS * KV % NT == 0 && BLK <= NT && RS % 16 == 0, "whole chunks, at most one block per thread");
  f32x4_t r[NR];
  int how, kleft;  // kleft: k in range from the tile's first one on (a chunk of H_KC may straddle it)

  static __device__ __forceinline__ unsigned thread() { return threadIdx.x & (NT - 1); }

  // Rows past the operand lie past its buffer's end and read zero; so do k rows past K (H_MC). Values past K within a
  // row (H_KC) are the next row's, cleared on the way to LDS; m/n past the operand in an H_MC row are the next row's
  // and reach only results that are not stored. Offsets are relative to the tile's own first element: 128 rows stay
  // under 2 GiB for leading dimensions below 2^21 (the host clears vec above, and every element is then addressed by
  // itself).
  template <typename LD>
  __device__ __forceinline__ void load_kc(LD ld, int sh, int stride) {
    const unsigned t = thread();
    unsigned off = (t / KV * stride + t % KV * 4) << sh;
#pragma unroll
    for (int i = 0; i < NC; ++i, off += (unsigned)(RS * stride) << sh) r[i] = ld((int)off);
  }
  template <typename LD>
  __device__ __forceinline__ void load_mc(LD ld, int sh, int stride) {
    const unsigned t = thread();
    unsigned off = BLK < NT && t >= BLK ? (unsigned)kOob : (t / RB * 4 * stride + t % RB * 4) << sh;
#pragma unroll
    for (int j = 0; j < 4; ++j, off += (unsigned)stride << sh) r[j] = ld((int)off);
  }
  template <typename T>
  __device__ __forceinline__ void load_elem(const void* __restrict__ p, const CvOperand& o, int mn0, int k0, int rows,
                                            int kend) {
    int t = threadIdx.x & (NT - 1);
    asm volatile("" : "+v"(t));  // the addresses are recomputed for each tile rather than kept in registers
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int mn = mn0 + t / KV + i * RS, k = k0 + t % KV * 4;
#pragma unroll
      for (int e = 0; e < 4; ++e) r[i][e] = ld_elem<T>(p, o, mn, k + e, rows, kend);
    }
  }

  // mn0, k0: the tile's origin; rows, kend: the operand's extent (kend: end of this k range)
  __device__ __forceinline__ void load(const void* __restrict__ p, const CvOperand& o, int mn0, int k0, int rows, int kend) {
    int h = ANY ? o.mode : MODE;
    kleft = kend - k0;
    if constexpr (ANY) {
      if (o.mode == SYM) {
        if (mn0 + ROWS <= k0) h = H_KC;
        else if (mn0 >= k0 + 4 * KV) h = o.sign == 0 ? H_ZERO : H_MC;
        else h = H_ELEM;
      }
      if (!o.vec && h != H_ZERO) h = H_ELEM;
      how = h;
      if (h == H_ZERO) {
#pragma unroll
        for (int i = 0; i < NC; ++i) r[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        return;
      }
      if (h == H_ELEM) {
        if (o.bf16) load_elem<bf16_t>(p, o, mn0, k0, rows, kend);
        else load_elem<float>(p, o, mn0, k0, rows, kend);
        return;
      }
    }
    // the stored rows and columns this tile reads start at (r0, c0); the buffer ends with the operand's last element
    // (whole dwords: each is checked by itself)
    const int sh = BF || (ANY && o.bf16) ? 1 : 2, stride = (int)o.ld;
    const bool kc = h == H_KC;
    const int r0 = kc ? mn0 : k0, c0 = kc ? k0 : mn0, nrow = kc ? rows : kend, ncol = kc ? kend : rows;
    const __amdgpu_buffer_rsrc_t rs =
        make_rsrc(reinterpret_cast<const char*>(p) + (((long long)r0 * o.ld + c0) << sh),
                  ((((nrow - 1 - r0) * o.ld + ncol - c0) << sh) + 3) & ~3LL);
    auto f4 = [&](int off) { return ld_f32x4(rs, off); };
    auto b4 = [&](int off) { return ld_bf16x4(rs, off); };
    if constexpr (ANY) {
      if (o.bf16) {
        if (kc) load_kc(b4, 1, stride);
        else load_mc(b4, 1, stride);
      } else {
        if (kc) load_kc(f4, 2, stride);
        else load_mc(f4, 2, stride);
      }
    } else if constexpr (MODE == KC) {
      if constexpr (BF) load_kc(b4, 1, stride);
      else load_kc(f4, 2, stride);
    } else {
      if constexpr (BF) load_mc(b4, 1, stride);
      else load_mc(f4, 2, stride);
    }
  }

  // calls put(row, chunk, i, 4 values) for each chunk of the tile this thread holds: row `row` + i rows
  template <typename P>
  __device__ __forceinline__ void each(const CvOperand& o, P put) const {
    unsigned t = thread();
    if constexpr (MODE == MC) asm volatile("" : "+v"(t));  // its LDS addresses, recomputed for each tile: few registers
    if (ANY ? how == H_MC : MODE == MC) {
      if (BLK == NT || t < BLK) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          f32x4_t x = {r[0][c], r[1][c], r[2][c], r[3][c]};
          if (ANY && o.mode == SYM && o.sign < 0) x = -x;
          put(t % RB * 4, t / RB, c, x);
        }
      }
    } else if ((!ANY || how == H_KC) && kleft < 4 * KV) {  // the last tile: values past K are another row's
      const int k = t % KV * 4;
#pragma unroll
      for (int i = 0; i < NC; ++i)
        put(t / KV, t % KV, i * RS, f32x4_t{k < kleft ? r[i][0] : 0.f, k + 1 < kleft ? r[i][1] : 0.f,
                                            k + 2 < kleft ? r[i][2] : 0.f, k + 3 < kleft ? r[i][3] : 0.f});
    } else {
#pragma unroll
      for (int i = 0; i < NC; ++i) put(t / KV, t % KV, i * RS, r[i]);
    }
  }

  // zeroes the elements whose row is their k (a tile that starts at equal rows and k)
  __device__ __forceinline__ void clear_own() {
    const unsigned t = thread();
    if (ANY ? how == H_MC : MODE == MC) {
#pragma unroll
      for (int j = 0; j < 4; ++j) r[j][j] = t % RB == t / RB ? 0.f : r[j][j];
    } else {
#pragma unroll
      for (int i = 0; i < NC; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) r[i][e] = t / KV + i * RS == t % KV * 4 + e ? 0.f : r[i][e];
    }
  }

  // into NP bf16 planes of KS slices of TROWS rows x 32 k, from row `row0` on (a multiple of 16)
  // (three planes: of the values times `scale`, +- kSplitScale)
  template <int NP, int TROWS>
  __device__ __forceinline__ void store(unsigned char* lds, int row0, const CvOperand& o, float scale) const {
    lds += row0 * 64;
    each(o, [&](unsigned row, unsigned kv, int i, f32x4_t x) {
      if constexpr (NP == 3) x = f32x4_t{x.x * scale, x.y * scale, x.z * scale, x.w * scale};
      // rows i apart (below 4 from a multiple of 4, or a multiple of 16) keep the slot's XOR: a constant offset
      unsigned char* q = lds + (kv >> 3) * (TROWS * 64) + cv_slot(row, (kv & 7) >> 1) + (kv & 1) * 8 + i * 64;
      const uint2 h = make_uint2(cvt2(x.x, x.y), cvt2(x.z, x.w));
      *reinterpret_cast<uint2*>(q) = h;
      if constexpr (NP == 3) {
        const f32x4_t d = {x.x - lo_f32(h.x), x.y - hi_f32(h.x), x.z - lo_f32(h.y), x.w - hi_f32(h.y)};
        const uint2 m = make_uint2(cvt2(d.x, d.y), cvt2(d.z, d.w));
        *reinterpret_cast<uint2*>(q + KS * TROWS * 64) = m;
        *reinterpret_cast<uint2*>(q + 2 * KS * TROWS * 64) =
            make_uint2(cvt2(d.x - lo_f32(m.x), d.y - hi_f32(m.x)), cvt2(d.z - lo_f32(m.y), d.w - hi_f32(m.y)));
      }
    });
  }
  // fp32 rows of 32 KS k, the 16-byte pieces XORed with the row
  __device__ __forceinline__ void store_f32(unsigned char* lds, int row0, const CvOperand& o) const {
    each(o, [&](unsigned row, unsigned kv, int i, f32x4_t x) {
      *reinterpret_cast<f32x4_t*>(lds + ((row0 + row + i) * KV + (kv ^ ((row + i) & 7))) * 16) = x;
    });
  }
};

constexpr int cv_ks(int BM) { return BM == 64 ? 2 : 1; }          // 32-k slices per LDS stage
constexpr int cv_hr(int BM) { return BM == 128 ? 32 : BM / 2; }  // rows of a wave's block per epilogue pass
constexpr int cv_smem(int NP, int BM, int BN, int WN, int KG) {
  const int planes = (WN == 4 ? 2 : KG) * NP * (BM + BN) * 64 * cv_ks(BM);
  const int f32 = (BM + BN) * 128 * cv_ks(BM), epi = 2 * WN * cv_hr(BM) * (BN / WN + 4) * 4;
  const int m = planes > f32 ? planes : f32;
  return m > epi ? m : epi;
}

}  // namespace

// LAY: bit 0 = A stored m-contiguous, bit 1 = B stored n-contiguous, bits 3 and 4 = A and B in bf16 (else fp32),
// bit 5 = Gram product with its rows' own k apart; 4: any operands
template <int NP, int BM, int BN, int WN, int KG, int EPI, int LAY>
__global__ void __launch_bounds__(WN == 4 || KG == 2 ? 512 : 256, 2) gemm_cv_kernel(const CvArgs p) {
  // Two groups of four waves, half a step apart, or (KG = 1) one. WN = 4: the groups own the upper and lower half of the
  // tile's rows and share both operands; KG = 2: both own the whole tile and alternate k tiles, their sums added at the
  // end.
  constexpr bool SHARE = WN == 4;
  static_assert(!SHARE || KG == 1, "one split of the work");
  constexpr int KS = cv_ks(BM), BK = KS32 * KS;
  constexpr int TM = BM / 2, TN = BN / WN;
  // MFMA tiles of MT x MT over KM k: 32 x 32 x 16 on the large tile (half the fragment registers and instructions per
  // product), 16 x 16 x 32 on the others. Lane (r, g) = (lane % MT, lane / MT) holds the 8 k of piece g of row r and the
  // results of column r, rows acc_row(g, e).
  constexpr int MT = SHARE ? 32 : 16, KM = SHARE ? 16 : 32, FM = TM / MT, FN = TN / MT, NE = MT * MT / 64;
  using Acc = std::conditional_t<SHARE, f32x16_t, f32x4_t>;
  auto acc_row = [](int g, int e) INL { return SHARE ? 8 * (e >> 2) + 4 * g + (e & 3) : 4 * g + e; };
  extern __shared__ __align__(16) unsigned char smem[];
  constexpr int AB = KS * BM * 64, BB = KS * BN * 64;  // bytes of one plane
  constexpr int STAGE = NP * (AB + BB);

  const int G = p.ntiles * p.nb * p.splitk;
  int logical = p.order ? xcd_run(blockIdx.x, G) : (int)blockIdx.x;
  const int split = logical % p.splitk;
  logical /= p.splitk;
  const int b = logical / p.ntiles, tile = logical % p.ntiles;
  int ti, tj;
  if (p.tri) {
    ti = 0;
    int rem = tile, rowlen = p.tiles_n;
    while (rem >= rowlen) { rem -= rowlen; ++ti; rowlen = p.tiles_n - ti * BM / BN; }
    tj = ti * BM / BN + rem;
  } else if (p.order) {  // groups of 4 tile rows, column-major inside a group: neighbours share operand panels in L2
    constexpr int GM = 4;
    const int grp = tile / (GM * p.tiles_n), r0 = grp * GM;
    const int gm = min(GM, p.tiles_m - r0), idx = tile - r0 * p.tiles_n;
    ti = r0 + idx % gm;
    tj = idx / gm;
  } else {
    ti = tile / p.tiles_n;
    tj = tile % p.tiles_n;
  }
  const int m0 = ti * BM, n0 = tj * BN;
  const CvOperand oa = p.a, ob = p.b;
  const void* __restrict__ Ap = p.A[b];
  const void* __restrict__ Bp = p.tri ? p.A[b] : p.B[b];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int h = SHARE || KG == 2 ? __builtin_amdgcn_readfirstlane(wave >> 2) : 0;  // the wave's group
  const int wm = SHARE ? h : (wave >> 1) & 1, wn = wave % WN, r = lane % MT, g = lane / MT;

  int kbeg = split * p.kchunk;
  const int kend = min(p.K, kbeg + p.kchunk);
  if (p.kbeg) kbeg = max(kbeg, m0 / BK * BK);
  const int nk = kend > kbeg ? (kend - kbeg + BK - 1) / BK : 0;

  // sums folded so far, the current block's, and (three planes, small tiles) all five small products' of the whole k range
  constexpr bool SM = NP == 3 && !SHARE;
  constexpr bool GRAM = (LAY & 32) != 0;
  // an accumulation block has 2^bs k tiles: 128 k, or the large tile's 64 (see the file's comment)
  constexpr int BT = 128 / BK, BS = BT == 4 ? 2 : 1;
  static_assert(BT == 1 << BS, "a power of two");
  const int bs = SHARE && NP == 3 && p.K <= 1280 ? BS - 1 : BS;
  auto block_end = [&](int kt, int n) INL { return (kt + 1 & (1 << bs) - 1) == 0 || kt + 1 == n; };
  Acc acc[FM][FN], blk[FM][FN], sm[FM][FN];
  auto each_acc = [&](auto f) INL {
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j)
#pragma unroll
        for (int e = 0; e < NE; ++e) f(i, j, e);
  };
  auto zero = [&]() INL { each_acc([&](int i, int j, int e) INL { acc[i][j][e] = blk[i][j][e] = sm[i][j][e] = 0.f; }); };
  auto fold = [&](bool neg) INL {
    const float sg = neg ? -1.f : 1.f;
    each_acc([&](int i, int j, int e) INL {
      acc[i][j][e] = fmaf(sg, blk[i][j][e], acc[i][j][e]);  // an exact product: one rounding, as of the sum
      blk[i][j][e] = 0.f;
    });
  };
  constexpr int RA = SHARE ? BM / 2 : BM, RB = SHARE ? BN / 2 : BN;  // rows a group stages
  const int ha = SHARE ? h * RA : 0, hb = SHARE ? h * RB : 0;
  CvTile<RA, KS, LAY & 4 ? SYM : LAY & 1 ? MC : KC, (LAY & 8) != 0> la;
  CvTile<RB, KS, LAY & 4 ? SYM : LAY & 2 ? MC : KC, (LAY & 16) != 0> lb;
  auto load_a = [&](int kt) INL { la.load(Ap, oa, m0 + ha, kbeg + kt * BK, p.M, kend); };
  auto load_b = [&](int kt) INL { lb.load(Bp, ob, n0 + hb, kbeg + kt * BK, p.N, kend); };
  // One stage's MFMAs, the products that need only B's first plane first. On the large tile, whose waves multiply alone
  // on their SIMD, A fragments are read one row of tiles ahead (and B's next k step with them) and the MFMAs start before
  // all of a step's fragments have arrived; the small tiles' waves overlap each other, and fewer registers are better.
  auto mma_planes = [&](const unsigned char* As) INL {
    const unsigned char* Bs = As + NP * AB;
    constexpr int NK = BK / KM, NQ = NK * FM;  // k steps, rows of tiles
    bf16x8_t aq[2][NP], bq[2][NP][FN];
    // piece of row `row` for k step t
    auto at = [&](const unsigned char* plane, int rows, int row, int t) INL {
      const int piece = SHARE ? 2 * t + g : 4 * t + g;
      return *reinterpret_cast<const bf16x8_t*>(plane + (piece >> 2) * rows * 64 + cv_slot(row, piece & 3));
    };
    auto rd_a = [&](int q) INL {
#pragma unroll
      for (int x = NP - 1; x >= 0; --x) aq[q & 1][x] = at(As + x * AB, BM, wm * TM + q % FM * MT + r, q / FM);
    };
    auto rd_b = [&](int t) INL {
#pragma unroll
      for (int x = 0; x < NP; ++x)
#pragma unroll
        for (int j = 0; j < FN; ++j) bq[t & 1][x][j] = at(Bs + x * BB, BN, wn * TN + j * MT + r, t);
    };
    if (SHARE) {
      rd_a(0);
      rd_b(0);
    }
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      if (!SHARE) {
        if (q % FM == 0) rd_b(q / FM);
        rd_a(q);
      } else if (q + 1 < NQ) {
        rd_a(q + 1);
        if ((q + 1) % FM == 0) rd_b((q + 1) / FM);
      }
      if (SHARE) __builtin_amdgcn_sched_barrier(0);
      const int i = q % FM, t = q / FM;
      auto mfma = [&](int xa, int xb, int j, const Acc& c) INL {
        if constexpr (SHARE) return __builtin_amdgcn_mfma_f32_32x32x16_bf16(aq[q & 1][xa], bq[t & 1][xb][j], c, 0, 0, 0);
        else return __builtin_amdgcn_mfma_f32_16x16x32_bf16(aq[q & 1][xa], bq[t & 1][xb][j], c, 0, 0, 0);
      };
      auto term = [&](Acc(&to)[FN], int xa, int xb) INL {
#pragma unroll
        for (int j = 0; j < FN; ++j) to[j] = mfma(xa, xb, j, to[j]);
      };
      const Acc nil = {};
      if constexpr (SM) {
        Acc top[FN];
#pragma unroll
        for (int j = 0; j < FN; ++j) top[j] = mfma(0, 0, j, nil);
        term(sm[i], 2, 0);
        term(sm[i], 1, 0);
        term(sm[i], 1, 1);
        term(sm[i], 0, 1);
        term(sm[i], 0, 2);
#pragma unroll
        for (int j = 0; j < FN; ++j) blk[i][j] += top[j];
      } else {
        if constexpr (NP == 3) {
          term(blk[i], 2, 0);
          term(blk[i], 1, 0);
        }
        term(blk[i], 0, 0);
        if constexpr (NP == 3) {
          term(blk[i], 1, 1);
          term(blk[i], 0, 1);
          term(blk[i], 0, 2);
        }
      }
      if (SHARE) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // fp32 MFMAs on the fp32 rows: lane group g holds the four k of one 16-byte piece of both operands, one k per MFMA
  unsigned char* const Bf = smem + BM * BK * 4;
  auto mma_f32 = [&]() INL {
    constexpr int PG = 64 / MT;  // pieces per step: one per lane group
#pragma unroll 1
    for (int s = 0; s < BK / 4 / PG; ++s) {
      auto at = [&](const unsigned char* rows, int row) INL {
        return *reinterpret_cast<const f32x4_t*>(rows + (row * 8 * KS + ((PG * s + g) ^ (row & 7))) * 16);
      };
#pragma unroll
      for (int i = 0; i < FM; ++i) {
        const f32x4_t a = at(smem, wm * TM + i * MT + r);
#pragma unroll
        for (int j = 0; j < FN; ++j) {
          const f32x4_t bb = at(Bf, wn * TN + j * MT + r);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if constexpr (SHARE) blk[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(a[e], bb[e], blk[i][j], 0, 0, 0);
            else blk[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[e], bb[e], blk[i][j], 0, 0, 0);
          }
        }
      }
    }
  };
  // each operand's tile in registers is converted and stored and the tile kt requested into its place at once
  // (neg: A's values negated)
  auto stage = [&](unsigned char* st, bool neg, int kt) INL {
    la.template store<NP, BM>(st, ha, oa, neg ? -kSplitScale : kSplitScale);
    load_a(kt);
    lb.template store<NP, BN>(st + NP * AB, hb, ob, kSplitScale);
    load_b(kt);
  };
  // k tile kt holds the own k of its rows, in a Gram product's diagonal tile
  static_assert(!GRAM || (SM && BK == BM && BM == BN), "the k of a diagonal tile's rows are one tile");
  auto own_k = [&](int kt) INL { return m0 == n0 && kbeg + kt * BK == m0; };
  // tile i belongs to a negated block
  auto odd = [&](int i) INL { return NP == 3 && SHARE && (i >> bs & 1) != 0; };
  zero();
  if (nk > 0 && (NP == 1 || !p.f32)) {
    if constexpr (SHARE) {
      // Two steps per tile: in each, one group (one wave of it per SIMD) multiplies tile kt while the other converts its
      // rows of tile kt + 1 into the other LDS stage and requests those of tile kt + 2. The stage being written is never
      // the one read in the same step, and a tile's loads have two steps to arrive.
      auto at = [&](int kt) INL { return smem + (kt & 1) * STAGE; };
      // (One loop for both: group 1 runs one tile ahead in its staging and half a step behind in its barriers.)
      load_a(0);
      load_b(0);
      for (int kt = -h; kt < nk; ++kt) {
        stage(at(kt + h), odd(kt + h), kt + h + 1);
        __syncthreads();
        if (kt >= 0) {
          mma_planes(at(kt));
          if (block_end(kt, nk)) fold(odd(kt));
          __syncthreads();
        }
      }
      if (h == 0) __syncthreads();
    } else {
      // Group h of KG takes the k tiles h, h + KG, ... through its own LDS stage, group 1 one step behind: while one
      // converts, the other multiplies. (A tile past the last is zeros.) Group 1's sums are added to group 0's.
      load_a(h);
      load_b(h);
      const int n = (nk + KG - 1) / KG;
      unsigned char* const st = smem + h * STAGE;
      if (h == 1) __syncthreads();
      for (int i = 0; i < n; ++i) {
        if (GRAM && own_k(KG * i + h)) la.clear_own();
        stage(st, odd(i), (i + 1) * KG + h);
        __syncthreads();
        mma_planes(st);
        if (block_end(i, n)) fold(odd(i));
        __syncthreads();
      }
      if (KG == 2 && h == 0) __syncthreads();
      if constexpr (SM) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) acc[i][j] += sm[i][j];
      }
      Acc* const px = reinterpret_cast<Acc*>(smem) + (tid & 255);
      if (KG == 2 && h == 1) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) px[(i * FN + j) * 256] = acc[i][j];
      }
      if constexpr (KG == 2) {
        __syncthreads();
        if (h == 0) {
#pragma unroll
          for (int i = 0; i < FM; ++i)
#pragma unroll
            for (int j = 0; j < FN; ++j) acc[i][j] += px[(i * FN + j) * 256];
        }
        __syncthreads();
      }
    }
  }
  const bool out = SHARE || h == 0;  // the wave holds results
  if constexpr (NP == 3) each_acc([&](int i, int j, int e) INL { acc[i][j][e] *= 1.f / (kSplitScale * kSplitScale); });
  if constexpr (NP == 3) {  // the same tile by fp32 MFMAs: on request, or where a sum is not finite
    bool fin = !p.f32;
    if (out) each_acc([&](int i, int j, int e) INL { fin = fin && fabsf(acc[i][j][e]) < INFINITY; });
    const bool again = __syncthreads_or(!fin);
    if constexpr (GRAM) {  // the rows' own k: one exact product, one rounding
      // element (mn, k) of A, both from m0 on, by 32-bit offsets from (m0, m0); zero past the operand's end
      constexpr bool ANY = (LAY & 4) != 0;  // rows in bf16, in either layout
      const bool mc = ANY ? oa.mode == MC : (LAY & 1) != 0;
      const int ld = (int)oa.ld, nrow = (mc ? p.K : p.M) - m0, ncol = (mc ? p.M : p.K) - m0;
      const int sm = mc ? 1 : ld, sk = mc ? ld : 1, sh = ANY ? 1 : 2;
      const __amdgpu_buffer_rsrc_t rs = make_rsrc(reinterpret_cast<const char*>(Ap) + ((m0 * (oa.ld + 1)) << sh),
                                                  ((nrow - 1) * oa.ld + ncol) << sh);
      auto at = [&](int mn, int k) INL {
        const int off = m0 + k < p.K ? (mn * sm + k * sk) << sh : kOob;
        if constexpr (ANY) return bf16_to_f32(__builtin_amdgcn_raw_buffer_load_b16(rs, off, 0, 0));
        else return __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rs, off, 0, 0));
      };
      if (!again && out && m0 == n0 && m0 < p.K) {
        float d[FM][NE];
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int e = 0; e < NE; ++e) {
            const int k = wm * TM + i * MT + acc_row(g, e);
            d[i][e] = at(k, k);
          }
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j) {
            const int mn = wn * TN + j * MT + r, k = wm * TM + i * MT + acc_row(g, 0);
            f32x4_t x;  // k .. k + 3: one load where they are neighbours (past K they are another row's)
            if constexpr (!ANY && !(LAY & 1)) x = ld_f32x4(rs, m0 + k < p.K ? (mn * ld + k) * 4 : kOob);
            else x = f32x4_t{at(mn, k), at(mn, k + 1), at(mn, k + 2), at(mn, k + 3)};
#pragma unroll
            for (int e = 0; e < NE; ++e) acc[i][j][e] = fmaf(d[i][e], m0 + k + e < p.K ? x[e] : 0.f, acc[i][j][e]);
          }
      }
    }
    if (again) {
      zero();
      for (int kt = 0; kt < nk; ++kt) {
        if (out) {
          load_a(kt);
          load_b(kt);
          la.store_f32(smem, ha, oa);
          lb.store_f32(Bf, hb, ob);
        }
        __syncthreads();
        if (out) {
          mma_f32();
          if (block_end(kt, nk)) fold(false);
        }
        __syncthreads();
      }
    }
  }

  // Epilogue through LDS (idle now), HR rows of each wave's block at a time: (1) the wave parks its accumulators in its
  // own slot; (2) row pass: 4 consecutive columns of a row per lane, the epilogue's arithmetic, C; (3) column pass: 4
  // consecutive rows of a column per lane, for the SYRK mirror and the Procrustes traces.
  constexpr int HR = cv_hr(BM), EP = TN + 4;
  float* const ep = reinterpret_cast<float*>(smem) + (SHARE ? wave : wave & 3) * HR * EP;
  float* __restrict__ C = p.C[b] + (long long)split * p.M * p.ldc;
  const float* __restrict__ X1 = p.X1[b];
  const float* __restrict__ X2 = p.X2[b];
  constexpr bool L1 = EPI == EPI_FACTOR || EPI == EPI_PROC || EPI == EPI_STRACE;
  float c0 = 0.f, c1 = 0.f;
  if constexpr (EPI != EPI_STORE && EPI != EPI_SUMSQ) c0 = p.s[b][0];
  if constexpr (EPI == EPI_FACTOR || EPI == EPI_PROC) c1 = p.s[b][1];
  const bool packed = p.tri && p.out_mode == 2, mirror = p.tri && p.out_mode == 1;
  const bool colpass = mirror || EPI == EPI_RQ || EPI == EPI_STRACE;
  const bool inside = m0 + BM <= p.M && n0 + BN <= p.N && (!p.tri || n0 >= m0 + BM) && !packed;
  float t1 = 0.f, t2 = 0.f;
  auto ld4 = [](const float* q) {
    const f32x4u_t v = *reinterpret_cast<const f32x4u_t*>(q);
    return make_float4(v[0], v[1], v[2], v[3]);
  };
  auto st4 = [](float* q, float4 v) { *reinterpret_cast<f32x4u_t*>(q) = f32x4u_t{v.x, v.y, v.z, v.w}; };

  auto half = [&](auto h_c) INL {
    constexpr int hf = decltype(h_c)::value;
    if (out) {
#pragma unroll
      for (int i = 0; i < HR / MT; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
#pragma unroll
          for (int e = 0; e < NE; ++e) ep[(i * MT + acc_row(g, e)) * EP + j * MT + r] = acc[hf * (HR / MT) + i][j][e];
    }
    __syncthreads();
    const int row0 = m0 + wm * TM + hf * HR, col0 = n0 + wn * TN;
    auto row_pass = [&](auto in_c) INL {
      constexpr bool IN = decltype(in_c)::value;
      constexpr int IT = HR * (TN / 4) / 64, U = IT < 4 ? IT : 4;
#pragma unroll 1
      for (int it0 = 0; it0 < IT; it0 += U) {
        float4 x1[U], x2[U];
        if constexpr (IN && L1) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            const int idx = lane + 64 * (it0 + u);
            const long long xo = (long long)(row0 + idx / (TN / 4)) * p.ldx + col0 + idx % (TN / 4) * 4;
            x1[u] = ld4(X1 + xo);
            if constexpr (EPI == EPI_PROC) x2[u] = ld4(X2 + xo);
          }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const int idx = lane + 64 * (it0 + u);
          const int lr = idx / (TN / 4), lc = idx % (TN / 4) * 4;
          const int row = row0 + lr, col = col0 + lc;
          float4* const slot = reinterpret_cast<float4*>(ep + lr * EP + lc);
          float v[4];
          *reinterpret_cast<float4*>(v) = *slot;
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool ok = IN || (row < p.M && col + e < p.N && !(p.tri && row > col + e));
            float q1 = 0.f, q2 = 0.f;
            if constexpr (L1) q1 = IN ? (&x1[u].x)[e] : ok ? X1[(long long)row * p.ldx + col + e] : 0.f;
            if constexpr (EPI == EPI_PROC) q2 = IN ? (&x2[u].x)[e] : ok ? X2[(long long)row * p.ldx + col + e] : 0.f;
            if constexpr (EPI == EPI_FACTOR) v[e] = q1 - c0 * (v[e] - c1 * q1);
            else if constexpr (EPI == EPI_PROC) v[e] = q1 + c0 * q2 + 0.5f * c0 * c0 * c1 * v[e];
            else if constexpr (EPI == EPI_STRACE) v[e] = (c0 * v[e]) * c0;
            else if constexpr (EPI == EPI_RQ) v[e] = c0 * v[e];
            else v[e] = p.alpha * v[e];
            if constexpr (EPI == EPI_RQ) { if (ok && row == col + e) t1 += v[e]; }
            if constexpr (EPI == EPI_SUMSQ) { if (ok) t1 += v[e] * v[e]; }
            if constexpr (EPI == EPI_STRACE) { if (ok) t2 += v[e] * q1; }
            if constexpr (EPI == EPI_STORE) {
              if (p.beta != 0.f && ok) v[e] += p.beta * C[(long long)row * p.ldc + col + e];
            }
            if constexpr (!IN) {
              if (!ok) continue;
              if (packed) C[(long long)row * p.N - (long long)row * (row - 1) / 2 + (col + e - row)] = v[e];
              else C[(long long)row * p.ldc + col + e] = v[e];
            }
          }
          const float4 o = make_float4(v[0], v[1], v[2], v[3]);
          *slot = o;
          if constexpr (IN) st4(C + (long long)row * p.ldc + col, o);
        }
      }
    };
    if (out) {
      if (inside) row_pass(std::true_type{});
      else row_pass(std::false_type{});
    }
    __syncthreads();
    if (!colpass) return;
    auto col_pass = [&](auto in_c) INL {
      constexpr bool IN = decltype(in_c)::value;
      constexpr int IT = TN * (HR / 4) / 64;
#pragma unroll 2
      for (int it = 0; it < IT; ++it) {
        const int idx = lane + 64 * it;
        const int lc = idx / (HR / 4), lr = idx % (HR / 4) * 4;
        const int col = col0 + lc, row = row0 + lr;
        float v[4];
        bool ok[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          v[e] = ep[(lr + e) * EP + lc];
          ok[e] = IN || (row + e < p.M && col < p.N && !(p.tri && row + e > col));
        }
        if constexpr (EPI == EPI_RQ || EPI == EPI_STRACE) {  // X1 at (col, row .. row + 3)
          const float* x = X1 + (long long)col * p.ldx + row;
          float4 q = make_float4(0.f, 0.f, 0.f, 0.f);
          if constexpr (IN) q = ld4(x);
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool use = ok[e] && (IN || EPI == EPI_RQ || row + e < col);  // EPI_STRACE: strictly below, mirrored
            const float xe = IN ? (&q.x)[e] : use ? x[e] : 0.f;
            if (use) t2 += EPI == EPI_RQ ? c0 * xe * v[e] : v[e] * xe;
          }
        }
        auto put = [&](float* dst) INL {  // 4 consecutive values at (col, row ..), off the diagonal
          if constexpr (IN) {
            st4(dst, make_float4(v[0], v[1], v[2], v[3]));
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              if (ok[e] && row + e != col) dst[e] = v[e];
          }
        };
        if (mirror) put(C + (long long)col * p.ldc + row);
      }
    };
    if (out) {
      if (inside) col_pass(std::true_type{});
      else col_pass(std::false_type{});
    }
    __syncthreads();
  };
  half(std::integral_constant<int, 0>{});
  if constexpr (TM > HR) half(std::integral_constant<int, 1>{});
  if constexpr (EPI == EPI_RQ || EPI == EPI_SUMSQ || EPI == EPI_STRACE) {
    __shared__ float red[16];
    t1 = block_sum(t1, red);
    if constexpr (EPI != EPI_SUMSQ) t2 = block_sum(t2, red);
    if (tid == 0) {
      p.part[b][2 * tile] = t1;
      p.part[b][2 * tile + 1] = t2;
    }
  }
}

// operands beyond plain rows (bf16 ones: plain stores of the bf16 precision)
static bool gemm_cv_any(const CvArgs& a, int prec) {
  auto any = [&](const CvOperand& o) { return (o.bf16 && !(prec == 1 && a.epi == EPI_STORE)) || o.mode == SYM || !o.vec; };
  return any(a.a) || any(a.b);
}
bool gemm_cv_wide(const CvArgs& a, int prec) {
  return !gemm_cv_any(a, prec) && !(a.a.mode == MC && a.b.mode == KC) && a.a.bf16 == a.b.bf16;
}

static void cv_tile(int cfg, int& bm, int& bn) {
  bm = cfg == 0 ? 128 : cfg == 2 ? 32 : 64;
  bn = cfg == 0 ? 256 : 64;
}

int gemm_cv_tiles(long long M, long long N, int tri, int cfg) {
  int bm, bn;
  cv_tile(cfg, bm, bn);
  const long long tm = (M + bm - 1) / bm, tn = (N + bn - 1) / bn;
  if (!tri) return (int)(tm * tn);
  long long t = 0;  // a tile row starts at the column tile that holds its first row
  for (long long i = 0; i < tm; ++i) t += tn - i * bm / bn;
  return (int)t;
}

template <int NP, int BM, int BN, int WN, int KG, int EPI, int LAY>
static hipError_t launch_cv(const CvArgs& a, hipStream_t st) {
  constexpr int smem = cv_smem(NP, BM, BN, WN, KG), nt = WN == 4 || KG == 2 ? 512 : 256;
  auto fn = gemm_cv_kernel<NP, BM, BN, WN, KG, EPI, LAY>;
  // once per instantiation (a function-local static is initialised once, also under concurrent first calls)
  static const hipError_t attr =
      hipFuncSetAttribute(reinterpret_cast<const void*>(fn), hipFuncAttributeMaxDynamicSharedMemorySize, smem);
  if (attr != hipSuccess) return attr;
  const int G = a.ntiles * a.nb * a.splitk;
  hipLaunchKernelGGL(fn, dim3(G), dim3(nt), smem, st, a);
  const hipError_t e = hipGetLastError();
  note_launch(reinterpret_cast<const void*>(fn), G, nt, smem);
  return e;
}

// Plain stores of the bf16 precision with operands in bf16 (bits 8: A, 16: B). With the storage type known only at run
// time a tile's loads had no step to arrive in: 2048^3 130 us, now 50, 16 x 4096 x 4096 172-192, now 45-52.
template <int BM, int BN, int WN, int KG, int ST>
static hipError_t launch_cv_b16(const CvArgs& a, int lay, hipStream_t st) {
  switch (lay) {
    case 0: return launch_cv<1, BM, BN, WN, KG, EPI_STORE, ST>(a, st);
    case 1:
      if constexpr (BM < 128) return launch_cv<1, BM, BN, WN, KG, EPI_STORE, ST + 1>(a, st);
      return hipErrorInvalidValue;
    case 2: return launch_cv<1, BM, BN, WN, KG, EPI_STORE, ST + 2>(a, st);
    default: return launch_cv<1, BM, BN, WN, KG, EPI_STORE, ST + 3>(a, st);
  }
}

// The layouts each epilogue's callers have: plain stores any, sums of squares (P1 X, X P2) A k-contiguous, the factor
// and Procrustes products (term1 Q, R Q, R RQ, M Q) A k- and B n-contiguous, the trace SYRK k-contiguous.
template <int NP, int BM, int BN, int WN, int KG>
static hipError_t launch_cv_epi(const CvArgs& a, hipStream_t st) {
  const int lay = (a.a.mode == MC ? 1 : 0) | (a.b.mode == MC ? 2 : 0);
  if constexpr (NP == 1) {
    if (a.a.bf16 && a.b.bf16) return launch_cv_b16<BM, BN, WN, KG, 24>(a, lay, st);
    if constexpr (BM < 128) {
      if (a.a.bf16) return launch_cv_b16<BM, BN, WN, KG, 8>(a, lay, st);
      if (a.b.bf16) return launch_cv_b16<BM, BN, WN, KG, 16>(a, lay, st);
    }
  }
  if constexpr (NP == 3 && BM == 64) {
    if (a.gram && lay == 0) return launch_cv<NP, BM, BN, WN, KG, EPI_STORE, 32>(a, st);
    if (a.gram && lay == 3) return launch_cv<NP, BM, BN, WN, KG, EPI_STORE, 35>(a, st);
  }
  if (a.epi == EPI_STORE) {
    switch (lay) {
      case 0: return launch_cv<NP, BM, BN, WN, KG, EPI_STORE, 0>(a, st);
      case 1:
        if constexpr (BM < 128) return launch_cv<NP, BM, BN, WN, KG, EPI_STORE, 1>(a, st);
        return hipErrorInvalidValue;  // its registers spill there, and no call of the optimizer has it
      case 2: return launch_cv<NP, BM, BN, WN, KG, EPI_STORE, 2>(a, st);
      default: return launch_cv<NP, BM, BN, WN, KG, EPI_STORE, 3>(a, st);
    }
  }
  if (a.epi == EPI_SUMSQ && lay == 0) return launch_cv<NP, BM, BN, WN, KG, EPI_SUMSQ, 0>(a, st);
  if (a.epi == EPI_SUMSQ && lay == 2) return launch_cv<NP, BM, BN, WN, KG, EPI_SUMSQ, 2>(a, st);
  if constexpr (BM > 32) {
    if (a.epi == EPI_FACTOR && lay == 2) return launch_cv<NP, BM, BN, WN, KG, EPI_FACTOR, 2>(a, st);
    if (a.epi == EPI_PROC && lay == 2) return launch_cv<NP, BM, BN, WN, KG, EPI_PROC, 2>(a, st);
    if (a.epi == EPI_RQ && lay == 2) return launch_cv<NP, BM, BN, WN, KG, EPI_RQ, 2>(a, st);
    if (a.epi == EPI_STRACE && lay == 0) return launch_cv<NP, BM, BN, WN, KG, EPI_STRACE, 0>(a, st);
  }
  return hipErrorInvalidValue;
}

// Operands beyond plain rows (gemm_cv_any): 64- and 32-row tiles. Beside the plain products only the factor update's A
// may be a triangle; the other epilogues' operands are fp32 rows short of 2^21 (their sides).
template <int NP, int BM, int KG>
static hipError_t launch_cv_any(const CvArgs& a, hipStream_t st) {
  if constexpr (NP == 3 && BM == 64) {
    if (a.gram) return launch_cv<NP, BM, 64, 2, KG, EPI_STORE, 36>(a, st);
  }
  switch (a.epi) {
    case EPI_STORE: return launch_cv<NP, BM, 64, 2, KG, EPI_STORE, 4>(a, st);
    case EPI_SUMSQ: return launch_cv<NP, BM, 64, 2, KG, EPI_SUMSQ, 4>(a, st);
    default: break;
  }
  if constexpr (BM > 32) {
    if (a.epi == EPI_FACTOR) return launch_cv<NP, BM, 64, 2, KG, EPI_FACTOR, 4>(a, st);
  }
  return hipErrorInvalidValue;
}

template <int NP>
static hipError_t launch_cv_cfg(const CvArgs& a, int cfg, hipStream_t st) {
  if (gemm_cv_any(a, NP == 1)) {
    if (cfg == 2) return launch_cv_any<NP, 32, 2>(a, st);
    return cfg == 3 ? launch_cv_any<NP, 64, 2>(a, st) : launch_cv_any<NP, 64, 1>(a, st);
  }
  if (cfg == 0) return launch_cv_epi<NP, 128, 256, 4, 1>(a, st);
  if (cfg == 1) return launch_cv_epi<NP, 64, 64, 2, 1>(a, st);
  if (cfg == 2) return launch_cv_epi<NP, 32, 64, 2, 2>(a, st);
  return launch_cv_epi<NP, 64, 64, 2, 2>(a, st);
}

// prec 0: fp32 (three planes), 1: bf16 (one plane). splitk > 1 and kbeg as in CvArgs.
hipError_t gemm_cv_launch(CvArgs& a, int prec, int cfg, hipStream_t st) {
  int bm, bn;
  cv_tile(cfg, bm, bn);
  a.tiles_m = (a.M + bm - 1) / bm;
  a.tiles_n = (a.N + bn - 1) / bn;
  a.ntiles = gemm_cv_tiles(a.M, a.N, a.tri, cfg);
  return prec == 1 ? launch_cv_cfg<1>(a, cfg, st) : launch_cv_cfg<3>(a, cfg, st);
}

}  // namespace psgdk
