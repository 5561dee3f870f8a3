// The K/V prologue on gfx950: two launches, both HBM-bound streaming passes.
//
//   1. stats pass  (kv_stats_kernel):  reads K and V once (with smooth_v: twice, see VMode).
//        * K: per-column fp64 partial sums over the block's rows (the smooth_k mean), written to the
//          workspace as C1 partials per plane -- no atomics, so the sum order is fixed;
//        * V: per-token scale sv = max(RN(vmax/448), 1e-12), e4m3 quantization, and the transposed
//          store V8T[d][n] through an LDS tile; SV is written; the block's max sv goes to the
//          workspace for the fold.
//   2. quant pass  (k_quant_kernel):   reads K again.
//        * reduces the C1 mean partials of its plane in a fixed order (every block gets the same
//          bits), mu = fp32(sum / N);
//        * S = max(1, max sv) from the stats partials; SV' = RN(SV / S) in place for its rows;
//        * K per-token quantization: int8 (round half to even, clamp) or e4m3.
//
// The arithmetic restates kernels/hip/h34_prologue.hip:116-211 (K and V quantizers),
// :259-282 (fp64 mean) and sageattention/sk1_backend/__init__.py:561-579 (the S fold) of the
// reference. The mean is fp64-accumulated from exactly widened inputs like the reference's; the
// summation order differs, which cannot change the bits whenever the fp64 sum is exact (fp16 data
// of magnitude below 2^10 at N below 2^19 -- every served shape of interest).
//
// Thread layout of both passes: 256 threads = CG = D/8 column groups (cg, 8 columns = one 16-byte
// load) x RG = 256/CG row groups (rg). In a step of STEP = 8*RG rows a thread holds 8 consecutive
// rows of 8 columns, so it has 8 consecutive tokens of a column (one 8-byte word of the transposed
// V tile) and 8 rows whose scales the CG lanes that share them work out together (row_absmax).
//
// What bounds the passes: HBM bandwidth, if enough bytes are in flight and the arithmetic stays
// out of the way. On gfx950 a wave64 add, multiply, fma, AND or move takes about 2.3 cycles of its
// SIMD, other VALU operations (max, min, selects, shifts, DPP moves, 16 -> 32-bit and 32 -> 64-bit
// conversions) about 4.3 and reciprocals and e4m3 packs 8.2, so the per-row work (absmax, scale,
// reciprocal) is shared out over the row's lanes and e4m3 bytes are converted two tokens at a time.
// Measured (both passes, fp16, head_dim 128, 48 planes, before / after that and the changes below):
// N = 1024 21.7 / 16.0 us, N = 8771 99.4 / 80.4 us (436 MB moved, 5.4 TB/s), N = 47520 577 / 546 us;
// 8 planes of 4096 21.1 / 11.5 us (its 96 mean partials were read one after another). A copy runs
// at 5.1-5.6 TB/s on the same card and a read at 6.2 (7.0 with nontemporal loads).
#include "sage_device.h"
#include "sage_launch.h"

namespace sage {

constexpr int PT = 256;          // threads per block

template <int D>
struct Geo {
  static constexpr int CG = D / 8, RG = PT / CG, STEP = 8 * RG, VTS = STEP + 16;
};

// Both grids are sized to one round of resident blocks on the device's compute units (a block is 4
// waves, one per SIMD; MI355X has 256 CUs): at most 128 VGPRs, so 4 blocks fit per CU, and each
// wave has 8 rows of 16-byte loads in flight (128 KB per CU). A partly filled second round costs a
// streaming pass as much as a full one. Three blocks per CU that request the next step's rows
// before they work on this one's were no faster (N = 8771: 79.5 us against 80.8).
// Each plane gets c = slots / BH blocks (at least 1) of equal row counts; a block's rows are
// a whole number of its steps (128 rows for head_dim 128, 256 for 64), so no step reaches into
// the next block's rows. A larger step, or fewer CUs, only lowers C1, so the head_dim-128
// geometry on MAX_CUS bounds the workspace for every call; a device with more CUs than that runs
// the MAX_CUS grids.
constexpr int64_t MAX_CUS = 256;
constexpr int64_t STATS_BLOCKS_PER_CU = 4;
constexpr int64_t QUANT_BLOCKS_PER_CU = 4;

PrologueGeom prologue_geom(int64_t BH, int64_t N, int64_t N_pad, int64_t step, int64_t cus) {
  auto cdiv = [](int64_t a, int64_t b) { return (a + b - 1) / b; };
  auto blocks_per_plane = [&](int64_t slots) { return BH < slots ? slots / BH : (int64_t)1; };
  const int64_t cu = (cus <= 0 || cus > MAX_CUS) ? MAX_CUS : cus;
  const int64_t Nc = cdiv(N, 64) * 64;
  PrologueGeom g;
  g.R1 = cdiv(cdiv(Nc, blocks_per_plane(cu * STATS_BLOCKS_PER_CU)), step) * step;
  g.C1 = cdiv(Nc, g.R1);
  g.R2 = cdiv(cdiv(N_pad, blocks_per_plane(cu * QUANT_BLOCKS_PER_CU)), step) * step;
  g.C2 = cdiv(N_pad, g.R2);
  return g;
}

// Workspace: K's mean partials, V's mean partials (smooth_v), the per-block max of sv -- each
// region 256-byte aligned. The V region is always reserved, so the size does not depend on flags.
static size_t part_region_bytes(int64_t BH, const PrologueGeom& g) {
  return ((size_t)BH * g.C1 * HD * sizeof(double) + 255) / 256 * 256;
}

size_t prologue_workspace_bytes(int64_t BH, int64_t N) {
  const int64_t Nc = (N + 63) / 64 * 64;
  const PrologueGeom g = prologue_geom(BH, N, Nc);
  const size_t smax = (size_t)BH * g.C1 * sizeof(float);
  return 2 * part_region_bytes(BH, g) + ((smax + 255) / 256 * 256);
}

// ---------------------------------------------------------------------------------------------
// Device pieces shared by the two passes.
// ---------------------------------------------------------------------------------------------

// 16-byte load; NT: a nontemporal one, for V, which is not read again. K's two reads are plain
// ones: what the second pass then finds in the 256 MB last-level cache is worth more (48 planes
// of 8771 rows: 80 us; all nontemporal 90, none 86).
template <typename X>
using global_ptr = const __attribute__((address_space(1))) X*;
template <bool NT, typename T>
__device__ __forceinline__ u32x4 load16(global_ptr<T> p) {
  return NT ? __builtin_nontemporal_load((global_ptr<u32x4>)p) : *(global_ptr<u32x4>)p;
}

// The 8 rows n .. n+7 at `row` (the thread's columns of row n; sr: the row stride in elements). Rows
// at or past the plane's end N read as zero. The step's pointer is opaque, so that the compiler
// forms the rows' addresses from it here instead of keeping eight running pointers in registers.
// It stays a pointer to global memory: through a generic one the loads would be flat ones, which
// waits for LDS, scalar loads and barriers would also have to drain.
// CLAMP: where the plane ends within the 8 rows, the ones past the end are read as its last row and
// cleared, for loads under conditions of their own wait for one another. For smooth_v's passes, which
// read V twice: all three passes, 200 planes of 300 rows 25.7 -> 25.1 us, 1000 of 300 72.0 -> 71.0.
// Without smooth_v it is no gain (48 planes of 4250 rows 42.9 / 42.9 us) and a loss where one row is
// left over (3000 planes of 65 51.1 -> 52.5).
template <bool NT, bool CLAMP, typename T>
__device__ __forceinline__ void load_rows(const T* row, int n, int64_t sr, int N, u32x4 (&w)[8]) {
  global_ptr<T> p = (global_ptr<T>)row;
  asm volatile("" : "+v"(p));
  if (n + 8 <= N) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = load16<NT, T>(p + i * sr);
  } else if (CLAMP && n < N) {
#pragma unroll
    for (int i = 0; i < 8; ++i) w[i] = load16<NT, T>(p + (n + i < N ? i : N - 1 - n) * sr);
#pragma unroll
    for (int i = 0; i < 8; ++i)
      if (n + i >= N) w[i] = (u32x4){0u, 0u, 0u, 0u};
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      w[i] = (n + i < N) ? load16<NT, T>(p + i * sr) : (u32x4){0u, 0u, 0u, 0u};
  }
}
template <typename T>
__device__ __forceinline__ void unpack_rows(const u32x4 (&w)[8], float (&f)[8][8]) {
#pragma unroll
  for (int i = 0; i < 8; ++i) unpack8<T>(w[i], f[i]);
}

// Two tokens' e4m3 bytes of one column into the low (HI = 0) or high half of a word. The low half
// is written first: the word has no value before it, and the convert keeps the high half of an
// operand that the next one overwrites, so a's own bits do (as in fp8x4).
template <bool HI>
__device__ __forceinline__ void fp8_pair(u32& w, float a, float b) {
  w = (u32)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, HI ? (int)w : __float_as_int(a), HI);
}

// Sum over c of part[c * D] (c = first, first + step, ...), eight loads in flight at a time.
__device__ __forceinline__ double sum_partials(const double* __restrict__ p, int first, int step,
                                               int count, int D) {
  double s = 0.0;
  int c = first;
  for (; c + 7 * step < count; c += 8 * step) {
    double v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = p[(int64_t)(c + i * step) * D];
#pragma unroll
    for (int i = 0; i < 8; ++i) s += v[i];
  }
  for (; c < count; c += step) s += p[(int64_t)c * D];
  return s;
}

// The mean of column tid % D from the plane's C1 partials, by all 256 threads: PT/D of them share a
// column, each taking every (PT/D)-th partial, and their sums are added in thread order. The order
// is fixed, so every block of a plane gets the same bits. Returns it for tid < D; `buf` holds PT
// doubles.
template <int D>
__device__ __forceinline__ float mean_of_partials(const double* __restrict__ part, int C1, int64_t N,
                                                  double* buf, int tid) {
  constexpr int W = PT / D;
  buf[tid] = sum_partials(part + tid % D, tid / D, W, C1, D);
  __syncthreads();
  double s = 0.0;
  if (tid < D) {
#pragma unroll
    for (int i = 0; i < W; ++i) s += buf[i * D + tid];
  }
  return (float)(s / (double)N);
}

// fp64 column sums of the block's rows: thread (cg, rg)'s sums of its 8 columns, added over the RG
// row groups in order and written to dst[0 .. D-1]. `red` holds RG x D doubles.
template <int D>
__device__ __forceinline__ void store_partials(const double (&s)[8], double* red, double* dst,
                                               int tid) {
  using G = Geo<D>;
  const int cg = tid % G::CG, rg = tid / G::CG;
  __syncthreads();
#pragma unroll
  for (int e = 0; e < 8; ++e) red[rg * D + 8 * cg + e] = s[e];
  __syncthreads();
  if (tid < D) {
    double t = 0.0;
#pragma unroll
    for (int r = 0; r < G::RG; ++r) t += red[r * D + tid];
    dst[tid] = t;
  }
}

template <typename T, int D, bool CLAMP>
__device__ __forceinline__ void column_sums(const T* __restrict__ p, int r_begin, int r_end,
                                            int64_t sr, int N, int rg, double (&s)[8]) {
  const int end = r_end < N ? r_end : N;
  const T* q = p + (int64_t)(r_begin + 8 * rg) * sr;
  for (int n0 = r_begin; n0 < end; n0 += Geo<D>::STEP, q += Geo<D>::STEP * sr) {
    u32x4 w[8];
    load_rows<false, CLAMP>(q, n0 + 8 * rg, sr, N, w);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      float f[8];
      unpack8<T>(w[i], f);
#pragma unroll
      for (int e = 0; e < 8; ++e) s[e] += (double)f[e];
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Stats pass. grid (C1, BH), block 256. A block first quantizes its rows of V, then sums its rows
// of K, which are then the data that the quant pass finds in the last-level cache.
// In a STEP-row step, thread (cg, rg) owns rows 8rg .. 8rg+7 and columns 8cg .. 8cg+7, so for each
// of its 8 columns it holds 8 consecutive tokens: one 8-byte word of the transposed tile. The LDS
// tile is [D d][STEP+16 B]; the 8-byte chunk of tokens 8rg..8rg+7 of row d sits at chunk position
// rg ^ (d >> 3), which spreads the column writes over the banks. The tile goes out in rows of
// 16-byte chunks, STEP/16 adjacent lanes to a row, so that a store instruction fills whole lines.
// ---------------------------------------------------------------------------------------------
// V_QUANT: V quantized as it is (and K's mean partials when smooth_k) -- the whole stats pass.
// V_SUMS: K's and V's mean partials only (smooth_v, first launch).
// V_CENTERED: V's mean from its partials (written to VMEAN), V - mean quantized (smooth_v, second
//             launch; K is not read).
// K_ONLY: K's mean partials only (the smooth_k mean on its own; V is not read).
enum VMode { V_QUANT = 0, V_SUMS = 1, V_CENTERED = 2, K_ONLY = 3 };

template <typename T, int VMODE, int D>
__global__ __launch_bounds__(PT) __attribute__((amdgpu_waves_per_eu(STATS_BLOCKS_PER_CU))) void kv_stats_kernel(
    const T* __restrict__ K, const T* __restrict__ V, u8* __restrict__ V8T, float* __restrict__ SV,
    double* __restrict__ part, double* __restrict__ vpart, float* __restrict__ VMEAN,
    float* __restrict__ smax, int64_t H, int64_t N64, int64_t Np64, int64_t R1, int64_t C1,
    int64_t k_sb, int64_t k_sh, int64_t k_sr, int64_t v_sb, int64_t v_sh, int64_t v_sr,
    int smooth_k) {
  using G = Geo<D>;
  constexpr int STEP = G::STEP, VT_STRIDE = G::VTS, RG = G::RG, CG = G::CG;
  static_assert(RG * D * sizeof(double) <= D * VT_STRIDE, "reduction buffer");
  __shared__ __attribute__((aligned(16))) u8 tile[D * VT_STRIDE];
  __shared__ float wmax[PT / 64];
  __shared__ float vmu_s[D];
  double* red = (double*)tile;  // RG x D doubles = 16 KB

  const int tid = threadIdx.x, cg = tid % CG, rg = tid / CG;
  // 1-D grid: block = bh * C1 + c (any number of planes; the block count is below 2^24)
  const u32 bh32 = blockIdx.x / (u32)C1, c32 = blockIdx.x - bh32 * (u32)C1;
  const u32 b32 = bh32 / (u32)H, h32 = bh32 - b32 * (u32)H;
  const int64_t bh = bh32, b = b32, h = h32;
  // row numbers fit 32 bits: the entry points bound N_pad by 2^31 / 128
  const int N = (int)N64, N_pad = (int)Np64;
  const int r_begin = (int)c32 * (int)R1;
  // the plane's last block also covers the pure pad rows up to N_pad
  const int r_end =
      (c32 == (u32)C1 - 1 || r_begin + (int)R1 > N_pad) ? N_pad : r_begin + (int)R1;
  const int64_t pidx = bh * C1 + c32;   // this block's partials

  if (VMODE == V_SUMS) {
    double vs[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    column_sums<T, D, VMODE == V_SUMS>(V + b * v_sb + h * v_sh + 8 * cg, r_begin, r_end, v_sr, N, rg, vs);
    store_partials<D>(vs, red, vpart + pidx * D, tid);
  }

  if (VMODE == V_QUANT || VMODE == V_CENTERED) {
    const T* vp = V + b * v_sb + h * v_sh + 8 * cg;
    u8* vt = V8T + bh * D * Np64;
    // V's sequence mean (V_CENTERED): every block of the plane reduces the same partials in the
    // same order, so all of them subtract the same bits.
    if (VMODE == V_CENTERED) {
      const float m = mean_of_partials<D>(vpart + bh * C1 * D, (int)C1, N64, red, tid);
      if (tid < D) {
        vmu_s[tid] = m;
        if (c32 == 0) VMEAN[bh * D + tid] = m;
      }
      __syncthreads();
    }
    float sv_max = 0.0f;
    const T* vq = vp + (int64_t)(r_begin + 8 * rg) * v_sr;
    float* svp = SV + bh * Np64;
    for (int n0 = r_begin; n0 < r_end; n0 += STEP, vq += STEP * v_sr) {
      const int n = n0 + 8 * rg;
      float f[8][8];
      {
        u32x4 vw[8];
        load_rows<VMODE == V_QUANT, VMODE == V_CENTERED>(vq, n, v_sr, N, vw);
        unpack_rows<T>(vw, f);
      }
      if (VMODE == V_CENTERED) {
        // read from LDS in each step: eight registers fewer across it
        int at = 8 * cg;
        asm volatile("" : "+v"(at));
        float vmu[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) vmu[e] = vmu_s[at + e];
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int e = 0; e < 8; ++e) f[i][e] -= vmu[e];
      }
      // the rows' maxima; lane l of the row group gets row l & 7's, and that row's scale
      // sv = max(RN(vmax / 448), 1e-12) and reciprocal: the row's quotients RN(v / sv) come from
      // one correctly rounded reciprocal (div_by: bit-identical to a division per element)
      const float vmax = row_absmax<CG, VMODE == V_CENTERED || std::is_same_v<T, f16>>(f, cg);
      const float sv = fmaxf(div_by(vmax, P_SCALE, RCP_P_SCALE), SCALE_FLOOR);
      const float rsv = __fdiv_rn(1.0f, sv);
      {
        const int row = n + (cg & 7);
        const float svl = row < N ? sv : 0.0f;
        if (cg < 8 && row < N_pad) svp[row] = svl;
        sv_max = fmaxf(sv_max, svl);
      }
      // e4m3 bytes, two rows (tokens) at a time: col[e] holds tokens 0..3, 4..7 of column e
      u32 col[8][2];
      static_for<0, 4>([&](auto ic) {
        constexpr int i = 2 * decltype(ic)::value;
        const float s0 = group_bcast<CG, i>(sv), s1 = group_bcast<CG, i + 1>(sv);
        const float y0 = group_bcast<CG, i>(rsv), y1 = group_bcast<CG, i + 1>(rsv);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const float a = fminf(div_by(f[i][e], s0, y0), P_SCALE);
          const float d = fminf(div_by(f[i + 1][e], s1, y1), P_SCALE);
          fp8_pair<(i & 2) != 0>(col[e][i >> 2], a, d);
        }
      });
      if (VMODE == V_CENTERED && n + 8 > N) {
        // pad rows stay zero (without a mean they are: their values are loaded as zero)
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const int left = N - (n + 4 * k);   // live tokens of this half
          const u32 keep = left >= 4 ? ~0u : left <= 0 ? 0u : (1u << (8 * left)) - 1u;
#pragma unroll
          for (int e = 0; e < 8; ++e) col[e][k] &= keep;
        }
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = 8 * cg + e;
        const int pos = rg ^ cg;  // d >> 3 == cg
        *(u32x2*)(tile + d * VT_STRIDE + 8 * pos) = (u32x2){col[e][0], col[e][1]};
      }
      __syncthreads();
      {
        // LPR lanes per row d, 16 bytes (token chunks 2j, 2j + 1) each
        constexpr int LPR = STEP / 16, RPI = PT / LPR;
        const int j = tid % LPR;
        const int nb = n0 + 16 * j;
        if (nb < N_pad) {
          u8* vo = vt + (int64_t)(tid / LPR) * Np64 + nb;
#pragma unroll
          for (int k = 0; k < D / RPI; ++k) {
            const int d = RPI * k + tid / LPR;
            const int p0 = (2 * j) ^ (d >> 3);
            u32x4 x = *(const u32x4*)(tile + d * VT_STRIDE + 8 * (p0 & ~1));
            if (p0 & 1) x = (u32x4){x.z, x.w, x.x, x.y};
            *(u32x4*)(vo + (int64_t)(RPI * k) * Np64) = x;
          }
        }
      }
      __syncthreads();
    }
    // block max of sv over live rows
    float mx = max_row16(sv_max);
#pragma unroll
    for (int o = 16; o < 64; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 64));
    if ((tid & 63) == 0) wmax[tid >> 6] = mx;
    __syncthreads();
    if (tid == 0) smax[pidx] = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  }

  if ((smooth_k && VMODE != V_CENTERED) || VMODE == K_ONLY) {
    double ks[8] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    column_sums<T, D, VMODE == V_SUMS>(K + b * k_sb + h * k_sh + 8 * cg, r_begin, r_end, k_sr, N, rg, ks);
    store_partials<D>(ks, red, part + pidx * D, tid);
  }
}

// ---------------------------------------------------------------------------------------------
// Quant pass. grid (C2, BH), block 256, the stats pass's steps and thread layout. A block requests
// its first rows of K and then reduces the partials of S and of the mean; loads return in the order
// of their requests, so the reductions begin when the rows are there. (The partials requested
// first, with eight rows by every thread, both passes: 48 planes of 1024 rows 15.4 -> 14.5 us, but
// 1000 planes of 64 rows 17.8 -> 18.4.)
// ---------------------------------------------------------------------------------------------
template <typename T, bool KINT8, int D>
__global__ __launch_bounds__(PT) __attribute__((amdgpu_waves_per_eu(QUANT_BLOCKS_PER_CU))) void k_quant_kernel(
    const T* __restrict__ K, u8* __restrict__ K8, float* __restrict__ SK, float* __restrict__ SV,
    const double* __restrict__ part, const float* __restrict__ smax, float* __restrict__ MEAN,
    float* __restrict__ S_out, float* __restrict__ KC, int64_t H, int64_t N64, int64_t Np64,
    int64_t R2, int64_t C2, int64_t C1,
    int64_t k_sb, int64_t k_sh, int64_t k_sr, int smooth_k, int fold) {
  using G = Geo<D>;
  constexpr int CG = G::CG, STEP = G::STEP;
  __shared__ double red[PT];
  __shared__ float mu_s[D];
  __shared__ float wmax[PT / 64];

  const int tid = threadIdx.x, cg = tid % CG, rg = tid / CG;
  // 1-D grid: block = bh * C2 + c2 (any number of planes; the block count is below 2^24)
  const u32 bh32 = blockIdx.x / (u32)C2, c32 = blockIdx.x - bh32 * (u32)C2;
  const u32 b32 = bh32 / (u32)H, h32 = bh32 - b32 * (u32)H;
  const int64_t bh = bh32, b = b32, h = h32;
  // row numbers fit 32 bits: the entry points bound N_pad by 2^31 / 128
  const int N = (int)N64, N_pad = (int)Np64;
  const int r_begin = (int)c32 * (int)R2;
  const int r_end = (r_begin + (int)R2 < N_pad) ? r_begin + (int)R2 : N_pad;
  const T* kq = K + b * k_sb + h * k_sh + 8 * cg + (int64_t)(r_begin + 8 * rg) * k_sr;

  u32x4 kw[8];
  load_rows<false, false>(kq, r_begin + 8 * rg, k_sr, N, kw);

  // S = max(1, max sv) and the mean
  float m = 1.0f;
  for (int i = tid; i < (int)C1; i += PT) m = fmaxf(m, smax[bh * C1 + i]);
  m = max_row16(m);
#pragma unroll
  for (int o = 16; o < 64; o <<= 1) m = fmaxf(m, __shfl_xor(m, o, 64));
  if ((tid & 63) == 0) wmax[tid >> 6] = m;
  float mean = 0.0f;   // without smooth_k: k - 0 is k
  if (smooth_k) {
    mean = mean_of_partials<D>(part + bh * C1 * D, (int)C1, N64, red, tid);
    if (MEAN != nullptr && c32 == 0 && tid < D) MEAN[bh * D + tid] = mean;
  }
  if (tid < D) mu_s[tid] = mean;
  __syncthreads();
  const float S = fmaxf(fmaxf(wmax[0], wmax[1]), fmaxf(wmax[2], wmax[3]));
  if (c32 == 0 && tid == 0) S_out[bh] = S;
  float mu[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) mu[e] = mu_s[8 * cg + e];

  float* skp = SK + bh * Np64;
  float* svp = SV + bh * Np64;
  float* kcp = KC ? KC + bh * Np64 * 2 : nullptr;
  u8* k8 = K8 + bh * Np64 * D + 8 * cg;
  // V's fold SV' = RN(SV / S) in place, and the main loop's per-key constants RN(SV'*448) (KC,
  // optional: per 64-key block 64 floats of SK and 64 of these)
  for (int row = r_begin + tid; row < r_end; row += PT) {
    const float sv = svp[row];
    const float svf = fold ? __fdiv_rn(sv, S) : sv;
    if (fold) svp[row] = svf;
    if (kcp) kcp[(row / 64) * 128 + 64 + (row & 63)] = svf * P_SCALE;
  }

  for (int n0 = r_begin; n0 < r_end; n0 += STEP) {
    const int n = n0 + 8 * rg;
    float f[8][8];
    unpack_rows<T>(kw, f);
    kq += STEP * k_sr;
#pragma unroll
    for (int i = 0; i < 8; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) f[i][e] -= mu[e];
    // row cg & 7's scale sk = max(RN(kmax / 127 or 448), 1e-12) and reciprocal
    const float kmax = row_absmax<CG, true>(f, cg);
    const float sk = fmaxf(KINT8 ? div_by(kmax, I8_MAX, RCP_I8_MAX)
                                 : div_by(kmax, P_SCALE, RCP_P_SCALE), SCALE_FLOOR);
    const float rsk = __fdiv_rn(1.0f, sk);
    const int row = n + cg;
    if (cg < 8 && row < N_pad) {
      const float ske = row < N ? sk : 1.0f;
      skp[row] = ske;
      if (kcp) kcp[(row / 64) * 128 + (row & 63)] = ske;
    }
    // the quotients RN((k - mu) / sk) of each row, and their bytes
    u8* k8r = k8 + (int64_t)n * D;
    static_for<0, 8>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const float s = group_bcast<CG, i>(sk), y = group_bcast<CG, i>(rsk);
      float x[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) x[e] = div_by(f[i][e], s, y);
      u32x2 word;
      if (KINT8) {
        word = (u32x2){i8x4(x[0], x[1], x[2], x[3]), i8x4(x[4], x[5], x[6], x[7])};
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = fminf(x[e], P_SCALE);
        word = (u32x2){fp8x4(x[0], x[1], x[2], x[3]), fp8x4(x[4], x[5], x[6], x[7])};
      }
      if (n + i >= N) word = (u32x2){0u, 0u};   // pad rows
      if (n + i < N_pad) *(u32x2*)(k8r + i * D) = word;
    });
    if (n0 + STEP < r_end) load_rows<false, false>(kq, n + STEP, k_sr, N, kw);
  }
}

template <typename T, int D>
static hipError_t launch_prologue_t(const PrologueArgs& a, hipStream_t stream) {
  const int64_t BH = a.B * a.H;
  const PrologueGeom g = prologue_geom(BH, a.N, a.N_pad, Geo<D>::STEP, a.cus);
  // region offsets as sized for head_dim 128 (prologue_workspace_bytes)
  const size_t part_bytes = part_region_bytes(BH, prologue_geom(BH, a.N, a.N_pad));
  double* part = (double*)a.workspace;
  double* vpart = (double*)((char*)a.workspace + part_bytes);
  float* smax = (float*)((char*)a.workspace + 2 * part_bytes);
  const dim3 grid1((unsigned)(g.C1 * BH));
  if (a.smooth_v) {
    // V's mean first (with K's partials), then V - mean quantized
    hipLaunchKernelGGL((kv_stats_kernel<T, V_SUMS, D>), grid1, dim3(PT), 0, stream, (const T*)a.k,
                       (const T*)a.v, (u8*)a.v8t, a.sv, part, vpart, a.vmean, smax, a.H, a.N,
                       a.N_pad, g.R1, g.C1, a.k_sb, a.k_sh, a.k_sr, a.v_sb, a.v_sh, a.v_sr,
                       a.smooth_k);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL((kv_stats_kernel<T, V_CENTERED, D>), grid1, dim3(PT), 0, stream,
                       (const T*)a.k, (const T*)a.v, (u8*)a.v8t, a.sv, part, vpart, a.vmean, smax,
                       a.H, a.N, a.N_pad, g.R1, g.C1, a.k_sb, a.k_sh, a.k_sr, a.v_sb, a.v_sh,
                       a.v_sr, a.smooth_k);
  } else {
    hipLaunchKernelGGL((kv_stats_kernel<T, V_QUANT, D>), grid1, dim3(PT), 0, stream, (const T*)a.k,
                       (const T*)a.v, (u8*)a.v8t, a.sv, part, vpart, a.vmean, smax, a.H, a.N,
                       a.N_pad, g.R1, g.C1, a.k_sb, a.k_sh, a.k_sr, a.v_sb, a.v_sh, a.v_sr,
                       a.smooth_k);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const dim3 grid2((unsigned)(g.C2 * BH));
  if (a.k_int8)
    hipLaunchKernelGGL((k_quant_kernel<T, true, D>), grid2, dim3(PT), 0,
                       stream, (const T*)a.k, (u8*)a.k8, a.sk, a.sv, part, smax, a.mean, a.s, a.kconst, a.H,
                       a.N, a.N_pad, g.R2, g.C2, g.C1, a.k_sb, a.k_sh, a.k_sr, a.smooth_k, a.fold);
  else
    hipLaunchKernelGGL((k_quant_kernel<T, false, D>), grid2, dim3(PT), 0,
                       stream, (const T*)a.k, (u8*)a.k8, a.sk, a.sv, part, smax, a.mean, a.s, a.kconst, a.H,
                       a.N, a.N_pad, g.R2, g.C2, g.C1, a.k_sb, a.k_sh, a.k_sr, a.smooth_k, a.fold);
  return hipGetLastError();
}

// MEAN from the stats pass's K partials: the reduction of k_quant_kernel (same order, same
// rounding), one block per plane.
template <int D>
__global__ __launch_bounds__(PT) void mean_reduce_kernel(const double* __restrict__ part,
                                                        float* __restrict__ MEAN, int64_t N,
                                                        int64_t C1) {
  __shared__ double red[PT];
  const int64_t bh = blockIdx.x;
  const int tid = threadIdx.x;
  const float mean = mean_of_partials<D>(part + bh * C1 * D, (int)C1, N, red, tid);
  if (tid < D) MEAN[bh * D + tid] = mean;
}

template <typename T, int D>
static hipError_t launch_kseq_mean_t(const PrologueArgs& a, hipStream_t stream) {
  const int64_t BH = a.B * a.H;
  const PrologueGeom g = prologue_geom(BH, a.N, a.N_pad, Geo<D>::STEP, a.cus);
  double* part = (double*)a.workspace;
  hipLaunchKernelGGL((kv_stats_kernel<T, K_ONLY, D>), dim3((unsigned)(g.C1 * BH)), dim3(PT), 0,
                     stream, (const T*)a.k, (const T*)a.k, nullptr, nullptr, part, nullptr, nullptr,
                     nullptr, a.H, a.N, a.N_pad, g.R1, g.C1, a.k_sb, a.k_sh, a.k_sr, a.k_sb,
                     a.k_sh, a.k_sr, 1);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL((mean_reduce_kernel<D>), dim3((unsigned)BH), dim3(PT), 0, stream, part, a.mean,
                     a.N, g.C1);
  return hipGetLastError();
}

hipError_t launch_kseq_mean(const PrologueArgs& a, hipStream_t stream) {
  if (a.D == 64)
    return a.dtype == 1 ? launch_kseq_mean_t<bf16, 64>(a, stream)
                        : launch_kseq_mean_t<f16, 64>(a, stream);
  return a.dtype == 1 ? launch_kseq_mean_t<bf16, 128>(a, stream)
                      : launch_kseq_mean_t<f16, 128>(a, stream);
}

hipError_t launch_prologue(const PrologueArgs& a, hipStream_t stream) {
  if (a.D == 64)
    return a.dtype == 1 ? launch_prologue_t<bf16, 64>(a, stream)
                        : launch_prologue_t<f16, 64>(a, stream);
  return a.dtype == 1 ? launch_prologue_t<bf16, 128>(a, stream)
                      : launch_prologue_t<f16, 128>(a, stream);
}

}  // namespace sage
