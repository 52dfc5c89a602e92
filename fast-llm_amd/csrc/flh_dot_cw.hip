// flh_dot_cw.hip -- several activation columns (speculative verify, grouped
// MoE experts) on the int8 matrix cores, one accumulator chain per wave.
//
// The reference folds a row's integer dots into four independent chains,
// a[b & 3] over its blocks b (32 weights for Q8_0 / Q5_0 / IQ, a superblock of 256
// for Q4_K / Q6_K), and adds (a0 + a1) + (a2 + a3) at the end
// (src/runtime/quants.h:438-594).  Here a workgroup of four waves owns 16 rows
// at a time and wave k runs chain k of all of them, so a chain is a register
// from the first block to the last and its order is the reference's: every
// output is bitwise the single-column result.
//
// The four waves share one ring of chunks.  A chunk is a run of 16 rows'
// consecutive blocks (Q8_0, Q5_0: 512 columns, 4 blocks per wave; Q4_K, Q6_K:
// 1024 columns, one superblock per wave), 352-840 contiguous bytes per row,
// followed by the same columns' quantised activations: a chunk brings
// everything its multiplications read, and rows of any length take this
// kernel.  Pieces of this size stream at the rate of contiguous memory (16 x
// 144 bytes stop at 4.4 TB/s).
//
// A fifth wave issues the chunks by direct-to-LDS 16-byte loads, D - 1 ahead,
// and waits for them; one barrier per chunk publishes it and frees the stage
// read before.  The four consumers then run nothing but LDS reads, matrix
// instructions and their chain.  With the loads dealt to the consumers, their
// issue, waits and branches sat on every chunk's critical path (one wave per
// SIMD where a matrix has one tile per CU): Q8_0 4096x14336 with 4 columns
// 21.5 us, 15.0 with the producer; streaming alone takes 13.8.
//
// The A operand is block-diagonal: row n holds column n / 4 of a group of 4
// on k-slice n % 4 only (Q6_K: column n / 2 of 8 on the slices of sub-block n %
// 2), so 16-lane row j of the result holds column j's dots with the four blocks
// of lane rows 0-3: Q8_0 / Q5_0 the chain's four blocks in the chunk, in order
// (their scales are gathered from the lane rows once per chunk, for all
// columns), Q4_K the superblock's sub-blocks, scaled and added as integers.  With
// column n % 4 on slice n / 4 (each lane row its own block's dots) results and
// scales had to be transposed per group, eight lane-row swaps: Q8_0 28672x4096
// with 16 columns 34.6 -> 32.8 us, IQ2_XXS 4096x14336 29.0 -> 25.4, Q4_K 16.4 ->
// 14.9, Q6_K vocabulary 128256x4096 with 5 / 16 columns 89.9 -> 88.9, 120 -> 114.
// A lane reads one block's contiguous bytes; 8 bytes of every block per lane (a
// plain A operand) took 742 LDS cycles per chunk instead of about 140.  (Rows r and
// r + 8 of a Q8_0 or Q6_K stage share banks: 65 % of the LDS-active cycles are
// conflicts, about 540 cycles a wave of Q8_0 14336x4096 with 4 columns; Q4_K 37 %.)
//
// IQ2_XXS / IQ3_XXS: 1024 columns a chunk, 8 blocks per wave in two halves that
// run as Q8_0's; a lane expands its block from the codebook and a table of sign
// masks in LDS (the consumers copy both in while the first chunks fly).  Rows lie
// at 2-byte offsets, so a row of any number of superblocks is taken from the
// 16-byte boundary below, as Q6_K's.  Bound by the expansion and the folds:
// 28672x4096 IQ2_XXS with 4 / 8 / 16 columns 20.6 / 28.6 / 42 us, 27.6 / 41 / 82 one
// lane per half superblock; 3840x3840 with 16 columns 44 -> 10.2 (register kernel before);
// six of 64 experts of 1536x2560, 3 tokens: 237 -> 60 us a layer.
//
// Bound by the weight stream with few columns (28672x4096 Q8_0 with 4 24.2 us, 5.2
// TB/s; streaming the chunks alone takes 25.1 where the whole kernel took 25.9), by
// the consumers beyond: with 16 columns 32.8 us, and staging fewer activation
// bytes (32-row tiles, or only the columns that are there) changes nothing.
#include "flh_kstream.h"
#include "flh_internal.h"
#include "flh_status.h"

namespace flh {

typedef int v4i __attribute__((ext_vector_type(4)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// cache policy of the weight DMA (2 = nontemporal)
constexpr int CW_AUX = 2;

// UB: weight bytes per 256 columns; CU: 256-column units per chunk; WSEG:
// 16-byte segments of a row's chunk (Q6_K, IQ2_XXS, IQ3_XXS: its bytes from a
// 16-byte boundary up to 14 bytes below); UA: appendix bytes per unit; ASEG: segments per
// column of a chunk's activations.
template <int FMT> struct CW;
template <> struct CW<FMT_Q8_0> { static constexpr uint32_t UB = 272, CU = 2, WSEG = 34, UA = 288, ASEG = 36; };
template <> struct CW<FMT_Q5_0> { static constexpr uint32_t UB = 176, CU = 2, WSEG = 22, UA = 288, ASEG = 36; };
template <> struct CW<FMT_Q4_K> { static constexpr uint32_t UB = 144, CU = 4, WSEG = 36, UA = 292, ASEG = 73; };
template <> struct CW<FMT_Q6_K> { static constexpr uint32_t UB = 210, CU = 4, WSEG = 54, UA = 292, ASEG = 73; };
template <> struct CW<FMT_IQ2_XXS> { static constexpr uint32_t UB = 66, CU = 4, WSEG = 18, UA = 288, ASEG = 72; };
template <> struct CW<FMT_IQ3_XXS> { static constexpr uint32_t UB = 98, CU = 4, WSEG = 26, UA = 288, ASEG = 72; };
// the codebook formats; the formats whose superblocks are 2-byte aligned
__host__ __device__ constexpr bool cw_iq(int fmt) { return fmt == FMT_IQ2_XXS || fmt == FMT_IQ3_XXS; }
__host__ __device__ constexpr bool cw_gran(int fmt) { return fmt == FMT_Q6_K || cw_iq(fmt); }

// DMA instructions of a chunk: the rows' segments, the columns' segments, and
// (32-weight blocks) the blocks' {d, s} words of every column again, as a
// table [column][16 blocks][chain][4] whose four words a lane reads at once.
template <int FMT, int NC> struct CwPlan {
    static constexpr bool KF = FMT == FMT_Q4_K || FMT == FMT_Q6_K;
    static constexpr uint32_t NW = (16 * CW<FMT>::WSEG + 63) / 64, NA = (NC * CW<FMT>::ASEG + 63) / 64;
    static constexpr uint32_t NX = KF ? 0 : NC * CW<FMT>::CU / 8, NT = NW + NA + NX;
    static constexpr uint32_t XOFF = (NW + NA) * 1024, STG = XOFF + NX * 256;
};
// A chunk of `units` 256-column units of a column is staged in 16-byte pieces
// that end where its bytes end, and so begin up to 12 bytes below it (q8_K: 292
// bytes a unit; a whole chunk is whole pieces): nothing is read past the column,
// wherever it lies (K formats: at any 4-byte boundary, where 16-byte
// direct-to-LDS loads are as fast).
template <int FMT> __device__ __forceinline__ uint32_t cw_xshift(uint32_t units) { return (0u - units * CW<FMT>::UA) & 15u; }
constexpr uint32_t CW_WAVES = 5;                                  // four consumers and the producer
constexpr uint32_t CW_ZERO = 320;                                 // zero bytes that off-diagonal lanes read
// LDS: [D][STG] ring | [4][16][16] sums | zeros | codebook (2 KiB), sign masks (1 KiB)
template <int FMT, int NC> __host__ __device__ constexpr size_t cw_smem(int D) {
    return (size_t)D * CwPlan<FMT, NC>::STG + 4096 + CW_ZERO + (cw_iq(FMT) ? 3072 : 0);
}

// Activation column p starts xoff(p) bytes after base() (the launcher bounds
// the offsets to 32 bits), output column p at y(p).
struct CwColsStrided {
    const float * x0;
    float * y0;
    uint32_t xs, ys;
    __device__ const float * base() const { return x0; }
    __device__ uint32_t xoff(uint32_t p) const { return p * xs * 4; }
    __device__ float * y(uint32_t p) const { return y0 + (size_t)p * ys; }
};
struct CwColsMoe {
    const float * x0;
    float * y0;
    uint32_t xs, ys;
    const uint32_t * xi;                                          // __shared__ [NC]
    const uint32_t * yi;                                          // __shared__ [NC]
    __device__ const float * base() const { return x0; }
    __device__ uint32_t xoff(uint32_t p) const { return lds_ld32(&xi[p]) * xs * 4; }
    __device__ float * y(uint32_t p) const { return y0 + (size_t)lds_ld32(&yi[p]) * ys; }
};

// All four 16-lane rows' values: g[t] = the v of lane row t.
__device__ __forceinline__ void cw_gather(uint32_t v, uint32_t (&g)[4]) {
    const auto a = __builtin_amdgcn_permlane32_swap(v, v, false, false);   // rows 0 1 0 1, 2 3 2 3
    const auto b = __builtin_amdgcn_permlane16_swap(a[0], a[0], false, false);
    const auto c = __builtin_amdgcn_permlane16_swap(a[1], a[1], false, false);
    g[0] = b[0]; g[1] = b[1]; g[2] = c[0]; g[3] = c[1];
}
// d_w * d_x of two halves (the low or the high one of a, the low one of b) as
// binary32: exact (22 significant bits), so the same as the product of the
// widened values; as a mixed-precision fma with nz = -0.0 (kept opaque) it is
// one instruction instead of two conversions and a multiplication.
// (cw_fmul: of a binary32 and a half, rounded once)
__device__ __forceinline__ float cw_fmul(uint32_t a, uint32_t b, float nz) {
    typedef _Float16 h2v __attribute__((ext_vector_type(2)));
    return __builtin_fmaf(__uint_as_float(a), (float)__builtin_bit_cast(h2v, b).x, nz);
}
template <bool HI>
__device__ __forceinline__ float cw_hmul(uint32_t a, uint32_t b, float nz) {
    typedef _Float16 h2v __attribute__((ext_vector_type(2)));
    const h2v x = __builtin_bit_cast(h2v, a), y = __builtin_bit_cast(h2v, b);
    return __builtin_fmaf((float)(HI ? x.y : x.x), (float)y.x, nz);
}
// dwords at an LDS offset
typedef const __attribute__((address_space(3))) uint32_t * lds32;
typedef const __attribute__((address_space(3))) u32x2 * lds64;
typedef const __attribute__((address_space(3))) uint16_t * lds16;
typedef __attribute__((address_space(3))) uint32_t * lds32w;
typedef __attribute__((address_space(3))) u32x2 * lds64w;
__device__ __forceinline__ lds32 lp32(uint32_t off) { return (lds32)(uintptr_t)off; }
__device__ __forceinline__ u32x2 lp64(uint32_t off) { return *(lds64)(uintptr_t)off; }

// at most `behind` (<= B) chunks of N DMA instructions outstanding
template <int B, int N>
__device__ __forceinline__ void cw_wait(uint32_t behind) {
    if (behind >= (uint32_t)B) {
        WAIT_VM(B * N);
        return;
    }
    if constexpr (B > 0) cw_wait<B - 1, N>(behind);
}

// The thread's index, opaque: a kernel that holds several forms of the body
// must not compute all their addresses up front (230 registers, one workgroup
// per CU).
__device__ __forceinline__ uint32_t cw_tid() {
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));
    return t;
}

// The producer wave: streams the chunks of rows [rbeg, rend), D - 1 ahead.
// vo: per instruction the lane's byte offset from the chunk's start in the
// tile's first row (rows), or in column 0's appendix (columns, table); the
// chunk's own start is scalar, so a chunk costs no vector work.
template <int FMT, int NC, int D, typename COLS>
__device__ __forceinline__ void cw_produce(const uint8_t * __restrict__ w, uint32_t cols, const COLS & C, uint32_t nx,
                                           uint32_t rbeg, uint32_t rend, uint8_t * sm) {
    using P = CW<FMT>;
    using L = CwPlan<FMT, NC>;
    constexpr bool KF = L::KF;
    constexpr uint32_t NT = L::NT, STG = L::STG, NW = L::NW, NA = L::NA;
    constexpr uint32_t CB = P::CU * P::UB, CA = P::CU * P::UA;
    static_assert((D - 2) * (int)NT <= 60, "vmcnt counts to 63");
    const uint32_t lane = cw_tid() & 63;
    const uint32_t nsb = cols >> 8, nch = (nsb + P::CU - 1) / P::CU, lastu = nsb - (nch - 1) * P::CU;
    const uint32_t RB = nsb * P::UB, ntile = (rend - rbeg + 15) >> 4, total = ntile * nch;
    const uint8_t * const x0 = reinterpret_cast<const uint8_t *>(C.base()) + (KF ? xqk_off(cols) : xq_off(cols));
    constexpr uint32_t ALIM = 16 * P::ASEG - 16;                  // a column's last segment
    uint32_t vo[NT];
    auto w_off = [&](uint32_t ln, uint32_t q, uint32_t nv, uint32_t lim) -> uint32_t {
        const uint32_t s = min(64 * q + ln, 16 * P::WSEG - 1);
        return min(s / P::WSEG, nv) * RB + (cw_gran(FMT) ? 0u : min(16 * (s % P::WSEG), lim));
    };
    auto a_off = [&](uint32_t ln, uint32_t q, uint32_t lim) -> uint32_t {
        const uint32_t s = min(64 * (q - NW) + ln, NC * P::ASEG - 1), n = s / P::ASEG;
        return C.xoff(n < nx ? n : 0) + min(16 * (s % P::ASEG), lim);
    };
    auto x_off = [&](uint32_t ln, uint32_t q, uint32_t lim) -> uint32_t {
        const uint32_t e = 64 * (q - NW - NA) + ln, n = e / (8 * P::CU), i = e % (8 * P::CU);
        return C.xoff(n < nx ? n : 0) + 36 * min((i & ~15u) + 4 * (i & 3) + ((i >> 2) & 3), lim);
    };
#pragma unroll
    for (uint32_t q = NW; q < NT; ++q) vo[q] = q < NW + NA ? a_off(lane, q, ALIM) : x_off(lane, q, 8 * P::CU - 1);
    uint32_t qt = 0, qc = 0, qslot = 0;                           // next chunk to issue
    auto issue_next = [&]() __attribute__((always_inline)) {
        if (qt >= ntile) return;
        const uint32_t row0 = rbeg + 16 * qt, nv = min(15u, rend - 1 - row0);   // nv: last row of the tile
        if (qc == 0 && (qt == 0 || nv < 15)) {                    // the offsets differ only in a partial tile
#pragma unroll
            for (uint32_t q = 0; q < NW; ++q) vo[q] = w_off(lane, q, nv, 0xFFFFu);
        }
        uint8_t * stage = sm + (size_t)qslot * STG;
        const uint8_t * wb = w + (size_t)row0 * RB + (size_t)qc * CB;
        const uint8_t * xb = x0 + (size_t)qc * CA - (qc + 1 < nch ? 0u : cw_xshift<FMT>(lastu));
        if (qc + 1 < nch || lastu == P::CU || cw_gran(FMT)) {
            const uint32_t sh = (uint32_t)(uintptr_t)wb & 15u;    // the chunk's offset in its granule
            const bool part = qc + 1 == nch && lastu < P::CU;     // (these formats only)
            const uint32_t wbytes = (part ? lastu : P::CU) * P::UB;
            uint32_t ln = lane;
            asm volatile("" : "+v"(ln));                          // (see below)
#pragma unroll
            for (uint32_t q = 0; q < NW; ++q) {
                if constexpr (cw_gran(FMT)) {
                    // segments from the boundary below the row's chunk to the
                    // granule of its last byte
                    const uint32_t s = min(64 * q + lane, 16 * P::WSEG - 1) % P::WSEG;
                    const uint32_t o = min(((sh + vo[q]) & ~15u) + 16 * s, (sh + vo[q] + wbytes - 1) & ~15u);
                    __builtin_amdgcn_global_load_lds(GPTR(wb - sh + o), LPTR(stage + 1024 * q), 16, 0, CW_AUX);
                } else {
                    __builtin_amdgcn_global_load_lds(GPTR(wb + vo[q]), LPTR(stage + 1024 * q), 16, 0, CW_AUX);
                }
            }
#pragma unroll
            for (uint32_t q = NW; q < NW + NA; ++q)
                __builtin_amdgcn_global_load_lds(GPTR(xb + (part ? a_off(ln, q, (lastu * P::UA - 1) & ~15u) : vo[q])),
                                                 LPTR(stage + 1024 * q), 16, 0, 0);
#pragma unroll
            for (uint32_t q = NW + NA; q < NT; ++q)
                __builtin_amdgcn_global_load_lds(GPTR(xb + (part ? x_off(ln, q, 8 * lastu - 1) : vo[q])),
                                                 LPTR(stage + L::XOFF + 256 * (q - NW - NA)), 4, 0, 0);
        } else {                                                  // a partial last chunk: no read past the row or column
            // its offsets are made anew (the opaque lane): kept next to the whole
            // chunk's they took the producer over 128 registers, and waves that
            // need more leave a CU one workgroup (Q4_K 28672x4096 with 16 columns
            // 31.7 us, 24.9 within 128)
            uint32_t ln = lane;
            asm volatile("" : "+v"(ln));
#pragma unroll
            for (uint32_t q = 0; q < NW; ++q)
                __builtin_amdgcn_global_load_lds(GPTR(wb + w_off(ln, q, nv, lastu * P::UB - 16)), LPTR(stage + 1024 * q), 16, 0,
                                                 CW_AUX);
#pragma unroll
            for (uint32_t q = NW; q < NW + NA; ++q)
                __builtin_amdgcn_global_load_lds(GPTR(xb + a_off(ln, q, (lastu * P::UA - 1) & ~15u)), LPTR(stage + 1024 * q), 16,
                                                 0, 0);
#pragma unroll
            for (uint32_t q = NW + NA; q < NT; ++q)
                __builtin_amdgcn_global_load_lds(GPTR(xb + x_off(ln, q, 8 * lastu - 1)),
                                                 LPTR(stage + L::XOFF + 256 * (q - NW - NA)), 4, 0, 0);
        }
        qslot = qslot + 1 == (uint32_t)D ? 0 : qslot + 1;
        if (++qc == nch) { qc = 0; ++qt; }
    };
#pragma unroll 1
    for (int d = 0; d + 1 < D; ++d) issue_next();
    uint32_t c = 0;
#pragma unroll 1
    for (uint32_t g = 0; g < total; ++g) {
        cw_wait<D - 2, (int)NT>(min(total - 1 - g, (uint32_t)(D - 2)));
        lds_barrier();                                            // chunk g is whole; chunk g - 1 has been read
        issue_next();
        if (++c == nch) { c = 0; lds_barrier(); }                 // the consumers' sums
    }
}

// The consumer waves: wave k runs chain k of 16 rows at a time.
template <int FMT, int NC, int D, typename COLS>
__device__ __forceinline__ void cw_consume(const uint8_t * __restrict__ w, uint32_t cols, const COLS & C, uint32_t nx,
                                           uint32_t rbeg, uint32_t rend, uint8_t * sm) {
    using P = CW<FMT>;
    using L = CwPlan<FMT, NC>;
    constexpr bool KF = L::KF;
    constexpr uint32_t STG = L::STG, WROW = 16 * P::WSEG, AROW = 16 * P::ASEG, CB = P::CU * P::UB;
    const uint32_t tid = cw_tid(), lane = tid & 63;
    const uint32_t k = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint32_t r = lane & 15, j = lane >> 4;
    const uint32_t nsb = cols >> 8, nch = (nsb + P::CU - 1) / P::CU, lastu = nsb - (nch - 1) * P::CU;
    const uint32_t RB = nsb * P::UB, ntile = (rend - rbeg + 15) >> 4;
    float * AC = reinterpret_cast<float *>(sm + (size_t)D * STG);     // [4][16 columns][16 rows]
    const uint32_t zr = lds_off(reinterpret_cast<uint8_t *>(AC) + 4096);
    constexpr int NG = FMT == FMT_Q6_K ? (NC == 16 ? 2 : 1) : NC / 4;   // groups of 8 (Q6_K) or 4 columns
    constexpr int NACC = FMT == FMT_Q6_K ? 2 * NG : NG;
    float acc[NACC];
    // the lane's i-th output column
    auto col_of = [&](int i) -> uint32_t {
        if constexpr (FMT != FMT_Q6_K) return 4 * i + j;
        else return 8 * (i >> 1) + 2 * j + (i & 1);
    };
    [[maybe_unused]] float nz = -0.0f;
    asm volatile("" : "+v"(nz));                                  // kept as a register
    const uint32_t p = tid >> 4;                                  // this thread's (column, row) of the sums
    uint32_t slot = 0;
    [[maybe_unused]] const uint32_t grid = zr + CW_ZERO;
    if constexpr (cw_iq(FMT)) {                                   // (read after the first chunk's barrier)
        if constexpr (FMT == FMT_IQ2_XXS) {
            *(lds64w)(uintptr_t)(grid + 8 * tid) = u32x2{(uint32_t)k_iq2_grid[tid], (uint32_t)(k_iq2_grid[tid] >> 32)};
        } else {
            *(lds32w)(uintptr_t)(grid + 4 * tid) = k_iq3_grid[tid];
        }
        const uint32_t sg = iq_sign8(tid & 127u);
        *(lds64w)(uintptr_t)(grid + 2048 + 8 * (tid & 127u)) = u32x2{iq_neg4(sg), iq_neg4(sg >> 4)};
    }
    for (uint32_t t = 0; t < ntile; ++t) {
        const uint32_t row = rbeg + 16 * t + (tid & 15);
        const bool mine = p < nx && row < rend;
        // (every thread loads: a guarded load would be waited for here)
        float * const yp = C.y(min(p, nx - 1)) + min(row, rend - 1);
        const float y0 = *yp;
#pragma unroll
        for (int i = 0; i < NACC; ++i) acc[i] = 0.f;
        for (uint32_t c = 0; c < nch; ++c) {
            lds_barrier();
            const uint32_t st = lds_off(sm + (size_t)slot * STG);
            const uint32_t units = c + 1 == nch ? lastu : P::CU;
            const uint32_t xs = st + 1024 * L::NW + cw_xshift<FMT>(units), xt = st + L::XOFF;   // the columns, the table
            slot = slot + 1 == (uint32_t)D ? 0 : slot + 1;
            if constexpr (cw_iq(FMT)) {
                // lane (r, j): blocks b = 16 h + 4 j + k of row r, group 4 (j & 1) + k
                // of superblock 2 h + j / 2; the row's chunk starts sh bytes into its window
                const uint32_t wrow = min(rbeg + 16 * t + r, rend - 1);
                const uint32_t sh = ((uint32_t)(uintptr_t)w + wrow * RB + c * CB) & 15u;
                const bool diag = (r & 3) == j;
#pragma unroll
                for (uint32_t h = 0; h < 2; ++h) {
                    if (2 * h >= units) break;
                    const uint32_t g = 4 * (j & 1) + k, sb = st + r * WROW + sh + P::UB * (2 * h + (j >> 1));
                    const uint32_t hd = *(lds16)(uintptr_t)sb;
                    // w1 and the grid indices, from aligned dwords
                    const uint32_t ga = sb + 2 + 8 * g, s2 = ga & 2u;
                    const lds32 gp = lp32(ga - s2);
                    const uint32_t i0 = alignb(gp[1], gp[0], s2);
                    uint32_t w1 = alignb(gp[2], gp[1], s2), E[8];
                    if constexpr (FMT == FMT_IQ2_XXS) {           // an 8-byte entry per run
#pragma unroll
                        for (int l = 0; l < 4; ++l) {
                            const u32x2 e = lp64(grid + 8 * ((i0 >> (8 * l)) & 0xFFu));
                            E[2 * l] = e.x;
                            E[2 * l + 1] = e.y;
                        }
                    } else {                                      // two 4-byte entries per run
                        const uint32_t i1 = w1;
                        const lds32 wp = lp32(ga - s2 + 64 - 4 * g);
                        w1 = alignb(wp[1], wp[0], s2);
#pragma unroll
                        for (int l = 0; l < 8; ++l)
                            E[l] = *lp32(grid + 4 * (((l < 4 ? i0 : i1) >> (8 * (l & 3))) & 0xFFu));
                    }
#pragma unroll
                    for (int l = 0; l < 4; ++l) {
                        const u32x2 n = lp64(grid + 2048 + 8 * ((w1 >> (7 * l)) & 127u));
                        E[2 * l] = iq_apply(E[2 * l], n.x);
                        E[2 * l + 1] = iq_apply(E[2 * l + 1], n.y);
                    }
                    uint32_t db[4];
                    cw_gather(__float_as_uint(iq_db(FMT, h2f(hd), w1)), db);
                    const v4i b0 = {(int)E[0], (int)E[1], (int)E[2], (int)E[3]}, b1 = {(int)E[4], (int)E[5], (int)E[6], (int)E[7]};
#pragma unroll
                    for (int gr = 0; gr < NG; ++gr) {             // A as for Q8_0 below
                        const lds32 ap = lp32(diag ? xs + (4 * gr + (r >> 2)) * AROW + 36 * (16 * h + 4 * j + k) + 4 : zr);
                        const v4i a0 = {(int)ap[0], (int)ap[1], (int)ap[2], (int)ap[3]};
                        const v4i a1 = {(int)ap[4], (int)ap[5], (int)ap[6], (int)ap[7]};
                        const u32x4a dx = *(const __attribute__((address_space(3))) u32x4a *)(uintptr_t)(
                            xt + 32 * P::CU * (4 * gr + j) + 64 * h + 16 * k);
                        v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0, v4i{0, 0, 0, 0}, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1, d, 0, 0, 0);
                        acc[gr] = fmaf(cw_fmul(db[0], dx[0], nz), (float)d[0], acc[gr]);
                        acc[gr] = fmaf(cw_fmul(db[1], dx[1], nz), (float)d[1], acc[gr]);
                        const float a2 = fmaf(cw_fmul(db[2], dx[2], nz), (float)d[2], acc[gr]);
                        const float a3 = fmaf(cw_fmul(db[3], dx[3], nz), (float)d[3], a2);
                        acc[gr] = units > 2 * h + 1 ? a3 : acc[gr];   // (blocks 2 and 3 lie in the second superblock)
                    }
                }
            } else if constexpr (!KF) {
                // lane (r, j): block b = 4 j + k of row r
                auto chain = [&](auto kc) __attribute__((always_inline)) {
                    constexpr int K = decltype(kc)::value, BB = FMT == FMT_Q8_0 ? 34 : 22;
                    constexpr int B8 = (BB * K) & ~7, O = BB * K - B8;   // the block starts O bytes into its window
                    uint32_t W[10];
#pragma unroll
                    for (int i = 0; i < (FMT == FMT_Q8_0 ? 5 : 4); ++i) {
                        const u32x2 v = lp64(st + r * WROW + 4 * BB * j + B8 + 8 * i);
                        W[2 * i] = v.x;
                        W[2 * i + 1] = v.y;
                    }
                    constexpr int QO = O + (FMT == FMT_Q8_0 ? 2 : 6), Q0 = QO >> 2, QS = QO & 3;   // quants
                    auto word = [&](int i, int o0, int os) -> uint32_t {
                        return os ? alignb(W[o0 + i + 1], W[o0 + i], os) : W[o0 + i];
                    };
                    uint32_t B[8];
                    if constexpr (FMT == FMT_Q8_0) {
#pragma unroll
                        for (int i = 0; i < 8; ++i) B[i] = word(i, Q0, QS);
                    } else {
                        constexpr int HO = O + 2;
                        const uint32_t qh = word(0, HO >> 2, HO & 3);
#pragma unroll
                        for (int i = 0; i < 8; ++i) {             // elements 16..31: the high nibbles
                            const uint32_t q = word(i & 3, Q0, QS);
                            const uint32_t v = ((i < 4 ? q : q >> 4) & 0x0F0F0F0Fu) | (spread4((qh >> (4 * i)) & 0xFu) << 4);
                            B[i] = (v + 0x70707070u) ^ 0x80808080u;   // q - 16 per byte
                        }
                    }
                    const v4i b0 = {(int)B[0], (int)B[1], (int)B[2], (int)B[3]}, b1 = {(int)B[4], (int)B[5], (int)B[6], (int)B[7]};
                    const bool diag = (r & 3) == j;
                    uint32_t dw[4];
                    cw_gather(W[O >> 2], dw);
                    constexpr bool HI = (O & 2) != 0;
#pragma unroll
                    for (int gr = 0; gr < NG; ++gr) {
                        // A row n: column n / 4 of the group, non-zero on k-slice
                        // n % 4 only, so lane row j receives column j's dots with
                        // the blocks t = 0..3 that lane rows 0..3 hold
                        const lds32 ap = lp32(diag ? xs + (4 * gr + (r >> 2)) * AROW + 36 * (4 * j + K) + 4 : zr);
                        const v4i a0 = {(int)ap[0], (int)ap[1], (int)ap[2], (int)ap[3]};
                        const v4i a1 = {(int)ap[4], (int)ap[5], (int)ap[6], (int)ap[7]};
                        const u32x4a dx = *(const __attribute__((address_space(3))) u32x4a *)(uintptr_t)(
                            xt + 32 * P::CU * (4 * gr + j) + 16 * K);
                        v4i d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a0, b0, v4i{0, 0, 0, 0}, 0, 0, 0);
                        d = __builtin_amdgcn_mfma_i32_16x16x64_i8(a1, b1, d, 0, 0, 0);
                        acc[gr] = fmaf(cw_hmul<HI>(dw[0], dx[0], nz), (float)d[0], acc[gr]);
                        acc[gr] = fmaf(cw_hmul<HI>(dw[1], dx[1], nz), (float)d[1], acc[gr]);
                        const float a2 = fmaf(cw_hmul<HI>(dw[2], dx[2], nz), (float)d[2], acc[gr]);
                        const float a3 = fmaf(cw_hmul<HI>(dw[3], dx[3], nz), (float)d[3], a2);
                        acc[gr] = units > 1 ? a3 : acc[gr];       // (a half chunk: blocks 2 and 3 are not there)
                    }
                };
                switch (k) {
                    case 0: chain(std::integral_constant<int, 0>()); break;
                    case 1: chain(std::integral_constant<int, 1>()); break;
                    case 2: chain(std::integral_constant<int, 2>()); break;
                    default: chain(std::integral_constant<int, 3>()); break;
                }
            } else if constexpr (FMT == FMT_Q4_K) {
                if (k < units) {
                    // lane (r, j): the header and qs bytes 32 j .. 32 j + 31 of row r's
                    // superblock: sub-blocks 2 j (low nibbles) and 2 j + 1 (high)
                    typedef const __attribute__((address_space(3))) u32x4a * lds128;
                    const uint32_t wb = st + r * WROW + 144 * k;
                    const u32x4a hd = *(lds128)(uintptr_t)wb;
                    const u32x4a qa = *(lds128)(uintptr_t)(wb + 16 + 32 * j), qb = *(lds128)(uintptr_t)(wb + 32 + 32 * j);
                    v4i lo[2], hi[2];
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        lo[0][i] = (int)(qa[i] & 0x0F0F0F0Fu);
                        lo[1][i] = (int)(qb[i] & 0x0F0F0F0Fu);
                        hi[0][i] = (int)((qa[i] >> 4) & 0x0F0F0F0Fu);
                        hi[1][i] = (int)((qb[i] >> 4) & 0x0F0F0F0Fu);
                    }
                    // the row's 6-bit scales, the mins of sub-blocks 2 j, 2 j + 1 (SWAR,
                    // fl_q4k_scale_min)
                    const uint32_t sc[2] = {hd.y & 0x3F3F3F3Fu, (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u)};
                    const uint32_t wmn = j < 2 ? hd.z & 0x3F3F3F3Fu : ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
                    const uint32_t m16 = (wmn >> (16 * (j & 1)));
                    const int n0 = (int)((m16 & 0xFFu) * 0x01010101u), n1 = (int)(((m16 >> 8) & 0xFFu) * 0x01010101u);
                    const v4i mv0 = {n0, n0, n0, n0}, mv1 = {n1, n1, n1, n1};
                    const float d = h2f(hd.x & 0xFFFFu), dmin = h2f(hd.x >> 16);
                    const bool diag = (r & 3) == j;
#pragma unroll
                    for (int gr = 0; gr < NG; ++gr) {
                        // A row n: column n / 4 of the group, non-zero on k-slice n % 4
                        // only, so lane row j receives column j's dots with the
                        // sub-blocks 2 i (d0) and 2 i + 1 (d1) of lane row i
                        const uint32_t xc = xs + 4 * gr * AROW + 292 * k;
                        const lds32 ap = lp32(diag ? xc + (r >> 2) * AROW + 36 + 64 * j : zr);
                        v4i a[4];
#pragma unroll
                        for (int i = 0; i < 4; ++i) a[i] = v4i{(int)ap[4 * i], (int)ap[4 * i + 1], (int)ap[4 * i + 2], (int)ap[4 * i + 3]};
                        const v4i z = {0, 0, 0, 0};
                        v4i d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], lo[0], z, 0, 0, 0);
                        v4i d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[2], hi[0], z, 0, 0, 0);
                        // the min term sum_g m_g sum x_g: the same A against the min in every byte
                        v4i dm = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[0], mv0, z, 0, 0, 0);
                        d0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[1], lo[1], d0, 0, 0, 0);
                        d1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[3], hi[1], d1, 0, 0, 0);
                        dm = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[1], mv0, dm, 0, 0, 0);
                        dm = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[2], mv1, dm, 0, 0, 0);
                        dm = __builtin_amdgcn_mfma_i32_16x16x64_i8(a[3], mv1, dm, 0, 0, 0);
                        int ti = 0;
#pragma unroll
                        for (int i = 0; i < 4; ++i) {
                            const uint32_t s2 = sc[i >> 1] >> (16 * (i & 1));
                            ti += __mul24((int)(s2 & 0xFFu), d0[i]) + __mul24((int)((s2 >> 8) & 0xFFu), d1[i]);
                        }
                        const int tm = (dm[0] + dm[1]) + (dm[2] + dm[3]);
                        const float dk = __uint_as_float(*lp32(xc + j * AROW));
                        acc[gr] = fmaf(d * dk, (float)ti, acc[gr]);
                        acc[gr] = fmaf(-(dmin * dk), (float)tm, acc[gr]);
                    }
                }
            } else if constexpr (FMT == FMT_Q6_K) {
                if (k < units) {
                    // the row's chunk starts sh bytes into its window
                    const uint32_t wrow = min(rbeg + 16 * t + r, rend - 1);
                    const uint32_t sh = ((uint32_t)(uintptr_t)w + wrow * RB + c * CB) & 15u;
                    const uint32_t wb = st + r * WROW + sh + 210 * k, s2 = wb & 2u;
                    // six runs of 8 bytes (ql at 64 h + 32 b + 8 j, qh at 128 + 32 h
                    // + 8 j), the 16 scales and d, from aligned dwords
                    const lds32 rp = lp32(wb - s2 + 8 * j), sp = lp32(wb - s2 + 192);
                    uint32_t W[6][2];
#pragma unroll
                    for (int q = 0; q < 6; ++q) {
                        const uint32_t d0 = rp[8 * q], d1 = rp[8 * q + 1], d2 = rp[8 * q + 2];
                        W[q][0] = alignb(d1, d0, s2);
                        W[q][1] = alignb(d2, d1, s2);
                    }
                    const uint32_t SC[4] = {alignb(sp[1], sp[0], s2), alignb(sp[2], sp[1], s2), alignb(sp[3], sp[2], s2),
                                            alignb(sp[4], sp[3], s2)};
                    const float d = h2f((s2 ? sp[4] >> 16 : sp[4]) & 0xFFFFu);
                    // 4 (q - 32) per byte: the six bits at the top, the highest one
                    // inverted (qh: once for its four groups)
                    uint32_t Bv[8][2];
#pragma unroll
                    for (int m = 0; m < 8; ++m) {                 // half m / 4, group m % 4
                        const int hh = m >> 2, gg = m & 3;
#pragma unroll
                        for (int u = 0; u < 2; ++u) {
                            const uint32_t ql = W[2 * hh + (gg & 1)][u], qh = W[4 + hh][u] ^ 0xAAAAAAAAu;
                            const uint32_t nib = (gg < 2 ? ql << 2 : ql >> 2) & 0x3C3C3C3Cu;
                            Bv[m][u] = nib | ((qh << (6 - 2 * gg)) & 0xC0C0C0C0u);
                        }
                    }
#pragma unroll
                    for (int gr = 0; gr < NG; ++gr) {
                        // A row n: column 8 gr + n / 2, non-zero on the k-slices of
                        // sub-block 2 m + n % 2 only, so lane row j receives the dots of
                        // columns 2 j (dd[0], dd[1]) and 2 j + 1 with both sub-blocks
                        const uint32_t xc = xs + ((8 * gr + (r >> 1)) & (NC - 1)) * AROW + 292 * k + 8 * j;
                        const lds32 ap = lp32((r & 1) == (j >> 1) ? xc + 36 : zr);
                        int ia[2] = {0, 0};
#pragma unroll
                        for (int m = 0; m < 8; ++m) {
                            const v4i dd = __builtin_amdgcn_mfma_i32_16x16x32_i8(
                                (long)(((uint64_t)ap[8 * m + 1] << 32) | ap[8 * m]),
                                (long)(((uint64_t)Bv[m][1] << 32) | Bv[m][0]), v4i{0, 0, 0, 0}, 0, 0, 0);
                            const int s0 = (int)(int8_t)(SC[m >> 1] >> (16 * (m & 1)));
                            const int s1 = (int)(int8_t)(SC[m >> 1] >> (16 * (m & 1) + 8));
                            ia[0] += __mul24(s0, dd[0]) + __mul24(s1, dd[1]);
                            ia[1] += __mul24(s0, dd[2]) + __mul24(s1, dd[3]);
                        }
                        const uint32_t c0 = (8 * gr + 2 * j) & (NC - 1);
                        const float dk0 = __uint_as_float(*lp32(xs + c0 * AROW + 292 * k));
                        const float dk1 = __uint_as_float(*lp32(xs + (c0 + 1) * AROW + 292 * k));
                        acc[2 * gr] = fmaf(d * dk0, (float)(ia[0] >> 2), acc[2 * gr]);
                        acc[2 * gr + 1] = fmaf(d * dk1, (float)(ia[1] >> 2), acc[2 * gr + 1]);
                    }
                }
            }
        }
        // (a0 + a1) + (a2 + a3): wave k leaves chain k, thread (column, row) adds
        // (the next tile's first chunk barrier orders these reads before its stores)
#pragma unroll
        for (int i = 0; i < NACC; ++i) AC[k * 256 + col_of(i) * 16 + r] = acc[i];
        lds_barrier();
        if (mine) *yp = y0 + ((AC[tid] + AC[tid + 256]) + (AC[tid + 512] + AC[tid + 768]));
    }
}

// Rows [rbeg, rend) of the matrix for nx <= NC columns.
template <int FMT, int NC, int D, typename COLS>
__device__ __forceinline__ void cw_body(const uint8_t * __restrict__ w, uint32_t cols, const COLS & C, uint32_t nx,
                                        uint32_t rbeg, uint32_t rend, uint8_t * sm) {
    uint8_t * zr = sm + (size_t)D * CwPlan<FMT, NC>::STG + 4096;
    if (threadIdx.x < CW_ZERO / 4) lds_st32(zr + 4 * threadIdx.x, 0u);   // (read after the first chunk's barrier)
    if (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) == CW_WAVES - 1)
        cw_produce<FMT, NC, D>(w, cols, C, nx, rbeg, rend, sm);
    else
        cw_consume<FMT, NC, D>(w, cols, C, nx, rbeg, rend, sm);
}

// Workgroup g's rows of G: whole 16-row tiles (a partial one costs a whole
// one's work), the first workgroups one more, so that the two that share a CU
// (g and g + 256) get one of each.
__device__ __forceinline__ void cw_rows(uint32_t rows, uint32_t g, uint32_t G, uint32_t & rbeg, uint32_t & rend) {
    const uint32_t T = (rows + 15) >> 4, base = T / G, rem = T - base * G;
    const uint32_t t0 = g * base + min(g, rem), t1 = t0 + base + (g < rem ? 1u : 0u);
    rbeg = min(16 * t0, rows);
    rend = min(16 * t1, rows);
}

template <int FMT, int NC, int D>
__global__ __launch_bounds__(64 * CW_WAVES, 4) void k_dot_cw(DotArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t cw_sm[];
    const uint8_t * w = a.w + (a.id_slot ? (size_t)(*a.id_slot) * a.estride : 0);
    const CwColsStrided C{a.x, a.y, a.xstride, a.ystride};
    uint32_t rbeg, rend;
    cw_rows(a.rows, blockIdx.x, gridDim.x, rbeg, rend);
    cw_body<FMT, NC, D>(w, a.cols, C, a.nx, rbeg, rend, cw_sm);
}

// Ring depth within `lds` bytes and the vmcnt range.  Up to one 16-row tile per
// CU: a workgroup alone on its CU, the ring deep (Q8_0 4096x14336 with 4 columns
// 14.9 us, 17.7 with 3 stages; Q6_K with 8 columns 15.9 / 18.4).  More tiles: 3
// stages and two workgroups per CU, or three where 4 columns' stages are small
// (Q4_K 28672x4096 with 3 columns 15.3 us, 16.6 with two workgroups and a deep
// ring; Q8_0 11264x2048 7.6 / 8.8; Q6_K's stages are larger: 25.0 with two,
// 28.9 with three).
template <int FMT, int NC> constexpr int cw_depth(int most, size_t lds) {
    int d = 2;
    while (d < most && cw_smem<FMT, NC>(d + 1) <= lds && (d - 1) * (int)CwPlan<FMT, NC>::NT <= 60) ++d;
    return d;
}
constexpr size_t CW_LDS1 = 150 * 1024, CW_LDS2 = 80 * 1024;       // one or two workgroups per CU
// Grouped experts: the routed experts share the grid (moe_assign); the
// workgroup streams its rows of its expert once for up to 16 of the expert's
// pairs, in the smallest of the 4-, 8- and 16-column forms that holds them: the
// counts differ from expert to expert (8 tokens, 2 of 8 experts: 2 on average,
// often 5), and one form for all of them, sized for the average, read the
// weights of every fuller expert twice.
template <int FMT, int NC> constexpr int cw_moe_depth() { return cw_depth<FMT, NC>(3, CW_LDS2); }
template <int FMT> constexpr size_t cw_moe_smem() {
    size_t m = cw_smem<FMT, 4>(cw_moe_depth<FMT, 4>());
    for (size_t n : {cw_smem<FMT, 8>(cw_moe_depth<FMT, 8>()), cw_smem<FMT, 16>(cw_moe_depth<FMT, 16>())}) m = n > m ? n : m;
    return m;
}
template <int FMT>
__global__ __launch_bounds__(64 * CW_WAVES, 4) void k_moe_cw(MoeArgs a) {
    extern __shared__ __attribute__((aligned(16))) uint8_t cw_sm[];
    __shared__ uint32_t pairs[256], rids[256], npairs, cxi[16], cyi[16];
    const uint32_t tid = threadIdx.x;
    if (tid == 0) npairs = 0;
    const uint32_t * ids = moe_route(a, rids);
    uint32_t g, G;
    const uint32_t e = moe_assign(ids, a.ntok * a.top_k, a.n_expert, blockIdx.x, gridDim.x, g, G);   // (barriers)
    if (e >= a.n_expert) return;
    if (tid < a.ntok * a.top_k && ids[tid] == e) pairs[atomicAdd(&npairs, 1u)] = tid;
    __syncthreads();
    const uint32_t np = npairs;
    const uint8_t * w = a.w + (size_t)e * a.estride;
    uint32_t rbeg, rend;
    cw_rows(a.rows, g, G, rbeg, rend);
    if (rbeg >= rend) return;
    for (uint32_t p0 = 0; p0 < np; p0 += 16) {
        const uint32_t nx = min(16u, np - p0);
        if (tid < 16) {
            const uint32_t ts = pairs[p0 + (tid < nx ? tid : 0)];
            cxi[tid] = a.x_per_slot ? ts : ts / a.top_k;
            cyi[tid] = ts;
        }
        __syncthreads();
        const CwColsMoe C{a.x, a.y, a.xstride, a.ystride, cxi, cyi};
        if (nx <= 4) cw_body<FMT, 4, cw_moe_depth<FMT, 4>()>(w, a.cols, C, nx, rbeg, rend, cw_sm);
        else if (nx <= 8) cw_body<FMT, 8, cw_moe_depth<FMT, 8>()>(w, a.cols, C, nx, rbeg, rend, cw_sm);
        else cw_body<FMT, 16, cw_moe_depth<FMT, 16>()>(w, a.cols, C, nx, rbeg, rend, cw_sm);
        __syncthreads();
    }
}

// ----------------------------------------------------------------- launch --
static bool cw_takes(int fmt, const void * w, uint64_t estride, const void * x, uint32_t xstride, uint32_t ncol,
                     uint32_t cols) {
    if (cols == 0 || cols > 16384 || (cols & 255) || ((uintptr_t)x & 3)) return false;   // (longer rows are refused everywhere)
    if (fmt != FMT_Q4_K && fmt != FMT_Q6_K && (((uintptr_t)x & 15) || (xstride & 3))) return false;
    // 32-bit lane offsets
    if ((uint64_t)ncol * xstride * 4 + x_alloc_bytes(cols) >= (1ull << 32) || 16ull * cols * 2 >= (1ull << 32)) return false;
    // Q6_K and IQ rows are placed from their own 16-byte boundaries; the others' rows
    // and pieces are whole 16-byte segments of an aligned matrix
    const uintptr_t al = cw_gran(fmt) ? 1 : 15;
    return !((uintptr_t)w & al) && !(estride & al);
}

template <int FMT, int NC, int D>
static int cw_go(const DotArgs & a, uint32_t G, hipStream_t s) {
    constexpr size_t smb = cw_smem<FMT, NC>(D);
    const void * kern = (const void *)k_dot_cw<FMT, NC, D>;
    if (int rc = lds_fits(kern, smb, "k_dot_cw")) return rc;
    (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smb);
    hipLaunchKernelGGL((k_dot_cw<FMT, NC, D>), dim3(G), dim3(64 * CW_WAVES), smb, s, a);
    return hip_check(hipGetLastError(), "k_dot_cw launch");
}
template <int FMT, int NC> static int cw_plan(const DotArgs & a, hipStream_t s) {
    const uint32_t T = (a.rows + 15) / 16, cus = (uint32_t)num_cus();
    if (T <= cus) return cw_go<FMT, NC, cw_depth<FMT, NC>(6, CW_LDS1)>(a, T, s);
    const uint32_t wgs = (tune().cw_wpc ? tune().cw_wpc : NC == 4 && FMT != FMT_Q6_K ? 3 : 2) * cus;
    return cw_go<FMT, NC, cw_depth<FMT, NC>(3, CW_LDS2)>(a, T < wgs ? T : wgs, s);
}
template <int FMT> static int cw_launch(const DotArgs & a, hipStream_t s) {
    return a.nx <= 4 ? cw_plan<FMT, 4>(a, s) : a.nx <= 8 ? cw_plan<FMT, 8>(a, s) : cw_plan<FMT, 16>(a, s);
}

// Whether a matrix with nx columns is faster here than on the format's other
// kernel (us here / there, medians of back-to-back launches over matrices in
// HBM).  A workgroup takes whole 16-row tiles of whole rows: with half as many
// tiles as CUs, or fewer, a launch takes as long as one tile however few there
// are, about 4.3 + 0.75 us per chunk of a row, and kernels that split the rows
// further are faster on all but short rows.  Elsewhere:
//  * Q4_K against k_dot_mfma (k_dot_kstream with 2 columns of up to 4096), whose
//    tiles are 16 x 144-byte pieces but which stages the columns once per
//    workgroup.  4 columns 14336x4096 9.7 / 10.3, 4096x14336 9.4 / 11.3; 8
//    columns 6144x3840 7.4 / 8.1, 14336x4096 11.3 / 11.8, 8192x14336 16.6 / 26.9;
//    16 columns 14336x4096 14.6 / 14.7, 28672x4096 21.8 / 21.7 (the columns are as
//    many bytes as the weights), where that kernel takes several passes
//    28672x5120 27.8 / 46.2.  Rows that end in part of a chunk cost a whole one:
//    8 columns 28672x2304 14.8 / 13.4, 28672x3840 18.1 / 17.4 (20480x2816 11.9 /
//    11.8), 16 columns 9216x3328 13.2 / 12.6 (6144x3328 8.9 / 9.5).  Few long rows:
//    5 columns 512x14336 11.6 / 11.3; 2 columns 100x4096 4.9 / 4.4.
//  * Q6_K against the streaming kernel.  2 columns 4096x14336 15.6 / 16.2,
//    3072x14336 15.4 / 14.0, 14336x4096 14.5 / 12.1; 4 columns 4096x4096 7.8 / 8.0,
//    2048x4096 7.5 / 6.8, 1024x8192 10.4 / 7.0, 1024x2048 5.0 / 5.9; 8 columns
//    2048x4096 7.5 / 8.1, 1024x4096 7.5 / 6.8, 1024x8192 10.6 / 9.9, 512x14336 15.0
//    / 16.5, 14336x4096 15.6 / 33.
//  * Q8_0 and Q5_0 against k_dot_sbl_nx (rows of up to 8192 columns) and the
//    register kernel.  2 columns Q8_0 14336x4096 15.3 / 14.4, 4096x8192 9.9 / 11.5,
//    2048x8192 9.4 / 8.1, 4096x14336 14.2 / 20.1, Q5_0 14336x4096 12.3 / 14.2,
//    2048x4096 6.5 / 5.8; 4 columns Q8_0 1024x1792 5.1 / 4.8, 14336x4096 15.7 /
//    18.1; 5 columns Q5_0 512x8192 11.3 / 10.1 (8 columns 11.4 / 11.7), Q8_0 256x6144
//    8.9 / 8.1; 16 columns 14336x4096 20 / 52.  One column against k_dot_sbl: rows
//    wider than its one pass per lane group holds well, Q8_0 4096x14336 14.3 / 18.6,
//    8192x8192 14.1 / 17.1, Q5_0 8192x14336 17.8 / 29.6; not 14336x4096 15.2 / 13.4,
//    2048x5632 7.6 / 6.3.
//  * IQ2_XXS and IQ3_XXS against k_dot_sbl_nx (rows of up to 8192 columns, a
//    multiple of 2048), k_dot_sbl (one column) and the register kernel.  2 columns
//    IQ2_XXS 14336x4096 13.8 / 12.5, 28672x4096 21.3 / 23.2, IQ3_XXS 28672x2048 14.7 /
//    13.8; 4 columns IQ2_XXS 4096x4096 7.3 / 7.7, 2048x4096 7.2 / 6.2, 1024x8192
//    10.5 / 7.0; 8 columns 2048x4096 8.9 / 8.3, 2048x8192 12.9 / 14.0 (5 columns 13.0
//    / 12.2), 1024x8192 12.9 / 11.9; 16 columns 14336x4096 25.7 / 42.6.  Other row
//    lengths: 2 columns 1024x2816 5.9 / 5.8, 2048x2816 6.3 / 7.9, 1024x14336 15.8 /
//    14.8; 4 columns 256x1792 IQ3_XXS 4.9 / 4.5, 512x2816 5.8 / 5.7; 3840x3840 with 1
//    / 16 6.5 / 7.7, 10.2 / 44; one column of few rows, 1024x2816 5.4 / 5.1,
//    2048x16384 17.4 / 15.2, 256x16384 16.9 / 10.8.
static bool cw_wins(int fmt, uint32_t rows, uint32_t cols, uint32_t nx) {
    const uint32_t T = (rows + 15) / 16, cus = (uint32_t)num_cus();
    const bool half = 2 * T <= cus, quarter = 4 * T <= cus, sixteenth = 16 * T <= cus;   // of the chip, at most
    if (fmt == FMT_Q4_K) {
        const bool part = (cols & 1023) && cols > 1024;
        if (nx > 8) return cols > 4096 || rows <= (part ? 8192u : 16384u);
        if (nx > 4) return !(part && rows > 20480) && !(half && cols > 8192);
        return !(nx == 2 && sixteenth && cols > 2048 && cols <= 4096);
    }
    if (fmt == FMT_Q6_K) {
        if (nx == 2) return cols > 8192 && T >= cus;
        if (nx <= 4) return !(half && cols > 2048);
        return nx > 8 || !((cols <= 8192 ? quarter : sixteenth) && cols > 2816);
    }
    if (cw_iq(fmt)) {
        const bool sbl = !(cols & 2047) && cols <= 8192;
        if (nx == 1) return ((cols & 2047) || cols > 16128) && (cols > 8192 ? !half : rows >= 2048);
        if (nx == 2) return sbl ? rows > 16384 && cols > 2048 : !(quarter && cols > 1024);
        if (nx <= 4 && sbl) return !(half && cols > 2048);
        if (nx <= 4) return !(sixteenth && cols > 1024) && !((cols > 8192 ? quarter : 5 * T <= cus) && cols > 2048);
        return nx > 8 || !(sbl && cols > 2048 && (cols <= 6144 || nx <= 6 ? half : quarter));
    }
    if (nx == 1) return cols > 4096 && T >= cus;
    if (nx == 2 && half && cols > 2048 && cols <= 8192) return false;
    if (nx <= 4 && quarter && cols > (fmt == FMT_Q8_0 && nx > 2 ? 1536u : 2048u)) return false;
    if (nx > 4 && nx <= 8 && sixteenth && cols > 4096 && cols <= 6144) return false;
    if (fmt == FMT_Q5_0 && (nx == 5 || nx == 6) && quarter && cols > 4096 && cols <= 8192) return false;
    return nx > 2 || fmt == FMT_Q5_0 || cols > 4096;
}
static bool cw_on(int fmt) {
    const Tune & t = tune();
    return t.cw && !(fmt == FMT_Q4_K && (t.no_mfma || t.mf_forced)) && !(fmt == FMT_Q6_K && t.no_q6mf);
}

int launch_dot_cw(int fmt, const DotArgs & a, hipStream_t s) {
    if (!cw_on(fmt) || (tune().cw == 1 && !cw_wins(fmt, a.rows, a.cols, a.nx))) return FLH_ERR_UNSUPPORTED;
    if (a.nx < 1 || a.nx > 16 || !cw_takes(fmt, a.w, a.estride, a.x, a.xstride, a.nx, a.cols)) return FLH_ERR_UNSUPPORTED;
    if (a.rows == 0) return FLH_OK;
    switch (fmt) {
        case FMT_Q8_0: return cw_launch<FMT_Q8_0>(a, s);
        case FMT_Q5_0: return cw_launch<FMT_Q5_0>(a, s);
        case FMT_Q4_K: return cw_launch<FMT_Q4_K>(a, s);
        case FMT_Q6_K: return cw_launch<FMT_Q6_K>(a, s);
        case FMT_IQ2_XXS: return cw_launch<FMT_IQ2_XXS>(a, s);
        case FMT_IQ3_XXS: return cw_launch<FMT_IQ3_XXS>(a, s);
        default: return FLH_ERR_UNSUPPORTED;
    }
}

template <int FMT> static int cw_moe(const MoeArgs & a, hipStream_t s) {
    constexpr size_t smb = cw_moe_smem<FMT>();
    uint32_t wgs = (tune().cw_wpc ? tune().cw_wpc : 2) * (uint32_t)num_cus();
    if (tune().cw_gmax && wgs > tune().cw_gmax) wgs = tune().cw_gmax;
    // a workgroup per expert at least (moe_assign); a partitioned device has as few as 32 CUs
    if (wgs < moe_rows(a)) wgs = moe_rows(a);
    const void * kern = (const void *)k_moe_cw<FMT>;
    if (int rc = lds_fits(kern, smb, "k_moe_cw")) return rc;
    (void)hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)smb);
    hipLaunchKernelGGL((k_moe_cw<FMT>), dim3(wgs), dim3(64 * CW_WAVES), smb, s, a);
    return hip_check(hipGetLastError(), "k_moe_cw launch");
}
// Whether grouped experts of several tokens are faster here than on the format's
// other kernel, which reads an expert once for each of its pairs (us here /
// there; 8 experts take 2 of 8, 128 take 8 of 128).  So the line is a number of
// pairs per expert that some token takes, on average:
//  * Q8_0, Q5_0 and the IQ formats against the routed k_dot_sbl (rows of up to
//    8192 columns).  That launch is about one workgroup per CU and as many for
//    every pair, so where the pairs do not divide the CUs some wait for a second turn:
//    Q8_0 3072x2048, 64 experts, 6 of them a token, 2 / 4 tokens 18.5 / 26.4, 29.8 /
//    47.7.  Elsewhere Q8_0 256x1024 of 8 with 2 / 16 tokens 5.6 / 4.5, 6.3 / 4.9, of
//    128 with 8 / 16 8.0 / 6.7, 10.2 / 9.6 (Q5_0 9.6 / 9.3); 1024x2048 of 8 with 4
//    / 8 7.4 / 6.3, 7.7 / 8.5, of 128 with 8 / 16 26.7 / 23.2, 38.2 / 43.2; 3072x2048
//    of 8 with 4 / 8 11.5 / 10.8, 13.5 / 18.0; 4096x4096 of 8 with 2 / 4 15.3 / 15.2,
//    22.9 / 25.4 (Q5_0 13.1 / 14.1 with 2), of 128 with 4 / 8 92 / 89, 164 / 174;
//    IQ2_XXS 3072x2048 of 8 with 4 / 8 12.3 / 10.7, 13.5 / 16.5, of 128 with 8 / 16
//    62 / 51, 98 / 97; 4096x4096 of 8 with 4 24.1 / 22.2, of 128 with 8 / 16 151 /
//    141, 249 / 275; 14336x4096 of 8 with 2 / 4 39 / 35, 56 / 65.
//  * Q6_K against the streaming kernel: two tokens 3072x2048 of 8 10.9 / 9.0,
//    14336x4096 38 / 31, 4096x14336 42.7 / 44.5; three 14336x4096 50 / 53.
static bool cw_moe_wins(int fmt, const MoeArgs & a) {
    const uint64_t weights = (uint64_t)a.rows * a.cols;
    const uint32_t pairs = a.ntok * a.top_k, cus = (uint32_t)num_cus();
    if (fmt == FMT_Q4_K || a.cols < 256 || a.cols > 8192 || pairs == 0) return true;
    if (fmt == FMT_Q6_K) return a.ntok > 2 || cus % pairs || weights < (1u << 21);
    // that launch's workgroups for a pair: no more than there are chunks of rows
    const uint32_t rpc = 32 / (a.cols >> 8), chunks = (a.rows + rpc - 1) / rpc;
    uint32_t per = (cus + pairs - 1) / pairs;
    if (per > chunks) per = chunks;
    if (per * pairs > cus) return true;
    float routed = 1.f;                                           // experts that some token takes, on average
    for (uint32_t t = 0; t < a.ntok; ++t) routed *= 1.f - (float)a.top_k / (float)a.n_expert;
    routed = (float)a.n_expert * (1.f - routed);
    float most;
    if (weights <= (1u << 18) && pairs <= 64) return false;
    if (cw_iq(fmt)) most = weights <= (1u << 23) ? 1.6f : weights <= (1u << 24) ? 1.47f : 1.2f;
    else most = weights <= (1u << 18) ? 1.6f : weights > (1u << 23) ? 1.12f : pairs <= 32 ? 1.53f : 1.3f;
    return (float)pairs > most * routed;
}
int launch_moe_cw(int fmt, const MoeArgs & a, hipStream_t s, bool any) {
    if (!cw_on(fmt) || (!any && tune().cw == 1 && !cw_moe_wins(fmt, a))) return FLH_ERR_UNSUPPORTED;
    const uint64_t pairs = (uint64_t)a.ntok * a.top_k;
    if (pairs > 256 || a.n_expert > 256 || !cw_takes(fmt, a.w, a.estride, a.x, a.xstride, (uint32_t)pairs, a.cols))
        return FLH_ERR_UNSUPPORTED;
    if (a.rows == 0 || pairs == 0) return FLH_OK;
    switch (fmt) {
        case FMT_Q8_0: return cw_moe<FMT_Q8_0>(a, s);
        case FMT_Q5_0: return cw_moe<FMT_Q5_0>(a, s);
        case FMT_Q4_K: return cw_moe<FMT_Q4_K>(a, s);
        case FMT_Q6_K: return cw_moe<FMT_Q6_K>(a, s);
        case FMT_IQ2_XXS: return cw_moe<FMT_IQ2_XXS>(a, s);
        case FMT_IQ3_XXS: return cw_moe<FMT_IQ3_XXS>(a, s);
        default: return FLH_ERR_UNSUPPORTED;
    }
}

}  // namespace flh
