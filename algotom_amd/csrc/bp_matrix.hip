// Back-projection of slice stacks on the matrix cores.
//
// One pixel's interpolation at one angle is a product of two weights with two
// neighbouring detector samples, and the weights are the same for every
// slice.  A 4 x 4 pixel block spans at most 3 (|cos| + |sin|) <= 4.25
// detector columns, so its samples of one angle always lie in 8 columns that
// start at an even column.  Four angles of one block are therefore one
//     (16 pixels) x (4 angles x 8 columns) . (4 angles x 8 columns) x 16 slices
// product: v_mfma_f32_16x16x32_f16 with a weight operand that holds two
// non-zero entries per pixel and angle.  Building it costs about 30 VALU
// instructions per block and four angles, shared by every slice of the
// workgroup; the vector kernel (bp_tiled_kernel) pays 3.4 (16-bit) to 8.9
// (reference typing) per pixel, angle and slice.
//
// Precision.  16-bit factors appear as two-term splits:
//   * a float32 sample s, scaled by a power of two per slice so that
//     2^14 <= max|s| < 2^15, is h + l with h = f16(s), l = f16(s - h): 23 bits
//     (22 where l rounds up), down to a last step of 2^-24 (2^-39 of the
//     slice's maximum).  16-bit storage is one f16 value: float16 itself, a
//     bfloat16 scaled in the same way, which is exact down to 2^-32 of the
//     maximum;
//   * the fraction of the detector position, rounded to nearest on 22 bits,
//     is 2^-11 a + 2^-22 b, and so is its complement; a, b <= 2^11 are
//     integers, and an integer n <= 2048 read as a float16 bit pattern is
//     exactly n 2^-24 (subnormals and the first two binades share one step),
//     so a and b need no conversion;
//   * every product (h + l)(a + b) is exact in float32; the matrix unit sums
//     four angles in float32 and truncates, the total is rounded.
// That is a bit less per sample than float32 and less per weight than the
// float64 fraction of ATH_ACC_F32SEQ, against a quarter of its roundings of the
// sum: from about 100 angles on the error against float64 is below
// that of ATH_ACC_F32SEQ.  Relative 2-norm, 128 / 361 / 1801 / 3601 angles, the
// largest of 131 to 2560 columns: white noise 1.8 / 2.3 / 4.3 / 5.8e-7 against
// 2.0 / 3.3 / 7.4 / 10.5e-7, filtered projections 1.1 / 1.5 / 3.1 / 4.4e-7
// against 1.8 / 2.8 / 6.2 / 8.8e-7, positive ones 0.9 / 1.5 / 3.2 / 4.5e-7
// against 1.6 / 2.9 / 6.3 / 8.9e-7 (37 angles of noise: 1.6 against 1.1e-7).
//
// A slice with a non-finite (or > 2^100) sample would spread it over the 8
// columns of a window, and one whose ordinary samples are small beside a few
// huge ones would lose them (range_kernel); such slices are redone by the
// vector kernel in the caller's accumulation.
//
// Measured (64 x 1801 x 2560, with the mask): float32 42 ms against 181 ms
// for ATH_ACC_F32SEQ (17.9 against 4.2 updates per ps), float16 31
// against 75 ms; 16 slices 14.9 against 46 ms.  What bounds it is VALU issue,
// 41 instructions per block and four angles of 32 slices (76 % busy with the
// matrix unit 41 %; simple 32-bit instructions take 1.2 ns per wave here,
// permutes, shift-adds and float64 2.0, a matrix instruction 7.4 of which it
// holds up the VALU for about 4).  Tried and left out: 8 waves per CU instead
// of 16 (45 ms), four slice groups (48), records of four pairs for float32
// (one product less, but twice the LDS stores: 17.4 against 15.8 ms for 16
// slices), 2:4 sparse products (the weights would have to change lanes).
//
// Layout.  split_kernel writes the stack as (group of 16 slices, angle,
// column pair, slice) entries: the f16 pair of two columns, high parts then
// low parts.  A workgroup's strip of one angle is contiguous there.  It is
// staged in LDS as one 16-byte record per (column pair i, slice): the pairs
// i and i + 1 (high and low part each), or i .. i + 3 for 16-bit storage, so an
// operand is read with aligned ds_read_b128 at any even column: a 4-byte
// aligned 16-byte LDS read runs at 16 B per clock and CU here, an aligned
// one at 208.  Records are double buffered: the next four angles are loaded
// into registers before a step's arithmetic and stored after it.
#include <cmath>
#include <type_traits>

#include "ath_internal.h"

namespace ath {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef float float4_t __attribute__((ext_vector_type(4)));
typedef unsigned uint2_t __attribute__((ext_vector_type(2)));
typedef unsigned uint4_t __attribute__((ext_vector_type(4)));
typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));

// LDS by its 32-bit offset
typedef __attribute__((address_space(3))) uint4_t* LdsQuad;
typedef __attribute__((address_space(3))) uint2_t* LdsPair;
typedef __attribute__((address_space(3))) half8_t* LdsHalf8;

constexpr int kThreads = 1024;
constexpr int kWaves = kThreads / 64;
constexpr unsigned kPatchX = 8, kPatchY = 4;  // tiles
constexpr int kGroup = 16;     // slices per matrix operand
constexpr int kStep = 4;       // angles per matrix operand
// |sample| above 2^100 (bit pattern) goes to the vector kernel
constexpr unsigned kMaxBits = 0x71800000u;
constexpr unsigned kRedo = 0xffffffffu;  // in place of a slice's max|s|
constexpr int kSpanCols = 32;            // columns of a span (range_kernel)

// SG slice groups per workgroup share the weights of its pixels; every tile
// keeps 64 accumulator registers per lane.
//   rows: records per angle.  A window starts at record e, 2 e < b <= 2 e + 2,
//   b the block's lowest position less L (and a slack of 2^-20), L the tile's
//   lowest position (less 2^-19) rounded down to even: 0 < b < 2 + 2^-19 +
//   diag - 3, diag = sqrt((X-1)^2 + (Y-1)^2); the last record read is e + 2.
//   wx: waves side by side (the others are below each other).
// Tile corners lie on one 64-column grid, and a position is built from its
// column's grid point, so that a slice's bits do not depend on the tile.
template <int SG> struct Tile;
template <> struct Tile<2> {
    static constexpr int X = 32, Y = 32, rows = 24, wx = 2;
};
template <> struct Tile<1> {
    static constexpr int X = 64, Y = 32, rows = 40, wx = 2;
};
template <int SG> constexpr bool rows_cover() {
    // e <= ceil(b / 2) - 1 and e + 2 <= rows - 1, i.e. b <= 2 (rows - 2)
    constexpr int X = Tile<SG>::X - 1, Y = Tile<SG>::Y - 1;
    constexpr int m = 2 * (Tile<SG>::rows - 2);  // diag - 0.99 <= m
    return 100 * 100 * (X * X + Y * Y) <= (100 * m + 99) * (100 * m + 99);
}
static_assert(rows_cover<2>() && rows_cover<1>(), "rows");

// zero pairs past the last row, which a tile at its end may stage
constexpr int kTailPairs = 64;
static_assert(kTailPairs >= Tile<1>::rows + 16, "tail");

struct MatArgs {
    unsigned* op;           // split samples
    unsigned* smax;         // per slice: bits of max|s|
    uint2* spans;           // per slice and span of columns, see split
    float2* trig;           // per angle: cos, sin
    size_t nop;             // entries of op (the zero tail follows)
    double pos0;            // centre + kPosMagic
    int scaled;             // samples carry the power of two of smax
    int npair;              // column pairs per row
    int nzero, ntail;       // words to clear from smax on, and of the tail
    int max_rows;           // workgroups per slice that look for its maximum
    int group0, group_end;  // slice groups of the launch
    int group_op, group_have;  // slice groups that op holds
    unsigned patches_x, patches_y;
};

// The kernels run one stack, whose MatJob is a launch argument, or many
// (BATCH: jobs[0 .. njobs) in device memory, a workgroup's by its index).
enum Stage { kClear, kMaxima, kSplit, kRange, kPairs, kSingle, kStages };
struct MatJob {
    BpRedoJob r;
    MatArgs m;
    unsigned begin[kStages];  // the job's first workgroup of a batch's launch
};

// the workgroup's job, and its number in it
template <bool BATCH>
__device__ __forceinline__ const MatJob& find_job(
    const MatJob* __restrict__ jobs, int njobs, const MatJob& one, int stage,
    unsigned& block) {
    block = blockIdx.x;
    if constexpr (!BATCH) return one;
    int lo = 0, hi = njobs - 1;  // last job with begin <= block
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (jobs[mid].begin[stage] <= block) lo = mid;
        else hi = mid - 1;
    }
    block -= jobs[lo].begin[stage];
    return jobs[lo];
}

__device__ __forceinline__ double det_pos(double xc_c, double yc, double s,
                                          double cen) {
    return fma(yc, s, xc_c) + cen;  // as bp_tiled_kernel
}

// power of two that takes max|s| (its bits) into [2^14, 2^15); 0 where the
// samples are all zero or the vector kernel takes the slice
__device__ __forceinline__ int scale_exp(unsigned bits) {
    if (bits == 0u || bits > kMaxBits) return 0;
    return 14 - ilogbf(__uint_as_float(bits));
}

// scaled samples that are large or huge for range_kernel
constexpr float kLarge = 0.25f, kHuge = 8.0f;
__host__ __device__ inline int span_count(int ncol) {
    return (ncol + kSpanCols - 1) / kSpanCols;
}

template <typename T> __device__ __forceinline__ float widen(T v);
template <> __device__ __forceinline__ float widen<float>(float v) { return v; }
template <> __device__ __forceinline__ float widen<__half>(__half v) {
    return __half2float(v);
}
template <>
__device__ __forceinline__ float widen<__hip_bfloat16>(__hip_bfloat16 v) {
    return __bfloat162float(v);
}

template <bool BATCH>
__global__ __launch_bounds__(256) void clear_kernel(
    const MatJob* __restrict__ jobs, int njobs, MatJob one) {
    unsigned b;
    const MatJob& job = find_job<BATCH>(jobs, njobs, one, kClear, b);
    const MatArgs& m = job.m;
    const int i = b * 256 + threadIdx.x;
    if (i < job.r.a.nrow) {
        const float th = -job.r.a.angles[i];
        m.trig[i] =
            make_float2((float)cos((double)th), (float)sin((double)th));
    }
    if (i < m.nzero) m.smax[i] = 0u;
    if (i < m.ntail) m.op[m.nop + i] = 0u;
}

// max|s| per slice, max_rows workgroups each.  Integer order of the bit
// patterns is the order of the magnitudes, with infinities and NaN on top.
template <typename T, bool BATCH>
__global__ __launch_bounds__(256) void slice_max_kernel(
    const MatJob* __restrict__ jobs, int njobs, MatJob one) {
    unsigned b;
    const MatJob& job = find_job<BATCH>(jobs, njobs, one, kMaxima, b);
    const BpArgs& a = job.r.a;
    const int nslice = a.nslice, ncol = a.ncol, step = job.m.max_rows;
    const T* sino = static_cast<const T*>(a.sino);
    const int j = b / step;
    unsigned m = 0u;
    for (int r = b % step; r < a.nrow; r += step) {
        const T* row = sino + ((size_t)r * nslice + j) * ncol;
        for (int c = threadIdx.x; c < ncol; c += 256)
            m = max(m, __float_as_uint(fabsf(widen(row[c]))));
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) m = max(m, (unsigned)__shfl_xor((int)m, o));
    __shared__ unsigned part[4];
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        m = max(max(part[0], part[1]), max(part[2], part[3]));
        if (m) atomicMax(&job.m.smax[j], m);
    }
}

// (row, slice, column) samples -> (group, angle, pair, slice) entries.  A
// block handles 128 columns of one angle's 16 slices through LDS, so both
// the reads (columns) and the writes (slices) are contiguous.  Scaled samples
// are counted on the way for range_kernel: spans[slice][span] = (angles in
// which few of the span's samples are kLarge, those in which few are kHuge <<
// 16, angles in which all are zero); ordinary slices have few of them and add
// next to nothing.
template <typename T, int PL, bool BATCH>
__global__ __launch_bounds__(256) void split_kernel(
    const MatJob* __restrict__ jobs, int njobs, MatJob one) {
    constexpr int COLS = 128, SPANS = COLS / kSpanCols;
    __shared__ float tile[kGroup][COLS + 1];
    // not zero, large << 8, huge << 16 (32 at most each)
    __shared__ unsigned count[SPANS][kGroup];
    unsigned b;
    const MatJob& job = find_job<BATCH>(jobs, njobs, one, kSplit, b);
    const BpArgs& a = job.r.a;
    const int nrow = a.nrow, nslice = a.nslice, ncol = a.ncol;
    const int npair = job.m.npair, scaled = job.m.scaled;
    const T* sino = static_cast<const T*>(a.sino);
    // one stack: grid.y is the row (its workgroups can be more than 2^24)
    const unsigned nblock = (ncol + COLS - 1) / COLS;
    const int c0 = (int)(b % nblock) * COLS;
    b /= nblock;
    const int row = BATCH ? (int)(b % nrow) : (int)blockIdx.y;
    const int gl = BATCH ? (int)(b / nrow) : (int)b;
    const int g = job.m.group_op + gl;
    const int tid = threadIdx.x;
    for (int e = tid; e < kGroup * COLS; e += 256) {
        const int n = e / COLS, c = c0 + e % COLS, j = g * kGroup + n;
        float v = 0.0f;
        if (j < nslice && c < ncol)
            v = widen(sino[((size_t)row * nslice + j) * ncol + c]);
        tile[n][e % COLS] = v;
    }
    if (tid < SPANS * kGroup) count[tid / kGroup][tid % kGroup] = 0u;
    __syncthreads();
    const int n = tid & 15, j = g * kGroup + n;
    const unsigned bits = j < nslice ? job.m.smax[j] : 0u;
    const bool bad = bits > kMaxBits;  // redone by the vector kernel
    const int ex = scaled ? scale_exp(bits) : 0;
    unsigned* base =
        job.m.op + (((size_t)gl * nrow + row) * npair) * (kGroup * PL);
    for (int i = tid >> 4; i < COLS / 2; i += 16) {
        const int p = c0 / 2 + i;
        if (p >= npair) break;
        float s0 = tile[n][2 * i], s1 = tile[n][2 * i + 1];
        if (bad) s0 = s1 = 0.0f;
        s0 = ldexpf(s0, ex);
        s1 = ldexpf(s1, ex);
        if (scaled) {
            const auto rank = [](float v) {
                const float u = fabsf(v);
                return (unsigned)(u != 0.0f) + ((unsigned)(u >= kLarge) << 8) +
                       ((unsigned)(u >= kHuge) << 16);
            };
            const unsigned m = rank(s0) + rank(s1);
            if (m) atomicAdd(&count[i / (kSpanCols / 2)][n], m);
        }
        const half2_t h = {(_Float16)s0, (_Float16)s1};
        unsigned* dst = base + ((size_t)p * kGroup + n) * PL;
        if constexpr (PL == 2) {
            const half2_t l = {(_Float16)(s0 - (float)h[0]),
                               (_Float16)(s1 - (float)h[1])};
            *reinterpret_cast<uint2_t*>(dst) =
                uint2_t{__builtin_bit_cast(unsigned, h),
                        __builtin_bit_cast(unsigned, l)};
        } else {
            *dst = __builtin_bit_cast(unsigned, h);
        }
    }
    if (!scaled) return;
    __syncthreads();
    const int sp = tid / kGroup;
    if (sp < SPANS && j < nslice && c0 + sp * kSpanCols < ncol) {
        const unsigned m = count[sp][n];
        const unsigned some = m & 255u, large = m >> 8 & 255u, huge = m >> 16;
        uint2* at = job.m.spans + (size_t)j * span_count(ncol) +
                    c0 / kSpanCols + sp;
        if (some == 0u)
            atomicAdd(&at->y, 1u);
        else if (8u * huge < some)
            atomicAdd(&at->x, 0x10000u + (8u * large < some ? 1u : 0u));
    }
}

// Sends the slices whose samples the split does not hold well enough to the
// vector kernel.  A term of the split ends 2^-40 below the slice's maximum: a
// sample of less than 2^-16 of it has 24 bits no more.  That is nothing to a
// pixel that also sees larger ones (the sum's own rounding is coarser), but a
// pixel whose samples are all small, beside a few that are huge (a hot pixel
// or column), would lose its value.  The floor's error of a pixel, 2^-26
// sqrt(2 n / 3) for n angles, stays below that of a float32 sum after every
// angle, r 2^-25 n / sqrt(2), from 128 angles on if the rms of its samples is r
// >= 2^-4 (with the maximum scaled to 2^14 .. 2^15).  A pixel at a distance d
// from the axis sees the columns within d of the centre, so a slice stays if
// for every d, in steps of a span of 32 columns, of the (span, angle) pairs in
// there that are not all zero
//   * half have one sample in 8 of kLarge = 2^-2 or more (r >= 2^-4), or
//   * one in 16 has one sample in 8 of kHuge = 2^3 or more: an object in air
//     whose edges fade out, which every pixel sees from 2 / (16 pi) of
//     the angles at least (r >= 2^-1).
template <bool BATCH>
__global__ __launch_bounds__(256) void range_kernel(
    const MatJob* __restrict__ jobs, int njobs, MatJob one) {
    unsigned b;
    const MatJob& job = find_job<BATCH>(jobs, njobs, one, kRange, b);
    const int nrow = job.r.a.nrow, ns = span_count(job.r.a.ncol);
    const int j = job.m.group_op * kGroup + (int)b;
    const double center = job.r.a.center;
    const uint2* sp = job.m.spans + (size_t)j * ns;
    bool any = false;
    for (int k = threadIdx.x; k < ns; k += 256) any |= (sp[k].x & 0xffffu) != 0u;
    if (!__syncthreads_or(any)) return;
    const int mid = (int)fmin(fmax(center / kSpanCols, 0.0), ns - 1.0);
    bool redo = false;
    for (int d = threadIdx.x; d < ns; d += 256) {
        unsigned long long low = 0, faint = 0, some = 0;
        for (int k = max(mid - d, 0); k <= min(mid + d, ns - 1); ++k) {
            low += sp[k].x & 0xffffu;
            faint += sp[k].x >> 16;
            some += (unsigned)nrow - sp[k].y;
        }
        redo |= 2 * low > some && 16 * (some - faint) < some;
    }
    if (__syncthreads_or(redo) && threadIdx.x == 0) job.m.smax[j] = kRedo;
}

__device__ __forceinline__ double clamp_pos(double f, double w1) {
    return fmin(fmax(f, 0.0), w1);
}

// a wave-uniform value in scalar registers
__device__ __forceinline__ double to_scalar(double v) {
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Geometry of one angle for a tile.  Positions are fixed point in the low
// word of a double: 1.5 * 2^25 puts 27 fraction bits there (5 integer bits:
// enough for the offset within a window; the 2 folds in the 1 of
// -e = (127 - e) + 1 mod 16), 2^-23 rounds to the 22 bits that are kept;
// 1.5 * 2^28 puts 24 fraction bits (8 integer bits: enough for a tile).
constexpr double kPosMagic = 50331648.0 + 2.0 + 1.0 / 8388608.0;
constexpr double kWinMagic = 402653184.0;
constexpr double kSlack = 1.0 / 1048576.0;
struct alignas(16) Angle {
    double c, s;       // cos, sin
    double pos;        // position = c x + s y + pos, less L, plus kPosMagic
    double win;        // win - (c x + s y): kWinMagic less the lowest
                       // position of the block centred at (x, y), less L,
                       // plus the slack
    int L;             // tile's first column (even)
    int inner;         // every pixel of the tile is in range
    int valid;         // the angle exists
    int pad;
};

// Tile (tx, ty) of slice groups grp .. grp + SG - 1
template <int PL, int SG>
__device__ __forceinline__ void matrix_tile(const BpArgs& a, const MatArgs& ma,
                                            int tx, int ty, int grp) {
    using TL = Tile<SG>;
    constexpr int S = SG * kGroup;
    constexpr int ROWS = TL::rows;
    constexpr int BX = TL::X / 4 / TL::wx;   // blocks per wave, side by side
    static_assert(TL::Y / 4 * TL::wx == kWaves, "one row of blocks per wave");
    // staging: a strip is the records of one (angle, slice group); a wave
    // loads a SHARE-th of one, a 16-lane group RUN consecutive records
    constexpr int SHARE = kWaves / (kStep * SG);
    constexpr int WROWS = ROWS / SHARE;
    constexpr int RUN = (WROWS + 3) / 4;
    // a record: two pairs' high and low parts, or four pairs (WIDE)
    constexpr bool WIDE = PL == 1;
    constexpr int EXTRA = WIDE ? 3 : 1;               // pairs past a record
    constexpr int kTerms = 2 * PL;                    // products per group
    constexpr unsigned kRow = S * 16;
    constexpr unsigned kBuf = kStep * ROWS * kRow;    // one step's records
    static_assert(WROWS * SHARE == ROWS && SHARE * kStep * SG == kWaves,
                  "rows split evenly");
    using Raw = typename std::conditional<PL == 2, uint2_t, unsigned>::type;
    constexpr int kPairBytes = kGroup * sizeof(Raw);  // one pair, 16 slices

    // [8] selectors, three steps' angles [3][kStep], then records
    // [2][kStep][ROWS][S], an angle's rows in descending order (the window
    // counts down, see place)
    extern __shared__ uint4_t lds[];
    const unsigned sh = (unsigned)(size_t)(LdsQuad)lds;
    constexpr unsigned kAngAt = 8 * 16;
    Angle* const angles = reinterpret_cast<Angle*>(lds + 8);
    constexpr unsigned kRecAt = kAngAt + 3 * kStep * sizeof(Angle);

    const int tid = threadIdx.x, lane = tid & 63;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n16 = lane & 15, k4 = lane >> 4;
    const int x0 = tx * TL::X, y0 = ty * TL::Y;
    const int xw = x0 + 4 * BX * (wv % TL::wx);       // this wave's pixels
    const int yw = y0 + 4 * (wv / TL::wx);
    const int C = a.ncol, N = a.nrow;
    const double ic = a.icenter, cen = a.center, w1 = (double)(C - 1);

    float4_t acc[BX][SG];
#pragma unroll
    for (int i = 0; i < BX; ++i)
#pragma unroll
        for (int g = 0; g < SG; ++g) acc[i][g] = float4_t{0, 0, 0, 0};

    // a tile whose every pixel the mask removes needs no sums
    if (!tile_masked<TL::X, TL::Y>(a, x0, y0)) {
        // selectors of the byte permutation that places (1 - w, w) at columns
        // d, d + 1 of the window's 8: entry d <= 6, one word per column
        // pair; entry 7 places nothing (pixels out of range)
        if (tid < 32) {
            const int d = tid >> 2, p = tid & 3;
            unsigned sel = 0;
            for (int h = 0; h < 2; ++h) {
                const int col = 2 * p + h;
                const unsigned v = d == 7 ? 0x0c0cu
                                   : col == d ? 0x0100u
                                   : col == d + 1 ? 0x0302u : 0x0c0cu;
                sel |= v << (16 * h);
            }
            reinterpret_cast<unsigned*>(lds)[tid] = sel;
        }

        // the lane's pixel and, for the windows, the block's centre, both in
        // the grid column of 64 that holds the tile
        const int xg = x0 & ~63;
        const double xl = (double)(xg + (n16 & 3)) - ic;
        const double yl = (double)(yw + (n16 >> 2)) - ic;
        const double xb = to_scalar((double)xg + 1.5 - ic);
        const double yb = to_scalar((double)yw + 1.5 - ic);

        auto trig = [&](int a0) { return ma.trig[min(a0 + k4, N - 1)]; };
        // lanes 0, 16, 32, 48 of one wave: the angles of the step at a0
        auto geometry = [&](int a0, float2 tf, unsigned slot) {
            const double2 t = make_double2((double)tf.x, (double)tf.y);
            const double xm = (double)x0 + 0.5 * (TL::X - 1) - ic;
            const double ym = (double)y0 + 0.5 * (TL::Y - 1) - ic;
            const double fm = det_pos(xm * t.x, ym, t.y, cen);
            const double ext = fma(0.5 * (TL::Y - 1), fabs(t.y),
                                   0.5 * (TL::X - 1) * fabs(t.x));
            const double lo = fm - ext - 2.0 * kSlack;
            const double hi = fm + ext + 2.0 * kSlack;
            Angle g;
            g.c = t.x;
            g.s = t.y;
            g.L = (int)clamp_pos(lo, w1) & ~1;
            g.valid = a0 + k4 < N;
            g.inner = g.valid && lo >= 0.0 && hi <= w1;
            g.pad = 0;
            // rounded to fixed point before L is taken off, so that the bits
            // of a block do not depend on the tile it lies in
            g.pos = ma.pos0 - (double)g.L;
            g.win = (kWinMagic -
                     (cen - fma(1.5, fabs(t.x) + fabs(t.y), kSlack))) +
                    (double)g.L;
            if (n16 == 0) angles[slot * kStep + k4] = g;
        };

        // this wave's share of a strip
        const int sk = wv / SHARE / SG, sg = wv / SHARE % SG;
        const int row0 = wv % SHARE * WROWS + k4 * RUN;
        const int row_end = wv % SHARE * WROWS + WROWS;
        const unsigned lane_at = (unsigned)(row0 * kGroup + n16) * sizeof(Raw);
        // (an idle last group repeats the one before it)
        const int gr = min(grp + sg, ma.group_have - 1) - ma.group_op;
        Raw raw[RUN + EXTRA];
        // (pairs past the row's end are the next row's, or the buffer's zero
        // tail: finite, and their weights are zero)
        auto load = [&](int a0, unsigned slot) {
            const int ai = min(a0 + sk, N - 1);
            const int L =
                __builtin_amdgcn_readfirstlane(angles[slot * kStep + sk].L);
            const char* src =
                reinterpret_cast<const char*>(ma.op) +
                (((size_t)gr * N + ai) * ma.npair + (L >> 1)) * kPairBytes;
#pragma unroll
            for (int u = 0; u < RUN + EXTRA; ++u)
                raw[u] = *reinterpret_cast<const Raw*>(
                    src + (lane_at + u * kPairBytes));
        };
        auto store = [&](unsigned buf) {
            // row RUN - 1 of the run lies lowest
            const unsigned dst =
                sh + kRecAt + buf * kBuf +
                (sk * ROWS + ROWS - RUN - row0) * kRow +
                (sg * kGroup + n16) * 16;
#pragma unroll
            for (int u = 0; u < RUN; ++u) {
                const Raw* r = raw + u;
                if (RUN * 4 != WROWS && row0 + u >= row_end) continue;
                const unsigned at = dst + (RUN - 1 - u) * kRow;
                if constexpr (PL == 2) {
                    // two 8-byte stores: one instruction, no copies of the
                    // entry that two records share
                    *(LdsPair)(at) = r[0];
                    *(LdsPair)(at + 8) = r[1];
                } else {
                    *(LdsQuad)(at) = uint4_t{r[0], r[1], r[2], r[3]};
                }
            }
        };

        // One block of pixels goes through four stages, a stage per turn of
        // the block loop, so that LDS latencies and the matrix unit's own lie
        // behind other blocks' work: its weights' halves and selectors
        // (place), the weight operands and the records they meet (operands),
        // the products, and the sum into the total.
        struct Place {
            unsigned pa, pb, at;
            uint4_t sel;
        };
        struct Operands {
            half8_t w[kTerms];
            half8_t r[SG][PL == 2 ? 2 : 1];
        };
        struct Sums {
            float4_t t[SG];
        };
        // p: the lane's position; e: 127 - the window's record (its sign
        // takes one shift-add off the offset in the window)
        auto place = [&](unsigned p, unsigned e, unsigned lbase) {
            Place k;
            const unsigned rel = (e << 28) + p;
            k.sel = *(LdsQuad)(((rel >> 23) & 0x70u) | sh);
            k.at = e * kRow + lbase;
            const unsigned T = p & 0x07ffffe0u;        // w, 22 bits
            const unsigned Q = 0x08000000u - T;        // 1 - w
            k.pa = __builtin_amdgcn_perm(T, Q, 0x07060302u);
            k.pb = __builtin_amdgcn_perm(T, Q, 0x05040100u);
            k.pb = __builtin_bit_cast(
                unsigned,
                (ushort2_t)(__builtin_bit_cast(ushort2_t, k.pb) >> 5));
            // 2^-24 a -> 2^-13 a, so that a and b share the scale 2^-2
            const half2_t up = {(_Float16)2048.0f, (_Float16)2048.0f};
            k.pa = __builtin_bit_cast(unsigned,
                                      __builtin_bit_cast(half2_t, k.pa) * up);
            return k;
        };
        auto operands = [&](const Place& k) {
            Operands o;
#pragma unroll
            for (int g = 0; g < SG; ++g) {
                if constexpr (PL == 2) {
                    // the record and the second one after it
                    o.r[g][0] = *(LdsHalf8)(k.at + 2 * kRow + g * kGroup * 16);
                    o.r[g][1] = *(LdsHalf8)(k.at + g * kGroup * 16);
                } else {
                    o.r[g][0] = *(LdsHalf8)(k.at + g * kGroup * 16);
                }
            }
            unsigned wa[4], wb[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                wa[q] = __builtin_amdgcn_perm(0u, k.pa, k.sel[q]);
                wb[q] = __builtin_amdgcn_perm(0u, k.pb, k.sel[q]);
            }
            if constexpr (!WIDE) {
                // records hold a pair's high and low parts side by side
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    o.w[h] = __builtin_bit_cast(
                        half8_t, (uint4_t{wb[2 * h], wb[2 * h], wb[2 * h + 1],
                                          wb[2 * h + 1]}));
                    o.w[2 + h] = __builtin_bit_cast(
                        half8_t, (uint4_t{wa[2 * h], wa[2 * h], wa[2 * h + 1],
                                          wa[2 * h + 1]}));
                }
            } else {
                o.w[0] = __builtin_bit_cast(
                    half8_t, (uint4_t{wb[0], wb[1], wb[2], wb[3]}));
                o.w[1] = __builtin_bit_cast(
                    half8_t, (uint4_t{wa[0], wa[1], wa[2], wa[3]}));
            }
            return o;
        };
        // A step's sum starts from zero and is added to the total in the
        // vector unit: the matrix unit truncates, and into the total that
        // would be a bias (1801 angles of positive samples: -7e-7).
        auto products = [&](const Operands& o) {
            Sums u;
#pragma unroll
            for (int g = 0; g < SG; ++g) u.t[g] = float4_t{0, 0, 0, 0};
            // (small terms first: they are truncated at their own size)
#pragma unroll
            for (int q = 0; q < kTerms; ++q)
#pragma unroll
                for (int g = 0; g < SG; ++g)
                    u.t[g] = __builtin_amdgcn_mfma_f32_16x16x32_f16(
                        o.w[q], o.r[g][PL == 2 ? q & 1 : 0], u.t[g], 0, 0, 0);
            return u;
        };
        auto total = [&](const Sums& u, float4_t (&ac)[SG]) {
#pragma unroll
            for (int g = 0; g < SG; ++g)
#pragma unroll
                for (int q = 0; q < 4; ++q) ac[g][q] += u.t[g][q];
        };
        // the other stages' instructions between the matrix instructions
        auto interleave = [&]() {
            constexpr int M = kTerms * SG;
            constexpr int V = (PL == 1 ? 22 : 30) + 4 * SG;
#pragma unroll
            for (int q = 0; q < M; ++q) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, (V + M - 1) / M,
                                                     0);
            }
        };

        if (wv == 0) {
            geometry(0, trig(0), 0);
            geometry(kStep, trig(kStep), 1);
        }
        __syncthreads();
        load(0, 0);
        store(0);
        __syncthreads();
        // step t: its angles are in slot t % 3; the samples of step t + 1 are
        // loaded and stored, and one wave works out the angles of step t + 2
        unsigned cur = 0, buf = 0, turn = 0;
        float2 tr = trig(2 * kStep);
        for (int a0 = 0; a0 < N; a0 += kStep) {
            const unsigned next = cur == 2 ? 0 : cur + 1;
            const unsigned after = next == 2 ? 0 : next + 1;
            if (wv == (int)turn) geometry(a0 + 2 * kStep, tr, after);
            turn = turn + 1 == kWaves ? 0 : turn + 1;
            // (past the last angle these repeat it)
            load(a0 + kStep, next);
            const Angle* g = angles + cur * kStep + k4;
            const double c = g->c, s = g->s;
            // record 127 - e of the lane's angle and the second one after it
            // (lower) start e rows past here
            const unsigned lbase =
                sh + kRecAt + buf * kBuf +
                (unsigned)(k4 * ROWS + ROWS - 1 - 127 - (WIDE ? 0 : 2)) * kRow +
                n16 * 16;
            const double fr = fma(yl, s, fma(xl, c, g->pos));
            unsigned p[BX], e[BX];
            if (__all(g->inner)) {
                const double bn = fma(-yb, s, fma(-xb, c, g->win));
#pragma unroll
                for (int i = 0; i < BX; ++i) {
                    const double m = (double)(xw - xg + 4 * i);
                    p[i] = (unsigned)__double2loint(fma(m, c, fr));
                    e[i] = (unsigned)__double2loint(fma(-m, c, bn)) >> 25;
                }
            } else {
                // some pixel or angle is out of range: the vector kernel's
                // exact position decides which; windows that start in the
                // row and in-range pixels' weights are those above (a tile of
                // the other shape may take the same block there), other
                // windows are clamped to the row
                const double l = (double)g->L;
                const double bn = fma(-yb, s, fma(-xb, c, g->win));
                // (where the tile is in range a window starts kSlack - 2^-23
                // or more past L, so the clamps change none)
                const double q_end = kWinMagic - (w1 - l + 0.5 * kSlack);
                const bool valid = g->valid;
                // (16 bits: opaque, so that the columns' coordinates are not
                // kept in registers across the angle loop; in float32 the
                // copies would spill)
                double xo = xl, yo = yl;
                if constexpr (PL == 1) asm volatile("" : "+v"(xo), "+v"(yo));
#pragma unroll
                for (int i = 0; i < BX; ++i) {
                    const double m = (double)(xw - xg + 4 * i);
                    const double q = fmin(fmax(fma(-m, c, bn), q_end),
                                          kWinMagic - 0.5 * kSlack);
                    e[i] = (unsigned)__double2loint(q) >> 25;
                    const double f = det_pos((xo + m) * c, yo, s, cen);
                    const bool in = f >= 0.0 && f <= w1;
                    const double edge = clamp_pos(f, w1) - l + kPosMagic;
                    p[i] = (unsigned)__double2loint(in ? fma(m, c, fr) : edge);
                    // selector 7: no weights
                    unsigned none = e[i];
                    asm volatile("" : "+v"(none));
                    if (!valid || (!in && !a.edge_pad))
                        p[i] = 0x38000000u - (none << 28);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            Place pl = place(p[0], e[0], lbase);
            Operands op = operands(pl);
            if (BX > 1) pl = place(p[1], e[1], lbase);
            Sums su;
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int i = 0; i < BX; ++i) {
                const Sums next_su = products(op);
                if (i > 0) total(su, acc[i - 1]);
                if (i + 1 < BX) op = operands(pl);
                if (i + 2 < BX) pl = place(p[i + 2], e[i + 2], lbase);
                su = next_su;
                interleave();
                __builtin_amdgcn_sched_barrier(0);
                // the samples have arrived: their stores go beside the
                // other waves' products
                if (i == BX * 3 / 4 - 1) store(buf ^ 1);
            }
            total(su, acc[BX - 1]);
            tr = trig(a0 + 3 * kStep);
            cur = next;
            buf ^= 1;
            __syncthreads();
        }
    }

    // lane: slice n16 of each group; rows 4 g + r of the product are the
    // pixels (x + r, y + g), g = lane >> 4
    const bool vec = (C & 3) == 0 && (reinterpret_cast<size_t>(a.recon) & 15) == 0;
#pragma unroll
    for (int g = 0; g < SG; ++g) {
        const int j = (grp + g) * kGroup + n16;
        if (j >= a.nslice) continue;
        const unsigned bits = ma.smax[j];
        if (bits > kMaxBits) continue;  // the vector kernel's
        const int ex = 2 - (ma.scaled ? scale_exp(bits) : 0);
        const int y = yw + k4;
        if (y >= C) continue;
        float* row = a.recon + ((size_t)y * a.nslice + j) * C;
        const long long dy = y - a.mask_c;
#pragma unroll
        for (int i = 0; i < BX; ++i) {
            const int x = xw + 4 * i;
            __builtin_amdgcn_sched_barrier(0);
            float4_t v;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                float t = ldexpf(acc[i][g][q], ex);
                if (a.use_mask) {
                    const long long dx = x + q - a.mask_c;
                    t *= (double)(dx * dx + dy * dy) <= a.mask_r2 ? 1.0f
                                                                  : 0.0f;
                }
                if (a.apply_scale) {
                    t = t * a.pi32;
                    t = t / a.denom;
                }
                v[q] = t;
            }
            if (vec && x + 3 < C) {
                *reinterpret_cast<float4_t*>(row + x) = v;
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q)
                    if (x + q < C) row[x + q] = v[q];
            }
        }
    }
}

// Workgroups go to the 8 XCDs in turn.  An XCD's consecutive ones take a
// kPatchX x kPatchY patch of tiles, whose strips of an angle overlap: one
// L2 then holds them for as many angles as the workgroups drift apart.
// One stack: slice groups x patches (a multiple of 8) x tiles of a patch.  A
// batch has no workgroups to spare for patches that hang over small images:
// every XCD takes an eighth of a stack's tiles, four rows of them at a time.
template <int PL, int SG, bool BATCH>
__global__ __launch_bounds__(kThreads) void bp_matrix_kernel(
    const MatJob* __restrict__ jobs, int njobs, MatJob one) {
    unsigned b;
    const MatJob& job = find_job<BATCH>(jobs, njobs, one,
                                        SG == 2 ? kPairs : kSingle, b);
    const BpArgs& a = job.r.a;
    const MatArgs& ma = job.m;
    const int tiles_x = (a.ncol + Tile<SG>::X - 1) / Tile<SG>::X;
    const int tiles_y = (a.ncol + Tile<SG>::Y - 1) / Tile<SG>::Y;
    int tx, ty, grp;
    if constexpr (BATCH) {
        // pairs from group 0 on, a last odd group
        const unsigned tiles = tiles_x * tiles_y, groups = ma.group_have;
        const unsigned items = SG == 2 ? tiles * (groups / 2) : tiles;
        const unsigned c = b & 7u;  // workgroups of one XCD are 8 apart
        const unsigned i = c * (items >> 3) + min(c, items & 7u) + (b >> 3);
        const unsigned t = i % tiles, row4 = tiles_x * kPatchY;
        const unsigned y0 = t / row4 * kPatchY, in = t % row4;
        const unsigned h = min(kPatchY, tiles_y - y0);
        tx = in / h;
        ty = y0 + in % h;
        grp = SG == 2 ? i / tiles * 2 : groups - 1;
    } else {
        const unsigned xcd = b & 7u, seq = b >> 3;
        const unsigned patch = (seq / (kPatchX * kPatchY)) * 8u + xcd;
        const unsigned in = seq % (kPatchX * kPatchY);
        const unsigned px = patch % ma.patches_x, pr = patch / ma.patches_x;
        tx = px * kPatchX + in % kPatchX;
        ty = (pr % ma.patches_y) * kPatchY + in / kPatchX;
        grp = ma.group0 + (pr / ma.patches_y) * SG;
        if (tx >= tiles_x || ty >= tiles_y || grp >= ma.group_end) return;
    }
    matrix_tile<PL, SG>(a, ma, tx, ty, grp);
}

// workgroups of 256 threads in a grid's x: its work items are a 32-bit number
constexpr long long kMaxBlocks = (1LL << 24) - 1;

template <int SG> constexpr size_t matrix_lds() {
    return (size_t)(2 * kStep * Tile<SG>::rows * SG * kGroup + 8) *
               sizeof(uint4_t) +
           3 * kStep * sizeof(Angle);
}

template <int PL, int SG, bool BATCH>
int launch_kernel(const MatJob* jobs, int njobs, const MatJob& one,
                  long long blocks, hipStream_t stream) {
    if (blocks > kMaxBlocks / 4)
        return set_error(ATH_ERR_UNSUPPORTED, "back-projection grid too large");
    auto kern = bp_matrix_kernel<PL, SG, BATCH>;
    const int st = allow_dynamic_lds(reinterpret_cast<const void*>(kern),
                                     matrix_lds<SG>());
    if (st != ATH_OK) return st;
    hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(kThreads),
                       matrix_lds<SG>(), stream, jobs, njobs, one);
    return check_hip(hipGetLastError(), "bp_matrix_kernel launch");
}

template <int PL, int SG>
int launch_matrix(MatJob job, int groups, hipStream_t stream) {
    const int ncol = job.r.a.ncol;
    const int tiles_x = (ncol + Tile<SG>::X - 1) / Tile<SG>::X;
    const int tiles_y = (ncol + Tile<SG>::Y - 1) / Tile<SG>::Y;
    MatArgs& ma = job.m;
    ma.group_end = ma.group0 + groups;
    ma.patches_x = (tiles_x + kPatchX - 1) / kPatchX;
    ma.patches_y = (tiles_y + kPatchY - 1) / kPatchY;
    const long long patches =
        (long long)ma.patches_x * ma.patches_y * (groups / SG);
    return launch_kernel<PL, SG, false>(
        nullptr, 0, job, (patches + 7) / 8 * 8 * (kPatchX * kPatchY), stream);
}

// rounds of 256 workgroups that `units` slice groups (or pairs) take
template <int SG> double rounds_of(int ncol, int units) {
    const double tiles = (double)((ncol + Tile<SG>::X - 1) / Tile<SG>::X) *
                         ((ncol + Tile<SG>::Y - 1) / Tile<SG>::Y);
    return std::ceil(tiles * units / 256.0);
}

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }
int groups_of(int nslice) { return (nslice + kGroup - 1) / kGroup; }
int planes_of(int dtype) { return dtype == ATH_F32 ? 2 : 1; }

// Slice groups split and summed at a time: as many pairs as 2 GiB of split
// samples hold, so that the workspace stays small beside a large stack (64 x
// 1801 x 2560 takes 1.2 GB).
int part_groups(int planes, int nrow, int ncol, int groups) {
    const size_t bytes = (size_t)nrow * ((ncol + 1) / 2) * kGroup * 4 * planes;
    const size_t n = ((size_t)2 << 30) / bytes / 2 * 2;
    return (int)std::min<size_t>(groups, std::max<size_t>(n, 2));
}

// Lays a stack's job out in `work` (null: only counts) with `part` slice
// groups of split samples; returns the bytes.
size_t set_job(MatJob& job, const BpArgs& a, int dtype, int part, char* work) {
    const size_t nmax = (size_t)groups_of(a.nslice) * kGroup;
    const int planes = planes_of(dtype);
    // maxima, then the spans' counts: cleared together
    const size_t nzero = nmax * (1 + 2 * (size_t)span_count(a.ncol));
    const size_t trig_at = align256(nzero * sizeof(unsigned));
    const size_t op_at = trig_at + align256((size_t)a.nrow * sizeof(float2));
    MatArgs& m = job.m;
    m.smax = reinterpret_cast<unsigned*>(work);
    m.spans = reinterpret_cast<uint2*>(work + nmax * sizeof(unsigned));
    m.trig = reinterpret_cast<float2*>(work + trig_at);
    m.op = reinterpret_cast<unsigned*>(work + op_at);
    m.npair = (a.ncol + 1) / 2;
    m.nop = (size_t)part * kGroup * a.nrow * m.npair * planes;
    m.pos0 = a.center + kPosMagic;
    m.scaled = dtype != ATH_F16;
    m.nzero = (int)nzero;
    m.ntail = kTailPairs * kGroup * planes;
    m.max_rows = std::min(a.nrow, 128);
    m.group0 = m.group_op = 0;
    m.group_have = part;
    m.group_end = 0;
    m.patches_x = m.patches_y = 0;
    // slices with non-finite or huge samples are the vector kernel's
    job.r.a = a;
    job.r.a.only_above = m.smax;
    job.r.a.above = kMaxBits;
    job.r.begin = 0;
    for (unsigned& b : job.begin) b = 0;
    return op_at + (m.nop + m.ntail) * sizeof(unsigned);
}

int split_block_columns(const MatJob& j) { return (j.r.a.ncol + 127) / 128; }
long long clear_blocks(const MatJob& j) {
    return ((long long)std::max({j.r.a.nrow, j.m.nzero, j.m.ntail}) + 255) /
           256;
}
long long max_blocks(const MatJob& j) {
    return (long long)j.r.a.nslice * j.m.max_rows;
}
long long split_blocks(const MatJob& j, int groups) {
    return (long long)split_block_columns(j) * j.r.a.nrow * groups;
}

#define ATH_MATRIX_LAUNCH(KERNEL, BLOCKS, ROWS, JOBS, NJOBS, ONE)             \
    do {                                                                      \
        const long long n_ = (BLOCKS);                                        \
        if (n_ > kMaxBlocks)                                                  \
            return set_error(ATH_ERR_UNSUPPORTED,                             \
                             "back-projection grid too large");               \
        if (n_ > 0) {                                                         \
            hipLaunchKernelGGL((KERNEL), dim3((unsigned)n_, ROWS), dim3(256), \
                               0, s, JOBS, NJOBS, ONE);                       \
            const int st_ = check_hip(hipGetLastError(), #KERNEL " launch");  \
            if (st_ != ATH_OK) return st_;                                    \
        }                                                                     \
    } while (0)

template <typename T, int PL>
int run_matrix(const BpArgs& a, int dtype, int acc, char* work,
               hipStream_t s) {
    const int groups = groups_of(a.nslice);
    const int part = part_groups(PL, a.nrow, a.ncol, groups);
    MatJob job;
    set_job(job, a, dtype, part, work);
    const MatJob* none = nullptr;
    ATH_MATRIX_LAUNCH(clear_kernel<false>, clear_blocks(job), 1, none, 0, job);
    ATH_MATRIX_LAUNCH((slice_max_kernel<T, false>), max_blocks(job), 1, none,
                      0, job);
    for (int g0 = 0; g0 < groups; g0 += part) {
        const int n = std::min(part, groups - g0);
        job.m.group0 = job.m.group_op = g0;
        job.m.group_have = g0 + n;
        ATH_MATRIX_LAUNCH((split_kernel<T, PL, false>),
                          (long long)split_block_columns(job) * n, a.nrow,
                          none, 0, job);
        if (job.m.scaled)
            ATH_MATRIX_LAUNCH(range_kernel<false>,
                              std::min(n * kGroup, a.nslice - g0 * kGroup),
                              1, none, 0, job);
        // Pairs of groups; a last odd group by itself unless an idle one
        // beside it is cheaper, which it is where the launch does not fill the
        // chip twice (rounds of 256 workgroups, at the measured 0.69 against
        // 0.88 us per angle)
        int pairs = n / 2;
        if (n & 1) {
            const double with = rounds_of<2>(a.ncol, pairs + 1) * 0.69;
            const double apart = rounds_of<2>(a.ncol, pairs) * 0.69 +
                                 rounds_of<1>(a.ncol, 1) * 0.88;
            if (with < apart) ++pairs;
        }
        if (pairs) {
            const int st = launch_matrix<PL, 2>(job, 2 * pairs, s);
            if (st != ATH_OK) return st;
            job.m.group0 += 2 * pairs;
        }
        if (n > 2 * pairs) {
            const int st = launch_matrix<PL, 1>(job, 1, s);
            if (st != ATH_OK) return st;
        }
    }
    // (workgroups of other slices leave at once)
    return back_projection(job.r.a, dtype, acc, 0, 0, s);
}

// ---- many stacks in one set of launches ------------------------------------
// Stack by stack the small ones would leave most of the chip idle, one after
// another.  64 stacks of 361 x 6 x 128, filter included: 15.6 ms so, 1.6 ms here
// (the vector kernel's work list 1.7); 16 of 721 x 16 x 512 8.6 and 6.6 (15.0);
// 8 of 901 x 12 x 1024, which fill the chip by themselves, 12.5 and 12.5 (24.7).
struct MatPlan {
    int njobs, dtype, acc;
    unsigned blocks[kStages], redo_blocks;
};
constexpr size_t kPlanJobs = 256;
static_assert(sizeof(MatPlan) <= kPlanJobs, "plan header");

template <typename T, int PL>
int run_batch(const MatPlan& p, const MatJob* jobs, hipStream_t s) {
    const MatJob one{};
    const unsigned* n = p.blocks;
    ATH_MATRIX_LAUNCH(clear_kernel<true>, n[kClear], 1, jobs, p.njobs, one);
    ATH_MATRIX_LAUNCH((slice_max_kernel<T, true>), n[kMaxima], 1, jobs,
                      p.njobs, one);
    ATH_MATRIX_LAUNCH((split_kernel<T, PL, true>), n[kSplit], 1, jobs, p.njobs,
                      one);
    if (p.dtype != ATH_F16)
        ATH_MATRIX_LAUNCH(range_kernel<true>, n[kRange], 1, jobs, p.njobs,
                          one);
    int st = ATH_OK;
    if (n[kPairs])
        st = launch_kernel<PL, 2, true>(jobs, p.njobs, one, n[kPairs], s);
    if (st == ATH_OK && n[kSingle])
        st = launch_kernel<PL, 1, true>(jobs, p.njobs, one, n[kSingle], s);
    if (st != ATH_OK) return st;
    return back_projection_redo(&jobs->r, sizeof(MatJob), p.njobs,
                                p.redo_blocks, p.dtype, p.acc, s);
}
#undef ATH_MATRIX_LAUNCH

// what the matrix path takes
int check_matrix(const BpArgs& a, int dtype, int acc) {
    if (a.ncol > kMaxMatrixCols || a.nrow > 65535 || a.nslice > 65535)
        return set_error(ATH_ERR_UNSUPPORTED,
                         "matrix back-projection: at most 32768 columns, "
                         "65535 angles and 65535 slices");
    if (dtype == ATH_F32) {
        if (acc != ATH_ACC_F32SEQ && acc != ATH_ACC_F32)
            return set_error(ATH_ERR_INVALID_ARG,
                             "matrix back-projection: acc must be "
                             "ATH_ACC_F32SEQ or ATH_ACC_F32");
        return ATH_OK;
    }
    if (acc != ATH_ACC_F32)
        return set_error(ATH_ERR_UNSUPPORTED,
                         "back-projection: float16/bfloat16 sinograms need "
                         "acc = ATH_ACC_F32");
    if (dtype != ATH_F16 && dtype != ATH_BF16)
        return set_error(ATH_ERR_INVALID_ARG,
                         "back-projection: bad sinogram dtype");
    return ATH_OK;
}

}  // namespace

size_t back_projection_matrix_workspace(int dtype, int nrow, int nslice,
                                        int ncol) {
    BpArgs a{};
    a.nrow = nrow;
    a.nslice = nslice;
    a.ncol = ncol;
    MatJob job;
    return set_job(job, a, dtype,
                   part_groups(planes_of(dtype), nrow, ncol,
                               groups_of(nslice)),
                   nullptr);
}

int back_projection_matrix(const BpArgs& a, int dtype, int acc, void* work,
                           hipStream_t s) {
    const int st = check_matrix(a, dtype, acc);
    if (st != ATH_OK) return st;
    char* w = static_cast<char*>(work);
    if (dtype == ATH_F32) return run_matrix<float, 2>(a, dtype, acc, w, s);
    if (dtype == ATH_F16) return run_matrix<__half, 1>(a, dtype, acc, w, s);
    return run_matrix<__hip_bfloat16, 1>(a, dtype, acc, w, s);
}

size_t matrix_batch_plan_bytes(int njobs) {
    return kPlanJobs + (size_t)njobs * sizeof(MatJob);
}

size_t matrix_batch_job_bytes(int dtype, int nrow, int nslice, int ncol) {
    BpArgs a{};
    a.nrow = nrow;
    a.nslice = nslice;
    a.ncol = ncol;
    MatJob job;
    return align256(set_job(job, a, dtype, groups_of(nslice), nullptr));
}

void matrix_batch_begin(void* plan, int dtype, int acc) {
    MatPlan p{};
    p.dtype = dtype;
    p.acc = acc;
    *static_cast<MatPlan*>(plan) = p;
}

int matrix_batch_add(void* plan, const BpArgs& a, void* work) {
    MatPlan& p = *static_cast<MatPlan*>(plan);
    const int st = check_matrix(a, p.dtype, p.acc);
    if (st != ATH_OK) return st;
    MatJob& j = reinterpret_cast<MatJob*>(static_cast<char*>(plan) +
                                          kPlanJobs)[p.njobs];
    const int groups = groups_of(a.nslice);
    set_job(j, a, p.dtype, groups, static_cast<char*>(work));
    j.m.max_rows = std::min(a.nrow, 32);
    const auto tiles = [&](int x, int y) {
        return (long long)((a.ncol + x - 1) / x) * ((a.ncol + y - 1) / y);
    };
    long long n[kStages];
    n[kClear] = clear_blocks(j);
    n[kMaxima] = max_blocks(j);
    n[kSplit] = split_blocks(j, groups);
    n[kRange] = a.nslice;
    n[kPairs] = tiles(Tile<2>::X, Tile<2>::Y) * (groups / 2);
    n[kSingle] = groups & 1 ? tiles(Tile<1>::X, Tile<1>::Y) : 0;
    const long long redo = redo_tiles(a.nslice, a.ncol);
    const char* large = "matrix back-projection: batch too large";
    for (int k = 0; k < kStages; ++k)
        if (p.blocks[k] + n[k] >
            (k == kPairs || k == kSingle ? kMaxBlocks / 4 : kMaxBlocks))
            return set_error(ATH_ERR_UNSUPPORTED, large);
    if (p.redo_blocks + redo > kMaxBlocks)
        return set_error(ATH_ERR_UNSUPPORTED, large);
    for (int k = 0; k < kStages; ++k) {
        j.begin[k] = p.blocks[k];
        p.blocks[k] += (unsigned)n[k];
    }
    j.r.begin = p.redo_blocks;
    p.redo_blocks += (unsigned)redo;
    ++p.njobs;
    return ATH_OK;
}

int back_projection_matrix_batched(const void* plan, const void* plan_dev,
                                   hipStream_t s) {
    const MatPlan& p = *static_cast<const MatPlan*>(plan);
    const MatJob* jobs = reinterpret_cast<const MatJob*>(
        static_cast<const char*>(plan_dev) + kPlanJobs);
    if (p.dtype == ATH_F32) return run_batch<float, 2>(p, jobs, s);
    if (p.dtype == ATH_F16) return run_batch<__half, 1>(p, jobs, s);
    return run_batch<__hip_bfloat16, 1>(p, jobs, s);
}

}  // namespace ath
