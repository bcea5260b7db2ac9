// Baseline W4A16 GEMV (the reference's second extension, w4a16_ext.w4a16_gemv):
//
//   C[n] = fp16_rn((acc[n] - zW[n]) * sW[n]),   acc[n] = sum_k wv(n, k) * A[k]
//
// W int32 [N, K/8] row-major; nibble j (bits 4j..4j+3) of word k/8 of row n is the signed 4-bit
// weight wv(n, k) at k = 8*(k/8) + j (src/baseline/kernel.cu:19-28).  A fp16 [K]; sW, zW fp16 [N];
// fp32 epilogue (kernel.cu:31-33).
//
// Exact accumulation on the int8 matrix cores.  Every finite fp16 value a is an integer multiple
// of 2^-24 with |a * 2^24| < 2^40, so X = a * 2^24 is an exact integer.  Written in six signed
// base-256 digits, X = sum_j L_j * 256^j with L_j in [-128, 127] (the bytes of X + 0x808080808080,
// each minus 128), the dot product becomes six integer dot products
//     acc * 2^24 = sum_j 256^j * P_j,   P_j = sum_k wv(n, k) * L_j(k),
// and P_j is exact in int32 for K <= 2^20 (|wv * L| <= 1024).  One v_mfma_i32_16x16x64_i8 takes
// 16 rows of signed weight bytes (A operand) against a B operand whose columns 0..5 are the digit
// planes L_0..L_5 (columns 6..15 zero).  The int64 sum is rounded once to fp32, so the result is
// the exact dot product correctly rounded, whatever the split of K.  The reference accumulates in
// fp32 in k order (kernel.cu:22-30); its result differs from this one by that order's rounding
// error only.  Non-finite inputs follow IEEE semantics, which for this sum do not depend on the
// order: a NaN term, 0 * inf, or +inf together with -inf give NaN, otherwise any infinite term
// gives that infinity.
//
// Workgroup = 8 waves on 16 or 32 rows.  K is processed in segments of 4096: each of the 512 threads
// converts 8 A values into the digit table in LDS (laid out as the B operands), then each wave
// multiplies a contiguous eighth of the segment's 128-wide superchunks.  Lane (r, g) = (lane %
// 16, lane / 16) loads 16 bytes of row r per superchunk: the 32 weights at k = 128p + 32g .. +31,
// two MFMAs' worth (k offsets 0..15 and 16..31 of its group).  The MFMA output tiles of the 8
// waves (row 4g + i, digit r in lane (r, g), element i) are summed in LDS (exact integers).
//
// The A operand holds the nibbles offset by 8 (n ^ 8 = wv + 8, unsigned, two operations per dword
// instead of four), and one more MFMA per B operand with a weight of one in every row gives the digit
// sums, so P_j = sum_k (wv + 8) L_j - 8 sum_k L_j (below 15 * 128 * 2^20 < 2^31 before the
// subtraction).
//
// What bounds it: the launch and the first round trip at small N K (K = N = 4096: 4.5 us, 4.7 before this
// loop), the weight stream at large (N = 28672, K = 8192: 28.4 us, 4.2 TB/s, 33.6 before).  Rows that are
// not whole 16-byte units cost what others do: N = 9184, K = 888 3.9 us against 11.6 with 4-byte loads,
// N = 20000, K = 2000 7.1 against 19.0; two segments in flight: N = 4096, K = 14336 9.7 against 13.3; short K,
// only the loads that are multiplied: N = 8192, K = 512 3.3 against 4.0 (both timed in turn).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "w4a16.h"
#include "w4a16_device.h"
#include "w4a16_internal.h"

namespace w4a16 {

namespace {

// Workgroup barrier that orders LDS only (global loads stay in flight).
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

typedef int32_t i4v __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;                  // rows per MFMA row tile
constexpr int kWaves = 8;                  // waves per workgroup, splitting each segment's k range
constexpr int kThreads = kWaves * 64;
constexpr int kSeg = 4096;                 // k per digit-table segment
constexpr int kSuper = 128;                // k per superchunk (16 bytes of a row per lane)
constexpr int kDigits = 6;                 // base-256 digits of a * 2^24
constexpr int kSuperBytes = 2 * 4 * kDigits * 16;   // table bytes per superchunk (768)
constexpr int kPerWave = kSeg / kSuper / kWaves;   // superchunks per wave and segment (4)

static_assert(kSeg % (kSuper * kWaves) == 0, "segment must split evenly over the waves");
static_assert(kSeg / 8 == kThreads, "the table build gives each thread one 8-k unit");

// The balanced digits of a finite fp16 a (callers pass 0 for inputs that must count as 0), split at
// 2^24: a * 2^24 = hi * 2^24 + lo with hi an integer and lo in [-0x808080, 0x7F7F7F], so lo gives
// digits 0..2 and hi digits 3..5.  hi = rne(a + 1/510): the window of lo is off centre by 1/510, and
// the sum stays on the right side of it for every fp16 value (checked exhaustively, see the tests).
// Adding 2^23 + 0x408080 rounds to an integer and leaves hi + 0x408080 in the low mantissa bytes;
// lo + 0x808080 is formed exactly by one fma.  Seven fp32 operations per value.
constexpr float kHiMagic = 8388608.0f + 4227200.0f;          // 2^23 + 0x408080
constexpr float kHiBias = 0.00196f;                          // about 1/510
__device__ __forceinline__ void split_fixed(float f, uint32_t& lo, uint32_t& hi) {
    const float m = (f + kHiBias) + kHiMagic;
    hi = __builtin_bit_cast(uint32_t, m);
    lo = (uint32_t)__builtin_fmaf(f - (m - kHiMagic), 16777216.0f, 8421504.0f);
}

// 4x4 byte transpose: out[j] byte i = byte j of in[i] (v_perm_b32 picks bytes of {src0, src1},
// selector values 0..3 = src1, 4..7 = src0).
__device__ __forceinline__ void byte_transpose(const uint32_t (&in)[4], uint32_t (&out)[4]) {
    const uint32_t u01l = __builtin_amdgcn_perm(in[1], in[0], 0x05010400u);
    const uint32_t u01h = __builtin_amdgcn_perm(in[1], in[0], 0x07030602u);
    const uint32_t u23l = __builtin_amdgcn_perm(in[3], in[2], 0x05010400u);
    const uint32_t u23h = __builtin_amdgcn_perm(in[3], in[2], 0x07030602u);
    out[0] = __builtin_amdgcn_perm(u23l, u01l, 0x05040100u);
    out[1] = __builtin_amdgcn_perm(u23l, u01l, 0x07060302u);
    out[2] = __builtin_amdgcn_perm(u23h, u01h, 0x05040100u);
    out[3] = __builtin_amdgcn_perm(u23h, u01h, 0x07060302u);
}

// Digit dwords of four values: d[j] byte i = digit j of value i as a signed byte.  The bytes of lo
// are the digits plus 128 (XOR 0x80); of hi likewise, the third plus 64 (0x3F..0x41).
__device__ __forceinline__ void digit_dwords(const uint32_t (&lo)[4], const uint32_t (&hi)[4], uint32_t (&d)[kDigits]) {
    uint32_t t[4];
    byte_transpose(lo, t);
#pragma unroll
    for (int j = 0; j < 3; ++j) d[j] = t[j] ^ 0x80808080u;
    byte_transpose(hi, t);
    d[3] = t[0] ^ 0x80808080u;
    d[4] = t[1] ^ 0x80808080u;
    d[5] = (t[2] + 0x40404040u) ^ 0x80808080u;
}

// The even (shift 0) or odd (shift 4) nibbles of a word as bytes offset by 8: n ^ 8 = wv + 8.
__device__ __forceinline__ uint32_t offset_nibbles(uint32_t w, int shift) {
    return ((w >> shift) ^ 0x08080808u) & 0x0F0F0F0Fu;
}

// IEEE class of the non-finite terms of row n (only called when A holds inf or NaN).
// Returns 0 (none), 1 (+inf), 2 (-inf) or 3 (NaN).
__device__ int nonfinite_class(const uint32_t* __restrict__ wrow, const uint16_t* __restrict__ A, int K) {
    bool pos = false, neg = false, nan = false;
    for (int k = 0; k < K; ++k) {
        const uint32_t h = A[k];
        if (((h >> 10) & 31u) != 31u) continue;
        const int nib = (int)((wrow[k >> 3] >> (4 * (k & 7))) & 15u);
        const int wv = nib >= 8 ? nib - 16 : nib;
        if ((h & 1023u) != 0 || wv == 0) nan = true;
        else if ((wv < 0) != ((h & 0x8000u) != 0)) neg = true;
        else pos = true;
    }
    return nan || (pos && neg) ? 3 : pos ? 1 : neg ? 2 : 0;
}

// Lanes load 16 bytes of their row at any 4-byte alignment (K % 8 == 0 makes rows whole words; the
// hardware takes dword-aligned 16-byte loads).  A lane whose 4 words cross the row's end loads the
// row's last 4 words and shifts them down when they are used; lanes past the end multiply zero digits
// (the table is zero for k >= K), so what they load does not matter.  NARROW: rows of fewer than 4 words.
// XVEC: A is 16-byte aligned (one 16-byte load per 8 values); otherwise eight 2-byte loads.
//
// MULTI (K > 4096): two segments are in flight (the loads of segment s + 2 are issued once segment s is
// multiplied) and two digit tables leave one barrier per segment, which waits for LDS only.  Every load is issued
// unconditionally (clamped addresses) so the compiler's waits count exactly the loads in flight; the
// pointers are not __restrict__, or it would move the loads down to their use.
// RT: row tiles of 16 per workgroup.  Each digit-table B operand feeds RT + 1 MFMAs, so the A
// conversion (done once per workgroup and segment) is shared by 16 RT rows.
// PW: superchunks per wave that are loaded, at least those the longest segment gives a wave: 1 up to K = 1024,
// 2 up to 2048, 3 up to 3072.  A wave waits for all of its loads before it leaves, also for those that it does not multiply,
// and always loading kPerWave cost N = 24576, K = 512 9.7 us against 4.7 with one and two row tiles (7.8 before this loop).
typedef u4 u4_a4 __attribute__((aligned(4)));

template <bool NARROW, bool XVEC, int RT, bool MULTI, int PW>
__global__ void __launch_bounds__(kThreads)
gemv_kernel(const uint32_t* W, const uint16_t* A, const uint16_t* sW, const uint16_t* zW, uint16_t* C, int N, int K) {
    constexpr int ROWS = kRows * RT;
    constexpr int kTable = kSeg / kSuper * kSuperBytes;
    __shared__ __align__(16) uint8_t table[(MULTI ? 2 : 1) * kTable];
    __shared__ int32_t part[kWaves][ROWS][8];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int r = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * ROWS;
    const int kw = K >> 3;                                   // words per row
    const char* wbase = reinterpret_cast<const char*>(W + (size_t)row0 * kw);
    uint32_t woff[RT];                                       // bytes from wbase, below 32 * 2^19
#pragma unroll
    for (int t = 0; t < RT; ++t) woff[t] = (uint32_t)(min(row0 + kRows * t + r, N - 1) - row0) * (uint32_t)kw * 4u;
    i4v acc[RT], sums = {0, 0, 0, 0};
#pragma unroll
    for (int t = 0; t < RT; ++t) acc[t] = i4v{0, 0, 0, 0};
    int nonfinite = 0;

    // superchunks of segment `seg`, and this wave's share (a contiguous range starting at p0)
    auto shape = [&](int seg, int& nsc, int& per) {
        nsc = (min(kSeg, K - seg) + kSuper - 1) / kSuper;
        per = (nsc + kWaves - 1) / kWaves;
    };
    // Request the A values of this thread's 8-k unit and this wave's weights for segment `seg` (past
    // the end, MULTI: one cached address, unused).
    auto issue = [&](int seg, u4& xa, u4 (&wq)[RT][PW]) {
        const uint32_t live = !MULTI || seg < K ? 0xFFFFFFFFu : 0u;
        int nsc, per;
        shape(min(seg, K - 1), nsc, per);
        const int k0 = seg + 8 * tid;
        const uint16_t* src = A + (k0 < K ? k0 : 0);
        if constexpr (XVEC) {
            xa = *reinterpret_cast<const u4*>(src);
        } else {
            uint32_t d[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) d[e] = (uint32_t)src[2 * e] | ((uint32_t)src[2 * e + 1] << 16);
            xa = u4{d[0], d[1], d[2], d[3]};
        }
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const int p = wave * per + min(i, per - 1);      // past the share: repeat its last one
            const int wi = ((seg + p * kSuper) >> 3) + 4 * g;   // first word of the lane's 32 weights
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                if constexpr (NARROW) {
                    uint32_t d[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        d[e] = *reinterpret_cast<const uint32_t*>(wbase + woff[t] + 4u * (uint32_t)min(wi + e, kw - 1));
                    wq[t][i] = u4{d[0], d[1], d[2], d[3]};
                } else {
                    wq[t][i] = *reinterpret_cast<const u4_a4*>(wbase + ((woff[t] + 4u * (uint32_t)min(wi, kw - 4)) & live));
                }
            }
        }
        asm volatile("" ::: "memory");
    };
    // Digits of this thread's unit into a table (units past the segment's superchunks are
    // never read; units past K write zero digits).
    auto build = [&](int seg, const u4& xa, uint8_t* tab) {
        int nsc, per;
        shape(seg, nsc, per);
        const int u = tid;
        if (u >= nsc * (kSuper / 8)) return;
        const bool in = seg + 8 * u < K;
        uint32_t hw[4] = {in ? xa.x : 0u, in ? xa.y : 0u, in ? xa.z : 0u, in ? xa.w : 0u};
        // inf / NaN count as 0 here (their class is applied in the epilogue); rare, so one test
        // per 8 values and the zeroing behind a branch
        bool special = false;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const uint32_t ee = hw[q] & 0x7C007C00u;
            special |= (ee & 0xFFFFu) == 0x7C00u || (ee >> 16) == 0x7C00u;
        }
        if (special) {
            nonfinite = 1;
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t ee = hw[q] & 0x7C007C00u;
                hw[q] &= ((ee & 0xFFFFu) == 0x7C00u ? 0xFFFF0000u : 0xFFFFFFFFu) &
                         ((ee >> 16) == 0x7C00u ? 0x0000FFFFu : 0xFFFFFFFFu);
            }
        }
        uint32_t le[4], he[4], lo[4], ho[4];                 // k offsets 0, 2, 4, 6 and 1, 3, 5, 7
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            split_fixed((float)__builtin_bit_cast(_Float16, (uint16_t)(hw[i] & 0xFFFFu)), le[i], he[i]);
            split_fixed((float)__builtin_bit_cast(_Float16, (uint16_t)(hw[i] >> 16)), lo[i], ho[i]);
        }
        uint32_t de[kDigits], dd[kDigits];
        digit_dwords(le, he, de);
        digit_dwords(lo, ho, dd);
        const int p = u >> 4, rr = (u & 15) * 8;             // superchunk, k offset in it
        const int gg = rr >> 5, m = (rr >> 4) & 1, h = (rr >> 3) & 1;
        uint8_t* dst = tab + p * kSuperBytes + ((m * 4 + gg) * kDigits) * 16 + 8 * h;
#pragma unroll
        for (int j = 0; j < kDigits; ++j) *reinterpret_cast<uint2*>(dst + 16 * j) = uint2{de[j], dd[j]};
    };
    auto multiply = [&](int seg, const u4 (&wq)[RT][PW], const uint8_t* tab) {
        int nsc, per;
        shape(seg, nsc, per);
        const i4v ones = {0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const int p = wave * per + i;
            if (i >= per || p >= nsc) break;
            i4v b[2];
#pragma unroll
            for (int m = 0; m < 2; ++m) {
                // columns past the digits repeat the last one; nobody reads them
                b[m] = *reinterpret_cast<const i4v*>(tab + p * kSuperBytes + ((m * 4 + g) * kDigits + min(r, kDigits - 1)) * 16);
                sums = __builtin_amdgcn_mfma_i32_16x16x64_i8(ones, b[m], sums, 0, 0, 0);
            }
            const int wi = ((seg + p * kSuper) >> 3) + 4 * g;
            const bool crosses = !NARROW && ((seg + (p + 1) * kSuper) >> 3) > kw && (kw & 3) != 0;   // wave-uniform
#pragma unroll
            for (int t = 0; t < RT; ++t) {
                u4 w = wq[t][i];
                if (crosses) {
                    const int sh = wi - min(wi, kw - 4);     // 0..3, more where the lane is past the end
                    const bool one = sh & 1, two = sh & 2;
                    const u4 v = u4{one ? w.y : w.x, one ? w.z : w.y, one ? w.w : w.z, w.w};
                    w = u4{two ? v.z : v.x, two ? v.w : v.y, v.z, v.w};
                }
#pragma unroll
                for (int m = 0; m < 2; ++m) {
                    const uint32_t w0 = m ? w.z : w.x, w1 = m ? w.w : w.y;
                    const i4v a = {(int32_t)offset_nibbles(w0, 0), (int32_t)offset_nibbles(w0, 4),
                                   (int32_t)offset_nibbles(w1, 0), (int32_t)offset_nibbles(w1, 4)};
                    acc[t] = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b[m], acc[t], 0, 0, 0);
                }
            }
        }
    };

    u4 xa0, wq0[RT][PW];
    if constexpr (MULTI) {
        u4 xa1, wq1[RT][PW];
        issue(0, xa0, wq0);
        issue(kSeg, xa1, wq1);
        for (int seg = 0; seg < K; seg += 2 * kSeg) {
            build(seg, xa0, table);
            lds_barrier();                                   // also: every wave is done with the other table
            multiply(seg, wq0, table);
            issue(seg + 2 * kSeg, xa0, wq0);
            if (seg + kSeg < K) build(seg + kSeg, xa1, table + kTable);
            lds_barrier();
            if (seg + kSeg < K) multiply(seg + kSeg, wq1, table + kTable);
            issue(seg + 3 * kSeg, xa1, wq1);
        }
    } else if (K > 0) {
        issue(0, xa0, wq0);
        build(0, xa0, table);
        lds_barrier();
        multiply(0, wq0, table);
    }

    if (r < kDigits) {
#pragma unroll
        for (int t = 0; t < RT; ++t)
#pragma unroll
            for (int i = 0; i < 4; ++i) part[wave][kRows * t + 4 * g + i][r] = acc[t][i] - 8 * sums[i];
    }
    const bool any_nonfinite = __syncthreads_or(nonfinite);
    if (tid < ROWS && row0 + tid < N) {
        const int n = row0 + tid;
        int64_t total = 0;
#pragma unroll
        for (int j = 0; j < kDigits; ++j) {
            int32_t pj = 0;
#pragma unroll
            for (int w = 0; w < kWaves; ++w) pj += part[w][tid][j];
            total += (int64_t)pj << (8 * j);
        }
        float s = (float)total * 0x1p-24f;                   // the exact sum, rounded once
        if (any_nonfinite) {
            const int cls = nonfinite_class(W + (size_t)n * kw, A, K);
            if (cls == 3) s = __builtin_nanf("");
            else if (cls == 1) s = __builtin_inff();
            else if (cls == 2) s = -__builtin_inff();
        }
        // fp32 subtract and multiply, then fp16 rounding: two roundings, as the reference's
        // __float2half((acc - z) * s).  Left alone, the compiler folds the multiply and the
        // conversion into one v_fma_mixlo_f16, which rounds the exact product once (measured: one
        // fp16 ulp apart in 1 of 14336 outputs); the empty asm makes the fp32 product a value of
        // its own.
        const float z = (float)__builtin_bit_cast(_Float16, zW[n]);
        const float sc = (float)__builtin_bit_cast(_Float16, sW[n]);
        float prod = (s - z) * sc;
        asm volatile("" : "+v"(prod));
        C[n] = __builtin_bit_cast(uint16_t, (_Float16)prod);
    }
}

}  // namespace

}  // namespace w4a16

using namespace w4a16;

extern "C" int w4a16_gemv(const int32_t* W, const uint16_t* A, const uint16_t* sW, const uint16_t* zW,
                          uint16_t* C, int64_t N, int64_t K, void* stream) {
    if (N < 0 || K < 0 || N >= (int64_t)1 << 31) {
        w4a16_set_last_error("dimensions out of range");
        return W4A16_ERR_INVALID;
    }
    if (K % 8 != 0) {
        w4a16_set_last_error("K must be a multiple of 8");
        return W4A16_ERR_INVALID;
    }
    if (K > W4A16_GEMV_MAX_K) {
        w4a16_set_last_error("K must be at most 1048576 (exact int32 digit sums)");
        return W4A16_ERR_INVALID;
    }
    if (N == 0) return W4A16_OK;
    if (!sW || !zW || !C || (K > 0 && (!W || !A))) {             // W and A may be empty when K == 0
        w4a16_set_last_error("null pointer");
        return W4A16_ERR_INVALID;
    }
    if (reinterpret_cast<uintptr_t>(W) % 4 != 0 ||
        (reinterpret_cast<uintptr_t>(A) | reinterpret_cast<uintptr_t>(sW) | reinterpret_cast<uintptr_t>(zW) |
         reinterpret_cast<uintptr_t>(C)) % 2 != 0) {
        w4a16_set_last_error("W must be 4-byte aligned, A, sW, zW and C 2-byte aligned");
        return W4A16_ERR_INVALID;
    }
    hipStream_t st = reinterpret_cast<hipStream_t>(stream);
    // Row tiles per workgroup, measured as the time of two over that of one (weights from HBM):
    //  * K <= 1024: two once one tile each is more than a workgroup per CU; the digits of A and the launch are
    //    most of the call (N = 8192: 0.89-0.98, N = 9000..12288 0.97-1.02, N = 28672 0.77-0.82; N = 4096 1.01-1.04);
    //  * K <= 2048: two when that does not leave a CU a row tile more to do, or from six per CU (N = 7168, two
    //    per CU 0.94-0.99; N = 14336, four 0.96-0.98; N = 24576, six 0.84-0.93; N = 9000, three 1.04-1.05);
    //  * longer: one.  K <= 3072: N = 9000..12288 1.11-1.15, N = 14336, 16384 1.01-1.09, N = 28672 1.01-1.06, but
    //    N = 22016..24576 and 40960 0.92-1.01; K <= 4096: 1.13-1.17, 1.03-1.06, 1.05-1.10 and 0.96-1.05.
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) == hipSuccess) {
        w4a16_device_limits lim;
        if (w4a16_query_device(dev, &lim) == W4A16_OK && lim.cu_count > 0) cus = lim.cu_count;
    }
    const bool narrow = K < 32, multi = K > kSeg;
    const int64_t per_cu = ((N + kRows - 1) / kRows + cus - 1) / cus;
    const bool two = !narrow && K <= kSeg / 2 && per_cu > 1 && (K <= kSeg / 4 || per_cu % 2 == 0 || per_cu > 5);
    const int rt = two ? 2 : 1;
    const dim3 grid((unsigned)((N + rt * kRows - 1) / (rt * kRows)));
    const bool xvec = reinterpret_cast<uintptr_t>(A) % 16 == 0;
    auto pick = [&](auto nx_c, auto rt_c, auto multi_c, auto pw_c) {
        constexpr bool X = decltype(nx_c)::value, L = decltype(multi_c)::value;
        constexpr int R = decltype(rt_c)::value, P = decltype(pw_c)::value;
        return xvec ? gemv_kernel<X, true, R, L, P> : gemv_kernel<X, false, R, L, P>;
    };
    constexpr std::integral_constant<int, 1> c1;
    constexpr std::integral_constant<int, 2> c2;
    constexpr std::integral_constant<int, 3> c3;
    constexpr std::integral_constant<int, kPerWave> c4;
    constexpr std::false_type no;
    constexpr std::true_type yes;
    auto kernel = narrow              ? pick(yes, c1, no, c1)
                  : K <= kSeg / 4     ? (two ? pick(no, c2, no, c1) : pick(no, c1, no, c1))
                  : K <= kSeg / 2     ? (two ? pick(no, c2, no, c2) : pick(no, c1, no, c2))
                  : K <= 3 * kSeg / 4 ? pick(no, c1, no, c3)
                  : multi             ? pick(no, c1, yes, c4)
                                      : pick(no, c1, no, c4);
    hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, reinterpret_cast<const uint32_t*>(W), A, sW, zW, C, (int)N,
                       (int)K);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        w4a16_set_last_error(hipGetErrorString(e));
        return W4A16_ERR_HIP;
    }
    return W4A16_OK;
}
