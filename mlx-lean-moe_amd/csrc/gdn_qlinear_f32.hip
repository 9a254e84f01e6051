// Affine-quantized projections of float32 activations at prompt sizes
// (gdn_quantized_matmul_f32): y = x W^T for float32 x (M, K) and MLX-packed
// 4- or 8-bit codes, in float32 accuracy on the bf16 matrix cores.
//
// Both factors are taken exactly. A code less an integer c of [0, 255] is a
// bf16 value; a float32 x is the sum of three bf16 values (its 24
// significant bits cut into three 8-bit pieces). So with
//   P[m][n] = sum over one quantization group's k of x[m][k] (q[n][k] - c)
// (three MFMAs a fragment pair, float32 sums of exact products), X[m][g] the
// group's sum of x and b' = b + c s,
//   y[m][n] = sum over groups of s[n][g] P + b'[n][g] X[m][g]:
// no weight is rounded and no product is, which leaves the float32 sums
// (777 rows of 2048 normal values against 12352 columns of 4-bit codes in
// groups of 64: 1.2e-7 from float64, where the float32 library product of
// rounded weights is 8.1e-7 off and takes 345 us to this one's 125-129).
// c is the group's own: the integer nearest to -b / s, the code of the weight
// nearest to zero, so that |b'| <= |s| / 2 and the two terms of a weight w are
// at most 3 |w| together (0 for w = 0; with one c for all, an x thousands of
// times the rest left the rounding of c s x where its weight is 0). Where -b /
// s lies outside [0, 255], c is the nearer end and the terms have one sign.
//
// Two launches (three where K is split): the preparation cuts x, sums its
// groups and lays s and b' out group-major; the product kernel does the rest.
#include "gdn_common.h"
#include "gdn_host.h"
#include "gdn_qlinear.h"

namespace gdn {
namespace {

constexpr int kBK = 64;             // k per step
constexpr int kParts = 3;           // bf16 pieces of a float32
constexpr int kPK = kParts * kBK;   // a row's pieces of one step
constexpr int kXS = kPK + 8;        // row stride of the LDS tile, bf16: 16 rows cover the banks
constexpr int kTN = 4;              // 16-column tiles of a wave
constexpr int kBN = 4 * 16 * kTN;   // columns of a workgroup (4 waves)
constexpr int kMaxTM = 5;           // 16-row tiles of a workgroup, at most (6 spill)
constexpr int kCUs = 256;

GDN_DEV f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// ---------------------------------------------------------------------------
// preparation
// ---------------------------------------------------------------------------

// Rows whose pieces would not be exact (a non-finite x, a row of magnitudes
// whose last piece leaves bf16's range), and rows and columns whose partial
// sums could overflow where the products with the weights do not, are
// multiplied apart (float_rows; flags of rows and of 64 columns). Inside the
// limits no partial sum over K <= 2^20 of a scaled P (|q - c| <= 2^8: 2^20 2^16
// 2^8 2^80) or of b' X (|b'| <= 2^24 + 2^8 2^16 = 2^25: 2^20 2^25 2^80), nor
// their sum, reaches 2^127.
constexpr float kRowMax = 0x1p80f, kRowMin = 0x1p-90f;
constexpr float kScaleMax = 0x1p16f, kBiasMax = 0x1p24f;
constexpr int kFlagCols = 64;
constexpr int kFlagGroups = 32;  // quantization groups of a column flag
__host__ __device__ constexpr int flag_chunks(int groups) { return (groups + kFlagGroups - 1) / kFlagGroups; }
__host__ __device__ constexpr int64_t padded_columns(int64_t n) { return (n + kBN - 1) / kBN * kBN; }

// Blocks 0 .. M - 1: row m of x as bf16 pieces, pieces[m][step][part][64]
// (part 0 the upper 8 significant bits; truncation, so no piece can round up
// to infinity), its group sums (in double, rounded once) and its flag.
// The blocks after them, 64 columns by 32 groups each, a thread 8 consecutive
// ones of a column with all its loads in flight (a thread walking all of its
// column's groups took 18 us for 128 rows and 1024 columns of 128 groups, this
// 8): s, b (o_t) and b' = b + c s in float32, group-major, c as a byte
// (c_t[group][64-column block][n % 16][n / 16 % 4]: a word for the four columns
// of a lane of the product) and the flag (at flags[M + column block * chunks +
// chunk]). The rows of s, b and c have padded_columns(N) columns; those past N
// are read for outputs that are not stored.
template <class SB>
__global__ __launch_bounds__(256) void prepare_f32_kernel(
    const float* __restrict__ x, const typename SB::storage* __restrict__ scales,
    const typename SB::storage* __restrict__ biases, uint16_t* __restrict__ pieces, float* __restrict__ xsum,
    int* __restrict__ flags, float* __restrict__ s_t, float* __restrict__ b_t, float* __restrict__ o_t,
    uint8_t* __restrict__ c_t, int M, int N, int K, int group_size) {
    const int G = K / group_size;
    if (int(blockIdx.x) >= M) {
        constexpr int kPer = kFlagGroups / 4;  // groups of a thread
        const int at = int(blockIdx.x) - M, block = at / flag_chunks(G), lane = threadIdx.x & 63;
        const int g0 = at % flag_chunks(G) * kFlagGroups + int(threadIdx.x >> 6) * kPer;
        const int64_t stride = padded_columns(N), n = int64_t(block) * kFlagCols + lane;
        const int64_t row = (n < N ? n : N - 1) * G;
        float s[kPer], b[kPer];
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int g = g0 + i < G ? g0 + i : G - 1;
            s[i] = SB::load(scales, row + g);
            b[i] = SB::load(biases, row + g);
        }
        bool far = false;
#pragma unroll
        for (int i = 0; i < kPer; ++i) {
            const int64_t g = g0 + i;
            if (n >= N || g >= G) continue;
            far |= !(fabsf(s[i]) < kScaleMax && fabsf(b[i]) < kBiasMax);
            const float c = fminf(fmaxf(rintf(-b[i] / s[i]), 0.f), 255.f);  // s = 0: any, b' = b
            s_t[g * stride + n] = s[i];
            o_t[g * stride + n] = b[i];
            c_t[g * stride + block * kFlagCols + (lane % 16) * 4 + lane / 16] = uint8_t(c);
            b_t[g * N + n] = __builtin_fmaf(c, s[i], b[i]);
        }
        far = __syncthreads_or(far);
        if (threadIdx.x == 0) flags[blockIdx.x] = far;
        return;
    }
    const int64_t m = blockIdx.x;
    const int chunks = K / 8, lanes = group_size / 8;  // 8-element chunks; chunks of a group
    bool odd = false;
    float top = 0.f;
    for (int c0 = 0; c0 < chunks; c0 += 256) {
        const int c = c0 + int(threadIdx.x);
        double sum = 0.0;
        if (c < chunks) {
            const float4 lo4 = *reinterpret_cast<const float4*>(x + m * K + 8 * c);
            const float4 hi4 = *reinterpret_cast<const float4*>(x + m * K + 8 * c + 4);
            const float v[8] = {lo4.x, lo4.y, lo4.z, lo4.w, hi4.x, hi4.y, hi4.z, hi4.w};
            uint32_t part[kParts][4];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                odd |= !(fabsf(v[j]) < kRowMax);
                top = fmaxf(top, fabsf(v[j]));
                sum += double(v[j]);
                const float h = __uint_as_float(__float_as_uint(v[j]) & 0xFFFF0000u);
                const float r = v[j] - h;  // exact
                const float mid = __uint_as_float(__float_as_uint(r) & 0xFFFF0000u);
                const uint32_t bits[kParts] = {__float_as_uint(h), __float_as_uint(mid), __float_as_uint(r - mid)};
#pragma unroll
                for (int p = 0; p < kParts; ++p)
                    part[p][j / 2] = j & 1 ? (part[p][j / 2] | (bits[p] & 0xFFFF0000u)) : bits[p] >> 16;
            }
            uint16_t* dst = pieces + (m * K + (c / 8) * kBK) * kParts + 8 * (c % 8);
#pragma unroll
            for (int p = 0; p < kParts; ++p)
                *reinterpret_cast<uint4*>(dst + kBK * p) = make_uint4(part[p][0], part[p][1], part[p][2], part[p][3]);
        }
        // a group's 4, 8 or 16 chunks lie in consecutive lanes (K is a
        // multiple of the group, so a group never ends inside `chunks`)
        for (int d = 1; d < lanes; d *= 2) sum += __shfl_xor(sum, d);
        if (c < chunks && c % lanes == 0) xsum[m * G + c / lanes] = float(sum);
    }
    odd |= __syncthreads_or(odd);
    const bool small = top < kRowMin, zero = top == 0.f;
    const bool all_small = !__syncthreads_or(!small), all_zero = !__syncthreads_or(!zero);
    if (threadIdx.x == 0) flags[m] = odd || (all_small && !all_zero);
}

// ---------------------------------------------------------------------------
// product
// ---------------------------------------------------------------------------

// 8 codes less c as bf16 (exact: the float's upper half). A masked 4-bit code
// in a byte is the e4m3 value q 2^-9, so one conversion gives two.
template <int kBits>
GDN_DEV bf16x8 centred_fragment(const uint32_t* words, float c) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    u32x4 d;
    float f[8];
    if constexpr (kBits == 4) {
        const uint32_t half[2] = {words[0] & 0x0F0F0F0Fu, (words[0] >> 4) & 0x0F0F0F0Fu};  // codes 0 2 4 6, 1 3 5 7
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const auto lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(half[i], 512.f, false);
            const auto hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(half[i], 512.f, true);
            f[i] = lo[0] - c;
            f[2 + i] = lo[1] - c;
            f[4 + i] = hi[0] - c;
            f[6 + i] = hi[1] - c;
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) f[j] = float((words[j / 4] >> (8 * (j % 4))) & 255u) - c;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i)
        d[i] = __builtin_amdgcn_perm(__float_as_uint(f[2 * i + 1]), __float_as_uint(f[2 * i]), 0x07060302u);
    return __builtin_bit_cast(bf16x8, d);
}

// The workgroup's rows of x (past M - 1 repeating it) by a wave's 64 columns
// from n0 over the k range [k0, k1), from the float32 weights s q + b on the
// float32 matrix cores: what the pieces and group sums cannot carry
// (infinities, NaN, the ends of the range). Lane (lr, lq) holds row or column
// lr and k 4 lq .. of each 16, the next 16's operands in registers meanwhile.
// All of 777 rows flagged, 2048 -> 12352, take 612 us, one row 383, ordinary
// rows 130 (a thread a column and a serial chain a row took 234 ms and 950 us).
template <int kBits, int kTM>
GDN_DEV void float_rows(const float* __restrict__ x, const uint32_t* __restrict__ w, const float* __restrict__ s_t,
                        const float* __restrict__ o_t, int m0, int n0, int M, int N, int K, int group_size, int k0,
                        int k1, int lr, int lq, f32x4 (&v)[kTM][kTN]) {
    constexpr int kPer = 32 / kBits;
    const int64_t stride = padded_columns(N);
    const float* xr[kTM];
    const uint32_t* wr[kTN];
#pragma unroll
    for (int a = 0; a < kTM; ++a) {
        const int64_t m = m0 + 16 * a + lr;
        xr[a] = x + (m < M ? m : M - 1) * K + 4 * lq;
#pragma unroll
        for (int b = 0; b < kTN; ++b) v[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
#pragma unroll
    for (int b = 0; b < kTN; ++b) {
        const int64_t n = n0 + 16 * b + lr;
        wr[b] = w + (n < N ? n : N - 1) * (K / kPer);
    }
    struct Operands {
        f32x4 x[kTM];
        uint32_t wd[kTN];
        float s[kTN], o[kTN];
    };
    const auto fetch = [&](int k) {
        Operands p;
        const int kl = k + 4 * lq;
        const int64_t at = kl / group_size * stride + n0 + lr;
#pragma unroll
        for (int a = 0; a < kTM; ++a) p.x[a] = *reinterpret_cast<const f32x4*>(xr[a] + k);
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            p.wd[b] = wr[b][kl / kPer];
            p.s[b] = s_t[at + 16 * b];
            p.o[b] = o_t[at + 16 * b];
        }
        return p;
    };
    Operands p = fetch(k0);
#pragma unroll 1
    for (int k = k0; k < k1; k += 16) {
        const Operands next = fetch(k + 16 < k1 ? k + 16 : k);
        f32x4 wf[kTN];
#pragma unroll
        for (int b = 0; b < kTN; ++b)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t q = p.wd[b] >> (kBits * ((4 * lq) % kPer) + kBits * j) & ((1u << kBits) - 1u);
                wf[b][j] = __builtin_fmaf(p.s[b], float(q), p.o[b]);
            }
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int a = 0; a < kTM; ++a)
#pragma unroll
                for (int b = 0; b < kTN; ++b)
                    v[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(p.x[a][j], wf[b][j], v[a][b], 0, 0, 0);
        p = next;
    }
}

// A workgroup holds 16 kTM rows by 256 columns, each of its 4 waves all the
// rows by 64 columns, so a piece of x read from LDS serves four MFMAs and the
// codes go from memory to the wave's own B fragments, converted once per
// workgroup. A step is 64 k: x's pieces through two LDS tiles (one barrier a
// step), the next step's pieces, codes and scales in registers meanwhile. Two
// workgroups share a CU (256 registers a thread). At 777 rows, 2048 -> 12352,
// the matrix cores are busy half the time (118 GFLOP of bf16 products against
// 2.1 PFLOP/s: 56 us of 125): with two waves on a SIMD a wave's LDS reads,
// conversions and scaling are not all covered. A wave in its MFMAs goes before
// one that loads or converts (131 us without). Fetching the codes two steps
// ahead, or the next row tile's fragments, spilled or gained nothing. One c for
// all groups (no c_t, a shift in place of the fp8 conversion and subtraction)
// takes the same time at this size, 8-bit K = 4096 153 us to 157.
//
// kG32: groups of 32 (an MFMA's k), each scaled by itself; else one group (64
// or half of 128) a step. Lane quarter q = l / 16 holds k 8 q .. of each
// 32-block, or 16 q .. of the step (one 8-byte load of 4-bit codes).
//
// Split K: blockIdx.y = j takes steps [j steps / S, (j + 1) steps / S) and
// stores its float32 block at out + j M N, to be added in order afterwards.
template <int kBits, int kTM, bool kG32>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) void qlinear_f32_kernel(
    const uint16_t* __restrict__ pieces, const float* __restrict__ xsum, const int* __restrict__ flags,
    const float* __restrict__ s_t, const float* __restrict__ b_t, const float* __restrict__ o_t,
    const uint32_t* __restrict__ c_t, const float* __restrict__ x, const uint32_t* __restrict__ w, float* out,
    const float* residual, int M, int N, int K, int group_size, int mt, int tiles) {
    constexpr int kBM = 16 * kTM;
    constexpr int kPiecesPerRow = kPK / 8;
    constexpr int kXLoads = (kBM * kPiecesPerRow + 255) / 256;
    constexpr int kWords = 2 * kBits / 4;  // packed words of a lane's 16 codes of a step
    __shared__ __attribute__((aligned(16))) uint16_t xs[2][kBM * kXS];

    // Tiles in row-major order within a column block, an eighth of them to
    // each XCD (workgroups go round-robin over the XCDs): a column block's
    // codes are read into one XCD's L2.
    const int per_xcd = (tiles + 7) / 8;
    const int t = int(blockIdx.x % 8) * per_xcd + int(blockIdx.x / 8);
    if (t >= tiles || int(blockIdx.x / 8) >= per_xcd) return;
    const int m0 = (t % mt) * kBM, n0 = (t / mt) * kBN;
    const int tid = threadIdx.x, l = tid & 63, lr = l & 15, lq = l >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int steps = K / kBK / int(gridDim.y), step0 = steps * int(blockIdx.y);
    const int g0 = step0 * kBK / group_size, g1 = (step0 + steps) * kBK / group_size;

    int col[kTN];
#pragma unroll
    for (int b = 0; b < kTN; ++b) {
        const int n = n0 + 16 * kTN * wv + 16 * b + lr;
        col[b] = n < N ? n : N - 1;  // clamped columns are not stored
    }

    // x: rows clamped to M - 1 (not stored); pieces past the tile repeat its last
    const uint16_t* xtile = pieces + int64_t(m0) * K * kParts;
    uint32_t xo[kXLoads];  // byte offsets from a uniform base, as below: no address arithmetic in the loop
    int xl[kXLoads];
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) {
        int idx = tid + 256 * i;
        idx = idx < kBM * kPiecesPerRow ? idx : kBM * kPiecesPerRow - 1;
        const int row = idx / kPiecesPerRow, seg = idx % kPiecesPerRow;
        const int r = m0 + row < M ? row : M - 1 - m0;
        xo[i] = (uint32_t(r) * uint32_t(K * kParts) + 8 * seg) * 2;
        xl[i] = row * kXS + 8 * seg;
    }
    u16x8 xr[kXLoads];
    auto fetch_x = [&](int s) {
        const char* src = reinterpret_cast<const char*>(xtile + int64_t(s) * kPK);
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) xr[i] = *reinterpret_cast<const u16x8*>(src + xo[i]);
    };
    auto stage_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) *reinterpret_cast<u16x8*>(xs[buf] + xl[i]) = xr[i];
    };

    const int64_t wpr = int64_t(K) * kBits / 32;
    uint32_t wo[kTN];
#pragma unroll
    for (int b = 0; b < kTN; ++b) {
        wo[b] = (uint32_t(col[b] - n0) * uint32_t(wpr) + lq * (kG32 ? kWords / 2 : kWords)) * 4;
    }
    static_assert(kFlagCols == 16 * kTN, "a wave's columns share a flag and a word of c");
    const int blocks = (N + kFlagCols - 1) / kFlagCols, wblock = n0 / kFlagCols + wv;
    const int64_t sstride = padded_columns(N);
    // a step's codes (words of MFMA block kb at [b][kb kWords / 2 ..]), scales and c
    struct Codes {
        uint32_t wd[kTN][kWords];
        float sc[kTN][kG32 ? 2 : 1];
        uint32_t centre[kG32 ? 2 : 1];  // a byte a column
    };
    Codes c;
    auto fetch_w = [&](int s) {
        const char* wtile = reinterpret_cast<const char*>(w + n0 * wpr + s * kBK * kBits / 32);
        const int g = s * kBK / group_size;
#pragma unroll
        for (int i = 0; i < (kG32 ? 2 : 1); ++i) c.centre[i] = (c_t + ((g + i) * sstride + n0) / 4 + 16 * wv)[lr];
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const uint32_t* src = reinterpret_cast<const uint32_t*>(wtile + wo[b]);
#pragma unroll
            for (int i = 0; i < kWords; ++i) c.wd[b][i] = src[kG32 ? i / (kWords / 2) * kBits + i % (kWords / 2) : i];
#pragma unroll
            for (int i = 0; i < (kG32 ? 2 : 1); ++i)
                c.sc[b][i] = (s_t + (g + i) * sstride + n0 + 16 * kTN * wv)[lr + 16 * b];
        }
    };

    const int last = step0 + steps - 1;
    fetch_x(step0);
    fetch_w(step0);

    // the bias terms first: X times b' over the range's groups, in float32
    // MFMAs of four groups (lanes past the last group carry zeros)
    f32x4 acc[kTM][kTN];
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int G = K / group_size;
    for (int g = g0; g < g1; g += 4) {
        const bool in = g + lq < g1;
        const int gl = in ? g + lq : g1 - 1;
        float xa[kTM], bb[kTN];
#pragma unroll
        for (int a = 0; a < kTM; ++a) {
            const int m = m0 + 16 * a + lr;
            xa[a] = xsum[int64_t(m < M ? m : M - 1) * G + gl];
        }
#pragma unroll
        for (int b = 0; b < kTN; ++b) bb[b] = b_t[int64_t(gl) * N + col[b]];
#pragma unroll
        for (int a = 0; a < kTM; ++a)
#pragma unroll
            for (int b = 0; b < kTN; ++b)
                acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(in ? xa[a] : 0.f, in ? bb[b] : 0.f, acc[a][b], 0, 0, 0);
    }

    stage_x(0);
    for (int s = step0; s <= last; ++s) {
        bf16x8 bf[kTN][2];
        float scale[kTN][kG32 ? 2 : 1];
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
#pragma unroll
            for (int kb = 0; kb < 2; ++kb)
                bf[b][kb] = centred_fragment<kBits>(&c.wd[b][kb * kWords / 2], float((c.centre[kG32 ? kb : 0] >> (8 * b)) & 255u));
#pragma unroll
            for (int i = 0; i < (kG32 ? 2 : 1); ++i) scale[b][i] = c.sc[b][i];
        }
        __builtin_amdgcn_sched_barrier(0);  // the codes' registers first: fetches hoisted above them spill
        const int next = s < last ? s + 1 : last;  // the last step again, unused
        fetch_x(next);
        fetch_w(next);
        __builtin_amdgcn_sched_barrier(0);
        __syncthreads();
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int a = 0; a < kTM; ++a) {
            const uint16_t* xrow = xs[(s - step0) & 1] + (16 * a + lr) * kXS;
            bf16x8 af[kParts][2];
#pragma unroll
            for (int p = 0; p < kParts; ++p)
#pragma unroll
                for (int kb = 0; kb < 2; ++kb)
                    af[p][kb] = *reinterpret_cast<const bf16x8*>(xrow + kBK * p + (kG32 ? 32 * kb + 8 * lq : 16 * lq + 8 * kb));
            f32x4 part[kTN];
            auto scaled = [&](int i) {
#pragma unroll
                for (int b = 0; b < kTN; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) acc[a][b][e] = __builtin_fmaf(scale[b][i], part[b][e], acc[a][b][e]);
            };
#pragma unroll
            for (int kb = 0; kb < 2; ++kb) {
                if (kG32 || kb == 0) {
#pragma unroll
                    for (int b = 0; b < kTN; ++b) part[b] = f32x4{0.f, 0.f, 0.f, 0.f};
                }
#pragma unroll
                for (int p = kParts - 1; p >= 0; --p)  // the small pieces first
#pragma unroll
                    for (int b = 0; b < kTN; ++b) part[b] = mfma_bf16(af[p][kb], bf[b][kb], part[b]);
                if constexpr (kG32) scaled(kb);
            }
            if constexpr (!kG32) scaled(0);
        }
        __builtin_amdgcn_s_setprio(0);
        stage_x((s - step0 + 1) & 1);
    }

    // flagged rows, and the wave's own 64 columns when flagged, are left to
    // float_rows below
    const int col0 = n0 / kFlagCols, chunks = flag_chunks(G);
    int any = 0;
    if (tid < kBM) any = flags[m0 + tid < M ? m0 + tid : M - 1];
    for (int i = tid; i < kBN / kFlagCols * chunks && col0 + i / chunks < blocks; i += 256)
        any |= flags[M + col0 * chunks + i];
    any = __syncthreads_or(any);
    int far = 0;
    if (any && wblock < blocks)
        for (int i = 0; i < chunks; ++i) far |= flags[M + wblock * chunks + i];
    float* dst = out + int64_t(blockIdx.y) * M * N;
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + 16 * a + 4 * lq + i;
            if (m >= M || far || (any && flags[m])) continue;
#pragma unroll
            for (int b = 0; b < kTN; ++b) {
                const int n = n0 + 16 * kTN * wv + 16 * b + lr;
                if (n >= N) continue;
                const int64_t e = int64_t(m) * N + n;
                dst[e] = acc[a][b][i] + (residual ? residual[e] : 0.f);
            }
        }
    if (!any || wblock >= blocks) return;
    float_rows<kBits, kTM>(x, w, s_t, o_t, m0, n0 + 16 * kTN * wv, M, N, K, group_size, step0 * kBK, (last + 1) * kBK,
                           lr, lq, acc);
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int m = m0 + 16 * a + 4 * lq + i;
            if (m >= M || !(far || flags[m])) continue;
#pragma unroll
            for (int b = 0; b < kTN; ++b) {
                const int n = n0 + 16 * kTN * wv + 16 * b + lr;
                if (n >= N) continue;
                const int64_t e = int64_t(m) * N + n;
                dst[e] = acc[a][b][i] + (residual ? residual[e] : 0.f);
            }
        }
}

// ---------------------------------------------------------------------------
// launch
// ---------------------------------------------------------------------------

struct F32Plan {
    int tm, splits;
    int64_t pieces, xsum, flags, s_t, b_t, o_t, c_t, partial, bytes;  // workspace offsets
};

// Rows of a workgroup and splits of K: the least time by the matrix cores'
// share of the fullest CU, ceil(workgroups / 256) steps (fixed + per row tile)
// (0.1 and 0.2 us as measured), and a split's partial blocks written and read.
F32Plan plan_f32(int M, int N, int K, int group_size) {
    F32Plan p{};
    double best = 1e30;
    const int64_t nt = (N + kBN - 1) / kBN;
    for (int tm = 2; tm <= kMaxTM; ++tm)
        for (int s = 1; s <= 16; s *= 2) {
            if (K % (kBK * s) || K / s % group_size) break;
            const int64_t wgs = (int64_t(M) + 16 * tm - 1) / (16 * tm) * nt * s;
            const double us = double((wgs + kCUs - 1) / kCUs) * (K / kBK / s) * (0.1 + 0.2 * tm) +
                              (s > 1 ? 3.0 + double(s) * M * N * 8 / 4e6 : 0.0);
            if (us < best) {
                best = us;
                p.tm = tm;
                p.splits = s;
            }
        }
    const auto up = [](int64_t b) { return (b + 255) & ~int64_t(255); };
    const int64_t G = K / group_size;
    p.xsum = up(int64_t(M) * K * kParts * 2);
    p.flags = p.xsum + up(M * G * 4);
    p.s_t = p.flags + up((int64_t(M) + int64_t(N + kFlagCols - 1) / kFlagCols * flag_chunks(int(G))) * 4);
    p.b_t = p.s_t + up(padded_columns(N) * G * 4);
    p.o_t = p.b_t + up(N * G * 4);
    p.c_t = p.o_t + up(padded_columns(N) * G * 4);
    p.partial = p.c_t + up(padded_columns(N) * G);
    p.bytes = p.partial + (p.splits > 1 ? int64_t(p.splits) * M * N * 4 : 0);
    return p;
}

template <int kBits, bool kG32>
auto kernel_of(int tm) {
    switch (tm) {
        case 2: return qlinear_f32_kernel<kBits, 2, kG32>;
        case 3: return qlinear_f32_kernel<kBits, 3, kG32>;
        case 4: return qlinear_f32_kernel<kBits, 4, kG32>;
        default: return qlinear_f32_kernel<kBits, 5, kG32>;
    }
}

bool f32_sizes_ok(int64_t M, int64_t N, int64_t K, int group_size) {
    // 32-bit lane offsets; grids of less than 2^32 threads (256 a block): the
    // preparation's rows and column blocks, the product's smallest tiles
    constexpr int64_t kBlocks = 1 << 24;
    return (group_size == 32 || group_size == 64 || group_size == 128) && K % kBK == 0 && K % group_size == 0 &&
           M <= kBlocks && N <= kBlocks && K <= (1 << 20) &&
           M + (N + kFlagCols - 1) / kFlagCols * flag_chunks(int(K) / group_size) < kBlocks &&
           ((M + 31) / 32) * ((N + kBN - 1) / kBN) < kBlocks - 8;
}

}  // namespace
}  // namespace gdn

using namespace gdn;

extern "C" int64_t gdn_quantized_matmul_f32_workspace_size(int M, int N, int K, int bits, int group_size) {
    if (M < 1 || N < 1 || K < 1 || (bits != 4 && bits != 8) || !f32_sizes_ok(M, N, K, group_size)) return 0;
    return plan_f32(M, N, K, group_size).bytes;
}

extern "C" int gdn_quantized_matmul_f32(const float* x, const void* w, const void* scales, const void* biases,
                                        int sb_dtype, float* y, const float* residual, int M, int N, int K, int bits,
                                        int group_size, void* workspace, int64_t workspace_bytes, void* stream) {
    const char* fn = "gdn_quantized_matmul_f32";
    GDN_REQUIRE(M >= 0 && N > 0 && K > 0, "%s: bad sizes M=%d N=%d K=%d", fn, M, N, K);
    GDN_REQUIRE(w && scales && biases, "%s: null weight, scales or biases", fn);
    GDN_REQUIRE(valid_dtype(sb_dtype), "%s: bad scales/biases dtype", fn);
    if (bits != 4 && bits != 8) return fail(GDN_EUNSUPPORTED, "%s: %d-bit weights (4 and 8 are implemented)", fn, bits);
    GDN_REQUIRE(f32_sizes_ok(M, N, K, group_size),
                "%s: group_size must be 32, 64 or 128, K=%d a multiple of 64 and of it, and M=%d N=%d fit the grid", fn,
                K, M, N);
    if (M == 0) return 0;
    GDN_REQUIRE(x && y, "%s: null x or y", fn);
    GDN_REQUIRE((reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(w) |
                 reinterpret_cast<uintptr_t>(workspace)) % 16 == 0,
                "%s: x, weight and workspace must be 16-byte aligned", fn);
    const int64_t xb = int64_t(M) * K * 4, yb = int64_t(M) * N * 4;
    GDN_REQUIRE(!overlaps(x, xb, y, yb), "%s: y overlaps x", fn);
    GDN_REQUIRE(!residual || residual == y || !overlaps(residual, yb, y, yb), "%s: residual partially overlaps y", fn);
    const F32Plan p = plan_f32(M, N, K, group_size);
    GDN_REQUIRE(workspace && workspace_bytes >= p.bytes, "%s: workspace of %lld bytes, need %lld", fn,
                (long long)workspace_bytes, (long long)p.bytes);

    hipStream_t s = as_stream(stream);
    char* ws = static_cast<char*>(workspace);
    auto* pieces = reinterpret_cast<uint16_t*>(ws);
    auto* xsum = reinterpret_cast<float*>(ws + p.xsum);
    auto* flags = reinterpret_cast<int*>(ws + p.flags);
    auto* s_t = reinterpret_cast<float*>(ws + p.s_t);
    auto* b_t = reinterpret_cast<float*>(ws + p.b_t);
    auto* o_t = reinterpret_cast<float*>(ws + p.o_t);
    auto* c_t = reinterpret_cast<uint8_t*>(ws + p.c_t);
    auto* partial = reinterpret_cast<float*>(ws + p.partial);
    const int64_t sb_blocks = (int64_t(N) + kFlagCols - 1) / kFlagCols * flag_chunks(K / group_size);
    const auto prepare = [&](auto sb) {
        using SB = decltype(sb);
        using St = typename SB::storage;
        hipLaunchKernelGGL(prepare_f32_kernel<SB>, dim3(unsigned(M + sb_blocks)), dim3(256), 0, s, x,
                           static_cast<const St*>(scales), static_cast<const St*>(biases), pieces, xsum, flags, s_t,
                           b_t, o_t, c_t, M, N, K, group_size);
    };
    if (sb_dtype == GDN_F32) prepare(ActF32{});
    else if (sb_dtype == GDN_BF16) prepare(ActBF16{});
    else prepare(ActF16{});
    if (int rc = check_launch("gdn_quantized_matmul_f32/prepare")) return rc;

    const int mt = (M + 16 * p.tm - 1) / (16 * p.tm), tiles = mt * ((N + kBN - 1) / kBN);
    const auto kernel = bits == 4 ? (group_size == 32 ? kernel_of<4, true>(p.tm) : kernel_of<4, false>(p.tm))
                                  : (group_size == 32 ? kernel_of<8, true>(p.tm) : kernel_of<8, false>(p.tm));
    hipLaunchKernelGGL(kernel, dim3(unsigned((tiles + 7) / 8 * 8), unsigned(p.splits)), dim3(256), 0, s, pieces, xsum,
                       flags, s_t, b_t, o_t, reinterpret_cast<const uint32_t*>(c_t), x,
                       static_cast<const uint32_t*>(w), p.splits > 1 ? partial : y, p.splits > 1 ? nullptr : residual,
                       M, N, K, group_size, mt, tiles);
    if (int rc = check_launch(fn)) return rc;
    if (p.splits > 1)
        return launch_split_sum(partial, p.splits, int64_t(M) * N, y, GDN_F32, residual, s, "gdn_quantized_matmul_f32/sum");
    return 0;
}
