// Affine-quantized projections of bf16 rows above the decode sizes
// (gdn_quantized_matmul with M > 64): the weights enter the MFMAs as
// bf16(scale q + bias), one rounding, as the tiled kernel of gdn_qlinear.hip
// takes them.
#include <type_traits>

#include "gdn_common.h"
#include "gdn_host.h"
#include "gdn_qlinear.h"

namespace gdn {
namespace {

constexpr int kTN = 4;               // 16-column tiles of a wave
constexpr int kNW = 2;               // waves side by side in N
constexpr int kKW = 4;               // waves sharing a step's k
constexpr int kBN = 16 * kTN * kNW;  // columns of a workgroup
constexpr int kSlice = 64;           // a wave's k of a step
constexpr int kStep = kSlice * kKW;  // k of a step
constexpr int kXS = kStep + 8;       // row stride of the x tile: 16 rows cover the banks
constexpr int kMaxTM = 7;
constexpr int kMaxRows = 511;
// Bytes of scales and biases the LDS holds (of a workgroup's columns over its k range)
constexpr int kSBBytes = 32 * 1024;
constexpr int kCUs = 256;

GDN_DEV f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// 8 weights of one group as bf16. A masked 4-bit code in a byte is the e4m3
// value q 2^-9 (the subnormals and the first binade share their spacing), so
// one conversion gives two codes' floats.
template <int kBits>
GDN_DEV bf16x8 weight_fragment(const uint32_t* words, float s, float b) {
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
    float q[8];
    if constexpr (kBits == 4) {
        const uint32_t half[2] = {words[0] & 0x0F0F0F0Fu, (words[0] >> 4) & 0x0F0F0F0Fu};  // codes 0 2 4 6, 1 3 5 7
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const auto lo = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(half[i], 512.f, false);
            const auto hi = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(half[i], 512.f, true);
            q[i] = lo[0];
            q[2 + i] = lo[1];
            q[4 + i] = hi[0];
            q[6 + i] = hi[1];
        }
    } else {
#pragma unroll
        for (int j = 0; j < 8; ++j) q[j] = float((words[j / 4] >> (8 * (j % 4))) & 255u);
    }
    u32x4 d;
#pragma unroll
    for (int i = 0; i < 4; ++i) d[i] = pack_bf16x2(__builtin_fmaf(s, q[2 * i], b), __builtin_fmaf(s, q[2 * i + 1], b));
    return __builtin_bit_cast(bf16x8, d);
}

// A workgroup of 8 waves holds 16 kTM rows by 128 columns: wave (n, q) takes
// columns [64 n, 64 n + 64) and the q-th 64 k of each 256-k step for all the
// rows, so a weight is converted once per workgroup, in the registers it is
// multiplied from, and a fragment of x read from LDS serves four MFMAs. x
// goes through two LDS tiles (one barrier a step, the next step's in
// registers meanwhile). The four k quarters' float32 blocks are added through
// LDS at the end, in order: wave q finishes column tile q of its 64 columns.
// 200 rows, 2048 -> 12352, 4-bit: 26.7 us against 42.1 with 128 x 128 tiles of
// 256 threads (weights through LDS, one wave a SIMD). Of that the final sum
// and the stores take 5 us and the chip holds 194 such workgroups on 256 CUs.
// Scales and biases sit in LDS (eight scattered 2-byte loads a step cost 10
// us), the codes come two steps ahead (one ahead: 38 us).
//
// Split K: blockIdx.y = j takes the j-th of gridDim.y equal k ranges and
// stores its float32 block at partial + j M N.
template <int kBits, int kTM, class SB, class Y>
__global__ __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2))) void qlinear_mid_kernel(
    const uint16_t* __restrict__ x, const uint32_t* __restrict__ w, const typename SB::storage* __restrict__ scales,
    const typename SB::storage* __restrict__ biases, typename Y::storage* y, float* partial, const void* residual,
    int M, int N, int K, int group_size, int mt, int tiles) {
    constexpr int kBM = 16 * kTM;
    constexpr int kSegs = kStep / 8;                 // 16-byte pieces of a row's step
    constexpr int kXLoads = kBM * kSegs / 512;
    constexpr int kWords = 2 * kBits / 4;            // packed words of a lane's 16 codes of a step
    constexpr int kXBytes = 2 * kBM * kXS * 2;
    constexpr int kRound = (kTM + 1) / 2;            // row tiles of one round of the final sum
    constexpr int kSumBytes = kNW * kKW * (kKW - 1) * kRound * 64 * 16;
    struct __attribute__((aligned(2 * sizeof(typename SB::storage)))) ScaleBias {
        typename SB::storage s, b;
    };
    __shared__ __attribute__((aligned(16))) unsigned char lds[kXBytes > kSumBytes ? kXBytes : kSumBytes];
    __shared__ ScaleBias sb[kSBBytes / sizeof(ScaleBias)];  // [group][column]
    uint16_t* xs = reinterpret_cast<uint16_t*>(lds);

    // an eighth of the tiles to each XCD, row tiles of a column block together
    const int per_xcd = (tiles + 7) / 8;
    const int t = int(blockIdx.x % 8) * per_xcd + int(blockIdx.x / 8);
    if (t >= tiles) return;
    const int m0 = (t % mt) * kBM, n0 = (t / mt) * kBN;
    const int tid = threadIdx.x, l = tid & 63, lr = l & 15, lq = l >> 4;
    const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wn = wv / kKW, wq = wv % kKW;
    const int steps = K / kStep / int(gridDim.y), k0 = steps * int(blockIdx.y) * kStep;

    // operands: a uniform base and fixed 32-bit byte offsets; rows and columns
    // past the edge repeat the last one (not stored)
    uint32_t xo[kXLoads];
    int xl[kXLoads];
#pragma unroll
    for (int i = 0; i < kXLoads; ++i) {
        const int idx = tid + 512 * i, row = idx / kSegs, seg = idx % kSegs;
        const int r = m0 + row < M ? row : M - 1 - m0;
        xo[i] = (uint32_t(r) * uint32_t(K) + 8 * seg) * 2;
        xl[i] = row * kXS + 8 * seg;
    }
    const uint16_t* xtile = x + int64_t(m0) * K + k0;
    u16x8 xr[kXLoads];
    auto fetch_x = [&](int s) {
        const char* src = reinterpret_cast<const char*>(xtile + s * kStep);
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) xr[i] = *reinterpret_cast<const u16x8*>(src + xo[i]);
    };
    auto stage_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kXLoads; ++i) *reinterpret_cast<u16x8*>(xs + buf * kBM * kXS + xl[i]) = xr[i];
    };

    // lane (column lr, quarter lq) holds k 16 lq .. + 15 of the wave's slice
    const int64_t wpr = int64_t(K) * kBits / 32, G = K / group_size;
    const uint32_t* wtile = w + n0 * wpr + k0 * kBits / 32;
    uint32_t wo[kTN];
#pragma unroll
    for (int b = 0; b < kTN; ++b) {
        const int n = n0 + 16 * (kTN * wn + b) + lr, c = (n < N ? n : N - 1) - n0;
        wo[b] = (uint32_t(c) * uint32_t(wpr) + (wq * kSlice + 16 * lq) * kBits / 32) * 4;
    }
    uint32_t wd[2][kTN][kWords];
    auto fetch_w = [&](uint32_t (&dst)[kTN][kWords], int s) {
        const char* src = reinterpret_cast<const char*>(wtile + s * (kStep * kBits / 32));
#pragma unroll
        for (int b = 0; b < kTN; ++b) {
            const uint32_t* p = reinterpret_cast<const uint32_t*>(src + wo[b]);
#pragma unroll
            for (int i = 0; i < kWords; ++i) dst[b][i] = p[i];
        }
    };

    f32x4 acc[kTM][kTN];
#pragma unroll
    for (int a = 0; a < kTM; ++a)
#pragma unroll
        for (int b = 0; b < kTN; ++b) acc[a][b] = f32x4{0.f, 0.f, 0.f, 0.f};

    fetch_x(0);
    fetch_w(wd[0], 0);
    fetch_w(wd[1], steps > 1 ? 1 : 0);
    {
        const int groups = steps * kStep / group_size, g0 = k0 / group_size;
        for (int i = tid; i < kBN * groups; i += 512) {
            const int c = i / groups, g = i % groups;
            const int64_t at = int64_t(n0 + c < N ? n0 + c : N - 1) * G + g0 + g;
            sb[g * kBN + c] = ScaleBias{scales[at], biases[at]};
        }
    }
    stage_x(0);
    __syncthreads();
    // Codes are fetched two steps ahead (their scattered 8-byte pieces come
    // from HBM: one step ahead each step waited for them), x's one.
    auto step = [&](int s, uint32_t (&codes)[kTN][kWords]) {
        const ScaleBias* row = sb + uint32_t(s * kStep + wq * kSlice + 16 * lq) / uint32_t(group_size) * kBN + 16 * kTN * wn + lr;
        fetch_x(s + 1 < steps ? s + 1 : s);  // past the end: repeats, unused
        __builtin_amdgcn_sched_barrier(0);
        if (s) __syncthreads();
        const uint16_t* xrow = xs + (s & 1) * kBM * kXS + lr * kXS + wq * kSlice + 16 * lq;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
            bf16x8 bf[kTN];
#pragma unroll
            for (int b = 0; b < kTN; ++b) {
                const ScaleBias p = row[16 * b];
                bf[b] = weight_fragment<kBits>(&codes[b][kb * kWords / 2], SB::load(&p.s, 0), SB::load(&p.b, 0));
            }
            if (kb == 1) fetch_w(codes, s + 2 < steps ? s + 2 : s);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int a = 0; a < kTM; ++a) {
                const bf16x8 af = *reinterpret_cast<const bf16x8*>(xrow + 16 * a * kXS + 8 * kb);
#pragma unroll
                for (int b = 0; b < kTN; ++b) acc[a][b] = mfma_bf16(af, bf[b], acc[a][b]);
            }
            __builtin_amdgcn_sched_barrier(0);
        }
        stage_x((s + 1) & 1);
    };
    int s = 0;
    for (; s + 1 < steps; s += 2) {
        step(s, wd[0]);
        step(s + 1, wd[1]);
    }
    if (s < steps) step(s, wd[0]);

    // add the quarters: wave q of each column half keeps column tile q
    static_assert(kTN == kKW, "one column tile of a wave's 64 columns for each of its quarters");
    f32x4* sum = reinterpret_cast<f32x4*>(lds);
    const auto slot = [&](int owner, int from, int a) {  // from: the owner's other quarters in order
        return (((wn * kKW + owner) * (kKW - 1) + from) * kRound + a) * 64 + l;
    };
#pragma unroll
    for (int r = 0; r < kTM; r += kRound) {
        __syncthreads();  // the tile's (then the previous round's) readers are done
#pragma unroll
        for (int b = 0; b < kTN; ++b)
            if (b != wq) {
#pragma unroll
                for (int a = 0; a < kRound; ++a)
                    if (r + a < kTM) sum[slot(b, wq < b ? wq : wq - 1, a)] = acc[r + a][b];
            }
        __syncthreads();
#pragma unroll
        for (int a = 0; a < kRound; ++a) {
            if (r + a >= kTM) continue;
            f32x4 v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < kKW; ++q) {
                // the wave's own tile by a uniform choice (an index would put acc in memory)
                f32x4 own = acc[r + a][0];
#pragma unroll
                for (int b = 1; b < kTN; ++b)
                    if (wq == b) own = acc[r + a][b];
                f32x4 add = own;
                if (q != wq) add = sum[slot(wq, q < wq ? q : q - 1, a)];
                v = q == 0 ? add : v + add;
            }
            const int n = n0 + 16 * (kTN * wn + wq) + lr;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int m = m0 + 16 * (r + a) + 4 * lq + i;
                if (m >= M || n >= N) continue;
                const int64_t e = int64_t(m) * N + n;
                if (partial)
                    partial[int64_t(blockIdx.y) * M * N + e] = v[i];
                else
                    Y::store(y, e, residual ? round_to(v[i], Y::code) + load_any(residual, e, Y::code) : v[i]);
            }
        }
    }
}

struct MidPlan {
    int tm, splits;
};

// Rows of a workgroup (at most 112) and splits of K: the least of rounds over
// the CUs times steps times a step's time (0.5 us + 0.09 a row tile), plus a
// workgroup's start and final sum and, split, the partial blocks' traffic.
MidPlan mid_plan(int M, int N, int K, int group_size, int sb_dtype, int64_t ws_bytes) {
    MidPlan p{0, 1};
    double best = 1e30;
    for (int tm = 4; tm <= kMaxTM; ++tm)
        for (int s = 1; s <= 16; s *= 2) {
            if (K % (kStep * s) || (s > 1 && int64_t(s) * M * N * 4 > ws_bytes)) break;
            if (int64_t(K / s / group_size) * kBN * 2 * dtype_size(sb_dtype) > kSBBytes) continue;
            const int64_t wgs = (int64_t(M) + 16 * tm - 1) / (16 * tm) * ((N + kBN - 1) / kBN) * s;
            const double us = double((wgs + kCUs - 1) / kCUs) * (3.0 + (K / kStep / s) * (0.5 + 0.09 * tm)) +
                              (s > 1 ? 3.0 + double(s) * M * N * 8 / 4e6 : 0.0);
            if (us < best) {
                best = us;
                p = MidPlan{tm, s};
            }
        }
    return p;
}

template <int kBits, class SB, class Y>
auto mid_kernel_of(int tm) {
    switch (tm) {
        case 4: return qlinear_mid_kernel<kBits, 4, SB, Y>;
        case 5: return qlinear_mid_kernel<kBits, 5, SB, Y>;
        case 6: return qlinear_mid_kernel<kBits, 6, SB, Y>;
        default: return qlinear_mid_kernel<kBits, 7, SB, Y>;
    }
}

struct MidArgs {
    const void *x, *scales, *biases;
    const uint32_t* w;
    void* y;
    const void* residual;
    float* partial;
    int M, N, K, group_size;
    hipStream_t s;
};

template <int kBits, class SB, class Y>
int launch_mid_t(const MidArgs& a, MidPlan p) {
    const int mt = (a.M + 16 * p.tm - 1) / (16 * p.tm), tiles = mt * ((a.N + kBN - 1) / kBN);
    hipLaunchKernelGGL((mid_kernel_of<kBits, SB, Y>(p.tm)), dim3(unsigned((tiles + 7) / 8 * 8), unsigned(p.splits)),
                       dim3(512), 0, a.s, static_cast<const uint16_t*>(a.x), a.w,
                       static_cast<const typename SB::storage*>(a.scales),
                       static_cast<const typename SB::storage*>(a.biases), static_cast<typename Y::storage*>(a.y),
                       p.splits > 1 ? a.partial : nullptr, a.residual, a.M, a.N, a.K, a.group_size, mt, tiles);
    return check_launch("gdn_quantized_matmul");
}

template <int kBits, class SB>
int launch_mid_y(const MidArgs& a, int y_dtype, MidPlan p) {
    if (y_dtype == GDN_F32 || p.splits > 1) return launch_mid_t<kBits, SB, ActF32>(a, p);
    if (y_dtype == GDN_BF16) return launch_mid_t<kBits, SB, ActBF16>(a, p);
    return launch_mid_t<kBits, SB, ActF16>(a, p);
}

template <int kBits>
int launch_mid_sb(const MidArgs& a, int sb_dtype, int y_dtype, MidPlan p) {
    if (sb_dtype == GDN_F32) return launch_mid_y<kBits, ActF32>(a, y_dtype, p);
    if (sb_dtype == GDN_BF16) return launch_mid_y<kBits, ActBF16>(a, y_dtype, p);
    return launch_mid_y<kBits, ActF16>(a, y_dtype, p);
}

}  // namespace

// Up to kMaxRows rows: with more of them than workgroups want, the 128 x 128
// tiles read x less often (2048 -> 12352 at 4096 rows 352 us there, 397 here,
// even at 2048; 1024 -> 12352 at 600 rows 36 and 46). The same where this
// kernel's workgroups, one a CU, need a second round and the 128 x 128 tiles,
// two a CU, one: at 256 rows of 12352 columns (291 and 194 of them) K = 256
// takes 16 us here and 12 there, 1024 27 and 25 (groups of 32: 29 and 26),
// 2048 45 and 44 (53 and 45), 4096 79 and 81. And where both need two but the
// work of a round is short: K = 512, 384 rows 22.0 and 21.3, 511 rows 26.1 and
// 22.0; K = 1024, 384 rows 29.6 and 33.8, 511 rows, five row tiles to four,
// 34.7 and 34.5 (8-bit 38.1 and 33.6). 32-bit byte offsets inside a tile bound
// K; the scales of a k range have to fit the LDS (ws_bytes: the workspace a
// split may use).
bool mid_kernel_takes(int M, int N, int K, int group_size, int sb_dtype, int64_t ws_bytes) {
    if (M <= 64 || M > kMaxRows || N < 1 || K < 1 || K % kStep || K % group_size || K > (1 << 20)) return false;
    const MidPlan p = mid_plan(M, N, K, group_size, sb_dtype, ws_bytes);
    if (p.tm == 0) return false;
    const int64_t wgs = (int64_t(M) + 16 * p.tm - 1) / (16 * p.tm) * ((int64_t(N) + kBN - 1) / kBN);
    const int64_t tiled = (int64_t(M) + 127) / 128 * ((int64_t(N) + 127) / 128);
    return p.splits > 1 || wgs <= kCUs || (tiled > kCUs && K >= 1024 && (K > 1024 || M <= 448));
}

int64_t mid_workspace_bytes(int M, int N, int K, int group_size, int sb_dtype) {
    if (!mid_kernel_takes(M, N, K, group_size, sb_dtype, INT64_MAX)) return 0;
    const MidPlan p = mid_plan(M, N, K, group_size, sb_dtype, INT64_MAX);
    return p.splits > 1 ? int64_t(p.splits) * M * N * 4 : 0;
}

int launch_mid(const void* x, const uint32_t* w, const void* scales, const void* biases, int sb_dtype, void* y,
               int y_dtype, const void* residual, int M, int N, int K, int bits, int group_size, void* workspace,
               int64_t ws_bytes, hipStream_t s) {
    const MidPlan p = mid_plan(M, N, K, group_size, sb_dtype, workspace ? ws_bytes : 0);
    const MidArgs a{x, scales, biases, w, y, residual, static_cast<float*>(workspace), M, N, K, group_size, s};
    if (int rc = bits == 4 ? launch_mid_sb<4>(a, sb_dtype, y_dtype, p) : launch_mid_sb<8>(a, sb_dtype, y_dtype, p))
        return rc;
    if (p.splits > 1)
        return launch_split_sum(a.partial, p.splits, int64_t(M) * N, y, y_dtype, residual, s, "gdn_quantized_matmul/sum");
    return 0;
}

}  // namespace gdn
