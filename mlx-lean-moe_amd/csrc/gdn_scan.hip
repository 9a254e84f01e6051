// Sequential gated-delta scans over token runs.
//
// scan_reference_kernel: one thread per state row, the reference's exact
// operation order (gated_delta.py:35-39), any Dk/Dv and dtype mix. A test aid
// and the use_kernel=False path.
//
// scan_kernel: the state tile stays in registers across the token loop.
// 32 lanes own one state row (Dk/32 contiguous values each), 8 rows per
// 256-thread workgroup. Per token the lanes form S.k and S.q in one pass
// over the (undecayed) row and one 32-lane reduction, then
//     delta = beta (v - g S.k),  y = g S.q + delta (k.q),  S <- g S + delta k^T
// which is the reference's step (decay, read, delta, update, output)
// rearranged so that a token needs one reduction instead of two.
#include <type_traits>

#include "gdn_common.h"
#include "gdn_host.h"

namespace gdn {

__global__ void scan_reference_kernel(const void* q, const void* k, int qk_dtype, const void* v,
                                      int v_dtype, const void* g, int g_dtype, const void* beta,
                                      int beta_dtype, const void* state_in, void* state_out,
                                      int state_dtype, void* y, int y_dtype, const int32_t* cu,
                                      int N, int64_t L_uniform, int Hk, int Hv, int Dk, int Dv) {
    const int64_t gid = int64_t(blockIdx.x) * blockDim.x + threadIdx.x;
    if (gid >= int64_t(N) * Hv * Dv) return;
    const int run = int(gid / (int64_t(Hv) * Dv));
    const int h = int((gid / Dv) % Hv);
    const int dv = int(gid % Dv);
    const int hk = h / (Hv / Hk);
    float S[256];
    const int64_t sbase = ((int64_t(run) * Hv + h) * Dv + dv) * Dk;
    for (int j = 0; j < Dk; ++j) S[j] = load_any(state_in, sbase + j, state_dtype);
    const int64_t t0 = cu ? cu[run] : run * L_uniform;
    const int64_t t1 = cu ? cu[run + 1] : t0 + L_uniform;
    for (int64_t t = t0; t < t1; ++t) {
        const int64_t kb = (t * Hk + hk) * Dk;
        const float gt = load_any(g, t * Hv + h, g_dtype);
        const float bt = load_any(beta, t * Hv + h, beta_dtype);
        float read = 0.f;
        for (int j = 0; j < Dk; ++j) S[j] *= gt;
        for (int j = 0; j < Dk; ++j) read += S[j] * load_any(k, kb + j, qk_dtype);
        const float delta = (load_any(v, (t * Hv + h) * Dv + dv, v_dtype) - read) * bt;
        float out = 0.f;
        for (int j = 0; j < Dk; ++j) S[j] += load_any(k, kb + j, qk_dtype) * delta;
        for (int j = 0; j < Dk; ++j) out += S[j] * load_any(q, kb + j, qk_dtype);
        store_any(y, (t * Hv + h) * Dv + dv, y_dtype, out);
    }
    for (int j = 0; j < Dk; ++j) store_any(state_out, sbase + j, state_dtype, S[j]);
}

constexpr int kScanThreads = 256;
constexpr int kScanRows = kScanThreads / 32;
// Tokens staged at a time. (With 256 key channels 16 tokens take 66 KB, two
// workgroups a CU; 8 tokens at four a CU took 253 us against 232, 400 tokens,
// Hv = 32.)
constexpr int kScanBlock = 16;

// N consecutive elements of a row as loaded (raw), converted where they are
// used: a conversion at the load would wait for it. kVec: the operands are
// aligned for one load of the N.
template <class Act, int N, bool kVec>
struct RawRow {
    typename Act::storage x[N];
    GDN_DEV void load(const typename Act::storage* p) {
        if constexpr (kVec) {
            typedef typename Act::storage vec __attribute__((ext_vector_type(N)));
            const vec v = *reinterpret_cast<const vec*>(p);
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] = v[j];
        } else {
#pragma unroll
            for (int j = 0; j < N; ++j) x[j] = p[j];
        }
    }
    GDN_DEV float at(int j) const { return Act::load(x, j); }
};

// The scan is a serial chain over tokens, so its time is tokens x the chain's
// length: per token the two 32-lane sums and the update, about 40 vector
// instructions at one or two waves a SIMD. Fetching each token's inputs one
// token ahead put a whole memory latency on that chain (1.3 us a token); so
// the workgroup stages kScanBlock tokens of q, k (as floats), v, g, beta and
// the row-independent k.q in LDS, with the next block's loads in flight
// meanwhile, reads a token's operands one token ahead, and stores y once a
// block. 41 tokens, Hk = 16, Hv = 32, d = 128: 55 -> 13 us
// (bf16; 63 tokens float32 85 -> 18 us, 400 tokens at d = 256 2.9 ms -> 0.23,
// at d = 64 530 -> 69 us), about 0.21 us a token and 4.5 us a call.
template <class Act, int NPL, bool kVec>
__global__ __launch_bounds__(kScanThreads) void scan_kernel(
    const typename Act::storage* __restrict__ q, const typename Act::storage* __restrict__ k,
    const void* __restrict__ v, int v_dtype, const void* __restrict__ g, int g_dtype,
    const void* __restrict__ beta, int beta_dtype, const void* state_in, void* state_out,
    int state_dtype, void* __restrict__ y, int y_dtype, const int32_t* __restrict__ cu, int N,
    int64_t L_uniform, int Hk, int Hv, int Dv) {
    constexpr int Dk = 32 * NPL, TB = kScanBlock, kStage = TB / kScanRows;
    __shared__ __attribute__((aligned(16))) float ks[2][TB][Dk], qs[2][TB][Dk];
    __shared__ float4 gs[2][TB];  // g, beta, k.q
    __shared__ float vs[2][TB][kScanRows], ys[2][TB][kScanRows];
    const int tiles = (Dv + kScanRows - 1) / kScanRows;
    const int tile = blockIdx.x % tiles;
    const int h = (blockIdx.x / tiles) % Hv;
    const int run = blockIdx.x / (tiles * Hv);
    const int tid = threadIdx.x, l32 = tid & 31, grp = tid >> 5;
    const int row = tile * kScanRows + grp;
    const bool active = row < Dv;
    const int hk = h / (Hv / Hk);
    const int col = l32 * NPL;

    const int64_t t0 = cu ? cu[run] : run * L_uniform;
    const int64_t t1 = cu ? cu[run + 1] : t0 + L_uniform;

    // Block staging: 32-lane group i loads the q and k rows of tokens i and
    // i + 8 (their k.q summed over the group), threads 0-127 the rows' v,
    // 128-143 g, 144-159 beta. Tokens past the run repeat its last (unused).
    RawRow<Act, NPL, kVec> kr[kStage], qr[kStage];
    float vg = 0.f;
    auto fetch = [&](int64_t tb) {
        const auto at = [&](int i) { return tb + i < t1 ? tb + i : t1 - 1; };
#pragma unroll
        for (int i = 0; i < kStage; ++i) {
            const int64_t o = (at(grp + kScanRows * i) * Hk + hk) * Dk + col;
            kr[i].load(k + o);
            qr[i].load(q + o);
        }
        if (tid < TB * kScanRows) {
            const int r = tile * kScanRows + tid % kScanRows;
            vg = load_any(v, (at(tid / kScanRows) * Hv + h) * Dv + (r < Dv ? r : Dv - 1), v_dtype);
        } else if (tid < TB * kScanRows + TB) {
            vg = load_any(g, at(tid - TB * kScanRows) * Hv + h, g_dtype);
        } else if (tid < TB * kScanRows + 2 * TB) {
            vg = load_any(beta, at(tid - TB * kScanRows - TB) * Hv + h, beta_dtype);
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int i = 0; i < kStage; ++i) {
            const int t = grp + kScanRows * i;
            float kq = 0.f;
#pragma unroll
            for (int j = 0; j < NPL; ++j) {
                const float kj = kr[i].at(j), qj = qr[i].at(j);
                kq += kj * qj;
                ks[buf][t][col + j] = kj;
                qs[buf][t][col + j] = qj;
            }
            kq = group_sum<32>(kq);
            if (l32 == 0) gs[buf][t].z = kq;
        }
        if (tid < TB * kScanRows) vs[buf][tid / kScanRows][tid % kScanRows] = vg;
        else if (tid < TB * kScanRows + TB) gs[buf][tid - TB * kScanRows].x = vg;
        else if (tid < TB * kScanRows + 2 * TB) gs[buf][tid - TB * kScanRows - TB].y = vg;
    };
    auto store_y = [&](int buf, int64_t tb) {
        const int64_t t = tb + tid / kScanRows;
        const int r = tile * kScanRows + tid % kScanRows;
        if (tid < TB * kScanRows && t < t1 && r < Dv)
            store_any(y, (t * Hv + h) * Dv + r, y_dtype, ys[buf][tid / kScanRows][tid % kScanRows]);
    };
    if (t0 < t1) fetch(t0);

    float S[NPL];
    const int64_t sbase = ((int64_t(run) * Hv + h) * Dv + row) * Dk + col;
#pragma unroll
    for (int j = 0; j < NPL; ++j) S[j] = active ? load_any(state_in, sbase + j, state_dtype) : 0.f;

    struct Token {
        float k[NPL], q[NPL], v;
        float4 g;
    };
    auto read = [&](int buf, int t) {
        Token x;
#pragma unroll
        for (int j = 0; j < NPL; ++j) {
            x.k[j] = ks[buf][t][col + j];
            x.q[j] = qs[buf][t][col + j];
        }
        x.g = gs[buf][t];
        x.v = vs[buf][t][grp];
        return x;
    };
    auto step = [&](const Token& x, int buf, int t) {
        float sk = 0.f, sq = 0.f;
#pragma unroll
        for (int j = 0; j < NPL; ++j) {
            sk += S[j] * x.k[j];
            sq += S[j] * x.q[j];
        }
        sk = group_sum<32>(sk);
        sq = group_sum<32>(sq);
        const float delta = __builtin_fmaf(-x.g.x, sk, x.v) * x.g.y;
        const float out = __builtin_fmaf(x.g.x, sq, delta * x.g.z);
#pragma unroll
        for (int j = 0; j < NPL; ++j) S[j] = __builtin_fmaf(x.g.x, S[j], delta * x.k[j]);
        if (l32 == 0) ys[buf][t][grp] = out;
    };
    int buf = 0;
    for (int64_t tb = t0; tb < t1; tb += TB, buf ^= 1) {
        stage(buf);
        __syncthreads();
        if (tb > t0) store_y(buf ^ 1, tb - TB);
        if (tb + TB < t1) fetch(tb + TB);
        const int n = int(t1 - tb < TB ? t1 - tb : TB);
        Token cur = read(buf, 0);
        if (n == TB) {
#pragma unroll 4
            for (int t = 0; t < TB; ++t) {
                const Token next = read(buf, t + 1 < TB ? t + 1 : t);
                step(cur, buf, t);
                cur = next;
            }
        } else {
            for (int t = 0; t < n; ++t) {
                const Token next = read(buf, t + 1);  // t + 1 <= n < TB
                step(cur, buf, t);
                cur = next;
            }
        }
    }
    if (t0 < t1) {
        __syncthreads();
        store_y(buf ^ 1, t0 + (t1 - t0 - 1) / TB * TB);
    }
    if (active) {
#pragma unroll
        for (int j = 0; j < NPL; ++j) store_any(state_out, sbase + j, state_dtype, S[j]);
    }
}

static int check_scan_args(const char* who, const void* q, const void* k, int qk_dtype,
                           const void* v, int v_dtype, const void* g, int g_dtype,
                           const void* beta, int beta_dtype, const void* state_in,
                           void* state_out, int state_dtype, void* y, int y_dtype,
                           const int32_t* cu, int N, int64_t T_total, int Hk, int Hv, int Dk,
                           int Dv) {
    GDN_REQUIRE(N > 0 && T_total >= 0 && Hk > 0 && Hv > 0 && Dk > 0 && Dv > 0,
                "%s: bad sizes", who);
    GDN_REQUIRE(Hv % Hk == 0, "%s: Hv=%d is not a multiple of Hk=%d", who, Hv, Hk);
    GDN_REQUIRE(valid_dtype(qk_dtype) && valid_dtype(v_dtype) && valid_dtype(g_dtype) &&
                    valid_dtype(beta_dtype) && valid_dtype(state_dtype) && valid_dtype(y_dtype),
                "%s: bad dtype", who);
    GDN_REQUIRE(cu || T_total % N == 0, "%s: T_total not divisible by N without cu_seqlens", who);
    GDN_REQUIRE(state_in && state_out, "%s: null state", who);
    GDN_REQUIRE(T_total == 0 || (q && k && v && g && beta && y), "%s: null pointer", who);
    return 0;
}

}  // namespace gdn

using namespace gdn;

extern "C" int gdn_scan_reference(const void* q, const void* k, int qk_dtype, const void* v,
                                  int v_dtype, const void* g, int g_dtype, const void* beta,
                                  int beta_dtype, const void* state_in, void* state_out,
                                  int state_dtype, void* y, int y_dtype,
                                  const int32_t* cu_seqlens, int N, int64_t T_total, int Hk,
                                  int Hv, int Dk, int Dv, void* stream) {
    if (int rc = check_scan_args("gdn_scan_reference", q, k, qk_dtype, v, v_dtype, g, g_dtype,
                                 beta, beta_dtype, state_in, state_out, state_dtype, y, y_dtype,
                                 cu_seqlens, N, T_total, Hk, Hv, Dk, Dv))
        return rc;
    GDN_REQUIRE(Dk <= 256, "gdn_scan_reference: Dk=%d exceeds 256", Dk);
    const int64_t rows = int64_t(N) * Hv * Dv;
    const int threads = 64;
    const int64_t blocks = (rows + threads - 1) / threads;
    const int64_t L_uniform = cu_seqlens ? 0 : T_total / N;
    hipLaunchKernelGGL(scan_reference_kernel, dim3(unsigned(blocks)), dim3(threads), 0,
                       as_stream(stream), q, k, qk_dtype, v, v_dtype, g, g_dtype, beta,
                       beta_dtype, state_in, state_out, state_dtype, y, y_dtype, cu_seqlens, N,
                       L_uniform, Hk, Hv, Dk, Dv);
    return check_launch("gdn_scan_reference");
}

extern "C" int gdn_scan(const void* q, const void* k, int qk_dtype, const void* v, int v_dtype,
                        const void* g, int g_dtype, const void* beta, int beta_dtype,
                        const void* state_in, void* state_out, int state_dtype, void* y,
                        int y_dtype, const int32_t* cu_seqlens, int N, int64_t T_total, int Hk,
                        int Hv, int Dk, int Dv, void* stream) {
    if (int rc = check_scan_args("gdn_scan", q, k, qk_dtype, v, v_dtype, g, g_dtype, beta,
                                 beta_dtype, state_in, state_out, state_dtype, y, y_dtype,
                                 cu_seqlens, N, T_total, Hk, Hv, Dk, Dv))
        return rc;
    const int64_t tiles = (Dv + kScanRows - 1) / kScanRows;
    const int64_t blocks = int64_t(N) * Hv * tiles;
    const int64_t L_uniform = cu_seqlens ? 0 : T_total / N;
    hipStream_t s = as_stream(stream);
    const uintptr_t addr = reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k);
    const auto launch = [&](auto act, auto npl) {
        using Act = decltype(act);
        constexpr int NPL = decltype(npl)::value;
        using St = typename Act::storage;
        // one load per lane of NPL elements where both operands allow it
        const bool vec = addr % (NPL * sizeof(St)) == 0;
        hipLaunchKernelGGL((vec ? scan_kernel<Act, NPL, true> : scan_kernel<Act, NPL, false>),
                           dim3(unsigned(blocks)), dim3(kScanThreads), 0, s, static_cast<const St*>(q),
                           static_cast<const St*>(k), v, v_dtype, g, g_dtype, beta, beta_dtype, state_in,
                           state_out, state_dtype, y, y_dtype, cu_seqlens, N, L_uniform, Hk, Hv, Dv);
    };
    const auto by_dtype = [&](auto npl) {
        if (qk_dtype == GDN_F32) launch(ActF32{}, npl);
        else if (qk_dtype == GDN_BF16) launch(ActBF16{}, npl);
        else launch(ActF16{}, npl);
    };
    switch (Dk) {
        case 32: by_dtype(std::integral_constant<int, 1>{}); break;
        case 64: by_dtype(std::integral_constant<int, 2>{}); break;
        case 128: by_dtype(std::integral_constant<int, 4>{}); break;
        case 256: by_dtype(std::integral_constant<int, 8>{}); break;
        default:
            return fail(GDN_EUNSUPPORTED, "gdn_scan: Dk=%d not in {32, 64, 128, 256}", Dk);
    }
    return check_launch("gdn_scan");
}
