// Prefill front-end: causal depthwise conv + SiLU + conv-state roll, then the
// q/k scaling, for N packed token runs (linear_attention.py:61-79,103-113).
//
// Two kernels. The tiled one covers the production shape (Dk = Dv = 128,
// K = 4, 16-byte aligned operands): a wave holds four
// 128-channel groups (q, k or v heads) of one token, 8 channels a lane, and
// walks a tile of 4-16 tokens with the previous three input rows in registers, so
// each qkv row is read once per tile plus a three-row halo, with 16-byte
// loads and stores; the q/k RMS norm is a 16-lane DPP sum. The general
// one (any head size and K) gives each token a block: every channel's K-tap
// conv goes to LDS, then one wave per q/k head normalises. In both, extra
// blocks each write one run's new conv state (the last K-1 rows of
// concat(state, tokens)), so conv_state_out must not overlap conv_state_in.
#include <type_traits>

#include "gdn_common.h"
#include "gdn_conv.h"
#include "gdn_host.h"

namespace gdn {

constexpr int kFrontThreads = 256;

// Row j of a run's new conv state is row len + j of concat(state, tokens).
template <class Act>
GDN_DEV void write_conv_state(const typename Act::storage* __restrict__ qkv, int64_t qs,
                              const void* __restrict__ cs_in, int conv_dtype,
                              typename Act::storage* __restrict__ cs_out,
                              const int32_t* __restrict__ cu, int run, int64_t L_uniform, int C,
                              int S) {
    const int64_t start = cu ? cu[run] : run * L_uniform;
    const int64_t len = cu ? cu[run + 1] - cu[run] : L_uniform;
    for (int c = threadIdx.x; c < C; c += blockDim.x) {
        for (int j = 0; j < S; ++j) {
            const int64_t idx = len + j;
            const float x = idx < S
                ? Act::round(load_any(cs_in, (int64_t(run) * S + idx) * C + c, conv_dtype))
                : Act::load(qkv, (start + idx - S) * qs + c);
            Act::store(cs_out, (int64_t(run) * S + j) * C + c, x);
        }
    }
}

template <class Act>
__global__ __launch_bounds__(kFrontThreads) void frontend_kernel(
    const typename Act::storage* __restrict__ qkv, int64_t qs, const void* __restrict__ cs_in,
    int conv_dtype, typename Act::storage* __restrict__ cs_out, const float* __restrict__ w,
    const int32_t* __restrict__ cu, int N, int64_t T, int64_t L_uniform,
    typename Act::storage* __restrict__ qo, typename Act::storage* __restrict__ ko,
    typename Act::storage* __restrict__ vo, int Hk, int Hv, int Dk, int Dv, int K) {
    extern __shared__ float conv_out[];  // C floats
    const int C = 2 * Hk * Dk + Hv * Dv;
    const int64_t blk = blockIdx.x;
    const int tid = threadIdx.x;
    const int S = K - 1;  // conv state rows

    if (blk >= T) {
        const int run = int(blk - T);
        if (run < N) write_conv_state<Act>(qkv, qs, cs_in, conv_dtype, cs_out, cu, run, L_uniform, C, S);
        return;
    }

    const int64_t t = blk;
    const int run = cu ? find_run(cu, N, t) : int(t / L_uniform);
    const int64_t start = cu ? cu[run] : run * L_uniform;
    const int64_t pos = t - start;  // position inside the run
    // the conv and SiLU of each channel, with the tiled kernel's instruction
    // sequence (conv_chain, silu_act; for float32 that is the decode step's)
    for (int c = tid; c < C; c += kFrontThreads) {
        float acc[1] = {Act::round(conv_chain(K, [&](int j) {
            const int64_t idx = pos + j;  // index into concat(state, run tokens)
            const float x = idx < S
                ? Act::round(load_any(cs_in, (int64_t(run) * S + idx) * C + c, conv_dtype))
                : Act::load(qkv, (start + idx - S) * qs + c);
            return float2{Act::round(w[int64_t(c) * K + j]), x};
        }))};
        silu_act<Act::code>(acc);
        conv_out[c] = Act::round(acc[0]);
    }
    __syncthreads();

    // the q/k scaling: 128-wide bf16 heads with the tiled kernels' rms_norm8
    // (lane l takes channels 8 (l % 16) .. + 7, the wave's four DPP rows the
    // same head, the first storing it); others in double, each value rounded
    // once (rms_rr), as the decode step scales them
    const int wave = tid / kWave, lane = tid % kWave;
    const float inv = 1.f / sqrtf(float(Dk));
    const float scale_q = Act::round(inv * inv), scale_k = Act::round(inv);
    for (int head = wave; head < 2 * Hk; head += kFrontThreads / kWave) {
        const float* src = conv_out + head * Dk;
        const bool is_q = head < Hk;
        const float sc = is_q ? scale_q : scale_k;
        typename Act::storage* dst = is_q ? qo + (t * Hk + head) * Dk : ko + (t * Hk + head - Hk) * Dk;
        if (Act::code == GDN_BF16 && Dk == 128) {
            const int c8 = 8 * (lane & 15);
            float o[8], n[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = src[c8 + e];
            rms_norm8(o, n);
            if (lane < 16) {
#pragma unroll
                for (int e = 0; e < 8; ++e) Act::store(dst, c8 + e, sc * n[e]);
            }
        } else {
            double ss = 0.0;
            for (int e = lane; e < Dk; e += kWave) ss = fma(double(src[e]), double(src[e]), ss);
            const double rr = rms_rr(group_sum<kWave>(ss), Dk);
            for (int e = lane; e < Dk; e += kWave)
                Act::store(dst, e, sc * round_once(double(src[e]) * rr, Act::code));
        }
    }
    const float* vsrc = conv_out + 2 * Hk * Dk;
    for (int e = tid; e < Hv * Dv; e += kFrontThreads) Act::store(vo, t * Hv * Dv + e, vsrc[e]);
}


// A lane's 8 channels of a 128-channel group held by 16 lanes, in the tiled
// kernel's activation type: the loads and stores of a token's row, the conv
// state and taps as the general kernel rounds them, and its conv, SiLU and
// scaled norm. bf16: channels 8l .. 8l + 7 (16 bytes). float32: channels
// 4l .. 4l + 3 and 64 + 4l .. (two 16-byte pieces, each 256 contiguous bytes
// over the 16 lanes); SiLU from expf and an IEEE divide and the norm in
// double, each value rounded once, as the decode step does.
template <class Act>
struct Lane8;

template <>
struct Lane8<ActBF16> {
    using Raw = uint4;
    static constexpr int kAhead = 8;  // rows in flight
    static GDN_DEV int first(int l16) { return 8 * l16; }
    static GDN_DEV Raw load(const uint16_t* p) { return *reinterpret_cast<const uint4*>(p); }
    static GDN_DEV void unpack(const Raw& r, float (&x)[8]) { unpack8(r, x); }
    static GDN_DEV void store(uint16_t* p, const float (&o)[8]) { *reinterpret_cast<uint4*>(p) = pack8(o); }
    template <int kConvDt>
    static GDN_DEV void state(const void* p, int64_t at, float (&x)[8]) { load_state8<kConvDt>(p, at, x); }
    static GDN_DEV void taps(const float* w, int64_t c0, float (&wr)[8][4]) { load_conv_w8(w, c0, wr); }
    static GDN_DEV void conv_silu(const float (&wr)[8][4], const float (&win)[3][8], const float (&x)[8],
                                  float (&o)[8]) {
        conv_silu8(wr, win, x, o);
    }
    static GDN_DEV void norm(const float (&o)[8], float sc, float (&n)[8]) {
        rms_norm8(o, n);
#pragma unroll
        for (int e = 0; e < 8; ++e) n[e] = sc * n[e];
    }
};

template <>
struct Lane8<ActF32> {
    struct Raw {
        float4 a, b;
    };
    static constexpr int kAhead = 4;
    static GDN_DEV int first(int l16) { return 4 * l16; }
    static GDN_DEV Raw load(const float* p) {
        return {*reinterpret_cast<const float4*>(p), *reinterpret_cast<const float4*>(p + 64)};
    }
    static GDN_DEV void unpack(const Raw& r, float (&x)[8]) {
        const float v[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = v[e];
    }
    static GDN_DEV void store(float* p, const float (&o)[8]) {
        *reinterpret_cast<float4*>(p) = make_float4(o[0], o[1], o[2], o[3]);
        *reinterpret_cast<float4*>(p + 64) = make_float4(o[4], o[5], o[6], o[7]);
    }
    template <int kConvDt>
    static GDN_DEV void state(const void* p, int64_t at, float (&x)[8]) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            if constexpr (kConvDt == GDN_F32) {
                const float4 v = *reinterpret_cast<const float4*>(static_cast<const float*>(p) + at + 64 * h);
                x[4 * h] = v.x, x[4 * h + 1] = v.y, x[4 * h + 2] = v.z, x[4 * h + 3] = v.w;
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) x[4 * h + e] = load_any(p, at + 64 * h + e, kConvDt);
            }
        }
    }
    static GDN_DEV void taps(const float* w, int64_t c0, float (&wr)[8][4]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float4 v = *reinterpret_cast<const float4*>(w + (c0 + (e & 3) + 64 * (e >> 2)) * 4);
            wr[e][0] = v.x, wr[e][1] = v.y, wr[e][2] = v.z, wr[e][3] = v.w;
        }
    }
    static GDN_DEV void conv_silu(const float (&wr)[8][4], const float (&win)[3][8], const float (&x)[8],
                                  float (&o)[8]) {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const float xs[4] = {win[0][e], win[1][e], win[2][e], x[e]};
            o[e] = conv_chain(4, [&](int j) { return float2{wr[e][j], xs[j]}; });
        }
        silu_act<GDN_F32>(o);
    }
    static GDN_DEV void norm(const float (&o)[8], float sc, float (&n)[8]) {
        double ss = 0.0;
#pragma unroll
        for (int e = 0; e < 8; ++e) ss = fma(double(o[e]), double(o[e]), ss);
        const double rr = rms_rr(group_sum<16>(ss), 128);
#pragma unroll
        for (int e = 0; e < 8; ++e) n[e] = sc * float(double(o[e]) * rr);
    }
};

constexpr int kMaxTileTokens = 16;  // tokens a wave walks, at most
constexpr int kTileWaves = 4;    // waves a block, four channel groups each

constexpr int kStateChunk = kTileWaves * kWave * 8;  // conv-state elements a block writes

// Tiles of kTileTokens = TT tokens (16, or 8 or 4 for short inputs).
// grid (n_state + n_tiles, ceil(G / 16)) for G = 2 Hk + Hv channel groups of
// 128. The first n_state columns write the runs' new conv states, flattened
// to N (K-1) C elements, kStateChunk a block (8 independent elements a
// thread; dispatched first, they overlap the tiles); block (n_state + x, y)
// covers tokens [TT x, TT x + TT) of groups [16 y, 16 y + 16).
//
// The three-row window holds rows t-3 .. t-1 of concat(run's conv state,
// run's tokens) for the token t in hand: it is loaded so at the tile's first
// token and reloaded from the conv state where a run starts inside the tile,
// and each token shifts itself in.
//
// float32, T = 1531, C = 8192 (50 MB in, 50 MB out): 25 us (3.9 TB/s) against
// 117 us on the general kernel (a block per token, scalar loads, every tap's
// row read again); what is left over the copy's 20 us is the expf and divide
// of SiLU.
template <class Act, int kConvDt, int kTileTokens>
__global__ __launch_bounds__(kTileWaves * kWave) void frontend_tiled_kernel(
    const typename Act::storage* __restrict__ qkv, int64_t qs, const void* __restrict__ cs_in,
    typename Act::storage* __restrict__ cs_out, const float* __restrict__ w, const int32_t* __restrict__ cu,
    int N, int64_t T, int64_t L_uniform, int n_state, typename Act::storage* __restrict__ qo,
    typename Act::storage* __restrict__ ko, typename Act::storage* __restrict__ vo, int Hk, int Hv) {
    using Lane = Lane8<Act>;
    constexpr int D = 128, K = 4, S = K - 1;
    const int G = 2 * Hk + Hv;
    const int C = G * D;
    if (int(blockIdx.x) < n_state) {
        const int64_t total = int64_t(N) * S * C;
        const int64_t first = (int64_t(blockIdx.x) * gridDim.y + blockIdx.y) * kStateChunk + threadIdx.x;
        float x[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) {  // all loads first: they do not wait on each other
            const int64_t e = first + int64_t(i) * kTileWaves * kWave;
            if (e < total) {
                const int run = int(e / (int64_t(S) * C));
                const int j = int(e / C % S), c = int(e % C);
                const int64_t start = cu ? cu[run] : run * L_uniform;
                const int64_t idx = (cu ? cu[run + 1] - cu[run] : L_uniform) + j;  // in concat(state, run)
                x[i] = idx < S ? Act::round(load_any(cs_in, (int64_t(run) * S + idx) * C + c, kConvDt))
                               : Act::load(qkv, (start + idx - S) * qs + c);
            }
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const int64_t e = first + int64_t(i) * kTileWaves * kWave;
            if (e < total) Act::store(cs_out, e, x[i]);
        }
        return;
    }
    const int wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const int g0 = (int(blockIdx.y) * kTileWaves + wave) * 4;  // the wave's first group
    if (g0 >= G) return;  // the whole wave idles; the kernel has no barrier
    const int g = g0 + lane / 16;
    const bool live = g < G;
    const int c0 = (live ? g : G - 1) * D + Lane::first(lane % 16);  // this lane's first channel
    const int64_t t0 = (int64_t(blockIdx.x) - n_state) * kTileTokens;

    // the tile's rows, kAhead in flight (the last tile's missing ones repeat
    // row T-1, unused)
    constexpr int kAhead = kTileTokens < Lane::kAhead ? kTileTokens : Lane::kAhead;
    const auto row_at = [&](int i) {
        const int64_t t = t0 + i < T ? t0 + i : T - 1;
        return Lane::load(qkv + t * qs + c0);
    };
    typename Lane::Raw raw[kAhead];
#pragma unroll
    for (int i = 0; i < kAhead; ++i) raw[i] = row_at(i);
    int run = cu ? find_run(cu, N, t0) : int(t0 / L_uniform);
    int64_t start = cu ? cu[run] : run * L_uniform;
    int64_t next = cu ? cu[run + 1] : start + L_uniform;
    float win[S][8];
#pragma unroll
    for (int j = 0; j < S; ++j) {
        const int64_t row = t0 - S + j;
        if (row >= start) {
            Lane::unpack(Lane::load(qkv + row * qs + c0), win[j]);
        } else {  // concat index row - start + S of the run's conv state
            Lane::template state<kConvDt>(cs_in, (int64_t(run) * S + (row - start + S)) * C + c0, win[j]);
        }
    }
    float wr[8][K];
    Lane::taps(w, c0, wr);

    const float inv = 1.f / sqrtf(float(D));
    const float sc = g < Hk ? Act::round(inv * inv) : Act::round(inv);
    const bool is_v = g >= 2 * Hk;
    // whether the wave holds a q or k head (uniform: a wave may also hold v
    // heads when Hk is not a multiple of 4; their lanes keep o)
    const bool qk_wave = __builtin_amdgcn_readfirstlane(int(g0 < 2 * Hk)) != 0;
    typename Act::storage* dst = g < Hk ? qo + int64_t(g) * D
                  : !is_v ? ko + int64_t(g - Hk) * D
                          : vo + int64_t(g - 2 * Hk) * D;
    const int64_t dst_row = is_v ? int64_t(Hv) * D : int64_t(Hk) * D;
    dst += Lane::first(lane % 16);

#pragma unroll
    for (int i = 0; i < kTileTokens; ++i) {
        const int64_t t = t0 + i;
        if (t < T && t >= next) {  // a run starts at t (uniform): its conv state is the window
            run = cu ? find_run(cu, N, t) : int(t / L_uniform);
            start = t;
            next = cu ? cu[run + 1] : t + L_uniform;
#pragma unroll
            for (int j = 0; j < S; ++j)
                Lane::template state<kConvDt>(cs_in, (int64_t(run) * S + j) * C + c0, win[j]);
        }
        float x[8];
        Lane::unpack(raw[i % kAhead], x);
        if (i + kAhead < kTileTokens) raw[i % kAhead] = row_at(i + kAhead);
        float o[8];
        Lane::conv_silu(wr, win, x, o);
        if (qk_wave) {  // q and k heads: scaled RMS norm (v lanes keep o)
            float n[8];
            Lane::norm(o, sc, n);
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = is_v ? o[e] : n[e];
        }
        if (live && t < T) Lane::store(dst + t * dst_row, o);
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            win[0][e] = win[1][e];
            win[1][e] = win[2][e];
            win[2][e] = x[e];
        }
    }
}

}  // namespace gdn

using namespace gdn;

extern "C" int gdn_frontend(const void* qkv, int64_t qkv_stride, const void* conv_state_in, void* conv_state_out,
                            int conv_dtype, const float* conv_weight, const int32_t* cu_seqlens,
                            int N, int64_t T_total, void* q_out, void* k_out, void* v_out, int Hk,
                            int Hv, int Dk, int Dv, int K, int act_dtype, void* stream) {
    GDN_REQUIRE(N > 0 && T_total >= 0 && Hk > 0 && Hv > 0 && Dk > 0 && Dv > 0 && K >= 1,
                "gdn_frontend: bad sizes");
    GDN_REQUIRE(Hv % Hk == 0, "gdn_frontend: Hv=%d is not a multiple of Hk=%d", Hv, Hk);
    GDN_REQUIRE(valid_dtype(conv_dtype), "gdn_frontend: bad conv dtype");
    GDN_REQUIRE(act_dtype == GDN_F32 || act_dtype == GDN_BF16,
                "gdn_frontend: activations must be float32 or bfloat16");
    GDN_REQUIRE(cu_seqlens || T_total % N == 0,
                "gdn_frontend: T_total=%lld not divisible by N=%d without cu_seqlens",
                (long long)T_total, N);
    const int64_t C = 2LL * Hk * Dk + int64_t(Hv) * Dv;
    GDN_REQUIRE(C * 4 <= 64 * 1024, "gdn_frontend: conv_dim %lld exceeds the LDS tile", (long long)C);
    GDN_REQUIRE(qkv_stride >= C, "gdn_frontend: qkv_stride %lld below conv_dim %lld",
                (long long)qkv_stride, (long long)C);
    const int64_t S = K - 1;
    if (S > 0) {
        GDN_REQUIRE(conv_state_in && conv_state_out, "gdn_frontend: null conv state");
        GDN_REQUIRE(!overlaps(conv_state_in, N * S * C * dtype_size(conv_dtype), conv_state_out,
                              N * S * C * dtype_size(act_dtype)),
                    "gdn_frontend: conv_state_out overlaps conv_state_in");
    }
    if (T_total == 0 && S == 0) return 0;
    GDN_REQUIRE(conv_weight && (T_total == 0 || (qkv && q_out && k_out && v_out)),
                "gdn_frontend: null pointer");
    const int64_t L_uniform = cu_seqlens ? 0 : T_total / N;
    const auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    if (Dk == 128 && Dv == 128 && K == 4 && T_total > 0 && aligned(qkv) &&
        qkv_stride * dtype_size(act_dtype) % 16 == 0 &&
        aligned(conv_state_in) && aligned(conv_weight) && aligned(q_out) && aligned(k_out) &&
        aligned(v_out)) {
        const int G = 2 * Hk + Hv;
        const int gy = (G + 4 * kTileWaves - 1) / (4 * kTileWaves);
        // tiles of 16 tokens, or of 8 or 4 where that leaves under 1024
        // workgroups (a wave walks its tile's tokens one after another)
        int tile = kMaxTileTokens;
        while (tile > 4 && (T_total + tile - 1) / tile * gy < 1024) tile /= 2;
        const int64_t n_tiles = (T_total + tile - 1) / tile;
        const int64_t chunks = (int64_t(N) * S * C + kStateChunk - 1) / kStateChunk;
        const int64_t n_state = (chunks + gy - 1) / gy;
        const int64_t gx = n_state + n_tiles;
        GDN_REQUIRE(gx < (1LL << 31) / (kTileWaves * kWave) && gy < 65536,
                    "gdn_frontend: %lld tokens exceed the grid", (long long)T_total);
        const auto launch = [&](auto act, auto tt) {
            using Act = decltype(act);
            using St = typename Act::storage;
            constexpr int TT = decltype(tt)::value;
            const auto kern = conv_dtype == GDN_F32    ? frontend_tiled_kernel<Act, GDN_F32, TT>
                              : conv_dtype == GDN_BF16 ? frontend_tiled_kernel<Act, GDN_BF16, TT>
                                                       : frontend_tiled_kernel<Act, GDN_F16, TT>;
            hipLaunchKernelGGL(kern, dim3(unsigned(gx), unsigned(gy)), dim3(kTileWaves * kWave), 0,
                               as_stream(stream), static_cast<const St*>(qkv), qkv_stride, conv_state_in,
                               static_cast<St*>(conv_state_out), conv_weight, cu_seqlens, N, T_total, L_uniform,
                               int(n_state), static_cast<St*>(q_out), static_cast<St*>(k_out),
                               static_cast<St*>(v_out), Hk, Hv);
        };
        const auto by_tile = [&](auto act) {
            if (tile == 16) launch(act, std::integral_constant<int, 16>{});
            else if (tile == 8) launch(act, std::integral_constant<int, 8>{});
            else launch(act, std::integral_constant<int, 4>{});
        };
        if (act_dtype == GDN_F32) by_tile(ActF32{});
        else by_tile(ActBF16{});
        return check_launch("gdn_frontend");
    }
    const int64_t blocks = T_total + (S > 0 ? N : 0);
    if (blocks == 0) return 0;
    const size_t lds = size_t(C) * sizeof(float);
    if (act_dtype == GDN_F32) {
        hipLaunchKernelGGL(frontend_kernel<ActF32>, dim3(unsigned(blocks)), dim3(kFrontThreads),
                           lds, as_stream(stream), static_cast<const float*>(qkv), qkv_stride, conv_state_in,
                           conv_dtype, static_cast<float*>(conv_state_out), conv_weight,
                           cu_seqlens, N, T_total, L_uniform, static_cast<float*>(q_out),
                           static_cast<float*>(k_out), static_cast<float*>(v_out), Hk, Hv, Dk,
                           Dv, K);
    } else {
        hipLaunchKernelGGL(frontend_kernel<ActBF16>, dim3(unsigned(blocks)), dim3(kFrontThreads),
                           lds, as_stream(stream), static_cast<const uint16_t*>(qkv), qkv_stride,
                           conv_state_in, conv_dtype, static_cast<uint16_t*>(conv_state_out),
                           conv_weight, cu_seqlens, N, T_total, L_uniform,
                           static_cast<uint16_t*>(q_out), static_cast<uint16_t*>(k_out),
                           static_cast<uint16_t*>(v_out), Hk, Hv, Dk, Dv, K);
    }
    return check_launch("gdn_frontend");
}
