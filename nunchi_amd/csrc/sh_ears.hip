// Kernels of the ears (imi/core/ears.cpp:198-407) for gfx950. Every fp32 operation is the one the oracle
// restatement of imi's ears performs, in the same order; the exceptions are the C library's erff (GELU) and the
// double log10 of the mel, here the device's routines.
//
// The float tables run on the matrix cores in imi_wg_group12's order (k_etab below).
#include "sh_ears.h"
#include "sh_device.h"

namespace sh {
namespace {

constexpr int ET = 256;

__device__ __forceinline__ float gelu_erf(float x) { return 0.5f * x * (1.0f + erff(x * 0.70710678118654752f)); }

// where feature e of position p sits in a table's input (sh_ears.h)
__device__ __forceinline__ size_t xat(int e, int p, int ldx) {
    return ((((size_t)(e >> 5) * (ldx >> 4) + (p >> 4)) * 2 + ((e >> 4) & 1)) * 64 + (e & 3) * 16 + (p & 15)) * 4 + ((e >> 2) & 3);
}

// a lane's 8 weights of a 32-column chunk, raw: F16 bits (one 16-byte load) or F32 (two)
template <bool F32W> struct wraw;
template <> struct wraw<false> { uint4 a; };
template <> struct wraw<true> { float4 a, b; };

template <bool F32W>
__device__ __forceinline__ wraw<F32W> wload(const void* w, size_t tile, int lane) {
    wraw<F32W> r;
    if constexpr (F32W) {
        const float4* p = static_cast<const float4*>(w) + tile * 128 + lane;
        r.a = p[0];
        r.b = p[64];
    } else {
        r.a = static_cast<const uint4*>(w)[tile * 64 + lane];
    }
    return r;
}
template <bool F32W>
__device__ __forceinline__ float wval(const wraw<F32W>& r, int s) {   // (s known at compile time)
    if constexpr (F32W) {
        const float o[8] = {r.a.x, r.a.y, r.a.z, r.a.w, r.b.x, r.b.y, r.b.z, r.b.w};
        return o[s];
    } else {
        const unsigned v[4] = {r.a.x, r.a.y, r.a.z, r.a.w};
        return h2f((uint16_t)((v[s >> 1] >> (16 * (s & 1))) & 0xffffu));
    }
}

// The float tables on the matrix cores, in imi_wg_group12's order (imi/core/tables.cpp:522-556): one chain
// acc = fma(w, x, acc) per row and position over the columns in order. v_mfma_f32_16x16x4_f32 runs four columns of 16
// rows x 16 positions: its four K steps are four fused multiply-adds in order, each rounded once, bit for bit the VALU's
// fmaf chain (no mismatch in 11 M random chains: 3 M of spread exponents, 8 M with denormals, signed zeros and overflow; the
// ears' bit-for-bit tests rest on it). A chain then takes 8 cycles a column, the rate of one
// matrix core in fp32, with a single chain per wave in flight; v_mfma_f32_4x4x1_16b_f32, one column per instruction,
// is as fast only with two waves to cover its 15-cycle dependency, and wants a weight conversion and an operand word per
// lane for every 64 x 4 outputs and column, where this takes them for 16 x 16 outputs and four columns.
// A wave is 16 rows x 16 MP positions, a workgroup 4 waves over 64 rows. Lane l supplies row l % 16, column l / 16 of the
// four (a) and position l % 16 of that column (b); it holds rows 4 (l / 16) .. + 3 at position l % 16. Tables and inputs
// are laid out so that a lane's operands of 32 columns are whole 16-byte words and a wave reads 1 KB pieces (a vector
// load costs its wave about as many cycles as one of these products), requested DC chunks of 32 columns ahead. Every
// global load is unconditional (chunk indices clamped; past the table's last column nothing is multiplied), so the
// compiler's wait counts stay exact.
// At 384 positions, against one column per v_mfma_f32_4x4x1_16b_f32: b|c|x 2304 x 768 33.7 -> 21.2 us, gate|up 4096 x 768
// 45.5 -> 30.1, o and pw2 768 x 768 20.3 -> 12.8, down 768 x 2048 47.7 -> 26.3, mlp.3 2048 x 2048 63.7 -> 37.8, pre_encode
// 768 x 4096 91.7 -> 47.6; at 29 positions b|c|x 16.9 -> 8.8, gate|up 17.7 -> 9.7, down 39.3 -> 17.2, pre_encode 76.2 ->
// 30.8. (With this product but feature-major inputs, read a word per step: b|c|x 28.0, gate|up 44.0, mlp.3 51.3, pre_encode
// 65.3; at 29 positions gate|up 12.6.) The matrix cores are busy 14 % (o, pw2) to 48 % (mlp.3) of the time at 384
// positions: a 768-row table has 1152 tiles for 1024 SIMDs, a wave's chain takes 8 cycles a column (2048 columns 6.8 us),
// and its loads (3 KB per 32 columns and 16 x 16 outputs) are issued between the products.
template <int EPI, bool F32W, int MP>
__global__ __launch_bounds__(ET) void k_etab(etab_args a) {
    typedef float v4f __attribute__((ext_vector_type(4)));
    constexpr int DC = MP == 4 ? 2 : MP == 2 ? 4 : 8;
    constexpr bool EXPE = EPI == EE_GLU || EPI == EE_SILU;   // epilogues that take e^x
    __shared__ uint64_t eE[ET / 64][EXPE ? 32 : 1];         // expf's table, a copy per wave (no memory round trip)
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), li = lane & 15, lq = lane >> 4;
    const int nt = a.W.rows_pad / 16, tile = (int)blockIdx.x * (ET / 64) + wv, p0 = (int)blockIdx.y * 16 * MP;
    if (tile >= nt) return;   // (whole waves; no barriers below)
    const uint64_t et = EXPE ? kExp2Tab[lane & 31] : 0;      // (requested first: its wait needs nothing later)
    const int K = a.W.cols, nst = K / 4, nch = (K + 31) / 32, np = a.ldx / 16;
    const float4* xs[MP];   // (position tiles past ldx re-read the last one)
#pragma unroll
    for (int m = 0; m < MP; m++) xs[m] = reinterpret_cast<const float4*>(a.x) + (size_t)min(p0 / 16 + m, np - 1) * 128 + lane;
    wraw<F32W> wr[DC];
    float4 xr[DC][2][MP];
    auto request = [&](int c, int d) {
        const int cc = min(c, nch - 1);
        wr[d] = wload<F32W>(a.W.w, (size_t)cc * nt + tile, lane);
#pragma unroll
        for (int h = 0; h < 2; h++)
#pragma unroll
            for (int m = 0; m < MP; m++) xr[d][h][m] = xs[m][((size_t)cc * np * 2 + h) * 64];
    };
    auto step = [&](int d, int s, int m) {
        const float4 v = xr[d][s >> 2][m];
        return (s & 3) == 0 ? v.x : (s & 3) == 1 ? v.y : (s & 3) == 2 ? v.z : v.w;
    };
    v4f acc[MP];
#pragma unroll
    for (int m = 0; m < MP; m++) acc[m] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int d = 0; d < DC; d++) request(d, d);
    int c = 0;
    for (; 8 * (c + DC) <= nst; c += DC) {
#pragma unroll
        for (int d = 0; d < DC; d++) {
#pragma unroll
            for (int s = 0; s < 8; s++)
#pragma unroll
                for (int m = 0; m < MP; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(wval<F32W>(wr[d], s), step(d, s, m), acc[m], 0, 0, 0);
            request(c + d + DC, d);
        }
    }
#pragma unroll
    for (int d = 0; d < DC; d++)
#pragma unroll
        for (int s = 0; s < 8; s++)
            if (8 * (c + d) + s < nst) {
#pragma unroll
                for (int m = 0; m < MP; m++)
                    acc[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(wval<F32W>(wr[d], s), step(d, s, m), acc[m], 0, 0, 0);
            }
    // lane l holds rows rb .. rb + 3 of position p0 + 16 m + l % 16
    const int rb = 16 * tile + 4 * lq;
    if (EXPE && lane < 32) eE[wv][EXPE ? lane : 0] = et;
    __builtin_amdgcn_wave_barrier();
    const uint64_t* etab = eE[wv];
    const int kind = a.out_kind;
    const int pend = kind != EO_POS ? min(a.ldx, a.ldo) : a.P;   // feature-major outputs also fill the padded positions
    auto put = [&](int row, int p, float v) {
        float* d = kind == EO_POS ? a.out + (size_t)p * a.ldo + row : kind == EO_FEAT ? a.out + (size_t)row * a.ldo + p
                                                                                     : a.out + xat(row, p, a.ldo);
        *d = EPI == EE_ADD ? *d + v : v;
    };
#pragma unroll
    for (int m = 0; m < MP; m++) {
        const int p = p0 + 16 * m + li;
        if constexpr (EPI == EE_GLU) {   // rows 0-7 of each 16 are gates, 8-15 the matching ups (lanes + 32)
            v4f up;
#pragma unroll
            for (int i = 0; i < 4; i++) up[i] = __shfl_xor(acc[m][i], 32);
            if (lq < 2 && p < pend) {
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    const int ro = 8 * tile + 4 * lq + i;
                    if (ro < a.W.rows / 2) put(ro, p, silu_t(acc[m][i], etab) * up[i]);
                }
            }
        } else if constexpr (EPI == EE_POWER) {   // rows (2j, 2j + 1) = (re, im) of bin j
            if (p < pend) {
#pragma unroll
                for (int h = 0; h < 2; h++) {
                    const int ro = (rb >> 1) + h;
                    if (ro < a.W.rows / 2) put(ro, p, fmaf(acc[m][2 * h], acc[m][2 * h], acc[m][2 * h + 1] * acc[m][2 * h + 1]));
                }
            }
        } else if (p < pend) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const int row = rb + i;
                if (row >= a.W.rows) break;
                const float v = acc[m][i] + (a.bias ? a.bias[row] : 0.0f);
                put(row, p, EPI == EE_SILU ? silu_t(v, etab) : EPI == EE_GELU ? gelu_erf(v) : v);
            }
        }
    }
}

// (these fill table inputs: a thread writes the four features e, e + 4, e + 8, e + 12 that are one 16-byte word)
__device__ __forceinline__ int quad_feature(int g) { return 16 * (g >> 2) + (g & 3); }

__global__ __launch_bounds__(ET) void k_eframes(const float* pcm, int n, const float* hann, int n_fft, int hop,
                                                int n_fr, float* fx, int ldf) {
    const int fr = blockIdx.x * ET + threadIdx.x, k0 = quad_feature(blockIdx.y);
    if (fr >= ldf) return;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = k0 + 4 * q;
        const long i = (long)fr * hop + k;
        v[q] = k < n_fft && fr < n_fr && i < n ? hann[k] * pcm[i] : 0.0f;
    }
    *reinterpret_cast<float4*>(fx + xat(k0, fr, ldf)) = make_float4(v[0], v[1], v[2], v[3]);
}

// imi sums all n_bin terms in bin order; a term with a zero filter weight is fma(0, pw, s) = s exactly (pw is a sum of
// two squares, finite and >= 0), so each mel only runs over its filter's nonzero bins [lo, hi), in order
__global__ __launch_bounds__(ET) void k_emel(const float* pw, int ldp, const float* fb, const int2* span, int n_bin,
                                             int n_mel, int n_fr, float* mel) {
    const int fr = blockIdx.x * ET + threadIdx.x, m = blockIdx.y;
    if (fr >= n_fr) return;
    const float* w = fb + (size_t)m * n_bin;
    const int2 sp = span[m];
    double s = 0.0;
    for (int b = sp.x; b < sp.y; b++) s = fma((double)w[b], (double)pw[(size_t)b * ldp + fr], s);
    mel[(size_t)fr * n_mel + m] = (float)((log10(s < 1e-12 ? 1e-12 : s) + 4.0) / 4.0);
}

// thread per (t, f) and 8 channels: the 9 taps' inputs are requested first (addresses clamped into the image) and
// shared by the channels; a tap outside the image leaves o as it is (a select, not a multiply by zero, so o keeps its
// bits exactly as imi's skipped tap does)
constexpr int E0_CPT = 8;
__global__ __launch_bounds__(ET) void k_econv0(const float* mel, int n_fr, int n_mel, const float* w9, const float* b,
                                               int C, int T2, int F2, float* a0) {
    __shared__ uint64_t etab[32];   // expf's table (each lookup in constant memory is a gather: 63 -> 53 us at 3072 frames)
    if (threadIdx.x < 32) etab[threadIdx.x] = kExp2Tab[threadIdx.x];
    __syncthreads();
    const int i = blockIdx.x * ET + threadIdx.x, c0 = blockIdx.y * E0_CPT;
    if (i >= T2 * F2) return;
    const int t = i / F2, f = i - t * F2;
    float v[9];
    bool ok[9];
#pragma unroll
    for (int j = 0; j < 9; j++) {
        const int ti = 2 * t + j % 3 - 1, fi = 2 * f + j / 3 - 1;   // j = kh * 3 + kw: kw along time, kh along freq
        ok[j] = ti >= 0 && ti < n_fr && fi >= 0 && fi < n_mel;
        const int tc = ti < 0 ? 0 : ti >= n_fr ? n_fr - 1 : ti, fc = fi < 0 ? 0 : fi >= n_mel ? n_mel - 1 : fi;
        v[j] = mel[(size_t)tc * n_mel + fc];
    }
#pragma unroll
    for (int cc = 0; cc < E0_CPT; cc++) {
        const int c = c0 + cc;
        if (c >= C) break;
        float o = b[c];
#pragma unroll
        for (int j = 0; j < 9; j++) {
            const float u = fmaf(v[j], w9[(size_t)j * C + c], o);
            o = ok[j] ? u : o;
        }
        a0[(size_t)c * T2 * F2 + i] = silu_t(o, etab);
    }
}

__global__ __launch_bounds__(ET) void k_edw(const float* in, int Ti, int Fi, int ldi, const float* w9, const float* b,
                                            int C, int To, int Fo, float* out, int ldo) {
    const int i = blockIdx.x * ET + threadIdx.x, c0 = quad_feature(blockIdx.y);
    if (i >= To * Fo) return;
    const int t = i / Fo, f = i - t * Fo;
    int at[9];
    bool ok[9];
#pragma unroll
    for (int j = 0; j < 9; j++) {
        const int ti = 2 * t + j % 3 - 1, fi = 2 * f + j / 3 - 1;
        ok[j] = ti >= 0 && ti < Ti && fi >= 0 && fi < Fi;
        const int tc = ti < 0 ? 0 : ti >= Ti ? Ti - 1 : ti, fc = fi < 0 ? 0 : fi >= Fi ? Fi - 1 : fi;
        at[j] = tc * Fi + fc;
    }
    float o[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int c = min(c0 + 4 * q, C - 1);
        const float* src = in + (size_t)c * ldi;
        o[q] = b[c];
#pragma unroll
        for (int j = 0; j < 9; j++) {
            const float u = fmaf(src[at[j]], w9[(size_t)j * C + c], o[q]);
            o[q] = ok[j] ? u : o[q];
        }
    }
    *reinterpret_cast<float4*>(out + xat(c0, i, ldo)) = make_float4(o[0], o[1], o[2], o[3]);
}

__global__ __launch_bounds__(ET) void k_eflat(const float* a, int lda, int K, int F8, int P, float* xf, int ldf) {
    const int p = blockIdx.x * ET + threadIdx.x, k0 = quad_feature(blockIdx.y);
    if (p >= ldf) return;
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int k = min(k0 + 4 * q, K - 1), c = k / F8, f = k - c * F8;
        v[q] = p < P ? a[(size_t)c * lda + (size_t)p * F8 + f] : 0.0f;
    }
    *reinterpret_cast<float4*>(xf + xat(k0, p, ldf)) = make_float4(v[0], v[1], v[2], v[3]);
}

// a workgroup is 16 positions x 64 features: each wave forms 4 positions' scales in imi's order (every workgroup of a
// position forms the same scale), then h is written as a table input, a thread the four features of one 16-byte
// word. Bound by memory round trips: a width of 256, 512 or 768 (NT = E / 32; 0 takes any) has every operand requested
// before the chains (768: 5.4 -> 4.9 us a launch at 384 positions, 5.0 -> 4.1 at 29)
template <int NT>
__global__ __launch_bounds__(ET) void k_enorm(const float* x, const float* w, int E, int P, int ldh, float eps, float* h) {
    __shared__ float sc[16];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, p0 = blockIdx.x * 16, e0 = blockIdx.y * 64;
    // this thread's four values and weights, requested before the scales' chains
    const int pl = threadIdx.x & 15, p = p0 + pl, e = min(e0 + quad_feature((int)threadIdx.x >> 4), E - 13);
    float xv[4], wv4[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        xv[q] = x[(size_t)min(p, P - 1) * E + e + 4 * q];
        wv4[q] = w[e + 4 * q];
    }
    const int hf = lane >> 5, pq = wv * 4 + hf;   // half-wave hf forms positions p0 + 4 wv + hf and + 2 + hf
    const float* r0 = x + (size_t)min(p0 + pq, P - 1) * E;
    const float* r1 = x + (size_t)min(p0 + pq + 2, P - 1) * E;
    float sq[2];
    rms_scale_half<2, NT>({r0, r1}, E, eps, sq);
    if ((lane & 31) == 0) {
        sc[pq] = sq[0];
        sc[pq + 2] = sq[1];
    }
    __syncthreads();
    const float s = sc[pl];
    if (e0 + quad_feature((int)threadIdx.x >> 4) >= E) return;   // (E is a multiple of 32)
    float v[4];
#pragma unroll
    for (int q = 0; q < 4; q++) v[q] = p < P ? xv[q] * s * wv4[q] : 0.0f;
    *reinterpret_cast<float4*>(h + xat(e, p, ldh)) = make_float4(v[0], v[1], v[2], v[3]);
}

__global__ __launch_bounds__(ET) void k_econv(const float* big, int ld, const float* w, int E, int d_conv, int P,
                                              float* act, int lda) {
    const int e = blockIdx.x * ET + threadIdx.x, p = blockIdx.y;
    if (e >= E) return;
    if (p >= P) { act[xat(e, p, lda)] = 0.0f; return; }
    float co = 0.0f;
    for (int k = 0; k < d_conv; k++) {
        const int t = p - (d_conv - 1) + k;
        if (t < 0) continue;
        const float* rw = big + (size_t)t * ld;
        co = fmaf(w[(size_t)k * E + e], rw[e] * rw[2 * E + e], co);
    }
    act[xat(e, p, lda)] = big[(size_t)p * ld + E + e] * co;
}

// one wave per (position, head slot): the n_head query heads, then the n_kv key heads
template <int DPL>
__global__ __launch_bounds__(ET) void k_eqk(float* big, int ld, int n_head, int n_kv, int D, const float* q_norm,
                                            const float* k_norm, const float2* cs, int P, float eps) {
    __shared__ float stg[ET / 64][EA_MAX_D];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, ns = n_head + n_kv;
    const int u = blockIdx.x * (ET / 64) + wv;
    if (u >= P * ns) return;
    const int p = u / ns, sl = u - p * ns;
    float* v = big + (size_t)p * ld + (sl < n_head ? sl * D : n_head * D + (sl - n_head) * D);
    float r[DPL];
    head_norm_rope<DPL>(v, sl < n_head ? q_norm : k_norm, stg[wv], cs + (size_t)p * (D / 2), D, eps, r);
#pragma unroll
    for (int c = 0; c < DPL; c++)
        if (lane + 64 * c < D) v[lane + 64 * c] = r[c];
}

// one wave per (position, query head): lane t < nk scores key s0 + t (fma chain over the dimensions), the exponentials
// are summed in key order by lane 0, lane i runs dimension i's chain o = fma(e_t, v_t, o) over the keys
__global__ __launch_bounds__(ET) void k_eattn(const float* big, int ld, int n_head, int n_kv, int D, int window, int P,
                                              float* act, int lda) {
    __shared__ float qs[ET / 64][EA_MAX_D];
    __shared__ float es[ET / 64][EA_MAX_WIN];
    __shared__ float sums[ET / 64];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
    const int u = blockIdx.x * (ET / 64) + wv;
    if (u >= P * n_head) return;
    const int p = u / n_head, hh = u - p * n_head, kv = hh / (n_head / n_kv);
    const int Hq = n_head * D, Hk = n_kv * D;
    const int s0 = p - window + 1 > 0 ? p - window + 1 : 0, nk = p - s0 + 1;
    for (int i = lane; i < D; i += 64) qs[wv][i] = big[(size_t)p * ld + hh * D + i];
    __builtin_amdgcn_wave_barrier();
    const float scale = 1.0f / sqrtf((float)D);
    float sc = -__builtin_inff();
    if (lane < nk) {
        const float* k = big + (size_t)(s0 + lane) * ld + Hq + kv * D;
        float s = 0.0f;
        for (int i = 0; i < D; i++) s = fmaf(qs[wv][i], k[i], s);
        sc = s * scale;
    }
    float mx = sc;
    for (int o = 32; o > 0; o >>= 1) {
        const float t = __shfl_xor(mx, o);
        mx = mx < t ? t : mx;
    }
    if (lane < nk) es[wv][lane] = expf_glibc(sc - mx);
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
        float sum = 0.0f;
        for (int t = 0; t < nk; t++) sum += es[wv][t];
        sums[wv] = sum;
    }
    __builtin_amdgcn_wave_barrier();
    const float sum = sums[wv];
    for (int i = lane; i < D; i += 64) {
        float o = 0.0f;
        for (int t = 0; t < nk; t++) o = fmaf(es[wv][t], big[(size_t)(s0 + t) * ld + Hq + Hk + kv * D + i], o);
        act[xat(hh * D + i, p, lda)] = o / sum;
    }
}

// one wave per position: h = x * rms(x) * post_ln into LDS; lane 0 forms the double mean and variance in order;
// then fma((float)(h - mu) * inv, ln_w, ln_b)
__global__ __launch_bounds__(ET) void k_efinal(const float* x, const float* post_ln, const float* ln_w,
                                               const float* ln_b, int E, int P, float eps, float* h, int ldh) {
    extern __shared__ float hs_all[];
    __shared__ double st[ET / 64][2];
    const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6, p = blockIdx.x * (ET / 64) + wv;
    if (p >= ldh) return;
    if (p >= P) {
        for (int e = lane; e < E; e += 64) h[xat(e, p, ldh)] = 0.0f;
        return;
    }
    float* hs = hs_all + (size_t)wv * E;
    const float* xp = x + (size_t)p * E;
    const float s = E == 768 ? rms_scale_wave_g<24>(xp, eps) : rms_scale_wave(xp, E, eps);
    for (int e = lane; e < E; e += 64) hs[e] = xp[e] * s * post_ln[e];
    __builtin_amdgcn_wave_barrier();
    if (lane == 0) {
        double mu = 0.0, var = 0.0;
        // (E is a multiple of 32; 32 values read ahead of their adds, which alone are in order: 40 -> 34 us)
        for (int k = 0; k < E; k += 32) {
            float v[32];
#pragma unroll
            for (int u = 0; u < 32; u++) v[u] = hs[k + u];
#pragma unroll
            for (int u = 0; u < 32; u++) mu += (double)v[u];
        }
        mu /= E;
        for (int k = 0; k < E; k += 32) {
            float v[32];
#pragma unroll
            for (int u = 0; u < 32; u++) v[u] = hs[k + u];
#pragma unroll
            for (int u = 0; u < 32; u++) {
                const double d = (double)v[u] - mu;
                var = fma(d, d, var);
            }
        }
        st[wv][0] = mu;
        st[wv][1] = (double)(float)(1.0 / sqrt(var / E + 1e-5));
    }
    __builtin_amdgcn_wave_barrier();
    const double mu = st[wv][0];
    const float inv = (float)st[wv][1];
    for (int e = lane; e < E; e += 64) h[xat(e, p, ldh)] = fmaf((float)((double)hs[e] - mu) * inv, ln_w[e], ln_b[e]);
}

inline unsigned blocks(long n) { return (unsigned)((n + ET - 1) / ET); }
inline unsigned quads(int n) { return (unsigned)((n + 15) / 16 * 4); }   // feature quads (quad_feature)

}  // namespace

hipError_t launch_etab(int epi, const etab_args& a, hipStream_t s) {
    if (a.W.cols % 8 || a.W.cols < 8 || a.W.rows_pad % 16 || a.ldx % 16 || a.ldx < 16 ||
        (a.out_kind == EO_FEAT && a.ldo % 4) || (a.out_kind == EO_TABLE && a.ldo % 16)) return hipErrorInvalidValue;
    const unsigned gx = (unsigned)((a.W.rows_pad + 63) / 64);
    // position tiles per wave: the most that keeps enough waves in flight
    const auto waves = [&](int mp) { return 4L * gx * ((a.ldx + 16 * mp - 1) / (16 * mp)); };
    const int mp = waves(4) >= 2048 ? 4 : waves(2) >= 2048 ? 2 : 1;
    const dim3 grid(gx, (unsigned)((a.ldx + 16 * mp - 1) / (16 * mp)));
#define SH_ETAB(E)                                                                                        \
    case E:                                                                                               \
        if (a.W.f32) {                                                                                    \
            if (mp == 4) SH_ETAB_MF(E, true, 4); else if (mp == 2) SH_ETAB_MF(E, true, 2); else SH_ETAB_MF(E, true, 1); \
        } else {                                                                                          \
            if (mp == 4) SH_ETAB_MF(E, false, 4); else if (mp == 2) SH_ETAB_MF(E, false, 2); else SH_ETAB_MF(E, false, 1); \
        }                                                                                                 \
        break;
#define SH_ETAB_MF(E, F, N) hipLaunchKernelGGL((k_etab<E, F, N>), grid, dim3(ET), 0, s, a)
    switch (epi) {
        SH_ETAB(EE_STORE) SH_ETAB(EE_ADD) SH_ETAB(EE_SILU) SH_ETAB(EE_GELU) SH_ETAB(EE_GLU) SH_ETAB(EE_POWER)
        default: return hipErrorInvalidValue;
    }
#undef SH_ETAB
#undef SH_ETAB_MF
    return hipGetLastError();
}

hipError_t launch_eframes(const float* pcm, int n, const float* hann, int n_fft, int hop, int n_fr, float* fx, int ldf,
                          hipStream_t s) {
    hipLaunchKernelGGL(k_eframes, dim3(blocks(ldf), quads(n_fft)), dim3(ET), 0, s, pcm, n, hann, n_fft, hop, n_fr, fx, ldf);
    return hipGetLastError();
}
hipError_t launch_emel(const float* pw, int ldp, const float* fb, const int2* span, int n_bin, int n_mel, int n_fr,
                       float* mel, hipStream_t s) {
    hipLaunchKernelGGL(k_emel, dim3(blocks(n_fr), n_mel), dim3(ET), 0, s, pw, ldp, fb, span, n_bin, n_mel, n_fr, mel);
    return hipGetLastError();
}
hipError_t launch_econv0(const float* mel, int n_fr, int n_mel, const float* w9, const float* b, int C, float* a0,
                         hipStream_t s) {
    const int T2 = (n_fr + 1) / 2, F2 = n_mel / 2;
    hipLaunchKernelGGL(k_econv0, dim3(blocks((long)T2 * F2), (C + E0_CPT - 1) / E0_CPT), dim3(ET), 0, s, mel, n_fr, n_mel,
                       w9, b, C, T2, F2, a0);
    return hipGetLastError();
}
hipError_t launch_edw(const float* in, int Ti, int Fi, int ldi, const float* w9, const float* b, int C, float* out,
                      int ldo, hipStream_t s) {
    const int To = (Ti + 1) / 2, Fo = Fi / 2;
    hipLaunchKernelGGL(k_edw, dim3(blocks((long)To * Fo), quads(C)), dim3(ET), 0, s, in, Ti, Fi, ldi, w9, b, C, To, Fo, out, ldo);
    return hipGetLastError();
}
hipError_t launch_eflat(const float* a, int lda, int C, int F8, int P, float* xf, int ldf, hipStream_t s) {
    hipLaunchKernelGGL(k_eflat, dim3(blocks(ldf), quads(C * F8)), dim3(ET), 0, s, a, lda, C * F8, F8, P, xf, ldf);
    return hipGetLastError();
}
hipError_t launch_enorm(const float* x, const float* w, int E, int P, float eps, float* h, int ldh, hipStream_t s) {
    if (E % 32) return hipErrorInvalidValue;
    if (ldh % 16) return hipErrorInvalidValue;
    const dim3 grid((unsigned)(ldh / 16), (unsigned)((E + 63) / 64));
    switch (E) {
        case 256: hipLaunchKernelGGL((k_enorm<8>), grid, dim3(ET), 0, s, x, w, E, P, ldh, eps, h); break;
        case 512: hipLaunchKernelGGL((k_enorm<16>), grid, dim3(ET), 0, s, x, w, E, P, ldh, eps, h); break;
        case 768: hipLaunchKernelGGL((k_enorm<24>), grid, dim3(ET), 0, s, x, w, E, P, ldh, eps, h); break;
        default: hipLaunchKernelGGL((k_enorm<0>), grid, dim3(ET), 0, s, x, w, E, P, ldh, eps, h);
    }
    return hipGetLastError();
}
hipError_t launch_econv(const float* big, int ld, const float* w, int E, int d_conv, int P, float* act, int lda,
                        hipStream_t s) {
    hipLaunchKernelGGL(k_econv, dim3(blocks(E), lda), dim3(ET), 0, s, big, ld, w, E, d_conv, P, act, lda);
    return hipGetLastError();
}
hipError_t launch_eqk(float* big, int ld, int n_head, int n_kv, int D, const float* q_norm, const float* k_norm,
                      const float2* cs, int P, float eps, hipStream_t s) {
    if (D % 32 || D > EA_MAX_D) return hipErrorInvalidValue;
    const unsigned g = (unsigned)(((long)P * (n_head + n_kv) + 3) / 4);
    if (D > 64) hipLaunchKernelGGL((k_eqk<2>), dim3(g), dim3(ET), 0, s, big, ld, n_head, n_kv, D, q_norm, k_norm, cs, P, eps);
    else hipLaunchKernelGGL((k_eqk<1>), dim3(g), dim3(ET), 0, s, big, ld, n_head, n_kv, D, q_norm, k_norm, cs, P, eps);
    return hipGetLastError();
}
hipError_t launch_eattn(const float* big, int ld, int n_head, int n_kv, int D, int window, int P, float* act, int lda,
                        hipStream_t s) {
    if (D > EA_MAX_D || window < 1 || window > EA_MAX_WIN) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_eattn, dim3((unsigned)(((long)P * n_head + 3) / 4)), dim3(ET), 0, s, big, ld, n_head, n_kv, D,
                       window, P, act, lda);
    return hipGetLastError();
}
hipError_t launch_efinal(const float* x, const float* post_ln, const float* ln_w, const float* ln_b, int E, int P,
                         float eps, float* h, int ldh, hipStream_t s) {
    if (E % 32 || E > 4096) return hipErrorInvalidValue;
    hipLaunchKernelGGL(k_efinal, dim3((unsigned)((ldh + 3) / 4)), dim3(ET), (size_t)4 * E * sizeof(float), s, x, post_ln,
                       ln_w, ln_b, E, P, eps, h, ldh);
    return hipGetLastError();
}

}  // namespace sh
