// codec_kernels.hip -- gfx950 kernels of the audio codec decoder.
//
// Every matrix product runs on v_mfma_f32_16x16x4_f32: fp32 activations times the file's
// weights widened to fp32 (exact for fp16), fp32 accumulation -- the arithmetic of the
// reference's gemm_par on F16/F32 matrices (csrc/src/gemv.cpp:343-363) in another
// summation order.
//
// v_mfma_f32_16x16x4_f32 lane layout: lane l gives A[l%16][k] and B[k][l%16] for the
// k = l/16 of the step, and holds D[4(l/16)+i][l%16], i = 0..3.  Which 4 values of
// the contraction index form a step is free as long as A and B agree; here lane group
// g = l/16 walks 8 (GEMM) or 16 (attention) consecutive indices of its own, so every
// operand is read with 16-byte vector loads.
#include <math.h>

#include "codec.h"
#include "mh_device.h"

namespace mh {
namespace {

typedef float floatx4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

__device__ __forceinline__ float exp_f(float x) {  // e^x; e^-inf = 0
    return __builtin_amdgcn_exp2f(x * 1.4426950408889634f);
}

// 8 consecutive weights of one row, raw (fp16: one 16-byte load; fp32: two).
template <int WF32>
struct W8 {
    uint4 r[WF32 ? 2 : 1];
    __device__ __forceinline__ void load(const void *w, size_t off) {
        if constexpr (WF32) {
            const uint4 *p = reinterpret_cast<const uint4 *>(static_cast<const float *>(w) + off);
            r[0] = p[0];
            r[1] = p[1];
        } else {
            r[0] = *reinterpret_cast<const uint4 *>(static_cast<const uint16_t *>(w) + off);
        }
    }
    __device__ __forceinline__ void zero() {
#pragma unroll
        for (int i = 0; i < (WF32 ? 2 : 1); ++i) r[i] = make_uint4(0, 0, 0, 0);
    }
    __device__ __forceinline__ float get(int s) const {
        if constexpr (WF32) {
            const uint32_t u = s < 4 ? (&r[0].x)[s] : (&r[1].x)[s - 4];
            return __uint_as_float(u);
        } else {
            const uint32_t u = (&r[0].x)[s >> 1];
            return h2f((uint16_t)((s & 1) ? (u >> 16) : (u & 0xffffu)));
        }
    }
};

// What element (m, nn) of a product needs besides its sum, loaded before any element is stored:
// a load behind a store that may alias it costs its own round trip (QKV in large tiles 28.5 ->
// 23.8 us a launch of an utterance, f2 and proj 22.5 -> 20.7; in an 8-frame chunk, with the
// operands requested first of all, QKV 7.4 -> 6.7, f1 6.3 -> 5.8).
struct EpiIn {
    float2 cs;       // CEPI_QKV: cos and sin of the element's RoPE pair
    float *out;      // CEPI_QKV: where it goes
    float y, ls, b;  // CEPI_RESID: the residual and its layer scale; CEPI_STORE: the bias
};

template <int EPI>
__device__ __forceinline__ EpiIn epi_load(const CodecGemmArgs &g, int m, int nn) {
    EpiIn e;
    if constexpr (EPI == CEPI_QKV) {
        // q to its buffer, k and v to the ring slot of the row's position; cos and sin from the
        // piece's table (loaded for v too: no branch)
        const int region = nn / kCodecDModel, c = nn - region * kCodecDModel;
        const int slot = (*g.pos0 + m) % g.ring;
        float *dst = region == 0 ? g.q : (region == 1 ? g.kc : g.vc);
        e.out = dst + (size_t)(region == 0 ? m : slot) * kCodecDModel + c;
        e.cs = g.rope[(size_t)m * (kCodecHeadDim / 2) + ((c & (kCodecHeadDim - 1)) >> 1)];
    } else if constexpr (EPI == CEPI_RESID) {
        e.y = g.y[(size_t)m * g.ldy + nn];
        e.ls = g.ls[nn];
    } else if constexpr (EPI == CEPI_STORE) {
        e.b = g.bias ? g.bias[nn] : 0.f;
    }
    return e;
}

// partner: the sum of column nn ^ 1 of the row (CEPI_QKV: interleaved RoPE, audio_layer.cpp:30-44)
template <int EPI>
__device__ __forceinline__ void epi_store(const CodecGemmArgs &g, const EpiIn &e, int m, int nn, float v, float partner) {
    if constexpr (EPI == CEPI_QKV) {
        float out = v;
        if (nn < 2 * kCodecDModel) out = (nn & 1) ? partner * e.cs.y + v * e.cs.x : v * e.cs.x - partner * e.cs.y;
        *e.out = out;
    } else if constexpr (EPI == CEPI_STORE) {
        const int p = g.patch;
        g.y[((size_t)m * p + nn % p) * g.ldy + nn / p] = g.bias ? v + e.b : v;
    } else if constexpr (EPI == CEPI_GELU) {
        // audio_gelu (audio_layer.cpp:46)
        g.y[(size_t)m * g.ldy + nn] = 0.5f * v * (1.0f + erff(v * 0.7071067811865476f));
    } else {
        g.y[(size_t)m * g.ldy + nn] = e.y + e.ls * v;
    }
}

// Y[m][n] = sum_k A[m][k] W[n][k] over a 16-row x 16-column tile.  The contraction is
// cut into chunks of 32 columns; wave w takes chunks [w nch/4, (w+1) nch/4) of every
// round of 1024 columns and reads its A and W straight from global memory (each lane
// 8 consecutive columns of one A row and one W row per chunk, all of the wave's chunks in
// flight before the first MFMA); the 4 partial tiles are summed in LDS and thread t
// finishes element (t / 16, t % 16).  Prologues transform A as it is loaded:
// CPRO_LN with per-row (mean, 1/std) from LDS, CPRO_MERGE with wave w = head w.
// chunks of 32 per wave per round: rounds of 1024 columns, or all of K = 256 under a prologue
template <int PRO>
constexpr int kWaveChunks = PRO == CPRO_ROWS ? 8 : 2;

template <int PRO, int EPI, int WF32>
__global__ __launch_bounds__(256) void codec_gemm_kernel(const CodecGemmArgs g) {
    __shared__ float red[4][256];
    __shared__ float2 rowst[16];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
    const int m0 = blockIdx.y * 16, n0 = blockIdx.x * 16;
    const int am = m0 + col;        // A row this lane feeds
    const bool avalid = am < g.M;
    const int n = n0 + col;          // W row this lane feeds (N % 16 == 0: always valid)
    constexpr int WC = kWaveChunks<PRO>;
    const int fm = m0 + (t >> 4), fn = n0 + (t & 15);  // the element this thread finishes
    const EpiIn ein = epi_load<EPI>(g, min(fm, g.M - 1), fn);

    // CPRO_MERGE: this lane's (row am, head = wave) split weights e^(m_s - M) / sum_s e^(m_s - M) l_s.
    // Every split's statistics are loaded before any is used (a loop over the splits waited for
    // each in turn: 10.7 us for the proj launch of an 8-frame chunk)
    float fs[PRO == CPRO_MERGE ? kCodecMaxSplits : 1], inv_den = 0.f;
    if constexpr (PRO == CPRO_MERGE) {
        float2 st[kCodecMaxSplits];
        const float2 *sp = g.st + (size_t)(avalid ? am : 0) * kCodecHeads + wave;
#pragma unroll
        for (int s = 0; s < kCodecMaxSplits; ++s)
            st[s] = s < g.splits ? sp[(size_t)s * g.M * kCodecHeads] : make_float2(-INFINITY, 0.f);
        float mx = -INFINITY, den = 0.f;
#pragma unroll
        for (int s = 0; s < kCodecMaxSplits; ++s) mx = fmaxf(mx, st[s].x);
#pragma unroll
        for (int s = 0; s < kCodecMaxSplits; ++s) {
            fs[s] = s < g.splits ? exp_f(st[s].x - mx) : 0.f;
            den += fs[s] * st[s].y;
        }
        inv_den = 1.0f / den;
    }

    floatx4 acc0 = {0.f, 0.f, 0.f, 0.f}, acc1 = {0.f, 0.f, 0.f, 0.f};
    for (int k0 = 0; k0 < g.K; k0 += 32 * 4 * WC) {
        const int nch = min(4 * WC, (g.K - k0) >> 5);
        const int c0 = wave * nch / 4, c1 = (wave + 1) * nch / 4;
        float4 av[WC][2];
        W8<WF32> wr[WC];
#pragma unroll
        for (int c = 0; c < WC; ++c) {
            const int kk = k0 + 32 * (c0 + c) + 8 * grp;
            if (c0 + c < c1) {
                wr[c].load(g.w, (size_t)n * g.K + kk);
                if constexpr (PRO == CPRO_MERGE) {
                    const float *op = g.o + (size_t)(avalid ? am : 0) * kCodecDModel + kk;
                    float4 o[kCodecMaxSplits][2];
#pragma unroll
                    for (int s = 0; s < kCodecMaxSplits; ++s)
                        if (s < g.splits) {  // (uniform)
                            const float4 *os = reinterpret_cast<const float4 *>(op + (size_t)s * g.M * kCodecDModel);
                            o[s][0] = os[0];
                            o[s][1] = os[1];
                        }
                    av[c][0] = av[c][1] = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
                    for (int s = 0; s < kCodecMaxSplits; ++s)
                        if (s < g.splits && avalid) {
                            const float f = fs[s];
                            av[c][0].x += f * o[s][0].x;
                            av[c][0].y += f * o[s][0].y;
                            av[c][0].z += f * o[s][0].z;
                            av[c][0].w += f * o[s][0].w;
                            av[c][1].x += f * o[s][1].x;
                            av[c][1].y += f * o[s][1].y;
                            av[c][1].z += f * o[s][1].z;
                            av[c][1].w += f * o[s][1].w;
                        }
                } else {
                    const float4 *src = reinterpret_cast<const float4 *>(g.a + (size_t)(avalid ? am : 0) * g.lda + kk);
                    av[c][0] = avalid ? src[0] : make_float4(0.f, 0.f, 0.f, 0.f);
                    av[c][1] = avalid ? src[1] : make_float4(0.f, 0.f, 0.f, 0.f);
                }
            } else {
                wr[c].zero();
                av[c][0] = av[c][1] = make_float4(0.f, 0.f, 0.f, 0.f);
            }
        }
        float lw[PRO == CPRO_LN ? WC : 1][8], lb[PRO == CPRO_LN ? WC : 1][8];
        if constexpr (PRO == CPRO_LN) {  // K == 256: one round of two chunks a wave; the loads above are in flight
#pragma unroll
            for (int c = 0; c < WC; ++c) {
                const float4 *wp = reinterpret_cast<const float4 *>(g.ln_w + 32 * (c0 + c) + 8 * grp);
                const float4 *bp = reinterpret_cast<const float4 *>(g.ln_b + 32 * (c0 + c) + 8 * grp);
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    const float4 w = wp[i], b = bp[i];
                    lw[c][4 * i] = w.x, lw[c][4 * i + 1] = w.y, lw[c][4 * i + 2] = w.z, lw[c][4 * i + 3] = w.w;
                    lb[c][4 * i] = b.x, lb[c][4 * i + 1] = b.y, lb[c][4 * i + 2] = b.z, lb[c][4 * i + 3] = b.w;
                }
            }
            // audio_layernorm (audio_layer.cpp:17-28): two-pass mean / variance over 256, eps 1e-5
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const int r = 4 * wave + j, m = m0 + r;
                if (m < g.M) {  // uniform over the wave
                    const float4 x = *reinterpret_cast<const float4 *>(g.a + (size_t)m * g.lda + 4 * lane);
                    const float mean = wave_sum((x.x + x.y) + (x.z + x.w)) / 256.0f;
                    const float d0 = x.x - mean, d1 = x.y - mean, d2 = x.z - mean, d3 = x.w - mean;
                    const float var = wave_sum((d0 * d0 + d1 * d1) + (d2 * d2 + d3 * d3)) / 256.0f;
                    if (lane == 0) rowst[r] = make_float2(mean, 1.0f / sqrtf(var + 1e-5f));
                } else if (lane == 0) {
                    rowst[r] = make_float2(0.f, 0.f);
                }
            }
            lds_barrier();
        }
#pragma unroll
        for (int c = 0; c < WC; ++c) {
            if (c0 + c < c1) {
                float a[8] = {av[c][0].x, av[c][0].y, av[c][0].z, av[c][0].w,
                              av[c][1].x, av[c][1].y, av[c][1].z, av[c][1].w};
                if constexpr (PRO == CPRO_LN) {
                    const float2 rs = rowst[col];
#pragma unroll
                    for (int i = 0; i < 8; ++i) a[i] = avalid ? (a[i] - rs.x) * rs.y * lw[c][i] + lb[c][i] : 0.f;
                } else if constexpr (PRO == CPRO_MERGE) {
#pragma unroll
                    for (int i = 0; i < 8; ++i) a[i] *= inv_den;
                }
                acc0 = mfma4(a[0], wr[c].get(0), acc0);
                acc1 = mfma4(a[1], wr[c].get(1), acc1);
                acc0 = mfma4(a[2], wr[c].get(2), acc0);
                acc1 = mfma4(a[3], wr[c].get(3), acc1);
                acc0 = mfma4(a[4], wr[c].get(4), acc0);
                acc1 = mfma4(a[5], wr[c].get(5), acc1);
                acc0 = mfma4(a[6], wr[c].get(6), acc0);
                acc1 = mfma4(a[7], wr[c].get(7), acc1);
            }
        }
    }
    const floatx4 acc = acc0 + acc1;
#pragma unroll
    for (int i = 0; i < 4; ++i) red[wave][(4 * grp + i) * 16 + col] = acc[i];
    lds_barrier();
    const float v = (red[0][t] + red[1][t]) + (red[2][t] + red[3][t]);
    float partner = 0.f;
    if constexpr (EPI == CEPI_QKV) {
        const int tp = t ^ 1;
        partner = (red[0][tp] + red[1][tp]) + (red[2][tp] + red[3][tp]);
    }
    if (fm < g.M) epi_store<EPI>(g, ein, fm, fn, v, partner);
}

// The same product for pieces with many rows: a workgroup takes 32 MT rows x 32 NT columns,
// its 4 waves 2 x 2 of 16 MT x 16 NT, each over the whole contraction.  What bounds it is the
// fp32 matrix rate (64 flop per SIMD and cycle), so operands come straight from global memory
// -- per 32 columns a wave loads 2 MT + NT vectors for 8 MT NT MFMAs of 32 cycles -- with the next
// chunk in flight.  CPRO_LN (K = 256): the rows are read once, 8 / MT threads a row, normalised
// in registers and kept in LDS (rows of 260 floats: the 16 rows of a 16-byte read fall into
// different banks).  Consecutive workgroups go to different XCDs, so the tiles are numbered
// such that all column tiles of a row tile run on one XCD and its L2 holds their rows.
// (An utterance of 203 frames, with decode()'s long pieces: 6.66 ms in 32-frame pieces of 16 x 16
// tiles, 2.75 ms now.)
template <int PRO, int EPI, int WF32, int MT, int NT>
__global__ __launch_bounds__(256) void codec_tile_kernel(const CodecGemmArgs g, int ntiles, int mtiles) {
    constexpr int kLdA = kCodecDModel + 4;
    __shared__ float as[PRO == CPRO_LN ? 32 * MT : 1][kLdA];
    const int id = blockIdx.x, xcd = id & 7, slot = id >> 3;
    const int mt0 = (slot / ntiles) * 8 + xcd;
    if (mt0 >= mtiles) return;
    const int m0 = mt0 * 32 * MT, n0 = (slot % ntiles) * 32 * NT;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
    const int wm = (wave >> 1) * 16 * MT, wn = n0 + (wave & 1) * 16 * NT;

    size_t woff[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) woff[j] = (size_t)min(wn + 16 * j + col, g.N - 1) * g.K + 8 * grp;
    const float *arow[MT];
#pragma unroll
    for (int i = 0; i < MT; ++i) arow[i] = g.a + (size_t)min(m0 + wm + 16 * i + col, g.M - 1) * g.lda + 8 * grp;

    W8<WF32> wr[2][NT];
    float4 av[2][MT][2];
    auto load = [&](int s, int kk) {
#pragma unroll
        for (int j = 0; j < NT; ++j) wr[s][j].load(g.w, woff[j] + kk);
        if constexpr (PRO != CPRO_LN)
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                const float4 *p = reinterpret_cast<const float4 *>(arow[i] + kk);
                av[s][i][0] = p[0];
                av[s][i][1] = p[1];
            }
    };
    load(0, 0);
    if constexpr (PRO == CPRO_LN) {
        // audio_layernorm (audio_layer.cpp:17-28): two-pass mean / variance over 256, eps 1e-5
        constexpr int TPR = 8 / MT, V = kCodecDModel / 4 / TPR;  // threads and float4s per row
        const int r = t / TPR, q = t % TPR;
        const float4 *src = reinterpret_cast<const float4 *>(g.a + (size_t)min(m0 + r, g.M - 1) * g.lda) + q;
        float4 x[V];
#pragma unroll
        for (int i = 0; i < V; ++i) x[i] = src[TPR * i];
        auto row_sum = [&](float v) {
            v += xshfl<1>(v);
            v += xshfl<2>(v);
            if constexpr (TPR == 8) v += xshfl<4>(v);
            return v;
        };
        float sum = 0.f;
#pragma unroll
        for (int i = 0; i < V; ++i) sum += (x[i].x + x[i].y) + (x[i].z + x[i].w);
        const float mean = row_sum(sum) / 256.0f;
        float sq = 0.f;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            x[i].x -= mean;
            x[i].y -= mean;
            x[i].z -= mean;
            x[i].w -= mean;
            sq += (x[i].x * x[i].x + x[i].y * x[i].y) + (x[i].z * x[i].z + x[i].w * x[i].w);
        }
        const float inv = 1.0f / sqrtf(row_sum(sq) / 256.0f + 1e-5f);
        const float4 *lw = reinterpret_cast<const float4 *>(g.ln_w) + q, *lb = reinterpret_cast<const float4 *>(g.ln_b) + q;
#pragma unroll
        for (int i = 0; i < V; ++i) {
            const float4 w = lw[TPR * i], b = lb[TPR * i];
            *reinterpret_cast<float4 *>(&as[r][4 * (q + TPR * i)]) =
                make_float4(x[i].x * inv * w.x + b.x, x[i].y * inv * w.y + b.y, x[i].z * inv * w.z + b.z,
                            x[i].w * inv * w.w + b.w);
        }
        lds_barrier();
    }

    // sums of 64 columns at a time in two chains (even and odd columns), then those: the chains
    // of the 16 x 16 tile's waves are no longer (one chain over K = 1024 measured twice their
    // error after all layers, 7e-7 against 4e-7, one chain per 64 columns 4.4e-7)
    floatx4 acc[2][MT][NT], tot[MT][NT];
    auto clear = [](floatx4 (&v)[MT][NT]) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) v[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};
    };
    auto flush = [&] {
#pragma unroll
        for (int i = 0; i < MT; ++i)
#pragma unroll
            for (int j = 0; j < NT; ++j) tot[i][j] += acc[0][i][j] + acc[1][i][j];
        clear(acc[0]);
        clear(acc[1]);
    };
    clear(acc[0]);
    clear(acc[1]);
    clear(tot);
    auto step = [&](int s, int kk) {
        float a[MT][8];
#pragma unroll
        for (int i = 0; i < MT; ++i) {
            float4 x0, x1;
            if constexpr (PRO == CPRO_LN) {
                const float4 *p = reinterpret_cast<const float4 *>(&as[wm + 16 * i + col][kk + 8 * grp]);
                x0 = p[0];
                x1 = p[1];
            } else {
                x0 = av[s][i][0];
                x1 = av[s][i][1];
            }
            a[i][0] = x0.x;
            a[i][1] = x0.y;
            a[i][2] = x0.z;
            a[i][3] = x0.w;
            a[i][4] = x1.x;
            a[i][5] = x1.y;
            a[i][6] = x1.z;
            a[i][7] = x1.w;
        }
#pragma unroll
        for (int k = 0; k < 8; ++k)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = 0; j < NT; ++j) acc[k & 1][i][j] = mfma4(a[i][k], wr[s][j].get(k), acc[k & 1][i][j]);
    };
    int kk = 0;
    for (; kk + 64 <= g.K; kk += 64) {
        load(1, kk + 32);
        step(0, kk);
        if (kk + 64 < g.K) load(0, kk + 64);
        step(1, kk + 32);
        flush();
    }
    if (kk < g.K) {  // K an odd number of chunks
        step(0, kk);
        flush();
    }

    EpiIn ein[MT][4][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int j = 0; j < NT; ++j)
                ein[i][e][j] = epi_load<EPI>(g, min(m0 + wm + 16 * i + 4 * grp + e, g.M - 1), min(wn + 16 * j + col, g.N - 1));
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int m = m0 + wm + 16 * i + 4 * grp + e;
#pragma unroll
            for (int j = 0; j < NT; ++j) {
                const int nn = wn + 16 * j + col;
                const float v = tot[i][j][e];
                const float partner = EPI == CEPI_QKV ? xshfl<1>(v) : 0.f;
                if (m < g.M && nn < g.N) epi_store<EPI>(g, ein[i][e][j], m, nn, v, partner);
            }
        }
}

// Windowed causal attention of 16 query rows x one head over the ring's keys
// (attention_window_avx2, attn_avx2.cpp:93-204): key position kp is visible to the
// query at position qp iff 0 <= qp - kp < window.  Grid (row tiles, heads, splits):
// split z takes a contiguous share of the tile's 16-key blocks, its WV waves every WVth
// block of it, each with a running max / sum (online softmax); the waves merge in LDS
// and the split writes its unnormalised output and (max, sum) for the proj GEMM's
// merge prologue.
//   S^T = K Q^T: A = K[key kb + l%16][16g + t], B = Q[q l%16][16g + t], t = 0..15
//   O^T = V^T P^T per 4-column group j: A = V[key kb + 4g + s][4(l%16) + j], B = P[q][kb + 4g + s]
// so the lane with q = l%16 holds S^T for keys kb + 4g + i and O for columns 16g..16g+15.
//
// Many unsplit tiles (XCD) are a linear grid: workgroups go to the 8 XCDs in turn and within one to
// its 32 CUs in turn, so an XCD works on every other tile of one head, whose keys its L2 keeps, and
// its tiles go out longest first (an utterance's first rows see few keys), every other round of
// 32 backwards, so that a CU which drew a long tile draws a short one next.
// With two register sets for the keys in turn and no division a key, a 203-frame utterance spends
// 0.80 ms here, 1.13 before.
template <int WV, bool XCD>
__global__ __launch_bounds__(64 * WV) void codec_attn_kernel(const CodecAttnArgs a) {
    // a wave's rows, 68 floats apart (16-byte reads and writes fall into different banks), then
    // their maxima and sums
    constexpr int kRow = kCodecHeadDim + 4, kStat = 16 * kRow;
    __shared__ __align__(16) float red[WV][kStat + 32];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6, col = lane & 15, grp = lane >> 4;
    int tile = blockIdx.x, h = blockIdx.y;
    if constexpr (XCD) {
        const int xcd = blockIdx.x & 7, at = blockIdx.x >> 3, n = gridDim.x >> 3;
        const int row = at >> 5, in_row = min(32, n - 32 * row);
        const int rank = 32 * row + ((row & 1) ? in_row - 1 - (at & 31) : at & 31);
        h = xcd >> 1;
        tile = ((a.M + 15) >> 4) - 1 - 2 * rank - (xcd & 1);
        if (tile < 0) return;  // uniform (an odd number of tiles)
    }
    const int m0 = tile * 16, split = blockIdx.z;
    const int P0 = *a.pos0;
    const int mlast = min(m0 + 15, a.M - 1);
    const int klo = max(0, P0 + m0 - a.window + 1), khi = P0 + mlast;
    const int nkb = (khi - klo + 16) >> 4;
    const int per = (nkb + a.splits - 1) / a.splits;
    const int b0 = split * per, b1 = min(nkb, b0 + per);
    const int mq = m0 + col, qpos = P0 + mq;
    const bool qvalid = mq < a.M;
    const int hoff = h * kCodecHeadDim;

    float qv[16];
    {
        const float4 *src = reinterpret_cast<const float4 *>(a.q + (size_t)(qvalid ? mq : 0) * kCodecDModel + hoff + 16 * grp);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = qvalid ? src[i] : make_float4(0.f, 0.f, 0.f, 0.f);
            qv[4 * i] = v.x;
            qv[4 * i + 1] = v.y;
            qv[4 * i + 2] = v.z;
            qv[4 * i + 3] = v.w;
        }
    }
    float mrun = -INFINITY, lrun = 0.f;
    floatx4 o[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) o[j] = floatx4{0.f, 0.f, 0.f, 0.f};

    // block b's operands: K rows kb + l%16 (this lane's 16 columns of the head), V rows
    // kb + 4g + s (4 columns); keys past khi read as key khi (their scores are masked)
    // the ring slot of key klo + i (i < ring: the ring holds the window and the piece)
    const int slot0 = klo % a.ring, span = khi - klo;
    auto slot = [&](int i) {
        const int s = slot0 + min(i, span);
        return (size_t)(s < a.ring ? s : s - a.ring) * kCodecDModel;
    };
    auto load_block = [&](int b, float (&kv)[16], float4 (&vv)[4]) {
        const float4 *src = reinterpret_cast<const float4 *>(a.kc + slot(16 * b + col) + hoff + 16 * grp);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const float4 v = src[i];
            kv[4 * i] = v.x;
            kv[4 * i + 1] = v.y;
            kv[4 * i + 2] = v.z;
            kv[4 * i + 3] = v.w;
        }
#pragma unroll
        for (int s = 0; s < 4; ++s)
            vv[s] = *reinterpret_cast<const float4 *>(a.vc + slot(16 * b + 4 * grp + s) + hoff + 4 * col);
    };
    auto block = [&](int b, const float (&kv)[16], const float4 (&vv)[4]) {
        const int kb = klo + 16 * b;
        floatx4 sc0 = {0.f, 0.f, 0.f, 0.f}, sc1 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 16; i += 2) {
            sc0 = mfma4(kv[i], qv[i], sc0);
            sc1 = mfma4(kv[i + 1], qv[i + 1], sc1);
        }
        const floatx4 sc = sc0 + sc1;
        float p[4], bmax = -INFINITY;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int kp = kb + 4 * grp + i;
            const bool vis = qvalid && kp <= qpos && qpos - kp < a.window;
            p[i] = vis ? sc[i] * 0.125f : -INFINITY;  // 1/sqrt(64)
            bmax = fmaxf(bmax, p[i]);
        }
        bmax = fmaxf(bmax, xshfl<16>(bmax));
        bmax = fmaxf(bmax, xshfl<32>(bmax));
        const float mnew = fmaxf(mrun, bmax);
        const float msafe = mnew == -INFINITY ? 0.f : mnew;
        const float alpha = exp_f(mrun - msafe);
#pragma unroll
        for (int i = 0; i < 4; ++i) p[i] = exp_f(p[i] - msafe);
        lrun = lrun * alpha + ((p[0] + p[1]) + (p[2] + p[3]));
        mrun = mnew;
#pragma unroll
        for (int j = 0; j < 4; ++j) o[j] *= alpha;
#pragma unroll
        for (int s = 0; s < 4; ++s) {
            o[0] = mfma4(vv[s].x, p[s], o[0]);
            o[1] = mfma4(vv[s].y, p[s], o[1]);
            o[2] = mfma4(vv[s].z, p[s], o[2]);
            o[3] = mfma4(vv[s].w, p[s], o[3]);
        }
    };
    // the wave's next block is in flight while one is computed, in the other of two register
    // sets; a request past the last block reads the last key again
    float k0[16], k1[16];
    float4 v0[4], v1[4];
    if (b0 + wave < b1) load_block(b0 + wave, k0, v0);
    for (int b = b0 + wave; b < b1; b += 2 * WV) {
        load_block(b + WV, k1, v1);
        block(b, k0, v0);
        if (b + WV >= b1) break;
        load_block(b + 2 * WV, k0, v0);
        block(b + WV, k1, v1);
    }
    lrun += xshfl<16>(lrun);
    lrun += xshfl<32>(lrun);
    // lane (grp, col) holds O[q col][16 grp + 4 i + j] = o[j][i]: rows of the head in LDS
    float *R = red[wave];
#pragma unroll
    for (int i = 0; i < 4; ++i)
        *reinterpret_cast<float4 *>(&R[col * kRow + 16 * grp + 4 * i]) = make_float4(o[0][i], o[1][i], o[2][i], o[3][i]);
    if (grp == 0) {
        R[kStat + col] = mrun;
        R[kStat + 16 + col] = lrun;
    }
    lds_barrier();
    constexpr int E = 16 / WV, TR = 64 / E;  // columns a thread finishes, threads a row
    const int q = t / TR, d = E * (t % TR), m = m0 + q;
    if (m >= a.M) return;
    float mx = -INFINITY;
#pragma unroll
    for (int w = 0; w < WV; ++w) mx = fmaxf(mx, red[w][kStat + q]);
    const float msafe = mx == -INFINITY ? 0.f : mx;
    float l = 0.f, acc[E] = {};
#pragma unroll
    for (int w = 0; w < WV; ++w) {
        const float f = exp_f(red[w][kStat + q] - msafe);
        l += f * red[w][kStat + 16 + q];
        float r[E];
        if constexpr (E == 4)
            *reinterpret_cast<float4 *>(r) = *reinterpret_cast<const float4 *>(&red[w][q * kRow + d]);
        else
            *reinterpret_cast<float2 *>(r) = *reinterpret_cast<const float2 *>(&red[w][q * kRow + d]);
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] += f * r[e];
    }
    if (a.splits == 1) {
        const float inv = 1.0f / l;
#pragma unroll
        for (int e = 0; e < E; ++e) acc[e] *= inv;
    }
    const size_t row = (size_t)split * a.M + m;
    float *out = a.o + row * kCodecDModel + hoff + d;
    if constexpr (E == 4)
        *reinterpret_cast<float4 *>(out) = make_float4(acc[0], acc[1], acc[2], acc[3]);
    else
        *reinterpret_cast<float2 *>(out) = make_float2(acc[0], acc[1]);
    if (d == 0 && a.splits > 1) a.st[row * kCodecHeads + h] = make_float2(mx, l);
}

// Workgroup t < frames: z[t][r] = sum_i (b_i[r] + sum_k W_i[r][k] cb_i[code_it][k]), i in order
// (decoder.cpp:224-240); the 16 quantizers' loads are all in flight together (one after the
// other: 9.1 us).  The workgroups after those: cos and sin of every stage's positions, which
// each layer's q and k then read (sincosf per element of every QKV launch before).
__global__ __launch_bounds__(512) void codec_front_kernel(const CodecFrontArgs a) {
    if ((int)blockIdx.x >= a.frames) {
        int e = ((int)blockIdx.x - a.frames) * 512 + threadIdx.x;  // entry: stage, row, frequency
        const int f = e & 31;
        e >>= 5;
#pragma unroll
        for (int s = 0; s < kCodecStages; ++s) {
            if (e < a.rows[s]) {
                float sn, cs;
                sincosf((float)(a.pos0[s] + e) * a.freq[f], &sn, &cs);
                a.rope[s][(size_t)e * 32 + f] = make_float2(cs, sn);
                return;
            }
            e -= a.rows[s];
        }
        return;
    }
    const int t = blockIdx.x, r = threadIdx.x;
    float4 e0[kCodecNq], e1[kCodecNq], w0[kCodecNq], w1[kCodecNq];
    float b[kCodecNq];
#pragma unroll
    for (int i = 0; i < kCodecNq; ++i) {
        const int code = a.codes[(size_t)i * a.code_stride + t];
        const float4 *e = reinterpret_cast<const float4 *>(a.cb[i] + (size_t)code * kCodecCbDim);
        const float4 *w = reinterpret_cast<const float4 *>(a.cw[i] + (size_t)r * kCodecCbDim);
        e0[i] = e[0];
        e1[i] = e[1];
        w0[i] = w[0];
        w1[i] = w[1];
        b[i] = a.cbias[i][r];
    }
    float z = 0.f;
#pragma unroll
    for (int i = 0; i < kCodecNq; ++i) {
        float acc = b[i];
        acc += w0[i].x * e0[i].x;
        acc += w0[i].y * e0[i].y;
        acc += w0[i].z * e0[i].z;
        acc += w0[i].w * e0[i].w;
        acc += w1[i].x * e1[i].x;
        acc += w1[i].y * e1[i].y;
        acc += w1[i].z * e1[i].z;
        acc += w1[i].w * e1[i].w;
        z += acc;
    }
    a.z[(size_t)t * kCodecZ + r] = z;
}

struct Rows4 {
    int r[kCodecStages];
};

__global__ void codec_advance_kernel(int *pos0, Rows4 rows) {
    if (threadIdx.x < kCodecStages) pos0[threadIdx.x] += rows.r[threadIdx.x];
}

// Tiles of 64 x 64, or else 32 x 32, from this many of them on: about one per CU, so that the chip
// fills before a workgroup's own time grows.  Launches of one utterance in tiles of 16, 32 and 64 (us; N x K):
//   768 x 256 (QKV):  224 rows 8.6, 6.7, 12.1; 352 11.6, 7.4, 12.1; 832 19.3, 10.2, 12.4;
//                     1024 22.4, 10.4, 12.9; 1792 35.3, 16.7, 18.3; 3328 59.2, 26.3, 26.7
//   1024 x 256 (f1):  224 rows 11.1, 7.0, 12.8; 640 19.3, 10.1, 13.4; 768 22.0, 10.2, 13.6; 3328 74.7, 32.3, 34.3
//   256 x 1024 (f2):  1024 rows 14.2, 14.9, 29.3; 1152 16.6, 23.1, 29.4; 1664 21.8, 23.1, 29.5;
//                     2560 29.9, 33.8, 29.9; 3328 37.6, 45.0, 30.4
//   256 x 256 (proj): 896 rows 7.9, 7.8, 8.0; 1152 6.9, 7.8, 10.0; 1664 8.4, 8.0, 10.1; 2816 12.4, 10.5, 10.3
// By them one line for all shapes is a compromise: 32 x 32 is already ahead at 120 tiles and still at
// 1300 for the two wide products, and a long K does better in 16 x 16 until 64 x 64 fill the chip.
constexpr long kTile64Min = 192, kTile32Min = 256;

template <int PRO, int EPI, int MT, int NT>
void launch_tile(const CodecGemmArgs &g, hipStream_t s) {
    const int mt = (g.M + 32 * MT - 1) / (32 * MT), nt = (g.N + 32 * NT - 1) / (32 * NT);
    const dim3 grid(8 * nt * ((mt + 7) / 8));
    if (g.w_f32)
        hipLaunchKernelGGL((codec_tile_kernel<PRO, EPI, 1, MT, NT>), grid, dim3(256), 0, s, g, nt, mt);
    else
        hipLaunchKernelGGL((codec_tile_kernel<PRO, EPI, 0, MT, NT>), grid, dim3(256), 0, s, g, nt, mt);
}

template <int PRO, int EPI>
int launch_w(const CodecGemmArgs &g, hipStream_t s) {
    (void)hipGetLastError();  // report only this launch's error, not a stale one
    if constexpr (PRO != CPRO_MERGE) {
        const long tiles64 = (long)((g.M + 63) / 64) * ((g.N + 63) / 64), tiles32 = (long)((g.M + 31) / 32) * ((g.N + 31) / 32);
        if (tiles64 >= kTile64Min) {
            launch_tile<PRO, EPI, 2, 2>(g, s);
            return hipGetLastError() == hipSuccess ? 0 : MOSS_HIP_EDEVICE;
        }
        if (tiles32 >= kTile32Min) {
            launch_tile<PRO, EPI, 1, 1>(g, s);
            return hipGetLastError() == hipSuccess ? 0 : MOSS_HIP_EDEVICE;
        }
    }
    const dim3 grid(g.N / 16, (g.M + 15) / 16);
    if (g.w_f32)
        hipLaunchKernelGGL((codec_gemm_kernel<PRO, EPI, 1>), grid, dim3(256), 0, s, g);
    else
        hipLaunchKernelGGL((codec_gemm_kernel<PRO, EPI, 0>), grid, dim3(256), 0, s, g);
    return hipGetLastError() == hipSuccess ? 0 : MOSS_HIP_EDEVICE;
}

}  // namespace

int codec_gemm_launch(int pro, int epi, const CodecGemmArgs &g, hipStream_t s) {
    if (g.M <= 0 || g.N <= 0 || g.K <= 0 || g.N % 16 || g.K % 32 || (!g.a && pro != CPRO_MERGE) || !g.w)
        return MOSS_HIP_EINVAL;
    if ((pro == CPRO_LN || pro == CPRO_MERGE) && g.K != kCodecDModel) return MOSS_HIP_EINVAL;
    if (pro == CPRO_ROWS && (g.lda % 4 || g.lda < g.K)) return MOSS_HIP_EINVAL;
    if (pro == CPRO_MERGE && (!g.o || !g.st || g.splits < 1 || g.splits > kCodecMaxSplits)) return MOSS_HIP_EINVAL;
    if (epi == CEPI_QKV && (g.N != 3 * kCodecDModel || !g.q || !g.kc || !g.vc || g.ring <= 0 || !g.pos0 || !g.rope))
        return MOSS_HIP_EINVAL;
    if (epi == CEPI_STORE && (g.patch < 1 || g.N % g.patch)) return MOSS_HIP_EINVAL;
    if (epi == CEPI_RESID && !g.ls) return MOSS_HIP_EINVAL;
    switch (pro * 4 + epi) {
        case CPRO_ROWS * 4 + CEPI_STORE: return launch_w<CPRO_ROWS, CEPI_STORE>(g, s);
        case CPRO_ROWS * 4 + CEPI_RESID: return launch_w<CPRO_ROWS, CEPI_RESID>(g, s);
        case CPRO_LN * 4 + CEPI_QKV: return launch_w<CPRO_LN, CEPI_QKV>(g, s);
        case CPRO_LN * 4 + CEPI_GELU: return launch_w<CPRO_LN, CEPI_GELU>(g, s);
        case CPRO_MERGE * 4 + CEPI_RESID: return launch_w<CPRO_MERGE, CEPI_RESID>(g, s);
        default: return MOSS_HIP_EUNSUPPORTED;
    }
}

int codec_attn_launch(const CodecAttnArgs &a, hipStream_t s) {
    (void)hipGetLastError();  // report only this launch's error, not a stale one
    if (a.M <= 0 || a.splits < 1 || a.window <= 0 || a.ring <= 0 || !a.q || !a.kc || !a.vc || !a.pos0 || !a.o || !a.st)
        return MOSS_HIP_EINVAL;
    const int tiles = (a.M + 15) / 16;
    static_assert(kCodecHeads == 4, "two XCDs a head");
    // more than one workgroup per CU: tiles by XCD and length, 4 waves (1024 rows, 256 workgroups: 17.2 us,
    // 16.5 in order with 8 waves; 1152 rows 20.0 and 21.4, 1664 24.8 and 32.3, 3328 55.8 and 68.2)
    if (a.splits == 1 && tiles * kCodecHeads > 256)
        hipLaunchKernelGGL((codec_attn_kernel<4, true>), dim3(8 * ((tiles + 1) / 2)), dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((codec_attn_kernel<8, false>), dim3(tiles, kCodecHeads, a.splits), dim3(512), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : MOSS_HIP_EDEVICE;
}

int codec_front_launch(const CodecFrontArgs &a, hipStream_t s) {
    (void)hipGetLastError();  // report only this launch's error, not a stale one
    if (a.frames <= 0 || !a.codes || !a.z || a.code_stride < a.frames || !a.pos0 || !a.freq) return MOSS_HIP_EINVAL;
    long rows = 0;
    for (int i = 0; i < kCodecStages; ++i) {
        if (a.rows[i] <= 0 || !a.rope[i]) return MOSS_HIP_EINVAL;
        rows += a.rows[i];
    }
    const dim3 grid(a.frames + (unsigned)((rows * 32 + 511) / 512));
    hipLaunchKernelGGL(codec_front_kernel, grid, dim3(kCodecZ), 0, s, a);
    return hipGetLastError() == hipSuccess ? 0 : MOSS_HIP_EDEVICE;
}

int codec_advance_launch(int *pos0, const int *rows, hipStream_t s) {
    (void)hipGetLastError();  // report only this launch's error, not a stale one
    Rows4 r;
    for (int i = 0; i < kCodecStages; ++i) r.r[i] = rows[i];
    hipLaunchKernelGGL(codec_advance_kernel, dim3(1), dim3(64), 0, s, pos0, r);
    return hipGetLastError() == hipSuccess ? 0 : MOSS_HIP_EDEVICE;
}

}  // namespace mh
