// gemm_tile.hip -- the W8A16 / W8A8 GEMM for many rows: 64 x 64 tiles, the activations
// staged in LDS.
//
// The same products and the same sums as gemm_mfma.hip (per scale block a 32-deep MFMA, times
// the block scale, accumulated in fp32; K in 4 runs of blocks, added in order), so the results
// are the same bits.  There a workgroup owns 16 rows: a weight is read, widened and scaled again
// for every 16 rows, and at 1000 rows 2268 workgroups pull 226 MB through the L2s for one QKV
// product.  Here a wave owns 64 rows x 16 columns: a weight is widened once per 64 rows, and the
// rows come from LDS, where the workgroup's four waves put them once.  What bounds it is the
// instructions of a wave (per 16 x 16 x 32 product 2 MFMAs and 4 FMAs with the block scale, and
// the widening): tiles of 64 x 128 and 64 x 192 with 4 or 8 waves, which read less again, measured
// 19.5 to 26 us where this takes 19.0 (QKV, 1000 rows, A16; 22.8 in 16-row tiles).  The 1000-row A16
// prefill went from 1.82 to 1.67 ms.
#include "mh_gemm.h"

namespace mh {
namespace {

constexpr int TM = 64, TN = 64;
constexpr int kOutStride = TN + 4;  // floats from one row of the finished tile in LDS to the next
// the runs of blocks that are summed apart and then in order: gemm_mfma.hip's waves
constexpr int kRuns = 4;

// scale blocks per staged chunk: divides every run of blocks of the model's products
// (K = 768: 6 a run)
constexpr int KB = 2;
template <bool A8>
constexpr int kChunkBytes = KB * 4 * (A8 ? 512 + 64 : 2048);  // W8A8: the quants, then the scales as [block][row]
// register sets a wave streams chunks through: one chunk in LDS and its weights here, three
// more in flight (a chunk is ~0.15 us of work, a load ~0.6 us)
constexpr int kSets = 4;

constexpr int kPastEnd = 0x40000000;  // operands are smaller (tile_gemm_fits)

template <bool A8>
struct TileSrc {
    rsrc_t a, ad, w;
    int va, vad;  // staging: this lane's activations (and scale) at block 0
    int vw, vs;   // this lane's weights and scale
};

// A lane's share of a chunk of activations on the way to LDS: the wave stages 16 rows, the
// lane the 8 columns it would hold as an MFMA operand.
template <bool A8, bool AT>
struct StageA {
    floatx4 x[A8 ? 1 : KB][2];  // fp32 columns 0..3, 4..7, or the hi and lo halves
    uint2 q[A8 ? KB : 1];
    uint32_t d;  // the scale of row lane % 16 in block lane / 16 % 2
};

template <bool A8>
struct ChunkW {
    uint2 q[KB];
    uint32_t d[KB];
};

template <bool A8, bool AT>
__device__ __forceinline__ void load_a(StageA<A8, AT> &c, int b0, int off, const TileSrc<A8> &s) {
#pragma unroll
    for (int j = 0; j < KB; ++j) {
        if constexpr (A8) {
            constexpr int QB = AT ? 512 : 32;
            const auto q = __builtin_amdgcn_raw_buffer_load_b64(s.a, s.va + off + QB * j, QB * b0, 0);
            c.q[j] = make_uint2(q[0], q[1]);
        } else {
            constexpr int XB = AT ? 2048 : 128, XH = AT ? 1024 : 16;
            c.x[j][0] = __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(s.a, s.va + off + XB * j, XB * b0, 0));
            c.x[j][1] =
                __builtin_bit_cast(floatx4, __builtin_amdgcn_raw_buffer_load_b128(s.a, s.va + off + XB * j + XH, XB * b0, 0));
        }
    }
    if constexpr (A8) c.d = __builtin_amdgcn_raw_buffer_load_b32(s.ad, s.vad + off, (AT ? 64 : 4) * b0, 0);
}

template <bool A8, bool TL>
__device__ __forceinline__ void load_w(ChunkW<A8> &c, int b0, int off, const TileSrc<A8> &s) {
    constexpr int UB = TL ? kTileBytes : kBlockBytes;
#pragma unroll
    for (int j = 0; j < KB; ++j) {
        const auto q = __builtin_amdgcn_raw_buffer_load_b64(s.w, s.vw + off + UB * j, UB * b0, 0);
        c.q[j] = make_uint2(q[0], q[1]);
        c.d[j] = __builtin_amdgcn_raw_buffer_load_b16(s.w, s.vs + off + UB * j, UB * b0, 0);
    }
}

// One chunk of activations into LDS, per block and 16 rows in the matrix-core order (a wave
// writes and later reads 64 consecutive 16- or 8-byte runs: no bank conflicts), the W8A8
// block scales behind them as [block][row].
template <bool A8, bool AT>
__device__ __forceinline__ void stage_a(const StageA<A8, AT> &c, uint8_t *buf, int sr, int lane) {
#pragma unroll
    for (int j = 0; j < KB; ++j) {
        if constexpr (A8) {
            *reinterpret_cast<uint2 *>(buf + (j * 4 + sr) * 512 + 8 * lane) = c.q[j];
        } else {
            half8 hi, lo;
            if constexpr (AT) {
                hi = __builtin_bit_cast(half8, c.x[j][0]);
                lo = __builtin_bit_cast(half8, c.x[j][1]);
            }
            if constexpr (!AT) {
                float x[8];
#pragma unroll
                for (int i = 0; i < 8; ++i) x[i] = c.x[j][i >> 2][i & 3];
                split_hi_lo(x, hi, lo);
            }
            uint8_t *u = buf + (j * 4 + sr) * 2048 + 16 * lane;
            *reinterpret_cast<half8 *>(u) = hi;
            *reinterpret_cast<half8 *>(u + 1024) = lo;
        }
    }
    if constexpr (A8) {
        *reinterpret_cast<uint32_t *>(buf + KB * 2048 + ((lane >> 4) & 1) * 256 + 4 * (16 * sr + (lane & 15))) = c.d;
    }
}

// Block j of a chunk: the 4 row subtiles times the wave's 16 columns.
template <bool A8>
__device__ __forceinline__ void mma_block(const uint8_t *buf, int j, int lane, const ChunkW<A8> &c, floatx4 (&acc)[4]) {
#pragma clang fp contract(off)
    const float d = h2f((uint16_t)c.d[j]);
    if constexpr (A8) {
        const floatx4 *da = reinterpret_cast<const floatx4 *>(buf + KB * 2048 + j * 256) + (lane >> 4);
        const long bq = (long)(((uint64_t)c.q[j].y << 32) | c.q[j].x);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const long aq = *reinterpret_cast<const long *>(buf + (j * 4 + r) * 512 + 8 * lane);
            const floatx4 ad = da[4 * r];  // rows 16 r + 4 (lane / 16) + i
            const intx4 p = __builtin_amdgcn_mfma_i32_16x16x32_i8(aq, bq, intx4{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float scale = d * ad[i];
                acc[r][i] = fmaf((float)p[i], scale, acc[r][i]);
            }
        }
    } else {
        const half8 bw = i8x8_to_h8(c.q[j]);
        floatx4 blk[4];
        half8 lo[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint8_t *u = buf + (j * 4 + r) * 2048 + 16 * lane;
            const half8 hi = *reinterpret_cast<const half8 *>(u);
            lo[r] = *reinterpret_cast<const half8 *>(u + 1024);
            blk[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(hi, bw, floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
        }
#pragma unroll
        for (int r = 0; r < 4; ++r) blk[r] = __builtin_amdgcn_mfma_f32_16x16x32_f16(lo[r], bw, blk[r], 0, 0, 0);
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[r][i] = fmaf(blk[r][i], d, acc[r][i]);
    }
}

__device__ __forceinline__ void load8(float (&v)[8], const float *p) {
    const float4 a = reinterpret_cast<const float4 *>(p)[0], b = reinterpret_cast<const float4 *>(p)[1];
    v[0] = a.x, v[1] = a.y, v[2] = a.z, v[3] = a.w;
    v[4] = b.x, v[5] = b.y, v[6] = b.z, v[7] = b.w;
}
__device__ __forceinline__ void store8(float *p, const float (&v)[8]) {
    reinterpret_cast<float4 *>(p)[0] = make_float4(v[0], v[1], v[2], v[3]);
    reinterpret_cast<float4 *>(p)[1] = make_float4(v[4], v[5], v[6], v[7]);
}
// 8 columns from k (a multiple of 8) of row m as hi / lo halves (hlt_at)
__device__ __forceinline__ void store8_hl(uint8_t *hl, int m, int k, int K, const float (&v)[8]) {
    half8 hi, lo;
    split_hi_lo(v, hi, lo);
    uint8_t *u = hl + hlt_at(m, k, K);
    *reinterpret_cast<half8 *>(u) = hi;
    *reinterpret_cast<half8 *>(u + 1024) = lo;
}

// What the epilogue looks up for a row, requested when the workgroup starts.
struct RowInfo {
    int pos = 0;
    size_t slot = 0;  // EPI_QKV: the row's K/V slot of head 0, in values
    bool kv = false;  // EPI_QKV: K and V are written
};

template <int EPI>
__device__ __forceinline__ RowInfo row_info(const GemmArgs &g, int m) {
    RowInfo r;
    if constexpr (EPI == EPI_QKV) {
        r.pos = g.row_pos ? g.row_pos[m] : g.pos0 + m * g.pos_stride;
        const int s = g.row_stream ? g.row_stream[m] : m * g.stream_stride;
        const int page = g.page_table ? g.page_table[(size_t)s * g.table_stride + r.pos / g.page_size] : s;
        r.slot = ((size_t)page * kHeads * g.page_size + r.pos % g.page_size) * kHeadDim;
        r.kv = g.row_active == nullptr || g.row_active[m];
    }
    return r;
}

// The epilogue's operands of 8 columns of a row.
template <int EPI>
struct Ops8 {
    float b[EPI == EPI_GELU || EPI == EPI_QKV ? 8 : 1];
    float4 c, s;  // EPI_QKV: RoPE factors of the 4 pairs
};

template <int EPI>
__device__ __forceinline__ void ops_load(Ops8<EPI> &o, const GemmArgs &g, const RowInfo &ri, int n) {
    if constexpr (EPI == EPI_GELU || EPI == EPI_QKV) load8(o.b, g.bias + n);
    if constexpr (EPI == EPI_QKV) {
        const size_t at = (size_t)ri.pos * kRopeHalf + ((n & 63) >> 1);
        o.c = *reinterpret_cast<const float4 *>(g.rope_cos + at);
        o.s = *reinterpret_cast<const float4 *>(g.rope_sin + at);
    }
}

// Columns n .. n + 7 of row m finished: gemm_finish's arithmetic (gemm_mfma.hip), 8 at a
// time.  `live` is m < M: the other lanes take part in the exchanges and store nothing.
template <int EPI, int KV>
__device__ __forceinline__ void finish8(const GemmArgs &g, const Ops8<EPI> &o, const RowInfo &ri, int m, int n, bool live, float (&v)[8]) {
#pragma clang fp contract(off)
    if constexpr (EPI == EPI_F32) {
        if (live) store8(g.y + (size_t)m * g.ldy + n, v);
    } else if constexpr (EPI == EPI_GELU) {
        float h[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) h[e] = gelu_new(v[e] + o.b[e]);
        if (g.q8_out != nullptr) {  // uniform: a 32-block is the 4 lanes of a row (quant_block32's arithmetic)
            float amax = 0.0f;
#pragma unroll
            for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf(h[e]));
            amax = fmaxf(amax, xshfl<16>(amax));
            amax = fmaxf(amax, xshfl<32>(amax));
            const float d = amax / 127.0f;
            const float id = d > 0.0f ? 1.0f / d : 0.0f;
            uint32_t w[2] = {0, 0};
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                int q = (int)rintf(h[e] * id);
                q = q < -127 ? -127 : (q > 127 ? 127 : q);
                w[e >> 2] |= (uint32_t)(uint8_t)q << (8 * (e & 3));
            }
            if (live) {
                *reinterpret_cast<uint2 *>(g.q8_out + q8t_at(m, n, g.N)) = make_uint2(w[0], w[1]);
                if ((n & 31) == 0) g.d8_out[d8t_at(m, n >> 5, g.N)] = d;
                if (g.y != nullptr) store8(g.y + (size_t)m * g.ldy + n, h);
            }
        } else if (live) {
            if (g.y_hl != nullptr)
                store8_hl(g.y_hl, m, n, g.N, h);
            else
                store8(g.y + (size_t)m * g.ldy + n, h);
        }
    } else {  // EPI_QKV: 8 columns lie in one head of one section (q, k or v)
        const int sec = n / kHidden;
        float out[8];
        const float c[4] = {o.c.x, o.c.y, o.c.z, o.c.w}, sn[4] = {o.s.x, o.s.y, o.s.z, o.s.w};
#pragma unroll
        for (int e = 0; e < 8; e += 2) {
            const float v0 = v[e] + o.b[e], v1 = v[e + 1] + o.b[e + 1];
            if (sec < 2) {
                const float p0 = v0 * c[e >> 1], p1 = v1 * sn[e >> 1];
                const float r0 = v1 * c[e >> 1], r1 = v0 * sn[e >> 1];
                out[e] = p0 - p1;
                out[e + 1] = r0 + r1;
            } else {
                out[e] = v0;
                out[e + 1] = v1;
            }
        }
        if (!live) return;
        if (sec == 0) {
            store8(g.q_out + (size_t)m * kHidden + n, out);
        } else if (ri.kv) {
            const size_t at = ri.slot + (size_t)((n - sec * kHidden) >> 6) * g.page_size * kHeadDim + (n & 63);
            void *pool = sec == 1 ? g.k_pool : g.v_pool;
            if constexpr (KV == KV_F16) {
                uint32_t w[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) w[e] = (uint32_t)f2h(out[2 * e]) | (uint32_t)f2h(out[2 * e + 1]) << 16;
                *reinterpret_cast<uint4 *>((__half *)pool + at) = make_uint4(w[0], w[1], w[2], w[3]);
            } else {
                store8((float *)pool + at, out);
            }
        }
    }
}

template <int EPI, int KV, bool A8, bool TL, bool AT>
__global__ __launch_bounds__(256, 3) void gemm_tile_kernel(GemmArgs g) {
    constexpr int CB = kChunkBytes<A8>;
    constexpr int kSmem = 2 * CB > 4 * TM * kOutStride ? 2 * CB : 4 * TM * kOutStride;
    __shared__ __align__(16) uint8_t smem[kSmem];
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int l16 = lane & 15, kq = lane >> 4;
    const int m_base = blockIdx.y * TM, n_base = blockIdx.x * TN;
    const int nb = g.K >> 5;
    const int m = m_base + 16 * wave + l16;  // the row this lane stages and finishes
    const int srow = min(m, g.M - 1);        // rows past M read row M-1, never stored
    const RowInfo ri = row_info<EPI>(g, srow);
    TileSrc<A8> src;
    {
        const uint32_t a_elems = (uint32_t)((g.M - 1) * g.lda + g.K);
        if constexpr (AT) {  // rows padded to 16: a unit past the last row tile reads 0
            const uint32_t units = (uint32_t)((g.M + 15) / 16) * (uint32_t)nb;
            const int unit = (m_base / 16 + wave) * nb;
            src.a = make_rsrc(A8 ? (const void *)g.a8 : (const void *)g.a_hl, units * (A8 ? 512u : 2048u));
            src.va = unit * (A8 ? 512 : 2048) + (A8 ? 8 : 16) * lane;
            if constexpr (A8) {
                src.ad = make_rsrc(g.d8, units * 64u);
                src.vad = (unit + (kq & 1)) * 64 + 4 * l16;
            }
        } else if constexpr (A8) {
            src.a = make_rsrc(g.a8, a_elems);
            src.va = srow * g.lda + 8 * kq;
            src.ad = make_rsrc(g.d8, 4u * (uint32_t)((g.M - 1) * (g.lda / 32) + nb));
            src.vad = 4 * (srow * (g.lda / 32) + (kq & 1));
        } else {
            src.a = make_rsrc(g.a, 4u * a_elems);
            src.va = 4 * (srow * g.lda + 8 * kq);
        }
        src.w = make_rsrc(TL ? g.wm : g.w, (uint32_t)(g.N / 16) * (uint32_t)nb * kTileBytes);
        const int sub = (n_base >> 4) + wave;
        if constexpr (TL) {
            src.vw = sub * nb * kTileBytes + 8 * lane;
            src.vs = sub * nb * kTileBytes + 512 + 2 * l16;
        } else {
            const int grp = 4 * sub + (l16 >> 2), krow = l16 & 3;
            src.vw = grp * nb * kBlockBytes + 8 + 32 * krow + 8 * kq;
            src.vs = grp * nb * kBlockBytes + 2 * krow;
        }
    }
    const int nch = nb / KB;
    StageA<A8, AT> a[kSets];
    ChunkW<A8> w[kSets];
    // chunk c into its set; a chunk past the last is not fetched (its offset is past every
    // resource), but stays an instruction: under a branch, every wait for an older load
    // would have to wait for all of them
    auto load = [&](int u, int c) {
        const int off = c < nch ? 0 : kPastEnd;
        load_a<A8, AT>(a[u], c * KB, off, src);
        load_w<A8, TL>(w[u], c * KB, off, src);
    };
#pragma unroll
    for (int u = 0; u + 1 < kSets; ++u) load(u, u);
    floatx4 acc[4], tot[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) acc[r] = tot[r] = floatx4{0.f, 0.f, 0.f, 0.f};
    const int per_run = nch / kRuns;  // chunks of a run of blocks that is summed apart
    int left = per_run;
    stage_a<A8, AT>(a[0], smem, wave, lane);
    lds_barrier();
    // chunk i is in LDS half i % 2 and its weights in set i % 4; chunk i + 3 is requested before
    // its products, chunk i + 1 goes to the other half after them
    for (int i = 0; i < nch; i += kSets) {
#pragma unroll
        for (int u = 0; u < kSets; ++u) {
            load((u + 3) % kSets, i + u + 3);
            const uint8_t *buf = smem + (u & 1) * CB;
#pragma unroll
            for (int j = 0; j < KB; ++j) mma_block<A8>(buf, j, lane, w[u], acc);
            if (--left == 0) {  // uniform
                left = per_run;
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    tot[r] += acc[r];
                    acc[r] = floatx4{0.f, 0.f, 0.f, 0.f};
                }
            }
            stage_a<A8, AT>(a[(u + 1) % kSets], smem + ((u + 1) & 1) * CB, wave, lane);
            lds_barrier();
        }
    }
    // finish: the tile crosses LDS so that a lane ends with 8 columns of a row, in the lane order of
    // the matrix-core layouts; a wave finishes 16 rows, 32 columns at a time
    Ops8<EPI> o[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) ops_load<EPI>(o[hf], g, ri, n_base + 32 * hf + 8 * kq);
    float *tile = reinterpret_cast<float *>(smem);
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int i = 0; i < 4; ++i) tile[(16 * r + 4 * kq + i) * kOutStride + 16 * wave + l16] = tot[r][i];
    lds_barrier();
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
        float v[8];
        load8(v, tile + (16 * wave + l16) * kOutStride + 32 * hf + 8 * kq);
        finish8<EPI, KV>(g, o[hf], ri, m, n_base + 32 * hf + 8 * kq, m < g.M, v);
    }
}

template <int EPI, int KV, bool A8, bool TL, bool AT>
hipError_t launch_k(const GemmArgs &g, hipStream_t s) {
    (void)hipGetLastError();  // report only this launch's error, not a stale one
    hipLaunchKernelGGL((gemm_tile_kernel<EPI, KV, A8, TL, AT>), dim3(g.N / TN, (g.M + TM - 1) / TM), dim3(256), 0, s, g);
    return hipGetLastError();
}

template <int EPI, int KV, bool TL>
hipError_t launch_t(const GemmArgs &g, hipStream_t s) {
    if (g.a8 != nullptr)
        return g.a8_tiled ? launch_k<EPI, KV, true, TL, true>(g, s) : launch_k<EPI, KV, true, TL, false>(g, s);
    return g.a_hl != nullptr ? launch_k<EPI, KV, false, TL, true>(g, s) : launch_k<EPI, KV, false, TL, false>(g, s);
}

template <int EPI, int KV>
hipError_t launch_e(const GemmArgs &g, hipStream_t s) {
    return g.wm != nullptr ? launch_t<EPI, KV, true>(g, s) : launch_t<EPI, KV, false>(g, s);
}

bool aligned16(const void *p) { return ((uintptr_t)p & 15) == 0; }
}  // namespace

// The call goes to 64 x 64 tiles where those fill the chip: from 384 workgroups on for fp32
// activations, from 512 for int8 (its products cost a third less, so a workgroup's start and
// end weigh more).  Under that a workgroup is on a CU alone or with one other and takes ~14 us
// from start to end, while the 16-row tiles of gemm_mfma.hip still spread over all CUs
// (measured inside prefills, here / there; A16: QKV of 512 rows, 288 workgroups 14.2 / 14.0 us,
// fc_in of 512, 384: 15.8 / 17.0, QKV of 768, 432: 14.9 / 18.6, of 1000, 576: 19.0 / 22.8, fc_in
// of 1000, 768: 21.2 / 30.0; W8A8: fc_in of 512, 384: 13.6 / 12.9, QKV of 1000: 15.4 / 17.7,
// fc_in of 1000: 16.5 / 21.8).  A long K (fc_out) is a chain of 48 chunks here, and its four
// slices measured 22.0 / 22.4 us at 1000 rows, 21.2 / 18 at 768: it stays there.
bool tile_gemm_fits(const GemmArgs &g, Epilogue epi) {
    if ((epi != EPI_QKV && epi != EPI_GELU && epi != EPI_F32) || g.ln_w != nullptr || g.pick_pairs != nullptr) return false;
    if (g.N % TN || g.K % (32 * KB * kRuns) || g.K % (32 * KB * kSets) || g.K > 1024) return false;
    const int64_t wgs = (int64_t)(g.N / TN) * ((g.M + TM - 1) / TM);
    if (wgs < (g.a8 ? 512 : 384)) return false;
    // operand offsets are 32-bit byte offsets below kPastEnd
    const int64_t a_bytes = (int64_t)((g.M + 15) / 16 * 16) * g.lda * (g.a8 ? 1 : 4);
    if (a_bytes >= kPastEnd || (int64_t)(g.N / 16) * (g.K / 32) * kTileBytes >= kPastEnd) return false;
    // the epilogue moves 16 bytes at a time
    if (!aligned16(g.y) || !aligned16(g.bias) || g.ldy % 4) return false;
    return epi != EPI_QKV || (aligned16(g.q_out) && aligned16(g.k_pool) && aligned16(g.v_pool) && aligned16(g.rope_cos) &&
                              aligned16(g.rope_sin));
}

hipError_t launch_gemm_tile(const GemmArgs &g, Epilogue epi, KvType kv, hipStream_t s) {
    switch (epi) {
        case EPI_F32: return launch_e<EPI_F32, KV_F16>(g, s);
        case EPI_GELU: return launch_e<EPI_GELU, KV_F16>(g, s);
        case EPI_QKV: return kv == KV_F32 ? launch_e<EPI_QKV, KV_F32>(g, s) : launch_e<EPI_QKV, KV_F16>(g, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace mh
