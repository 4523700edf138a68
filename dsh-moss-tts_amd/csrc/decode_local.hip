// decode_local.hip -- a frame's local half of the single-stream decode in one launch (gfx950).
//
// Replaces the local steps of a frame (local_step, reference csrc/src/llm.cpp:259-264:
// block_forward of the one local layer at local position lpos, llm.cpp:230-246),
// the channels' audio heads (audio_logits, llm.cpp:686-688: logits = aemb[ch] .
// local_ln_f(x)), the picks and the end gate.  Within each step lpos = 0 .. 16 the
// stages hand their outputs on through LL words (mh_ll.h), as in decode_layer.hip:
//   Q  lpos 0 only, b < 144: LN1 + QKV of the block input (the global hidden
//      state), RoPE, k/v into the local cache                  -> LL q|k|v
//   A  b < 12: head h = b: the step's input -- for lpos >= 2 the code of the
//      previous channel, picked here (penalised argmax of its logits, or a draw
//      from them, or the forced code) -- and the head's q|k|v:
//      from the QKV stage (lpos 0) or from the precomputed row of (lpos,
//      code); k/v into the local cache; the head's attention over keys
//      0..lpos (at most 17)                                    -> LL attn + code
//   P  b < 192: proj + residual (the raw input row is aemb[ch][code]) -> LL x + attn
//   M  b < 192: LN2 + fc_in + gelu_new                          -> LL h
//   F  b < 192: fc_out + residual -> x_out (memory) and, lpos >= 1, LL x_out
//   H  b < 64, lpos >= 1: local ln_f + the audio head GEMV     -> logits (memory, LL)
// (192 workgroups, one per CU; the GEMV stages take one wave per 4-row group,
// or four for the K slices of proj and fc_out).
//
// Precomputed q|k|v rows.  For lpos >= 1 the block input is an embedding row
// -- wte[slot] at lpos 1, aemb[lpos - 2][code] at lpos >= 2 -- and RoPE uses
// the fixed position lpos, so q|k|v = RoPE_lpos(attn_w . LN1(row) + attn_b) is
// a function of (lpos, code) only.  The host computes every such row once, at
// load, with the one-GEMV kernel of the per-operator path (the same per-row
// arithmetic), so the table holds exactly the values that path computes live.
#include "mh_gemv.h"
#include "mh_ll.h"
#include "mh_ops.h"
#include "mh_sample.h"

namespace mh {
namespace {

// LL regions (words); consecutive steps differ in lpos, so in tag
constexpr int kLQ = 0;                  // q | k | v (lpos 0)
constexpr int kLA = kLQ + 3 * kHidden;  // attention output (768) and the step's input code (1)
constexpr int kLX = kLA + kHidden + 1;  // x after the attention sub-block
constexpr int kLH = kLX + kHidden;      // fc_in output
constexpr int kLO = kLH + kFF;          // block output (head input)
constexpr int kLL = kLO + kHidden;      // head logits, the next step's pick input (1024)
constexpr int kLG = kLL + kCodebook;    // position 0's block output, the end gate's input (768)
constexpr int kLD = kLG + kHidden;      // sampled frames: the end gate is done (1)
static_assert(kLD + 1 <= kLayerWords, "local LL layout fits the exchange buffer");

// Stage timestamps (100 MHz device clock) of the last launch, per workgroup,
// in builds with -DMH_STAGE_TRACE only.
#ifdef MH_STAGE_TRACE
}  // namespace
__device__ unsigned long long mh_local_ts[kLayerGrid][32];
namespace {
// Kept in LDS by thread 0 and written out at the end of the launch: a global
// store inside a stage would make the next barrier wait for it.
#define STAGE_DECL                                         \
    __shared__ unsigned long long stage_ts_lds[32];        \
    if (threadIdx.x == 0)                                  \
        for (int i_ = 0; i_ < 32; ++i_) stage_ts_lds[i_] = i_ == 16 ? __builtin_amdgcn_s_memtime() : 0
#define STAGE_TS(k)                                                               \
    do {                                                                          \
        if (threadIdx.x == 0) stage_ts_lds[k] = __builtin_amdgcn_s_memrealtime(); \
    } while (0)
#define STAGE_FLUSH()                                                          \
    do {                                                                       \
        if (threadIdx.x == 0) {                                                \
            stage_ts_lds[17] = __builtin_amdgcn_s_memtime();                   \
            stage_ts_lds[18] = __builtin_amdgcn_s_memrealtime();               \
            for (int i_ = 0; i_ < 32; ++i_) mh_local_ts[blockIdx.x][i_] = stage_ts_lds[i_]; \
        }                                                                      \
    } while (0)
#else
#define STAGE_DECL \
    do {           \
    } while (0)
#define STAGE_TS(k) \
    do {            \
    } while (0)
#define STAGE_FLUSH() \
    do {              \
    } while (0)
#endif

template <bool SAMPLED>
__device__ __forceinline__ SampleLds &sample_lds() {  // in LDS only where a kernel draws
    __shared__ SampleLds l;
    return l;
}

// A8: every GEMV in W8A8 (quant_act_lds), the reference's decode with MOSS_A16 unset.
// SAMPLED: the frame draws its codes (sampler.cpp:30-78) unless it is one of the call's greedy
// first frames.  Each of the 12 attention workgroups makes the same draw from its own copy of
// the call's xoshiro stream, so a pick costs its ~4 us of sorting and no hand-off; one launch
// per position with a sampler kernel after each measured 0.88 ms per frame's local half
// (17 x 16 us + 16 x 38 us, W8A8).
template <bool A8, bool SAMPLED>
__global__ __launch_bounds__(256) void decode_local_kernel(LocalArgs a) {
#pragma clang fp contract(off)
    __shared__ float act[kFF + 1];
    __shared__ float da[kFF / 32];  // block scales of act (A8)
    __shared__ float xm[kHidden];
    __shared__ float qkv[3 * kHidden];             // q | k | v of this position
    __shared__ float sc[kHeads][kLocalLen + 1];
    __shared__ float part[4][4];
    __shared__ float pbv[4];
    __shared__ int pbi[4];
    __shared__ float lgt[kCodebook];  // the previous step's logits (chained launches)
    __shared__ GateLds gl;
    SampleLds &sl = sample_lds<SAMPLED>();

    __shared__ int wait_failed;  // set when a wait of this workgroup runs out
    if (threadIdx.x == 0) wait_failed = 0;
    __syncthreads();
    STAGE_DECL;
    STAGE_TS(0);
    DevState *st = a.state;
    if (st->stop) return;  // written only between frames: the same for every workgroup
    const uint32_t tag_base = (uint32_t)(st->pos + 1) << 5;
    int budget = a.poll_budget > 0 ? a.poll_budget : kPollBudget;
    uint64_t *LL = a.ll;
    // SAMPLED: this frame's stream.  The end gate draws first (llm.cpp:678) when it samples at all;
    // workgroup 0 stores the state after the frame's last draw.
    bool draws = false;
    uint32_t rng[4], gate_rng[4];
    if constexpr (SAMPLED) {
        const SampleCfg c = st->cfg;
        draws = !c.greedy && st->frame >= c.greedy_frames;
#pragma unroll
        for (int i = 0; i < 4; ++i) gate_rng[i] = rng[i] = st->rng[i];
        if (!c.end_greedy && st->frame >= st->min_frames) (void)rng_next(rng);
    }

    // ---- the end gate (llm.cpp:653-679) in a workgroup of its own (the last):
    // ln_f of position 0's block output, the 2-row W8A8 gate, the stop rule.  The
    // channel steps do not wait for it: a frame the gate ends is dropped by the
    // host, and every state it touches is rewritten before it is read again.
    if ((int)blockIdx.x == kLayerGrid) {
        const int t = threadIdx.x;
        float lw[3], lb[3];
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            lw[i] = a.lnf_w[t + 256 * i];
            lb[i] = a.lnf_b[t + 256 * i];
        }
        const bool ok = ll_gather<3>(LL + kLG, kHidden, tag_base | 12u, xm, budget);
        if (sync_failed(!ok, &wait_failed)) {
            if (t == 0) atomicOr(a.err, 1u);
            return;
        }
        float o[3];
        layernorm_768_lds(xm, lw, lb, o);
#pragma unroll
        for (int i = 0; i < 3; ++i) act[t + 256 * i] = o[i];
        __syncthreads();
        // no other workgroup waits for this one in a greedy frame, so by now workgroup 0 may have
        // counted the frame in st->frame; a sampled frame's stream it stores after kLD only
        gate_block(act, a.wte, st, gl, SAMPLED ? gate_rng : st->rng, a.frame);
        if constexpr (SAMPLED)
            if (t == 0) ll_put(LL + kLD, 1.0f, tag_base | 12u);
        return;
    }

    auto pick = [&](const PickIn &in) {  // by every thread of the workgroup, the same in all of them
        if constexpr (SAMPLED)
            if (draws) return pick_penalised(in, st->rep_penalty, st->cfg, rng_uniform(rng), sl);
        const int idx = greedy_pick_reduce(in, st->rep_penalty, pbv, pbi);
        return idx >= kCodebook ? 0 : idx;  // every value NaN: the reference's scan stays at 0
    };

    // positions 0 .. 16, the bounds hidden from the compiler: knowing them, it compiles a loop whose
    // launch takes 219.5 us where one with the bounds as kernel arguments takes 217.5; this one takes
    // 214.1 where that takes 214.8 (another card)
    int first = 0, last = kNVq;
    asm("" : "+s"(first), "+s"(last));
#pragma unroll 1
    for (int lpos = first; lpos <= last; ++lpos) {
        const int n = lpos + 1;
        const uint32_t tag = tag_base | (uint32_t)(12 + lpos);
        // per-step copies of the indices: nothing derived from them is held across steps
        const int t = tix();
        const int b = bix();
        const int ch_in = lpos >= 2 ? lpos - 2 : -1;  // channel whose code is this step's input
        const uint8_t *aemb_in = ch_in >= 0 ? a.aemb[ch_in] : nullptr;
        const uint8_t *head_w = lpos >= 1 ? a.aemb[lpos - 1] : nullptr;
        float *logits_out = lpos >= 1 ? a.logits + (size_t)(lpos - 1) * kCodebook : nullptr;
        const bool live = lpos == 0;  // the block input is the global hidden state: QKV computed here
        const bool picking = !live && ch_in >= 0;  // from the previous step's logits
        // W8A8 quantiser capture of this position (tests only; null in the library's own use)
        float *const cap = A8 && a.cap ? a.cap + (size_t)lpos * MOSS_HIP_CAP_STEP : nullptr;

        // ---- stage Q (lpos 0): LN1 + QKV of the block input, one wave per group
        if (live) {
            if (b < 3 * kHidden / 16) {
                GemvStage<1, 6, kHidden> gs;
                gs.prefetch(a.attn_w, b);
                const int r = gs.row();
                QkvEpi e;
                if (gs.storer()) e.load(a.attn_b, a.rope_cos, a.rope_sin, r, lpos);
                float o[3], lw[3], lb[3];
#pragma unroll
                for (int i = 0; i < 3; ++i) {
                    xm[t + 256 * i] = a.x_in[t + 256 * i];
                    lw[i] = a.ln1_w[t + 256 * i];
                    lb[i] = a.ln1_b[t + 256 * i];
                }
                __syncthreads();
                layernorm_768_lds(xm, lw, lb, o);
#pragma unroll
                for (int i = 0; i < 3; ++i) act[t + 256 * i] = o[i];
                __syncthreads();
                if constexpr (A8) {
                    float *cp = b == 0 ? cap : nullptr;  // (uniform)
                    if (cp) {
                        cap_copy(cp + MOSS_HIP_CAP_XIN, xm, kHidden);
                        cap_copy(cp + MOSS_HIP_CAP_LN1, act, kHidden);
                        __syncthreads();  // before the quantiser rewrites runs other threads copy
                    }
                    quant_act_lds_k<kHidden>(act, da);
                    __syncthreads();
                    if (cp) {
                        cap_copy(cp + MOSS_HIP_CAP_LN1_Q, act, kHidden);
                        cap_copy(cp + MOSS_HIP_CAP_LN1_D, da, kHidden / 32);
                    }
                }
                const float yv = gs.template dot<A8>(act, part, da);
                const float partner = xshfl<4>(yv);
                if (gs.storer()) ll_put(LL + kLQ + r, e.apply(r, yv, partner), tag);  // k, v cached by stage A
                __syncthreads();
            }
        }

        // ---- stage A (b < 12): head h = b of the local attention (llm.cpp:189-217
        // over the local cache, keys 0..lpos) in the reference's order:
        // s_p = (q_h . k_p) * 0.125 summed over d in order; e_p = exp(s_p - max),
        // the in-order sum, w_p = e_p * (1 / sum); o[d] = sum_p w_p v_p[d] in order.
        // Wave 0 computes: lane p < 17 a score, lane d the output dimension d.
        if (b < kHeads) {
            const int h = b, lane = t & 63;
            const bool w0 = t < 64;
            const int kmax = max(lpos - 1, 0);
            // loads complete in issue order: the pick's logits first
            PickIn pin;
            if (picking)  // counts now, values once the previous step's head has stored them
#pragma unroll
                for (int k = 0; k < kCodebook / 256; ++k)
                    pin.cnt[k] = st->rep_penalty != 1.0f ? a.counts[(size_t)ch_in * kCodebook + t + 256 * k] : 0;
            // the cache rows (keys 0 .. lpos-1, written by earlier steps) before
            // anything else; the key at lpos, and the clamped ones past it, take
            // this step's row below
            float4 kr[kHeadDim / 4];
            float vv[kLocalLen];
            if (w0) {
                const float *krow = a.lk + ((size_t)h * kLocalLen + min(lane, kmax)) * kHeadDim;
#pragma unroll
                for (int c = 0; c < kHeadDim / 4; ++c) kr[c] = *(const float4 *)(krow + 4 * c);
#pragma unroll
                for (int p = 0; p < kLocalLen; ++p) vv[p] = a.lv[((size_t)h * kLocalLen + min(p, kmax)) * kHeadDim + lane];
            }
            // q, k, v of head h at lpos
            if (live) {
                const int seg = min(t >> 6, 2), i = seg * kHidden + h * kHeadDim + (t & 63);
                const bool ok = ll_wait1(LL + kLQ + i, t < 3 * kHeadDim, tag, &qkv[i], budget);
                // this position's k, v into the local cache (llm.cpp:224-225) by the workgroup
                // that reads them at the later positions: same-workgroup ordering, no fence
                if (ok && t < 3 * kHeadDim && seg > 0)
                    (seg == 1 ? a.lk : a.lv)[((size_t)h * kLocalLen + lpos) * kHeadDim + (t & 63)] = qkv[i];
                if (sync_failed(!ok, &wait_failed)) {
                    if (t == 0) atomicOr(a.err, 1u);
                    return;
                }
            } else {
                const float *row = a.qkv_table;  // lpos 1: wte[slot]
                if (picking) {  // the pick of channel ch_in (llm.cpp:689-697)
                    // waves 1-3 poll the logits: wave 0's cache-row loads, issued
                    // above, would hold back its polls (loads complete in order)
                    bool ok = true;
                    if (t >= 64)
                        ok = ll_gather_by<(kCodebook + 191) / 192, 192>(LL + kLL, kCodebook, tag - 1, lgt, budget, t - 64);
                    if (sync_failed(!ok, &wait_failed)) {
                        if (t == 0) atomicOr(a.err, 1u);
                        return;
                    }
#pragma unroll
                    for (int k = 0; k < kCodebook / 256; ++k) pin.vals[k] = lgt[t + 256 * k];
                    const int idx = pick(pin);
                    const int used = st->forced_on ? a.forced[st->frame * kNVq + ch_in] : idx;
                    if (b == 0 && t == 0) {
                        st->codes[ch_in] = idx;
                        st->row[ch_in + 1] = used;
                    }
                    if (b == 0 && t == 0) ll_put(LL + kLA + kHidden, __int_as_float(used), tag);  // for stage P
                    row = a.qkv_table + (1 + (size_t)ch_in * kCodebook + used) * 3 * kHidden;
                }
                STAGE_TS(1);
                if (t < 3 * kHeadDim) {
                    const int seg = t >> 6, i = seg * kHidden + h * kHeadDim + (t & 63);
                    const float v = row[i];
                    qkv[i] = v;
                    if (seg > 0)  // this position's k, v into the local cache (llm.cpp:224-225), for later steps
                        (seg == 1 ? a.lk : a.lv)[((size_t)h * kLocalLen + lpos) * kHeadDim + (t & 63)] = v;
                }
                __syncthreads();
            }
            STAGE_TS(2);
            if constexpr (A8)
                if (cap && t < 3 * kHeadDim) {
                    const int i = (t >> 6) * kHidden + h * kHeadDim + (t & 63);
                    cap[MOSS_HIP_CAP_QKV + i] = qkv[i];
                }
            if (w0) {
                const float *qh = &qkv[h * kHeadDim];
                if (min(lane, n - 1) == lpos)
#pragma unroll
                    for (int c = 0; c < kHeadDim / 4; ++c) kr[c] = *(const float4 *)&qkv[kHidden + h * kHeadDim + 4 * c];
                float dot = 0.0f;
#pragma unroll
                for (int c = 0; c < kHeadDim / 4; ++c) {
                    const float4 qv = *(const float4 *)(qh + 4 * c);
                    dot = dot + qv.x * kr[c].x;
                    dot = dot + qv.y * kr[c].y;
                    dot = dot + qv.z * kr[c].z;
                    dot = dot + qv.w * kr[c].w;
                }
                dot *= 0.125f;
                if (lane < kLocalLen) sc[0][lane] = dot;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                float sv[kLocalLen];
#pragma unroll
                for (int p = 0; p < kLocalLen; ++p) sv[p] = sc[0][p];
                float mx = -1e30f;
#pragma unroll
                for (int p = 0; p < kLocalLen; ++p)
                    if (p < n) mx = fmaxf(mx, sv[p]);
                const float e = lane < n ? expf(dot - mx) : 0.0f;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (lane < kLocalLen) sc[0][lane] = e;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
#pragma unroll
                for (int p = 0; p < kLocalLen; ++p) sv[p] = sc[0][p];
                float sum = 0.0f;
#pragma unroll
                for (int p = 0; p < kLocalLen; ++p)
                    if (p < n) sum += sv[p];
                const float wgt = e * (1.0f / sum);  // 0 for keys past n
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (lane < kLocalLen) sc[0][lane] = wgt;
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                const float vnew = qkv[2 * kHidden + h * kHeadDim + lane];
                float o = 0.0f;
#pragma unroll
                for (int p = 0; p < kLocalLen; ++p) o = o + sc[0][p] * (min(p, n - 1) == lpos ? vnew : vv[p]);
                ll_put(LL + kLA + h * kHeadDim + lane, o, tag);
            }
            STAGE_TS(3);
            __syncthreads();
        }

        // ---- stage P: proj + residual (4 waves per group)
        if (b < kHidden / 4) {
            GemvStage<4, 2, kHidden> gs;
            gs.prefetch(a.proj_w, b);
            const int r = gs.row();
            const float eb = gs.storer() ? a.proj_b[r] : 0.0f;
            const bool with_code = !live && ch_in >= 0;  // the raw input row is aemb[ch_in][used]
            float eres = 0.0f;
            if (gs.storer() && !with_code) eres = (live ? a.x_in : a.x_slot)[r];
            const bool ok = ll_gather<(kHidden + 1 + 255) / 256>(LL + kLA, kHidden + (with_code ? 1 : 0), tag, act, budget);
            if (sync_failed(!ok, &wait_failed)) {
                if (t == 0) atomicOr(a.err, 1u);
                return;
            }
            if (gs.storer() && with_code)  // lookup_row (llm.cpp:697)
                eres = q8x4_elem(aemb_in, kHidden / 32, __float_as_int(act[kHidden]), r);
            if constexpr (A8) {  // act[0, 768) only: the code at act[kHidden] stays
                float *cp = b == 0 ? cap : nullptr;
                if (cp) {  // a barrier before the quantiser rewrites runs other threads copy
                    cap_copy(cp + MOSS_HIP_CAP_ATT, act, kHidden);
                    __syncthreads();
                }
                quant_act_lds_k<kHidden>(act, da);
                __syncthreads();
                if (cp) {
                    cap_copy(cp + MOSS_HIP_CAP_ATT_Q, act, kHidden);
                    cap_copy(cp + MOSS_HIP_CAP_ATT_D, da, kHidden / 32);
                }
            }
            const float yv = gs.template dot<A8>(act, part, da);
            if (gs.storer()) {
                ll_put(LL + kLX + r, eres + (yv + eb), tag);  // llm.cpp:239
                if constexpr (A8)
                    if (cap) cap[MOSS_HIP_CAP_XM + r] = eres + (yv + eb);
            }
            STAGE_TS(4);
            __syncthreads();  // act is reused by stage F
        }

        // ---- stage M: LN2 + fc_in + gelu_new, one wave per group, every workgroup
        {
            GemvStage<1, 6, kHidden> gs;
            gs.prefetch(a.fc_in_w, b);
            const int r = gs.row();
            const float eb = gs.storer() ? a.fc_in_b[r] : 0.0f;
            float lw[3], lb[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                lw[i] = a.ln2_w[t + 256 * i];
                lb[i] = a.ln2_b[t + 256 * i];
            }
            const bool ok = ll_gather<3>(LL + kLX, kHidden, tag, xm, budget);
            if (sync_failed(!ok, &wait_failed)) {
                if (t == 0) atomicOr(a.err, 1u);
                return;
            }
            STAGE_TS(5);
            float o[3];
            layernorm_768_lds(xm, lw, lb, o);
#pragma unroll
            for (int i = 0; i < 3; ++i) act[t + 256 * i] = o[i];
            __syncthreads();
            if constexpr (A8) {
                float *cp = b == 0 ? cap : nullptr;
                if (cp) {  // a barrier before the quantiser rewrites runs other threads copy
                    cap_copy(cp + MOSS_HIP_CAP_LN2, act, kHidden);
                    __syncthreads();
                }
                quant_act_lds_k<kHidden>(act, da);
                __syncthreads();
                if (cp) {
                    cap_copy(cp + MOSS_HIP_CAP_LN2_Q, act, kHidden);
                    cap_copy(cp + MOSS_HIP_CAP_LN2_D, da, kHidden / 32);
                }
            }
            const float yv = gs.template dot<A8>(act, part, da);
            if (gs.storer()) {
                ll_put(LL + kLH + r, gelu_new(yv + eb), tag);  // llm.cpp:243
                if constexpr (A8)
                    if (cap) cap[MOSS_HIP_CAP_H + r] = gelu_new(yv + eb);
            }
            STAGE_TS(6);
            __syncthreads();  // every wave is done with act before stage F gathers into it
        }

        // ---- stage F: fc_out + residual (4 waves per group)
        if (b < kHidden / 4) {
            GemvStage<4, 6, kFF> gs;
            gs.prefetch(a.fc_out_w, b);
            const int r = gs.row();
            const float eb = gs.storer() ? a.fc_out_b[r] : 0.0f;
            ll_gather_slice<kFF>(LL + kLH, tag, act, budget, &wait_failed);
            if constexpr (A8) {  // the slice's 24 blocks, quantised by the wave that reads them
                const int w = __builtin_amdgcn_readfirstlane(t >> 6);
                quant_act_lds_k<kFF / 4, 64>(act + (kFF / 4) * w, da + (kFF / 128) * w, t & 63);
                __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
                __builtin_amdgcn_wave_barrier();
                if (b == 0 && cap) {
                    __syncthreads();
                    cap_copy(cap + MOSS_HIP_CAP_H_Q, act, kFF);
                    cap_copy(cap + MOSS_HIP_CAP_H_D, da, kFF / 32);
                }
            }
            STAGE_TS(7);
            const float yv = gs.template dot<A8>(act, part, da);
            if (*(volatile int *)&wait_failed) {  // read after the dot's barriers
                if (t == 0) atomicOr(a.err, 1u);
                return;
            }
            if (gs.storer()) {
                const float xo = xm[r] + (yv + eb);  // llm.cpp:245
                a.x_out[r] = xo;
                if constexpr (A8)
                    if (cap) cap[MOSS_HIP_CAP_XOUT + r] = xo;
                if (head_w) ll_put(LL + kLO + r, xo, tag);
                if (live) ll_put(LL + kLG + r, xo, tag);  // the gate workgroup's input
            }
            STAGE_TS(8);
            __syncthreads();
        }

        // ---- stage H: local ln_f + audio head (4 waves per group)
        if (head_w && b < kCodebook / 16) {
            GemvStage<1, 6, kHidden> gs;
            gs.prefetch(head_w, b);
            float lw[3], lb[3];
#pragma unroll
            for (int i = 0; i < 3; ++i) {
                lw[i] = a.lnf_w[t + 256 * i];
                lb[i] = a.lnf_b[t + 256 * i];
            }
            const bool ok = ll_gather<3>(LL + kLO, kHidden, tag, xm, budget);
            if (sync_failed(!ok, &wait_failed)) {
                if (t == 0) atomicOr(a.err, 1u);
                return;
            }
            STAGE_TS(9);
            float o[3];
            layernorm_768_lds(xm, lw, lb, o);  // normalize(lx, local_lnf) (llm.cpp:262)
#pragma unroll
            for (int i = 0; i < 3; ++i) act[t + 256 * i] = o[i];
            __syncthreads();
            if constexpr (A8) {
                float *cp = b == 0 ? cap : nullptr;
                if (cp) {  // a barrier before the quantiser rewrites runs other threads copy
                    cap_copy(cp + MOSS_HIP_CAP_LNF, act, kHidden);
                    __syncthreads();
                }
                quant_act_lds_k<kHidden>(act, da);
                __syncthreads();
                if (cp) {
                    cap_copy(cp + MOSS_HIP_CAP_LNF_Q, act, kHidden);
                    cap_copy(cp + MOSS_HIP_CAP_LNF_D, da, kHidden / 32);
                }
            }
            const float yv = gs.template dot<A8>(act, part, da);
            if (gs.storer()) {
                logits_out[gs.row()] = yv;
                ll_put(LL + kLL + gs.row(), yv, tag);  // the next pick
            }
            STAGE_TS(10);
        }

        // ---- after the last position: the pick of its channel, as
        // sample_kernel does for the last channel (workgroup 0)
        if (lpos == last && b == 0) {
            const int ch = lpos - 1;
            PickIn pin;
#pragma unroll
            for (int k = 0; k < kCodebook / 256; ++k)
                pin.cnt[k] = st->rep_penalty != 1.0f ? a.counts[(size_t)ch * kCodebook + t + 256 * k] : 0;
            bool ok = ll_gather<kCodebook / 256>(LL + kLL, kCodebook, tag, lgt, budget);
            if constexpr (SAMPLED) ok = ll_wait1(LL + kLD, t == 0, tag_base | 12u, &pbv[0], budget) && ok;
            if (sync_failed(!ok, &wait_failed)) {
                if (t == 0) atomicOr(a.err, 1u);
                return;
            }
#pragma unroll
            for (int k = 0; k < kCodebook / 256; ++k) pin.vals[k] = lgt[t + 256 * k];
            const int idx = pick(pin);
            const int used = st->forced_on ? a.forced[st->frame * kNVq + ch] : idx;
            if (t < ch) a.counts[(size_t)t * kCodebook + st->row[t + 1]] += 1;  // the frame's earlier channels
            if (t == 0) {
                st->codes[ch] = idx;
                st->row[ch + 1] = used;
                a.counts[(size_t)ch * kCodebook + used] += 1;
                st->row[0] = kSlotToken;
                st->frame += 1;
                if constexpr (SAMPLED)
#pragma unroll
                    for (int i = 0; i < 4; ++i) st->rng[i] = rng[i];
            }
        }
    }  // lpos
    STAGE_FLUSH();
}

}  // namespace

#ifdef MH_STAGE_TRACE
// [kLayerGrid][32] timestamps of the last launch (profiling builds only)
extern "C" int mh_local_trace_read(unsigned long long *out) {
    return (int)hipMemcpyFromSymbol(out, HIP_SYMBOL(mh_local_ts), sizeof(mh_local_ts));
}
#endif

hipError_t decode_local_occupancy(int *per_cu) {
    const void *k[4] = {(const void *)decode_local_kernel<false, false>, (const void *)decode_local_kernel<true, false>,
                        (const void *)decode_local_kernel<false, true>, (const void *)decode_local_kernel<true, true>};
    for (int i = 0; i < 4; ++i) {
        int p = 0;
        const hipError_t e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&p, k[i], 256, 0);
        if (e != hipSuccess) return e;
        *per_cu = i == 0 || p < *per_cu ? p : *per_cu;
    }
    return hipSuccess;
}

hipError_t launch_decode_local(const LocalArgs &a, hipStream_t s) {
    (void)hipGetLastError();  // report only this launch's error, not a stale one
    if (!a.attn_w || !a.proj_w || !a.fc_in_w || !a.fc_out_w || !a.lk || !a.lv || !a.state || !a.ll || !a.err ||
        !a.x_out || !a.logits || !a.lnf_w || !a.lnf_b || !a.x_in || !a.rope_cos || !a.rope_sin || !a.wte ||
        !a.qkv_table || !a.x_slot || !a.counts || !a.forced)
        return hipErrorInvalidValue;
    for (const uint8_t *w : a.aemb)
        if (!w) return hipErrorInvalidValue;
    static_assert(kNVq + 1 == kLocalLen, "positions 0 .. 16");
    const dim3 grid(kLayerGrid + 1);  // one more workgroup for the end gate
    if (a.a8 && a.sampled)
        hipLaunchKernelGGL((decode_local_kernel<true, true>), grid, dim3(256), 0, s, a);
    else if (a.a8)
        hipLaunchKernelGGL((decode_local_kernel<true, false>), grid, dim3(256), 0, s, a);
    else if (a.sampled)
        hipLaunchKernelGGL((decode_local_kernel<false, true>), grid, dim3(256), 0, s, a);
    else
        hipLaunchKernelGGL((decode_local_kernel<false, false>), grid, dim3(256), 0, s, a);
    return hipGetLastError();
}

}  // namespace mh
