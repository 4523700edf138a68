// codec_model.hip -- host driver of the GPU audio codec decoder (see codec.h).
#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstring>
#include <vector>

#include "codec.h"
#include "llm_model.h"

namespace mh {
namespace {

constexpr int kStageIds[kCodecStages] = {1, 3, 5, 7};       // decoder.cpp:42
constexpr int kPatches[kCodecStages] = {4, 2, 2, 2};        // decoder.cpp:43
constexpr int kLayerCounts[kCodecStages] = {4, 2, 2, 4};    // decoder.cpp:44
constexpr int kContexts[kCodecStages] = {500, 800, 1200, 1600};  // decoder.cpp:21
constexpr int kDtF16 = 0, kDtF32 = 3;  // DType (csrc/include/moss/common.h:26)
constexpr int kMaxPieceFrames = 1024;
// decode() runs an utterance in equal pieces of at most this many frames (of max_chunk_frames,
// where the caller set it).  Longer ones are faster and hold more: us a frame of utterances of 104,
// 203, 300 and 1000 frames, and MB of rings and activations, at 32 frames 25.5, 23.2, 22.7, 21.4 (38 +
// 12); 64: 17.9, 18.3, 15.7, 15.1 (51 + 22); 104: 13.2, 13.3, 13.5, 13.6 (66 + 36); 208: 13.4, 11.1, 12.3,
// 10.8 (107 + 72); 512: 13.4, 11.1, 10.6, 8.8 (227 + 176).  104 keeps a handle's decode() near 100 MB; a
// caller with long utterances and the room sets max_chunk_frames.
constexpr int kWholePiece = 104;

size_t align256(size_t n) { return (n + 255) & ~(size_t)255; }

// rows a piece of `frames` frames has at stage s: frames * 4, * 8, * 16, * 32
int stage_rows(int frames, int s) {
    int r = frames;
    for (int i = 0; i <= s; ++i) r *= kPatches[i];
    return r;
}

}  // namespace

Codec::Codec(const void *blob, size_t bytes, const moss_hip_codec_options &opt) {
    device_ = opt.device;
    fmax_ = opt.max_chunk_frames > 0 ? opt.max_chunk_frames : 32;
    if (fmax_ > kMaxPieceFrames) throw Status(MOSS_HIP_EINVAL, "max_chunk_frames > 1024");
    whole_max_ = opt.max_chunk_frames > 0 ? fmax_ : kWholePiece;
    eager_ = opt.eager != 0;
    const uint8_t *b = static_cast<const uint8_t *>(blob);
    auto idx = parse_moss_index(b, bytes);

    // Resolve every tensor AudioDecoder::load asks for (decoder.cpp:28-68) before touching the GPU.
    struct Place {
        uint64_t src, n;
        size_t dst;
    };
    std::vector<Place> places;
    size_t arena = 0;
    auto place = [&](const MossEntry &e, uint64_t n) {
        places.push_back({e.off, n, arena});
        const size_t at = arena;
        arena += align256(n);
        return at;
    };
    auto vec = [&](const std::string &name, uint32_t n) -> size_t {
        auto it = idx.find(name);
        if (it == idx.end() || !is_vector(it->second)) throw Status(MOSS_HIP_EFORMAT, "missing vector: " + name);
        const MossEntry &e = it->second;
        if (e.dims[0] * e.dims[1] != n || e.dtype != kDtF32 || e.nbytes < (uint64_t)n * 4)
            throw Status(MOSS_HIP_EFORMAT, "bad vector: " + name);
        return place(e, (uint64_t)n * 4);
    };
    // a matrix of rows x cols (either may be -1 = taken from the file); fp16 or fp32
    auto mat = [&](const std::string &name, int rows, int cols, int *rows_out, int *cols_out, int *f32) -> size_t {
        auto it = idx.find(name);
        if (it == idx.end() || is_vector(it->second)) throw Status(MOSS_HIP_EFORMAT, "missing matrix: " + name);
        const MossEntry &e = it->second;
        if (e.dtype != kDtF16 && e.dtype != kDtF32)
            throw Status(MOSS_HIP_EUNSUPPORTED, "matrix " + name + " has dtype " + std::to_string(e.dtype) +
                                                    "; only F16 (0) and F32 (3) are supported");
        const int r = (int)e.dims[0], c = (int)e.dims[1];
        if ((rows >= 0 && r != rows) || (cols >= 0 && c != cols)) throw Status(MOSS_HIP_EFORMAT, "bad matrix shape: " + name);
        const uint64_t n = (uint64_t)r * c * (e.dtype == kDtF32 ? 4 : 2);
        if (e.nbytes < n) throw Status(MOSS_HIP_EFORMAT, "matrix truncated: " + name);
        if (rows_out) *rows_out = r;
        if (cols_out) *cols_out = c;
        if (f32) *f32 = e.dtype == kDtF32;
        return place(e, n);
    };

    // quantizer front (decoder.cpp:31-38, 224-245): fp32 codebooks and projections
    size_t o_cb[kCodecNq], o_cw[kCodecNq], o_cbias[kCodecNq];
    for (int i = 0; i < kCodecNq; ++i) {
        const std::string p = "q" + std::to_string(i);
        int f32 = 0;
        o_cb[i] = mat(p + ".cb", kCodecCb, kCodecCbDim, nullptr, nullptr, &f32);
        if (!f32) throw Status(MOSS_HIP_EUNSUPPORTED, p + ".cb must be F32");
        o_cw[i] = mat(p + ".out.w", kCodecZ, kCodecCbDim, nullptr, nullptr, &f32);
        if (!f32) throw Status(MOSS_HIP_EUNSUPPORTED, p + ".out.w must be F32");
        o_cbias[i] = vec(p + ".out.b", kCodecZ);
    }
    int c0 = 0;
    const size_t o_qw = mat("q.out.w", -1, kCodecZ, &c0, nullptr, &qout_f32_);
    const size_t o_qb = vec("q.out.b", (uint32_t)c0);
    if (c0 % 16) throw Status(MOSS_HIP_EUNSUPPORTED, "q.out.w rows must be a multiple of 16");

    struct LayerOff {
        size_t attn, proj, f1, f2, n1w, n1b, n2w, n2b, ls1, ls2;
    };
    std::vector<LayerOff> loff;
    size_t o_in[kCodecStages], o_out[kCodecStages];
    int cin = c0;
    for (int s = 0; s < kCodecStages; ++s) {
        const std::string p = "d" + std::to_string(kStageIds[s]) + ".";
        StageW &S = stages_[s];
        S.patch = kPatches[s];
        if (cin % S.patch) throw Status(MOSS_HIP_EFORMAT, "stage input width does not divide by the patch");
        S.cin = cin / S.patch;
        if (S.cin % 32) throw Status(MOSS_HIP_EUNSUPPORTED, p + "in.w: columns must be a multiple of 32");
        o_in[s] = mat(p + "in.w", kCodecDModel, S.cin, nullptr, nullptr, &S.in_f32);
        o_out[s] = mat(p + "out.w", -1, kCodecDModel, &S.cout, nullptr, &S.out_f32);
        if (S.cout % 16) throw Status(MOSS_HIP_EUNSUPPORTED, p + "out.w: rows must be a multiple of 16");
        S.window = opt.contexts[s] > 0 ? opt.contexts[s] : kContexts[s];
        S.layer0 = (int)layers_.size();
        S.nlayers = kLayerCounts[s];
        for (int n = 0; n < S.nlayers; ++n) {
            const std::string lp = p + "l" + std::to_string(n) + ".";
            LayerW L{};
            LayerOff lo{};
            lo.attn = mat(lp + "attn.w", 3 * kCodecDModel, kCodecDModel, nullptr, nullptr, &L.attn_f32);
            lo.proj = mat(lp + "proj.w", kCodecDModel, kCodecDModel, nullptr, nullptr, &L.proj_f32);
            lo.f1 = mat(lp + "f1.w", -1, kCodecDModel, &L.ffn, nullptr, &L.f1_f32);
            if (L.ffn % 32) throw Status(MOSS_HIP_EUNSUPPORTED, lp + "f1.w: rows must be a multiple of 32");
            lo.f2 = mat(lp + "f2.w", kCodecDModel, L.ffn, nullptr, nullptr, &L.f2_f32);
            lo.n1w = vec(lp + "n1.w", kCodecDModel);
            lo.n1b = vec(lp + "n1.b", kCodecDModel);
            lo.n2w = vec(lp + "n2.w", kCodecDModel);
            lo.n2b = vec(lp + "n2.b", kCodecDModel);
            lo.ls1 = vec(lp + "ls1", kCodecDModel);
            lo.ls2 = vec(lp + "ls2", kCodecDModel);
            ffn_max_ = std::max(ffn_max_, L.ffn);
            layers_.push_back(L);
            loff.push_back(lo);
        }
        cin = S.cout;
    }
    // decode_chunk's final patch_forward(x, 240) (decoder.cpp:218-220) keeps one value per row
    if (cin != kCodecFinalPatch) throw Status(MOSS_HIP_EUNSUPPORTED, "the last stage must have 240 output channels");
    spf_ = stage_rows(1, kCodecStages - 1) * kCodecFinalPatch;

    hip_check(hipSetDevice(device_), "hipSetDevice");
    hip_check(hipStreamCreateWithFlags(&stream_, hipStreamNonBlocking), "hipStreamCreate");
    {
        std::vector<uint8_t> host(arena, 0);
        for (const Place &p : places) std::memcpy(host.data() + p.dst, b + p.src, p.n);
        hip_check(hipMalloc(&wdev_, arena), "hipMalloc(codec weights)");
        hip_check(hipMemcpy(wdev_, host.data(), arena, hipMemcpyHostToDevice), "upload codec weights");
    }
    auto fptr = [&](size_t o) { return reinterpret_cast<const float *>(wdev_ + o); };
    for (int i = 0; i < kCodecNq; ++i) {
        front_cb_[i] = fptr(o_cb[i]);
        front_w_[i] = fptr(o_cw[i]);
        front_b_[i] = fptr(o_cbias[i]);
    }
    qout_w_ = wdev_ + o_qw;
    qout_b_ = fptr(o_qb);
    for (int s = 0; s < kCodecStages; ++s) {
        stages_[s].in = wdev_ + o_in[s];
        stages_[s].out = wdev_ + o_out[s];
    }
    for (size_t i = 0; i < layers_.size(); ++i) {
        LayerW &L = layers_[i];
        const LayerOff &lo = loff[i];
        L.attn = wdev_ + lo.attn;
        L.proj = wdev_ + lo.proj;
        L.f1 = wdev_ + lo.f1;
        L.f2 = wdev_ + lo.f2;
        L.n1w = fptr(lo.n1w);
        L.n1b = fptr(lo.n1b);
        L.n2w = fptr(lo.n2w);
        L.n2b = fptr(lo.n2b);
        L.ls1 = fptr(lo.ls1);
        L.ls2 = fptr(lo.ls2);
    }

    // RoPE frequencies exactly as audio_rope forms them (audio_layer.cpp:34-35), in fp32
    float freq[kCodecHeadDim / 2];
    for (int i = 0; i < kCodecHeadDim / 2; ++i)
        freq[i] = std::exp(-std::log(10000.0f) * 2.0f * static_cast<float>(i) / kCodecHeadDim);
    hip_check(hipMalloc(&freq_, sizeof(freq)), "hipMalloc(freq)");
    hip_check(hipMemcpy(freq_, freq, sizeof(freq), hipMemcpyHostToDevice), "upload freq");

    c0_ = c0;
    alloc_work(work_, fmax_);
    hip_check(hipHostMalloc(&codes_host_, sizeof(int32_t) * kCodecNq * fmax_), "hipHostMalloc(codes)");
    hip_check(hipHostMalloc(&out_host_, sizeof(float) * (size_t)fmax_ * spf_), "hipHostMalloc(samples)");
    for (auto &set : ev_)
        for (auto &e : set) hip_check(hipEventCreate(&e), "hipEventCreate");
    for (auto &e : done_) hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate");
    alloc_state(stream_state_, fmax_);
    clear_state(stream_state_);
    hip_check(hipStreamSynchronize(stream_), "codec init");

    char buf[160];
    std::snprintf(buf, sizeof(buf), "gpu decoder device=%d bytes=%zu ffn=%d windows=%d/%d/%d/%d pieces<=%d frames, decode %d",
                  device_, arena, ffn_max_, stages_[0].window, stages_[1].window, stages_[2].window, stages_[3].window,
                  fmax_, whole_max_);
    info_ = buf;
}

Codec::~Codec() {
    (void)hipSetDevice(device_);
    if (stream_) (void)hipStreamSynchronize(stream_);
    for (auto &kv : graphs_) (void)hipGraphExecDestroy(kv.second);
    free_state(stream_state_);
    free_state(whole_state_);
    free_work(work_);
    free_work(whole_work_);
    if (whole_codes_) (void)hipFree(whole_codes_);
    for (auto &set : ev_)
        for (auto &e : set)
            if (e) (void)hipEventDestroy(e);
    for (auto &e : done_)
        if (e) (void)hipEventDestroy(e);
    if (wdev_) (void)hipFree(wdev_);
    if (freq_) (void)hipFree(freq_);
    if (codes_host_) (void)hipHostFree(codes_host_);
    if (out_host_) (void)hipHostFree(out_host_);
    for (float *p : whole_host_)
        if (p) (void)hipHostFree(p);
    if (stream_) (void)hipStreamDestroy(stream_);
}

// Key splits of a stage's attention for a piece of `rows` rows: enough workgroups (row tiles x
// 4 heads x splits, of 8 waves) for one per CU, each split keeping >= 16 key blocks of 16 (two per
// wave) of the steady-state window.  Every column tile of proj merges all splits of its rows
// again, so twice as many splits of 4 waves made proj of an 8-frame chunk 8.4 us a launch where it is 5.2 now.
int Codec::splits_for(int stage, int rows) const {
    const int tiles = (rows + 15) / 16;
    const int blocks = (stages_[stage].window + 15 + 15) / 16;
    const int want = (256 + tiles * kCodecHeads - 1) / (tiles * kCodecHeads);
    return std::max(1, std::min(std::min(want, blocks / 16), kCodecMaxSplits));
}

namespace {
// Parts of one allocation, each on a 256-byte boundary: what they take in all, then where they lie.
struct Parts {
    uint8_t *base = nullptr;
    size_t bytes = 0;
    template <class T>
    void take(T *&p, size_t n) {
        p = base ? reinterpret_cast<T *>(base + bytes) : nullptr;
        bytes += align256(std::max<size_t>(n, 1) * sizeof(T));
    }
};
}  // namespace

// Buffers for pieces of up to `frames` frames.
void Codec::alloc_work(CodecWork &w, int frames) {
    size_t xmax = (size_t)frames * c0_;  // q.out output = stage 0 input
    for (int s = 0; s + 1 < kCodecStages; ++s) xmax = std::max(xmax, (size_t)stage_rows(frames, s) * stages_[s].cout);
    const size_t rmax = (size_t)stage_rows(frames, kCodecStages - 1);
    size_t part_rows = 0, rope_rows = 0;
    for (int f = 1; f <= frames; ++f)
        for (int s = 0; s < kCodecStages; ++s) {
            const int r = stage_rows(f, s);
            part_rows = std::max(part_rows, (size_t)splits_for(s, r) * r);
        }
    for (int s = 0; s < kCodecStages; ++s) rope_rows += stage_rows(frames, s);
    auto parts = [&](uint8_t *base) {
        Parts p{base};
        p.take(w.codes, (size_t)kCodecNq * frames);
        p.take(w.z, (size_t)frames * kCodecZ);
        p.take(w.xa, xmax);
        p.take(w.xb, xmax);
        p.take(w.y, rmax * kCodecDModel);
        p.take(w.qb, rmax * kCodecDModel);
        p.take(w.h, rmax * ffn_max_);
        p.take(w.ao, part_rows * kCodecDModel);
        p.take(w.ast, part_rows * kCodecHeads);
        p.take(w.rope, rope_rows * (kCodecHeadDim / 2));
        p.take(w.out, (size_t)frames * spf_);
        return p.bytes;
    };
    hip_check(hipMalloc(&w.mem, parts(nullptr)), "hipMalloc(codec activations)");
    parts(w.mem);
}

void Codec::free_work(CodecWork &w) {
    if (w.mem) (void)hipFree(w.mem);
    w = CodecWork{};
}

// What decode() keeps from its first call on: its state, its activations (the stream's serve where
// the caller sized the pieces), pinned room for the samples of one piece, or two, and the codes of
// the longest utterance so far.  All but the codes are made for the longest piece at once, one
// allocation each: grown with the pieces asked for, ring by ring, a handle's utterances of 30, 40, 70
// and 100 frames took 2.2, 2.9, 6.4 and 6.7 ms, now 0.8, 0.9, 1.2 and 1.4.
void Codec::ensure_whole(int frames, int pieces) {
    if (!whole_state_.mem) alloc_state(whole_state_, whole_max_);
    if (whole_max_ != fmax_ && !whole_work_.mem) alloc_work(whole_work_, whole_max_);
    for (int i = 0; i < std::min(pieces, 2); ++i)
        if (!whole_host_[i])
            hip_check(hipHostMalloc(&whole_host_[i], sizeof(float) * (size_t)whole_max_ * spf_), "hipHostMalloc(samples)");
    const size_t n = (size_t)kCodecNq * frames;
    if (n > whole_codes_n_) {
        if (whole_codes_) hip_check(hipFree(whole_codes_), "free codes");
        whole_codes_ = nullptr;
        whole_codes_n_ = 0;
        const size_t room = (n + 16383) / 16384 * 16384;  // 1024 frames more at a time
        hip_check(hipMalloc(&whole_codes_, sizeof(int32_t) * room), "hipMalloc(codes)");
        whole_codes_n_ = room;
    }
}

// Rings for pieces of up to `frames` frames.
void Codec::alloc_state(CodecState &st, int frames) {
    auto parts = [&](uint8_t *base) {
        Parts p{base};
        p.take(st.pos0, kCodecStages);
        st.k.clear();
        st.v.clear();
        for (int s = 0; s < kCodecStages; ++s) {
            st.ring[s] = stages_[s].window + stage_rows(frames, s);
            for (int n = 0; n < stages_[s].nlayers; ++n) {
                float *k, *v;
                p.take(k, (size_t)st.ring[s] * kCodecDModel);
                p.take(v, (size_t)st.ring[s] * kCodecDModel);
                st.k.push_back(k);
                st.v.push_back(v);
            }
        }
        return p.bytes;
    };
    const size_t bytes = parts(nullptr);
    hip_check(hipMalloc(&st.mem, bytes), "hipMalloc(codec rings)");
    parts(st.mem);
    // zero once: a ring slot is only read after this stream wrote it, but keep it finite
    hip_check(hipMemsetAsync(st.mem, 0, bytes, stream_), "clear rings");
}

void Codec::free_state(CodecState &st) {
    if (st.mem) (void)hipFree(st.mem);
    st = CodecState{};
}

void Codec::clear_state(CodecState &st) {
    hip_check(hipMemsetAsync(st.pos0, 0, sizeof(int) * kCodecStages, stream_), "reset positions");
}

void Codec::reset_stream() {
    hip_check(hipSetDevice(device_), "hipSetDevice");
    clear_state(stream_state_);
    hip_check(hipStreamSynchronize(stream_), "reset_stream");
}

void Codec::check_codes(const int32_t *codes, int frames) const {
    if (frames <= 0 || !codes) throw Status(MOSS_HIP_EINVAL, "frames must be > 0 and codes non-null");
    for (size_t i = 0; i < (size_t)kCodecNq * frames; ++i)
        if (codes[i] < 0 || codes[i] >= kCodecCb) throw Status(MOSS_HIP_EINVAL, "code out of [0, 1024)");
}

static void ok(int rc, const char *what) {
    if (rc != 0) throw Status(rc, std::string("codec launch failed: ") + what);
}

// The launches of one piece: front, q.out (+ patch 4), four stages, position advance.
void Codec::enqueue(CodecState &st, CodecWork &w, const int32_t *codes, int stride, int frames, hipEvent_t *stage_ev) {
    hipStream_t s = stream_;
    CodecFrontArgs fa;
    fa.codes = codes;
    fa.code_stride = stride;
    fa.frames = frames;
    fa.pos0 = st.pos0;
    fa.freq = freq_;
    float2 *rope = w.rope;
    for (int si = 0; si < kCodecStages; ++si) {
        fa.rows[si] = stage_rows(frames, si);
        fa.rope[si] = rope;
        rope += (size_t)fa.rows[si] * (kCodecHeadDim / 2);
    }
    for (int i = 0; i < kCodecNq; ++i) {
        fa.cb[i] = front_cb_[i];
        fa.cw[i] = front_w_[i];
        fa.cbias[i] = front_b_[i];
    }
    fa.z = w.z;
    ok(codec_front_launch(fa, s), "front");
    float *xin = w.xa, *xother = w.xb;
    {
        CodecGemmArgs g;
        g.a = w.z;
        g.lda = kCodecZ;
        g.w = qout_w_;
        g.w_f32 = qout_f32_;
        g.M = frames;
        g.N = stages_[0].cin * stages_[0].patch;
        g.K = kCodecZ;
        g.bias = qout_b_;
        g.y = xin;
        g.patch = stages_[0].patch;
        g.ldy = stages_[0].cin;
        ok(codec_gemm_launch(CPRO_ROWS, CEPI_STORE, g, s), "q.out");
    }
    int rows[kCodecStages];
    for (int si = 0; si < kCodecStages; ++si) {
        const StageW &S = stages_[si];
        const int M = stage_rows(frames, si);
        rows[si] = M;
        const int splits = splits_for(si, M);
        {
            CodecGemmArgs g;
            g.a = xin;
            g.lda = S.cin;
            g.w = S.in;
            g.w_f32 = S.in_f32;
            g.M = M;
            g.N = kCodecDModel;
            g.K = S.cin;
            g.y = w.y;
            g.ldy = kCodecDModel;
            ok(codec_gemm_launch(CPRO_ROWS, CEPI_STORE, g, s), "stage in");
        }
        for (int n = 0; n < S.nlayers; ++n) {
            const int li = S.layer0 + n;
            const LayerW &L = layers_[li];
            CodecGemmArgs q;
            q.a = w.y;
            q.lda = kCodecDModel;
            q.ln_w = L.n1w;
            q.ln_b = L.n1b;
            q.w = L.attn;
            q.w_f32 = L.attn_f32;
            q.M = M;
            q.N = 3 * kCodecDModel;
            q.K = kCodecDModel;
            q.q = w.qb;
            q.kc = st.k[li];
            q.vc = st.v[li];
            q.ring = st.ring[si];
            q.pos0 = st.pos0 + si;
            q.rope = fa.rope[si];
            ok(codec_gemm_launch(CPRO_LN, CEPI_QKV, q, s), "qkv");
            CodecAttnArgs a;
            a.q = w.qb;
            a.kc = st.k[li];
            a.vc = st.v[li];
            a.ring = st.ring[si];
            a.window = S.window;
            a.M = M;
            a.splits = splits;
            a.pos0 = st.pos0 + si;
            a.o = w.ao;
            a.st = w.ast;
            ok(codec_attn_launch(a, s), "attention");
            CodecGemmArgs p;
            if (splits > 1) {
                p.o = w.ao;
                p.st = w.ast;
                p.splits = splits;
            } else {
                p.a = w.ao;
                p.lda = kCodecDModel;
            }
            p.w = L.proj;
            p.w_f32 = L.proj_f32;
            p.M = M;
            p.N = kCodecDModel;
            p.K = kCodecDModel;
            p.y = w.y;
            p.ldy = kCodecDModel;
            p.ls = L.ls1;
            ok(codec_gemm_launch(splits > 1 ? CPRO_MERGE : CPRO_ROWS, CEPI_RESID, p, s), "proj");
            CodecGemmArgs f;
            f.a = w.y;
            f.lda = kCodecDModel;
            f.ln_w = L.n2w;
            f.ln_b = L.n2b;
            f.w = L.f1;
            f.w_f32 = L.f1_f32;
            f.M = M;
            f.N = L.ffn;
            f.K = kCodecDModel;
            f.y = w.h;
            f.ldy = L.ffn;
            ok(codec_gemm_launch(CPRO_LN, CEPI_GELU, f, s), "f1");
            CodecGemmArgs f2;
            f2.a = w.h;
            f2.lda = L.ffn;
            f2.w = L.f2;
            f2.w_f32 = L.f2_f32;
            f2.M = M;
            f2.N = kCodecDModel;
            f2.K = L.ffn;
            f2.y = w.y;
            f2.ldy = kCodecDModel;
            f2.ls = L.ls2;
            ok(codec_gemm_launch(CPRO_ROWS, CEPI_RESID, f2, s), "f2");
        }
        {
            CodecGemmArgs g;
            g.a = w.y;
            g.lda = kCodecDModel;
            g.w = S.out;
            g.w_f32 = S.out_f32;
            g.M = M;
            g.N = S.cout;
            g.K = kCodecDModel;
            if (si + 1 < kCodecStages) {
                g.y = xother;
                g.patch = stages_[si + 1].patch;
                g.ldy = stages_[si + 1].cin;
            } else {  // patch 240: the samples, row-major
                g.y = w.out;
                g.patch = kCodecFinalPatch;
                g.ldy = 1;
            }
            ok(codec_gemm_launch(CPRO_ROWS, CEPI_STORE, g, s), "stage out");
        }
        std::swap(xin, xother);
        if (stage_ev) hip_check(hipEventRecord(stage_ev[si + 1], s), "hipEventRecord");
    }
    ok(codec_advance_launch(st.pos0, rows, s), "advance");
}

void Codec::run_piece(CodecState &st, const int32_t *codes, int frames, float *out, bool graph) {
    hipStream_t s = stream_;
    hip_check(hipMemcpyAsync(work_.codes, codes, sizeof(int32_t) * kCodecNq * frames, hipMemcpyHostToDevice, s),
              "upload codes");
    if (graph) {
        auto it = graphs_.find(frames);
        if (it == graphs_.end()) {
            hipGraph_t g = nullptr;
            hipGraphExec_t ge = nullptr;
            hip_check(hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal), "begin capture");
            try {
                enqueue(st, work_, work_.codes, frames, frames, nullptr);
            } catch (...) {
                (void)hipStreamEndCapture(s, &g);
                if (g) (void)hipGraphDestroy(g);
                throw;
            }
            hip_check(hipStreamEndCapture(s, &g), "end capture");
            const hipError_t e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
            (void)hipGraphDestroy(g);
            hip_check(e, "hipGraphInstantiate");
            it = graphs_.emplace(frames, ge).first;
        }
        hip_check(hipGraphLaunch(it->second, s), "hipGraphLaunch");
    } else {
        enqueue(st, work_, work_.codes, frames, frames, nullptr);
    }
    const size_t n = (size_t)frames * spf_;
    hip_check(hipMemcpyAsync(out_host_, work_.out, n * sizeof(float), hipMemcpyDeviceToHost, s), "download samples");
    hip_check(hipStreamSynchronize(s), "codec piece");
    std::memcpy(out, out_host_, n * sizeof(float));
}

// codes [16][frames] -> the piece [f0, f0 + n) gathered into the pinned staging buffer
static void gather_codes(const int32_t *codes, int frames, int f0, int n, int32_t *dst) {
    for (int i = 0; i < kCodecNq; ++i) std::memcpy(dst + (size_t)i * n, codes + (size_t)i * frames + f0, sizeof(int32_t) * n);
}

void Codec::decode_chunk(const int32_t *codes, int frames, float *out) {
    check_codes(codes, frames);
    hip_check(hipSetDevice(device_), "hipSetDevice");
    for (int f0 = 0; f0 < frames; f0 += fmax_) {
        const int n = std::min(fmax_, frames - f0);
        gather_codes(codes, frames, f0, n, codes_host_);
        run_piece(stream_state_, codes_host_, n, out + (size_t)f0 * spf_, !eager_);
    }
}

void Codec::decode(const int32_t *codes, int frames, float *out) {
    check_codes(codes, frames);
    const auto t0 = std::chrono::steady_clock::now();
    hip_check(hipSetDevice(device_), "hipSetDevice");
    // Equal pieces, each a long run of launches: while one computes, the host copies the samples
    // of the one before out of pinned memory.  (32-frame pieces, each waited for: 6.7 ms for 203
    // frames, a third of it launches too small for the chip and the copy.)
    const int pieces = (frames + whole_max_ - 1) / whole_max_, piece = (frames + pieces - 1) / pieces;
    ensure_whole(frames, pieces);
    CodecWork &work = whole_work_.mem ? whole_work_ : work_;
    clear_state(whole_state_);
    hip_check(hipMemcpyAsync(whole_codes_, codes, sizeof(int32_t) * kCodecNq * frames, hipMemcpyHostToDevice, stream_),
              "upload codes");
    double stage[kCodecStages] = {0, 0, 0, 0};
    auto finish = [&](int p) {  // the samples and stage times of piece p
        const int b = p & 1, f0 = p * piece, n = std::min(piece, frames - f0);
        hip_check(hipEventSynchronize(done_[b]), "codec decode");
        std::memcpy(out + (size_t)f0 * spf_, whole_host_[b], (size_t)n * spf_ * sizeof(float));
        for (int s = 0; s < kCodecStages; ++s) {
            float ms = 0.f;
            hip_check(hipEventElapsedTime(&ms, ev_[b][s], ev_[b][s + 1]), "hipEventElapsedTime");
            stage[s] += ms;
        }
    };
    for (int p = 0; p < pieces; ++p) {
        const int b = p & 1, f0 = p * piece, n = std::min(piece, frames - f0);
        hip_check(hipEventRecord(ev_[b][0], stream_), "hipEventRecord");
        enqueue(whole_state_, work, whole_codes_ + f0, frames, n, ev_[b]);
        hip_check(hipMemcpyAsync(whole_host_[b], work.out, (size_t)n * spf_ * sizeof(float), hipMemcpyDeviceToHost,
                                 stream_),
                  "download samples");
        hip_check(hipEventRecord(done_[b], stream_), "hipEventRecord");
        if (p > 0) finish(p - 1);
    }
    finish(pieces - 1);
    for (int s = 0; s < kCodecStages; ++s) stage_ms_[s] = stage[s];
    last_ms_ = std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t0).count();
}

}  // namespace mh
