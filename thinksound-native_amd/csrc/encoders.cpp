// encoders.cpp — ClipModel and T5Model: the reference's text encoders on HIP (src/clip.cpp, src/t5.cpp).
#include "encoders.h"

#include <math.h>
#include <string.h>

#include <algorithm>
#include <map>

#include "gguf.h"

namespace tsn {

namespace {

struct Layout {   // device arena: named regions at float offsets
    std::map<std::string, size_t> at;
    size_t size = 0;
    size_t put(const std::string &n, size_t numel) {
        at[n] = size;
        size += (numel + 3) & ~(size_t)3;   // 16-byte aligned regions
        return at[n];
    }
};

// stage the host tensors into the arena layout (the tensors of `group` go one after the other at
// the region of group[0]), upload once
int fill_arena(Runtime *rt, const std::vector<ManifestEntry> &man, const float *host, const Layout &lay,
               const std::map<std::string, std::pair<std::string, size_t>> &group, float *dev) {
    std::vector<float> stage(lay.size, 0.0f);
    for (const auto &e : man) {
        size_t dst;
        const auto g = group.find(e.name);
        if (g != group.end()) dst = lay.at.at(g->second.first) + g->second.second;
        else dst = lay.at.at(e.name);
        memcpy(stage.data() + dst, host + e.offset, (size_t)e.numel * sizeof(float));
    }
    return rt->dev.upload(dev, stage.data(), stage.size() * sizeof(float));
}

} // namespace

int t5_bucket(int rel, int n_bucket, int max_dist) {
    const int half = n_bucket / 2;
    int b = rel > 0 ? half : 0;
    const int n = rel < 0 ? -rel : rel;
    const int exact = half / 2;
    if (n < exact) return b + n;
    const int v = exact + (int)(log((double)n / exact) / log((double)max_dist / exact) * (half - exact));
    return b + std::min(v, half - 1);
}

/* ---------------- specs and manifests ---------------- */

ClipSpec clip_spec_default() { return ClipSpec{1024, 24, 16, 77, 49408, 1e-5f}; }
T5Spec t5_spec_default() { return T5Spec{2048, 5120, 24, 32, 77, 32128, 32, 128, 1e-6f}; }

int clip_spec_check(const ClipSpec &s) {
    TSN_REQUIRE(s.H > 0 && s.H % 64 == 0 && s.NH * 64 == s.H, "clip spec: heads of 64 (H = 64 NH)");
    TSN_REQUIRE(s.NL > 0 && s.ctx > 0 && s.ctx <= 128 && s.vocab > 0, "clip spec: layers, context 1..128, vocabulary");
    return TSN_OK;
}

int t5_spec_check(const T5Spec &s) {
    TSN_REQUIRE(s.d > 0 && s.d % 64 == 0 && s.NH * 64 == s.d, "t5 spec: heads of 64 (d = 64 NH)");
    TSN_REQUIRE(s.d_ff > 0 && s.d_ff % 32 == 0, "t5 spec: d_ff a multiple of 32");
    TSN_REQUIRE(s.NL > 0 && s.ctx > 0 && s.ctx <= 128 && s.vocab > 0, "t5 spec: layers, context 1..128, vocabulary");
    TSN_REQUIRE(s.n_bucket >= 4 && s.n_bucket % 4 == 0 && s.max_dist > s.n_bucket / 4,
                "t5 spec: relative buckets (a multiple of 4) and a max distance past the exact range");
    return TSN_OK;
}

int clip_spec_from_gguf(const char *path, ClipSpec *out) {
    TSN_REQUIRE(out, "clip gguf: null spec");
    GgufReader g;
    TSN_TRY(g.open(path));
    ClipSpec s = clip_spec_default();
    s.H = (int)g.get_i64("clip.hidden", s.H);
    s.NL = (int)g.get_i64("clip.layers", s.NL);
    s.NH = (int)g.get_i64("clip.heads", s.NH);
    s.ctx = (int)g.get_i64("clip.ctx", s.ctx);
    if (const GgufTensorInfo *t = g.find("tok_emb")) s.vocab = (int)t->ne[1];
    TSN_TRY(clip_spec_check(s));
    *out = s;
    return TSN_OK;
}

int t5_spec_from_gguf(const char *path, T5Spec *out) {
    TSN_REQUIRE(out, "t5 gguf: null spec");
    GgufReader g;
    TSN_TRY(g.open(path));
    T5Spec s = t5_spec_default();
    s.d = (int)g.get_i64("t5.d_model", s.d);
    s.d_ff = (int)g.get_i64("t5.d_ff", s.d_ff);
    s.NL = (int)g.get_i64("t5.n_layers", s.NL);
    s.NH = (int)g.get_i64("t5.n_heads", s.NH);
    s.n_bucket = (int)g.get_i64("t5.rel_buckets", s.n_bucket);
    s.max_dist = (int)g.get_i64("t5.rel_max_dist", s.max_dist);
    s.eps = (float)g.get_f64("t5.eps", s.eps);
    if (const GgufTensorInfo *t = g.find("tok_emb")) s.vocab = (int)t->ne[1];
    TSN_TRY(t5_spec_check(s));
    *out = s;
    return TSN_OK;
}

std::vector<ManifestEntry> clip_manifest(const ClipSpec &s) {
    std::vector<ManifestEntry> v;
    int64_t off = 0;
    auto add = [&](const std::string &n, int64_t numel) {
        v.push_back({n, numel, off});
        off += numel;
    };
    const int64_t H = s.H;
    add("tok_emb", (int64_t)s.vocab * H);
    add("pos_emb", (int64_t)s.ctx * H);
    for (int l = 0; l < s.NL; ++l) {
        const std::string b = "blk." + std::to_string(l);
        add(b + ".ln1.w", H); add(b + ".ln1.b", H);
        add(b + ".q.w", H * H); add(b + ".q.b", H);
        add(b + ".k.w", H * H); add(b + ".k.b", H);
        add(b + ".v.w", H * H); add(b + ".v.b", H);
        add(b + ".out.w", H * H); add(b + ".out.b", H);
        add(b + ".ln2.w", H); add(b + ".ln2.b", H);
        add(b + ".fc1.w", 4 * H * H); add(b + ".fc1.b", 4 * H);
        add(b + ".fc2.w", H * 4 * H); add(b + ".fc2.b", H);
    }
    add("out_ln.w", H);
    add("out_ln.b", H);
    add("text_proj", H * H);
    return v;
}

std::vector<ManifestEntry> t5_manifest(const T5Spec &s) {
    std::vector<ManifestEntry> v;
    int64_t off = 0;
    auto add = [&](const std::string &n, int64_t numel) {
        v.push_back({n, numel, off});
        off += numel;
    };
    const int64_t d = s.d, F = s.d_ff;
    add("tok_emb", (int64_t)s.vocab * d);
    for (int l = 0; l < s.NL; ++l) {
        const std::string b = "blk." + std::to_string(l);
        add(b + ".attn_norm", d);
        add(b + ".q", d * d); add(b + ".k", d * d); add(b + ".v", d * d); add(b + ".o", d * d);
        add(b + ".ffn_norm", d);
        add(b + ".wi_0", F * d); add(b + ".wi_1", F * d); add(b + ".wo", d * F);
    }
    add("rel_bias", (int64_t)s.n_bucket * s.NH);
    add("out_norm", d);
    return v;
}

// K splits of a QKV GEMM: attention reads every split of k and v in each of a head's workgroups. 77 rows, 1024
// wide: 2 splits 4% a prompt more than 4; 2048 wide: 4 and 2 the same, 5 2% more.
constexpr int QKV_SPLITS = 4;

int EncoderRunner::create_common(int ctx, int width, int ffn, int ffn_cols) {
    TSN_TRY(alloc(enc_operand_bytes(ctx, width), (void **)&A_));
    TSN_TRY(alloc(enc_operand_bytes(ctx, ffn), (void **)&F_));
    ws_bytes_ = std::max(ENC_WS_BYTES, (size_t)ctx * std::max(3 * (size_t)width, (size_t)ffn_cols) * sizeof(float));
    return alloc(ws_bytes_, (void **)&ws_);
}

int EncoderRunner::gemm(const uint16_t *A, const float *W, const float *b, int M, int N, int K, EncParts &out, int most) {
    EncGemmArgs g{A, W, ws_, ws_bytes_, M, N, K, most, 1, 0};
    TSN_TRY(run("enc_gemm_kernel", 2.0 * M * N * K, 4.0 * ((double)N * K + M * (double)N) + 6.0 * M * (double)K,
                [&] { return launch_enc_gemm(g, rt->dev.stream()); }));
    out = EncParts{ws_, (long long)M * N, g.splits, N, b};
    return TSN_OK;
}

int EncoderRunner::pack_weights(const std::vector<RawWeight> &ws) {
    size_t most = 0;
    for (const RawWeight &w : ws) most = std::max(most, (size_t)w.N * w.K * sizeof(float));
    void *tmp;
    TSN_TRY(alloc(most, &tmp));
    const hipStream_t st = rt->dev.stream();
    for (const RawWeight &w : ws) {
        TSN_TRY(rt->dev.copy_d2d(tmp, w.p, (size_t)w.N * w.K * sizeof(float)));
        TSN_TRY(launch_enc_weight_pack((const float *)tmp, w.p, w.N, w.K, st));
    }
    return release(tmp);
}

/* ---------------- CLIP ---------------- */

int ClipModel::create(Runtime *r, const ClipSpec &sp) {
    TSN_REQUIRE(r, "clip: null runtime");
    TSN_TRY(clip_spec_check(sp));
    rt = r;
    s = sp;
    const size_t n = s.ctx, H = s.H;
    TSN_TRY(alloc(n * H * 4, (void **)&X_));
    return create_common(s.ctx, s.H, 4 * s.H, 4 * s.H);
}

int ClipModel::upload_weights(const float *host, size_t numel) { return upload(host, numel); }

int ClipModel::load_gguf(const char *path) {
    GgufReader g;
    TSN_TRY(g.open(path));
    std::vector<float> host;
    TSN_TRY(gguf_read_manifest(g, clip_manifest(s), host));
    return upload(host.data(), host.size());
}

int ClipModel::upload(const float *host, size_t numel) {
    TSN_REQUIRE(rt && host, "clip: not created / null weights");
    TSN_REQUIRE(!ready_, "clip: weights already uploaded");
    const auto man = clip_manifest(s);
    const size_t total = (size_t)(man.back().offset + man.back().numel);
    TSN_REQUIRE(numel == total, "clip: weight count does not match the manifest (" + std::to_string(total) + ")");
    const size_t H = s.H;
    Layout lay;
    std::map<std::string, std::pair<std::string, size_t>> group;
    for (const auto &e : man) {
        const std::string &n = e.name;
        const std::string stem = n.compare(0, 4, "blk.") == 0 ? n.substr(0, n.find('.', 4)) : "";
        const std::string leaf = stem.empty() ? n : n.substr(stem.size() + 1);
        if (leaf == "q.w" || leaf == "k.w" || leaf == "v.w") {   // one [3H][H] weight per layer
            const size_t j = leaf[0] == 'q' ? 0 : leaf[0] == 'k' ? 1 : 2;
            if (j == 0) lay.put(stem + ".qkv.w", enc_weight_floats(3 * s.H, s.H));
            group[n] = {stem + ".qkv.w", j * H * H};
        } else if (leaf == "q.b" || leaf == "k.b" || leaf == "v.b") {
            const size_t j = leaf[0] == 'q' ? 0 : leaf[0] == 'k' ? 1 : 2;
            if (j == 0) lay.put(stem + ".qkv.b", 3 * H);
            group[n] = {stem + ".qkv.b", j * H};
        } else {
            lay.put(n, (size_t)e.numel);
        }
    }
    float *dev;
    TSN_TRY(alloc(lay.size * sizeof(float), (void **)&dev));
    TSN_TRY(fill_arena(rt, man, host, lay, group, dev));
    auto P = [&](const std::string &n) { return (const float *)(dev + lay.at.at(n)); };
    tok_ = P("tok_emb");
    pos_ = P("pos_emb");
    L_.resize(s.NL);
    std::vector<RawWeight> pw;
    for (int l = 0; l < s.NL; ++l) {
        const std::string b = "blk." + std::to_string(l);
        Layer &L = L_[l];
        L.ln1w = P(b + ".ln1.w"); L.ln1b = P(b + ".ln1.b"); L.bqkv = P(b + ".qkv.b"); L.bo = P(b + ".out.b");
        L.ln2w = P(b + ".ln2.w"); L.ln2b = P(b + ".ln2.b"); L.b1 = P(b + ".fc1.b"); L.b2 = P(b + ".fc2.b");
        L.Wqkv = P(b + ".qkv.w"); L.Wo = P(b + ".out.w"); L.W1 = P(b + ".fc1.w"); L.W2 = P(b + ".fc2.w");
        pw.push_back({dev + lay.at.at(b + ".qkv.w"), 3 * s.H, s.H});
        pw.push_back({dev + lay.at.at(b + ".out.w"), s.H, s.H});
        pw.push_back({dev + lay.at.at(b + ".fc1.w"), 4 * s.H, s.H});
        pw.push_back({dev + lay.at.at(b + ".fc2.w"), s.H, 4 * s.H});
    }
    lnw_ = P("out_ln.w");
    lnb_ = P("out_ln.b");
    proj_ = P("text_proj");
    TSN_TRY(pack_weights(pw));
    ready_ = true;
    return TSN_OK;
}

int ClipModel::encode(const int32_t *ids, float *per_token, float *global) {
    TSN_REQUIRE(ready_, "clip: weights not uploaded");
    TSN_REQUIRE(ids && per_token && global, "clip: null ids or outputs");
    const int n = s.ctx, H = s.H;
    int eos = 0;
    EncIds id{};
    for (int i = 0; i < n; ++i) {
        TSN_REQUIRE(ids[i] >= 0 && ids[i] < s.vocab, "clip: token id outside the vocabulary");
        if (ids[i] > ids[eos]) eos = i;   // first position of the largest id (src/clip.cpp:45-46)
        id.id[i] = ids[i];
    }
    TSN_TRY(rt->dev.make_current());
    const hipStream_t st = rt->dev.stream();
    const int mt = enc_row_blocks(n);
    // X += the pending GEMM result (if any), then LN into the operand A_ or, last, per_token
    auto norm = [&](const EncParts &p, const float *w, const float *b, float *y) {
        EncNormArgs a{X_, X_, p, w, b, y, y ? nullptr : A_, mt, n, H, s.eps};
        return run("enc_norm_kernel<true>", 0, 4.0 * n * H * (p.ws ? p.splits + 3 : 2),
                   [&] { return launch_enc_norm(a, true, st); });
    };
    EncParts p{}, none{};
    TSN_TRY(run("embed_rows_kernel", 0, 12.0 * n * H, [&] { return launch_embed_rows(id, tok_, pos_, X_, n, H, st); }));
    for (int l = 0; l < s.NL; ++l) {
        const Layer &w = L_[l];
        TSN_TRY(norm(l ? p : none, w.ln1w, w.ln1b, nullptr));
        TSN_TRY(gemm(A_, w.Wqkv, w.bqkv, n, 3 * H, H, p, QKV_SPLITS));
        EncAttnArgs a{p, A_, mt, n, s.NH, 0.125f, 2, nullptr, {0, 0, 0, 0}, eos};
        TSN_TRY(run("enc_attn_kernel", 4.0 * s.NH * n * (double)n * 64, 4.0 * n * H * (3 * p.splits + 1.5),
                    [&] { return launch_enc_attention(a, st); }));
        TSN_TRY(gemm(A_, w.Wo, w.bo, n, H, H, p));
        TSN_TRY(norm(p, w.ln2w, w.ln2b, nullptr));
        TSN_TRY(gemm(A_, w.W1, w.b1, n, 4 * H, H, p));
        TSN_TRY(run("enc_act_kernel<false>", 0, 4.0 * n * 4 * H * (p.splits + 1.5),
                    [&] { return launch_enc_act(p, false, F_, n, 4 * H, st); }));
        TSN_TRY(gemm(F_, w.W2, w.b2, n, H, 4 * H, p));
    }
    TSN_TRY(norm(p, lnw_, lnb_, per_token));
    // pooled: text_proj · per_token[eos] (src/clip.cpp:88-91)
    GemvArgs v;
    memset(&v, 0, sizeof v);
    v.W = proj_; v.ldw = H; v.wdt = DT_F32; v.X = per_token + (size_t)eos * H; v.ldx = H; v.Y = global; v.ldy = H;
    v.N = H; v.K = H; v.nb = 1;
    return run("gemv_kernel", 2.0 * H * H, 4.0 * H * H, [&] { return launch_gemv(v, st); });
}

/* ---------------- T5 ---------------- */

int T5Model::create(Runtime *r, const T5Spec &sp) {
    TSN_REQUIRE(r, "t5: null runtime");
    TSN_TRY(t5_spec_check(sp));
    rt = r;
    s = sp;
    const size_t n = s.ctx, d = s.d;
    TSN_TRY(alloc(n * d * 4, (void **)&X_));
    TSN_TRY(alloc((2 * n - 1) * s.NH * 4, (void **)&rel_));
    return create_common(s.ctx, s.d, s.d_ff, 2 * s.d_ff);
}

int T5Model::upload_weights(const float *host, size_t numel) { return upload(host, numel); }

int T5Model::load_gguf(const char *path) {
    GgufReader g;
    TSN_TRY(g.open(path));
    std::vector<float> host;
    TSN_TRY(gguf_read_manifest(g, t5_manifest(s), host));
    return upload(host.data(), host.size());
}

int T5Model::upload(const float *host, size_t numel) {
    TSN_REQUIRE(rt && host, "t5: not created / null weights");
    TSN_REQUIRE(!ready_, "t5: weights already uploaded");
    const auto man = t5_manifest(s);
    const size_t total = (size_t)(man.back().offset + man.back().numel);
    TSN_REQUIRE(numel == total, "t5: weight count does not match the manifest (" + std::to_string(total) + ")");
    const size_t d = s.d, F = s.d_ff;
    Layout lay;
    std::map<std::string, std::pair<std::string, size_t>> group;
    for (const auto &e : man) {
        const std::string &n = e.name;
        const std::string stem = n.compare(0, 4, "blk.") == 0 ? n.substr(0, n.find('.', 4)) : "";
        const std::string leaf = stem.empty() ? n : n.substr(stem.size() + 1);
        if (leaf == "q" || leaf == "k" || leaf == "v") {
            const size_t j = leaf == "q" ? 0 : leaf == "k" ? 1 : 2;
            if (j == 0) lay.put(stem + ".qkv", enc_weight_floats(3 * s.d, s.d));
            group[n] = {stem + ".qkv", j * d * d};
        } else if (leaf == "wi_0" || leaf == "wi_1") {   // one [2F][d] weight: wi_0 rows, then wi_1 rows
            const size_t j = leaf == "wi_0" ? 0 : 1;
            if (j == 0) lay.put(stem + ".wi", enc_weight_floats(2 * s.d_ff, s.d));
            group[n] = {stem + ".wi", j * F * d};
        } else if (leaf == "wo") {
            lay.put(n, enc_weight_floats(s.d, s.d_ff));
        } else {
            lay.put(n, (size_t)e.numel);
        }
    }
    float *dev;
    TSN_TRY(alloc(lay.size * sizeof(float), (void **)&dev));
    TSN_TRY(fill_arena(rt, man, host, lay, group, dev));
    auto P = [&](const std::string &n) { return (const float *)(dev + lay.at.at(n)); };
    tok_ = P("tok_emb");
    L_.resize(s.NL);
    std::vector<RawWeight> pw;
    auto at = [&](const std::string &n) {   // host tensor
        return host + std::find_if(man.begin(), man.end(), [&](const ManifestEntry &e) { return e.name == n; })->offset;
    };
    for (int l = 0; l < s.NL; ++l) {
        const std::string b = "blk." + std::to_string(l);
        Layer &L = L_[l];
        L.an = P(b + ".attn_norm"); L.fn = P(b + ".ffn_norm");
        L.Wqkv = P(b + ".qkv"); L.Wo = P(b + ".o"); L.Wi = P(b + ".wi"); L.Wout = P(b + ".wo");
        pw.push_back({dev + lay.at.at(b + ".qkv"), 3 * s.d, s.d});
        pw.push_back({dev + lay.at.at(b + ".o"), s.d, s.d});
        pw.push_back({dev + lay.at.at(b + ".wi"), 2 * s.d_ff, s.d});
        pw.push_back({dev + lay.at.at(b + ".wo"), s.d, s.d_ff});
    }
    on_ = P("out_norm");
    // the bias of each head by distance k - q in -(ctx - 1) .. ctx - 1: bucket(k - q) (src/t5.cpp:47-53)
    const float *rb = at("rel_bias");
    const int span = 2 * s.ctx - 1;
    std::vector<float> rel((size_t)span * s.NH);
    for (int h = 0; h < s.NH; ++h)
        for (int i = 0; i < span; ++i)
            rel[(size_t)h * span + i] = rb[(size_t)t5_bucket(i - (s.ctx - 1), s.n_bucket, s.max_dist) * s.NH + h];
    TSN_TRY(rt->dev.upload(rel_, rel.data(), rel.size() * sizeof(float)));
    TSN_TRY(pack_weights(pw));
    ready_ = true;
    return TSN_OK;
}

int T5Model::encode(const int32_t *ids, float *out) {
    TSN_REQUIRE(ready_, "t5: weights not uploaded");
    TSN_REQUIRE(ids && out, "t5: null ids or output");
    const int n = s.ctx, d = s.d, F = s.d_ff;
    EncIds id{};
    uint32_t keys[4] = {0, 0, 0, 0};
    for (int i = 0; i < n; ++i) {
        TSN_REQUIRE(ids[i] >= 0 && ids[i] < s.vocab, "t5: token id outside the vocabulary");
        id.id[i] = ids[i];
        if (ids[i] != 0) keys[i >> 5] |= 1u << (i & 31);   // keys of id 0 (pad) masked (src/t5.cpp:90-94)
    }
    TSN_TRY(rt->dev.make_current());
    const hipStream_t st = rt->dev.stream();
    const int mt = enc_row_blocks(n);
    // X += the pending GEMM result (if any), then RMS into the operand A_ or, last, out
    auto rms = [&](const EncParts &p, const float *w, float *y) {
        EncNormArgs a{X_, X_, p, w, nullptr, y, y ? nullptr : A_, mt, n, d, s.eps};
        return run("enc_norm_kernel<false>", 0, 4.0 * n * d * (p.ws ? p.splits + 3 : 2),
                   [&] { return launch_enc_norm(a, false, st); });
    };
    EncParts p{}, none{};
    TSN_TRY(run("embed_rows_kernel", 0, 8.0 * n * d, [&] { return launch_embed_rows(id, tok_, nullptr, X_, n, d, st); }));
    for (int l = 0; l < s.NL; ++l) {
        const Layer &w = L_[l];
        TSN_TRY(rms(l ? p : none, w.an, nullptr));
        TSN_TRY(gemm(A_, w.Wqkv, nullptr, n, 3 * d, d, p, QKV_SPLITS));
        // scale 1: T5 folds 1/sqrt(d_kv) into q (src/t5.cpp:70)
        EncAttnArgs a{p, A_, mt, n, s.NH, 1.0f, 1, rel_, {keys[0], keys[1], keys[2], keys[3]}, 0};
        TSN_TRY(run("enc_attn_kernel", 4.0 * s.NH * n * (double)n * 64, 4.0 * n * d * (3 * p.splits + 1.5),
                    [&] { return launch_enc_attention(a, st); }));
        TSN_TRY(gemm(A_, w.Wo, nullptr, n, d, d, p));
        TSN_TRY(rms(p, w.fn, nullptr));
        TSN_TRY(gemm(A_, w.Wi, nullptr, n, 2 * F, d, p));
        TSN_TRY(run("enc_act_kernel<true>", 0, 4.0 * n * F * (2 * p.splits + 1.5),
                    [&] { return launch_enc_act(p, true, F_, n, F, st); }));
        TSN_TRY(gemm(F_, w.Wout, nullptr, n, d, F, p));
    }
    return rms(p, on_, out);
}

} // namespace tsn
