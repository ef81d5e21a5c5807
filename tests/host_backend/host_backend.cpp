// backend.cpp over the host HIP calls of hip/hip_runtime.h, with kernels that
// only move rows: copies copy, a decode step appends a row that names itself,
// rotating a key leaves it as it is (so a window's rotated rows equal its
// keys). What each scenario shows is the order of the host's and the streams'
// accesses and what the error paths leave behind.
//
// host_backend SCENARIO: prints "ok" or the first difference.
#include "../../plamo-3-translate.c_amd/csrc/backend.cpp"

#include <memory>
#include <string>

#include "../../include/plamo_synthetic.h"

namespace plamo {
static int fail_after = -1;  // launches until one fails; -1: none

static hipError_t queue(hipStream_t s, std::function<void()> f = [] {}) {
    if (fail_after >= 0 && fail_after-- == 0) return hipErrorInvalidValue;
    s->add(std::move(f));
    return hipSuccess;
}

hipError_t launch_copy_rows(hipStream_t s, const CopyRow *table, uint32_t entries) {
    if (!entries) return hipSuccess;
    return queue(s, [=] {
        for (uint32_t i = 0; i < entries; ++i)
            memcpy(table[i].dst, table[i].src, table[i].floats * 4);
    });
}
hipError_t launch_copy_block(hipStream_t s, const void *src, void *dst, uint64_t bytes) {
    return queue(s, [=] { memcpy(dst, src, bytes); });
}
hipError_t launch_copy_blocks(hipStream_t s, const CopyBlocks &b) {
    return queue(s, [=] {
        for (uint32_t i = 0; i < b.count; ++i) memcpy(b.dst[i], b.src[i], b.words[i] * 4);
    });
}
hipError_t launch_rerotate(hipStream_t s, const float *k, float *rot, const float *, uint64_t rows,
                           uint32_t kh, uint32_t dim) {
    return queue(s, [=] { memcpy(rot, k, rows * kh * dim * 4); });
}
hipError_t launch_embed(hipStream_t s, const uint16_t *, const uint32_t *, const StepParams *params,
                        uint32_t, uint32_t, float *, StepParams *publish) {
    return queue(s, [=] {
        if (publish) *publish = *params;
    });
}
hipError_t launch_gemv(hipStream_t s, const uint16_t *, uint64_t rows, uint64_t,
                       const Prologue &pro, float *y, uint64_t half, int) {
    return queue(s, [=] {
        memset(y, 0, (half ? half : rows) * 4);
        if (pro.status_out) *pro.status_out = *pro.status;
    });
}
// The new row of layer l at count n: 1000 (l + 1) + n + token / 128, V its negative.
static float row_value(uint32_t layer, uint32_t count, uint32_t token) {
    return 1000.0f * (layer + 1) + count + token / 128.0f;
}
static void append_row(const DecodeAttention &a) {
    const uint32_t width = a.kh * a.dim, count = a.params->count[a.layer];
    const float x = row_value(a.layer, count, a.params->token);
    const uint64_t at = (uint64_t)count * width;
    for (uint32_t i = 0; i < width; ++i) {
        a.k_raw[at + i] = a.k_rot[at + i] = x;
        a.v[at + i] = -x;
        if (a.stage) {
            a.stage[i] = a.stage[2 * width + i] = x;
            a.stage[width + i] = -x;
        }
        if (a.host_k) a.host_k[at + i] = a.host_rot[at + i] = x;
        if (a.host_v) a.host_v[at + i] = -x;
    }
}
hipError_t launch_decode_attention(hipStream_t s, const DecodeAttention &a) {
    return queue(s, [=] { append_row(a); });
}
hipError_t launch_attention_o(hipStream_t s, const AttentionO &f) {
    return queue(s, [=] { append_row(f.a); });
}
bool decode_attention_supported(uint32_t, uint32_t) { return true; }
bool attention_o_supported(uint32_t, uint32_t, uint64_t) { return true; }
uint32_t decode_attention_splits(uint64_t) { return 1; }
hipError_t launch_fill(hipStream_t s, uint32_t *p, uint64_t words, uint32_t value) {
    return queue(s, [=] { std::fill(p, p + words, value); });
}
hipError_t configure_gemv(uint64_t) { return hipSuccess; }

// Not looked at here: launched, without effect.
hipError_t launch_rope_table(hipStream_t s, const float *, float, uint32_t, uint64_t, uint64_t,
                             float *, bool) {
    return queue(s);
}
uint64_t gemm_plane_elems(uint64_t tokens, uint64_t cols) { return 3 * tokens * cols; }
hipError_t launch_gemm(hipStream_t s, const float *, uint64_t, const uint16_t *, uint64_t, uint64_t,
                       uint64_t, float *, uint64_t, const GemmWorkspace *, bool) {
    return queue(s);
}
uint32_t gemm_planes_rows(uint64_t, uint64_t, const GemmWorkspace *) { return 0; }
uint16_t *gemm_swiglu_planes(uint64_t, uint64_t, uint64_t, const GemmWorkspace *) { return nullptr; }
PairWeight pair_rows_from(const PairWeight &w, uint32_t) { return w; }
bool pair_supported(uint64_t, uint64_t) { return true; }
uint64_t pair_frag_elems(uint64_t rows, uint64_t cols) { return rows * cols; }
uint64_t pair_exp_count(uint64_t rows) { return rows; }
uint32_t pair_padded(uint64_t tokens) { return (uint32_t)tokens; }
hipError_t launch_pair_weights(hipStream_t s, const uint16_t *, const PairWeight &, float *,
                               const int32_t *) {
    return queue(s);
}
hipError_t launch_pair_rows(hipStream_t s, const float *, uint64_t, uint64_t, uint64_t,
                            const PairRows &) {
    return queue(s);
}
hipError_t launch_pair_balance(hipStream_t s, const float *, uint64_t, int32_t *, float *) {
    return queue(s);
}
hipError_t launch_gemm_pair(hipStream_t s, const PairRows &, const PairWeight &, uint64_t, float *,
                            uint64_t, const GemmWorkspace &) {
    return queue(s);
}
hipError_t launch_gemm_pair_swiglu(hipStream_t s, const PairRows &, const PairWeight &, uint64_t,
                                   const PairRows &, const GemmWorkspace &) {
    return queue(s);
}
hipError_t launch_norm_rows(hipStream_t s, const float *, uint64_t, const uint16_t *, float,
                            float *, uint64_t, uint64_t, uint64_t, const PairRows *,
                            const SplitRows *) {
    return queue(s);
}
hipError_t launch_residual_norm_rows(hipStream_t s, float *, const float *, const uint16_t *, float,
                                     const uint16_t *, float, float *, uint64_t, uint64_t, uint64_t,
                                     const PairRows *, const SplitRows *) {
    return queue(s);
}
hipError_t launch_residual_rows(hipStream_t s, float *, const float *, const uint16_t *, float,
                                uint64_t, uint64_t) {
    return queue(s);
}
hipError_t launch_swiglu_rows(hipStream_t s, const float *, float *, uint64_t, uint64_t) {
    return queue(s);
}
hipError_t launch_gemm_swiglu(hipStream_t s, const float *, uint64_t, const uint16_t *, uint64_t,
                              uint64_t, uint64_t, float *, float *, const GemmWorkspace *, bool,
                              uint16_t *) {
    return queue(s);
}
hipError_t launch_qkv_post(hipStream_t s, const QkvPost &) { return queue(s); }
hipError_t launch_prompt_attention(hipStream_t s, const PromptAttention &) { return queue(s); }
bool prompt_attention_matrix(uint32_t, uint32_t, uint32_t) { return true; }
uint64_t prompt_attention_scratch(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, uint32_t, int) {
    return 0;
}
bool pair_attention_supported(uint32_t, uint32_t, uint32_t, uint32_t, uint32_t) { return true; }
uint64_t pair_attention_scratch(uint32_t, uint32_t, uint32_t, uint32_t) { return 256; }
hipError_t launch_pair_attention(hipStream_t s, const PromptAttention &, void *) { return queue(s); }
hipError_t launch_window_store(hipStream_t s, float *, float *, float *, const float *,
                               const float *, uint64_t, const float *, float *, uint64_t, uint64_t,
                               uint64_t, uint32_t, uint32_t) {
    return queue(s);
}
hipError_t launch_argmax_rows(hipStream_t s, const float *, uint64_t, uint64_t, uint32_t *, void *) {
    return queue(s);
}
uint64_t argmax_scratch_bytes(uint64_t) { return 16; }
}  // namespace plamo

namespace {

void check(bool ok, const char *what, uint64_t layer = 0, uint64_t row = 0) {
    if (ok) return;
    printf("%s (layer %llu, row %llu)\n", what, (unsigned long long)layer, (unsigned long long)row);
    exit(1);
}

struct Request {
    plamo_synthetic *syn;
    plamo_synthetic_instance *inst;
    struct model *model;
    plamo_metal *metal;
    Request(uint64_t layers, uint64_t window, uint64_t pattern, bool pinned,
            plamo_metal_packing packing = PLAMO_PACK_AUTO) {
        plamo_synthetic_config cfg;
        char err[256] = "";
        plamo_synthetic_defaults(&cfg, 64, layers, 4, 2, 16, 96, 40);
        cfg.window = window;
        cfg.global_capacity = 512;
        cfg.pattern = pattern;
        syn = plamo_synthetic_build(&cfg, 1, err, sizeof err);
        inst = syn ? plamo_synthetic_instantiate(syn, pinned, err, sizeof err) : nullptr;
        plamo_metal_config config{};
        const plamo_mapping *map = syn ? plamo_synthetic_weights(syn) : nullptr;
        config.maps = map;
        config.count = 1;
        config.packing = packing;
        metal = inst ? plamo_metal_open(&config, err, sizeof err) : nullptr;
        check(metal, err);
        model = plamo_synthetic_model(inst);
    }
    ~Request() {
        plamo_metal_close(metal);
        plamo_synthetic_release(inst);
        plamo_synthetic_free(syn);
    }
    struct cache *cache(uint64_t i) { return model->layers[i]->mixer->cache; }
    struct rotation *rotation(uint64_t i) { return model->layers[i]->mixer->rotation; }
    // `rows` host rows that name themselves; their rotations are current.
    void fill(uint64_t rows, float salt) {
        for (uint64_t i = 0; i < model->count; ++i) {
            struct cache *c = cache(i);
            const uint64_t n = std::min<uint64_t>(rows, c->capacity);
            for (uint64_t r = 0; r < n; ++r)
                for (uint64_t j = 0; j < c->width; ++j) {
                    c->k[r * c->width + j] = salt + 100.0f * i + r;
                    c->v[r * c->width + j] = -(salt + 100.0f * i + r);
                }
            memcpy(rotation(i)->out, c->k, n * c->width * 4);
            c->count = rotation(i)->processed_count = n;
            rotation(i)->scale_bits = float_bits(model->scales[i]);
        }
    }
    // Device rows equal the host's, and the host's rotated rows its keys.
    void same(const char *when) {
        for (uint64_t i = 0; i < model->count; ++i) {
            const struct cache *c = cache(i);
            const Layer &d = metal->layers[i];
            for (uint64_t r = 0; r < c->count; ++r) {
                const uint64_t at = r * c->width, n = c->width * 4;
                check(!memcmp(d.k + at, c->k + at, n), (std::string(when) + ": device K").c_str(), i, r);
                check(!memcmp(d.v + at, c->v + at, n), (std::string(when) + ": device V").c_str(), i, r);
                check(!memcmp(d.rot + at, c->k + at, n), (std::string(when) + ": device rotation").c_str(), i, r);
                check(rotation(i)->processed_count == c->count, (std::string(when) + ": processed").c_str(), i, r);
                check(!memcmp(rotation(i)->out + at, c->k + at, n), (std::string(when) + ": host rotation").c_str(), i, r);
            }
        }
    }
};

// A step on full windows whose rows the host has just edited: the upload reads
// the edited rows, not the rows the step moves meanwhile.
void edited_window(bool pinned) {
    Request q(3, 20, 3, pinned);
    q.fill(21, 10.0f);
    check(plamo_metal_forward(q.metal, q.model, 1) == 1, "first step");
    q.same("first step");
    for (int again = 0; again < 2; ++again) {
        q.fill(21, 5000.0f + again);
        std::vector<float> want(q.cache(0)->k, q.cache(0)->k + 21 * q.cache(0)->width);
        check(plamo_metal_forward(q.metal, q.model, 2) == 1, "step after an edit");
        const struct cache *c = q.cache(0);
        check(!memcmp(c->k, want.data() + c->width, 20 * c->width * 4), "host K moved by one");
        q.same("step after an edit");
        check(plamo_metal_forward(q.metal, q.model, 3) == 1, "next step");
        q.same("next step");
    }
}

// A launch that fails anywhere in a step on full windows: -1, the host's rows
// as they were, and no rotations of the moved window left as current.
void failed_launch(bool pinned) {
    Request q(6, 20, 6, pinned);
    q.fill(21, 10.0f);
    check(plamo_metal_forward(q.metal, q.model, 1) == 1, "first step");
    std::vector<std::vector<float>> before;
    for (uint64_t i = 0; i < q.model->count; ++i)
        for (float *rows : {q.cache(i)->k, q.cache(i)->v})
            before.emplace_back(rows, rows + q.cache(i)->count * q.cache(i)->width);
    int launches = 0;
    for (bool failed = true; failed; ++launches) {
        fail_after = launches;
        const int result = plamo_metal_forward(q.metal, q.model, 2);
        failed = fail_after < 0;
        fail_after = -1;
        check(result == (failed ? -1 : 1), "result", 0, launches);
        if (!failed) break;
        for (uint64_t i = 0; i < q.model->count; ++i) {
            const struct cache *c = q.cache(i);
            const uint64_t n = c->count * c->width * 4;
            check(!memcmp(c->k, before[2 * i].data(), n), "host K", i, launches);
            check(!memcmp(c->v, before[2 * i + 1].data(), n), "host V", i, launches);
            check(q.rotation(i)->processed_count == 0 || !memcmp(q.rotation(i)->out, c->k, n),
                  "rotations of other rows", i, launches);
        }
    }
    check(launches > 24, "launches of a step", 0, launches);
    q.same("step after failures");
    check(plamo_metal_forward(q.metal, q.model, 3) == 1, "next step");
    q.same("next step");
}

// One layer with a small full window, at `layer` of eight whose other windows
// are not full: its rotated rows reach the host wherever it stands.
void lone_window(uint64_t layer) {
    Request q(8, 100, 0, true);
    q.cache(layer)->capacity = 20;
    q.fill(20, 10.0f);
    for (uint32_t token = 1; token < 4; ++token) {
        check(plamo_metal_forward(q.metal, q.model, token) == 1, "step", layer);
        q.same("step");
    }
}

// Device memory that holds the weights twice, but not the rows of a longer
// context beside both: the fragments make room, in a prompt, in a decode step
// and for weights preloaded later. A caller who asks for raw weights has none.
void fragments_make_room() {
    for (int turn = 0; turn < 3; ++turn) {
        host::device_limit = 96 << 20;
        Request q(3, 400, 3, true);
        check(plamo_metal_prepare_model(q.metal, q.model) == 1, "prepare");
        check(q.metal->pair_ready, "fragments laid out", 0, turn);
        std::vector<uint32_t> ids(300, 1);
        std::vector<uint16_t> weights(1 << 20);
        check(plamo_metal_prefill(q.metal, q.model, ids.data(), 20, nullptr) == 1, "prompt");
        check(q.metal->pair_ready, "fragments kept", 0, turn);
        // Not a byte more; for the step, three layers' rows doubled less half
        // of the fragments.
        host::device_limit = host::device_bytes;
        if (turn == 1)
            host::device_limit += (400 << 10) - host::device[q.metal->pair_block] / 2;
        if (turn == 0) {
            check(plamo_metal_prefill(q.metal, q.model, ids.data(), 24, nullptr) == 1, "longer prompt");
        } else if (turn == 1) {
            q.fill(256, 10.0f);
            check(plamo_metal_forward(q.metal, q.model, 1) == 1, "step past the rows");
        } else {
            check(plamo_metal_preload(q.metal, weights.data(), 1 << 10) == 1, "preload");
        }
        check(!q.metal->pair_ready && !q.metal->pair_block, "fragments given back", 0, turn);
        plamo_metal_info info;
        plamo_metal_get_info(q.metal, &info);
        check(info.errors == 0, info.note);
        check(plamo_metal_prefill(q.metal, q.model, ids.data(), 7, nullptr) == 1, "next prompt");
    }
    host::device_limit = ~(size_t)0;
    Request raw(3, 400, 3, true, PLAMO_PACK_RAW);
    std::vector<uint32_t> ids(20, 1);
    check(plamo_metal_prepare_model(raw.metal, raw.model) == 1, "prepare, raw");
    check(plamo_metal_prefill(raw.metal, raw.model, ids.data(), 20, nullptr) == 1, "prompt, raw");
    check(!raw.metal->pair_ready && !raw.metal->pair_block, "raw weights alone");
}

}  // namespace

int main(int argc, char **argv) {
    setenv("PLAMO_HIP_EAGER_DECODE", "1", 1);
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "edited_window")
        edited_window(true);
    else if (what == "edited_window_pageable")
        edited_window(false);
    else if (what == "failed_launch")
        failed_launch(true);
    else if (what == "failed_launch_pageable")
        failed_launch(false);
    else if (what == "lone_window")
        for (uint64_t layer = 0; layer < 8; ++layer) lone_window(layer);
    else if (what == "fragments_make_room")
        fragments_make_room();
    else
        check(false, "unknown scenario");
    printf("ok\n");
    return 0;
}
