// Lifetime checks of libgemma_hip's C ABI on the CPU, linked against
// hip_stub.cpp / kernel_stub.cpp and built with AddressSanitizer by
// tests/test_lifetime.py.
//
//   lifetime_test          every destroy order of context, model, cache and
//                          Q4_0 tensor is free of use-after-free and leaks;
//                          a model and its cache keep working after their
//                          context's destroy; a second destroy, or a call on
//                          a destroyed or never-created handle, is
//                          GH_ERR_STATE
//   lifetime_test exit     only the order in which Python finalisers ran at
//                          interpreter exit when a model outlived its
//                          context (context first, then model, then cache)
//   lifetime_test race     one thread steps (and takes a greedy sample)
//                          while another creates and destroys caches, Q4_0
//                          tensors and models on the same context, as a
//                          garbage collector's finaliser thread does; a
//                          watchdog fails the run if the two deadlock
//   lifetime_test config   gh_model_create's checks
//   lifetime_test oom      a prefill whose longest pass does not fit in the
//                          device memory takes shorter ones
//   lifetime_test cut FMT HIDDEN FFN N ...
//                          per N: token tile, splits, blocks per split and
//                          blocks of the four GEMMs of a prefill of N tokens
//                          (8 q heads, 4 kv heads, head_dim 256)
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <thread>
#include <vector>

#include "../../gemma.hs_amd/csrc/common.h"

extern "C" size_t hip_stub_live_bytes(void);
extern "C" size_t hip_stub_mallocs(void);
extern "C" void hip_stub_set_device_bytes(size_t n);
namespace gh {
extern std::vector<int> prefill_passes;
}

#define CHECK(c)                                                                                   \
    do {                                                                                           \
        if (!(c)) {                                                                                \
            std::fprintf(stderr, "FAIL %s:%d: %s (last error: %s)\n", __FILE__, __LINE__, #c,     \
                         gh_last_error());                                                         \
            return 1;                                                                              \
        }                                                                                          \
    } while (0)

namespace {

struct Handles {
    gh_ctx* ctx = nullptr;
    gh_model* m = nullptr;
    gh_kv* kv = nullptr;
    gh_q4* t = nullptr;
};

int make(Handles& h) {
    CHECK(gh_ctx_create(0, &h.ctx) == GH_OK);
    gh_config c;
    CHECK(gh_config_preset("tiny", &c) == GH_OK);
    CHECK(gh_model_create(h.ctx, &c, &h.m) == GH_OK);
    CHECK(gh_synth_model(h.m, 7, 1, 0.02f, 0.01f, 0.02f) == GH_OK);
    CHECK(gh_kv_create(h.m, 16, &h.kv) == GH_OK);
    std::vector<uint8_t> raw(64 * 18, 0);
    CHECK(gh_q4_0_upload(h.ctx, raw.data(), 64, 32, 0, &h.t) == GH_OK);
    int32_t next = -1;
    CHECK(gh_step(h.m, h.kv, 3, nullptr, nullptr, &next) == GH_OK);
    return 0;
}

int destroy(Handles& h, char what) {
    switch (what) {
        case 'c': return gh_ctx_destroy(h.ctx);
        case 'm': return gh_model_destroy(h.m);
        case 'k': return gh_kv_destroy(h.kv);
        default: return gh_q4_0_free(h.t);
    }
}

int any_order() {
    const char* orders[] = {"cmkt", "ckmt", "mckt", "mkct", "kcmt", "kmct", "tcmk", "ctkm"};
    for (const char* order : orders) {
        Handles h;
        if (make(h)) return 1;
        for (const char* p = order; *p; ++p) {
            CHECK(destroy(h, *p) == GH_OK);
            const bool model_open = !std::strchr(order, 'm') || std::strchr(p + 1, 'm');
            const bool kv_open = std::strchr(p + 1, 'k') != nullptr;
            if (*p == 'c' && model_open && kv_open) {
                // the context is released, not freed: its model still steps
                int32_t next = -1;
                CHECK(gh_step(h.m, h.kv, 5, nullptr, nullptr, &next) == GH_OK);
            }
            if (*p == 'm' && kv_open) {
                int32_t next = -1;
                CHECK(gh_step(h.m, h.kv, 5, nullptr, nullptr, &next) == GH_ERR_STATE);
                int32_t len = -1;
                CHECK(gh_kv_length(h.kv, &len) == GH_OK && len >= 1);
            }
        }
        for (char w : {'c', 'm', 'k', 't'}) CHECK(destroy(h, w) == GH_ERR_STATE);
    }
    // gh_kv_truncate rewinds within [0, length]; gh_model_plan reports the
    // step's plan (graph mode, five phases, the tied head) and its length
    {
        Handles h;
        if (make(h)) return 1;
        char plan[512];
        size_t n = 0;
        CHECK(gh_model_plan(h.m, plan, sizeof plan, &n) == GH_OK && n > 0 && n < sizeof plan);
        CHECK(std::strncmp(plan, "step=", 5) == 0 && std::strstr(plan, " gate_up=S") && std::strstr(plan, " lm=tied") &&
              std::strstr(plan, " env="));
        char small[8];
        size_t n2 = 0;
        CHECK(gh_model_plan(h.m, small, sizeof small, &n2) == GH_OK && n2 == n && std::strlen(small) == 7);
        CHECK(gh_model_plan(h.m, nullptr, 4, &n2) == GH_ERR_INVALID);
        int32_t len = -1;
        CHECK(gh_kv_truncate(h.kv, 2) == GH_ERR_RANGE);
        CHECK(gh_kv_truncate(h.kv, -1) == GH_ERR_RANGE);
        CHECK(gh_kv_truncate(h.kv, 0) == GH_OK && gh_kv_length(h.kv, &len) == GH_OK && len == 0);
        for (char w : {'k', 'm', 't', 'c'}) CHECK(destroy(h, w) == GH_OK);
    }
    // handles that were never returned by the library
    int local = 0;
    CHECK(gh_model_destroy(reinterpret_cast<gh_model*>(&local)) == GH_ERR_STATE);
    CHECK(gh_kv_length(reinterpret_cast<gh_kv*>(&local), &local) == GH_ERR_STATE);
    CHECK(gh_ctx_sync(reinterpret_cast<gh_ctx*>(&local)) == GH_ERR_STATE);
    // a handle of the wrong kind
    Handles h;
    if (make(h)) return 1;
    CHECK(gh_kv_destroy(reinterpret_cast<gh_kv*>(h.m)) == GH_ERR_STATE);
    gh_kv_release(h.kv);
    gh_model_release(h.m);
    gh_q4_0_release(h.t);
    gh_ctx_release(h.ctx);
    gh_ctx_release(h.ctx);  // void: a second release is ignored
    return 0;
}

// Concurrent use and destruction on one context (finalisers run on their
// own thread under a -threaded RTS, gemma.cabal:102).
int race() {
    Handles h;
    if (make(h)) return 1;
    void* buf = nullptr;
    CHECK(gh_buf_alloc(h.ctx, 1024 * sizeof(float), &buf) == GH_OK);
    std::atomic<bool> done{false};
    std::atomic<int> failed{0};
    std::thread watchdog([&] {
        for (int i = 0; i < 600 && !done.load(); ++i) std::this_thread::sleep_for(std::chrono::milliseconds(100));
        if (!done.load()) {
            std::fprintf(stderr, "DEADLOCK: stepping and destroying threads did not finish in 60 s\n");
            std::fflush(stderr);
            std::_Exit(3);
        }
    });
    const int iters = 300;
    std::thread stepper([&] {
        for (int i = 0; i < iters; ++i) {
            int32_t next = -1, tok = -1, len = -1;
            if (gh_kv_truncate(h.kv, 0) != GH_OK) failed = 1;
            if (gh_step(h.m, h.kv, (i * 7) % 1024, nullptr, nullptr, &next) != GH_OK) failed = 2;
            if (gh_sample_logits(h.ctx, (const float*)buf, 1024, 0.0f, 1, 0, &tok) != GH_OK) failed = 3;
            if (gh_kv_length(h.kv, &len) != GH_OK || len != 1) failed = 4;
        }
    });
    std::thread finaliser([&] {
        gh_config c;
        if (gh_config_preset("tiny", &c) != GH_OK) failed = 10;
        std::vector<uint8_t> raw(64 * 18, 0);
        for (int i = 0; i < iters; ++i) {
            gh_kv* kv2 = nullptr;
            if (gh_kv_create(h.m, 8, &kv2) != GH_OK) failed = 11;
            gh_q4* t2 = nullptr;
            if (gh_q4_0_upload(h.ctx, raw.data(), 64, 32, 0, &t2) != GH_OK) failed = 12;
            gh_kv_release(kv2);
            gh_q4_0_release(t2);
            if (i % 30 == 0) {
                gh_model* m2 = nullptr;
                if (gh_model_create(h.ctx, &c, &m2) != GH_OK) failed = 13;
                gh_kv* kv3 = nullptr;
                if (gh_kv_create(m2, 4, &kv3) != GH_OK) failed = 14;
                gh_model_release(m2);  // released first: freed with its cache
                gh_kv_release(kv3);
            }
        }
    });
    stepper.join();
    finaliser.join();
    done = true;
    watchdog.join();
    CHECK(failed.load() == 0);
    CHECK(gh_buf_free(h.ctx, buf) == GH_OK);
    for (char w : {'t', 'c', 'k', 'm'}) CHECK(destroy(h, w) == GH_OK);
    return 0;
}

// gh_model_create rejects configurations the kernels do not support, and
// creates nothing for them.
int config_checks() {
    gh_ctx* ctx = nullptr;
    CHECK(gh_ctx_create(0, &ctx) == GH_OK);
    gh_config base;
    CHECK(gh_config_preset("gemma3-4b", &base) == GH_OK);
    gh_model* m = nullptr;
    CHECK(gh_model_create(ctx, &base, &m) == GH_OK && m);
    CHECK(gh_model_destroy(m) == GH_OK);
    auto rejects = [&](void (*edit)(gh_config&)) {
        gh_config c = base;
        edit(c);
        gh_model* bad = nullptr;
        return gh_model_create(ctx, &c, &bad) == GH_ERR_INVALID && bad == nullptr;
    };
    CHECK(rejects([](gh_config& c) { c.hidden = 3104; }));
    CHECK(rejects([](gh_config& c) { c.hidden = 1000; }));
    CHECK(rejects([](gh_config& c) { c.head_dim = 64; }));
    CHECK(rejects([](gh_config& c) { c.n_kv_heads = 3; }));
    CHECK(rejects([](gh_config& c) { c.n_heads = 48; }));  // group 12
    CHECK(rejects([](gh_config& c) { c.sliding_window = -1; }));
    CHECK(rejects([](gh_config& c) { c.global_every = -6; }));
    CHECK(rejects([](gh_config& c) { c.rope_theta_local = 0.0f; }));
    CHECK(rejects([](gh_config& c) { c.rope_theta_global = -1e6f; }));
    CHECK(rejects([](gh_config& c) { c.rope_theta_global = 1.0f / 0.0f; }));
    CHECK(rejects([](gh_config& c) { c.rms_eps = -1e-6f; }));
    CHECK(rejects([](gh_config& c) { c.rms_eps = 0.0f / 0.0f; }));
    CHECK(rejects([](gh_config& c) { c.mode = 7; }));
    CHECK(rejects([](gh_config& c) { c.max_seq = 0; }));
    gh_config wide = base;
    wide.hidden = 3072;
    CHECK(gh_model_create(ctx, &wide, &m) == GH_OK);
    CHECK(gh_model_destroy(m) == GH_OK);
    CHECK(gh_ctx_destroy(ctx) == GH_OK);
    return 0;
}

// A prefill takes the longest passes whose buffers fit: the whole prompt (to
// 2048 tokens), 1024 or 512; only what not even 512 fit in is GH_ERR_OOM.
int prefill_oom() {
    gh_ctx* ctx = nullptr;
    gh_config c;
    CHECK(gh_ctx_create(0, &ctx) == GH_OK);
    CHECK(gh_config_preset("tiny", &c) == GH_OK);
    const std::vector<int32_t> toks(1900, 3);
    // bytes of the buffers for passes of n tokens; a prefill of 1900 tokens with `room` beside the model
    auto run = [&](int n, size_t room, size_t* used, int* rc) {
        gh_model* m = nullptr;
        gh_kv* kv = nullptr;
        CHECK(gh_model_create(ctx, &c, &m) == GH_OK);
        CHECK(gh_synth_model(m, 7, 1, 0.02f, 0.01f, 0.02f) == GH_OK);
        CHECK(gh_kv_create(m, 2048, &kv) == GH_OK);
        int32_t next = -1;
        CHECK(gh_step(m, kv, 3, nullptr, nullptr, &next) == GH_OK);
        const size_t before = hip_stub_live_bytes();
        gh::prefill_passes.clear();
        hip_stub_set_device_bytes(room == SIZE_MAX ? room : before + room);
        *rc = gh_prefill(m, kv, toks.data(), n, nullptr, nullptr, &next);
        hip_stub_set_device_bytes(SIZE_MAX);
        *used = hip_stub_live_bytes() - before;
        if (*rc != GH_OK) {  // the failed call left nothing behind, and the next one works
            int32_t len = -1;
            CHECK(gh_kv_length(kv, &len) == GH_OK && len == 1 && *used == 0);
            gh::prefill_passes.clear();
            CHECK(gh_prefill(m, kv, toks.data(), n, nullptr, nullptr, &next) == GH_OK);
        }
        CHECK(gh_kv_destroy(kv) == GH_OK && gh_model_destroy(m) == GH_OK);
        return 0;
    };
    const std::vector<int> one{1900}, two{1024, 876}, four{512, 512, 512, 364};
    size_t used = 0, b512 = 0, b1024 = 0, b2048 = 0;
    int rc = GH_OK;
    if (run(512, SIZE_MAX, &b512, &rc) || run(1024, SIZE_MAX, &b1024, &rc) || run(1900, SIZE_MAX, &b2048, &rc)) return 1;
    CHECK(b512 < b1024 && b1024 < b2048 && gh::prefill_passes == one);
    if (run(1900, b2048, &used, &rc)) return 1;
    CHECK(rc == GH_OK && used == b2048 && gh::prefill_passes == one);
    if (run(1900, b2048 - 1, &used, &rc)) return 1;
    CHECK(rc == GH_OK && used < b2048 && used > b1024 && gh::prefill_passes == one);
    if (run(1900, b1024, &used, &rc)) return 1;
    CHECK(rc == GH_OK && used == b1024 && gh::prefill_passes == two);
    if (run(1900, b1024 - 1, &used, &rc)) return 1;
    CHECK(rc == GH_OK && used == b512 && gh::prefill_passes == four);
    if (run(1900, b512 - 1, &used, &rc)) return 1;
    CHECK(rc == GH_ERR_OOM && gh::prefill_passes == one);
    if (run(300, b512 - 1, &used, &rc)) return 1;
    CHECK(rc == GH_OK && used < b512);
    // prompts each longer than the one before: the buffers double, in one block
    gh_model* m = nullptr;
    gh_kv* kv = nullptr;
    CHECK(gh_model_create(ctx, &c, &m) == GH_OK);
    CHECK(gh_synth_model(m, 7, 1, 0.02f, 0.01f, 0.02f) == GH_OK);
    CHECK(gh_kv_create(m, 2048, &kv) == GH_OK);
    int32_t next = -1;
    CHECK(gh_step(m, kv, 3, nullptr, nullptr, &next) == GH_OK);
    const size_t mallocs = hip_stub_mallocs();
    for (int n = 2; n <= 1900; n += 26) {
        CHECK(gh_kv_truncate(kv, 0) == GH_OK);
        CHECK(gh_prefill(m, kv, toks.data(), n, nullptr, nullptr, &next) == GH_OK);
    }
    CHECK(hip_stub_mallocs() - mallocs <= 5);
    CHECK(gh_kv_destroy(kv) == GH_OK && gh_model_destroy(m) == GH_OK);
    CHECK(gh_ctx_destroy(ctx) == GH_OK);
    return 0;
}

int print_cuts(int argc, char** argv) {
    CHECK(argc > 5);
    const int fmt = std::atoi(argv[2]);
    gh_ctx* ctx = nullptr;
    gh_config c;
    gh_model* m = nullptr;
    CHECK(gh_ctx_create(0, &ctx) == GH_OK);
    CHECK(gh_config_preset("gemma3-4b", &c) == GH_OK);
    c.hidden = std::atoi(argv[3]);
    c.ffn = std::atoi(argv[4]);
    c.n_layers = 1;
    CHECK(gh_model_create(ctx, &c, &m) == GH_OK);
    auto set = [&](const char* name, size_t rows, size_t cols) {
        const std::vector<uint8_t> zeros(fmt == gh::FMT_Q4 ? rows * (cols / 32) * 18 : rows * cols * 4);
        return gh_model_set_tensor(m, name, fmt == gh::FMT_Q4 ? GH_DTYPE_Q4_0 : GH_DTYPE_F32, zeros.data(), zeros.size());
    };
    const size_t H = c.hidden, F = c.ffn, Q = (size_t)c.n_heads * c.head_dim;
    CHECK(set("blk.0.attn_q.weight", Q, H) == GH_OK && set("blk.0.attn_output.weight", H, Q) == GH_OK);
    CHECK(set("blk.0.ffn_gate.weight", F, H) == GH_OK && set("blk.0.ffn_down.weight", H, F) == GH_OK);
    const gh::LayerDev& L = m->layers[0];
    for (int i = 5; i < argc; ++i) {
        const int n = std::atoi(argv[i]);
        std::printf("%d", n);
        for (const gh::DMat* w : {&L.qkv, &L.o, &L.gu, &L.down}) {
            const gh::PfCut k = gh::pf_cut(*w, gh::pf_rows_padded(w->fmt, n));
            std::printf(" %d,%d,%d,%d,%d", k.mt, k.S, k.per, w->nblk, w->cols);
        }
        std::printf("\n");
    }
    CHECK(gh_model_destroy(m) == GH_OK && gh_ctx_destroy(ctx) == GH_OK);
    return 0;
}

}  // namespace

int main(int argc, char** argv) {
    if (argc > 1 && std::strcmp(argv[1], "config") == 0) {
        if (config_checks()) return 1;
        std::printf("config ok\n");
        return 0;
    }
    if (argc > 1 && std::strcmp(argv[1], "cut") == 0) return print_cuts(argc, argv);
    if (argc > 1 && std::strcmp(argv[1], "oom") == 0) {
        if (prefill_oom()) return 1;
        std::printf("oom ok\n");
        return 0;
    }
    if (argc > 1 && std::strcmp(argv[1], "race") == 0) {
        if (race()) return 1;
        std::printf("race ok\n");
        return 0;
    }
    if (argc > 1 && std::strcmp(argv[1], "exit") == 0) {
        Handles h;
        if (make(h)) return 1;
        gh_q4_0_free(h.t);
        gh_ctx_destroy(h.ctx);
        gh_model_destroy(h.m);
        gh_kv_destroy(h.kv);
        std::printf("exit order ok\n");
        return 0;
    }
    if (any_order()) return 1;
    std::printf("lifetime ok\n");
    return 0;
}
