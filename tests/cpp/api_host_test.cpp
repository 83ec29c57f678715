// Tests of the library's host code (csrc/api.hip) without a GPU: its object, a HIP runtime that only keeps books
// (fake_hip.hpp), and launchers that remember what they were given.
//   api_host_test NAME   runs one test, "ok" at its end
#include "fake_hip.hpp"

#include <algorithm>
#include <array>
#include <atomic>
#include <cstdint>
#include <cstdio>
#include <ctime>
#include <functional>

#include "../../include/rt_attn.h"
#include "../../rustorch_amd/csrc/flash_tile_lds.hpp"
#include "../../rustorch_amd/csrc/rt_kernels.hpp"

static int g_failed = 0;
#define CHECK(cond)                                                     \
    do {                                                                \
        if (!(cond)) {                                                  \
            std::printf("FAIL %s:%d: %s\n", __FILE__, __LINE__, #cond); \
            ++g_failed;                                                 \
        }                                                               \
    } while (0)

// ---- the launchers ---------------------------------------------------------------------------------------------
static std::mutex g_mutex;
static std::vector<rt::DecodeSplitParams> g_decode;
static std::vector<rt::FlashTileParams> g_tile;
static int g_rows = 0;
static bool g_f32_split = false;
static std::vector<std::string> g_bwd;  // the gradients' kernels, as launched: "both", "dq", "dkdv", "delta"

// the kernels of decode.hip, by their names
static void note_launch(const std::string& name, dim3 grid, void** args, hipStream_t s) {
    if (name.find("attn_rows") != std::string::npos) g_rows++;
    for (const char* k : {"both", "dq", "dkdv", "delta"})
        if (name.find(std::string("flash_bwd_f32_") + k) != std::string::npos || name.find(std::string("flash_bwd_rows_") + k) != std::string::npos) {
            fake::Inside here;
            g_bwd.push_back(k);
        }
    if (name.find("decode_latency") == std::string::npos && name.find("decode_split") == std::string::npos) return;
    fake::log("decode", s);
    std::lock_guard<std::mutex> lock(g_mutex);
    g_decode.push_back(*(rt::DecodeSplitParams*)args[0]);
}

namespace rt {
hipError_t launch_flash_f32(hipStream_t s, const FlashF32Params& p) {
    fake::log("flash_f32", s);
    const size_t n = (size_t)p.batch * p.heads * p.seq * p.dim;
    for (size_t i = 0; i < n; i++) p.out[i] = p.q[i] + 2.0f * p.k[i] + 4.0f * p.v[i];
    return hipSuccess;
}
bool flash_f32_takes_split(const FlashF32Params&, bool) { return g_f32_split; }
hipError_t launch_flash_tile_bf16(hipStream_t s, const FlashTileParams& p) {
    fake::log("tile", s);
    fake::Inside here;
    std::lock_guard<std::mutex> lock(g_mutex);
    g_tile.push_back(p);
    return hipSuccess;
}
bool flash_tile_bf16_supported(int dim) { return dim <= 256 && dim % 8 == 0; }
bool flash_tile_bf16_addressable(long long, long long) { return true; }
bool flash_wide_bf16_supported(const FlashTileParams&) { return false; }
hipError_t launch_flash_wide_bf16(hipStream_t, const FlashTileParams&) { return hipSuccess; }
hipError_t launch_decode_prepare(hipStream_t, const DecodePrepareParams&) { return hipSuccess; }
}  // namespace rt

// ---- a machine that refuses -------------------------------------------------------------------------------------
static std::atomic<long> g_news{0};
static std::atomic<long> g_news_left{-1};  // this many allocations of the host are granted to the calling thread; -1: all
static thread_local bool g_counted = false;
void* operator new(size_t n) {
    if (g_counted) g_news++;
    if (g_counted && !fake::inside && g_news_left.load() >= 0 && g_news_left.fetch_sub(1) == 0) throw std::bad_alloc();
    return malloc(n ? n : 1);
}
void operator delete(void* p) noexcept { free(p); }
void operator delete(void* p, size_t) noexcept { free(p); }

static std::atomic<bool> g_refuse_threads{false};
#include <dlfcn.h>
extern "C" int pthread_create(pthread_t* t, const pthread_attr_t* a, void* (*f)(void*), void* arg) noexcept {
    if (g_refuse_threads) return EAGAIN;
    static auto real = (int (*)(pthread_t*, const pthread_attr_t*, void* (*)(void*), void*))dlsym(RTLD_NEXT, "pthread_create");
    return real(t, a, f, arg);
}

alignas(256) static char g_buf[1 << 16];  // an address for whatever is not looked into

static int online(hipStream_t s, int kv_len, void* out = g_buf) {
    return rt_gqa_decode_online_bf16(s, g_buf, g_buf, g_buf, out, 8, 2, kv_len, 64, 8192, nullptr);
}
static int chunk(hipStream_t s) { return rt_gqa_decode_chunk_bf16(s, g_buf, g_buf, g_buf, g_buf, nullptr, 4096, 1, 16, 8, 2, 64, 8192, nullptr); }

// ---- tests -----------------------------------------------------------------------------------------------------

// The launches of a batched call work in the caller's workspace alone, under whatever handle: none shares memory, or the
// id it goes by, with another.
static void batched_calls_share_nothing() {
    const size_t need = rt_gqa_decode_workspace_bytes(2, 8, 2, 64, 3000);
    std::vector<std::vector<char>> ws(4, std::vector<char>(need + 16));
    int32_t lens[2] = {3000, 500};
    auto call = [&](int i, hipStream_t s) {
        void* w = (void*)(((uintptr_t)ws[(size_t)i].data() + 15) & ~(uintptr_t)15);
        CHECK(rt_gqa_decode_batched_bf16(s, g_buf, g_buf, g_buf, g_buf, lens, 2, 8, 2, 64, 3000, w, need, nullptr) == RT_OK);
    };
    std::thread a(call, 0, hipStreamPerThread), b(call, 1, hipStreamPerThread);
    a.join();
    b.join();
    call(2, nullptr);
    call(3, nullptr);
    CHECK(g_decode.size() == 4);
    for (size_t i = 0; i < g_decode.size(); i++) {
        CHECK(g_decode[i].n_splits > 1 && (g_decode[i].launch_id & 255) == 0);
        for (size_t j = 0; j < i; j++) CHECK(g_decode[i].launch_id != g_decode[j].launch_id && g_decode[i].ws != g_decode[j].ws);
    }
    hipStream_t s;
    (void)hipStreamCreate(&s);
    ((fake::Stream*)s)->capturing = true;  // a replay would bring the same id
    call(0, s);
    CHECK(g_decode.back().n_splits == 0);
}

// hipStreamPerThread is a stream of every thread: what calls on it do in shared scratch has an order.
static void calls_on_the_per_thread_stream_take_turns() {
    CHECK(rt_init(0, nullptr) == RT_OK);
    std::vector<std::thread> threads;
    for (int i = 0; i < 4; i++)
        threads.emplace_back([i] {
            for (int n = 0; n < 50; n++) CHECK((i % 2 ? online(hipStreamPerThread, n % 2 ? 2000 : 8192) : chunk(hipStreamPerThread)) == RT_OK);
        });
    for (auto& t : threads) t.join();
    const auto& ops = fake::state().ops;
    void* event = nullptr;
    size_t launches = 0;
    for (size_t i = 0; i < ops.size(); i++) {
        if (ops[i].what != "decode" && ops[i].what != "tile") continue;
        launches++;
        CHECK(i > 0 && i + 1 < ops.size());
        const auto &before = ops[i - 1], &after = ops[i + 1];
        CHECK(before.what == "wait" && before.thread == ops[i].thread && before.stream == ops[i].stream);
        CHECK(after.what == "record" && after.thread == ops[i].thread && after.stream == ops[i].stream);
        CHECK(before.event == after.event && (!event || event == before.event));
        event = before.event;
    }
    CHECK(launches == 200);
    // what needs no scratch waits for nobody, nor does an ordinary stream
    fake::state().ops.clear();
    CHECK(online(hipStreamPerThread, 300) == RT_OK);
    CHECK(online(nullptr, 2000) == RT_OK && chunk(nullptr) == RT_OK);
    for (auto& o : fake::state().ops) CHECK(o.what == "decode" || o.what == "tile");
    // under capture there is nothing to wait for: no scratch, and so no splits
    fake::state().per_thread_capturing = true;
    CHECK(online(hipStreamPerThread, 8000) == RT_OK && g_decode.back().n_splits == 1);
    CHECK(online(hipStreamPerThread, 8000, g_buf + 2) == RT_OK && g_rows == 1);
    CHECK(chunk(hipStreamPerThread) == RT_OK && g_tile.back().n_splits <= 1);
    fake::state().per_thread_capturing = false;
    CHECK(rt_shutdown(nullptr) == RT_OK);
    CHECK(online(hipStreamPerThread, 2000) == RT_OK);
    CHECK(fake::state().errors == 0);
}

// A host-slice call whose results come by chunks, checked.
static int host_call(uint64_t seq, uint64_t heads = 4) {
    rt_attention_shape shape = {1, heads, seq, 64, 64, 64};
    const size_t n = heads * seq * 64;
    std::vector<float> q(n), k(n), v(n), out(n, -1.0f);
    for (size_t i = 0; i < n; i++) q[i] = (float)(i % 1000), k[i] = (float)(i % 777), v[i] = (float)(i % 501);
    const int rc = rt_flash_forward_f32(&shape, q.data(), n, k.data(), n, v.data(), n, out.data(), n, nullptr);
    size_t wrong = 0;
    for (size_t i = 0; i < n; i++) wrong += out[i] != q[i] + 2.0f * k[i] + 4.0f * v[i];
    CHECK(rc != RT_OK || wrong == 0);
    return rc;
}

static void host_slices_follow_the_current_device() {
    for (int dev : {0, 1, 0, 1}) {
        (void)hipSetDevice(dev);
        CHECK(host_call(1024) == RT_OK);   // kept block
        CHECK(host_call(20000) == RT_OK);  // ring more than once, block of its own, copies shared with the helpers
    }
    CHECK(rt_shutdown(nullptr) == RT_OK);
    CHECK(fake::state().memory.empty());
    CHECK(host_call(1024) == RT_OK);
    CHECK(fake::state().errors == 0);
}

// A call whose copies are shared waits for its kernel as any other: no core is busy meanwhile.
static void no_thread_spins_through_the_kernel() {
    rt_attention_shape shape = {1, 4, 20000, 64, 64, 64};
    std::vector<float> x(4 * 20000 * 64, 1.0f), out(x.size());
    auto call = [&] { return rt_flash_forward_f32(&shape, x.data(), x.size(), x.data(), x.size(), x.data(), x.size(), out.data(), x.size(), nullptr); };
    auto cpu_ms = [&] {
        const clock_t before = clock();  // of all threads
        CHECK(call() == RT_OK);
        return (double)(clock() - before) * 1e3 / CLOCKS_PER_SEC;
    };
    (void)cpu_ms();
    const double idle = cpu_ms();
    fake::state().busy_ms = 500;
    CHECK(cpu_ms() < idle + 250.0);
    CHECK(fake::state().busy_ms == 0);
}

static void a_host_without_threads_copies_by_itself() {
    g_refuse_threads = true;
    CHECK(host_call(20000) == RT_OK);
    g_refuse_threads = false;
    CHECK(host_call(20000) == RT_OK);
}

// Whichever allocation fails: the entry returns an error, and the next call is as if nothing had been.
static void a_host_without_memory_is_an_error() {
    static float q[3 * 5 * 64], out[3 * 5 * 64];
    static std::vector<float> big(4 * 20000 * 64, 1.0f), big_out(big.size());
    rt_attention_shape small_shape = {1, 3, 5, 64, 64, 64}, big_shape = {1, 4, 20000, 64, 64, 64};
    const size_t n = 3 * 5 * 64;
    rt_err_detail err;
    hipStream_t s = nullptr;
    const std::vector<std::function<int()>> calls = {
        [&] { return rt_flash_forward_masked_f32(&small_shape, q, n, q, n, q, n, RT_MASK_NONE, nullptr, 0, out, n, &err); },
        [&] { return rt_flash_forward_masked_f32(&big_shape, big.data(), big.size(), big.data(), big.size(), big.data(), big.size(),
                                                 RT_MASK_NONE, nullptr, 0, big_out.data(), big.size(), &err); },
        [&] { return rt_gqa_forward_f32(q, n, q, n, q, n, out, n, 1, 3, 3, 5, 5, 64, &err); },
        [&] { return rt_flash_backward_f32(&small_shape, q, n, q, n, q, n, q, n, out, n, out, n, out, n, &err); },
        [&] { return rt_mha_flash_forward_f32(q, n, q, n, q, n, out, n, 1, 5, 3, 64, &err); },
        [&] { return rt_mha_forward_masked_f32(q, n, q, n, q, n, nullptr, 0, out, n, 1, 5, 5, 3, 64, &err); },
        [&] { return rt_gqa_decode_online_bf16(s, g_buf, g_buf, g_buf, g_buf, 8, 2, 2000, 64, 8192, &err); },
        [&] { return rt_gqa_decode_chunk_bf16(s, g_buf, g_buf, g_buf, g_buf, nullptr, 4096, 1, 16, 8, 2, 64, 8192, &err); },
    };
    CHECK(rt_init(0, nullptr) == RT_OK);
    for (size_t i = 0; i < calls.size(); i++) {
        int failures = 0;
        for (long k = 0; k < 1000; k++) {
            (void)rt_shutdown(nullptr);
            (void)hipStreamCreate(&s);  // (nothing is kept for it yet)
            g_news_left = k;
            g_counted = true;
            const int rc = calls[i]();
            g_counted = false;
            const bool all_granted = g_news_left > 0;
            g_news_left = -1;
            CHECK(rc == RT_OK || (rc == RT_ERR_HIP && err.hip_error == hipErrorOutOfMemory));
            CHECK(calls[i]() == RT_OK);
            failures += rc != RT_OK;
            if (rc == RT_OK && all_granted) break;
        }
        CHECK(failures > 0);
    }
    CHECK(host_call(20000) == RT_OK);
    (void)rt_shutdown(nullptr);
    CHECK(fake::state().memory.empty());
}

// One-launch decode: what it leaves fits the memory of every entry, and what the kernel counts on holds.
static void partials_and_words_fit() {
    int split = 0;
    for (int batch : {1, 2, 3, 7, 16, 64, 200, 4000})
        for (int kv : {1, 2, 8, 32})
            for (int group : {1, 3, 16})
                for (int dim : {64, 128, 256})
                    for (int max_seq : {1, 100, 384, 385, 513, 1056, 2048, 5000, 8192, 100000})
                        for (int cus : {64, 256, 304}) {
                            const int heads = kv * group;
                            const int n = rt::decode_latency_splits(batch, heads, kv, dim, max_seq, max_seq, cus);
                            CHECK(n >= 0 && n <= 24);
                            if (n <= 1) continue;
                            split++;
                            const size_t used = (size_t)batch * heads * n * (dim + 2) * 4 + (size_t)batch * kv * 128;
                            CHECK(used <= rt::decode_split_workspace_bytes(batch, heads, dim, max_seq) && used <= rt::kStreamSlotBytes);
                            CHECK((long long)n * batch * kv <= cus);
                        }
    CHECK(split > 0);
}

// The prefill plan is what dealing the jobs one by one gives (jobs of 256 rows, rounds back and forth over the workers of
// an XCD, or over all), and it costs a call no allocation.
static void the_prefill_plan_deals_as_the_kernel_does() {
    auto by_hand = [](const rt::FlashBf16Params& p, bool rank_major, int workers, int heads, int n_qtiles) {
        std::vector<float> load((size_t)workers, 0.0f);
        for (int q = 0; q < n_qtiles * heads; q++) {
            const int round = q / workers, at = q % workers, rank = rank_major ? q / heads : q % n_qtiles;
            const int keys = p.mask == rt::kMaskCausal ? std::min(p.seq, (n_qtiles - rank) * 256) : p.seq;
            load[(size_t)(round % 2 ? workers - 1 - at : at)] += (float)((keys + 127) / 128) + 2.5f;
        }
        float most = 0.0f;
        for (float x : load) most = std::max(most, x);
        return most;
    };
    int ranked = 0;
    for (int cus : {256, 304, 64, 12})
        for (int batch : {1, 2, 3, 8})
            for (int heads : {1, 5, 8, 12, 28, 32, 40})
                for (int seq : {512, 777, 1024, 1501, 2048, 3000, 4096, 9000})
                    for (int mask : {rt::kMaskNone, rt::kMaskCausal}) {
                        rt::FlashBf16Params p{};
                        p.batch = batch;
                        p.heads = p.kv_heads = heads;
                        p.group = 1;
                        p.seq = seq;
                        p.dim = 128;
                        p.mask = mask;
                        p.n_workers = cus;
                        g_news = 0;
                        g_counted = true;
                        const float got = rt::plan_flash_bf16(p);
                        g_counted = false;
                        CHECK(g_news == 0);
                        const int n_qtiles = (seq + 255) / 256, n_bh = batch * heads, w = std::min(cus, n_qtiles * n_bh);
                        const bool by_xcd = n_bh % 8 == 0 && w % 8 == 0;
                        const int workers = by_xcd ? w / 8 : w, list = by_xcd ? n_bh / 8 : n_bh;
                        if (n_qtiles * list > 16 * workers) continue;  // the mean stands for it
                        const float rank = by_hand(p, true, workers, list, n_qtiles), head = by_hand(p, false, workers, list, n_qtiles);
                        CHECK(got == (by_xcd ? std::min(rank, head) : rank));
                        CHECK(p.rank_major == (by_xcd && rank < head));
                        ranked += p.rank_major;
                    }
    CHECK(ranked > 0);
}

// bf16 tile kernel, tiles straight to LDS: ahead of its first barrier no 16 bytes of LDS are written by two waves, nor twice by
// one (a request's arrival has no order with a wave's own clearing), and a wave's query rows are its own requests' alone.
template <int DP>
static void one_writer(int dim) {
    using L = rt::TileLds<DP>;
    std::vector<int> writer(5 * L::STAGE_BYTES / 16, -1);
    auto write = [&](int at, int wave) {
        CHECK(at % 16 == 0 && at + 16 <= 5 * L::STAGE_BYTES && writer[(size_t)at / 16] == -1);
        writer[(size_t)at / 16] = wave;
    };
    for (int wave = 0; wave < 4; wave++)
        for (int lane = 0; lane < 64; lane++) {
            for (int n = 0; n < L::REQUESTS; n++) {
                const int at = L::block(wave, n) + 16 * lane, row = at / L::ROW_BYTES, slot = at / 16 % L::SPR;
                CHECK(row < L::KT);
                for (int stage = 0; stage < 4; stage++) {  // K(0), K(1) and V(0) are requested, V(1) behind the barrier
                    const bool inside = 8 * (slot ^ (stage < 2 ? L::swz_k(row) : L::swz_v(row))) < dim;
                    if ((inside && stage < 3) || (!inside && stage < L::CLEARED)) write(stage * L::STAGE_BYTES + at, wave);
                }
            }
            for (int n = 0; n < L::Q_REQUESTS; n++) write(L::q_block(wave, n) + 16 * lane, wave);
        }
    for (int at = 0; at < 2 * L::STAGE_BYTES; at += 16) CHECK(writer[(size_t)at / 16] >= 0);  // K: whole rows
    for (int row = 0; row < 128; row++)
        for (int slot = 0; slot < L::SPR; slot++) CHECK(writer[(size_t)(L::Q_AT / 16 + row * L::SPR + slot)] == row / 32);
    CHECK(L::KEEP_AT == L::Q_AT + L::STAGE_BYTES && L::V_AT + L::STAGE_BYTES == L::Q_AT);
}
static void a_tiles_lds_has_one_writer() {
    for (int dim = 8; dim <= 32; dim += 8) one_writer<32>(dim);
    for (int dim = 40; dim <= 64; dim += 8) one_writer<64>(dim);
    for (int dim = 72; dim <= 96; dim += 8) one_writer<96>(dim);
    for (int dim = 104; dim <= 128; dim += 8) one_writer<128>(dim);
    for (int dim = 136; dim <= 256; dim += 8) one_writer<256>(dim);
}

// How many spans a chunk's keys are cut into, of every case of tests/test_gpu_chunk_split.py and on either side of the rule's ends.
static void a_chunks_keys_are_cut_as_its_tests_say() {
    hipStream_t s;
    CHECK(hipStreamCreate(&s) == hipSuccess);
    auto spans = [&](int batch, int seq_new, int heads, int kv, int dim, int keys) {
        g_tile.clear();
        CHECK(rt_gqa_decode_chunk_bf16(s, g_buf, g_buf, g_buf, g_buf, (const int32_t*)g_buf, 0, batch, seq_new, heads, kv, dim, keys, nullptr) == RT_OK);
        return g_tile.size() == 1 ? g_tile[0].n_splits : -1;
    };
    // test_spans_fold_to_the_whole
    CHECK(spans(1, 1, 7, 1, 128, 1024) == 16);
    CHECK(spans(1, 11, 6, 2, 128, 1500) == 24);
    CHECK(spans(2, 43, 3, 1, 96, 700) == 11);
    CHECK(spans(1, 31, 1, 1, 8, 4096) == 64);
    CHECK(spans(1, 3, 64, 2, 200, 2000) == 21);
    CHECK(spans(1, 100, 16, 2, 256, 2048) == 8);
    // test_spans_of_a_tile: as many as tiles, but for two of them
    CHECK(spans(1, 2, 16, 16, 64, 900) == 15);
    CHECK(spans(1, 4, 8, 2, 64, 1473) == 24);
    CHECK(spans(3, 4, 32, 8, 128, 200) <= 1);
    CHECK(spans(1, 8, 16, 2, 256, 300) == 10);
    CHECK(spans(2, 5, 12, 12, 80, 321) == 6);
    CHECK(spans(4, 4, 16, 16, 64, 800) == 7);
    CHECK(spans(3, 2, 8, 8, 64, 900) == 15);
    CHECK(spans(2, 4, 16, 16, 64, 800) == 13);
    CHECK(spans(1, 4, 32, 8, 128, 200) == 4);
    // units that fill the chip, and fewer than four tiles, are not cut
    CHECK(spans(16, 2, 16, 16, 64, 4096) <= 1 && spans(8, 2, 16, 16, 64, 4096) > 1);
    CHECK(spans(1, 4, 32, 8, 128, 192) <= 1 && spans(1, 4, 32, 8, 128, 193) == 4);
}

// Head dims above 128: a chunk whose lengths the launch does not know may be short, whatever the cache holds, and keeps the form for it; as
// long as its new positions it is.
static void a_chunk_of_unknown_lengths_keeps_the_short_walk() {
    hipStream_t s;
    CHECK(hipStreamCreate(&s) == hipSuccess);
    auto direct = [&](int batch, int seq_new, int heads, int kv, int dim, bool device) {
        g_tile.clear();
        CHECK(rt_gqa_decode_chunk_bf16(s, g_buf, g_buf, g_buf, g_buf, device ? (const int32_t*)g_buf : nullptr, 8192, batch, seq_new, heads, kv, dim, 8192,
                                       nullptr) == RT_OK);
        CHECK(g_tile.size() == 1);
        return rt::flash_tile_bf16_direct(g_tile[0]);
    };
    for (int dim : {136, 160, 256}) {
        for (auto [batch, seq_new, heads, kv] : {std::array{9, 8, 8, 8}, std::array{32, 100, 16, 16}, std::array{4, 200, 16, 2}, std::array{1, 100, 16, 2}, std::array{32, 16, 32, 8},
                                                 std::array{5, 96, 28, 28}, std::array{4, 255, 16, 16}})
            CHECK(!direct(batch, seq_new, heads, kv, dim, true));
        CHECK(direct(4, 300, 16, 16, dim, true) && direct(2, 1024, 16, 8, dim, true) && direct(1, 1024, 32, 8, dim, true) && direct(8, 1100, 16, 4, dim, true));
        CHECK(direct(32, 100, 16, 16, dim, false) && direct(4, 200, 16, 2, dim, false) && direct(1, 100, 16, 2, dim, false) && direct(5, 96, 28, 28, dim, false));
    }
}

// The gradients run side by side only where they share no memory with what either kernel reads, nor with each other.
static void gradients_that_share_memory_take_turns() {
    const std::vector<std::string> one = {"both"}, two = {"dq", "dkdv"};
    for (bool split : {false, true})
        for (int dim : {64, 32, 200}) {
            g_f32_split = split;
            const rt_attention_shape shape = {1, 8, 100, (uint64_t)dim};
            const size_t rows = 800, n = rows * (size_t)dim;
            std::vector<float> memory(9 * (n + 64));
            float* x[9];  // q k v d_out o dq dk dv, and the row statistic
            for (int i = 0; i < 9; i++) x[i] = (float*)(((uintptr_t)memory.data() + 63) / 64 * 64) + i * n;  // side by side
            std::vector<float> ws(rows);
            auto launched = [&](float* dq, float* dk, float* dv) {
                g_bwd.clear();
                CHECK(rt_flash_backward_saved_f32_dev(nullptr, &shape, x[0], x[1], x[2], x[4], x[8], x[3], dq, dk, dv, ws.data(),
                                                      rows * sizeof(float), nullptr) == RT_OK);
                return g_bwd;
            };
            CHECK(launched(x[5], x[6], x[7]) == (dim <= 128 ? one : two));
            CHECK(launched(x[5], x[1], x[2]) == two);              // dk over k, dv over v
            CHECK(launched(x[5], x[2], x[7]) == two);
            CHECK(launched(x[4], x[6], x[7]) == two);              // dq over out, dk over out, dv over out
            CHECK(launched(x[5], x[4], x[7]) == two);
            CHECK(launched(x[5], x[6], x[4]) == two);
            CHECK(launched(x[5], x[5], x[7]) == two);              // one buffer for two gradients
            CHECK(launched(x[5], x[6], x[6] + n - 4) == two);      // the last four values
            CHECK(launched(x[5], x[6], x[8] - n + 4) == two);      // the statistic's first
        }
    g_f32_split = false;
}

// Head dims above 128, either side of the lines between the two forms of the tile kernel: workgroups that leave the chip room or fill it.
static void wide_heads_take_the_form_that_pays() {
    struct Case {
        int batch, heads, group, seq, dim, mask, window;
        bool lens, direct;
    };
    for (const Case& c : {Case{2, 16, 1, 95, 256, rt::kMaskCausal, 0, false, false}, Case{2, 16, 1, 96, 256, rt::kMaskCausal, 0, false, true},
                          Case{12, 16, 1, 128, 256, rt::kMaskCausal, 0, false, true}, Case{13, 16, 1, 128, 256, rt::kMaskCausal, 0, false, false},
                          Case{32, 16, 1, 256, 256, rt::kMaskCausal, 0, false, false}, Case{32, 16, 1, 300, 256, rt::kMaskCausal, 0, false, true},
                          Case{8, 32, 4, 128, 256, rt::kMaskCausal, 0, false, false}, Case{8, 32, 4, 129, 256, rt::kMaskCausal, 0, false, true}, Case{8, 32, 4, 97, 224, rt::kMaskCausal, 0, false, true},
                          Case{32, 16, 1, 128, 160, rt::kMaskNone, 0, false, true}, Case{32, 16, 1, 129, 160, rt::kMaskNone, 0, false, false},
                          Case{32, 16, 1, 160, 160, rt::kMaskNone, 0, false, false}, Case{32, 16, 1, 161, 160, rt::kMaskNone, 0, false, true},
                          Case{8, 32, 4, 97, 256, rt::kMaskNone, 0, false, true}, Case{32, 16, 1, 128, 256, rt::kMaskPadding, 0, false, true},
                          Case{4, 16, 1, 1000, 256, rt::kMaskCausal, 255, false, false}, Case{4, 16, 1, 1000, 256, rt::kMaskCausal, 256, false, true},
                          Case{4, 16, 1, 1000, 224, rt::kMaskCausal, 256, false, false}, Case{4, 40, 5, 1000, 224, rt::kMaskCausal, 64, false, true},
                          Case{8, 8, 4, 1000, 224, rt::kMaskCausal, 64, false, false},
                          Case{1, 16, 1, 1000, 256, rt::kMaskCausal, 64, false, true}, Case{16, 16, 1, 351, 160, rt::kMaskCausal, 0, true, false}, Case{16, 16, 1, 352, 160, rt::kMaskCausal, 0, true, true},
                          Case{16, 16, 1, 352, 256, rt::kMaskCausal, 0, true, true}, Case{16, 12, 1, 511, 256, rt::kMaskCausal, 0, true, false}, Case{5, 16, 1, 159, 256, rt::kMaskCausal, 0, true, false}, Case{4, 16, 1, 159, 256, rt::kMaskCausal, 0, true, true},
                          Case{16, 16, 1, 600, 256, rt::kMaskCausal, 0, true, true}, Case{4, 16, 1, 200, 256, rt::kMaskCausal, 0, true, true}}) {
        rt::FlashTileParams p{};
        p.batch = c.batch;
        p.heads = c.heads;
        p.group = c.group;
        p.kv_heads = c.heads / c.group;
        p.pack = 1;
        p.seq_q = p.seq_kv = c.seq;
        p.dim = c.dim;
        p.mask = c.mask;
        p.window = c.window;
        p.n_cus = 256;
        int32_t lens = 0;
        if (c.lens) p.q_lens = p.kv_lens = &lens;
        CHECK(rt::flash_tile_bf16_direct(p) == c.direct);
    }
    hipStream_t s;
    CHECK(hipStreamCreate(&s) == hipSuccess);
    struct Chunk {
        int batch, seq_new, heads, kv, dim, keys;
        bool direct;
    };
    for (const Chunk& c : {Chunk{32, 100, 16, 16, 160, 200, false}, Chunk{32, 100, 16, 16, 160, 300, true}, Chunk{32, 30, 8, 8, 192, 400, false},
                           Chunk{32, 30, 8, 8, 192, 700, true}, Chunk{32, 100, 16, 16, 256, 500, false}, Chunk{32, 100, 16, 16, 256, 1000, true},
                           Chunk{64, 4, 32, 8, 256, 2000, false}, Chunk{4, 300, 16, 16, 256, 300, true},
                           Chunk{32, 30, 32, 8, 256, 249, false}, Chunk{32, 30, 32, 8, 256, 250, true}, Chunk{16, 66, 16, 16, 256, 249, false}, Chunk{16, 66, 16, 16, 256, 250, true},
                           Chunk{17, 66, 16, 16, 256, 999, false}, Chunk{16, 10, 8, 8, 256, 139, false}, Chunk{16, 10, 8, 8, 256, 140, true}}) {
        g_tile.clear();
        CHECK(rt_gqa_decode_chunk_bf16(s, g_buf, g_buf, g_buf, g_buf, nullptr, c.keys, c.batch, c.seq_new, c.heads, c.kv, c.dim, 2048, nullptr) == RT_OK);
        CHECK(g_tile.size() == 1 && g_tile[0].n_splits <= 1 && rt::flash_tile_bf16_direct(g_tile[0]) == c.direct);
    }
}

// Above head dim 64 the gradients that run side by side read delta from the workspace: one that shares memory with a gradient gives
// the call to the kernels that have no use for it.
static void wide_gradients_read_the_workspace() {
    const rt_attention_shape shape = {1, 8, 16, 96};
    const size_t rows = 128, n = rows * 96;
    std::vector<float> memory(10 * (n + 64));
    float* x[10];  // q k v d_out o dq dk dv, the row statistic and a workspace
    for (int i = 0; i < 10; i++) x[i] = (float*)(((uintptr_t)memory.data() + 63) / 64 * 64) + i * n;
    auto launched = [&](float* ws) {
        g_bwd.clear();
        CHECK(rt_flash_backward_saved_f32_dev(nullptr, &shape, x[0], x[1], x[2], x[4], x[8], x[3], x[5], x[6], x[7], ws, rows * sizeof(float), nullptr) == RT_OK);
        return g_bwd;
    };
    const std::vector<std::string> wide = {"delta", "dkdv"}, f32 = {"both"};
    CHECK(launched(x[9]) == wide);
    for (int i = 5; i < 8; i++) CHECK(launched(x[i]) == f32 && launched(x[i] + n - 4) == f32);
}

int main(int argc, char** argv) {
    fake::on_launch() = note_launch;
    const std::map<std::string, std::function<void()>> tests = {
        {"partials_and_words_fit", partials_and_words_fit},
        {"batched_calls_share_nothing", batched_calls_share_nothing},
        {"calls_on_the_per_thread_stream_take_turns", calls_on_the_per_thread_stream_take_turns},
        {"host_slices_follow_the_current_device", host_slices_follow_the_current_device},
        {"the_prefill_plan_deals_as_the_kernel_does", the_prefill_plan_deals_as_the_kernel_does},
        {"a_tiles_lds_has_one_writer", a_tiles_lds_has_one_writer},
        {"gradients_that_share_memory_take_turns", gradients_that_share_memory_take_turns},
        {"wide_gradients_read_the_workspace", wide_gradients_read_the_workspace},
        {"a_chunks_keys_are_cut_as_its_tests_say", a_chunks_keys_are_cut_as_its_tests_say},
        {"wide_heads_take_the_form_that_pays", wide_heads_take_the_form_that_pays},
        {"a_chunk_of_unknown_lengths_keeps_the_short_walk", a_chunk_of_unknown_lengths_keeps_the_short_walk},
        {"no_thread_spins_through_the_kernel", no_thread_spins_through_the_kernel},
        {"a_host_without_threads_copies_by_itself", a_host_without_threads_copies_by_itself},
        {"a_host_without_memory_is_an_error", a_host_without_memory_is_an_error},
    };
    if (argc == 2 && tests.count(argv[1])) tests.at(argv[1])();
    else {
        for (auto& t : tests) std::printf("%s\n", t.first.c_str());
        return argc == 1 ? 0 : 2;
    }
    if (!g_failed) std::printf("ok\n");
    return g_failed ? 1 : 0;
}
