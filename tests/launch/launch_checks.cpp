// What the host launches, checked on a machine without a GPU: the library's
// objects against fake_hip.cpp.  `launch_checks NAME` runs one check.
#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <functional>
#include <map>
#include <set>
#include <string>
#include <thread>
#include <vector>

#include "fake_hip.hpp"
#include "kernels.hpp"
#include "model.hpp"
#include "train.hpp"

using namespace meshgpt;

namespace {

void expect(bool ok, const std::string &what) {
    if (ok) return;
    std::fprintf(stderr, "check failed: %s\n", what.c_str());
    std::exit(1);
}

// The status of the Error that f throws, 0 when it returns.
template <class F>
int status_of(F &&f) {
    try {
        f();
    } catch (const Error &e) {
        return e.status;
    }
    return 0;
}

GptConfig shape(size_t W, size_t H, size_t C, size_t L = 2, size_t A = 4, size_t F = 6) {
    GptConfig c;
    c.vocab_size = 64;
    c.context = C;
    c.width = W;
    c.heads = H;
    c.layers = L;
    c.attention_mesh_depth = A;
    c.ffn_mesh_depth = F;
    return c;
}

void generate(MeshGpt &m, size_t batch, size_t prompt, size_t count, float temperature = 0.0f) {
    const std::vector<uint32_t> prompts(batch * prompt, 1);
    std::vector<uint32_t> out(batch * (prompt + count));
    m.generate_tokens(prompts.data(), batch, prompt, count, temperature, 7, out.data());
}

// Programs that between them take each route.
std::vector<std::pair<const char *, std::function<void()>>> programs() {
    return {
        {"window", [] {
             MeshGpt m(0, shape(32, 4, 32), 7, 2);
             generate(m, 2, 5, 60);
         }},
        {"long prefill", [] {
             MeshGpt m(0, shape(128, 2, 630), 7, 8);
             const std::vector<uint32_t> prompts(8 * 600, 1);
             m.prefill(prompts.data(), 8, 600, 0.0f, 7, 620);
             m.decode(2);
             std::vector<uint32_t> out(8 * 600);
             m.read_tokens(out.data(), 8, 600);
         }},
        {"decode", [] {
             setenv("MG_DISABLE_PERSISTENT", "1", 1);
             MeshGpt m(0, shape(128, 4, 256), 7, 64);
             generate(m, 64, 16, 20);
             unsetenv("MG_DISABLE_PERSISTENT");
         }},
        {"logits", [] {
             MeshGpt m(0, shape(64, 4, 64), 7);
             const std::vector<uint32_t> tokens(1024, 1);
             std::vector<float> out(1024 * 64);
             for (size_t sequence : {4, 32, 64}) m.logits(tokens.data(), 1024, sequence, false, out.data(), out.size());
             m.hidden_states(tokens.data(), 1024, 64, out.data(), out.size());
         }},
        {"training", [] {
             for (size_t W : {32, 256}) {
                 MeshGpt m(0, shape(W, 4, 64), 7);
                 const std::vector<uint32_t> tokens(256, 1);
                 for (size_t sequence : {4, 32, 64}) m.train_batch(tokens.data(), tokens.data(), 256, sequence, {});
             }
         }},
        {"sampler", [] {
             for (size_t V : {64, 1000, 50000}) {
                 const std::vector<float> logits(2 * V, 0.0f);
                 uint64_t rng[2] = {1, 2};
                 uint32_t tokens[2];
                 sample_logits(0, logits.data(), 2, V, 0.5f, rng, tokens);
             }
         }},
    };
}

// A launch that the runtime refuses is reported by the call that made it, for
// every kernel that the programs launch.
void refused_launches() {
    for (const auto &program : programs()) {
        std::set<std::string> kernels;
        fake::on_launch = [&](const fake::Launch &l) { kernels.insert(l.kernel); };
        program.second();
        fake::on_launch = nullptr;
        expect(!kernels.empty(), std::string(program.first) + " launches kernels");
        for (const std::string &k : kernels) {
            fake::refuse = k;
            expect(status_of(program.second) == kDeviceError, std::string(program.first) + " reports a refused " + k);
            fake::refuse.clear();
        }
        expect(status_of(program.second) == 0, std::string(program.first) + " runs after refusals");
    }
    // Windows that need more LDS than a launch has unasked.
    MeshGpt m(0, shape(128, 4, 32, 2), 7, 1);
    fake::refuse_attributes = true;
    expect(status_of([&] { generate(m, 1, 30, 40); }) == kDeviceError, "a refused LDS size is reported");
    fake::refuse_attributes = false;
    expect(status_of([&] { generate(m, 1, 30, 40); }) == 0, "and the model goes on");
}

// An error that a program's own HIP calls left on the thread, or an allocation
// that failed and was reported, is no launch error of the next call.
void foreign_errors() {
    for (const auto &program : programs()) {
        void *p = nullptr;
        (void)hipMalloc(&p, size_t(1) << 50);
        expect(status_of(program.second) == 0, std::string(program.first) + " after a foreign error");
    }
    MeshGpt m(0, shape(32, 4, 32), 7, 1);
    fake::memory = 0;
    expect(status_of([&] { generate(m, 100000, 5, 8); }) == kOutOfMemory, "no memory for a batch");
    fake::memory = size_t(1) << 33;
    expect(status_of([&] { generate(m, 1, 5, 8); }) == 0, "a smaller batch after it");
}

// No launch of whole windows holds the GPU for long: 50 ms at 1 us for a layer
// of a stack, or five for its block's attention, and a round of 256 sequences
// (the most that a window of 64 rows of 128 channels takes).
void window_launches() {
    for (size_t layers : {1, 2, 12, 40})
        for (size_t depth : {1, 6, 14})
            for (size_t batch : {1, 300, 1024}) {
                MeshGpt m(0, shape(128, 8, 64, layers, depth, depth), 7, 1);
                size_t steps = 0;
                fake::on_launch = [&](const fake::Launch &l) {
                    if (l.kernel.find("window_kernel") == std::string::npos) return;
                    const auto *a = static_cast<const kern::WindowArgs *>(l.args[0]);
                    const double us = double(a->steps) * double((batch + 255) / 256) * double(layers) * double(5 * depth + 5);
                    expect(a->steps == 1 || us <= 50000.0, "a launch of " + std::to_string(us) + " us");
                    steps += size_t(a->steps);
                };
                generate(m, batch, 64, 5000);
                fake::on_launch = nullptr;
                expect(steps == 4999 || steps == 5000, "every token past the context from a window");
            }
}

// The route of tokens inside and past the context, by what each was measured to
// take where the persistent decode does not run: 'w' a window, 'c' the cached
// decode, 'p' a prefill a token.
void window_routes() {
    struct Case {
        size_t W, H, C, L, A, F, batch;
        char inside, past;
    };
    const Case cases[] = {
        {32, 4, 64, 2, 4, 6, 4096, 'w', 'w'},  {32, 4, 32, 12, 9, 9, 16, 'w', 'w'},   {64, 4, 64, 2, 4, 6, 1024, 'w', 'w'},
        {64, 4, 64, 6, 9, 9, 128, 'w', 'w'},   {64, 4, 64, 6, 9, 9, 1024, 'c', 'w'},  {64, 4, 64, 12, 9, 9, 16, 'c', 'w'},
        {128, 4, 32, 2, 4, 6, 1024, 'w', 'w'}, {128, 4, 32, 12, 9, 9, 16, 'c', 'w'},  {128, 4, 32, 12, 9, 9, 512, 'c', 'w'},
        {128, 4, 64, 2, 4, 6, 128, 'w', 'w'},  {128, 4, 64, 2, 4, 6, 512, 'w', 'w'},  {128, 4, 64, 2, 4, 6, 4096, 'c', 'w'},
        {128, 4, 64, 12, 4, 6, 16, 'c', 'w'},  {128, 4, 64, 12, 4, 6, 256, 'c', 'w'}, {128, 4, 64, 12, 9, 9, 16, 'c', 'p'},
        {128, 8, 64, 12, 9, 9, 16, 'c', 'w'},  {128, 4, 48, 12, 9, 9, 16, 'c', 'w'},  {128, 4, 64, 12, 9, 9, 256, 'c', 'w'},
    };
    setenv("MG_DISABLE_PERSISTENT", "1", 1);
    for (const Case &c : cases) {
        MeshGpt m(0, shape(c.W, c.H, c.C, c.L, c.A, c.F), 7, c.batch);
        size_t windows = 0;
        fake::on_launch = [&](const fake::Launch &l) {
            if (l.kernel.find("window_kernel") != std::string::npos)
                windows += size_t(static_cast<const kern::WindowArgs *>(l.args[0])->steps);
        };
        const std::string what = "W" + std::to_string(c.W) + " context " + std::to_string(c.C) + " batch " +
                                 std::to_string(c.batch) + " blocks " + std::to_string(c.L) + " stacks of " +
                                 std::to_string(c.A);
        generate(m, c.batch, 4, c.C - 4);
        expect(windows == (c.inside == 'w' ? c.C - 4 : 0), what + ": inside the context");
        windows = 0;
        generate(m, c.batch, c.C + 1, 3);
        expect(windows == (c.past == 'w' ? 3 : 0), what + ": past the context");
        windows = 0;
        generate(m, c.batch, c.C - 3, 9);  // four tokens inside the context
        expect(windows >= (c.past == 'w' ? 5u : 0u) && windows <= (c.past == 'w' ? 9u : 4u), what + ": across it");
        fake::on_launch = nullptr;
    }
    unsetenv("MG_DISABLE_PERSISTENT");
}

// Every launch of the training chain has the shape that its kernel divides by.
void chain_shapes() {
    setenv("MG_FORCE_TRAIN_CHAIN", "1", 1);
    MeshGpt m(0, shape(128, 4, 32, 3), 7);
    unsetenv("MG_FORCE_TRAIN_CHAIN");
    size_t launches = 0;
    fake::on_launch = [&](const fake::Launch &l) {
        if (l.kernel.find("backward_chain_kernel") == std::string::npos) return;
        const auto *a = static_cast<const kern::train::BackwardChain *>(l.args[0]);
        expect(a->H == 4 && a->sequence == 32 && a->rows == 64 && a->ma.W == 128, "a launch's shape");
        ++launches;
    };
    const std::vector<uint32_t> tokens(64, 1);
    m.train_batch(tokens.data(), tokens.data(), 64, 32, {});
    fake::on_launch = nullptr;
    expect(launches == 4, "one launch before, between and after three blocks");
}

// A prefill that fits without the split attention's planes, or without the last
// rows' buffers, runs without them where there is no memory for them.
void scratch_limits() {
    const std::vector<uint32_t> prompts(8 * 600, 1);
    std::set<std::string> kernels;
    auto prefill = [&] {
        MeshGpt m(0, shape(256, 4, 640), 7, 8);
        kernels.clear();
        fake::on_launch = [&](const fake::Launch &l) { kernels.insert(l.kernel); };
        m.prefill(prompts.data(), 8, 600, 0.0f, 7, 620);
        m.decode(2);
        fake::on_launch = nullptr;
    };
    auto launched = [&](const char *name) {
        for (const std::string &k : kernels)
            if (k.find(name) != std::string::npos) return true;
        return false;
    };
    prefill();
    expect(launched("attn_split_kernel") && launched("last_merge_kernel"), "both where there is memory");
    setenv("MG_DISABLE_SPLIT_PREFILL", "1", 1);
    fake::peak = 0;
    prefill();
    unsetenv("MG_DISABLE_SPLIT_PREFILL");
    fake::memory = fake::peak;
    expect(status_of(prefill) == 0, "a prefill in the memory that it took without planes");
    expect(!launched("attn_split_kernel") && launched("attn_prefill_mfma_kernel"), "on the FP32 kernel");
    fake::memory -= 3 * 8 * 256 * 4;  // less than the last rows' buffers take
    expect(status_of(prefill) == 0, "a prefill without the last rows' buffers");
    expect(!launched("last_merge_kernel"), "with every row in the last block");
    fake::memory = size_t(1) << 33;

    // What an earlier prefill left there makes room for a later call of any kind.
    const std::vector<uint32_t> tokens(12 * 500, 1);
    std::vector<float> out(12 * 500 * 64);
    std::vector<uint32_t> generated(40 * 8);
    const std::function<void(MeshGpt &)> later[] = {
        [&](MeshGpt &m) { m.logits(tokens.data(), 12 * 500, 500, false, out.data(), out.size()); },
        [&](MeshGpt &m) { m.generate_tokens(tokens.data(), 40, 4, 4, 0.0f, 7, generated.data()); },
        [&](MeshGpt &m) { m.train_batch(tokens.data(), tokens.data(), 64, 32, {}); },
    };
    for (const auto &call : later) {
        size_t need = 0;
        for (const char *off : {"1", "0"}) {
            setenv("MG_DISABLE_SPLIT_PREFILL", off, 1);
            MeshGpt m(0, shape(256, 4, 640), 7, 8);
            fake::peak = 0;
            m.prefill(prompts.data(), 8, 600, 0.0f, 7, 620);
            if (need) fake::memory = std::max(need, fake::used);
            expect(status_of([&] { call(m); }) == 0, "a call in the memory that it took without planes");
            need = fake::peak;
            fake::memory = size_t(1) << 33;
        }
        unsetenv("MG_DISABLE_SPLIT_PREFILL");
    }
}

// The training chains are taken for the row counts at which they were measured
// faster, the forward one in every cross_entropy.
void chain_routes() {
    struct Case {
        size_t W, A, F, rows;
        bool butterfly, forward, backward;
    };
    const Case cases[] = {
        {32, 4, 6, 256, false, true, true},    {64, 4, 6, 256, true, true, true},     {32, 4, 6, 4096, true, true, false},
        {128, 4, 6, 64, false, true, false},   {128, 4, 6, 2048, true, true, true},   {128, 4, 6, 256, true, false, false},
        {128, 4, 6, 8192, false, true, false}, {64, 7, 7, 256, false, true, false},   {64, 7, 7, 2048, false, true, false},
        {64, 7, 7, 256, true, false, false},   {64, 7, 7, 2048, true, true, false},   {128, 5, 5, 2048, false, false, false}};
    for (const Case &c : cases) {
        GptConfig g = shape(c.W, 4, 32, 1, c.A, c.F);
        g.connectivity = c.butterfly ? MeshConnectivity::Butterfly : MeshConnectivity::Neighbor;
        MeshGpt m(0, g, 7);
        bool forward = false, backward = false;
        fake::on_launch = [&](const fake::Launch &l) {
            forward |= l.kernel.find("forward_chain_kernel") != std::string::npos;
            backward |= l.kernel.find("backward_chain_kernel") != std::string::npos;
        };
        const std::string what = "W" + std::to_string(c.W) + ", " + std::to_string(c.A) + " layers, " +
                                 std::to_string(c.rows) + " rows" + (c.butterfly ? ", butterfly" : "");
        const std::vector<uint32_t> tokens(c.rows, 1);
        m.train_batch(tokens.data(), tokens.data(), c.rows, 4, {});
        expect(forward == c.forward && backward == c.backward, what);
        forward = false;
        m.cross_entropy(tokens.data(), tokens.data(), c.rows, 4);
        expect(forward == (c.A <= 4 || c.W <= 64), what + ", the loss alone");
        fake::on_launch = nullptr;
    }
}

// Split attention is taken for the sizes at which it was measured faster.
void split_routes() {
    struct Case {
        size_t H, n, batch;
        bool split;
    };
    const Case cases[] = {{2, 288, 8, false},  {2, 288, 64, true},   {2, 320, 48, false}, {2, 330, 48, true}, {2, 384, 16, false},
                          {2, 449, 16, false}, {2, 449, 32, true},   {4, 449, 1, true},   {4, 447, 1, false}, {2, 576, 1, true},
                          {2, 287, 64, false}, {4, 2048, 1, true}};
    for (const Case &c : cases) {
        MeshGpt m(0, shape(128, c.H, 2048, 1), 7);
        bool split = false;
        fake::on_launch = [&](const fake::Launch &l) { split |= l.kernel.find("attn_split_kernel") != std::string::npos; };
        const std::vector<uint32_t> tokens(c.n * c.batch, 1);
        std::vector<float> out(c.n * c.batch * 64);
        m.logits(tokens.data(), tokens.size(), c.n, false, out.data(), out.size());
        fake::on_launch = nullptr;
        expect(split == c.split, std::to_string(c.batch * c.H) + " pairs of " + std::to_string(c.n) + " rows");
    }
}

// A result is looked through on the host up to the size at which the device's
// launches cost less.
void finite_checks() {
    MeshGpt m(0, shape(32, 4, 32), 7);
    for (size_t rows : {8, 728, 1536, 1544, 8000}) {
        bool device = false;
        fake::on_launch = [&](const fake::Launch &l) { device |= l.kernel.find("nonfinite_kernel") != std::string::npos; };
        const std::vector<uint32_t> tokens(rows, 1);
        std::vector<float> out(rows * 64);
        m.logits(tokens.data(), rows, 8, false, out.data(), out.size());
        fake::on_launch = nullptr;
        expect(device == (rows * 64 > 98304), std::to_string(rows * 64) + " values");
    }
}

// Before a batch there are no logits, which is no error.
void no_batch() {
    MeshGpt m(0, shape(32, 4, 32), 7);
    expect(status_of([&] { expect(m.last_logits().empty(), "no logits"); }) == 0, "last_logits before a batch");
}

// Threads that read a model's results at once each get theirs.
void threads_reading() {
    MeshGpt m(0, shape(1024, 16, 64, 8, 10, 10), 7, 64);
    const std::vector<uint32_t> prompts(64 * 40, 1);
    m.prefill(prompts.data(), 64, 40, 0.0f, 7, 50);
    const std::vector<float> weights = m.parameters();  // four chunks
    std::vector<std::thread> readers;
    std::atomic<int> wrong{0};
    for (int t = 0; t < 4; ++t)
        readers.emplace_back([&, t] {
            std::vector<uint32_t> tokens(64 * 40);
            for (int i = 0; i < 40; ++i) {
                if (t < 2) {
                    wrong += m.parameters() != weights;
                } else {
                    m.read_tokens(tokens.data(), 64, 40);
                    wrong += tokens != prompts && tokens != std::vector<uint32_t>(64 * 40, 0);  // no kernel gathers here
                    for (float v : m.last_logits()) wrong += v != 0.0f;
                }
            }
        });
    for (std::thread &r : readers) r.join();
    expect(wrong == 0, std::to_string(wrong) + " reads held another's data");
}

// A batch that finds no memory leaves a model that smaller batches can use, with
// all the buffers that their launches name.
void batch_without_memory() {
    for (size_t room : {0, 1 << 20, 1 << 22, 1 << 24}) {
        MeshGpt m(0, shape(32, 4, 32), 7, 2);
        fake::peak = 0;
        generate(m, 2, 5, 8);
        fake::memory = fake::peak + room;
        expect(status_of([&] { generate(m, 100000, 5, 8); }) == kOutOfMemory, "no memory for a batch");
        size_t windows = 0;
        fake::on_launch = [&](const fake::Launch &l) {
            if (l.kernel.find("window_kernel") == std::string::npos) return;
            const auto *a = static_cast<const kern::WindowArgs *>(l.args[0]);
            expect(a->tokens && a->len && a->rng && a->logits && a->flags && a->kc && a->vc, "every buffer is there");
            expect(a->layer_elems * 2 * 4 <= fake::size_of(a->kc), "the cache holds the layers");
            ++windows;
        };
        expect(status_of([&] { generate(m, 2, 5, 8); }) == 0 && windows == 1, "a smaller batch after it");
        fake::on_launch = nullptr;
        fake::memory = size_t(1) << 33;
    }
}

// Kernels that carry mesh values times log2(e) run models whose weights keep
// these below 1e38: a row of at most sqrt(128) through the V mesh's four layers,
// seven times that at most into the projection's.  Small weights settle it on
// the host; large or trained ones by the gain of each layer.
void wide_routes() {
    for (float gain : {0.0f, 1.0f, 3.0e4f, 4.0e4f, 1.0e30f})
        for (float largest : {1.0f, 1.0e6f, 0.0f}) {  // 0: after a training step
            MeshGpt m(0, shape(128, 4, 64), 7, 2);
            std::vector<float> weights = m.parameters();
            weights[10 * 128] = largest;
            size_t asked = 0;
            std::set<std::string> kernels;
            fake::on_launch = [&](const fake::Launch &l) {
                kernels.insert(l.kernel);
                if (l.kernel.find("layer_gains_kernel") == std::string::npos) return;
                expect(l.grid.x == 2 * (4 * 4 + 6), "a gain for each layer of the blocks");
                std::fill_n(*static_cast<float **>(l.args[2]), l.grid.x, gain);
                ++asked;
            };
            m.set_parameters(weights.data(), weights.size());
            if (largest == 0.0f) {
                const std::vector<uint32_t> tokens(64, 1);
                m.train_batch(tokens.data(), tokens.data(), 64, 32, {});
            }
            generate(m, 2, 70, 3);
            fake::on_launch = nullptr;
            expect(asked == (largest == 1.0f ? 0u : 1u), "the layers' gains are asked for once where they are needed");
            const char *form = asked && gain > 3.5e4f ? "ELb0EEEv" : "ELb1EEEv";
            for (const std::string &k : kernels)
                if (k.find("rows_block_kernel") != std::string::npos || k.find("window_kernel") != std::string::npos)
                    expect(k.find(form) != std::string::npos, "gain " + std::to_string(gain) + ": " + k);
        }
    // The largest weight may be any; one that is not finite is refused as ever.
    MeshGpt m(0, shape(128, 4, 64), 7, 2);
    std::vector<float> weights = m.parameters();
    for (float bad : {INFINITY, -INFINITY, NAN}) {
        weights[5] = bad;
        expect(status_of([&] { m.set_parameters(weights.data(), weights.size()); }) == kNonfinite, "a weight refused");
    }
    weights[5] = -3.0e38f;
    expect(status_of([&] { m.set_parameters(weights.data(), weights.size()); }) == 0, "a large weight taken");
}

const std::map<std::string, void (*)()> kChecks = {
    {"wide_routes", wide_routes},
    {"batch_without_memory", batch_without_memory},
    {"threads_reading", threads_reading},
    {"no_batch", no_batch},
    {"finite_checks", finite_checks},
    {"split_routes", split_routes},
    {"chain_routes", chain_routes},
    {"scratch_limits", scratch_limits},
    {"chain_shapes", chain_shapes},
    {"window_routes", window_routes},
    {"window_launches", window_launches},
    {"refused_launches", refused_launches},
    {"foreign_errors", foreign_errors},
};

}  // namespace

int main(int argc, char **argv) {
    const auto check = kChecks.find(argc > 1 ? argv[1] : "");
    if (check == kChecks.end()) {
        for (const auto &c : kChecks) std::puts(c.first.c_str());
        return 2;
    }
    check->second();
    std::puts("ok");
}
