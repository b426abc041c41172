// Llama-family model, AdamW and the training step on the device-resident
// tape, plus their C ABI. Mirrors paperkiln src/llama.cpp (LlamaBlock::forward
// :25-60, Llama::forward :71-89), nn::AdamW (src/nn.cpp:301-321) and the step
// shape of tools/mtstudio.cpp:456-480. The per-block activation checkpoint is
// the reference's checkpoint() (src/autograd.cpp:68-102) on HBM tensors; its
// receipt here is bytes from the allocator's high-water mark, not a node count.
#include <algorithm>
#include <cmath>
#include <cstring>
#include <exception>
#include <mutex>
#include <string>
#include <thread>
#include <unordered_map>
#include <vector>

#include "pk_internal.h"
#include "tape.h"

namespace pk {
namespace {

// splitmix64 + Box-Muller, the same stream as paperkiln_amd/synth.py randn():
// the reference initialises from libstdc++'s mt19937 + normal_distribution
// (nn.cpp:14-21), which is not reproducible outside libstdc++.
struct Rng {
    uint64_t seed;
    static uint64_t mix(uint64_t z) {
        z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
        z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
        return z ^ (z >> 31);
    }
    double u01(uint64_t idx) const {  // idx is 1-based
        const uint64_t z = mix(seed + idx * 0x9E3779B97F4A7C15ull);
        return (static_cast<double>(z >> 11) + 0.5) * (1.0 / 9007199254740992.0);
    }
};
std::vector<float> randn_host(uint64_t seed, size_t n, float std_) {
    const size_t m = (n + 1) / 2;
    Rng r{seed};
    std::vector<float> out(2 * m);
    for (size_t i = 0; i < m; ++i) {
        const double u1 = r.u01(i + 1), u2 = r.u01(m + i + 1);
        const double rad = std::sqrt(-2.0 * std::log(u1)), th = 2.0 * M_PI * u2;
        out[2 * i] = static_cast<float>(rad * std::cos(th) * std_);
        out[2 * i + 1] = static_cast<float>(rad * std::sin(th) * std_);
    }
    out.resize(n);
    return out;
}

Var make_param(int64_t r, int64_t c, const std::vector<float>& host) {
    Tensor t = Tensor::make(r, c, PK_F32);
    hip_check(hipMemcpy(t.ptr(), host.data(), sizeof(float) * r * c, hipMemcpyHostToDevice), "hipMemcpy");
    Var v = make_var(std::move(t), true);
    v->is_param = true;
    return v;
}

// A device slab read back into many host arrays. One blocking copy per array from pageable memory runs at about
// 7 GB/s (141 MB of a 35 M parameter model took 20 ms): the runtime copies through its own staging on one thread, and
// that thread also takes the page faults of freshly allocated arrays. Here the slab comes down in chunks through pinned
// staging, and several host threads, each with two chunks of its own, copy them out while the next ones arrive (the
// link moves 141 MB in 2.5 ms, one thread copies it into fresh pages in 10 ms, eight in 2 ms).
class SlabReader {
public:
    // A copy and its event cost the stream 14 us beside 26 a MiB, and what the threads then wait for is pages: 141 MB took, in chunks of
    // 0.5, 1, 2 and 4 MiB by 8 threads, 6.9, 5.7, 5.6 and 5.9 ms, of 2 MiB by 12 5.3; 15 MB of 1 and 2 MiB 0.79 and 0.65.
    static constexpr int64_t CHUNK = int64_t{1} << 19;  // floats: 2 MiB
    static constexpr int MAX_THREADS = 12;              // so the staging is at most 48 MiB
    SlabReader() = default;
    SlabReader(const SlabReader&) = delete;
    SlabReader& operator=(const SlabReader&) = delete;
    ~SlabReader() {
        if (staging_) (void)hipHostFree(staging_);
    }
    struct Piece {
        int64_t begin, count;  // floats of the slab, ascending and disjoint
        float* host;
    };
    void read(const float* slab, const std::vector<Piece>& pieces, hipStream_t stream) {
        if (pieces.empty()) return;
        const int64_t total = pieces.back().begin + pieces.back().count, chunks = (total + CHUNK - 1) / CHUNK;
        // a thread costs about as much to start as it takes to copy a chunk: two chunks or more for each
        const int hw = std::max(1, static_cast<int>(std::thread::hardware_concurrency()));
        const int threads = static_cast<int>(std::clamp<int64_t>(chunks / 2, 1, std::min(hw, MAX_THREADS)));
        reserve(static_cast<size_t>(threads) * 2);
        int device = 0;
        hip_check(hipGetDevice(&device), "hipGetDevice");
        std::vector<std::exception_ptr> failed(threads);
        auto work = [&](int w) {
            try {
                hip_check(hipSetDevice(device), "hipSetDevice");
                copy_out(slab, pieces, total, chunks, w, threads, stream);
            } catch (...) {
                failed[w] = std::current_exception();
            }
        };
        std::vector<std::thread> pool;
        try {
            for (int w = 1; w < threads; ++w) pool.emplace_back(work, w);
        } catch (...) {  // no more threads to be had: their chunks are copied here
            for (int w = static_cast<int>(pool.size()) + 1; w < threads; ++w) work(w);
        }
        work(0);
        for (auto& t : pool) t.join();
        for (const auto& e : failed)
            if (e) std::rethrow_exception(e);
    }

private:
    float* staging_ = nullptr;
    size_t chunks_ = 0;
    void reserve(size_t chunks) {
        if (chunks <= chunks_) return;
        if (staging_) hip_check(hipHostFree(staging_), "hipHostFree");
        staging_ = nullptr;
        chunks_ = 0;
        void* p = nullptr;
        hip_check(hipHostMalloc(&p, sizeof(float) * CHUNK * chunks, hipHostMallocDefault), "hipHostMalloc");
        staging_ = static_cast<float*>(p);
        chunks_ = chunks;
    }
    // worker w's share, chunks w, w + threads, ...: the next one is on its way while the present one is copied out
    void copy_out(const float* slab, const std::vector<Piece>& pieces, int64_t total, int64_t chunks, int w, int threads,
                  hipStream_t stream) {
        struct Event {
            hipEvent_t e = nullptr;
            Event() { hip_check(hipEventCreateWithFlags(&e, hipEventDisableTiming), "hipEventCreate"); }
            ~Event() { (void)hipEventDestroy(e); }
        } arrived[2];
        auto fetch = [&](int64_t c, int slot) {
            const int64_t n = std::min(CHUNK, total - c * CHUNK);
            hip_check(hipMemcpyAsync(staging_ + (2 * w + slot) * CHUNK, slab + c * CHUNK, sizeof(float) * n,
                                     hipMemcpyDeviceToHost, stream), "hipMemcpyAsync");
            hip_check(hipEventRecord(arrived[slot].e, stream), "hipEventRecord");
        };
        int slot = 0;
        fetch(w, 0);
        for (int64_t c = w; c < chunks; c += threads, slot ^= 1) {
            if (c + threads < chunks) fetch(c + threads, slot ^ 1);
            hip_check(hipEventSynchronize(arrived[slot].e), "hipEventSynchronize");
            const float* src = staging_ + (2 * w + slot) * CHUNK;
            const int64_t lo = c * CHUNK, hi = std::min(lo + CHUNK, total);
            auto p = std::upper_bound(pieces.begin(), pieces.end(), lo,
                                      [](int64_t v, const Piece& q) { return v < q.begin + q.count; });
            for (; p != pieces.end() && p->begin < hi; ++p) {
                const int64_t from = std::max(lo, p->begin), to = std::min(hi, p->begin + p->count);
                std::memcpy(p->host + (from - p->begin), src + (from - lo), sizeof(float) * (to - from));
            }
        }
    }
};

struct Block {
    Var ln1_w, ln2_w, q, k, v, o, gate, up, down;
};

struct Model {
    pk_llama_config cfg;
    // The model's own tape state (stream, element type, parameter shadows) and the lock that keeps two host
    // threads from running the same model at once; every C entry holds both for the length of the call.
    TapeContext ctx;
    std::mutex mu;
    int64_t head_chunk_rows = 0;  // rows of the tied head evaluated at a time (linear_cross_entropy); 0 = its default
    Var embed, norm_w;
    std::vector<Block> blocks;
    std::vector<std::pair<std::string, Var>> named;
    bool checkpoint_blocks = false;
    // Master weights, gradients and the two AdamW moments (nn.cpp:293-299) each live in ONE
    // allocation, [1, slab_len] fp32, with every parameter's tensors as views at the same offset:
    // zero_grad, the clip norm and the optimiser step are then one launch each, not one per parameter.
    Tensor pslab, gslab, mslab, vslab;
    SlabReader reader;
    // Cosines and sines of RoPE's angles for every position that a sequence of this model has had, laid out once like the weights.
    std::shared_ptr<Buffer> turns;
    int64_t turned_positions = 0;
    void turn_positions(int64_t seq_len) {
        if (seq_len <= turned_positions) return;
        const int dk = cfg.d / cfg.n_heads;
        auto table = std::make_shared<Buffer>(sizeof(float) * seq_len * std::max(dk / 2 * 2, 2));
        k_rope_table(cfg.rope_theta, dk, seq_len, static_cast<float*>(table->p));
        // Waited for, once per growth: a pass that fails behind this one leaves the table to the next, which may be on another stream.
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        turns = std::move(table);
        turned_positions = seq_len;
    }
    long t = 0;
    // Pinned staging for what a pass sends up (ids, targets, positions): one host copy and asynchronous transfers
    // instead of three transfers from pageable memory with a wait each. Written only between passes (a pass ends
    // with a wait for its stream).
    int* stage = nullptr;
    size_t stage_cap = 0;
    ~Model() {
        if (stage) (void)hipHostFree(stage);
    }
    int* staging(size_t n_ints) {
        if (n_ints > stage_cap) {
            if (stage) hip_check(hipHostFree(stage), "hipHostFree");
            stage = nullptr;
            stage_cap = 0;
            void* p = nullptr;
            hip_check(hipHostMalloc(&p, sizeof(int) * n_ints, hipHostMallocDefault), "hipHostMalloc");
            stage = static_cast<int*>(p);
            stage_cap = n_ints;
        }
        return stage;
    }

    void reg(const std::string& name, const Var& p) { named.emplace_back(name, p); }

    Model(const pk_llama_config& c, unsigned seed) : cfg(c) {
        if (c.d % c.n_heads != 0) shape_fail("llama: d must divide by n_heads");
        const int64_t d = c.d, ff = c.d_ff;
        auto lin = [&](int64_t in, int64_t out, unsigned s) {
            return make_param(in, out, randn_host(static_cast<uint64_t>(s) * 7919u + 1u, in * out, 0.02f));
        };
        const std::vector<float> ones(d, 1.0f);
        embed = make_param(c.vocab, d, randn_host(static_cast<uint64_t>(seed + 11) * 104729u + 3u, c.vocab * d, 0.02f));
        reg("embed_tokens.weight", embed);
        for (int i = 0; i < c.n_layers; ++i) {
            const unsigned s = seed + 100u * static_cast<unsigned>(i + 1);
            const std::string p = "layers." + std::to_string(i) + ".";
            Block b;
            b.ln1_w = make_param(1, d, ones);
            b.ln2_w = make_param(1, d, ones);
            b.q = lin(d, d, s + 1);
            b.k = lin(d, d, s + 2);
            b.v = lin(d, d, s + 3);
            b.o = lin(d, d, s + 4);
            b.gate = lin(d, ff, s + 5);
            b.up = lin(d, ff, s + 6);
            b.down = lin(ff, d, s + 7);
            reg(p + "input_layernorm.weight", b.ln1_w);
            reg(p + "post_attention_layernorm.weight", b.ln2_w);
            reg(p + "self_attn.q_proj.weight", b.q);
            reg(p + "self_attn.k_proj.weight", b.k);
            reg(p + "self_attn.v_proj.weight", b.v);
            reg(p + "self_attn.o_proj.weight", b.o);
            reg(p + "mlp.gate_proj.weight", b.gate);
            reg(p + "mlp.up_proj.weight", b.up);
            reg(p + "mlp.down_proj.weight", b.down);
            blocks.push_back(b);
        }
        norm_w = make_param(1, d, ones);
        reg("norm.weight", norm_w);
        if (!c.tie_embeddings) throw std::runtime_error("llama: only the tied head (lm_head = embed_tokens) is built");
        build_slabs();
    }

    void build_slabs() {
        std::vector<int64_t> off;
        int64_t total = 0;
        for (const auto& kv : named) {  // 256-byte granules keep every view aligned for the GEMMs
            off.push_back(total);
            total += (kv.second->data.numel() + 63) / 64 * 64;
        }
        pslab = Tensor::make(1, total, PK_F32);
        gslab = Tensor::make(1, total, PK_F32);
        k_fill(pslab, 0.0f);
        k_fill(gslab, 0.0f);
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        for (size_t i = 0; i < named.size(); ++i) {
            Variable& p = *named[i].second;
            auto view = [&](const Tensor& slab) {
                Tensor t = slab;
                t.rows = p.data.rows;
                t.cols = p.data.cols;
                t.off_bytes = off[i] * static_cast<int64_t>(sizeof(float));
                return t;
            };
            Tensor w = view(pslab);
            hip_check(hipMemcpy(w.ptr(), p.data.ptr(), sizeof(float) * p.data.numel(), hipMemcpyDeviceToDevice), "hipMemcpy");
            p.data = w;
            p.grad = view(gslab);
        }
    }

    std::vector<Var> parameters() const {
        std::vector<Var> out;
        for (const auto& kv : named) out.push_back(kv.second);
        return out;
    }

    // LlamaBlock::forward, llama.cpp:25-60. The 3H slice_cols + H fused_attention +
    // concat_cols nodes of :47-53 are one attention node reading heads in place.
    Var block_forward(const Block& b, const Var& x, const std::shared_ptr<Buffer>& pos, int64_t seq_len) const {
        const int dk = cfg.d / cfg.n_heads;
        std::shared_ptr<ops::Turned> turned;
        Var qkv = ops::rms_linear3_rope(x, b.ln1_w, b.q, b.k, b.v, pos, cfg.rope_theta, dk, cfg.rope_all_heads ? cfg.n_heads : 1, turns,
                                        seq_len == 0 ? x->data.rows : seq_len, turned);
        const float sc = 1.0f / std::sqrt(static_cast<float>(dk));
        Var x1 = ops::linear_add(ops::attention_turned(qkv, turned, cfg.n_heads, sc, seq_len, true, cfg.window, cfg.sinks), b.o, x);
        // re-run at backward time, the block's own output is not needed again (the gradient arrives from outside): the
        // down projection is recorded but not multiplied
        return ops::rms_gated_mlp(x1, b.ln2_w, b.gate, b.up, b.down, !recomputing());
    }

    // Llama::forward (llama.cpp:71-89) from the embedded tokens up to the final norm; positions restart per sequence.
    Var hidden(Var h, const std::shared_ptr<Buffer>& pos_dev, int64_t seq_len) const {
        for (const Block& blk : blocks) {
            if (checkpoint_blocks && grad_enabled()) {
                const Block* bp = &blk;
                h = checkpoint([this, bp, pos_dev, seq_len](const Var& in) { return block_forward(*bp, in, pos_dev, seq_len); },
                               h);
            } else {
                h = block_forward(blk, h, pos_dev, seq_len);
            }
        }
        return ops::rmsnorm(h, norm_w);
    }
};

thread_local std::string g_llama_err;
template <typename F>
int guarded(F&& f) {
    try {
        f();
        return PK_OK;
    } catch (const std::exception& e) {
        g_llama_err = e.what();
        set_error(g_llama_err);
        return status_of(e);
    }
}

// AdamW on every parameter with the copies that the products read. False, with nothing done, where the kernel does not take
// them (or a parameter has two copies).
bool adamw_with_copies(const Model& m, float lr, float b1, float b2, float eps, float wd, float c1, float c2, const Clip& clip) {
    std::unordered_map<const Variable*, CastJob> copies;
    for (const ShadowCopy& s : shadow_copies())
        if (!copies.emplace(s.of, s.job).second) return false;
    std::vector<AdamWPart> parts;
    size_t found = 0;
    for (const auto& kv : m.named) {
        const Tensor& p = kv.second->data;
        AdamWPart part{p.off_bytes / static_cast<int64_t>(sizeof(float)), p.numel(), p.cols, Tensor(), 0};
        const auto it = copies.find(kv.second.get());
        if (it != copies.end()) {
            part.copy = it->second.dst;
            part.col_off = it->second.col_off;
            ++found;
        }
        if (p.buf != m.pslab.buf || kv.second->grad.buf != m.gslab.buf || kv.second->grad.off_bytes != p.off_bytes) return false;
        parts.push_back(std::move(part));
    }
    return found == copies.size() && k_adamw_parts(m.pslab, m.gslab, m.mslab, m.vslab, parts, lr, b1, b2, eps, wd, c1, c2, clip);
}

Model* model_of(void* handle) {
    if (!handle) throw Error(PK_ERR_ARGUMENT, "null model handle");
    return static_cast<Model*>(handle);
}
// Runs f(model) as the model's own tape: its lock held, its context current on this thread.
template <typename F>
int with_model(void* handle, F&& f) {
    return guarded([&] {
        Model* m = model_of(handle);
        std::lock_guard<std::mutex> lk(m->mu);
        ContextScope scope(m->ctx);
        f(m);
    });
}

}  // namespace
}  // namespace pk

using namespace pk;

extern "C" {

int pk_alloc(size_t bytes, void** out) {
    return guarded([&] {
        if (!out) throw Error(PK_ERR_ARGUMENT, "pk_alloc: null result pointer");
        *out = dev_alloc(bytes);
    });
}
int pk_free(void* p) {
    return guarded([&] {
        if (!dev_free(p)) throw Error(PK_ERR_ARGUMENT, "pk_free: not a pointer pk_alloc returned (or already freed)");
    });
}
size_t pk_live_bytes(void) { return dev_live_bytes(); }
size_t pk_peak_bytes(void) { return dev_peak_bytes(); }
void pk_reset_peak(void) { dev_reset_peak(); }
void pk_trim(void) { dev_trim(); }

int pk_llama_create(const pk_llama_config* cfg, unsigned seed, void** handle) {
    return guarded([&] {
        if (!cfg || !handle) throw Error(PK_ERR_ARGUMENT, "pk_llama_create: null argument");
        // the parameters are created under a context of the model's element type, which the model then keeps
        TapeContext ctx;
        ContextScope scope(ctx);
        set_compute_dtype(cfg->compute_dtype);
        Model* m = new Model(*cfg, seed);
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        m->ctx = ctx;
        *handle = m;
    });
}
int pk_llama_destroy(void* h) {
    return guarded([&] {
        if (!h) return;
        Model* m = static_cast<Model*>(h);
        {
            std::lock_guard<std::mutex> lk(m->mu);
            ContextScope scope(m->ctx);
            hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
            m->ctx.shadows.reset();  // the shadows' memory goes back tagged with the model's stream
        }
        TapeContext last = m->ctx;  // parameters and slabs are freed under the model's stream as well
        ContextScope scope(last);
        delete m;
    });
}
int pk_llama_num_params(void* h) { return h ? static_cast<int>(static_cast<Model*>(h)->named.size()) : -1; }
int pk_llama_param_info(void* h, int i, char* name, size_t name_len, int64_t* rows, int64_t* cols) {
    return with_model(h, [&](Model* m) {
        if (i < 0 || i >= static_cast<int>(m->named.size())) throw Error(PK_ERR_ARGUMENT, "parameter index out of range");
        if (name && name_len) std::snprintf(name, name_len, "%s", m->named[i].first.c_str());
        if (rows) *rows = m->named[i].second->data.rows;
        if (cols) *cols = m->named[i].second->data.cols;
    });
}
int pk_llama_set_param(void* h, int i, const float* host) {
    return with_model(h, [&](Model* m) {
        if (i < 0 || i >= static_cast<int>(m->named.size()) || !host) throw Error(PK_ERR_ARGUMENT, "parameter index out of range or null data");
        const Tensor& t = m->named[i].second->data;
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        hip_check(hipMemcpy(t.ptr(), host, sizeof(float) * t.numel(), hipMemcpyHostToDevice), "hipMemcpy");
        invalidate_shadows();
    });
}
int pk_llama_get_param(void* h, int i, float* host) {
    return with_model(h, [&](Model* m) {
        if (i < 0 || i >= static_cast<int>(m->named.size()) || !host) throw Error(PK_ERR_ARGUMENT, "parameter index out of range or null data");
        const Tensor& t = m->named[i].second->data;
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        hip_check(hipMemcpy(host, t.ptr(), sizeof(float) * t.numel(), hipMemcpyDeviceToHost), "hipMemcpy");
    });
}
int pk_llama_get_grad(void* h, int i, float* host) {
    return with_model(h, [&](Model* m) {
        if (i < 0 || i >= static_cast<int>(m->named.size()) || !host) throw Error(PK_ERR_ARGUMENT, "parameter index out of range or null data");
        const Var& p = m->named[i].second;
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        if (p->grad.empty())
            std::memset(host, 0, sizeof(float) * p->data.numel());
        else
            hip_check(hipMemcpy(host, p->grad.ptr(), sizeof(float) * p->data.numel(), hipMemcpyDeviceToHost), "hipMemcpy");
    });
}
int pk_llama_get_all(void* h, int grads, float* const* hosts) {
    return with_model(h, [&](Model* m) {
        if (!hosts) throw Error(PK_ERR_ARGUMENT, "pk_llama_get_all: null argument");
        const Tensor& slab = grads ? m->gslab : m->pslab;
        std::vector<SlabReader::Piece> pieces;
        for (size_t i = 0; i < m->named.size(); ++i) {
            const Tensor& t = grads ? m->named[i].second->grad : m->named[i].second->data;
            if (!hosts[i]) throw Error(PK_ERR_ARGUMENT, "pk_llama_get_all: null data");
            if (t.buf != slab.buf) throw std::runtime_error("a parameter's storage is no longer the model's own");
            pieces.push_back(SlabReader::Piece{t.off_bytes / static_cast<int64_t>(sizeof(float)), t.numel(), hosts[i]});
        }
        m->reader.read(static_cast<const float*>(slab.ptr()), pieces, tape_stream());
    });
}
int pk_llama_set_head_chunk(void* h, int64_t rows) {
    return with_model(h, [&](Model* m) {
        if (rows <= 0) throw Error(PK_ERR_ARGUMENT, "pk_llama_set_head_chunk: rows must be positive");
        m->head_chunk_rows = rows;
    });
}

int pk_llama_loss_backward(void* h, const int* host_ids, const int* host_targets, int64_t n, int64_t seq_len,
                           int checkpoint_blocks, int do_backward, int fused_head, float* loss, pk_llama_stats* stats,
                           void* stream) {
    return with_model(h, [&](Model* m) {
        if (!host_ids || !host_targets || !loss || n <= 0) throw Error(PK_ERR_ARGUMENT, "pk_llama_loss_backward: null or empty argument");
        set_tape_stream(static_cast<hipStream_t>(stream));  // the model keeps it: the optimiser step runs there too
        for (int64_t i = 0; i < n; ++i)
            if (host_ids[i] < 0 || host_ids[i] >= m->cfg.vocab) throw std::runtime_error("embedding: id out of range");
        for (int64_t i = 0; i < n; ++i)
            if (host_targets[i] < 0 || host_targets[i] >= m->cfg.vocab)
                throw std::runtime_error("cross_entropy: target out of range");
        m->checkpoint_blocks = checkpoint_blocks != 0;
        const int64_t sl = seq_len == 0 ? n : seq_len;
        if (n % sl != 0) shape_fail("ids not a multiple of seq_len");
        // ids, targets and positions (which restart per sequence, llama.cpp:73-76) go up from pinned memory without a wait, with
        // zero_grad: every parameter's gradient is a view of one slab
        int* st = m->staging(static_cast<size_t>(3 * n + 1));
        std::memcpy(st, host_ids, sizeof(int) * n);
        std::memcpy(st + n, host_targets, sizeof(int) * n);
        for (int64_t i = 0; i < n; ++i) st[2 * n + i] = static_cast<int>(i % sl);
        auto sent = std::make_shared<Buffer>(sizeof(int) * 3 * n);
        auto third = [&](int k) {  // a view that keeps the whole transfer's memory
            return std::shared_ptr<Buffer>(new Buffer(static_cast<int*>(sent->p) + k * n, sizeof(int) * n),
                                           [sent](Buffer* b) { delete b; });
        };
        auto ids = third(0), tg = third(1), pos_dev = third(2);
        // Everything allocated from here on, until backward returns, is activation memory.
        // The copies of the parameters that the products read come first: they are not activations.
        for (const auto& b : m->blocks) {
            prepare_shadow_cat({b.q, b.k, b.v});
            prepare_shadow(b.o);
            prepare_shadow_cat({b.gate, b.up});
            prepare_shadow(b.down);
        }
        prepare_shadow(m->embed);
        m->turn_positions(sl);
        const size_t base = dev_live_bytes();  // the allocator's host-side counters: nothing to wait for
        dev_reset_peak();
        const size_t live0 = live_variables();
        Tensor rows = Tensor::make(n, m->cfg.d, compute_dtype());
        // The head's product writes the embedding's whole gradient before anything is added to it, so that part of the slab, its first, is not
        // cleared before: a 32000 x 512 table's 65 MB written once and read once less (this launch 22.2 -> 15.3 us, the head's two products
        // [32000, 512] over 4096 rows 117 -> 112.5 each).
        const Variable& em = *m->embed;
        const bool head_writes = fused_head && do_backward && grad_enabled() && em.requires_grad && em.is_param && em.grad.buf == m->gslab.buf &&
                                 em.grad.off_bytes == m->gslab.off_bytes;
        Tensor clear = m->gslab;
        if (head_writes) {
            const int64_t written = std::min(clear.cols, (em.data.numel() + 63) / 64 * 64);
            clear.off_bytes += written * static_cast<int64_t>(sizeof(float));
            clear.cols -= written;
        }
        if (!k_begin_pass(clear, st, static_cast<int*>(sent->p), 3 * n, m->embed->data, rows))
            k_embedding_fwd(m->embed->data, static_cast<const int*>(ids->p), rows);
        Var hid = m->hidden(ops::embedding_of(m->embed, ids, std::move(rows)), pos_dev, seq_len);
        // the loss comes back into the pinned staging's spare word; one wait behind the last kernel ends the pass
        float* hl = reinterpret_cast<float*>(st + 3 * n);
        Var l = fused_head ? ops::linear_cross_entropy_to(hid, m->embed, tg, m->head_chunk_rows, do_backward != 0, hl, head_writes)
                           : ops::cross_entropy(ops::matmul_nt(hid, m->embed), tg);
        hid.reset();
        // the allocator's counters move when the host allocates and frees, not when the GPU gets there: no wait here
        if (stats) {
            stats->live_vars_after_forward = static_cast<int64_t>(live_variables() - live0);
            stats->activation_bytes_after_forward = static_cast<int64_t>(dev_live_bytes() - base);
        }
        if (do_backward) backward(l);
        if (!fused_head) k_word_to_pinned(l->data.ptr(), hl);
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        if (stats) stats->peak_activation_bytes = static_cast<int64_t>(dev_peak_bytes() - base);
        *loss = *hl;
    });
}

int pk_llama_adamw_step(void* h, float lr, float b1, float b2, float eps, float wd, float max_norm, float* total_norm) {
    return with_model(h, [&](Model* m) {
        if (m->mslab.empty()) {
            m->mslab = Tensor::make(1, m->pslab.cols, PK_F32);
            m->vslab = Tensor::make(1, m->pslab.cols, PK_F32);
            k_fill(m->mslab, 0.0f);
            k_fill(m->vslab, 0.0f);
        }
        // ops::clip_grad_norm over the slab (the padding between parameters is zero), in double as the reference
        // (ops.cpp:1047-1053); the AdamW pass applies it, and the norm reaches the host with the wait at the end
        std::unique_ptr<Buffer> scratch;
        float* const norm = reinterpret_cast<float*>(m->staging(1));
        *norm = 0.0f;
        Clip clip;
        if (max_norm > 0.0f) {
            scratch = std::make_unique<Buffer>(sizeof(double) * (SUMSQ_MAX_PARTS + 1));
            double* const parts = static_cast<double*>(scratch->p);
            clip = Clip{parts, k_sumsq_parts(m->gslab, parts), max_norm, reinterpret_cast<float*>(parts + SUMSQ_MAX_PARTS), norm};
        }
        ++m->t;
        const float c1 = 1.0f - std::pow(b1, static_cast<float>(m->t));
        const float c2 = 1.0f - std::pow(b2, static_cast<float>(m->t));
        // every parameter of this model receives a gradient each step, so the reference's "skip a
        // parameter that never accumulated" (nn.cpp:309) never applies; padding stays at zero
        if (!adamw_with_copies(*m, lr, b1, b2, eps, wd, c1, c2, clip)) {
            if (clip.part_dev) k_clip_factor(clip.part_dev, clip.n, clip.max_norm, clip.factor, clip.norm_pinned);
            k_adamw(m->pslab, m->gslab, m->mslab, m->vslab, lr, b1, b2, eps, wd, c1, c2, clip.factor);
            refresh_shadows();  // the copies of the weights follow them, in one launch
        }
        hip_check(hipStreamSynchronize(tape_stream()), "hipStreamSynchronize");
        if (total_norm) *total_norm = *norm;
    });
}

}  // extern "C"
