#include "cloth_batch.h"

#include <algorithm>
#include <cmath>
#include <stdexcept>

#include "threads.h"

namespace chysx {
namespace cloth {

int ClothBatch::add_instance(ClothSimulator& sim) {
    if (std::find(sims_.begin(), sims_.end(), &sim) != sims_.end())
        throw std::invalid_argument("ClothBatch::add_instance: simulator already in the batch");
    sims_.push_back(&sim);
    bound_ = false;
    return static_cast<int>(sims_.size()) - 1;
}

bool ClothBatch::remove_instance(ClothSimulator& sim) {
    const auto it = std::find(sims_.begin(), sims_.end(), &sim);
    if (it == sims_.end()) return false;
    sims_.erase(it);
    bound_ = false;
    return true;
}

void ClothBatch::clear() noexcept {
    sims_.clear();
    bound_ = false;
}

namespace {
// Plans of a choice that are missing, each made by one of a few threads (0.2
// to 0.3 us a row: half a second for 2 M rows on one).
void make_plans(const std::vector<ClothSimulator*>& sims, engine::ResidentChoice c) {
    std::vector<ClothSimulator*> todo;
    for (ClothSimulator* s : sims)
        if (s->plan_missing(c)) todo.push_back(s);
    for_each_on_threads(todo.size(), 8, [&](std::size_t i) { todo[i]->make_plan(c); });
}
}  // namespace

std::vector<chx_instance> ClothBatch::descriptors(float dt, std::uintptr_t cuda_stream) {
    std::vector<int> rows;
    std::vector<chx_instance> ds;
    rows.reserve(sims_.size());
    ds.reserve(sims_.size());
    for (ClothSimulator* s : sims_) {
        ds.push_back(s->prepare_instance(dt, cuda_stream));
        rows.push_back(ds.back().n_rows);
        if (bf16_ && ds.back().n_rows > 0 && ds.back().diag_c == nullptr)
            throw std::invalid_argument(
                "ClothBatch: BF16 mode needs every instance switched with set_bf16_blocks(true)");
    }
    // the resident solve wants all plans in one form: they go to the device
    // only when every cloth has one
    for (const engine::ResidentChoice& c : engine::resident_choices(rows, bf16_)) {
        make_plans(sims_, c);
        if (!std::all_of(sims_.begin(), sims_.end(), [&](ClothSimulator* s) { return s->plan_fits(c); })) continue;
        for (std::size_t i = 0; i < sims_.size(); ++i) sims_[i]->attach_plan(ds[i], c, cuda_stream);
        break;
    }
    return ds;
}

void ClothBatch::finalize(float dt, std::uintptr_t cuda_stream) {
    if (sims_.empty()) throw std::runtime_error("ClothBatch::finalize: no instances");
    runner_.bind_many(descriptors(dt, cuda_stream), cuda_stream);
    bound_ = true;
}

void ClothBatch::step(float dt, std::uintptr_t cuda_stream) {
    if (!(dt > 0.0f)) throw std::invalid_argument("ClothBatch::step: dt must be positive");
    ProfileRange range("chysx::cloth::batch_step");
    if (!bound_) finalize(dt, cuda_stream);
    else runner_.update_many(descriptors(dt, cuda_stream), cuda_stream);
    if (graph_) runner_.step_graph(cuda_stream);
    else runner_.step(cuda_stream);
}

void ClothBatch::assemble(float dt, std::uintptr_t cuda_stream) {
    if (!(dt > 0.0f)) throw std::invalid_argument("ClothBatch::assemble: dt must be positive");
    if (!bound_) finalize(dt, cuda_stream);
    else runner_.update_many(descriptors(dt, cuda_stream), cuda_stream);
    runner_.assemble(cuda_stream);
}

void ClothBatch::solve(std::uintptr_t cuda_stream) {
    if (!bound_) throw std::runtime_error("ClothBatch::solve: call assemble() first");
    runner_.solve(true, cuda_stream);
}

int ClothBatch::num_rows() const noexcept {
    int n = 0;
    for (const ClothSimulator* s : sims_) n += s->buffers().particle_count();
    return n;
}

std::size_t ClothBatch::device_bytes() const noexcept {
    std::size_t b = 0;
    for (const ClothSimulator* s : sims_) b += s->device_bytes();
    return b;
}

std::vector<std::pair<int, int>> ClothBatch::instance_sizes() const {
    std::vector<std::pair<int, int>> out;
    for (const ClothSimulator* s : sims_) out.emplace_back(s->buffers().particle_count(), s->pattern().nnz());
    return out;
}

std::vector<int> ClothBatch::last_pcg_iterations(std::uintptr_t cuda_stream) {
    std::vector<int> it;
    std::vector<double> rr, bb;
    if (bound_) runner_.read_stats(it, rr, bb, cuda_stream);
    return it;
}

std::vector<double> ClothBatch::last_relative_residuals(std::uintptr_t cuda_stream) {
    std::vector<int> it;
    std::vector<double> rr, bb, out;
    if (!bound_) return out;
    runner_.read_stats(it, rr, bb, cuda_stream);
    out.resize(rr.size());
    for (std::size_t i = 0; i < rr.size(); ++i) out[i] = bb[i] > 0.0 ? std::sqrt(rr[i] / bb[i]) : std::sqrt(rr[i]);
    return out;
}

}  // namespace cloth
}  // namespace chysx
