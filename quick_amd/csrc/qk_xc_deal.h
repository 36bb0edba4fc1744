// qk_xc_deal.h -- the order of a chunk's GEMM tasks over the accelerator dies.
//
// Block b of a launch runs on XCD b % 8, each with 32 CUs and an L2 of its own.
// Dealt by batch (each batch to the XCD with the fewest V tasks so far, tasks of
// batch -1 filling the shorter queues), the tiles that a batch's tasks share come
// from one L2; but a batch of m functions has up to 325 V tasks at m = 1,600, and
// with few batches most of the GPU waits for one XCD.  So a chunk is dealt by
// batch where every task then has a CU to itself (no queue above 32), or where it
// has at least 64 batches an XCD to even out, and otherwise goes out in batch order.
// Measured, batch order against by batch, us per evaluation: 200 functions and 8
// batches 251 / 198, 32 batches 254 / 255, 250 batches 501 / 520; 1,600 functions
// and 1 batch 863 / 1,205, 16 batches 1,172 / 1,262, 125 batches 2,288 / 2,358,
// 1,000 batches 4,810 / 4,789; (H2O)64 on 11,361 batches, xc_rho_gemm 9.9 / 9.65 ms.
#pragma once
#include <algorithm>
#include <cstddef>
#include <vector>

namespace qk {

constexpr int kXcds = 8, kXcdCus = 32;   // accelerator dies, each with its own L2; CUs of one
constexpr int kXcDealBatches = 64 * kXcds;

// Task: an aggregate of integers, the first the batch
template <class Task>
class XcDeal {
    struct Batch { size_t rho, v; };   // first task of each kind
    std::vector<Batch> batches;
    std::vector<Task> all_rho, all_v;

    static void spread(const std::vector<Task>* q, std::vector<Task>& out) {
        size_t len = 0;
        for (int x = 0; x < kXcds; ++x) len = std::max(len, q[x].size());
        for (size_t i = 0; i < len; ++i)
            for (int x = 0; x < kXcds; ++x) out.push_back(i < q[x].size() ? q[x][i] : Task{-1, 0, 0, 0});
    }

public:
    void begin_batch() { batches.push_back({all_rho.size(), all_v.size()}); }
    void rho(const Task& t) { all_rho.push_back(t); }
    void v(const Task& t) { all_v.push_back(t); }
    // appends the chunk's tasks in launch order and starts the next chunk
    void finish(std::vector<Task>& rho_out, std::vector<Task>& v_out) {
        std::vector<Task> rq[kXcds], vq[kXcds];
        size_t longest = 0;
        batches.push_back({all_rho.size(), all_v.size()});
        for (size_t b = 0; b + 1 < batches.size(); ++b) {
            int x = 0;
            for (int k = 1; k < kXcds; ++k)
                if (vq[k].size() < vq[x].size()) x = k;
            rq[x].insert(rq[x].end(), all_rho.begin() + batches[b].rho, all_rho.begin() + batches[b + 1].rho);
            vq[x].insert(vq[x].end(), all_v.begin() + batches[b].v, all_v.begin() + batches[b + 1].v);
            longest = std::max({longest, rq[x].size(), vq[x].size()});
        }
        if (longest <= (size_t)kXcdCus || batches.size() > (size_t)kXcDealBatches) {
            spread(rq, rho_out);
            spread(vq, v_out);
        } else {
            rho_out.insert(rho_out.end(), all_rho.begin(), all_rho.end());
            v_out.insert(v_out.end(), all_v.begin(), all_v.end());
        }
        batches.clear();
        all_rho.clear();
        all_v.clear();
    }
};

}  // namespace qk
