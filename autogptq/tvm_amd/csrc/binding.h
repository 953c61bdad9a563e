// Shared by the translation units of the torch operator library (binding.cpp: torch.ops.gptq_hip.* and the torch class;
// python_call.cpp: the module call from Python): the per-stream workspaces and a layer's constant tensors bound to one
// row count.
#pragma once
#include <ATen/ATen.h>

#include <mutex>
#include <optional>

#include "gptq_hip.h"

namespace gptq_torch {

using at::Tensor;
using OptTensor = std::optional<Tensor>;

inline const void *ptr(const OptTensor &t) { return t.has_value() && t->defined() ? t->data_ptr() : nullptr; }
inline bool has(const OptTensor &t) { return t.has_value() && t->defined(); }

// x, or a copy of it where the kernels' 16-byte loads ask for one (a contiguous view at an odd offset)
inline Tensor aligned(const Tensor &x) { return (uintptr_t)x.data_ptr() % 16 == 0 ? x : x.clone(); }

void raise(int rc, const char *what, int64_t M, int64_t K, int64_t N, int64_t bits, int64_t gs);

int workspace_kind(const gptq_hip_plan &plan);

// The workspace of a stream for the launches of one call (none for nbytes = 0).  Held over all of them: a call is up to three
// launches that hand x or partial sums on through the workspace, and those of another thread on the same stream must not
// come between.
struct Workspace {
    std::mutex busy;
    Tensor bytes;
};
class WorkspaceLease {
public:
    WorkspaceLease(const Tensor &like, size_t nbytes, void *stream, int kind = 0);
    void *data() const { return ws ? ws->bytes.data_ptr() : nullptr; }
    size_t size() const { return ws ? (size_t)ws->bytes.numel() : 0; }

private:
    Workspace *ws = nullptr;
    std::unique_lock<std::mutex> held;
};

// One layer's constant tensors, a row count and the plan for it: what a call needs beside x.
// kind: 0 = checkpoint tensors (qweight, qzeros, scales, g_idx?), 1 = sorted copy (qweight_sorted, qzeros, scales,
// kmap), 2 = tiled copy (qtile, sz, -, xsrc?, kinv?).
struct Bound {
    int kind = 0, bits = 0, group_size = 0;
    int M = 0, K = 0, N = 0;
    Tensor a, b, c;
    OptTensor d, e, bias;
    gptq_hip_plan plan{};
    size_t ws_need = 0;

    // fills plan and ws_need for M, K and N; a status of the library
    int choose();
    // y = x @ W (+ bias) on the current stream of the layer's device; x fp16 [M, K] and y fp16 [M, N], contiguous,
    // on that device, which is the current one.  A status of the library.
    int launch(const Tensor &x, void *y, void *stream) const;
};

// the same product as the operator torch.ops.gptq_hip.*, through the dispatcher
Tensor dispatch(const Bound &q, const Tensor &x);

// the operators' checks of a layer's tensors (devices, dtypes, shapes), once, when they are bound
void check_bound(const Bound &q);

}  // namespace gptq_torch
