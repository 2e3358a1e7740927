// PyTorch-ROCm extension over the C ABI in include/snd_scan.h.
//
// Exports the reference's operator pair with the reference's argument and return lists
// (kernels/selective_nd_scan/src/cusoflex/selective_scan_oflex.cpp:179-187,282 and :286-297,432-438,
// pybind :442-445):
//     fwd(u, delta, A, B, C, D?, delta_bias?, delta_softplus, out_float, A_decay?) -> [out, x, x_v, x_sd]
//     bwd(u, delta, A, B, C, D?, delta_bias?, dout, x?, x_v?, delta_softplus, A_decay?, x_sd?)
//         -> [du, ddelta, dA, dB, dC, dD, ddelta_bias, dA_decay]
// which does what a host binding has to do: the reference's TORCH_CHECKs (:188-245, :298-391), allocation of outputs / saved
// state / scratch, device guard, current-stream lookup, and mapping of a non-zero library status to a c10::Error (Python
// RuntimeError).  On top of it stand the differentiable scan and, over snd_block.h, the norm and linear layers of a block and
// everything between its projections, as native autograd functions: what they share is said at NoAutocast, check_elements
// and once_differentiable.
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <ATen/hip/impl/HIPGuardImplMasqueradingAsCUDA.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/extension.h>

#include <algorithm>
#include <atomic>
#include <cstdlib>
#include <initializer_list>
#include <vector>

#include "snd_block.h"
#include "snd_scan.h"

namespace {

#define CHECK_SHAPE(x, ...) \
    TORCH_CHECK(x.sizes() == torch::IntArrayRef({__VA_ARGS__}), #x " must have shape (" #__VA_ARGS__ ")")

// bytes rounded up to the 2 MiB grid that large allocations start on (the grid snd_plan's placement advice refers to)
int64_t round_2mib(int64_t bytes) { return (bytes + (2 << 20) - 1) / (2 << 20) * (2 << 20); }

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::ScalarType::Float: return SND_F32;
        case at::ScalarType::Half: return SND_F16;
        case at::ScalarType::BFloat16: return SND_BF16;
        default: TORCH_CHECK(false, "selective_nd_scan: unsupported dtype ", toString(t)); return -1;
    }
}

void check_status(int st, const char *what) {
    TORCH_CHECK(st == SND_OK, "selective_nd_scan ", what, " failed: ", snd_status_string(st), " (status ", st, ")");
}

struct Checked {
    int batch, dim, nrows, ncols, dstate, n_groups, delta_dim;
    bool u_shared;                 // u is [batch, dim / n_groups, H, W]: one feature map scanned by every group
    snd_shape shape;
    snd_plan plan;
};

// The checks of selective_scan_oflex.cpp:188-245 (shared by fwd and bwd).
Checked check_inputs(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B,
                     const at::Tensor &C, const c10::optional<at::Tensor> &D_,
                     const c10::optional<at::Tensor> &delta_bias_, const c10::optional<at::Tensor> &A_decay_) {
    auto input_type = u.scalar_type();
    TORCH_CHECK(input_type == at::ScalarType::Float || input_type == at::ScalarType::Half ||
                input_type == at::ScalarType::BFloat16, "u must be float32, float16 or bfloat16");
    TORCH_CHECK(A.scalar_type() == at::ScalarType::Float, "A must be float32");
    TORCH_CHECK(delta.scalar_type() == input_type && B.scalar_type() == input_type && C.scalar_type() == input_type,
                "u, delta, B, C must share one dtype");
    TORCH_CHECK(u.is_cuda() && delta.is_cuda() && A.is_cuda() && B.is_cuda() && C.is_cuda(),
                "all tensors must be on the GPU");
    TORCH_CHECK(u.dim() == 4 && delta.dim() == 4 && A.dim() == 2 && B.dim() == 5 && C.dim() == 5,
                "expected u, delta 4-D; A 2-D; B, C 5-D");
    TORCH_CHECK(u.stride(-1) == 1 || u.size(-1) == 1, "u must be contiguous in its last dimension");
    TORCH_CHECK(delta.stride(-1) == 1 || delta.size(-1) == 1, "delta must be contiguous in its last dimension");

    Checked c;
    // dim is A's (the reference takes it from u, selective_scan_oflex.cpp:206): u may carry only
    // dim / n_groups channels, shared by all groups (the CrossScan of one feature map without copies)
    c.batch = u.size(0); c.dim = A.size(0); c.nrows = u.size(2); c.ncols = u.size(3);
    c.dstate = A.size(1); c.n_groups = B.size(1); c.delta_dim = delta.size(1);
    c.u_shared = u.size(1) != c.dim;
    TORCH_CHECK(!c.u_shared || u.size(1) * c.n_groups == c.dim,
                "u must have dim = A.size(0) channels, or dim / n_groups channels shared by the groups");
    TORCH_CHECK(c.dim % c.n_groups == 0, "dims should be dividable by n_groups");
    TORCH_CHECK(c.dim % c.delta_dim == 0, "dims should be dividable by delta_dim");
    TORCH_CHECK(c.dstate <= SND_MAX_DSTATE, "selective_scan only supports state dimension <= 16");
    const int batch_size = c.batch, dim = c.dim, nrows = c.nrows, ncols = c.ncols, dstate = c.dstate,
              n_groups = c.n_groups, delta_dim = c.delta_dim;
    CHECK_SHAPE(u, batch_size, c.u_shared ? dim / n_groups : dim, nrows, ncols);
    CHECK_SHAPE(delta, batch_size, delta_dim, nrows, ncols);
    CHECK_SHAPE(A, dim, dstate);
    CHECK_SHAPE(B, batch_size, n_groups, dstate, nrows, ncols);
    TORCH_CHECK(B.stride(-1) == 1 || B.size(-1) == 1, "B must be contiguous in its last dimension");
    CHECK_SHAPE(C, batch_size, n_groups, dstate, nrows, ncols);
    TORCH_CHECK(C.stride(-1) == 1 || C.size(-1) == 1, "C must be contiguous in its last dimension");
    if (A_decay_.has_value()) {
        const auto &A_decay = A_decay_.value();
        TORCH_CHECK(A_decay.scalar_type() == at::ScalarType::Float && A_decay.is_cuda());
        CHECK_SHAPE(A_decay, 1);
    }
    if (D_.has_value()) {
        const auto &D = D_.value();
        TORCH_CHECK(D.scalar_type() == at::ScalarType::Float && D.is_cuda());
        TORCH_CHECK(D.stride(-1) == 1 || D.size(-1) == 1);
        CHECK_SHAPE(D, dim);
    }
    if (delta_bias_.has_value()) {
        const auto &delta_bias = delta_bias_.value();
        TORCH_CHECK(delta_bias.scalar_type() == at::ScalarType::Float && delta_bias.is_cuda());
        TORCH_CHECK(delta_bias.stride(-1) == 1 || delta_bias.size(-1) == 1);
        CHECK_SHAPE(delta_bias, delta_dim);
    }
    c.shape = snd_shape{c.batch, c.dim, c.nrows, c.ncols, c.dstate, c.n_groups, c.delta_dim, dtype_code(input_type)};
    check_status(snd_make_plan(&c.shape, &c.plan), "plan");
    return c;
}

// Default snd_schedule of fwd and bwd (0 = chosen by shape) when a call does not name one; set_schedule()
// is for tests and tuning.  Calls that pass `schedule` themselves never read it.
std::atomic<int> g_schedule{SND_SCHED_AUTO};
// Opt-in check of the pipelined schedules' error word after every launch (costs a stream sync):
// SND_CHECK_PIPELINE=1 in the environment, or set_debug(True).
std::atomic<bool> g_check_pipeline{[] { const char *e = std::getenv("SND_CHECK_PIPELINE"); return e && e[0] && e[0] != '0'; }()};

int resolve_schedule(int64_t schedule) {
    if (schedule < 0) return g_schedule.load();
    TORCH_CHECK(schedule >= SND_SCHED_AUTO && schedule <= SND_SCHED_WAVEFRONT,
                "schedule must be 0 (auto), 1 (plane), 2 (strips), 3 (bands) or 4 (row-segment wavefront)");
    return (int)schedule;
}
// whether a call with this schedule runs one of the pipelined tile schedules (they need the workspace)
bool pipelined(int sched, int auto_choice) {
    const int s = sched == SND_SCHED_AUTO ? auto_choice : sched;
    return s == SND_SCHED_STRIPS || s == SND_SCHED_BANDS;
}
bool wavefront(int sched, const snd_plan &plan) {
    return sched == SND_SCHED_WAVEFRONT || (sched == SND_SCHED_AUTO && plan.auto_schedule == SND_SCHED_WAVEFRONT);
}
void check_pipeline(const at::Tensor &ws, hipStream_t stream, const char *what) {
    if (!ws.defined() || !g_check_pipeline.load()) return;
    const int st = snd_workspace_error(ws.data_ptr(), (snd_stream_t)stream);
    TORCH_CHECK(st == SND_OK, "selective_nd_scan ", what, ": ", snd_status_string(st), " (status ", st, ")");
}

void fill_fwd(snd_fwd_params &p, const Checked &c, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A,
              const at::Tensor &B, const at::Tensor &C, const c10::optional<at::Tensor> &D_,
              const c10::optional<at::Tensor> &delta_bias_, const c10::optional<at::Tensor> &A_decay_,
              bool delta_softplus) {
    memset(&p, 0, sizeof(p));
    p.shape = c.shape;
    p.u_shared = c.u_shared ? 1 : 0;
    p.delta_softplus = delta_softplus ? 1 : 0;
    p.u = u.data_ptr(); p.delta = delta.data_ptr(); p.B = B.data_ptr(); p.C = C.data_ptr();
    p.A = A.data_ptr<float>();
    p.D = D_.has_value() ? D_.value().data_ptr<float>() : nullptr;
    p.delta_bias = delta_bias_.has_value() ? delta_bias_.value().data_ptr<float>() : nullptr;
    p.A_decay = A_decay_.has_value() ? A_decay_.value().data_ptr<float>() : nullptr;
    p.u_batch_stride = u.stride(0); p.u_d_stride = u.stride(1); p.u_h_stride = u.stride(2);
    p.delta_batch_stride = delta.stride(0); p.delta_d_stride = delta.stride(1); p.delta_h_stride = delta.stride(2);
    p.A_d_stride = A.stride(0); p.A_dstate_stride = A.stride(1);
    p.B_batch_stride = B.stride(0); p.B_group_stride = B.stride(1); p.B_dstate_stride = B.stride(2); p.B_h_stride = B.stride(3);
    p.C_batch_stride = C.stride(0); p.C_group_stride = C.stride(1); p.C_dstate_stride = C.stride(2); p.C_h_stride = C.stride(3);
}

// Fused CrossMerge arguments: weights are one float32 per channel, contiguous, on the inputs' device.
void check_merge(const Checked &c, bool merge, const c10::optional<at::Tensor> &w, const at::Tensor &u) {
    if (!merge) {
        TORCH_CHECK(!w.has_value(), "merge_weights given without merge=True");
        return;
    }
    if (w.has_value()) {
        const at::Tensor &t = w.value();
        TORCH_CHECK(t.scalar_type() == at::ScalarType::Float && t.is_cuda() && t.is_contiguous() && t.numel() == c.dim &&
                        t.device() == u.device(),
                    "merge_weights must be a contiguous float32 GPU tensor with dim = ", c.dim, " elements");
    }
}

// Everything a scan call takes beside its tensors.
struct Options {
    bool delta_softplus = false, out_float = true;
    int64_t directions = 0;
    int sched = SND_SCHED_AUTO;
    bool merge = false;
};
typedef c10::optional<at::Tensor> OptTensor;

snd_job clear_job(void *ptr, int64_t bytes) {
    snd_job j{};
    j.kind = SND_JOB_CLEAR;
    j.out = ptr;
    j.outer = bytes;
    return j;
}
// out[o][i] = sum over the rows of in[o][row][i] (one row: a cast)
snd_job sum_job(const at::Tensor &in, int64_t outer, int rows, int64_t cols, const at::Tensor &out) {
    snd_job j{};
    j.kind = SND_JOB_SUM;
    j.in = in.data_ptr();
    j.out = out.data_ptr();
    j.outer = outer; j.rows = rows; j.cols = cols;
    j.in_dtype = dtype_code(in.scalar_type());
    j.out_dtype = dtype_code(out.scalar_type());
    return j;
}
void run_jobs(const snd_job *jobs, int n, hipStream_t stream, const char *what) {
    if (n > 0) check_status(snd_run_jobs(jobs, n, (snd_stream_t)stream), what);
}
at::Tensor floats(int64_t n, const at::Tensor &like) { return at::empty({n}, like.options().dtype(at::kFloat)); }

// The forward launch: clears what it accumulates into, and runs the kernel.  x == nullptr: no state is saved (x_v is then
// scratch of this call).
at::Tensor launch_fwd(const Checked &c, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B,
                      const at::Tensor &C, const OptTensor &D_, const OptTensor &delta_bias_, const OptTensor &A_decay_,
                      const Options &o, const OptTensor &merge_weights_, float *x, float *x_v, float *x_sd) {
    const auto f32 = u.options().dtype(at::kFloat);
    // merged: one fp32 channel per feature, to which every group adds its weighted result
    at::Tensor out = o.merge ? at::empty({c.batch, c.dim / c.n_groups, c.nrows, c.ncols}, f32)
                             : at::empty({c.batch, c.dim, c.nrows, c.ncols}, o.out_float ? f32 : u.options());
    auto stream = at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    snd_fwd_params p;
    fill_fwd(p, c, u, delta, A, B, C, D_, delta_bias_, A_decay_, o.delta_softplus);
    p.out = out.data_ptr();
    p.out_dtype = dtype_code(out.scalar_type());
    p.out_batch_stride = out.stride(0); p.out_d_stride = out.stride(1); p.out_h_stride = out.stride(2);
    p.schedule = o.sched;
    p.directions = (int32_t)o.directions;
    p.merge = o.merge ? 1 : 0;
    p.merge_weights = o.merge && merge_weights_.has_value() ? merge_weights_.value().data_ptr<float>() : nullptr;
    // scratch for the pipelined schedules, and for wide planes without saved state (only when it will be used); released to
    // the caching allocator in stream order
    const bool wave = wavefront(o.sched, c.plan), states = o.sched == SND_SCHED_AUTO && c.plan.wave_per_state;
    const bool need_ws = wave ? !x && c.plan.wavefront_workspace : !states && pipelined(o.sched, c.plan.auto_schedule);
    at::Tensor ws, scratch;
    if (need_ws) {
        ws = floats((c.plan.fwd_workspace_bytes + 3) / 4, u);
        p.workspace = ws.data_ptr();
        p.workspace_bytes = c.plan.fwd_workspace_bytes;
    }
    if (!x) {                                       // (where a wave takes whole rows it carries them in registers and touches none of it)
        const int64_t slabs = std::min(4, (int)c.plan.n_chunks_y);
        scratch = floats(wave || states ? 4 : c.plan.x_v_elems / c.plan.n_chunks_y * slabs, u);
        x_v = scratch.data_ptr<float>();
    }
    p.x = x; p.x_v = x_v; p.x_sd = x_sd;
    snd_job jobs[2];
    int nj = 0;
    if (o.merge && !snd_fwd_merge_stores(&c.shape, o.sched, (int)o.directions)) jobs[nj++] = clear_job(out.data_ptr(), out.numel() * 4);
    if (need_ws && !wave) jobs[nj++] = clear_job(ws.data_ptr(), snd_clear_bytes(&c.shape, o.sched, 0));
    run_jobs(jobs, nj, stream, "fwd");
    check_status(snd_fwd_cleared(&p, (snd_stream_t)stream), "fwd");
    check_pipeline(ws, stream, "fwd");
    return out;
}

void check_call(const Options &o) {
    TORCH_CHECK(o.directions == SND_DIR_TOPLEFT || o.directions == SND_DIR_CORNERS, "directions must be 0 (top-left) or 1 (four corners)");
    TORCH_CHECK(!o.merge || o.out_float, "the fused merge accumulates in float32: out_float must be true");
}

std::vector<at::Tensor> selective_scan_fwd(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A,
                                           const at::Tensor &B, const at::Tensor &C, const OptTensor &D_,
                                           const OptTensor &delta_bias_, bool delta_softplus, bool out_float,
                                           const OptTensor &A_decay_, int64_t directions, int64_t schedule, bool merge,
                                           const OptTensor &merge_weights_) {
    Options o{delta_softplus, out_float, directions, SND_SCHED_AUTO, merge};
    TORCH_CHECK(directions == SND_DIR_TOPLEFT || directions == SND_DIR_CORNERS, "directions must be 0 (top-left) or 1 (four corners)");
    const Checked c = check_inputs(u, delta, A, B, C, D_, delta_bias_, A_decay_);
    check_merge(c, merge, merge_weights_, u);
    check_call(o);
    o.sched = resolve_schedule(schedule);
    at::hip::HIPGuardMasqueradingAsCUDA device_guard{u.device()};
    const auto f32 = u.options().dtype(at::kFloat);
    at::Tensor x = at::empty({c.batch, c.dim, c.dstate, c.plan.n_chunks_x, c.plan.x_inner}, f32);
    at::Tensor x_v = at::empty({c.batch, c.dim, c.dstate, c.plan.n_chunks_y, c.plan.xv_inner}, f32);
    at::Tensor x_sd = at::empty({c.batch, c.dim, c.dstate, c.plan.n_chunks_x, c.plan.x_inner}, f32);
    at::Tensor out = launch_fwd(c, u, delta, A, B, C, D_, delta_bias_, A_decay_, o, merge_weights_, x.data_ptr<float>(),
                                x_v.data_ptr<float>(), x_sd.data_ptr<float>());
    return {out, x, x_v, x_sd};
}

struct Grads {
    at::Tensor du, ddelta, dA, dB, dC, dD, ddelta_bias, dA_decay, dmerge, dweights;
};

// The backward launch with its passes before (accumulators and sync words cleared, merge weights floored) and after it
// (dB / dC cast to the input dtype, du folded over the groups that share u and ddelta over the channels that share a
// delta, host.cpp:432-438; d merge_weights), each side one launch.
// want_weights: dweights = d merge_weights, of `weight_numel` elements (per channel, or per group), and the weights enter
// floored (SND_MERGE_WEIGHT_FLOOR); otherwise they enter as they are and only dmerge = weight * d(weight) is returned.
Grads launch_bwd(const Checked &c, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A, const at::Tensor &B,
                 const at::Tensor &C, const OptTensor &D_, const OptTensor &delta_bias_, const OptTensor &A_decay_, const at::Tensor &dout,
                 const float *x, const float *x_v, const float *x_sd, const Options &o, const OptTensor &merge_weights_,
                 bool floor_weights, int64_t weight_numel) {
    const int64_t dim = c.dim, HW = (int64_t)c.nrows * c.ncols;
    auto stream = at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream();
    Grads g;
    g.du = at::empty({c.batch, dim, c.nrows, c.ncols}, u.options());
    g.ddelta = at::empty({c.batch, dim, c.nrows, c.ncols}, u.options());
    // the accumulated gradients are zero-filled as host.cpp:395-403 does.  dB and dC share one buffer; the small ones (dA, dD,
    // ddelta_bias, dA_decay) share another, so that a parameter gradient kept by the optimizer never pins the large buffer.
    const int64_t nA = dim * c.dstate, nBC = B.numel();
    auto round64 = [](int64_t v) { return (v + 63) / 64 * 64; };
    // dB and dC are accumulated at equal offsets at the same time.  Where that matters (the row-segment kernels on
    // tensors of 2 MiB and more) dC starts a chosen distance past the 2 MiB-rounded end of dB (snd_plan.dC_skew_bytes:
    // not a multiple of 2 MiB apart); everywhere else it follows dB directly.
    const bool spread = c.plan.auto_schedule == SND_SCHED_WAVEFRONT && nBC * 4 >= (int64_t)(2 << 20);
    const int64_t oC = spread ? (round_2mib(nBC * 4) + c.plan.dC_skew_bytes) / 4 : round64(nBC);
    at::Tensor accBC = floats(oC + nBC, u);
    g.dB = accBC.narrow(0, 0, nBC).view(B.sizes());
    g.dC = accBC.narrow(0, oC, nBC).view(C.sizes());
    const bool merge = o.merge, weights = merge && merge_weights_.has_value();
    const int64_t oD = round64(nA), oBias = oD + round64(dim), oDec = oBias + round64(dim), oMerge = oDec + 64, nP = oMerge + (merge ? round64(dim) : 0);
    at::Tensor accP = floats(nP, u);
    g.dA = accP.narrow(0, 0, nA).view({dim, c.dstate});
    if (D_.has_value()) g.dD = accP.narrow(0, oD, dim);
    if (delta_bias_.has_value()) g.ddelta_bias = accP.narrow(0, oBias, dim);
    if (A_decay_.has_value()) g.dA_decay = accP.narrow(0, oDec, 1);
    if (merge) g.dmerge = accP.narrow(0, oMerge, dim);   // weight * d(weight) per channel
    at::Tensor ws, wfloor;                          // (the row-segment kernels need no workspace, except for planes taken in column groups or halves)
    if (!wavefront(o.sched, c.plan) || c.plan.wavefront_workspace) ws = floats((c.plan.bwd_workspace_bytes + 3) / 4, u);

    snd_job jobs[8];
    int nj = 0;
    // one job over both accumulators where the gap between them is small beside them
    if ((oC - nBC) * 4 <= nBC) {
        jobs[nj++] = clear_job(accBC.data_ptr(), (oC + nBC) * 4);
    } else {
        jobs[nj++] = clear_job(g.dB.data_ptr(), nBC * 4);
        jobs[nj++] = clear_job(g.dC.data_ptr(), nBC * 4);
    }
    jobs[nj++] = clear_job(accP.data_ptr(), nP * 4);
    if (ws.defined()) jobs[nj++] = clear_job(ws.data_ptr(), snd_clear_bytes(&c.shape, o.sched, 1));
    if (weights && floor_weights) {
        wfloor = floats(dim, u);
        snd_job j{};
        j.kind = SND_JOB_WEIGHT_FLOOR;
        j.in = merge_weights_.value().data_ptr();
        j.out = wfloor.data_ptr();
        j.outer = 1; j.cols = dim; j.rows = 1;
        jobs[nj++] = j;
    }
    run_jobs(jobs, nj, stream, "bwd");

    snd_bwd_params p;
    memset(&p, 0, sizeof(p));
    fill_fwd(p.f, c, u, delta, A, B, C, D_, delta_bias_, A_decay_, o.delta_softplus);
    p.f.x = const_cast<float *>(x); p.f.x_v = const_cast<float *>(x_v); p.f.x_sd = const_cast<float *>(x_sd);
    p.dout = dout.data_ptr();
    p.dout_dtype = dtype_code(dout.scalar_type());
    p.dout_batch_stride = dout.stride(0); p.dout_d_stride = dout.stride(1); p.dout_h_stride = dout.stride(2);
    p.du = g.du.data_ptr(); p.ddelta = g.ddelta.data_ptr();
    p.dA = g.dA.data_ptr<float>(); p.dB = g.dB.data_ptr<float>(); p.dC = g.dC.data_ptr<float>();
    p.dD = g.dD.defined() ? g.dD.data_ptr<float>() : nullptr;
    p.ddelta_bias = g.ddelta_bias.defined() ? g.ddelta_bias.data_ptr<float>() : nullptr;
    p.dA_decay = g.dA_decay.defined() ? g.dA_decay.data_ptr<float>() : nullptr;
    p.workspace = ws.defined() ? ws.data_ptr() : nullptr;
    p.workspace_bytes = ws.defined() ? c.plan.bwd_workspace_bytes : 0;
    p.f.schedule = o.sched;
    p.f.directions = (int32_t)o.directions;
    p.f.merge = merge ? 1 : 0;
    p.f.merge_weights = wfloor.defined() ? wfloor.data_ptr<float>() : weights ? merge_weights_.value().data_ptr<float>() : nullptr;
    p.dmerge = merge ? g.dmerge.data_ptr<float>() : nullptr;
    check_status(snd_bwd_cleared(&p, (snd_stream_t)stream), "bwd");
    if (o.sched == SND_SCHED_STRIPS || o.sched == SND_SCHED_BANDS || (o.sched == SND_SCHED_AUTO && c.plan.auto_bwd_jobs != 0))
        check_pipeline(ws, stream, "bwd");

    nj = 0;
    if (B.scalar_type() != at::kFloat) {
        at::Tensor cast = at::empty({2 * round64(nBC)}, B.options());
        at::Tensor dBc = cast.narrow(0, 0, nBC).view(B.sizes()), dCc = cast.narrow(0, round64(nBC), nBC).view(C.sizes());
        jobs[nj++] = sum_job(g.dB, 1, 1, nBC, dBc);
        jobs[nj++] = sum_job(g.dC, 1, 1, nBC, dCc);
        g.dB = dBc;
        g.dC = dCc;
    }
    at::Tensor du_all, dd_all, db_all;              // (kept until the launch below is enqueued)
    if (dim != c.delta_dim) {
        const int rep = dim / c.delta_dim;
        dd_all = g.ddelta;
        g.ddelta = at::empty({c.batch, c.delta_dim, c.nrows, c.ncols}, u.options());
        jobs[nj++] = sum_job(dd_all, (int64_t)c.batch * c.delta_dim, rep, HW, g.ddelta);
        if (delta_bias_.has_value()) {
            db_all = g.ddelta_bias;
            g.ddelta_bias = floats(c.delta_dim, u);
            jobs[nj++] = sum_job(db_all, c.delta_dim, rep, 1, g.ddelta_bias);
        }
    }
    if (c.u_shared) {   // one feature map scanned by every group: its gradient is the sum over the groups
        du_all = g.du;
        g.du = at::empty({c.batch, dim / c.n_groups, c.nrows, c.ncols}, u.options());
        jobs[nj++] = sum_job(du_all, c.batch, c.n_groups, dim / c.n_groups * HW, g.du);
    }
    if (weights && weight_numel > 0) {
        g.dweights = floats(weight_numel, u);
        snd_job j{};
        j.kind = weight_numel == dim ? SND_JOB_WEIGHT : SND_JOB_WEIGHT_GROUP;
        j.in = g.dmerge.data_ptr(); j.in2 = merge_weights_.value().data_ptr(); j.out = g.dweights.data_ptr();
        j.outer = c.n_groups; j.cols = dim / c.n_groups; j.rows = 1;
        jobs[nj++] = j;
    }
    run_jobs(jobs, nj, stream, "bwd");
    return g;
}

void check_dout(const Checked &c, const at::Tensor &u, const at::Tensor &dout, bool merge) {
    const int batch_size = c.batch, dim = c.dim, nrows = c.nrows, ncols = c.ncols;
    TORCH_CHECK(dout.scalar_type() == u.scalar_type() || dout.scalar_type() == at::ScalarType::Float,
                "dout must be float32 or the input dtype");
    TORCH_CHECK(dout.is_cuda());
    TORCH_CHECK(dout.stride(-1) == 1 || dout.size(-1) == 1, "dout must be contiguous in its last dimension");
    CHECK_SHAPE(dout, batch_size, merge ? dim / c.n_groups : dim, nrows, ncols);   // merged: the gradient of the merged output
}

std::vector<at::Tensor> selective_scan_bwd(const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A,
                                           const at::Tensor &B, const at::Tensor &C, const OptTensor &D_,
                                           const OptTensor &delta_bias_, const at::Tensor &dout, const OptTensor &x_,
                                           const OptTensor &x_v_, bool delta_softplus, const OptTensor &A_decay_,
                                           const OptTensor &x_sd_, int64_t directions, int64_t schedule, bool merge,
                                           const OptTensor &merge_weights_) {
    Options o{delta_softplus, true, directions, SND_SCHED_AUTO, merge};
    check_call(o);
    const Checked c = check_inputs(u, delta, A, B, C, D_, delta_bias_, A_decay_);
    check_merge(c, merge, merge_weights_, u);
    const int batch_size = c.batch, dim = c.dim, dstate = c.dstate;
    check_dout(c, u, dout, merge);
    // the saved state is required: gradients computed without it would belong to another function
    TORCH_CHECK(x_.has_value() && x_v_.has_value() && x_sd_.has_value(),
                "bwd needs the x, x_v and x_sd tensors returned by fwd");
    const auto &x = x_.value(), &x_v = x_v_.value(), &x_sd = x_sd_.value();
    const int nChunksX = c.plan.n_chunks_x, nChunksY = c.plan.n_chunks_y, x_inner = c.plan.x_inner,
              xv_inner = c.plan.xv_inner;
    for (const at::Tensor *t : {&x, &x_v, &x_sd}) {
        TORCH_CHECK(t->scalar_type() == at::ScalarType::Float && t->is_cuda() && t->is_contiguous(),
                    "saved state must be contiguous float32 GPU tensors");
    }
    CHECK_SHAPE(x, batch_size, dim, dstate, nChunksX, x_inner);
    CHECK_SHAPE(x_sd, batch_size, dim, dstate, nChunksX, x_inner);
    CHECK_SHAPE(x_v, batch_size, dim, dstate, nChunksY, xv_inner);
    o.sched = resolve_schedule(schedule);
    at::hip::HIPGuardMasqueradingAsCUDA device_guard{u.device()};
    Grads g = launch_bwd(c, u, delta, A, B, C, D_, delta_bias_, A_decay_, dout, x.data_ptr<float>(), x_v.data_ptr<float>(),
                         x_sd.data_ptr<float>(), o, merge_weights_, false, 0);
    std::vector<at::Tensor> result = {g.du, g.ddelta, g.dA, g.dB, g.dC, g.dD, g.ddelta_bias, g.dA_decay};
    if (merge) result.push_back(g.dmerge);
    return result;
}

at::Tensor rows_contiguous(const at::Tensor &t) { return t.stride(-1) == 1 || t.size(-1) == 1 ? t : t.contiguous(); }
OptTensor optional_of(const at::Tensor &t) { return t.defined() ? OptTensor(t) : OptTensor(); }

// Held by the functions below in both directions.  Their types are settled before they are called, and the raw pointers they
// pass on are of those types: no call inside them may be cast.  In the backward autocast is in whatever state backward() was
// called under (the engine hands it to its threads), which need not be the forward's.
struct NoAutocast {
    c10::impl::ExcludeDispatchKeyGuard off{c10::autocast_dispatch_keyset};
};
// A tensor whose pointer goes to a kernel as `numel` elements of `type`: the result of a library call, or one saved for the
// backward (saved-tensor hooks may hand back another than was saved).
void check_elements(const at::Tensor &t, at::ScalarType type, const at::Device &device, int64_t numel, const char *what) {
    TORCH_CHECK(t.defined() && t.scalar_type() == type && t.device() == device && t.is_contiguous() && t.numel() == numel,
                "selective_nd_scan: ", what, " is not a contiguous ", toString(type), " tensor of ", numel, " elements on ", device);
}

// Gradients that come out of kernels have no graph behind them.  Under create_graph they leave through a node that raises
// when it is differentiated: a second derivative is refused instead of being short of a term.
torch::autograd::variable_list once_differentiable(torch::autograd::variable_list r, const char *what) {
    if (!at::GradMode::is_enabled()) return r;
    torch::autograd::variable_list given;
    for (const at::Tensor &t : r)
        if (t.defined()) given.push_back(t.detach().set_requires_grad(true));
    auto refuse = std::make_shared<torch::autograd::DelayedError>(std::string(what) + " can be differentiated once: its gradients have no derivative", (int64_t)given.size());
    const torch::autograd::variable_list out = (*refuse)(std::move(given));
    size_t k = 0;
    for (at::Tensor &t : r)
        if (t.defined()) t = out[k++];
    return r;
}

// The differentiable scan.  The saved state is one buffer [x | x_sd | x_v] that only the backward reads.
// The block mapping is resolved once, in the forward, and the backward runs the same one: the two kernel families keep
// different saved-state layouts, so a default changed between a forward and its backward must not reach it.
struct ScanFn : public torch::autograd::Function<ScanFn> {
    static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &u, const at::Tensor &delta, const at::Tensor &A,
                              const at::Tensor &B, const at::Tensor &C, const OptTensor &D_, const OptTensor &delta_bias_,
                              const OptTensor &A_decay_, const OptTensor &weights_, bool delta_softplus, bool out_float,
                              int64_t directions, bool merge) {
        at::AutoDispatchBelowADInplaceOrView below;
        NoAutocast no_autocast;
        Options o{delta_softplus, out_float, directions, resolve_schedule(-1), merge};
        OptTensor w;
        const Checked c = check_inputs(u, delta, A, B, C, D_, delta_bias_, A_decay_);
        if (weights_.has_value())                   // [G], [G, 1] or [G, D/G] -> one per channel
            w = weights_.value().to(at::kFloat).reshape({c.n_groups, -1}).expand({c.n_groups, c.dim / c.n_groups}).contiguous().view(-1);
        check_merge(c, merge, w, u);
        check_call(o);
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{u.device()};
        const int64_t nx = (c.plan.x_elems + 63) / 64 * 64;
        at::Tensor state = floats(2 * nx + c.plan.x_v_elems, u);
        float *st = state.data_ptr<float>();
        at::Tensor out = launch_fwd(c, u, delta, A, B, C, D_, delta_bias_, A_decay_, o, w, st, st + 2 * nx, st + nx);
        ctx->save_for_backward({u, delta, A, B, C, D_.value_or(at::Tensor()), delta_bias_.value_or(at::Tensor()), A_decay_.value_or(at::Tensor()),
                                w.value_or(at::Tensor()), state});
        ctx->saved_data["softplus"] = delta_softplus;
        ctx->saved_data["directions"] = directions;
        ctx->saved_data["sched"] = (int64_t)o.sched;
        ctx->saved_data["merge"] = merge;
        if (weights_.has_value()) {
            ctx->saved_data["w_shape"] = weights_.value().sizes().vec();
            ctx->saved_data["w_dtype"] = (int64_t)weights_.value().scalar_type();
        }
        return out;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        return once_differentiable(gradients(ctx, std::move(grads)), "selective_nd_scan");
    }
    static torch::autograd::variable_list gradients(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        at::NoGradGuard no_grad;
        NoAutocast no_autocast;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &u = saved[0], &delta = saved[1], &A = saved[2], &B = saved[3], &C = saved[4], &state = saved[9];
        const OptTensor D_ = optional_of(saved[5]), delta_bias_ = optional_of(saved[6]), A_decay_ = optional_of(saved[7]), w = optional_of(saved[8]);
        torch::autograd::variable_list r(13);
        if (!grads[0].defined()) return r;
        Options o{ctx->saved_data["softplus"].toBool(), true, ctx->saved_data["directions"].toInt(), (int)ctx->saved_data["sched"].toInt(),
                  ctx->saved_data["merge"].toBool()};
        const Checked c = check_inputs(u, delta, A, B, C, D_, delta_bias_, A_decay_);
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{u.device()};
        const at::Tensor dout = rows_contiguous(grads[0]);
        check_dout(c, u, dout, o.merge);
        check_merge(c, o.merge, w, u);
        const int64_t nx = (c.plan.x_elems + 63) / 64 * 64;
        check_elements(state, at::kFloat, u.device(), 2 * nx + c.plan.x_v_elems, "the saved state");
        const float *st = state.data_ptr<float>();
        int64_t wn = 0;
        if (w.has_value()) {
            wn = 1;
            for (int64_t s : ctx->saved_data["w_shape"].toIntVector()) wn *= s;
        }
        Grads g = launch_bwd(c, u, delta, A, B, C, D_, delta_bias_, A_decay_, dout, st, st + 2 * nx, st + nx, o, w, true, wn);
        r[0] = g.du; r[1] = g.ddelta; r[2] = g.dA; r[3] = g.dB; r[4] = g.dC; r[5] = g.dD; r[6] = g.ddelta_bias; r[7] = g.dA_decay;
        if (wn > 0) r[8] = g.dweights.view(ctx->saved_data["w_shape"].toIntVector()).to((at::ScalarType)ctx->saved_data["w_dtype"].toInt());
        return r;
    }
};

// Whether a forward-mode tangent is attached (it is where requires_grad() says no, and the raw path would drop it).
bool has_tangent(const at::Tensor &t) { return t._fw_grad(/*level=*/0).defined(); }

// selective_nd_scan / selective_nd_scan_merged: the differentiable function where a gradient can be asked for, the forward
// that saves no state where none can.
at::Tensor scan(const at::Tensor &u_, const at::Tensor &delta_, const at::Tensor &A, const at::Tensor &B_, const at::Tensor &C_,
                const OptTensor &D_, const OptTensor &delta_bias_, bool delta_softplus, bool out_float, const OptTensor &A_decay_,
                int64_t directions, bool merge, const OptTensor &weights_) {
    TORCH_CHECK(u_.dim() == 4 && delta_.dim() == 4 && A.dim() == 2 && B_.dim() == 5 && C_.dim() == 5, "expected u, delta 4-D; A 2-D; B, C 5-D");
    const at::Tensor u = rows_contiguous(u_), delta = rows_contiguous(delta_), B = rows_contiguous(B_), C = rows_contiguous(C_);
    for (const at::Tensor *t : {&u, &delta, &A, &B, &C}) TORCH_CHECK(!has_tangent(*t), "selective_nd_scan has no forward-mode derivative");
    for (const OptTensor *t : {&D_, &delta_bias_, &A_decay_, &weights_})
        TORCH_CHECK(!t->has_value() || !has_tangent(t->value()), "selective_nd_scan has no forward-mode derivative");
    bool grad = false;
    if (at::GradMode::is_enabled()) {
        for (const at::Tensor *t : {&u, &delta, &A, &B, &C}) grad = grad || t->requires_grad();
        for (const OptTensor *t : {&D_, &delta_bias_, &A_decay_, &weights_}) grad = grad || (t->has_value() && t->value().requires_grad());
    }
    if (grad) return ScanFn::apply(u, delta, A, B, C, D_, delta_bias_, A_decay_, weights_, delta_softplus, out_float, directions, merge);
    at::AutoDispatchBelowADInplaceOrView below;
    Options o{delta_softplus, out_float, directions, resolve_schedule(-1), merge};
    const Checked c = check_inputs(u, delta, A, B, C, D_, delta_bias_, A_decay_);
    OptTensor w;
    if (weights_.has_value())
        w = weights_.value().to(at::kFloat).reshape({c.n_groups, -1}).expand({c.n_groups, c.dim / c.n_groups}).contiguous().view(-1);
    check_merge(c, merge, w, u);
    check_call(o);
    at::hip::HIPGuardMasqueradingAsCUDA device_guard{u.device()};
    return launch_fwd(c, u, delta, A, B, C, D_, delta_bias_, A_decay_, o, w, nullptr, nullptr, nullptr);
}

// ---------------------------------------------------------------- the passes of a VSS block around its scan
hipStream_t current_stream() { return at::hip::getCurrentHIPStreamMasqueradingAsCUDA().stream(); }
at::Tensor f32c(const at::Tensor &t) { return t.to(at::kFloat).contiguous(); }
// (undefined: an optional tensor that was not given)
void check_device(const char *what, const at::Tensor &x, std::initializer_list<at::Tensor> others) {
    TORCH_CHECK(x.is_cuda(), what, ": the tensors must be on the GPU");
    for (const at::Tensor &t : others) TORCH_CHECK(!t.defined() || t.device() == x.device(), what, ": the tensors must be on one device");
}
const float *ptr_or_null(const OptTensor &t) { return t.has_value() ? t.value().data_ptr<float>() : nullptr; }

// LayerNorm over the last axis of a contiguous x, its result in `out_dtype` (what the next layer reads under autocast); gamma and
// beta fp32.  Its gradients are torch calls on the saved inputs under create_graph, where they are differentiated again, and where
// deterministic algorithms are asked for: the kernel adds up dgamma and dbeta with atomics.
struct NormFn : public torch::autograd::Function<NormFn> {
    static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &x, const at::Tensor &gamma, const at::Tensor &beta, double eps,
                              int64_t out_dtype) {
        at::AutoDispatchBelowADInplaceOrView below;
        NoAutocast no_autocast;
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{x.device()};
        const int64_t C = x.size(-1), tokens = x.numel() / C;
        at::Tensor y = at::empty(x.sizes(), x.options().dtype((at::ScalarType)out_dtype)), stats = floats(2 * tokens, x);
        check_status(snd_block_norm_fwd(x.data_ptr(), dtype_code(x.scalar_type()), gamma.data_ptr<float>(), beta.data_ptr<float>(), (float)eps, tokens, (int)C,
                                        y.data_ptr(), dtype_code(y.scalar_type()), stats.data_ptr<float>(), (snd_stream_t)current_stream()), "norm");
        ctx->save_for_backward({x, gamma, stats});
        ctx->saved_data["eps"] = eps;
        return y;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        NoAutocast no_autocast;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &x = saved[0], &gamma = saved[1], &stats = saved[2];
        torch::autograd::variable_list r(5);
        if (!grads[0].defined()) return r;
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{x.device()};
        const int64_t C = x.size(-1), tokens = x.numel() / C;
        check_elements(x, x.scalar_type(), grads[0].device(), grads[0].numel(), "x");
        check_elements(gamma, at::kFloat, x.device(), C, "gamma");
        check_elements(stats, at::kFloat, x.device(), 2 * tokens, "the statistics");
        if (at::GradMode::is_enabled() || at::globalContext().deterministicAlgorithms()) {
            const at::Tensor xf = x.to(at::kFloat), d = grads[0].to(at::kFloat), xc = xf - xf.mean(-1, true);
            const at::Tensor rstd = (xc * xc).mean(-1, true).add(ctx->saved_data["eps"].toDouble()).rsqrt(), xh = xc * rstd, dn = d * gamma;
            r[0] = (rstd * (dn - dn.mean(-1, true) - xh * (dn * xh).mean(-1, true))).to(x.scalar_type());
            r[1] = (d * xh).reshape({tokens, C}).sum(0);
            r[2] = d.reshape({tokens, C}).sum(0);
            return r;
        }
        const at::Tensor dy = grads[0].contiguous();
        at::Tensor dx = at::empty_like(x), acc = at::zeros({2, C}, x.options().dtype(at::kFloat));
        check_status(snd_block_norm_bwd(dy.data_ptr(), dtype_code(dy.scalar_type()), x.data_ptr(), dtype_code(x.scalar_type()), gamma.data_ptr<float>(),
                                        stats.data_ptr<float>(), tokens, (int)C, dx.data_ptr(), acc.data_ptr<float>(), acc.data_ptr<float>() + C,
                                        (snd_stream_t)current_stream()), "norm");
        r[0] = dx;
        r[1] = acc[0];
        r[2] = acc[1];
        return r;
    }
};
at::Tensor block_norm(const at::Tensor &x, const at::Tensor &gamma, const at::Tensor &beta, double eps, const at::Tensor &like) {
    TORCH_CHECK(x.dim() >= 1 && gamma.dim() == 1 && beta.dim() == 1 && gamma.size(0) == x.size(-1) && beta.size(0) == x.size(-1),
                "block_norm: the last axis of x has another size than gamma or beta");
    check_device("block_norm", x, {gamma, beta});
    return NormFn::apply(x.contiguous(), f32c(gamma), f32c(beta), eps, (int64_t)like.scalar_type());
}

// A linear layer in the 16-bit type of x (what autocast makes of F.linear) whose weight and bias gradients are summed over the
// tokens by the extension's kernel where linear_wgrad_pays says so: the library's product has a block per tile of the result and
// walks all tokens in each, the kernel splits the tokens over the grid and pays with atomics.
// Kernel / library (product, sum over the tokens, casts), bf16, us, by tokens:
//     M x N           784        3136       12544        32768       100352       401408
//     768 x 384     11 / 41    19 / 48    34 /  97     66 / 183    187 / 372    740 / 1102
//     1024 x 512    13 / 45    23 / 51    51 / 106    115 / 203    339 / 476   1352 / 1439
//     1536 x 384    15 / 41    24 / 53    56 / 102    124 / 209    398 / 532   1751 / 1659
//     1024 x 768    18 / 41    28 / 49    65 / 102    151 / 231    471 / 575   1997 / 1513
//     1024 x 1024   19 / 40    31 / 49    85 / 107    203 / 233    653 / 585   2765 / 1641
// Up to 2^19 elements it is the kernel at any number of tokens: its sums are fp32, the library's result is rounded to 16 bits.
// From there on the line is where a slower kernel met the library (1024 x 768: 218 / 228 at 32768 tokens, 689 / 574 at 100352); as it is now
// the kernel would be faster beyond it, up to 100352 tokens at 1024 x 768 and up to 32768 at 1024 x 1024.
bool linear_wgrad_pays(int64_t tokens, int64_t M, int64_t N) {
    return M % 2 == 0 && N % 2 == 0 && (M * N <= (int64_t)1 << 19 || (M * N <= (int64_t)3 << 18 && tokens <= 1 << 15));
}
struct LinearFn : public torch::autograd::Function<LinearFn> {
    static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &x, const at::Tensor &w_, const OptTensor &b_) {
        at::AutoDispatchBelowADInplaceOrView below;
        NoAutocast no_autocast;
        const auto T = x.scalar_type();
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{x.device()};
        at::Tensor w = w_, b = b_.value_or(at::Tensor());
        if (b.defined() && w.scalar_type() == at::kFloat && b.scalar_type() == at::kFloat && w.is_contiguous() && b.is_contiguous()) {
            w = at::empty(w_.sizes(), x.options());  // both casts in one launch
            b = at::empty(b_.value().sizes(), x.options());
            const snd_job jobs[] = {sum_job(w_, 1, 1, w_.numel(), w), sum_job(b_.value(), 1, 1, b.numel(), b)};
            run_jobs(jobs, 2, current_stream(), "linear");
        } else {
            w = w.to(T).contiguous();
            if (b.defined()) b = b.to(T);
        }
        ctx->save_for_backward({x, w});
        if (!w.is_same(w_)) ctx->saved_data["w_in"] = w_;   // (the copy saved above has no history; used under create_graph alone)
        ctx->saved_data["w"] = (int64_t)w_.scalar_type();
        ctx->saved_data["b"] = b_.has_value() ? (int64_t)b_.value().scalar_type() : (int64_t)-1;
        return at::linear(x, w, optional_of(b));
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        NoAutocast no_autocast;
        const auto sv = ctx->get_saved_variables();
        const at::Tensor &x = sv[0];
        at::Tensor w = sv[1];
        torch::autograd::variable_list r(3);
        if (!grads[0].defined()) return r;
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{x.device()};
        const int64_t M = w.size(0), N = w.size(1), tokens = x.numel() / N, btype = ctx->saved_data["b"].toInt();
        check_elements(x, w.scalar_type(), w.device(), tokens * N, "x");
        const auto wtype = (at::ScalarType)ctx->saved_data["w"].toInt();
        const bool graph = at::GradMode::is_enabled();      // create_graph: torch calls on the inputs, which can be differentiated again
        if (graph && ctx->saved_data.count("w_in")) {       // the values of the saved copy, the history of the parameter
            const at::Tensor now = ctx->saved_data["w_in"].toTensor().to(x.scalar_type());
            w = w + (now - now.detach());
        }
        const at::Tensor dy = grads[0].to(x.scalar_type()).contiguous().view({tokens, M}), x2 = x.view({tokens, N});
        if (ctx->needs_input_grad(0)) r[0] = at::mm(dy, w).view(x.sizes());
        // (edges: x, weight and, where there is one, bias)
        const bool dw = ctx->needs_input_grad(1), db = btype >= 0 && ctx->needs_input_grad(2);
        if (dw && !graph && !at::globalContext().deterministicAlgorithms() && linear_wgrad_pays(tokens, M, N)) {
            const int64_t nw = (M * N + 15) / 16 * 16;     // (the kernel adds up with atomics)
            at::Tensor acc = at::zeros({nw + M}, x.options().dtype(at::kFloat));
            float *p = acc.data_ptr<float>();
            check_status(snd_block_linear_wgrad(dy.data_ptr(), x2.data_ptr(), tokens, (int)M, (int)N, dtype_code(x.scalar_type()), p, db ? p + nw : nullptr,
                                                (snd_stream_t)current_stream()), "linear");
            r[1] = acc.narrow(0, 0, M * N).view({M, N}).to(wtype);
            if (db) r[2] = acc.narrow(0, nw, M).to((at::ScalarType)btype);
        } else {
            if (dw) r[1] = at::mm(dy.t(), x2).to(wtype);
            if (db) r[2] = dy.sum(0).to((at::ScalarType)btype);
        }
        return r;
    }
};
at::Tensor block_linear(const at::Tensor &x, const at::Tensor &w, const OptTensor &b, const at::Tensor &like) {
    TORCH_CHECK(x.dim() >= 1 && w.dim() == 2 && w.size(1) == x.size(-1) && (!b.has_value() || (b.value().dim() == 1 && b.value().size(0) == w.size(0))),
                "block_linear: the shapes of x, weight and bias do not fit");
    TORCH_CHECK(like.scalar_type() == at::kHalf || like.scalar_type() == at::kBFloat16, "block_linear: the type of `like` must be float16 or bfloat16");
    check_device("block_linear", x, {w, b.value_or(at::Tensor())});
    return LinearFn::apply(x.to(like.scalar_type()).contiguous(), w, b);
}

// Whether kernels may stand in for torch layers on these tensors (an optional one that was not given is None): they lie on one
// GPU and are ordinary tensors (a DTensor, FakeTensor or other subclass has no memory of its own to point to), and nothing around
// the call has to see the layers' own calls - tracing, a function transform, a dispatch mode, a forward-mode tangent.
bool plain(const std::vector<OptTensor> &ts) {
    if (at::tracer::impl::is_dispatch_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
        c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
        return false;
    const at::Tensor *first = nullptr;
    for (const OptTensor &o : ts) {
        if (!o.has_value()) continue;
        const at::Tensor &t = o.value();
        if (!t.is_cuda() || t.layout() != at::kStrided || t.key_set().has(c10::DispatchKey::Python) || has_tangent(t)) return false;
        if (first && t.device() != first->device()) return false;
        first = &t;
    }
    return true;
}

// Everything between in_proj and out_proj of SS2DCrossScan: xz [B, H, W, 2 * inner] -> [B, H, W, inner].
struct Ss2dFn : public torch::autograd::Function<Ss2dFn> {
    static snd_block_shape shape_of(const at::Tensor &xz, const at::Tensor &wdt, const at::Tensor &A) {
        snd_block_shape s;
        s.batch = (int)xz.size(0); s.nrows = (int)xz.size(1); s.ncols = (int)xz.size(2); s.inner = (int)(xz.size(3) / 2);
        s.n_groups = (int)wdt.size(0); s.rank = (int)wdt.size(2); s.dstate = (int)A.size(1);
        s.dtype = dtype_code(xz.scalar_type());
        return s;
    }
    static at::Tensor forward(torch::autograd::AutogradContext *ctx, const at::Tensor &xz_, const at::Tensor &conv_w_, const OptTensor &conv_b_,
                              const at::Tensor &wx_, const at::Tensor &wdt_, const at::Tensor &dt_bias_, const at::Tensor &A_logs_, const at::Tensor &D_,
                              const OptTensor &mw_, const at::Tensor &gamma_, const at::Tensor &beta_, double eps, bool grad) {
        at::AutoDispatchBelowADInplaceOrView below;
        NoAutocast no_autocast;
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{xz_.device()};
        const snd_stream_t stream = (snd_stream_t)current_stream();
        const at::Tensor xz = xz_.contiguous(), conv_w = f32c(conv_w_), wdt = f32c(wdt_), gamma = f32c(gamma_), beta = f32c(beta_), Dv = f32c(D_);
        const at::Tensor dt_bias = f32c(dt_bias_).view(-1), A_logs = f32c(A_logs_), wx32 = f32c(wx_);
        const OptTensor conv_b = conv_b_.has_value() ? OptTensor(f32c(conv_b_.value())) : OptTensor();
        const snd_block_shape s = shape_of(xz, wdt, A_logs);
        const int64_t B = s.batch, H = s.nrows, W = s.ncols, Di = s.inner, K = s.n_groups, N = s.dstate, R = s.rank, M = R + 2 * N, HW = H * W;
        at::Tensor u = at::empty({B, Di, H, W}, xz.options()), pre = grad ? at::empty({B, Di, H, W}, xz.options()) : at::Tensor();
        check_status(snd_block_conv_fwd(&s, xz.data_ptr(), conv_w.data_ptr<float>(), ptr_or_null(conv_b), grad ? pre.data_ptr() : nullptr, u.data_ptr(), stream),
                     "block");
        at::Tensor A = at::empty_like(A_logs), wx = at::empty({1, K * M, Di}, xz.options()), wxt = grad ? at::empty({1, Di, K * M}, xz.options()) : at::Tensor();
        check_status(snd_block_params(A_logs.data_ptr<float>(), (int)A.numel(), wx32.data_ptr<float>(), (int)(K * M), (int)Di, s.dtype, A.data_ptr<float>(),
                                      wx.data_ptr(), grad ? wxt.data_ptr() : nullptr, stream), "block");
        const at::Tensor proj = at::bmm(wx.expand({B, K * M, Di}), u.view({B, Di, HW}));                 // [B, K * (R + 2N), HW]
        check_elements(proj, xz.scalar_type(), xz.device(), B * K * M * HW, "the projection");
        at::Tensor delta = at::empty({B, K * Di, H, W}, xz.options());
        check_status(snd_block_dt_fwd(&s, proj.data_ptr(), wdt.data_ptr<float>(), delta.data_ptr(), stream), "block");
        const at::Tensor p5 = proj.view({B, K, M, H, W}), Bs = p5.narrow(2, R, N), Cs = p5.narrow(2, R + N, N);
        OptTensor w;
        if (mw_.has_value()) w = f32c(mw_.value()).reshape({K, -1}).expand({K, Di}).contiguous().view(-1);
        Options o{true, true, SND_DIR_CORNERS, resolve_schedule(-1), true};
        const Checked c = check_inputs(u, delta, A, Bs, Cs, Dv, dt_bias, OptTensor());
        check_merge(c, true, w, u);
        const int64_t nx = (c.plan.x_elems + 63) / 64 * 64;
        at::Tensor state;
        float *st = nullptr;
        if (grad) {
            state = floats(2 * nx + c.plan.x_v_elems, u);
            st = state.data_ptr<float>();
        }
        const at::Tensor y = launch_fwd(c, u, delta, A, Bs, Cs, Dv, dt_bias, OptTensor(), o, w, st, st ? st + 2 * nx : nullptr, st ? st + nx : nullptr);
        at::Tensor out = at::empty({B, H, W, Di}, xz.options()), stats = grad ? floats(2 * B * HW, u) : at::Tensor();
        check_status(snd_block_gate_fwd(&s, y.data_ptr<float>(), xz.data_ptr(), gamma.data_ptr<float>(), beta.data_ptr<float>(), (float)eps, out.data_ptr(),
                                        grad ? stats.data_ptr<float>() : nullptr, stream), "block");
        if (!grad) return out;
        ctx->save_for_backward({xz, conv_w, conv_b.value_or(at::Tensor()), wxt, wdt, dt_bias, A, Dv, w.value_or(at::Tensor()), gamma, beta, u, pre, proj, delta, y,
                                stats, state});
        ctx->saved_data["sched"] = (int64_t)o.sched;
        if (mw_.has_value()) ctx->saved_data["mw_shape"] = mw_.value().sizes().vec();
        const at::Tensor *params[] = {&conv_w_, conv_b_.has_value() ? &conv_b_.value() : nullptr, &wx_, &wdt_, &dt_bias_, &A_logs_, &D_,
                                      mw_.has_value() ? &mw_.value() : nullptr, &gamma_, &beta_};
        std::vector<int64_t> types;
        for (const at::Tensor *t : params) types.push_back(t ? (int64_t)t->scalar_type() : -1);
        ctx->saved_data["types"] = types;
        return out;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        return once_differentiable(gradients(ctx, std::move(grads)), "SS2DCrossScan");
    }
    static torch::autograd::variable_list gradients(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        at::NoGradGuard no_grad;
        NoAutocast no_autocast;
        const auto sv = ctx->get_saved_variables();
        torch::autograd::variable_list r(13);
        if (!grads[0].defined()) return r;
        const at::Tensor &xz = sv[0], &conv_w = sv[1], &wxt = sv[3], &wdt = sv[4], &dt_bias = sv[5], &A = sv[6], &Dv = sv[7], &gamma = sv[9], &beta = sv[10],
                         &u = sv[11], &pre = sv[12], &proj = sv[13], &delta = sv[14], &y = sv[15], &stats = sv[16], &state = sv[17];
        const OptTensor conv_b = optional_of(sv[2]), w = optional_of(sv[8]);
        at::hip::HIPGuardMasqueradingAsCUDA device_guard{xz.device()};
        const snd_stream_t stream = (snd_stream_t)current_stream();
        const snd_block_shape s = shape_of(xz, wdt, A);
        const int64_t B = s.batch, H = s.nrows, W = s.ncols, Di = s.inner, K = s.n_groups, N = s.dstate, R = s.rank, M = R + 2 * N, HW = H * W;
        const at::Tensor dout = grads[0].to(xz.scalar_type()).contiguous();
        const auto T = xz.scalar_type();
        const struct { const at::Tensor *t; at::ScalarType type; int64_t numel; const char *what; } saved[] = {
            {&dout, T, B * HW * Di, "the gradient"}, {&xz, T, B * HW * 2 * Di, "xz"}, {&wxt, T, Di * K * M, "the projection's weight"}, {&u, T, B * Di * HW, "u"},
            {&pre, T, B * Di * HW, "the convolution"}, {&proj, T, B * K * M * HW, "the projection"}, {&delta, T, B * K * Di * HW, "delta"},
            {&y, at::kFloat, B * Di * HW, "y"}, {&stats, at::kFloat, 2 * B * HW, "the statistics"}, {&conv_w, at::kFloat, Di * 9, "the convolution's weight"},
            {&wdt, at::kFloat, K * Di * R, "the step sizes' weight"}, {&gamma, at::kFloat, Di, "gamma"}, {&beta, at::kFloat, Di, "beta"}};
        for (const auto &v : saved) check_elements(*v.t, v.type, grads[0].device(), v.numel, v.what);
        // the accumulated parameter gradients: conv weight and bias, the two projections, gamma, beta
        const int64_t sizes[] = {Di * 9, Di, K * M * Di, K * Di * R, Di, Di};
        int64_t off[7] = {0};
        for (int i = 0; i < 6; ++i) off[i + 1] = off[i] + (sizes[i] + 15) / 16 * 16;
        at::Tensor acc = at::zeros({off[6]}, xz.options().dtype(at::kFloat));
        float *ap = acc.data_ptr<float>();
        at::Tensor dy = at::empty_like(y), dxz = at::empty_like(xz);
        check_status(snd_block_gate_bwd(&s, dout.data_ptr(), y.data_ptr<float>(), xz.data_ptr(), gamma.data_ptr<float>(), beta.data_ptr<float>(),
                                        stats.data_ptr<float>(), dy.data_ptr<float>(), dxz.data_ptr(), ap + off[4], ap + off[5], stream), "block");
        const at::Tensor p5 = proj.view({B, K, M, H, W}), Bs = p5.narrow(2, R, N), Cs = p5.narrow(2, R + N, N);
        Options o{true, true, SND_DIR_CORNERS, (int)ctx->saved_data["sched"].toInt(), true};
        const Checked c = check_inputs(u, delta, A, Bs, Cs, Dv, dt_bias, OptTensor());
        check_merge(c, true, w, u);
        const int64_t nx = (c.plan.x_elems + 63) / 64 * 64;
        check_elements(state, at::kFloat, u.device(), 2 * nx + c.plan.x_v_elems, "the saved state");
        const float *st = state.data_ptr<float>();
        int64_t wn = 0;
        if (w.has_value()) {
            wn = 1;
            for (int64_t v : ctx->saved_data["mw_shape"].toIntVector()) wn *= v;
        }
        Grads g = launch_bwd(c, u, delta, A, Bs, Cs, Dv, dt_bias, OptTensor(), dy, st, st + 2 * nx, st + nx, o, w, true, wn);
        at::Tensor dproj = at::empty_like(proj);
        check_status(snd_block_dt_bwd(&s, g.ddelta.data_ptr(), g.dB.data_ptr(), g.dC.data_ptr(), wdt.data_ptr<float>(), dproj.data_ptr(), stream), "block");
        check_status(snd_block_wgrad(g.ddelta.data_ptr(), K * Di * HW, Di * HW, proj.data_ptr(), K * M * HW, M * HW, (int)B, (int)K, (int)Di, (int)R, HW, s.dtype,
                                     ap + off[3], stream), "block");
        check_status(snd_block_wgrad(dproj.data_ptr(), K * M * HW, 0, u.data_ptr(), Di * HW, 0, (int)B, 1, (int)(K * M), (int)Di, HW, s.dtype, ap + off[2],
                                     stream), "block");
        const at::Tensor du = at::baddbmm(g.du.view({B, Di, HW}), wxt.expand({B, Di, K * M}), dproj);
        check_elements(du, xz.scalar_type(), xz.device(), B * Di * HW, "du");
        check_status(snd_block_conv_bwd(&s, du.data_ptr(), pre.data_ptr(), xz.data_ptr(), conv_w.data_ptr<float>(), dxz.data_ptr(), ap + off[0],
                                        conv_b.has_value() ? ap + off[1] : nullptr, stream), "block");
        const std::vector<int64_t> types = ctx->saved_data["types"].toIntVector();
        auto part = [&](int i, at::IntArrayRef shape, int type) { return acc.narrow(0, off[i], sizes[i]).view(shape).to((at::ScalarType)types[type]); };
        r[0] = dxz;
        r[1] = part(0, {Di, 1, 3, 3}, 0);
        if (conv_b.has_value()) r[2] = part(1, {Di}, 1);
        r[3] = part(2, {K, M, Di}, 2);
        r[4] = part(3, {K, Di, R}, 3);
        r[5] = g.ddelta_bias.view({K, Di}).to((at::ScalarType)types[4]);
        r[6] = g.dA.mul_(A).to((at::ScalarType)types[5]);
        r[7] = g.dD.to((at::ScalarType)types[6]);
        if (wn > 0) r[8] = g.dweights.view(ctx->saved_data["mw_shape"].toIntVector()).to((at::ScalarType)types[7]);
        r[9] = part(4, {Di}, 8);
        r[10] = part(5, {Di}, 9);
        return r;
    }
};
at::Tensor ss2d(const at::Tensor &xz, const at::Tensor &conv_w, const OptTensor &conv_b, const at::Tensor &wx, const at::Tensor &wdt, const at::Tensor &dt_bias,
                const at::Tensor &A_logs, const at::Tensor &D, const OptTensor &mw, const at::Tensor &gamma, const at::Tensor &beta, double eps) {
    TORCH_CHECK(xz.dim() == 4 && xz.size(3) % 2 == 0, "ss2d: xz must be [batch, rows, cols, 2 * inner]");
    const int64_t Di = xz.size(3) / 2;
    TORCH_CHECK(wx.dim() == 3 && wdt.dim() == 3 && A_logs.dim() == 2, "ss2d: projections are 3-D, A_logs is 2-D");
    const int64_t K = wx.size(0), R = wdt.size(2), N = A_logs.size(1);
    TORCH_CHECK(wx.size(1) == R + 2 * N && wx.size(2) == Di && wdt.size(0) == K && wdt.size(1) == Di && dt_bias.numel() == K * Di && A_logs.size(0) == K * Di &&
                    D.numel() == K * Di && gamma.numel() == Di && beta.numel() == Di && conv_w.sizes() == at::IntArrayRef({Di, 1, 3, 3}) &&
                    (!conv_b.has_value() || conv_b.value().numel() == Di) && (!mw.has_value() || mw.value().sizes() == at::IntArrayRef({K}) || mw.value().sizes() == at::IntArrayRef({K, 1}) ||
                     mw.value().sizes() == at::IntArrayRef({K, Di})),
                "ss2d: parameter shapes do not fit");
    check_device("ss2d", xz, {conv_w, conv_b.value_or(at::Tensor()), wx, wdt, dt_bias, A_logs, D, mw.value_or(at::Tensor()), gamma, beta});
    bool grad = false;
    if (at::GradMode::is_enabled()) {
        for (const at::Tensor *t : {&xz, &conv_w, &wx, &wdt, &dt_bias, &A_logs, &D, &gamma, &beta}) grad = grad || t->requires_grad();
        for (const OptTensor *t : {&conv_b, &mw}) grad = grad || (t->has_value() && t->value().requires_grad());
    }
    return Ss2dFn::apply(xz, conv_w, conv_b, wx, wdt, dt_bias, A_logs, D, mw, gamma, beta, eps, grad);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    // the reference's positional lists (selective_scan_oflex.cpp:179-187,286-297) plus trailing optional
    // arguments: the per-group scan origin the reference leaves as a TODO (fwd.cuh:140), the block mapping
    // of this call (-1: the module default), and the fused CrossMerge (out / dout have dim / n_groups
    // channels, merge_weights [dim] float32 or None for the plain sum; bwd then returns a ninth tensor,
    // merge_weights * d merge_weights per channel)
    namespace py = pybind11;
    m.def("fwd", &selective_scan_fwd, "Selective nd scan forward (gfx950)", py::arg("u"), py::arg("delta"), py::arg("A"),
          py::arg("B"), py::arg("C"), py::arg("D"), py::arg("delta_bias"), py::arg("delta_softplus"), py::arg("out_float"),
          py::arg("A_decay"), py::arg("directions") = 0, py::arg("schedule") = -1, py::arg("merge") = false,
          py::arg("merge_weights") = py::none());
    m.def("bwd", &selective_scan_bwd, "Selective nd scan backward (gfx950)", py::arg("u"), py::arg("delta"), py::arg("A"),
          py::arg("B"), py::arg("C"), py::arg("D"), py::arg("delta_bias"), py::arg("dout"), py::arg("x"), py::arg("x_v"),
          py::arg("delta_softplus"), py::arg("A_decay"), py::arg("x_sd"), py::arg("directions") = 0, py::arg("schedule") = -1,
          py::arg("merge") = false, py::arg("merge_weights") = py::none());
    m.def("scan", &scan, "selective_nd_scan / selective_nd_scan_merged (differentiable)", py::arg("u"), py::arg("delta"), py::arg("A"),
          py::arg("B"), py::arg("C"), py::arg("D"), py::arg("delta_bias"), py::arg("delta_softplus"), py::arg("out_float"),
          py::arg("A_decay"), py::arg("directions"), py::arg("merge"), py::arg("merge_weights"));
    m.def("block_norm", &block_norm, "LayerNorm over the last axis, in the type of `like`", py::arg("x"), py::arg("gamma"), py::arg("beta"), py::arg("eps"), py::arg("like"));
    m.def("block_linear", &block_linear, "A linear layer in the 16-bit type of `like`", py::arg("x"), py::arg("weight"), py::arg("bias"), py::arg("like"));
    m.def("plain", &plain, "Whether kernels may stand in for torch layers on these tensors", py::arg("tensors"));
    m.def("ss2d", &ss2d, "SS2DCrossScan between its in and out projections", py::arg("xz"), py::arg("conv_w"), py::arg("conv_b"), py::arg("x_proj"),
          py::arg("dt_proj"), py::arg("dt_bias"), py::arg("A_logs"), py::arg("D"), py::arg("merge_weights"), py::arg("gamma"), py::arg("beta"), py::arg("eps"));
    m.def("set_schedule", [](int mode) {
        TORCH_CHECK(mode >= SND_SCHED_AUTO && mode <= SND_SCHED_WAVEFRONT, "schedule must be 0 (auto), 1 (plane), 2 (strips), 3 (bands) or 4 (row-segment wavefront)");
        g_schedule.store(mode);
    }, "Default block mapping of calls that pass no schedule: 0 auto, 1 one block per plane chunk, 2 pipelined row strips, 3 bands");
    m.def("get_schedule", [] { return g_schedule.load(); }, "The default block mapping calls use when they name none (see set_schedule)");
    m.def("set_debug", [](bool on) { g_check_pipeline.store(on); },
          "Check the pipelined schedules' error word after every launch (a stream sync per call) and raise if a hand-over wait timed out");
    m.def("init", [](int device) { check_status(snd_init(device), "init"); },
          "Per-device set-up (kernel attributes); call once before capturing launches into a HIP graph");
}
