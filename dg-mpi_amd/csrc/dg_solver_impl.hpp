// The solver handle behind the C ABI (shared by the host files of the
// library).
#pragma once

#include <hip/hip_runtime.h>

#include <mutex>
#include <string>
#include <vector>

#include "dg_config.hpp"
#include "dg_kernels.hpp"

namespace dg {

// hipMalloc on the current device.  When the device is full, the two-pass
// stage's scratch arrays on it are taken back first (their owners run the
// fused stage from then on): no allocation of the library is refused for them.
hipError_t device_malloc(void** p, size_t bytes);
template <class T>
hipError_t device_malloc(T** p, size_t bytes) {
    return device_malloc(reinterpret_cast<void**>(p), bytes);
}

// Scratch of the two-pass stage, which its owner can do without.  mu is held
// from the look at p until the launches that use it are on the stream (by a
// batch until they are done): device_malloc of any thread may free it.
struct Scratch {
    void* p = nullptr;
    int device = 0;
    std::mutex mu;
    // allocates it on the current device, where that leaves as much free as
    // `arrays`, the bytes of the arrays it serves: the caller's own states of
    // the case, or a second handle for it, then still fit
    void take(size_t bytes, size_t arrays);
    void drop();
    ~Scratch() { drop(); }
};

}  // namespace dg

struct dg_solver {
    dg::CaseConfig cfg;
    dg::KTables tab;
    dg::KGeom geo;
    dg::KIC ic;
    int P = 0;
    int ns = 5;                        // state variables: dim + 2
    size_t ncoef = 0;                  // E * nb * ns
    double dt = 0.0;                   // case time step (0 until known)
    double time = 0.0;
    int device = 0;
    hipStream_t stream = nullptr;      // stream the handle launches on
    hipStream_t own_stream = nullptr;  // stream created by dg_create
    double* U0 = nullptr;              // solution (Solver::Uc)
    double* Ua = nullptr;              // stage states
    double* Ub = nullptr;
    double* acc = nullptr;             // RK accumulator
    float* cmp = nullptr;              // Stepper.compensated: rounding error of U0 (FP32)
    dg::Scratch faces;                 // lifted fluxes of the two-pass stage (null: the fused stage)
    double* work = nullptr;            // per-element reduction output
    double* X = nullptr;               // mapped box: element node coordinates [E][8][3]
    double* imm = nullptr;             // mapped box: inverse mass matrices [E][nb][nb]
    unsigned* frec = nullptr;          // general path: face records [E][6][2]
    double* nev = nullptr;             // general path: normal evaluation points
    dg::KTables* dtab = nullptr;       // device copy of tab
    // learned-closure stepping (dg_closure_step):
    // corrections [E][40] and the fallback counter, allocated on first use
    float* cl_C = nullptr;
    unsigned long long* cl_cnt = nullptr;
    std::vector<double> mesh_xyz;      // given mesh: node coordinates [n][dim]
    std::vector<long> mesh_e2n;        // given mesh: element nodes [E][8] (2D: [E][4])
    std::string err;
};

// A stage or the residual of the handle's case; corr: the closure's
// correction or null.  The two passes share the handle's scratch array: its
// users are ordered by the handle's stream, each pair of launches enqueued
// under the lock.  A residual on a stream of the caller's, or captured into
// a graph that may be replayed on any stream, takes the fused kernel, which
// needs no scratch.
inline hipError_t launch_solver_stage(dg_solver* s, const dg::StageArgs& a, const float* corr, hipStream_t st) {
    const int flux = (int)s->cfg.flux;
    std::unique_lock<std::mutex> lk(s->faces.mu);
    if (s->faces.p) {
        hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
        if (a.mode != dg::MODE_RESIDUAL
                ? dg::two_pass_steps(s->P, s->geo, s->geo.E)
                : st == s->stream && hipStreamIsCapturing(st, &cap) == hipSuccess && cap == hipStreamCaptureStatusNone)
            return dg::launch_stage_two_pass(s->P, flux, a, s->faces.p, corr, s->dtab, s->geo, st);
    }
    lk.unlock();
    if (corr) return dg::launch_stage_corrected(s->P, flux, a, corr, s->dtab, s->geo, st);
    return dg::launch_stage(s->P, flux, a, s->dtab, s->geo, st);
}
