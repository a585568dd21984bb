// DG transport on the device: DGTransport<DG> (dynamics/src/include/DGTransport.hpp:27-152,
// dynamics/src/DGTransport.cpp) and the CG -> DG projection it is fed with
// (Interpolations::CG2DG, dynamics/src/Interpolations.cpp:74-122).
#pragma once
#include "nsdg_internal.hpp"

namespace nsdg {

// LimitMax(field, maxv) and LimitMin(field, minv) (dgLimit.hpp:16-84), in that order.
struct Limits {
    bool doMax = false, doMin = false;
    double maxv = 0, minv = 0;
    static Limits max(double v) { return { true, false, v, 0 }; }
    static Limits min(double v) { return { false, true, 0, v }; }
    static Limits both(double hi, double lo) { return { true, true, hi, lo }; }
};

// Runtime-degree interface over TransportImpl<DG>.
struct TransportBase {
    virtual ~TransportBase() = default;
    virtual int dg() const = 0;
    virtual void setScheme(int rk) = 0;
    virtual void setVelocityHost(const double* vx, const double* vy) = 0; // N_e x DG host layout
    virtual void prepareAdvectionHost(int cg, const double* u, const double* v) = 0;
    virtual void reinitNormalVelocity() = 0;
    // SoA field on the device; tally (optional, N_e doubles) accumulates each element's
    // Dirichlet outflow in Tools::MeanValue units; lim is applied to the new field
    virtual void step(double dt, double* phiDev, double* tally = nullptr, const Limits& lim = {}) = 0;
    // tally (optional) accumulates the change of each element's MeanValue contribution
    virtual void limit(double* phiDev, const Limits& lim, double* tally = nullptr) = 0;
    virtual double* velx() = 0;
    virtual double* vely() = 0;
};

// Copies from the device to host memory, done when the call returns, and the device scratch
// of the layout conversion. Of one handle, so used by one thread at a time.
// The runtime copies into pageable memory through its own staging, one chunk and one core
// at a time. From kMinSplit bytes up the range is split over a few threads, each with two
// pinned slots: a kernel stores into one while a core empties the other. (Copies into the
// slots by the copy engine fell to 4.7 GB/s for hundreds of copies at a time in processes with
// several handles: 67 MB in 14.3 ms, by the runtime 6.3, by the kernel 2.3.)
// Plain against split, into fresh pages (whose faults the threads share): 8 MiB 2.2 -> 2.0 ms,
// 16 MiB 4.5 -> 3.8, 32 MiB 8.9 -> 5.6; into pages in use: 8 MiB 0.47 -> 0.36, 32 MiB 1.85 -> 0.97;
// the first copy of a handle, which pins its slots, into pages in use: 8 MiB 0.53 -> 0.46, 16
// MiB 1.02 -> 0.67; a new transport handle with one step at 512 x 512 (13 MB) 5.24 -> 5.11. Below
// 6 MiB a copy stays with the runtime (4 MiB 0.23 ms, through slots 0.24 to 0.26 and 0.32 the
// first time); two threads take it up to 24 MiB and one more for each 8 MiB beyond, so that a
// copy pays for its slots.
// Page-locked and device destinations stay with the runtime (2048 x 2048 cell means 0.6 ms),
// and so do uploads: it reads pageable memory faster (preparing the 512 x 512 box took 15
// ms through the slots, 11 without).
struct HostIO {
    static constexpr size_t kMinSplit = size_t(6) << 20, kShare = size_t(1) << 23; // bytes
    static constexpr size_t kSlot = size_t(1) << 16;                            // values
    static constexpr int kThreads = 4;
    DBuf<double> scratch;
    HostIO() = default;
    HostIO(const HostIO&) = delete;
    HostIO& operator=(const HostIO&) = delete;
    ~HostIO();
    void toHost(double* host, const double* dev, size_t values, hipStream_t s);

private:
    double* pinned = nullptr; // 2 slots per thread, for `threads` threads
    int threads = 0;
    hipEvent_t done[2 * kThreads] = {};
    void reserve(int n);
    void release();
    void part(double* host, const double* dev, size_t values, int t, hipStream_t s);
};

// Owning wrapper used by the C ABI (mesh + transport + stream).
struct TransportHandle {
    hipStream_t stream = nullptr;
    Profiler prof;
    DeviceMesh mesh;
    std::unique_ptr<TransportBase> t;
    DBuf<double> field;
    HostIO io;
    ~TransportHandle();
};

std::unique_ptr<TransportBase> makeTransport(int dg, DeviceMesh& mesh, hipStream_t s, Profiler& p);

// CG -> DG projection operators and launch (u, v to the advection velocity, output fields).
struct CG2DGOps {
    int cg = 0, dg = 0;
    DBuf<double> ops;
    void build(int cg, int dg, const DeviceMesh& mesh, hipStream_t s);
    // dst: SoA DG x ne; src: CG node vector. Two fields at once when src2/dst2 are set.
    void apply(const DeviceMesh& mesh, const double* src, double* dst, const double* src2, double* dst2,
        hipStream_t s, Profiler& p) const;
};

// Host <-> device layout conversion (ModelArray N x ncomp <-> SoA ncomp x N).
void uploadSoA(HostIO& io, const double* host, size_t n, int ncomp, double* dst, hipStream_t s);
void downloadSoA(HostIO& io, const double* src, size_t n, int ncomp, double* host, hipStream_t s);
void deviceFill(double* p, size_t n, double v, hipStream_t s);
void deviceCopy(double* dst, const double* src, size_t n, hipStream_t s);

} // namespace nsdg
