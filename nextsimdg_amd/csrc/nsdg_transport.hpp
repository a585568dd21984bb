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
// pinned slots, one filled by the copy engine while a core empties the other. Plain against
// split, into fresh pages (whose faults the threads share): 8 MiB 2.2 -> 1.2 to 1.5 ms, 32 MiB
// 8.9 -> 5.4; into pages in use: 4 MiB 0.23 -> 0.24, 8 MiB 0.47 -> 0.44, 32 MiB 1.8 -> 1.6; the
// first copy of a handle, which pins its slots, into pages in use: 4 MiB 0.27 -> 0.32, 8 MiB
// 0.53 -> 0.54, 16 MiB 1.02 -> 0.93. Below 6 MiB a copy stays with the runtime; two threads take
// it up to 24 MiB and one more for each 8 MiB beyond, so that a copy pays for its slots; eight
// threads copied no faster than four and took twice as long to pin theirs. Slots of 256 KiB:
// 32 MiB 2.4 ms.
// Page-locked and device destinations stay with the runtime (2048 x 2048 cell means 0.6 ms),
// and so do uploads: it reads pageable memory faster (preparing the 512 x 512 box took 15
// ms through the slots, 11 without).
struct HostIO {
    static constexpr size_t kMinSplit = size_t(6) << 20, kSlot = size_t(1) << 19, kShare = size_t(1) << 23;
    static constexpr int kThreads = 4;
    DBuf<double> scratch;
    HostIO() = default;
    HostIO(const HostIO&) = delete;
    HostIO& operator=(const HostIO&) = delete;
    ~HostIO();
    void toHost(void* host, const void* src, size_t bytes, hipStream_t s);

private:
    char* pinned = nullptr; // 2 slots per thread, for `threads` threads
    int threads = 0;
    hipEvent_t done[2 * kThreads] = {};
    void reserve(int n);
    void release();
    void part(char* host, const char* dev, size_t bytes, int t, hipStream_t s);
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
