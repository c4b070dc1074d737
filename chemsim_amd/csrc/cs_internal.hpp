// Internal definitions shared by the translation units of libchemsim_hip.so.
#pragma once

#include <hip/hip_runtime.h>

#include <climits>
#include <cstdint>
#include <cstdio>
#include <cstring>
#include <exception>
#include <memory>
#include <mutex>
#include <vector>
#include <string>

#include "../../include/chemsim.h"

namespace cs {

// ---------------------------------------------------------------- errors --
void set_error(const std::string& msg);
void clear_error();

struct Error {
    int code;
    std::string msg;
};

#define CS_HIP(expr)                                                                        \
    do {                                                                                    \
        hipError_t e_ = (expr);                                                             \
        if (e_ != hipSuccess)                                                               \
            throw ::cs::Error{CS_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_)}; \
    } while (0)

#define CS_REQUIRE(cond, code, msg)                        \
    do {                                                   \
        if (!(cond)) throw ::cs::Error{(code), (msg)};     \
    } while (0)

// Runs f, converting exceptions into a status code + thread-local message.
template <class F>
int guarded(F&& f)
{
    try {
        clear_error();
        f();
        return CS_OK;
    } catch (const Error& e) {
        set_error(e.msg);
        return e.code;
    } catch (const std::bad_alloc&) {
        set_error("host allocation failed");
        return CS_ERR_NOMEM;
    } catch (...) {
        set_error("unknown error");
        return CS_ERR_ARG;
    }
}

// ------------------------------------------------------------- constants --
// D2Q9 directions of lbm.rs:221-231 and the opposite map of lbm.rs:298-309.
constexpr int CX[9] = {0, 1, 0, -1, 0, 1, -1, -1, 1};
constexpr int CY[9] = {0, 0, 1, 0, -1, 1, 1, -1, -1};
constexpr int OPP[9] = {0, 3, 4, 1, 2, 7, 8, 5, 6};

// Per-run constants in the working precision T (float or double):
// K = -dt/tau (lbm.rs:357); A, B, C of compute_equilibrium (lbm.rs:54-66);
// weights (lbm.rs:209-219); Ladd lid terms 6 w_i (c_i . u_lid); deviation
// storage bases w_i * rho0 and rho0; Zou-He boundary values.  Only distinct
// values are stored (three weight classes; the lid terms of directions
// 3, 4, 7, 8 are the negatives of 1, 2, 5, 6), so a kernel keeps them all in
// scalar registers.
template <class T>
struct Consts {
    T K, A, B, C, cs2;
    T wp, wm, hdt;  // TRT: 1/tau_plus, 1/tau_minus, -dt * 0.5 (lbm.rs:431-440)
    T dx, beta;     // KBC: delta_x, 1 / (2 nu / cs^2 + 1) (lbm.rs:478, 547-550)
    T sfq[3];       // Regularized: w / (2 cs^4) of the rest, axis, diagonal classes (lbm.rs:651)
    T wq[3];     // w of the rest, axis and diagonal directions
    T baseq[3];  // w * rho0 of the same classes
    T lidq[4];   // lid term of directions 1, 2, 5, 6
    T in_ux, in_uy, out_rho;
    T rho0;

    __host__ __device__ static constexpr int wclass(int i) { return i == 0 ? 0 : (i < 5 ? 1 : 2); }
    __host__ __device__ T w(int i) const { return wq[wclass(i)]; }
    __host__ __device__ T base(int i) const { return baseq[wclass(i)]; }
    __host__ __device__ T lid(int i) const
    {
        switch (i) {
        case 1: return lidq[0];
        case 2: return lidq[1];
        case 3: return -lidq[0];
        case 4: return -lidq[1];
        case 5: return lidq[2];
        case 6: return lidq[3];
        case 7: return -lidq[2];
        case 8: return -lidq[3];
        default: return T(0);
        }
    }
};

Consts<float> make_consts_f32(const cs_params& p);
Consts<double> make_consts_f64(const cs_params& p);
// Constants of the deviation storages (A, B, C rounded once from f64).
Consts<float> make_consts_dev_f32(const cs_params& p);
bool is_dev_storage(int storage);

// Node info word (one per cell, built on the device from the flags):
//   bits 0..8   source cell of direction i is solid (wall or lid)
//   bits 9..17  source cell of direction i is a moving lid
//   bits 24..27 the cell's own flag
constexpr uint32_t NODE_TYPE_SHIFT = 24;

inline bool is_solid_flag(int t) { return t == CS_WALL || t == CS_LID; }

size_t storage_bytes(int storage);

// Device staging of the moment calls' result planes, kept from call to call
// (hipMalloc and hipFree of a 2 MB buffer take about as long as copying it to the
// host, and hipFree waits for the whole device): as many buffers as calls run at
// once, of at most STAGING_KEEP bytes together, shared by the handles of a
// context and freed with the last of them -- one buffer per handle would hold 12
// to 24 bytes per cell of every lattice that was ever read.  What does not fit is
// allocated for the call.  Eight threads that each read the velocity of their own
// 512^2 lattice: 400 us per call of all of them, 905 with one buffer for the
// context, 1075 with an allocation per call.
constexpr size_t STAGING_KEEP = (size_t)64 << 20;
class KeptStaging {
public:
    struct Buf {
        void* p = nullptr;
        size_t bytes = 0;
    };
    KeptStaging() { idle_.reserve(MOST); }
    KeptStaging(const KeptStaging&) = delete;
    KeptStaging& operator=(const KeptStaging&) = delete;
    ~KeptStaging()
    {
        for (const Buf& b : idle_) (void)hipFree(b.p);
    }
    // A buffer of at least `bytes` for the caller alone; null if none may be kept for it.
    Buf take(size_t bytes)
    {
        std::vector<Buf> drop;
        {
            std::lock_guard<std::mutex> lk(mu_);
            auto fit = idle_.end(), big = idle_.end();
            for (auto i = idle_.begin(); i != idle_.end(); ++i) {
                if (i->bytes >= bytes && (fit == idle_.end() || i->bytes < fit->bytes)) fit = i;
                if (big == idle_.end() || i->bytes > big->bytes) big = i;
            }
            if (fit != idle_.end()) {
                const Buf b = *fit;
                idle_.erase(fit);
                return b;
            }
            if (bytes > STAGING_KEEP) return Buf{};
            // grow the largest idle one, and drop others while the rest is too much
            while (big != idle_.end()) {
                drop.push_back(*big);
                kept_ -= big->bytes;
                --count_;
                idle_.erase(big);
                big = kept_ + bytes > STAGING_KEEP ? idle_.begin() : idle_.end();
            }
            if (kept_ + bytes > STAGING_KEEP || count_ == MOST) bytes = 0;
            else {
                kept_ += bytes;
                ++count_;
            }
        }
        for (const Buf& b : drop) (void)hipFree(b.p);
        Buf b;
        if (bytes == 0) return b;
        const hipError_t e = hipMalloc(&b.p, bytes);
        if (e != hipSuccess) {
            std::lock_guard<std::mutex> lk(mu_);
            kept_ -= bytes;
            --count_;
            CS_HIP(e);
        }
        b.bytes = bytes;
        return b;
    }
    void give(const Buf& b)
    {
        std::lock_guard<std::mutex> lk(mu_);
        idle_.push_back(b);  // within the reserve: count_ <= MOST
    }

private:
    static constexpr int MOST = 64;
    std::mutex mu_;
    std::vector<Buf> idle_;
    size_t kept_ = 0;  // bytes of the idle buffers and of those in use
    int count_ = 0;    // their number
};
class Staging {
public:
    // For work on `stream`, which is waited for before the buffer is given back.
    Staging(KeptStaging& kept, size_t bytes, hipStream_t stream) : kept_(kept), stream_(stream), buf_(kept.take(bytes))
    {
        if (!buf_.p) CS_HIP(hipMalloc(&own_, bytes));
    }
    ~Staging()
    {
        if (std::uncaught_exceptions() > 0) (void)hipStreamSynchronize(stream_);  // else its user has waited
        if (own_) (void)hipFree(own_);
        if (buf_.p) kept_.give(buf_);
    }
    Staging(const Staging&) = delete;
    Staging& operator=(const Staging&) = delete;
    void* get() const { return own_ ? own_ : buf_.p; }

private:
    KeptStaging& kept_;
    hipStream_t stream_;
    KeptStaging::Buf buf_;
    void* own_ = nullptr;
};

// Copies the device planes src, src + n, ... to the caller's arrays and waits.
// Small planes come over in one copy into host scratch: a pageable copy waits
// for its own end, so three of them take three latencies.  moments_f64 of a
// 16^2 lattice 50 -> 28 us, velocity of 128^2 (128 KiB) 37 -> 30 us; 180^2
// (760 KiB) 72 -> 68 us; from 1 MiB on the second copy on the host costs more
// than it saves (velocity of 360^2 75 us plane by plane, 83 us together).
constexpr size_t PLANES_TOGETHER = (size_t)768 << 10;
template <class Out>
inline void planes_to_host(const Out* src, int64_t n, Out* const* outs, int count, hipStream_t stream)
{
    const size_t plane = sizeof(Out) * (size_t)n;
    if (count > 1 && plane * (size_t)count <= PLANES_TOGETHER) {
        const std::unique_ptr<Out[]> tmp(new Out[(size_t)n * (size_t)count]);
        CS_HIP(hipMemcpyAsync(tmp.get(), src, plane * (size_t)count, hipMemcpyDeviceToHost, stream));
        CS_HIP(hipStreamSynchronize(stream));
        for (int j = 0; j < count; ++j) std::memcpy(outs[j], tmp.get() + j * n, plane);
        return;
    }
    for (int j = 0; j < count; ++j)
        CS_HIP(hipMemcpyAsync(outs[j], src + j * n, plane, hipMemcpyDeviceToHost, stream));
    CS_HIP(hipStreamSynchronize(stream));
}

}  // namespace cs

struct cs_lattice;
namespace cs {
// n fused steps on the lattice's stream (cs_lattice_step without the checks).
void do_steps(cs_lattice* l, int n);
// Temporally blocked steps (lattice_tb.hip): the plan this lattice takes --
// steps per launch K in the low byte (tb_plan_steps), the region side above
// it (0: one-step kernels; cpt_override: the cs_set_cells_per_thread value)
// -- and one launch of that plan (advances cur, steps and time by K).
int tb_steps(const cs_lattice* l, int cpt_override);
inline int tb_plan_steps(int plan) { return plan & 0xFF; }
// The plan of 4 steps per launch for the remainder of a run of 8-step launches
// (BGK lattices; 0 when there is none).
int tb_remainder_plan(const cs_lattice* l, int plan);
void launch_tb(cs_lattice* l, int plan);
// The streaming variant of the temporally blocked step (lattice_ts.hip):
// whether this lattice takes it, whether its 4-step remainder does too, and one
// launch of k (8 or 4) steps.
bool ts_takes(const cs_lattice* l);
bool ts_takes_remainder(const cs_lattice* l);
void launch_ts(cs_lattice* l, int k);
// The render passes of the current populations into d_out (device, h*w pixels
// of `channels` bytes: 3 = RGB, 4 = RGBA with alpha 255), enqueued on the
// lattice's stream; allocates the lattice's render scratch on first use.
void render_enqueue(cs_lattice* l, int mode, int overlay, uint8_t* d_out, int channels);
}  // namespace cs

// ----------------------------------------------------------------- handles --
struct cs_ctx {
    int device = 0;
    hipDeviceProp_t prop{};
    std::mutex staging_mu;
    std::weak_ptr<cs::KeptStaging> staging_now;
    // The staging of this context's handles: made for the first, freed with the last.
    std::shared_ptr<cs::KeptStaging> staging()
    {
        std::lock_guard<std::mutex> lk(staging_mu);
        auto s = staging_now.lock();
        if (!s) staging_now = s = std::make_shared<cs::KeptStaging>();
        return s;
    }
};

struct cs_lattice {
    cs_ctx* ctx = nullptr;      // may be gone while the lattice steps: the kernel choice reads cus
    int cus = 0;                // the device's compute units
    int w = 0, h = 0, storage = CS_F32;
    // Populations are row-interleaved: row r holds planes 0..8 of that row
    // one after another, so element (i, r, c) is at i * plane + r * pitch + c
    // with plane = the padded row length and pitch = 9 * plane.  A thread
    // block then reads and writes a few contiguous row groups instead of
    // 9 streams 1/9 of the buffer apart.
    int pitch = 0;          // population row stride, elements
    int64_t plane = 0;      // population plane stride, elements
    int cpitch = 0;         // row pitch of the per-cell arrays (flags, node), elements
    void* buf[2] = {nullptr, nullptr};
    int cur = 0;            // buf[cur] holds the current populations
    uint8_t* flags = nullptr;   // h*pitch flags (device) or null
    uint32_t* node = nullptr;   // h*pitch node info (device) or null
    bool has_flags = false;
    bool has_io = false;        // the flags hold an inlet or outlet cell
    cs_params params{};
    cs::Consts<float> k32{};
    cs::Consts<double> k64{};
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    float* snap = nullptr;      // 2 planes (ux, uy) of h*pitch
    bool has_snap = false;
    double* partials = nullptr; // reduction partials
    int npartials = 0;
    double* dscratch = nullptr; // small device scratch for reduction results
    int* iscratch = nullptr;
    double time = 0.0;
    uint64_t steps = 0;         // fused steps taken (keys the stochastic rounding)
    std::shared_ptr<cs::KeptStaging> staging;  // the context's: result planes of the moment calls
    void* render_buf = nullptr; // render pass scratch (fields, partials, RGB)
    // Launch-bound lattices replay captured runs of fused steps: one graph per
    // starting buffer parity, valid for the parameters, geometry and launch
    // shape they were captured with (cleared when any of them changes).
    hipGraphExec_t step_graph[2] = {nullptr, nullptr};
    int graph_cpt = INT_MIN;    // cells-per-thread override at capture (INT_MIN: none captured)
    int graph_tb = 0;           // temporally blocked plan (tb_steps) at capture
};
