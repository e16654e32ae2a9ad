// dugks_adjoint.hip -- discrete adjoint of the DUGKS step on MI355X (gfx950), behind the
// dugks_adjoint_* entry points of include/dugks.h.
//
// The fused step engine (dugks_engine.hip) never materialises gbar+, its gradients or the face
// values of a step, and the reverse sweep needs all of them, so the adjoint runs its own FP64 step
// in a plain materialised form: one kernel per phase, one workgroup per cell or face, the lanes
// strided over the velocities and every velocity sum a deterministic workgroup reduction.  The
// per-point work lives in adjoint_core.h and the sweep in adjoint_driver.h; this file supplies the
// HIP backend: device memory, one stream (default priority), HIP events, and the kernel that runs a
// phase over its points.

#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <new>
#include <string>
#include <vector>

#include "../../include/dugks.h"
#include "adjoint_driver.h"
#include "lane_sums.h"

namespace {

constexpr long NT_FILL = 2048;            // half of the device's wave slots at 4 waves a SIMD
constexpr int SUM_MAX = 32;               // widest workgroup reduction of adjoint_core.h
constexpr size_t ROWS_MAX = 32 * 1024;   // LDS for the two rows of a workgroup: 5 of them on a CU

// Executor of adjoint_core.h inside a workgroup of NT lanes; ROWS: its two rows are in LDS.
template <int NT, bool ROWS>
struct GX {
    static constexpr bool local_rows = ROWS;
    double *lds, *rows;

    __host__ __device__ double *row(int i, int nv) { return rows + (size_t)i * nv; }

    template <class F>
    __host__ __device__ void for_k(int nv, F fn)
    {
#if defined(__HIP_DEVICE_COMPILE__)
        for (int k = threadIdx.x; k < nv; k += NT) fn(k);
#else
        (void)nv;
        (void)fn;
#endif
    }

    // Deterministic workgroup sum of v[N], result in every lane: over the lanes of each wavefront,
    // then the wavefront totals added in order.
    template <int N>
    __host__ __device__ void sum(double *v)
    {
        static_assert(N <= SUM_MAX, "reduction width");
#if defined(__HIP_DEVICE_COMPILE__)
        const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
        lane_sums<N>(v, lane);
        const int q = lane_value<N>(lane, 0);
        __syncthreads();
        if (q >= 0) lds[wave * N + q] = v[0];
        __syncthreads();
#pragma unroll
        for (int i = 0; i < N; ++i) {
            double s = 0.0;
#pragma unroll
            for (int w = 0; w < NT / 64; ++w) s += lds[w * N + i];
            v[i] = s;
        }
#else
        (void)v;
#endif
    }

    __host__ __device__ bool leader() const
    {
#if defined(__HIP_DEVICE_COMPILE__)
        return threadIdx.x == 0;
#else
        return true;
#endif
    }
};

// k_face_adj takes 146 registers left alone, 3 waves a SIMD: 323 us for 16000 faces of 32^2 velocities,
// 294 with 4 waves.  The others fit, or spill inside their loops when held to more.
template <class Tag>
constexpr int min_waves()
{
    return std::is_same_v<Tag, adj::k_face_adj> ? 4 : 1;
}

template <class Tag, int NT, bool ROWS, class Fn>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(min_waves<Tag>(), 8))) void k_points(Fn fn)
{
    __shared__ double lds[(NT / 64) * SUM_MAX];
    extern __shared__ __align__(16) double rows[];
    GX<NT, ROWS> x{lds, rows};
    fn(x, (int)blockIdx.x);
}

struct HipBackend {
    int device = 0, nv = 0;   // nv: velocities of a point
    hipStream_t stream = nullptr;
    hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
    bool bad = false;
    std::string msg;
    std::vector<void *> owned;

    bool check(hipError_t e, const char *what)
    {
        if (e != hipSuccess && !bad) {
            bad = true;
            msg = std::string(what) + ": " + hipGetErrorString(e);
        }
        return e == hipSuccess;
    }

    int init(int dev)
    {
        device = dev;
        int n = 0;
        if (hipGetDeviceCount(&n) != hipSuccess || n <= 0) return DUGKS_ERR_DEVICE;
        if (dev < 0 || dev >= n) return DUGKS_ERR_INVALID;
        if (!check(hipSetDevice(dev), "hipSetDevice")) return DUGKS_ERR_DEVICE;
        if (!check(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking), "hipStreamCreate")) return DUGKS_ERR_DEVICE;
        for (auto &e : ev)
            if (!check(hipEventCreate(&e), "hipEventCreate")) return DUGKS_ERR_DEVICE;
        return DUGKS_OK;
    }

    ~HipBackend()
    {
        if (stream) (void)hipStreamSynchronize(stream);
        for (void *p : owned) (void)hipFree(p);
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
        if (stream) (void)hipStreamDestroy(stream);
    }

    template <class T>
    T *alloc(size_t n)
    {
        void *p = nullptr;
        const size_t bytes = std::max<size_t>(n, 1) * sizeof(T);
        if (!check(hipMalloc(&p, bytes), "hipMalloc")) return nullptr;
        owned.push_back(p);
        check(hipMemsetAsync(p, 0, bytes, stream), "hipMemsetAsync");
        return (T *)p;
    }

    void release(void *p)
    {
        check(hipStreamSynchronize(stream), "hipStreamSynchronize");
        for (size_t i = 0; i < owned.size(); ++i)
            if (owned[i] == p) {
                check(hipFree(p), "hipFree");
                owned.erase(owned.begin() + i);
                return;
            }
    }

    void upload(void *d, const void *h, size_t bytes)
    {
        if (bytes) check(hipMemcpyAsync(d, h, bytes, hipMemcpyHostToDevice, stream), "upload");
        check(hipStreamSynchronize(stream), "upload");
    }
    void download(void *h, const void *d, size_t bytes)
    {
        if (bytes) check(hipMemcpyAsync(h, d, bytes, hipMemcpyDeviceToHost, stream), "download");
        check(hipStreamSynchronize(stream), "download");
    }
    void copy(void *d, const void *s, size_t bytes)
    {
        if (bytes) check(hipMemcpyAsync(d, s, bytes, hipMemcpyDeviceToDevice, stream), "copy");
    }
    void zero(void *d, size_t bytes)
    {
        if (bytes) check(hipMemsetAsync(d, 0, bytes, stream), "memset");
    }

    template <class Tag, int NT, class Fn>
    void launch_nt(int n, Fn fn)
    {
        const size_t rows = 2 * (size_t)nv * sizeof(double);
        if constexpr (adj::uses_rows<Tag>::value) {
            if (rows <= ROWS_MAX) {
                hipLaunchKernelGGL((k_points<Tag, NT, true, Fn>), dim3(n), dim3(NT), rows, stream, fn);
                return;
            }
        }
        hipLaunchKernelGGL((k_points<Tag, NT, false, Fn>), dim3(n), dim3(NT), 0, stream, fn);
    }

    template <class Tag, class Fn>
    void launch(int n, Fn fn)
    {
        if (n <= 0 || bad) return;
        // Lanes of a point: 64 up to 128 velocities (50^2 cells of 9^2: 8.5 ms for 60 steps, 9.2 with 128), 128
        // beyond (200 x 40 cells of 32^2: 128 ms, 166 with 64), and more while the points give the
        // device fewer than NT_FILL waves (20^2 cells of 28^2: 14.2 ms with 128, 11.3 with 256)
        int nt = nv <= 128 ? 64 : 128;
        while (nt < 256 && nt < nv && (long)n * (nt / 64) < NT_FILL) nt *= 2;
        if (nt == 64) launch_nt<Tag, 64>(n, fn);
        else if (nt == 128) launch_nt<Tag, 128>(n, fn);
        else launch_nt<Tag, 256>(n, fn);
        check(hipGetLastError(), "kernel launch");
    }

    double free_bytes()
    {
        size_t fr = 0, tot = 0;
        if (hipMemGetInfo(&fr, &tot) != hipSuccess) return 0.0;
        return (double)fr;
    }

    void tic(int i) { check(hipEventRecord(ev[i], stream), "hipEventRecord"); }
    double ms(int a, int b)
    {
        float t = 0.0f;
        if (hipEventElapsedTime(&t, ev[a], ev[b]) != hipSuccess) return 0.0;
        return t;
    }
    void sync() { check(hipStreamSynchronize(stream), "hipStreamSynchronize"); }
    void clear_error()
    {
        (void)hipGetLastError();
        bad = false;
        msg.clear();
    }
};

}  // namespace

struct dugks_adjoint {
    adj::Engine<HipBackend> e;
};

extern "C" {

int dugks_adjoint_create(const dugks_case *cs, dugks_adjoint **out)
{
    if (!out) return DUGKS_ERR_INVALID;
    *out = nullptr;
    if (!cs) return DUGKS_ERR_INVALID;
    dugks_adjoint *a = new (std::nothrow) dugks_adjoint();
    if (!a) return DUGKS_ERR_MEMORY;
    int rc = a->e.be.init(cs->device);
    if (rc != DUGKS_OK) {
        a->e.err = "no usable HIP device: " + a->e.be.msg;
    } else {
        rc = a->e.create(cs);
        a->e.be.nv = a->e.p.nv;
    }
    *out = a;   // returned also on failure so that dugks_adjoint_last_error can explain it
    return rc;
}

int dugks_adjoint_run(dugks_adjoint *a, const double *rho, const double *U, const double *T, double dt,
                      int32_t n_steps, int32_t first_step, int32_t checkpoint_every, const double *face_coef,
                      double *J, double *dJ_dTw)
{
    if (!a) return DUGKS_ERR_INVALID;
    if (a->e.be.bad) return a->e.fail(DUGKS_ERR_DEVICE, "device error: " + a->e.be.msg);
    if (!a->e.p.xi) return a->e.fail(DUGKS_ERR_STATE, "adjoint was not created");
    if (hipSetDevice(a->e.be.device) != hipSuccess) return a->e.fail(DUGKS_ERR_DEVICE, "hipSetDevice failed");
    return a->e.run(rho, U, T, dt, n_steps, first_step, checkpoint_every, face_coef, J, dJ_dTw);
}

int dugks_adjoint_get_macro(dugks_adjoint *a, double *rho, double *U, double *T, double *q)
{
    if (!a) return DUGKS_ERR_INVALID;
    return a->e.macro(rho, U, T, q);
}

int dugks_adjoint_last_ms(dugks_adjoint *a, double *forward_ms, double *reverse_ms)
{
    if (!a) return DUGKS_ERR_INVALID;
    if (!a->e.have_run) return a->e.fail(DUGKS_ERR_STATE, "no run yet");
    if (forward_ms) *forward_ms = a->e.fwd_ms;
    if (reverse_ms) *reverse_ms = a->e.rev_ms;
    return DUGKS_OK;
}

void dugks_adjoint_destroy(dugks_adjoint *a) { delete a; }

const char *dugks_adjoint_last_error(dugks_adjoint *a)
{
    if (!a) return "null adjoint handle";
    return a->e.err.c_str();
}

}  // extern "C"
