/*
 * Host side of the Newton initial-guess network: parameter storage (FP32
 * master weights + BF16 copies on the device), forward pass, and one
 * training step (MSE loss, backward through the three SiLU layers, Adam).
 * The input layer is 32 wide on the device: 16 features and 16 zero
 * columns, so every matrix-core tile is full.
 */
#include <algorithm>
#include <cmath>
#include <cstring>
#include <mutex>
#include <random>
#include <vector>
#include "ngmi_internal.h"
#include "mlp_types.h"

namespace ngmi {
int launch_gemm_bf16(const unsigned short *A, const unsigned short *B, const float *bias, unsigned short *Cb, int M,
                     int N, int K, hipStream_t s, const int *Mdev);
__global__ void k_f32_to_bf16(const float *x, unsigned short *y, int64_t n);
__global__ void k_train_transpose(const unsigned short *wb, unsigned short *wbt);
int launch_train_step(const TrainBufs &B, const float *X, const float *target, int M, const AdamStep &A, hipStream_t s);
__global__ void k_head(const unsigned short *H, const unsigned short *w, const float *b, float *y, int M, int K,
                       const int *Mdev);
int launch_guess_net(const unsigned short *wb, const float *wf, const float *X, int *count, int maxRows,
                     const int64_t *dest, const double2 *base, double *x, float *yout,
                     unsigned long long *rows_total, hipStream_t s);
}  // namespace ngmi

using namespace ngmi;

namespace {
constexpr int IN_PAD = MLP_IN_PAD;
constexpr int H = MLP_HID;
constexpr int64_t OFF_W1 = MLP_OFF_W1, OFF_B1 = MLP_OFF_B1, OFF_W2 = MLP_OFF_W2, OFF_B2 = MLP_OFF_B2,
                  OFF_W3 = MLP_OFF_W3, OFF_B3 = MLP_OFF_B3, OFF_W4 = MLP_OFF_W4, OFF_B4 = MLP_OFF_B4,
                  NPARAM = MLP_NPARAM;

/* work buffers of the layer-by-layer inference: packed input and two
 * activation buffers (ping-pong), BF16 */
struct InferBufs {
    int cap = 0;   /* rows */
    unsigned short *xb = nullptr, *a = nullptr, *b = nullptr;
    ~InferBufs() { release(); }
    void release()
    {
        for (unsigned short **p : {&xb, &a, &b}) {
            (void)hipFree(*p);
            *p = nullptr;
        }
        cap = 0;
    }
    int ensure(int rows)
    {
        if (rows <= cap) return NGMI_OK;
        release();
        NGMI_HIP(hipMalloc(&xb, (size_t)rows * IN_PAD * 2));
        NGMI_HIP(hipMalloc(&a, (size_t)rows * H * 2));
        NGMI_HIP(hipMalloc(&b, (size_t)rows * H * 2));
        cap = rows;
        return NGMI_OK;
    }
};
}  // namespace

struct ngmi_mlp {
    float *w = nullptr, *g = nullptr, *m = nullptr, *v = nullptr;   /* NPARAM each */
    unsigned short *wb = nullptr, *wbt = nullptr;                   /* BF16 copy; W2, W3 transposed */
    int cap = 0;                                                    /* training rows allocated */
    unsigned short *xo = nullptr, *h1 = nullptr, *h2 = nullptr, *h3 = nullptr;
    unsigned short *dz1 = nullptr, *dz2 = nullptr, *dz3 = nullptr;
    float *df1 = nullptr, *df2 = nullptr, *df3 = nullptr, *y = nullptr, *dy = nullptr, *cols = nullptr;
    int64_t step = 0;
    /* ngmi_mlp_forward's and the transient's: a transient keeps the pointers
     * in its captured passes, and may run beside a forward call */
    InferBufs fwd, guess;
    ~ngmi_mlp()
    {
        void *ps[] = {w, g, m, v, wb, wbt, xo, h1, h2, h3, dz1, dz2, dz3, df1, df2, df3, y, dy, cols};
        for (void *p : ps) (void)hipFree(p);
    }
    int ensure(int rows)   /* a multiple of 32 */
    {
        if (rows <= cap) return NGMI_OK;
        cap = 0;
        void **ps[] = {(void **)&xo, (void **)&h1, (void **)&h2, (void **)&h3, (void **)&dz1, (void **)&dz2,
                       (void **)&dz3, (void **)&df1, (void **)&df2, (void **)&df3, (void **)&y, (void **)&dy,
                       (void **)&cols};
        const size_t r = (size_t)rows, hb = r * H * 2, hf = r * H * 4;
        const size_t bytes[] = {r * IN_PAD * 2, hb, hb, hb, hb, hb, hb, hf, hf, hf, r * 4, r * 4,
                                (size_t)TR_PARTS * TR_PART * 4};
        for (void **p : ps) {
            (void)hipFree(*p);
            *p = nullptr;
        }
        for (size_t i = 0; i < sizeof(ps) / sizeof(*ps); i++) NGMI_HIP(hipMalloc(ps[i], bytes[i]));
        cap = rows;
        return NGMI_OK;
    }
};

namespace {

int blocks(int64_t n) { return (int)((n + 255) / 256); }

/* X (device fp32, M x 16, row-major) -> padded BF16 input rows */
__global__ void k_pack_input(const float *__restrict__ X, unsigned short *__restrict__ xb, int M,
                             int Mpad, const int *__restrict__ Mdev = nullptr)
{
    if (Mdev) {
        M = min(M, *Mdev);
        Mpad = min(Mpad, (M + 31) / 32 * 32);
    }
    const int64_t n = (int64_t)Mpad * IN_PAD;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (int64_t)gridDim.x * blockDim.x) {
        const int r = (int)(i / IN_PAD), c = (int)(i % IN_PAD);
        xb[i] = f2bf((r < M && c < MLP_IN) ? X[(int64_t)r * MLP_IN + c] : 0.0f);
    }
}

/* the BF16 copies of the master weights */
int refresh_bf16(ngmi_mlp *n)
{
    hipLaunchKernelGGL(k_f32_to_bf16, dim3(blocks(NPARAM)), dim3(256), 0, 0, n->w, n->wb, (int64_t)NPARAM);
    NGMI_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_train_transpose, dim3(H), dim3(H), 0, 0, n->wb, n->wbt);
    NGMI_HIP(hipGetLastError());
    NGMI_HIP(hipDeviceSynchronize());
    return NGMI_OK;
}

}  // namespace

namespace {
/* inference over at most maxRows rows (the first *dcount when dcount is
 * set) with caller-provided work buffers: xb (Mpad x 32 BF16 input rows),
 * ia and ib (Mpad x 256 BF16 activations, ping-pong) */
int forward_infer(const ngmi_mlp *n, const float *X, float *y, int maxRows, int Mpad, unsigned short *xb,
                  unsigned short *ia, unsigned short *ib, const int *dcount, hipStream_t s)
{
    int rc;
    hipLaunchKernelGGL(k_pack_input, dim3(std::min(blocks((int64_t)Mpad * IN_PAD), 2048)), dim3(256), 0, s,
                       X, xb, maxRows, Mpad, dcount);
    NGMI_HIP(hipGetLastError());
    const unsigned short *wb = n->wb;
    if ((rc = launch_gemm_bf16(xb, wb + OFF_W1, n->w + OFF_B1, ia, Mpad, H, IN_PAD, s, dcount))) return rc;
    if ((rc = launch_gemm_bf16(ia, wb + OFF_W2, n->w + OFF_B2, ib, Mpad, H, H, s, dcount))) return rc;
    if ((rc = launch_gemm_bf16(ib, wb + OFF_W3, n->w + OFF_B3, ia, Mpad, H, H, s, dcount))) return rc;
    hipLaunchKernelGGL(k_head, dim3(std::min(blocks(maxRows), 1024)), dim3(256), 0, s, ia, wb + OFF_W4,
                       n->w + OFF_B4, y, maxRows, H, dcount);
    NGMI_HIP(hipGetLastError());
    return NGMI_OK;
}

/* Work memory of ngmi_mlp_forward_noalloc: NGMI_MLP_NOALLOC_MAX_ROWS rows of
 * packed BF16 input (32 wide) and two BF16 activation buffers (256 wide),
 * 17 MB, in device memory of every GPU the library runs on until the
 * process ends.  Host code addresses it only through the pointer
 * hipGetSymbolAddress returns for the current device. */
constexpr int64_t NOALLOC_XB = (int64_t)NGMI_MLP_NOALLOC_MAX_ROWS * IN_PAD;
constexpr int64_t NOALLOC_ACT = (int64_t)NGMI_MLP_NOALLOC_MAX_ROWS * H;
}  // namespace

static __device__ __align__(256) unsigned short scratch[NOALLOC_XB + 2 * NOALLOC_ACT];

namespace {
constexpr int MAX_DEVICES = 64;
std::mutex scratch_mu;
unsigned short *scratch_ptr[MAX_DEVICES] = {};

/* the device address of this device's scratch, looked up once per device */
int scratch_for_current_device(unsigned short **out)
{
    int dev = 0;
    NGMI_HIP(hipGetDevice(&dev));
    if (dev < 0 || dev >= MAX_DEVICES) {
        set_error("mlp_forward_noalloc: device %d beyond the %d the library tracks", dev, MAX_DEVICES);
        return NGMI_E_DEVICE;
    }
    std::lock_guard<std::mutex> lk(scratch_mu);
    if (!scratch_ptr[dev]) {
        void *p = nullptr;
        const hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !p) {
            set_error("mlp_forward_noalloc: hipGetSymbolAddress failed: %s", hipGetErrorString(e));
            return NGMI_E_DEVICE;
        }
        scratch_ptr[dev] = (unsigned short *)p;
    }
    *out = scratch_ptr[dev];
    return NGMI_OK;
}
}  // namespace

namespace ngmi {
/* forward over the first *dcount of at most maxRows rows (device-side count) */
int mlp_forward_rows(ngmi_mlp *n, const float *X, float *y, int maxRows, const int *dcount,
                     hipStream_t s)
{
    const int Mpad = (maxRows + 31) / 32 * 32;
    int rc = n->guess.ensure(Mpad);
    if (rc) return rc;
    return forward_infer(n, X, y, maxRows, Mpad, n->guess.xb, n->guess.a, n->guess.b, dcount, s);
}

/* the fused inference of the transient's guess pass: rows from count[0]
 * (cleared, with the finish counter count[1], by the kernel) */
int mlp_guess_rows(const ngmi_mlp *n, const float *X, int *count, int maxRows, const int64_t *dest,
                   const double2 *base, double *x, float *yout, unsigned long long *rows_total, hipStream_t s)
{
    return launch_guess_net(n->wb, n->w, X, count, maxRows, dest, base, x, yout, rows_total, s);
}
}  // namespace ngmi

extern "C" {

ngmi_mlp *ngmi_mlp_new(unsigned long long seed)
{
    ngmi_mlp *n = new ngmi_mlp;
    std::vector<float> w(NPARAM, 0.0f);
    std::mt19937_64 g(seed);
    auto init = [&](int64_t off, int fan_out, int fan_in, int used_in) {
        const double lim = std::sqrt(6.0 / (fan_in + fan_out));
        std::uniform_real_distribution<double> u(-lim, lim);
        for (int o = 0; o < fan_out; o++)
            for (int i = 0; i < fan_in; i++)
                w[off + (int64_t)o * fan_in + i] = i < used_in ? (float)u(g) : 0.0f;
    };
    init(OFF_W1, H, IN_PAD, MLP_IN);
    init(OFF_W2, H, H, H);
    init(OFF_W3, H, H, H);
    {
        std::uniform_real_distribution<double> u(-1e-3, 1e-3);
        for (int k = 0; k < H; k++) w[OFF_W4 + k] = (float)u(g);
    }
    if (hipMalloc(&n->w, NPARAM * 4) != hipSuccess || hipMalloc(&n->g, NPARAM * 4) != hipSuccess ||
        hipMalloc(&n->m, NPARAM * 4) != hipSuccess || hipMalloc(&n->v, NPARAM * 4) != hipSuccess ||
        hipMalloc(&n->wb, NPARAM * 2) != hipSuccess || hipMalloc(&n->wbt, 2 * MLP_SZ_W2 * 2) != hipSuccess ||
        hipMemcpy(n->w, w.data(), NPARAM * 4, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(n->m, 0, NPARAM * 4) != hipSuccess || hipMemset(n->v, 0, NPARAM * 4) != hipSuccess ||
        hipMemset(n->g, 0, NPARAM * 4) != hipSuccess) {
        set_error("ngmi_mlp_new: device allocation failed");
        delete n;
        return nullptr;
    }
    if (refresh_bf16(n)) {
        delete n;
        return nullptr;
    }
    return n;
}

void ngmi_mlp_free(ngmi_mlp *n) { delete n; }

int64_t ngmi_mlp_num_params(void) { return NPARAM; }

int ngmi_mlp_get_params(const ngmi_mlp *n, float *host, int grads)
{
    if (!n || !host) return NGMI_E_PANIC;
    NGMI_HIP(hipMemcpy(host, grads ? n->g : n->w, NPARAM * 4, hipMemcpyDeviceToHost));
    return NGMI_OK;
}

int ngmi_mlp_set_params(ngmi_mlp *n, const float *host)
{
    if (!n || !host) return NGMI_E_PANIC;
    NGMI_HIP(hipMemcpy(n->w, host, NPARAM * 4, hipMemcpyHostToDevice));
    return refresh_bf16(n);
}

/* y[M] = network(X[M x 16]); device pointers */
int ngmi_mlp_forward(ngmi_mlp *n, const float *X, float *y, int M, void *stream)
{
    if (!n || M < 0) return NGMI_E_PANIC;
    if (M == 0) return NGMI_OK;
    const hipStream_t s = (hipStream_t)stream;
    if (tune_get(TUNE_GUESS_FUSED))
        return launch_guess_net(n->wb, n->w, X, nullptr, M, nullptr, nullptr, nullptr, y, nullptr, s);
    const int Mpad = (M + 31) / 32 * 32;
    const int rc = n->fwd.ensure(Mpad);
    if (rc) return rc;
    return forward_infer(n, X, y, M, Mpad, n->fwd.xb, n->fwd.a, n->fwd.b, nullptr, s);
}

/* ngmi_mlp_forward without allocating: the work buffers are the library's
 * fixed per-device scratch, so calls that overlap on one GPU race */
int ngmi_mlp_forward_noalloc(const ngmi_mlp *n, const float *X, float *y, int M, void *stream)
{
    if (!n || M < 0 || (M > 0 && (!X || !y))) {
        set_error("mlp_forward_noalloc: bad arguments");
        return NGMI_E_PANIC;
    }
    if (M > NGMI_MLP_NOALLOC_MAX_ROWS) {
        set_error("mlp_forward_noalloc: %d rows exceed the scratch maximum of %d", M, NGMI_MLP_NOALLOC_MAX_ROWS);
        return NGMI_E_PARMVAL;
    }
    if (M == 0) return NGMI_OK;
    unsigned short *base = nullptr;
    int rc = scratch_for_current_device(&base);
    if (rc) return rc;
    const int Mpad = (M + 31) / 32 * 32;
    return forward_infer(n, X, y, M, Mpad, base, base + NOALLOC_XB, base + NOALLOC_XB + NOALLOC_ACT, nullptr,
                         (hipStream_t)stream);
}

/* gradients of the mean squared error over M samples into the gradient
 * buffer; with lr > 0 also one Adam step (beta 0.9 / 0.999, eps 1e-8) */
int ngmi_mlp_train_step(ngmi_mlp *n, const float *X, const float *target, int M, float lr,
                        float *loss_host, void *stream)
{
    if (!n || M <= 0) return NGMI_E_PANIC;
    const hipStream_t s = (hipStream_t)stream;
    const int Mpad = (M + 31) / 32 * 32;
    int rc = n->ensure(Mpad);
    if (rc) return rc;
    AdamStep A{lr, 0.9f, 0.999f, 1e-8f, 1.0f, 1.0f};
    if (lr > 0) {
        n->step++;
        A.c1 = 1.0f - std::pow(A.b1, (float)n->step);
        A.c2 = 1.0f - std::pow(A.b2, (float)n->step);
    }
    const TrainBufs B{n->w,  n->g,  n->m,   n->v,   n->wb,  n->wbt, n->y,   n->dy,  n->xo,  n->h1,
                      n->h2, n->dz1, n->dz2, n->dz3, n->h3, n->df1, n->df2, n->df3, n->cols};
    if ((rc = launch_train_step(B, X, target, M, A, s))) return rc;
    if (loss_host) {
        std::vector<float> yh(M), th(M);
        NGMI_HIP(hipMemcpyAsync(yh.data(), n->y, (size_t)M * 4, hipMemcpyDeviceToHost, s));
        NGMI_HIP(hipMemcpyAsync(th.data(), target, (size_t)M * 4, hipMemcpyDeviceToHost, s));
        NGMI_HIP(hipStreamSynchronize(s));
        double acc = 0;
        for (int i = 0; i < M; i++) acc += (double)(yh[i] - th[i]) * (yh[i] - th[i]);
        *loss_host = (float)(acc / M);
    }
    return NGMI_OK;
}

}  // extern "C"
