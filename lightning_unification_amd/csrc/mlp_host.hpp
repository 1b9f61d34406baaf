// Host side of the learned surrogate: a d0 -> d1 -> d2 -> d3 MLP (GELU on the
// two hidden layers) whose weights live in HBM as FP32 masters plus BF16
// copies for the matrix cores.  Forward, backward and Adam run as the kernels
// of kernels_mlp.hpp on one stream, seven launches a training step (three
// forward, the last with the loss; three backward, one per layer; Adam);
// training data stays resident on the device (features in BF16, targets in
// FP32) and minibatches are contiguous slices of it.  Every BF16 array's rows
// are padded with zeros to a multiple of kMlpPad columns, and row counts to
// that of a workgroup's block, so the products read whole blocks.
//
// Parameter layout (host and device, FP32): W1 [d0 x d1] row-major, b1 [d1],
// W2 [d1 x d2], b2 [d2], W3 [d2 x d3], b3 [d3].  y = act2 W3 + b3 with
// act_k = GELU(act_{k-1} W_k + b_k), act_0 = x.
#pragma once

#include <hip/hip_runtime.h>

#include <cmath>
#include <vector>

#include "kernels_mlp.hpp"

namespace plamd {

struct Mlp {
    int d[4];
    int maxb;
    size_t woff[3], boff[3], nparam = 0;
    hipStream_t stream = nullptr;
    float *p32 = nullptr, *grad = nullptr, *mom = nullptr, *vel = nullptr; // nparam each
    int ld[4];                             // padded widths
    MlpLayout lay{};
    uint16_t *pbf = nullptr;               // padded BF16 weights, W1 then W2 then W3
    uint16_t *xb = nullptr, *a1 = nullptr, *a2 = nullptr;     // padded BF16 activations
    uint16_t *dyb = nullptr, *dz1 = nullptr, *dz2 = nullptr;  // padded BF16 gradients
    float *z1 = nullptr, *z2 = nullptr, *y = nullptr;
    float *cp1 = nullptr, *cp2 = nullptr, *cp3 = nullptr;     // column sums per row block of dz1, dz2, dy
    float *tb = nullptr, *colw = nullptr, *xf = nullptr;
    double *lpart = nullptr; // loss partials of up to kLossParts / (partials a step) steps
    uint16_t *data_x = nullptr;
    float *data_t = nullptr;
    int64_t ndata = 0;
    int64_t step = 0, cursor = 0;
    static constexpr size_t kLossParts = 1 << 16;

    Mlp(int d0, int d1, int d2, int d3, int max_batch, uint64_t seed) : d{d0, d1, d2, d3}, maxb(max_batch) {
        for (int l = 0; l < 3; l++) {
            woff[l] = nparam;
            nparam += static_cast<size_t>(d[l]) * d[l + 1];
            boff[l] = nparam;
            nparam += d[l + 1];
        }
        HIP_OK(hipStreamCreateWithFlags(&stream, hipStreamNonBlocking));
        auto alloc = [](auto **p, size_t count) {
            HIP_OK(hipMalloc(reinterpret_cast<void **>(p), std::max<size_t>(count, 1) * sizeof(**p)));
        };
        alloc(&p32, nparam);
        alloc(&grad, nparam);
        alloc(&mom, nparam);
        alloc(&vel, nparam);
        size_t nbf = 0;
        for (int l = 0; l < 4; l++) {
            ld[l] = (d[l] + kMlpPad - 1) / kMlpPad * kMlpPad;
        }
        for (int l = 0; l < 3; l++) {
            lay.woff[l] = static_cast<int64_t>(woff[l]);
            lay.boff[l] = static_cast<int64_t>(boff[l]);
            lay.cols[l] = d[l + 1];
            lay.bf[l] = static_cast<int64_t>(nbf);
            lay.ld[l] = ld[l + 1];
            nbf += static_cast<size_t>(ld[l]) * ld[l + 1];
        }
        alloc(&pbf, nbf);
        HIP_OK(hipMemsetAsync(pbf, 0, nbf * sizeof(uint16_t), stream)); // the padding stays zero
        const size_t B = row_pad(maxb), nblk = B / 32;
        alloc(&xf, static_cast<size_t>(maxb) * d0);
        alloc(&xb, B * ld[0]);
        alloc(&a1, B * ld[1]);
        alloc(&a2, B * ld[2]);
        alloc(&z1, B * ld[1]);
        alloc(&z2, B * ld[2]);
        alloc(&dz1, B * ld[1]);
        alloc(&dz2, B * ld[2]);
        alloc(&dyb, B * ld[3]);
        alloc(&y, static_cast<size_t>(maxb) * d3);
        alloc(&tb, static_cast<size_t>(maxb) * d3);
        alloc(&colw, d3);
        alloc(&cp1, nblk * ld[1]);
        alloc(&cp2, nblk * ld[2]);
        alloc(&cp3, nblk * ld[3]);
        alloc(&lpart, std::max(kLossParts, loss_parts(maxb)));
        // He-uniform weights (GELU), zero biases; SplitMix64 draws
        std::vector<float> h(nparam, 0.0f);
        uint64_t s = seed;
        auto next = [&s]() {
            uint64_t z = (s += 0x9E3779B97F4A7C15ull);
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            z ^= z >> 31;
            return static_cast<double>(z >> 11) * 0x1.0p-53;
        };
        for (int l = 0; l < 3; l++) {
            const double lim = std::sqrt(6.0 / d[l]);
            for (size_t e = 0; e < static_cast<size_t>(d[l]) * d[l + 1]; e++) {
                h[woff[l] + e] = static_cast<float>((2.0 * next() - 1.0) * lim);
            }
        }
        set_params(h.data());
        std::vector<float> ones(d3, 1.0f);
        HIP_OK(hipMemcpy(colw, ones.data(), d3 * sizeof(float), hipMemcpyHostToDevice));
    }

    ~Mlp() {
        for (void *p : {static_cast<void *>(p32), static_cast<void *>(grad), static_cast<void *>(mom),
                        static_cast<void *>(vel), static_cast<void *>(pbf), static_cast<void *>(xf),
                        static_cast<void *>(xb), static_cast<void *>(a1), static_cast<void *>(a2),
                        static_cast<void *>(z1), static_cast<void *>(z2), static_cast<void *>(dz1),
                        static_cast<void *>(dz2), static_cast<void *>(dyb), static_cast<void *>(y),
                        static_cast<void *>(cp1), static_cast<void *>(cp2), static_cast<void *>(cp3),
                        static_cast<void *>(tb), static_cast<void *>(colw), static_cast<void *>(lpart),
                        static_cast<void *>(data_x), static_cast<void *>(data_t)}) {
            if (p) {
                (void)hipFree(p);
            }
        }
        if (stream) {
            (void)hipStreamDestroy(stream);
        }
    }

    // rows a padded array holds for n used ones (whole workgroup blocks)
    static size_t row_pad(int64_t n) { return static_cast<size_t>((n + 63) / 64 * 64); }
    static unsigned tiles(int rows, int cols, int tile_rows) {
        return static_cast<unsigned>((rows + tile_rows - 1) / tile_rows) * static_cast<unsigned>((cols + 63) / 64);
    }
    size_t loss_parts(int B) const { return tiles(B, d[3], 32); }
    static unsigned blocks(int64_t n) { return static_cast<unsigned>((n + 255) / 256); }

    void set_params(const float *host) {
        HIP_OK(hipMemcpyAsync(p32, host, nparam * sizeof(float), hipMemcpyHostToDevice, stream));
        hipLaunchKernelGGL(k_weights_to_bf16, dim3(blocks(nparam)), dim3(256), 0, stream, p32, pbf, lay,
                           static_cast<int64_t>(nparam));
        HIP_OK(hipGetLastError());
        HIP_OK(hipMemsetAsync(mom, 0, nparam * sizeof(float), stream));
        HIP_OK(hipMemsetAsync(vel, 0, nparam * sizeof(float), stream));
        HIP_OK(hipStreamSynchronize(stream));
        step = 0;
    }

    void forward_layer(const GemmArgs &g) {
        hipLaunchKernelGGL(k_mlp_forward, dim3(tiles(g.M, g.N, 32)), dim3(kMlpThreads), 0, stream, g);
        HIP_OK(hipGetLastError());
    }

    // y[B x d3] for padded BF16 features x; with targets t, dloss/dy (dyb, its
    // column sums in cp3) and the loss partials at `loss` instead of y
    void forward(const uint16_t *x, int B, const float *t = nullptr, double *loss = nullptr) {
        GemmArgs g{};
        g.A = x, g.lda = ld[0], g.B = pbf + lay.bf[0], g.ldb = ld[1], g.M = B, g.N = d[1], g.K = d[0];
        g.bias = p32 + boff[0], g.Z = z1, g.act = a1, g.ldact = ld[1], g.epi = kEpiGelu;
        forward_layer(g);
        g.A = a1, g.lda = ld[1], g.B = pbf + lay.bf[1], g.ldb = ld[2], g.N = d[2], g.K = d[1];
        g.bias = p32 + boff[1], g.Z = z2, g.act = a2, g.ldact = ld[2];
        forward_layer(g);
        g.A = a2, g.lda = ld[2], g.B = pbf + lay.bf[2], g.ldb = ld[3], g.N = d[3], g.K = d[2];
        g.bias = p32 + boff[2], g.Z = nullptr, g.act = dyb, g.ldact = ld[3], g.C = y;
        g.target = t, g.colw = colw, g.loss = loss, g.colpart = cp3, g.epi = t ? kEpiLoss : kEpiOut;
        forward_layer(g);
    }

    // Layer l's weight and bias gradients from its dz (padded BF16, column
    // sums cp) and input act, and dzp of the layer before through Zp.
    void backward_layer(int l, int B, const uint16_t *act, const uint16_t *dz, const float *cp, uint16_t *dzp,
                        float *Zp, float *cpp) {
        GemmArgs w{}, z{};
        w.A = act, w.lda = ld[l], w.B = dz, w.ldb = ld[l + 1], w.M = d[l], w.N = d[l + 1], w.K = B;
        w.C = grad + woff[l], w.epi = kEpiGrad;
        const unsigned nw = tiles(w.M, w.N, 64);
        unsigned nz = 0;
        if (dzp) {
            z.A = dz, z.lda = ld[l + 1], z.B = pbf + lay.bf[l], z.ldb = ld[l + 1], z.M = B, z.N = d[l],
            z.K = d[l + 1];
            z.Z = Zp, z.act = dzp, z.ldact = ld[l], z.colpart = cpp, z.epi = kEpiGeluGrad;
            nz = tiles(z.M, z.N, 32);
        }
        const ColsumArgs cs{cp, (B + 31) / 32, ld[l + 1], d[l + 1], grad + boff[l]};
        const unsigned nc = static_cast<unsigned>((d[l + 1] + 63) / 64);
        hipLaunchKernelGGL(k_mlp_backward, dim3(nw + nz + nc), dim3(kMlpThreads), 0, stream, w, nw, z, nz, cs);
        HIP_OK(hipGetLastError());
    }

    // gradients of the weighted MSE into `grad`, queued (after forward with targets)
    void backward(const uint16_t *x, int B) {
        backward_layer(2, B, a2, dyb, cp3, dz2, z2, cp2);
        backward_layer(1, B, a1, dz2, cp2, dz1, z1, cp1);
        backward_layer(0, B, x, dz1, cp1, nullptr, nullptr, nullptr);
    }

    // sum over `steps` steps of the batch loss, each step's partials added in order
    double read_losses(int64_t steps, int B) {
        const size_t per = loss_parts(B);
        std::vector<double> part(static_cast<size_t>(steps) * per);
        HIP_OK(hipMemcpyAsync(part.data(), lpart, part.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
        HIP_OK(hipStreamSynchronize(stream));
        double tot = 0;
        for (int64_t s = 0; s < steps; s++) {
            double v = 0;
            for (size_t i = 0; i < per; i++) {
                v += part[s * per + i];
            }
            tot += v / B;
        }
        return tot;
    }

    void adam(float lr) {
        step++;
        const float b1 = 0.9f, b2 = 0.999f;
        const float c1 = 1.0f - std::pow(b1, static_cast<float>(step));
        const float c2 = 1.0f - std::pow(b2, static_cast<float>(step));
        hipLaunchKernelGGL(k_adam, dim3(blocks(nparam)), dim3(256), 0, stream, p32, pbf, lay, mom, vel, grad,
                           static_cast<int64_t>(nparam), lr, b1, b2, 1e-8f, c1, c2);
        HIP_OK(hipGetLastError());
    }

    void check_batch(int64_t n) const {
        if (n < 1 || n > maxb) {
            throw InvalidArg("batch size must be in [1, " + std::to_string(maxb) + "]");
        }
    }

    void upload_x(const float *x_host, int n) {
        check_batch(n);
        HIP_OK(hipMemcpyAsync(xf, x_host, static_cast<size_t>(n) * d[0] * sizeof(float), hipMemcpyHostToDevice,
                              stream));
        hipLaunchKernelGGL(k_to_bf16, dim3(blocks(static_cast<int64_t>(n) * ld[0])), dim3(256), 0, stream, xf, xb,
                           static_cast<int64_t>(n), d[0], ld[0]);
        HIP_OK(hipGetLastError());
    }

    void predict(const float *x_host, int n, float *y_host) {
        upload_x(x_host, n);
        forward(xb, n);
        HIP_OK(hipMemcpyAsync(y_host, y, static_cast<size_t>(n) * d[3] * sizeof(float), hipMemcpyDeviceToHost,
                              stream));
        HIP_OK(hipStreamSynchronize(stream));
    }

    double gradients(const float *x_host, const float *t_host, int n, float *g_host) {
        upload_x(x_host, n);
        HIP_OK(hipMemcpyAsync(tb, t_host, static_cast<size_t>(n) * d[3] * sizeof(float), hipMemcpyHostToDevice,
                              stream));
        forward(xb, n, tb, lpart);
        backward(xb, n);
        const double loss = read_losses(1, n);
        HIP_OK(hipMemcpy(g_host, grad, nparam * sizeof(float), hipMemcpyDeviceToHost));
        return loss;
    }

    void load_data(const float *x_host, const float *t_host, int64_t n) {
        for (void *p : {static_cast<void *>(data_x), static_cast<void *>(data_t)}) {
            if (p) {
                HIP_OK(hipFree(p));
            }
        }
        data_x = nullptr;
        data_t = nullptr;
        ndata = n;
        cursor = 0;
        HIP_OK(hipMalloc(reinterpret_cast<void **>(&data_x), row_pad(n + 63) * ld[0] * sizeof(uint16_t)));
        HIP_OK(hipMalloc(reinterpret_cast<void **>(&data_t), std::max<int64_t>(n, 1) * d[3] * sizeof(float)));
        // features through the FP32 staging buffer, maxb rows at a time
        for (int64_t r = 0; r < n; r += maxb) {
            const int64_t m = std::min<int64_t>(maxb, n - r);
            HIP_OK(hipMemcpyAsync(xf, x_host + r * d[0], m * d[0] * sizeof(float), hipMemcpyHostToDevice, stream));
            hipLaunchKernelGGL(k_to_bf16, dim3(blocks(m * ld[0])), dim3(256), 0, stream, xf, data_x + r * ld[0],
                               m, d[0], ld[0]);
            HIP_OK(hipGetLastError());
            HIP_OK(hipStreamSynchronize(stream));
        }
        HIP_OK(hipMemcpy(data_t, t_host, n * d[3] * sizeof(float), hipMemcpyHostToDevice));
    }

    // `steps` Adam steps over consecutive minibatches of the loaded data
    double train(int64_t steps, int batch, float lr) {
        check_batch(batch);
        if (ndata < batch) {
            throw InvalidArg("load at least one batch of data first");
        }
        // the steps' loss partials stay on the device until there is no room
        // for another step's, so the queue runs without a wait per step
        const size_t per = loss_parts(batch);
        const int64_t room = std::max<int64_t>(1, static_cast<int64_t>(kLossParts / per));
        double tot = 0;
        int64_t held = 0;
        for (int64_t s = 0; s < steps; s++) {
            if (cursor + batch > ndata) {
                cursor = 0;
            }
            const uint16_t *x = data_x + cursor * ld[0];
            const float *t = data_t + cursor * d[3];
            cursor += batch;
            forward(x, batch, t, lpart + held * per);
            backward(x, batch);
            adam(lr);
            if (++held == room || s + 1 == steps) {
                tot += read_losses(held, batch);
                held = 0;
            }
        }
        HIP_OK(hipStreamSynchronize(stream));
        return steps ? tot / steps : 0.0;
    }
};

} // namespace plamd
