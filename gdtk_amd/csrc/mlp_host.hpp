// mlp_host.hpp -- the network handle of the C ABI (defined in mlp.cpp).
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <vector>

#include "host_common.hpp"
#include "mlp_launch.hpp"

namespace gdtk {

struct Mlp {
    int n_in = 0, H = 0, NH = 0, n_out = 0;
    int nlayer = 0;  // NH + 1
    std::vector<int> in_w, out_w;
    std::vector<size_t> woff, boff;
    size_t nparam = 0;
    DevArr<float> params, grads, am, av;
    int adam_t = 0;
    // BF16-aware training: the forward pass uses BF16-rounded inputs, weights (wq, refreshed
    // after every update) and hidden activations, as the inference kernel does; gradients
    // pass the roundings unchanged and update the FP32 masters.
    int bf16_train = 0;
    DevArr<float> wq;
    // the inner layers' weights (wq's with bf16_train) in the operand order of the training passes
    DevArr<float> packed_w;
    bool wq_fresh = false;  // wq (with bf16_train) and packed_w follow params
    // BF16 inference fragments and the concatenated biases
    DevArr<unsigned short> frag;
    DevArr<float> bias_cat;
    bool packed = false;
    // training batch buffers (the layouts of MlpPass)
    int bcap = 0;
    std::vector<DevArr<float>> act, dz;
    DevArr<float> xb, yb, yout, loss, gparts;
    DevArr<int> idx;
    hipStream_t stream = nullptr;

    ~Mlp() {
        if (stream) (void)hipStreamDestroy(stream);
    }

    void layout() {
        nlayer = NH + 1;
        in_w.assign(nlayer, H);
        out_w.assign(nlayer, H);
        in_w[0] = n_in;
        out_w[nlayer - 1] = n_out;
        woff.resize(nlayer);
        boff.resize(nlayer);
        size_t o = 0;
        for (int l = 0; l < nlayer; ++l) {
            woff[l] = o;
            o += (size_t)out_w[l] * in_w[l];
            boff[l] = o;
            o += out_w[l];
        }
        nparam = o;
    }

    void ensure_batch(int B) {
        if (B <= bcap) return;
        bcap = 0;  // until every buffer has been allocated
        const size_t cells = (size_t)mlp_blocks(B) * 16;
        act.clear();
        dz.clear();
        act.resize(nlayer);
        dz.resize(nlayer);
        MlpPass q{};
        for (int l = 0; l < nlayer; ++l) {
            act[l].alloc(cells * ((in_w[l] + 15) / 16 * 16));
            dz[l].alloc(cells * ((out_w[l] + 15) / 16 * 16));
            q.in_w[l] = in_w[l];
            q.out_w[l] = out_w[l];
        }
        xb.alloc((size_t)B * n_in);
        yb.alloc((size_t)B * n_out);
        yout.alloc((size_t)B * n_out);
        loss.alloc((size_t)mlp_blocks(B));
        gparts.alloc((size_t)mlp_grad_splits(q, nlayer, B) * nparam);
        bcap = B;
    }

    // The batch's inputs at x[k xk + row xc] (rows idx[b], or b), targets likewise.
    MlpPass pass(int B, const float* x, size_t xk, size_t xc, const float* y, size_t yk, size_t yc, const int* rows,
                 hipStream_t s) {
        MlpPass q{};
        q.B = B;
        q.n_in = n_in;
        q.n_out = n_out;
        q.bf16 = bf16_train;
        q.x = x;
        q.y = y;
        q.xk = xk;
        q.xc = xc;
        q.yk = yk;
        q.yc = yc;
        q.idx = rows;
        q.y_out = yout.p;
        q.loss = loss.p;
        const float* Wm = weights(s);
        for (int l = 0; l < nlayer; ++l) {
            q.W[l] = Wm + woff[l];
            const bool in = l > 0 && l < nlayer - 1;
            q.Wf[l] = in ? packed_w.p + (size_t)(l - 1) * 2 * H * H : nullptr;
            q.Wb[l] = in ? q.Wf[l] + H * H : nullptr;
            q.b[l] = params.p + boff[l];  // the biases stay FP32 (as in inference)
            q.act[l] = act[l].p;
            q.dz[l] = dz[l].p;
            q.in_w[l] = in_w[l];
            q.out_w[l] = out_w[l];
            q.woff[l] = woff[l];
            q.boff[l] = boff[l];
        }
        return q;
    }

    size_t inner() const { return (size_t)(nlayer - 2); }
    const float* weights(hipStream_t s) {
        if (!wq_fresh) {
            if (bf16_train) {
                wq.reserve(nparam);
                HIPCHK(launch_round_bf16(nparam, params.p, wq.p, s));
            }
            packed_w.reserve(inner() * 2 * H * H);
            HIPCHK(launch_mlp_operands(nparam, bf16_train ? wq.p : params.p, packed_w.p, H, woff[1], inner(), s));
            wq_fresh = true;
        }
        return bf16_train ? wq.p : params.p;
    }

    // Loss and gradient shares of a batch; the number of shares in gparts.
    int loss_grad(const MlpPass& q, hipStream_t s) {
        const int nz = mlp_grad_splits(q, nlayer, q.B);
        HIPCHK(launch_mlp_pass(H, NH, q, 1, s));
        HIPCHK(launch_mlp_weight_grad(q, nlayer, nz, nparam, gparts.p, s));
        return nz;
    }

    double read_loss(int B, hipStream_t s) {
        const int np = mlp_blocks(B);
        std::vector<float> h((size_t)np);
        HIPCHK(hipMemcpyAsync(h.data(), loss.p, np * sizeof(float), hipMemcpyDeviceToHost, s));
        HIPCHK(hipStreamSynchronize(s));
        double acc = 0.0;
        for (float v : h) acc += v;
        return acc / ((double)B * n_out);
    }

    void adam(float lr, int nz, hipStream_t s) {
        ++adam_t;
        HIPCHK(launch_mlp_adam(nparam, nz, gparts.p, params.p, am.p, av.p, bf16_train ? wq.p : nullptr, packed_w.p, H,
                               woff[1], inner(), lr, 0.9f, 0.999f, 1.0e-8f, adam_t, s));
        packed = false;
        wq_fresh = true;
    }

    void pack(hipStream_t s) {
        if (packed) return;
        size_t nfrag = 0;
        std::vector<size_t> foff(nlayer);
        for (int l = 0; l < nlayer; ++l) {
            foff[l] = nfrag;
            nfrag += (size_t)((out_w[l] + 15) / 16) * ((in_w[l] + 31) / 32) * 64 * 8;
        }
        frag.reserve(nfrag);
        size_t nb = 0;
        for (int l = 0; l < nlayer; ++l) nb += out_w[l];
        bias_cat.reserve(nb);
        size_t bo = 0;
        for (int l = 0; l < nlayer; ++l) {
            HIPCHK(launch_mlp_pack(params.p + woff[l], out_w[l], in_w[l], l > 0 ? 1 : 0, frag.p + foff[l], s));
            HIPCHK(hipMemcpyAsync(bias_cat.p + bo, params.p + boff[l], out_w[l] * sizeof(float),
                                  hipMemcpyDeviceToDevice, s));
            bo += out_w[l];
        }
        packed = true;
    }
};

Mlp& get_mlp(int h);
// BF16 inference of n cells: x SoA [n_in][n] -> y SoA [n_out][n] (device arrays).
// Inference over x, y [n_in/n_out][n]; with count (device memory, may be null) only the
// first *count cells are evaluated (the arrays keep the stride n).
void mlp_infer(Mlp& m, int n, const float* x, float* y, hipStream_t s, const unsigned* count = nullptr);

}  // namespace gdtk
