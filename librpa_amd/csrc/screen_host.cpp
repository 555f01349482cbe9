// Block-norm screening of the chi0 build: plan-time block tables, per-tau features and skip
// flags, training-sample export and the MLP training loop.
//
// A chi0 output block (I, J, R) at tau is skipped when the norm-product bound
//   ||chi0s(I,J,R)||_F <= c_I c_J (g+_IJ gm- + g-_IJ gm+ + 2 gm+ gm-)
// (c_A: sum of the Frobenius norms of atom A's folded Cs blocks; g: Frobenius norms of the
// G_IJ(R, +-tau) blocks, gm: their maxima) is below the threshold, or, in learned mode, when
// the MLP's prediction of ln ||chi0s(I,J,R)||_F is.  Every term of the chi0 label sums
// (thirdparty/LibRI/include/RI/physics/RPA.hpp:104-138) is a contraction <C^I_mu, G C^J_nu G'^T>,
// which the bound majorises term by term.  Skipped blocks are exactly zero in chi0(R, tau).
#include <algorithm>
#include <cmath>
#include <random>

#include "rpa.h"
#include "screen.h"

namespace lra {

void RpaEngine::screen_plan(const Dataset &ds) {
    const int nout = (int)outs.size();
    const long long gpm_r = (long long)NAO * 2 * NAO;
    gblocks.assign(2 * (size_t)nout, BlockRef{});
    feat_static.assign(5 * (size_t)nout, 0.0f);
    std::vector<long long> eo(nout);
    std::vector<int> es(nout);
    const bool geo = ds.lat_set && ds.pos.size() >= 3 * (size_t)natom;
    for (int o = 0; o < nout; ++o) {
        const auto &O = outs[o];
        for (int s = 0; s < 2; ++s)
            gblocks[2 * (size_t)o + s] = {O.r * gpm_r + ao[O.I] * 2LL * NAO + 2 * ao[O.J] + (long long)s * nb[O.J],
                                          nb[O.I], nb[O.J]};
        double d = 0;
        if (geo) {
            double v[3];
            for (int c = 0; c < 3; ++c) {
                v[c] = ds.pos[3 * (size_t)O.J + c] - ds.pos[3 * (size_t)O.I + c];
                for (int a = 0; a < 3; ++a) v[c] += cells[O.r][a] * ds.latvec[3 * a + c];
            }
            d = std::sqrt(v[0] * v[0] + v[1] * v[1] + v[2] * v[2]);
        }
        float *f = &feat_static[5 * (size_t)o];
        f[0] = (float)(d / 10.0);
        f[1] = (float)(nb[O.I] / 27.0);
        f[2] = (float)(nb[O.J] / 27.0);
        f[3] = (float)std::log(std::max(cnorm[O.I], 1e-300));
        f[4] = (float)std::log(std::max(cnorm[O.J], 1e-300));
        eo[o] = O.eoff;
        es[o] = na[O.I] * na[O.J];
    }
    d_gblocks = upload(gblocks, stream);
    d_eoff = upload(eo, stream);
    d_esize = upload(es, stream);
    d_gnorm.alloc(sizeof(double) * 2 * std::max(1, nout) * nbatch);
    d_feat.alloc(sizeof(float) * MLP_NFEAT * std::max(1, nout) * nbatch);
    d_pred.alloc(sizeof(float) * std::max(1, nout) * nbatch);
}

void RpaEngine::screen_taus(int it, const double *taus, int nz) {
    const int nout = (int)outs.size();
    if (nout == 0) return;
    auto &prof = profiler();
    prof.begin("chi0_screen", stream);
    const long long zg = (long long)nR * NAO * 2 * NAO;
    for (int z = 0; z < nz; ++z) {
        double *gn = d_gnorm.as<double>() + (size_t)z * 2 * nout;
        if (cur == Prec::F64)
            launch_block_norms<double>(d_Gpm.as<double>() + z * zg, 2LL * NAO, d_gblocks.as<BlockRef>(), 2 * nout, gn, stream);
        else
            launch_block_norms<float>(d_Gpm.as<float>() + z * zg, 2LL * NAO, d_gblocks.as<BlockRef>(), 2 * nout, gn, stream);
    }
    gnorm_h.resize(2 * (size_t)nout * nz);
    HIP_CHECK(hipMemcpyAsync(gnorm_h.data(), d_gnorm.get(), sizeof(double) * gnorm_h.size(), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
    feat_h.resize((size_t)MLP_NFEAT * nout * nz);
    skip_out.assign((size_t)nout * nz, 0);
    for (int z = 0; z < nz; ++z) {
        const double *gn = gnorm_h.data() + (size_t)z * 2 * nout;
        float *fz = feat_h.data() + (size_t)z * MLP_NFEAT * nout;
        double gpx = 0, gmx = 0;
        for (int o = 0; o < nout; ++o) {
            gpx = std::max(gpx, gn[2 * (size_t)o]);
            gmx = std::max(gmx, gn[2 * (size_t)o + 1]);
        }
        const float ltau = (float)std::log(taus[z]), lgm = (float)std::log(gpx * gmx + 1e-300);
        for (int o = 0; o < nout; ++o) {
            const float *fs = &feat_static[5 * (size_t)o];
            float *f = fz + (size_t)MLP_NFEAT * o;
            f[0] = fs[0]; f[1] = fs[1]; f[2] = fs[2]; f[3] = ltau; f[4] = fs[3]; f[5] = fs[4];
            f[6] = (float)std::log(gn[2 * (size_t)o] * gn[2 * (size_t)o + 1] + 1e-300);
            f[7] = lgm;
        }
        if (collect) std::copy(fz, fz + (size_t)MLP_NFEAT * nout, features.begin() + (size_t)(it + z) * MLP_NFEAT * nout);
        if (screen_mode == 0) continue;
        for (int o = 0; o < nout; ++o) {
            const auto &O = outs[o];
            const double bound = cnorm[O.I] * cnorm[O.J] *
                                 (gn[2 * (size_t)o] * gmx + gn[2 * (size_t)o + 1] * gpx + 2.0 * gpx * gmx);
            if (bound < screen_thr) skip_out[(size_t)z * nout + o] = 1;
        }
    }
    if (screen_mode == 0) {
        prof.end("chi0_screen", stream);
        return;
    }
    if (screen_mode == 2) {
        // standardise with the model's scaling, predict ln ||chi0s|| on the device
        const float *mean = screen_model.data() + MLP_NPARAM, *scale = mean + MLP_NFEAT;
        const float tmean = screen_model[MLP_NPARAM + 2 * MLP_NFEAT], tscale = screen_model[MLP_NPARAM + 2 * MLP_NFEAT + 1];
        std::vector<float> xs(feat_h.size());
        for (size_t i = 0; i < xs.size(); ++i) xs[i] = (feat_h[i] - mean[i % MLP_NFEAT]) / scale[i % MLP_NFEAT];
        HIP_CHECK(hipMemcpyAsync(d_feat.get(), xs.data(), sizeof(float) * xs.size(), hipMemcpyHostToDevice, stream));
        launch_mlp_forward(d_model.as<float>(), d_feat.as<float>(), nout * nz, d_pred.as<float>(), stream);
        pred_h.resize((size_t)nout * nz);
        HIP_CHECK(hipMemcpyAsync(pred_h.data(), d_pred.get(), sizeof(float) * pred_h.size(), hipMemcpyDeviceToHost, stream));
        HIP_CHECK(hipStreamSynchronize(stream));
        const double lthr = std::log(screen_thr);
        for (size_t i = 0; i < pred_h.size(); ++i)
            if ((double)pred_h[i] * tscale + tmean < lthr) skip_out[i] = 1;
    }
    double fl = 0, fls = 0, nsk = 0;
    for (size_t i = 0; i < skip_out.size(); ++i) {
        fl += out_flops[i % nout];
        if (skip_out[i]) fls += out_flops[i % nout];
        nsk += skip_out[i];
    }
    HIP_CHECK(hipMemcpyAsync(d_skip.get(), skip_out.data(), skip_out.size(), hipMemcpyHostToDevice, stream));
    scr_blocks += (double)nout * nz;
    scr_skipped += nsk;
    scr_flops += fl;
    scr_flops_skipped += fls;
    prof.end("chi0_screen", stream);
}

void RpaEngine::chi0_norms(std::vector<double> &out) {
    if (host_staged) LRA_THROW("chi0 block norms need the device-resident chi0 store (too large here)");
    const int nout = (int)outs.size();
    out.assign((size_t)ntau_done * nout, 0.0);
    if (out.empty()) return;
    DevBuf d((size_t)ntau_done * nout * sizeof(double));
    if (prec == Prec::F64)
        launch_chi0_block_norms<double>(d_chi0s.as<double>(), E_tot, ntau_done, d_eoff.as<long long>(),
                                        d_esize.as<int>(), nout, d.as<double>(), stream);
    else
        launch_chi0_block_norms<float>(d_chi0s.as<float>(), E_tot, ntau_done, d_eoff.as<long long>(),
                                       d_esize.as<int>(), nout, d.as<double>(), stream);
    HIP_CHECK(hipMemcpyAsync(out.data(), d.get(), sizeof(double) * out.size(), hipMemcpyDeviceToHost, stream));
    HIP_CHECK(hipStreamSynchronize(stream));
}

double mlp_train(const float *X, const float *t, int n, int iters, double lr, int seed, float *model) {
    if (n < 2) LRA_THROW("mlp_train: need at least two samples");
    if (iters < 1) LRA_THROW("mlp_train: iters must be positive");
    // feature / target standardisation (a constant feature keeps scale 1)
    std::vector<double> mean(MLP_NFEAT, 0.0), var(MLP_NFEAT, 0.0);
    double tm = 0, tv = 0;
    for (int s = 0; s < n; ++s) {
        for (int k = 0; k < MLP_NFEAT; ++k) mean[k] += X[(size_t)s * MLP_NFEAT + k];
        tm += t[s];
    }
    for (int k = 0; k < MLP_NFEAT; ++k) mean[k] /= n;
    tm /= n;
    for (int s = 0; s < n; ++s) {
        for (int k = 0; k < MLP_NFEAT; ++k) {
            const double d = X[(size_t)s * MLP_NFEAT + k] - mean[k];
            var[k] += d * d;
        }
        tv += (t[s] - tm) * (t[s] - tm);
    }
    std::vector<float> sc(MLP_NFEAT);
    for (int k = 0; k < MLP_NFEAT; ++k) {
        const double sd = std::sqrt(var[k] / n);
        sc[k] = sd > 1e-6 ? (float)sd : 1.0f;
    }
    const double tsd = std::sqrt(tv / n) > 1e-12 ? std::sqrt(tv / n) : 1.0;
    std::vector<float> xs((size_t)n * MLP_NFEAT), ts(n);
    for (int s = 0; s < n; ++s) {
        for (int k = 0; k < MLP_NFEAT; ++k)
            xs[(size_t)s * MLP_NFEAT + k] = (float)((X[(size_t)s * MLP_NFEAT + k] - mean[k]) / sc[k]);
        ts[s] = (float)((t[s] - tm) / tsd);
    }
    // fan-in scaled uniform weights, zero biases
    std::vector<float> p(MLP_NPARAM, 0.0f);
    std::mt19937_64 rng((unsigned long long)seed);
    std::uniform_real_distribution<double> u(-1.0, 1.0);
    for (int i = 0; i < MLP_NFEAT * MLP_H; ++i) p[i] = (float)(u(rng) / std::sqrt((double)MLP_NFEAT));
    const int ow2 = MLP_NFEAT * MLP_H + MLP_H, ow3 = ow2 + MLP_H * MLP_H + MLP_H;
    for (int i = 0; i < MLP_H * MLP_H; ++i) p[ow2 + i] = (float)(u(rng) / std::sqrt((double)MLP_H));
    for (int i = 0; i < MLP_H; ++i) p[ow3 + i] = (float)(u(rng) / std::sqrt((double)MLP_H));
    hipStream_t s = 0;
    DevBuf dX = upload(xs, s), dt = upload(ts, s), dp = upload(p, s);
    DevBuf dg(sizeof(float) * MLP_NPARAM), dm(sizeof(float) * MLP_NPARAM), dv(sizeof(float) * MLP_NPARAM),
        dl(sizeof(double));
    HIP_CHECK(hipMemsetAsync(dm.get(), 0, dm.bytes(), s));
    HIP_CHECK(hipMemsetAsync(dv.get(), 0, dv.bytes(), s));
    MlpWork w;
    for (int step = 1; step <= iters; ++step) {
        // learning rate decays geometrically to lr / 20 over the run
        const float lr_s = (float)(lr * std::pow(0.05, (double)(step - 1) / iters));
        mlp_loss_grad(dp.as<float>(), dX.as<float>(), dt.as<float>(), n, dg.as<float>(), dl.as<double>(), w, s);
        launch_adam(dp.as<float>(), dg.as<float>(), dm.as<float>(), dv.as<float>(), MLP_NPARAM, lr_s, step, s);
    }
    mlp_loss_grad(dp.as<float>(), dX.as<float>(), dt.as<float>(), n, dg.as<float>(), dl.as<double>(), w, s);
    double loss = 0;
    HIP_CHECK(hipMemcpy(&loss, dl.get(), sizeof(double), hipMemcpyDeviceToHost));
    HIP_CHECK(hipMemcpy(model, dp.get(), sizeof(float) * MLP_NPARAM, hipMemcpyDeviceToHost));
    for (int k = 0; k < MLP_NFEAT; ++k) {
        model[MLP_NPARAM + k] = (float)mean[k];
        model[MLP_NPARAM + MLP_NFEAT + k] = sc[k];
    }
    model[MLP_NPARAM + 2 * MLP_NFEAT] = (float)tm;
    model[MLP_NPARAM + 2 * MLP_NFEAT + 1] = (float)tsd;
    return loss;
}

}  // namespace lra
