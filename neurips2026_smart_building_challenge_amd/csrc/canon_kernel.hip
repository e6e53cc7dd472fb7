// Canonical policy interface of the env (env kwargs canonical = 1, residual),
// on the device: the env's own observation stays in an internal row, and two
// small kernels around the step give the policy its canonical view.
//
//   canon_pre_kernel   (before the step) the policy's canonical action row and
//                      the base controller's proposal -> the env's native
//                      action row (residual: base + res_scale p, run bits
//                      (2 base - 1) + res_dscale p > 0; absolute: p, run bits
//                      p > -0.5; p clamped to [-1, 1], non-finite -> 0, times
//                      the comfort guard's trust when it is on), which the step
//                      kernel then decodes as any action row
//                      (complete_port/gpu/sb_gpu_base.inc:371-404 decode_res_k);
//   canon_post_kernel  (after the step or reset) from the env's new observation:
//                      the pid_water base controller's proposal for the next
//                      step and its PID state (zeroed when the env starts an
//                      episode; complete_port/submission/pidw_base.py
//                      PIDWaterResetPolicy, zones of an AHU in observation
//                      order, its float32 / float64 arithmetic op by op), the
//                      comfort guard's trust (sb_gpu_base.inc:230-265), and the
//                      canonical observation into the trainer's row
//                      (sb_gpu_base.inc:287-369).
#include <hip/hip_runtime.h>
#include <math.h>

#include "canon.h"
#include "sbenv_internal.h"

namespace sbk {

// numpy's pairwise sum of n < 128 values (8 accumulators), then / n
template <class T>
__device__ __forceinline__ T np_mean(const T* a, int n) {
#pragma clang fp contract(off)
    T r;
    if (n < 8) {
        r = T(0);
        for (int i = 0; i < n; i++) r = r + a[i];
    } else {
        T q[8];
        for (int j = 0; j < 8; j++) q[j] = a[j];
        int i = 8;
        for (; i < n - (n % 8); i += 8)
            for (int j = 0; j < 8; j++) q[j] = q[j] + a[i + j];
        r = ((q[0] + q[1]) + (q[2] + q[3])) + ((q[4] + q[5]) + (q[6] + q[7]));
        for (; i < n; i++) r = r + a[i];
    }
    return r / (T)n;
}

// The same by a wavefront, the 8 accumulators on lanes 0..7 (every lane of the
// wavefront calls it); the mean on lane 0.
template <class T>
__device__ __forceinline__ T np_mean_wave(const T* a, int n, int lane) {
#pragma clang fp contract(off)
    if (n < 8) return np_mean(a, n);
    const int j = lane & 7;
    T q = a[j];
    int i = 8;
    for (; i < n - (n % 8); i += 8) q = q + a[i + j];
    for (int o = 1; o < 8; o <<= 1) q = q + __shfl_xor(q, o);
    for (; i < n; i++) q = q + a[i];
    return q / (T)n;
}

// pidw_base.py _cyclic_feature_to_index: float32 arctan2 (rounded from
// float64), + 2 pi when negative, floor(period * angle / (2 pi)) in float32
__device__ __forceinline__ int cyclic(float s, float c, int period) {
#pragma clang fp contract(off)
    float ang = (float)atan2((double)s, (double)c);
    if (ang < 0.0f) ang = ang + (float)(2.0 * 3.141592653589793);
    const float v = ((float)period * ang) / (float)(2.0 * 3.141592653589793);
    return (int)floorf(v);
}

__device__ __forceinline__ double clipd(double x, double lo, double hi) { return x < lo ? lo : (x > hi ? hi : x); }

// One workgroup of 4 wavefronts per env. What bounds it is the chain of its
// phases' latencies, so everything it reads goes out in one burst (the
// observation row and its native values to LDS, each thread's own indices to
// registers): wavefronts 0 and 1 take a zone slot per lane (its command, its
// trust, its 9 features), wavefront 2 an AHU per lane (PID, 16 features),
// wavefront 3 the hot-water loop and the global features; the observation row
// is put together in LDS and written in one piece. 42 us as one wavefront
// that looked each feature's fields up in turn, 8 us so (300 envs of 81
// zones on 9 AHUs).
constexpr int kPostThreads = 256;
__global__ __launch_bounds__(kPostThreads) void canon_post_kernel(CanonArgs A) {
#pragma clang fp contract(off)
    const int e = blockIdx.x, tid = (int)threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if (e >= A.n) return;
    const CanonTab& C = A.tabs[A.envs[e].layout];
    const float* o = A.raw_obs + (size_t)e * SB_OBS;
    // so: the env's observation; sn: its native values, then a zero for absent fields
    __shared__ float so[SB_OBS], sn[SB_OBS + 1], sr[SB_OBS];
    __shared__ float sb[SB_ACT], sw[SB_ACT], sT[SBC_ZS], st[SBC_ZS], sai[2 * SBC_K], swk[SBC_K], s32[SBC_ZS];
    __shared__ double spid[2 * SBC_K], seff[SBC_K], s64[SBC_ZS];
    __shared__ int sact[SBC_K], sheat[SBC_K], scold;
    const bool fresh = A.reset || A.terminals[e] == 1.0f;   // a new episode starts here
#pragma unroll
    for (int q = 0; q < SB_OBS / kPostThreads; q++) {
        const int i = q * kPostThreads + tid;
        const float x = o[i];
        so[i] = x;
        sn[i] = x * C.fstd[i] + C.fmean[i];
        sr[i] = 0.0f;
    }
    for (int i = tid; i < SB_ACT; i += kPostThreads) {
        sb[i] = 0.0f;
        sw[i] = 1.0f;
    }
    if (tid < 2 * SBC_K) {
        spid[tid] = fresh ? 0.0 : A.pid[(size_t)e * 2 * SBC_K + tid];
        sai[tid] = 0.0f;
    }
    if (tid == 0) {
        sn[SB_OBS] = 0.0f;
        scold = 1;
    }
    const int s = tid < SBC_ZS ? tid : 0;   // wavefronts 0 and 1: this lane's zone slot
    const int zT = tid < SBC_ZS ? C.zT[s] : -1, zAd = C.zAd[s], zAr = C.zAr[s];
    const int zH = C.zH[s], zC = C.zC[s], zD = C.zD[s], zR = C.zR[s];
    int zpos = s % SBC_ZPA, ns = 0;         // its place among the building's zones, and their number
#pragma unroll
    for (int k = 0; k < SBC_K; k++) {
        const int z = k < C.K ? C.zc[k] : 0;
        if (k < s / SBC_ZPA) zpos += z;
        ns += z;
    }
    const int ka = lane < SBC_K ? lane : 0;   // wavefront 2: this lane's AHU
    int aq[8];
#pragma unroll
    for (int m = 0; m < 8; m++) aq[m] = C.aObs[ka][m];
    const int aT = C.aT[ka], aP = C.aP[ka], aRec = C.aRec[ka], aRun = C.aRun[ka], azc = C.zc[ka];
    const int hW = C.hW, hDPa = C.hDPa, hRun = C.hRun;
    // hour of the day on even lanes, day of the week on odd ones
    const int g0 = max(C.g[(lane & 1) * 8], 0), g1 = max(C.g[(lane & 1) * 8 + 4], 0);
    __syncthreads();
    auto nat = [&](int i) { return sn[i >= 0 ? i : SB_OBS]; };
    const int cyc = cyclic(so[g0], so[g1], (lane & 1) ? 7 : 24);
    const int hour = __builtin_amdgcn_readlane(cyc, 0), day = __builtin_amdgcn_readlane(cyc, 1);
    const bool work = day < 5 && C.morning <= hour && hour < C.evening;
    const double lo = work ? C.comfort_lo : C.eco_lo, hi = work ? C.comfort_hi : C.eco_hi;
    const float lof = (float)lo, hif = (float)hi;
    // zone commands (PIDProportionalReheatPolicy._command_zones) and the
    // guard's trust per zone
    if (zT >= 0) {
        const float T = so[zT] * C.tstd + C.tmean;
        sT[s] = T;
        float err = 0.0f;
        if (T < lof) err = lof - T;
        else if (T > hif) err = hif - T;
        const float damper = fminf(1.0f, fabsf(err) / 2.0f);
        if (zAd >= 0) sb[zAd] = 2.0f * damper - 1.0f;
        const float opening = fminf(1.0f, fmaxf(0.0f, err) / 2.0f);
        if (zAr >= 0) sb[zAr] = 2.0f * opening - 1.0f;
        if (A.guard) {
            const float dev = T < lof ? lof - T : (A.hot && T > hif ? T - hif : 0.0f);
            const float t = fminf(1.0f, fmaxf(0.0f, 1.0f - (dev - A.d0) / A.d1));
            st[s] = t;
            if (zAd >= 0) sw[zAd] = t;
            if (zAr >= 0) sw[zAr] = t;
        }
        // the zones' shortfalls in order, for the hot-water reset
        const float d = lof - T;
        s32[zpos] = d;
        s64[zpos] = d > 0.0f ? (double)d : 0.0;
        if (!(d > 0.0f)) scold = 0;
    }
    __syncthreads();
    // one lane per AHU: its PID loop on the mean zone temperature, fan
    // pressure, run command and economiser (PIDWorstZonePolicy.get_action with
    // PIDEconomizerPolicy's average-zone error and recirculation)
    if (wave == 2 && lane < C.K) {
        const int k = lane, nz = azc;
        sact[k] = 0;
        sheat[k] = 0;
        seff[k] = 0.0;
        if (aRec >= 0) sb[aRec] = 1.0f;
        if (nz > 0) {
            const double avg = (double)np_mean<float>(sT + SBC_ZPA * k, nz);
            sai[2 * k + 1] = (float)avg;
            double error = 0.0;
            if (avg < lo) error = lo - avg;
            else if (avg > hi) error = hi - avg;
            double* ps = spid + 2 * k;
            if (error == 0.0) {
                ps[0] = ps[0] * 0.5;
                ps[1] = 0.0;
                if (aT >= 0) sb[aT] = -1.0f;
                if (aP >= 0) sb[aP] = -1.0f;
                if (aRun >= 0) sb[aRun] = 0.0f;
            } else {
                ps[0] = clipd(ps[0] + error, -10.0, 10.0);
                const double deriv = error - ps[1];
                ps[1] = error;
                const double u = clipd(0.5 * error + 0.02 * ps[0] + 0.1 * deriv, -1.0, 1.0);
                sai[2 * k] = (float)u;
                seff[k] = u;
                sact[k] = 1;
                sheat[k] = error > 0.0;
                const double pressure = clipd(2.0 * fabs(u) - 1.0, -1.0, 1.0);
                if (aT >= 0) sb[aT] = (float)u;
                if (aP >= 0) sb[aP] = (float)pressure;
                if (aRun >= 0) sb[aRun] = 1.0f;
                if (aRec >= 0) {
                    double rec = 1.0;
                    if (!(u >= 0.0) && aq[0] >= 0) {
                        const double outside = (double)so[aq[0]], inside = avg;
                        if (isfinite(outside) && !(outside >= inside)) {
                            double pa = (pressure + 1.0) * 0.5 * 2000.0;
                            pa = pa > 200.0 ? pa : 200.0;
                            if (!(inside - outside <= pa * 0.00322)) {
                                double target = 285.0 + (u + 1.0) * 0.5 * 20.0;
                                target = target > lo ? target : lo;
                                if (!(inside <= target)) {
                                    const double f = (inside - target) / (inside - outside);
                                    rec = 2.0 * clipd(1.0 - f, 0.0, 1.0) - 1.0;
                                }
                            }
                        }
                    }
                    sb[aRec] = (float)rec;
                }
            }
        }
        if (A.guard) {
            float wk = 1.0f;
            for (int j = 0; j < nz; j++) wk = fminf(wk, st[SBC_ZPA * k + j]);
            if (aT >= 0) sw[aT] = wk;
            if (aP >= 0) sw[aP] = wk;
            if (aRec >= 0) sw[aRec] = wk;
            if (aRun >= 0) sw[aRun] = wk;
            swk[k] = wk;
        }
    }
    // zone features (residual_policy.py _features), beside the AHUs
    if (zT >= 0) {
        const float T = nat(zT), Hs = nat(zH), Cs = nat(zC);
        float* r = sr + SBC_FZ * s;
        r[0] = 1.0f;
        r[1] = (T - 295.0f) / 5.0f;
        r[2] = (T - Hs) / 2.0f;
        r[3] = (Cs - T) / 2.0f;
        r[4] = (Hs - 294.0f) / 3.0f;
        r[5] = zD >= 0 ? 2.0f * nat(zD) - 1.0f : 0.0f;
        r[6] = zR >= 0 ? 2.0f * nat(zR) - 1.0f : 0.0f;
        r[7] = zAd >= 0 ? sb[zAd] : 0.0f;
        r[8] = zAr >= 0 ? sb[zAr] : 0.0f;
    }
    __syncthreads();
    if (wave == 3) {
        // the hot-water loop (PIDPolicy's water actions, then
        // PIDWaterResetPolicy's reset: the greater of the mean zone shortfall
        // over 4 K and the 0.25 quantile of the AHUs' heating effort)
        const bool mine = lane < C.K;
        const bool act = mine && sact[ka] != 0;
        const unsigned long long acts = __ballot(act);
        const bool any_act = acts != 0ull, any_heat = __ballot(mine && sheat[ka] != 0) != 0ull;
        float water = any_heat ? 1.0f : -1.0f;
        if (hW >= 0 && any_heat) {
            // a shortfall of 0 is a Python 0.0 in the reference's list, which
            // makes numpy's mean float64; with none the mean is float32
            double shortfall = 0.0;
            if (ns > 0) shortfall = scold ? (double)np_mean_wave<float>(s32, ns, lane) : np_mean_wave<double>(s64, ns, lane);
            const double demand = shortfall / 4.0;
            double sat = 0.0;
            const int ne = __popcll(acts);
            if (ne > 0) {
                // numpy quantile, method linear: virtual index (n - 1) q, numpy's
                // _lerp; the sorted efforts by their ranks
                const double h = act && seff[ka] > 0.0 ? seff[ka] : 0.0;
                int rank = 0;
#pragma unroll
                for (int k = 0; k < SBC_K; k++) {
                    const double x = __shfl(h, k);
                    if ((acts >> k) & 1ull) rank += x < h || (x == h && k < lane);
                }
                const double vi = (double)(ne - 1) * 0.25;
                int i0 = (int)floor(vi), i1 = i0 + 1;
                if (vi >= (double)(ne - 1)) i0 = i1 = ne - 1;
                const double h0 = __shfl(h, __ffsll((long long)__ballot(act && rank == i0)) - 1);
                const double h1 = __shfl(h, __ffsll((long long)__ballot(act && rank == i1)) - 1);
                const double t = vi - floor(vi);
                const double diff = h1 - h0;
                sat = t >= 0.5 ? h1 - diff * (1.0 - t) : h0 + diff * t;
            }
            const double m = demand > sat ? demand : sat;
            water = (float)(2.0 * clipd(m + 0.0, 0.0, 1.0) - 1.0);
        }
        if (lane == 0) {
            if (hW >= 0) sb[hW] = water;
            if (hDPa >= 0) sb[hDPa] = any_act ? 1.0f : -1.0f;
            if (hRun >= 0) sb[hRun] = any_act ? 1.0f : 0.0f;
            if (A.guard) {
                float wb = 1.0f;
                for (int k = 0; k < C.K; k++) wb = fminf(wb, swk[k]);
                if (hW >= 0) sw[hW] = wb;
                if (hDPa >= 0) sw[hDPa] = wb;
                if (hRun >= 0) sw[hRun] = wb;
            }
            const int* q = C.hObs;
            float* r = sr + SBC_OH;
            r[0] = 1.0f;
            r[1] = (nat(q[0]) - 330.0f) / 20.0f;
            r[2] = (nat(q[1]) - 330.0f) / 20.0f;
            r[3] = nat(q[2]) / 10.0f;
            r[4] = nat(q[3]) / 10.0f;
            r[5] = 2.0f * nat(q[4]) - 1.0f;
            r[6] = nat(q[5]) / 10.0f;
            r[7] = hW >= 0 ? sb[hW] : 0.0f;
            r[8] = hDPa >= 0 ? sb[hDPa] : 0.0f;
            r[9] = hRun >= 0 ? 2.0f * sb[hRun] - 1.0f : 0.0f;
        }
        if (lane < SBC_FG) {
            const int i = C.g[lane];
            sr[SBC_OG + lane] = i >= 0 ? so[i] : 0.0f;
        }
    } else if (wave == 2 && lane < C.K) {
        const int k = lane;
        float* r = sr + SBC_OA + SBC_FA * k;
        r[0] = 1.0f;
        r[1] = (nat(aq[0]) - 283.0f) / 15.0f;
        r[2] = nat(aq[1]) / 1000.0f;
        r[3] = nat(aq[2]) / 10.0f;
        r[4] = nat(aq[3]) / 10.0f;
        r[5] = aq[4] >= 0 ? (nat(aq[4]) - 295.0f) / 5.0f : 0.0f;
        r[6] = 2.0f * nat(aq[5]) - 1.0f;
        r[7] = nat(aq[6]) / 10.0f;
        r[8] = 2.0f * nat(aq[7]) - 1.0f;
        r[9] = aT >= 0 ? sb[aT] : 0.0f;
        r[10] = aP >= 0 ? sb[aP] : 0.0f;
        r[11] = aRec >= 0 ? sb[aRec] : 0.0f;
        r[12] = aRun >= 0 ? 2.0f * sb[aRun] - 1.0f : 0.0f;
        r[13] = azc > 0 ? (sai[2 * k + 1] - 295.0f) / 5.0f : 0.0f;
        r[14] = (float)(spid[2 * k] / 10.0);
        r[15] = sai[2 * k];
    }
    __syncthreads();
    for (int i = tid; i < SB_ACT; i += kPostThreads) {
        A.base[(size_t)e * SB_ACT + i] = sb[i];
        A.trust[(size_t)e * SB_ACT + i] = sw[i];
    }
    if (tid < 2 * SBC_K) {
        A.pid[(size_t)e * 2 * SBC_K + tid] = spid[tid];
        A.ainfo[(size_t)e * 2 * SBC_K + tid] = sai[tid];
    }
    // the padding past the canonical features is zeroed by a reset only
    float* out = A.obs + (size_t)e * SB_OBS;
    for (int f = tid; f < (A.reset ? SB_OBS : SBC_OBS); f += kPostThreads) out[f] = sr[f];
}

__global__ __launch_bounds__(64) void canon_pre_kernel(CanonArgs A) {
#pragma clang fp contract(off)
    const int e = blockIdx.x, lane = (int)threadIdx.x;
    if (e >= A.n) return;
    const CanonTab& C = A.tabs[A.envs[e].layout];
    const float* prow = A.actions + (size_t)e * SB_ACT;
    float* row = A.native + (size_t)e * SB_ACT;
    for (int col = lane; col < SB_ACT; col += 64) {
        const int i = C.act_of_col[col];
        float v = 0.0f;
        if (i >= 0) {
            const int sl = C.slot_of_action[i];
            float p = 0.0f;
            if (sl >= 0) {
                p = prow[sl];
                p = isfinite(p) ? fminf(1.0f, fmaxf(-1.0f, p)) : 0.0f;
                if (A.guard) p = p * A.trust[(size_t)e * SB_ACT + i];
            }
            const float b = A.base[(size_t)e * SB_ACT + i];
            if (C.act_disc[i]) {
                const bool on = A.resid ? (2.0f * b - 1.0f) + A.dscale * p > 0.0f : p > -0.5f;
                v = on ? 1.0f : 0.0f;
            } else {
                const float m = A.resid ? b + A.scale * p : p;
                v = fminf(1.0f, fmaxf(-1.0f, m));
            }
        }
        row[col] = v;
    }
}

}  // namespace sbk

extern "C" int sbk_launch_canon(const sbk::CanonArgs* a, int post, hipStream_t s) {
    if (a->n <= 0) return (int)hipErrorInvalidValue;
    if (post) hipLaunchKernelGGL(sbk::canon_post_kernel, dim3(a->n), dim3(sbk::kPostThreads), 0, s, *a);
    else hipLaunchKernelGGL(sbk::canon_pre_kernel, dim3(a->n), dim3(64), 0, s, *a);
    return (int)hipGetLastError();
}
