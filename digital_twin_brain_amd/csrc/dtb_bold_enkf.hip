// dtb_bold_enkf.hip -- Balloon-Windkessel BOLD step and the diffusion EnKF
// analysis on device arrays.
#include <algorithm>
#include <cmath>
#include <mutex>

#include "dtb_internal.hpp"

namespace dtb {

// models/bold_model_pytorch.py:69-77, in the reference's update order:
// d_s from the old s and f_in; q and v from the old f_in, q, v; f_in += s dt
// with the old s, clamped at 0; s += d_s dt; output from the new q, v.
template <typename T>
__global__ void bold_kernel(int64_t n, T eps, T ts, T tf, T t0, T div_alpha, T E0, T V0, T dt, T* __restrict__ s,
                            T* __restrict__ q, T* __restrict__ v, T* __restrict__ f, const T* __restrict__ u,
                            T* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const T si = s[i], qi = q[i], vi = v[i], fi = f[i];
    const T d_s = eps * u[i] - si / ts - (fi - T(1)) / tf;
    const T q_part = fi > T(0) ? T(1) - pow(T(1) - E0, T(1) / fi) : T(1);
    const T qn = qi + (fi * q_part / E0 - qi * pow(vi, div_alpha - T(1))) / t0 * dt;
    const T vn = vi + (fi - pow(vi, div_alpha)) / t0 * dt;
    T fn = fi + si * dt;
    fn = fn > T(0) ? fn : T(0);
    const T sn = si + d_s * dt;
    s[i] = sn;
    q[i] = qn;
    v[i] = vn;
    f[i] = fn;
    out[i] = V0 * (T(7) * E0 * (T(1) - qn) + T(2) * (T(1) - qn / vn) + (T(2) * E0 - T(0.2)) * (T(1) - vn));
}

// `steps` consecutive steps of bold_kernel with a constant input per voxel,
// the state kept in registers: the same per-step arithmetic in the same order.
__global__ void bold_run_kernel(int64_t n, int32_t steps, double eps, double ts, double tf, double t0,
                                double div_alpha, double E0, double V0, double dt, double* __restrict__ s,
                                double* __restrict__ q, double* __restrict__ v, double* __restrict__ f,
                                const double* __restrict__ u, double* __restrict__ out)
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    double si = s[i], qi = q[i], vi = v[i], fi = f[i];
    const double ui = u[i];
    double o = out[i];
    for (int32_t k = 0; k < steps; ++k) {
        const double d_s = eps * ui - si / ts - (fi - 1.0) / tf;
        const double q_part = fi > 0.0 ? 1.0 - pow(1.0 - E0, 1.0 / fi) : 1.0;
        const double qn = qi + (fi * q_part / E0 - qi * pow(vi, div_alpha - 1.0)) / t0 * dt;
        const double vn = vi + (fi - pow(vi, div_alpha)) / t0 * dt;
        double fn = fi + si * dt;
        fn = fn > 0.0 ? fn : 0.0;
        si = si + d_s * dt;
        qi = qn;
        vi = vn;
        fi = fn;
        o = V0 * (7.0 * E0 * (1.0 - qn) + 2.0 * (1.0 - qn / vn) + (2.0 * E0 - 0.2) * (1.0 - vn));
    }
    s[i] = si;
    q[i] = qi;
    v[i] = vi;
    f[i] = fi;
    out[i] = o;
}

template <typename T>
static int bold_step(int64_t n, const double* par, T* s, T* q, T* v, T* f, const T* u, T* out, void* stream)
{
    DTB_REQUIRE(n >= 0, "n must be >= 0");
    DTB_REQUIRE(par != nullptr, "par is NULL");
    if (n == 0) return DTB_OK;
    DTB_REQUIRE(s && q && v && f && u && out, "state, input and output arrays are required");
    hipLaunchKernelGGL(bold_kernel<T>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n,
                       (T)par[0], (T)par[1], (T)par[2], (T)par[3], (T)(1.0 / par[4]), (T)par[5], (T)par[6], (T)par[7],
                       s, q, v, f, u, out);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

// ------------------------------------------------------------------- EnKF
// data_assimilation/DataAssimilation.py:40-60.  w[E][V][S], last state =
// BOLD.  wd = w - mean_e(w); c_v = sum_e wd_ev^2/(E-1) + sigma;
// K_ev = wd_ev(last)/c_v/(E-1); innov_ev = y_v + sqrt(sigma) xi_ev - w_ev(last)
// w += rho innov_ev sum_e' K_e'v wd_e'vs + (1-rho) sum_e' A_ee' wd_e'vs,
// A_ee' = sum_v innov_ev K_e'v / V.
//
// Two kernels, both bound by latency at the sizes of an assimilation window
// (256 members, 90 voxels, 10 states: 1.8 MB and 0.13 GFLOP), so the work is
// spread until no thread walks a long chain of dependent loads:
//   enkf_voxel_kernel   one workgroup per voxel, one wavefront per state with
//                       its lanes over the members: ensemble mean,
//                       deviations, gain, innovation and the local term, all
//                       sums of one voxel, with one barrier (the gains)
//   enkf_update_kernel  one workgroup per 16 members x 64 CT states: its 16
//                       rows of A from the innovations and gains, then the
//                       global term A wd, both on the FP64 matrix cores
// 256 x 90 x 10: 9.4 + 17 us.  (Six launches with a thread per output element,
// each summing over the members or voxels by itself, took 394 us.)
constexpr int kEnkfWaves = 16;        // wavefronts of the voxel kernel
constexpr int kEnkfLdsMembers = 4096; // members whose gains stay in LDS (larger ensembles re-read them)
constexpr int kEnkfRegs = 8;          // members per lane held in registers (up to 512 members)
typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ inline double wave_sum_f64(double v)
{
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
    return v;
}

// HELD: at most kEnkfWaves states and 64 kEnkfRegs members, so each wavefront
// keeps its one state's deviations in registers; else they are read again
// from wd.  GLDS: the gains are exchanged through LDS, else through tempT.
template <bool HELD, bool GLDS>
__global__ __launch_bounds__(64 * kEnkfWaves) void enkf_voxel_kernel(int32_t E, int32_t V, int32_t S,
                                                                     const double* __restrict__ w, double sigma,
                                                                     const double* __restrict__ y,
                                                                     const double* __restrict__ xi, double* wd,
                                                                     double* tempT, double* __restrict__ innovT,
                                                                     double* __restrict__ gsum)
{
    extern __shared__ double s_gain[]; // [E] gains
    const int32_t v = blockIdx.x;
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int64_t VS = (int64_t)V * S;
    double* tv = tempT + (int64_t)v * E;
    double* iv = innovT + (int64_t)v * E;
    double* gain = GLDS ? s_gain : tv;
    double d[kEnkfRegs];
    for (int32_t s = wid; s < S; s += kEnkfWaves) {
        const double* src = w + (int64_t)v * S + s;
        double* dst = wd + (int64_t)v * S + s;
        const bool last = s == S - 1;
        double noise[kEnkfRegs];
        double a = 0.0;
        if (HELD) {
#pragma unroll
            for (int k = 0; k < kEnkfRegs; ++k) {
                const int32_t e = lane + 64 * k;
                d[k] = e < E ? src[e * VS] : 0.0;
                noise[k] = last && e < E ? xi[(int64_t)e * V + v] : 0.0;
            }
#pragma unroll
            for (int k = 0; k < kEnkfRegs; ++k) a += d[k];
        } else {
#pragma unroll 8
            for (int32_t e = lane; e < E; e += 64) a += src[e * VS];
        }
        const double mean = wave_sum_f64(a) / E;
        double q = 0.0;
        const double yv = y[v], sq = sqrt(sigma);
        if (HELD) {
#pragma unroll
            for (int k = 0; k < kEnkfRegs; ++k) {
                const int32_t e = lane + 64 * k;
                if (e >= E) continue;
                if (last) iv[e] = yv + sq * noise[k] - d[k];
                d[k] -= mean;
                dst[e * VS] = d[k];
                q += d[k] * d[k];
            }
        } else {
#pragma unroll 4
            for (int32_t e = lane; e < E; e += 64) {
                const double x = src[e * VS], dx = x - mean;
                dst[e * VS] = dx;
                q += dx * dx;
                if (last) iv[e] = yv + sq * xi[(int64_t)e * V + v] - x;
            }
        }
        if (last) {
            const double c = wave_sum_f64(q) / (E - 1) + sigma;
            if (HELD) {
#pragma unroll
                for (int k = 0; k < kEnkfRegs; ++k) {
                    const int32_t e = lane + 64 * k;
                    if (e >= E) continue;
                    const double g = d[k] / c / (E - 1);
                    gain[e] = g;
                    if (GLDS) tv[e] = g;
                }
            } else {
                for (int32_t e = lane; e < E; e += 64) {
                    const double g = dst[e * VS] / c / (E - 1);
                    gain[e] = g;
                    if (GLDS) tv[e] = g;
                }
            }
        }
    }
    __syncthreads();
    for (int32_t s = wid; s < S; s += kEnkfWaves) {
        double a = 0.0;
        if (HELD) {
#pragma unroll
            for (int k = 0; k < kEnkfRegs; ++k)
                if (lane + 64 * k < E) a += gain[lane + 64 * k] * d[k];
        } else {
            const double* src = wd + (int64_t)v * S + s; // this lane's own stores
#pragma unroll 8
            for (int32_t e = lane; e < E; e += 64) a += gain[e] * src[e * VS];
        }
        a = wave_sum_f64(a);
        if (lane == 0) gsum[(int64_t)v * S + s] = a;
    }
}

// w += rho innov gsum + (1 - rho) A wd, A_ef = sum_v innov_ev temp_fv / V.
// A workgroup of four wavefronts takes 16 members (blockIdx.y) and 64 CT
// columns of wd (blockIdx.x).  It computes its 16 rows of A, kEnkfChunk
// members f at a time, into LDS and multiplies them with wd: every workgroup
// of a row repeats that small product (E x V x 16), which costs less than a
// launch between the two.  v_mfma_f64_16x16x4: lane l holds A[l % 16][l / 16]
// and B[l / 16][l % 16]; register r of the result is D[4 r + l / 16][l % 16].
// The chains of loads bound it, so they are issued in batches ahead of the
// products: all of a chunk's wd values (CT = 1) before its A is computed, and
// the gains eight steps at a time.
// CT = 1 while the workgroups then still fit the device about twice (the
// columns' loads spread over more of them), else 4 (A repeated less often).
constexpr int kEnkfChunk = 256;
constexpr int kEnkfBatch = 8;            // steps of four voxels whose loads are in flight together
constexpr int kEnkfRow = kEnkfChunk + 4; // LDS row: 16 rows x 4 columns of a fragment fall on distinct banks

template <int CT>
__global__ __launch_bounds__(256) void enkf_update_kernel(int32_t E, int32_t V, int32_t S, double rho,
                                                          const double* __restrict__ wd,
                                                          const double* __restrict__ tempT,
                                                          const double* __restrict__ innovT,
                                                          const double* __restrict__ gsum, double* __restrict__ w)
{
    __shared__ double sA[16 * kEnkfRow];
    __shared__ double sR[3][256]; // partial tiles of A
    const int wid = threadIdx.x >> 6, lane = threadIdx.x & 63;
    const int lr = lane & 15, lk = lane >> 4;
    const int64_t VS = (int64_t)V * S;
    const int32_t e0 = blockIdx.y * 16;
    const int64_t x0 = ((int64_t)blockIdx.x * 4 + wid) * 16 * CT;
    f64x4 acc[CT];
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[j] = f64x4{0.0, 0.0, 0.0, 0.0};
    const int32_t er = min(e0 + lr, E - 1); // rows and columns past the edge repeat the last one and are not stored
    for (int32_t f0 = 0; f0 < E; f0 += kEnkfChunk) {
        const int32_t nf = min(kEnkfChunk, E - f0);
        double bv[CT == 1 ? kEnkfChunk / 4 : 1];
        if (CT == 1) {
            const int64_t x = min(x0 + lr, VS - 1);
#pragma unroll
            for (int k = 0; k < kEnkfChunk / 4; ++k)
                bv[k] = 4 * k + lk < nf ? wd[(int64_t)(f0 + 4 * k + lk) * VS + x] : 0.0;
        }
        // columns f0 .. f0 + nf of A; wavefront wid takes the 16-column tiles wid, wid + 4, ...
        f64x4 a4[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) a4[j] = f64x4{0.0, 0.0, 0.0, 0.0};
        // With one or two tiles (32 members or fewer) four or two wavefronts
        // share each, a range of voxels apiece: what is left then is the chain
        // of loads over the voxels (a call of 2 members x 2,000 voxels x 10: 342
        // -> 92 us, 207 in six launches).
        const int nt = (nf + 15) / 16;
        const int parts = nt == 1 ? 4 : nt == 2 ? 2 : 1;
        if (parts > 1) { // uniform
            const int tile = wid % nt, part = wid / nt;
            const int32_t per = ((V + parts - 1) / parts + 3) / 4 * 4;
            const int32_t vend = min(V, (part + 1) * per), f = f0 + tile * 16 + lr;
            for (int32_t v0 = part * per; v0 < vend; v0 += 4 * kEnkfBatch) {
                double in[kEnkfBatch], tv[kEnkfBatch];
#pragma unroll
                for (int u = 0; u < kEnkfBatch; ++u) {
                    const int32_t v = v0 + 4 * u + lk;
                    const int64_t row = (int64_t)min(v, V - 1) * E;
                    in[u] = v < vend ? innovT[row + er] : 0.0;
                    tv[u] = v < vend && f < E ? tempT[row + f] : 0.0;
                }
#pragma unroll
                for (int u = 0; u < kEnkfBatch; ++u)
                    a4[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(in[u], tv[u], a4[0], 0, 0, 0);
            }
            double* red = sR[nt == 1 ? max(part - 1, 0) : tile];
            if (part > 0) {
#pragma unroll
                for (int r = 0; r < 4; ++r) red[r * 64 + lane] = a4[0][r];
            }
            __syncthreads(); // and the chunk before has been used
            if (part == 0) {
                for (int q = 1; q < parts; ++q)
#pragma unroll
                    for (int r = 0; r < 4; ++r) a4[0][r] += sR[nt == 1 ? q - 1 : tile][r * 64 + lane];
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    sA[(4 * r + lk) * kEnkfRow + tile * 16 + lr] = f < E ? a4[0][r] / V : 0.0;
            }
        }
        for (int32_t v0 = 0; parts == 1 && v0 < V; v0 += 4 * kEnkfBatch) {
            double in[kEnkfBatch], tv[kEnkfBatch][4];
#pragma unroll
            for (int u = 0; u < kEnkfBatch; ++u) {
                const int32_t v = v0 + 4 * u + lk;
                const int64_t row = (int64_t)min(v, V - 1) * E;
                const bool ok = v < V;
                in[u] = ok ? innovT[row + er] : 0.0;
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const int32_t f = f0 + (wid + 4 * j) * 16 + lr;
                    tv[u][j] = ok && f < E ? tempT[row + f] : 0.0; // columns past the last member are zero
                }
            }
#pragma unroll
            for (int u = 0; u < kEnkfBatch; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j)
                    a4[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(in[u], tv[u][j], a4[j], 0, 0, 0);
        }
        if (parts == 1 && f0 > 0) __syncthreads(); // the chunk before has been used
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int r = 0; r < 4 && parts == 1; ++r) {
                const int fl = (wid + 4 * j) * 16 + lr;
                sA[(4 * r + lk) * kEnkfRow + fl] = f0 + fl < E ? a4[j][r] / V : 0.0;
            }
        __syncthreads();
        if (CT == 1) {
#pragma unroll
            for (int k = 0; k < kEnkfChunk / 4; ++k) {
                if (4 * k >= nf) break; // uniform
                acc[0] = __builtin_amdgcn_mfma_f64_16x16x4f64(sA[lr * kEnkfRow + 4 * k + lk], bv[k], acc[0], 0, 0, 0);
            }
        } else {
#pragma unroll 8
            for (int32_t f = 0; f < nf; f += 4) {
                const double av = sA[lr * kEnkfRow + f + lk];
                const bool ok = f + lk < nf;
                const double* src = wd + (int64_t)(f0 + (ok ? f + lk : 0)) * VS;
                double b4[CT];
#pragma unroll
                for (int j = 0; j < CT; ++j) b4[j] = ok ? src[min(x0 + 16 * j + lr, VS - 1)] : 0.0;
#pragma unroll
                for (int j = 0; j < CT; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av, b4[j], acc[j], 0, 0, 0);
            }
        }
    }
#pragma unroll
    for (int j = 0; j < CT; ++j) {
        const int64_t x = x0 + 16 * j + lr;
        if (x >= VS) continue;
        const int64_t v = x / S;
        const double gs = gsum[x];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int32_t e = e0 + 4 * r + lk;
            if (e < E) w[e * VS + x] += rho * innovT[v * E + e] * gs + (1.0 - rho) * acc[j][r];
        }
    }
}

// The analysis on a caller-chosen scratch of enkf_scratch_doubles doubles:
// wd [E*V*S], the gains and innovations of each voxel [V*E] and gsum [V*S].
// Every scratch element is written before it is read.
static size_t enkf_scratch_doubles(int32_t E, int32_t V, int32_t S)
{
    const size_t EVS = (size_t)E * V * S, VS = (size_t)V * S, EV = (size_t)E * V;
    return EVS + 2 * EV + VS;
}

static int enkf_launch(int32_t E, int32_t V, int32_t S, double* w, double sigma, const double* y, double rho,
                       const double* xi, hipStream_t st, double* scratch)
{
    const size_t EVS = (size_t)E * V * S, VS = (size_t)V * S, EV = (size_t)E * V;
    double* wd = scratch;
    double* tempT = wd + EVS;
    double* innovT = tempT + EV;
    double* gsum = innovT + EV;
    const dim3 vt(64 * kEnkfWaves);
    if (E <= 64 * kEnkfRegs && S <= kEnkfWaves)
        hipLaunchKernelGGL((enkf_voxel_kernel<true, true>), dim3((unsigned)V), vt, sizeof(double) * (size_t)E, st, E, V,
                           S, w, sigma, y, xi, wd, tempT, innovT, gsum);
    else if (E <= kEnkfLdsMembers)
        hipLaunchKernelGGL((enkf_voxel_kernel<false, true>), dim3((unsigned)V), vt, sizeof(double) * (size_t)E, st, E,
                           V, S, w, sigma, y, xi, wd, tempT, innovT, gsum);
    else
        hipLaunchKernelGGL((enkf_voxel_kernel<false, false>), dim3((unsigned)V), vt, 0, st, E, V, S, w, sigma, y, xi,
                           wd, tempT, innovT, gsum);
    const size_t rows = ((size_t)E + 15) / 16;
    if (rows * ((VS + 63) / 64) <= 512)
        hipLaunchKernelGGL(enkf_update_kernel<1>, dim3((unsigned)((VS + 63) / 64), (unsigned)rows), dim3(256), 0, st, E,
                           V, S, rho, wd, tempT, innovT, gsum, w);
    else
        hipLaunchKernelGGL(enkf_update_kernel<4>, dim3((unsigned)((VS + 255) / 256), (unsigned)rows), dim3(256), 0, st,
                           E, V, S, rho, wd, tempT, innovT, gsum, w);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

// Scratch for the analysis, kept per device and grown on demand.
struct EnkfScratch {
    double* p = nullptr;
    size_t cap = 0;
};
static std::mutex g_enkf_mu;
static EnkfScratch g_enkf[64];

static int enkf(int32_t E, int32_t V, int32_t S, double* w, double sigma, const double* y, double rho,
                const double* xi, void* stream)
{
    DTB_REQUIRE(E >= 2 && V >= 1 && S >= 1, "EnKF needs E >= 2, V >= 1, S >= 1");
    DTB_REQUIRE(w && y && xi, "w, y and xi are required");
    int dev = 0;
    DTB_TRY_HIP(hipGetDevice(&dev));
    DTB_REQUIRE(dev >= 0 && dev < 64, "device index out of range");
    const size_t need = enkf_scratch_doubles(E, V, S);
    std::lock_guard<std::mutex> lk(g_enkf_mu);
    EnkfScratch& sc = g_enkf[dev];
    if (sc.cap < need) {
        if (sc.p) {
            DTB_TRY_HIP(hipDeviceSynchronize());
            DTB_TRY_HIP(hipFree(sc.p));
        }
        sc.p = nullptr;
        sc.cap = 0;
        DTB_TRY_HIP(hipMalloc(&sc.p, need * sizeof(double)));
        sc.cap = need;
    }
    hipStream_t st = (hipStream_t)stream;
    DTB_TRY(enkf_launch(E, V, S, w, sigma, y, rho, xi, st, sc.p));
    // the scratch is shared by later calls on this device
    DTB_TRY_HIP(hipStreamSynchronize(st));
    return DTB_OK;
}

// Allocation-free analysis: the scratch is a fixed device array, one copy per
// GPU, held until the process ends.  Its host-side name is not a device
// address, so each device's address comes from hipGetSymbolAddress, taken
// once per device with that device current, and only that address is handed
// to the kernels.
constexpr size_t kEnkfScratchMax = (size_t)1 << 19; // doubles (4 MiB): E = 256, V = 90, S = 10 needs 277,380
static __device__ __align__(256) double scratch[kEnkfScratchMax];
static std::mutex g_scratch_mu;
static double* g_scratch_ptr[64] = {nullptr};

static int enkf_noalloc(int32_t E, int32_t V, int32_t S, double* w, double sigma, const double* y, double rho,
                        const double* xi, void* stream)
{
    DTB_REQUIRE(E >= 2 && V >= 1 && S >= 1, "EnKF needs E >= 2, V >= 1, S >= 1");
    DTB_REQUIRE(w && y && xi, "w, y and xi are required");
    DTB_REQUIRE((size_t)E <= kEnkfScratchMax && (size_t)V <= kEnkfScratchMax && (size_t)S <= kEnkfScratchMax,
                "allocation-free EnKF: E=%d, V=%d, S=%d exceeds the fixed scratch of %zu doubles "
                "(use dtb_enkf_analysis_f64)", E, V, S, kEnkfScratchMax);
    // the documented limit, which also counts a mean [V*S] and a matrix [E*E]
    const size_t need = enkf_scratch_doubles(E, V, S) + (size_t)V * S + (size_t)E * E;
    DTB_REQUIRE(need <= kEnkfScratchMax,
                "allocation-free EnKF: E=%d, V=%d, S=%d counts %zu scratch doubles, the fixed scratch holds %zu "
                "(use dtb_enkf_analysis_f64)", E, V, S, need, kEnkfScratchMax);
    int dev = 0;
    DTB_TRY_HIP(hipGetDevice(&dev));
    DTB_REQUIRE(dev >= 0 && dev < 64, "device index out of range");
    double* p = nullptr;
    {
        std::lock_guard<std::mutex> lk(g_scratch_mu);
        if (!g_scratch_ptr[dev]) {
            void* a = nullptr;
            const hipError_t e = hipGetSymbolAddress(&a, HIP_SYMBOL(scratch));
            if (e != hipSuccess || !a) {
                set_error("hipGetSymbolAddress of the EnKF scratch failed on device %d: %s", dev, hipGetErrorString(e));
                return DTB_RUNTIME_ERROR;
            }
            g_scratch_ptr[dev] = static_cast<double*>(a);
        }
        p = g_scratch_ptr[dev];
    }
    return enkf_launch(E, V, S, w, sigma, y, rho, xi, (hipStream_t)stream, p);
}

} // namespace dtb

extern "C" {

int dtb_bold_step_f32(int64_t n, const double* par, float* s, float* q, float* v, float* f, const float* u,
                      float* out, void* stream)
{
    return dtb::bold_step<float>(n, par, s, q, v, f, u, out, stream);
}

int dtb_bold_step_f64(int64_t n, const double* par, double* s, double* q, double* v, double* f, const double* u,
                      double* out, void* stream)
{
    return dtb::bold_step<double>(n, par, s, q, v, f, u, out, stream);
}

int dtb_bold_run_f64(int64_t n, int32_t steps, const double* par, double* s, double* q, double* v, double* f,
                     const double* u, double* out, void* stream)
{
    DTB_REQUIRE(n >= 0 && steps >= 0, "n and steps must be >= 0");
    DTB_REQUIRE(par != nullptr, "par is NULL");
    if (n == 0 || steps == 0) return DTB_OK;
    DTB_REQUIRE(s && q && v && f && u && out, "state, input and output arrays are required");
    hipLaunchKernelGGL(dtb::bold_run_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, (hipStream_t)stream, n,
                       steps, par[0], par[1], par[2], par[3], 1.0 / par[4], par[5], par[6], par[7], s, q, v, f, u, out);
    DTB_TRY_HIP(hipGetLastError());
    return DTB_OK;
}

int dtb_enkf_analysis_f64(int32_t E, int32_t V, int32_t S, double* w, double sigma, const double* y, double rho,
                          const double* xi, void* stream)
{
    return dtb::enkf(E, V, S, w, sigma, y, rho, xi, stream);
}

int dtb_enkf_analysis_f64_noalloc(int32_t E, int32_t V, int32_t S, double* w, double sigma, const double* y,
                                  double rho, const double* xi, void* stream)
{
    return dtb::enkf_noalloc(E, V, S, w, sigma, y, rho, xi, stream);
}

} // extern "C"
