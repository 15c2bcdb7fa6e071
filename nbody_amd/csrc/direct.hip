// direct.hip -- O(N^2) sums: the FP32 direct solver, the reference's naive
// force law, and the FP64 sums that the force error is measured against.
#include <algorithm>

#include "common.h"
#include "launch.h"

namespace nbh {

// ---------------------------------------------------------------------------
// Direct sum on the GPU (replaces NaiveSimulation::step's O(N^2) loop,
// naive_simulation.cpp:8-35), softened law: FP32 positions relative to the
// system's box centre, packed once: x, y, z and charge in arrays in which every
// system is followed by DS_PAD zeros, so that a chunk past its end reads no
// other system's values (which may overflow FP32, and 0 times infinity is NaN).
__global__ void direct_pack_kernel(State S, uint32_t n, const uint32_t* sys_off, int nsys, const double4* box,
                                   float* pk) {
    const uint32_t t = blockIdx.x * blockDim.x + threadIdx.x;
    const uint32_t m = direct_pack_len(n, nsys);
    if (t >= m) return;
    uint32_t at;
    float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
    if (t < n) {
        int lo = 0, hi = nsys - 1;
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (sys_off[mid] <= t) lo = mid; else hi = mid - 1;
        }
        const double4 bx = box[lo];
        const double h = 0.5 * bx.w;
        v = make_float4((float)(S.x[t] - (bx.x + h)), (float)(S.y[t] - (bx.y + h)), (float)(S.z[t] - (bx.z + h)),
                        (float)S.charge[t]);
        at = t + lo * DS_PAD;
    } else {
        const uint32_t s = (t - n) / DS_PAD;
        at = sys_off[s + 1] + (t - n);
    }
    pk[at] = v.x;
    pk[m + at] = v.y;
    pk[2 * m + at] = v.z;
    pk[3 * m + at] = v.w;
}

// One workgroup per 64 targets (one per lane).  Each target's force is one
// FP32 sum over the sources in order, a serial chain: with a thread per target
// doing all of a pair's work, N / 64 wavefronts share the GPU (256 on 1024
// SIMDs at N = 16,384: 842 us a sum).  Here the chain holds only what has to
// be in order: 13 producer wavefronts compute q / r^3 for 8 sources each of a
// chunk of 104 into LDS while three consumers, one per component, add the
// chunk before it: a subtraction and an FMA per source.  The sums are bit for
// bit those of the one-thread chain.  Per source and 64 targets the producers
// issue 14 slots (the rsq takes four) and the consumers 6: 150 us at N =
// 16,384 if the four SIMDs of a CU never wait; measured 190 us.  (The sum cut
// into 16 slices takes 129 us, but rounds differently.)  Sources are the same
// for every lane of a wavefront and come through scalar loads.  The potential
// has no such order: each producer keeps a partial sum.  NORMAL: eps^2 is a normal float, so that
// v_rsq_f32 needs no denormal scaling (rsqrtf's).
constexpr int DS_PROD = 13, DS_PER = 8, DS_CH = DS_PROD * DS_PER, DS_WAVES = DS_PROD + 3;
static_assert(DS_PAD >= DS_CH, "a chunk past the particles reads the padding");
template <bool NORMAL>
__global__ __launch_bounds__(WAVE * DS_WAVES) void direct_f32_kernel(State S, const float* __restrict__ pk, uint32_t m,
                                                                     const uint32_t* __restrict__ sys_off, float G,
                                                                     float eps2, double kick_dt) {
    __shared__ float4 w3s[2][DS_CH / 4][WAVE];  // q / r^3 of four sources
    __shared__ float part[DS_PROD + 3][WAVE];
    const uint32_t b = sys_off[blockIdx.y], e = sys_off[blockIdx.y + 1];
    const uint32_t i0 = b + blockIdx.x * WAVE;
    if (i0 >= e) return;
    const int lane = lane_id();
    const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t i = i0 + lane, it = min(i, e - 1);
    // (m: the arrays' length, in 32 bits: with 64-bit strides the kernel took half
    // as long again at N = 65,536)
    const uint32_t pad = blockIdx.y * DS_PAD;  // the system's particles stand so much further on
    const uint32_t nch = (e - b + DS_CH - 1) / DS_CH;
    if (wv < 3) {  // consumers: component wv
        const float* src = pk + wv * m + (b + pad);
        const float me = pk[wv * m + it + pad];
        float acc = 0.f;
        for (uint32_t c = 0; c <= nch; ++c) {
            if (c > 0) {
                const float* q = src + (size_t)(c - 1) * DS_CH;
#pragma unroll 2
                for (int g = 0; g < DS_CH / 4; ++g) {
                    const float4 w = w3s[(c - 1) & 1][g][lane];
                    acc = fmaf(q[4 * g] - me, w.x, acc);
                    acc = fmaf(q[4 * g + 1] - me, w.y, acc);
                    acc = fmaf(q[4 * g + 2] - me, w.z, acc);
                    acc = fmaf(q[4 * g + 3] - me, w.w, acc);
                }
            }
            __syncthreads();
        }
        part[DS_PROD + wv][lane] = acc;
    } else {
        const int pw = wv - 3;
        const float px = pk[it + pad], py = pk[m + it + pad], pz = pk[2 * m + it + pad];
        float ph = 0.f;
        for (uint32_t c = 0; c <= nch; ++c) {
            if (c < nch) {
                const uint32_t j0 = b + c * DS_CH + pw * DS_PER;  // uniform
                const float *sx = pk + (j0 + pad), *sy = sx + m, *sz = sy + m, *sq = sz + m;
                float w3[DS_PER];
                auto pairs = [&](auto&& skip) {
#pragma unroll
                    for (int k = 0; k < DS_PER; ++k) {
                        const float rx = sx[k] - px, ry = sy[k] - py, rz = sz[k] - pz;
                        const float r2 = fmaf(rx, rx, fmaf(ry, ry, fmaf(rz, rz, eps2)));
                        const float inv = skip(k) ? 0.f : NORMAL ? __builtin_amdgcn_rsqf(r2) : rsqrtf(r2);
                        const float w = sq[k] * inv;
                        w3[k] = w * inv * inv;
                        ph += w;
                    }
                };
                // the self pair and the slots past the system's end contribute nothing
                if (j0 + DS_PER <= e && (j0 + DS_PER <= i0 || j0 >= i0 + WAVE)) pairs([](int) { return false; });
                else pairs([&](int k) { return j0 + k == i || j0 + k >= e; });
#pragma unroll
                for (int g = 0; g < DS_PER / 4; ++g)
                    w3s[c & 1][pw * (DS_PER / 4) + g][lane] =
                        make_float4(w3[4 * g], w3[4 * g + 1], w3[4 * g + 2], w3[4 * g + 3]);
            }
            __syncthreads();
        }
        part[pw][lane] = ph;
    }
    __syncthreads();
    if (wv != 0 || i >= e) return;
    float ph = 0.f;
    for (int w = 0; w < DS_PROD; ++w) ph += part[w][lane];
    const float fac = (float)(S.charge[i] / S.mass[i]) * G;
    const float ax = fac * part[DS_PROD][lane], ay = fac * part[DS_PROD + 1][lane], az = fac * part[DS_PROD + 2][lane];
    S.ax[i] = ax; S.ay[i] = ay; S.az[i] = az;
    S.pot[i] = -G * ph;
    if (kick_dt != 0.0) {
        S.vx[i] += (double)ax * kick_dt;
        S.vy[i] += (double)ay * kick_dt;
        S.vz[i] += (double)az * kick_dt;
    }
}

// The same sums with one thread per target that does all of a pair's work,
// source tiles in LDS: about 12 issue slots a pair where the pipeline takes 20,
// once there are targets enough to fill the GPU with (direct_by_pipeline).
constexpr int DT_THREADS = 256;
template <bool NORMAL>
__global__ __launch_bounds__(DT_THREADS) void direct_thread_kernel(State S, const uint32_t* __restrict__ sys_off,
                                                                   const double4* __restrict__ box, float G,
                                                                   float eps2, double kick_dt) {
    __shared__ float4 tile[DT_THREADS];
    const uint32_t b = sys_off[blockIdx.y], e = sys_off[blockIdx.y + 1];
    const uint32_t i = b + blockIdx.x * DT_THREADS + threadIdx.x;
    if (b + blockIdx.x * DT_THREADS >= e) return;
    const double4 bx = box[blockIdx.y];
    const double h = 0.5 * bx.w, cx = bx.x + h, cy = bx.y + h, cz = bx.z + h;
    const bool valid = i < e;
    auto offset = [&](uint32_t j) {
        return make_float4((float)(S.x[j] - cx), (float)(S.y[j] - cy), (float)(S.z[j] - cz), (float)S.charge[j]);
    };
    const float4 me = offset(valid ? i : e - 1);
    float ax = 0.f, ay = 0.f, az = 0.f, ph = 0.f;
    for (uint32_t j0 = b; j0 < e; j0 += DT_THREADS) {
        const uint32_t j = j0 + threadIdx.x;
        __syncthreads();
        if (j < e) tile[threadIdx.x] = offset(j);
        __syncthreads();
        const uint32_t jn = min((uint32_t)DT_THREADS, e - j0);
        if (!valid) continue;
        for (uint32_t k = 0; k < jn; ++k) {
            const float4 q = tile[k];
            const float rx = q.x - me.x, ry = q.y - me.y, rz = q.z - me.z;
            const float r2 = fmaf(rx, rx, fmaf(ry, ry, fmaf(rz, rz, eps2)));
            // the self pair contributes nothing (r2 = 0 when unsoftened)
            const float inv = j0 + k == i ? 0.f : NORMAL ? __builtin_amdgcn_rsqf(r2) : rsqrtf(r2);
            const float w = q.w * inv;
            const float w3 = w * inv * inv;
            ax = fmaf(rx, w3, ax);
            ay = fmaf(ry, w3, ay);
            az = fmaf(rz, w3, az);
            ph += w;
        }
    }
    if (!valid) return;
    const float fac = (float)(S.charge[i] / S.mass[i]) * G;
    ax *= fac; ay *= fac; az *= fac;
    S.ax[i] = ax; S.ay[i] = ay; S.az[i] = az;
    S.pot[i] = -G * ph;
    if (kick_dt != 0.0) {
        S.vx[i] += (double)ax * kick_dt;
        S.vy[i] += (double)ay * kick_dt;
        S.vz[i] += (double)az * kick_dt;
    }
}

// The reference's naive force law (compat): separation (dx, dx, dx), no
// softening (naive_simulation.cpp:10-17), with each pair's term formed as the
// reference forms it in FP32 (uncentred x difference, r = sqrt(d d + d d +
// d d), force = (k q_i q_j) d / (r r r), divided by m_i; no contraction into
// FMAs) and summed in FP64, so one evaluation differs from the reference only
// by its FP32 summation order.  One thread per target, source tiles in LDS.
constexpr int DC_THREADS = 256;
__global__ __launch_bounds__(DC_THREADS) void direct_compat_kernel(State S, const uint32_t* sys_off, float G,
                                                                   double kick_dt) {
    __shared__ float2 tile[DC_THREADS];  // x, charge
    const int s = blockIdx.y;
    const uint32_t b = sys_off[s], e = sys_off[s + 1];
    const uint32_t i = b + blockIdx.x * DC_THREADS + threadIdx.x;
    if (b + blockIdx.x * DC_THREADS >= e) return;
    const bool valid = i < e;
    const float px = valid ? (float)S.x[i] : 0.f;
    float ph = 0;
    double acd = 0.0;  // sum of the reference's per-pair kicks / dt
    const float qi = valid ? (float)S.charge[i] : 0.f, mi = valid ? (float)S.mass[i] : 1.f;
    for (uint32_t j0 = b; j0 < e; j0 += DC_THREADS) {
        const uint32_t j = j0 + threadIdx.x;
        __syncthreads();
        tile[threadIdx.x] = j < e ? make_float2((float)S.x[j], (float)S.charge[j]) : make_float2(0, 0);
        __syncthreads();
        const uint32_t jn = min((uint32_t)DC_THREADS, e - j0);
        if (!valid) continue;
        for (uint32_t k = 0; k < jn; ++k) {
            // IEEE single operations in the reference's order: no FMA
            // contraction; sqrtf and '/' are correctly rounded in HIP
#pragma clang fp contract(off)
            if (j0 + k == i) continue;
            const float2 q = tile[k];
            const float d = q.x - px;
            const float r = sqrtf(d * d + d * d + d * d);
            const float f = G * (qi * q.y) * d / (r * r * r);
            acd += (double)(f / mi);
            ph += q.y / r;
        }
    }
    if (!valid) return;
    const float a = (float)acd;
    S.ax[i] = a; S.ay[i] = a; S.az[i] = a;
    S.pot[i] = -G * ph;
    if (kick_dt != 0.0) {
        S.vx[i] += (double)a * kick_dt;
        S.vy[i] += (double)a * kick_dt;
        S.vz[i] += (double)a * kick_dt;
    }
}

// The pipeline shortens the chain of each target, the thread-per-target form
// takes fewer slots a pair: the first wins while there are few targets, in
// systems large enough to fill and drain its chunks.  Sum kernels, us, pipeline
// and threads (eps > 0), either side of the line:
//   size x systems
//   128 x 1     11.1  9.5     200 x 1      11.0  12.4
//   200 x 128   14.3 13.3     200 x 64     12.5  13.1
//   512 x 128   33.6 28.0     512 x 64     20.3  26.8
//   1000 x 64   52.2 50.7     1000 x 48    39.6  46.2
//   4096 x 64    612  435     4096 x 20     182   215
//   65536 x 2   4070 3362     65536 x 1    2092  2732
//   131072 x 1  8144 6667     90000 x 1    4005  4548
//   262144 x 1 31960 24905    16384 x 1     174   675
// (every system has a workgroup, also one of few particles)
static bool direct_by_pipeline(uint32_t n, uint32_t max_sys_n, int nsys) {
    return max_sys_n >= 192 && n <= std::min<uint64_t>(24576u + 24ull * max_sys_n, 98304u) && nsys <= 512;
}
size_t direct_pack_bytes(uint32_t n, uint32_t max_sys_n, int nsys) {
    return direct_by_pipeline(n, max_sys_n, nsys) ? 16 * (size_t)direct_pack_len(n, nsys) : 0;
}

void launch_direct_f32(const State& S, uint32_t n, uint32_t max_sys_n, const uint32_t* sys_off, int nsys,
                       const double4* box, float G, float eps2, int compat_law, double kick_dt, float* pk,
                       hipStream_t st) {
    if (compat_law) {
        hipLaunchKernelGGL(direct_compat_kernel, dim3(ceil_div(max_sys_n, DC_THREADS), nsys), dim3(DC_THREADS), 0, st,
                           S, sys_off, G, kick_dt);
        return;
    }
    const bool normal = eps2 >= 1.17549435e-38f;
    if (!direct_by_pipeline(n, max_sys_n, nsys)) {
        const dim3 grid(ceil_div(max_sys_n, DT_THREADS), nsys), block(DT_THREADS);
        if (normal)
            hipLaunchKernelGGL(direct_thread_kernel<true>, grid, block, 0, st, S, sys_off, box, G, eps2, kick_dt);
        else
            hipLaunchKernelGGL(direct_thread_kernel<false>, grid, block, 0, st, S, sys_off, box, G, eps2, kick_dt);
        return;
    }
    const uint32_t m = direct_pack_len(n, nsys);
    hipLaunchKernelGGL(direct_pack_kernel, dim3(ceil_div(m, 256)), dim3(256), 0, st, S, n, sys_off, nsys, box, pk);
    const dim3 grid(ceil_div(max_sys_n, WAVE), nsys), block(WAVE * DS_WAVES);
    if (normal)
        hipLaunchKernelGGL(direct_f32_kernel<true>, grid, block, 0, st, S, pk, m, sys_off, G, eps2, kick_dt);
    else
        hipLaunchKernelGGL(direct_f32_kernel<false>, grid, block, 0, st, S, pk, m, sys_off, G, eps2, kick_dt);
}

// ---------------------------------------------------------------------------
// FP64 direct sum for selected targets (sorted slots).  NW of a workgroup's 8
// wavefronts take T targets together and stride over the sources with one
// source per lane, so that each source is loaded once for T targets (one
// target per wavefront read 32 bytes per pair from L2, 12 TB/s at 262,144
// sources x 4096 targets, which bound it).  1/r is v_rsq_f64 (relative error
// e/2 ~ 2^-27) and one third-order step y (1 + e/2 + 3/8 e^2), e = 1 - r^2 y^2,
// whose remainder ~e^3 is below the rounding; 1/sqrt took ~50 instructions of
// the pair's ~70.  262,144 x 4096: 2.5 -> 1.06 ms, of 0.68 ms that the pairs'
// FP64 instructions take.
constexpr int DD_WAVES = 8;
template <int T, int NW>
__global__ __launch_bounds__(WAVE * DD_WAVES) void direct_fp64_kernel(State S, const uint32_t* __restrict__ sys_off,
                                                                      int nsys, const uint32_t* __restrict__ targets,
                                                                      uint32_t nt, double G, double eps2, double* acc,
                                                                      double* pot) {
    __shared__ double part[DD_WAVES][T][4];
    const int lane = lane_id();
    const uint32_t wv = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE);
    const uint32_t w0 = (blockIdx.x * (DD_WAVES / NW) + wv / NW) * T;  // the group's targets
    const uint32_t n = sys_off[nsys];
    uint32_t id[T];
    double px[T], py[T], pz[T], a[T][4];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        // (no such particle, or past the last target: the sums are dropped)
        const uint32_t i = targets[min(w0 + t, nt - 1)];
        id[t] = i;
        const uint32_t k = i < n ? i : 0u;
        px[t] = S.x[k]; py[t] = S.y[k]; pz[t] = S.z[k];
        a[t][0] = a[t][1] = a[t][2] = a[t][3] = 0.0;
    }
    // T > 1: one system (the launcher's rule)
    uint32_t b = 0, e = n;
    if (T == 1 && nsys > 1) {
        int lo = 0, hi = nsys - 1;
        while (lo < hi) { int mid = (lo + hi + 1) >> 1; if (sys_off[mid] <= id[0]) lo = mid; else hi = mid - 1; }
        b = sys_off[lo];
        e = sys_off[lo + 1];
    }
    if (w0 >= nt) e = b;
    for (uint32_t j = b + (wv % NW) * WAVE + lane; j < e; j += WAVE * NW) {
        const double sx = S.x[j], sy = S.y[j], sz = S.z[j], q = S.charge[j];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const double rx = sx - px[t], ry = sy - py[t], rz = sz - pz[t];
            const double r2 = rx * rx + ry * ry + rz * rz + eps2;
            const double y = __builtin_amdgcn_rsq(r2);
            const double err = fma(-r2 * y, y, 1.0);
            const double yn = fma(y * err, fma(0.375, err, 0.5), y);
            // (r2 = 0 or infinite: err is NaN, and y is the limit)
            const double inv = fabs(err) < 1.0 ? yn : y;
            const double w = j == id[t] ? 0.0 : q * inv;
            const double w3 = j == id[t] ? 0.0 : w * inv * inv;
            a[t][0] = fma(rx, w3, a[t][0]);
            a[t][1] = fma(ry, w3, a[t][1]);
            a[t][2] = fma(rz, w3, a[t][2]);
            a[t][3] += w;
        }
    }
    {
        // (a sum a lane: the 4 T sums one after the other took 24 T shuffles, and
        // half of the kernel's time at n = 5003)
        group_reduce_scatter<4 * T, 6>(&a[0][0]);
        int at, cnt;
        rs_slot(4 * T, 6, lane, at, cnt);
        if (cnt > 0) (&part[wv][0][0])[at] = a[0][0];
    }
    __syncthreads();
    for (uint32_t v = threadIdx.x; v < 4 * T * (DD_WAVES / NW); v += WAVE * DD_WAVES) {
        const int g = v / (4 * T), t = v / 4 % T, k = v % 4;
        const uint32_t w = (blockIdx.x * (DD_WAVES / NW) + g) * T + t;
        if (w >= nt) continue;
        const uint32_t i = targets[w];
        double sum = 0.0;
        for (int q = 0; q < NW; ++q) sum += part[g * NW + q][t][k];
        // no such particle: report NaN
        if (k < 3) acc[3 * (size_t)w + k] = i < n ? S.charge[i] / S.mass[i] * G * sum : NAN;
        else pot[w] = i < n ? -G * sum : NAN;
    }
}

template <int T, int NW>
static void launch_direct_fp64_t(const State& S, const uint32_t* sys_off, int nsys, const uint32_t* targets,
                                 uint32_t nt, double G, double eps2, double* acc, double* pot, hipStream_t st) {
    hipLaunchKernelGGL((direct_fp64_kernel<T, NW>), dim3(ceil_div(nt, T * (DD_WAVES / NW))), dim3(WAVE * DD_WAVES), 0,
                       st, S, sys_off, nsys, targets, nt, G, eps2, acc, pot);
}
void launch_direct_fp64(const State& S, uint32_t n, const uint32_t* sys_off, int nsys, const uint32_t* targets,
                        uint32_t nt, double G, double eps2, double* acc, double* pot, hipStream_t st) {
    if (!nt) return;
    if (nsys == 1) {
        // eight targets where that leaves two workgroups a CU, four where it
        // leaves one, us with 1, 4 and 8 at 262,144 sources: 512 targets 244,
        // 284, 606; 1024 491, 307, 613; 2048 929, 562, 630; 4096 1810, 1047,
        // 1056; 16,384 7172, 3999, 3871; at 5003 sources: 1024 16, 12, 18;
        // 4096 45, 29, 29
        if (nt >= 4096) launch_direct_fp64_t<8, 8>(S, sys_off, nsys, targets, nt, G, eps2, acc, pot, st);
        else if (nt >= 1024) launch_direct_fp64_t<4, 8>(S, sys_off, nsys, targets, nt, G, eps2, acc, pot, st);
        else launch_direct_fp64_t<1, 8>(S, sys_off, nsys, targets, nt, G, eps2, acc, pot, st);
        return;
    }
    // of several systems each target has its own sources, and one wavefront
    // does where there are targets enough and their systems are small, us with
    // one and eight, size x targets: 8 x 65,536 35, 241; 512 x 4096 11, 20;
    // 2048 x 2048 14, 16; 2048 x 1024 13, 11; 1000 x 1024 9.4, 9.0; 8192 x 8192
    // 133, 122; 40,000 x 2048 245, 151
    const uint32_t mean = n / (uint32_t)nsys;
    if (nt >= 1024 && mean <= (nt < 2048 ? 1024u : 4096u))
        launch_direct_fp64_t<1, 1>(S, sys_off, nsys, targets, nt, G, eps2, acc, pot, st);
    else
        launch_direct_fp64_t<1, 8>(S, sys_off, nsys, targets, nt, G, eps2, acc, pot, st);
}

// slots[k] = slot_of[targets[k]] (targets checked by the host)
__global__ void map_slots_kernel(const uint32_t* slot_of, const int64_t* targets, uint32_t nt, uint32_t* slots) {
    const uint32_t k = blockIdx.x * blockDim.x + threadIdx.x;
    if (k < nt) slots[k] = slot_of[targets[k]];
}
void launch_map_slots(const uint32_t* slot_of, const int64_t* targets, uint32_t nt, uint32_t* slots, hipStream_t st) {
    hipLaunchKernelGGL(map_slots_kernel, dim3(ceil_div(nt, 256)), dim3(256), 0, st, slot_of, targets, nt, slots);
}

// Sorted slot of each target given in input order, by a scan of the id array
// (one wavefront per target; an id array is a permutation, so every index in
// [0, n) is found once; anything else gets 0xffffffff).  Costs a read of the
// ids per target, an eighth of what the FP64 sum then reads per target.
__global__ __launch_bounds__(256) void find_slots_kernel(const uint32_t* __restrict__ id, uint32_t n,
                                                         const int64_t* __restrict__ targets, uint32_t nt,
                                                         uint32_t* slots) {
    const uint32_t w = (blockIdx.x * blockDim.x + threadIdx.x) / WAVE;
    if (w >= nt) return;
    const int64_t t = targets[w];
    uint32_t found = 0xffffffffu;
    for (uint32_t j0 = 0; j0 < n && found == 0xffffffffu; j0 += WAVE) {
        const uint32_t j = j0 + lane_id();
        const uint64_t hit = __ballot(j < n && (int64_t)id[j] == t);
        if (hit) found = j0 + (uint32_t)__ffsll((unsigned long long)hit) - 1;
    }
    if (lane_id() == 0) slots[w] = found;
}
void launch_find_slots(const uint32_t* id, uint32_t n, const int64_t* targets, uint32_t nt, uint32_t* slots,
                       hipStream_t st) {
    hipLaunchKernelGGL(find_slots_kernel, dim3(ceil_div(nt, 4)), dim3(256), 0, st, id, n, targets, nt, slots);
}

}  // namespace nbh
