// eq_channels.hip -- flow channels coupled to the traps, and per-node wall
// values (fenicsInterface::stepDiffusion with MICROFLUIDIC_TRAP and a channel
// trap type, src/fHSL.cpp:110-152).
//
// A channel is a 1-D P1 interval mesh over the trap's columns (fenicsChannel,
// src/fHSL.h:240-332, with zero channel extensions: src/fHSL.cpp:262-275).
// Its values are the trap's Dirichlet data on that wall (DirichletBC bound to
// the channel Function, src/fHSL.cpp:514, 531).  After every trap solve:
//   flux_j = dt*D*(u_inner,j - u_wall,j)/wellScaling          (src/fHSL.cpp:54-96)
//   repeat substeps times:  c += flux/substeps;  Crank-Nicolson step of
//     dt/substeps of   w(c - c0) + k D w' (c0+c)'/2 + k v (c0+c)'/2 w
//                      + k r_{1,2} ((c0+c)/2 - s_{1,2}) w |_{x=0, W}
//   (fenics/AdvectionDiffusion.ufl:62-64), a tridiagonal system solved by the
//   Thomas algorithm (diagonally dominant for the reference's step control,
//   src/main.cpp:414-430).
// Channels are independent, and their matrices stay the same from step to step:
// the Thomas factors are laid out once with the channel, which leaves two
// first-order recurrences a substep, run as prefix scans of affine maps.
#include <hip/hip_runtime.h>

#include <array>
#include <vector>

#include "eq_internal.h"

namespace eqk {

struct ChannelDev {
    eq_channel_desc ch;
    double* c;         // channel values (nx+1), also the wall's Dirichlet data
    double* dp;        // scratch (nx+1 each): the forward sweep's values
    const double* cp;  // Thomas factors: upper / pivot,
    const double* im;  // 1 / pivot,
    const double* am;  // lower / pivot
    const double* u;   // node (0,0) of the trap field
    int32_t nx, ny, pitch, top; // top: 1 = channel above the trap (wall row ny)
    double hc, D, dt;
};

// Row i of the channel's tridiagonal system for one substep, and of its
// right-hand side: lower, diagonal, upper each; r0 the Robin source.
struct ChannelRow {
    double a, b, c, ra, rb, rc, r0;
};
__host__ __device__ __forceinline__ ChannelRow channel_row(const eq_channel_desc& ch, int i, int N, double k, double hc,
                                                           double D)
{
    const double v = ch.v, m1 = hc / 6.0, m2 = 2.0 * hc / 6.0;
    // D K + v C (+ Robin); nodes 0 and N lie on one element
    double Tl = -D / hc - 0.5 * v, Td = 2.0 * D / hc, Tu = -D / hc + 0.5 * v, md = 2.0 * m2, r0 = 0.0;
    if (i == 0) {
        Td = D / hc - 0.5 * v + ch.r_left;
        md = m2;
        r0 = k * ch.r_left * ch.s_left;
    } else if (i == N) {
        Td = D / hc + 0.5 * v + ch.r_right;
        md = m2;
        r0 = k * ch.r_right * ch.s_right;
    }
    ChannelRow R{m1 + 0.5 * k * Tl, md + 0.5 * k * Td, m1 + 0.5 * k * Tu,
                 m1 - 0.5 * k * Tl, md - 0.5 * k * Td, m1 - 0.5 * k * Tu, r0};
    if (i == 0) R.a = R.ra = 0.0;
    if (i == N) R.c = R.rc = 0.0;
    return R;
}

// One block a channel, consecutive rows a thread.  A substep is
//   dp_i = im_i r_i - am_i dp_(i-1),  x_i = dp_i - cp_i x_(i+1):
// a thread composes its rows' maps, the block scans the compositions, the
// thread applies its carry.  Bound by the latency of the two scans (about 3 us
// a substep); one thread walking the rows with two divisions each took 750 us
// for three substeps of 438 rows; the case's whole step, two species with two
// channels, went from 1.08 to 0.34 ms.
constexpr int kChanThreads = 512;

// the map value -> p value + q of everything before (after, if DOWN) this
// thread, applied to zero: the thread's carry
template <bool DOWN>
__device__ __forceinline__ double scan_carry(double p, double q, double (*red)[2])
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    constexpr int W = kChanThreads / 64;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const double pp = DOWN ? __shfl_down(p, off, 64) : __shfl_up(p, off, 64);
        const double qq = DOWN ? __shfl_down(q, off, 64) : __shfl_up(q, off, 64);
        if (DOWN ? lane + off < 64 : lane >= off) {
            q = p * qq + q;
            p = p * pp;
        }
    }
    if (lane == (DOWN ? 0 : 63)) {
        red[w][0] = p;
        red[w][1] = q;
    }
    __syncthreads();
    double in = 0.0; // at this wave's edge
    if (DOWN)
        for (int k = W - 1; k > w; --k) in = red[k][0] * in + red[k][1];
    else
        for (int k = 0; k < w; ++k) in = red[k][0] * in + red[k][1];
    // the neighbour's inclusive map on the wave's edge value
    const double pe = DOWN ? __shfl_down(p, 1, 64) : __shfl_up(p, 1, 64);
    const double qe = DOWN ? __shfl_down(q, 1, 64) : __shfl_up(q, 1, 64);
    __syncthreads(); // red is free again
    return lane == (DOWN ? 63 : 0) ? in : pe * in + qe;
}

__global__ __launch_bounds__(kChanThreads) void k_channels(const ChannelDev* __restrict__ chans)
{
    __shared__ double red[kChanThreads / 64][2];
    const ChannelDev C = chans[blockIdx.x];
    const int N = C.nx;
    const int nsub = C.ch.substeps > 0 ? C.ch.substeps : 1;
    const double k = C.dt / nsub;
    const double* inner = C.u + (C.top ? (int64_t)(C.ny - 1) * C.pitch : C.pitch);
    const double* wall = C.u + (C.top ? (int64_t)C.ny * C.pitch : 0);
    const double fscale = C.dt * C.D / C.ch.well_scaling / (double)nsub;
    const int L = (N + kChanThreads) / kChanThreads; // rows a thread
    const int i0 = (int)threadIdx.x * L, i1 = min(i0 + L, N + 1);
    auto value = [&](int i) { return i >= 0 && i <= N ? C.c[i] + fscale * (inner[i] - wall[i]) : 0.0; };
    for (int s = 0; s < nsub; ++s) {
        double p = 1.0, q = 0.0;
        double prev = i0 < i1 ? value(i0 - 1) : 0.0, cur = i0 < i1 ? value(i0) : 0.0;
        for (int i = i0; i < i1; ++i) {
            const ChannelRow R = channel_row(C.ch, i, N, k, C.hc, C.D);
            const double next = value(i + 1);
            const double g = C.im[i] * (R.ra * prev + R.rb * cur + R.rc * next + R.r0);
            C.dp[i] = g;
            q = g - C.am[i] * q;
            p = -C.am[i] * p;
            prev = cur;
            cur = next;
        }
        double d = scan_carry<false>(p, q, red);
        for (int i = i0; i < i1; ++i) {
            d = C.dp[i] - C.am[i] * d;
            C.dp[i] = d;
        }
        p = 1.0;
        q = 0.0;
        for (int i = i1 - 1; i >= i0; --i) {
            q = C.dp[i] - C.cp[i] * q;
            p = -C.cp[i] * p;
        }
        double x = scan_carry<true>(p, q, red);
        for (int i = i1 - 1; i >= i0; --i) {
            x = C.dp[i] - C.cp[i] * x;
            C.c[i] = x;
        }
        __syncthreads(); // the neighbours' values of the next substep
    }
}

} // namespace eqk

using namespace eqk;

namespace {

// re-send level 0's problem table after a change of its wall-value pointers
int upload_level0(eq_batch* b)
{
    Level& L = b->levels[0];
    EQ_HIP(hipStreamSynchronize(b->stream));
    const int rc = pull_well_values(b); // keep the wall values the wells wrote
    if (rc) return rc;
    EQ_HIP(hipMemcpy(L.d_probs, L.probs.data(), sizeof(LevelProb) * L.probs.size(), hipMemcpyHostToDevice));
    return EQ_OK;
}

int wall_length(const LevelProb& P, int wall) { return (wall == kTop || wall == kBottom) ? P.nx + 1 : P.ny + 1; }

} // namespace

namespace eqk {

// the channels after a solve (called by eq_batch_step)
int channels_after_step(eq_batch* b)
{
    if (b->chan_count == 0) return EQ_OK;
    double bytes = 0.0; // per channel: its values read and written, the trap's two rows read, per substep
    for (size_t p = 0; p < b->chan_desc.size(); ++p)
        for (int k = 0; k < 2; ++k)
            if (b->chan_desc[p][k].substeps > 0)
                bytes += 32.0 * (b->levels[0].probs[p].nx + 1) * b->chan_desc[p][k].substeps;
    launch(b, EQ_KERNEL_BOUNDARY, bytes, k_channels, dim3(b->chan_count), dim3(kChanThreads), 0, b->stream,
           (const ChannelDev*)b->d_chans);
    EQ_HIP(hipGetLastError());
    return EQ_OK;
}

void free_channels(eq_batch* b)
{
    for (auto& w : b->wall_vals)
        for (double* p : w) hipFree(p);
    b->wall_vals.clear();
    hipFree(b->d_chans);
    b->d_chans = nullptr;
    for (double* p : b->chan_scratch) hipFree(p);
    b->chan_scratch.clear();
}

} // namespace eqk

namespace {

// rebuild the device channel table from the host descriptions
int rebuild_channels(eq_batch* b)
{
    EQ_HIP(hipStreamSynchronize(b->stream)); // the old table and scratch are no longer in use
    for (double* p : b->chan_scratch) hipFree(p);
    b->chan_scratch.clear();
    std::vector<ChannelDev> v;
    const Level& L = b->levels[0];
    for (int p = 0; p < b->nprob; ++p) {
        for (int side = 0; side < 2; ++side) {
            const int wall = side == 0 ? kTop : kBottom;
            if (b->chan_desc[p][side].substeps == 0) continue; // no channel
            const LevelProb& P = L.probs[p];
            ChannelDev c{};
            c.ch = b->chan_desc[p][side];
            c.c = b->wall_vals[p][wall];
            const size_t n = (size_t)P.nx + 1;
            double* scratch = nullptr;
            if (hipMalloc((void**)&scratch, sizeof(double) * 4 * n) != hipSuccess)
                return set_error(EQ_ERR_NOMEM, "channel scratch");
            b->chan_scratch.push_back(scratch);
            c.hc = b->descs[p].width / P.nx;
            c.D = b->descs[p].D;
            c.dt = b->descs[p].dt;
            std::vector<double> fac(3 * n); // cp, im, am
            for (size_t i = 0; i < n; ++i) {
                const ChannelRow R = channel_row(c.ch, (int)i, P.nx, c.dt / c.ch.substeps, c.hc, c.D);
                const double m = i ? R.b - R.a * fac[i - 1] : R.b;
                fac[i] = R.c / m;
                fac[n + i] = 1.0 / m;
                fac[2 * n + i] = R.a / m;
            }
            EQ_HIP(hipMemcpy(scratch + n, fac.data(), sizeof(double) * 3 * n, hipMemcpyHostToDevice));
            c.dp = scratch;
            c.cp = scratch + n;
            c.im = scratch + 2 * n;
            c.am = scratch + 3 * n;
            c.u = b->u + P.origin;
            c.nx = P.nx;
            c.ny = P.ny;
            c.pitch = P.pitch;
            c.top = side == 0 ? 1 : 0;
            v.push_back(c);
        }
    }
    hipFree(b->d_chans);
    b->d_chans = nullptr;
    b->chan_count = (int32_t)v.size();
    if (v.empty()) return EQ_OK;
    if (hipMalloc(&b->d_chans, sizeof(ChannelDev) * v.size()) != hipSuccess)
        return set_error(EQ_ERR_NOMEM, "channel table");
    EQ_HIP(hipMemcpy(b->d_chans, v.data(), sizeof(ChannelDev) * v.size(), hipMemcpyHostToDevice));
    return EQ_OK;
}

// device array of one wall's per-node values (allocated on first use)
int ensure_wall_array(eq_batch* b, int32_t prob, int32_t wall, double** out)
{
    if ((int)b->wall_vals.size() < b->nprob) b->wall_vals.resize(b->nprob, std::array<double*, 4>{});
    double*& a = b->wall_vals[prob][wall];
    if (!a) {
        const int n = wall_length(b->levels[0].probs[prob], wall);
        if (hipMalloc((void**)&a, sizeof(double) * n) != hipSuccess) return set_error(EQ_ERR_NOMEM, "wall values");
        EQ_HIP(hipMemset(a, 0, sizeof(double) * n));
    }
    *out = a;
    return EQ_OK;
}

} // namespace

extern "C" {

int eq_batch_set_wall_values(eq_batch* b, int32_t prob, int32_t wall, const double* values, size_t n)
{
    if (!b) return set_error(EQ_ERR_INVALID, "NULL batch");
    if (prob < 0 || prob >= b->nprob) return set_error(EQ_ERR_INVALID, "problem index out of range");
    if (wall < 0 || wall > 3) return set_error(EQ_ERR_INVALID, "wall index out of range");
    hipSetDevice(b->device);
    LevelProb& P = b->levels[0].probs[prob];
    if (!(P.dmask & (1 << wall))) return set_error(EQ_ERR_INVALID, "the wall is not Dirichlet");
    if ((wall == kTop || wall == kBottom) && (int)b->chan_desc.size() > prob &&
        b->chan_desc[prob][wall == kTop ? 0 : 1].substeps != 0)
        return set_error(EQ_ERR_INVALID, "the wall's values come from its channel");
    if (!values) {
        P.gw[wall] = nullptr;
        return upload_level0(b);
    }
    if (n != (size_t)wall_length(P, wall)) return set_error(EQ_ERR_INVALID, "wrong number of wall values");
    double* a = nullptr;
    int rc = ensure_wall_array(b, prob, wall, &a);
    if (rc) return rc;
    EQ_HIP(hipStreamSynchronize(b->stream));
    EQ_HIP(hipMemcpy(a, values, sizeof(double) * n, hipMemcpyHostToDevice));
    P.gw[wall] = a;
    return upload_level0(b);
}

int eq_batch_set_channels(eq_batch* b, int32_t prob, const eq_channel_desc* top, const eq_channel_desc* bottom)
{
    if (!b) return set_error(EQ_ERR_INVALID, "NULL batch");
    if (prob < 0 || prob >= b->nprob) return set_error(EQ_ERR_INVALID, "problem index out of range");
    hipSetDevice(b->device);
    LevelProb& P = b->levels[0].probs[prob];
    const eq_channel_desc* d[2] = {top, bottom};
    const int walls[2] = {kTop, kBottom};
    for (int side = 0; side < 2; ++side) {
        if (!d[side]) continue;
        if (!(P.dmask & (1 << walls[side]))) return set_error(EQ_ERR_INVALID, "a channel's wall must be Dirichlet");
        if (!(d[side]->well_scaling > 0) || d[side]->substeps < 1)
            return set_error(EQ_ERR_INVALID, "channel needs well_scaling > 0 and substeps >= 1");
    }
    if ((int)b->chan_desc.size() < b->nprob) b->chan_desc.resize(b->nprob);
    for (int side = 0; side < 2; ++side) {
        eq_channel_desc& slot = b->chan_desc[prob][side];
        if (!d[side]) {
            if (slot.substeps != 0) P.gw[walls[side]] = nullptr;
            slot = eq_channel_desc{};
            continue;
        }
        double* a = nullptr;
        int rc = ensure_wall_array(b, prob, walls[side], &a);
        if (rc) return rc;
        EQ_HIP(hipMemset(a, 0, sizeof(double) * wall_length(P, walls[side]))); // channels start at zero
        slot = *d[side];
        P.gw[walls[side]] = a;
    }
    int rc = upload_level0(b);
    if (rc) return rc;
    return rebuild_channels(b);
}

int eq_batch_channel_values(eq_batch* b, int32_t prob, double* top, double* bottom)
{
    if (!b) return set_error(EQ_ERR_INVALID, "NULL batch");
    if (prob < 0 || prob >= b->nprob) return set_error(EQ_ERR_INVALID, "problem index out of range");
    hipSetDevice(b->device);
    const LevelProb& P = b->levels[0].probs[prob];
    double* out[2] = {top, bottom};
    for (int side = 0; side < 2; ++side) {
        if (!out[side]) continue;
        if ((int)b->chan_desc.size() <= prob || b->chan_desc[prob][side].substeps == 0)
            return set_error(EQ_ERR_INVALID, "no channel on that side");
        const int rc = rows_to_host(b, b->wall_vals[prob][side == 0 ? kTop : kBottom], 1024, 1024, out[side],
                                    sizeof(double) * (P.nx + 1));
        if (rc) return rc;
    }
    return EQ_OK;
}

} // extern "C"
