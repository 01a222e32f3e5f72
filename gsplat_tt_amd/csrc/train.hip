// train.hip - one training step of the splat rasterizer on gfx950: projection of
// the optimizer-space parameters, per-tile forward with the 3DGS blend rules and
// the L1 gradient, per-tile blend backward with per-Gaussian reduction, the
// analytic projection backward, and sparse Adam over the visible rows.
//
// Follows the reference's training oracle gsplat/train_oracle.py:
//   projection + colour + 3-sigma visibility  :125-181
//   blend (skip alpha < alpha_min, stop without blending when
//   T (1 - alpha) < t_min, alpha clamp)         :183-233
//   sparse Adam                                  :434-470
// and the L1 gradient of gsplat/train_loss.py:166-171. Every Gaussian that can
// reach alpha_min somewhere is kept: its footprint uses the opacity-aware
// radius k = sqrt(2 ln(op / alpha_min)) (uncapped) and the per-pair tile cull at
// the same floor, so the tiled forward blends exactly the pairs the per-pixel
// oracle blends.
#include <type_traits>

#include "gs_common.h"
#include "gs_internal.h"

namespace gs {
namespace {

constexpr int kTThreads = 512;
constexpr int kTItems = 4;
constexpr int kTPart = kTThreads * kTItems;
static_assert(kTPart == (int)kProjPartition && kTThreads == 512, "projection partition size");

constexpr float kC0 = 0.28209479177387814f;
constexpr float kC1 = 0.4886025119029199f;
__constant__ float kC2[5] = {1.0925484305920792f, -1.0925484305920792f, 0.31539156525252005f,
                             -1.0925484305920792f, 0.5462742152960396f};
__constant__ float kC3[7] = {-0.5900435899266435f, 2.890611442640554f, -0.4570457994644658f,
                             0.3731763325901154f, -0.4570457994644658f, 1.445305721320277f,
                             -0.5900435899266435f};

// Real SH basis (3DGS order) of direction (x, y, z) up to DEG, and optionally its
// gradient with respect to (x, y, z) taken as a polynomial.
template <int DEG, bool GRAD>
__device__ __forceinline__ void sh_basis(float x, float y, float z, float* b, float (*g)[3]) {
    b[0] = kC0;
    if (GRAD) g[0][0] = g[0][1] = g[0][2] = 0.0f;
    if (DEG >= 1) {
        b[1] = -kC1 * y;
        b[2] = kC1 * z;
        b[3] = -kC1 * x;
        if (GRAD) {
            g[1][0] = 0.0f; g[1][1] = -kC1; g[1][2] = 0.0f;
            g[2][0] = 0.0f; g[2][1] = 0.0f; g[2][2] = kC1;
            g[3][0] = -kC1; g[3][1] = 0.0f; g[3][2] = 0.0f;
        }
    }
    if (DEG >= 2) {
        const float xx = x * x, yy = y * y, zz = z * z;
        b[4] = kC2[0] * x * y;
        b[5] = kC2[1] * y * z;
        b[6] = kC2[2] * (2.0f * zz - xx - yy);
        b[7] = kC2[3] * x * z;
        b[8] = kC2[4] * (xx - yy);
        if (GRAD) {
            g[4][0] = kC2[0] * y; g[4][1] = kC2[0] * x; g[4][2] = 0.0f;
            g[5][0] = 0.0f; g[5][1] = kC2[1] * z; g[5][2] = kC2[1] * y;
            g[6][0] = -2.0f * kC2[2] * x; g[6][1] = -2.0f * kC2[2] * y; g[6][2] = 4.0f * kC2[2] * z;
            g[7][0] = kC2[3] * z; g[7][1] = 0.0f; g[7][2] = kC2[3] * x;
            g[8][0] = 2.0f * kC2[4] * x; g[8][1] = -2.0f * kC2[4] * y; g[8][2] = 0.0f;
        }
        if (DEG >= 3) {
            b[9] = kC3[0] * y * (3.0f * xx - yy);
            b[10] = kC3[1] * x * y * z;
            b[11] = kC3[2] * y * (4.0f * zz - xx - yy);
            b[12] = kC3[3] * z * (2.0f * zz - 3.0f * xx - 3.0f * yy);
            b[13] = kC3[4] * x * (4.0f * zz - xx - yy);
            b[14] = kC3[5] * z * (xx - yy);
            b[15] = kC3[6] * x * (xx - 3.0f * yy);
            if (GRAD) {
                g[9][0] = 6.0f * kC3[0] * x * y; g[9][1] = kC3[0] * (3.0f * xx - 3.0f * yy);
                g[9][2] = 0.0f;
                g[10][0] = kC3[1] * y * z; g[10][1] = kC3[1] * x * z; g[10][2] = kC3[1] * x * y;
                g[11][0] = -2.0f * kC3[2] * x * y;
                g[11][1] = kC3[2] * (4.0f * zz - xx - 3.0f * yy);
                g[11][2] = 8.0f * kC3[2] * y * z;
                g[12][0] = -6.0f * kC3[3] * x * z; g[12][1] = -6.0f * kC3[3] * y * z;
                g[12][2] = kC3[3] * (6.0f * zz - 3.0f * xx - 3.0f * yy);
                g[13][0] = kC3[4] * (4.0f * zz - 3.0f * xx - yy);
                g[13][1] = -2.0f * kC3[4] * x * y; g[13][2] = 8.0f * kC3[4] * x * z;
                g[14][0] = 2.0f * kC3[5] * x * z; g[14][1] = -2.0f * kC3[5] * y * z;
                g[14][2] = kC3[5] * (xx - yy);
                g[15][0] = kC3[6] * (3.0f * xx - 3.0f * yy); g[15][1] = -6.0f * kC3[6] * x * y;
                g[15][2] = 0.0f;
            }
        }
    }
}

// Per-Gaussian projection values (train_oracle.py:125-181), fp32.
struct Geo {
    float x, y, z, iz;
    bool valid;
    float u, v;
    float qn[4], qinv;
    float Rq[9];
    float s[3];
    float S[6];       // cov3d: s00 s01 s02 s11 s12 s22
    float T0[3], T1[3];
    float a, b, c;    // low-passed 2D covariance
    float A, B, C;    // conic
};

__device__ __forceinline__ float s3(const float* S, int i, int k) {
    const int lo = i < k ? i : k, hi = i < k ? k : i;
    return lo == 0 ? S[hi] : (lo == 1 ? S[2 + hi] : S[5]);
}

// Layout of a parameter row (gs_internal.h).
template <int DEG>
struct Row {
    static constexpr int K = (DEG + 1) * (DEG + 1);
    static constexpr int V = (11 + 3 * K + 3) / 4;  // float4 per row
    static constexpr int S = 4 * V;
};

// The first three float4 of a row: mean, log-scale, quaternion, opacity logit
// and the first SH value.
struct Head {
    float4 a, b, c;
};
__device__ __forceinline__ Head load_head(const float4* row) { return Head{row[0], row[1], row[2]}; }

// SH values 0 .. 3K-1 of a row (the padding after them is zero).
template <int DEG>
__device__ __forceinline__ void load_sh(const float4* row, const Head& h, float* sh) {
    sh[0] = h.c.w;
#pragma unroll
    for (int q = 3; q < Row<DEG>::V; ++q) {
        const float4 f = row[q];
        const float t[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (4 * (q - 3) + 1 + e < 3 * Row<DEG>::K) sh[4 * (q - 3) + 1 + e] = t[e];
    }
}

__device__ __forceinline__ void geometry(const Head& h, const TrainCam& cam, Geo& g) {
    const float mx = h.a.x, my = h.a.y, mz = h.a.z;
    const float* R = cam.r;
    g.x = R[0] * mx + R[1] * my + R[2] * mz + cam.t[0];
    g.y = R[3] * mx + R[4] * my + R[5] * mz + cam.t[1];
    g.z = R[6] * mx + R[7] * my + R[8] * mz + cam.t[2];
    g.valid = g.z > cam.near;
    const float zs = g.valid ? g.z : 1.0f;
    g.iz = 1.0f / zs;
    g.u = cam.fx * g.x * g.iz + cam.cx;
    g.v = cam.fy * g.y * g.iz + cam.cy;
    const float q0 = h.b.z, q1 = h.b.w, q2 = h.c.x, q3 = h.c.y;
    g.qinv = 1.0f / sqrtf(q0 * q0 + q1 * q1 + q2 * q2 + q3 * q3);
    const float w = q0 * g.qinv, x = q1 * g.qinv, y = q2 * g.qinv, z = q3 * g.qinv;
    g.qn[0] = w; g.qn[1] = x; g.qn[2] = y; g.qn[3] = z;
    float* Q = g.Rq;
    Q[0] = 1.0f - 2.0f * (y * y + z * z); Q[1] = 2.0f * (x * y - w * z); Q[2] = 2.0f * (x * z + w * y);
    Q[3] = 2.0f * (x * y + w * z); Q[4] = 1.0f - 2.0f * (x * x + z * z); Q[5] = 2.0f * (y * z - w * x);
    Q[6] = 2.0f * (x * z - w * y); Q[7] = 2.0f * (y * z + w * x); Q[8] = 1.0f - 2.0f * (x * x + y * y);
    g.s[0] = expf(h.a.w);
    g.s[1] = expf(h.b.x);
    g.s[2] = expf(h.b.y);
    float M[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int k = 0; k < 3; ++k) M[3 * r + k] = Q[3 * r + k] * g.s[k];
    int idx = 0;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int k = r; k < 3; ++k)
            g.S[idx++] = M[3 * r] * M[3 * k] + M[3 * r + 1] * M[3 * k + 1] + M[3 * r + 2] * M[3 * k + 2];
    const float j00 = cam.fx * g.iz, j02 = -cam.fx * g.x * g.iz * g.iz;
    const float j11 = cam.fy * g.iz, j12 = -cam.fy * g.y * g.iz * g.iz;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        g.T0[k] = j00 * R[k] + j02 * R[6 + k];
        g.T1[k] = j11 * R[3 + k] + j12 * R[6 + k];
    }
    float CT0[3], CT1[3];
#pragma unroll
    for (int r = 0; r < 3; ++r) {
        CT0[r] = s3(g.S, r, 0) * g.T0[0] + s3(g.S, r, 1) * g.T0[1] + s3(g.S, r, 2) * g.T0[2];
        CT1[r] = s3(g.S, r, 0) * g.T1[0] + s3(g.S, r, 1) * g.T1[1] + s3(g.S, r, 2) * g.T1[2];
    }
    g.a = g.T0[0] * CT0[0] + g.T0[1] * CT0[1] + g.T0[2] * CT0[2] + cam.lowpass;
    g.b = g.T1[0] * CT0[0] + g.T1[1] * CT0[1] + g.T1[2] * CT0[2];
    g.c = g.T1[0] * CT1[0] + g.T1[1] * CT1[1] + g.T1[2] * CT1[2] + cam.lowpass;
    const float det = g.a * g.c - g.b * g.b;
    g.A = g.c / det;
    g.B = -g.b / det;
    g.C = g.a / det;
}

// SH colour + 0.5 of a row's Gaussian; the coefficients are read as they are used.
template <int DEG>
__device__ __forceinline__ void colour(const Head& h, const float4* row, const TrainCam& cam,
                                       float* raw, float* dir, float& dnorm) {
    const float dx = h.a.x - cam.ccx, dy = h.a.y - cam.ccy, dz = h.a.z - cam.ccz;
    dnorm = sqrtf(dx * dx + dy * dy + dz * dz);
    dir[0] = dx / dnorm; dir[1] = dy / dnorm; dir[2] = dz / dnorm;
    float b[16];
    sh_basis<DEG, false>(dir[0], dir[1], dir[2], b, nullptr);
    float acc[3] = {0.0f, 0.0f, 0.0f};
    acc[0] += b[0] * h.c.w;
#pragma unroll
    for (int q = 3; q < Row<DEG>::V; ++q) {
        const float4 f = row[q];
        const float t[4] = {f.x, f.y, f.z, f.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 4 * (q - 3) + 1 + e;  // SH value 3k + channel
            if (j < 3 * Row<DEG>::K) acc[j % 3] += b[j / 3] * t[e];
        }
    }
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) raw[ch] = acc[ch] + 0.5f;
}

__device__ __forceinline__ bool finite3(float x, float y, float z) {
    const float inf = __builtin_inff();
    return fabsf(x) < inf && fabsf(y) < inf && fabsf(z) < inf;
}

__device__ __forceinline__ float sigmoidf(float x) { return 1.0f / (1.0f + expf(-x)); }

// Projection of the optimizer-space parameters; stable compaction of the
// Gaussians that can reach alpha_min somewhere in the image. As the render's
// projection: the geometry of a thread's four rows first, held in LDS (in
// registers, with the colours, it left one workgroup on a CU), the partition's
// count published, then the colours of the kept rows, which are the largest
// reads, then the walk over the predecessors. BINNED as there.
// (1M Gaussians, SH1: 48.5 -> 40.3 us; with the tile counts' scan.)
// ITEMS as there too (a 20K step's loop 1263 -> 1235 us, a 50K gradient call 722 -> 713).
template <int DEG, bool BINNED, int ITEMS>
__global__ __launch_bounds__(kTThreads, 4) void k_train_project(
    TrainParamsDev P, TrainCam cam, Compact out, float4* __restrict__ trec,
    uint32_t* __restrict__ cidx, uint8_t* __restrict__ visible, uint64_t* lb_state,
    uint32_t* ticket, uint32_t* count_out, uint32_t* __restrict__ part_hist, TrainDebug dbg) {
    constexpr int V = Row<DEG>::V, kWaves = kTThreads / GS_WAVE;
    __shared__ uint32_t s_vid;
    __shared__ uint32_t s_cnt[ITEMS][kWaves], s_ccnt[ITEMS][kWaves];
    __shared__ uint32_t s_hist[BINNED ? 1 : 4][256];
    __shared__ float4 s_iv[2][ITEMS][kTThreads];
    __shared__ uint64_t s_excl;
    const int tid = threadIdx.x, w = tid / GS_WAVE, lane = lane_id();
    if (tid == 0) s_vid = atomicAdd(ticket, 1u);
    if (!BINNED)
        for (int k = tid; k < 1024; k += kTThreads) (&s_hist[0][0])[k] = 0;
    __syncthreads();
    const uint32_t vid = s_vid;
    const int64_t base = (int64_t)vid * (kTThreads * ITEMS);
    const int64_t n = P.n;
    bool keep[ITEMS];
    float ops[ITEMS], m2[ITEMS];
    uint32_t coff[ITEMS];
    uint64_t bal[ITEMS];
    // the heads of a thread's rows together (past the end: the last row's)
    Head head[ITEMS];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it)
        head[it] = load_head(P.rows + min(base + it * kTThreads + tid, n - 1) * V);
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        const int64_t i = base + it * kTThreads + tid;
        Geo g;
        geometry(head[it], cam, g);
        const float op = sigmoidf(head[it].c.z);
        // sparse-Adam rows: 3-sigma box overlaps the image (train_oracle.py:175-181)
        const float rx3 = ceilf(3.0f * sqrtf(fmaxf(g.a, 0.0f)));
        const float ry3 = ceilf(3.0f * sqrtf(fmaxf(g.c, 0.0f)));
        const bool vis = g.valid && (g.u + rx3 > 0.0f) && (g.u - rx3 < (float)cam.W) &&
                         (g.v + ry3 > 0.0f) && (g.v - ry3 < (float)cam.H);
        // blendable: alpha = op exp(power) >= alpha_min somewhere in the image
        bool k = i < n && g.valid && op >= cam.alpha_min && g.a * g.c - g.b * g.b > 0.0f;
        float m2thr = 0.0f, rx = 0.0f, ry = 0.0f;
        if (k) {
            m2thr = 2.0f * logf(op / cam.alpha_min);
            const float kk = sqrtf(m2thr);
            rx = ceilf(kk * sqrtf(fmaxf(g.a, 0.0f)));
            ry = ceilf(kk * sqrtf(fmaxf(g.c, 0.0f)));
            k = rx > 0.0f && ry > 0.0f && (g.u + rx > 0.0f) && (g.u - rx < (float)cam.W) &&
                (g.v + ry > 0.0f) && (g.v - ry < (float)cam.H);
        }
        keep[it] = k;
        ops[it] = op;
        m2[it] = m2thr;
        if (i < n) {
            visible[i] = vis ? 1 : 0;
            if (!k) cidx[i] = 0xFFFFFFFFu;
            if (dbg.means2d != nullptr) {  // parity outputs, the colours of all
                float raw[3], dir[3], dn;
                colour<DEG>(head[it], P.rows + i * V, cam, raw, dir, dn);
                dbg.means2d[2 * i] = g.u;
                dbg.means2d[2 * i + 1] = g.v;
                dbg.conic[3 * i] = g.A;
                dbg.conic[3 * i + 1] = g.B;
                dbg.conic[3 * i + 2] = g.C;
                dbg.opacity[i] = op;
                for (int ch = 0; ch < 3; ++ch)
                    dbg.colors[3 * i + ch] = raw[ch] < 0.0f ? 0.0f : raw[ch];
                dbg.depth[i] = g.z;
                dbg.valid[i] = g.valid ? 1 : 0;
            }
        }
        s_iv[0][it][tid] = make_float4(g.u, g.v, rx, ry);
        s_iv[1][it][tid] = make_float4(g.a, g.b, g.c, g.z);
        bal[it] = __ballot(k);
        if (lane == 0) s_cnt[it][w] = (uint32_t)__popcll(bal[it]);
        if constexpr (BINNED) {
            const uint32_t c = k ? rect_tiles(g.u, g.v, rx, ry, cam.tiles_x, cam.tiles_y, 16) : 0u;
            const uint32_t incl = wave_incl_scan(c);
            coff[it] = incl - c;
            if (lane == GS_WAVE - 1) s_ccnt[it][w] = incl;
        } else {
            const uint32_t key = __float_as_uint(g.z);
            hist_add_wave(s_hist[0], key & 255u, k);
            hist_add_wave(s_hist[1], (key >> 8) & 255u, k);
            hist_add_wave(s_hist[2], (key >> 16) & 255u, k);
            hist_add_wave(s_hist[3], key >> 24, k);
        }
    }
    __syncthreads();
    if (!BINNED)
        for (int k = tid; k < 1024; k += kTThreads)
            part_hist[(size_t)vid * 1024 + k] = (&s_hist[0][0])[k];
    // exclusive prefixes of the (item, wave) counts in source order: lane
    // it * waves + w of a wave scan
    static_assert(ITEMS * kWaves <= GS_WAVE, "one count per lane");
    uint32_t total, my_off[ITEMS];
    uint64_t ctotal = 0;
    {
        const uint32_t c = lane < ITEMS * kWaves ? (&s_cnt[0][0])[lane] : 0u;
        const uint32_t incl = wave_incl_scan(c);
        total = (uint32_t)__builtin_amdgcn_readlane((int)incl, GS_WAVE - 1);
#pragma unroll
        for (int it = 0; it < ITEMS; ++it)
            my_off[it] = (uint32_t)__builtin_amdgcn_readlane((int)(incl - c), it * kWaves + w);
        if constexpr (BINNED) {
            const uint32_t cc = lane < ITEMS * kWaves ? (&s_ccnt[0][0])[lane] : 0u;
            const uint32_t ci = wave_incl_scan(cc);
            ctotal = (uint32_t)__builtin_amdgcn_readlane((int)ci, GS_WAVE - 1);
#pragma unroll
            for (int it = 0; it < ITEMS; ++it)
                coff[it] += (uint32_t)__builtin_amdgcn_readlane((int)(ci - cc), it * kWaves + w);
        }
    }
    const uint64_t agg = BINNED ? binned_pack(total, ctotal) : (uint64_t)total;
    if (w == 0) lookback_publish(lb_state, vid, agg);
    float col[ITEMS][3];
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        if (!keep[it]) continue;
        const float4* row = P.rows + (base + it * kTThreads + tid) * V;
        float dir[3], dn;
        colour<DEG>(load_head(row), row, cam, col[it], dir, dn);
        if (!finite3(col[it][0], col[it][1], col[it][2])) *cam.odd = 1u;
    }
    if (w == 0) {
        const uint64_t excl = lookback_walk(lb_state, vid, agg, cam.ctl);
        if (lane == 0) {
            s_excl = excl;
            if (vid == gridDim.x - 1) {
                if constexpr (BINNED)
                    binned_totals(excl + agg, count_out, cam.binned, cam.ctl);
                else
                    *count_out = (uint32_t)(excl + agg);
            }
        }
    }
    __syncthreads();
    const uint64_t excl = BINNED ? binned_count(s_excl) : s_excl;
    const uint64_t ltm = lanemask_lt();
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
        if (!keep[it]) continue;
        const int64_t i = base + it * kTThreads + tid;
        const uint64_t m = excl + my_off[it] + (uint64_t)__popcll(bal[it] & ltm);
        const float4 q0 = s_iv[0][it][tid], q1 = s_iv[1][it][tid];
        const float a = q1.x, b = q1.y, c = q1.z, det = a * c - b * b;
        out.rc[2 * m + 0] = q0;
        out.rc[2 * m + 1] = make_float4(a, b, c, m2[it]);
        out.dkey[m] = __float_as_uint(q1.w);
        trec[3 * m + 0] = make_float4(q0.x, q0.y, ops[it], m2[it]);
        trec[3 * m + 1] = make_float4(c / det, -b / det, a / det, 0.0f);
        trec[3 * m + 2] = make_float4(col[it][0] < 0.0f ? 0.0f : col[it][0],
                                      col[it][1] < 0.0f ? 0.0f : col[it][1],
                                      col[it][2] < 0.0f ? 0.0f : col[it][2], 0.0f);
        out.src[m] = (uint32_t)i;
        cidx[i] = (uint32_t)m;
        if constexpr (BINNED)
            binned_write(cam.binned, m, binned_cands(s_excl) + coff[it],
                         rect_tiles(q0.x, q0.y, q0.z, q0.w, cam.tiles_x, cam.tiles_y, 16));
        if (cam.grad2d != nullptr) {  // the step's backward adds into these
#pragma unroll
            for (int k = 0; k < 9; ++k) cam.grad2d[9 * m + k] = 0.0f;
        }
    }
}

// ---------------------------------------------------------------------------
// Blend forward and backward. One wave64 (its own workgroup, no barriers
// between waves) owns a 16x4 pixel band of a 16x16 tile, lane = row * 16 +
// column, and walks the tile's depth-ordered entries 64 at a time: lane q tests
// entry q against the whole band (band_keeps) and the kept ones are packed into
// LDS, so that the per-pixel work is spent on entries that reach the band. The
// next batch's records are loaded while this one is walked. Both are bound by
// VALU issue, the longest tile lists by the latency of one wave's chain, which is
// why a band is a workgroup of its own: four waves per tile finish independently.
// Measured against 256-thread tile workgroups that evaluated every entry at
// every pixel behind a barrier per batch (per step, 1M Gaussians at 1280x720):
// forward 286 -> 124 us, backward 609 -> 318 us; 20K Gaussians at 200x152:
// 58 -> 17 and 74 -> 26 us.
// ---------------------------------------------------------------------------
constexpr int kBandRows = 4;
constexpr int kBandsPerTile = 16 / kBandRows;

// False only when alpha = op exp(-q/2) stays below alpha_min at every pixel
// centre of the band whose first centre is (x0, y0): the least q over the
// rectangle of centres, on the edges facing the Gaussian's centre, is past
// m2thr = 2 ln(op / alpha_min). The margin covers the rounding of this test and
// of the per-pixel evaluation (a few ulp of the largest term), so no entry that
// any pixel would blend is dropped; NaN keeps.
__device__ __forceinline__ bool band_keeps(float4 r0, float4 r1, float x0, float y0) {
    const float A = r1.x, B = r1.y, C = r1.z;
    const float ul = x0 - r0.x, uh = ul + 15.0f;
    const float vl = y0 - r0.y, vh = vl + (float)(kBandRows - 1);
    const bool xin = ul <= 0.0f && uh >= 0.0f, yin = vl <= 0.0f && vh >= 0.0f;
    const float uf = ul > 0.0f ? ul : uh, vf = vl > 0.0f ? vl : vh;
    const float vs = fminf(fmaxf(-B * uf * __builtin_amdgcn_rcpf(C), vl), vh);
    const float us = fminf(fmaxf(-B * vf * __builtin_amdgcn_rcpf(A), ul), uh);
    const float a1 = A * uf * uf, b1 = 2.0f * B * uf * vs, c1 = C * vs * vs;
    const float a2 = A * us * us, b2 = 2.0f * B * us * vf, c2 = C * vf * vf;
    const float tol = 4e-6f;
    const float q1 = (a1 + b1 + c1) - tol * (a1 + fabsf(b1) + c1);
    const float q2 = (a2 + b2 + c2) - tol * (a2 + fabsf(b2) + c2);
    const float lim = r0.w + 1e-4f;
    const bool far1 = !xin && q1 > lim, far2 = !yin && q2 > lim;
    // the nearest point lies on one of the facing edges: dropped when each of them is far
    return !((far1 || xin) && (far2 || yin) && !(xin && yin));
}

// One entry at one pixel: power = -0.5 (A dx^2 + 2 B dx dy + C dy^2) in the order
// of train_oracle.py:199-203, each operation rounded, the same in the forward
// and the backward, so both see the same alpha.
struct Splat {
    float dx, dy, adx, cdy, power, w, raw;
};
__device__ __forceinline__ Splat splat_at(float px, float py, float u, float v, float A, float B,
                                          float C, float op) {
    Splat s;
    s.dx = px - u;
    s.dy = py - v;
    s.adx = A * s.dx;
    s.cdy = C * s.dy;
    s.power = -0.5f * (s.adx * s.dx + 2.0f * B * s.dx * s.dy + s.cdy * s.dy);
    s.w = __expf(fminf(s.power, 0.0f));
    s.raw = op * s.w;
    return s;
}

// Forward of one band (3DGS rules, train_oracle.py:196-229). Writes the image,
// the final transmittance, the entry index where the pixel stopped, and - with
// a target - the L1 gradient and the loss.
__global__ __launch_bounds__(GS_WAVE) void k_train_fwd(const float4* __restrict__ trec,
                                                       const uint32_t* __restrict__ sid,
                                                       const uint32_t* __restrict__ ranges,
                                                       TrainFwdParams fp) {
    __shared__ float4 s0[GS_WAVE], s1[GS_WAVE];
    __shared__ float2 s2[GS_WAVE];
    // after an earlier give-up the sorted ids may be wrong: read nothing (the
    // flag was raised by an earlier launch, so every thread sees the same value)
    if (upstream_failed(fp.ctl)) return;
    const bool any_odd = __builtin_amdgcn_readfirstlane((int)*fp.odd) != 0;
    const int lane = threadIdx.x;
    const int tile = blockIdx.x / kBandsPerTile, band = blockIdx.x % kBandsPerTile;
    const int tx = tile % fp.tiles_x, ty = tile / fp.tiles_x;
    const int px = tx * 16 + (lane & 15), py = ty * 16 + band * kBandRows + (lane >> 4);
    const bool inside = px < fp.width && py < fp.height;
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const float bx0 = (float)(tx * 16) + 0.5f, by0 = (float)(ty * 16 + band * kBandRows) + 0.5f;
    const uint32_t start = ranges[2 * tile], end = ranges[2 * tile + 1];
    float T = 1.0f, cr = 0.0f, cg = 0.0f, cb = 0.0f;
    bool done = !inside;
    uint32_t stop = end - start;
    uint32_t blended = 0;  // of the wave
    if (start < end && __ballot(inside) != 0ull) {
        uint32_t gi = sid[min(start + lane, end - 1)];
        float4 r0 = trec[3 * (size_t)gi + 0], r1 = trec[3 * (size_t)gi + 1],
               r2 = trec[3 * (size_t)gi + 2];
        gi = sid[min(start + GS_WAVE + lane, end - 1)];
        for (uint32_t base = start; base < end; base += GS_WAVE) {
            const bool keep = base + lane < end && band_keeps(r0, r1, bx0, by0);
            const uint64_t mask = __ballot(keep);
            // kept entries whose colours are not finite
            const uint64_t odd = any_odd ? __ballot(keep && !finite3(r2.x, r2.y, r2.z)) : 0ull;
            const int cnt = __popcll(mask);
            __syncthreads();  // one wave: orders the LDS reads of the batch before
            if (keep) {
                const int k = __popcll(mask & lanemask_lt());
                s0[k] = make_float4(r0.x, r0.y, r0.z, r1.x);
                s1[k] = make_float4(r1.y, r1.z, r2.x, r2.y);
                s2[k] = make_float2(r2.z, __uint_as_float(base - start + lane));
            }
            if (lane >= cnt && lane < ((cnt + 3) & ~3)) {  // opacity 0: blends nowhere
                s0[lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                s1[lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
                s2[lane] = make_float2(0.0f, 0.0f);
            }
            r0 = trec[3 * (size_t)gi + 0];
            r1 = trec[3 * (size_t)gi + 1];
            r2 = trec[3 * (size_t)gi + 2];
            gi = sid[min(base + 2 * GS_WAVE + lane, end - 1)];
            __syncthreads();
            // An entry that the pixel does not blend adds 0 times its colour, but where a
            // colour of the batch is not finite the sums are selected instead (1M Gaussians
            // at 1280x720: 117 us with and without that walk, 119 when it is unrolled as the
            // other, 123.5 with selects in every batch; 20K 21.2 without, 21.5 with it).
            const auto blend = [&](int k, auto select) {
                const float4 e0 = s0[k], e1 = s1[k];
                const float2 e2 = s2[k];
                const Splat s = splat_at(pxc, pyc, e0.x, e0.y, e0.w, e1.x, e1.y, e0.z);
                const float alpha = fminf(s.raw, fp.alpha_max);
                const bool live = alpha >= fp.alpha_min && !done;
                const float tn = T * (1.0f - alpha);
                const bool hit = live && tn < fp.t_min;
                const bool bl = live && !hit;
                done = done || hit;
                stop = hit ? __float_as_uint(e2.y) : stop;
                const float at = bl ? alpha * T : 0.0f;
                if constexpr (decltype(select)::value) {
                    cr = bl ? cr + at * e1.z : cr;
                    cg = bl ? cg + at * e1.w : cg;
                    cb = bl ? cb + at * e2.x : cb;
                } else {
                    cr += at * e1.z;
                    cg += at * e1.w;
                    cb += at * e2.x;
                }
                T = bl ? tn : T;
                blended += (uint32_t)__popcll(__ballot(bl));
            };
            if (__builtin_expect(odd == 0ull, 1)) {
                for (int k = 0; k < cnt; k += 4) {
#pragma unroll
                    for (int j = 0; j < 4; ++j) blend(k + j, std::false_type{});
                    if (__ballot(!done) == 0ull) break;
                }
            } else {
#pragma unroll 1
                for (int k = 0; k < cnt && __ballot(!done) != 0ull; ++k) blend(k, std::true_type{});
            }
            if (__ballot(!done) == 0ull) break;
        }
    }
    double lsum = 0.0;
    if (inside) {
        const size_t p = (size_t)py * fp.width + px;
        const float o[3] = {cr + T * fp.bg[0], cg + T * fp.bg[1], cb + T * fp.bg[2]};
        fp.image[3 * p + 0] = o[0];
        fp.image[3 * p + 1] = o[1];
        fp.image[3 * p + 2] = o[2];
        fp.final_T[p] = T;
        fp.stop[p] = stop;
        if (fp.target != nullptr) {
#pragma unroll
            for (int ch = 0; ch < 3; ++ch) {
                const float d = o[ch] - fp.target[3 * p + ch];
                const float sg = d > 0.0f ? 1.0f : (d < 0.0f ? -1.0f : 0.0f);
                fp.dimage[3 * p + ch] = sg * fp.grad_scale;
                lsum += (double)fabsf(d);
            }
        }
    }
    // sums into one of kTrainSumSlots groups (one address for all of a
    // launch's thousands of waves would serialise them); the host adds the groups
    TrainSums* const slot = fp.sums + blockIdx.x % kTrainSumSlots;
    if (fp.target != nullptr) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) lsum += __shfl_xor(lsum, o, GS_WAVE);
        if (lane == 0) atomicAdd(&slot->l1, lsum);
    }
    uint32_t pc = inside ? stop : 0u;  // a band's 64 stops, each below 2^26
    unsigned long long pcw = pc;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) pcw += __shfl_xor(pcw, o, GS_WAVE);
    if (lane == 0) {
        atomicAdd(&slot->considered, pcw);
        atomicAdd(&slot->blended, (unsigned long long)blended);
    }
}

// ---------------------------------------------------------------------------
// Full 3DGS loss (train_oracle.py:253-279): SSIM with an 11-tap Gaussian window
// (sigma 1.5), zero padding, S = A B / (C D); the image gradient in the
// fused-SSIM form of train_loss.py:5-19. A workgroup takes one channel of 32 x 22
// pixels: 32 halo rows are one row-pass unit of four adjacent outputs per thread
// (14 values read for four of 11 taps each), the column pass gives each thread
// three outputs of a column from 13 rows, and products go into fused adds (which
// also drop a rounding): a quarter of the LDS reads and half of the VALU issue of
// one output per thread on 16 x 16 tiles. Bound by both still (800x600, forward and
// backward: 35.3 -> 25.1 and 38.6 -> 23.3 us; 501x333: 16.0 -> 10.8 and 13.6 -> 9.9).
// The gradient's terms are formed from products, not as quotients of S by A and B, which
// pass through 0 (0 / 0 there; two divisions a pixel for seven: 25.1 -> 23.5 us).
// ---------------------------------------------------------------------------
constexpr int kSsimW = 32, kSsimH = 22, kSsimR = 5;
constexpr int kSsimEW = kSsimW + 2 * kSsimR, kSsimEH = kSsimH + 2 * kSsimR;  // with the halo
constexpr int kSsimX = 44, kSsimHs = 36;  // row strides in LDS, whole float4
constexpr int kSsimCol = 3;               // outputs of a column per thread
constexpr int kSsimHRows = 256 / kSsimW * kSsimCol + 2 * kSsimR;  // rows that the column pass reads
static_assert(kSsimEH * (kSsimW / 4) == 256, "one row-pass unit per thread");
static_assert(256 / kSsimW * kSsimCol >= kSsimH && kSsimHRows >= kSsimEH, "the columns are covered");

// Sixteen values of an LDS row: the taps of four adjacent outputs.
__device__ __forceinline__ void load14(const float* row, float (&v)[16]) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 q = reinterpret_cast<const float4*>(row)[i];
        v[4 * i] = q.x;
        v[4 * i + 1] = q.y;
        v[4 * i + 2] = q.z;
        v[4 * i + 3] = q.w;
    }
}
// The column filter of Q planes at kSsimCol outputs from row r0 of column c.
template <int Q>
__device__ __forceinline__ void ssim_columns(const float (*h)[kSsimHRows][kSsimHs], int r0, int c,
                                             const float* g, float (&acc)[kSsimCol][Q]) {
#pragma unroll
    for (int j = 0; j < kSsimCol; ++j)
#pragma unroll
        for (int q = 0; q < Q; ++q) acc[j][q] = 0.0f;
#pragma unroll
    for (int r = 0; r < kSsimCol + 2 * kSsimR; ++r) {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const float v = h[q][r0 + r][c];
#pragma unroll
            for (int j = 0; j < kSsimCol; ++j)
                if (r >= j && r - j <= 2 * kSsimR) acc[j][q] = fmaf(g[r - j], v, acc[j][q]);
        }
    }
}

// Forward: mu_x, mu_y, E_xx, E_yy, E_xy -> S and the three per-pixel terms
// w dS/dmu_x, w dS/dE_xx, w dS/dE_xy (planes by term and channel), sum of S.
__global__ __launch_bounds__(256) void k_ssim_fwd(SsimParams sp) {
    __shared__ __attribute__((aligned(16))) float s_x[kSsimEH][kSsimX], s_y[kSsimEH][kSsimX];
    __shared__ __attribute__((aligned(16))) float s_h[5][kSsimHRows][kSsimHs];
    __shared__ double s_sum[4];
    const int tid = threadIdx.x;
    const int tiles_x = (sp.width + kSsimW - 1) / kSsimW;
    const int tiles = tiles_x * ((sp.height + kSsimH - 1) / kSsimH);
    const int ch = blockIdx.x / tiles, t = blockIdx.x % tiles;
    const int x0 = t % tiles_x * kSsimW, y0 = t / tiles_x * kSsimH;
    const size_t npx = (size_t)sp.width * sp.height;
    for (int i = tid; i < kSsimEH * kSsimEW; i += 256) {
        const int r = i / kSsimEW, c = i % kSsimEW;
        const int gx = x0 - kSsimR + c, gy = y0 - kSsimR + r;
        float xv = 0.0f, yv = 0.0f;
        if (gx >= 0 && gx < sp.width && gy >= 0 && gy < sp.height) {
            const size_t q = ((size_t)gy * sp.width + gx) * 3 + ch;
            xv = sp.image[q];
            yv = sp.target[q];
        }
        s_x[r][c] = xv;
        s_y[r][c] = yv;
    }
    __syncthreads();
    {
        const int r = tid / (kSsimW / 4), c = tid % (kSsimW / 4) * 4;
        float v[5][16], h[5][4] = {};
        load14(&s_x[r][c], v[0]);
        load14(&s_y[r][c], v[1]);
#pragma unroll
        for (int i = 0; i < kSsimR * 2 + 4; ++i) {
            v[2][i] = v[0][i] * v[0][i];
            v[3][i] = v[1][i] * v[1][i];
            v[4][i] = v[0][i] * v[1][i];
        }
#pragma unroll
        for (int q = 0; q < 5; ++q)
#pragma unroll
            for (int k = 0; k < 2 * kSsimR + 1; ++k)
#pragma unroll
                for (int j = 0; j < 4; ++j) h[q][j] = fmaf(sp.g[k], v[q][j + k], h[q][j]);
#pragma unroll
        for (int q = 0; q < 5; ++q)
            *reinterpret_cast<float4*>(&s_h[q][r][c]) = make_float4(h[q][0], h[q][1], h[q][2], h[q][3]);
    }
    __syncthreads();
    const int lx = tid % kSsimW, r0 = tid / kSsimW * kSsimCol;
    float m[kSsimCol][5];
    ssim_columns<5>(s_h, r0, lx, sp.g, m);
    double ssum = 0.0;
#pragma unroll
    for (int j = 0; j < kSsimCol; ++j) {
        const int px = x0 + lx, py = y0 + r0 + j;
        if (r0 + j < kSsimH && px < sp.width && py < sp.height) {
            const float mu_x = m[j][0], mu_y = m[j][1], e_xx = m[j][2], e_yy = m[j][3];
            const float c1 = 0.01f * 0.01f, c2 = 0.03f * 0.03f;
            const float mxy = mu_x * mu_y;
            const float A = 2.0f * mxy + c1;
            const float B = 2.0f * fmaf(-mu_x, mu_y, m[j][4]) + c2;
            const float C = mu_x * mu_x + mu_y * mu_y + c1;
            const float D = fmaf(-mu_x, mu_x, e_xx) + fmaf(-mu_y, mu_y, e_yy) + c2;
            const float icd = 1.0f / (C * D), S = A * B * icd;
            const float d_mu = 2.0f * sp.w * icd * fmaf(mu_y, B - A, mu_x * S * (C - D));
            float* map = sp.maps + (size_t)ch * npx + (size_t)py * sp.width + px;
            map[0] = d_mu;
            map[3 * npx] = -sp.w * S / D;
            map[6 * npx] = 2.0f * sp.w * A * icd;
            ssum += (double)S;
        }
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) ssum += __shfl_xor(ssum, o, GS_WAVE);
    if (lane_id() == 0) s_sum[tid / GS_WAVE] = ssum;
    __syncthreads();
    if (tid == 0)
        atomicAdd(&sp.sums[blockIdx.x % kTrainSumSlots].ssim,
                  (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]));
}

// Backward: dimage += G*(w dS/dmu_x) + 2 x G*(w dS/dE_xx) + y G*(w dS/dE_xy)
// (G symmetric, so its adjoint is the same zero-padded filter).
__global__ __launch_bounds__(256) void k_ssim_bwd(SsimParams sp) {
    __shared__ __attribute__((aligned(16))) float s_m[3][kSsimEH][kSsimX];
    __shared__ __attribute__((aligned(16))) float s_h[3][kSsimHRows][kSsimHs];
    const int tid = threadIdx.x;
    const int tiles_x = (sp.width + kSsimW - 1) / kSsimW;
    const int tiles = tiles_x * ((sp.height + kSsimH - 1) / kSsimH);
    const int ch = blockIdx.x / tiles, t = blockIdx.x % tiles;
    const int x0 = t % tiles_x * kSsimW, y0 = t / tiles_x * kSsimH;
    const size_t npx = (size_t)sp.width * sp.height;
    const float* map = sp.maps + (size_t)ch * npx;
    for (int i = tid; i < kSsimEH * kSsimEW; i += 256) {
        const int r = i / kSsimEW, c = i % kSsimEW;
        const int gx = x0 - kSsimR + c, gy = y0 - kSsimR + r;
        const bool in = gx >= 0 && gx < sp.width && gy >= 0 && gy < sp.height;
        const size_t q = in ? (size_t)gy * sp.width + gx : 0;
#pragma unroll
        for (int p = 0; p < 3; ++p) s_m[p][r][c] = in ? map[(size_t)(3 * p) * npx + q] : 0.0f;
    }
    __syncthreads();
    {
        const int r = tid / (kSsimW / 4), c = tid % (kSsimW / 4) * 4;
#pragma unroll
        for (int p = 0; p < 3; ++p) {
            float v[16], h[4] = {};
            load14(&s_m[p][r][c], v);
#pragma unroll
            for (int k = 0; k < 2 * kSsimR + 1; ++k)
#pragma unroll
                for (int j = 0; j < 4; ++j) h[j] = fmaf(sp.g[k], v[j + k], h[j]);
            *reinterpret_cast<float4*>(&s_h[p][r][c]) = make_float4(h[0], h[1], h[2], h[3]);
        }
    }
    __syncthreads();
    const int lx = tid % kSsimW, r0 = tid / kSsimW * kSsimCol;
    float m[kSsimCol][3];
    ssim_columns<3>(s_h, r0, lx, sp.g, m);
#pragma unroll
    for (int j = 0; j < kSsimCol; ++j) {
        const int px = x0 + lx, py = y0 + r0 + j;
        if (r0 + j < kSsimH && px < sp.width && py < sp.height) {
            const size_t q = ((size_t)py * sp.width + px) * 3 + ch;
            sp.dimage[q] += m[j][0] + 2.0f * sp.image[q] * m[j][1] + sp.target[q] * m[j][2];
        }
    }
}

// dimage = scale * sign(image - target), sum |image - target| (stage path).
__global__ __launch_bounds__(256) void k_l1(const float* __restrict__ image,
                                            const float* __restrict__ target, int64_t count,
                                            float scale, float* __restrict__ dimage,
                                            TrainSums* sums) {
    __shared__ double s_sum[4];
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    double a = 0.0;
    if (i < count) {
        const float d = image[i] - target[i];
        dimage[i] = (d > 0.0f ? 1.0f : (d < 0.0f ? -1.0f : 0.0f)) * scale;
        a = (double)fabsf(d);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) a += __shfl_xor(a, o, GS_WAVE);
    if (lane_id() == 0) s_sum[threadIdx.x / GS_WAVE] = a;
    __syncthreads();
    if (threadIdx.x == 0)
        atomicAdd(&sums[blockIdx.x % kTrainSumSlots].l1,
                  (s_sum[0] + s_sum[1]) + (s_sum[2] + s_sum[3]));
}

// v plus the value a DPP move brings into the lane (all lanes active).
template <int CTRL>
__device__ __forceinline__ float dpp_add(float keep, float give) {
    const int x = __builtin_amdgcn_update_dpp(0, __float_as_int(give), CTRL, 0xF, 0xF, false);
    return keep + __int_as_float(x);
}
constexpr int kDppXor1 = 0xB1;         // quad_perm 1,0,3,2
constexpr int kDppXor2 = 0x4E;         // quad_perm 2,3,0,1
constexpr int kDppHalfMirror = 0x141;  // lane 7 - l of each 8
constexpr int kDppRor8 = 0x128;        // lane l ^ 8 of each 16

// Lanes 0-31: the sum of a over lane pairs (l, l + 32); lanes 32-63: that of b.
__device__ __forceinline__ float pack32(float a, float b) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
// Even rows of 16 lanes: the sum of a over the row and the next one; odd rows: that of b.
__device__ __forceinline__ float pack16(float a, float b) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false,
                                                    false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// Sums the nine terms of two entries over the 64 lanes, all 18 of them in one
// register: at each halving of the lanes, two registers become one, half of the
// lanes carrying on with the one's term and half with the other's, so that the
// 18 sums take 43 vector instructions (one by one, six each: 108). Lane l
// returns the sum of term_of_lane(l) of entry l / 32.
__device__ __forceinline__ float sum_terms(const float (&a)[9], const float (&b)[9], bool bit3,
                                           bool bit2, bool bit1) {
    float r[9];
#pragma unroll
    for (int i = 0; i < 9; ++i) r[i] = pack32(a[i], b[i]);
    float q[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = pack16(r[i], r[i + 4]);
    float s8 = pack16(r[8], r[8]);
    float x0 = dpp_add<kDppRor8>(bit3 ? q[1] : q[0], bit3 ? q[0] : q[1]);
    float x1 = dpp_add<kDppRor8>(bit3 ? q[3] : q[2], bit3 ? q[2] : q[3]);
    s8 = dpp_add<kDppRor8>(s8, s8);
    float x = dpp_add<kDppHalfMirror>(bit2 ? x1 : x0, bit2 ? x0 : x1);
    s8 = dpp_add<kDppHalfMirror>(s8, s8);
    x = dpp_add<kDppXor2>(bit1 ? s8 : x, bit1 ? x : s8);
    return dpp_add<kDppXor1>(x, x);
}
__device__ __forceinline__ int term_of_lane(int l) {
    return (l & 2) ? 8 : ((l >> 4) & 1) * 4 + ((l >> 2) & 1) * 2 + ((l >> 3) & 1);
}

// Backward of one pixel by its lane, an atomic per term of each entry that it blends.
__device__ __forceinline__ void backward_alone(const float4* __restrict__ trec,
                                               const uint32_t* __restrict__ ids, uint32_t stop,
                                               float pxc, float pyc, float T, float g0, float g1,
                                               float g2, const TrainBwdParams& bp) {
    float behind = bp.bg[0] * g0 + bp.bg[1] * g1 + bp.bg[2] * g2;
#pragma unroll 1
    for (uint32_t e = stop; e-- > 0;) {
        const size_t gi = ids[e];
        const float4 r0 = trec[3 * gi + 0], r1 = trec[3 * gi + 1], r2 = trec[3 * gi + 2];
        const Splat s = splat_at(pxc, pyc, r0.x, r0.y, r1.x, r1.y, r1.z, r0.z);
        const float alpha = fminf(s.raw, bp.alpha_max);
        if (!(alpha >= bp.alpha_min)) continue;
        T = T * __builtin_amdgcn_rcpf(1.0f - alpha);
        const float d = __builtin_fmaf(r2.x, g0, __builtin_fmaf(r2.y, g1, r2.z * g2)) - behind;
        behind = __builtin_fmaf(alpha, d, behind);
        const float at = alpha * T;
        const float dop = s.raw > bp.alpha_max ? 0.0f : T * d;
        const float dp = s.power <= 0.0f ? dop * s.raw : 0.0f;
        const float dpx = dp * s.dx, dpy = dp * s.dy;
        float* const dst = bp.grad2d + 9 * gi;
        atomicAdd(dst + 0, dp * __builtin_fmaf(r1.y, s.dy, s.adx));
        atomicAdd(dst + 1, dp * __builtin_fmaf(r1.y, s.dx, s.cdy));
        atomicAdd(dst + 2, -0.5f * dpx * s.dx);
        atomicAdd(dst + 3, -dpx * s.dy);
        atomicAdd(dst + 4, -0.5f * dpy * s.dy);
        atomicAdd(dst + 5, dop * s.w);
        atomicAdd(dst + 6, at * g0);
        atomicAdd(dst + 7, at * g1);
        atomicAdd(dst + 8, at * g2);
    }
}

// Backward of one band: entries from the last one any of its pixels considered
// down to the first; per pixel the reverse recursion T_i = T_{i+1}/(1 - alpha_i)
// and, with s_i = c_i . g, behind_i = behind_{i+1} + alpha_{i+1} (s_{i+1} -
// behind_{i+1}) starting from the background's bg . g (the colours behind an
// entry are only ever needed through their product with the pixel's gradient),
// dL/dalpha_i = T_i (s_i - behind_i). A lane that does not blend the entry has
// alpha 0, which leaves T and behind as they are and contributes exact zeros - of finite
// values. A pixel whose gradient is not finite, or that blends a colour that is not (its
// image is not either), takes no part but goes its entries alone (backward_alone), and
// the others see such a colour as 0. (287 -> 289 us at 1M Gaussians, 33.9 at 20K; by
// selects, of behind in every pair and of the colours' terms in the bands of such
// gradients, 292 and 34.8.)
// The nine per-pair terms (dmx dmy dA dB dC dop dr dg db) of two entries at a
// time are summed over the wave (sum_terms) and 18 lanes add them to the
// Gaussians' accumulators, one atomic each. 1/(1 - alpha) is one reciprocal
// estimate.
__global__ __launch_bounds__(GS_WAVE) void k_train_bwd(const float4* __restrict__ trec,
                                                       const uint32_t* __restrict__ sid,
                                                       const uint32_t* __restrict__ ranges,
                                                       TrainBwdParams bp) {
    __shared__ float4 s0[GS_WAVE], s1[GS_WAVE], s2[GS_WAVE];
    if (upstream_failed(bp.ctl)) return;
    const bool any_odd = __builtin_amdgcn_readfirstlane((int)*bp.odd) != 0;
    const int lane = threadIdx.x;
    const int tile = blockIdx.x / kBandsPerTile, band = blockIdx.x % kBandsPerTile;
    const int tx = tile % bp.tiles_x, ty = tile / bp.tiles_x;
    const int px = tx * 16 + (lane & 15), py = ty * 16 + band * kBandRows + (lane >> 4);
    const bool inside = px < bp.width && py < bp.height;
    const float pxc = (float)px + 0.5f, pyc = (float)py + 0.5f;
    const float bx0 = (float)(tx * 16) + 0.5f, by0 = (float)(ty * 16 + band * kBandRows) + 0.5f;
    const uint32_t start = ranges[2 * tile], end = ranges[2 * tile + 1];
    float T = 1.0f, g0 = 0.0f, g1 = 0.0f, g2 = 0.0f;
    uint32_t stop = 0;
    if (inside) {
        const size_t p = (size_t)py * bp.width + px;
        T = bp.final_T[p];
        stop = bp.stop[p];
        g0 = bp.dimage[3 * p + 0];
        g1 = bp.dimage[3 * p + 1];
        g2 = bp.dimage[3 * p + 2];
    }
    // the band's last considered entry: entries past it are skipped
    uint32_t nmax = stop;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) nmax = max(nmax, (uint32_t)__shfl_xor((int)nmax, o, GS_WAVE));
    nmax = min((uint32_t)__builtin_amdgcn_readfirstlane((int)nmax), end - start);
    if (nmax == 0) return;
    // this lane's share of a pair's sums: its term, and the term's scale
    const int term = term_of_lane(lane);
    const bool writes = (lane & 3) == 0 || (lane & 31) == 2;
    const float scale = term == 3 ? -1.0f : ((term == 2 || term == 4) ? -0.5f : 1.0f);
    const bool bit3 = lane & 8, bit2 = lane & 4, bit1 = lane & 2;
    // lane q holds the batch's entry hi - 1 - q (the walk's order)
    int32_t hi = (int32_t)nmax;
    uint32_t gi = sid[start + max(hi - 1 - lane, 0)];
    float4 r0 = trec[3 * (size_t)gi + 0], r1 = trec[3 * (size_t)gi + 1],
           r2 = trec[3 * (size_t)gi + 2];
    uint32_t gn = sid[start + max(hi - 1 - GS_WAVE - lane, 0)];
    bool alone = !finite3(g0, g1, g2);
    if (any_odd && inside) {
        const float* img = bp.image + 3 * ((size_t)py * bp.width + px);
        alone = alone || !finite3(img[0], img[1], img[2]);
    }
    if (__builtin_expect(alone, 0)) {
        backward_alone(trec, sid + start, min(stop, end - start), pxc, pyc, T, g0, g1, g2, bp);
        stop = 0;
        g0 = g1 = g2 = 0.0f;
    }
    float behind = bp.bg[0] * g0 + bp.bg[1] * g1 + bp.bg[2] * g2;
    for (; hi > 0; hi -= GS_WAVE) {
        const bool keep = hi - 1 - lane >= 0 && band_keeps(r0, r1, bx0, by0);
        if (any_odd && !finite3(r2.x, r2.y, r2.z)) r2 = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        const uint64_t mask = __ballot(keep);
        const int cnt = __popcll(mask);
        __syncthreads();  // one wave: orders the LDS reads of the batch before
        if (keep) {
            const int k = __popcll(mask & lanemask_lt());
            s0[k] = make_float4(r0.x, r0.y, r0.z, r1.x);
            s1[k] = make_float4(r1.y, r1.z, r2.x, r2.y);
            s2[k] = make_float4(r2.z, __uint_as_float((uint32_t)(hi - 1 - lane)),
                                __uint_as_float(gi), 0.0f);
        }
        if (lane == cnt && (cnt & 1)) {  // opacity 0, past every stop: blends nowhere
            s0[lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            s1[lane] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
            s2[lane] = make_float4(0.0f, __uint_as_float(0xFFFFFFFFu), 0.0f, 0.0f);
        }
        gi = gn;
        r0 = trec[3 * (size_t)gi + 0];
        r1 = trec[3 * (size_t)gi + 1];
        r2 = trec[3 * (size_t)gi + 2];
        gn = sid[start + max(hi - 1 - 2 * GS_WAVE - lane, 0)];
        __syncthreads();
        for (int k = 0; k < cnt; k += 2) {
            float v[2][9];
            bool any = false;
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const float4 e0 = s0[k + j], e1 = s1[k + j], e2 = s2[k + j];
                const Splat s = splat_at(pxc, pyc, e0.x, e0.y, e0.w, e1.x, e1.y, e0.z);
                const float alpha = fminf(s.raw, bp.alpha_max);
                const bool live = __float_as_uint(e2.y) < stop && alpha >= bp.alpha_min;
                any = any || live;
                const float a = live ? alpha : 0.0f;
                const float Tn = T * __builtin_amdgcn_rcpf(1.0f - a);
                const float d = __builtin_fmaf(e1.z, g0, __builtin_fmaf(e1.w, g1, e2.x * g2)) -
                                behind;
                behind = __builtin_fmaf(a, d, behind);
                T = Tn;
                const float at = a * Tn;
                // no gradient through the clamps
                const float dop = (live && !(s.raw > bp.alpha_max)) ? Tn * d : 0.0f;
                const float dp = s.power <= 0.0f ? dop * s.raw : 0.0f;
                const float dpx = dp * s.dx, dpy = dp * s.dy;
                v[j][0] = dp * __builtin_fmaf(e1.x, s.dy, s.adx);
                v[j][1] = dp * __builtin_fmaf(e1.x, s.dx, s.cdy);
                v[j][2] = dpx * s.dx;
                v[j][3] = dpx * s.dy;
                v[j][4] = dpy * s.dy;
                v[j][5] = dop * s.w;
                v[j][6] = at * g0;
                v[j][7] = at * g1;
                v[j][8] = at * g2;
            }
            if (__ballot(any) == 0ull) continue;
            const float sum = sum_terms(v[0], v[1], bit3, bit2, bit1);
            const uint32_t g = __float_as_uint(s2[k + (lane >> 5)].z);
            if (writes && sum != 0.0f) atomicAdd(bp.grad2d + 9 * (size_t)g + term, sum * scale);
        }
    }
}

// Optimizer-space gradient row (Row<DEG>::S values into out) of a Gaussian from
// its accumulated 2D gradients gg: dmx dmy dA dB dC dop dr dg db.
template <int DEG>
__device__ __forceinline__ void row_gradient(const float4* row, const TrainCam& cam,
                                             const float (&gg)[9], float4* out) {
    constexpr int K = Row<DEG>::K;
    const Head head = load_head(row);
    Geo g;
    geometry(head, cam, g);
    const float gu = gg[0], gv = gg[1], gA = gg[2], gB = gg[3], gC = gg[4], gop = gg[5];
    // conic = inv(S2): dL/dS2 = -Q Gq Q, Gq = [[gA, gB/2], [gB/2, gC]]
    const float hB = 0.5f * gB;
    const float P00 = g.A * gA + g.B * hB, P01 = g.A * hB + g.B * gC;
    const float P10 = g.B * gA + g.C * hB, P11 = g.B * hB + g.C * gC;
    const float G00 = -(P00 * g.A + P01 * g.B);
    const float G01 = -(P00 * g.B + P01 * g.C);
    const float G11 = -(P10 * g.B + P11 * g.C);
    // dL/dcov3 = T^T G2 T ; dL/dT = 2 G2 T cov3
    float G3[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int k = 0; k < 3; ++k)
            G3[3 * r + k] = G00 * g.T0[r] * g.T0[k] + G01 * (g.T0[r] * g.T1[k] + g.T1[r] * g.T0[k]) +
                            G11 * g.T1[r] * g.T1[k];
    float TC0[3], TC1[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        TC0[k] = g.T0[0] * s3(g.S, 0, k) + g.T0[1] * s3(g.S, 1, k) + g.T0[2] * s3(g.S, 2, k);
        TC1[k] = g.T1[0] * s3(g.S, 0, k) + g.T1[1] * s3(g.S, 1, k) + g.T1[2] * s3(g.S, 2, k);
    }
    float dT0[3], dT1[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        dT0[k] = 2.0f * (G00 * TC0[k] + G01 * TC1[k]);
        dT1[k] = 2.0f * (G01 * TC0[k] + G11 * TC1[k]);
    }
    const float* R = cam.r;
    const float dj00 = dT0[0] * R[0] + dT0[1] * R[1] + dT0[2] * R[2];
    const float dj02 = dT0[0] * R[6] + dT0[1] * R[7] + dT0[2] * R[8];
    const float dj11 = dT1[0] * R[3] + dT1[1] * R[4] + dT1[2] * R[5];
    const float dj12 = dT1[0] * R[6] + dT1[1] * R[7] + dT1[2] * R[8];
    const float iz = g.iz, iz2 = iz * iz, fx = cam.fx, fy = cam.fy;
    float gx = gu * fx * iz - dj02 * fx * iz2;
    float gy = gv * fy * iz - dj12 * fy * iz2;
    float gz = -(gu * fx * g.x + gv * fy * g.y + dj00 * fx + dj11 * fy) * iz2 +
               2.0f * (dj02 * fx * g.x + dj12 * fy * g.y) * iz2 * iz;
    if (!g.valid) gx = gy = gz = 0.0f;
    float gm[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) gm[k] = R[k] * gx + R[3 + k] * gy + R[6 + k] * gz;
    // cov3 = M M^T, M = Rq diag(s): dM = 2 G3 M
    float M[9];
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int k = 0; k < 3; ++k) M[3 * r + k] = g.Rq[3 * r + k] * g.s[k];
    float gR[9], gls[3];
#pragma unroll
    for (int k = 0; k < 3; ++k) gls[k] = 0.0f;
#pragma unroll
    for (int r = 0; r < 3; ++r)
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float dM = 2.0f * (G3[3 * r] * M[k] + G3[3 * r + 1] * M[3 + k] +
                                     G3[3 * r + 2] * M[6 + k]);
            gls[k] += dM * g.Rq[3 * r + k];
            gR[3 * r + k] = dM * g.s[k];
        }
    float gq[4];
    {
        const float w = g.qn[0], x = g.qn[1], y = g.qn[2], z = g.qn[3];
        const float gw = 2.0f * (-z * gR[1] + y * gR[2] + z * gR[3] - x * gR[5] - y * gR[6] + x * gR[7]);
        const float gxq = 2.0f * (y * gR[1] + z * gR[2] + y * gR[3] - 2.0f * x * gR[4] - w * gR[5] +
                                  z * gR[6] + w * gR[7] - 2.0f * x * gR[8]);
        const float gyq = 2.0f * (-2.0f * y * gR[0] + x * gR[1] + w * gR[2] + x * gR[3] + z * gR[5] -
                                  w * gR[6] + z * gR[7] - 2.0f * y * gR[8]);
        const float gzq = 2.0f * (-2.0f * z * gR[0] - w * gR[1] + x * gR[2] + w * gR[3] -
                                  2.0f * z * gR[4] + y * gR[5] + x * gR[6] + y * gR[7]);
        const float dot = w * gw + x * gxq + y * gyq + z * gzq;
        gq[0] = (gw - w * dot) * g.qinv;
        gq[1] = (gxq - x * dot) * g.qinv;
        gq[2] = (gyq - y * dot) * g.qinv;
        gq[3] = (gzq - z * dot) * g.qinv;
    }
    if (!g.valid) {
        gq[0] = gq[1] = gq[2] = gq[3] = 0.0f;
        gls[0] = gls[1] = gls[2] = 0.0f;
    }
#pragma unroll
    for (int k = 0; k < 3; ++k) gls[k] *= g.s[k];
    const float op = sigmoidf(head.c.z);
    const float gol = gop * op * (1.0f - op);
    // colour = max(SH(d) + 0.5, 0)
    float sh[3 * K];
    load_sh<DEG>(row, head, sh);
    float raw[3], dir[3], dn;
    colour<DEG>(head, row, cam, raw, dir, dn);
    float gcol[3];
#pragma unroll
    for (int ch = 0; ch < 3; ++ch) gcol[ch] = raw[ch] >= 0.0f ? gg[6 + ch] : 0.0f;
    float b[16], db[16][3];
    sh_basis<DEG, true>(dir[0], dir[1], dir[2], b, db);
    if (K > 1) {
        float gd[3] = {0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int k = 1; k < K; ++k) {
            const float c = sh[3 * k] * gcol[0] + sh[3 * k + 1] * gcol[1] + sh[3 * k + 2] * gcol[2];
            gd[0] += c * db[k][0];
            gd[1] += c * db[k][1];
            gd[2] += c * db[k][2];
        }
        const float dd = dir[0] * gd[0] + dir[1] * gd[1] + dir[2] * gd[2];
#pragma unroll
        for (int k = 0; k < 3; ++k) gm[k] += (gd[k] - dir[k] * dd) / dn;
    }
    out[0] = make_float4(gm[0], gm[1], gm[2], gls[0]);
    out[1] = make_float4(gls[1], gls[2], gq[0], gq[1]);
    out[2] = make_float4(gq[2], gq[3], gol, b[0] * gcol[0]);
#pragma unroll
    for (int q = 3; q < Row<DEG>::V; ++q) {
        float t[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int j = 4 * (q - 3) + 1 + e;  // SH value 3k + channel
            t[e] = j < 3 * K ? b[j < 3 * K ? j / 3 : 0] * gcol[j % 3] : 0.0f;
        }
        out[q] = make_float4(t[0], t[1], t[2], t[3]);
    }
}

// Moments of four values of a row: float, or bf16 bits (uint16_t) read exactly
// into fp32, updated in fp32, the update taken from the fp32 values, stored
// rounded to nearest even (train_oracle.py:445-470 with moment_dtype bfloat16,
// t2_param_backward.py:195-224): half the moments' bytes.
__device__ __forceinline__ float4 mom_load(const float* a, size_t f) {
    return reinterpret_cast<const float4*>(a)[f];
}
__device__ __forceinline__ float4 mom_load(const uint16_t* a, size_t f) {
    const ushort4 u = reinterpret_cast<const ushort4*>(a)[f];
    return make_float4(bf16_to_f32(u.x), bf16_to_f32(u.y), bf16_to_f32(u.z), bf16_to_f32(u.w));
}
__device__ __forceinline__ void mom_store(float* a, size_t f, float4 x) {
    reinterpret_cast<float4*>(a)[f] = x;
}
__device__ __forceinline__ void mom_store(uint16_t* a, size_t f, float4 x) {
    reinterpret_cast<ushort4*>(a)[f] = make_ushort4(f32_to_bf16_rne(x.x), f32_to_bf16_rne(x.y),
                                                    f32_to_bf16_rne(x.z), f32_to_bf16_rne(x.w));
}

// Sparse Adam of one value (train_oracle.py:434-470), fp32 arithmetic, bias
// correction folded into the step size and sqrt(1 - beta2^t) by the host.
__device__ __forceinline__ void adam_value(float& p, float& m, float& v, float g, float step,
                                           const AdamParams& ap) {
    m = ap.beta1 * m + ap.one_minus_beta1 * g;
    v = ap.beta2 * v + ap.one_minus_beta2 * g * g;
    const float den = sqrtf(v) / ap.sqrt_bc2 + ap.eps;
    p = p - step * (m / den);
}
template <typename MOM>
__device__ __forceinline__ void adam_float4(float4* P, MOM* m, MOM* v, size_t f, float4 g,
                                            float4 step, const AdamParams& ap) {
    float4 p = P[f], mm = mom_load(m, f), vv = mom_load(v, f);
    adam_value(p.x, mm.x, vv.x, g.x, step.x, ap);
    adam_value(p.y, mm.y, vv.y, g.y, step.y, ap);
    adam_value(p.z, mm.z, vv.z, g.z, step.z, ap);
    adam_value(p.w, mm.w, vv.w, g.w, step.w, ap);
    P[f] = p;
    mom_store(m, f, mm);
    mom_store(v, f, vv);
}

// Gradients of every Gaussian, and with ADAM the sparse Adam of the visible rows
// in the same pass (the gradient row then never comes back from HBM). A
// workgroup owns R rows. First a thread per row forms the gradient of a row
// that blended somewhere into LDS and the rows with work are listed; then the
// workgroup streams those rows, one float4 per lane, so that every access to
// G, the parameters and the moments is contiguous within a row and the rows
// without work (invisible, gradient zero as before) are not touched at all.
constexpr uint32_t kRowGrad = 1u << 16, kRowZero = 1u << 17, kRowAdam = 1u << 18;
constexpr int kGradThreads = 256;
template <int DEG, bool ADAM, typename MOM>
__global__ __launch_bounds__(kGradThreads) void k_train_grads(
    TrainParamsDev P, TrainCam cam, const uint32_t* __restrict__ cidx,
    const float* __restrict__ grad2d, float4* __restrict__ G, uint8_t* __restrict__ gnz,
    MOM* __restrict__ m, MOM* __restrict__ v, const uint8_t* __restrict__ visible, AdamParams ap,
    HostCopy report) {
    constexpr int V = Row<DEG>::V;
    constexpr int R = DEG < 2 ? kGradThreads : kGradThreads / 2;  // rows: 16 to 30 KB of LDS
    __shared__ float4 s_g[R][V];
    __shared__ float4 s_step[V];
    __shared__ uint32_t s_list[R];
    __shared__ uint32_t s_count;
    // the step's counters and sums are final by now, whether it failed or not
    if (blockIdx.x == 0) host_copy(report, threadIdx.x, kGradThreads);
    if (upstream_failed(cam.ctl)) return;
    const int tid = threadIdx.x;
    const int64_t row0 = (int64_t)blockIdx.x * R;
    if (tid == 0) s_count = 0;
    if (ADAM && tid < V)
        s_step[tid] = make_float4(ap.step[4 * tid], ap.step[4 * tid + 1], ap.step[4 * tid + 2],
                                  ap.step[4 * tid + 3]);
    __syncthreads();
    const int64_t i = row0 + tid;
    if (tid < R) {
        uint32_t act = 0;
        if (i < P.n) {
            const uint32_t ci = cidx[i];
            float gg[9];
            bool any = false;
#pragma unroll
            for (int k = 0; k < 9; ++k) {
                gg[k] = ci != 0xFFFFFFFFu ? grad2d[9 * (size_t)ci + k] : 0.0f;
                any |= gg[k] != 0.0f;
            }
            const bool was = gnz[i] != 0;
            if (any) {
                row_gradient<DEG>(P.rows + i * V, cam, gg, s_g[tid]);
                act = kRowGrad;
            } else if (was) {
                act = kRowZero;
            }
            if (any != was) gnz[i] = any ? 1 : 0;
            if (ADAM && visible[i]) act |= kRowAdam;
        }
        const uint64_t mask = __ballot(act != 0u);
        uint32_t at = 0;
        if (lane_id() == 0 && mask != 0ull) at = atomicAdd(&s_count, (uint32_t)__popcll(mask));
        at = (uint32_t)__builtin_amdgcn_readfirstlane((int)at);
        if (act != 0u) s_list[at + (uint32_t)__popcll(mask & lanemask_lt())] = act | (uint32_t)tid;
    }
    __syncthreads();
    const uint32_t total = s_count * V;
    for (uint32_t k = tid; k < total; k += kGradThreads) {
        const uint32_t e = s_list[k / V], q = k % V, r = e & 0xFFFFu;
        const size_t f = (size_t)(row0 + r) * V + q;
        float4 g = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (e & kRowGrad) g = s_g[r][q];
        if (e & (kRowGrad | kRowZero)) G[f] = g;
        if (ADAM && (e & kRowAdam)) adam_float4(P.rows, m, v, f, g, s_step[q], ap);
    }
}

// The sparse Adam alone, from gradient rows: a lane per float4 of the visible
// rows.
template <int DEG, typename MOM>
__global__ __launch_bounds__(256) void k_sparse_adam(TrainParamsDev P, MOM* __restrict__ m,
                                                     MOM* __restrict__ v,
                                                     const float4* __restrict__ G,
                                                     const uint8_t* __restrict__ visible,
                                                     AdamParams ap) {
    constexpr int V = Row<DEG>::V;
    __shared__ float4 s_step[V];
    if (threadIdx.x < V)
        s_step[threadIdx.x] = make_float4(ap.step[4 * threadIdx.x], ap.step[4 * threadIdx.x + 1],
                                          ap.step[4 * threadIdx.x + 2], ap.step[4 * threadIdx.x + 3]);
    __syncthreads();
    const size_t f = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (f >= (size_t)P.n * V || !visible[f / V]) return;
    adam_float4(P.rows, m, v, f, G[f], s_step[f % V], ap);
}

// Rows <-> the caller's arrays: a thread per value, the arrays' side contiguous,
// the rows' side within a few lines (bound by HBM, 8 MB of either in a few us).
__device__ __forceinline__ float row_get(const float* r, size_t k) { return r[k]; }
__device__ __forceinline__ float row_get(const uint16_t* r, size_t k) { return bf16_to_f32(r[k]); }
__device__ __forceinline__ void row_put(float* r, size_t k, float x) { r[k] = x; }
__device__ __forceinline__ void row_put(uint16_t* r, size_t k, float x) {
    r[k] = f32_to_bf16_rne(x);
}
template <typename T, bool SPLIT>
__global__ __launch_bounds__(256) void k_train_rows(T* __restrict__ rows, int64_t row0,
                                                    int64_t count, int vals, int stride,
                                                    float* __restrict__ arrays) {
    const int64_t k = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (k >= count * vals) {
        // a joined row's padding
        const int64_t e = k - count * vals, pad = stride - vals;
        if (!SPLIT && e < count * pad)
            row_put(rows, (size_t)(row0 + e / pad) * stride + vals + e % pad, 0.0f);
        return;
    }
    const int start[6] = {0, 3, 6, 10, 11, vals};
    int q = 0;
    while (k >= count * start[q + 1]) ++q;
    const int w = start[q + 1] - start[q];
    const int64_t j = k - count * start[q];
    const size_t r = (size_t)(row0 + j / w) * stride + start[q] + j % w;
    if (SPLIT) arrays[k] = row_get(rows, r);
    else row_put(rows, r, arrays[k]);
}

}  // namespace

hipError_t launch_train_rows(void* rows, int64_t row0, int64_t count, int sh_degree, float* arrays,
                             bool split, bool bf16, hipStream_t st) {
    if (count <= 0) return hipSuccess;
    if (sh_degree < 0 || sh_degree > 3) return hipErrorInvalidValue;
    const int vals = train_row_values(sh_degree), stride = train_row_floats(sh_degree);
    const unsigned grid = (unsigned)((count * stride + 255) / 256);
    if (split && bf16)
        k_train_rows<uint16_t, true><<<grid, 256, 0, st>>>(static_cast<uint16_t*>(rows), row0,
                                                           count, vals, stride, arrays);
    else if (split)
        k_train_rows<float, true><<<grid, 256, 0, st>>>(static_cast<float*>(rows), row0, count,
                                                        vals, stride, arrays);
    else if (bf16)
        k_train_rows<uint16_t, false><<<grid, 256, 0, st>>>(static_cast<uint16_t*>(rows), row0,
                                                            count, vals, stride, arrays);
    else
        k_train_rows<float, false><<<grid, 256, 0, st>>>(static_cast<float*>(rows), row0, count,
                                                         vals, stride, arrays);
    return hipGetLastError();
}

hipError_t launch_train_project(const TrainParamsDev& P, const TrainCam& cam, Compact out,
                                float4* trec, uint32_t* cidx, uint8_t* visible,
                                uint64_t* lb_state, uint32_t* ticket, uint32_t* count_out,
                                uint32_t* part_hist, const TrainDebug& dbg, hipStream_t st) {
    if (P.n <= 0) return hipSuccess;
    const int items = cam.binned.offs != nullptr ? project_items(P.n) : kTItems;
    const unsigned grid = (unsigned)((P.n + kTThreads * items - 1) / (kTThreads * items));
#define GS_TP_I(D, B, I)                                                                   \
    k_train_project<D, B, I><<<grid, kTThreads, 0, st>>>(P, cam, out, trec, cidx, visible,  \
                                                         lb_state, ticket, count_out,      \
                                                         part_hist, dbg)
#define GS_TP(D)                                                                           \
    if (cam.binned.offs == nullptr) GS_TP_I(D, false, kTItems);                            \
    else if (items == 1) GS_TP_I(D, true, 1);                                              \
    else GS_TP_I(D, true, kTItems)
    switch (P.sh_degree) {
        case 0: GS_TP(0); break;
        case 1: GS_TP(1); break;
        case 2: GS_TP(2); break;
        case 3: GS_TP(3); break;
        default: return hipErrorInvalidValue;
    }
#undef GS_TP
#undef GS_TP_I
    return hipGetLastError();
}

hipError_t launch_train_fwd(const float4* trec, const uint32_t* sid, const uint32_t* ranges,
                            const TrainFwdParams& fp, hipStream_t st) {
    const int tiles = fp.tiles_x * fp.tiles_y;
    if (tiles <= 0) return hipSuccess;
    k_train_fwd<<<tiles * kBandsPerTile, GS_WAVE, 0, st>>>(trec, sid, ranges, fp);
    return hipGetLastError();
}

hipError_t launch_ssim(const SsimParams& sp, hipStream_t st) {
    if (sp.width <= 0 || sp.height <= 0) return hipSuccess;
    const unsigned grid = 3u * (unsigned)(((sp.width + kSsimW - 1) / kSsimW) *
                                          ((sp.height + kSsimH - 1) / kSsimH));
    k_ssim_fwd<<<grid, 256, 0, st>>>(sp);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    k_ssim_bwd<<<grid, 256, 0, st>>>(sp);
    return hipGetLastError();
}

hipError_t launch_l1(const float* image, const float* target, int64_t count, float scale,
                     float* dimage, TrainSums* sums, hipStream_t st) {
    if (count <= 0) return hipSuccess;
    k_l1<<<(unsigned)((count + 255) / 256), 256, 0, st>>>(image, target, count, scale, dimage,
                                                          sums);
    return hipGetLastError();
}

hipError_t launch_train_bwd(const float4* trec, const uint32_t* sid, const uint32_t* ranges,
                            const TrainBwdParams& bp, hipStream_t st) {
    const int tiles = bp.tiles_x * bp.tiles_y;
    if (tiles <= 0) return hipSuccess;
    k_train_bwd<<<tiles * kBandsPerTile, GS_WAVE, 0, st>>>(trec, sid, ranges, bp);
    return hipGetLastError();
}

namespace {
template <int DEG>
hipError_t train_grads_deg(const TrainParamsDev& P, const TrainCam& cam, const uint32_t* cidx,
                           const float* grad2d, float4* G, uint8_t* gnz, void* m, void* v,
                           const uint8_t* visible, const AdamParams* adam, bool bf16_moments,
                           const HostCopy& report, hipStream_t st) {
    constexpr int R = DEG < 2 ? kGradThreads : kGradThreads / 2;
    const unsigned grid = (unsigned)((P.n + R - 1) / R);
    if (adam == nullptr)
        k_train_grads<DEG, false, float><<<grid, kGradThreads, 0, st>>>(
            P, cam, cidx, grad2d, G, gnz, nullptr, nullptr, nullptr, AdamParams{}, report);
    else if (bf16_moments)
        k_train_grads<DEG, true, uint16_t><<<grid, kGradThreads, 0, st>>>(
            P, cam, cidx, grad2d, G, gnz, static_cast<uint16_t*>(m), static_cast<uint16_t*>(v),
            visible, *adam, report);
    else
        k_train_grads<DEG, true, float><<<grid, kGradThreads, 0, st>>>(
            P, cam, cidx, grad2d, G, gnz, static_cast<float*>(m), static_cast<float*>(v), visible,
            *adam, report);
    return hipGetLastError();
}

template <int DEG>
hipError_t sparse_adam_deg(const TrainParamsDev& P, void* m, void* v, const float4* G,
                           const uint8_t* visible, const AdamParams& ap, bool bf16_moments,
                           hipStream_t st) {
    const unsigned grid = (unsigned)(((size_t)P.n * Row<DEG>::V + 255) / 256);
    if (bf16_moments)
        k_sparse_adam<DEG, uint16_t><<<grid, 256, 0, st>>>(
            P, static_cast<uint16_t*>(m), static_cast<uint16_t*>(v), G, visible, ap);
    else
        k_sparse_adam<DEG, float><<<grid, 256, 0, st>>>(P, static_cast<float*>(m),
                                                        static_cast<float*>(v), G, visible, ap);
    return hipGetLastError();
}
}  // namespace

hipError_t launch_train_grads(const TrainParamsDev& P, const TrainCam& cam, const uint32_t* cidx,
                              const float* grad2d, float4* G, uint8_t* gnz, void* m, void* v,
                              const uint8_t* visible, const AdamParams* adam, bool bf16_moments,
                              const HostCopy& report, hipStream_t st) {
    if (P.n <= 0) return hipSuccess;
#define GS_TG(D) \
    train_grads_deg<D>(P, cam, cidx, grad2d, G, gnz, m, v, visible, adam, bf16_moments, report, st)
    switch (P.sh_degree) {
        case 0: return GS_TG(0);
        case 1: return GS_TG(1);
        case 2: return GS_TG(2);
        case 3: return GS_TG(3);
        default: return hipErrorInvalidValue;
    }
#undef GS_TG
}

hipError_t launch_sparse_adam(const TrainParamsDev& P, void* m, void* v, const float4* G,
                              const uint8_t* visible, const AdamParams& ap, bool bf16_moments,
                              hipStream_t st) {
    if (P.n <= 0) return hipSuccess;
    switch (P.sh_degree) {
        case 0: return sparse_adam_deg<0>(P, m, v, G, visible, ap, bf16_moments, st);
        case 1: return sparse_adam_deg<1>(P, m, v, G, visible, ap, bf16_moments, st);
        case 2: return sparse_adam_deg<2>(P, m, v, G, visible, ap, bf16_moments, st);
        case 3: return sparse_adam_deg<3>(P, m, v, G, visible, ap, bf16_moments, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace gs
