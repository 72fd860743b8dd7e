// One decode position of consecutive blocks, two launches per block:
// UnifiedBlock.step (model.py:96-111, run.c:193-265) on the deferred state of
// decode.hip (S_base and up to kMaxPending pending terms), for batches whose
// position takes two launches less time than it takes the host to enqueue the
// per-kernel form's (kMaxCost).
//
// There a position is bound by launches and memory latency, not by bytes: the
// per-kernel form (RMSNorm + conv, three GEMMs, address, state read: 6 launches
// and their host work) took 93 us per block and position at 8 sequences of the
// 110M widths and 99 us per block of the default model at one, against 14 and
// 1 us of bytes; this form takes 30 and 11 us. What depends on what leaves two
// phases with one grid-wide dependency between them, the address's row sum:
//
//   in    h, u (RMSNorm, conv) formed by every workgroup for itself;
//         pre = K u, v = W_v h, 32 rows per workgroup;  z = relu(pre + b)^2;
//         c <- lam c + (1 - lam) w + r_prev;  r_prev appended as pending key,
//         v as pending value;  this tile's part of the row sum of z and of the
//         pending keys' read-outs pr_j . (z / c)
//   out   the parts summed in a fixed order; q = z / c / denom;
//         out = x + lam^m (S_base q) + sum_j lam^(m-1-j) v_j (pr_j . q) + mu (w q);
//         r_prev <- z / denom;  the conv window shifted
//
// r and w q never reach memory. Every sum has a fixed order.
#include "ulm_common.h"

#include <algorithm>

namespace ulm {

// decode.hip
int launch_decode_write_back(float *S, const float *pv, const float *pr, int m, const float *g, int N, int D, int A,
                             hipStream_t s);

namespace step {

constexpr int kMaxPending = 16;   // as decode.hip
constexpr int kMaxN = 256;        // sequences
// Microseconds up to which a block's position takes this form (cost below): the
// per-kernel form's eight calls take 88 of host time, whatever their sizes, and
// from about 250 MB of state on 94 of the device's. 16 positions of one block, us,
// this form / per kernel, at (sequences, features, slots) and the cost:
//   (256, 64, 128)     27    405 / 1440        (26, 768, 4096)    92   1656 / 1635
//   (16, 768, 3072)    52    898 / 1421        (48, 768, 2048)    99   1539 / 1498
//   (256, 64, 1024)    54    825 / 1418        (256, 288, 712)   108   1731 / 1450
//   (128, 288, 712)    61    913 / 1422        (128, 768, 768)   141   2146 / 1452
//   (40, 512, 3072)    80   1359 / 1433        (256, 512, 512)   153   2436 / 1445
//   (32, 768, 3072)    90   1330 / 1504        (256, 768, 400)   210   3520 / 1781
constexpr double kMaxCost = 92;
constexpr int kWgN = 16;          // sequences per workgroup of the first phase
constexpr int kLdsFloats = 15 * 1024;   // of dynamic LDS per workgroup: 60 KB
constexpr int kRows = 4;          // weight rows per wave
constexpr int kWaves = 8;         // waves per workgroup of the first phase
constexpr int kTile = kRows * kWaves;   // rows per workgroup: 32, half a wave's lanes in the epilogue
constexpr int kMaxTaps = 8;
constexpr int kCus = 256;
constexpr int kGroup = 4;         // sequences per workgroup of the second phase
constexpr int kParts = kMaxPending + 2;   // row stride of the partial sums: z, then the pending terms

struct Layer {
    const float *norm_w, *conv_w, *key_w, *key_b, *log_eps, *val_w, *mu_w, *w, *g;
    float *buf, *S, *c, *r_prev, *pv, *pr;
    float eps;
    int m;   // terms already pending: this position's is term m
};

// V consecutive floats at p, in one access where V is 4 (16-byte aligned)
template <int V> struct Vec {
    float e[V];
    __device__ __forceinline__ void load(const float *p) {
        if constexpr (V == 4) {
            const f32x4 t = *reinterpret_cast<const f32x4 *>(p);
#pragma unroll
            for (int i = 0; i < 4; ++i) e[i] = t[i];
        } else {
            e[0] = *p;
        }
    }
};

// x (N, D) -> z (N, A) and the partial sums part[n][i][tile], i = 0 the row sum
// of z, 1 + j term j; h (N, D). Workgroups below nta take 32 slots each (rows of
// key_w, contracted with u), the others 32 features (rows of val_w, with h).
// The weight rows, c, r_prev and the pending keys are loaded before anything
// waits, so one memory latency covers them and the prologue's own loads.
// V = 4: D % 4 == 0, every row 16-byte aligned, else V = 1. A launch runs its
// code once, and at these sizes its instructions are what it takes: 10 us at
// N = 8 and the 110M widths, of which the 12 MB of weights are 2; 5.5 us at
// N = 1 and the default model's. (38 us with the sums over lanes in select
// chains, below.)
template <int NT, int V>
__global__ __launch_bounds__(kWaves * 64) void decode_in_kernel(Layer L, const float *__restrict__ x,
                                                                float *__restrict__ z, float *__restrict__ zq,
                                                                float *__restrict__ part, float *__restrict__ hout, int N, int D, int A, int Kc,
                                                                int nta, int per_wg) {
    extern __shared__ __align__(16) float su[];   // [Nl][D] u or h
    __shared__ float res[kTile][NT + 1];
    constexpr int KS = 3;                          // column slices of 64 V per register set
    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64);
    const int n0 = blockIdx.y * per_wg, Nl = min(per_wg, N - n0);   // this workgroup's sequences
    const bool slots = static_cast<int>(blockIdx.x) < nta;
    const int tile = slots ? blockIdx.x : blockIdx.x - nta;
    const int rows = slots ? A : D, row0 = tile * kTile;
    const float *__restrict__ W = slots ? L.key_w : L.val_w;
    // weights of this wave's rows, columns d0 .. d0 + 64 V KS - 1 (past D: the row's last columns, their products dropped)
    Vec<V> wv[kRows][KS];
    auto load_w = [&](int d0) {
#pragma unroll
        for (int i = 0; i < kRows; ++i) {
            const float *wr = W + static_cast<size_t>(min(row0 + wave * kRows + i, rows - 1)) * D;
#pragma unroll
            for (int k = 0; k < KS; ++k) wv[i][k].load(wr + min(d0 + (64 * k + lane) * V, D - V));
        }
    };
    // h, or u = conv over [buf, h]: kWaves / NS waves per sequence (NS: NT up to
    // kWaves), each taking every (kWaves / NS)-th slice of 64 V columns; every
    // wave sums its sequence's squares by itself, so that nothing waits on a
    // barrier. Loads complete in order, so what is waited for first is asked for
    // first: x, the conv's operands, then the weights and the epilogue's operands.
    constexpr int NS = NT < kWaves ? NT : kWaves, WS = kWaves / NS;   // sequences at a time, waves per sequence
    constexpr int HB = (KS + WS - 1) / WS;                            // slices per wave held in registers
    const int kw = Kc - 1;
    const int wn = wave / WS, wp = wave % WS;
    Vec<V> xs[KS], xv[HB], nv[HB], sv[HB][3], cv[HB][4];
    auto load_x = [&](int n, int d0) {
#pragma unroll
        for (int k = 0; k < KS; ++k) xs[k].load(x + static_cast<size_t>(n0 + n) * D + min(d0 + (64 * k + lane) * V, D - V));
    };
    auto load_h = [&](int n, int k0) {
#pragma unroll
        for (int u = 0; u < HB; ++u) {
            const int d = min((64 * (k0 + u * WS) + lane) * V, D - V), i = (n0 + n) * D + d;
            xv[u].load(x + i);
            nv[u].load(L.norm_w + d);
            if (slots && Kc == 4) {
#pragma unroll
                for (int j = 0; j < 3; ++j) sv[u][j].load(L.buf + i * 3 + j * V);
#pragma unroll
                for (int j = 0; j < 4; ++j) cv[u][j].load(L.conv_w + d * 4 + j * V);
            }
        }
    };
    if (wn < Nl) {
        load_x(wn, 0);
        load_h(wn, wp);
    }
    load_w(0);
    // the epilogue's operands: thread (sequence n, row r)
    const int er = tid % kTile, en = tid / kTile;
    const bool live = en < Nl && row0 + er < rows;
    const uint32_t ea = (n0 + (live ? en : 0)) * A + (slots && live ? row0 + er : 0);
    float c0 = 0.f, rp = 0.f, w0 = 0.f, b0 = 0.f, pk[kMaxPending - 1];
    if (slots) {
        c0 = L.c[ea];
        rp = L.r_prev[ea];
        w0 = L.w[live ? row0 + er : 0];
        b0 = L.key_b[live ? row0 + er : 0];
        // terms past the pending ones read the first again, unused: no branch between the loads
#pragma unroll
        for (int j = 0; j < kMaxPending - 1; ++j) pk[j] = ld_row(L.pr + static_cast<size_t>(j < L.m ? j : 0) * N * A, 4u * ea);
    }
    const float lam = __expf(L.g[0]);
    for (int n = wn; n < Nl; n += NS) {
        float ss = 0.f;
        for (int d0 = 0; d0 < D; d0 += 64 * V * KS) {
            if (n != wn || d0 > 0) load_x(n, d0);
#pragma unroll
            for (int k = 0; k < KS; ++k) {
                const bool in = d0 + (64 * k + lane) * V < D;
#pragma unroll
                for (int e = 0; e < V; ++e) ss += in ? xs[k].e[e] * xs[k].e[e] : 0.f;
            }
        }
        ss = wave_sum(ss);
        const float inv = rsqrtf(ss / static_cast<float>(D) + L.eps);
        for (int k0 = wp; k0 * 64 * V < D; k0 += HB * WS) {
            if (n != wn || k0 != wp) load_h(n, k0);
#pragma unroll
            for (int u = 0; u < HB; ++u) {
                const int d = (64 * (k0 + u * WS) + lane) * V;
                if (d < D) {
                    float y[V];
#pragma unroll
                    for (int e = 0; e < V; ++e) y[e] = (xv[u].e[e] * inv) * nv[u].e[e];
                    if (!slots) {
                        if (tile == 0)
#pragma unroll
                            for (int e = 0; e < V; ++e) hout[(n0 + n) * D + d + e] = y[e];
                    } else if (Kc == 4) {
#pragma unroll
                        for (int e = 0; e < V; ++e) {
                            float t = 0.f;
#pragma unroll
                            for (int j = 0; j < 3; ++j)
                                t += cv[u][(e * 4 + j) / V].e[(e * 4 + j) % V] * sv[u][(e * 3 + j) / V].e[(e * 3 + j) % V];
                            y[e] = t + cv[u][(e * 4 + 3) / V].e[(e * 4 + 3) % V] * y[e];
                        }
                    } else {
                        const float *st = L.buf + static_cast<size_t>((n0 + n) * D + d) * kw;
                        const float *cw = L.conv_w + static_cast<size_t>(d) * Kc;
#pragma unroll
                        for (int e = 0; e < V; ++e) {
                            float t = 0.f;
                            for (int j = 0; j < kw; ++j) t += cw[e * Kc + j] * st[e * kw + j];
                            y[e] = t + cw[e * Kc + kw] * y[e];
                        }
                    }
#pragma unroll
                    for (int e = 0; e < V; ++e) su[n * D + d + e] = y[e];
                }
            }
        }
    }
    __syncthreads();
    float acc[kRows * NT];
#pragma unroll
    for (int i = 0; i < kRows * NT; ++i) acc[i] = 0.f;
    for (int d0 = 0; d0 < D; d0 += 64 * V * KS) {
        if (d0 > 0) load_w(d0);
#pragma unroll
        for (int k = 0; k < KS; ++k) {
            const int d = d0 + (64 * k + lane) * V;
            if (d < D) {
#pragma unroll
                for (int n = 0; n < NT; ++n) {
                    Vec<V> t;
                    t.load(su + min(n, Nl - 1) * D + d);
#pragma unroll
                    for (int i = 0; i < kRows; ++i)
#pragma unroll
                        for (int e = 0; e < V; ++e) acc[i * NT + n] += wv[i][k].e[e] * t.e[e];
                }
            }
        }
    }
    constexpr int VS = kRows * NT;
    const float dot = reduce_scatter<VS, 32>(acc, lane);
    if (lane % (64 / VS) == 0) {
        const int i = lane / (64 / VS);
        res[wave * kRows + i / NT][i % NT] = dot;
    }
    __syncthreads();
    if (en >= Nl) return;   // whole half-waves
    const float y = res[er][en < NT ? en : 0];
    if (!slots) {
        if (live) L.pv[(static_cast<size_t>(L.m) * N + n0 + en) * D + row0 + er] = y;
        return;
    }
    float p = y + b0;
    p = p > 0.f ? p : 0.f;
    const float zv = live ? p * p : 0.f;
    const float cn = lam * c0 + (1.f - lam) * w0 + rp;
    const float zc = live ? zv / cn : 0.f;
    if (live) {
        z[ea] = zv;
        zq[ea] = zc;
        L.c[ea] = cn;
        L.pr[static_cast<size_t>(L.m) * N * A + ea] = rp;
    }
    float dots[kMaxPending];
#pragma unroll
    for (int j = 0; j < kMaxPending - 1; ++j) dots[j] = live && j < L.m ? pk[j] * zc : 0.f;
    dots[kMaxPending - 1] = 0.f;
    // this position's own key goes last, into the slot past the others
    float own = live ? rp * zc : 0.f, zs = zv;
    for (int mask = 16; mask >= 1; mask >>= 1) {
        own += __shfl_xor(own, mask, kWave);
        zs += __shfl_xor(zs, mask, kWave);
    }
    const float dj = reduce_scatter<kMaxPending, 16>(dots, lane);
    float *pn = part + static_cast<size_t>(n0 + en) * kParts * nta + tile;
    const int hl = lane % 32;
    if (hl == 0) pn[0] = zs;
    if (hl == 1) pn[static_cast<size_t>(1 + L.m) * nta] = own;
    if (hl % 2 == 0 && hl / 2 < L.m) pn[static_cast<size_t>(1 + hl / 2) * nta] = dj;
}

// The read-out of one position: NG sequences n0 .. of one feature per wave,
// blockDim / 64 features per workgroup. The wave walks the slots in slices of
// 256: a slice of mu's row, times w's, and of each sequence's row of S_base,
// against q's slice in LDS, KB slices at a time with the next KB in flight. q
// goes into LDS without the address's 1 / denom, which multiplies the read-out
// instead: the stream waits for q alone, and wave i sums sequence n0 + i's
// parts beside it. 18 us at N = 8 and the 110M widths (75 MB of S_base), 5.6 us
// at N = 1 and the default model's (20 and 6.2 with the parts, the address and
// the windows loaded where they are used); a whole row of one sequence after the other,
// with its prologue ahead of the stream, took 24. A % 4 == 0, nta <= 128.
template <int NG>
__global__ __launch_bounds__(512) void decode_out_kernel(Layer L, const float *__restrict__ x,
                                                          const float *__restrict__ z, const float *__restrict__ zq,
                                                          const float *__restrict__ part, const float *__restrict__ h,
                                                          float *__restrict__ out, int N, int D, int A, int Kc,
                                                          int nta) {
    extern __shared__ __align__(16) float sq[];      // [NG][A] z / c
    __shared__ float sums[kGroup][2 * kMaxPending];   // z's row sum, then lam^(m - j) (pr_j . (z / c))
    static_assert(NG <= kGroup && kParts <= 32, "a lane pair per value");
    constexpr int KB = 2;
    const int tid = threadIdx.x, lane = tid % 64;
    const int wave = __builtin_amdgcn_readfirstlane(tid / 64), waves = blockDim.x / 64;
    const int n0 = blockIdx.y * NG, ng = min(NG, N - n0);
    const int d = blockIdx.x * waves + wave;
    const int dc = min(d, D - 1);
    const int A4 = A / 4, mt = L.m + 1;
    const uint32_t last = 16u * (A4 - 1);
    f32x4 sv[2][KB][NG], mv[2][KB], wv[2][KB];
    const float *mrow = L.mu_w + static_cast<size_t>(dc) * A, *srow = L.S + (static_cast<size_t>(n0) * D + dc) * A;
    const size_t sn = static_cast<size_t>(D) * A;   // between two sequences' rows
    auto at16 = [](const float *p, uint32_t off) { return reinterpret_cast<const f32x4 *>(reinterpret_cast<const char *>(p) + off); };
    auto load = [&](int k0, int b) {
#pragma unroll
        for (int u = 0; u < KB; ++u) {
            const uint32_t off = min(16u * (lane + 64 * (k0 + u)), last);
#pragma unroll
            for (int n = 0; n < NG; ++n) sv[b][u][n] = __builtin_nontemporal_load(at16(srow + (n < ng ? n : 0) * sn, off));
            mv[b][u] = *at16(mrow, off);
            wv[b][u] = *at16(L.w, off);
        }
    };
    // Loads complete in order and the stream waits for q alone, so q is asked for
    // first; then everything else that is small, so that nothing is asked for at
    // the end: the parts (wave i: sequence n0 + i's; values past the m + 2 in use
    // read the row sum's again, unused), this thread's share of the address and of
    // the conv windows.
    constexpr int QB = 8;
    const f32x4 *zr = reinterpret_cast<const f32x4 *>(zq + static_cast<size_t>(n0) * A);
    const int nq = ng * A4, nt = blockDim.x;
    f32x4 qv[QB];
#pragma unroll
    for (int u = 0; u < QB; ++u) qv[u] = zr[min(tid + u * nt, nq - 1)];   // the sequences' rows are contiguous
    const float *pn = part + static_cast<size_t>(n0 + min(wave, ng - 1)) * kParts * nta;
    float v[32], v2[kParts];
#pragma unroll
    for (int i = 0; i < kParts; ++i) v[i] = ld_row(pn + (i <= mt ? i : 0) * nta, 4u * min(lane, nta - 1));
#pragma unroll
    for (int i = 0; i < kParts; ++i) v2[i] = ld_row(pn + (i <= mt ? i : 0) * nta, 4u * min(lane + 64, nta - 1));
    const int gi = blockIdx.x * nt + tid;   // 16-byte slice gi of the sequences' addresses
    const f32x4 zv = reinterpret_cast<const f32x4 *>(z + static_cast<size_t>(n0) * A)[min(gi, nq - 1)];
    const int kw = Kc - 1, wi = gi;         // pair (sequence, feature) wi of the sequences' windows
    const bool shifts = kw > 0 && wi < ng * D;
    float *win = L.buf + (static_cast<size_t>(n0) * D + (shifts ? wi : 0)) * kw;
    const float hv = h[static_cast<size_t>(n0) * D + (shifts ? wi : 0)];
    // one tap leaves no window (and a null buffer): h stands in for it, unused
    const float *win_in = kw > 0 ? win : h;
    float st[kMaxTaps - 1];
#pragma unroll
    for (int j = 1; j < kMaxTaps - 1; ++j) st[j] = win_in[j < kw ? j : 0];
    load(0, 0);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int u = 0; u < QB; ++u)
        if (tid + u * nt < nq) reinterpret_cast<f32x4 *>(sq)[tid + u * nt] = qv[u];
    for (int i = tid + QB * nt; i < nq; i += nt) reinterpret_cast<f32x4 *>(sq)[i] = zr[i];
    const float lam = __expf(L.g[0]);
    __syncthreads();
    float acc[4] = {0.f, 0.f, 0.f, 0.f};
    if (wave < ng) {
#pragma unroll
        for (int i = 0; i < 32; ++i)
            v[i] = i < kParts ? (lane < nta ? v[i] : 0.f) + (lane + 64 < nta ? v2[i < kParts ? i : 0] : 0.f) : 0.f;
        float s = reduce_scatter<32, 32>(v, lane);
        for (int e = lane / 2 - 1; e >= 0 && e < L.m; ++e) s *= lam;   // term j's weight
        if (lane % 2 == 0) sums[wave][lane / 2] = s;
    }
    if (shifts) {
#pragma unroll
        for (int j = 1; j < kMaxTaps - 1; ++j)
            if (j < kw) win[j - 1] = st[j];
        win[kw - 1] = hv;
    }
    // lane j's pending value
    float pvl[NG];
#pragma unroll
    for (int n = 0; n < NG; ++n)
        pvl[n] = L.pv[(static_cast<size_t>(min(lane, L.m)) * N + n0 + (n < ng ? n : 0)) * D + dc];
    const float eps = __expf(fminf(fmaxf(L.log_eps[0], -10.f), 10.f));
    float lm = lam;
    for (int j = 0; j < L.m; ++j) lm *= lam;
    auto add = [&](int k0, int b) {
#pragma unroll
        for (int u = 0; u < KB; ++u) {
            const int j = lane + 64 * (k0 + u);
            const bool in = j < A4;
            const f32x4 mw = mv[b][u] * wv[b][u];
#pragma unroll
            for (int n = 0; n < NG; ++n) {
                const f32x4 t = (lm * sv[b][u][n] + mw) * reinterpret_cast<const f32x4 *>(sq + n * A)[in ? j : 0];
                const float s = (t[0] + t[1]) + (t[2] + t[3]);
                acc[n] += in ? s : 0.f;
            }
        }
    };
    const int nk = (A4 + 63) / 64;
    // loads past the row read its last 16 bytes, one line, and count for nothing:
    // under a condition the compiler would wait for every load in flight
    for (int k0 = 0; k0 < nk; k0 += 2 * KB) {
        load(k0 + KB, 1);
        __builtin_amdgcn_sched_barrier(0);   // the next slices' loads go out before this arithmetic
        add(k0, 0);
        load(k0 + 2 * KB, 0);
        __builtin_amdgcn_sched_barrier(0);
        add(k0 + KB, 1);
    }
    __syncthreads();
    // the address itself, read by the next position (the grid has a thread for every slice: four features' waves at
    // least per workgroup; the loop covers the shapes where it has not)
    if (gi < nq) reinterpret_cast<f32x4 *>(L.r_prev + static_cast<size_t>(n0) * A)[gi] = zv * (1.f / (eps + sums[gi / A4][0]));
    for (int i = gi + gridDim.x * nt; i < nq; i += gridDim.x * nt)
        reinterpret_cast<f32x4 *>(L.r_prev + static_cast<size_t>(n0) * A)[i] =
            reinterpret_cast<const f32x4 *>(z + static_cast<size_t>(n0) * A)[i] * (1.f / (eps + sums[i / A4][0]));
#pragma unroll
    for (int n = 0; n < NG; ++n) acc[n] += lane < mt && n < ng ? pvl[n] * sums[n][1 + lane] : 0.f;
    const float y = reduce_scatter<4, 32>(acc, lane);   // lane 16 n: sequence n0 + n
    const int n = lane / 16;
    if (lane % 16 == 0 && n < ng && d < D) {
        const size_t o = static_cast<size_t>(n0 + n) * D + d;
        out[o] = x[o] + y * (1.f / (eps + sums[n][0]));
    }
}

// the workspace: z, z / c, the parts, h and two rows of block outputs
struct Ws {
    float *z, *zq, *part, *h, *x0, *x1;
    size_t bytes;
};
Ws layout(void *base, int N, int D, int A) {
    Carver c(base);
    Ws w{};
    const int nta = (A + kTile - 1) / kTile;
    w.z = c.take<float>(static_cast<size_t>(N) * A);
    w.zq = c.take<float>(static_cast<size_t>(N) * A);
    w.part = c.take<float>(static_cast<size_t>(N) * kParts * nta);
    w.h = c.take<float>(static_cast<size_t>(N) * D);
    w.x0 = c.take<float>(static_cast<size_t>(N) * D);
    w.x1 = c.take<float>(static_cast<size_t>(N) * D);
    w.bytes = c.off;
    return w;
}

template <int NT>
int launch_in(const Layer &L, const float *x, const Ws &ws, int N, int D, int A, int Kc, int groups, hipStream_t s) {
    const int nta = (A + kTile - 1) / kTile, ntd = (D + kTile - 1) / kTile, per = (N + groups - 1) / groups;
    const size_t lds = static_cast<size_t>(per) * D * sizeof(float);
    const dim3 grid(nta + ntd, groups), wg(kWaves * 64);
    uintptr_t bits = static_cast<uintptr_t>(D) * sizeof(float);
    for (const float *p : {L.norm_w, L.conv_w, L.key_w, L.val_w, static_cast<const float *>(L.buf), x})
        bits |= reinterpret_cast<uintptr_t>(p);
    if (bits % 16 == 0)
        decode_in_kernel<NT, 4><<<grid, wg, lds, s>>>(L, x, ws.z, ws.zq, ws.part, ws.h, N, D, A, Kc, nta, per);
    else
        decode_in_kernel<NT, 1><<<grid, wg, lds, s>>>(L, x, ws.z, ws.zq, ws.part, ws.h, N, D, A, Kc, nta, per);
    return check_launch("decode_in_kernel");
}

// A position's microseconds in this form, within 10% where it is near the line
// (30 shapes, 1 to 256 sequences, 16 to 2048 features, 64 to 4096 slots): two
// launches; S_base, mu and the key rows; the value rows; z, c and the pending
// keys, several passes of N A floats; and h and u, which every workgroup of the
// first phase forms for itself, with what a wave of the second one does per
// feature before it walks the slots.
double cost(double N, double D, double A) { return 14 + 1e-6 * N * (0.70 * D * A + 0.185 * D * D + 75 * A + 540 * D); }

// sequences per workgroup of the first phase, their u in LDS: evenly over the fewest groups of at most kWgN
int in_groups(int N, int D) {
    const int most = std::min(kWgN, kLdsFloats / D);
    return most ? (N + most - 1) / most : 0;
}

int launch_block(const Layer &L, const float *x, float *out, const Ws &ws, int N, int D, int A, int Kc, hipStream_t s) {
    const int ig = in_groups(N, D), ip = (N + ig - 1) / ig, gi = (N + ip - 1) / ip;
    if (ip == 1) ULM_TRY(launch_in<1>(L, x, ws, N, D, A, Kc, gi, s));
    else if (ip == 2) ULM_TRY(launch_in<2>(L, x, ws, N, D, A, Kc, gi, s));
    else if (ip <= 4) ULM_TRY(launch_in<4>(L, x, ws, N, D, A, Kc, gi, s));
    else if (ip <= 8) ULM_TRY(launch_in<8>(L, x, ws, N, D, A, Kc, gi, s));
    else ULM_TRY(launch_in<16>(L, x, ws, N, D, A, Kc, gi, s));
    const int nta = (A + kTile - 1) / kTile;
    // sequences per workgroup, evenly, their q within 60 KB of LDS (A <= 4096: three at least)
    const int most = std::min(kGroup, kLdsFloats / A);
    const int groups = (N + most - 1) / most, per = (N + groups - 1) / groups;
    // one feature per wave; as many waves per workgroup (4 to 8) as make about one workgroup per CU, since a second
    // one on some CUs would take twice as long as the rest (the prologue is repeated by each)
    const int waves = std::clamp((D * groups + kCus - 1) / kCus, 4, 8);
    const dim3 grid((D + waves - 1) / waves, (N + per - 1) / per), wg(64 * waves);
    const size_t lds = static_cast<size_t>(per) * A * sizeof(float);
#define ULM_OUT(G) decode_out_kernel<G><<<grid, wg, lds, s>>>(L, x, ws.z, ws.zq, ws.part, ws.h, out, N, D, A, Kc, nta)
    if (per == 1) ULM_OUT(1);
    else if (per == 2) ULM_OUT(2);
    else if (per == 3) ULM_OUT(3);
    else ULM_OUT(4);
#undef ULM_OUT
    return check_launch("decode_out_kernel");
}

}  // namespace step
}  // namespace ulm

using namespace ulm;

// the shapes this form takes; at least one sequence's u fits the LDS of a workgroup
static bool step_supported(int N, int D, int A, int Kc) {
    return N >= 1 && N <= step::kMaxN && D >= 1 && A >= 4 && A % 4 == 0 && A <= 4096 && Kc >= 1 && Kc <= step::kMaxTaps &&
           step::in_groups(N, D) > 0 && step::cost(N, D, A) <= step::kMaxCost;
}

extern "C" size_t ulm_decode_step_workspace_bytes(int N, int D, int A, int Kc) {
    return step_supported(N, D, A, Kc) ? step::layout(nullptr, N, D, A).bytes : 0;
}

extern "C" int ulm_decode_step(const ulm_decode_layer *layers, int n_layers, const float *x, float *out,
                               void *workspace, size_t workspace_bytes, int N, int D, int A, int Kc, void *stream) {
    ULM_REQUIRE(step_supported(N, D, A, Kc), "ulm_decode_step: unsupported sizes N=%d D=%d A=%d Kc=%d", N, D, A, Kc);
    ULM_REQUIRE(layers && n_layers >= 1 && x && out && workspace, "ulm_decode_step: null pointer");
    ULM_REQUIRE(x != out, "ulm_decode_step: out must not alias x");
    const step::Ws ws = step::layout(workspace, N, D, A);
    ULM_REQUIRE(workspace_bytes >= ws.bytes && reinterpret_cast<uintptr_t>(workspace) % 16 == 0,
                "ulm_decode_step: workspace of %zu bytes, need %zu, 16-byte aligned", workspace_bytes, ws.bytes);
    for (int i = 0; i < n_layers; ++i) {
        const ulm_decode_layer &l = layers[i];
        ULM_REQUIRE(l.norm_w && l.conv_w && l.key_w && l.key_b && l.log_eps && l.val_w && l.mu_w && l.w && l.g && l.S && l.c &&
                        l.r_prev && l.pv && l.pr && (Kc == 1 || l.conv_buf),
                    "ulm_decode_step: null pointer in layer %d", i);
        ULM_REQUIRE(l.pending >= 0 && l.pending < step::kMaxPending, "ulm_decode_step: layer %d holds %lld terms", i,
                    static_cast<long long>(l.pending));
        for (const void *p : {static_cast<const void *>(l.mu_w), static_cast<const void *>(l.w),
                              static_cast<const void *>(l.S), static_cast<const void *>(l.c),
                              static_cast<const void *>(l.r_prev), static_cast<const void *>(l.pr)})   // pr: the write-back's
            ULM_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0,
                        "ulm_decode_step: layer %d: mu_w, w, S, c, r_prev and pr must be 16-byte aligned", i);
    }
    hipStream_t s = static_cast<hipStream_t>(stream);
    for (int i = 0; i < n_layers; ++i) {
        const ulm_decode_layer &l = layers[i];
        step::Layer L{l.norm_w, l.conv_w, l.key_w, l.key_b, l.log_eps, l.val_w, l.mu_w, l.w, l.g, l.conv_buf, l.S, l.c,
                      l.r_prev, l.pv, l.pr, static_cast<float>(l.norm_eps), static_cast<int>(l.pending)};
        float *y = i + 1 == n_layers ? out : (i % 2 ? ws.x1 : ws.x0);
        ULM_TRY(step::launch_block(L, x, y, ws, N, D, A, Kc, s));
        x = y;
        if (l.pending + 1 == step::kMaxPending)
            ULM_TRY(launch_decode_write_back(l.S, l.pv, l.pr, step::kMaxPending, l.g, N, D, A, s));
    }
    return ULM_OK;
}
