// Gated GQA attention decode on gfx950 (Model::Impl::attention_preout, reference
// model.cpp:129-157, which the reference runs on the host even on its device path).
//
// Split-KV ("flash decoding") over a fixed grid: workgroup (range j of kAttnSplit, kv head;
// the ranges that short contexts leave empty are dispatched last: 4 KV heads at 200 positions
// 9.5 us, head-major 10.7) serves the `group` = heads/kv_heads query heads that share the KV head, so
// each K/V row is read once for all of them, over range j of the positions 0..pos. The
// ranges are whole sub-chunks of kAttnSub positions, as many per range as it takes to
// cover the context with the ranges in use (attn_per). Every workgroup recomputes the RMSNorm + RoPE of its query heads and of
// the new key (a few KiB of work); the workgroup whose range holds the current position
// also appends the new k/v to the caches and uses them straight from LDS. Each
// workgroup writes an unnormalised partial (o, running max, sum of exponentials); a
// second small kernel merges the (at most kAttnSplit) partials, divides, and applies the
// sigmoid output gate. (A last-workgroup merge inside the first kernel needs
// agent-scope fences, which write back and invalidate an L2 on this part: measured
// 29.3 us per call at 512 positions against 9.9 us for the two kernels, and 2.9 us more
// even at 16 positions, where four workgroups take part. Without fences -- partials
// written with agent-scope atomic stores, s_waitcnt 0 and a barrier before a relaxed
// ticket, the last range of each KV head merging with agent-scope loads -- it is
// correct and still slower past a few ranges, one workgroup reading every partial:
// 8.3 / 9.7 / 17.3 / 26.6 / 31.9 us at 16 / 100 / 512 / 1024 / 4096 positions against
// 8.7 / 8.6 / 9.0 / 9.5 / 15.6 us for the two kernels, 569 against 592 tok/s.)
//
// Inside a workgroup (8 waves) every wave owns kAttnSub/8 positions of each sub-chunk
// and keeps their K and V rows in registers, lane l holding dims E*l .. E*l+E-1 (head_dim = 64*E,
// one 16-byte access per row at E = 4). A score is then E products and one wave sum,
// with the query heads in registers too; each wave runs an online softmax (its own
// running maximum and sum) over its rows and accumulates their P.V, and the eight
// waves are merged (max-rescaled) through LDS. Measured on the 9B attention shape
// (16 Q / 4 KV heads x 256; one attention + merge, replayed from a graph): 10.3, 13.4
// and 17.5 µs at 512, 2048 and 4096 positions, against 11.6, 16.2 and 23.0 µs with
// 4-wave workgroups and 14.8, 15.1 and 18.4 µs for the earlier design (64-position
// chunks, one workgroup each, keys staged in LDS, one score per lane); 9.1, 11.4 and
// 15.7 µs for this kernel on a later box. Measured alternatives that did not pay, same
// box each: computing the RoPE angles in the kernel instead of reading the table (9.9
// against 9.2 µs at 512), issuing the norm-input loads before the position read (9.13
// against 9.10), loading each range's first K/V rows before the position is known
// (no gain, and the ranges past the position then read rows they never use).
//
// The grid does not depend on the position, so the launch can be replayed from a
// hipGraph: the position is read from device memory and ranges past it return at once.
// Barriers order LDS only (lds_barrier), so none of them waits for the K/V rows in flight.
#include <algorithm>

#include "common.hpp"
#include "kernels.hpp"

namespace emprise {
namespace {

constexpr int kAttnWaves = 8;
constexpr int kMaxGroup = 8;
constexpr int kAttnLong = 512;  // sub-chunks (8192 positions) past which kAttnSplit ranges are faster

// E consecutive floats (lane l of a wave owns dims E*l .. E*l+E-1 of a head): one
// 16-, 8- or 4-byte access.
template <int E> __device__ __forceinline__ void ldv(float (&v)[E], const float* p) {
    if constexpr (E == 4) {
        const float4 t = *reinterpret_cast<const float4*>(p);
        v[0] = t.x, v[1] = t.y, v[2] = t.z, v[3] = t.w;
    } else if constexpr (E == 2) {
        const float2 t = *reinterpret_cast<const float2*>(p);
        v[0] = t.x, v[1] = t.y;
    } else {
        v[0] = *p;
    }
}
template <int E> __device__ __forceinline__ void stv(float* p, const float (&v)[E]) {
    if constexpr (E == 4) *reinterpret_cast<float4*>(p) = make_float4(v[0], v[1], v[2], v[3]);
    else if constexpr (E == 2) *reinterpret_cast<float2*>(p) = make_float2(v[0], v[1]);
    else *p = v[0];
}

// The `len` positions are cut into nsub = ceil(len / CH) sub-chunks, and range j takes
// `per` = ceil(nsub / ranges) consecutive ones (ranges past the end are empty). The combine
// kernel recomputes the same split to know how many partials exist.
//
// ranges: kAttnFew while they give every CU a workgroup and the range is short, else
// kAttnSplit, two workgroups per CU, so that 16 waves' rows are in flight. The second 64
// partials cost the merge a round trip behind the position read (4 KV heads x 256, graph
// replays, us with 128 and 64 ranges: 14.0 / 12.6 at 2000 positions, 17.1 / 16.2 at 4000, 19.6 /
// 19.2 at 6000, 22.2 / 22.5 at 8000, 23.0 / 23.9 at 8250, 28.1 / 31.6 at 12000, 35.9 / 39.6 at
// 16000; the empty workgroups of a short context cost nothing that shows, 8.6 at 200 either way).
// Two KV heads fill the chip only with 128 (10.4 / 12.0 at 4000).
__device__ __forceinline__ int attn_per(int len, int kv_heads) {
    const int nsub = (len + kAttnSub - 1) / kAttnSub;
    const int ranges = kv_heads * kAttnFew < 256 || nsub > kAttnLong ? kAttnSplit : kAttnFew;
    return (nsub + ranges - 1) / ranges;
}

// Eight wave-wide sums at once: halving exchanges across lanes l^32 and l^16
// (v_permlane32_swap / v_permlane16_swap, each pair of values trading the halves the
// other lane keeps) and l^8 (a row rotation) leave lane l with value
// (l>>3 & 1) + 2*(l>>4 & 1) + 4*(l>>5 & 1) summed over 8 lanes, and a three-step butterfly
// inside each group of 8 lanes completes it (the same bits in all 8); value j is then
// read from lane 8j. About half the instructions of eight wave_sum, and a shorter chain.
__device__ __forceinline__ void wave_sum8(const float (&x)[8], float (&out)[8]) {
    float y[4], z[2];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x[j]), __float_as_uint(x[j + 4]), false, false);
        y[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);  // lanes 0-31: value j, 32-63: value j+4
    }
#pragma unroll
    for (int j = 0; j < 2; ++j) {
        const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(y[j]), __float_as_uint(y[j + 2]), false, false);
        z[j] = __uint_as_float(r[0]) + __uint_as_float(r[1]);  // even rows of 16: slot j, odd rows: slot j+2
    }
    const bool hi8 = (threadIdx.x & 8) != 0;
    float w = (hi8 ? z[1] : z[0]) + dpp_f<0x128, 0xf>(0.f, hi8 ? z[0] : z[1]);  // row_ror:8
    w += dpp_f<0xb1, 0xf>(0.f, w);   // quad_perm [1,0,3,2]
    w += dpp_f<0x4e, 0xf>(0.f, w);   // quad_perm [2,3,0,1]
    w += dpp_f<0x141, 0xf>(0.f, w);  // row_half_mirror
#pragma unroll
    for (int j = 0; j < 8; ++j) out[j] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(w), 8 * j));
}

// Bound by the K/V rows in flight: with registers and LDS for up to 4 query heads per KV head
// (97 and 39 KiB at head_dim 256, instead of 149 and 76 KiB for 8) two workgroups share a CU.
// 30000 positions of 4 KV heads x 256: 66.6 -> 52.7 us (3.7 -> 4.7 TB/s); 2 x 64: 49.2 -> 28.8.
template <int E, int MG>  // head_dim = 64 * E, at most MG query heads per KV head
__global__ __launch_bounds__(kAttnWaves * 64, MG <= 4 ? 4 : 2) void attention_kernel(AttnArgs a) {
    constexpr int HD = 64 * E, CH = kAttnSub, PW = CH / kAttnWaves;  // rows per wave and sub-chunk
    __shared__ __align__(16) float qs[MG][HD];
    __shared__ __align__(16) float knew[HD], vnew[HD];
    __shared__ float wstat[kAttnWaves][MG][2];  // per wave and head: max, sum
    __shared__ __align__(16) float acc_lds[kAttnWaves][MG][HD];

    const int group = a.heads / a.kv_heads;
    const int range = blockIdx.x / a.kv_heads, kvh = blockIdx.x - range * a.kv_heads;
    const int pos = *a.position;
    if (pos < 0 || pos >= a.context) return;  // the host keeps positions inside the caches
    const int rpos = a.rope_position ? *a.rope_position : pos;
    if (rpos < 0 || rpos >= a.context) return;  // the RoPE table has `context` rows
    const int len = pos + 1;
    const int nsub = (len + CH - 1) / CH, per = attn_per(len, a.kv_heads);
    const int sub0 = range * per, sub1 = min(nsub, sub0 + per);
    if (sub0 >= sub1) return;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int qd = a.heads * HD * 2, kvd = a.kv_heads * HD;
    const float* kin = a.qkv + qd + (size_t)kvh * HD;
    const float* vin = a.qkv + qd + kvd + (size_t)kvh * HD;
    const size_t row_stride = (size_t)a.kv_heads * HD;
    const float* kb = a.keys + (size_t)kvh * HD + E * lane;
    const float* vb = a.values + (size_t)kvh * HD + E * lane;

    // The wave's K and V rows of sub-chunk `sub` (positions sub*CH + wave + 8i); rows
    // past `len` are loaded clamped and never used; the row at `pos` is not written yet,
    // may hold anything, NaN included, and is replaced by the new k/v.
    auto load_rows = [&](float (&kr)[PW][E], float (&vr)[PW][E], int sub) {
        const int t0 = sub * CH, tn = min(CH, len - t0);
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const size_t t = (size_t)(t0 + min(wave + kAttnWaves * i, tn - 1));
            ldv<E>(kr[i], kb + t * row_stride);
            ldv<E>(vr[i], vb + t * row_stride);
        }
    };

    // Loads, in the order they are needed: the inputs of the q/k RMSNorms (wave w
    // normalises heads w, w+8, ... and, as head `group`, the new key), then the wave's
    // K and V rows of the first sub-chunk. The norm inputs are loaded unconditionally
    // (clamped heads) so waiting for them never waits for the K/V rows, whose latency
    // overlaps the norms and RoPE.
    constexpr int NJ = (MG + kAttnWaves) / kAttnWaves;  // heads per wave, incl. the key
    float xin[NJ][E], qn[E], kn[E];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int g = min(wave + kAttnWaves * j, group);
        const float* src = g < group ? a.qkv + (size_t)(kvh * group + g) * HD * 2 : kin;
        ldv<E>(xin[j], src + E * lane);
    }
    ldv<E>(qn, a.q_norm + E * lane);
    ldv<E>(kn, a.k_norm + E * lane);
    const float vin_d = vin[min((int)threadIdx.x, HD - 1)];
    // this thread's first RoPE pair (idx = threadIdx.x below): its (cos, sin) from the table
    const int half = a.rotary / 2;
    const float2 cs0 = half > 0 ? a.rope[(size_t)rpos * half + min((int)threadIdx.x, (group + 1) * half - 1) % half]
                                : make_float2(1.f, 0.f);
    float kr[PW][E], vr[PW][E];
    load_rows(kr, vr, sub0);

    // RMSNorm of the query heads and of the new key (model.cpp:133-134)
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
        const int g = wave + kAttnWaves * j;
        if (g <= group) {
            float ss = 0.f;
#pragma unroll
            for (int e = 0; e < E; ++e) ss += xin[j][e] * xin[j][e];
            ss = wave_sum(ss);
            const float scale = 1.f / sqrtf(ss / (float)HD + a.eps);
            float y[E];
#pragma unroll
            for (int e = 0; e < E; ++e) y[e] = xin[j][e] * (scale * (g < group ? qn[e] : kn[e]));
            stv<E>((g < group ? qs[g] : knew) + E * lane, y);
        }
    }
    if (threadIdx.x < HD) vnew[threadIdx.x] = vin_d;
    lds_barrier();
    // NEOX RoPE over the first `rotary` dims (model.cpp:121-127); one thread per pair,
    // the angles' cos and sin from the backend's table (rope_table_kernel), which the
    // batched prefill reads as well
    for (int idx = threadIdx.x; idx < (group + 1) * half; idx += blockDim.x) {
        const int g = idx / half, i = idx % half;
        float* row = g < group ? qs[g] : knew;
        const float2 cs = idx == (int)threadIdx.x ? cs0 : a.rope[(size_t)rpos * half + i];
        const float c = cs.x, s = cs.y;
        const float x0 = row[i], x1 = row[i + half];
        row[i] = x0 * c - x1 * s;
        row[i + half] = x0 * s + x1 * c;
    }
    lds_barrier();
    if (sub1 == nsub) {  // this range holds `pos`: append k/v to the caches
        for (int d = threadIdx.x; d < HD; d += blockDim.x) {
            a.keys[((size_t)pos * a.kv_heads + kvh) * HD + d] = knew[d];
            a.values[((size_t)pos * a.kv_heads + kvh) * HD + d] = vnew[d];
        }
    }

    // Lane l holds dims E*l .. E*l+E-1 of every query head and of each row, so a score
    // is E products and one wave sum (model.cpp:143-150). Each wave runs an online
    // softmax over its rows of the range's sub-chunks (running maximum, sum and P.V),
    // with the next sub-chunk's rows loading while the current one is used; the four
    // waves are merged (max-rescaled) through LDS at the end.
    float qv[MG][E];
#pragma unroll
    for (int g = 0; g < MG; ++g)
        if (g < group) ldv<E>(qv[g], qs[g] + E * lane);
    const float inv_root = 1.f / sqrtf((float)HD);
    float mw[MG], lw[MG], acc[MG][E];
#pragma unroll
    for (int g = 0; g < MG; ++g) {
        mw[g] = -INFINITY;
        lw[g] = 0.f;
#pragma unroll
        for (int e = 0; e < E; ++e) acc[g][e] = 0.f;
    }
    for (int sub = sub0; sub < sub1; ++sub) {
        const int t0 = sub * CH, tn = min(CH, len - t0);
        float kn2[PW][E], vn2[PW][E];
        if (sub + 1 < sub1) load_rows(kn2, vn2, sub + 1);
        float sc[PW][MG];
#pragma unroll
        for (int i = 0; i < PW; ++i) {
            const int tt = wave + kAttnWaves * i;
            if (t0 + tt == pos) {
                ldv<E>(kr[i], knew + E * lane);
                ldv<E>(vr[i], vnew + E * lane);
            }
        }
        if (PW * 4 == 8 && MG == 4 && group == 4) {
            // the wave's eight scores (PW rows x 4 heads) reduced together
            float d[8], s8[8];
#pragma unroll
            for (int i = 0; i < PW; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    float p = 0.f;
#pragma unroll
                    for (int e = 0; e < E; ++e) p = fmaf(qv[g][e], kr[i][e], p);
                    d[(4 * i + g) & 7] = p;
                }
            wave_sum8(d, s8);
#pragma unroll
            for (int i = 0; i < PW; ++i)
#pragma unroll
                for (int g = 0; g < 4; ++g) sc[i][g] = s8[(4 * i + g) & 7] * inv_root;
        } else {
#pragma unroll
            for (int i = 0; i < PW; ++i)
#pragma unroll
                for (int g = 0; g < MG; ++g) {
                    if (g < group) {
                        float p = 0.f;
#pragma unroll
                        for (int e = 0; e < E; ++e) p = fmaf(qv[g][e], kr[i][e], p);
                        sc[i][g] = wave_sum(p) * inv_root;
                    }
                }
        }
#pragma unroll
        for (int g = 0; g < MG; ++g) {
            if (g < group) {
                float m = mw[g];
#pragma unroll
                for (int i = 0; i < PW; ++i)
                    if (wave + kAttnWaves * i < tn) m = fmaxf(m, sc[i][g]);
                if (m != -INFINITY) {  // the wave has rows in this sub-chunk
                    const float r = mw[g] == -INFINITY ? 0.f : expf(mw[g] - m);
                    lw[g] *= r;
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[g][e] *= r;
                    mw[g] = m;
                }
                // (rows past `len` hold a clamped copy of the row at `pos`, which the
                // cache does not have yet: never touched, not even times 0)
#pragma unroll
                for (int i = 0; i < PW; ++i) {
                    if (wave + kAttnWaves * i < tn) {
                        const float p = expf(sc[i][g] - m);
                        lw[g] += p;
#pragma unroll
                        for (int e = 0; e < E; ++e) acc[g][e] = fmaf(p, vr[i][e], acc[g][e]);
                    }
                }
            }
        }
        if (sub + 1 < sub1) {
#pragma unroll
            for (int i = 0; i < PW; ++i)
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    kr[i][e] = kn2[i][e];
                    vr[i][e] = vn2[i][e];
                }
        }
    }
#pragma unroll
    for (int g = 0; g < MG; ++g) {
        if (g < group) {
            stv<E>(acc_lds[wave][g] + E * lane, acc[g]);
            if (lane == 0) {
                wstat[wave][g][0] = mw[g];
                wstat[wave][g][1] = lw[g];
            }
        }
    }
    lds_barrier();
    // Merge of the waves into the range's partial: o, max, sum. Lane w*8+g of every
    // wave computes the weight exp(m_w - M_g) of wave w for head g. (Every loop below is
    // uniform per wave: head_dim is a multiple of 64, so a wave's 64 consecutive items
    // share one head, and __shfl never reads an inactive lane.)
    float wgt = 0.f, mg = -INFINITY;
    if (lane < kAttnWaves * MG) {
        const int w = lane / MG, g = lane % MG;
        if (g < group) {
#pragma unroll
            for (int v = 0; v < kAttnWaves; ++v) mg = fmaxf(mg, wstat[v][g][0]);
            const float m = wstat[w][g][0];
            wgt = m == -INFINITY ? 0.f : expf(m - mg);
        }
    }
    const int stride = HD + 2;
    float* part = a.partial + ((size_t)kvh * kAttnSplit + range) * group * stride;
    for (int idx = threadIdx.x; idx < group * HD; idx += blockDim.x) {
        const int g = idx / HD, d = idx % HD;
        float o = 0.f;
#pragma unroll
        for (int w = 0; w < kAttnWaves; ++w) o = fmaf(__shfl(wgt, w * MG + g, 64), acc_lds[w][g][d], o);
        part[g * stride + d] = o;
    }
    if (wave == 0) {
        const int g = lane < MG ? lane : 0;
        float l = 0.f;
#pragma unroll
        for (int w = 0; w < kAttnWaves; ++w) l = fmaf(__shfl(wgt, w * MG + g, 64), wstat[w][g][1], l);
        const float m = __shfl(mg, g, 64);
        if (lane < group) {
            part[lane * stride + HD] = m;
            part[lane * stride + HD + 1] = l;
        }
    }
}

// Merges the range partials of one query head and 64 of its output dims:
// o = sum_c e^(m_c - M) o_c / sum_c e^(m_c - M) l_c, then the sigmoid output gate
// (model.cpp:153). The loads of the first kAttnFew partials -- the gate, each wave's share
// of the o values (ranges w, w+4, ...), the statistics -- go out
// together with the position's, before it is known which ranges hold positions (the
// slots of the others are loaded but never used); the four waves' sums are added
// through LDS. Loading only the ranges that hold positions makes those loads wait for
// the position read: measured 1.2 us slower per call at 512 positions and 2.3 us at
// 1024-4096 (graph replay), for half the merge's fetched bytes at 512.
// Partials past kAttnFew exist only where they pay for that wait (attn_per).
constexpr int kCombineBatch = kAttnFew / 4;  // ranges per wave
static_assert(kAttnSplit == 2 * kAttnFew, "two batches");
__global__ __launch_bounds__(256) void attention_combine_kernel(AttnArgs a) {
    __shared__ float wts[kAttnSplit];
    __shared__ float red[8];
    __shared__ float part[4][64];
    const int hd = a.head_dim, group = a.heads / a.kv_heads, dblocks = hd / 64;
    const int head = blockIdx.x / dblocks, db = blockIdx.x - head * dblocks;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int kvh = head / group, g = head - kvh * group, stride = hd + 2;
    const float* base = a.partial + ((size_t)kvh * kAttnSplit * group + g) * stride;
    const size_t cstride = (size_t)group * stride;
    const int d = db * 64 + lane;
    const int pos = *a.position;
    const float gate = a.qkv[(size_t)head * hd * 2 + hd + d];
    float ov[kCombineBatch];
#pragma unroll
    for (int i = 0; i < kCombineBatch; ++i) ov[i] = base[(size_t)(wave + 4 * i) * cstride + d];
    const int cs = min((int)threadIdx.x, kAttnFew - 1);
    float m_c = base[(size_t)cs * cstride + hd], l_c = base[(size_t)cs * cstride + hd + 1];
    if (pos < 0 || pos >= a.context) return;
    const int nsub = pos / kAttnSub + 1, per = attn_per(pos + 1, a.kv_heads);
    const int nchunks = (nsub + per - 1) / per;  // ranges holding positions
    const bool own = (int)threadIdx.x < nchunks;
    float more[kCombineBatch];
    if (nchunks > kAttnFew) {
#pragma unroll
        for (int i = 0; i < kCombineBatch; ++i) {
            const int c = min(kAttnFew + wave + 4 * i, nchunks - 1);
            more[i] = base[(size_t)c * cstride + d];
        }
        if (own && (int)threadIdx.x >= kAttnFew) {
            m_c = base[(size_t)threadIdx.x * cstride + hd];
            l_c = base[(size_t)threadIdx.x * cstride + hd + 1];
        }
    }
    const float mloc = wave_max(own ? m_c : -INFINITY);
    if (lane == 0) red[wave] = mloc;
    lds_barrier();
    const float M = fmaxf(fmaxf(red[0], red[1]), fmaxf(red[2], red[3]));
    const float w = own ? expf(m_c - M) : 0.f;
    if ((int)threadIdx.x < kAttnSplit) wts[threadIdx.x] = w;
    const float dloc = wave_sum(own ? w * l_c : 0.f);
    lds_barrier();  // every weight is in wts; red is free again
    if (lane == 0) red[4 + wave] = dloc;
    float num = 0.f;
#pragma unroll
    for (int i = 0; i < kCombineBatch; ++i) {
        const int c = wave + 4 * i;
        if (c < nchunks) num = fmaf(wts[c], ov[i], num);
    }
    if (nchunks > kAttnFew) {
#pragma unroll
        for (int i = 0; i < kCombineBatch; ++i) {
            const int c = kAttnFew + wave + 4 * i;
            if (c < nchunks) num = fmaf(wts[c], more[i], num);
        }
    }
    part[wave][lane] = num;
    lds_barrier();
    if (wave == 0) {
        const float den = (red[4] + red[5]) + (red[6] + red[7]);
        const float o = (part[0][lane] + part[1][lane]) + (part[2][lane] + part[3][lane]);
        a.out[(size_t)head * hd + d] = (o / den) * sigmoidf_(gate);
    }
}

// (cos, sin) of angle = pos / base^(2i / rotary) for every position < context and
// i < rotary / 2 (model.cpp:121-127), with the expressions attention_kernel used inline.
__global__ __launch_bounds__(256) void rope_table_kernel(float2* t, int context, int rotary, float base) {
    const int half = rotary / 2;
    const size_t n = (size_t)context * half;
    for (size_t idx = (size_t)blockIdx.x * blockDim.x + threadIdx.x; idx < n; idx += (size_t)gridDim.x * blockDim.x) {
        const int pos = (int)(idx / half), i = (int)(idx % half);
        const float angle = (float)pos / powf(base, 2.f * (float)i / (float)rotary);
        t[idx] = make_float2(cosf(angle), sinf(angle));
    }
}

// ---- batched form: `count` consecutive prompt positions (the prefill) --------------------
//
// Position t (absolute first + t) attends over keys 0..first+t. attn_prep_batch_kernel
// normalises and rotates the queries and new keys exactly as attention_kernel does and
// appends k/v to the caches; attn_split_kv_kernel writes the keys and values of 0..first+
// count-1 as matrix operands; attn_flash_kernel then runs the scores, an online softmax and
// P.V tile by tile, so no score goes through memory, and applies the sigmoid gate
// (model.cpp:129-157). With few query rows the keys are split over workgroups and
// attn_merge_batch_kernel joins their partial results.
//
// Scores run on the fp16 matrix cores from two fp16 pieces per FP32 operand: x = 2^e (xh +
// 2^-11 xl), 22 significant bits of every value down to 2^-28 of its vector's largest, e taken
// per query and per key, three products of four (xl yl is below 2^-22 of its term), those with a
// low piece in a sum of their own, FP32 sums. P.V carries P and V whole, as three bf16 pieces of 8
// bits each (with FP32's range, so it does not matter how the values' sizes differ), in the six products above 2^-24 of their
// term, a tile's summed apart from O. Each product has 16 queries on the lane index: S^T = K Q^T
// leaves lane (query l%16, group g = l/16) the scores of keys 4g .. 4g+3 of two 16-key halves,
// which is the operand of O^T = V^T P^T if V^T lists the 32 keys in that order -- so it does, and
// P goes from one product to the next in registers.
//
// Bound by the matrix cores and, about as much, by LDS reads (80 KiB per wave and tile): 2048
// positions behind 4096 of the 9B shape (16 Q / 4 KV heads x 256) are 172 GFLOP, four and a half
// times that in 16-bit products; 750 us for all the kernels here, of which the split 21 and the
// prep 24. As two FP32 GEMMs per head with the scores in memory and a softmax pass between them it
// took 2570 us and 805 MB of scratch, with 1.4e-6 of error against 64 bits, now 4e-7 (relative,
// whole output). P.V from two fp16 pieces with an exponent per tile of values took 579 us, with
// 8.8e-7, but lost all digits of values much smaller than others in their tile or before it.

// Workgroup = one position; wave w normalises head vectors w, w+8, ... of the group's
// q heads (all kv heads' groups) and the kv heads' new keys.
template <int E>
__global__ __launch_bounds__(512) void attn_prep_batch_kernel(AttnBatchArgs a) {
    constexpr int HD = 64 * E;
    extern __shared__ __align__(16) float rows[];  // (heads + kv_heads) x HD
    const int t = blockIdx.x, pos = a.first + t;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, waves = blockDim.x >> 6;
    const int nh = a.heads + a.kv_heads, qd = a.heads * HD * 2, kvd = a.kv_heads * HD;
    const float* row = a.qkv + (size_t)t * a.stride;
    for (int v = wave; v < nh; v += waves) {
        const bool is_q = v < a.heads;
        const float* src = is_q ? row + (size_t)v * HD * 2 : row + qd + (size_t)(v - a.heads) * HD;
        const float* w = is_q ? a.q_norm : a.k_norm;
        float x[E], ss = 0.f;
        ldv<E>(x, src + E * lane);
#pragma unroll
        for (int e = 0; e < E; ++e) ss += x[e] * x[e];
        ss = wave_sum(ss);
        const float scale = 1.f / sqrtf(ss / (float)HD + a.eps);
        float wv[E], y[E];
        ldv<E>(wv, w + E * lane);
#pragma unroll
        for (int e = 0; e < E; ++e) y[e] = x[e] * (scale * wv[e]);
        stv<E>(rows + (size_t)v * HD + E * lane, y);
    }
    __syncthreads();
    const int half = a.rotary / 2;
    for (int idx = threadIdx.x; idx < nh * half; idx += blockDim.x) {
        const int v = idx / half, i = idx % half;
        float* r = rows + (size_t)v * HD;
        const float2 cs = a.rope[(size_t)pos * half + i];
        const float c = cs.x, s = cs.y;
        const float x0 = r[i], x1 = r[i + half];
        r[i] = x0 * c - x1 * s;
        r[i + half] = x0 * s + x1 * c;
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < a.heads * HD; idx += blockDim.x) a.q[(size_t)t * a.heads * HD + idx] = rows[idx];
    for (int idx = threadIdx.x; idx < kvd; idx += blockDim.x) {
        a.keys[(size_t)pos * kvd + idx] = rows[(size_t)a.heads * HD + idx];
        a.values[(size_t)pos * kvd + idx] = row[qd + kvd + idx];
    }
}

typedef _Float16 half8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4v __attribute__((ext_vector_type(4)));

constexpr int kKeyTile = kAttnKeyTile;
constexpr int kFlashRows = 128;  // query rows (position x head of a KV head's group) per workgroup
constexpr int kFlashThreads = 64 * kFlashRows / 16;
constexpr float kLag = 8.f;      // a row's maximum may pass its reference by this (powers of two)
constexpr float kLow = 2048.f;   // the low fp16 pieces of queries and keys are carried 2^11 times as large

// The exponent that brings a vector of largest magnitude mx to [2^14, 2^15).
__device__ __forceinline__ int piece_exp(float mx) {
    int e = 0;
    if (mx > 0.f && mx < INFINITY) {
        (void)frexpf(mx, &e);
        e = max(e - 15, -126);
    }
    return e;
}
__device__ __forceinline__ void split8(const float (&v)[8], float up, half8& hi, half8& lo) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        const float w = v[k] * up;
        hi[k] = (_Float16)w;
        lo[k] = (_Float16)((w - (float)hi[k]) * kLow);
    }
}
// x = p0 + p1 + p2, each the next 8 significant bits of it as bf16 (a NaN stays one; an
// infinity becomes one).
__device__ __forceinline__ void split3(const float (&v)[8], bf16x8 (&p)[3]) {
    uint32_t w[3][4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
        uint32_t b[3][2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float x = v[2 * k + i];
            b[0][i] = __float_as_uint(x);
            const float r = x - __uint_as_float(b[0][i] & 0xffff0000u);
            b[1][i] = __float_as_uint(r);
            b[2][i] = __float_as_uint(r - __uint_as_float(b[1][i] & 0xffff0000u));
        }
#pragma unroll
        for (int n = 0; n < 3; ++n) w[n][k] = __builtin_amdgcn_perm(b[n][1], b[n][0], 0x07060302u);  // the upper halves
    }
#pragma unroll
    for (int n = 0; n < 3; ++n) p[n] = __builtin_bit_cast(bf16x8, u32x4v{w[n][0], w[n][1], w[n][2], w[n][3]});
}

// Maximum / sum over lanes l, l^16, l^32, l^48 (the lane groups that share a query).
template <class F> __device__ __forceinline__ float over_groups(float x, F f) {
    const auto a = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    x = f(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const auto b = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
    return f(__uint_as_float(b[0]), __uint_as_float(b[1]));
}
__device__ __forceinline__ float max_groups(float x) {
    return over_groups(x, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float sum_groups(float x) {
    return over_groups(x, [](float a, float b) { return a + b; });
}

// Operands of the keys and values of one 32-key tile of one KV head (rows past the last
// key are zero). Keys: half kt, slice s (32 dims), piece p, lane (key l%16, dims 8(l/16) ..
// +7) -> ((kt*HD/32 + s)*2 + p)*512 + 8l halves, 2^e per key in ke. Values: dims tile dt,
// piece p, lane (dim l%16, g) -> (dt*3 + p)*512 + 8l: keys 4g .. 4g+3, 16+4g .. 16+4g+3.
template <int HD>
__global__ __launch_bounds__(256) void attn_split_kv_kernel(AttnBatchArgs a) {
    constexpr int CK = HD / 64;            // 8-dim pieces of a key per thread
    constexpr int CV = HD / 64;            // (dims tile, lane) items per thread
    const int tile = blockIdx.x, kvh = blockIdx.y, tid = threadIdx.x;
    const int L = a.first + a.count, kvd = a.kv_heads * HD, tiles = (L + kKeyTile - 1) / kKeyTile;
    const size_t at = (size_t)kvh * tiles + tile;
    {
        const int key = tid >> 3, j = tid & 7, pos = tile * kKeyTile + key;
        float v[CK][8], mx = 0.f;
#pragma unroll
        for (int i = 0; i < CK; ++i) {
            const float* src = a.keys + (size_t)min(pos, L - 1) * kvd + (size_t)kvh * HD + 8 * (8 * i + j);
            float lo4[4], hi4[4];
            ldv<4>(lo4, src);
            ldv<4>(hi4, src + 4);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[i][k] = pos < L ? lo4[k] : 0.f;
                v[i][4 + k] = pos < L ? hi4[k] : 0.f;
                mx = fmaxf(mx, fmaxf(fabsf(v[i][k]), fabsf(v[i][4 + k])));
            }
        }
        mx = fmaxf(mx, dpp_f<0xb1, 0xf>(mx, mx));   // over the key's 8 threads
        mx = fmaxf(mx, dpp_f<0x4e, 0xf>(mx, mx));
        mx = fmaxf(mx, dpp_f<0x141, 0xf>(mx, mx));
        const int e = piece_exp(mx);
        const float up = ldexpf(1.f, -e);
        if (j == 0) a.ke[at * kKeyTile + key] = ldexpf(1.f, e);
        _Float16* dst = reinterpret_cast<_Float16*>(a.kf) + at * (kKeyTile * HD * 2) + (size_t)(key >> 4) * (HD / 32) * 1024;
#pragma unroll
        for (int i = 0; i < CK; ++i) {
            const int c = 8 * i + j, lane = (c & 3) * 16 + (key & 15);  // dims 8c: slice c/4, group c%4
            half8 hi, lo;
            split8(v[i], up, hi, lo);
            *reinterpret_cast<half8*>(dst + (c >> 2) * 1024 + lane * 8) = hi;
            *reinterpret_cast<half8*>(dst + (c >> 2) * 1024 + 512 + lane * 8) = lo;
        }
    }
    uint16_t* dst = a.vf + at * (kKeyTile * HD * 3);
#pragma unroll
    for (int i = 0; i < CV; ++i) {
        const int item = i * 256 + tid, dt = item >> 6, lane = item & 63, g = lane >> 4;
        float v[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const int pos = tile * kKeyTile + (k >> 2) * 16 + 4 * g + (k & 3);
            const float x = a.values[(size_t)min(pos, L - 1) * kvd + (size_t)kvh * HD + dt * 16 + (lane & 15)];
            v[k] = pos < L ? x : 0.f;
        }
        bf16x8 p[3];
        split3(v, p);
#pragma unroll
        for (int n = 0; n < 3; ++n) *reinterpret_cast<bf16x8*>(dst + (dt * 3 + n) * 512 + lane * 8) = p[n];
    }
}

// Key tiles with a key of the query rows of a half-tile.
__device__ __forceinline__ int flash_tiles(const AttnBatchArgs& a, int rows, int half) {
    const int t_last = (min(rows, (half + 1) * (kFlashRows / 2)) - 1) / (a.heads / a.kv_heads);
    return (a.first + t_last) / kKeyTile + 1;
}

// 128 query rows of one KV head (row r: position r / group, head kvh*group + r % group)
// over the key tiles of one split: 8 waves of 16 rows, queries and outputs in registers, the
// tile's key and value operands shared through LDS, double-buffered. (Four waves of 32 rows
// with 512 registers read half as much LDS but leave one wave per SIMD, with nothing beside
// its softmax and its waits: 843 us against 660 at that stage.)
template <int HD>
__global__ __launch_bounds__(kFlashThreads, 2) void attn_flash_kernel(AttnBatchArgs a) {
    constexpr int TH = kFlashThreads, NS = HD / 32, ND = HD / 16;
    constexpr int KN = kKeyTile * HD * 4 / 16, VN = kKeyTile * HD * 6 / 16;  // 16-byte pieces of a tile's keys, values
    constexpr int KL = KN / TH, VL = (VN + TH - 1) / TH;
    constexpr int KD = 1, VD = 3;  // operands are read this many steps ahead of their products
    // keys of two tiles, values of two tiles; at the end one array for the outputs of all waves
    __shared__ __align__(16) u32x4v KV[2 * KN + 2 * VN];
    static_assert(sizeof(KV) >= (size_t)kFlashRows * HD * sizeof(float), "outputs in KV");
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, qj = lane & 15;
    const int kvh = blockIdx.x, group = a.heads / a.kv_heads, rows = a.count * group;
    const int tiles_all = (a.first + a.count + kKeyTile - 1) / kKeyTile;
    // half-tiles p and n-1-p: waves 0..3 (one per SIMD) have the rows with few keys, waves 4..7
    // those with many, so that every workgroup has about the same work
    const int halves = (rows + kFlashRows / 2 - 1) / (kFlashRows / 2), far = halves - 1 - (int)blockIdx.y;
    const bool near = wave < TH / 128;
    const int half = near ? (int)blockIdx.y : far;
    const int row0 = half * (kFlashRows / 2) + (near ? wave : wave - TH / 128) * 16;
    const int tile0 = blockIdx.z * a.split_tiles;
    const int tile1 = min(flash_tiles(a, rows, far), tile0 + a.split_tiles);
    if (tile0 >= tile1) return;
    const int mine = min(tile1, flash_tiles(a, rows, half));  // this wave's last tile
    const bool active = row0 < rows && tile0 < mine && !(near && half == far);

    const u32x4v* kf = reinterpret_cast<const u32x4v*>(a.kf) + (size_t)kvh * tiles_all * KN;
    const u32x4v* vf = reinterpret_cast<const u32x4v*>(a.vf) + (size_t)kvh * tiles_all * VN;
    u32x4v rk[KL], rv[VL];
    auto load_keys = [&](int tile) {
#pragma unroll
        for (int k = 0; k < KL; ++k) rk[k] = kf[(size_t)tile * KN + k * TH + tid];
    };
    auto load_values = [&](int tile) {
#pragma unroll
        for (int k = 0; k < VL; ++k) rv[k] = vf[(size_t)tile * VN + min(k * TH + tid, VN - 1)];
    };
    auto store_keys = [&](int b) {
#pragma unroll
        for (int k = 0; k < KL; ++k) KV[b * KN + k * TH + tid] = rk[k];
    };
    auto store_values = [&](int b) {
#pragma unroll
        for (int k = 0; k < VL; ++k)
            if (VN % TH == 0 || k * TH + tid < VN) KV[2 * KN + b * VN + k * TH + tid] = rv[k];
    };
    load_keys(tile0);
    load_values(tile0);

    // the wave's queries as operands: lane (query l%16, dims 32s + 8g .. +7)
    half8 qh[NS], ql[NS];
    float qs;                                      // 2^e / sqrt(head_dim) * log2(e): scores in units of log 2
    const int row = min(row0 + qj, rows - 1), last = a.first + row / group;  // the query's last key
    {
        const int t = row / group, h = kvh * group + (row - t * group);
        const float* src = a.q + ((size_t)t * a.heads + h) * HD + 8 * g;
        float v[NS][8], mx = 0.f;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            float lo4[4], hi4[4];
            ldv<4>(lo4, src + 32 * s);
            ldv<4>(hi4, src + 32 * s + 4);
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                v[s][k] = lo4[k], v[s][4 + k] = hi4[k];
                mx = fmaxf(mx, fmaxf(fabsf(lo4[k]), fabsf(hi4[k])));
            }
        }
        const int e = piece_exp(max_groups(mx));
        const float up = ldexpf(1.f, -e);
#pragma unroll
        for (int s = 0; s < NS; ++s) split8(v[s], up, qh[s], ql[s]);
        qs = ldexpf(1.44269504088896340736f / sqrtf((float)HD), e);
    }

    // a tile's scores in log 2 units (S^T of its two key halves), masked, and their maximum
    float x[8], mx;
    float4 ke[2];  // the tile's 2^e
    auto load_scales = [&](int tile) {
        const float* e = a.ke + ((size_t)kvh * tiles_all + tile) * kKeyTile + 4 * g;
        ke[0] = *reinterpret_cast<const float4*>(e);
        ke[1] = *reinterpret_cast<const float4*>(e + 16);
    };
    auto scores = [&](int b, floatx4 (&S)[2], floatx4 (&R)[2]) {
        const half8* K = reinterpret_cast<const half8*>(KV + b * KN);
#pragma unroll
        for (int kt = 0; kt < 2; ++kt) S[kt] = R[kt] = floatx4{0.f, 0.f, 0.f, 0.f};
        half8 kh[KD + 1][2], kl[KD + 1][2];
        auto operands = [&](int s) {
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) {
                kh[s % (KD + 1)][kt] = K[((kt * NS + s) * 2) * 64 + lane];
                kl[s % (KD + 1)][kt] = K[((kt * NS + s) * 2 + 1) * 64 + lane];
            }
        };
#pragma unroll
        for (int s = 0; s < KD && s < NS; ++s) operands(s);
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            if (s + KD < NS) operands(s + KD);
            const int r = s % (KD + 1);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) R[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kl[r][kt], qh[s], R[kt], 0, 0, 0);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) S[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh[r][kt], qh[s], S[kt], 0, 0, 0);
#pragma unroll
            for (int kt = 0; kt < 2; ++kt) R[kt] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kh[r][kt], ql[s], R[kt], 0, 0, 0);
            if (s + KD < NS) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);  // LDS reads, then
            __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);                  // products
        }
    };
    auto scaled = [&](const floatx4 (&S)[2], const floatx4 (&R)[2], int tile) {
        const float e[8] = {ke[0].x, ke[0].y, ke[0].z, ke[0].w, ke[1].x, ke[1].y, ke[1].z, ke[1].w};
        const int key0 = tile * kKeyTile + 4 * g;
        mx = -INFINITY;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const float s = fmaf(R[k >> 2][k & 3], 1.f / kLow, S[k >> 2][k & 3]);
            x[k] = key0 + (k >> 2) * 16 + (k & 3) <= last ? (s * e[k]) * qs : -INFINITY;
            mx = fmaxf(mx, x[k]);
        }
        mx = max_groups(mx);
    };

    floatx4 O[ND], S[2], R[2];
    float m = -INFINITY, l = 0.f;  // the reference of the scores, a whole number; the sum of 2^(score - m - kLag)
#pragma unroll
    for (int d = 0; d < ND; ++d) O[d] = floatx4{0.f, 0.f, 0.f, 0.f};
    load_scales(tile0);
    store_keys(0);
    store_values(0);
    load_keys(min(tile0 + 1, tile1 - 1));
    load_values(min(tile0 + 1, tile1 - 1));
    lds_barrier();
    if (active) {
        scores(0, S, R);
        scaled(S, R, tile0);
    }
    store_keys(1);
    load_keys(min(tile0 + 2, tile1 - 1));
    lds_barrier();
    // Iteration `tile`: the keys two tiles on and the values of the next go to LDS (loaded an
    // iteration before, into what the last one finished with); then the softmax of this tile
    // beside the next tile's scores, and the scaling of those beside P.V, so that the vector
    // work stands next to matrix work that does not wait for it.
    for (int tile = tile0, buf = 0; tile < tile1; ++tile, buf ^= 1) {
        store_keys(buf);
        store_values(buf ^ 1);
        load_keys(min(tile + 3, tile1 - 1));
        load_values(min(tile + 2, tile1 - 1));
        if (active && tile < mine) {
            load_scales(min(tile + 1, tile1 - 1));
            const bf16x8* V = reinterpret_cast<const bf16x8*>(KV + 2 * KN + buf * VN);
            // m follows the maximum only where that passes it by kLag, so O is seldom rescaled;
            // as a whole number it makes the rescaling exact
            if (__ballot(mx > m + kLag)) {
                const float mn = mx > m + kLag ? ceilf(mx) : m;
                const float f = mn == m ? 1.f : __builtin_amdgcn_exp2f(m - mn);
                m = mn;
                l *= f;
#pragma unroll
                for (int d = 0; d < ND; ++d) O[d] *= f;
            }
            const float off = m == -INFINITY ? 0.f : -kLag - m;  // (no key of the row yet: all x are -inf)
            bf16x8 P[3];
            {
                float p[8], sum = 0.f;
#pragma unroll
                for (int k = 0; k < 8; ++k) sum += p[k] = __builtin_amdgcn_exp2f(x[k] + off);
                l += sum;
                split3(p, P);
            }
            scores(buf ^ 1, S, R);
            scaled(S, R, tile + 1);
            // P.V of two dims tiles at a time: the products of pieces i and j for i + j <= 2, the
            // smallest first, in a sum of their own, so that O is rounded once per tile; step
            // (d, n) uses piece 2 - n of the values
            floatx4 T[2];
            bf16x8 v[VD + 1][2];
            auto operands = [&](int i) {
#pragma unroll
                for (int u = 0; u < 2; ++u) v[i % (VD + 1)][u] = V[((2 * (i / 3) + u) * 3 + 2 - i % 3) * 64 + lane];
            };
            constexpr int N = 3 * (ND / 2);
#pragma unroll
            for (int i = 0; i < VD && i < N; ++i) operands(i);
#pragma unroll
            for (int i = 0; i < N; ++i) {
                if (i + VD < N) operands(i + VD);
#pragma unroll
                for (int n = i % 3; n >= 0; --n)
#pragma unroll
                    for (int u = 0; u < 2; ++u)
                        T[u] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(v[i % (VD + 1)][u], P[n], i % 3 ? T[u] : floatx4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                if (i % 3 == 2) {
#pragma unroll
                    for (int u = 0; u < 2; ++u) O[2 * (i / 3) + u] += T[u];
                }
                if (i + VD < N) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                if (i % 3 == 0) __builtin_amdgcn_sched_group_barrier(0x008, 2, 0);
                else if (i % 3 == 1) __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
                else __builtin_amdgcn_sched_group_barrier(0x008, 6, 0);
            }
        }
        lds_barrier();
    }
    if (!active) return;

    // lane: query l%16, dims 16d + 4g .. +3
    const float total = sum_groups(l);
    if (gridDim.z > 1) {
        if (row0 + qj >= rows) return;
        const size_t at = ((size_t)blockIdx.z * a.kv_heads + kvh) * rows + row;
        float* dst = a.part + at * HD;
#pragma unroll
        for (int d = 0; d < ND; ++d) *reinterpret_cast<floatx4*>(dst + 16 * d + 4 * g) = O[d];
        if (g == 0) *reinterpret_cast<float2*>(a.stat + at * 2) = make_float2(m, total);
        return;
    }
    // through this wave's share of LDS, row by row: consecutive lanes write consecutive dims, and
    // the gate's code stands here once (unrolled over the outputs it was 30 KB)
    float* tile = reinterpret_cast<float*>(KV) + wave * (16 * HD);
#pragma unroll
    for (int d = 0; d < ND; ++d) {
        floatx4 o;
#pragma unroll
        for (int k = 0; k < 4; ++k) o[k] = O[d][k] / total;
        *reinterpret_cast<floatx4*>(tile + qj * HD + 16 * d + 4 * g) = o;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int n = min(16, rows - row0);
#pragma unroll 1
    for (int i = 0; i < n; ++i) {
        const int r = row0 + i, t = r / group, h = kvh * group + (r - t * group);
        const float* gate = a.qkv + (size_t)t * a.stride + (size_t)h * HD * 2 + HD;
        float* dst = a.out + (size_t)t * a.out_stride + (size_t)h * HD;
#pragma unroll
        for (int c = lane; c < HD; c += 64) dst[c] = tile[i * HD + c] * sigmoidf_(gate[c]);
    }
}

// Joins the splits of one query row (workgroup = KV head x row, a thread per dim): sum_s
// 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s, then the sigmoid gate. A split whose keys
// all lie past those of the row's half-tile was not run.
__global__ __launch_bounds__(256) void attn_merge_batch_kernel(AttnBatchArgs a, int splits) {
    const int hd = a.head_dim, group = a.heads / a.kv_heads, rows = a.count * group;
    const int kvh = blockIdx.x, r = blockIdx.y, d = threadIdx.x;
    const int t = r / group, h = kvh * group + (r - t * group);
    const int n = min(splits, (flash_tiles(a, rows, r / (kFlashRows / 2)) + a.split_tiles - 1) / a.split_tiles);
    const size_t step = (size_t)a.kv_heads * rows, at = (size_t)kvh * rows + r;
    float M = -INFINITY;
    for (int s = 0; s < n; ++s) M = fmaxf(M, a.stat[(at + s * step) * 2]);
    float num = 0.f, den = 0.f;
    for (int s = 0; s < n; ++s) {
        const float2 st = *reinterpret_cast<const float2*>(a.stat + (at + s * step) * 2);
        const float w = __builtin_amdgcn_exp2f(st.x - M);  // (0 for a split none of whose keys the row has)
        den = fmaf(w, st.y, den);
        num = fmaf(w, a.part[(at + s * step) * hd + d], num);
    }
    const float gate = a.qkv[(size_t)t * a.stride + (size_t)h * hd * 2 + hd + d];
    a.out[(size_t)t * a.out_stride + (size_t)h * hd + d] = num / den * sigmoidf_(gate);
}

}  // namespace

int attention_batch_splits(int heads, int kv_heads, int first, int count) {
    const int rows = count * (heads / kv_heads), wgs = kv_heads * ((rows + kFlashRows - 1) / kFlashRows);
    const int tiles = (first + count + kKeyTile - 1) / kKeyTile;
    // one workgroup per CU, each with at least two tiles
    return std::max(1, std::min(256 / wgs, tiles / 2));
}

hipError_t launch_attention_batch(const AttnBatchArgs& a0, hipStream_t stream) {
    AttnBatchArgs a = a0;
    const int hd = a.head_dim, L = a.first + a.count;
    if (a.count < 1 || a.heads % a.kv_heads || (hd != 64 && hd != 128 && hd != 256)) return hipErrorInvalidValue;
    const size_t prep_lds = (size_t)(a.heads + a.kv_heads) * hd * sizeof(float);
    const int rows = a.count * (a.heads / a.kv_heads), tiles = (L + kKeyTile - 1) / kKeyTile;
    int splits = a.part ? attention_batch_splits(a.heads, a.kv_heads, a.first, a.count) : 1;
    a.split_tiles = (tiles + splits - 1) / splits;
    splits = (tiles + a.split_tiles - 1) / a.split_tiles;
    const dim3 kv_grid(tiles, a.kv_heads), grid(a.kv_heads, (rows + kFlashRows - 1) / kFlashRows, splits);
    if (grid.y > 65535 || rows > 0x7fffffff / 2) return hipErrorInvalidValue;
#define EMPRISE_ATTN_CASE(HD)                                                                             \
    case HD:                                                                                              \
        launch_kernel(attn_prep_batch_kernel<HD / 64>, dim3(a.count), dim3(512), prep_lds, stream, a);     \
        launch_kernel(attn_split_kv_kernel<HD>, kv_grid, dim3(256), 0, stream, a);                         \
        launch_kernel(attn_flash_kernel<HD>, grid, dim3(kFlashThreads), 0, stream, a);                         \
        break;
    switch (hd) {
        EMPRISE_ATTN_CASE(64)
        EMPRISE_ATTN_CASE(128)
        EMPRISE_ATTN_CASE(256)
    }
#undef EMPRISE_ATTN_CASE
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || splits == 1) return e;
    launch_kernel(attn_merge_batch_kernel, dim3(a.kv_heads, rows), dim3(hd), 0, stream, a, splits);
    return hipGetLastError();
}

hipError_t launch_rope_table(float2* table, int context, int rotary, float base, hipStream_t stream) {
    const size_t n = (size_t)context * (rotary / 2);
    if (!n) return hipSuccess;
    launch_kernel(rope_table_kernel, dim3((unsigned)std::min<size_t>((n + 255) / 256, 1024)), dim3(256), 0, stream,
                  table, context, rotary, base);
    return hipGetLastError();
}

size_t attention_partial_floats(int heads, int kv_heads, int head_dim, int context) {
    (void)context;  // (the combine kernel reads kAttnFew slots at every context length)
    return (size_t)kv_heads * kAttnSplit * (heads / kv_heads) * (head_dim + 2);
}

hipError_t launch_attention(const AttnArgs& a, hipStream_t stream) {
    if (a.heads % a.kv_heads || a.heads / a.kv_heads > kMaxGroup || a.rotary > a.head_dim || a.rotary % 2)
        return hipErrorInvalidValue;
    // no more ranges than the caches have sub-chunks (2 KV heads x 64, 1024-position caches: 7.9 us
    // at 16 positions, 8.5 with the empty ranges)
    const dim3 grid(a.kv_heads * std::min(kAttnSplit, (a.context + kAttnSub - 1) / kAttnSub)), block(kAttnWaves * 64);
    const bool few = a.heads / a.kv_heads <= 4;
    switch (a.head_dim) {
    case 64: launch_kernel(few ? attention_kernel<1, 4> : attention_kernel<1, 8>, grid, block, 0, stream, a); break;
    case 128: launch_kernel(few ? attention_kernel<2, 4> : attention_kernel<2, 8>, grid, block, 0, stream, a); break;
    case 256: launch_kernel(few ? attention_kernel<4, 4> : attention_kernel<4, 8>, grid, block, 0, stream, a); break;
    default: return hipErrorInvalidValue;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    launch_kernel(attention_combine_kernel, dim3(a.heads * (a.head_dim / 64)), dim3(256), 0, stream, a);
    return hipGetLastError();
}

}  // namespace emprise
