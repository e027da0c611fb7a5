// Tiled prefill attention for gfx950: the softmax's caller over a whole
// prompt chunk, on the matrix cores.
//
// Reference: the GPU engine's --flash-prefill tier (attention_flash,
// src/gpu/gpu_engine.cpp:3292-3372, with k_flash_softmax 1481-1545 and
// k_flash_finish 1547-1560) over the KV ring of k_kv_append (481-492): query
// row t (position pos0 + t) of head h attends keys j in [lo_t, pos0 + t],
// lo_t = window > 0 ? max(0, pos0 + t - window + 1) : 0, key j in slot
// j % slots of kv head h / (q_heads / kv_heads);
//   S = q.k * scaling, masked keys excluded; per key tile the running
//   (max, sumexp) fold, the accumulator rescale, and P = bf16(e) for the p.v
//   product (e summed in f32); out = acc / sumexp (f32).
// The same numerical contract as the reference's tier: a tile-wise summation
// schedule with bf16 probabilities in the second product, gated on an
// envelope rather than bits.
//
// Layout of the work: a work-group serves one KV head and 256 (or 128, pf_plan)
// (query row, head) pairs of its GQA group, row-major (51.2 rows of a 5-head
// group), 32 pairs a wave; every K/V tile staged in LDS serves all of them, and
// every fragment a wave reads from LDS feeds 32 pairs (v_mfma_f32_32x32x16_bf16).
// Per 64-key step j:
//   staging   coalesced 16-byte loads (whole 256-byte key rows per
//             instruction) of V(j+1) and K(j+3), in registers through most of
//             the step, then written to the free LDS buffers (rows padded so
//             that no read conflicts: counted 0); one barrier per step;
//   S^T       of step j+1: A = 32 keys x 16 dims of K from LDS, B = the wave's
//             32 pairs (registers): C lane (pair n, h) holds 32 keys of its pair;
//   softmax   of step j, per pair in f32 (hardware exp2 of fma(score, scale,
//             -ref)); the pair's two lanes meet in one permlane swap for the
//             maximum, the sum stays apart until the end; a pair's reference
//             maximum moves only when passed by more than 8 (log2 units), so
//             most steps rescale nothing;
//   O^T       += V^T P^T: A = V through the transposing ds_read_b64_tr_b16, B =
//             P straight from the S^T layout; a pair's output stays in its lanes.
// What bounds it: the matrix cores and the vector units, which a SIMD runs at
// once only if they alternate within a wave's own stream (measured: 16 products
// and 112 fma after each other 469 ns a wave, alternating 307; two waves a SIMD,
// one of products and one of fma, 400 where 257 would be full overlap). So the
// scores are formed a step ahead, and the 32 products of a step go out one by
// one with the softmax's instructions spread between them in a fixed order.
// 4096 tokens of 40 / 8 heads, causal: 203 -> 184 us (0.93 PFLOP/s; 1.03 behind a
// 16384-token context) against the earlier 16-row tiles, whose products and
// softmax ran one after the other. A step takes 1.8 us where its products alone
// would take 1.0 (at the 1.9-2.0 GHz the card holds under them); the rest is LDS
// reads (0.4), staging (0.25) and the 7 us a work-group starts and ends with. By
// the counters the matrix cores are busy 45 % of the kernel's cycles and the LDS
// 29 %, without a bank conflict; 5 of the 256 registers spill.
#include "mg_device.hpp"
#include "mg_internal.hpp"
#include "mg_prefill_plan.hpp"

#include <type_traits>

namespace mg
{
    constexpr int kPfAhead = 4;                // K fragments read ahead of the products
    constexpr int kPfVAhead = 3;               // V fragments read ahead

    // out rows need no more than a float's alignment
    typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

    // W waves of 32 (query row, head) pairs each: pair p of the work-group's kv
    // head is query row p / hpg, head p % hpg, so a wave's columns may mix rows
    // and heads (each column is masked and normalised on its own). SPLIT: the
    // work-group takes steps [part * per, (part + 1) * per) of its tile's keys
    // and leaves (reference, sum, unnormalised output) of its pairs in pm / pl / po.
    template <int D, int W, bool SPLIT>
    __global__ __launch_bounds__(64 * W, W / 4) void k_attn_prefill(const uint16_t *__restrict__ q,
                                                            const uint16_t *__restrict__ kc,
                                                            const uint16_t *__restrict__ vc, PfArgs a,
                                                            float *__restrict__ out, float *__restrict__ pm,
                                                            float *__restrict__ pl_, float *__restrict__ po)
    {
        constexpr int KS = kPfKeys, NK = D / 16, ND = D / 32; // k-steps of a score tile, 32-dim output tiles
        // LDS row strides (elements)
        constexpr int SK = D + 8, SV = D + 32;
        constexpr int NTHR = 64 * W, PW = 32 * W;
        constexpr int LPR = D / 8;                       // 16-byte pieces per key row
        constexpr int NPC = KS * LPR;                    // pieces per tile of K (or V)
        static_assert(NPC % NTHR == 0, "whole pieces per thread");
        constexpr int PPH = NPC / NTHR;                  // staged pieces per thread (K or V)
        constexpr int KPP = NTHR / LPR;                  // keys between a thread's pieces
        __shared__ __align__(16) uint16_t lk[3 * KS * SK];
        __shared__ __align__(16) uint16_t lv[2 * KS * SV];
        const int wv = __builtin_amdgcn_readfirstlane(int(threadIdx.x >> 6)), lane = threadIdx.x & 63, tid = threadIdx.x;
        const int n = lane & 31, h = lane >> 5;
        // the last pair tiles attend the most keys: they start first
        const uint32_t parts = SPLIT ? uint32_t(a.parts) : 1u;
        const uint32_t per_tile = uint32_t(a.nkv) * parts;
        const uint32_t ot = blockIdx.x / per_tile;
        const uint32_t qt = ot < a.nfirst ? a.nfirst - 1 - ot : a.nqt - 1 - (ot - a.nfirst);
        const uint32_t gp = blockIdx.x % per_tile;
        const int64_t g = gp / parts;
        const uint32_t part = gp % parts;
        const uint32_t pb0 = qt * PW;                                           // the work-group's first pair
        const uint32_t pl = (pb0 + PW < a.npair ? pb0 + PW : a.npair) - 1;      // its last live pair
        const PfSpan ks = pf_span(a.pos0, a.window, a.hpg, a.hw, pb0, pl);
        // key positions below are offsets from klo; this work-group's are [s0, s1]
        const int s0 = SPLIT ? int(part) * a.per * KS : 0;
        if (SPLIT && s0 > ks.span) return; // a part past the tile's keys (the whole work-group)
        const int s1 = SPLIT && s0 + a.per * KS - 1 < ks.span ? s0 + a.per * KS - 1 : ks.span;
        const uint32_t pw0 = pb0 + 32 * wv; // this wave's first pair

        // this lane's pair: its query row and head, its keys [ql, qp]
        const uint32_t pr = pw0 + n;
        const uint32_t pc = pr <= pl ? pr : pl;
        const uint32_t row = pc / a.hpg;
        const int64_t hd = g * a.hpg + (pc - row * a.hpg);
        const int base0 = int(a.pos0 - ks.klo);
        const int qp = base0 + int(row);
        const int64_t lo = a.window > 0 ? int64_t(qp) - a.window + 1 : 0;
        const int ql = lo > 0 ? int(lo) : 0;
        // the steps every row of the work-group attends whole: [f0, f1)
        const int64_t wl = a.window > 0 ? int64_t(ks.span) - a.window + 1 : 0;
        const int fs = wl > s0 ? s0 + (int(wl) - s0 + KS - 1) / KS * KS : s0;
        const int f0 = fs < s1 + 1 ? fs : s1 + 1;
        const int fe = base0 + int(pb0 / a.hpg) + 1 < s1 + 1 ? base0 + int(pb0 / a.hpg) + 1 : s1 + 1; // first masked key
        const int f1 = fe > f0 ? f0 + (fe - f0) / KS * KS : f0;

        // B of S^T: lane (pair n, h) holds q[row][head][16 kb + 8h ..]
        bf16x8 qop[NK];
#pragma unroll
        for (int kb = 0; kb < NK; ++kb) {
            Vec<uint32_t, 4> w = __builtin_bit_cast(Vec<uint32_t, 4>, ld_bf16x8(q + row * a.ldq + hd * D + 16 * kb + 8 * h));
#pragma unroll
            for (int i = 0; i < 4; ++i) w.v[i] ^= a.qsign;
            qop[kb] = __builtin_bit_cast(bf16x8, w);
        }

        // staging, K and V separately (one of them in registers at a time):
        // piece u of thread tid is key tid / LPR + KPP u of the step, 16 bytes
        // at column tid % LPR. A key past s1 re-reads s1's row (masked for
        // every row but those attending it, so nothing stands behind a branch).
        const int skey = tid / LPR, scol = 8 * (tid % LPR);
        const uint32_t ring = a.slots < 0x7fffffff ? uint32_t(a.slots) : 0x7fffffffu;
        const uint32_t slot0 = uint32_t(ks.klo < a.slots ? ks.klo : ks.klo % a.slots); // ring slot of key 0
        const uint32_t rowb = uint32_t(a.nkv * D * 2);     // bytes between a ring's slots
        const char *kg = reinterpret_cast<const char *>(kc + g * D + scol), *vg = reinterpret_cast<const char *>(vc + g * D + scol);
        auto stage = [&](u32x4(&stg)[PPH], const char *src, int jb) {
#pragma unroll
            for (int u = 0; u < PPH; ++u) {
                const int j = jb + skey + KPP * u;
                uint32_t sl = slot0 + uint32_t(j < s1 ? j : s1);
                sl = sl >= ring ? sl - ring : sl;
                stg[u] = *reinterpret_cast<const u32x4 *>(src + uint64_t(sl) * rowb);
            }
        };
        auto commit = [&](const u32x4(&stg)[PPH], uint16_t *dst, int stride) {
#pragma unroll
            for (int u = 0; u < PPH; ++u) *reinterpret_cast<u32x4 *>(dst + (skey + KPP * u) * stride + scol) = stg[u];
        };

        // O^T: lane (pair n, h) holds dims 32 t + 8 (r / 4) + 4h + r % 4 of its pair
        f32x16 o[ND];
#pragma unroll
        for (int t = 0; t < ND; ++t)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[t][r] = 0.0f;
        float m = -__builtin_huge_valf(), l = 0.0f;

        // The K fragment of product x of a score tile pair: lane (key n, h) holds
        // dims 16 (x / 2) + 8h.. of key 32 (x % 2) + n
        auto kread = [&](const uint16_t *sk, int x) {
            return *reinterpret_cast<const bf16x8 *>(sk + 32 * (x % 2) * SK + 16 * (x / 2));
        };
        const int koff = n * SK + 8 * h;
        // V^T of product x of the p.v products: lane (dim 32 (x % ND) + l % 32, h)
        // gets keys 16 (x / ND) + 8 g + 4h + 0..3 from the transposing read (lane
        // 4j + c of each 16 addresses key .. + j, dims 4c.. of the 16)
        auto vread = [&](const uint16_t *vr, int x) {
            const bf16x4 v0 = lds_read_tr(vr + 16 * (x / ND) * SV + 32 * (x % ND));
            const bf16x4 v1 = lds_read_tr(vr + (16 * (x / ND) + 8) * SV + 32 * (x % ND));
            return bf16x8{v0[0], v0[1], v0[2], v0[3], v1[0], v1[1], v1[2], v1[3]};
        };
        const int voff = (4 * h + ((lane & 15) >> 2)) * SV + 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        auto fmax2 = [](float x, float y) { return __builtin_fmaxf(x, y); };
        auto mask = [&](f32x16(&s)[2], int jb) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    const int j = jb + 32 * t + 8 * (r / 4) + 4 * h + r % 4;
                    s[t][r] = (j > qp || j < ql) ? -__builtin_huge_valf() : float(s[t][r]);
                }
        };

        // At the top of step j its scores S(j) (lane (pair n, h) holds keys
        // 32 t + 8 (r / 4) + 4h + r % 4, unscaled: scale2 > 0 multiplies inside
        // the exponent) and their maximum mx are in registers, K(j+1) and K(j+2)
        // in lk at k1 and k2 and V(j) in lv[cur]; the other two buffers, read
        // before the last barrier, are free for K(j+3) and V(j+1). (K is a step
        // further ahead so that the next step's first fragments are read before
        // the barrier: no product waits for the LDS right after it.)
        int cur = 0, k1 = KS * SK, k2 = 2 * KS * SK, k3 = 0;
        bf16x8 ka[kPfAhead + 1]; // K(j+1)'s first fragments
        float mx;
        auto step = [&](f32x16(&s)[2], f32x16(&sn)[2], int jb, auto masked, auto last_) {
            constexpr bool LAST = decltype(last_)::value;
            u32x4 stk[PPH], stv[PPH];
            if constexpr (!LAST) {
                stage(stv, vg, jb + KS); // in flight through the step
                stage(stk, kg, jb + 3 * KS);
            }
            // lazy reference: a pair's reference moves only when its new
            // maximum passes the old by more than 8 (log2 units), so its
            // weights stay at most 2^8 (exact to scale in f32 and bf16)
            // and most steps rescale nothing; a pair with nothing attended
            // yet (m = -inf) takes the first finite maximum
            const bool mv = mx > m + 8.0f;
            if (__builtin_amdgcn_ballot_w64(mv) != 0) {
                const float mn = mv ? mx : m;
                const float corr = __builtin_amdgcn_exp2f(m - (mn == -__builtin_huge_valf() ? 0.0f : mn));
                if (mv) {
                    l *= corr;
#pragma unroll
                    for (int t = 0; t < ND; ++t)
#pragma unroll
                        for (int r = 0; r < 16; ++r) o[t][r] *= corr;
                }
                m = mn;
            }
            // a pair with nothing attended yet keeps a zero reference: its
            // weights are 2^-inf = 0 and nothing is rescaled into NaN
            const float mref = m == -__builtin_huge_valf() ? 0.0f : m;
            // P as B of the p.v product of 16 keys: element 4g + e of group i is
            // key 16 i + 8 g + 4h + e; two weights at a time
            bf16x8 pb[4];
            float ps[2] = {0.0f, 0.0f};
            auto weights = [&](int pr0, int pr1) {
#pragma unroll
                for (int w = pr0; w < pr1; ++w)
#pragma unroll
                    for (int d = 0; d < 2; ++d) {
                        const int i = w / 4, e = 2 * (w % 4) + d;
                        const float p = __builtin_amdgcn_exp2f(__builtin_fmaf(s[i / 2][8 * (i % 2) + e], a.scale2, -mref));
                        pb[i][e] = __bf16(p);
                        ps[d] += p;
                        __asm__ volatile("" : "+v"(ps[d])); // the sum here, not after the products
                    }
            };
            const uint16_t *vr = lv + cur * (KS * SV) + voff;
            bf16x8 va[kPfVAhead + 1];
            // The products go out one at a time, each with the fragment a few
            // products ahead and a share of the vector work under it: a wave's
            // own vector instructions run under its products, another wave's
            // only in part.
            if constexpr (!LAST) {
                // S(j+1) = K(j+1) Q^T, with the weights of three of S(j)'s four key groups
                constexpr int NX = 2 * NK;
                const uint16_t *sk = lk + k1 + koff;
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sn[t][r] = 0.0f;
#pragma unroll
                for (int x = 0; x < NX; ++x) {
                    __builtin_amdgcn_sched_barrier(0);
                    if (x + kPfAhead < NX) ka[(x + kPfAhead) % (kPfAhead + 1)] = kread(sk, x + kPfAhead);
                    sn[x % 2] = mfma_bf16_32(ka[x % (kPfAhead + 1)], qop[x / 2], sn[x % 2]);
                    weights(12 * x / NX, 12 * (x + 1) / NX);
                    if (x >= NX - kPfVAhead) va[x - NX + kPfVAhead] = vread(vr, x - NX + kPfVAhead);
                }
                __builtin_amdgcn_sched_barrier(0);
            } else {
                weights(0, 12);
#pragma unroll
                for (int x = 0; x < kPfVAhead; ++x) va[x] = vread(vr, x);
            }
            // O^T += V^T P^T, with the last group's weights and S(j+1)'s maximum
            constexpr int NX = 4 * ND;
            if constexpr (!LAST && decltype(masked)::value) mask(sn, jb + KS);
            float nx = -__builtin_huge_valf();
#pragma unroll
            for (int x = 0; x < NX; ++x) {
                __builtin_amdgcn_sched_barrier(0);
                if (x + kPfVAhead < NX) va[(x + kPfVAhead) % (kPfVAhead + 1)] = vread(vr, x + kPfVAhead);
                o[x % ND] = mfma_bf16_32(va[x % (kPfVAhead + 1)], pb[x / ND], o[x % ND]);
                if (x < NX / 2) weights(12 + 4 * x / (NX / 2), 12 + 4 * (x + 1) / (NX / 2));
                if constexpr (!LAST) {
#pragma unroll
                    for (int r = 32 * x / NX; r < 32 * (x + 1) / NX; ++r) nx = __builtin_fmaxf(nx, sn[r / 16][r % 16]);
                    __asm__ volatile("" : "+v"(nx));
                }
                if constexpr (!LAST) {
                    if (x == NX / 2) commit(stv, lv + (cur ^ 1) * (KS * SV), SV);
                    if (x == NX / 2 + 1) commit(stk, lk + k3, SK);
                    if (x >= NX - kPfAhead) ka[x - NX + kPfAhead] = kread(lk + k2 + koff, x - NX + kPfAhead);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            l += ps[0] + ps[1];
            if constexpr (!LAST) {
                mx = lane_pair<32>(nx, fmax2) * a.scale2;
                __syncthreads(); // the next buffers are written; these are free again
                cur ^= 1;
                const int k0 = k1;
                k1 = k2;
                k2 = k3;
                k3 = k0;
            }
        };
        f32x16 sa[2], sb[2];
        {
            u32x4 t0[PPH], t1[PPH], t2[PPH], t3[PPH];
            stage(t0, kg, s0);
            stage(t1, kg, s0 + KS);
            stage(t2, kg, s0 + 2 * KS);
            stage(t3, vg, s0);
            auto first = [&](const uint16_t *sk, int j0, bool whole) {
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int r = 0; r < 16; ++r) sa[t][r] = 0.0f;
#pragma unroll
                for (int x = 0; x < 2 * NK; ++x) sa[x % 2] = mfma_bf16_32(kread(sk, x), qop[x / 2], sa[x % 2]);
                if (!whole) mask(sa, j0);
                float nx = -__builtin_huge_valf();
#pragma unroll
                for (int r = 0; r < 32; ++r) nx = __builtin_fmaxf(nx, sa[r / 16][r % 16]);
                return lane_pair<32>(nx, fmax2) * a.scale2;
            };
            // A later part starts from the reference its pairs have in an unsplit
            // call, their maximum over the first step that holds keys of theirs
            // (one step but for windows over tiles of many rows): the weights, as
            // rounded to bf16, are then the same however the keys are split, unless
            // a reference moves in an earlier part. (Through V(1)'s buffer; 100
            // tokens of 32 / 2 heads at 9000: 34.7 -> 35.3 us.)
            if constexpr (SPLIT)
                for (int j0 = 0; j0 < s0 && (j0 == 0 || j0 <= wl); j0 += KS) {
                    u32x4 tr[PPH];
                    stage(tr, kg, j0);
                    commit(tr, lv + KS * SV, SK);
                    __syncthreads();
                    const float mj = first(lv + KS * SV + koff, j0, false);
                    m = m == -__builtin_huge_valf() ? mj : m;
                    __syncthreads();
                }
            commit(t0, lk, SK);
            commit(t1, lk + k1, SK);
            commit(t2, lk + k2, SK);
            commit(t3, lv, SV);
            __syncthreads();
            mx = first(lk + koff, s0, f0 == s0 && f1 > s0);
#pragma unroll
            for (int x = 0; x < kPfAhead; ++x) ka[x] = kread(lk + k1 + koff, x);
            __syncthreads(); // lk[0] is free for K(3)
        }
        // steps by whether the step after them (whose scores they form) is masked
        using yes = std::true_type;
        using no = std::false_type;
        auto move = [&]() {
            sa[0] = sb[0];
            sa[1] = sb[1];
        };
        int jb = s0;
        for (; jb + KS <= s1 && jb + KS < f0; jb += KS) {
            step(sa, sb, jb, yes{}, no{});
            move();
        }
        for (; jb + 2 * KS < f1; jb += 2 * KS) {
            step(sa, sb, jb, no{}, no{});
            step(sb, sa, jb + KS, no{}, no{});
        }
        if (jb + KS < f1) {
            step(sa, sb, jb, no{}, no{});
            move();
            jb += KS;
        }
        for (; jb + KS <= s1; jb += KS) {
            step(sa, sb, jb, yes{}, no{});
            move();
        }
        step(sa, sb, jb, no{}, yes{});

        l = lane_pair<32>(l, [](float x, float y) { return x + y; });
        if (pr > pl) return;
        float *dst;
        float f = 1.0f;
        if constexpr (SPLIT) {
            // the part's (reference, sum, output) of pair i of tile (qt, g) at
            // slot ((qt nkv + g) parts + part) PW + i
            const int64_t i = ((int64_t(qt) * a.nkv + g) * parts + part) * PW + (pr - pb0);
            if (h == 0) {
                pm[i] = m;
                pl_[i] = l;
            }
            dst = po + i * D;
        } else {
            f = l > 0.0f ? 1.0f / l : 0.0f; // out = acc / sumexp
            dst = out + row * a.ldo + hd * D;
        }
#pragma unroll
        for (int t = 0; t < ND; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const f32x4u w = {o[t][4 * r] * f, o[t][4 * r + 1] * f, o[t][4 * r + 2] * f, o[t][4 * r + 3] * f};
                *reinterpret_cast<f32x4u *>(dst + 32 * t + 8 * r + 4 * h) = w;
            }
    }

    // The parts of one (row, head) pair merged: M = max of the references,
    // out = sum 2^(m_p - M) o_p / sum 2^(m_p - M) l_p over the parts holding
    // keys the row attends. WPP waves a pair (a power of two, 4 waves a
    // work-group): D / 4 lanes take one part's output in 16-byte pieces, so a
    // wave has 64 / (D / 4) parts in flight per load.
    template <int D, int WPP>
    __global__ __launch_bounds__(256) void k_attn_prefill_merge(PfArgs a, const float *__restrict__ pm,
                                                                const float *__restrict__ pl,
                                                                const float *__restrict__ po, float *__restrict__ out)
    {
        constexpr int LPP = D / 4, GPW = 64 / LPP; // lanes per part, parts per wave and load
        constexpr int PPB = 4 / WPP;               // pairs per work-group
        __shared__ float so[4][D];
        __shared__ float sl[4];
        const int wv = threadIdx.x >> 6, lane = threadIdx.x & 63, ww = wv % WPP;
        const int64_t x = int64_t(blockIdx.x) * PPB + wv / WPP; // pair of all kv heads
        const bool live = x < a.nkv * int64_t(a.npair);
        const int64_t xc = live ? x : 0;
        const int64_t g = xc / a.npair;
        const uint32_t pr = uint32_t(xc - g * a.npair);
        const uint32_t PW = 1u << a.lw, qt = pr >> a.lw, pb0 = qt << a.lw;
        const PfSpan ks = pf_span(a.pos0, a.window, a.hpg, a.hw, pb0, pb0 + PW < a.npair ? pb0 + PW - 1 : a.npair - 1);
        const uint32_t row = pr / a.hpg;
        // the row's keys are [ql, qp] of the tile's: the parts that hold them
        const int qp = int(a.pos0 - ks.klo) + int(row), pk = a.per * kPfKeys;
        const int64_t lo = a.window > 0 ? int64_t(qp) - a.window + 1 : 0;
        const int f = (lo > 0 ? int(lo) : 0) / pk, e = qp / pk; // first and last part
        const int64_t base = ((int64_t(qt) * a.nkv + g) * a.parts << a.lw) + (pr - pb0);
        float M = -__builtin_huge_valf();
        for (int p = f + lane; p <= e; p += 64) M = __builtin_fmaxf(M, pm[base + (int64_t(p) << a.lw)]);
        M = dpp_max(M);
        const float ref = M == -__builtin_huge_valf() ? 0.0f : M;
        const int grp = lane / LPP, d0 = 4 * (lane % LPP);
        float L = 0.0f;
        float o[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll 4
        for (int p = f + ww * GPW + grp; p <= e; p += GPW * WPP) {
            const int64_t i = base + (int64_t(p) << a.lw);
            const float w = __builtin_amdgcn_exp2f(pm[i] - ref);
            const Vec<float, 4> v = *reinterpret_cast<const Vec<float, 4> *>(po + i * D + d0);
            L = __builtin_fmaf(w, pl[i], L);
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = __builtin_fmaf(w, v.v[k], o[k]);
        }
        // the wave's part groups, in order of the lane halves (quarters)
        auto add = [](float x, float y) { return x + y; };
        if constexpr (GPW == 4) L = lane_pair<16>(L, add);
        L = lane_pair<32>(L, add);
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            if constexpr (GPW == 4) o[k] = lane_pair<16>(o[k], add);
            o[k] = lane_pair<32>(o[k], add);
        }
        if constexpr (WPP > 1) {
            if (grp == 0)
                *reinterpret_cast<Vec<float, 4> *>(&so[wv][d0]) = Vec<float, 4>{{o[0], o[1], o[2], o[3]}};
            if (lane == 0) sl[wv] = L;
            __syncthreads();
            if (ww != 0) return;
            L = 0.0f;
#pragma unroll
            for (int k = 0; k < 4; ++k) o[k] = 0.0f;
#pragma unroll
            for (int i = 0; i < WPP; ++i) {
                L += sl[wv + i];
#pragma unroll
                for (int k = 0; k < 4; ++k) o[k] += so[wv + i][d0 + k];
            }
        }
        if (!live || grp != 0) return;
        const float inv = L > 0.0f ? 1.0f / L : 0.0f;
        const int64_t hd = g * a.hpg + (pr - row * a.hpg);
        float *dst = out + row * a.ldo + hd * D + d0;
#pragma unroll
        for (int k = 0; k < 4; ++k) dst[k] = o[k] * inv;
    }

    void launch_attn_prefill(mg_ctx *c, const uint16_t *q, int64_t ldq, const uint16_t *kc, const uint16_t *vc,
                             int64_t T, int64_t nq, int64_t nkv, int64_t D, int64_t slots, int64_t pos0,
                             int64_t window, double scaling, float *out, int64_t ldo)
    {
        need(nq > 0 && nkv > 0 && nq % nkv == 0, "attn_prefill: q_heads must be a multiple of kv_heads");
        const int64_t hpg = nq / nkv;
        need(D == 64 || D == 128, "attn_prefill: head_dim must be 64 or 128");
        need(T >= 0 && pos0 >= 0 && slots > 0, "attn_prefill: bad shape");
        need(q && kc && vc && out, "attn_prefill: NULL tensor");
        if (ldq == 0) ldq = nq * D;
        if (ldo == 0) ldo = nq * D;
        need(ldq >= nq * D && ldo >= nq * D && ldq % 8 == 0, "attn_prefill: token stride too small or unaligned");
        need(aligned16(q) && aligned16(kc) && aligned16(vc), "attn_prefill: q and caches must be 16-byte aligned");
        if (T == 0) return;
        const int64_t lo0 = window > 0 ? (pos0 - window + 1 > 0 ? pos0 - window + 1 : 0) : 0;
        need(pos0 + T - 1 - lo0 + 1 <= slots,
             "attn_prefill: the attended keys do not fit the cache ring (pos0 + T - lo > cache_slots)");
        const int64_t npair = T * hpg;
        need(npair <= int64_t(0x7fffffff) && npair / 256 * nkv <= int64_t(0x7ffffff), "attn_prefill: too many query tiles");
        // the kernel scales inside the exponent by a positive factor: a negative
        // scaling flips the sign of q instead (exact in bf16 and in the products),
        // and a zero one becomes 2^-126, under which every exponent of a finite
        // score is below 2^-100 in magnitude and exp2 returns 1 as it does at 0
        const float s2 = float(double(float(scaling)) * 1.4426950408889634);
        PfArgs a{nkv, ldq, ldo, slots, pos0, window, uint32_t(npair), uint32_t(hpg), 0, 0, 0, 0, 1, 0,
                 s2 == 0.0f ? 0x1p-126f : __builtin_fabsf(s2), s2 < 0.0f ? 0x80008000u : 0u};
        pf_plan(a, c->num_cus, c->work_bytes, D);
        const int64_t tiles = int64_t(a.nqt) * nkv;
        // the tiles past a whole number of rounds are the shortest, and start
        // first: longest first alone leaves them to the end of the last round,
        // on part of the CUs (4096 tokens of 40 / 8 heads: 190 -> 185 us)
        if (a.parts == 1 && tiles > c->num_cus) a.nfirst = uint32_t(tiles % c->num_cus / nkv);
        const int64_t slots_out = tiles * a.parts << a.lw;
        float *po = static_cast<float *>(c->work);
        float *pm = po + slots_out * D, *pl = pm + slots_out;
        const dim3 grid{unsigned(tiles * a.parts), 1u, 1u};
        auto go = [&](auto kern) {
            hipLaunchKernelGGL(kern, grid, dim3(64u << (a.lw - 5)), 0, c->stream, q, kc, vc, a, out, pm, pl, po);
        };
        auto by_width = [&](auto wide, auto narrow) { a.lw == 8 ? go(wide) : go(narrow); };
        if (a.parts == 1) {
            if (D == 128)
                by_width(k_attn_prefill<128, 8, false>, k_attn_prefill<128, 4, false>);
            else
                by_width(k_attn_prefill<64, 8, false>, k_attn_prefill<64, 4, false>);
            check_launch("k_attn_prefill");
            return;
        }
        if (D == 128)
            by_width(k_attn_prefill<128, 8, true>, k_attn_prefill<128, 4, true>);
        else
            by_width(k_attn_prefill<64, 8, true>, k_attn_prefill<64, 4, true>);
        check_launch("k_attn_prefill");
        auto merge = [&](auto kern, int64_t ppb) {
            hipLaunchKernelGGL(kern, dim3(unsigned((npair * nkv + ppb - 1) / ppb)), dim3(256), 0, c->stream, a, pm, pl, po, out);
        };
        // four waves a pair once a pair has more parts than one wave has in flight
        if (D == 128)
            a.parts > 16 ? merge(k_attn_prefill_merge<128, 4>, 1) : merge(k_attn_prefill_merge<128, 1>, 4);
        else
            a.parts > 16 ? merge(k_attn_prefill_merge<64, 4>, 1) : merge(k_attn_prefill_merge<64, 1>, 4);
        check_launch("k_attn_prefill_merge");
    }
} // namespace mg
