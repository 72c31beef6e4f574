// Attention-JVP backward for key axes beyond one workgroup, 16-wide form (gfx950): a row-owned and a
// column-owned launch (mathematics in sjvp_bwd.hpp) with 16 owned positions per wavefront,
// so that several wavefronts share a SIMD and a workgroup's copies overlap another's arithmetic.
//   bwd_row16_kernel   4 waves x 16 queries; streams K, V (, K_dot, V_dot)        -> dQ (, dQ_dot)
//   bwd_col16_kernel   4 waves x 16 keys;    streams Q (, Q_dot, G) (, dO) + stats -> dK, dV (, dK_dot, dV_dot)
// (workgroups of four waves: at 160-200 registers two or three of them share a CU)
// NC = 2: a wave owns 2 x 16 positions and every operand that it reads from LDS feeds twice as many matrix instructions
// (the transposing reads deliver 128 bytes per clock and CU, one operand of 1 KB in the time of half a matrix
// instruction of each of its four SIMDs: with 16 positions and no tangents every operand feeds one instruction, and the
// LDS is what such a kernel waits for).  Only where 256 registers hold it: measured beside the dispatch.
// The owned rows are loaded straight into registers (each lane its own 16-byte pieces), the streamed
// side goes through an LDS ring filled by LDS-DMA (IO = kIoDma), or, where the rows do not start on 16-byte boundaries
// or hold fp32 elements, through registers one stage ahead (sjvp_staged16.hpp).  Each gradient is accumulated in fp32 registers by
// exactly one wavefront and written once: deterministic, no atomics.
//
// Row sums.  The row-owned kernel starts from s4' = rowsum(G*O), s7d' = rowsum(G*TO) + rowsum(dO*O),
// formed from the 16-bit outputs, whose rounding leaves s4' = s4 + e4, s7d' = s7d + e7.  With the exact
// sums, sum_j dS_dot_ij = sum_j dS_ij = 0 for every query i; with the rounded ones the sums over the
// keys come out as rho4 = -e4 and rho7 = -e7.  A wave owns whole query rows, so it accumulates both
// residues in fp32 beside its tiles (per-lane adds) and
//   - leaves the corrected sums s4' + rho4 = sum_j P W, s7d' + rho7 = sum_j P (N W + XY) in the
//     workspace: the column-owned kernel works with the sums the reference's preprocess kernel forms
//     from the probabilities (semicat/jvp_utils/flash_jvp_backward.py:2266-2287).  They are stored
//     negated: both kernels start the accumulators of W and XY from minus the sums, so that W - s4 and
//     XY - s7d come out of the matrix cores and cost no vector instruction;
//   - flags its workgroup where a residue is not small against the row's |dS_dot| / |dS| mass (sharp
//     rows, gradients formed by cancellation).  A second launch of the same kernel (PASS = 2) runs the
//     flagged workgroups again with the corrected sums, so that their dQ, dQ_dot are formed from tiles
//     that were rounded without the residue in them; the others leave at once.
// BwdParams::rowfix: 0 no second launch; 1 as described; 2 every workgroup runs twice and the first
// launch (PASS = 1) only measures (the reference's preprocess + backward structure).
#pragma once
#include "sjvp_bwd.hpp"
#include "sjvp_staged16.hpp"

namespace sjvp {

constexpr int kXWaves16 = 4;
constexpr int kXThreads16 = 64 * kXWaves16;
constexpr int kXOwned16 = 16 * kXWaves16;  // owned positions per workgroup

// sum over the 16-bit pairs of a[i]*b[i]
template <typename T>
__device__ __forceinline__ float dot8(const u32x4& a, const u32x4& b) {
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) s = T::dot2(a[i], b[i], s);
    return s;
}

// ---------------------------------------------------------------------------------------------
// Row-owned kernel.  LDS: [ring of K | V (| K_dot | V_dot) stages][sink]; the ring doubles as store
// staging after the last stage.
template <int HD, int R, bool HAS_G, int SPLIT = 1>
struct Row16Smem {
    static constexpr int nt = HAS_G ? 4 : 2;
    static constexpr int slot = nt * Slab<HD>::elems;
    static constexpr int loop = R * slot * (int)sizeof(elem_t);
    static constexpr int after = SPLIT > 1 ? Split16Smem<HD, kXWaves16, HAS_G ? 2 : 1>::bytes : 0;
    static constexpr int sink = loop > after ? loop : after;
    static constexpr int bytes = sink + kSink16;
    static_assert(R * slot >= kXWaves16 * StoreStage16<HD>::elems, "ring too small to stage stores");
};

// (the body of the kernel as a function of the workgroup's index and the number of workgroups, so that the
// second launch can also ride at the end of the column-owned launch, see bwd_col16_repair_kernel)
// SPLIT > 1 (launches of few workgroups): the SPLIT waves of a group share 16 queries and take every SPLIT-th stage each, SPLIT
// stages to a barrier (ring of 2 SPLIT); their sums meet in LDS at the end, in a fixed order.
template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int PASS, int IO, int NC = 1, int SPLIT = 1,
          int DT = HD / 16>
__device__ __forceinline__ void bwd_row16_body(const BwdParams p, const int block, const int blocks) {
    constexpr bool DMA = IO == kIoDma;
    constexpr bool SECOND = PASS == 2;   // second launch: sums from the workspace, flagged workgroups only
    constexpr bool MEASURE = PASS == 1;  // first launch of "always": residues and sums only, no gradients
    extern __shared__ __align__(16) unsigned char smem_raw[];
    using SM = Row16Smem<HD, R, HAS_G, SPLIT>;
    elem_t* ring = reinterpret_cast<elem_t*>(smem_raw);
    constexpr int SE = Slab<HD>::elems;
    constexpr int KL = HD / 32, KC = (DT + 1) / 2;  // 32-column chunks of a row, and those with columns below D
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int g = lane >> 4;
    static_assert(NC == 1 || PASS == 0, "the passes of the repair go by blocks of 64 rows");
    static_assert(SPLIT == 1 || (PASS == 0 && NC == 1 && R == 2 * SPLIT), "a step is a stage for every part");
    const int part = SPLIT > 1 ? wave % SPLIT : 0, group = wave / SPLIT;
    constexpr int OWNED = NC * kXOwned16 / SPLIT;
    const int q_blocks = p.Lr / OWNED;  // statistic rows up to Lr are all covered
    // Workgroups run through the heads in descending order: this launch follows the forward, which
    // ran through them in ascending order, so it starts on what the caches still hold (the
    // column-owned launch after it ascends again).
    const int bid = blocks - 1 - xcd_linear_id(block, blocks);
    const int bh = bid / q_blocks;
    const int qb = bid % q_blocks;
    const int b = bh / p.H, h = bh % p.H;
    const int q0 = qb * OWNED;
    const int wrow = q0 + group * 16 * NC;  // the wave's first query; the lane's are wrow + 16 u + n
    const bool wave_active = wrow < p.Lq;
    if constexpr (SECOND) {
        if (p.rowfix == 1 && p.flags[bid] == 0) return;  // nothing to repair in this workgroup's rows
    }

    // The own rows are requested first, as B operands; the set-up of the stage copies runs while they travel.
    u32x4 qB[NC][KL], tqB[NC][KL], gB[NC][KL], doB[NC][KL];
    u32x4 oR[NC][KL], toR[NC][KL];
    float lse_in[NC], mu_in[NC];
    const int64_t so = (int64_t)bh * p.Lr + wrow + n;  // rows below Lr exist in every statistic
    if (DMA && p.q_side_uniform && p.D == HD && q0 + OWNED <= p.Lq) {
        // the common case: whole rows that all exist, every tensor with q's strides
        const int64_t slice = b * p.q.sb + h * p.q.sh;
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const uint32_t at = ((uint32_t)(wrow + 16 * u + n) * (uint32_t)p.q.sl + 8u * (uint32_t)g) * (uint32_t)sizeof(elem_t);
            load_b_operands16_at<HD>(qB[u], p.q.ptr + slice, at);
            if constexpr (!SECOND) load_b_operands16_at<HD>(oR[u], p.o.ptr + slice, at);
            if constexpr (HAS_G) {
                load_b_operands16_at<HD>(tqB[u], p.tq.ptr + slice, at);
                load_b_operands16_at<HD>(gB[u], p.dTO.ptr + slice, at);
                if constexpr (!SECOND) load_b_operands16_at<HD>(toR[u], p.to.ptr + slice, at);
            }
            if constexpr (HAS_DO) load_b_operands16_at<HD>(doB[u], p.dO.ptr + slice, at);
        }
    } else {
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const bool qvalid = wrow + 16 * u + n < p.Lq;
            const int64_t qrow = IO == kIoAny ? own_row(wrow + 16 * u + n, p.Lq) : wrow + 16 * u + n;
            load_b_operands16<T, HD, IO, true>(qB[u], p.q.head(b, h) + qrow * p.q.sl, g, p.D, qvalid);
            if constexpr (!SECOND) load_b_operands16<T, HD, IO, true>(oR[u], p.o.head(b, h) + qrow * p.o.sl, g, p.D, qvalid);
            if constexpr (HAS_G) {
                load_b_operands16<T, HD, IO, true>(tqB[u], p.tq.head(b, h) + qrow * p.tq.sl, g, p.D, qvalid);
                load_b_operands16<T, HD, IO, true>(gB[u], p.dTO.head(b, h) + qrow * p.dTO.sl, g, p.D, qvalid);
                if constexpr (!SECOND) load_b_operands16<T, HD, IO, true>(toR[u], p.to.head(b, h) + qrow * p.to.sl, g, p.D, qvalid);
            }
            if constexpr (HAS_DO) load_b_operands16<T, HD, IO, true>(doB[u], p.dO.head(b, h) + qrow * p.dO.sl, g, p.D, qvalid);
        }
    }
#pragma unroll
    for (int u = 0; u < NC; ++u) {  // requested with the rows: they are awaited together
        lse_in[u] = p.lse[so + 16 * u];
        mu_in[u] = HAS_G ? p.mu[so + 16 * u] : 0.f;
    }

    using StagePlan = std::conditional_t<DMA, CopyPlan<HD, SM::nt, 1, kXThreads16>,
                                         StagedPlan<T, HD, SM::nt, kXThreads16, IO>>;
    constexpr int SPT = StagePlan::N;
    StagePlan plan[DMA ? 1 : SPLIT];
#pragma unroll
    for (int u = 0; u < (DMA ? 1 : SPLIT); ++u) {
        if constexpr (HAS_G)
            init_plan(plan[u], tid, p.D, smem_raw + SM::sink, Src{p.k.head(b, h), p.k.sl}, Src{p.v.head(b, h), p.v.sl},
                      Src{p.tk.head(b, h), p.tk.sl}, Src{p.tv.head(b, h), p.tv.sl});
        else
            init_plan(plan[u], tid, p.D, smem_raw + SM::sink, Src{p.k.head(b, h), p.k.sl}, Src{p.v.head(b, h), p.v.sl});
        if constexpr (!DMA && SPLIT > 1) plan[u].take(u, SPLIT);
    }
    const int ns = (p.Lk + kStageRows - 1) / kStageRows;
    int issued = 0;
    auto issue_next = [&](int u = 0) {  // u: place of the stage in its step
        issue_plan(plan[DMA ? 0 : u], ring + (issued % R) * SM::slot, p.Lk - issued * kStageRows,
                   p.D == HD && (issued + 1) * kStageRows <= p.Lk);
        ++issued;
    };
    auto issue_step = [&]() {
#pragma unroll
        for (int u = 0; u < SPLIT; ++u)
            if (SPLIT == 1 || issued < ns) issue_next(u);
    };
    auto commit_step = [&]() {
        if constexpr (!DMA) {
#pragma unroll
            for (int u = 0; u < SPLIT; ++u) plan[u].commit();
        }
    };
    // The first step (stage 0) only for now: the loads of the own rows are awaited by a wait for everything this wave has
    // outstanding (the compiler cannot tell them from the stage copies), so the later stages are issued once
    // the own rows are in registers and land under the first stage's arithmetic.
    issue_step();
    if constexpr (IO == kIoAny) {
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const bool qvalid = wrow + 16 * u + n < p.Lq;
            finish_b_operands16<HD, IO>(qB[u], g, p.D, qvalid);
            if constexpr (!SECOND) finish_b_operands16<HD, IO>(oR[u], g, p.D, qvalid);
            if constexpr (HAS_G) {
                finish_b_operands16<HD, IO>(tqB[u], g, p.D, qvalid);
                finish_b_operands16<HD, IO>(gB[u], g, p.D, qvalid);
                if constexpr (!SECOND) finish_b_operands16<HD, IO>(toR[u], g, p.D, qvalid);
            }
            if constexpr (HAS_DO) finish_b_operands16<HD, IO>(doB[u], g, p.D, qvalid);
        }
    }
    // The own rows as whole pieces, behind the copies: used by their elements alone (the row sums below), a piece is joined
    // element by element where the two paths above meet, and an element that changes its register there is awaited in front
    // of the copies (D = 128, 1476 queries on 10 keys, cotangent on TO: 372 us against 331).
    if constexpr (!SECOND) {
        auto arrived = [](u32x4& piece) __attribute__((always_inline)) { asm volatile("" : "+v"(piece)); };
#pragma unroll
        for (int u = 0; u < NC; ++u)
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                arrived(qB[u][c]);
                arrived(oR[u][c]);
                if constexpr (HAS_G) {
                    arrived(tqB[u][c]);
                    arrived(gB[u][c]);
                    arrived(toR[u][c]);
                }
                if constexpr (HAS_DO) arrived(doB[u][c]);
            }
    }

    // row sums s4 = rowsum(G*O), s7d = rowsum(G*TO) + rowsum(dO*O) from the lane's 16-byte pieces, combined
    // over the four lanes of a query.  The tiles W and XY are accumulated on top of -s4 and -s7d, so that W - s4 and
    // XY - s7d leave the matrix cores ready for use.
    float n4[NC], n7[NC], lse2[NC], mu[NC];
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        if constexpr (SECOND) {
            // the corrected sums the first launch left in the workspace (negated there)
            n4[u] = p.s4[so + 16 * u];
            n7[u] = p.s7d[so + 16 * u];
        } else {
            float s4 = 0.f, s7d = 0.f;
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                if constexpr (HAS_G) {
                    s4 += dot8<T>(gB[u][c], oR[u][c]);
                    s7d += dot8<T>(gB[u][c], toR[u][c]);
                }
                if constexpr (HAS_DO) s7d += dot8<T>(doB[u][c], oR[u][c]);
            }
            n4[u] = -group_sum(s4);
            n7[u] = -group_sum(s7d);
        }
        asm volatile("" : "+v"(lse_in[u]), "+v"(mu_in[u]));  // not before the copies of stage 0 are under way
        lse2[u] = lse_in[u] * kLog2e;
        mu[u] = HAS_G ? mu_in[u] : 0.f;
        asm volatile("" : "+v"(lse2[u]), "+v"(mu[u]), "+v"(n4[u]), "+v"(n7[u]));  // every load so far is awaited here
    }
    if constexpr (DMA) {
        while (issued < R && issued < ns) issue_next();
    } else {
        commit_step();
    }
    // every row below Lr gets its workspace entries (zeros beyond Lq except lse2, which is finite): the
    // column-owned kernel, which runs after this one, stages 32-row groups
    if constexpr (!SECOND) {
#pragma unroll
        for (int u = 0; u < NC; ++u)
            if (g == 0 && part == 0) p.lse2[so + 16 * u] = lse2[u];
    }
    const float sl2 = p.scale * kLog2e;
    f32x4 dq[NC][DT], dtq[NC][DT];
#pragma unroll
    for (int u = 0; u < NC; ++u)
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            dq[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            dtq[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    // First launch: this lane's part of sum_j dS_dot_ij, sum_j dS_ij (zero in exact arithmetic), and of
    // their absolute sums, which only set the scale of a threshold and are sampled on every fourth key.
    float r4[NC] = {}, r7[NC] = {}, a4[NC] = {}, a7[NC] = {};

    auto compute = [&](const elem_t* slot, int k0, auto ragged_tag) {
        const elem_t* sK = slot;
        const elem_t* sV = slot + SE;
        const elem_t* sTK = slot + 2 * SE;
        const elem_t* sTV = slot + 3 * SE;
        // tiles: rows = keys (registers), columns = this wave's queries (lanes)
        f32x4 s[NC][2], ts[NC][2], w[NC][2], xy[NC][2];
        auto scores = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                s[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                ts[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                w[u][t] = f32x4{n4[u], n4[u], n4[u], n4[u]};
                xy[u][t] = f32x4{n7[u], n7[u], n7[u], n7[u]};
            }
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const u32x4 ak = lds_a_rows16<HD>(sK, t, c, n, g);
                const u32x4 av = lds_a_rows16<HD>(sV, t, c, n, g);
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    s[u][t] = T::mfma16(ak, qB[u][c], s[u][t]);
                    if constexpr (HAS_G) ts[u][t] = T::mfma16(ak, tqB[u][c], ts[u][t]);
                }
                if constexpr (HAS_G) {
                    const u32x4 atk = lds_a_rows16<HD>(sTK, t, c, n, g);
#pragma unroll
                    for (int u = 0; u < NC; ++u) {
                        ts[u][t] = T::mfma16(atk, qB[u][c], ts[u][t]);
                        w[u][t] = T::mfma16(av, gB[u][c], w[u][t]);
                    }
                    const u32x4 atv = lds_a_rows16<HD>(sTV, t, c, n, g);
#pragma unroll
                    for (int u = 0; u < NC; ++u) xy[u][t] = T::mfma16(atv, gB[u][c], xy[u][t]);
                }
                if constexpr (HAS_DO) {
#pragma unroll
                    for (int u = 0; u < NC; ++u) xy[u][t] = T::mfma16(av, doB[u][c], xy[u][t]);
                }
            }
        };
        constexpr bool ragged = decltype(ragged_tag)::value;  // the stage reaches beyond Lk (only the last one can)
        // in place: w -> dS_dot, xy -> dS
        auto pointwise = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < NC; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    float pj = fast_exp2(fmaf(s[u][t][j], sl2, -lse2[u]));
                    // keys beyond Lk are zero rows; exp(-lse) may overflow when every real score is very
                    // negative, so their P is forced to zero
                    if constexpr (ragged) {
                        if (k0 + 16 * t + 4 * g + j >= p.Lk) pj = 0.f;
                    }
                    if constexpr (HAS_G) {
                        const float nn = fmaf(ts[u][t][j], p.scale, -mu[u]);
                        const float dts = pj * w[u][t][j];
                        w[u][t][j] = dts;
                        xy[u][t][j] = fmaf(dts, nn, pj * xy[u][t][j]);
                        if constexpr (!SECOND) {
                            r4[u] += dts;
                            if (j == 0) a4[u] += fabsf(dts);
                        }
                    } else {
                        xy[u][t][j] = pj * xy[u][t][j];
                    }
                    if constexpr (!SECOND) {
                        r7[u] += xy[u][t][j];
                        if (j == 0) a7[u] += fabsf(xy[u][t][j]);
                    }
                }
        };
        // the second key tile's MFMA chains run under the first tile's element-wise arithmetic
        scores(0);
        __builtin_amdgcn_sched_barrier(0);
        scores(1);
        pointwise(0);
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (MEASURE) {  // a launch that only measures the residues
            pointwise(1);
            return;
        }
        // the transposed operands of the output contractions are read one step ahead, the first ones
        // under the second tile's element-wise arithmetic
        u32x4 ak = lds_a_tr16<HD>(sK, 0, lane), atk;
        if constexpr (HAS_G) atk = lds_a_tr16<HD>(sTK, 0, lane);
        __builtin_amdgcn_sched_barrier(0);
        pointwise(1);
        u32x4 dsB[NC], dtsB[NC];
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            dsB[u] = pack_b16<T>(xy[u][0], xy[u][1]);
            if constexpr (HAS_G) dtsB[u] = pack_b16<T>(w[u][0], w[u][1]);
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            u32x4 nk, ntk;
            if (d + 1 < DT) {
                nk = lds_a_tr16<HD>(sK, 16 * (d + 1), lane);
                if constexpr (HAS_G) ntk = lds_a_tr16<HD>(sTK, 16 * (d + 1), lane);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                dq[u][d] = T::mfma16(ak, dsB[u], dq[u][d]);
                if constexpr (HAS_G) {
                    dtq[u][d] = T::mfma16(ak, dtsB[u], dtq[u][d]);
                    dq[u][d] = T::mfma16(atk, dtsB[u], dq[u][d]);
                }
            }
            __builtin_amdgcn_sched_barrier(0);
            ak = nk;
            if constexpr (HAS_G) atk = ntk;
        }
    };

    // The last stage, the only one that can reach beyond Lk, runs behind the loop in a form of its own: the
    // selects of its padded keys (a compare and two selects per tile element) stay out of the loop.
    auto stage = [&](int i, auto ragged_tag) {
        // copies issued after stage i: the later stages; anything else in flight (the own rows'
        // loads, the statistics) only makes the wait stricter
        if constexpr (DMA) wait_stages<SPT>(issued - 1 - i);
        workgroup_barrier();  // stage i has landed for every wave; stage i-1 is fully consumed
        if ((i > 0 || !DMA) && issued < ns) issue_next();
        if (wave_active) compute(ring + (i % R) * SM::slot, i * kStageRows, ragged_tag);
        commit_step();
    };
    if constexpr (SPLIT > 1) {
        const elem_t* part_ring = ring + part * SM::slot;
        for (int i = 0; i < ns; i += SPLIT) {
            if constexpr (DMA) wait_stages<SPT>(issued - SPLIT - i > 0 ? issued - SPLIT - i : 0);
            workgroup_barrier();  // as above, of a step
            if (i > 0 || !DMA) issue_step();
            const int mine = i + part;
            if (wave_active && mine < ns) {
                const elem_t* slot = part_ring + (i % R) * SM::slot;
                if (mine == ns - 1) compute(slot, mine * kStageRows, std::true_type{});
                else compute(slot, mine * kStageRows, std::false_type{});
            }
            commit_step();
        }
    } else {
        for (int i = 0; i < ns - 1; ++i) stage(i, std::false_type{});
        stage(ns - 1, std::true_type{});
    }
    if constexpr (!SECOND) {
        // the residues of the row sums (see the top of the file); the four lanes of a query hold its keys
        bool wanted = false;
        int own = n;
        asm volatile("" : "+v"(own));  // (formed anew: nothing of the address is held through the loop)
        const int64_t so = (int64_t)bh * p.Lr + wrow + own;
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            r4[u] = group_sum(r4[u]);
            r7[u] = group_sum(r7[u]);
            a4[u] = group_sum(a4[u]);
            a7[u] = group_sum(a7[u]);
            if constexpr (SPLIT > 1) {
                using SP = Split16Smem<HD, kXWaves16, HAS_G ? 2 : 1>;
                float* stat = reinterpret_cast<float*>(smem_raw + SP::red);
                workgroup_barrier();  // the ring has been read
                float* mine = stat + wave * 64 + n;
                if (g == 0) {
                    mine[0] = r4[u];
                    mine[16] = r7[u];
                    mine[32] = a4[u];
                    mine[48] = a7[u];
                }
                workgroup_barrier();
                const float* all = stat + SPLIT * group * 64 + n;
                r4[u] = r7[u] = a4[u] = a7[u] = 0.f;
#pragma unroll
                for (int s = 0; s < SPLIT; ++s) {
                    r4[u] += all[64 * s];
                    r7[u] += all[64 * s + 16];
                    a4[u] += all[64 * s + 32];
                    a7[u] += all[64 * s + 48];
                }
            }
            a4[u] *= 4.0f;
            a7[u] *= 4.0f;
            if (g == 0 && part == 0) {
                p.s4[so + 16 * u] = n4[u] - r4[u];  // minus the corrected sums: the column-owned kernel starts its tiles from them
                p.s7d[so + 16 * u] = n7[u] - r7[u];
            }
            // A residue matters where it is not small against the rounding of the tiles it is spread over:
            // |rho| against tau * sum_j |tile_ij|, tau = the unit roundoff of the 16-bit format.  NaN compares false.
            wanted = wanted || (wrow + 16 * u + n < p.Lq && (fabsf(r4[u]) > p.rowfix_tau * a4[u] || fabsf(r7[u]) > p.rowfix_tau * a7[u]));
        }
        if (p.rowfix == 1) {
            // one flag per 64 rows, which is what a workgroup of the second launch owns; the workgroups that share them
            // write a byte or two each
#pragma unroll
            for (int f = 0; f < NC; ++f) {
                const bool any = workgroup_barrier_or(wanted && wave / (kXWaves16 / NC) == f);
                if (tid != 0) continue;
                if constexpr (SPLIT == 1) p.flags[NC * bid + f] = any ? 1 : 0;
                else if constexpr (SPLIT == 2) reinterpret_cast<uint16_t*>(p.flags)[bid] = any ? 1 : 0;
                else reinterpret_cast<uint8_t*>(p.flags)[bid] = any ? 1 : 0;
            }
        }
        if constexpr (MEASURE) return;  // the second launch writes dQ, dQ_dot
    }
    if constexpr (SPLIT > 1) {
        static_assert(SPLIT <= 4, "flags are bytes of 16 rows");
        using SP = Split16Smem<HD, kXWaves16, HAS_G ? 2 : 1>;
        f32x4* red = reinterpret_cast<f32x4*>(smem_raw);
        elem_t* tile = reinterpret_cast<elem_t*>(smem_raw + SP::red + SP::stat) + wave * StoreStage16<HD>::elems;
        split_put<DT, kXWaves16>(red, 0, wave, lane, dq[0]);  // (the ring was given up in front of the residues)
        if constexpr (HAS_G) split_put<DT, kXWaves16>(red, 1, wave, lane, dtq[0]);
        workgroup_barrier();
        if (!wave_active) return;
        if (part == 0) {
            split_sum<DT, kXWaves16, SPLIT>(dq[0], red, 0, group, lane);
            store_rows16<T, HD, IO, false, DT>(tile, p.dq.head(b, h), p.dq.sl, wrow, p.Lq, p.D, dq[0], p.scale, lane);
        }
        if constexpr (HAS_G) {
            if (part == 1) {
                split_sum<DT, kXWaves16, SPLIT>(dq[0], red, 1, group, lane);
                store_rows16<T, HD, IO, false, DT>(tile, p.dtq.head(b, h), p.dtq.sl, wrow, p.Lq, p.D, dq[0], p.scale, lane);
            }
        }
        return;
    }
    workgroup_barrier();  // every wave is done reading the ring: it becomes the store staging area
    if (!wave_active) return;
    elem_t* stage_tile = ring + wave * StoreStage16<HD>::elems;
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int row0 = wrow + 16 * u;
        store_rows16<T, HD, IO, false, DT>(stage_tile, p.dq.head(b, h), p.dq.sl, row0, p.Lq, p.D, dq[u], p.scale, lane);
        if constexpr (HAS_G)
            store_rows16<T, HD, IO, false, DT>(stage_tile, p.dtq.head(b, h), p.dtq.sl, row0, p.Lq, p.D, dtq[u], p.scale, lane);
    }
}

template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int OCC, int PASS = 0, int IO = kIoDma, int NC = 1,
          int SPLIT = 1, int DT = HD / 16>
__global__ __launch_bounds__(kXThreads16, OCC) void bwd_row16_kernel(const BwdParams p) {
    bwd_row16_body<T, HD, R, HAS_DO, HAS_G, PASS, IO, NC, SPLIT, DT>(p, (int)blockIdx.x, (int)gridDim.x);
}

// ---------------------------------------------------------------------------------------------
// Column-owned kernel: a workgroup of four waves owns 64 keys and accumulates all their gradients (HD <= 64; the
// paired form below serves HD = 128).  LDS: [ring of Q | [Q_dot | G] | [dO] | lse2, mu, s4, s7d stages]
// [sink]; the ring doubles as store staging after the last stage.
template <int HD, int R, bool HAS_DO, bool HAS_G, int SPLIT = 1>
struct Col16Smem {
    static constexpr int nt = 1 + (HAS_G ? 2 : 0) + (HAS_DO ? 1 : 0);
    static constexpr int stat_elems = 4 * kStageRows * 2;  // 4 float arrays of 32, in elem_t units
    static constexpr int slot = nt * Slab<HD>::elems + stat_elems;
    static constexpr int loop = R * slot * (int)sizeof(elem_t);
    static constexpr int after = SPLIT > 1 ? Split16Smem<HD, kXWaves16, HAS_G ? 4 : 2>::bytes : 0;
    static constexpr int sink = loop > after ? loop : after;
    static constexpr int bytes = sink + kSink16;
    static_assert(R * slot >= kXWaves16 * StoreStage16<HD>::elems, "ring too small to stage stores");
};

// (SPLIT: as in the row-owned kernel)
template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int IO, int NC = 1, int SPLIT = 1,
          int DT = HD / 16>
__device__ __forceinline__ void bwd_col16_body(const BwdParams p, const int block, const int blocks) {
    constexpr bool DMA = IO == kIoDma;
    extern __shared__ __align__(16) unsigned char smem_raw[];
    using SM = Col16Smem<HD, R, HAS_DO, HAS_G, SPLIT>;
    elem_t* ring = reinterpret_cast<elem_t*>(smem_raw);
    constexpr int SE = Slab<HD>::elems;
    constexpr int oTQ = SE, oG = 2 * SE, oDO = (HAS_G ? 3 : 1) * SE, oST = SM::nt * SE;
    constexpr int KL = HD / 32, KC = (DT + 1) / 2;  // 32-column chunks of a row, and those with columns below D
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;
    const int g = lane >> 4;
    static_assert(SPLIT == 1 || (NC == 1 && R == 2 * SPLIT), "a step is a stage for every part");
    const int part = SPLIT > 1 ? wave % SPLIT : 0, group = wave / SPLIT;
    constexpr int OWNED = NC * kXOwned16 / SPLIT;
    const int k_blocks = (p.Lk + OWNED - 1) / OWNED;
    const int bid = xcd_linear_id(block, blocks);
    const int bh = bid / k_blocks;
    const int kb = bid % k_blocks;
    const int b = bh / p.H, h = bh % p.H;
    const int key0 = kb * OWNED;
    const int wrow = key0 + group * 16 * NC;  // the wave's first key; the lane's are wrow + 16 u + n
    const bool wave_active = wrow < p.Lk;

    using StagePlan = std::conditional_t<DMA, CopyPlan<HD, SM::nt, 1, kXThreads16>,
                                         StagedPlan<T, HD, SM::nt, kXThreads16, IO>>;
    constexpr int SPT = StagePlan::N + 1;  // plus one 4-byte copy of statistics
    StagePlan plan[DMA ? 1 : SPLIT];
    const int ns = (p.Lq + kStageRows - 1) / kStageRows;
    int issued = 0;
    auto issue_next = [&](int u = 0) {  // u: place of the stage in its step
        elem_t* slot = ring + (issued % R) * SM::slot;
        const int row0 = issued * kStageRows;
        issue_plan(plan[DMA ? 0 : u], slot, p.Lq - row0, p.D == HD && row0 + kStageRows <= p.Lq);
        // the four statistic arrays (lse2, mu, s4, s7d) of the stage's rows, one per wave, 32 lanes
        // each (rows < Lr exist in all of them); every wave issues exactly one 4-byte LDS-DMA
        // (the three workspace arrays lie one behind the other: chosen by arithmetic, which stays in scalar
        // registers, where a choice among four pointers becomes a table in memory)
        const int64_t plane = p.s4 - p.lse2;
        const float* src = p.lse2 + (wave == 0 ? 0 : wave == 3 ? 2 : 1) * plane;  // lse2 | s4 | s4 | s7d
        if (HAS_G && wave == 1) src = p.mu;
        float* st = reinterpret_cast<float*>(slot + oST);
        if (lane < 32) dma4(src + (int64_t)bh * p.Lr + row0 + lane, lds_addr(st) + (uint32_t)(wave * 32 * 4));
        ++issued;
    };
    auto issue_step = [&]() {
#pragma unroll
        for (int u = 0; u < SPLIT; ++u)
            if (SPLIT == 1 || issued < ns) issue_next(u);
    };
    auto commit_step = [&]() {
        if constexpr (!DMA) {
#pragma unroll
            for (int u = 0; u < SPLIT; ++u) plan[u].commit();
        }
    };
    // called behind the requests for the own rows on both paths below (see bwd_row16_kernel): set-up of the
    // stage copies, and the first step (stage 0) only for now
    auto begin_copies = [&]() __attribute__((always_inline)) {
        const Src q{p.q.head(b, h), p.q.sl};
#pragma unroll
        for (int u = 0; u < (DMA ? 1 : SPLIT); ++u) {
            if constexpr (HAS_G && HAS_DO)
                init_plan(plan[u], tid, p.D, smem_raw + SM::sink, q, Src{p.tq.head(b, h), p.tq.sl},
                          Src{p.dTO.head(b, h), p.dTO.sl}, Src{p.dO.head(b, h), p.dO.sl});
            else if constexpr (HAS_G)
                init_plan(plan[u], tid, p.D, smem_raw + SM::sink, q, Src{p.tq.head(b, h), p.tq.sl},
                          Src{p.dTO.head(b, h), p.dTO.sl});
            else
                init_plan(plan[u], tid, p.D, smem_raw + SM::sink, q, Src{p.dO.head(b, h), p.dO.sl});
            if constexpr (!DMA && SPLIT > 1) plan[u].take(u, SPLIT);
        }
        issue_step();
    };
    // the own rows are requested first; the set-up of the stage copies runs while they travel
    u32x4 kB[NC][KL], vB[NC][KL], tkB[NC][KL], tvB[NC][KL];
    if (DMA && p.k_side_uniform && p.D == HD && key0 + OWNED <= p.Lk) {
        // the common case: whole rows that all exist, every tensor with k's strides
        const int64_t slice = b * p.k.sb + h * p.k.sh;
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const uint32_t at = ((uint32_t)(wrow + 16 * u + n) * (uint32_t)p.k.sl + 8u * (uint32_t)g) * (uint32_t)sizeof(elem_t);
            load_b_operands16_at<HD>(kB[u], p.k.ptr + slice, at);
            load_b_operands16_at<HD>(vB[u], p.v.ptr + slice, at);
            if constexpr (HAS_G) {
                load_b_operands16_at<HD>(tkB[u], p.tk.ptr + slice, at);
                load_b_operands16_at<HD>(tvB[u], p.tv.ptr + slice, at);
            }
        }
        begin_copies();
    } else {
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const bool kvalid = wrow + 16 * u + n < p.Lk;
            const int64_t krow = IO == kIoAny ? own_row(wrow + 16 * u + n, p.Lk) : wrow + 16 * u + n;
            load_b_operands16<T, HD, IO>(kB[u], p.k.head(b, h) + krow * p.k.sl, g, p.D, kvalid);
            load_b_operands16<T, HD, IO>(vB[u], p.v.head(b, h) + krow * p.v.sl, g, p.D, kvalid);
            if constexpr (HAS_G) {
                load_b_operands16<T, HD, IO>(tkB[u], p.tk.head(b, h) + krow * p.tk.sl, g, p.D, kvalid);
                load_b_operands16<T, HD, IO>(tvB[u], p.tv.head(b, h) + krow * p.tv.sl, g, p.D, kvalid);
            }
        }
        begin_copies();
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const bool kvalid = wrow + 16 * u + n < p.Lk;
            finish_b_operands16<HD, IO>(kB[u], g, p.D, kvalid);
            finish_b_operands16<HD, IO>(vB[u], g, p.D, kvalid);
            if constexpr (HAS_G) {
                finish_b_operands16<HD, IO>(tkB[u], g, p.D, kvalid);
                finish_b_operands16<HD, IO>(tvB[u], g, p.D, kvalid);
            }
        }
    }
#pragma unroll
    for (int u = 0; u < NC; ++u)
#pragma unroll
        for (int c = 0; c < KC; ++c) {  // the own rows are awaited here
            asm volatile("" : "+v"(kB[u][c]));
            asm volatile("" : "+v"(vB[u][c]));
            if constexpr (HAS_G) {
                asm volatile("" : "+v"(tkB[u][c]));
                asm volatile("" : "+v"(tvB[u][c]));
            }
        }
    if constexpr (DMA) {
        while (issued < R && issued < ns) issue_next();
    } else {
        commit_step();
    }
    const float sl2 = p.scale * kLog2e;
    f32x4 dk[NC][DT], dv[NC][DT], dtk[NC][DT], dtv[NC][DT];
#pragma unroll
    for (int u = 0; u < NC; ++u)
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            dk[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            dv[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            dtk[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            dtv[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }

    auto compute = [&](const elem_t* slot) {
        const elem_t* sQ = slot;
        const elem_t* sTQ = slot + oTQ;
        const elem_t* sG = slot + oG;
        const elem_t* sDO = slot + oDO;
        const float* sStat = reinterpret_cast<const float*>(slot + oST);
        // tiles: rows = queries (registers), columns = this wave's keys (lanes).
        // The A operands of every contraction step are read from LDS one step ahead of the MFMAs
        // that use them (two register sets), so that a wave's matrix pipe does not sit out an LDS
        // round trip per step; the first operands of the gradient phase and the row statistics are
        // requested before the last score step and arrive during the element-wise work.
        struct AOps {
            u32x4 q, tq, g, d;
        };
        auto load_score = [&](int t, int c) {
            AOps a;
            a.q = lds_a_rows16<HD>(sQ, t, c, n, g);
            if constexpr (HAS_G) {
                a.tq = lds_a_rows16<HD>(sTQ, t, c, n, g);
                a.g = lds_a_rows16<HD>(sG, t, c, n, g);
            }
            if constexpr (HAS_DO) a.d = lds_a_rows16<HD>(sDO, t, c, n, g);
            return a;
        };
        auto load_grad = [&](int d) {
            AOps a;
            a.q = lds_a_tr16<HD>(sQ, 16 * d, lane);
            if constexpr (HAS_G) a.tq = lds_a_tr16<HD>(sTQ, 16 * d, lane);
            if constexpr (HAS_G) a.g = lds_a_tr16<HD>(sG, 16 * d, lane);
            if constexpr (HAS_DO) a.d = lds_a_tr16<HD>(sDO, 16 * d, lane);
            return a;
        };
        f32x4 s[NC][2], ts[NC][2], w[NC][2], xy[NC][2];
        f32x4 lse4[2], mu4[2];
#pragma unroll
        for (int u = 0; u < NC; ++u)
#pragma unroll
            for (int t = 0; t < 2; ++t) {
                s[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                ts[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
        // The workspace holds -s4 and -s7d: W and XY are accumulated on top of them, so that W - s4 and
        // XY - s7d leave the matrix cores ready for use.
        auto load_sums = [&](int t) __attribute__((always_inline)) {
            const int r0 = 16 * t + 4 * g;  // register j of tile t is query 16 t + 4 g + j
            if constexpr (HAS_G) w[0][t] = *reinterpret_cast<const f32x4*>(sStat + 2 * kStageRows + r0);
            xy[0][t] = *reinterpret_cast<const f32x4*>(sStat + 3 * kStageRows + r0);
#pragma unroll
            for (int u = 1; u < NC; ++u) {
                if constexpr (HAS_G) w[u][t] = w[0][t];
                xy[u][t] = xy[0][t];
            }
        };
        auto load_stats = [&](int t) __attribute__((always_inline)) {
            const int r0 = 16 * t + 4 * g;
            lse4[t] = *reinterpret_cast<const f32x4*>(sStat + 0 * kStageRows + r0);
            if constexpr (HAS_G) mu4[t] = *reinterpret_cast<const f32x4*>(sStat + 1 * kStageRows + r0);
        };
        auto score_step = [&](int t, int c, const AOps& a) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                s[u][t] = T::mfma16(a.q, kB[u][c], s[u][t]);
                if constexpr (HAS_G) {
                    ts[u][t] = T::mfma16(a.q, tkB[u][c], ts[u][t]);
                    ts[u][t] = T::mfma16(a.tq, kB[u][c], ts[u][t]);
                    w[u][t] = T::mfma16(a.g, vB[u][c], w[u][t]);
                    xy[u][t] = T::mfma16(a.g, tvB[u][c], xy[u][t]);
                }
                if constexpr (HAS_DO) xy[u][t] = T::mfma16(a.d, vB[u][c], xy[u][t]);
            }
        };
        // in place: s -> P, ts -> P_dot, w -> dS_dot, xy -> dS  (rows beyond Lq are zero rows of Q,
        // Q_dot, G, dO with finite statistics: they contribute nothing)
        auto pointwise = [&](int t) __attribute__((always_inline)) {
#pragma unroll
            for (int u = 0; u < NC; ++u)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float pj = fast_exp2(fmaf(s[u][t][j], sl2, -lse4[t][j]));
                    s[u][t][j] = pj;
                    if constexpr (HAS_G) {
                        const float nn = fmaf(ts[u][t][j], p.scale, -mu4[t][j]);
                        const float dts = pj * w[u][t][j];
                        w[u][t][j] = dts;
                        xy[u][t][j] = fmaf(dts, nn, pj * xy[u][t][j]);
                        ts[u][t][j] = pj * nn;
                    } else {
                        xy[u][t][j] = pj * xy[u][t][j];
                    }
                }
        };
        load_sums(0);
        AOps cur = load_score(0, 0);
        load_stats(0);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            AOps nxt;
            if (c + 1 < KC) {
                nxt = load_score(0, c + 1);
            } else {
                load_sums(1);
                nxt = load_score(1, 0);
            }
            __builtin_amdgcn_sched_barrier(0);  // keep the reads ahead of this step's MFMAs
            score_step(0, c, cur);
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
        // the second tile's MFMA chains run under the first tile's element-wise arithmetic
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            AOps nxt;
            if (c + 1 < KC) {
                nxt = load_score(1, c + 1);
            } else {
                load_stats(1);
                nxt = load_grad(0);
            }
            score_step(1, c, cur);
            cur = nxt;
        }
        pointwise(0);
        __builtin_amdgcn_sched_barrier(0);
        pointwise(1);
        u32x4 pB[NC], dsB[NC], pdB[NC], dtsB[NC];
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            pB[u] = pack_b16<T>(s[u][0], s[u][1]);
            dsB[u] = pack_b16<T>(xy[u][0], xy[u][1]);
            if constexpr (HAS_G) {
                pdB[u] = pack_b16<T>(ts[u][0], ts[u][1]);
                dtsB[u] = pack_b16<T>(w[u][0], w[u][1]);
            }
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            AOps nxt;
            if (d + 1 < DT) nxt = load_grad(d + 1);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                dk[u][d] = T::mfma16(cur.q, dsB[u], dk[u][d]);
                if constexpr (HAS_G) {
                    dtk[u][d] = T::mfma16(cur.q, dtsB[u], dtk[u][d]);
                    dk[u][d] = T::mfma16(cur.tq, dtsB[u], dk[u][d]);
                    dtv[u][d] = T::mfma16(cur.g, pB[u], dtv[u][d]);
                    dv[u][d] = T::mfma16(cur.g, pdB[u], dv[u][d]);
                }
                if constexpr (HAS_DO) dv[u][d] = T::mfma16(cur.d, pB[u], dv[u][d]);
            }
            __builtin_amdgcn_sched_barrier(0);
            cur = nxt;
        }
    };

    if constexpr (SPLIT > 1) {
        const elem_t* part_ring = ring + part * SM::slot;
        for (int i = 0; i < ns; i += SPLIT) {
            wait_stages<SPT>(DMA && issued - SPLIT - i > 0 ? issued - SPLIT - i : 0);
            workgroup_barrier();  // as below, of a step
            if (i > 0 || !DMA) issue_step();
            if (wave_active && i + part < ns) compute(part_ring + (i % R) * SM::slot);
            commit_step();
        }
        using SP = Split16Smem<HD, kXWaves16, HAS_G ? 4 : 2>;
        f32x4* red = reinterpret_cast<f32x4*>(smem_raw);
        elem_t* tile = reinterpret_cast<elem_t*>(smem_raw + SP::red + SP::stat) + wave * StoreStage16<HD>::elems;
        workgroup_barrier();  // every wave is done reading the ring
        split_put<DT, kXWaves16>(red, 0, wave, lane, dk[0]);
        split_put<DT, kXWaves16>(red, 1, wave, lane, dv[0]);
        if constexpr (HAS_G) {
            split_put<DT, kXWaves16>(red, 2, wave, lane, dtk[0]);
            split_put<DT, kXWaves16>(red, 3, wave, lane, dtv[0]);
        }
        workgroup_barrier();
        if (!wave_active) return;
#pragma unroll
        for (int k = 0; k < (HAS_G ? 4 : 2); ++k) {
            if (k % SPLIT != part) continue;  // wave-uniform
            const OutView out = k == 0 ? p.dk : k == 1 ? p.dv : k == 2 ? p.dtk : p.dtv;
            split_sum<DT, kXWaves16, SPLIT>(dk[0], red, k, group, lane);
            store_rows16<T, HD, IO, false, DT>(tile, out.head(b, h), out.sl, wrow, p.Lk, p.D, dk[0], k % 2 == 0 ? p.scale : 1.0f, lane);
        }
        return;
    }
    for (int i = 0; i < ns; ++i) {
        wait_stages<SPT>(DMA ? issued - 1 - i : 0);  // staged: the statistics still come by LDS-DMA
        workgroup_barrier();  // stage i has landed for every wave; stage i-1 is fully consumed
        if ((i > 0 || !DMA) && issued < ns) issue_next();
        if (wave_active) compute(ring + (i % R) * SM::slot);
        commit_step();
    }
    workgroup_barrier();  // every wave is done reading the ring: it becomes the store staging area
    if (!wave_active) return;
    elem_t* stage_tile = ring + wave * StoreStage16<HD>::elems;
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int row0 = wrow + 16 * u;
        store_rows16<T, HD, IO, false, DT>(stage_tile, p.dk.head(b, h), p.dk.sl, row0, p.Lk, p.D, dk[u], p.scale, lane);
        if constexpr (HAS_G)
            store_rows16<T, HD, IO, false, DT>(stage_tile, p.dtk.head(b, h), p.dtk.sl, row0, p.Lk, p.D, dtk[u], p.scale, lane);
        store_rows16<T, HD, IO, false, DT>(stage_tile, p.dv.head(b, h), p.dv.sl, row0, p.Lk, p.D, dv[u], 1.0f, lane);
        if constexpr (HAS_G)
            store_rows16<T, HD, IO, false, DT>(stage_tile, p.dtv.head(b, h), p.dtv.sl, row0, p.Lk, p.D, dtv[u], 1.0f, lane);
    }
}

template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int OCC, int IO = kIoDma, int NC = 1, int SPLIT = 1,
          int DT = HD / 16>
__global__ __launch_bounds__(kXThreads16, OCC) void bwd_col16_kernel(const BwdParams p) {
    bwd_col16_body<T, HD, R, HAS_DO, HAS_G, IO, NC, SPLIT, DT>(p, (int)blockIdx.x, (int)gridDim.x);
}

// The column-owned launch with the second launch of the row-owned kernel at its end: workgroups
// 0 .. col_blocks - 1 are the column-owned kernel's, the rest the row-owned kernel's second pass, which does
// not depend on the column pass (it rewrites dQ, dQ_dot of flagged workgroups from the sums the first pass
// left).  Nearly all of those workgroups leave at once; dealt out behind the column pass they fill the time in
// which its last workgroups run alone, where a launch of their own costs a few microseconds.
template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int OCC, int IO = kIoDma, int NC = 1, int SPLIT = 1,
          int RROW = R, int DT = HD / 16>
__global__ __launch_bounds__(kXThreads16, OCC) void bwd_col16_repair_kernel(const BwdParams p) {
    const int col_blocks = p.col_workgroups;
    if ((int)blockIdx.x < col_blocks)
        bwd_col16_body<T, HD, R, HAS_DO, HAS_G, IO, NC, SPLIT, DT>(p, (int)blockIdx.x, col_blocks);
    else
        bwd_row16_body<T, HD, RROW, HAS_DO, HAS_G, 2, IO, 1, 1, DT>(p, (int)blockIdx.x - col_blocks, (int)gridDim.x - col_blocks);
}

// ---------------------------------------------------------------------------------------------
// Column-owned kernel for the head dimension 128: a workgroup of eight waves owns 64 keys; waves
// 2 r and 2 r + 1 share keys 16 r .. 16 r + 15.  Four gradients of 16 x 128 do not fit one wave's
// registers beside the operands, so the pair splits the work without repeating any of it: member m
// forms the score-side tiles (S, S_dot, W, XY -> P, P_dot, dS_dot, dS) of the stage's query tile m
// (16 queries), the two exchange their packed tiles through LDS, and member m accumulates all four
// gradients for head-dimension columns 64 m .. 64 m + 63 (D <= 96: 48 m .. 48 m + 47) over the stage's 32 queries.  One launch,
// 12 tile contractions (6 + 6), the query side streamed once.
// LDS: [ring of Q | [Q_dot | G] | [dO] | lse2, mu, s4, s7d stages][exchange: 8 waves x 4 tiles][sink];
// the ring doubles as store staging after the last stage.
template <int HD, int R, bool HAS_DO, bool HAS_G>
struct Col16pSmem {
    static constexpr int nt = 1 + (HAS_G ? 2 : 0) + (HAS_DO ? 1 : 0);
    static constexpr int stat_elems = 4 * kStageRows * 2;
    static constexpr int slot = nt * Slab<HD>::elems + stat_elems;
    static constexpr int xch = kWaves16 * 4 * 64 * 4;  // u32x2 per lane, tile and wave, in elem_t units
    static constexpr int sink = (R * slot + xch) * (int)sizeof(elem_t);
    static constexpr int bytes = sink + kSink16;
    static_assert(R * slot >= kWaves16 * StoreStage16<64>::elems, "ring too small to stage stores");
};

template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int IO, int DT = HD / 16>
__device__ __forceinline__ void bwd_col16p_body(const BwdParams p, const int block, const int blocks) {
    constexpr bool DMA = IO == kIoDma;
    static_assert(HD == 128, "the paired form exists for the head dimension that needs it");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    using SM = Col16pSmem<HD, R, HAS_DO, HAS_G>;
    elem_t* ring = reinterpret_cast<elem_t*>(smem_raw);
    u32x2* xch = reinterpret_cast<u32x2*>(ring + R * SM::slot);  // [wave][tile 0..3][lane]
    constexpr int SE = Slab<HD>::elems;
    constexpr int oTQ = SE, oG = 2 * SE, oDO = (HAS_G ? 3 : 1) * SE, oST = SM::nt * SE;
    constexpr int KL = HD / 32, KC = (DT + 1) / 2;
    constexpr int DH = DT / 2;  // 16-wide head-dimension tiles per member
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int pr = wave >> 1, m = wave & 1;  // pair, member
    const int n = lane & 15;
    const int g = lane >> 4;
    const int k_blocks = (p.Lk + kXOwned16 - 1) / kXOwned16;
    const int bid = xcd_linear_id(block, blocks);
    const int bh = bid / k_blocks;
    const int kb = bid % k_blocks;
    const int b = bh / p.H, h = bh % p.H;
    const int key0 = kb * kXOwned16;
    const int krow = key0 + pr * 16 + n;
    const bool kvalid = krow < p.Lk;
    const bool pair_active = (key0 + pr * 16) < p.Lk;

    using StagePlan = std::conditional_t<DMA, CopyPlan<HD, SM::nt, 1, kThreads16>,
                                         StagedPlan<T, HD, SM::nt, kThreads16, IO>>;
    constexpr int SPT = StagePlan::N + 1;  // plus one 4-byte copy of statistics (or its placeholder)
    StagePlan plan;
    const int ns = (p.Lq + kStageRows - 1) / kStageRows;
    int issued = 0;
    auto issue_next = [&]() {
        elem_t* slot = ring + (issued % R) * SM::slot;
        const int row0 = issued * kStageRows;
        issue_plan(plan, slot, p.Lq - row0, p.D == HD && row0 + kStageRows <= p.Lq);
        // the four statistic arrays of the stage's rows by waves 0..3; the others issue a placeholder
        if (wave < 4) {
            const int64_t plane = p.s4 - p.lse2;  // see bwd_col16_body
            const float* src = p.lse2 + (wave == 0 ? 0 : wave == 3 ? 2 : 1) * plane;  // lse2 | s4 | s4 | s7d
            if (HAS_G && wave == 1) src = p.mu;
            float* st = reinterpret_cast<float*>(slot + oST);
            if (lane < 32) dma4(src + (int64_t)bh * p.Lr + row0 + lane, lds_addr(st) + (uint32_t)(wave * 32 * 4));
        } else if constexpr (DMA) {
            if (lane == 0) dma4(plan.any, plan.sink);
        }
        ++issued;
    };
    // called behind the requests for the own rows on both paths below (see bwd_row16_kernel): set-up of the
    // stage copies, and stage 0 only for now
    auto begin_copies = [&]() __attribute__((always_inline)) {
        const Src q{p.q.head(b, h), p.q.sl};
        if constexpr (HAS_G && HAS_DO)
            init_plan(plan, tid, p.D, smem_raw + SM::sink, q, Src{p.tq.head(b, h), p.tq.sl},
                      Src{p.dTO.head(b, h), p.dTO.sl}, Src{p.dO.head(b, h), p.dO.sl});
        else if constexpr (HAS_G)
            init_plan(plan, tid, p.D, smem_raw + SM::sink, q, Src{p.tq.head(b, h), p.tq.sl},
                      Src{p.dTO.head(b, h), p.dTO.sl});
        else
            init_plan(plan, tid, p.D, smem_raw + SM::sink, q, Src{p.dO.head(b, h), p.dO.sl});
        issue_next();
    };
    // the own rows are requested first; the set-up of the stage copies runs while they travel
    u32x4 kB[KL], vB[KL], tkB[KL], tvB[KL];
    if (DMA && p.k_side_uniform && p.D == HD && key0 + kXOwned16 <= p.Lk) {
        // the common case: whole rows that all exist, every tensor with k's strides
        const int64_t slice = b * p.k.sb + h * p.k.sh;
        const uint32_t at = ((uint32_t)krow * (uint32_t)p.k.sl + 8u * (uint32_t)g) * (uint32_t)sizeof(elem_t);
        load_b_operands16_at<HD>(kB, p.k.ptr + slice, at);
        load_b_operands16_at<HD>(vB, p.v.ptr + slice, at);
        if constexpr (HAS_G) {
            load_b_operands16_at<HD>(tkB, p.tk.ptr + slice, at);
            load_b_operands16_at<HD>(tvB, p.tv.ptr + slice, at);
        }
        begin_copies();
    } else {
        const int64_t row = IO == kIoAny ? own_row(krow, p.Lk) : krow;
        load_b_operands16<T, HD, IO>(kB, p.k.head(b, h) + row * p.k.sl, g, p.D, kvalid);
        load_b_operands16<T, HD, IO>(vB, p.v.head(b, h) + row * p.v.sl, g, p.D, kvalid);
        if constexpr (HAS_G) {
            load_b_operands16<T, HD, IO>(tkB, p.tk.head(b, h) + row * p.tk.sl, g, p.D, kvalid);
            load_b_operands16<T, HD, IO>(tvB, p.tv.head(b, h) + row * p.tv.sl, g, p.D, kvalid);
        }
        begin_copies();
        finish_b_operands16<HD, IO>(kB, g, p.D, kvalid);
        finish_b_operands16<HD, IO>(vB, g, p.D, kvalid);
        if constexpr (HAS_G) {
            finish_b_operands16<HD, IO>(tkB, g, p.D, kvalid);
            finish_b_operands16<HD, IO>(tvB, g, p.D, kvalid);
        }
    }
#pragma unroll
    for (int c = 0; c < KC; ++c) {  // the own rows are awaited here
        asm volatile("" : "+v"(kB[c]), "+v"(vB[c]));
        if constexpr (HAS_G) asm volatile("" : "+v"(tkB[c]), "+v"(tvB[c]));
    }
    if constexpr (DMA) {
        while (issued < R && issued < ns) issue_next();
    } else {
        plan.commit();
    }
    const float sl2 = p.scale * kLog2e;
    f32x4 dk[DH], dv[DH], dtk[DH], dtv[DH];
#pragma unroll
    for (int t = 0; t < DH; ++t) {
        dk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        dv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        dtk[t] = f32x4{0.f, 0.f, 0.f, 0.f};
        dtv[t] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    // packed tiles of this member's query tile: P, P_dot, dS, dS_dot (register j = query 16 m + 4 g + j)
    u32x2 mine[4];
    u32x2* my_x = xch + (wave * 4) * 64 + lane;
    const u32x2* other_x = xch + ((wave ^ 1) * 4) * 64 + lane;

    auto scores = [&](const elem_t* slot) {
        const elem_t* sQ = slot;
        const elem_t* sTQ = slot + oTQ;
        const elem_t* sG = slot + oG;
        const elem_t* sDO = slot + oDO;
        const float* sStat = reinterpret_cast<const float*>(slot + oST);
        // the workspace holds -s4 and -s7d: W and XY are accumulated on top of them
        const int r0 = 16 * m + 4 * g;
        f32x4 s = {0.f, 0.f, 0.f, 0.f}, ts = {0.f, 0.f, 0.f, 0.f};
        f32x4 w = *reinterpret_cast<const f32x4*>(sStat + 2 * kStageRows + r0);
        f32x4 xy = *reinterpret_cast<const f32x4*>(sStat + 3 * kStageRows + r0);
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            const u32x4 aq = lds_a_rows16<HD>(sQ, m, c, n, g);
            s = T::mfma16(aq, kB[c], s);
            if constexpr (HAS_G) {
                ts = T::mfma16(aq, tkB[c], ts);
                const u32x4 atq = lds_a_rows16<HD>(sTQ, m, c, n, g);
                ts = T::mfma16(atq, kB[c], ts);
                const u32x4 ag = lds_a_rows16<HD>(sG, m, c, n, g);
                w = T::mfma16(ag, vB[c], w);
                xy = T::mfma16(ag, tvB[c], xy);
            }
            if constexpr (HAS_DO) {
                const u32x4 ado = lds_a_rows16<HD>(sDO, m, c, n, g);
                xy = T::mfma16(ado, vB[c], xy);
            }
        }
        // rows beyond Lq are zero rows of Q, Q_dot, G, dO with finite statistics: they contribute nothing
        const f32x4 lse4 = *reinterpret_cast<const f32x4*>(sStat + 0 * kStageRows + r0);
        const f32x4 mu4 = *reinterpret_cast<const f32x4*>(sStat + 1 * kStageRows + r0);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const float pj = fast_exp2(fmaf(s[j], sl2, -lse4[j]));
            s[j] = pj;
            if constexpr (HAS_G) {
                const float nn = fmaf(ts[j], p.scale, -mu4[j]);
                const float dts = pj * w[j];
                w[j] = dts;
                xy[j] = fmaf(dts, nn, pj * xy[j]);
                ts[j] = pj * nn;
            } else {
                xy[j] = pj * xy[j];
            }
        }
        mine[0] = u32x2{T::pack2(s[0], s[1]), T::pack2(s[2], s[3])};
        mine[2] = u32x2{T::pack2(xy[0], xy[1]), T::pack2(xy[2], xy[3])};
        my_x[0 * 64] = mine[0];
        my_x[2 * 64] = mine[2];
        if constexpr (HAS_G) {
            mine[1] = u32x2{T::pack2(ts[0], ts[1]), T::pack2(ts[2], ts[3])};
            mine[3] = u32x2{T::pack2(w[0], w[1]), T::pack2(w[2], w[3])};
            my_x[1 * 64] = mine[1];
            my_x[3 * 64] = mine[3];
        }
    };
    // B operand over the stage's 32 queries from the pair's two packed tiles (query tile 0 first)
    auto both = [&](int which) {
        const u32x2 o = other_x[which * 64];
        return m == 0 ? u32x4{mine[which][0], mine[which][1], o[0], o[1]}
                      : u32x4{o[0], o[1], mine[which][0], mine[which][1]};
    };
    auto outputs = [&](const elem_t* slot) {
        const elem_t* sQ = slot;
        const elem_t* sTQ = slot + oTQ;
        const elem_t* sG = slot + oG;
        const elem_t* sDO = slot + oDO;
        const u32x4 pB = both(0), dsB = both(2);
        u32x4 pdB, dtsB;
        if constexpr (HAS_G) {
            pdB = both(1);
            dtsB = both(3);
        }
#pragma unroll
        for (int d = 0; d < DH; ++d) {
            const int d0 = 16 * DH * m + 16 * d;
            const u32x4 aq = lds_a_tr16<HD>(sQ, d0, lane);
            dk[d] = T::mfma16(aq, dsB, dk[d]);
            if constexpr (HAS_G) {
                dtk[d] = T::mfma16(aq, dtsB, dtk[d]);
                const u32x4 atq = lds_a_tr16<HD>(sTQ, d0, lane);
                dk[d] = T::mfma16(atq, dtsB, dk[d]);
                const u32x4 ag = lds_a_tr16<HD>(sG, d0, lane);
                dtv[d] = T::mfma16(ag, pB, dtv[d]);
                dv[d] = T::mfma16(ag, pdB, dv[d]);
            }
            if constexpr (HAS_DO) {
                const u32x4 ado = lds_a_tr16<HD>(sDO, d0, lane);
                dv[d] = T::mfma16(ado, pB, dv[d]);
            }
        }
    };

    for (int i = 0; i < ns; ++i) {
        wait_stages<SPT>(DMA ? issued - 1 - i : 0);  // staged: the statistics still come by LDS-DMA
        workgroup_barrier();  // stage i has landed for every wave; stage i-1 and the exchange area are free
        if ((i > 0 || !DMA) && issued < ns) issue_next();
        const elem_t* slot = ring + (i % R) * SM::slot;
        if (pair_active) scores(slot);
        workgroup_barrier();  // the partner's tiles are visible
        if (pair_active) outputs(slot);
        if constexpr (!DMA) plan.commit();
    }
    workgroup_barrier();  // every wave is done reading the ring: it becomes the store staging area
    if (!pair_active) return;
    elem_t* stage_tile = ring + wave * StoreStage16<64>::elems;
    const int row0 = key0 + pr * 16;
    const int dcol = 16 * DH * m;
    const int doff = IO == kIoF32 ? 2 * dcol : dcol;  // in the units of the views
    const int Dm = min(p.D - dcol, 16 * DH);  // columns of this member's half that exist (may be <= 0)
    store_rows16<T, 64, IO, false, DH>(stage_tile, p.dk.head(b, h) + doff, p.dk.sl, row0, p.Lk, Dm, dk, p.scale, lane);
    if constexpr (HAS_G)
        store_rows16<T, 64, IO, false, DH>(stage_tile, p.dtk.head(b, h) + doff, p.dtk.sl, row0, p.Lk, Dm, dtk, p.scale, lane);
    store_rows16<T, 64, IO, false, DH>(stage_tile, p.dv.head(b, h) + doff, p.dv.sl, row0, p.Lk, Dm, dv, 1.0f, lane);
    if constexpr (HAS_G)
        store_rows16<T, 64, IO, false, DH>(stage_tile, p.dtv.head(b, h) + doff, p.dtv.sl, row0, p.Lk, Dm, dtv, 1.0f, lane);
}

template <typename T, int HD, int R, bool HAS_DO, bool HAS_G, int IO = kIoDma, int DT = HD / 16>
__global__ __launch_bounds__(kThreads16, 2) void bwd_col16p_kernel(const BwdParams p) {
    bwd_col16p_body<T, HD, R, HAS_DO, HAS_G, IO, DT>(p, (int)blockIdx.x, (int)gridDim.x);
}

// The paired column-owned launch with the second pass of the row-owned kernel at its end (see
// bwd_col16_repair_kernel).  The row-owned kernel's workgroups have four waves, these eight: in a workgroup that
// takes a row item the upper four leave at once, and the barriers of the others count the waves that are left.
template <typename T, int HD, int R, int RROW, bool HAS_DO, bool HAS_G, int IO = kIoDma, int DT = HD / 16>
__global__ __launch_bounds__(kThreads16, 2) void bwd_col16p_repair_kernel(const BwdParams p) {
    const int col_blocks = p.col_workgroups;
    if ((int)blockIdx.x < col_blocks) {
        bwd_col16p_body<T, HD, R, HAS_DO, HAS_G, IO, DT>(p, (int)blockIdx.x, col_blocks);
    } else {
        if ((int)threadIdx.x >= kXThreads16) return;
        bwd_row16_body<T, HD, RROW, HAS_DO, HAS_G, 2, IO, 1, 1, DT>(p, (int)blockIdx.x - col_blocks, (int)gridDim.x - col_blocks);
    }
}

}  // namespace sjvp
