// Fused attention-JVP forward, 16-wide form (gfx950).
//
// Computes what the reference forward does (semicat/jvp_utils/ryu_triton.py:73-291: O, TO, M = lse,
// MU, LI in one online-softmax pass), decomposed for occupancy: a workgroup of eight wavefronts owns
// 128 queries of one (batch, head), 16 per wavefront as MFMA columns, and walks over the keys in
// stages of 32 streamed through an LDS ring by LDS-DMA.  A wavefront needs fewer than 128 registers,
// so several wavefronts per SIMD overlap their MFMA chains, exponentials and LDS reads, and two
// workgroups per CU overlap one's copies with the other's arithmetic.
#pragma once
#include "sjvp_fwd.hpp"
#include "sjvp_staged16.hpp"

namespace sjvp {

// LDS layout, SPB = 1 (one stage per barrier): [own: Q (, Q_dot) rows of the workgroup, four slabs
// each][ring: R slots of K, V (, K_dot, V_dot) stage slabs][sink].  SPB = 2 (long key axes: two stages
// per barrier, half as many barriers): [ring of four slots][sink]; the own rows, which every wave
// moves into registers before the first stage is consumed, land in slots 2 and 3 (exactly their
// size), which then join the ring.  After the last stage the ring doubles as the per-wave staging
// tiles of the output stores.
template <int HD, int R, bool JVP, int SPB = 1, bool DMA = true, int SPLIT = 1>
struct Fwd16Smem {
    static constexpr int nt = JVP ? 4 : 2;
    static constexpr int slot = nt * Slab<HD>::elems;
    static constexpr int own = DMA && SPLIT == 1 ? (JVP ? 2 : 1) * 4 * Slab<HD>::elems : 0;
    static_assert(SPB == 1 || SPLIT > 1 || (SPB == 2 && R == 4 && own == 2 * slot), "SPB = 2 needs a ring of four slots");
    static constexpr int own_off = SPB == 2 ? 2 * slot : 0;
    static constexpr int ring_off = SPB == 2 ? 0 : own;
    static constexpr int loop = (SPB == 2 ? R * slot : own + R * slot) * (int)sizeof(elem_t);
    static constexpr int after = SPLIT > 1 ? Split16Smem<HD, kWaves16, JVP ? 2 : 1>::bytes : 0;
    static constexpr int sink = loop > after ? loop : after;
    static constexpr int bytes = sink + kSink16;
    static_assert(R * slot >= kWaves16 * StoreStage16<HD>::elems, "ring too small to stage stores");
};

// ROPE: q, k and their tangents are rotated by p.rope as they are loaded (head dimension 64, one
// stage per barrier): the own rows in registers, each stage's K (, K_dot) slab in place in LDS.  Meant
// for key axes that one workgroup per (batch, head) walks once (every workgroup rotates the K rows it
// streams).
// IO: how the tensors lie in memory (sjvp_staged16.hpp); anything but kIoDma copies its stages through registers,
// one stage ahead, and loads its own rows straight into registers.
// NC: sets of 16 queries per wavefront (NC = 2: four wavefronts, every operand read from LDS feeds both sets; with tangents
// 202 registers and no gain: 96.6 us against 97.6 at B=8 H=16 L=1024 D=64, 105 against 101 at B=128 H=12 L=256).
// SPLIT > 1 (launches of few workgroups): the SPLIT waves of a group share 16 queries and take every SPLIT-th stage each, SPLIT
// stages to a barrier; their partial sums are brought to one maximum and added in LDS, in a fixed order.
// DT: 16-wide tiles of the head dimension that hold columns below D.  D <= 48 in the class of 64 needs three of four: a quarter
// of the output products and of their transposing reads, which the LDS serves at half rate, are left out (here and in the
// backward pair).  Forward + backward, 4 / 3 tiles: B=4 H=6 333 x 205 D=48 cotangent on TO 35.0 / 32.6 us, B=8 H=8 L=300 D=36
// 60.2 / 57.7, B=8 H=16 L=1024 D=48 475 / 456, B=64 H=12 L=256 D=48 233 / 229.
// D <= 96 in the class of 128 needs six of eight, and three of the score products' four chunks: 8 / 6 tiles at B=8 H=16 L=1024
// D=80 1012 / 886 us, B=64 H=12 L=128 D=96 181 / 172, L=256 D=80 495 / 448, B=8 H=12 L=512 D=75 (staged) 320 / 292.
// D = 16 in the class of 32 needs one of two: B=64 H=12 L=256 134 / 120 us, B=8 H=16 L=1024 233 where D = 32 takes 251.
template <typename T, int HD, int R, bool JVP, int OCC, int SPB = 1, bool ROPE = false, int IO = kIoDma, int NC = 1,
          int SPLIT = 1, int DT = HD / 16>
__global__ __launch_bounds__(kThreads16 / NC, OCC) void fwd16_kernel(const FwdParams p) {
    constexpr int NT = kThreads16 / NC;  // threads of the workgroup
    static_assert(!ROPE || (HD == 64 && SPB == 1), "the folded rotation covers HD = 64, one stage per barrier");
    constexpr bool DMA = IO == kIoDma;
    static_assert(DMA || ((SPB == 1 || SPLIT > 1) && !ROPE), "staged copies run one stage ahead, unrotated");
    static_assert(SPLIT == 1 || (SPB == SPLIT && R == 2 * SPLIT && NC == 1 && !ROPE), "a step is a stage for every part");
    extern __shared__ __align__(16) unsigned char smem_raw[];
    using SM = Fwd16Smem<HD, R, JVP, SPB, DMA, SPLIT>;
    constexpr bool OWN_LDS = DMA && SPLIT == 1;  // the own rows come through LDS, else straight into registers
    elem_t* own = reinterpret_cast<elem_t*>(smem_raw) + SM::own_off;
    elem_t* ring = reinterpret_cast<elem_t*>(smem_raw) + SM::ring_off;
    constexpr int SE = Slab<HD>::elems;
    constexpr int KL = HD / 32;        // 32-column chunks of a row
    constexpr int KC = (DT + 1) / 2;  // those with columns below D: k-chunks of the score contraction

    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int n = lane & 15;  // owned query within the wave
    const int g = lane >> 4;  // lane group
    // with one workgroup per (batch, head) the identity is kept: the fused backward relies on head i
    // having run on XCD i % 8
    const int bid = p.q_blocks > 1 ? xcd_linear_id((int)blockIdx.x, (int)gridDim.x) : (int)blockIdx.x;
    const int bh = bid / p.q_blocks;
    const int qb = bid % p.q_blocks;
    const int b = bh / p.H, h = bh % p.H;
    const int part = SPLIT > 1 ? wave % SPLIT : 0, group = wave / SPLIT;
    const int q0 = qb * (kOwned16 / SPLIT);
    const int wrow = q0 + group * 16 * NC;  // the wave's first query; the lane's are wrow + 16 u + n
    const bool wave_active = wrow < p.Lq;

    u32x4 qB[NC][KL], tqB[NC][KL];
    using StagePlan = std::conditional_t<DMA, CopyPlan<HD, SM::nt, 1, NT>, StagedPlan<T, HD, SM::nt, NT, IO>>;
    constexpr int SPT = StagePlan::N;
    StagePlan plan[DMA ? 1 : SPLIT];
    // slot layout K | V | K_dot | V_dot (primal only: K | V)
    const Src sk{p.k.head(b, h), p.k.sl}, sv{p.v.head(b, h), p.v.sl};
    if constexpr (!OWN_LDS) {
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const bool qvalid = wrow + 16 * u + n < p.Lq;
            const int64_t qrow = IO == kIoAny ? own_row(wrow + 16 * u + n, p.Lq) : wrow + 16 * u + n;
            load_b_operands16<T, HD, IO>(qB[u], p.q.head(b, h) + qrow * p.q.sl, g, p.D, qvalid);
            if constexpr (JVP) load_b_operands16<T, HD, IO>(tqB[u], p.tq.head(b, h) + qrow * p.tq.sl, g, p.D, qvalid);
        }
    }
    if constexpr (DMA) {
        // own rows first (issued before the stages, so they land first), then the ring
        if constexpr (OWN_LDS) {
            CopyPlan<HD, JVP ? 8 : 4, 4, NT> own_plan;
            if constexpr (JVP)
                own_plan.init(tid, q0, p.D, smem_raw + SM::sink, Src{p.q.head(b, h), p.q.sl},
                              Src{p.tq.head(b, h), p.tq.sl});
            else
                own_plan.init(tid, q0, p.D, smem_raw + SM::sink, Src{p.q.head(b, h), p.q.sl});
            own_plan.issue(own, p.Lq - q0, p.D == HD && q0 + kOwned16 <= p.Lq);
        }
        if constexpr (JVP)
            plan[0].init(tid, 0, p.D, smem_raw + SM::sink, sk, sv, Src{p.tk.head(b, h), p.tk.sl},
                      Src{p.tv.head(b, h), p.tv.sl});
        else
            plan[0].init(tid, 0, p.D, smem_raw + SM::sink, sk, sv);
    } else {
#pragma unroll
        for (int u = 0; u < SPLIT; ++u) {
            if constexpr (JVP)
                plan[u].init(tid, p.D, sk, sv, Src{p.tk.head(b, h), p.tk.sl}, Src{p.tv.head(b, h), p.tv.sl});
            else
                plan[u].init(tid, p.D, sk, sv);
            plan[u].take(u, SPLIT);
        }
    }
    const int ns = (p.Lk + kStageRows - 1) / kStageRows;
    int issued = 0;
    auto issue_next = [&]() {
        elem_t* slot = ring + (issued % R) * SM::slot;
        issue_plan(plan[0], slot, p.Lk - issued * kStageRows, p.D == HD && (issued + 1) * kStageRows <= p.Lk);
        ++issued;
    };
    // staged copies: the stages of the next step (`ahead` of it in the ring), each through its own plan
    auto stage_step = [&](int first) {
        if constexpr (!DMA) {
#pragma unroll
            for (int u = 0; u < SPLIT; ++u)
                if (first + u < ns) plan[u].issue(ring + ((first + u) % R) * SM::slot, p.Lk - (first + u) * kStageRows);
        }
    };
    auto commit_step = [&]() {
        if constexpr (!DMA) {
#pragma unroll
            for (int u = 0; u < SPLIT; ++u) plan[u].commit();
        }
    };
    if constexpr (SPLIT > 1 && DMA) {
        // the stages of the first step only: the loads of the own rows are awaited by a wait for all that is outstanding
        while (issued < SPLIT && issued < ns) issue_next();
#pragma unroll
        for (int c = 0; c < KC; ++c) {
            asm volatile("" : "+v"(qB[0][c]));
            if constexpr (JVP) asm volatile("" : "+v"(tqB[0][c]));
        }
        while (issued < R && issued < ns) issue_next();
    } else if constexpr (DMA) {
        while (issued < (SPB == 2 ? 2 : R) && issued < ns) issue_next();
    } else {
        stage_step(0);
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const bool qvalid = wrow + 16 * u + n < p.Lq;
            finish_b_operands16<HD, IO>(qB[u], g, p.D, qvalid);
            if constexpr (JVP) finish_b_operands16<HD, IO>(tqB[u], g, p.D, qvalid);
        }
        commit_step();
        // The own rows are awaited here, once: left to their first use, the wait stands inside the loop and takes the next
        // stage's copies with it (B=50 H=10 L=292, D = 21 44 -> 48 us, D = 36 70 -> 73.5).
#pragma unroll
        for (int u = 0; u < NC; ++u)
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                asm volatile("" : "+v"(qB[u][c]));
                if constexpr (JVP) asm volatile("" : "+v"(tqB[u][c]));
            }
    }

    const float sl2 = p.scale * kLog2e;
    // per set of queries
    float m_i[NC];     // reference maximum (same in the four lanes of a query)
    float m_sub[NC];   // what the exponentials subtract: m_i, but 0 where no key of this lane's has a score above -inf yet
    float m_true[NC];  // maximum over the keys this lane has seen (for LI)
    float l_i[NC];     // exp-sum over the keys this lane has seen
    float mu_i[NC];    // sum of p * S_dot over the same keys
    // acc = sum P~ V;  tacc = sum (P~ * S_dot) V + P~ V_dot  (the reference's g_acc + p_tv_acc, which
    // only ever appear added together, ryu_triton.py:274-275)
    f32x4 acc[NC][DT], tacc[NC][DT];
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        m_i[u] = m_true[u] = -INFINITY;
        m_sub[u] = 0.f;
        l_i[u] = mu_i[u] = 0.f;
#pragma unroll
        for (int t = 0; t < DT; ++t) {
            acc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            tacc[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
    }

    // SPB = 1: the own rows and stage 0 were issued before the other stages; SPB = 2: everything
    if constexpr (SPLIT > 1) wait_stages<SPT>(DMA && issued > SPLIT ? issued - SPLIT : 0);
    else if constexpr (DMA) wait_stages<SPT>(SPB == 2 ? 0 : issued - 1);
    workgroup_barrier();
    if constexpr (OWN_LDS) {
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            const int r0 = wave * 16 * NC + 16 * u;  // of the workgroup's 128 rows, 32 to a slab
            const int r = (r0 & 31) + n;
            read_b_operands16<HD>(qB[u], own + (r0 >> 5) * SE, r, g);
            if constexpr (JVP) read_b_operands16<HD>(tqB[u], own + (4 + (r0 >> 5)) * SE, r, g);
            if constexpr (ROPE) {
                // the lane's two operands are columns 8g.. and 32 + 8g.. of its query: a rotation pair
                rope8<T>(qB[u][0], qB[u][1], p.rope, q0 + r0 + n, g, 1.0f);
                if constexpr (JVP) rope8<T>(tqB[u][0], tqB[u][1], p.rope, q0 + r0 + n, g, 1.0f);
            }
        }
    }
    // ROPE: rotate the K (, K_dot) slab of a landed stage in place; 128 items per slab
    auto rotate_stage = [&](elem_t* slot, int k0) {
        if constexpr (ROPE) {
            if (tid < 128) rope_slab_item<T>(slot, tid, p.rope, k0, 1.0f);
            else if (JVP && tid < 256) rope_slab_item<T>(slot + 2 * SE, tid - 128, p.rope, k0, 1.0f);
            workgroup_barrier();
        }
    };
    rotate_stage(ring, 0);
    if constexpr (SPB == 2 && OWN_LDS) {
        // the operands must have arrived in registers before the copies below overwrite their slots
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        workgroup_barrier();
        while (issued < R && issued < ns) issue_next();
    }

    auto compute = [&](const elem_t* slot, int k0) {
        const elem_t* sK = slot;
        const elem_t* sV = slot + SE;
        const elem_t* sTK = slot + 2 * SE;
        const elem_t* sTV = slot + 3 * SE;
        f32x4 s[NC][2], ts[NC][2];
#pragma unroll
        for (int t = 0; t < 2; ++t) {
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                s[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
                ts[u][t] = f32x4{0.f, 0.f, 0.f, 0.f};
            }
#pragma unroll
            for (int c = 0; c < KC; ++c) {
                const u32x4 a = lds_a_rows16<HD>(sK, t, c, n, g);
#pragma unroll
                for (int u = 0; u < NC; ++u) {
                    s[u][t] = T::mfma16(a, qB[u][c], s[u][t]);
                    if constexpr (JVP) ts[u][t] = T::mfma16(a, tqB[u][c], ts[u][t]);
                }
                if constexpr (JVP) {
                    const u32x4 at = lds_a_rows16<HD>(sTK, t, c, n, g);
#pragma unroll
                    for (int u = 0; u < NC; ++u) ts[u][t] = T::mfma16(at, qB[u][c], ts[u][t]);
                }
            }
        }
        if (k0 + kStageRows > p.Lk) {  // wave-uniform: only the last stage can be ragged
            // keys beyond Lk are zero rows in LDS (their S_dot is already 0)
#pragma unroll
            for (int u = 0; u < NC; ++u)
#pragma unroll
                for (int t = 0; t < 2; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
                        if (k0 + 16 * t + 4 * g + j >= p.Lk) s[u][t][j] = -INFINITY;
        }
        float mloc[NC];
        bool raise = false;
#pragma unroll
        for (int u = 0; u < NC; ++u) {
            mloc[u] = fmaxf(fmaxf(fmaxf(s[u][0][0], s[u][0][1]), fmaxf(s[u][0][2], s[u][0][3])),
                            fmaxf(fmaxf(s[u][1][0], s[u][1][1]), fmaxf(s[u][1][2], s[u][1][3]))) * sl2;
            m_true[u] = fmaxf(m_true[u], mloc[u]);
            raise = raise || mloc[u] > m_i[u] + kMaxSlack;
        }
        if (__builtin_amdgcn_ballot_w64(raise) != 0) {  // wave-uniform branch
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                const float m_new = fmaxf(m_i[u], group_max(mloc[u]));
                // 0 on the first tile.  A part of a split group may hold nothing but keys that score -inf.
                const float alpha = SPLIT == 1 || m_i[u] < m_new ? fast_exp2(m_i[u] - m_new) : 1.f;
                m_i[u] = m_new;
                m_sub[u] = SPLIT > 1 && m_new == -INFINITY ? 0.f : m_new;
                l_i[u] *= alpha;
                if constexpr (JVP) mu_i[u] *= alpha;
#pragma unroll
                for (int d = 0; d < DT; ++d) {
                    acc[u][d] *= alpha;
                    if constexpr (JVP) tacc[u][d] *= alpha;
                }
            }
        }
        u32x4 pb[NC], ptb[NC];
#pragma unroll
        for (int u = 0; u < NC; ++u) {
#pragma unroll
            for (int t = 0; t < 2; ++t)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float pj = fast_exp2(fmaf(s[u][t][j], sl2, SPLIT > 1 ? -m_sub[u] : -m_i[u]));
                    s[u][t][j] = pj;
                    l_i[u] += pj;
                    if constexpr (JVP) {
                        const float pt = pj * (ts[u][t][j] * p.scale);
                        ts[u][t][j] = pt;
                        mu_i[u] += pt;
                    }
                }
            pb[u] = pack_b16<T>(s[u][0], s[u][1]);
            if constexpr (JVP) ptb[u] = pack_b16<T>(ts[u][0], ts[u][1]);
        }
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            const u32x4 av = lds_a_tr16<HD>(sV, 16 * d, lane);
#pragma unroll
            for (int u = 0; u < NC; ++u) {
                acc[u][d] = T::mfma16(av, pb[u], acc[u][d]);
                if constexpr (JVP) tacc[u][d] = T::mfma16(av, ptb[u], tacc[u][d]);
            }
            if constexpr (JVP) {
                const u32x4 atv = lds_a_tr16<HD>(sTV, 16 * d, lane);
#pragma unroll
                for (int u = 0; u < NC; ++u) tacc[u][d] = T::mfma16(atv, pb[u], tacc[u][d]);
            }
        }
    };

    // One trip of the outer loop goes once round the ring, so that every LDS address of the
    // unrolled body is a per-lane constant plus an immediate offset.
    static_assert(R % SPB == 0, "a step must not wrap the ring");
    const elem_t* part_ring = ring + part * SM::slot;
    for (int i0 = 0; i0 < ns; i0 += R) {
#pragma unroll
        for (int h = 0; h < R; h += SPB) {
            const int i = i0 + h;
            if (i >= ns) break;
            if (i > 0) {
                // the stages of this step have landed for every wave; those of the last step are consumed
                if constexpr (DMA) wait_stages<SPT>(SPB > 1 ? 0 : issued - 1 - i);
                workgroup_barrier();
            }
            if constexpr (DMA) {
                if (i > 0) {
#pragma unroll
                    for (int u = 0; u < SPB; ++u)
                        if (issued < ns) issue_next();
                }
            } else {
                stage_step(i + SPB);
            }
            if (i > 0) rotate_stage(ring + h * SM::slot, i * kStageRows);
            if constexpr (SPLIT > 1) {
                if (wave_active && i + part < ns) compute(part_ring + h * SM::slot, (i + part) * kStageRows);
            } else if (wave_active) {
#pragma unroll
                for (int u = 0; u < SPB; ++u)
                    if (i + u < ns) compute(ring + (h + u) * SM::slot, (i + u) * kStageRows);
            }
            commit_step();
        }
    }
    workgroup_barrier();  // every wave is done reading the ring: it becomes the store staging area
    if constexpr (SPLIT > 1) {
        using SP = Split16Smem<HD, kWaves16, JVP ? 2 : 1>;
        f32x4* red = reinterpret_cast<f32x4*>(smem_raw);
        float* stat = reinterpret_cast<float*>(smem_raw + SP::red);
        elem_t* tile = reinterpret_cast<elem_t*>(smem_raw + SP::red + SP::stat) + wave * StoreStage16<HD>::elems;
        const int64_t so = (int64_t)bh * p.Lr + wrow + n;
        float l = group_sum(l_i[0]), mu_un = group_sum(mu_i[0]), m_all = -INFINITY, t_all = -INFINITY;
        if (p.li) m_true[0] = group_max(m_true[0]);
        float* mine = stat + wave * 64 + n;
        if (g == 0) {
            mine[0] = m_i[0];
            mine[16] = l;
            mine[32] = mu_un;
            mine[48] = m_true[0];
        }
        workgroup_barrier();
        const float* all = stat + SPLIT * group * 64 + n;
#pragma unroll
        for (int s = 0; s < SPLIT; ++s) {
            m_all = fmaxf(m_all, all[64 * s]);
            t_all = fmaxf(t_all, all[64 * s + 48]);
        }
        l = mu_un = 0.f;
#pragma unroll
        for (int s = 0; s < SPLIT; ++s) {
            const float f = fast_exp2(all[64 * s] - m_all);  // 0 for a part without keys
            l += f * all[64 * s + 16];
            mu_un += f * all[64 * s + 32];
        }
        const float inv_l = 1.0f / l, cmu = mu_un * inv_l, f = fast_exp2(m_i[0] - m_all);
#pragma unroll
        for (int d = 0; d < DT; ++d) {
            acc[0][d] *= f;
            if constexpr (JVP) tacc[0][d] = tacc[0][d] * f - cmu * acc[0][d];  // see below
        }
        if (g == 0 && part == 0) {
            // a group without queries gets what a zero query row produces
            p.lse[so] = wave_active ? (m_all + fast_log2(l)) * kLn2 : fast_log2((float)p.Lk) * kLn2;
            if constexpr (JVP) p.mu[so] = wave_active ? cmu : 0.f;
            if (p.li) p.li[so] = wave_active ? l * fast_exp2(m_all - t_all) : (float)p.Lk;
        }
        split_put<DT, kWaves16>(red, 0, wave, lane, acc[0]);
        if constexpr (JVP) split_put<DT, kWaves16>(red, 1, wave, lane, tacc[0]);
        workgroup_barrier();
        if (!wave_active) return;
        if (part == 0) {
            split_sum<DT, kWaves16, SPLIT>(acc[0], red, 0, group, lane);
            store_rows16<T, HD, IO, false, DT>(tile, p.o.head(b, h), p.o.sl, wrow, p.Lq, p.D, acc[0], inv_l, lane);
        }
        if constexpr (JVP) {
            if (part == 1) {
                split_sum<DT, kWaves16, SPLIT>(acc[0], red, 1, group, lane);
                store_rows16<T, HD, IO, false, DT>(tile, p.to.head(b, h), p.to.sl, wrow, p.Lq, p.D, acc[0], inv_l, lane);
            }
        }
        return;
    }
    elem_t* stage_tile = ring + wave * StoreStage16<HD>::elems;
#pragma unroll
    for (int u = 0; u < NC; ++u) {
        const int row0 = wrow + 16 * u;
        const int64_t so = (int64_t)bh * p.Lr + row0 + n;
        if (row0 >= p.Lq) {
            // All 16 rows lie beyond Lq: their statistic rows get the values a zero query row produces (and the
            // reference initialises them with): log(Lk), 0, Lk.
            if (g == 0) {
                p.lse[so] = fast_log2((float)p.Lk) * kLn2;
                if constexpr (JVP) p.mu[so] = 0.f;
                if (p.li) p.li[so] = (float)p.Lk;
            }
            continue;
        }
        // Combine the four lanes' partial sums (they cover disjoint keys of the same query).
        const float l = group_sum(l_i[u]);
        const float inv_l = 1.0f / l;
        float mu_un = 0.f;
        if constexpr (JVP) mu_un = group_sum(mu_i[u]);
        if (p.li) m_true[u] = group_max(m_true[u]);
        if (g == 0) {
            // Statistic rows up to Lr are all written: a padded query row (all-zero q, q_dot) yields
            // exactly the values the reference initialises them with: log(Lk), 0, Lk.
            p.lse[so] = (m_i[u] + fast_log2(l)) * kLn2;
            if constexpr (JVP) p.mu[so] = mu_un * inv_l;
            // LI is the exp-sum relative to the true row maximum (ryu_triton.py:291); l is relative
            // to m_i, which may lag behind it by up to kMaxSlack.
            if (p.li) p.li[so] = l * fast_exp2(m_i[u] - m_true[u]);
        }
        const float cmu = mu_un * inv_l;
        if constexpr (JVP) {
            // TO = (g_acc + p_tv_acc - mu_un * O) / l     (ryu_triton.py:274-275)
#pragma unroll
            for (int d = 0; d < DT; ++d) tacc[u][d] -= cmu * acc[u][d];
        }
        store_rows16<T, HD, IO, false, DT>(stage_tile, p.o.head(b, h), p.o.sl, row0, p.Lq, p.D, acc[u], inv_l, lane);
        if constexpr (JVP)
            store_rows16<T, HD, IO, false, DT>(stage_tile, p.to.head(b, h), p.to.sl, row0, p.Lq, p.D, tacc[u], inv_l, lane);
    }
}

}  // namespace sjvp
