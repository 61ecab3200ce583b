// Fused Lennard-Jones + Ewald real-space pair forces over the full neighbor
// list.  Replaces compute_force_iso / compute_energy_iso
// (src/Evaluators/PairEvaluateIso.h:8-358) instantiated with EvaluatorLJ
// (PairEvaluatorLJ.h:17-60) and ChargeEvaluatorEwald
// (ChargeEvaluatorEwald.h:11-63), the fusion the reference reaches through
// charge offloading (State.cpp:648-660, FixPair.cpp:89-97,
// EvaluatorWrapper.h:176-194).
//
// Design (gfx950): a team of P lanes (P = 4..32) owns one atom and strides
// through its row, so each row load is a P-wide coalesced segment and the
// neighbor positions (float4 x - lo, q) are gathered from cell-ordered memory
// that stays L2-resident.  Rows hold charged neighbors first and uncharged
// ones at the end, so an atom reads only the part that can interact with it:
// Coulomb needs q_i != 0 and charged neighbors, LJ needs a nonzero epsilon
// for the type pair (per-type flags say which part has such partners).  For
// TIP4P water an H or M site reads its charged part with Coulomb only and an
// O site its uncharged part with LJ only.  Arithmetic is FP32; the team's partial sums are
// combined with butterfly shuffles and added once per atom into the 64-bit
// fixed-point force buffer.  Energy and virial (0.5-weighted, full list) are
// reduced in FP64 per block and added with one fixed-point atomic per block.
#include <type_traits>

#include "erfc_fit.h"
#include "mdx_internal.h"

namespace mdx {

namespace {

struct PairArgs {
    int n;
    const float4 *xq;
    const int *type;
    int cap;
    const uint32_t *nl;
    const int *nlCount;
    const int *nlCountA;
    const int *typeFlags;
    const float *params;
    int ntypes;
    const BoxDev *bx;             // box lengths and alpha
    float spec[3];
    float qqr, rq2;
    unsigned long long *force;
    unsigned long long *acc;
    const int *vgate;  // EVM 2 inside a captured step: the barostat gate (0: no trace this step)
    RowMaxArgs rm;     // a captured build's row maxima in one extra workgroup (rm.on)
};

// EVM: 0 forces only; 1 energy and virial tensor; 2 the virial's trace only
// (sum r F, what a barostat needs), into ACC_VTRACE, skipped on steps whose
// barostat gate is 0
template <int P, bool LJ, bool COUL, int EVM>
__device__ __forceinline__ void pair_body(int blk, int nblk, PairArgs a) {
    constexpr bool EV = EVM == 1, VT = EVM == 2;
    if (a.rm.on && blk == nblk - 1) {  // uniform over the workgroup
        if (!a.rm.gate || *a.rm.gate != 0) row_max_wg(a.rm.na, a.rm.a, a.rm.nb, a.rm.b, a.rm.flags);
        return;
    }
    // box values into locals
    const float bL0 = a.bx->Lf[0], bL1 = a.bx->Lf[1], bL2 = a.bx->Lf[2];
    const float bI0 = a.bx->invLf[0], bI1 = a.bx->invLf[1], bI2 = a.bx->invLf[2];
    const float alphaB = a.bx->alphaF;
    __shared__ float sp[3 * kMaxTypes * kMaxTypes];
    __shared__ int sfl[kMaxTypes];
    __shared__ float smult[4];  // special-pair multiplier by tag
    __shared__ double wred[4][7];
    const int T2 = a.ntypes * a.ntypes;
    if (LJ) {
        for (int t = threadIdx.x; t < 3 * T2; t += blockDim.x) sp[t] = a.params[t];
        for (int t = threadIdx.x; t < a.ntypes; t += blockDim.x) sfl[t] = a.typeFlags[t];
    }
    if (threadIdx.x == 0) {
        smult[0] = 1.0f;
        smult[1] = a.spec[0];
        smult[2] = a.spec[1];
        smult[3] = a.spec[2];
    }
    __syncthreads();
    const int gt = blk * blockDim.x + threadIdx.x;
    const int i = gt / P;
    const int tl = threadIdx.x & (P - 1);
    float fx = 0.f, fy = 0.f, fz = 0.f;
    float e = 0.f, v0 = 0.f, v1 = 0.f, v2 = 0.f, v3 = 0.f, v4 = 0.f, v5 = 0.f;
    if (i < a.n) {
        const float4 pi = a.xq[i];
        const int ti = (LJ && a.ntypes > 1) ? a.type[i] : 0;
        const int fl = LJ ? sfl[ti] : 0;
        const int cnt = min(a.nlCount[i], a.cap);
        const int nA = min(a.nlCountA[i], cnt);
        const uint32_t *row = a.nl + (size_t)i * a.cap;
        const float twoAlphaRtPi = 2.0f * 0.5641895835477563f * alphaB;
        const float alpha2 = alphaB * alphaB;
        const float rq2 = a.rq2, qqi = a.qqr * pi.w;
        // One row entry.  What lies out of range is masked by a branch, not
        // added as a zero: lanes of a team take neighbouring entries of a row,
        // sorted by cell, so whole teams (16 lanes, a quarter of the wave) are
        // often out of range together, and the SIMD skips a quarter whose lanes
        // are all off.  Without the branches the kernel issued 13 % fewer
        // instructions and was no faster (88 us against 79 for 131,072 sites).
        // Reciprocals without the division's scaling, multipliers from a table
        // and loops without the other term: 131,072 water sites 82.6 -> 71.3 us,
        // 32,768 27.7 -> 24.6, 2,048 14.4 -> 12.0, 500,000 LJ atoms 107 -> 95.
        auto term = [&](auto L_, auto C_, uint32_t raw, const float4 &pj, float rc2, float eps24, float sig6) {
            constexpr bool L = decltype(L_)::value, C = decltype(C_)::value;
            float dx = pi.x - pj.x, dy = pi.y - pj.y, dz = pi.z - pj.z;
            dx -= bL0 * rintf(dx * bI0);
            dy -= bL1 * rintf(dy * bI1);
            dz -= bL2 * rintf(dz * bI2);
            // contracted by hand: the copies of this code must round alike
            const float r2 = fmaf(dz, dz, fmaf(dx, dx, dy * dy));
            asm volatile("" ::"v"(pj.w));  // keeps the charge in the record's load, out of the branch
            const bool inL = L && r2 < rc2, inC = C && r2 < rq2;
            if (!inL && !inC) return;
            const float m = smult[raw >> 30];
            float fs = 0.f;
            if (L && inL && m != 0.0f) {
                // the division's own special cases (coincident atoms) kept
                const float r2inv = __builtin_amdgcn_div_fixupf(rcp_exact(r2), r2, 1.0f);
                const float r6inv = r2inv * r2inv * r2inv;
                const float p1 = eps24 * 2.0f * sig6 * sig6;
                const float p2 = eps24 * sig6;
                fs += r6inv * r2inv * (p1 * r6inv - p2) * m;
                if (EV) {
                    const float s6r6 = sig6 * r6inv;
                    const float rc6 = rc2 * rc2 * rc2;
                    const float s6rc6 = sig6 / rc6;
                    e += 0.5f * (eps24 * (1.0f / 6.0f)) * (s6r6 * (s6r6 - 1.0f) - s6rc6 * (s6rc6 - 1.0f)) * m;
                }
            }
            if (C && (!L || inC)) {
                const float ls = __builtin_amdgcn_fmed3f(r2, 1e-10f, 3.4e38f);
                const float rinv = __builtin_amdgcn_rsqf(ls);  // ls is normal
                const float len = ls * rinv;
                const float qq = qqi * pj.w;
                // erfc(ar) - (1 - m); for a full exclusion (m = 0) this is -erf(ar).
                // erfc shares the Gaussian's exponential (erfc_fit.h)
                const float gauss = __expf(-alpha2 * ls);
                const float ec = erfc_from_gauss(alphaB * len, gauss) - (1.0f - m);
                const float s = qq * (ec * rinv + twoAlphaRtPi * gauss);
                fs += s * rinv * rinv;
                if (EV) e += 0.5f * qq * rinv * ec;
            }
            fx += dx * fs;
            fy += dy * fs;
            fz += dz * fs;
            if (VT) v0 += fs * r2;
            if (EV) {
                v0 += dx * fs * dx;
                v1 += dy * fs * dy;
                v2 += dz * fs * dz;
                v3 += dx * fs * dy;
                v4 += dx * fs * dz;
                v5 += dy * fs * dz;
            }
        };
        // A lane takes entries k0 + tl, + P, + 2P, ... of [k0, k1) in that order,
        // U of them per pass with all their loads in flight before any is used
        // (reading on past k1 instead of masking those loads costs 7 % where the
        // rows come from HBM).
        constexpr int U = 4;
        auto walk = [&](auto L_, auto C_, int k0, int k1) {
            constexpr bool L = decltype(L_)::value;
            const bool one = a.ntypes == 1;  // uniform: the only type pair stays in registers
            const float rc2a = L && one ? sp[0] : 0.f, eps24a = L && one ? sp[1] : 0.f, sig6a = L && one ? sp[2] : 0.f;
            for (int kb = k0 + tl; kb < k1; kb += U * P) {
                const uint32_t *rp = row + kb;
                uint32_t raw[U];
                float4 pj[U];
                int tj[U];
                bool ok[U];
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    ok[u] = kb + u * P < k1;
                    raw[u] = ok[u] ? rp[u * P] : (uint32_t)i;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    const uint32_t j = raw[u] & 0x3FFFFFFFu;
                    pj[u] = a.xq[j];
                    tj[u] = L && !one ? a.type[j] : 0;
                }
#pragma unroll
                for (int u = 0; u < U; ++u) {
                    float rc2 = rc2a, eps24 = eps24a, sig6 = sig6a;
                    if (L && !one) {
                        const int tp = ti * a.ntypes + tj[u];
                        rc2 = sp[tp];
                        eps24 = sp[T2 + tp];
                        sig6 = sp[2 * T2 + tp];
                    }
                    if (ok[u]) term(L_, C_, raw[u], pj[u], rc2, eps24, sig6);
                }
            }
        };
        // part 0: charged neighbors [0, nA); part 1: charge-free ones [nA, cnt).
        // The wave takes the code of the terms that any of its atoms needs there
        // (in TIP4P water part 0 is all Coulomb and part 1 all LJ).
        using Yes = std::true_type;
        using No = std::false_type;
        for (int part = 0; part < 2; ++part) {
            const bool lj = LJ && (fl & (1 << part));
            const bool coul = COUL && part == 0 && pi.w != 0.0f;
            const int k0 = part == 0 ? 0 : nA, k1 = part == 0 ? nA : cnt;
            if (LJ && !(COUL && part == 0)) {
                if (lj) walk(Yes{}, No{}, k0, k1);
            } else if (COUL && !(LJ && __any(lj))) {
                if (coul) walk(No{}, Yes{}, k0, k1);
            } else if (LJ && COUL) {
                if (lj && coul) walk(Yes{}, Yes{}, k0, k1);
                else if (lj) walk(Yes{}, No{}, k0, k1);
                else if (coul) walk(No{}, Yes{}, k0, k1);
            }
        }
    }
    fx = team_sum<P>(fx);
    fy = team_sum<P>(fy);
    fz = team_sum<P>(fz);
    if (tl == 0 && i < a.n) {
        fx_add(&a.force[3 * i + 0], fx);
        fx_add(&a.force[3 * i + 1], fy);
        fx_add(&a.force[3 * i + 2], fz);
    }
    if (VT && (!a.vgate || *a.vgate)) {  // one value for the whole workgroup
        double x = team_sum_d<64>(0.5 * (double)v0);
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
        if (lane == 0) wred[w][0] = x;
        __syncthreads();
        if (threadIdx.x == 0) {
            x = 0.0;
            for (int ww = 0; ww < (int)(blockDim.x >> 6); ++ww) x += wred[ww][0];
            fx_add(&acc_rep(a.acc)[ACC_VTRACE], x);
        }
    }
    if (EV) {
        double vals[7] = {e, 0.5 * v0, 0.5 * v1, 0.5 * v2, 0.5 * v3, 0.5 * v4, 0.5 * v5};
        const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
        for (int s = 0; s < 7; ++s) {
            double x = team_sum_d<64>(vals[s]);
            if (lane == 0) wred[w][s] = x;
        }
        __syncthreads();
        if (threadIdx.x < 7) {
            double x = 0.0;
            for (int ww = 0; ww < (int)(blockDim.x >> 6); ++ww) x += wred[ww][threadIdx.x];
            fx_add(&acc_rep(a.acc)[threadIdx.x == 0 ? ACC_PAIR : ACC_VIR + threadIdx.x - 1], x);
        }
    }
}

template <int P, bool LJ, bool COUL>
void launch3(Ctx &c, const PairArgs &a, int evm) {
    const int blocks = cdiv((long long)a.n * P, 256) + a.rm.on;
    if (evm == 1) launch<pair_body<P, LJ, COUL, 1>, 256>(c, blocks, 0, a);
    else if (evm == 2) launch<pair_body<P, LJ, COUL, 2>, 256>(c, blocks, 0, a);
    else launch<pair_body<P, LJ, COUL, 0>, 256>(c, blocks, 0, a);
}

template <int P>
void launch2(Ctx &c, const PairArgs &a, bool lj, bool coul, int evm) {
    if (lj && coul) launch3<P, true, true>(c, a, evm);
    else if (lj) launch3<P, true, false>(c, a, evm);
    else launch3<P, false, true>(c, a, evm);
}

}  // namespace

// Per-type flags of the LJ table against the charge classes present: bit 0 =
// nonzero epsilon with some type that has charged atoms, bit 1 = with some type
// that has uncharged atoms.  Recomputed when the system or the table changes.
std::vector<int> pair_type_flag_table(const Ctx &c) {
    std::vector<int> charged(kMaxTypes, 0), neutral(kMaxTypes, 0), fl(kMaxTypes, 0);
    for (size_t i = 0; i < c.typeHost.size(); ++i) (c.qHost[i] != 0.0f ? charged : neutral)[c.typeHost[i]] = 1;
    const int T = c.ntypes;
    for (int a = 0; a < T && c.ljOn; ++a)
        for (int b = 0; b < T; ++b) {
            if (c.ljEps[a * T + b] == 0.0) continue;
            if (charged[b]) fl[a] |= 1;
            if (neutral[b]) fl[a] |= 2;
        }
    return fl;
}

static void pair_type_flags(Ctx &c) {
    if (!c.pairTypeFlags) c.pairTypeFlags = dalloc<int>(c, kMaxTypes);
    const std::vector<int> fl = pair_type_flag_table(c);
    MDX_REQUIRE(!c.capture, 3, "pair type flags must be set before a step is captured");
    MDX_HIP(hipMemcpyAsync(c.pairTypeFlags, fl.data(), sizeof(int) * kMaxTypes, hipMemcpyHostToDevice, c.stream));
    MDX_HIP(hipStreamSynchronize(c.stream));
    c.pairFlagsDirty = false;
}

void pair_forces(Ctx &c, bool energy, bool virial) {
    const bool coul = c.ewaldReal && c.hasCharges;
    if (!c.ljOn && !coul) return;
    if (c.pairFlagsDirty) pair_type_flags(c);
    PairArgs a;
    a.n = c.n;
    a.xq = c.xq;
    a.type = c.type[c.cur];
    a.cap = c.cap;
    a.nl = c.nl;
    a.nlCount = c.nlCount;
    a.nlCountA = c.nlCountA;
    a.typeFlags = c.pairTypeFlags;
    a.params = c.ljParams;
    a.ntypes = c.ntypes;
    for (int d = 0; d < 3; ++d) {
        a.spec[d] = c.special[d];
    }
    a.bx = c.box;
    a.qqr = c.qqr;
    a.rq2 = c.rq2;
    a.force = c.force;
    a.acc = c.acc;
    a.vgate = baro_gate(c);
    a.rm = row_max_args(c);
    const int evm = (energy || virial) ? 1 : (c.vtrace ? 2 : 0);
    ProfScope ps(c, PK_PAIR);
    switch (c.pairTeam) {
        case 4: launch2<4>(c, a, c.ljOn, coul, evm); break;
        case 8: launch2<8>(c, a, c.ljOn, coul, evm); break;
        case 16: launch2<16>(c, a, c.ljOn, coul, evm); break;
        default: launch2<32>(c, a, c.ljOn, coul, evm); break;
    }
}

}  // namespace mdx
