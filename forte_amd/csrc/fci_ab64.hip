// fci_ab64.hip -- the FP64 alpha-beta term of sigma (H2_aabb, fci_vector_hamiltonian.cc:194-272) on
// v_mfma_f64_16x16x4_f64: per alpha row gather -> MFMA -> LDS scatter, every wave on its own columns.
#include "fci_device.h"
#include "fci_internal.h"

#include <algorithm>

namespace fci {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

constexpr int AB5_TH = 256;  // four waves; blocks of short rows have fewer

// registers of a wave: A operands, accumulators, B operands, row offsets, targets and the rest
constexpr int ab5_regs(int ks, int nmt) { return 2 * nmt * ks + 8 * nmt + 3 * ks + 2 * nmt + 40; }
constexpr int ab5_waves(int ks, int nmt) {
    const int r = ab5_regs(ks, nmt);
    return r > 250 ? 1 : r > 160 ? 2 : r > 120 ? 3 : 4;
}

// One block per alpha row Ja. A wave takes 16 beta columns at a time: lane (g, c) loads column c of the
// gathered rows X[e][Ib] = C[Ia_e][Ib] of the single excitations into Ja straight into the MFMA
// B-operand layout, multiplies them with every row tile of V[rs][e] = s_e (p_e q_e | rs), held in
// registers for the whole row, and scatters the products into the LDS row srow[Jb], Jb = E_rs Ib. The
// excitation behind the last one is the row Ja itself against sum_{q in Ja} (qq|rs).
//
// What bounds it: the matrix cores, 2 N_det 16 NMT 4 KS flops. An FP64 MFMA keeps the SIMD's vector
// instructions of every wave out for its 64 cycles (measured: the two add up), so a second wave on the
// SIMD hides no scatter; what counts is few vector instructions per product. Hence one wave with all row
// tiles (each B operand feeds NMT products, no sharing of tiles, staging or barriers between waves), up
// to 512 registers of A operands, and loads that need no address arithmetic beyond one addition. The
// scatter takes 5 vector instructions a value, 15 % of a chunk at n = 16.
// Measured (MI355X), before: row tiles over 4 waves, k-steps padded to 16 excitations, odd string counts
// through the general kernel: CAS(16,16) 62.4 -> 52.7 ms (61 TFLOP/s), CAS(14,14) 4.05 -> 2.58 ms,
// CAS(12,12) 0.212 -> 0.117 ms, 12 electrons in 13 orbitals (1716 x 1287) 1.42 -> 0.35 ms. Tried with the
// rows staged in LDS by the block and two waves a SIMD: 56 to 63 ms at CAS(16,16), whatever the prefetch.
template <int KS, int NMT>
__global__ __launch_bounds__(AB5_TH, ab5_waves(KS, NMT)) void k_ab5_f64(
    const double* __restrict__ C, double* __restrict__ S, int64_t Na, int64_t Nb, const uint32_t* __restrict__ into_a,
    int ns, const uint32_t* __restrict__ str_a, const uint16_t* __restrict__ outT, int ntile, int np,
    const double* __restrict__ vpk, const void* const* __restrict__ act, const double* const* __restrict__ C_t,
    double* const* __restrict__ S_t, const double* const* __restrict__ V_t) {
    extern __shared__ __attribute__((aligned(16))) double srow[];  // [ab_row_slots(Nb)]
    __shared__ uint32_t ent[KS * 4];
    __shared__ double vdg[NMT * 16];
    if (act) {
        if (!act[blockIdx.y]) return;
        C = C_t[blockIdx.y];
        S = S_t[blockIdx.y];
        vpk = V_t[blockIdx.y];
    }
    const GLOBAL_MEM char* Cg = (const GLOBAL_MEM char*)C;
    const GLOBAL_MEM double* vpkg = (const GLOBAL_MEM double*)vpk;
    const int64_t Ja = xcd_remap(blockIdx.x, Na);
    if (Ja >= Na) return;
    const int th = blockDim.x, nw = th >> 6;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, cl = lane & 15;
    for (int i = tid; i < KS * 4; i += th) ent[i] = i < ns ? into_a[Ja * ns + i] : kInvalid;
    for (int i = tid; i < int(ab_row_slots(Nb)); i += th) srow[i] = 0.0;
    const uint32_t occ = str_a[Ja];
    for (int r = tid; r < NMT * 16; r += th) {  // diagonal excitations: sum_{q in Ja} (qq|r)
        double d = 0.0, t[16];                      // every orbital's row is read, all loads in flight
#pragma unroll
        for (int q = 0; q < 16; ++q) t[q] = vpkg[(occ >> q) & 1u ? size_t(q * (q + 1) / 2 + q) * np + min(r, np - 1) : 0];
#pragma unroll
        for (int q = 0; q < 16; ++q) d += (occ >> q) & 1u ? t[q] : 0.0;
        vdg[r] = r < np ? d : 0.0;
    }
    __syncthreads();

    // A operands: row m of a tile holds pair 4 (m % 4) + m / 4, so that accumulator element v of lane
    // group g is pair 4 g + v, the order of the target table. The sign of the gathered row is folded
    // in; slots without an excitation read row Ja against zeros.
    double va[NMT][KS], b[KS];
    uint32_t roff[KS];  // byte offset of this lane's row of C (below 4 GB: at most 16 orbitals)
    double sg[KS];      // sign of the excitation, 0 where there is none
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
        const uint32_t en = ent[ks * 4 + g];
        const bool ex = en != kInvalid;
        roff[ks] = uint32_t((ex ? int64_t(en & kAddrMask) : Ja) * Nb * 8);
        sg[ks] = !ex ? 0.0 : (en >> 31) ? -1.0 : 1.0;
        const GLOBAL_MEM double* vrow = vpkg + (ex ? size_t((en >> 21) & 0x3FFu) * np : 0);
#pragma unroll
        for (int j = 0; j < NMT; ++j) va[j][ks] = vrow[min(j * 16 + 4 * (cl % 4) + cl / 4, np - 1)];
    }
    // all of these loads are in flight before the first one is used
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
        for (int j = 0; j < NMT; ++j) {
            const int rs = j * 16 + 4 * (cl % 4) + cl / 4;
            va[j][ks] *= j < NMT - 1 || rs < np ? sg[ks] : 0.0;
        }
        if (ks == ns / 4)  // uniform: the slot behind the last excitation
#pragma unroll
            for (int j = 0; j < NMT; ++j) {
                const double d = vdg[j * 16 + 4 * (cl % 4) + cl / 4];
                va[j][ks] = g == ns % 4 ? d : va[j][ks];
            }
    }
    // The waves run the same program; a quarter of a chunk apart, one scatters while the others multiply.
    // In step, all four would queue at the LDS (18 cycles an atomic) and then leave it idle.
    constexpr int QUARTER = KS * NMT / 4;  // of a chunk's products, in units of 64 cycles
    if (wave == 1) __builtin_amdgcn_s_sleep(QUARTER < 127 ? QUARTER : 127);
    if (wave == 2) __builtin_amdgcn_s_sleep(2 * QUARTER < 127 ? 2 * QUARTER : 127);
    if (wave == 3) __builtin_amdgcn_s_sleep(3 * QUARTER < 127 ? 3 * QUARTER : 127);
    const int nch = int((Nb + 15) / 16);
    const uint32_t lane_t = uint32_t(g * 256 + cl * 8);  // this lane's bytes within 16 columns of a tile's targets
    u2v tg[NMT];
    uint32_t coff = 0;  // byte offset of this lane's column in the chunk whose loads are being issued
    const GLOBAL_MEM char* tbase = nullptr;
    auto aim = [&](int ch) {
        coff = uint32_t(min(ch * 16 + cl, int(Nb) - 1)) * 8;  // columns past the end: computed, never kept
        tbase = (const GLOBAL_MEM char*)outT + int64_t(ch >> 1) * ntile * 1024 + (ch & 1) * 128;
    };
    // the loads stay where they are written: a wait then leaves every later one in flight, in the first
    // chunk as in the others (moved about, the first chunk's make the loop wait for all of them)
    auto load_b = [&](int ks) {
        b[ks] = *reinterpret_cast<const GLOBAL_MEM double*>(Cg + (roff[ks] + coff));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_t = [&](int j) {
        tg[j] = *reinterpret_cast<const GLOBAL_MEM u2v*>(tbase + j * 1024 + lane_t);
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wave < nch) {
        aim(wave);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) load_b(ks);
#pragma unroll
        for (int j = 0; j < NMT; ++j) load_t(j);
        // each B operand and target is replaced by the next chunk's as soon as it has been used, so the
        // loads are in flight for a whole chunk (the last chunk loads itself again)
        for (int ch = wave; ch < nch; ch += nw) {
            aim(ch + nw < nch ? ch + nw : ch);
            d4 acc[NMT];
#pragma unroll
            for (int j = 0; j < NMT; ++j) acc[j] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
            for (int ks = 0; ks < KS; ++ks) {
#pragma unroll
                for (int j = 0; j < NMT; ++j)
                    acc[j] = __builtin_amdgcn_mfma_f64_16x16x4f64(va[j][ks], b[ks], acc[j], 0, 0, 0);
                load_b(ks);
            }
#pragma unroll
            for (int j = 0; j < NMT; ++j) {
#pragma unroll
                for (int v = 0; v < 4; ++v) {
                    const uint32_t tw = v < 2 ? tg[j].x : tg[j].y;
                    const uint32_t sgn = v & 1 ? tw : tw << 16;
                    const uint32_t slot = v & 1 ? (tw >> 16) & 0x7FFFu : tw & 0x7FFFu;
                    const uint64_t bits = __builtin_bit_cast(uint64_t, double(acc[j][v]));
                    const uint32_t hi = uint32_t(bits >> 32) ^ (sgn & 0x80000000u);
                    atomicAdd(&srow[slot], __builtin_bit_cast(double, (uint64_t(hi) << 32) | uint32_t(bits)));
                }
                load_t(j);
            }
        }
    }
    __syncthreads();
    GLOBAL_MEM double* Srow = (GLOBAL_MEM double*)S + Ja * Nb;
    constexpr int U = 8;
    for (int i0 = tid; i0 < int(Nb); i0 += U * th) {
        double s[U];
#pragma unroll
        for (int u = 0; u < U; ++u) s[u] = Srow[min(i0 + u * th, int(Nb) - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * th;
            if (i < int(Nb)) Srow[i] = s[u] + srow[ab_slot(i)];
        }
    }
}

// Waves of a block: none without a chunk of the row. Rows of at most 8 chunks get one wave once there are rows
// for every SIMD: each wave loads all of A, and that is then most of its time. 16 orbitals, 12870 rows: 16
// strings 642 -> 178 us (586 in the kernel before this one), 120 strings 1063 -> 641 (1032).
unsigned block_waves(int64_t rows, int64_t nb) {
    const int64_t nch = (nb + 15) / 16;
    return nch <= 8 && rows >= 1024 ? 1 : unsigned(std::min<int64_t>(AB5_TH / 64, nch));
}

struct Ab5Launch {
    const SpinTables &a, &b;
    const double* C;
    double* S;
    const double* vpk;
    const BatchSigmaTabs* t;  // batched launch (null: the plain pointers)
    hipStream_t st;
    bool prepare;             // only set the kernel attribute
};

template <int KS, int NMT> void run(const Ab5Launch& l) {
    auto kern = k_ab5_f64<KS, NMT>;
    const size_t sh = size_t(ab_row_slots(l.b.nstr)) * sizeof(double);
    if (l.prepare || !l.t)
        HIPCHK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(sh)));
    if (l.prepare) return;
    const unsigned ny = l.t ? unsigned(l.t->nitem) : 1;
    kern<<<dim3(xcd_grid(l.a.nstr), ny), 64 * block_waves(l.a.nstr * ny, l.b.nstr), sh, l.st>>>(
        l.C, l.S, l.a.nstr, l.b.nstr, l.a.into.p, l.a.ns, l.a.str.p, l.b.outT.p, l.b.npp >> 4, l.b.np, l.vpk,
        l.t ? l.t->act : nullptr, l.t ? l.t->c : nullptr, l.t ? l.t->s : nullptr, l.t ? l.t->vpk : nullptr);
    HIPCHK(hipGetLastError());
}

// The smallest instance with room for ns excitations and the diagonal one in its k-steps of 4; false:
// none. Run when l is given. For every tile count (orbital count) the list holds the exact counts of
// its half-filled spaces and a few lower ones for other fillings (14 and 16 orbitals: also that of one
// electron or hole, whose few rows leave the chip idle; 16 rows of 12870 strings 569 -> 381 us, 500 before
// this kernel).
template <int NMT, int KS, int... More> bool pick(int ns, const Ab5Launch* l) {
    if (ns < 4 * KS) {
        if (l) run<KS, NMT>(*l);
        return true;
    }
    if constexpr (sizeof...(More) > 0) return pick<NMT, More...>(ns, l);
    return false;
}
bool dispatch(const SpinTables& a, const SpinTables& b, const Ab5Launch* l) {
    const int ns = a.ns;
    switch ((b.np + 15) / 16) {
        case 1: return pick<1, 2>(ns, l);
        case 2: return pick<2, 2, 3, 4>(ns, l);
        case 3: return pick<3, 4, 5, 6>(ns, l);
        case 4: return pick<4, 5, 7>(ns, l);
        case 5: return pick<5, 5, 7, 8, 9, 10>(ns, l);
        case 6: return pick<6, 6, 8, 10, 11>(ns, l);
        case 7: return pick<7, 4, 7, 9, 11, 13>(ns, l);
        case 8: return pick<8, 7, 10, 13, 15>(ns, l);
        case 9: return pick<9, 4, 8, 11, 14, 16, 17>(ns, l);
        default: return false;
    }
}

}  // namespace

// 16-bit targets (which bounds the row to 104 KB of LDS) and at most 16 orbitals
bool ab5_f64_ok(const SpinTables& a, const SpinTables& b) {
    return b.outT.p != nullptr && b.n <= 16 && dispatch(a, b, nullptr);
}
void ab5_f64(const double* C, double* S, const SpinTables& a, const SpinTables& b, const double* vpk, hipStream_t st) {
    const Ab5Launch l{a, b, C, S, vpk, nullptr, st, false};
    dispatch(a, b, &l);
}
void ab5_f64_batch(const SpinTables& a, const SpinTables& b, const BatchSigmaTabs& t, hipStream_t st) {
    const Ab5Launch l{a, b, nullptr, nullptr, nullptr, &t, st, false};
    dispatch(a, b, &l);
}
void ab5_f64_prepare(const SpinTables& a, const SpinTables& b) {
    const Ab5Launch l{a, b, nullptr, nullptr, nullptr, nullptr, nullptr, true};
    dispatch(a, b, &l);
}

}  // namespace fci
