// fci_ab32.hip -- the mixed-precision alpha-beta term of sigma (H2_aabb,
// fci_vector_hamiltonian.cc:194-272): FP32 vectors, BF16x3 products on v_mfma_f32_16x16x32_bf16 with
// FP32 accumulation; per alpha row gather -> MFMA -> LDS scatter, every wave on its own columns.
#include "fci_device.h"
#include "fci_internal.h"

#include <algorithm>

namespace fci {

namespace {

typedef float f4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf8 __attribute__((ext_vector_type(8)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
// two floats at 4-byte alignment: one 8-byte load whatever the parity of the row length
typedef float f2u __attribute__((ext_vector_type(2), aligned(4)));

// Registers of a wave with all row tiles: A operands, diagonal rows and targets per tile, the raw and the
// split columns. Where they pass 256, two waves share the row tiles of their columns (WM = 2, two waves a
// SIMD): with one wave a SIMD the products, the scatter's vector instructions and its LDS atomics run one
// after the other.
constexpr int ab5m_regs(int ks, int nt) { return nt * (8 * ks + 8) + 32 * ks + 8 * ks + 60; }
constexpr int ab5m_row_waves(int ks, int nmt) { return ab5m_regs(ks, nmt) > 264 ? 2 : 1; }
constexpr int ab5m_waves(int ks, int nmt) {
    const int wm = ab5m_row_waves(ks, nmt), r = ab5m_regs(ks, (nmt + wm - 1) / wm);
    return r > 168 ? 2 : r > 128 ? 3 : 4;
}

// One block per alpha row Ja. A wave takes 32 beta columns at a time: lane (g, c) loads columns 2c and
// 2c + 1 of the gathered rows X[e][Ib] = C[Ia_e][Ib] of the single excitations into Ja with one 8-byte
// load (whole 128-byte lines of four rows) straight into the B-operand layout of two column tiles,
// multiplies them with every row tile of V[rs][e] = s_e (p_e q_e | rs), held in registers for the whole
// row as BF16 hi and lo, adds the diagonal excitations' rank-1 term in FP32 and scatters into the LDS
// row srow[Jb], Jb = E_rs Ib (FP64: its LDS atomic costs a seventh of the FP32 one).
//
// Loads that are pinned a whole chunk ahead, a scatter without branches and any parity of the row length.
// What bounds it: nothing alone; LDS atomics (13.8 cycles each in a CU), the vector instructions of the
// scatter and the split, and the products (which overlap the vector instructions of the SIMD's other wave
// by about half) each take 40 to 65 % of the time. Measured (MI355X), against k_ab3_mixed / the general
// kernel: CAS(12,12) 94 -> 55 us, CAS(14,14) 1.12 -> 0.91 ms, odd: 12 electrons in 13 orbitals
// (1716 x 1287) 884 -> 189 us, 15 electrons in 15 orbitals (6435 x 6435) 20.1 -> 3.5 ms.
template <int KS, int NMT>
__global__ __launch_bounds__(256 * ab5m_row_waves(KS, NMT), ab5m_waves(KS, NMT)) void k_ab5_mixed(
    const float* __restrict__ C, float* __restrict__ S, int64_t Na, int64_t Nb, const uint32_t* __restrict__ into_a,
    int ns, const uint32_t* __restrict__ str_a, const uint16_t* __restrict__ outT, int ntile, int np,
    const float* __restrict__ vpk) {
    constexpr int WM = ab5m_row_waves(KS, NMT), NT = (NMT + WM - 1) / WM;
    const int TH = blockDim.x, NW = TH / (64 * WM);  // NW: column waves
    extern __shared__ __attribute__((aligned(16))) double srow[];  // [ab_row_slots(Nb)]
    __shared__ uint32_t ent[KS * 32];
    __shared__ __attribute__((aligned(16))) float vdg[NT * WM * 16];
    const int64_t Ja = xcd_remap(blockIdx.x, Na);
    if (Ja >= Na) return;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, cl = lane & 15;
    // row wave, column wave (waves w and w + 4 share a SIMD), first row tile
    const int rw = WM == 2 && wave >= NW, wc = wave - rw * NW, t0 = rw * NT;
    for (int i = tid; i < KS * 32; i += TH) ent[i] = i < ns ? into_a[Ja * ns + i] : kInvalid;
    for (int i = tid; i < int(ab_row_slots(Nb)); i += TH) srow[i] = 0.0;
    const uint32_t occ = str_a[Ja];
    for (int r = tid; r < NT * WM * 16; r += TH) {  // diagonal excitations: sum_{q in Ja} (qq|r)
        float d = 0.f, t[16];                        // every orbital's row is read, all loads in flight
#pragma unroll
        for (int q = 0; q < 16; ++q) t[q] = vpk[(occ >> q) & 1u ? size_t(q * (q + 1) / 2 + q) * np + min(r, np - 1) : 0];
#pragma unroll
        for (int q = 0; q < 16; ++q) d += (occ >> q) & 1u ? t[q] : 0.f;
        vdg[r] = r < np ? d : 0.f;
    }
    __syncthreads();

    bf8 ah[NT][KS], al[NT][KS];
    uint32_t roff[KS][8];  // byte offset of this lane's rows of C (below 4 GB: at most 15 orbitals)
    {
        float raw[NT][KS][8];
        uint32_t en[KS][8];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                en[ks][x] = ent[ks * 32 + 8 * g + x];
                const bool ex = en[ks][x] != kInvalid;
                roff[ks][x] = uint32_t((ex ? int64_t(en[ks][x] & kAddrMask) : 0) * Nb * 4);
                const float* vrow = vpk + (ex ? size_t((en[ks][x] >> 21) & 0x3FFu) * np : 0);
#pragma unroll
                for (int j = 0; j < NT; ++j) raw[j][ks][x] = vrow[min((t0 + j) * 16 + cl, np - 1)];
            }
        // all of these loads are in flight before the first one is used
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                // sign of the gathered row folded in; slots without an excitation read row 0 against zeros
                const float sg = en[ks][x] == kInvalid ? 0.f : (en[ks][x] >> 31) ? -1.f : 1.f;
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    __bf16 h, l;
                    split_bf16(raw[j][ks][x] * ((t0 + j) * 16 + cl < np ? sg : 0.f), h, l);
                    ah[j][ks][x] = h;
                    al[j][ks][x] = l;
                }
            }
    }
    f4 vd[NT];
#pragma unroll
    for (int j = 0; j < NT; ++j) vd[j] = *reinterpret_cast<const f4*>(vdg + (t0 + j) * 16 + 4 * g);

    // the waves run the same program: a part of a chunk apart, their scatters do not queue together
    constexpr int EIGHTH = (KS * NT * 12 + 31) / 32;  // of a chunk, in units of 64 cycles
    if (wave & 1) __builtin_amdgcn_s_sleep(EIGHTH);
    if (wave & 2) __builtin_amdgcn_s_sleep(2 * EIGHTH);
    if (wave & 4) __builtin_amdgcn_s_sleep(4 * EIGHTH);

    const GLOBAL_MEM char* Cg = (const GLOBAL_MEM char*)C;
    const int nch = int((Nb + 31) / 32);
    const uint32_t rja = uint32_t(Ja * Nb * 4);
    f2u x[KS][8], cx;
    u4v tg[NT];
    uint32_t coff = 0;  // byte offset of this lane's columns in the chunk whose loads are being issued
    const GLOBAL_MEM char* tbase = nullptr;
    auto aim = [&](int ch) {
        coff = uint32_t(min(ch * 32 + 2 * cl, int(Nb) - 2)) * 4;  // columns past the end: computed, never kept
        tbase = (const GLOBAL_MEM char*)outT + (int64_t(ch) * ntile + t0) * 1024;
    };
    // the loads stay where they are written: a wait then leaves every later one in flight
    auto load_x = [&]() {
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
            for (int i = 0; i < 8; ++i) {
                x[ks][i] = *reinterpret_cast<const GLOBAL_MEM f2u*>(Cg + (roff[ks][i] + coff));
                __builtin_amdgcn_sched_barrier(0);
            }
        cx = *reinterpret_cast<const GLOBAL_MEM f2u*>(Cg + (rja + coff));
        __builtin_amdgcn_sched_barrier(0);
    };
    auto load_t = [&](int j) {
        // (a wave's tiles past the last one: targets of its first, not used)
        tg[j] = *reinterpret_cast<const GLOBAL_MEM u4v*>(tbase + (t0 + j < NMT ? j : 0) * 1024 + uint32_t(lane * 16));
        __builtin_amdgcn_sched_barrier(0);
    };
    if (wc < nch) {
        aim(wc);
        __builtin_amdgcn_sched_barrier(0);
        load_x();
#pragma unroll
        for (int j = 0; j < NT; ++j) load_t(j);
        // the columns are loaded again as soon as they have been split, each target as soon as it has been
        // used: the loads are in flight for a whole chunk (the last chunk loads itself again)
        for (int ch = wc; ch < nch; ch += NW) {
            bf8 bh0[KS], bl0[KS], bh1[KS], bl1[KS];
            // odd Nb: the last column's pair was read one to the left
            const bool tail = ch * 32 + 2 * cl == int(Nb) - 1;
            float cd0 = tail ? cx.y : cx.x, cd1 = cx.y;
#pragma unroll
            for (int ks = 0; ks < KS; ++ks)
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    __bf16 h, l;
                    split_bf16(tail ? x[ks][i].y : x[ks][i].x, h, l);
                    bh0[ks][i] = h;
                    bl0[ks][i] = l;
                    split_bf16(x[ks][i].y, h, l);
                    bh1[ks][i] = h;
                    bl1[ks][i] = l;
                }
            __builtin_amdgcn_sched_barrier(0);
            aim(ch + NW < nch ? ch + NW : ch);
            load_x();
            f4 a0[2], a1[2];
            auto products = [&](int j) {
                f4 p0 = f4{0.f, 0.f, 0.f, 0.f}, p1 = f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int ks = 0; ks < KS; ++ks) {
                    p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[j][ks], bh0[ks], p0, 0, 0, 0);
                    p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[j][ks], bh1[ks], p1, 0, 0, 0);
                    p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[j][ks], bl0[ks], p0, 0, 0, 0);
                    p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[j][ks], bl1[ks], p1, 0, 0, 0);
                    p0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[j][ks], bh0[ks], p0, 0, 0, 0);
                    p1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[j][ks], bh1[ks], p1, 0, 0, 0);
                }
                a0[j & 1] = p0;
                a1[j & 1] = p1;
            };
            auto scatter = [&](int j) {
#pragma unroll
                for (int p = 0; p < 2; ++p)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const uint32_t tw = tg[j][p * 2 + v / 2];
                        const uint32_t sgn = (v & 1 ? tw : tw << 16) & 0x80000000u;
                        const uint32_t slot = v & 1 ? (tw >> 16) & 0x7FFFu : tw & 0x7FFFu;
                        const float a = (p ? a1[j & 1][v] : a0[j & 1][v]) + vd[j][v] * (p ? cd1 : cd0);
                        atomicAdd(&srow[slot], double(__uint_as_float(__float_as_uint(a) ^ sgn)));
                    }
            };
            // the products of a tile beside the scatter of the one before
            products(0);
#pragma unroll
            for (int j = 1; j <= NT; ++j) {
                if (j < NT && (WM == 1 || j + t0 < NMT)) products(j);
                if (WM == 1 || j - 1 + t0 < NMT) scatter(j - 1);
                load_t(j - 1);
            }
        }
    }
    __syncthreads();
    float* Srow = S + Ja * Nb;
    constexpr int U = 8;
    for (int i0 = tid; i0 < int(Nb); i0 += U * TH) {
        float s[U];
#pragma unroll
        for (int u = 0; u < U; ++u) s[u] = Srow[min(i0 + u * TH, int(Nb) - 1)];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int i = i0 + u * TH;
            if (i < int(Nb)) Srow[i] = float(double(s[u]) + srow[ab_slot(i)]);
        }
    }
}

struct Ab5mLaunch {
    const SpinTables &a, &b;
    const float* C;
    float* S;
    const float* vpk;
    hipStream_t st;
};

template <int KS, int NMT> void run(const Ab5mLaunch& l) {
    auto kern = k_ab5_mixed<KS, NMT>;
    const size_t sh = size_t(ab_row_slots(l.b.nstr)) * sizeof(double);
    HIPCHK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(sh)));
    // column waves: none without a chunk of the row (1365 rows of 15 strings, 15 orbitals: 45.4 -> 17.5 us, 42.4 in
    // the general kernel, which took these rows before)
    const unsigned nw = unsigned(std::min<int64_t>(4, (l.b.nstr + 31) / 32));
    kern<<<xcd_grid(l.a.nstr), 64 * nw * ab5m_row_waves(KS, NMT), sh, l.st>>>(
        l.C, l.S, l.a.nstr, l.b.nstr, l.a.into.p, l.a.ns, l.a.str.p, l.b.outT.p, l.b.npp >> 4, l.b.np, l.vpk);
    HIPCHK(hipGetLastError());
}

}  // namespace

// 16-bit targets, at most 15 orbitals (so at most 56 excitations and 8 row tiles), two strings or more
bool ab5_mixed_ok(const SpinTables& b) { return b.outT.p != nullptr && b.n <= 15 && b.nstr >= 2; }
void ab5_mixed(const float* C, float* S, const SpinTables& a, const SpinTables& b, const float* vpk, hipStream_t st) {
    const Ab5mLaunch l{a, b, C, S, vpk, st};
    const int nmt = (b.np + 15) / 16;
    const bool one = a.ns <= 32;
#define CASE(T) \
    case T: return one ? run<1, T>(l) : run<2, T>(l);
    switch (nmt) {
        case 1: return run<1, 1>(l);
        case 2: return run<1, 2>(l);
        case 3: return run<1, 3>(l);
        case 4: return run<1, 4>(l);
        CASE(5) CASE(6) CASE(7) CASE(8)
    }
#undef CASE
    throw Error(-1, "alpha-beta kernel: no instance for this shape");
}

}  // namespace fci
