// fci_rdm2.hip -- the 2-RDM products of up to 16 orbitals on v_mfma_f64_16x16x4_f64 (FCIVector::compute_rdms,
// fci_vector_rdm.cc:106-393): rows of the vectors staged through two LDS buffers, the next chunk's loads in
// registers, every wave with its own output tiles.
#include "fci_internal.h"

#include <algorithm>

namespace fci {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
// two doubles at 8-byte alignment: one 16-byte load whatever the parity of the row length
typedef double d2u __attribute__((ext_vector_type(2), aligned(8)));

constexpr int R2_TH = 256, R2_CK = 32, R2_RS = R2_CK + 2;  // four waves; columns per chunk; LDS row stride

// Stages 32 columns of NR rows (one 16-byte pair per lane: 16 lanes a row, 16 rows a pass) into LDS rows of 34.
// Columns past the end repeat earlier ones; the last one of an odd row comes with the one before it.
template <int NR> struct Stage {
    static constexpr int LD = (NR + 15) / 16;
    const double* p[LD];
    d2u v[LD];
    int ncol, cl;
    bool last = false;
    __device__ __forceinline__ void load(int c0) {
        const int col = c0 + 2 * cl;
        last = col == ncol - 1;
        const int c = min(col, ncol - 2);
#pragma unroll
        for (int i = 0; i < LD; ++i) v[i] = *reinterpret_cast<const d2u*>(p[i] + c);
    }
    __device__ __forceinline__ void store(double* xs, int r) {
#pragma unroll
        for (int i = 0; i < LD; ++i)
            *reinterpret_cast<double2*>(xs + (r + 16 * i) * R2_RS + 2 * cl) = make_double2(last ? v[i].y : v[i].x, v[i].y);
    }
};

// unpacks the triangular index P = hi (hi + 1) / 2 + lo
__device__ __forceinline__ void unpair(int P, int& hi, int& lo) {
    hi = int((sqrtf(float(8 * P + 1)) - 1.f) * 0.5f);
    if ((hi + 1) * (hi + 2) / 2 <= P) ++hi;
    if (hi * (hi + 1) / 2 > P) --hi;
    lo = P - hi * (hi + 1) / 2;
}

// the beta pair z (create r, annihilate s): the pairs r >= s where L and R are one vector, else all n^2
__device__ __forceinline__ void zpair(int z, int n, bool sym, int& r, int& s) {
    if (sym) {
        unpair(z, r, s);
    } else {
        r = z / n;
        s = z - r * n;
    }
}

// zT[chunk][z tile][lane][k-step]: the B operand of the alpha-beta product for 32 beta strings and 16 pairs z:
// lane (g, c), k-step ks is string Ib = 32 chunk + 4 ks + g, pair 16 tile + c; address of the string E_rs
// reaches from Ib | sign << 15, or nstr (a zero behind the row)
__global__ __launch_bounds__(256) void k_rdm2_targets(const uint32_t* __restrict__ out, const uint32_t* __restrict__ str,
                                                      int64_t nstr, int n, int nz, bool sym, uint16_t* __restrict__ zT) {
    const int nzt = (nz + 15) / 16;
    const int64_t x = int64_t(blockIdx.x) * 256 + threadIdx.x;
    if (x >= (nstr + 31) / 32 * nzt * 512) return;
    const int ks = int(x % 8), lane = int((x / 8) % 64);
    const int64_t q = x / 512;
    const int z = int(q % nzt) * 16 + lane % 16;
    const int64_t I = q / nzt * 32 + 4 * ks + lane / 16;
    uint32_t val = uint32_t(nstr);
    if (z < nz && I < nstr) {
        int r, s;
        zpair(z, n, sym, r, s);
        const int hi = max(r, s), lo = min(r, s);
        if ((str[I] >> s) & 1u) {
            const uint32_t t = out[int64_t(hi * (hi + 1) / 2 + lo) * nstr + I];
            if (t != kInvalid) val = (t & kAddrMask) | (t >> 31) << 15;
        }
    }
    zT[x] = uint16_t(val);
}

// Gamma[pr, qs] += sum <L| E^alpha_pq E^beta_rs |R>, block per alpha row Ja: out[e][z] = sum_Ib X[e][Ib] Z[z][Ib]
// with X the rows of R that the single excitations e reach from Ja, and Ja's own row for the diagonal ones,
// and Z[rs][Ib] = +-L[Ja][E_rs Ib]. X is staged; Z is gathered from the row L[Ja] in LDS straight into the
// B-operand layout, by the one wave that owns the pairs' tile, and feeds ET products. Signs of the alpha
// excitations are applied to the sums. Blocks of odd Ja hand their z tiles out two waves further on, so that
// two blocks on a CU load its SIMDs evenly. Where L and R are one vector (sym), Gamma[pr, qs] = Gamma[qs, pr]:
// only the pairs r >= s are formed, and each sum is added in both places.
//
// Bound by the FP64 matrix unit (64 cycles an instruction). CAS(14,14), 3432 x 3432: 3.35 ms with L = R (7 pair
// tiles, 1.7e11 operations, 51 TFLOP/s; the tile that one wave of four lacks costs an eighth) and 6.19 ms with two vectors
// (13 tiles, 51 TFLOP/s), where k_rdm2_ab_mfma, which stages both operands and takes the symmetric pairs of
// both directions, took 21.8 ms. CAS(16,16): 100 ms with L = R, and 452 ms with two vectors, whose sums do not fit
// the registers beside the rest (<5, 4>: 672 bytes of scratch a lane), against 757 for k_rdm2_ab_mfma either way;
// so that one is left to 17 orbitals and up.
template <int ET, int ZW>
__global__ __launch_bounds__(R2_TH, (ET * ZW <= 16 ? 2 : 1)) void k_rdm2_ab5(
    const double* __restrict__ L, const double* __restrict__ R, int64_t Na, int64_t Nb, const uint32_t* __restrict__ into_a,
    int ns, const uint32_t* __restrict__ str_a, const uint16_t* __restrict__ zT, int nz, bool sym, int n,
    double* __restrict__ g2ab) {
    extern __shared__ __attribute__((aligned(16))) double rsh[];
    __shared__ uint32_t ent[ET * 16];
    constexpr int NR = ET * 16, XS = NR * R2_RS;
    double* const Ls = rsh + 2 * XS;  // [Nb] and a zero
    const int64_t Ja = blockIdx.x;
    const int nzt = (nz + 15) / 16;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, cl = lane & 15;
    for (int i = tid; i < NR; i += R2_TH) ent[i] = i < ns ? into_a[Ja * ns + i] : uint32_t(Ja);
    for (int i = tid; i <= int(Nb); i += R2_TH) Ls[i] = i < int(Nb) ? L[Ja * Nb + i] : 0.0;
    __syncthreads();
    Stage<NR> sx;
    sx.ncol = int(Nb);
    sx.cl = tid & 15;
#pragma unroll
    for (int i = 0; i < Stage<NR>::LD; ++i) sx.p[i] = R + int64_t(ent[(tid >> 4) + 16 * i] & kAddrMask) * Nb;
    const int zg = (wave + 2 * int(Ja & 1)) & 3;  // z tiles zg, zg + 4, ...
    d4 acc[ZW][ET];
#pragma unroll
    for (int t = 0; t < ZW; ++t)
#pragma unroll
        for (int e = 0; e < ET; ++e) acc[t][e] = d4{0.0, 0.0, 0.0, 0.0};
    const int nch = int((Nb + R2_CK - 1) / R2_CK);
    u4v tg[ZW];
    auto load_t = [&](int ch) {
#pragma unroll
        for (int t = 0; t < ZW; ++t)  // (tiles past the last one: the first one's, not used)
            tg[t] = *reinterpret_cast<const u4v*>(zT + ((int64_t(ch) * nzt + (zg + 4 * t < nzt ? zg + 4 * t : 0)) * 64 + lane) * 8);
    };
    load_t(0);
    sx.load(0);
    sx.store(rsh, tid >> 4);
    __syncthreads();
    for (int ch = 0; ch < nch; ++ch) {
        const int nx = ch + 1 < nch ? ch + 1 : ch;
        sx.load(nx * R2_CK);
        u4v tc[ZW];
#pragma unroll
        for (int t = 0; t < ZW; ++t) tc[t] = tg[t];
        load_t(nx);
        const double* xa = rsh + (ch & 1) * XS + cl * R2_RS + g;
#pragma unroll
        for (int ks = 0; ks < R2_CK / 4; ++ks) {
            double a[ET], b[ZW];
#pragma unroll
            for (int e = 0; e < ET; ++e) a[e] = xa[e * 16 * R2_RS + ks * 4];
#pragma unroll
            for (int t = 0; t < ZW; ++t) {
                const uint32_t w = ks & 1 ? tc[t][ks / 2] : tc[t][ks / 2] << 16;  // sign in bit 31
                const uint64_t v = __builtin_bit_cast(uint64_t, Ls[(w >> 16) & 0x7FFFu]);
                b[t] = __builtin_bit_cast(double, v ^ (uint64_t(w & 0x80000000u) << 32));
            }
#pragma unroll
            for (int t = 0; t < ZW; ++t)
#pragma unroll
                for (int e = 0; e < ET; ++e) acc[t][e] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[e], b[t], acc[t][e], 0, 0, 0);
        }
        sx.store(rsh + ((ch + 1) & 1) * XS, tid >> 4);
        __syncthreads();
    }
    // D[row 4 v + g][column cl] of each tile: row = excitation e, column = z
    const uint32_t occ = str_a[Ja];
#pragma unroll
    for (int t = 0; t < ZW; ++t) {
        const int z = (zg + 4 * t) * 16 + cl;
        if (z >= nz) continue;
        int r, s;
        zpair(z, n, sym, r, s);
        auto add = [&](int p, int q, double x) {
            atomicAdd(&g2ab[((size_t(p) * n + r) * n + q) * n + s], x);
            if (sym && r != s) atomicAdd(&g2ab[((size_t(q) * n + s) * n + p) * n + r], x);
        };
#pragma unroll
        for (int e16 = 0; e16 < ET; ++e16)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int e = e16 * 16 + 4 * v + g;
                if (e < ns) {
                    const uint32_t en = ent[e];
                    const int P = int((en >> 21) & 0x3FFu);
                    int hi, lo;
                    unpair(P, hi, lo);
                    const int p = (occ >> hi) & 1u ? hi : lo, q = p == hi ? lo : hi;  // created p is occupied in Ja
                    const double x = acc[t][e16][v];
                    add(p, q, (en >> 31) ? -x : x);
                } else if (e == ns) {
                    for (uint32_t o = occ; o; o &= o - 1u) {
                        const int q = __ffs(o) - 1;
                        add(q, q, acc[t][e16][v]);
                    }
                }
            }
    }
}

// Same-spin 2-RDM through the pair cliques, block per clique K: acc[m][m'] += s_m s_m' sum_c L[I_m][c] R[I_m'][c].
// The four waves take every fourth k-step of all MT x MT tiles and add up through LDS; SAME: L and R are one
// vector, staged once, and only the tiles on and above the diagonal are formed. Bound by the matrix unit and,
// close behind, by reading every row once per clique that it is in (21 at half filling of 14 orbitals).
// CAS(14,14), per spin: 0.40 ms (0.54 with all tiles) where k_rdm2_clique took 3.45; that one is left to
// cliques of more than 64 members, whose sums don't fit a wave.
template <int MT, bool SAME>
__global__ __launch_bounds__(R2_TH, MT <= 3 ? 2 : 1) void k_rdm2_clique5(const double* __restrict__ L,
                                                                          const double* __restrict__ R, int64_t ncol,
                                                                          const uint32_t* __restrict__ clq, int M,
                                                                          double* __restrict__ out, int gdim) {
    extern __shared__ __attribute__((aligned(16))) double rsh[];
    __shared__ uint32_t mem[MT * 16];
    constexpr int NR = MT * 16, XS = NR * R2_RS, NB = SAME ? 1 : 2;
    const int64_t K = blockIdx.x;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, cl = lane & 15;
    for (int i = tid; i < NR; i += R2_TH) mem[i] = clq[K * M + min(i, M - 1)];
    __syncthreads();
    Stage<NR> sl, sr;
    sl.ncol = sr.ncol = int(ncol);
    sl.cl = sr.cl = tid & 15;
#pragma unroll
    for (int i = 0; i < Stage<NR>::LD; ++i) {
        const int64_t row = int64_t(mem[(tid >> 4) + 16 * i] & kAddrMask);
        sl.p[i] = L + row * ncol;
        sr.p[i] = R + row * ncol;
    }
    d4 acc[MT][MT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < MT; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    const int nch = int((ncol + R2_CK - 1) / R2_CK);
    sl.load(0);
    if (!SAME) sr.load(0);
    sl.store(rsh, tid >> 4);
    if (!SAME) sr.store(rsh + XS, tid >> 4);
    __syncthreads();
    for (int ch = 0; ch < nch; ++ch) {
        const int nx = ch + 1 < nch ? ch + 1 : ch;
        sl.load(nx * R2_CK);
        if (!SAME) sr.load(nx * R2_CK);
        const double* xa = rsh + (ch & 1) * NB * XS + cl * R2_RS + g;
#pragma unroll
        for (int k2 = 0; k2 < R2_CK / 16; ++k2) {
            const int k = (wave + 4 * k2) * 4;
            const bool in = ch * R2_CK + k + g < int(ncol);  // columns past the end repeat earlier ones
            double a[MT], b[MT];
#pragma unroll
            for (int i = 0; i < MT; ++i) a[i] = xa[i * 16 * R2_RS + k];
#pragma unroll
            for (int i = 0; i < MT; ++i) b[i] = SAME ? a[i] : xa[XS + i * 16 * R2_RS + k];
#pragma unroll
            for (int i = 0; i < MT; ++i) {
                a[i] = in ? a[i] : 0.0;
                b[i] = in ? b[i] : 0.0;
            }
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = SAME ? i : 0; j < MT; ++j) acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(a[i], b[j], acc[i][j], 0, 0, 0);
        }
        sl.store(rsh + ((ch + 1) & 1) * NB * XS, tid >> 4);
        if (!SAME) sr.store(rsh + ((ch + 1) & 1) * NB * XS + XS, tid >> 4);
        __syncthreads();
    }
    // the waves' sums, one after the other into [NR][NR]
    for (int w = 0; w < 4; ++w) {
        if (wave == w)
#pragma unroll
            for (int i = 0; i < MT; ++i)
#pragma unroll
                for (int j = SAME ? i : 0; j < MT; ++j)
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        double* d = rsh + (i * 16 + 4 * v + g) * NR + j * 16 + cl;
                        *d = w ? *d + acc[i][j][v] : acc[i][j][v];
                    }
        __syncthreads();
    }
    for (int x = tid; x < M * M; x += R2_TH) {
        const int m = x / M, mp = x - m * M;
        const uint32_t a = mem[m], b = mem[mp];
        const bool lower = SAME && m > mp;
        const double y = rsh[(lower ? mp : m) * NR + (lower ? m : mp)];
        atomicAdd(&out[size_t((a >> 21) & 0x3FFu) * gdim + ((b >> 21) & 0x3FFu)], ((a ^ b) >> 31) ? -y : y);
    }
}

template <int ET, int ZW>
void run_ab(const SpinTables& a, const SpinTables& b, const double* L, const double* R, const uint16_t* zT, int nz,
            double* g2ab, hipStream_t st) {
    const size_t sh = (size_t(2) * ET * 16 * R2_RS + size_t(b.nstr) + 1) * sizeof(double);
    auto kern = k_rdm2_ab5<ET, ZW>;
    HIPCHK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(sh)));
    kern<<<unsigned(a.nstr), R2_TH, sh, st>>>(L, R, a.nstr, b.nstr, a.into.p, a.ns, a.str.p, zT, nz, L == R, b.n, g2ab);
    HIPCHK(hipGetLastError());
}
template <int ET>
void run_ab_z(const SpinTables& a, const SpinTables& b, const double* L, const double* R, const uint16_t* zT, int nz,
              double* g2ab, hipStream_t st) {
    switch ((nz + 63) / 64) {
        case 1: return run_ab<ET, 1>(a, b, L, R, zT, nz, g2ab, st);
        case 2: return run_ab<ET, 2>(a, b, L, R, zT, nz, g2ab, st);
        case 3: return run_ab<ET, 3>(a, b, L, R, zT, nz, g2ab, st);
        default: return run_ab<ET, 4>(a, b, L, R, zT, nz, g2ab, st);
    }
}
template <int MT>
void run_clique(const SpinTables& sp, const double* L, const double* R, int64_t ncol, double* acc, int gdim, hipStream_t st) {
    auto go = [&](auto kern, int nb) {
        const size_t sh = std::max(size_t(2) * nb * MT * 16 * R2_RS, size_t(MT * 16) * (MT * 16)) * sizeof(double);
        HIPCHK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(sh)));
        kern<<<unsigned(sp.nK), R2_TH, sh, st>>>(L, R, ncol, sp.clq.p, sp.M, acc, gdim);
        HIPCHK(hipGetLastError());
    };
    if (L == R) go(k_rdm2_clique5<MT, true>, 1);
    else go(k_rdm2_clique5<MT, false>, 2);
}

}  // namespace

// At most 16 orbitals (5 excitation tiles, 4 tiles of ordered pairs a wave) and two beta strings; the row and
// the staging buffers take 147 KB of LDS at most
bool rdm2_ab5_ok(const SpinTables& a, const SpinTables& b) { return b.n <= 16 && b.nstr >= 2 && a.k > 0 && b.k > 0; }
void rdm2_ab5(const SpinTables& a, const SpinTables& b, const double* L, const double* R, double* g2ab, hipStream_t st) {
    const bool sym = L == R;
    const int nz = sym ? b.n * (b.n + 1) / 2 : b.n * b.n;
    const int64_t cnt = (b.nstr + 31) / 32 * ((nz + 15) / 16) * 512;
    DBuf<uint16_t> zT(cnt);
    k_rdm2_targets<<<unsigned((cnt + 255) / 256), 256, 0, st>>>(b.out.p, b.str.p, b.nstr, b.n, nz, sym, zT.p);
    HIPCHK(hipGetLastError());
    switch ((a.ns + 1 + 15) / 16) {
        case 1: run_ab_z<1>(a, b, L, R, zT.p, nz, g2ab, st); break;
        case 2: run_ab_z<2>(a, b, L, R, zT.p, nz, g2ab, st); break;
        case 3: run_ab_z<3>(a, b, L, R, zT.p, nz, g2ab, st); break;
        case 4: run_ab_z<4>(a, b, L, R, zT.p, nz, g2ab, st); break;
        default: run_ab_z<5>(a, b, L, R, zT.p, nz, g2ab, st); break;
    }
    HIPCHK(hipStreamSynchronize(st));  // zT is released here
}
// cliques of at most 64 members, two columns or more; acc is added to
bool rdm2_clique5_ok(const SpinTables& sp, int64_t ncol) { return sp.d == 2 && sp.M <= 64 && ncol >= 2; }
void rdm2_clique5(const SpinTables& sp, const double* L, const double* R, int64_t ncol, double* acc, int gdim, hipStream_t st) {
    switch ((sp.M + 15) / 16) {
        case 1: return run_clique<1>(sp, L, R, ncol, acc, gdim, st);
        case 2: return run_clique<2>(sp, L, R, ncol, acc, gdim, st);
        case 3: return run_clique<3>(sp, L, R, ncol, acc, gdim, st);
        default: return run_clique<4>(sp, L, R, ncol, acc, gdim, st);
    }
}

}  // namespace fci
