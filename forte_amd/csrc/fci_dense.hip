// fci_dense.hip -- the same-spin terms of sigma for small string spaces (H0, H1 and H2_aaaa / H2_bbbb,
// fci_vector_hamiltonian.cc:84-192) as one dense product per spin: S = s C + Haa C + C Hbb.
#include "fci_device.h"
#include "fci_internal.h"

#include <algorithm>

namespace fci {

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));

// Row I of the same-spin operator over the strings of one spin, from the pair cliques: every hole string K
// inside I contributes s_m s_m' g'[m][m'] to column I_m' (trans: row I of the operator's transpose, with
// g'[m'][m]; one-electron integrals need not be symmetric). One block per row; the members of a clique are
// different strings, so a thread owns each of them and the sum over K runs in a fixed order.
__global__ __launch_bounds__(64) void k_dense_same(const uint32_t* __restrict__ clq, int M, int64_t nstr,
                                                   const uint32_t* __restrict__ own, int nown,
                                                   const double* __restrict__ G, int gdim, bool trans,
                                                   double* __restrict__ H,
                                                   const double* const* __restrict__ G_t = nullptr,
                                                   double* const* __restrict__ H_t = nullptr) {
    extern __shared__ double row[];  // [nstr]
    if (G_t) {
        G = G_t[blockIdx.y];
        H = H_t[blockIdx.y];
    }
    const int64_t I = blockIdx.x;
    for (int i = threadIdx.x; i < int(nstr); i += 64) row[i] = 0.0;
    __syncthreads();
    for (int j = 0; j < nown; ++j) {
        const uint32_t slot = own[I * nown + j];
        const uint32_t e = clq[slot];
        const uint32_t* ent = clq + size_t(slot / uint32_t(M)) * M;
        const uint32_t ge = (e >> 21) & 0x3FFu;
        for (int m = threadIdx.x; m < M; m += 64) {
            const uint32_t f = ent[m], gf = (f >> 21) & 0x3FFu;
            const double t = G[trans ? size_t(gf) * gdim + ge : size_t(ge) * gdim + gf];
            row[f & kAddrMask] += ((e ^ f) >> 31) ? -t : t;
        }
        __syncthreads();
    }
    for (int i = threadIdx.x; i < int(nstr); i += 64) H[I * nstr + i] = row[i];
}

constexpr int DN_TH = 512;

// S (+)= s C + Ha C + C Hb, C and S Na x Nb, Ha Na x Na the alpha operator, Hb Nb x Nb the transpose of the
// beta operator (null: no such term), in FP64 whatever the vectors' type. Block: 32 WT x 32 WT outputs, four waves of 16 WT x 16 WT for the even k-steps and
// four for the odd ones (two a SIMD: one's LDS reads and waits beside the other's products), k in chunks of
// 64 / WT through two LDS buffers, the next chunk's loads in
// flight during the products. A rows are padded by 2 doubles (to 34 and 66) and B rows by 16 (to 80 and 48), so
// that the half waves' operand reads hit 64 banks.
template <class T, int WT>
__global__ __launch_bounds__(DN_TH) void k_dense_apply(const T* __restrict__ C, T* __restrict__ S, int Na, int Nb,
                                                     const double* __restrict__ Ha, const double* __restrict__ Hb,
                                                     T scale, int add, const void* const* __restrict__ act,
                                                     const T* const* __restrict__ C_t, T* const* __restrict__ S_t,
                                                     const double* const* __restrict__ Ha_t,
                                                     const double* const* __restrict__ Hb_t) {
    constexpr int TL = 32 * WT, KC = 64 / WT, AS = KC + 2, BS = TL + 16, NL = TL * KC / DN_TH;  // NL: loads per operand
    extern __shared__ __attribute__((aligned(16))) double dsh[];
    double* const As = dsh;                // [2][TL][AS]
    double* const Bs = dsh + 2 * TL * AS;  // [2][KC][BS]
    if (act) {
        if (!act[blockIdx.z]) return;
        C = C_t[blockIdx.z];
        S = S_t[blockIdx.z];
        Ha = Ha_t ? Ha_t[blockIdx.z] : nullptr;
        Hb = Hb_t ? Hb_t[blockIdx.z] : nullptr;
    }
    const GLOBAL_MEM T* Cg = (const GLOBAL_MEM T*)C;
    const int r0 = blockIdx.y * TL, c0 = blockIdx.x * TL;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, cl = lane & 15, wr = ((wave >> 1) & 1) * 16 * WT, wcol = (wave & 1) * 16 * WT, kg = wave >> 2;
    d4 acc[WT][WT];
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j) acc[i][j] = d4{0.0, 0.0, 0.0, 0.0};
    // First rows of Ha against C, then rows of C against Hb: operands A (row length lda) and B (lda rows of
    // Nb). Rows and columns past the end are computed and not stored. The loads take a uniform base that
    // advances with k and a constant offset per lane, no vector arithmetic (FP64 products keep the vector
    // instructions out); only the last, ragged chunk clamps k and stores zeros on both sides.
    const int ak = tid & (KC - 1), ar = tid / KC, bc = tid & (TL - 1), bk = tid / TL;
    auto product = [&](auto a0, const GLOBAL_MEM char* A, auto b0, const GLOBAL_MEM char* B, const int K) {
        using TA = decltype(a0);
        using TB = decltype(b0);
        uint32_t oa[NL], ob[NL];  // bytes (the matrices are far below 4 GB)
#pragma unroll
        for (int u = 0; u < NL; ++u) {
            oa[u] = uint32_t((int64_t(min(r0 + ar + (DN_TH / KC) * u, Na - 1)) * K + ak) * sizeof(TA));
            ob[u] = uint32_t((int64_t(bk + (DN_TH / TL) * u) * Nb + min(c0 + bc, Nb - 1)) * sizeof(TB));
        }
        TA ra[NL];
        TB rb[NL];
        const int nq = (K + KC - 1) / KC, nfull = K / KC;
        auto load = [&](int q) {
            const GLOBAL_MEM char* ba = A + int64_t(q) * KC * sizeof(TA);
            const GLOBAL_MEM char* bb = B + int64_t(q) * KC * Nb * sizeof(TB);
            if (q < nfull) {
#pragma unroll
                for (int u = 0; u < NL; ++u) ra[u] = *reinterpret_cast<const GLOBAL_MEM TA*>(ba + oa[u]);
#pragma unroll
                for (int u = 0; u < NL; ++u) rb[u] = *reinterpret_cast<const GLOBAL_MEM TB*>(bb + ob[u]);
            } else {
                const int left = K - q * KC;
#pragma unroll
                for (int u = 0; u < NL; ++u)
                    ra[u] = *reinterpret_cast<const GLOBAL_MEM TA*>(ba + oa[u] - uint32_t(max(0, ak - (left - 1)) * int(sizeof(TA))));
#pragma unroll
                for (int u = 0; u < NL; ++u) {
                    const int back = max(0, bk + (DN_TH / TL) * u - (left - 1));
                    rb[u] = *reinterpret_cast<const GLOBAL_MEM TB*>(bb + ob[u] - uint32_t(back * Nb * int(sizeof(TB))));
                }
            }
        };
        auto store = [&](int q) {
            double* a = As + (q & 1) * (TL * AS) + ar * AS + ak;
            double* b = Bs + (q & 1) * (KC * BS) + bk * BS + bc;
            if (q < nfull) {
#pragma unroll
                for (int u = 0; u < NL; ++u) a[(DN_TH / KC) * u * AS] = double(ra[u]);
#pragma unroll
                for (int u = 0; u < NL; ++u) b[(DN_TH / TL) * u * BS] = double(rb[u]);
            } else {
                const int left = K - q * KC;
#pragma unroll
                for (int u = 0; u < NL; ++u) a[(DN_TH / KC) * u * AS] = ak < left ? double(ra[u]) : 0.0;
#pragma unroll
                for (int u = 0; u < NL; ++u) b[(DN_TH / TL) * u * BS] = bk + (DN_TH / TL) * u < left ? double(rb[u]) : 0.0;
            }
        };
        load(0);
        store(0);
        __syncthreads();
        for (int q = 0; q < nq; ++q) {
            if (q + 1 < nq) load(q + 1);
            const double* a = As + (q & 1) * (TL * AS) + (wr + cl) * AS + g + 4 * kg;
            const double* b = Bs + (q & 1) * (KC * BS) + (g + 4 * kg) * BS + wcol + cl;
            double av[KC / 8][WT], bv[KC / 8][WT];  // all operand reads ahead of the products
#pragma unroll
            for (int ks = 0; ks < KC / 8; ++ks) {
#pragma unroll
                for (int i = 0; i < WT; ++i) av[ks][i] = a[i * 16 * AS + ks * 8];
#pragma unroll
                for (int j = 0; j < WT; ++j) bv[ks][j] = b[ks * 8 * BS + j * 16];
            }
#pragma unroll
            for (int ks = 0; ks < KC / 8; ++ks)
#pragma unroll
                for (int i = 0; i < WT; ++i)
#pragma unroll
                    for (int j = 0; j < WT; ++j)
                        acc[i][j] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[ks][i], bv[ks][j], acc[i][j], 0, 0, 0);
            if (q + 1 < nq) store(q + 1);
            __syncthreads();
        }
    };
    const GLOBAL_MEM char* Cc = (const GLOBAL_MEM char*)C;
    if (Ha) product(0.0, (const GLOBAL_MEM char*)Ha, T(0), Cc, Na);
    if (Hb) product(T(0), Cc, 0.0, (const GLOBAL_MEM char*)Hb, Nb);
    // the odd k-steps' halves through LDS (the staging buffers are done with: last barrier of the product)
    double* const half = dsh + (wave & 3) * (WT * WT * 256);
    if (kg) {
#pragma unroll
        for (int i = 0; i < WT; ++i)
#pragma unroll
            for (int j = 0; j < WT; ++j)
#pragma unroll
                for (int v = 0; v < 4; ++v) half[((i * WT + j) * 4 + v) * 64 + lane] = acc[i][j][v];
    }
    __syncthreads();
    if (kg) return;
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[i][j][v] += half[((i * WT + j) * 4 + v) * 64 + lane];
    GLOBAL_MEM T* Sg = (GLOBAL_MEM T*)S;
#pragma unroll
    for (int i = 0; i < WT; ++i)
#pragma unroll
        for (int j = 0; j < WT; ++j)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const int r = r0 + wr + i * 16 + 4 * v + g, c = c0 + wcol + j * 16 + cl;  // f64 output row
                if (r >= Na || c >= Nb) continue;
                const int64_t x = int64_t(r) * Nb + c;
                const double y = acc[i][j][v] + double(scale) * double(Cg[x]);
                Sg[x] = T(add ? double(Sg[x]) + y : y);
            }
}

size_t lds_bytes(int tl, int kc) { return size_t(2) * (tl * (kc + 2) + kc * (tl + 16)) * sizeof(double); }
template <class K> void allow_lds(K kern, size_t sh) {
    HIPCHK(hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, int(sh)));
}

template <class T>
void launch(const T* C, T* S, int64_t Na, int64_t Nb, const double* Ha, const double* Hb, T scale, bool add, int nitem,
            const void* const* act, const T* const* C_t, T* const* S_t, const double* const* Ha_t,
            const double* const* Hb_t, hipStream_t st) {
    auto tiles = [&](int64_t t) { return ((Na + t - 1) / t) * ((Nb + t - 1) / t); };
    auto go = [&](auto kern, int tl, int kc) {
        const size_t sh = lds_bytes(tl, kc);
        if (!act) allow_lds(kern, sh);  // batched launches are captured: dense_same_prepare did it
        kern<<<dim3(unsigned((Nb + tl - 1) / tl), unsigned((Na + tl - 1) / tl), unsigned(nitem)), DN_TH, sh, st>>>(
            C, S, int(Na), int(Nb), Ha, Hb, scale, add ? 1 : 0, act, C_t, S_t, Ha_t, Hb_t);
        HIPCHK(hipGetLastError());
    };
    // 64 x 64 outputs a block once they fill half of the chip
    if (tiles(64) * nitem >= 128) go(k_dense_apply<T, 2>, 64, 32);
    else go(k_dense_apply<T, 1>, 32, 64);
}

}  // namespace

// Spaces whose operator is held densely: both spins with at most 924 strings (12 orbitals), 462 with FP32
// vectors. The product costs N^2 instead of the cliques' nK M^2 multiply-adds a column (2.2 times at 12
// orbitals, 2.9 at 13), but needs no intermediate, no transposes and one launch instead of seven. Both
// same-spin terms, dense against cliques (MI355X, FP64): 6 orbitals 7 / 26 us (4 us of them the timing
// events), 8: 10 / 31, 10: 14 / 41, 11: 23 / 60, 12: 101 / 122, 13 (1716 x 1716): 456 / 451; FP32 at 11
// orbitals 23 / 53 us, at 12 orbitals (in FP64 inside) 101 / 74.
// One column and no beta term (fully polarized electrons): the cliques need no transposes, and for many strings in
// small cliques their two launches beat a product of which a tile uses one column: 924 strings in cliques of 28 (12
// orbitals, 6 electrons) 20.7 against 23.6 us, 792 in 21: 19.7 / 21.8, 715 in 15: 18.2 / 20.9; but 792 in 36: 24.6 /
// 21.8, 560 in 10: 23.3 / 17.9, 495 in 15: 16.6 / 17.0.
bool dense_same_use(const SpinTables& a, const SpinTables& b, size_t w) {
    if (b.d == 0 && b.nstr == 1 && a.nstr > 600 && a.M <= 28) return false;
    const int64_t most = w == 8 ? 924 : 462;
    return a.nstr <= most && b.nstr <= most;
}

void dense_same_device(const SpinTables& sp, const double* d_g, int gdim, bool trans, double* d_h, hipStream_t st) {
    k_dense_same<<<unsigned(sp.nstr), 64, size_t(sp.nstr) * sizeof(double), st>>>(sp.clq.p, sp.M, sp.nstr, sp.own.p,
                                                                                 sp.nown, d_g, gdim, trans, d_h);
    HIPCHK(hipGetLastError());
}
void dense_same_batch(const SpinTables& sp, const double* const* g_t, int gdim, bool trans, double* const* h_t,
                      int nprob, hipStream_t st) {
    k_dense_same<<<dim3(unsigned(sp.nstr), unsigned(nprob)), 64, size_t(sp.nstr) * sizeof(double), st>>>(
        sp.clq.p, sp.M, sp.nstr, sp.own.p, sp.nown, nullptr, gdim, trans, nullptr, g_t, h_t);
    HIPCHK(hipGetLastError());
}
template <class T>
void dense_same_apply(const T* C, T* S, int64_t Na, int64_t Nb, const double* Ha, const double* Hb, T scale, bool add,
                      hipStream_t st) {
    launch<T>(C, S, Na, Nb, Ha, Hb, scale, add, 1, nullptr, nullptr, nullptr, nullptr, nullptr, st);
}
template void dense_same_apply<double>(const double*, double*, int64_t, int64_t, const double*, const double*, double,
                                       bool, hipStream_t);
template void dense_same_apply<float>(const float*, float*, int64_t, int64_t, const double*, const double*, float, bool,
                                      hipStream_t);
void dense_same_prepare() {
    allow_lds(k_dense_apply<double, 2>, lds_bytes(64, 32));
    allow_lds(k_dense_apply<double, 1>, lds_bytes(32, 64));
}
void dense_same_apply_batch(int64_t Na, int64_t Nb, int nitem, const void* const* act, const double* const* C_t,
                            double* const* S_t, const double* const* Ha_t, const double* const* Hb_t, hipStream_t st) {
    launch<double>(nullptr, nullptr, Na, Nb, nullptr, nullptr, 0.0, false, nitem, act, C_t, S_t, Ha_t, Hb_t, st);
}

}  // namespace fci
