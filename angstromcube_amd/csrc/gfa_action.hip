// HIP kernels of the Green-function action y = (H - E S) x on gfx950.
//
// Data: x, y real_t[nnzb][2][64][64] (block, re/im plane, target point i, right-hand side j).
// Columns j are independent in every term, so a thread owns one (j, plane) pair and all loads and
// stores of a wave are 512 B (FP64) / 256 B (FP32) contiguous rows.
//
// Three launches per action:
//   1. k_sho_project  c_img = sum over the blocks touched by an atom image of H(x)H(y)H(z) x
//                     (include/green_dyadic.hxx:112-288, SHOprj), sum-factorised, split into
//                     chunks of blocks whose partial sums are reduced in a fixed order;
//   2. k_sho_atoms    collect images -> atom with Bloch phases, multiply the atom matrix
//                     (h - E s) dVol on the matrix cores, broadcast back with conjugate phases
//                     (include/green_dyadic.hxx:600-852, SHOsum + SHOmul + SHOsum);
//   3. the local kernel, per (block, column slice): (V - E) x (include/green_potential.hxx:16-139) + the
//                     three finite-difference Laplacians (include/green_kinetic.hxx:24-329) + the SHO add-back
//                     of the atoms touching the block with numax <= 5 (include/green_dyadic.hxx:325-518),
//                     written once.  Two kinds, picked per plan and precision by the autotuner: k_local (LDS
//                     accumulator) and k_plane (register accumulator per z plane).  The slice is staged in
//                     LDS; neighbour blocks come through L2.  Images with numax 6, 7 are added afterwards by
//                     k_sho_add_wide.
#include "gfa_device.hpp"

#include <algorithm>
#include <map>
#include <mutex>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <type_traits>

namespace gfa {

namespace {

constexpr int NBLK = 2 * 64 * 64;  // elements of one block

#ifndef LOCAL_TILE
#define LOCAL_TILE 6   // xy tile edge (blocks) of the local kernel's processing order (5 to 7 measured best)
#endif

#define HIP_TRY(call)                                                              \
    do {                                                                           \
        hipError_t const e_ = (call);                                              \
        if (hipSuccess != e_) {                                                    \
            err = std::string(#call) + ": " + hipGetErrorString(e_);               \
            return 2;                                                              \
        }                                                                          \
    } while (0)

template <int L> struct Sho { static constexpr int n3 = ((L + 1) * (L + 2) * (L + 3)) / 6, n2 = ((L + 1) * (L + 2)) / 2; };

// ---------------------------------------------------------------------------------------------
// 1D Hermite-Gauss functions on the 4 grid points of a block, per direction
// (include/green_dyadic.hxx:33-107): xi = ((cube*4 + i4 + 0.5) h - a) / sigma,
// H0 = exp(-xi^2/2) inside the projection radius, H_{n+1} = xi H_n - n/2 H_{n-1}.
// xi^2 is exported in float: the 3D sphere mask is evaluated in float as in the reference.
// Evaluated without contraction so that xi^2 rounds as on the host.
// ---------------------------------------------------------------------------------------------
template <typename real_t>
__device__ __forceinline__ void hermite_1d(real_t (*H)[3][4], float (*xi2)[4], int t, int lmax,
                                           double const* apos, float const* cpos, double const* hgrid) {
#pragma clang fp contract(off)
    int const dir = t >> 2, i4 = t & 3;
    double const h = hgrid[dir];
    double const cube = cpos[dir];
    double const a = apos[dir];
    double const sig_inv = apos[3] * apos[3];
    double const R2 = hgrid[3] * hgrid[3];
    double const xi = sig_inv * ((cube * 4 + i4 + 0.5) * h - a);
    double const x2 = xi * xi;
    xi2[dir][i4] = float(x2);
    double const H0 = (x2 < R2) ? exp(-0.5 * x2) : 0.0;
    H[0][dir][i4] = real_t(H0);
    double hn = H0, hm = 0;
    for (int nu = 0; nu < lmax; ++nu) {
        double const hp = xi * hn - (0.5 * nu) * hm;
        H[nu + 1][dir][i4] = real_t(hp);
        hm = hn; hn = hp;
    }
}

// The Hermite functions of every (atom image, target row) pair that the projection and the add-back use, computed
// once per plan with hermite_1d itself: htab[slot][8][3][4] (FP64, numax <= 7), and in smask[slot] the points (bit
// (z * 4 + y) * 4 + x) inside the projection sphere, tested in float from xi^2.
__global__ __launch_bounds__(64) void k_hermite_table(double* __restrict__ htab, uint64_t* __restrict__ smask,
                                                      uint32_t const* __restrict__ slot_img,
                                                      uint32_t const* __restrict__ slot_row,
                                                      double const* __restrict__ image_pos,
                                                      int8_t const* __restrict__ image_lmax,
                                                      float const* __restrict__ row_pos, double hx, double hy,
                                                      double hz, double rproj) {
    uint32_t const sl = blockIdx.x;
    int const t = threadIdx.x;
    uint32_t const img = slot_img[sl], row = slot_row[sl];
    double const hgrid[4] = {hx, hy, hz, rproj};
    __shared__ float xi2[3][4];
    if (t < 12)
        hermite_1d<double>(reinterpret_cast<double (*)[3][4]>(htab + size_t(sl) * 96), xi2, t, image_lmax[img],
                           image_pos + 4 * size_t(img), row_pos + 4 * size_t(row), hgrid);
    __syncthreads();
    float const R2 = float(rproj * rproj);
    float const d2z = xi2[2][t >> 4] - R2;
    float const d2yz = xi2[1][(t >> 2) & 3] + d2z;
    float const d2 = xi2[0][t & 3] + d2yz;
    uint64_t const in = __ballot((d2z < 0) && (d2yz < 0) && (d2 < 0));
    if (t == 0) smask[sl] = in;
}

// stage the table entry of `slot` into the LDS array H[L+1][3][4] (real_t); no barrier
template <typename real_t>
__device__ __forceinline__ void stage_hermite(real_t (*H)[3][4], double const* __restrict__ htab, uint32_t slot, int L,
                                              int tid, int T) {
    double const* src = htab + size_t(slot) * 96;
    for (int e = tid; e < (L + 1) * 12; e += T) H[e / 12][(e % 12) / 4][e % 4] = real_t(src[e]);
}

// ---------------------------------------------------------------------------------------------
// 1. projection: one work item = (atom image, column, chunk of blocks); 128 threads = (j, plane)
// ---------------------------------------------------------------------------------------------
template <typename real_t, int L>
__global__ __launch_bounds__(128) void k_sho_project(
    real_t* __restrict__ partial, real_t const* __restrict__ x, ProjChunk const* __restrict__ chunks,
    uint32_t const* __restrict__ bucket, uint32_t const* __restrict__ chunk_coef,
    uint32_t const* __restrict__ prj_blocks, uint8_t const* __restrict__ col_active,
    double const* __restrict__ htab, uint64_t const* __restrict__ smask, uint32_t const* __restrict__ prj_slot) {
    __shared__ real_t H[L + 1][3][4];
    uint32_t const ich = bucket[blockIdx.x];
    ProjChunk const ch = chunks[ich];
    if (col_active && !col_active[ch.col]) return;  // a retired column group
    int const tid = threadIdx.x, j = tid & 63, p = tid >> 6;
    constexpr int n3 = Sho<L>::n3, n2 = Sho<L>::n2;
    real_t czyx[n3];
#pragma unroll
    for (int s = 0; s < n3; ++s) czyx[s] = 0;
    for (uint32_t b = ch.begin; b < ch.end; ++b) {
        uint32_t const inzb = prj_blocks[b];
        uint64_t const in = smask[prj_slot[b]];   // uniform
        __syncthreads();
        stage_hermite<real_t>(H, htab, prj_slot[b], L, tid, 128);
        __syncthreads();
        real_t const* xb = x + size_t(inzb) * NBLK + p * 4096 + j;
#pragma unroll
        for (int z = 0; z < 4; ++z) {
            uint32_t const inz = uint32_t(in >> (16 * z)) & 0xffff;
            if (inz) {
                // the 16 points of the plane are loaded together (unconditionally, all in the block) and the
                // sphere mask is applied as a select, so the loads are in flight at once
                real_t v[16];
#pragma unroll
                for (int k = 0; k < 16; ++k) v[k] = xb[64 * (z * 16 + k)];
                real_t byx[n2];
#pragma unroll
                for (int k = 0; k < n2; ++k) byx[k] = 0;
#pragma unroll
                for (int y = 0; y < 4; ++y) {
                    uint32_t const iny = (inz >> (4 * y)) & 15;
                    if (iny) {
                        real_t ax[L + 1];
#pragma unroll
                        for (int k = 0; k <= L; ++k) ax[k] = 0;
#pragma unroll
                        for (int xx = 0; xx < 4; ++xx) {
                            real_t const ps = ((iny >> xx) & 1) ? v[y * 4 + xx] : real_t(0);
#pragma unroll
                            for (int k = 0; k <= L; ++k) ax[k] += ps * H[k][0][xx];
                        }
#pragma unroll
                        for (int iy = 0; iy <= L; ++iy) {
                            int const iyx0 = (iy * (2 * L + 3 - iy)) >> 1;
                            real_t const hy_ = H[iy][1][y];
#pragma unroll
                            for (int ix = 0; ix <= L - iy; ++ix) byx[iyx0 + ix] += ax[ix] * hy_;
                        }
                    }
                }
                int s = 0;
#pragma unroll
                for (int iz = 0; iz <= L; ++iz) {
                    real_t const hz_ = H[iz][2][z];
#pragma unroll
                    for (int iy = 0; iy <= L - iz; ++iy) {
                        int const iyx0 = (iy * (2 * L + 3 - iy)) >> 1;
#pragma unroll
                        for (int ix = 0; ix <= L - iz - iy; ++ix) czyx[s++] += byx[iyx0 + ix] * hz_;
                    }
                }
            }
        }
    }
    real_t* out = partial + size_t(chunk_coef[ich]) * 128 + p * 64 + j;
#pragma unroll
    for (int s = 0; s < n3; ++s) out[size_t(s) * 128] = czyx[s];
}

// ---------------------------------------------------------------------------------------------
// 1b. projection on the matrix cores (the dense form): per block of the chunk, C[s][n] += sum_i P[s][i] X[i][n]
//     with P[s][i] = H_x[ix_s](x_i) H_y[iy_s](y_i) H_z[iz_s](z_i) inside the projection sphere (0 outside), i the 64
//     points, n = plane * 64 + column.  P is built in LDS per block, X comes straight from global memory as the
//     B operand.  4 waves; wave w owns the columns n = 32 w .. 32 w + 31 (two 16-column tiles) and every
//     16-coefficient tile.  Operand layout of the 16x16x4 MFMA (64 lanes): A[m][k] from lane m + 16 k, B[k][n]
//     from lane n + 16 k; accumulator r of a lane holds D[row][lane % 16] with row = 4 (lane / 16) + r in FP32 and
//     row = lane / 16 + 4 r in FP64 (measured on gfx950).
// ---------------------------------------------------------------------------------------------
template <typename real_t> struct Mfma;
template <> struct Mfma<float> {
    typedef float __attribute__((ext_vector_type(4))) acc_t;
    static __device__ __forceinline__ acc_t mac(float a, float b, acc_t c) {
        return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int kl, int r) { return 4 * kl + r; }
};
template <> struct Mfma<double> {
    typedef double __attribute__((ext_vector_type(4))) acc_t;
    static __device__ __forceinline__ acc_t mac(double a, double b, acc_t c) {
        return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
    }
    static __device__ __forceinline__ int row(int kl, int r) { return kl + 4 * r; }
};

template <typename real_t, int L>
__global__ __launch_bounds__(256) void k_sho_project_mfma(
    real_t* __restrict__ partial, real_t const* __restrict__ x, ProjChunk const* __restrict__ chunks,
    uint32_t const* __restrict__ bucket, uint32_t const* __restrict__ chunk_coef,
    uint32_t const* __restrict__ prj_blocks, uint8_t const* __restrict__ col_active,
    double const* __restrict__ htab, uint64_t const* __restrict__ smask, uint32_t const* __restrict__ prj_slot) {
    using acc_t = typename Mfma<real_t>::acc_t;
    constexpr int NC = Sho<L>::n3, MT = (NC + 15) / 16, NCP = 16 * MT;
    __shared__ real_t P[64 * NCP];           // [point][coefficient], zero beyond NC and outside the sphere
    __shared__ real_t H[L + 1][3][4];
    __shared__ uint16_t sxyz[NCP];           // coefficient s -> ix | iy << 4 | iz << 8
    uint32_t const ich = bucket[blockIdx.x];
    ProjChunk const ch = chunks[ich];
    if (col_active && !col_active[ch.col]) return;  // a retired column group
    int const tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (tid == 0) {
        int s = 0;
        for (int iz = 0; iz <= L; ++iz)
            for (int iy = 0; iy <= L - iz; ++iy)
                for (int ix = 0; ix <= L - iz - iy; ++ix) sxyz[s++] = uint16_t(ix | (iy << 4) | (iz << 8));
        for (; s < NCP; ++s) sxyz[s] = 0xFFFF;
    }
    acc_t acc[MT][2];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[mt][t] = acc_t{0, 0, 0, 0};
    int const p = w >> 1, jb = (w & 1) * 32 + (lane & 15), kl = lane >> 4;   // B operand: column jb (+16), row kl
    for (uint32_t b = ch.begin; b < ch.end; ++b) {
        uint32_t const inzb = prj_blocks[b];
        // the B operands of the whole block (16 steps of 4 points, 2 column tiles), issued before P is built
        real_t const* xb = x + size_t(inzb) * NBLK + p * 4096 + jb;
        real_t bv[16][2];
#pragma unroll
        for (int ks = 0; ks < 16; ++ks) {
            bv[ks][0] = xb[(ks * 4 + kl) * 64];
            bv[ks][1] = xb[(ks * 4 + kl) * 64 + 16];
        }
        __syncthreads();   // P of the previous block is no longer read
        uint64_t const in = smask[prj_slot[b]];   // uniform
        stage_hermite<real_t>(H, htab, prj_slot[b], L, tid, 256);
        __syncthreads();
        for (int e = tid; e < 64 * NCP; e += 256) {
            int const i = e / NCP, s = e % NCP;
            int const xx = i & 3, yy = (i >> 2) & 3, zz = i >> 4;
            uint16_t const c = sxyz[s];
            real_t v = 0;
            if (c != 0xFFFF && ((in >> i) & 1))
                v = H[c & 15][0][xx] * H[(c >> 4) & 15][1][yy] * H[c >> 8][2][zz];
            P[e] = v;
        }
        __syncthreads();
#pragma unroll
        for (int ks = 0; ks < 16; ++ks) {
#pragma unroll
            for (int mt = 0; mt < MT; ++mt) {
                real_t const av = P[(ks * 4 + kl) * NCP + mt * 16 + (lane & 15)];
                acc[mt][0] = Mfma<real_t>::mac(av, bv[ks][0], acc[mt][0]);
                acc[mt][1] = Mfma<real_t>::mac(av, bv[ks][1], acc[mt][1]);
            }
        }
    }
    real_t* out = partial + size_t(chunk_coef[ich]) * 128 + p * 64 + jb;
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            int const s = mt * 16 + Mfma<real_t>::row(kl, r);
            if (s < NC) {
                out[size_t(s) * 128] = acc[mt][0][r];
                out[size_t(s) * 128 + 16] = acc[mt][1][r];
            }
        }
}

// ---------------------------------------------------------------------------------------------
// 2. per (atom, column): collect images with phase, multiply (h - E s) dVol, broadcast with conjugate phase.
//    The 64 right-hand sides of a column group are independent, so a work-group takes JS of them for one (atom,
//    column): 1,024 threads collect the chunk partial sums into LDS (thread = one right-hand side of one coefficient,
//    both planes, and where few coefficients leave threads over, one of P parts of the chunk list), then the waves
//    multiply on the matrix cores.  h and s are real, so with the collected c = (c_re, c_im) the products t = h c and
//    u = s c are real contractions, [16 rows of h and s] x [nc] x [16 right-hand sides of both planes] per wave on the
//    FP64 16x16x4 MFMA (operand layout as in k_sho_project_mfma), and d = t - E u.
//    Bound by latency: a plan has few (atom, column) pairs, and one pair's chain (chunk list, partial sums, matrix)
//    is what a launch takes.  The chunks of a pair are therefore one list in memory, read ahead of the sums, the
//    wave's first matrix columns are loaded before the collection, and JS is small enough for four (two) work-groups
//    per pair.  Measured, against one work-group of 8 waves per pair on the vector ALUs that read chunk by chunk, then
//    with 512 threads without parts, then as it is: FP64 numax 5, 215 pairs: 212, 79, 79 us; numax 7, 16 pairs: 428, 47,
//    42 us; numax 2, 2 pairs of 13 images: 63, 16, 13 us; numax 3, 4 pairs: 18 -> 15 us; FP32 numax 5, 1,370 pairs:
//    309, 187, 157 us.  P follows from the coefficients (and the precision), not from JS, so that the order of a pair's
//    sum follows from its chunk list alone; the length of the chunks follows from the whole plan (device_upload_plan),
//    so between plans of different sizes a sum may differ by rounding.  KA = 4 keeps 1,024 threads within 128 VGPRs with all of the parts' loads (8: the same times).
// ---------------------------------------------------------------------------------------------
// one chunk of the projection partial sums of an (atom, column): its first coefficient row and its atom image
struct CollectEntry {
    uint32_t coef, img;
};

// adds U chunks from e0 on (those below e1) to the sum below; their loads are in flight together
template <typename real_t, int U>
__device__ __forceinline__ void collect_chunks(real_t const* __restrict__ partial,
                                               CollectEntry const* __restrict__ coll, uint32_t e0, uint32_t e1,
                                               double const* __restrict__ image_phase, int s, int j, double& ar,
                                               double& ai) {
    double vr[U], vi[U], pr[U], pi[U];
#pragma unroll
    for (int q = 0; q < U; ++q) {   // beyond the end: the last chunk again, not added
        CollectEntry const en = coll[min(e0 + q, e1 - 1)];
        real_t const* src = partial + (size_t(en.coef) + s) * 128 + j;
        vr[q] = double(src[0]);
        vi[q] = double(src[64]);
        pr[q] = image_phase[2 * en.img];
        pi[q] = image_phase[2 * en.img + 1];
    }
#pragma unroll
    for (int q = 0; q < U; ++q)
        if (e0 + q < e1) {
            ar += pr[q] * vr[q] - pi[q] * vi[q];
            ai += pr[q] * vi[q] + pi[q] * vr[q];
        }
}

// sum over the chunks e0 .. e1 - 1 of an (atom, column) of the partial sums of coefficient s at right-hand side j,
// each with the Bloch phase of its image, in list order
template <typename real_t>
__device__ __forceinline__ void collect_coefficient(real_t const* __restrict__ partial,
                                                    CollectEntry const* __restrict__ coll, uint32_t e0, uint32_t e1,
                                                    double const* __restrict__ image_phase, int s, int j, double& ar,
                                                    double& ai) {
    ar = ai = 0;
    uint32_t e = e0;
    for (; e + 8 < e1; e += 16) collect_chunks<real_t, 16>(partial, coll, e, e1, image_phase, s, j, ar, ai);
    if (e < e1) collect_chunks<real_t, 8>(partial, coll, e, e1, image_phase, s, j, ar, ai);
}

constexpr int ATOM_T = 1024;   // threads of k_sho_atoms

template <typename real_t, int JS>
__global__ __launch_bounds__(ATOM_T) void k_sho_atoms(
    real_t* __restrict__ dcoef, real_t const* __restrict__ partial, uint32_t const* __restrict__ pairs,
    uint32_t const* __restrict__ coll_start, CollectEntry const* __restrict__ coll,
    uint32_t const* __restrict__ sum_start, uint32_t const* __restrict__ sum_index,
    uint32_t const* __restrict__ image_starts,
    int8_t const* __restrict__ atom_lmax, double const* __restrict__ atom_mat,
    uint64_t const* __restrict__ atom_mat_off, double const* __restrict__ image_phase, uint32_t nCols,
    double const* __restrict__ E_col, uint8_t const* __restrict__ col_active) {
    using acc_t = typename Mfma<double>::acc_t;
    constexpr int NS = 64 / JS, NJ = JS / 16;   // slices per pair, 16-column tiles per plane
    constexpr int KA = 4;                       // k-steps (of 4 columns of h and s) loaded together
    extern __shared__ double cs[];              // [plane][16-column tile][coefficient, padded to 4][16]
    // the pairs with a block of the column near the atom: those of small truncation spheres see few of the atoms,
    // and the coefficients of the others are never read
    uint32_t const slice = blockIdx.x % NS, pair = pairs[blockIdx.x / NS], c = pair % nCols, a = pair / nCols;
    if (col_active && !col_active[c]) return;  // a retired column group
    uint32_t const e0 = coll_start[pair], e1 = coll_start[pair + 1];
    int const tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const n = lane & 15, kl = lane >> 4;
    int const L = atom_lmax[a];
    int const nc = ((L + 1) * (L + 2) * (L + 3)) / 6, kp = (nc + 3) & ~3, nks = kp / 4, nu = ((nc + 15) / 16) * NJ;
    double const* HS = atom_mat + atom_mat_off[a];  // [2][nc][nc]: h dVol, s dVol
    double const Er = E_col[2 * c], Ei = E_col[2 * c + 1];

    double ah[KA], as[KA];   // the wave's rows of h and s: A[m = n][k = ks * 4 + kl]
    auto load_rows = [&](int mt, int ks0) {
        int const i = mt * 16 + n;
#pragma unroll
        for (int q = 0; q < KA; ++q) {
            int const k = (ks0 + q) * 4 + kl;
            bool const in = i < nc && k < nc;
            int const at = in ? i * nc + k : 0;
            double const h = HS[at], sv = HS[nc * nc + at];
            ah[q] = in ? h : 0.0;
            as[q] = in ? sv : 0.0;
        }
    };
    if (w < nu) load_rows(w / NJ, 0);

    // few coefficients: the threads take P parts of the chunk list, summed in part order below
    constexpr int SLOTS = ATOM_T / (sizeof(real_t) == 8 ? 16 : 32);
    int P = 1;
    while (2 * P * kp <= SLOTS) P *= 2;
    uint32_t const per = (e1 - e0 + P - 1) / P;
    int const jl = tid % JS;
    for (int t = tid / JS; t < P * kp; t += ATOM_T / JS) {
        int const part = __builtin_amdgcn_readfirstlane(t / kp), s = t - part * kp;   // kp and the wave: multiples of 4
        uint32_t const p0 = min(e0 + part * per, e1), p1 = min(p0 + per, e1);
        double ar = 0, ai = 0;
        if (s < nc) collect_coefficient<real_t>(partial, coll, p0, p1, image_phase, s, slice * JS + jl, ar, ai);
        double* dst = cs + (size_t(part) * 2 * NJ * kp + (jl >> 4) * kp + s) * 16 + (jl & 15);
        dst[0] = ar;
        dst[NJ * kp * 16] = ai;
    }
    __syncthreads();
    if (P > 1) {
        for (int t = tid; t < 2 * JS * kp; t += ATOM_T) {
            double v = cs[t];
            for (int part = 1; part < P; ++part) v += cs[part * 2 * JS * kp + t];
            cs[t] = v;
        }
        __syncthreads();
    }

    uint32_t const k0 = sum_start[a], k1 = sum_start[a + 1];
    // at most 8 * NJ = ATOM_T / 64 tiles: one per wave.  The loop has one turn, but as straight-line code, with its first
    // load_rows no longer kept apart, the kernel is slower (FP32 numax 5, 1,370 pairs: by 6%; FP64 numax 7, 16 pairs: 5%)
    for (int u = w; u < nu; u += ATOM_T / 64) {
        int const mt = u / NJ, jt = u % NJ;
        acc_t tr = {0, 0, 0, 0}, ti = {0, 0, 0, 0}, ur = {0, 0, 0, 0}, ui = {0, 0, 0, 0};
        double const* cr = cs + jt * kp * 16 + n;
        double const* ci = cs + (NJ + jt) * kp * 16 + n;
        for (int ks0 = 0; ks0 < nks; ks0 += KA) {
            if (u != w || ks0 > 0) load_rows(mt, ks0);
#pragma unroll
            for (int q = 0; q < KA; ++q) {
                if (ks0 + q < nks) {   // uniform
                    int const k = (ks0 + q) * 4 + kl;
                    double const br = cr[k * 16], bi = ci[k * 16];
                    tr = Mfma<double>::mac(ah[q], br, tr);
                    ti = Mfma<double>::mac(ah[q], bi, ti);
                    ur = Mfma<double>::mac(as[q], br, ur);
                    ui = Mfma<double>::mac(as[q], bi, ui);
                }
            }
        }
        // d = t - E u (include/green_dyadic.hxx:800-819, src/green_function.cxx:97-98), then every image's share
        double dr[4], di[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            dr[r] = tr[r] - (Er * ur[r] - Ei * ui[r]);
            di[r] = ti[r] - (Er * ui[r] + Ei * ur[r]);
        }
        for (uint32_t k = k0; k < k1; ++k) {
            uint32_t const img = sum_index[k];
            double const ph_re = image_phase[2 * img], ph_im = -image_phase[2 * img + 1];
            real_t* dst = dcoef + (size_t(image_starts[img]) * nCols + c) * 128 + slice * JS + jt * 16 + n;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int const i = mt * 16 + Mfma<double>::row(kl, r);
                if (i < nc) {
                    dst[size_t(i) * nCols * 128] = real_t(ph_re * dr[r] - ph_im * di[r]);
                    dst[size_t(i) * nCols * 128 + 64] = real_t(ph_re * di[r] + ph_im * dr[r]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------------------------------------
// 3. local part of the action: one work-group per (block, slice of JW of the 64 columns), 8 JW threads, each
//    owning points of one (column, plane).  The slice is staged in LDS; neighbour blocks are read with
//    branch-free addressing (an absent neighbour reads a zero block) so that all loads of a line are in flight
//    together.
// ---------------------------------------------------------------------------------------------
// 16 bytes of y, stored past the caches' replacement order (non-temporal): the output of the local kernels is read
// by the next kernel only, so keeping it out of L2 leaves room there for the neighbour blocks of x
__device__ __forceinline__ void st_y16(float* p, float4 const& v) {
    typedef float f4v __attribute__((ext_vector_type(4)));
    f4v t; t[0] = v.x; t[1] = v.y; t[2] = v.z; t[3] = v.w;
    __builtin_nontemporal_store(t, reinterpret_cast<f4v*>(p));
}
__device__ __forceinline__ void st_y16(double* p, double2 const& v) {
    typedef double d2v __attribute__((ext_vector_type(2)));
    d2v t; t[0] = v.x; t[1] = v.y;
    __builtin_nontemporal_store(t, reinterpret_cast<d2v*>(p));
}

// word indices in a block header: block, column group, potential cell (-1: none), add-list range [ADD0, ADD1),
// then the neighbour codes [direction][side][k < NH] (>= 0 block, -1 absent, <= -2 periodic image -code - 2)
enum : int { IH_BLK = 0, IH_COL = 1, IH_VEFF = 2, IH_ADD0 = 3, IH_ADD1 = 4, IH_NBR = 5 };
template <int NH>
struct alignas(64) ItemHead {
    uint32_t w[NH == 1 ? 16 : 32];
    __device__ int32_t code(int d, int sd, int k) const { return int32_t(w[IH_NBR + (d * 2 + sd) * NH + k]); }
};

// one add-list entry: atom image, its numax, the Hermite slot of (image, target row), its first coefficient
struct AddEntry {
    uint32_t img, L, slot, coef0;
};

template <typename real_t>
struct LocalArgs {
    real_t* y;
    real_t const* x;
    real_t const* dcoef;
    real_t const* zero;      // one block of zeros
    uint32_t const* items;   // block headers in processing order (cache-aware), ItemHead<NH> each
    AddEntry const* add_entry;   // [add nnz]
    double const* V;
    uint32_t const* add_start;   // [nnzb + 1] add-list range of each block (the add-back kernels after the local one)
    uint16_t const* colindx;
    uint64_t nitems;         // blocks to process (all, or the active ones) listed in items
    uint32_t nCols;
    uint32_t per_xcd;        // work-items per XCD in the XCD-contiguous mapping
    double const* E_col;     // [nCols][2] energy of each column group
    double const* htab;      // Hermite functions per (image, row) slot
    uint64_t const* smask;   // points inside the projection sphere per slot
    double* dot;             // if set: [nnzb][re, im][64] bilinear products sum_i x[b][i][j] y[b][i][j] per block
    int add_local;           // 1: the local kernel adds the numax <= 5 images; 0: k_sho_add_mfma adds them after it
    real_t c8[3][5];         // 8th-order weights per direction
    real_t c16[3][9];        // 16th-order weights per direction
    int nh[3];               // neighbour blocks per side used in direction d (1 or 2)
    real_t cdiag;            // sum of the centre weights of the three directions
    double phase[3][2][2];
};

// sum over the SHO coefficients c[iz][iy][ix] (ix fastest, iz + iy + ix <= L) of one atom image at the 16
// points (y, x) of the z plane zq, v(y, x) = sum c H_x[ix](x) H_y[iy](y) H_z[iz](zq), handed to out(y, x, v).
// Contracted z first (one value H_z[iz](zq) per thread), then y and x row by row: (L+1)(L+2)(L+3)/6 +
// 4 (L+1)(L+2)/2 + 16 (L+1) FMAs.  All loops are unrolled, with a scheduling barrier after every z layer so that at
// most one layer of coefficients is loaded ahead (rolled layers with a run-time size cost a copy of all sums per
// layer: more moves than FMAs); ROLL keeps the row loop rolled (out must then accept a run-time row y).  TIGHT adds a
// barrier after every row, for callers that are held to fewer registers.
// dsrc points to coefficient 0 of this thread's (plane, column); consecutive coefficients are dstride apart.
template <typename real_t, int L, bool ROLL, bool TIGHT, typename Out>
__device__ __forceinline__ void sho_plane(real_t const (*H)[3][4], real_t const* __restrict__ dsrc, size_t dstride,
                                          int zq, Out&& out) {
    constexpr int n2 = ((L + 1) * (L + 2)) / 2;
    real_t c2[n2];   // [iy][ix] triangular, row iy starts at iy (2L + 3 - iy) / 2
#pragma unroll
    for (int k = 0; k < n2; ++k) c2[k] = 0;
    int t = 0;
#pragma unroll
    for (int iz = 0; iz <= L; ++iz) {
        real_t const hz = H[iz][2][zq];
#pragma unroll
        for (int iy = 0; iy <= L - iz; ++iy)
#pragma unroll
            for (int ix = 0; ix <= L - iz - iy; ++ix, ++t)
                c2[(iy * (2 * L + 3 - iy)) / 2 + ix] += dsrc[size_t(t) * dstride] * hz;
        __builtin_amdgcn_sched_barrier(0);
    }
    auto row = [&](int y) {
        real_t by[L + 1];
#pragma unroll
        for (int ix = 0; ix <= L; ++ix) by[ix] = 0;
#pragma unroll
        for (int iy = 0; iy <= L; ++iy) {
            real_t const hy = H[iy][1][y];
#pragma unroll
            for (int ix = 0; ix <= L - iy; ++ix) by[ix] += c2[(iy * (2 * L + 3 - iy)) / 2 + ix] * hy;
        }
#pragma unroll
        for (int xx = 0; xx < 4; ++xx) {
            real_t v = 0;
#pragma unroll
            for (int ix = 0; ix <= L; ++ix) v += by[ix] * H[ix][0][xx];
            out(y, xx, v);
        }
        if constexpr (TIGHT) __builtin_amdgcn_sched_barrier(0);
    };
    if constexpr (ROLL) {
#pragma unroll 1
        for (int y = 0; y < 4; ++y) row(y);
    } else {
#pragma unroll
        for (int y = 0; y < 4; ++y) row(y);
    }
}

// sho_plane for a run-time numax LMIN <= L <= LMAX
template <typename real_t, int LMIN, int LMAX, bool ROLL, bool TIGHT, typename Out>
__device__ __forceinline__ void sho_plane_any(real_t const (*H)[3][4], real_t const* __restrict__ dsrc, size_t dstride,
                                              int zq, int L, Out&& out) {
    if constexpr (LMIN < LMAX) {
        if (L == LMIN) sho_plane<real_t, LMIN, ROLL, TIGHT>(H, dsrc, dstride, zq, out);
        else sho_plane_any<real_t, LMIN + 1, LMAX, ROLL, TIGHT>(H, dsrc, dstride, zq, L, out);
    } else {
        sho_plane<real_t, LMAX, ROLL, TIGHT>(H, dsrc, dstride, zq, out);
    }
}

// SHO add-back of one atom image (numax L <= 5) into this thread's z plane zq of an accumulator in LDS whose points are
// ostride apart: ys[(zq*16 + y*4 + x) * ostride]; in: the points inside the projection sphere
template <typename real_t>
__device__ __forceinline__ void sho_add_atom(real_t* __restrict__ ys, int ostride, real_t const (*H)[3][4], uint64_t in,
                                             real_t const* __restrict__ dsrc, size_t dstride, int zq, int L) {
    sho_plane_any<real_t, 0, 5, true, false>(H, dsrc, dstride, zq, L, [&](int y, int xx, real_t v) {
        real_t& o = ys[(zq * 16 + y * 4 + xx) * ostride];
        o += ((in >> (zq * 16 + y * 4 + xx)) & 1) ? v : real_t(0);
    });
}

// SHO add-back of one atom image (LMIN <= numax <= LMAX) into 16 register accumulators (z plane zq of one column and
// plane); in: the plane's points inside the projection sphere (16 bits)
template <typename real_t, int LMIN, int LMAX, bool TIGHT = false>
__device__ __forceinline__ void sho_add_regs(real_t (&out)[16], real_t const (*H)[3][4], uint32_t in,
                                             real_t const* __restrict__ dsrc, size_t dstride, int zq, int L) {
    sho_plane_any<real_t, LMIN, LMAX, false, TIGHT>(H, dsrc, dstride, zq, L, [&](int y, int xx, real_t v) {
        out[y * 4 + xx] += ((in >> (y * 4 + xx)) & 1) ? v : real_t(0);
    });
}

// The images of a block's add list are taken in batches whose coefficients fit a buffer of CAP rows in LDS, so that a
// work-group pays one round trip to memory and two barriers per batch: with numax 2 four images, numax 3 two (CAP 56) or
// three (CAP 64), numax 4 and 5 one at a time.
constexpr int BATCH = 4;
template <typename real_t>
struct BatchHermite { real_t H[BATCH][6][3][4]; };

// stages the next images (numax <= 5) of the add list from entry b on (column group col, columns from c0 on) into cs
// [coefficient][plane][JW] and bh, for all T threads of the work-group (it contains two barriers, and the buffers are
// free before the first); returns the entry after the batch.  The k-th image of the batch with numax L <= 5 has its
// coefficients behind those of the images before it.
template <typename real_t, int JW, int T, int CAP>
__device__ __forceinline__ uint32_t stage_batch(LocalArgs<real_t> const& a, uint32_t b, uint32_t b1, uint32_t col,
                                                int c0, real_t* cs, BatchHermite<real_t>& bh) {
    typedef real_t __attribute__((ext_vector_type(16 / sizeof(real_t)))) vec_t;
    constexpr int VE = 16 / sizeof(real_t), VPR = JW / VE;   // 16-byte vectors per row
    constexpr int NV = (2 * CAP * VPR + T - 1) / T;          // of them per thread in a full buffer
    int const tid = threadIdx.x;
    uint32_t slot[BATCH], coef[BATCH], row0[BATCH + 1];      // uniform; rows: 2 per coefficient
    int n = 0;
    row0[0] = 0;
#pragma unroll
    for (int q = 0; q < BATCH; ++q) {
        bool take = false;
        uint32_t nc = 0;
        slot[q] = q ? slot[0] : 0;   // entries beyond the batch are loaded like the first, and not used
        coef[q] = q ? coef[0] : 0;
        for (; b < b1; ++b) {
            AddEntry const e = a.add_entry[b];
            if (e.L > 5) continue;   // added by k_sho_add_wide
            nc = ((e.L + 1) * (e.L + 2) * (e.L + 3)) / 6;
            take = row0[q] + 2 * nc <= 2 * CAP;
            if (take) { slot[q] = e.slot; coef[q] = e.coef0; }
            break;
        }
        row0[q + 1] = row0[q] + (take ? 2 * nc : 0);
        if (take) { ++b; ++n; }
    }
    uint32_t const rows = row0[BATCH];
    vec_t t[NV];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        uint32_t const v = k * T + tid, row = v / VPR, cv = v % VPR;   // row = coefficient * 2 + plane
        uint32_t base = coef[0], r0 = 0;
#pragma unroll
        for (int q = 1; q < BATCH; ++q)
            if (row >= row0[q] && row0[q + 1] > row0[q]) { base = coef[q]; r0 = row0[q]; }
        uint32_t const r = (row < rows) ? row - r0 : 0;   // beyond the batch: a row of it again, not stored
        t[k] = *reinterpret_cast<vec_t const*>(a.dcoef + (size_t(base + (r >> 1)) * a.nCols + col) * 128 + (r & 1) * 64 +
                                               c0 + cv * VE);
    }
    real_t h[BATCH];
#pragma unroll
    for (int q = 0; q < BATCH; ++q) h[q] = real_t(a.htab[size_t(slot[q]) * 96 + (tid < 72 ? tid : 0)]);
    __syncthreads();   // the buffers are no longer read
#pragma unroll
    for (int q = 0; q < BATCH; ++q)
        if (q < n && tid < 72) bh.H[q][tid / 12][(tid % 12) / 4][tid % 4] = h[q];
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        uint32_t const v = k * T + tid, row = v / VPR, cv = v % VPR;
        if (row < rows) *reinterpret_cast<vec_t*>(cs + row * JW + cv * VE) = t[k];
    }
    __syncthreads();
    return b;
}

// the atom images (numax <= 5) of add-list entries b0 .. b1 - 1, added to out: the z plane zq of this thread's column,
// which is column c0 + jl of plane p.  cs: LDS for CAP coefficients [coefficient][plane][JW].
// Contains barriers: every thread of the work-group calls it; after it cs may still be read by other threads.
template <typename real_t, int JW, int T, int CAP, bool TIGHT = false>
__device__ __forceinline__ void add_images(LocalArgs<real_t> const& a, uint32_t b0, uint32_t b1, uint32_t col, int c0,
                                           int p, int jl, int zq, real_t* cs, BatchHermite<real_t>& bh,
                                           real_t (&out)[16]) {
    for (uint32_t b = b0; b < b1;) {
        uint32_t const be = stage_batch<real_t, JW, T, CAP>(a, b, b1, col, c0, cs, bh);
        real_t const* c = cs + p * JW + jl;
        for (int q = 0; b < be; ++b) {
            AddEntry const e = a.add_entry[b];
            if (e.L > 5) continue;
            uint32_t const in = uint32_t(a.smask[e.slot] >> (16 * zq));
            sho_add_regs<real_t, 0, 5, TIGHT>(out, bh.H[q], in, c, 2 * JW, zq, int(e.L));
            c += ((e.L + 1) * (e.L + 2) * (e.L + 3)) / 6 * (2 * JW);
            ++q;
        }
    }
}

// value of a neighbour block at point e (a compile-time element offset from the uniform pointer b) and byte
// offset `off` (this thread's column and plane), with the Bloch phase of a periodic image applied:
// f x_p - (+/-) g x_other; off_o is the byte offset of the other plane.  Uniform base + immediate + 32-bit
// vector offset is the global load's own addressing mode: no per-load address arithmetic.
template <typename real_t, bool IMG>
__device__ __forceinline__ real_t nb_value(real_t const* __restrict__ b, int e, uint32_t off, uint32_t off_o,
                                           real_t fr, real_t fi) {
    char const* bb = reinterpret_cast<char const*>(b + e);
    real_t v = *reinterpret_cast<real_t const*>(bb + off);
    if (IMG) v = fr * v - fi * *reinterpret_cast<real_t const*>(bb + off_o);
    return v;
}

// acc += the off-centre finite-difference weights applied to a window w of 4 (2 NH + 1) values centred at c, of the
// 16th order if O16 (the centre weights of the three directions are applied together with the potential)
template <typename real_t, int NH, int NW, bool O16>
__device__ __forceinline__ void stencil(real_t& acc, LocalArgs<real_t> const& a, int d, real_t const (&w)[NW], int c) {
    if constexpr (O16) {
#pragma unroll
        for (int m = 1; m <= 8; ++m) {
            int const lo = c - m, hi = c + m;
            acc += a.c16[d][m] * (w[lo < 0 ? 0 : lo] + w[hi >= NW ? NW - 1 : hi]);
        }
    } else {
#pragma unroll
        for (int m = 1; m <= 4; ++m) acc += a.c8[d][m] * (w[c - m] + w[c + m]);
    }
}

// f(O16) with the order of direction d as a compile-time flag.  The branch (uniform) is taken once per pass: inside the
// unrolled loops over the points it cost the 16th-order kernels half of their time (3,180 blocks FP32: k_plane 249 ->
// 112 us, k_lines 242 -> 111)
template <int NH, typename real_t, typename Fn>
__device__ __forceinline__ void with_order(LocalArgs<real_t> const& a, int d, Fn&& f) {
    if constexpr (NH == 2) {
        if (a.nh[d] == 2) { f(std::true_type()); return; }
    }
    f(std::false_type());
}

// One work-group per (block, JW-column slice), 8*JW threads.  LDS holds the slice of the block
// (xs) and the output accumulator (ys); passes: potential, kinetic x, y, z, SHO add-back, store.
// In the kinetic passes a thread owns 4 lines (4 points each) of one (column, plane); neighbour
// values come straight from global memory with branch-free addressing (absent -> zero block).
template <typename real_t, int NH, bool IMG, int JW, int LB>
__global__ __launch_bounds__(8 * JW) void k_local(LocalArgs<real_t> a) {
    constexpr int T = 8 * JW;
    constexpr int NW = 4 * (2 * NH + 1);   // points in a line window
    constexpr int NSLICE = 64 / JW;
    __shared__ real_t xs[2 * 64 * JW];
    __shared__ real_t ys[2 * 64 * JW];
    __shared__ real_t H[6][3][4];

    uint64_t lin = blockIdx.x;
    if (a.per_xcd) lin = uint64_t(blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    // slice-major: all blocks of column slice 0 in processing order, then slice 1, ...; the neighbour slices
    // a work-group reads were then read shortly before by work-groups of the same XCD
    uint64_t const item = lin % a.nitems;
    int const slice = int(lin / a.nitems);
    if (slice >= NSLICE) return;  // uniform over the work-group
    ItemHead<NH> const h = reinterpret_cast<ItemHead<NH> const*>(a.items)[item];   // one scalar load
    uint64_t const blk = h.w[IH_BLK];
    int const tid = threadIdx.x;

    // stage this column slice of the block in LDS with 16-byte loads
    using vec_t = typename std::conditional<sizeof(real_t) == 8, double2, float4>::type;
    constexpr int VE = 16 / sizeof(real_t), VPR = JW / VE;  // vectors per row
    {
        real_t const* src = a.x + blk * NBLK + slice * JW;
#pragma unroll
        for (int k = 0; k < 2 * 64 * VPR / T; ++k) {
            int const v = k * T + tid, row = v / VPR, cv = v % VPR;
            *reinterpret_cast<vec_t*>(xs + row * JW + cv * VE) = *reinterpret_cast<vec_t const*>(src + row * 64 + cv * VE);
        }
    }
    __syncthreads();

    // ---- potential: ys = (V - E) x ----
    {
        int32_t const iv = int32_t(h.w[IH_VEFF]);
        real_t const vm = (iv >= 0) ? real_t(1) : real_t(0);
        double const* Vb = a.V + uint64_t(iv >= 0 ? iv : 0) * 64;
        uint32_t const colE = h.w[IH_COL];
        real_t const E_re = real_t(a.E_col[2 * colE]), E_im = real_t(a.E_col[2 * colE + 1]);
#pragma unroll
        for (int k = 0; k < 2 * 64 * JW / T; ++k) {
            int const e = k * T + tid, jl = e % JW, row = e / JW, p = row >> 6, i = row & 63;
            real_t const Vim = E_im * real_t(1 - 2 * p);
            ys[e] = (real_t(Vb[i]) * vm + (a.cdiag - E_re)) * xs[e] + Vim * xs[((1 - p) * 64 + i) * JW + jl];
        }
    }

    // thread's (column, plane, line group) in the kinetic passes
    int const jl = tid % JW, p = (tid / JW) & 1, lg = tid / (2 * JW);   // lg in 0..3
    int const j = slice * JW + jl;
    real_t* ysp = ys + p * 64 * JW + jl;
    real_t const* xsp = xs + p * 64 * JW + jl;
    // byte offsets of this thread's column in its plane and in the other plane (neighbour loads)
    uint32_t const boff_p = uint32_t(p * 4096 + j) * sizeof(real_t), boff_o = uint32_t((1 - p) * 4096 + j) * sizeof(real_t);

#pragma unroll
    for (int d = 0; d < 3; ++d) {
        int const stride = (d == 0) ? 1 : ((d == 1) ? 4 : 16);
        // neighbour blocks of this direction (uniform over the work-group)
        real_t const* nb[2][NH];
        real_t fr[2][NH], fi[2][NH];
#pragma unroll
        for (int sd = 0; sd < 2; ++sd)
#pragma unroll
            for (int k = 0; k < NH; ++k) {
                int32_t const code = h.code(d, sd, k);
                uint64_t const idx = (code >= 0) ? uint64_t(code) : uint64_t(code <= -2 ? -code - 2 : 0);
                nb[sd][k] = (code == -1) ? a.zero : a.x + idx * NBLK;
                bool const img = IMG && (code <= -2);
                fr[sd][k] = img ? real_t(a.phase[d][sd][0]) : real_t(1);
                fi[sd][k] = img ? real_t(a.phase[d][sd][1]) * real_t(1 - 2 * p) : real_t(0);
            }
        __syncthreads();  // the previous pass has finished its updates of ys
#pragma unroll 1
        for (int rb = 0; rb < 4; rb += LB) {
        real_t w[LB][NW];
        int il0[LB];
#pragma unroll
        for (int r = 0; r < LB; ++r) {
            int const line = lg * 4 + rb + r;  // 0..15
            int i0;
            if (d == 0) i0 = line * 4;                               // line = z*4 + y
            else if (d == 1) i0 = (line >> 2) * 16 + (line & 3);     // line = z*4 + x
            else i0 = line;                                          // line = y*4 + x
            il0[r] = i0;
            uint32_t const line_p = boff_p + uint32_t(i0) * (64 * sizeof(real_t));   // first point of the line
            uint32_t const line_o = boff_o + uint32_t(i0) * (64 * sizeof(real_t));
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int const i = i0 + q * stride;
                w[r][4 * NH + q] = xsp[i * JW];
#pragma unroll
                for (int k = 0; k < NH; ++k) {
                    w[r][4 * (NH - 1 - k) + q] = nb_value<real_t, IMG>(nb[0][k], q * stride * 64, line_p, line_o, fr[0][k], fi[0][k]);
                    w[r][4 * (NH + 1 + k) + q] = nb_value<real_t, IMG>(nb[1][k], q * stride * 64, line_p, line_o, fr[1][k], fi[1][k]);
                }
            }
        }
        // off-centre weights only: the centre weights are applied with the potential
        with_order<NH>(a, d, [&](auto o16) {
#pragma unroll
            for (int r = 0; r < LB; ++r)
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    real_t t = 0;
                    stencil<real_t, NH, NW, decltype(o16)::value>(t, a, d, w[r], 4 * NH + q);
                    ysp[(il0[r] + q * stride) * JW] += t;
                }
        });
        }  // line batches
    }

    // ---- SHO add-back of the atom images (numax <= 5) touching this block; the coefficients of
    //      each image are staged in the LDS buffer of the block, which is free after the kinetic passes ----
    uint32_t const b0 = h.w[IH_ADD0], b1 = h.w[IH_ADD1];
    if (a.add_local && b1 > b0) {
        uint32_t const col = h.w[IH_COL];
        int const zq = lg;  // threads (jl, p, zq) own the z plane zq
        real_t* cs = xs;    // [nc][2][JW]
        for (uint32_t b = b0; b < b1; ++b) {
            AddEntry const e = a.add_entry[b];
            int const L = int(e.L);
            if (L > 5) continue;  // done by k_sho_add_wide
            int const nc = ((L + 1) * (L + 2) * (L + 3)) / 6;
            __syncthreads();
            stage_hermite<real_t>(H, a.htab, e.slot, L, tid, T);
            {
                real_t const* src = a.dcoef + (size_t(e.coef0) * a.nCols + col) * 128 + slice * JW;
                for (int v = tid; v < 2 * nc * VPR; v += T) {
                    int const row = v / VPR, cv = v % VPR;  // row = coefficient*2 + plane
                    *reinterpret_cast<vec_t*>(cs + row * JW + cv * VE) =
                        *reinterpret_cast<vec_t const*>(src + size_t(row >> 1) * a.nCols * 128 + (row & 1) * 64 + cv * VE);
                }
            }
            __syncthreads();
            sho_add_atom<real_t>(ysp, JW, H, a.smask[e.slot], cs + p * JW + jl, 2 * JW, zq, L);
        }
    }
    __syncthreads();

    // ---- store the slice with 16-byte stores ----
    {
        real_t* dst = a.y + blk * NBLK + slice * JW;
#pragma unroll
        for (int k = 0; k < 2 * 64 * VPR / T; ++k) {
            int const v = k * T + tid, row = v / VPR, cv = v % VPR;
            st_y16(dst + row * 64 + cv * VE, *reinterpret_cast<vec_t const*>(ys + row * JW + cv * VE));
        }
    }
    if (a.dot) {   // (x, y) = sum_i x_i y_i (no conjugation) per column, x re-read from global memory (L2)
        int const jl = tid % JW, grp = tid / JW;   // 8 groups of 8 points
        int const j = slice * JW + jl;
        real_t const* xb = a.x + blk * NBLK + j;
        double re = 0, im = 0;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            int const i = grp * 8 + q;
            double const yr = ys[i * JW + jl], yi = ys[(64 + i) * JW + jl];
            double const xr = xb[i * 64], xi = xb[4096 + i * 64];
            re += xr * yr - xi * yi;
            im += xr * yi + xi * yr;
        }
        __syncthreads();   // xs is free: the partial sums of the 8 groups
        double* red = reinterpret_cast<double*>(xs);
        red[(grp * 2 + 0) * JW + jl] = re;
        red[(grp * 2 + 1) * JW + jl] = im;
        __syncthreads();
        if (tid < JW) {
            double sr = 0, si = 0;
            for (int g = 0; g < 8; ++g) { sr += red[(g * 2) * JW + tid]; si += red[(g * 2 + 1) * JW + tid]; }
            a.dot[(blk * 2 + 0) * 64 + slice * JW + tid] = sr;
            a.dot[(blk * 2 + 1) * 64 + slice * JW + tid] = si;
        }
    }
}


// z-direction stencil for the thread's plane ZQ: window positions z' = ZQ - 4 NH .. ZQ + 4 NH along z at every
// (y, x); inside the block from LDS (own plane from registers), outside from the neighbour blocks
template <typename real_t, int NH, bool IMG, int JW, int ZQ, bool O16>
__device__ __forceinline__ void z_pass(LocalArgs<real_t> const& a, real_t (&acc)[16], real_t const (&own)[16],
                                       real_t const* __restrict__ xsp, real_t const* const (&nb)[2][NH],
                                       real_t const (&fr)[2][NH], real_t const (&fi)[2][NH], uint32_t boff_p, uint32_t boff_o) {
    constexpr int NWZ = 8 * NH + 1;   // z' = ZQ - 4 NH .. ZQ + 4 NH
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        real_t w[NWZ];
#pragma unroll
        for (int m = 0; m < NWZ; ++m) {
            int const z = ZQ - 4 * NH + m;   // z' relative to this block
            if (z == ZQ) w[m] = own[k];
            else if (z >= 0 && z < 4) w[m] = xsp[(z * 16 + k) * JW];
            else if (z < 0) {
                int const kb = (-z - 1) / 4, zz = z + 4 * (kb + 1);
                w[m] = nb_value<real_t, IMG>(nb[0][kb], (zz * 16 + k) * 64, boff_p, boff_o, fr[0][kb], fi[0][kb]);
            } else {
                int const kb = (z - 4) / 4, zz = z - 4 * (kb + 1);
                w[m] = nb_value<real_t, IMG>(nb[1][kb], (zz * 16 + k) * 64, boff_p, boff_o, fr[1][kb], fi[1][kb]);
            }
        }
        stencil<real_t, NH, NWZ, O16>(acc[k], a, 2, w, 4 * NH);
    }
}

// neighbour blocks of blk in direction d, NH per side: base pointers (an absent neighbour reads the zero block)
// and the Bloch phase of a periodic image as (fr, fi) for plane p (fr = 1, fi = 0 otherwise)
template <typename real_t, int NH, bool IMG>
__device__ __forceinline__ void neighbours(LocalArgs<real_t> const& a, int d, ItemHead<NH> const& h, int p,
                                           real_t const* (&nb)[2][NH], real_t (&fr)[2][NH], real_t (&fi)[2][NH]) {
#pragma unroll
    for (int sd = 0; sd < 2; ++sd)
#pragma unroll
        for (int k = 0; k < NH; ++k) {
            int32_t const code = h.code(d, sd, k);
            uint64_t const idx = (code >= 0) ? uint64_t(code) : uint64_t(code <= -2 ? -code - 2 : 0);
            nb[sd][k] = (code == -1) ? a.zero : a.x + idx * NBLK;
            bool const img = IMG && (code <= -2);
            fr[sd][k] = img ? real_t(a.phase[d][sd][0]) : real_t(1);
            fi[sd][k] = img ? real_t(a.phase[d][sd][1]) * real_t(1 - 2 * p) : real_t(0);
        }
}

// (V - E) x at the thread's 16 points (z plane zq of one column, plane p): own = x of plane p there, xso = x of the
// other plane in LDS (row stride JW), vz = the potential at the 16 points (0 where the block has no potential
// cell), E the column group's energy, whose imaginary part couples the two planes; the centre weights of the
// three finite-difference directions are applied here as well
template <typename real_t, int JW>
__device__ __forceinline__ void plane_potential(LocalArgs<real_t> const& a, double const (&vz)[16], double E_re,
                                                double E_im, int p, int zq, real_t const (&own)[16],
                                                real_t const* xso, real_t (&acc)[16]) {
    real_t const Vim = real_t(E_im) * real_t(1 - 2 * p);
    real_t const dg = a.cdiag - real_t(E_re);
#pragma unroll
    for (int k = 0; k < 16; ++k) acc[k] = (real_t(vz[k]) + dg) * own[k] + Vim * xso[(zq * 16 + k) * JW];
}

// kinetic x and y at the thread's 16 points: the lines of plane zq along x (the rows y) and along y (the columns
// x) through this block and NH neighbour blocks on each side, the neighbours straight from global memory.  zq is
// uniform within the wave, so the plane's offset goes into the (scalar) base pointers.
template <typename real_t, int NH, bool IMG>
__device__ __forceinline__ void plane_xy(LocalArgs<real_t> const& a, ItemHead<NH> const& h, int p, int zq,
                                         uint32_t boff_p, uint32_t boff_o, real_t const (&own)[16], real_t (&acc)[16]) {
    constexpr int NW = 4 * (2 * NH + 1);
#pragma unroll
    for (int d = 0; d < 2; ++d) {
        real_t const* nb[2][NH];
        real_t fr[2][NH], fi[2][NH];
        neighbours<real_t, NH, IMG>(a, d, h, p, nb, fr, fi);
        int const zqu = __builtin_amdgcn_readfirstlane(zq);
        real_t const* nbz[2][NH];
#pragma unroll
        for (int sd = 0; sd < 2; ++sd)
#pragma unroll
            for (int kk = 0; kk < NH; ++kk) nbz[sd][kk] = nb[sd][kk] + zqu * 16 * 64;
        with_order<NH>(a, d, [&](auto o16) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            real_t w[NW];   // the line through this block and NH neighbour blocks on each side
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int const k = (d == 0) ? (r * 4 + q) : (q * 4 + r);   // point of the plane on the line
                int const e = k * 64;   // plane zq is in the base pointers
#pragma unroll
                for (int kk = 0; kk < NH; ++kk) {
                    w[4 * (NH - 1 - kk) + q] = nb_value<real_t, IMG>(nbz[0][kk], e, boff_p, boff_o, fr[0][kk], fi[0][kk]);
                    w[4 * (NH + 1 + kk) + q] = nb_value<real_t, IMG>(nbz[1][kk], e, boff_p, boff_o, fr[1][kk], fi[1][kk]);
                }
                w[4 * NH + q] = own[k];
            }
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                int const k = (d == 0) ? (r * 4 + q) : (q * 4 + r);
                stencil<real_t, NH, NW, decltype(o16)::value>(acc[k], a, d, w, 4 * NH + q);
            }
        }
        });
    }
}

// The end of a register-plane kernel for one block slice: the SHO add-back of the atom images (numax <= 5)
// touching the block (add-list entries b0 .. b1 - 1, column group col), the store of the thread's 16 points and,
// if a.dot is set, the bilinear product (x, y) of every column of the slice.  cs is LDS of at least 2 * 56 * JW
// elements of its own (the coefficients of one image at a time, then the partial sums of the product); xsp and
// xso point to this thread's column of x in the LDS copy of the slice (its plane and the other one), which stays
// intact, so that x is not held in registers across the add-back.  Contains work-group barriers: every thread of
// the work-group calls it.
template <typename real_t, int JW>
__device__ __forceinline__ void plane_finish(LocalArgs<real_t> const& a, uint64_t blk, uint32_t col, uint32_t b0,
                                             uint32_t b1, int slice, int p, int zq, int jl, real_t (&acc)[16],
                                             real_t const* xsp, real_t const* xso, real_t* cs,
                                             BatchHermite<real_t>& bh) {
    constexpr int T = 8 * JW;
    int const tid = threadIdx.x, j = slice * JW + jl;
    if (a.add_local)   // zq is uniform within a wave
        add_images<real_t, JW, T, 56>(a, b0, b1, col, slice * JW, p, jl, __builtin_amdgcn_readfirstlane(zq), cs, bh, acc);

    real_t* dst = a.y + blk * NBLK + size_t(p * 4096 + j) + size_t(zq * 16) * 64;
#pragma unroll
    for (int k = 0; k < 16; ++k) __builtin_nontemporal_store(acc[k], &dst[size_t(k) * 64]);   // y is not re-read here
    if (a.dot) {
        // (x, y) = sum_i x_i y_i per column: plane 0 holds x_r, y_r (+ x_i from LDS), plane 1 x_i, y_i (+ x_r):
        // Re = sum x_r y_r - sum x_i y_i, Im = sum x_i y_r + sum x_r y_i
        real_t re_t = 0, im_t = 0;   // 16 products in the vector precision, then summed in FP64
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            re_t += xsp[(zq * 16 + k) * JW] * acc[k];
            im_t += xso[(zq * 16 + k) * JW] * acc[k];
        }
        double re = re_t, im = im_t;
        if (p == 1) re = -re;
        __syncthreads();   // cs is free
        double* red = reinterpret_cast<double*>(cs);   // [zq][p][re, im][JW]
        red[((zq * 2 + p) * 2 + 0) * JW + jl] = re;
        red[((zq * 2 + p) * 2 + 1) * JW + jl] = im;
        __syncthreads();
        if (tid < JW) {
            double sr = 0, si = 0;
            for (int g = 0; g < 8; ++g) { sr += red[(g * 2 + 0) * JW + tid]; si += red[(g * 2 + 1) * JW + tid]; }
            a.dot[(blk * 2 + 0) * 64 + slice * JW + tid] = sr;
            a.dot[(blk * 2 + 1) * 64 + slice * JW + tid] = si;
        }
    }
}

// Register-plane variant of the local kernel: one work-group per (block, JW-column slice), 8 JW threads; thread
// (jl, p, zq) owns the 16 points of z plane zq of column j = slice JW + jl, plane p, and accumulates potential,
// kinetic x, y, z and the SHO add-back in registers.  LDS holds the block slice (read by the z-stencil, the
// imaginary part of the potential and the bilinear product of the epilogue) and, apart, the coefficients of the
// add-back, so that x need not stay in registers across the add-back (95 VGPRs instead of 124 in FP32).  zq is
// uniform within a wave (2 JW >= 64), so the z-stencil is specialised per plane.
template <typename real_t, int NH, bool IMG, int JW>
__global__ __launch_bounds__(8 * JW) void k_plane(LocalArgs<real_t> a) {
    static_assert(2 * JW >= 64, "zq must be uniform within a wave");
    constexpr int T = 8 * JW;
    constexpr int NSLICE = 64 / JW;
    __shared__ real_t xs[2 * 64 * JW];
    __shared__ __align__(16) real_t cs[2 * 56 * JW];   // add-back coefficients (numax <= 5), then the (x, y) sums
    __shared__ BatchHermite<real_t> bh;

    uint64_t lin = blockIdx.x;
    if (a.per_xcd) lin = uint64_t(blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    // slice-major: all blocks of column slice 0 in processing order, then slice 1, ...; the neighbour slices
    // a work-group reads were then read shortly before by work-groups of the same XCD
    uint64_t const item = lin % a.nitems;
    int const slice = int(lin / a.nitems);
    if (slice >= NSLICE) return;  // uniform over the work-group
    ItemHead<NH> const h = reinterpret_cast<ItemHead<NH> const*>(a.items)[item];   // one scalar load
    uint64_t const blk = h.w[IH_BLK];
    int const tid = threadIdx.x;

    using vec_t = typename std::conditional<sizeof(real_t) == 8, double2, float4>::type;
    constexpr int VE = 16 / sizeof(real_t), VPR = JW / VE;
    {
        real_t const* src = a.x + blk * NBLK + slice * JW;
#pragma unroll
        for (int k = 0; k < 2 * 64 * VPR / T; ++k) {
            int const v = k * T + tid, row = v / VPR, cv = v % VPR;
            *reinterpret_cast<vec_t*>(xs + row * JW + cv * VE) = *reinterpret_cast<vec_t const*>(src + row * 64 + cv * VE);
        }
    }
    int const jl = tid % JW, p = (tid / JW) & 1, zq = tid / (2 * JW);
    // the potential at the thread's plane and the energy, loaded (scalar: zq is uniform within a wave) together
    // with the slice
    double vz[16];
    {
        int32_t const iv = int32_t(h.w[IH_VEFF]);
        double const* Vb = a.V + uint64_t(iv >= 0 ? iv : 0) * 64 + __builtin_amdgcn_readfirstlane(zq) * 16;
#pragma unroll
        for (int k = 0; k < 16; ++k) {
            double const v = Vb[k];   // in bounds also without a cell (row 0)
            vz[k] = (iv >= 0) ? v : 0.0;
        }
    }
    double const E_re = a.E_col[2 * h.w[IH_COL]], E_im = a.E_col[2 * h.w[IH_COL] + 1];
    __syncthreads();

    int const j = slice * JW + jl;
    real_t const* xsp = xs + p * 64 * JW + jl;
    real_t const* xso = xs + (1 - p) * 64 * JW + jl;
    // byte offsets of this thread's column in its plane and in the other plane (neighbour loads)
    uint32_t const boff_p = uint32_t(p * 4096 + j) * sizeof(real_t), boff_o = uint32_t((1 - p) * 4096 + j) * sizeof(real_t);

    real_t own[16], acc[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) own[k] = xsp[(zq * 16 + k) * JW];

    plane_potential<real_t, JW>(a, vz, E_re, E_im, p, zq, own, xso, acc);
    plane_xy<real_t, NH, IMG>(a, h, p, zq, boff_p, boff_o, own, acc);
    {
        real_t const* nb[2][NH];
        real_t fr[2][NH], fi[2][NH];
        neighbours<real_t, NH, IMG>(a, 2, h, p, nb, fr, fi);
        with_order<NH>(a, 2, [&](auto o16) {
            constexpr bool O = decltype(o16)::value;
            switch (zq) {
                case 0: z_pass<real_t, NH, IMG, JW, 0, O>(a, acc, own, xsp, nb, fr, fi, boff_p, boff_o); break;
                case 1: z_pass<real_t, NH, IMG, JW, 1, O>(a, acc, own, xsp, nb, fr, fi, boff_p, boff_o); break;
                case 2: z_pass<real_t, NH, IMG, JW, 2, O>(a, acc, own, xsp, nb, fr, fi, boff_p, boff_o); break;
                default: z_pass<real_t, NH, IMG, JW, 3, O>(a, acc, own, xsp, nb, fr, fi, boff_p, boff_o); break;
            }
        });
    }

    plane_finish<real_t, JW>(a, blk, h.w[IH_COL], h.w[IH_ADD0], h.w[IH_ADD1], slice, p, zq, jl, acc, xsp, xso, cs,
                             bh);
}

// ---------------------------------------------------------------------------------------------
// Line variant of the local kernel (kind 2).  One work-group per (block, JW-column slice).  A lane owns
// CPL = 16 / sizeof(real_t) adjacent columns of one plane, so that every global load and store moves 16 bytes per
// lane.  Thread (cq, p, l) owns line l = 0..15 of plane p in each direction: the x-line (y, z) = (l % 4, l / 4),
// the y-line (x, z) and the z-line (x, y) of the same two indices.  Every neighbour value the three stencils need
// is loaded once per work-group, straight into registers, and all of them are issued before the first stencil;
// the block's own y- and z-lines come from the LDS copy of the slice.  The y and z stencil sums meet the x-line
// accumulator (potential, x stencil, SHO add-back) in a second LDS buffer.
// ---------------------------------------------------------------------------------------------
template <typename real_t>
struct alignas(16) Lane {   // the 16 bytes of adjacent columns a lane owns at one point
    static constexpr int n = 16 / sizeof(real_t);
    real_t v[n];
};

__device__ __forceinline__ Lane<float> ld16(float const* p) {
    float4 const t = *reinterpret_cast<float4 const*>(p);
    return Lane<float>{{t.x, t.y, t.z, t.w}};
}
__device__ __forceinline__ Lane<double> ld16(double const* p) {
    double2 const t = *reinterpret_cast<double2 const*>(p);
    return Lane<double>{{t.x, t.y}};
}
__device__ __forceinline__ void st16(float* p, Lane<float> const& v) {
    *reinterpret_cast<float4*>(p) = float4{v.v[0], v.v[1], v.v[2], v.v[3]};
}
__device__ __forceinline__ void st16(double* p, Lane<double> const& v) {
    *reinterpret_cast<double2*>(p) = double2{v.v[0], v.v[1]};
}
template <typename real_t>
__device__ __forceinline__ void st16_nt(real_t* p, Lane<real_t> const& v) {   // non-temporal, for y
    if constexpr (sizeof(real_t) == 4) st_y16(p, float4{v.v[0], v.v[1], v.v[2], v.v[3]});
    else st_y16(p, double2{v.v[0], v.v[1]});
}
// 16 bytes at element e of the uniform base b plus the lane's byte offset off (the load's own addressing mode)
template <typename real_t>
__device__ __forceinline__ Lane<real_t> ldv(real_t const* __restrict__ b, int e, uint32_t off) {
    return ld16(reinterpret_cast<real_t const*>(reinterpret_cast<char const*>(b + e) + off));
}

// acc[q] += the off-centre stencil of direction d at point q of a line, for every column of the lane: the window
// is the own line (centre) and NH neighbour lines on each side (w[side][k][q], k = 0 nearest)
template <typename real_t, int NH>
__device__ __forceinline__ void line_stencil(Lane<real_t> (&acc)[4], LocalArgs<real_t> const& a, int d,
                                             Lane<real_t> const (&own)[4], Lane<real_t> const (&w)[2][NH][4]) {
    constexpr int NW = 4 * (2 * NH + 1);
    with_order<NH>(a, d, [&](auto o16) {
#pragma unroll
    for (int c = 0; c < Lane<real_t>::n; ++c) {
        real_t win[NW];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            win[4 * NH + q] = own[q].v[c];
#pragma unroll
            for (int k = 0; k < NH; ++k) {
                win[4 * (NH - 1 - k) + q] = w[0][k][q].v[c];
                win[4 * (NH + 1 + k) + q] = w[1][k][q].v[c];
            }
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
            stencil<real_t, NH, NW, decltype(o16)::value>(acc[q].v[c], a, d, win, 4 * NH + q);
    }
    });
}

// one z layer of sho_xline: the M = L - iz triangle of coefficients (iy + ix <= M, ix fastest) times
// H_z[iz](z) H_y[iy](y), accumulated into t[column][ix]
template <typename real_t, int L, int M>
__device__ __forceinline__ void xline_layer(real_t (&t)[Lane<real_t>::n][L + 1], real_t const* cs, int cstride,
                                            real_t hz, real_t const (*H)[3][4], int y) {
    int s = 0;
#pragma unroll
    for (int iy = 0; iy <= M; ++iy) {
        real_t const hzy = hz * H[iy][1][y];
#pragma unroll
        for (int ix = 0; ix <= M - iy; ++ix, ++s) {
            Lane<real_t> const cv = ld16(cs + s * cstride);
#pragma unroll
            for (int c = 0; c < Lane<real_t>::n; ++c) t[c][ix] += cv.v[c] * hzy;
        }
    }
}

// SHO add-back of one atom image (numax L) into the x-line (y, z) of a lane: the coefficients c[iz][iy][ix]
// (ix fastest) are contracted with H_z(z) H_y(y) first, t[ix], then t with H_x at the 4 points of the line; in: the
// line's points inside the projection sphere (4 bits).  The z layers run in a rolled loop, so that one layer of
// coefficients at a time is loaded ahead (unrolled, the kernel takes 256 VGPRs).
// cs points to coefficient 0 of the lane's plane and first column; consecutive coefficients are cstride apart.
template <typename real_t, int L>
__device__ __forceinline__ void sho_xline(Lane<real_t> (&acc)[4], real_t const (*H)[3][4], uint32_t in, real_t const* cs,
                                          int cstride, int y, int z) {
    constexpr int CPL = Lane<real_t>::n;
    real_t t[CPL][L + 1];
#pragma unroll
    for (int c = 0; c < CPL; ++c)
#pragma unroll
        for (int ix = 0; ix <= L; ++ix) t[c][ix] = 0;
#pragma unroll 1
    for (int iz = 0; iz <= L; ++iz) {
        real_t const hz = H[iz][2][z];
        switch (L - iz) {
            case 0: xline_layer<real_t, L, 0>(t, cs, cstride, hz, H, y); break;
            case 1: if constexpr (L >= 1) xline_layer<real_t, L, 1>(t, cs, cstride, hz, H, y); break;
            case 2: if constexpr (L >= 2) xline_layer<real_t, L, 2>(t, cs, cstride, hz, H, y); break;
            case 3: if constexpr (L >= 3) xline_layer<real_t, L, 3>(t, cs, cstride, hz, H, y); break;
            case 4: if constexpr (L >= 4) xline_layer<real_t, L, 4>(t, cs, cstride, hz, H, y); break;
            default: if constexpr (L >= 5) xline_layer<real_t, L, 5>(t, cs, cstride, hz, H, y); break;
        }
        cs += ((L - iz + 1) * (L - iz + 2)) / 2 * cstride;
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        bool const inside = (in >> q) & 1;
#pragma unroll
        for (int c = 0; c < CPL; ++c) {
            real_t v = 0;
#pragma unroll
            for (int ix = 0; ix <= L; ++ix) v += t[c][ix] * H[ix][0][q];
            acc[q].v[c] += inside ? v : real_t(0);
        }
    }
}

// the neighbour lines of direction d (NH blocks per side) of the lane's line starting at point i0, plane p and
// first column j0, into w, without the Bloch phase of periodic images (phase_lines)
template <typename real_t, int NH>
__device__ __forceinline__ void load_lines(LocalArgs<real_t> const& a, int d, ItemHead<NH> const& h, int p, int i0,
                                           int j0, Lane<real_t> (&w)[2][NH][4]) {
    int const stride = (d == 0) ? 1 : ((d == 1) ? 4 : 16);
    uint32_t const off = uint32_t(p * 4096 + i0 * 64 + j0) * sizeof(real_t);
#pragma unroll
    for (int sd = 0; sd < 2; ++sd)
#pragma unroll
        for (int k = 0; k < NH; ++k) {
            int32_t const code = h.code(d, sd, k);
            uint64_t const idx = (code >= 0) ? uint64_t(code) : uint64_t(code <= -2 ? -code - 2 : 0);
            real_t const* nb = (code == -1) ? a.zero : a.x + idx * NBLK;
#pragma unroll
            for (int q = 0; q < 4; ++q) w[sd][k][q] = ldv(nb, q * stride * 64, off);
        }
}

// the Bloch phase of the periodic-image neighbours of direction d (uniform over the work-group) on their loaded lines,
// f x_p - (+/-) g x_other: the same line of the other plane is in the lane LQ away, so nothing more is loaded
template <typename real_t, int NH, int LQ>
__device__ __forceinline__ void phase_lines(LocalArgs<real_t> const& a, int d, ItemHead<NH> const& h, int p,
                                            Lane<real_t> (&w)[2][NH][4]) {
#pragma unroll
    for (int sd = 0; sd < 2; ++sd)
#pragma unroll
        for (int k = 0; k < NH; ++k)
            if (h.code(d, sd, k) <= -2) {
                real_t const fr = real_t(a.phase[d][sd][0]), fi = real_t(a.phase[d][sd][1]) * real_t(1 - 2 * p);
#pragma unroll
                for (int q = 0; q < 4; ++q)
#pragma unroll
                    for (int c = 0; c < Lane<real_t>::n; ++c) {
                        real_t const o = __shfl_xor(w[sd][k][q].v[c], LQ, 64);
                        w[sd][k][q].v[c] = fr * w[sd][k][q].v[c] - fi * o;
                    }
            }
}

// PF: directions whose neighbour lines are issued before the first barrier (3: all; 2: x and y, z after the x
// stencil; 1: x, then y after the x stencil and z after the y stencil) -- loads in flight against occupancy.
// The 8th-order shapes without images and with PF 2 (in FP64 that of 16 columns) are held to 128 VGPRs (4 waves per
// SIMD; FP32, 158k blocks: 3,347 us against 3,616 with 154 VGPRs and 3 waves); with image phases the shuffles push
// every 8th-order shape past 168, so those are held to 168 (3 waves, 3 to 6 spills; at 128 they spill 53).  Measured, FP64,
// 16 columns, 2 directions: 512 blocks at a k-point 49 -> 32 us, 1,024 blocks 87 -> 57, 6,144 blocks 705 -> 368 against
// loading the other plane's lines as well; 45,896 blocks without images 2,118 -> 2,050 us from loading the potential
// before the barrier.  16th order: unbounded (184 VGPRs; held to 168, 11,474 blocks FP64 take 941 us instead of 829).
template <typename real_t, int NH, bool IMG, int JW, int PF>
constexpr bool lines_four_waves() {
    return NH == 1 && !IMG && PF == 2 && (sizeof(real_t) == 4 || JW == 16);
}
template <typename real_t, int NH, bool IMG, int JW, int PF>
__global__ __launch_bounds__((JW / Lane<real_t>::n) * 32,
                             (lines_four_waves<real_t, NH, IMG, JW, PF>() ? 4 : (IMG && NH == 1) ? 3 : 1))
void k_lines(LocalArgs<real_t> a) {
    using L16 = Lane<real_t>;
    constexpr bool W4 = lines_four_waves<real_t, NH, IMG, JW, PF>();
    constexpr int CPL = L16::n, LQ = JW / CPL, T = LQ * 32;
    constexpr int NSLICE = 64 / JW;
    __shared__ __align__(16) real_t xs[2 * 64 * JW];   // the slice [plane][point][column]
    __shared__ __align__(16) real_t ya[2 * 64 * JW];   // y + z stencil sums; then the coefficients of a batch of images
    __shared__ BatchHermite<real_t> bh;

    uint64_t lin = blockIdx.x;
    if (a.per_xcd) lin = uint64_t(blockIdx.x & 7) * a.per_xcd + (blockIdx.x >> 3);
    uint64_t const item = lin % a.nitems;   // slice-major, as in k_plane
    int const slice = int(lin / a.nitems);
    if (slice >= NSLICE) return;  // uniform over the work-group
    ItemHead<NH> const h = reinterpret_cast<ItemHead<NH> const*>(a.items)[item];   // one scalar load
    uint64_t const blk = h.w[IH_BLK];
    int const tid = threadIdx.x, cq = tid % LQ, p = (tid / LQ) & 1, l = tid / (2 * LQ);
    int const la = l & 3, lb = l >> 2;
    int const jc = cq * CPL, j0 = slice * JW + jc;
    // first points of the lines: x-line (y, z) = (la, lb), y-line (x, z) = (la, lb), z-line (x, y) = (la, lb)
    int const ix0 = lb * 16 + la * 4, iy0 = lb * 16 + la, iz0 = lb * 4 + la;

    L16 wx[2][NH][4], wy[2][NH][4], wz[2][NH][4];   // neighbour lines per direction
    load_lines<real_t, NH>(a, 0, h, p, ix0, j0, wx);
    if constexpr (PF >= 2) load_lines<real_t, NH>(a, 1, h, p, iy0, j0, wy);
    if constexpr (PF >= 3) load_lines<real_t, NH>(a, 2, h, p, iz0, j0, wz);
    // own x-line, to registers and to the LDS copy of the slice
    L16 own[4];
    {
        real_t const* src = a.x + blk * NBLK + p * 4096 + j0;
#pragma unroll
        for (int q = 0; q < 4; ++q) own[q] = ld16(src + (ix0 + q) * 64);
#pragma unroll
        for (int q = 0; q < 4; ++q) st16(xs + (p * 64 + ix0 + q) * JW + jc, own[q]);
    }
    // the potential on the x-line and the energy are loaded with the slice, before the barrier
    int32_t const iv = int32_t(h.w[IH_VEFF]);
    Lane<double> const V01 = ldv(a.V + uint64_t(iv >= 0 ? iv : 0) * 64, 0, uint32_t(ix0) * 8);
    Lane<double> const V23 = ldv(a.V + uint64_t(iv >= 0 ? iv : 0) * 64, 2, uint32_t(ix0) * 8);
    real_t const E_re = real_t(a.E_col[2 * h.w[IH_COL]]), E_im = real_t(a.E_col[2 * h.w[IH_COL] + 1]);
    __syncthreads();

    // ---- potential and x stencil on the x-line ----
    L16 acc[4];
    {
        L16 oth[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) oth[q] = ld16(xs + ((1 - p) * 64 + ix0 + q) * JW + jc);
        real_t const vm = (iv >= 0) ? real_t(1) : real_t(0);
        double const Vb[4] = {V01.v[0], V01.v[1], V23.v[0], V23.v[1]};
        real_t const Vim = E_im * real_t(1 - 2 * p);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            real_t const dg = real_t(Vb[q]) * vm + (a.cdiag - E_re);
#pragma unroll
            for (int c = 0; c < CPL; ++c) acc[q].v[c] = dg * own[q].v[c] + Vim * oth[q].v[c];
        }
        if (IMG) phase_lines<real_t, NH, LQ>(a, 0, h, p, wx);
        line_stencil<real_t, NH>(acc, a, 0, own, wx);
    }
    if constexpr (PF < 2) load_lines<real_t, NH>(a, 1, h, p, iy0, j0, wy);
    if constexpr (PF == 2) load_lines<real_t, NH>(a, 2, h, p, iz0, j0, wz);

    // ---- y stencil on the y-line, into ya ----
    {
        L16 o[4], s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[q] = ld16(xs + (p * 64 + iy0 + 4 * q) * JW + jc);
#pragma unroll
            for (int c = 0; c < CPL; ++c) s[q].v[c] = 0;
        }
        if (IMG) phase_lines<real_t, NH, LQ>(a, 1, h, p, wy);
        line_stencil<real_t, NH>(s, a, 1, o, wy);
#pragma unroll
        for (int q = 0; q < 4; ++q) st16(ya + (p * 64 + iy0 + 4 * q) * JW + jc, s[q]);
    }
    if constexpr (PF < 2) load_lines<real_t, NH>(a, 2, h, p, iz0, j0, wz);
    __syncthreads();
    // ---- z stencil on the z-line, added into ya ----
    {
        L16 o[4], s[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            o[q] = ld16(xs + (p * 64 + iz0 + 16 * q) * JW + jc);
            s[q] = ld16(ya + (p * 64 + iz0 + 16 * q) * JW + jc);
        }
        if (IMG) phase_lines<real_t, NH, LQ>(a, 2, h, p, wz);
        line_stencil<real_t, NH>(s, a, 2, o, wz);
#pragma unroll
        for (int q = 0; q < 4; ++q) st16(ya + (p * 64 + iz0 + 16 * q) * JW + jc, s[q]);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        L16 const s = ld16(ya + (p * 64 + ix0 + q) * JW + jc);
#pragma unroll
        for (int c = 0; c < CPL; ++c) acc[q].v[c] += s.v[c];
    }

    // ---- SHO add-back of the atom images (numax <= 5) touching the block; coefficients staged in ya ----
    if (a.add_local && h.w[IH_ADD1] > h.w[IH_ADD0]) {
        uint32_t const b1 = h.w[IH_ADD1], col = h.w[IH_COL];
        if constexpr (sizeof(real_t) == 4) {
            // FP32: for the add-back a thread takes a z plane of ONE column, as in k_plane, and the sums meet the x-lines
            // in ya.  Contracted for a whole plane an image costs 236 FMAs per 16 points at numax 5, for x-lines of
            // several columns 400 (158k blocks: 3,843 -> 3,347 us; without any add-back 2,893).  In FP64 the plane
            // of a column needs 202 VGPRs, or spills at 128.
            int const jl = tid % JW, pp = (tid / JW) & 1, zt = tid / (2 * JW);
            int const zq = JW >= 32 ? __builtin_amdgcn_readfirstlane(zt) : zt;   // uniform within a wave from 32 columns
            real_t out[16];
#pragma unroll
            for (int k = 0; k < 16; ++k) out[k] = 0;
            add_images<real_t, JW, T, 64, W4>(a, h.w[IH_ADD0], b1, col, slice * JW, pp, jl, zq, ya, bh, out);
            __syncthreads();   // the coefficients are no longer read
#pragma unroll
            for (int k = 0; k < 16; ++k) ya[(pp * 64 + zq * 16 + k) * JW + jl] = out[k];
            __syncthreads();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                L16 const s = ld16(ya + (p * 64 + ix0 + q) * JW + jc);
#pragma unroll
                for (int c = 0; c < CPL; ++c) acc[q].v[c] += s.v[c];
            }
        } else {
            for (uint32_t b = h.w[IH_ADD0]; b < b1;) {
                uint32_t const be = stage_batch<real_t, JW, T, 64>(a, b, b1, col, slice * JW, ya, bh);
                real_t const* cs = ya + p * JW + jc;
                for (int q = 0; b < be; ++b) {
                    AddEntry const e = a.add_entry[b];
                    if (e.L > 5) continue;
                    uint32_t const in = uint32_t(a.smask[e.slot] >> ix0) & 15;
                    switch (e.L) {
                        case 0: sho_xline<real_t, 0>(acc, bh.H[q], in, cs, 2 * JW, la, lb); break;
                        case 1: sho_xline<real_t, 1>(acc, bh.H[q], in, cs, 2 * JW, la, lb); break;
                        case 2: sho_xline<real_t, 2>(acc, bh.H[q], in, cs, 2 * JW, la, lb); break;
                        case 3: sho_xline<real_t, 3>(acc, bh.H[q], in, cs, 2 * JW, la, lb); break;
                        case 4: sho_xline<real_t, 4>(acc, bh.H[q], in, cs, 2 * JW, la, lb); break;
                        default: sho_xline<real_t, 5>(acc, bh.H[q], in, cs, 2 * JW, la, lb); break;
                    }
                    cs += ((e.L + 1) * (e.L + 2) * (e.L + 3)) / 6 * (2 * JW);
                    ++q;
                }
            }
        }
    }

    // ---- store the x-line ----
    {
        real_t* dst = a.y + blk * NBLK + p * 4096 + j0;
#pragma unroll
        for (int q = 0; q < 4; ++q) st16_nt(dst + (ix0 + q) * 64, acc[q]);
    }
    if (a.dot) {
        // (x, y) = sum_i x_i y_i per column: plane 0 holds x_r, y_r (+ x_i), plane 1 x_i, y_i (+ x_r):
        // Re = sum x_r y_r - sum x_i y_i, Im = sum x_i y_r + sum x_r y_i; 4 products in the vector precision,
        // then FP64 over the 32 lines and planes of the work-group in a fixed order
        L16 re_v, im_v;   // x of both planes at the x-line from the LDS copy of the slice
#pragma unroll
        for (int c = 0; c < CPL; ++c) re_v.v[c] = im_v.v[c] = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            L16 const xp = ld16(xs + (p * 64 + ix0 + q) * JW + jc), xo = ld16(xs + ((1 - p) * 64 + ix0 + q) * JW + jc);
#pragma unroll
            for (int c = 0; c < CPL; ++c) {
                re_v.v[c] += xp.v[c] * acc[q].v[c];
                im_v.v[c] += xo.v[c] * acc[q].v[c];
            }
        }
#pragma unroll
        for (int c = 0; c < CPL; ++c) re_v.v[c] = (p == 1) ? -re_v.v[c] : re_v.v[c];
        // through LDS, as re and im of [line and plane][column]: thread (column, re or im, part) sums 1 / PARTS of the
        // 32 lines and planes in FP64, then the first 2 JW threads the parts; as shuffles within a wave this
        // took 48 of 64 bits per thread in FP32 (inside a solve, 6,144 blocks with images 94.9 -> 86.3 us, 19,764 blocks
        // without 310 -> 294; FP64, 1,024 blocks with images 50.2 -> 49.0)
        constexpr int PARTS = T / (2 * JW), PER = 32 / PARTS;
        __syncthreads();   // xs and ya are free
        real_t* red = ya + (l * 2 + p) * (2 * JW) + jc;
        st16(red, re_v);
        st16(red + JW, im_v);
        __syncthreads();
        int const cc = tid % (2 * JW), part = tid / (2 * JW);   // cc < JW: re, otherwise im
        double sum = 0;
#pragma unroll
        for (int k = 0; k < PER; ++k) sum += double(ya[(part * PER + k) * (2 * JW) + cc]);
        double* const tot = reinterpret_cast<double*>(xs);   // [part][re, im][JW]
        tot[part * (2 * JW) + cc] = sum;
        __syncthreads();
        if (tid < 2 * JW) {
            sum = 0;
#pragma unroll
            for (int k = 0; k < PARTS; ++k) sum += tot[k * (2 * JW) + tid];
            a.dot[(blk * 2 + tid / JW) * 64 + slice * JW + tid % JW] = sum;
        }
    }
}

// SHO add-back on the matrix cores (the dense form), after the local kernel: for every block touched by atom images
// with numax <= 5, y[b][n][i] += sum_img sum_s P_img[i][s] D_img[s][n] (i the 64 points, n = plane * 64 + column,
// s the coefficients padded to 64).  One work-group per block; 4 waves, wave w owns the columns n = 32 w .. 32 w + 31
// and all four 16-point tiles.  P (the A operand, zero outside the sphere and beyond the coefficients) is built in
// LDS per image; the coefficients D (the B operand) are read from global memory.  Operand layout as in
// k_sho_project_mfma.
template <typename real_t>
__global__ __launch_bounds__(256) void k_sho_add_mfma(LocalArgs<real_t> a, uint32_t const* __restrict__ blocks,
                                                      uint8_t const* __restrict__ col_active) {
    using acc_t = typename Mfma<real_t>::acc_t;
    constexpr int NCP = 64;
    __shared__ real_t P[64 * NCP];   // [point][coefficient]
    __shared__ real_t H[6][3][4];
    __shared__ uint16_t sxyz[NCP];   // coefficient s -> ix | iy << 4 | iz << 8 of the current image's numax
    uint32_t const blk = blocks[blockIdx.x];
    uint32_t const col = a.colindx[blk];
    if (col_active && !col_active[col]) return;
    int const tid = threadIdx.x, lane = tid & 63, w = tid >> 6, kl = lane >> 4;
    acc_t acc[4][2];
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int t = 0; t < 2; ++t) acc[mt][t] = acc_t{0, 0, 0, 0};
    int const nb0 = 32 * w + (lane & 15);   // B operand column of tile 0 (tile 1: + 16)
    for (uint32_t b = a.add_start[blk]; b < a.add_start[blk + 1]; ++b) {
        AddEntry const e = a.add_entry[b];
        int const L = int(e.L);
        if (L > 5) continue;   // added by k_sho_add_wide
        int const nc = ((L + 1) * (L + 2) * (L + 3)) / 6;
        __syncthreads();   // P of the previous image is no longer read
        uint64_t const in = a.smask[e.slot];
        stage_hermite<real_t>(H, a.htab, e.slot, L, tid, 256);
        if (tid == 0) {
            int q = 0;
            for (int iz = 0; iz <= L; ++iz)
                for (int iy = 0; iy <= L - iz; ++iy)
                    for (int ix = 0; ix <= L - iz - iy; ++ix) sxyz[q++] = uint16_t(ix | (iy << 4) | (iz << 8));
            for (; q < NCP; ++q) sxyz[q] = 0xFFFF;
        }
        __syncthreads();
        for (int e = tid; e < 64 * NCP; e += 256) {
            int const i = e / NCP, c = e % NCP;
            int const xx = i & 3, yy = (i >> 2) & 3, zz = i >> 4;
            uint16_t const code = sxyz[c];
            real_t v = 0;
            if (code != 0xFFFF && ((in >> i) & 1))
                v = H[code & 15][0][xx] * H[(code >> 4) & 15][1][yy] * H[code >> 8][2][zz];
            P[e] = v;
        }
        __syncthreads();
        real_t const* dsrc = a.dcoef + (size_t(e.coef0) * a.nCols + col) * 128 + nb0;
        size_t const dstride = size_t(a.nCols) * 128;
        int const nks = (nc + 3) / 4;
        for (int ks = 0; ks < nks; ++ks) {
            int const sk = ks * 4 + kl;
            real_t const b0v = sk < nc ? dsrc[size_t(sk) * dstride] : real_t(0);
            real_t const b1v = sk < nc ? dsrc[size_t(sk) * dstride + 16] : real_t(0);
#pragma unroll
            for (int mt = 0; mt < 4; ++mt) {
                real_t const av = P[(mt * 16 + (lane & 15)) * NCP + ks * 4 + kl];
                acc[mt][0] = Mfma<real_t>::mac(av, b0v, acc[mt][0]);
                acc[mt][1] = Mfma<real_t>::mac(av, b1v, acc[mt][1]);
            }
        }
    }
    // y += acc: point mt * 16 + row, column n of tile t
    real_t* yb = a.y + size_t(blk) * NBLK;
#pragma unroll
    for (int mt = 0; mt < 4; ++mt)
#pragma unroll
        for (int t = 0; t < 2; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                int const i = mt * 16 + Mfma<real_t>::row(kl, r), n = nb0 + 16 * t;
                real_t& o = yb[(n >> 6) * 4096 + i * 64 + (n & 63)];
                o += acc[mt][t][r];
            }
}

// SHO add-back of the atom images with numax 6 or 7, y += P d, on the blocks listed in blocks[], after the local kernel
// (which adds numax <= 5).  One work-group of 8 JS threads per (block, JS columns): thread (j, p, zq) holds the 16
// points of z plane zq of one column and plane of y in registers, and the block's wide images are added one after the
// other from LDS copies of their coefficients, so that no two work-groups update the same values and y is read and
// written once.  JS fills 128-byte lines.
template <typename real_t>
__global__ __launch_bounds__(1024 / sizeof(real_t)) void k_sho_add_wide(LocalArgs<real_t> a,
                                                                        uint32_t const* __restrict__ blocks,
                                                                        uint8_t const* __restrict__ col_active) {
    typedef real_t __attribute__((ext_vector_type(16 / sizeof(real_t)))) vec_t;
    constexpr int JS = 128 / sizeof(real_t), T = 8 * JS, NS = 64 / JS, VE = 16 / sizeof(real_t), VPR = JS / VE;
    constexpr int NCMAX = Sho<7>::n3;
    constexpr int NV = (2 * NCMAX * VPR + T - 1) / T;   // 16-byte vectors of coefficients per thread
    __shared__ __align__(16) real_t cs[2 * NCMAX * JS];   // [coefficient][plane][JS]
    __shared__ real_t H[8][3][4];
    uint32_t const blk = blocks[blockIdx.x / NS];
    int const slice = blockIdx.x % NS;
    uint32_t const col = a.colindx[blk];
    if (col_active && !col_active[col]) return;
    int const tid = threadIdx.x, jl = tid % JS, p = (tid / JS) & 1, zq = tid / (2 * JS);
    real_t* yb = a.y + size_t(blk) * NBLK + p * 4096 + zq * 1024 + slice * JS + jl;
    real_t acc[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) acc[k] = yb[k * 64];
    for (uint32_t b = a.add_start[blk]; b < a.add_start[blk + 1]; ++b) {
        AddEntry const e = a.add_entry[b];
        int const L = int(e.L);
        if (L <= 5) continue;   // added by the local kernel
        int const rows = ((L + 1) * (L + 2) * (L + 3)) / 3;
        vec_t t[NV];
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            int const v = k * T + tid, row = v / VPR, cv = v % VPR;   // row = coefficient * 2 + plane
            if (row < rows)
                t[k] = *reinterpret_cast<vec_t const*>(a.dcoef + (size_t(e.coef0 + (row >> 1)) * a.nCols + col) * 128 +
                                                       (row & 1) * 64 + slice * JS + cv * VE);
        }
        __syncthreads();        // the previous image's coefficients are no longer read
        stage_hermite<real_t>(H, a.htab, e.slot, L, tid, T);
#pragma unroll
        for (int k = 0; k < NV; ++k) {
            int const v = k * T + tid, row = v / VPR, cv = v % VPR;
            if (row < rows) *reinterpret_cast<vec_t*>(cs + row * JS + cv * VE) = t[k];
        }
        __syncthreads();
        uint32_t const in = uint32_t(a.smask[e.slot] >> (16 * zq));
        sho_add_regs<real_t, 6, 7>(acc, H, in, cs + p * JS + jl, 2 * JS, zq, L);
    }
#pragma unroll
    for (int k = 0; k < 16; ++k) yb[k * 64] = acc[k];
}

template <typename T>
int dalloc(DevicePlan& d, T*& ptr, size_t n, std::string& err) {
    ptr = nullptr;
    if (n == 0) n = 1;
    void* p = nullptr;
    HIP_TRY(hipMalloc(&p, n * sizeof(T)));
    d.allocations.push_back(p);
    d.bytes += n * sizeof(T);
    ptr = (T*)p;
    return 0;
}

template <typename T>
int dupload(DevicePlan& d, T*& ptr, std::vector<T> const& v, std::string& err) {
    if (int s = dalloc(d, ptr, v.size(), err)) return s;
    if (!v.empty()) HIP_TRY(hipMemcpy(ptr, v.data(), v.size() * sizeof(T), hipMemcpyHostToDevice));
    return 0;
}

// items[i] = heads[order[i]] for i < n, one word per thread
__global__ __launch_bounds__(256) void k_gather_heads(uint32_t const* __restrict__ order, uint64_t n,
                                                      uint32_t const* __restrict__ heads, uint32_t* __restrict__ items,
                                                      int hw) {
    uint64_t const t = uint64_t(blockIdx.x) * 256 + threadIdx.x;
    if (t >= n * uint64_t(hw)) return;
    uint64_t const i = t / hw, w = t % hw;
    items[t] = heads[uint64_t(order[i]) * hw + w];
}

}  // namespace

int device_gather_heads(DevicePlan const& d, uint32_t const* order, uint64_t n, uint32_t* items, hipStream_t stream,
                        std::string& err) {
    if (n == 0) return 0;
    uint64_t const words = n * uint64_t(d.head_words);
    uint64_t const grid = (words + 255) / 256;
    if (grid > 0x7fffffffull) { err = "too many blocks for one launch"; return 1; }
    hipLaunchKernelGGL(k_gather_heads, dim3(uint32_t(grid)), dim3(256), 0, stream, order, n, d.heads, items,
                       d.head_words);
    HIP_TRY(hipGetLastError());
    return 0;
}

void device_free(DevicePlan& d) {
    for (void* p : d.allocations) (void)hipFree(p);
    d = DevicePlan();
}

double reference_flops(Plan const& p, int fp_bits) {
    (void)fp_bits;
    double const nnzb = double(p.nnzb);
    double n = 0;
    // potential: (1 + 2 [complex E]) * nnzb * 64^2 * 2 (include/green_potential.hxx:171-177)
    n += (1.0 + 2.0 * (p.E.imag() != 0)) * nnzb * 4096 * 2;
    // kinetic: nnzb * (2 nFD + 1) * 2 * 64^2 * 2 per direction (include/green_kinetic.hxx:381)
    for (int d = 0; d < 3; ++d) n += nnzb * (2.0 * p.kinetic[d].fd_range + 1) * 2 * 4096 * 2;
    // dyadic (include/dyadic_plan.hxx:93-103, src/dyadic_plan.cxx:103-135), R1C2 = 2, Noco = 1
    if (p.nAtomImages > 0) {
        double add = 0, gen = 0, mul = 0, sum = 0;
        for (uint32_t k = 0; k < p.sho_add.index.size(); ++k) {
            int const L = p.image_lmax[p.sho_add.index[k]];
            add += 64.0 * 2 * (64 * (L + 1) + 16 * ((L + 1) * (L + 2)) / 2 + 4 * ((L + 1) * (L + 2) * (L + 3)) / 6);
            gen += 12.0 * (7 + 4 * L);
        }
        for (uint32_t i = 0; i < p.nAtoms; ++i) mul += double(nsho(p.image_lmax[i])) * nsho(p.image_lmax[i]);
        mul *= 2.0 * p.nCols * 64;
        if (p.nAtomImages > p.nAtoms) {
            for (uint32_t i = 0; i < p.nAtomImages; ++i) sum += nsho(p.image_lmax[i]);
            sum *= 2.0 * p.nCols * 64;
        }
        n += mul * 4 + 2 * sum * 4 + 2 * gen + 2 * add * 2;
    }
    return n;
}

int device_upload_plan(Plan const& p, DevicePlan& d, std::string& err) {
    if (d.uploaded) return 0;
    HIP_TRY(hipGetDevice(&d.device));
    d.nnzb = p.nnzb; d.nCols = p.nCols; d.nRows = p.nRows;
    d.nAtoms = p.nAtoms; d.nAtomImages = p.nAtomImages;
    d.natomcoeffs = p.natomcoeffs();
    d.nh_max = 1;
    for (int dd = 0; dd < 3; ++dd) {
        d.fd_range[dd] = p.kinetic[dd].fd_range;
        if (p.kinetic[dd].fd_range == 8) d.nh_max = 2;
    }
    if (!d.tuned[1]) {
        // the FP32 default shape.  Up to the 8th order k_lines, 32 columns, 2 directions ahead: it adds the images in
        // the plane form of k_plane but reads and writes 16 bytes per lane (against k_plane with 32 columns: 158,112
        // blocks 3,347 us against 3,779, 19,764 blocks 424 against 472, 1,461 blocks 31.1 against 35.2, 6,144 blocks
        // with images 138 against 156, 64 blocks 15.0 against 16.6).  With a direction of the 16th order k_local, 32
        // columns, whose registers hold two lines instead of a plane or a direction (against k_plane: 3,246 blocks 91.5
        // us against 106, 22,948 blocks 765 against 915; mixed orders with images, 4,096 blocks 133 against 383)
        bool const wide = d.nh_max == 2;
        d.tune_kind[1] = wide ? 0 : 2; d.tune_jw[1] = 32; d.tune_lb[1] = 2;
    }
    int s = 0;
    if ((s = dupload(d, d.colindx, p.colindx, err))) return s;
    if ((s = dupload(d, d.veff, p.veff_index, err))) return s;
    if ((s = dupload(d, d.row_pos, p.row_pos, err))) return s;
    {   // processing order of the local kernel: per source column, xy tiles of TILE x TILE target blocks swept
        // along z, so that the 6 stencil neighbours of a block were read shortly before (z neighbours
        // TILE^2 blocks back); consecutive work items then share one XCD's L2
        int const TILE = LOCAL_TILE;
        std::vector<uint64_t> key(p.nnzb);
        int32_t lo[3] = {1 << 30, 1 << 30, 1 << 30};
        for (uint32_t r = 0; r < p.nRows; ++r)
            for (int k = 0; k < 3; ++k) lo[k] = std::min(lo[k], p.row_coords[3 * r + k]);
        for (uint64_t b = 0; b < p.nnzb; ++b) {
            int32_t const* g = &p.row_coords[3 * size_t(p.rowindx[b])];
            uint64_t const x = uint64_t(g[0] - lo[0]), y = uint64_t(g[1] - lo[1]), z = uint64_t(g[2] - lo[2]);
            uint64_t const tx = x / TILE, ty = y / TILE;
            uint64_t const txs = (ty & 1) ? (1023 - tx) : tx;  // serpentine over tiles
            key[b] = (uint64_t(p.colindx[b]) << 48) | (ty << 38) | (txs << 28) | (z << 8) | ((y % TILE) << 4) | (x % TILE);
        }
        std::vector<uint32_t> order(p.nnzb);
        for (uint64_t b = 0; b < p.nnzb; ++b) order[b] = uint32_t(b);
        std::sort(order.begin(), order.end(), [&](uint32_t u, uint32_t v) { return key[u] < key[v]; });
        d.h_order = std::move(order);
    }

    // neighbour codes from the finite-difference lists: the entry before (after) a block in its
    // list is its left (right) neighbour; halo entries 0 are absent, negative ones periodic images
    {
        int const NH = d.nh_max;
        std::vector<int32_t> nb(size_t(3) * 2 * NH * p.nnzb, -1);
        for (int dd = 0; dd < 3; ++dd) {
            auto const& kp = p.kinetic[dd];
            for (size_t l = 0; l + 1 < kp.start.size(); ++l) {
                int32_t const* L = &kp.list[kp.start[l]];
                int const len = int(kp.start[l + 1] - kp.start[l]);
                int const n = len - 2 * NHALO;
                for (int i = 0; i < n; ++i) {
                    uint32_t const inzb = uint32_t(L[NHALO + i] - CUBE_EXISTS);
                    for (int side = 0; side < 2; ++side) {
                        for (int k = 0; k < NH; ++k) {
                            int const pos = NHALO + i + (side ? (k + 1) : -(k + 1));
                            int32_t const e = L[pos];
                            int32_t code;
                            if (e > 0) code = e - CUBE_EXISTS;
                            else if (e == 0) code = -1;
                            else code = -2 - (-e - CUBE_EXISTS);
                            nb[((size_t(dd) * 2 + side) * NH + k) * p.nnzb + inzb] = code;
                            if (code <= -2) d.has_images = true;
                        }
                    }
                }
            }
        }

        // the local kernels' block headers: block, column group, potential cell, add-list range, neighbour codes
        int const HW = (NH == 1) ? 16 : 32;
        d.head_words = HW;
        std::vector<uint32_t> heads(size_t(HW) * p.nnzb, 0);
        for (uint64_t b = 0; b < p.nnzb; ++b) {
            uint32_t* h = &heads[size_t(HW) * b];
            h[IH_BLK] = uint32_t(b);
            h[IH_COL] = p.colindx[b];
            h[IH_VEFF] = uint32_t(p.veff_index[b]);
            h[IH_ADD0] = p.sho_add.start[b];
            h[IH_ADD1] = p.sho_add.start[b + 1];
            for (int c = 0; c < 6 * NH; ++c) h[IH_NBR + c] = uint32_t(nb[size_t(c) * p.nnzb + b]);
        }
        std::vector<uint32_t> items(heads.size());
        for (uint64_t i = 0; i < p.nnzb; ++i)
            std::copy_n(&heads[size_t(HW) * d.h_order[i]], HW, &items[size_t(HW) * i]);
        if ((s = dupload(d, d.heads, heads, err))) return s;
        if ((s = dupload(d, d.items, items, err))) return s;
    }

    // dyadic structures
    if ((s = dupload(d, d.add_start, p.sho_add.start, err))) return s;
    {   // blocks touched by atom images with numax > 5, whose add-back runs in a separate kernel after k_local
        std::vector<uint32_t> wide;
        for (uint64_t blk = 0; blk < p.nnzb; ++blk)
            for (uint32_t k = p.sho_add.start[blk]; k < p.sho_add.start[blk + 1]; ++k)
                if (p.image_lmax[p.sho_add.index[k]] > 5) { wide.push_back(uint32_t(blk)); break; }
        d.n_wide_blocks = uint32_t(wide.size());
        if ((s = dupload(d, d.wide_blocks, wide, err))) return s;
        // blocks touched by atom images with numax <= 5 (the add-back on the matrix cores)
        std::vector<uint32_t> narrow;
        for (uint64_t blk = 0; blk < p.nnzb; ++blk)
            for (uint32_t k = p.sho_add.start[blk]; k < p.sho_add.start[blk + 1]; ++k)
                if (p.image_lmax[p.sho_add.index[k]] <= 5) { narrow.push_back(uint32_t(blk)); break; }
        d.n_narrow_blocks = uint32_t(narrow.size());
        if ((s = dupload(d, d.narrow_blocks, narrow, err))) return s;
    }
    {   // add-list entries in one record each: image, numax, the slot of (image, target row) in the Hermite table
        // (the projection chunks below add their own slots), first coefficient of the image
        std::map<uint64_t, uint32_t> slot_of;
        std::vector<uint32_t> entry(4 * p.sho_add.index.size());
        for (uint64_t blk = 0; blk < p.nnzb; ++blk)
            for (uint32_t k = p.sho_add.start[blk]; k < p.sho_add.start[blk + 1]; ++k) {
                uint32_t const img = p.sho_add.index[k];
                uint64_t const key = (uint64_t(img) << 32) | p.rowindx[blk];
                entry[4 * size_t(k) + 0] = img;
                entry[4 * size_t(k) + 1] = uint32_t(p.image_lmax[img]);
                entry[4 * size_t(k) + 2] = slot_of.emplace(key, uint32_t(slot_of.size())).first->second;
                entry[4 * size_t(k) + 3] = p.image_starts[img];
            }
        d.slot_map = std::move(slot_of);
        if ((s = dupload(d, d.add_entry, entry, err))) return s;
    }
    if ((s = dupload(d, d.image_pos, p.image_pos, err))) return s;
    if ((s = dupload(d, d.image_lmax, p.image_lmax, err))) return s;
    if ((s = dupload(d, d.image_starts, p.image_starts, err))) return s;
    if ((s = dupload(d, d.sum_start, p.sho_sum.start, err))) return s;
    if ((s = dupload(d, d.sum_index, p.sho_sum.index, err))) return s;
    if ((s = dupload(d, d.atom_lmax, p.atom_lmax, err))) return s;
    if ((s = dupload(d, d.atom_mat_off, p.atom_mat_off, err))) return s;
    if ((s = dupload(d, d.atom_starts, p.atom_starts, err))) return s;
    d.ncoeffs = p.ncoeffs();
    d.max_atom_nc = 0;
    for (uint32_t a = 0; a < p.nAtoms; ++a) d.max_atom_nc = std::max<uint32_t>(d.max_atom_nc, nsho(p.atom_lmax[a]));

    // projection work items: (image, column) pairs split into chunks of at most K blocks
    {
        uint64_t pairs = 0;
        for (auto const& c : p.sho_prj) pairs += c.index.size();
        uint32_t K = uint32_t(std::min<uint64_t>(16, std::max<uint64_t>(2, pairs / 4096)));
        std::vector<ProjChunk> chunks;
        std::vector<uint32_t> blocks, coef(1, 0), pair_chunk(size_t(p.nAtomImages) * p.nCols + 1, 0);
        for (uint32_t img = 0; img < p.nAtomImages; ++img) {
            int const nc = nsho(p.image_lmax[img]);
            for (uint32_t c = 0; c < p.nCols; ++c) {
                auto const& s_ = p.sho_prj[c];
                uint32_t const b0 = s_.start[img], b1 = s_.start[img + 1];
                for (uint32_t b = b0; b < b1; b += K) {
                    ProjChunk ch;
                    ch.image = img; ch.col = c;
                    ch.begin = uint32_t(blocks.size());
                    for (uint32_t k = b; k < std::min(b1, b + K); ++k) blocks.push_back(s_.index[k]);
                    ch.end = uint32_t(blocks.size());
                    chunks.push_back(ch);
                    coef.push_back(coef.back() + uint32_t(nc));
                }
                pair_chunk[size_t(img) * p.nCols + c + 1] = uint32_t(chunks.size());
            }
        }
        d.nchunks = uint32_t(chunks.size());
        d.total_chunk_coefs = coef.back();
        std::vector<uint32_t> bucket;
        for (int L = 0; L <= 7; ++L) {
            d.bucket_start[L] = uint32_t(bucket.size());
            for (uint32_t k = 0; k < chunks.size(); ++k)
                if (p.image_lmax[chunks[k].image] == L) bucket.push_back(k);
        }
        d.bucket_start[8] = uint32_t(bucket.size());
        std::vector<uint32_t> prj_slot(blocks.size());
        for (auto const& chk : chunks)
            for (uint32_t b = chk.begin; b < chk.end; ++b) {
                uint64_t const key = (uint64_t(chk.image) << 32) | p.rowindx[blocks[b]];
                auto const it = d.slot_map.emplace(key, uint32_t(d.slot_map.size())).first;
                prj_slot[b] = it->second;
            }
        if ((s = dupload(d, d.chunks, chunks, err))) return s;
        if ((s = dupload(d, d.prj_blocks, blocks, err))) return s;
        if ((s = dupload(d, d.prj_slot, prj_slot, err))) return s;
        {   // the table itself, computed on the device by hermite_1d
            size_t const ns = std::max<size_t>(1, d.slot_map.size());
            std::vector<uint32_t> simg(ns, 0), srow(ns, 0);
            for (auto const& kv : d.slot_map) { simg[kv.second] = uint32_t(kv.first >> 32); srow[kv.second] = uint32_t(kv.first & 0xffffffffu); }
            uint32_t *dimg = nullptr, *drow = nullptr;
            if ((s = dupload(d, dimg, simg, err))) return s;
            if ((s = dupload(d, drow, srow, err))) return s;
            if ((s = dalloc(d, d.htab, ns * 96, err))) return s;
            if ((s = dalloc(d, d.smask, ns, err))) return s;
            if (!d.slot_map.empty()) {
                hipLaunchKernelGGL(k_hermite_table, dim3(uint32_t(d.slot_map.size())), dim3(64), 0, 0, d.htab, d.smask,
                                   dimg, drow, d.image_pos, d.image_lmax, d.row_pos, p.hg[0], p.hg[1], p.hg[2], p.r_proj);
                HIP_TRY(hipGetLastError());
                HIP_TRY(hipDeviceSynchronize());
            }
            d.nslots = uint32_t(d.slot_map.size());
            d.slot_map.clear();
        }
        if ((s = dupload(d, d.chunk_coef, coef, err))) return s;
        {   // the chunks of every (atom, column) in one list, images in the order of the collection; one upload of
            // [start of every pair | chunks | pairs with chunks]
            size_t const npair = size_t(p.nAtoms) * p.nCols;
            std::vector<uint32_t> t, list, pairs;
            t.reserve(2 * npair + 1 + 2 * chunks.size());
            list.reserve(2 * chunks.size());
            t.push_back(0);
            for (uint32_t a = 0; a < p.nAtoms; ++a)
                for (uint32_t c = 0; c < p.nCols; ++c) {
                    for (uint32_t k = p.sho_sum.start[a]; k < p.sho_sum.start[a + 1]; ++k) {
                        uint32_t const img = p.sho_sum.index[k];
                        size_t const ic = size_t(img) * p.nCols + c;
                        for (uint32_t ch = pair_chunk[ic]; ch < pair_chunk[ic + 1]; ++ch) {
                            list.push_back(coef[ch]);
                            list.push_back(img);
                        }
                    }
                    if (list.size() / 2 > t.back()) pairs.push_back(uint32_t(t.size() - 1));
                    t.push_back(uint32_t(list.size() / 2));
                }
            if (t.size() & 1) t.push_back(0);   // the 8-byte chunk records start on 8 bytes
            size_t const at_list = t.size(), at_pairs = at_list + list.size();
            t.insert(t.end(), list.begin(), list.end());
            t.insert(t.end(), pairs.begin(), pairs.end());
            if ((s = dupload(d, d.coll_start, t, err))) return s;
            d.coll = d.coll_start + at_list;
            d.atom_pairs = d.coll_start + at_pairs;
            d.n_atom_pairs = uint32_t(pairs.size());
        }
        if ((s = dupload(d, d.bucket_chunks, bucket, err))) return s;
    }

    if ((s = dalloc(d, d.V, p.ncell() * 64, err))) return s;
    if ((s = dalloc(d, d.atom_hs, p.atom_hs.size(), err))) return s;
    if ((s = dalloc(d, d.E_col, size_t(2) * p.nCols, err))) return s;
    if ((s = dalloc(d, d.image_phase, p.image_phase.size(), err))) return s;
    d.uploaded = true;
    return 0;
}

int device_upload_values(Plan const& p, DevicePlan& d, std::string& err) {
    HIP_TRY(hipMemcpy(d.V, p.V_cell.data(), p.V_cell.size() * sizeof(double), hipMemcpyHostToDevice));
    if (!p.atom_hs.empty())
        HIP_TRY(hipMemcpy(d.atom_hs, p.atom_hs.data(), p.atom_hs.size() * sizeof(double), hipMemcpyHostToDevice));
    HIP_TRY(hipMemcpy(d.E_col, p.E_col.data(), p.E_col.size() * sizeof(std::complex<double>), hipMemcpyHostToDevice));
    if (!p.image_phase.empty())
        HIP_TRY(hipMemcpy(d.image_phase, p.image_phase.data(), p.image_phase.size() * sizeof(double), hipMemcpyHostToDevice));
    return 0;
}

// ---------------------------------------------------------------------------------------------
// 4. adjoint gradient of L = Im sum_c w_c Tr[G_c], Tr over the diagonal block of column group c.
//    With dG = -A^-1 dA G and lambda_c = A^-H P_c: dL = -Im sum_c w_c <lambda_c, dA G_c>.
// ---------------------------------------------------------------------------------------------
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o, 64);
    return v;
}

// per block and point i: -Im(w_c sum_j conj(lambda[b][i][j]) G[b][i][j]), 0 outside the cell (no potential)
__global__ __launch_bounds__(256) void k_grad_v_blocks(double* __restrict__ gpart, double const* __restrict__ X,
                                                       double const* __restrict__ Lam, uint16_t const* __restrict__ colindx,
                                                       int32_t const* __restrict__ veff, double const* __restrict__ wE) {
    uint64_t const blk = blockIdx.x;
    int const j = threadIdx.x & 63, w = threadIdx.x >> 6;
    uint32_t const c = colindx[blk];
    double const wr = wE[4 * c], wi = wE[4 * c + 1];
    bool const inside = veff[blk] >= 0;
    for (int i = w; i < 64; i += 4) {
        size_t const er = (blk * 2 + 0) * 4096 + i * 64 + j, ei = er + 4096;
        double const gr = X[er], gi = X[ei], lr = Lam[er], li = Lam[ei];
        double const sr = wave_sum(lr * gr + li * gi), si = wave_sum(lr * gi - li * gr);
        if (j == 0) gpart[blk * 64 + i] = inside ? -(wr * si + wi * sr) : 0.0;
    }
}

// per cell block (bx, by, bz): the sum over the blocks that read its potential, in ascending block order, written in
// the caller's grid order [4 nbz][4 nby][4 nbx], so that the host copies it once and sorts nothing (a gradient on 64^3
// points, 11,688 blocks, 903 -> 691 us with the entries of k_grad_atoms below spread over more waves)
__global__ __launch_bounds__(64) void k_grad_v_cells(double* __restrict__ grid, double const* __restrict__ gpart,
                                                     uint32_t const* __restrict__ cell_start,
                                                     uint32_t const* __restrict__ cell_blocks, uint32_t nbx,
                                                     uint32_t nby) {
    uint32_t const v = blockIdx.x, bx = v % nbx, by = (v / nbx) % nby, bz = v / nbx / nby;
    int const i = threadIdx.x;
    double acc = 0;
    for (uint32_t k = cell_start[v]; k < cell_start[v + 1]; ++k) acc += gpart[uint64_t(cell_blocks[k]) * 64 + i];
    grid[((uint64_t(bz) * 4 + (i >> 4)) * (4 * uint64_t(nby)) + by * 4 + ((i >> 2) & 3)) * (4 * uint64_t(nbx)) + bx * 4 +
         (i & 3)] = acc;
}

// atom coefficients of one vector: per (atom, column group) the image partials collected with the Bloch phase,
// out[((atom_starts[a] + s) * nCols + c)][re/im][j] (the input of the atom-matrix multiply of k_sho_atoms).  One
// work-group per (atom, column, 4 coefficients), a wave per coefficient.
__global__ __launch_bounds__(256) void k_sho_collect(
    double* __restrict__ out, double const* __restrict__ partial, uint32_t const* __restrict__ coll_start,
    CollectEntry const* __restrict__ coll, int8_t const* __restrict__ atom_lmax,
    double const* __restrict__ image_phase, uint32_t nCols, uint32_t const* __restrict__ atom_starts) {
    uint32_t const pair = blockIdx.x, c = pair % nCols, a = pair / nCols;
    int const j = threadIdx.x & 63, s = blockIdx.y * 4 + (threadIdx.x >> 6);
    int const L = atom_lmax[a];
    if (s >= ((L + 1) * (L + 2) * (L + 3)) / 6) return;
    double ar, ai;
    collect_coefficient<double>(partial, coll, coll_start[pair], coll_start[pair + 1], image_phase, s, j, ar, ai);
    double* dst = out + ((size_t(atom_starts[a]) + s) * nCols + c) * 128 + j;
    dst[0] = ar;
    dst[64] = ai;
}

// per (atom a, row k, entry l): z_c = sum_j conj(cL[k][c][j]) cX[l][c][j];
// gmat[a] = [-Im sum_c w_c z_c][k][l] (dL/dM entries times 1) and [-Im sum_c w_c (-E_c) z_c][k][l].
// A wave per entry, 4 per work-group: latency-bound (16 atoms, numax 3, 8 column groups: 6,400 waves; with a wave per row
// looping over l, 320 waves, it took 70 us, now 11).
__global__ __launch_bounds__(256) void k_grad_atoms(double* __restrict__ gmat, double const* __restrict__ cX,
                                                    double const* __restrict__ cL, int8_t const* __restrict__ atom_lmax,
                                                    uint32_t const* __restrict__ atom_starts,
                                                    uint64_t const* __restrict__ atom_mat_off,
                                                    double const* __restrict__ wE, uint32_t nCols) {
    uint32_t const a = blockIdx.x;
    int const k = blockIdx.y, l = blockIdx.z * 4 + (threadIdx.x >> 6), j = threadIdx.x & 63;
    int const L = atom_lmax[a];
    int const nc = ((L + 1) * (L + 2) * (L + 3)) / 6;
    if (k >= nc || l >= nc) return;   // uniform over the wave; no barrier below
    size_t const base = size_t(atom_starts[a]) * nCols * 128;
    double const* pl = cL + base + size_t(k) * nCols * 128 + j;
    double const* px = cX + base + size_t(l) * nCols * 128 + j;
    double hr = 0, sr = 0;   // -Im of the two weighted sums
#pragma unroll 2
    for (uint32_t c = 0; c < nCols; ++c) {
        double const lr = pl[size_t(c) * 128], li = pl[size_t(c) * 128 + 64];
        double const xr = px[size_t(c) * 128], xi = px[size_t(c) * 128 + 64];
        double const zr = lr * xr + li * xi, zi = lr * xi - li * xr;   // conj(l) x
        double const w_r = wE[4 * c], w_i = wE[4 * c + 1], v_r = wE[4 * c + 2], v_i = wE[4 * c + 3];
        hr -= w_r * zi + w_i * zr;
        sr -= v_r * zi + v_i * zr;
    }
    hr = wave_sum(hr);
    sr = wave_sum(sr);
    if (j == 0) {
        gmat[atom_mat_off[a] + size_t(k) * nc + l] = hr;
        gmat[atom_mat_off[a] + size_t(nc) * nc + size_t(k) * nc + l] = sr;
    }
}

// Atomic density matrices, the right projection of the collected coefficients c of X onto the same image
// (SHOprj_right, include/green_dyadic.hxx:925-1036): D[i][j] = factor Im(phase sum_c sum_s c[i][c][s] p_j(c, s)) over the
// 64 points s of every source block c.  One work-group per (image, row i); wave w takes the source blocks w, w + 4, ...
// and a lane the entry j (nc <= 120: at most two), contracting x, y, z in turn (84 FMAs per component and block).
// desc[image] = {first coefficient row of its atom, offset of its matrix (low, high word)}, the float bits of col_pos
// follow.  As loops on the host, after a copy of all coefficients, this took about 150 us for 4 atoms of
// numax 3 and 8 source blocks; here 8 us.
__global__ __launch_bounds__(256) void k_density(double* __restrict__ D, double const* __restrict__ cX,
                                                 double const* __restrict__ image_pos,
                                                 int8_t const* __restrict__ image_lmax,
                                                 double const* __restrict__ image_phase,
                                                 uint32_t const* __restrict__ desc, uint32_t nai, uint32_t nCols,
                                                 double hx, double hy, double hz, double rproj, double factor) {
    __shared__ double A[4][2][64];      // masked coefficients of the wave's source block
    __shared__ double H[4][8][3][4];
    __shared__ float x2[4][3][4];
    __shared__ double part[4][2][128];
    uint32_t const img = blockIdx.x;
    int const i = blockIdx.y, tid = threadIdx.x, w = tid >> 6, lane = tid & 63;
    int const L = image_lmax[img], nc = ((L + 1) * (L + 2) * (L + 3)) / 6;
    if (i >= nc) return;   // uniform over the work-group
    float const* col_pos = reinterpret_cast<float const*>(desc + size_t(nai) * 3);
    double const* src0 = cX + (size_t(desc[3 * size_t(img)]) + i) * nCols * 128 + lane;
    int jx[2], jy[2], jz[2];   // exponents of the lane's entries
    for (int q = 0; q < 2; ++q) {
        int r = lane + 64 * q, iz = 0, iy = 0;
        if (r >= nc) r = 0;
        while (r >= ((L - iz + 1) * (L - iz + 2)) / 2) { r -= ((L - iz + 1) * (L - iz + 2)) / 2; ++iz; }
        while (r >= L - iz - iy + 1) { r -= L - iz - iy + 1; ++iy; }
        jx[q] = r; jy[q] = iy; jz[q] = iz;
    }
    int const nq = nc > 64 ? 2 : 1;
    double sre[2] = {0, 0}, sim[2] = {0, 0};
    float const R2 = float(rproj * rproj);
    double const hgrid[4] = {hx, hy, hz, rproj};
    for (uint32_t c0 = 0; c0 < nCols; c0 += 4) {
        uint32_t const c = c0 + w;
        bool const have = c < nCols;
        double const cr = have ? src0[size_t(c) * 128] : 0.0, ci = have ? src0[size_t(c) * 128 + 64] : 0.0;
        if (have && lane < 12)
            hermite_1d<double>(H[w], x2[w], lane, L, image_pos + 4 * size_t(img), col_pos + 4 * size_t(c), hgrid);
        __syncthreads();
        if (have) {
            float const d2z = x2[w][2][lane >> 4] - R2;
            float const d2yz = x2[w][1][(lane >> 2) & 3] + d2z;
            bool const in = (d2z < 0) && (d2yz < 0) && (x2[w][0][lane & 3] + d2yz < 0);
            A[w][0][lane] = in ? cr : 0.0;
            A[w][1][lane] = in ? ci : 0.0;
        }
        __syncthreads();
        if (have) {
            for (int q = 0; q < nq; ++q) {
                double const* Hx = H[w][jx[q]][0];
                double const* Hy = H[w][jy[q]][1];
                double const* Hz = H[w][jz[q]][2];
                double const x0 = Hx[0], x1 = Hx[1], x2_ = Hx[2], x3 = Hx[3];
#pragma unroll
                for (int p = 0; p < 2; ++p) {
                    double acc = 0;
#pragma unroll
                    for (int z = 0; z < 4; ++z) {
                        double by = 0;
#pragma unroll
                        for (int y = 0; y < 4; ++y) {
                            double const* r = &A[w][p][z * 16 + y * 4];
                            by += Hy[y] * (((r[0] * x0 + r[1] * x1) + r[2] * x2_) + r[3] * x3);
                        }
                        acc += Hz[z] * by;
                    }
                    if (p == 0) sre[q] += acc; else sim[q] += acc;
                }
            }
        }
        __syncthreads();   // A, H and x2 are free
    }
    for (int q = 0; q < nq; ++q) { part[w][0][lane + 64 * q] = sre[q]; part[w][1][lane + 64 * q] = sim[q]; }
    __syncthreads();
    if (tid < nc) {
        double const re = (part[0][0][tid] + part[1][0][tid]) + (part[2][0][tid] + part[3][0][tid]);
        double const im = (part[0][1][tid] + part[1][1][tid]) + (part[2][1][tid] + part[3][1][tid]);
        double const pr = image_phase[2 * size_t(img)], pi = image_phase[2 * size_t(img) + 1];
        uint64_t const off = uint64_t(desc[3 * size_t(img) + 1]) | uint64_t(desc[3 * size_t(img) + 2]) << 32;
        D[off + size_t(i) * nc + tid] = (re * pi + im * pr) * factor;
    }
}

// Local-kernel tile shapes.  kind 0: k_local (LDS accumulator), JW columns per work-group (16 or 32), LB
// kinetic lines per thread in flight (1, 2, 4).  kind 1: k_plane (register accumulator), JW = 32 or 64.
// kind 2: k_lines (16-byte lanes, line ownership), JW = 16 or 32, or 64 in FP32; LB = directions of neighbour
// lines issued up front (3 or 2; 16th-order stencils issue one direction at a time).
template <typename real_t, int NH, bool IMG>
static void launch_local(int kind, int jw, int lb, dim3 g, hipStream_t stream, LocalArgs<real_t> const& a) {
#define KL(JW_, LB_) hipLaunchKernelGGL((k_local<real_t, NH, IMG, JW_, LB_>), g, dim3(8 * JW_), 0, stream, a)
#define KP(JW_) hipLaunchKernelGGL((k_plane<real_t, NH, IMG, JW_>), g, dim3(8 * JW_), 0, stream, a)
#define KN(JW_, PF_) hipLaunchKernelGGL((k_lines<real_t, NH, IMG, JW_, PF_>), g, dim3((JW_ / Lane<real_t>::n) * 32), 0, stream, a)
    if (kind == 2) {   // lb: directions prefetched (3 or 2; 16th-order stencils always 1)
        if constexpr (NH == 2) {
            if (jw == 16) KN(16, 1);
            else if (jw == 64) { if constexpr (sizeof(real_t) == 4) KN(64, 1); }
            else KN(32, 1);
        } else if (lb == 2) {
            if (jw == 16) KN(16, 2);
            else if (jw == 64) { if constexpr (sizeof(real_t) == 4) KN(64, 2); }
            else KN(32, 2);
        } else {
            if (jw == 16) KN(16, 3);
            else if (jw == 64) { if constexpr (sizeof(real_t) == 4) KN(64, 3); }
            else KN(32, 3);
        }
    } else if (kind == 1) {
        if (jw == 64) KP(64); else KP(32);
    } else if (jw == 16) {
        if (lb == 1) KL(16, 1); else if (lb == 4) KL(16, 4); else KL(16, 2);
    } else {
        if (lb == 1) KL(32, 1); else if (lb == 4) KL(32, 4); else KL(32, 2);
    }
#undef KL
#undef KP
#undef KN
}

template <typename real_t>
static Workspace<real_t>& workspace(DevicePlan& d);
template <> Workspace<double>& workspace<double>(DevicePlan& d) { return d.ws64; }
template <> Workspace<float>& workspace<float>(DevicePlan& d) { return d.ws32; }

template <typename real_t>
int device_action(DevicePlan& d, ActionScalars const& s, real_t* y, real_t const* x, hipStream_t stream,
                  std::string& err, int parts, double* dot, Workspace<real_t>* ext) {
    auto& ws = ext ? *ext : workspace<real_t>(d);
    if (!ext) {
        // every buffer of this precision is allocated on the first call, so that later calls (also under graph
        // capture) allocate nothing; parts = 0 only allocates
        if (d.nAtomImages > 0 && !ws.dcoef) {
            if (int r = dalloc(d, ws.partial, size_t(d.total_chunk_coefs) * 128, err)) return r;
            if (int r = dalloc(d, ws.dcoef, size_t(d.natomcoeffs) * d.nCols * 128, err)) return r;
        }
        if (!ws.zero) {
            if (int r = dalloc(d, ws.zero, NBLK, err)) return r;
            HIP_TRY(hipMemsetAsync(ws.zero, 0, NBLK * sizeof(real_t), stream));
        }
    }
    if ((parts & ACTION_PROJECT) && d.nAtomImages > 0 && d.nchunks > 0) {
        for (int L = 0; L <= 7; ++L) {
            uint32_t const n = d.bucket_start[L + 1] - d.bucket_start[L];
            if (!n) continue;
            uint32_t const* bucket = d.bucket_chunks + d.bucket_start[L];
#define LAUNCH_PRJ(LL) hipLaunchKernelGGL((k_sho_project<real_t, LL>), dim3(n), dim3(128), 0, stream, ws.partial, x, \
                d.chunks, bucket, d.chunk_coef, d.prj_blocks, d.col_active, d.htab, d.smask, d.prj_slot)
#define LAUNCH_MFMA(LL) hipLaunchKernelGGL((k_sho_project_mfma<real_t, LL>), dim3(n), dim3(256), 0, stream, ws.partial, \
                x, d.chunks, bucket, d.chunk_coef, d.prj_blocks, d.col_active, d.htab, d.smask, d.prj_slot)
            if (d.prj_engine[sizeof(real_t) == 8 ? 0 : 1] == 1 && L <= 5) {   // the dense form on the matrix cores
                switch (L) {
                    case 0: LAUNCH_MFMA(0); break; case 1: LAUNCH_MFMA(1); break;
                    case 2: LAUNCH_MFMA(2); break; case 3: LAUNCH_MFMA(3); break;
                    case 4: LAUNCH_MFMA(4); break; default: LAUNCH_MFMA(5); break;
                }
            } else {
                switch (L) {
                    case 0: LAUNCH_PRJ(0); break; case 1: LAUNCH_PRJ(1); break;
                    case 2: LAUNCH_PRJ(2); break; case 3: LAUNCH_PRJ(3); break;
                    case 4: LAUNCH_PRJ(4); break; case 5: LAUNCH_PRJ(5); break;
                    case 6: LAUNCH_PRJ(6); break; default: LAUNCH_PRJ(7); break;
                }
            }
#undef LAUNCH_PRJ
#undef LAUNCH_MFMA
            HIP_TRY(hipGetLastError());
        }
        // right-hand sides per work-group: 16 fill 128-byte lines in FP64; in FP32 32 do, and 16 (twice the work-groups,
        // half lines) are taken while 32 would leave CUs without one, below 128 pairs = 256 work-groups.  Measured, FP32,
        // 16 against 32: numax 7, 88 pairs 61 us against 73, 264 pairs 131 against 118, 704 pairs 251 against 215; numax 5,
        // 140 pairs 46 against 38, 1,392 pairs 218 against 161; numax 3, 104 pairs 15.3 against 15.5, 312 pairs 34 against
        // 24; numax 2, 104 pairs 12.6 against 11.5, 832 pairs 55 against 37
        uint64_t const pairs = d.n_atom_pairs;
        int const JS = (sizeof(real_t) == 4 && pairs >= 128) ? 32 : 16;
        if (pairs * (64 / JS) > 0x7fffffffull) { err = "too many (atom, column) pairs for one launch"; return 1; }
        size_t const lds = size_t(2) * JS * std::max<size_t>((d.max_atom_nc + 3) & ~3u, ATOM_T / 16) * sizeof(double);
#define LAUNCH_ATOMS(JS_) hipLaunchKernelGGL((k_sho_atoms<real_t, JS_>), dim3(uint32_t(pairs) * (64 / JS_)), \
            dim3(ATOM_T), lds, stream, ws.dcoef, ws.partial, d.atom_pairs, d.coll_start, \
            reinterpret_cast<CollectEntry const*>(d.coll), d.sum_start, d.sum_index, d.image_starts, d.atom_lmax, d.atom_hs, d.atom_mat_off, d.image_phase, d.nCols, \
            d.E_col, d.col_active)
        if (JS == 32) LAUNCH_ATOMS(32); else LAUNCH_ATOMS(16);
#undef LAUNCH_ATOMS
        HIP_TRY(hipGetLastError());
    }
    if (!(parts & ACTION_LOCAL)) return 0;
    LocalArgs<real_t> a;
    a.y = y; a.x = x; a.dcoef = ws.dcoef; a.V = d.V;
    a.add_start = d.add_start; a.colindx = d.colindx;
    a.nCols = d.nCols;
    a.zero = ws.zero;
    a.items = d.active_order ? d.active_items : d.items;
    a.add_entry = reinterpret_cast<AddEntry const*>(d.add_entry);
    a.nitems = d.active_order ? d.n_active : d.nnzb;
    a.E_col = d.E_col;
    a.htab = d.htab; a.smask = d.smask;
    a.dot = dot;
    int const engine = d.prj_engine[sizeof(real_t) == 8 ? 0 : 1];
    a.add_local = (engine == 1) ? 0 : 1;
    static int const c8i[5] = {-14350, 8064, -1008, 128, -9};
    static int const c16i[9] = {-924708642, 538137600, -94174080, 22830080, -5350800, 1053696, -156800, 15360, -735};
    double cdiag = 0;
    for (int dd = 0; dd < 3; ++dd) {
        double const n8 = s.prefactor[dd] / 5040., n16 = s.prefactor[dd] / 302702400.;
        for (int m = 0; m < 5; ++m) a.c8[dd][m] = real_t(c8i[m] * n8);
        for (int m = 0; m < 9; ++m) a.c16[dd][m] = real_t(c16i[m] * n16);
        a.nh[dd] = (d.fd_range[dd] == 8) ? 2 : 1;
        cdiag += (a.nh[dd] == 2) ? c16i[0] * n16 : c8i[0] * n8;
        for (int u = 0; u < 2; ++u) for (int v = 0; v < 2; ++v) a.phase[dd][u][v] = s.phase[dd][u][v];
    }
    a.cdiag = real_t(cdiag);
    // work-groups are dealt round-robin to the 8 XCDs: give each XCD a contiguous range of
    // (block, column slice) items so that neighbour blocks meet in the same L2
    int const v = sizeof(real_t) == 8 ? 0 : 1;
    int const KIND = d.tune_kind[v], JW = d.tune_jw[v], LB = d.tune_lb[v];
    if (a.nitems == 0) return 0;
    uint64_t const items = uint64_t(64 / JW) * a.nitems;
    uint64_t const per = (items + 7) / 8;
    a.per_xcd = uint32_t(per);
    uint64_t const grid = per * 8;
    if (grid > 0x7fffffffull) { err = "too many blocks for one launch"; return 1; }
    dim3 const g{uint32_t(grid), 1, 1};
    if (d.nh_max == 2) {
        if (d.has_images) launch_local<real_t, 2, true>(KIND, JW, LB, g, stream, a);
        else launch_local<real_t, 2, false>(KIND, JW, LB, g, stream, a);
    } else {
        if (d.has_images) launch_local<real_t, 1, true>(KIND, JW, LB, g, stream, a);
        else launch_local<real_t, 1, false>(KIND, JW, LB, g, stream, a);
    }
    HIP_TRY(hipGetLastError());
    if (!a.add_local && d.n_narrow_blocks > 0) {   // the numax <= 5 images on the matrix cores
        hipLaunchKernelGGL((k_sho_add_mfma<real_t>), dim3(d.n_narrow_blocks), dim3(256), 0, stream, a, d.narrow_blocks,
                           d.col_active);
        HIP_TRY(hipGetLastError());
    }
    if (d.n_wide_blocks > 0) {
        uint64_t const wide = uint64_t(d.n_wide_blocks) * (64 * sizeof(real_t) / 128);   // column slices of 128 bytes
        if (wide > 0x7fffffffull) { err = "too many blocks for one launch"; return 1; }
        hipLaunchKernelGGL((k_sho_add_wide<real_t>), dim3(uint32_t(wide)), dim3(1024 / sizeof(real_t)), 0, stream, a,
                           d.wide_blocks, d.col_active);
        HIP_TRY(hipGetLastError());
    }
    return 0;
}

template int device_action<double>(DevicePlan&, ActionScalars const&, double*, double const*, hipStream_t, std::string&,
                                   int, double*, Workspace<double>*);
template int device_action<float>(DevicePlan&, ActionScalars const&, float*, float const*, hipStream_t, std::string&,
                                  int, double*, Workspace<float>*);

// ---------------------------------------------------------------------------------------------
// The action without allocation (gfa_action_noalloc): the projection partial sums, the addition coefficients
// and the zero block live in `scratch`, a fixed array of every GPU the library runs on (held until the process
// ends).  Its device address is taken once per device with hipGetSymbolAddress; the host-side name `scratch` is never handed to a kernel.  Calls that overlap on one GPU
// share the array and race.
// ---------------------------------------------------------------------------------------------
namespace {

static __device__ __align__(256) unsigned char scratch[NOALLOC_SCRATCH_BYTES];

constexpr int MAX_DEVICES = 64;
std::mutex g_scratch_mutex;
void* g_scratch_ptr[MAX_DEVICES] = {};

// the address of `scratch` on the current device (which must be `device`), looked up on its first use there
int scratch_address(int device, unsigned char** out, std::string& err) {
    if (device < 0 || device >= MAX_DEVICES) { err = "device ordinal out of range"; return 1; }
    std::lock_guard<std::mutex> lock(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void* ptr = nullptr;
        hipError_t const e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
        if (e != hipSuccess || !ptr) {
            err = std::string("hipGetSymbolAddress(scratch): ") + hipGetErrorString(e);
            return 2;
        }
        g_scratch_ptr[device] = ptr;
    }
    *out = static_cast<unsigned char*>(g_scratch_ptr[device]);
    return 0;
}

template <typename T>
__global__ __launch_bounds__(256) void k_fill_zero(T* __restrict__ p, uint32_t n) {
    uint32_t const i = blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = T(0);
}

size_t round256(size_t b) { return (b + 255) & ~size_t(255); }

}  // namespace

size_t noalloc_scratch_bytes(DevicePlan const& d, int fp_bits) {
    size_t const s = fp_bits == 64 ? 8 : 4;
    size_t b = round256(size_t(NBLK) * s);   // zero block
    if (d.nAtomImages > 0) {
        b += round256(size_t(d.total_chunk_coefs) * 128 * s);
        b += round256(size_t(d.natomcoeffs) * d.nCols * 128 * s);
    }
    return b;
}

template <typename real_t>
int device_action_noalloc(DevicePlan& d, ActionScalars const& s, real_t* y, real_t const* x, hipStream_t stream,
                          std::string& err) {
    size_t const need = noalloc_scratch_bytes(d, sizeof(real_t) == 8 ? 64 : 32);
    if (need > NOALLOC_SCRATCH_BYTES) {
        err = "the plan needs " + std::to_string(need) + " bytes of action scratch, more than the " +
              std::to_string(NOALLOC_SCRATCH_BYTES) + " of the allocation-free action";
        return 1;
    }
    unsigned char* base = nullptr;
    if (int r = scratch_address(d.device, &base, err)) return r;
    unsigned char* cur = base;
    auto take = [&](size_t bytes) { unsigned char* p = cur; cur += round256(bytes); return p; };
    Workspace<real_t> ws;
    ws.zero = reinterpret_cast<real_t*>(take(size_t(NBLK) * sizeof(real_t)));
    if (d.nAtomImages > 0) {
        ws.partial = reinterpret_cast<real_t*>(take(size_t(d.total_chunk_coefs) * 128 * sizeof(real_t)));
        ws.dcoef = reinterpret_cast<real_t*>(take(size_t(d.natomcoeffs) * d.nCols * 128 * sizeof(real_t)));
    }
    // the array keeps the previous call's contents: the zero block is cleared on every call (a kernel, so that
    // the call can be captured in a graph); the other regions are written before they are read
    hipLaunchKernelGGL((k_fill_zero<real_t>), dim3((NBLK + 255) / 256), dim3(256), 0, stream, ws.zero, uint32_t(NBLK));
    HIP_TRY(hipGetLastError());
    return device_action<real_t>(d, s, y, x, stream, err, ACTION_ALL, nullptr, &ws);
}
template int device_action_noalloc<double>(DevicePlan&, ActionScalars const&, double*, double const*, hipStream_t,
                                           std::string&);
template int device_action_noalloc<float>(DevicePlan&, ActionScalars const&, float*, float const*, hipStream_t,
                                          std::string&);

// Times every k_local tile shape on the caller's vectors (the whole action, reps launches each, HIP events on
// `stream`) and keeps the fastest for this precision.  y is overwritten.
template <typename real_t>
int device_autotune(DevicePlan& d, ActionScalars const& s, real_t* y, real_t const* x, hipStream_t stream, int reps,
                    double* best_ms, std::string& err) {
    int const v = sizeof(real_t) == 8 ? 0 : 1;
    static int const SHAPES[14][3] = {{0, 16, 1}, {0, 16, 2}, {0, 16, 4}, {0, 32, 1}, {0, 32, 2}, {0, 32, 4},
                                      {1, 32, 0}, {1, 64, 0}, {2, 16, 3}, {2, 32, 3}, {2, 64, 3}, {2, 16, 2},
                                      {2, 32, 2}, {2, 64, 2}};
    double best = 1e300;
    int bkind = d.tune_kind[v], bjw = d.tune_jw[v], blb = d.tune_lb[v];
    hipEvent_t e0 = nullptr, e1 = nullptr;
    // the shape in use before the call (or the fastest so far) is restored on every return, also on errors
    auto finish = [&](int status) {
        if (e0) (void)hipEventDestroy(e0);
        if (e1) (void)hipEventDestroy(e1);
        d.tune_kind[v] = bkind; d.tune_jw[v] = bjw; d.tune_lb[v] = blb;
        return status;
    };
    auto timed = [&]() -> int {
        HIP_TRY(hipEventCreate(&e0));
        HIP_TRY(hipEventCreate(&e1));
        for (auto const& sh : SHAPES) {
            int const kind = sh[0], jw = sh[1], lb = sh[2];
            if (kind == 2 && jw == 64 && sizeof(real_t) == 8) continue;   // no FP64 kind-2 shape of 64 columns
            d.tune_kind[v] = kind; d.tune_jw[v] = jw; d.tune_lb[v] = lb;
            if (int r = device_action<real_t>(d, s, y, x, stream, err)) return r;  // warm-up
            HIP_TRY(hipEventRecord(e0, stream));
            for (int k = 0; k < reps; ++k)
                if (int r = device_action<real_t>(d, s, y, x, stream, err)) return r;
            HIP_TRY(hipEventRecord(e1, stream));
            HIP_TRY(hipEventSynchronize(e1));
            float ms = 0;
            HIP_TRY(hipEventElapsedTime(&ms, e0, e1));
            double const t = double(ms) / std::max(1, reps);
            if (t < best) { best = t; bkind = kind; bjw = jw; blb = lb; }
        }
        return 0;
    };
    if (int r = timed()) return finish(r);
    // the projection's engine with the fastest shape: the vector form, then the matrix cores
    if (d.nAtomImages > 0 && d.nchunks > 0) {
        d.tune_kind[v] = bkind; d.tune_jw[v] = bjw; d.tune_lb[v] = blb;
        double tbest[2] = {1e300, 1e300};
        int const keep = d.prj_engine[v];
        for (int eng = 0; eng < 2; ++eng) {
            d.prj_engine[v] = eng;
            if (int r = device_action<real_t>(d, s, y, x, stream, err)) { d.prj_engine[v] = keep; return finish(r); }
            if (hipEventRecord(e0, stream) != hipSuccess) { d.prj_engine[v] = keep; return finish(2); }
            for (int k = 0; k < reps; ++k)
                if (int r = device_action<real_t>(d, s, y, x, stream, err)) { d.prj_engine[v] = keep; return finish(r); }
            float ms = 0;
            if (hipEventRecord(e1, stream) != hipSuccess || hipEventSynchronize(e1) != hipSuccess ||
                hipEventElapsedTime(&ms, e0, e1) != hipSuccess) {
                d.prj_engine[v] = keep;
                err = "autotune: event timing failed";
                return finish(2);
            }
            tbest[eng] = double(ms) / std::max(1, reps);
        }
        d.prj_engine[v] = tbest[1] < tbest[0] ? 1 : 0;
        best = std::min(tbest[0], tbest[1]);
    }
    d.tuned[v] = true;
    if (best_ms) *best_ms = best;
    return finish(0);
}
template int device_autotune<double>(DevicePlan&, ActionScalars const&, double*, double const*, hipStream_t, int, double*, std::string&);
template int device_autotune<float>(DevicePlan&, ActionScalars const&, float*, float const*, hipStream_t, int, double*, std::string&);

// The adjoint gradient (FP64): X solves (H - E_c S) X = B, Lam solves (H - conj(E_c) S) Lam = B column group by
// column group; wE[c] = {w_c, -E_c w_c}.  Results on the host: grad_V (dL/dV on the grid, unless null) and
// gmat_host at atom_mat_off (per contributing atom [2][nc][nc], the derivative with respect to the entries of
// (h dVol-scaled, s dVol-scaled) before the SHO prefactors, see gfa_gradient).
// projection of one FP64 vector onto every atom image and collection per (atom, column group) with the Bloch
// phases: out[((atom_starts[a] + s) * nCols + c)][re/im][j]
static int project_collect(DevicePlan& d, double const* vec, double* out, hipStream_t stream, std::string& err) {
    auto& ws = d.ws64;
    if (!ws.partial) {
        if (int r = dalloc(d, ws.partial, size_t(d.total_chunk_coefs) * 128, err)) return r;
        if (int r = dalloc(d, ws.dcoef, size_t(d.natomcoeffs) * d.nCols * 128, err)) return r;
    }
    for (int L = 0; L <= 7; ++L) {
        uint32_t const n = d.bucket_start[L + 1] - d.bucket_start[L];
        if (!n) continue;
        uint32_t const* bucket = d.bucket_chunks + d.bucket_start[L];
#define LAUNCH_PRJ(LL) hipLaunchKernelGGL((k_sho_project<double, LL>), dim3(n), dim3(128), 0, stream, ws.partial, vec, \
        d.chunks, bucket, d.chunk_coef, d.prj_blocks, (uint8_t const*)nullptr, d.htab, d.smask, d.prj_slot)
        switch (L) {
            case 0: LAUNCH_PRJ(0); break; case 1: LAUNCH_PRJ(1); break;
            case 2: LAUNCH_PRJ(2); break; case 3: LAUNCH_PRJ(3); break;
            case 4: LAUNCH_PRJ(4); break; case 5: LAUNCH_PRJ(5); break;
            case 6: LAUNCH_PRJ(6); break; default: LAUNCH_PRJ(7); break;
        }
#undef LAUNCH_PRJ
    }
    hipLaunchKernelGGL(k_sho_collect, dim3(d.nAtoms * d.nCols, (d.max_atom_nc + 3) / 4), dim3(256), 0, stream, out,
                       ws.partial, d.coll_start, reinterpret_cast<CollectEntry const*>(d.coll), d.atom_lmax,
                       d.image_phase, d.nCols, d.atom_starts);
    HIP_TRY(hipGetLastError());
    return 0;
}

int device_density_matrices(DevicePlan& d, Plan const& p, ActionScalars const& s, double const* X, double factor,
                            double* D, hipStream_t stream, std::string& err) {
    auto& w = d.dens;
    if (!w.desc) {   // kept with the plan, like the other work buffers
        std::vector<uint64_t> off(size_t(p.nAtoms) + 1, 0);
        for (uint32_t a = 0; a < p.nAtoms; ++a) off[a + 1] = off[a] + uint64_t(nsho(p.atom_lmax[a])) * nsho(p.atom_lmax[a]);
        w.n = off.back();
        std::vector<uint32_t> desc(size_t(p.nAtomImages) * 3 + p.col_pos.size());
        for (uint32_t i = 0; i < p.nAtomImages; ++i) {
            uint32_t const a = p.image_atom[i];
            desc[3 * size_t(i)] = p.atom_starts[a];
            desc[3 * size_t(i) + 1] = uint32_t(off[a]);
            desc[3 * size_t(i) + 2] = uint32_t(off[a] >> 32);
        }
        std::memcpy(desc.data() + size_t(p.nAtomImages) * 3, p.col_pos.data(), p.col_pos.size() * sizeof(float));
        if (!d.atom_coef)
            if (int r = dalloc(d, d.atom_coef, std::max<size_t>(1, size_t(d.ncoeffs) * d.nCols * 128), err)) return r;
        if (!w.D)
            if (int r = dalloc(d, w.D, std::max<size_t>(1, w.n), err)) return r;
        if (int r = dupload(d, w.desc, desc, err)) return r;
    }
    if (d.nAtoms == 0 || d.nchunks == 0 || w.n == 0) {
        std::fill(D, D + w.n, 0.0);
        return 0;
    }
    if (int r = project_collect(d, X, d.atom_coef, stream, err)) return r;
    hipLaunchKernelGGL(k_density, dim3(d.nAtomImages, d.max_atom_nc), dim3(256), 0, stream, w.D, d.atom_coef, d.image_pos,
                       d.image_lmax, d.image_phase, w.desc, d.nAtomImages, d.nCols, s.hgrid[0], s.hgrid[1], s.hgrid[2],
                       s.hgrid[3], factor);
    HIP_TRY(hipGetLastError());
    HIP_TRY(hipMemcpyAsync(D, w.D, size_t(w.n) * sizeof(double), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return 0;
}

int device_gradient(DevicePlan& d, Plan const& p, ActionScalars const& s, double const* X, double const* Lam,
                    std::vector<double> const& wE, double* grad_V, std::vector<double>& gmat_host,
                    hipStream_t stream, std::string& err) {
    auto& g = d.grad;
    if (!g.ready) {
        // cell -> blocks that read its potential, ascending block order
        std::vector<uint32_t> start(p.ncell() + 1, 0), blocks;
        for (uint64_t b = 0; b < p.nnzb; ++b) if (p.veff_index[b] >= 0) ++start[p.veff_index[b] + 1];
        for (uint64_t v = 0; v < p.ncell(); ++v) start[v + 1] += start[v];
        blocks.resize(start.back());
        std::vector<uint32_t> fill(start.begin(), start.end() - 1);
        for (uint64_t b = 0; b < p.nnzb; ++b) if (p.veff_index[b] >= 0) blocks[fill[p.veff_index[b]]++] = uint32_t(b);
        int r;
        if ((r = dupload(d, g.cell_start, start, err))) return r;
        if ((r = dupload(d, g.cell_blocks, blocks, err))) return r;
        if ((r = dalloc(d, g.gpart, size_t(p.nnzb) * 64, err))) return r;
        if ((r = dalloc(d, g.gcell, size_t(p.ncell()) * 64, err))) return r;
        if ((r = dalloc(d, g.wE, size_t(4) * p.nCols, err))) return r;
        size_t const nco = std::max<size_t>(1, size_t(d.ncoeffs) * d.nCols * 128);
        if ((r = dalloc(d, g.cX, nco, err))) return r;
        if ((r = dalloc(d, g.cL, nco, err))) return r;
        if ((r = dalloc(d, g.gmat, std::max<size_t>(1, p.atom_mat_off.back()), err))) return r;
        g.ready = true;
    }
    HIP_TRY(hipMemcpyAsync(g.wE, wE.data(), wE.size() * sizeof(double), hipMemcpyHostToDevice, stream));
    hipLaunchKernelGGL(k_grad_v_blocks, dim3(uint32_t(p.nnzb)), dim3(256), 0, stream, g.gpart, X, Lam, d.colindx,
                       d.veff, g.wE);
    hipLaunchKernelGGL(k_grad_v_cells, dim3(uint32_t(p.ncell())), dim3(64), 0, stream, g.gcell, g.gpart, g.cell_start,
                       g.cell_blocks, uint32_t(p.nb[0]), uint32_t(p.nb[1]));
    HIP_TRY(hipGetLastError());
    if (d.nAtoms > 0 && d.nchunks > 0) {
        for (int v = 0; v < 2; ++v)
            if (int r = project_collect(d, v ? Lam : X, v ? g.cL : g.cX, stream, err)) return r;
        hipLaunchKernelGGL(k_grad_atoms, dim3(d.nAtoms, d.max_atom_nc, (d.max_atom_nc + 3) / 4), dim3(256), 0, stream, g.gmat, g.cX, g.cL,
                           d.atom_lmax, d.atom_starts, d.atom_mat_off, g.wE, d.nCols);
        HIP_TRY(hipGetLastError());
    }
    gmat_host.assign(p.atom_mat_off.back(), 0.0);
    if (grad_V)   // (on a stream of its own, beside the kernels above, 691 -> 594 us in all; but creating one costs ms)
        HIP_TRY(hipMemcpyAsync(grad_V, g.gcell, size_t(p.ncell()) * 64 * sizeof(double), hipMemcpyDeviceToHost, stream));
    if (d.nAtoms > 0 && d.nchunks > 0 && !gmat_host.empty())
        HIP_TRY(hipMemcpyAsync(gmat_host.data(), g.gmat, gmat_host.size() * sizeof(double), hipMemcpyDeviceToHost, stream));
    HIP_TRY(hipStreamSynchronize(stream));
    return 0;
}

}  // namespace gfa
