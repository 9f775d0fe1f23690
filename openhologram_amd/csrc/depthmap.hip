// depthmap.hip -- depth-map layer hologram (angular-spectrum method) on gfx950.
//
// Replaces HologramGenerator's CPU/GPU paths (DM/Hologram/src/
// HologramGenerator_CPU.cpp:44-270, HologramGenerator_GPU.cpp:194-368,
// HologramKernel.cu:10-187, HologramGenerator.cpp:391-522).  Per colour:
//   u_l   = img/255 [img > 0] [idx == l]                  (CPU.cpp:57-66,139-141)
//   U     = rho sum_l exp(i k z_l) H_l . fftshift(FFT2(fftshift(u_l)))
//                                                          (CPU.cpp:152-160)
//   H_l   = exp(i k (-z_l) sqrt(1 - (lambda fx)^2 - (lambda fy)^2)) on the
//           reference's grids fx = -1/(2px) + x/Sx, fy = 1/(2py) - 1/Sy - y/Sy
//                                                          (CPU.cpp:196-216)
//   encode: keep centred spectrum rows [cropy1, cropy2], normalised inverse
//           fftwShift, times exp(i 2 pi yy/(4 py)), real part (CPU.cpp:231-270,
//           HologramGenerator.cpp:481-522)
// with the scene (w x h) embedded in an Nx x Ny transform grid (Nx = w,
// Ny = h reproduces the reference, which does not pad).
//
// The two fftshifts around each transform cancel against the shifts of the
// encode: with k in FFT order, U_ref(y(k)) = (-1)^(kx+ky) A(k) where
// A = sum_l m_l H_l(y(k)) FFT2(u_l), and the encoded field is IFFT2(crop(A)).
// So the pipeline works on plain FFTs and evaluates H at the reference's
// (off-by-one in fy) frequency of each FFT-order index:
//   fx = s(kx)/Sx,  |fy| = |s(ky) + 1|/Sy,  s(k) = k < N/2 ? k : k - N.
// The carrier exp(i k z_l) cancels the constant part of H, leaving the phase
//   (z_l lambda / 2)(fx^2 + fy^2) + (z_l/lambda) p(u),
//   p(u) = u^2/8 + u^3/16 + 5u^4/128 + 7u^5/256,  u = lambda^2 (fx^2 + fy^2),
// whose first term is reduced per axis in FP64.
//
// Passes (per colour; the depth index is shared):
//   dm_index  depth index of every pixel by a 256-entry table of the u8 depth
//             (built on the host; the reference makes one pass per level);
//   dm_cols   a workgroup owns 4 scene columns and every n-th layer; two
//             real columns are packed into one complex column, transformed
//             along y (length Ny) and separated; only rows ky <= Ny/2 are
//             stored (Hermitian symmetry of real input), and of these, for an
//             encoded output, only those whose row pair the crop keeps (half:
//             K below; 3 x 1920 x 1080 on 4096 x 2048, 256 layers: row pass
//             3196 -> 1720 us a colour by this alone), with a presence flag
//             per (layer, column group) -- absent groups are never written;
//   dm_rows   a workgroup owns the row pair (ky, Ny-ky): per layer it
//             transforms row ky along x once and obtains row Ny-ky from the
//             same transform by symmetry, multiplies both by H and
//             accumulates over its layers; then the encode crop, the inverse
//             row transforms, and the scene columns are stored.  Pairs that do
//             not fill the chip have their layers split over workgroups, whose
//             sums dm_rows_sum adds (rows_plan below);
//             Rows 0 and Ny/2 are real (transforms of real columns at the DC
//             and Nyquist frequencies): pair 0 packs them into one complex row
//             and separates the transform;
//   dm_final  inverse column transform, 1/(Nx Ny), the shift phase and the
//             real part (or the complex field) in the scene window.
#include <algorithm>
#include <cmath>
#include <vector>

#include "fft_engine.h"
#include "fft_kernels.h"
#include "fft_mixed.h"

namespace {

constexpr int GROUP = 4;        // scene columns per dm_cols workgroup (2 complex lines)
constexpr int MAX_LAYERS = 4096;

struct DmArgs {
    int w, h, Nx, Ny, ox, oy;
    int L, lo, hi;                 // layers 1..L, rendered range [lo, hi]
    int ngroups;
    const unsigned char* img;      // h x w, this colour
    const unsigned short* idx;     // h x w
    float2* I;                     // [L][ngroups][K][GROUP]: each column group's rows
                                   // contiguous (I_l(ky, x) at group x / GROUP)
    int K;                         // stored rows: ky = 0 .. K - 2, then Ny/2
    unsigned char* flags;          // [L][ngroups]
    unsigned char* any;            // [L]
    unsigned* fbits;               // [L][fwpl]: the flags as bits (group g: word g/32, bit g%32)
    int fwpl;                      // words per layer of fbits
    const double* lc;              // per layer: cx, cy, K (3 doubles)
    float ux, uy;                  // lambda^2 / Sx^2, lambda^2 / Sy^2
    int exact;                     // FP64 transfer path
    int horner;                    // equally spaced layers: chunked recurrence in dm_rows_h
    double dcx, dcy, dK;           // layer-step constants (z_{l+1} - z_l replacing z_l)
    double lam2_sx2, lam2_sy2, inv_lambda;
    float2 rho;
    int encode, cy1, cy2;          // crop range (centred rows) when encoding
    float2* T;                     // [Ny][w] after the inverse row transform
    float2* spectrum;              // optional centred spectrum [Ny][Nx]
    double scale;                  // 1/(Nx Ny)
    int n_main, nsplit, per;       // row pairs taken whole; workgroups per further pair, their layers
    int nsums;                     // ... and their partial sums:
    float2* part;                  // [pair][nsums][2][Nx]
    double* fringe;                // h x w (double) or
    float* fringe32;               // h x w (float) or
    float2* field;                 // h x w complex
};

__device__ __forceinline__ int sgnidx(int k, int n) { return k < n / 2 ? k : k - n; }

// ---- depth index -------------------------------------------------------------

// The depth index depends on the u8 depth value only: the host forms the
// 256-entry table (depth_index_table) and every pixel is one lookup.
__global__ void dm_index(const unsigned char* dep, int n, const double* table, unsigned short* idx) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    idx[i] = (unsigned short)table[dep[i]];
}

__global__ void dm_zero(unsigned char* p, int n) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0;
}

// Z = FFT(a + i b) of two real rows a, b; on entry z = Z(k), zc = conj Z(-k).
// On exit z = A(k) = (Z(k) + conj Z(-k))/2 and zc = B(k) = (Z(k) - conj Z(-k))/(2i).
__device__ __forceinline__ void split_real_pair(float2& z, float2& zc) {
    const float dx = z.x - zc.x, dy = z.y - zc.y;
    z = make_float2(0.5f * (z.x + zc.x), 0.5f * (z.y + zc.y));
    zc = make_float2(0.5f * dy, -0.5f * dx);
}

// ---- column pass ---------------------------------------------------------------

// A pixel's amplitude, rounded by itself (not fused into the additions after it)
__device__ __forceinline__ float pixel_value(unsigned img) {
#pragma clang fp contract(off)
    return (float)img * (1.f / 255.f);
}

// The pixels (idx << 16 | img) of grid rows row(m), M0 <= m < M1, of columns x
// and x + 1, and the layers they are in; 0 for a pixel that contributes nothing
// (alpha = [img > 0], CPU.cpp:61; a layer outside lo .. hi; no pixel).  Range-
// checked loads, all requested before the first is used.
template <int M0, int M1, int N, typename Row>
__device__ __forceinline__ void load_pixels(const DmArgs& a, int x, Row&& row, unsigned* mask, unsigned (&pa)[N],
                                            unsigned (&pb)[N]) {
    const unsigned npx = (unsigned)a.w * (unsigned)a.h;
    const auto ri = oph_buf_rsrc(a.img, npx), rd = oph_buf_rsrc(a.idx, npx * 2u);
    unsigned char im[2][N];
    unsigned short id[2][N];
#pragma unroll
    for (int m = M0; m < M1; ++m) {
        const int r = row(m) - a.oy;
        const bool in = r >= 0 && r < a.h;
        const unsigned o = (unsigned)r * (unsigned)a.w + (unsigned)x;
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const bool ok = in && x + c < a.w;
            im[c][m] = __builtin_amdgcn_raw_buffer_load_b8(ri, ok ? o + c : OPH_BUF_OOB, 0, 0);
            id[c][m] = __builtin_amdgcn_raw_buffer_load_b16(rd, ok ? 2u * (o + c) : OPH_BUF_OOB, 0, 0);
        }
    }
#pragma unroll
    for (int m = M0; m < M1; ++m)
#pragma unroll
        for (int c = 0; c < 2; ++c) {
            const unsigned d = id[c][m], i = im[c][m];
            const bool on = i > 0u && d >= (unsigned)a.lo && d <= (unsigned)a.hi;
            if (on) atomicOr(&mask[d >> 5], 1u << (d & 31));
            (c ? pb : pa)[m] = on ? d << 16 | i : 0u;
        }
}

// A thread owns 16 rows of a column pair (x0 + 2p, x0 + 2p + 1; neighbouring
// threads take the two pairs): their pixels stay in registers over all of the
// layers, a layer's values go straight into the transform's first radix-16
// stage, and the result is separated from registers -- only the mirrored
// rows that the stored ones need pass through LDS.  Bound by vector
// instructions and LDS; 1920 x 1080 on 2048 rows, 256 layers: 442 us a colour,
// against 921 with pixels, input and output of the transform in LDS and runs
// of layers instead of every chunks-th.
template <int LY>
__host__ __device__ constexpr bool cols_shared() { return LY > 4096; }   // the mirrored rows in the line itself
template <int LY>
__host__ __device__ constexpr int cols_mirror_stride(int K) { return cols_shared<LY>() ? 0 : (K + 31) / 32 * 32 + 16; }

// HALF: only the row pairs of an encoded output's crop are stored (K = Ny/4 +
// 3); its row Ny/2 is of no pair that is kept and stays zero.  MID: the scene's
// rows are among the middle ten sixteenths of the grid's.
template <int LY, bool HALF, bool MID>
__global__ __launch_bounds__(2 * (LY / 16)) void dm_cols(DmArgs a, int chunks,
                                                         const float2* __restrict__ twy) {
    constexpr int TPL = LY / 16;
    constexpr int NT = 2 * TPL;
    constexpr int M0 = MID ? 3 : 0, M1 = MID ? 13 : 16;
    extern __shared__ unsigned char smem[];
    const int p = threadIdx.x & 1, t = threadIdx.x >> 1;
    constexpr int PL = fft::skewed_len(LY, 2);
    constexpr bool SHARED = cols_shared<LY>();
    float2* line = reinterpret_cast<float2*>(smem) + p * PL;
    const int ms = cols_mirror_stride<LY>(a.K);
    float2* mirrors = reinterpret_cast<float2*>(smem) + 2 * PL;
    float2* mirror = SHARED ? line : mirrors + p * ms;               // Z(-k) at k = 1 .. K - 2
    unsigned* mask = reinterpret_cast<unsigned*>(mirrors + 2 * ms);  // layer bitmask
    // XCD-aware: neighbouring column groups (whose 32-byte row segments share
    // cache lines of I) run on the same XCD at the same time
    const int lin = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    const int g = lin % gridDim.x;
    const int chunk = lin / gridDim.x;   // layers lo + chunk, then every chunks-th
    const int nwords = (a.L + 32) / 32;
    for (int i = threadIdx.x; i < nwords; i += NT) mask[i] = 0u;
    __syncthreads();
    unsigned pa[16], pb[16];   // idx << 16 | img; 0: no contribution
    load_pixels<M0, M1>(a, g * GROUP + 2 * p, [&](int m) { return t + m * TPL; }, mask, pa, pb);
    fft::Twiddles<LY> Tw;   // (8192: too many registers with 1024 threads)
    if constexpr (!SHARED) Tw.load(twy, t);
    __syncthreads();
    const size_t gstride = (size_t)a.K * GROUP;
    const size_t lstride = gstride * a.ngroups;
    for (int l = a.lo + chunk; l <= a.hi; l += chunks) {
        if (!((mask[l >> 5] >> (l & 31)) & 1u)) continue;
        // the two real columns as one complex column
        float2 v[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            if (m < M0 || m >= M1) {
                v[m] = make_float2(0.f, 0.f);
                continue;
            }
            const unsigned wa = pa[m] >> 16 == (unsigned)l ? pa[m] : 0u;
            const unsigned wb = pb[m] >> 16 == (unsigned)l ? pb[m] : 0u;
            v[m] = make_float2(pixel_value(wa & 255u), pixel_value(wb & 255u));
        }
        if constexpr (SHARED)
            fft::line_regs_tw<LY, -1, M0, M1>(v, line, twy, t);
        else
            fft::line_regs<LY, -1, M0, M1>(v, line, Tw, t);
        if constexpr (!HALF) {
            // every element here, none computed within the branch that uses it
            // (a product and the addition after it would then round apart)
#pragma unroll
            for (int m = 0; m < 16; ++m) asm volatile("" : "+v"(v[m].x), "+v"(v[m].y));
        }
        // the mirrored rows (the previous layer's were read before the
        // barriers of this layer's transform; LY = 16 has none)
        if constexpr (SHARED || LY == 16) __syncthreads();
#pragma unroll
        for (int m = HALF ? 11 : 7; m < 16; ++m) {
            const int k = LY - (t + m * TPL);
            if (k < a.K - 1) mirror[k] = v[m];
        }
        __syncthreads();
        // separate: A(k) = (Z(k) + conj Z(-k))/2, B(k) = (Z(k) - conj Z(-k))/(2i)
        float2* dst = a.I + (size_t)(l - 1) * lstride + (size_t)g * gstride + 2 * p;
        constexpr float sc = 0.5f;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int k = t + m * TPL;
            if (m <= (HALF ? TPL == 1 ? 5 : 4 : 7) && k < a.K - 1) {
                const float2 z = v[m], zm = k == 0 ? z : mirror[k];
                *reinterpret_cast<float4*>(dst + (size_t)k * GROUP) =
                    make_float4(sc * (z.x + zm.x), sc * (z.y - zm.y), sc * (z.y + zm.y), sc * (zm.x - z.x));
            }
        }
        if (t == 0)
            *reinterpret_cast<float4*>(dst + (size_t)(a.K - 1) * GROUP) =
                HALF ? make_float4(0.f, 0.f, 0.f, 0.f) : make_float4(v[8].x, 0.f, v[8].y, 0.f);
        if (threadIdx.x == 0) {
            a.flags[(size_t)(l - 1) * a.ngroups + g] = 1;
            a.any[l - 1] = 1;
            atomicOr(&a.fbits[(size_t)(l - 1) * a.fwpl + (g >> 5)], 1u << (g & 31));
        }
        if constexpr (SHARED) __syncthreads();
    }
}

// ---- row pass ------------------------------------------------------------------

template <bool EXACT>
__device__ __forceinline__ float2 dm_transfer(const DmArgs& a, float tx, double ty, float usx, int sy,
                                              double K, float Kf, double sx2d) {
    const float u = fmaf(a.uy, (float)(sy * sy), usx);
    if (u >= 1.f) return make_float2(0.f, 0.f);
    float ph;
    if (!EXACT) {
        const float pu = u * u * fmaf(u, fmaf(u, fmaf(u, 7.f / 256.f, 5.f / 128.f), 1.f / 16.f), 0.125f);
        ph = tx + (float)ty + Kf * pu;
    } else {
        const double ud = a.lam2_sx2 * sx2d + a.lam2_sy2 * (double)sy * sy;
        if (ud >= 1.0) return make_float2(0.f, 0.f);
        double t = K * ud / (1.0 + sqrt(1.0 - ud));
        t -= rint(t);
        ph = (float)t;
    }
    return make_float2(cos_turns(ph), sin_turns(ph));
}

// Optional centred spectrum of one accumulated row, the encode crop, the
// inverse row transform and the store of the scene columns into T.
template <int LX>
__device__ __forceinline__ void finish_row(const DmArgs& a, const float2 (&acc)[16], int ky, float2* line,
                                           const float2* __restrict__ tw, int t) {
    constexpr int TPL = LX / 16;
    const int yc = (ky + a.Ny / 2) & (a.Ny - 1);
    if (a.spectrum) {
        // U_ref(y, x) = (-1)^(kx + ky) A(ky, kx), y, x centred indices
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int kx = t + m * TPL;
            const int xc = (kx + LX / 2) & (LX - 1);
            const float sg = ((kx + ky) & 1) ? -1.f : 1.f;
            a.spectrum[(size_t)yc * LX + xc] = make_float2(sg * acc[m].x, sg * acc[m].y);
        }
    }
    const bool kept = !a.encode || (yc >= a.cy1 && yc <= a.cy2);
    if (!kept) return;  // uniform over the workgroup
#pragma unroll
    for (int m = 0; m < 16; ++m) line[fft::lane_pad<LX>(t, m)] = acc[m];
    __syncthreads();
    fft::line_tw<LX, +1>(line, tw, t);
    float2* dst = a.T + (size_t)ky * a.w;
    for (int x = t; x < a.w; x += TPL) dst[x] = line[fft::pad16(x + a.ox)];
    __syncthreads();
}

template <int LX, bool EXACT>
__global__ __launch_bounds__(LX / 16) void dm_rows(DmArgs a, const float2* __restrict__ twx) {
    constexpr int TPL = LX / 16;
    constexpr int PL = fft::padded_len(LX);
    __shared__ float2 line[PL];
    const int t = threadIdx.x;
    const int kya = xcd_remap(blockIdx.x, gridDim.x);  // 0 .. K - 2
    const bool pair0 = kya == 0;              // real rows 0 and Ny/2 packed as re/im
    const int kyb = pair0 ? a.Ny / 2 : a.Ny - kya;
    const int sya = sgnidx(kya, a.Ny) + 1;
    const int syb = sgnidx(kyb, a.Ny) + 1;
    const size_t nyq = (size_t)(a.K - 1) * GROUP;  // row Ny/2 relative to row 0
    const size_t gstride = (size_t)a.K * GROUP;
    fft::Twiddles<LX> Tw;
    Tw.load(twx, t);
    float2 acca[16], accb[16];
    float usx[16];
    double sx2[16];
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        acca[m] = accb[m] = make_float2(0.f, 0.f);
        const int sx = sgnidx(t + m * TPL, LX);
        sx2[m] = (double)sx * sx;
        usx[m] = a.ux * (float)(sx * sx);
    }
    const size_t lstride = gstride * a.ngroups;
    for (int l = a.lo; l <= a.hi; ++l) {
        if (!a.any[l - 1]) continue;
        const float2* src = a.I + (size_t)(l - 1) * lstride + (size_t)kya * GROUP;
        const unsigned char* fl = a.flags + (size_t)(l - 1) * a.ngroups;
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int x = t + m * TPL - a.ox;
            float2 v = make_float2(0.f, 0.f);
            if (x >= 0 && x < a.w && fl[x / GROUP]) {
                const size_t o = (size_t)(x / GROUP) * gstride + x % GROUP;
                v = src[o];
                if (pair0) v.y = src[nyq + o].x;
            }
            line[fft::lane_pad<LX>(t, m)] = v;
        }
        __syncthreads();
        fft::line<LX, -1>(line, Tw, t);
        const double cx = a.lc[3 * (l - 1)], cy = a.lc[3 * (l - 1) + 1], K = a.lc[3 * (l - 1) + 2];
        const float Kf = (float)K;
        double tya = cy * (double)sya * sya;
        tya -= rint(tya);
        double tyb = cy * (double)syb * syb;
        tyb -= rint(tyb);
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int kx = t + m * TPL;
            double txd = cx * sx2[m];
            txd -= rint(txd);
            const float tx = (float)txd;
            float2 gv = line[fft::lane_pad<LX>(t, m)];
            const float2 gm = line[fft::pad16((LX - kx) & (LX - 1))];
            float2 gmc = make_float2(gm.x, -gm.y);
            if (pair0) split_real_pair(gv, gmc);
            const float2 ha = dm_transfer<EXACT>(a, tx, tya, usx[m], sya, K, Kf, sx2[m]);
            acca[m] = fft::cadd(acca[m], fft::cmul(ha, gv));
            const float2 hb = dm_transfer<EXACT>(a, tx, tyb, usx[m], syb, K, Kf, sx2[m]);
            accb[m] = fft::cadd(accb[m], fft::cmul(hb, gmc));
        }
        __syncthreads();
    }
    // rho (the same for every layer), optional centred spectrum, encode crop,
    // inverse row transform
#pragma unroll
    for (int m = 0; m < 16; ++m) {
        acca[m] = fft::cmul(acca[m], a.rho);
        accb[m] = fft::cmul(accb[m], a.rho);
    }
    finish_row<LX>(a, acca, kya, line, twx, t);
    finish_row<LX>(a, accb, kyb, line, twx, t);
}

// Row pass of power-of-two rows of 64 to 4096.  MODE 1 and 2 (a field lens, or
// a pitch that needs the transfer in full: 2) evaluate the transfer of every
// layer; against one thread per 16 elements (dm_rows below 64 and at 8192:
// 434 registers, one wave per SIMD, a line's loads waited for before its
// transform) a frame of 512^2, 64 layers fell from 482 to 69 us and of
// 4096 x 2048 from 1782 to 763; held to 168 or 128 registers it spills
// (1135, 1432 us).
//
// A scene in the middle half of the columns (HALF) loads half of the row and
// spares the first butterfly's operations on zeros; rows of 4096 go through
// line_r8_split4096 (together 1700 -> 1430 us at 4096 x 2048 encoded, 256
// layers; shorter rows keep the stage order and with it the bits of the learned
// pipeline's fields, and were not timed split).
//
// MODE 0: equally spaced layers (no field lens).  The transfer of
// layer l is H_l = exp(i 2 pi z_l Phi(kx, ky)) with one Phi for all layers,
// so over a chunk of 16 consecutive layers starting at c,
//   sum_j H_{c+j} G_{c+j} = H_c sum_j R^j G_{c+j},   R = exp(i 2 pi dz Phi),
// evaluated by Horner from the top layer down (T = T R + G_l): one complex
// multiply-add per element and layer instead of the phase reduction, series
// and sin/cos, which are evaluated once per chunk for the anchor H_c (the
// recurrence's rounding stays within ~16 ulp).  The row transforms are
// radix-8 with LX/8 threads (8 elements per thread) so that R and T of both
// rows fit in registers next to the transform; the chunk sums S accumulate
// in LDS, each element touched only by its owner thread.  The twiddle table
// and a bitmask of the present layers are copied to LDS at the start, so
// that inside the layer loop only the prefetched rows are global loads.
template <int LX, int MODE>
__host__ __device__ constexpr size_t rows_h_lds() {
    return (fft::padded_len(LX) + (MODE == 0 ? 2 * (size_t)LX : 0) + fft::table_len8(LX)) * sizeof(float2) +
           (size_t)(MAX_LAYERS / 32) * sizeof(unsigned);
}

// finish_row for the radix-8 layout (8 elements per thread)
template <int LX>
__device__ __forceinline__ void finish_row8(const DmArgs& a, const float2 (&acc)[8], int ky, float2* line,
                                            const float2* __restrict__ tw8, int t) {
    constexpr int TPL = LX / 8;
    const int yc = (ky + a.Ny / 2) & (a.Ny - 1);
    if (a.spectrum) {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int kx = t + m * TPL;
            const int xc = (kx + LX / 2) & (LX - 1);
            const float sg = ((kx + ky) & 1) ? -1.f : 1.f;
            a.spectrum[(size_t)yc * LX + xc] = make_float2(sg * acc[m].x, sg * acc[m].y);
        }
    }
    const bool kept = !a.encode || (yc >= a.cy1 && yc <= a.cy2);
    if (!kept) return;  // uniform over the workgroup
#pragma unroll
    for (int m = 0; m < 8; ++m) line[fft::pad16(t + m * TPL)] = acc[m];
    __syncthreads();
    fft::line_r8<LX, +1>(line, tw8, t);
    float2* dst = a.T + (size_t)ky * a.w;
    for (int x = t; x < a.w; x += TPL) dst[x] = line[fft::pad16(x + a.ox)];
    __syncthreads();
}

// PAIR0: workgroup 0, the real rows 0 and Ny/2 packed as re/im.  FBITS:
// the presence bits of every (layer, group) fit in LDS.
// Copies n elements of a table to LDS with NT threads, eight loads per
// thread requested before any is stored (a plain loop waits for each load
// before the next is issued).
template <int NT, typename E>
__device__ __forceinline__ void lds_copy(E* dst, const E* __restrict__ src, int n, int t) {
    for (int i0 = 0; i0 < n; i0 += 8 * NT) {
        E v[8];
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int i = i0 + t + j * NT;
            if (i < n) v[j] = src[i];
        }
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const int i = i0 + t + j * NT;
            if (i < n) dst[i] = v[j];
        }
    }
}

// lo .. hi: the layers taken (MODE 0: in chunks from lo).  part: the sums of
// both rows are written there instead of being finished; CHUNKS (MODE 0): of
// each chunk, one after the other.  HALF: the scene's
// columns are among the middle half of the grid's, so of a thread's eight
// inputs the outer four are zeros.
template <int LX, int MODE, bool PAIR0, bool FBITS, bool HALF, bool CHUNKS>
__device__ __forceinline__ void rows_h_body(const DmArgs& a, const float2* __restrict__ tw8, float2* sm, int kya,
                                            int lo, int hi, float2* part) {
    constexpr int TPL = LX / 8;
    constexpr int PL = fft::padded_len(LX);
    constexpr int CH = 16;
    constexpr int NTW = fft::table_len8(LX);
    constexpr bool SPLIT = LX == 4096;
    constexpr int M0 = HALF ? 2 : 0, M1 = HALF ? 6 : 8;
    float2* line = sm;
    float2* Sa = sm + PL;             // MODE 0, not CHUNKS: the chunk sums of both rows
    float2* Sb = Sa + LX;
    float2* tws = sm + PL + (MODE == 0 ? 2 * LX : 0);
    unsigned* amask = reinterpret_cast<unsigned*>(tws + NTW);
    // presence bits of every (layer, column group), when they fit in LDS:
    // then only present groups' rows of I are loaded
    unsigned* fb = amask + MAX_LAYERS / 32;
    const int t = threadIdx.x;
    lds_copy<TPL>(tws, tw8, NTW, t);
    for (int i = t; i < MAX_LAYERS / 32; i += TPL) amask[i] = 0u;
    if constexpr (FBITS) lds_copy<TPL>(fb, a.fbits, a.L * a.fwpl, t);
    __syncthreads();
    for (int i = t; i < a.L; i += TPL)
        if (a.any[i]) atomicOr(&amask[i >> 5], 1u << (i & 31));
    __syncthreads();
    auto present = [&](int l) -> bool { return (amask[(l - 1) >> 5] >> ((l - 1) & 31)) & 1u; };
    const int kyb = PAIR0 ? a.Ny / 2 : a.Ny - kya;
    const int sya = sgnidx(kya, a.Ny) + 1;
    const int syb = sgnidx(kyb, a.Ny) + 1;
    const size_t nyq = (size_t)(a.K - 1) * GROUP;
    const size_t gstride = (size_t)a.K * GROUP;
    // Thread t owns row a at kx = tk + m TPL (tk: as the transform leaves them) and row b at kb = -kx mod LX:
    // row b's transform at kb is conj Z(kx) of the thread's own element of
    // row a's transform Z, and the transfer depends on kx only through kx^2,
    // which is the same at kb, so one set of per-element factors serves both.
    const int tk = SPLIT ? fft::split_k(t) : t;
    const auto slot = [](int k) { return SPLIT ? (k & ~(TPL - 1)) + fft::split_slot(k & (TPL - 1)) : k; };
    float2 Ra[8], Rb[8];   // MODE 0
    float2 Ta[8], Tb[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) Ta[m] = Tb[m] = make_float2(0.f, 0.f);
    if constexpr (MODE == 0) {
        double tya = a.dcy * (double)sya * sya;
        tya -= rint(tya);
        double tyb = a.dcy * (double)syb * syb;
        tyb -= rint(tyb);
        const float dKf = (float)a.dK;
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int sx = sgnidx(tk + m * TPL, LX);
            const double sx2 = (double)sx * sx;
            double txd = a.dcx * sx2;
            txd -= rint(txd);
            const float usx = a.ux * (float)(sx * sx);
            Ra[m] = dm_transfer<false>(a, (float)txd, tya, usx, sya, a.dK, dKf, sx2);
            Rb[m] = dm_transfer<false>(a, (float)txd, tyb, usx, syb, a.dK, dKf, sx2);
            if constexpr (!CHUNKS) Sa[t + m * TPL] = Sb[t + m * TPL] = make_float2(0.f, 0.f);   // at its owner's place
        }
    }
    const size_t lstride = gstride * a.ngroups;
    // Layers are taken chunk by chunk, top layer first within a chunk.  The
    // row of the next present layer in that order is loaded into registers
    // (values and presence flags) before the current layer's transform, so
    // its latency hides behind the transform.
    auto next_layer = [&](int l) -> int {
        for (;;) {
            const int c = lo + (l - lo) / CH * CH;
            l = l > c ? l - 1 : (c + CH <= hi ? min(hi, c + 2 * CH - 1) : 0);
            if (l == 0 || present(l)) return l;
        }
    };
    float2 nv[8];
    unsigned nf;  // presence of the prefetched elements, bit m for element m
    auto fetch = [&](int l) {
        const float2* src = a.I + (size_t)(l - 1) * lstride + (size_t)kya * GROUP;
        if constexpr (FBITS) {
            // flags from LDS first; then range-checked buffer loads whose
            // offset is out of range for absent groups (no memory access, a
            // zero result, no branch): the rows of absent groups were never
            // written and are not read, and the loaded values need no mask
            nf = 0xFFu;
            const unsigned* fl = fb + (size_t)(l - 1) * a.fwpl;
            const auto rs = oph_buf_rsrc(a.I + (size_t)(l - 1) * lstride, (unsigned)(lstride * sizeof(float2)));
#pragma unroll
            for (int m = M0; m < M1; ++m) {
                const int x = t + m * TPL - a.ox;
                const int gx = x >> 2;  // x / GROUP for x >= 0
                const bool on = (x >= 0 && x < a.w) && ((fl[gx >> 5] >> (gx & 31)) & 1u);
                const unsigned o = (unsigned)(((size_t)gx * gstride + (x & 3) + (size_t)kya * GROUP) * sizeof(float2));
                if constexpr (PAIR0) {
                    const float2 lo = oph_buf_load_f2(rs, on ? o : OPH_BUF_OOB);
                    const float2 hi = oph_buf_load_f2(rs, on ? o + (unsigned)(nyq * sizeof(float2)) : OPH_BUF_OOB);
                    nv[m] = make_float2(lo.x, hi.x);
                } else {
                    nv[m] = oph_buf_load_f2(rs, on ? o : OPH_BUF_OOB);
                }
            }
            return;
        }
        const unsigned char* fl = a.flags + (size_t)(l - 1) * a.ngroups;
        nf = 0u;
#pragma unroll
        for (int m = M0; m < M1; ++m) {
            const int x = t + m * TPL - a.ox;
            const bool in = x >= 0 && x < a.w;
            const size_t o = (size_t)(x / GROUP) * gstride + x % GROUP;
            nf |= (in && fl[x / GROUP]) ? 1u << m : 0u;
            if constexpr (PAIR0)
                nv[m] = in ? make_float2(src[o].x, src[nyq + o].x) : make_float2(0.f, 0.f);
            else
                nv[m] = in ? src[o] : make_float2(0.f, 0.f);
        }
    };
    // MODE != 0: T += H_l G_l, the transfer evaluated for every layer
    auto add_layer = [&](int l, const float2 (&va)[8], const float2 (&vb)[8]) {
        const double cx = a.lc[3 * (l - 1)], cy = a.lc[3 * (l - 1) + 1], K = a.lc[3 * (l - 1) + 2];
        const float Kf = (float)K;
        double tya = cy * (double)sya * sya;
        tya -= rint(tya);
        double tyb = cy * (double)syb * syb;
        tyb -= rint(tyb);
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int sx = sgnidx(tk + m * TPL, LX);
            const double sx2 = (double)(sx * sx);
            double txd = cx * sx2;
            txd -= rint(txd);
            const float usx = a.ux * (float)(sx * sx);
            const float2 ha = dm_transfer<MODE == 2>(a, (float)txd, tya, usx, sya, K, Kf, sx2);
            Ta[m] = fft::cadd(Ta[m], fft::cmul(ha, va[m]));
            const float2 hb = dm_transfer<MODE == 2>(a, (float)txd, tyb, usx, syb, K, Kf, sx2);
            Tb[m] = fft::cadd(Tb[m], fft::cmul(hb, PAIR0 ? vb[m] : make_float2(va[m].x, -va[m].y)));
        }
    };
    int pl = min(hi, lo + CH - 1);
    if (!present(pl)) pl = next_layer(pl);
    if (pl) fetch(pl);
    for (int cs = lo; cs <= hi; cs += CH) {
        const int ce = min(hi, cs + CH - 1);
        bool anyc = false;
        for (int l = cs; l <= ce; ++l) anyc |= present(l);
        float2* sums = part + (size_t)((cs - lo) / CH) * 2 * LX;   // CHUNKS: this chunk's
        if (!anyc) {
            if constexpr (CHUNKS) {
#pragma unroll
                for (int m = 0; m < 16; ++m) sums[t + m * TPL] = make_float2(0.f, 0.f);
            }
            continue;
        }
        if constexpr (MODE == 0) {
#pragma unroll
            for (int m = 0; m < 8; ++m) Ta[m] = Tb[m] = make_float2(0.f, 0.f);
        }
        for (int l = ce; l >= cs; --l) {
            if constexpr (MODE == 0) {
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    Ta[m] = fft::cmul(Ta[m], Ra[m]);
                    Tb[m] = fft::cmul(Tb[m], Rb[m]);
                }
            }
            if (!present(l)) continue;
            // l is the prefetched layer
            float2 v[8], vb[8];   // vb: row b of PAIR0 (MODE != 0)
#pragma unroll
            for (int m = 0; m < 8; ++m)
                v[m] = m >= M0 && m < M1 && ((nf >> m) & 1u) ? nv[m] : make_float2(0.f, 0.f);
            pl = next_layer(l);
            if (pl) fetch(pl);
            if constexpr (SPLIT) {
                fft::line_r8_split4096<-1, HALF>(v, line, tws, t);
            } else {
                __syncthreads();  // the previous transform's readers are done with the line
                fft::line_r8_regs<LX, -1, false, HALF>(v, line, tws, t);
            }
            if constexpr (PAIR0) {
                // A(kx) = (Z(kx) + conj Z(-kx))/2 for row 0 and, row Ny/2
                // being real, B(-kx) = conj B(kx): exchange through the line
                __syncthreads();
#pragma unroll
                for (int m = 0; m < 8; ++m) line[fft::pad16(tk + m * TPL)] = v[m];
                __syncthreads();
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    const int kx = tk + m * TPL;
                    const float2 gm = line[fft::pad16((LX - kx) & (LX - 1))];
                    float2 z = v[m], zc = make_float2(gm.x, -gm.y);
                    split_real_pair(z, zc);
                    v[m] = z;
                    if constexpr (MODE == 0)
                        Tb[m] = fft::cadd(Tb[m], make_float2(zc.x, -zc.y));
                    else
                        vb[m] = make_float2(zc.x, -zc.y);
                }
            }
            if constexpr (MODE == 0) {
#pragma unroll
                for (int m = 0; m < 8; ++m) {
                    Ta[m] = fft::cadd(Ta[m], v[m]);
                    if constexpr (!PAIR0) Tb[m] = fft::cadd(Tb[m], make_float2(v[m].x, -v[m].y));
                }
            } else {
                add_layer(l, v, vb);
            }
        }
        if constexpr (MODE != 0) continue;
        // anchor: S += H_cs T
        if constexpr (MODE == 0) {
            const double cx = a.lc[3 * (cs - 1)], cy = a.lc[3 * (cs - 1) + 1], K = a.lc[3 * (cs - 1) + 2];
            const float Kf = (float)K;
            double tya = cy * (double)sya * sya;
            tya -= rint(tya);
            double tyb = cy * (double)syb * syb;
            tyb -= rint(tyb);
#pragma unroll
            for (int m = 0; m < 8; ++m) {
                const int sx = sgnidx(tk + m * TPL, LX), own = t + m * TPL;
                const double sx2 = (double)sx * sx;
                double txd = cx * sx2;
                txd -= rint(txd);
                const float usx = a.ux * (float)(sx * sx);
                const float2 ha = dm_transfer<false>(a, (float)txd, tya, usx, sya, K, Kf, sx2);
                const float2 hb = dm_transfer<false>(a, (float)txd, tyb, usx, syb, K, Kf, sx2);
                if constexpr (CHUNKS) {   // in natural order: row a at kx, row b at -kx
                    const int kx = tk + m * TPL;
                    sums[kx] = fft::cmul(ha, Ta[m]);
                    sums[LX + ((LX - kx) & (LX - 1))] = fft::cmul(hb, Tb[m]);
                } else {
                    Sa[own] = fft::cadd(Sa[own], fft::cmul(ha, Ta[m]));
                    Sb[own] = fft::cadd(Sb[own], fft::cmul(hb, Tb[m]));
                }
            }
        }
    }
    if constexpr (CHUNKS) return;
    // the rows in natural order: row a's sum at kx, row b's at -kx (MODE 0: the
    // sums are already in LDS, at their owners' places)
    if constexpr (MODE == 0) {
        __syncthreads();
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            const int k = t + m * TPL;
            Ta[m] = Sa[slot(k)];
            Tb[m] = Sb[slot((LX - k) & (LX - 1))];
        }
    } else {
        const auto reorder = [&](float2 (&v)[8], int sg) {
            __syncthreads();
#pragma unroll
            for (int m = 0; m < 8; ++m) line[fft::pad16((sg * (tk + m * TPL)) & (LX - 1))] = v[m];
            __syncthreads();
#pragma unroll
            for (int m = 0; m < 8; ++m) v[m] = line[fft::pad16(t + m * TPL)];
        };
        if constexpr (SPLIT) reorder(Ta, 1);
        reorder(Tb, -1);
    }
    if (part) {
#pragma unroll
        for (int m = 0; m < 8; ++m) {
            part[t + m * TPL] = Ta[m];
            part[LX + t + m * TPL] = Tb[m];
        }
        return;
    }
#pragma unroll
    for (int m = 0; m < 8; ++m) {
        Ta[m] = fft::cmul(Ta[m], a.rho);
        Tb[m] = fft::cmul(Tb[m], a.rho);
    }
    __syncthreads();
    finish_row8<LX>(a, Ta, kya, line, tws, t);
    finish_row8<LX>(a, Tb, kyb, line, tws, t);
}

// (two waves per SIMD: 256 registers, the budget of two 2048-point
// workgroups per CU or one 4096-point workgroup)
template <int LX, int MODE, bool FBITS, bool HALF>
__global__ __launch_bounds__(LX / 8, 2) void dm_rows_h(DmArgs a, const float2* __restrict__ tw8) {
    extern __shared__ float2 sm[];
    // XCD-aware: neighbouring rows, which share the cache lines of I, run on
    // the same XCD at the same time
    int kya, lo = a.lo, hi = a.hi;
    float2* part = nullptr;
    if ((int)blockIdx.x >= a.n_main) {
        // a pair beyond the last full round of workgroups: part j of its layers
        const int lin = xcd_remap(blockIdx.x - a.n_main, gridDim.x - a.n_main), left = a.K - 1 - a.n_main;
        const int j = lin / left, i = lin - j * left;
        lo = a.lo + j * a.per;
        hi = min(a.hi, lo + a.per - 1);
        kya = a.n_main + i;
        part = a.part + ((size_t)i * a.nsums + (MODE == 0 ? j * (a.per / 16) : j)) * 2 * LX;
    } else {
        kya = xcd_remap(blockIdx.x, a.n_main);  // 0 .. n_main - 1
    }
    if constexpr (MODE == 0) {
        if (part) {
            if (kya == 0)
                rows_h_body<LX, MODE, true, FBITS, HALF, true>(a, tw8, sm, 0, lo, hi, part);
            else
                rows_h_body<LX, MODE, false, FBITS, HALF, true>(a, tw8, sm, kya, lo, hi, part);
            return;
        }
    }
    if (kya == 0)
        rows_h_body<LX, MODE, true, FBITS, HALF, false>(a, tw8, sm, 0, lo, hi, part);
    else
        rows_h_body<LX, MODE, false, FBITS, HALF, false>(a, tw8, sm, kya, lo, hi, part);
}

// The pairs whose layers were split: their partial sums in order (with the
// chunked recurrence one per chunk, and these are the additions of a whole
// pair), then as a whole pair's
template <int LX>
__global__ __launch_bounds__(LX / 8) void dm_rows_h_sum(DmArgs a, const float2* __restrict__ tw8) {
    constexpr int TPL = LX / 8;
    __shared__ float2 line[fft::padded_len(LX)];
    const int t = threadIdx.x, i = blockIdx.x >> 1, row = blockIdx.x & 1, kya = a.n_main + i;
    const int ky = row == 0 ? kya : kya == 0 ? a.Ny / 2 : a.Ny - kya;
    const float2* p = a.part + ((size_t)i * a.nsums * 2 + row) * LX;
    float2 acc[8];
#pragma unroll
    for (int m = 0; m < 8; ++m) acc[m] = make_float2(0.f, 0.f);
    for (int j = 0; j < a.nsums; ++j)
#pragma unroll
        for (int m = 0; m < 8; ++m) acc[m] = fft::cadd(acc[m], p[(size_t)2 * j * LX + t + m * TPL]);
#pragma unroll
    for (int m = 0; m < 8; ++m) acc[m] = fft::cmul(acc[m], a.rho);
    finish_row8<LX>(a, acc, ky, line, tw8, t);
}

// ---- final column pass ---------------------------------------------------------

template <int LY, int B>
__global__ __launch_bounds__(B * (LY / 16)) void dm_final(DmArgs a, const float2* __restrict__ twy) {
    constexpr int TPL = LY / 16;
    constexpr int PL = fft::padded_len(LY);
    extern __shared__ float2 lds[];
    const int nthr = B * TPL;
    const int g = xcd_remap(blockIdx.x, gridDim.x);
    const int c0 = g * B;
    const int b = threadIdx.x / TPL, t = threadIdx.x % TPL;
    fft::Twiddles<LY> Tw;
    Tw.load(twy, t);
    // 16 elements per thread (LY B / nthr), all requested before any is
    // stored (range-checked buffer loads: dropped rows and columns beyond
    // the scene read zeros; T is at most 8192 x 8192 x 8 bytes)
    {
        const auto rt = oph_buf_rsrc(a.T, (unsigned)((size_t)a.Ny * a.w * sizeof(float2)));
        float2 v[16];
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int e = threadIdx.x + m * nthr;
            const int ky = e / B, x = c0 + e % B;
            const int yc = (ky + a.Ny / 2) & (a.Ny - 1);
            const bool kept = !a.encode || (yc >= a.cy1 && yc <= a.cy2);
            v[m] = oph_buf_load_f2(rt, x < a.w && kept ? ((unsigned)ky * (unsigned)a.w + (unsigned)x) * 8u : OPH_BUF_OOB);
        }
#pragma unroll
        for (int m = 0; m < 16; ++m) {
            const int e = threadIdx.x + m * nthr;
            lds[(e % B) * PL + fft::pad16(e / B)] = v[m];
        }
    }
    __syncthreads();
    fft::line<LY, +1>(lds + b * PL, Tw, t);
    const float sc = (float)a.scale;
    for (int e = threadIdx.x; e < a.h * B; e += nthr) {
        const int bb = e % B, r = e / B;
        const int x = c0 + bb;
        if (x >= a.w) continue;
        const float2 v0 = lds[bb * PL + fft::pad16(a.oy + r)];
        const float2 v = make_float2(v0.x * sc, v0.y * sc);
        const size_t o = (size_t)r * a.w + x;
        if (a.encode) {
            // exp(i 2 pi yy/(4 py)), yy = Sy/2 - py r - py, Sy = h py (CPU.cpp:376-390)
            double tt = a.h / 8.0 - (r + 1) / 4.0;
            tt -= rint(tt);
            const float ph = (float)tt;
            const float re = v.x * cos_turns(ph) - v.y * sin_turns(ph);
            if (a.fringe) a.fringe[o] = re;
            if (a.fringe32) a.fringe32[o] = re;
        } else {
            a.field[o] = v;
        }
    }
}

// ---- general lengths -------------------------------------------------------------
// The same three passes for grids whose sides are 2^a 3^b 5^c but not powers
// of two (the shipped 11520 x 2160 configuration, HD scenes transformed
// unpadded): mixed-radix line transforms (fft_mixed.h) by NT =
// fftm::threads(N) threads per line, in natural order thread t owning elements
// t + m NT (m < fftm::ept(N)), index arithmetic mod N (N even: the fftshifts are
// still the (-1)^k factors above).  No chunked recurrence: every layer's
// transfer is evaluated (dm_transfer).

#define OPH_DM_MIXED_LENGTHS(X) X(540) X(720) X(1080) X(1920) X(2160) X(3840) X(11520)

bool dm_mixed_length(int n) {
    switch (n) {
#define OPH_DMM_CASE(v) case v:
        OPH_DM_MIXED_LENGTHS(OPH_DMM_CASE)
#undef OPH_DMM_CASE
        return true;
        default: return false;
    }
}

// As dm_cols: pixels, a layer's values and its transform's result in registers
// (1080 rows, 1920 columns, 256 layers: 595 -> 390 us with 12 x 10 x 9 in place
// of 8 x 5 x 3 x 3 x 3).
template <int LY>
__host__ __device__ constexpr int cols_m_line() {   // lines 16 float2 apart modulo all banks
    return (fftm::padded_len(LY) + 31) / 32 * 32 + 16;
}

template <int LY>
__global__ __launch_bounds__(2 * fftm::threads(LY)) void dm_cols_m(DmArgs a, int chunks,
                                                                 const float2* __restrict__ twy) {
    using E = fftm::Ends<LY>;
    constexpr int NT = E::NT;
    extern __shared__ unsigned char smem[];
    const int p = threadIdx.x & 1, t = threadIdx.x >> 1;
    float2* line = reinterpret_cast<float2*>(smem) + p * cols_m_line<LY>();
    const int ms = cols_mirror_stride<0>(a.K);
    float2* mirrors = reinterpret_cast<float2*>(smem) + 2 * cols_m_line<LY>();
    float2* mirror = mirrors + p * ms;                               // Z(-k) at k = 1 .. K - 2
    unsigned* mask = reinterpret_cast<unsigned*>(mirrors + 2 * ms);  // layer bitmask
    const int lin = xcd_remap(blockIdx.y * gridDim.x + blockIdx.x, gridDim.x * gridDim.y);
    const int g = lin % gridDim.x;
    const int chunk = lin / gridDim.x;   // layers lo + chunk, then every chunks-th
    const int nwords = (a.L + 32) / 32;
    for (int i = threadIdx.x; i < nwords; i += 2 * NT) mask[i] = 0u;
    __syncthreads();
    unsigned pa[E::PER0 * E::R0], pb[E::PER0 * E::R0];
    load_pixels<0, E::PER0 * E::R0>(
        a, g * GROUP + 2 * p,
        [&](int m) {
            const int jj = t + m / E::R0 * NT;
            return jj < E::NB0 ? jj + m % E::R0 * E::NB0 : -1;   // (-1: no row)
        },
        mask, pa, pb);
    __syncthreads();
    const size_t gstride = (size_t)a.K * GROUP;
    const size_t lstride = gstride * a.ngroups;
    for (int l = a.lo + chunk; l <= a.hi; l += chunks) {
        if (!((mask[l >> 5] >> (l & 31)) & 1u)) continue;
        // the thread index through a zero the compiler cannot see through:
        // the transforms' LDS addresses are then formed per layer instead of
        // being hoisted out of the loop into ~100 registers
        int zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        const int tl = t + zero;
        float2 vi[E::PER0][E::R0], v[E::PERL][E::RL];
#pragma unroll
        for (int m = 0; m < E::PER0 * E::R0; ++m) {
            const unsigned wa = pa[m] >> 16 == (unsigned)l ? pa[m] : 0u;
            const unsigned wb = pb[m] >> 16 == (unsigned)l ? pb[m] : 0u;
            vi[m / E::R0][m % E::R0] = make_float2(pixel_value(wa & 255u), pixel_value(wb & 255u));
        }
        fftm::line_ends<LY, -1>(vi, v, line, twy, tl);
#pragma unroll
        for (int q = 0; q < E::PERL; ++q)
#pragma unroll
            for (int r = 0; r < E::RL; ++r) {
                const int j = tl + q * NT, k = LY - (j + r * E::NBL);
                if ((E::PERL * NT == E::NBL || j < E::NBL) && k < a.K - 1) mirror[k] = v[q][r];
            }
        __syncthreads();
        // separate: A(k) = (Z(k) + conj Z(-k))/2, B(k) = (Z(k) - conj Z(-k))/(2i)
        float2* dst = a.I + (size_t)(l - 1) * lstride + (size_t)g * gstride + 2 * p;
#pragma unroll
        for (int q = 0; q < E::PERL; ++q)
#pragma unroll
            for (int r = 0; r < E::RL; ++r) {
                const int j = tl + q * NT, k = j + r * E::NBL;
                const bool nyq = k == LY / 2;
                if ((E::PERL * NT == E::NBL || j < E::NBL) && (k < a.K - 1 || nyq)) {
                    const float2 z = v[q][r], zm = k == 0 || nyq ? z : mirror[k];
                    *reinterpret_cast<float4*>(dst + (size_t)(nyq ? a.K - 1 : k) * GROUP) =
                        make_float4(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y), 0.5f * (z.y + zm.y), 0.5f * (zm.x - z.x));
                }
            }
        if (threadIdx.x == 0) {
            a.flags[(size_t)(l - 1) * a.ngroups + g] = 1;
            a.any[l - 1] = 1;
            atomicOr(&a.fbits[(size_t)(l - 1) * a.fwpl + (g >> 5)], 1u << (g & 31));
        }
    }
}

// finish_row for a row already in the line, in natural order (synced); not
// called for rows that the crop drops, unless the spectrum is wanted.
template <int LX>
__device__ __forceinline__ void finish_row_m(const DmArgs& a, int ky, float2* line, const float2* __restrict__ tw,
                                             int t) {
    constexpr int NT = fftm::threads(LX);
    const int yc = (ky + a.Ny / 2) % a.Ny;
    if (a.spectrum) {
        for (int kx = t; kx < LX; kx += NT) {
            const int xc = (kx + LX / 2) % LX;
            const float sg = ((kx + ky) & 1) ? -1.f : 1.f;
            const float2 v = line[fft::pad16(kx)];
            a.spectrum[(size_t)yc * LX + xc] = make_float2(sg * v.x, sg * v.y);
        }
        __syncthreads();
    }
    if (a.encode && !(yc >= a.cy1 && yc <= a.cy2)) return;  // uniform over the workgroup
    fftm::line<LX, NT, +1>(line, tw, t);
    float2* dst = a.T + (size_t)ky * a.w;
    for (int x = t; x < a.w; x += NT) dst[x] = line[fft::pad16(x + a.ox)];
}
template <int LX>
__device__ __forceinline__ bool row_wanted_m(const DmArgs& a, int ky) {
    const int yc = (ky + a.Ny / 2) % a.Ny;
    return a.spectrum || !a.encode || (yc >= a.cy1 && yc <= a.cy2);
}

// Workgroups of three waves (2160): at two waves per SIMD only two fit a CU,
// at three, four.  Without the next layer's values its registers allow that
// (152, none spilled): a field of 2160^2 and 4 layers takes 235 us, of 32 950;
// with the values requested ahead 265 and 996 (and 248 and 1108 before either).
template <int LX>
__host__ __device__ constexpr bool rows_m_three() { return fftm::threads(LX) == 192; }

// Bound by vector instructions and the waits between a layer's stages.  1920 x
// 1080 encoded, 256 layers (272 pairs, of which one workgroup each fills two
// waves a CU: 2483 us): the layers split into 7 parts 795 us; the transform's
// ends in registers, 16 x 15 x 8 in place of 16 x 8 x 5 x 3, row b from the
// thread's own elements and the next layer's row requested before the
// transform 640 us.  Held to 168 or 128 registers it spills (1010, 1456 us).
template <int LX, bool EXACT>
__global__ __launch_bounds__(fftm::threads(LX), rows_m_three<LX>() ? 3 : 1) void dm_rows_m(DmArgs a, const float2* __restrict__ twx) {
    using E = fftm::Ends<LX>;
    constexpr int NT = E::NT;
    constexpr int N0 = E::PER0 * E::R0;
    constexpr bool PREF = N0 <= 16 && !rows_m_three<LX>();   // the next layer's values fit in registers
    extern __shared__ float2 line[];  // fftm::padded_len(LX)
    const int t = threadIdx.x;
    // XCD-aware, as dm_rows_h
    int kya, lo = a.lo, hi = a.hi;
    float2* part = nullptr;
    if ((int)blockIdx.x >= a.n_main) {
        const int lin = xcd_remap(blockIdx.x - a.n_main, gridDim.x - a.n_main), left = a.K - 1 - a.n_main;
        const int j = lin / left, i = lin - j * left;
        lo = a.lo + j * a.per;
        hi = min(a.hi, lo + a.per - 1);
        kya = a.n_main + i;
        part = a.part + ((size_t)i * a.nsums + j) * 2 * LX;
    } else {
        kya = xcd_remap(blockIdx.x, a.n_main);
    }
    const bool pair0 = kya == 0;              // real rows 0 and Ny/2 packed as re/im
    const int kyb = pair0 ? a.Ny / 2 : a.Ny - kya;
    const int sya = sgnidx(kya, a.Ny) + 1;
    const int syb = sgnidx(kyb, a.Ny) + 1;
    const size_t nyq = (size_t)(a.K - 1) * GROUP;
    const size_t gstride = (size_t)a.K * GROUP;
    const size_t lstride = gstride * a.ngroups;
    // Row a's sum at the transform's outputs kx = (t + q NT) + r NBL and row b's
    // at -kx, whose transform is conj Z(kx) and whose kx^2 is the same (as
    // dm_rows_h)
    float2 acca[E::PERL][E::RL], accb[E::PERL][E::RL];
#pragma unroll
    for (int q = 0; q < E::PERL; ++q)
#pragma unroll
        for (int r = 0; r < E::RL; ++r) acca[q][r] = accb[q][r] = make_float2(0.f, 0.f);
    const auto next_layer = [&](int l) {
        while (l <= hi && !a.any[l - 1]) ++l;
        return l;
    };
    // Input element m of layer l: range-checked buffer loads, first the presence
    // flag of its column group, then the value, whose offset is out of range (a
    // zero, no memory access) for absent groups and columns outside the image.
    const auto column = [&](int m, int tl) {
        const int j = tl + m / E::R0 * NT, x = j + m % E::R0 * E::NB0 - a.ox;
        return j < E::NB0 && x >= 0 && x < a.w ? x : -1;
    };
    const auto load_flags = [&](int l, int tl, unsigned char (&f)[N0]) {
        const auto rf = oph_buf_rsrc(a.flags + (size_t)(l - 1) * a.ngroups, (unsigned)a.ngroups);
#pragma unroll
        for (int m = 0; m < N0; ++m) {
            const int x = column(m, tl);
            f[m] = __builtin_amdgcn_raw_buffer_load_b8(rf, x >= 0 ? (unsigned)(x / GROUP) : OPH_BUF_OOB, 0, 0);
        }
    };
    const auto load_values = [&](int l, int tl, const unsigned char (&f)[N0], float2 (&v)[E::PER0][E::R0]) {
        const auto ri = oph_buf_rsrc(a.I + (size_t)(l - 1) * lstride, (unsigned)(lstride * sizeof(float2)));
#pragma unroll
        for (int m = 0; m < N0; ++m) {
            const int x = column(m, tl);
            const unsigned o = x >= 0 && f[m] ? (unsigned)(((size_t)(x / GROUP) * gstride + x % GROUP +
                                                            (size_t)kya * GROUP) * sizeof(float2))
                                              : OPH_BUF_OOB;
            v[m / E::R0][m % E::R0] = oph_buf_load_f2(ri, o);
            if (pair0)   // (workgroup 0 only)
                v[m / E::R0][m % E::R0].y = oph_buf_load_f2(ri, o == OPH_BUF_OOB ? o : o + (unsigned)(nyq * sizeof(float2))).x;
        }
    };
    // The values of the next present layer are requested before this layer's
    // transform, the flags of the one after it after them (PREF)
    unsigned char f[N0];
    float2 vi[E::PER0][E::R0], nv[E::PER0][E::R0];
    int l = next_layer(lo), ln = l <= hi ? next_layer(l + 1) : hi + 1;
    if (PREF && l <= hi) {
        load_flags(l, t, f);
        load_values(l, t, f, nv);
        if (ln <= hi) load_flags(ln, t, f);
    }
    while (l <= hi) {
        // the thread index through a zero the compiler cannot see through:
        // the transforms' LDS addresses are then formed per layer instead of
        // being hoisted out of the loop into ~100 registers
        int zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        const int tl = t + zero;
        if constexpr (PREF) {
#pragma unroll
            for (int m = 0; m < N0; ++m) vi[m / E::R0][m % E::R0] = nv[m / E::R0][m % E::R0];
            if (ln <= hi) {
                load_values(ln, tl, f, nv);
                const int l2 = next_layer(ln + 1);
                if (l2 <= hi) load_flags(l2, tl, f);
            }
        } else {
            load_flags(l, tl, f);
            load_values(l, tl, f, vi);
        }
        __syncthreads();  // the previous transform's readers are done with the line
        float2 v[E::PERL][E::RL];
        fftm::line_ends<LX, -1>(vi, v, line, twx, tl);
        const double cx = a.lc[3 * (l - 1)], cy = a.lc[3 * (l - 1) + 1], K = a.lc[3 * (l - 1) + 2];
        const float Kf = (float)K;
        double tya = cy * (double)sya * sya;
        tya -= rint(tya);
        double tyb = cy * (double)syb * syb;
        tyb -= rint(tyb);
        if (pair0) {
            __syncthreads();
#pragma unroll
            for (int q = 0; q < E::PERL; ++q)
#pragma unroll
                for (int r = 0; r < E::RL; ++r) {
                    const int j = tl + q * NT;
                    if (j < E::NBL) line[fft::pad16(j + r * E::NBL)] = v[q][r];
                }
            __syncthreads();
        }
#pragma unroll
        for (int q = 0; q < E::PERL; ++q)
#pragma unroll
            for (int r = 0; r < E::RL; ++r) {
                const int j = tl + q * NT, kx = j + r * E::NBL;
                if (E::PERL * NT == E::NBL || j < E::NBL) {
                    const int sx = sgnidx(kx, LX);
                    const double sx2 = (double)sx * sx;
                    const float usx = a.ux * (float)(sx * sx);
                    double txd = cx * sx2;
                    txd -= rint(txd);
                    const float tx = (float)txd;
                    float2 ga = v[q][r], gb = make_float2(ga.x, -ga.y);
                    if (pair0) {
                        const float2 gm = line[fft::pad16(kx == 0 ? 0 : LX - kx)];
                        gb = make_float2(gm.x, -gm.y);
                        split_real_pair(ga, gb);
                        gb.y = -gb.y;   // row Ny/2 is real: at -kx the conjugate
                    }
                    const float2 ha = dm_transfer<EXACT>(a, tx, tya, usx, sya, K, Kf, sx2);
                    acca[q][r] = fft::cadd(acca[q][r], fft::cmul(ha, ga));
                    const float2 hb = dm_transfer<EXACT>(a, tx, tyb, usx, syb, K, Kf, sx2);
                    accb[q][r] = fft::cadd(accb[q][r], fft::cmul(hb, gb));
                }
            }
        if constexpr (PREF) {
            l = ln;
            ln = l <= hi ? next_layer(l + 1) : hi + 1;
        } else {
            l = next_layer(l + 1);
        }
    }
    if (part) {
#pragma unroll
        for (int q = 0; q < E::PERL; ++q)
#pragma unroll
            for (int r = 0; r < E::RL; ++r) {
                const int j = t + q * NT, kx = j + r * E::NBL;
                if (j < E::NBL) {
                    part[kx] = acca[q][r];
                    part[LX + (kx == 0 ? 0 : LX - kx)] = accb[q][r];
                }
            }
        return;
    }
#pragma unroll
    for (int row = 0; row < 2; ++row) {
        const int ky = row == 0 ? kya : kyb;
        if (!row_wanted_m<LX>(a, ky)) continue;
        // into the line in natural order; no copy of the row in registers, and
        // each row's LDS addresses formed for it alone (as in the layer loop):
        // at 11520 the one or the other spills
        int zero;
        asm volatile("v_mov_b32 %0, 0" : "=v"(zero));
        const int tl = t + zero;
        __syncthreads();
#pragma unroll
        for (int q = 0; q < E::PERL; ++q)
#pragma unroll
            for (int r = 0; r < E::RL; ++r) {
                const int j = tl + q * NT, kx = j + r * E::NBL;
                if (j < E::NBL)
                    line[fft::pad16(row == 0 || kx == 0 ? kx : LX - kx)] =
                        fft::cmul(row == 0 ? acca[q][r] : accb[q][r], a.rho);
            }
        __syncthreads();
        finish_row_m<LX>(a, ky, line, twx, tl);
    }
}

// The partial sums of a pair's layers in order, then as a whole pair's
template <int LX>
__global__ __launch_bounds__(fftm::threads(LX)) void dm_rows_m_sum(DmArgs a, const float2* __restrict__ twx) {
    constexpr int NT = fftm::threads(LX), EPT = fftm::ept(LX);
    extern __shared__ float2 line[];  // fftm::padded_len(LX)
    const int t = threadIdx.x, i = blockIdx.x >> 1, row = blockIdx.x & 1, kya = a.n_main + i;
    const int ky = row == 0 ? kya : kya == 0 ? a.Ny / 2 : a.Ny - kya;
    const float2* p = a.part + ((size_t)i * a.nsums * 2 + row) * LX;
    float2 acc[EPT];
#pragma unroll
    for (int m = 0; m < EPT; ++m) acc[m] = make_float2(0.f, 0.f);
    for (int j = 0; j < a.nsums; ++j)
#pragma unroll
        for (int m = 0; m < EPT; ++m) {
            const int kx = t + m * NT;
            if (EPT * NT == LX || kx < LX) acc[m] = fft::cadd(acc[m], p[(size_t)2 * j * LX + kx]);
        }
    if (!row_wanted_m<LX>(a, ky)) return;
#pragma unroll
    for (int m = 0; m < EPT; ++m) {
        const int kx = t + m * NT;
        if (EPT * NT == LX || kx < LX) line[fft::pad16(kx)] = fft::cmul(acc[m], a.rho);
    }
    __syncthreads();
    finish_row_m<LX>(a, ky, line, twx, t);
}

template <int LY, int B>
__global__ __launch_bounds__(B * fftm::threads(LY)) void dm_final_m(DmArgs a, const float2* __restrict__ twy) {
    constexpr int NT = fftm::threads(LY);
    constexpr int PL = fftm::padded_len(LY);
    extern __shared__ float2 lds[];
    const int nthr = B * NT;
    const int g = xcd_remap(blockIdx.x, gridDim.x);
    const int c0 = g * B;
    const int b = threadIdx.x / NT, t = threadIdx.x % NT;
    for (int e = threadIdx.x; e < LY * B; e += nthr) {
        const int bb = e % B, ky = e / B;
        const int x = c0 + bb;
        const int yc = (ky + a.Ny / 2) % a.Ny;
        const bool kept = !a.encode || (yc >= a.cy1 && yc <= a.cy2);
        lds[bb * PL + fft::pad16(ky)] = (x < a.w && kept) ? a.T[(size_t)ky * a.w + x] : make_float2(0.f, 0.f);
    }
    __syncthreads();
    fftm::line<LY, NT, +1>(lds + b * PL, twy, t);
    const float sc = (float)a.scale;
    for (int e = threadIdx.x; e < a.h * B; e += nthr) {
        const int bb = e % B, r = e / B;
        const int x = c0 + bb;
        if (x >= a.w) continue;
        const float2 v0 = lds[bb * PL + fft::pad16(a.oy + r)];
        const float2 v = make_float2(v0.x * sc, v0.y * sc);
        const size_t o = (size_t)r * a.w + x;
        if (a.encode) {
            double tt = a.h / 8.0 - (r + 1) / 4.0;
            tt -= rint(tt);
            const float ph = (float)tt;
            const float re = v.x * cos_turns(ph) - v.y * sin_turns(ph);
            if (a.fringe) a.fringe[o] = re;
            if (a.fringe32) a.fringe32[o] = re;
        } else {
            a.field[o] = v;
        }
    }
}

// ---- launchers -------------------------------------------------------------------

// The context's entry of a kernel, which is allowed all of the LDS the first
// time (asked of the runtime once per context, not at every launch)
oph_ctx::KernelFit& full_lds(oph_ctx* ctx, const void* fn) {
    for (auto& k : ctx->kernel_fit)
        if (k.fn == fn) return k;
    hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    hipGetLastError();
    ctx->kernel_fit.push_back({fn, 0, 0});
    return ctx->kernel_fit.back();
}

// Workgroups of a kernel on a CU with this much dynamic LDS
template <typename F>
int rows_resident(oph_ctx* ctx, F kernel, int threads, size_t shm) {
    auto& k = full_lds(ctx, reinterpret_cast<const void*>(kernel));
    if (k.resident == 0 || k.shm != shm) {
        int n = 0;
        hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kernel, threads, shm);
        hipGetLastError();
        k.shm = shm;
        k.resident = std::max(n, 1);
    }
    return k.resident;
}

// The scenes that the column pass takes: its lines and four columns of pixels
// within the LDS.  The pixels are in registers, so the kernels need less; the
// limit is the call's and stays.
size_t cols_limit(int line, const DmArgs& a, size_t words) {
    return 2 * (size_t)line * sizeof(float2) + (size_t)a.h * GROUP * 4 + words;
}

template <int LY>
int launch_dm_cols(oph_ctx* ctx, const DmArgs& a, int chunks) {
    const float2* tw = oph_twiddles(ctx, LY);
    if (!tw) return OPH_ENOMEM;
    const size_t words = (size_t)((a.L + 32) / 32) * 4;
    const size_t shm = 2 * ((size_t)fft::skewed_len(LY, 2) + cols_mirror_stride<LY>(a.K)) * sizeof(float2) + words;
    if (std::max(shm, cols_limit(fft::padded_len(LY), a, words)) > 160 * 1024)
        return oph_fail(ctx, OPH_ENOTSUP, "scene height %d too large for the column pass", a.h);
    const auto launch = [&](auto* kernel) -> int {
        full_lds(ctx, reinterpret_cast<const void*>(kernel));
        OPH_LAUNCH(ctx, "dm_cols", kernel, dim3(a.ngroups, chunks), dim3(2 * (LY / 16)), shm, a, chunks, tw);
        return OPH_OK;
    };
    if constexpr (LY >= 512) {
        const bool half = a.K == LY / 4 + 3;
        const bool mid = a.oy >= 3 * (LY / 16) && a.oy + a.h <= 13 * (LY / 16);
        if (half) return mid ? launch(dm_cols<LY, true, true>) : launch(dm_cols<LY, true, false>);
        return mid ? launch(dm_cols<LY, false, true>) : launch(dm_cols<LY, false, false>);
    } else {
        return launch(dm_cols<LY, false, false>);
    }
}

// How the row pairs are spread over the chip, with `resident` workgroups of
// the row pass on a CU: the first n_main pairs (whole rounds of workgroups)
// are taken whole, the layers of each of the rest are split over nsplit
// workgroups of `per` layers.  The cost of a choice is its rounds times the
// layers of each; a part costs three layer times of its own (its set-up, its
// sums written and read again).  4096 x 2048 encoded needs 514 pairs: 2 rounds
// and a sixteenth, not 3.  (A frame of 720 x 540 and 256 layers, field: 2.29 ->
// 0.55 ms.)
//
// per is a multiple of 4.  For the chunked recurrence (chunk = 16 > 0) it is
// one of chunk, and each chunk's sums are stored, to be added chunk by chunk as
// a whole pair's are: a split pair has the bits of a whole one, whatever the
// size of the chip (the learned correction's BF16 network turns a last bit of
// its field into 1e-3).  Sums that would take over four times the memory of the
// layers' rows I are not formed.
void rows_plan(oph_ctx* ctx, DmArgs& a, int LX, int chunk, int resident) {
    const int pairs = a.K - 1, layers = a.hi - a.lo + 1;
    const int slots = std::max(ctx->cu_count, 1) * resident, gran = chunk ? chunk : 4;
    a.n_main = pairs;
    a.nsplit = a.nsums = 1;
    a.per = layers;
    if (layers < 2) return;   // (0: an empty range)
    const long long most = 4LL * a.L * a.ngroups * a.K * GROUP;
    long long best = (long long)((pairs + slots - 1) / slots) * layers;
    for (const int n_main : {pairs / slots * slots, 0})
        for (int n = 2; n <= 16; ++n) {
            const int per = ((layers + n - 1) / n + gran - 1) / gran * gran;
            const int parts = (layers + per - 1) / per, left = pairs - n_main;
            const int sums = chunk ? (layers + chunk - 1) / chunk : parts;
            if (parts < 2 || left == 0 || (long long)left * sums * 2 * LX > most) continue;
            const long long c = (long long)(n_main / slots) * layers +
                                ((long long)left * parts + slots - 1) / slots * (per + 3 + (chunk ? per / chunk : 0));
            if (c < best) {
                best = c;
                a.n_main = n_main;
                a.nsplit = parts;
                a.nsums = sums;
                a.per = per;
            }
        }
    if (a.n_main < pairs) {
        a.part = static_cast<float2*>(
            oph_scratch(ctx, SLOT_WORK0, (size_t)(pairs - a.n_main) * a.nsums * 2 * LX * sizeof(float2)));
        if (!a.part) {   // no room for them: every pair whole
            a.n_main = pairs;
            a.nsplit = a.nsums = 1;
            a.per = layers;
        }
    }
}

template <int LX, int MODE>
int launch_dm_rows_h(oph_ctx* ctx, const DmArgs& a) {
    const float2* tw8 = oph_twiddles(ctx, LX, 8);
    if (!tw8) return OPH_ENOMEM;
    const size_t fbytes = (size_t)a.L * a.fwpl * sizeof(unsigned);
    const bool fbits = rows_h_lds<LX, MODE>() + fbytes <= 160 * 1024;
    const size_t shm = rows_h_lds<LX, MODE>() + (fbits ? fbytes : 0);
    auto* kernel = fbits ? dm_rows_h<LX, MODE, true, false> : dm_rows_h<LX, MODE, false, false>;
    if constexpr (LX >= 512)
        if (fbits && a.w <= LX / 2) kernel = dm_rows_h<LX, MODE, true, true>;   // then ox >= LX/4
    DmArgs b = a;
    rows_plan(ctx, b, LX, MODE == 0 ? 16 : 0, rows_resident(ctx, kernel, LX / 8, shm));
    const int left = a.K - 1 - b.n_main;
    OPH_LAUNCH(ctx, "dm_rows", kernel, dim3(b.n_main + left * b.nsplit), dim3(LX / 8), shm, b, tw8);
    if (left > 0)
        OPH_LAUNCH(ctx, "dm_rows_sum", dm_rows_h_sum<LX>, dim3(2 * left), dim3(LX / 8), 0, b, tw8);
    return OPH_OK;
}

template <int LX>
int launch_dm_rows(oph_ctx* ctx, const DmArgs& a) {
    if constexpr (LX >= 64 && LX <= 4096) {
        if (a.horner) return launch_dm_rows_h<LX, 0>(ctx, a);
        return a.exact ? launch_dm_rows_h<LX, 2>(ctx, a) : launch_dm_rows_h<LX, 1>(ctx, a);
    } else {
        const float2* tw = oph_twiddles(ctx, LX);
        if (!tw) return OPH_ENOMEM;
        if (a.exact)
            OPH_LAUNCH(ctx, "dm_rows", (dm_rows<LX, true>), dim3(a.K - 1), dim3(LX / 16), 0, a, tw);
        else
            OPH_LAUNCH(ctx, "dm_rows", (dm_rows<LX, false>), dim3(a.K - 1), dim3(LX / 16), 0, a, tw);
        return OPH_OK;
    }
}

template <int LY>
int launch_dm_final(oph_ctx* ctx, const DmArgs& a) {
    const float2* tw = oph_twiddles(ctx, LY);
    if (!tw) return OPH_ENOMEM;
    constexpr int B = fftk::col_lines(LY) >= 4 ? 4 : fftk::col_lines(LY);
    const size_t shm = (size_t)B * fft::padded_len(LY) * sizeof(float2);
    static bool attr = false;
    if (!attr) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&dm_final<LY, B>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        hipGetLastError();
        attr = true;
    }
    OPH_LAUNCH(ctx, "dm_final", (dm_final<LY, B>), dim3((a.w + B - 1) / B), dim3(B * (LY / 16)), shm, a, tw);
    return OPH_OK;
}

template <int LY>
int launch_dm_cols_m(oph_ctx* ctx, const DmArgs& a, int chunks) {
    const float2* tw = oph_twiddles_mixed(ctx, LY);
    if (!tw) return OPH_ENOMEM;
    if constexpr (2 * (size_t)fftm::padded_len(LY) * sizeof(float2) > 150 * 1024) {
        (void)chunks;
        return oph_fail(ctx, OPH_ENOTSUP, "grid height %d too large for the column pass", LY);
    } else {
        const size_t words = (size_t)((a.L + 32) / 32) * 4;
        const size_t shm = 2 * ((size_t)cols_m_line<LY>() + cols_mirror_stride<0>(a.K)) * sizeof(float2) + words;
        if (std::max(shm, cols_limit(fftm::padded_len(LY), a, words)) > 160 * 1024)
            return oph_fail(ctx, OPH_ENOTSUP, "scene height %d too large for the column pass", a.h);
        full_lds(ctx, reinterpret_cast<const void*>(&dm_cols_m<LY>));
        OPH_LAUNCH(ctx, "dm_cols", dm_cols_m<LY>, dim3(a.ngroups, chunks), dim3(2 * fftm::threads(LY)), shm, a,
                   chunks, tw);
        return OPH_OK;
    }
}

template <int LX>
int launch_dm_rows_m(oph_ctx* ctx, const DmArgs& a) {
    const float2* tw = oph_twiddles_mixed(ctx, LX);
    if (!tw) return OPH_ENOMEM;
    const size_t shm = (size_t)fftm::padded_len(LX) * sizeof(float2);
    constexpr int NT = fftm::threads(LX);
    auto* kernel = a.exact ? dm_rows_m<LX, true> : dm_rows_m<LX, false>;
    DmArgs b = a;
    rows_plan(ctx, b, LX, 0, rows_resident(ctx, kernel, NT, shm));
    const int left = a.K - 1 - b.n_main;
    OPH_LAUNCH(ctx, "dm_rows", kernel, dim3(b.n_main + left * b.nsplit), dim3(NT), shm, b, tw);
    if (left > 0) {
        full_lds(ctx, reinterpret_cast<const void*>(&dm_rows_m_sum<LX>));
        OPH_LAUNCH(ctx, "dm_rows_sum", dm_rows_m_sum<LX>, dim3(2 * left), dim3(NT), shm, b, tw);
    }
    return OPH_OK;
}

// columns per dm_final_m workgroup: up to 4, at most 1024 threads and ~140 KB
__host__ __device__ constexpr int final_m_cols(int LY) {
    int b = 4;
    while (b > 1 && (b * fftm::threads(LY) > 1024 || (size_t)b * fftm::padded_len(LY) * 8 > 140 * 1024)) b /= 2;
    return b;
}

template <int LY>
int launch_dm_final_m(oph_ctx* ctx, const DmArgs& a) {
    const float2* tw = oph_twiddles_mixed(ctx, LY);
    if (!tw) return OPH_ENOMEM;
    constexpr int B = final_m_cols(LY);
    const size_t shm = (size_t)B * fftm::padded_len(LY) * sizeof(float2);
    static bool attr = false;
    if (!attr) {
        hipFuncSetAttribute(reinterpret_cast<const void*>(&dm_final_m<LY, B>),
                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)shm);
        hipGetLastError();
        attr = true;
    }
    OPH_LAUNCH(ctx, "dm_final", (dm_final_m<LY, B>), dim3((a.w + B - 1) / B), dim3(B * fftm::threads(LY)), shm,
               a, tw);
    return OPH_OK;
}

// Depth index of each u8 depth value d, as the reference forms it per pixel:
// mode 0 (FLAG_CHANGE_DEPTH_QUANTIZATION = 0): Q - d (0, no layer, below 0);
// mode 1, change_depth_quan (CPU.cpp:74-103): dmap = (1 - d/255)(far - near)
// + near, and every level l adds (l + 1) where dmap falls in
// [lev_l - dstep/2, lev_l + dstep/2) ([.., ..] for the last), capped at
// 65535.  Each product and sum is its own statement (no fused multiply-add),
// as the reference's double arithmetic.
void depth_index_table(int mode, int Q, const std::vector<double>& lev, double dstep, double near_m,
                       double far_m, double* table) {
    const int L = (int)lev.size();
    for (int d = 0; d < 256; ++d) {
        if (mode == 0) {
            const int v = Q - d;
            table[d] = (double)(unsigned short)(v < 0 ? 0 : v);
            continue;
        }
        const double dsrc = (double)d / 255.0;
        const double span = far_m - near_m;
        const double scaled = (1 - dsrc) * span;
        const double dmap = scaled + near_m;
        long long acc = 0;
        for (int l = 0; l < L; ++l) {
            const double half = dstep / 2.0;
            const double d1 = lev[l] - half, d2 = lev[l] + half;
            const bool t = (l < L - 1) ? (dmap >= d1 && dmap < d2) : (dmap >= d1 && dmap <= d2);
            if (t) acc += l + 1;
        }
        table[d] = (double)(acc > 65535 ? 65535 : acc);
    }
}

}  // namespace

extern "C" int oph_depthmap(oph_ctx* ctx, const oph_dm_spec* s, int ncolor, const double* lambdas,
                            const unsigned char* intensity, const unsigned char* depth, void* out, int flags) {
    int rc = oph_enter(ctx);
    if (rc) return rc;
    if (!s || !lambdas || !intensity || !depth || !out || ncolor < 1)
        return oph_fail(ctx, OPH_EINVAL, "null argument");
    const int w = s->w, h = s->h, Nx = s->Nx, Ny = s->Ny, L = s->num_depth;
    if (w <= 0 || h <= 0 || w > Nx || h > Ny) return oph_fail(ctx, OPH_EINVAL, "scene %dx%d must fit the grid %dx%d", w, h, Nx, Ny);
    // both sides powers of two, or both among the general lengths
    const bool mixed = !(fftk::supported(Nx) && fftk::supported(Ny));
    if (mixed && !(dm_mixed_length(Nx) && dm_mixed_length(Ny)))
        return oph_fail(ctx, OPH_ENOTSUP,
                        "grid %dx%d: sides must both be powers of two in 16..8192 or both among 540, 720, 1080, "
                        "1920, 2160, 3840, 11520", Nx, Ny);
    if (L < 1 || L > MAX_LAYERS) return oph_fail(ctx, OPH_EINVAL, "num_depth must be in 1..%d", MAX_LAYERS);
    if (!(s->pitch_x > 0) || !(s->pitch_y > 0) || !(s->far_m >= s->near_m))
        return oph_fail(ctx, OPH_EINVAL, "bad pitch or depth range");
    if (s->quant_mode != 0 && s->quant_mode != 1) return oph_fail(ctx, OPH_EINVAL, "quant_mode must be 0 or 1");
    if ((flags & OPH_ASYNC) && !(flags & OPH_DEVICE_PTR))
        return oph_fail(ctx, OPH_EINVAL, "OPH_ASYNC needs device pointers");
    for (int c = 0; c < ncolor; ++c)
        if (!(lambdas[c] > 0)) return oph_fail(ctx, OPH_EINVAL, "wavelength %d must be positive", c);
    const int fmt = flags & OPH_DM_OUT_MASK;
    const int hi = (s->layer_hi >= 1 && s->layer_hi <= L) ? s->layer_hi : L;
    // (a range that begins past its end is empty: lo = hi + 1, a field of zeros)
    const int lo = std::min(s->layer_lo >= 1 ? s->layer_lo : 1, hi + 1);

    // depth levels (GetDepthValues, HologramGenerator.cpp:393-401: repeated
    // addition; continued to exactly L entries) and the viewing-window
    // transform z_l = -f d/(d - f) (:432), or z_l = d without a field lens
    std::vector<double> lev(L);
    if (L > 1) {
        const double dstep = (s->far_m - s->near_m) / (L - 1);
        double v = s->near_m;
        for (int i = 0; i < L; ++i) { lev[i] = v; v += dstep; }
    } else {
        lev[0] = s->far_m - s->near_m;
    }
    const double dstep = L > 1 ? (s->far_m - s->near_m) / (L - 1) : (s->far_m + s->near_m) / 2;
    const double Sx = s->pitch_x * Nx, Sy = s->pitch_y * Ny;
    std::vector<double>& hc = ctx->host_scratch;
    // per colour and layer 3 constants, the L levels, the 256-entry depth-index table
    hc.assign((size_t)3 * L * ncolor + L + 256, 0.0);
    double zmax = 0.0;
    for (int c = 0; c < ncolor; ++c) {
        const double lam = lambdas[c];
        for (int l = 0; l < L; ++l) {
            const double d = lev[l];
            const double z = s->field_lens > 0.0 ? -s->field_lens * d / (d - s->field_lens) : d;
            double* o = &hc[(size_t)3 * (c * L + l)];
            o[0] = z * lam / (2.0 * Sx * Sx);
            o[1] = z * lam / (2.0 * Sy * Sy);
            o[2] = z / lam;
            zmax = fmax(zmax, fabs(z / lam));
        }
    }
    for (int l = 0; l < L; ++l) hc[(size_t)3 * L * ncolor + l] = lev[l];
    depth_index_table(s->quant_mode, s->default_q, lev, dstep, s->near_m, s->far_m, &hc[(size_t)3 * L * ncolor + L]);

    const size_t npx = (size_t)w * h;
    const int ngroups = (w + GROUP - 1) / GROUP;
    // Encoding keeps the centred rows [Ny/4 - 1, 3 Ny/4 - 2], ky from -(Ny/4 + 1)
    // to Ny/4 - 2: only the row pairs (ky, -ky) up to ky = Ny/4 + 1 are formed
    // (and row Ny/2, which shares row 0's transform); a field needs all
    const int K = fmt != OPH_DM_OUT_FIELD ? std::min(Ny / 2 + 1, Ny / 4 + 3) : Ny / 2 + 1;
    const size_t lstride = (size_t)K * GROUP * ngroups;
    // device buffers
    unsigned char* dimg = const_cast<unsigned char*>(intensity);
    unsigned char* ddep = const_cast<unsigned char*>(depth);
    if (!(flags & OPH_DEVICE_PTR)) {
        dimg = static_cast<unsigned char*>(oph_scratch(ctx, SLOT_IN, npx * (ncolor + 1)));
        if (!dimg) return OPH_ENOMEM;
        ddep = dimg + npx * ncolor;
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(dimg, intensity, npx * ncolor, hipMemcpyHostToDevice, ctx->stream));
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(ddep, depth, npx, hipMemcpyHostToDevice, ctx->stream));
    }
    const int fwpl = (ngroups + 31) / 32;
    const size_t aux_bytes = npx * 2 + (size_t)L * ngroups + L + 4 + (size_t)L * fwpl * 4 + 64 +
                             hc.size() * sizeof(double);
    unsigned char* aux = static_cast<unsigned char*>(oph_scratch(ctx, SLOT_AUX0, aux_bytes + 256));
    float2* I = static_cast<float2*>(oph_scratch(ctx, SLOT_WORK2, (size_t)L * lstride * sizeof(float2)));
    float2* T = static_cast<float2*>(oph_scratch(ctx, SLOT_WORK1, (size_t)Ny * w * sizeof(float2)));
    if (!aux || !I || !T) return OPH_ENOMEM;
    double* dlc = reinterpret_cast<double*>(aux);
    unsigned short* didx = reinterpret_cast<unsigned short*>(aux + hc.size() * sizeof(double));
    unsigned char* dflags = reinterpret_cast<unsigned char*>(didx + npx);
    unsigned char* dany = dflags + (size_t)L * ngroups;
    // the flag bits follow, at the next 4-byte boundary (word atomics)
    unsigned* dfbits = reinterpret_cast<unsigned*>((reinterpret_cast<uintptr_t>(dany + L) + 3) & ~(uintptr_t)3);
    const size_t nfl_bytes = reinterpret_cast<unsigned char*>(dfbits + (size_t)L * fwpl) - dflags;
    OPH_HIP_CHECK(ctx, hipMemcpyAsync(dlc, hc.data(), hc.size() * sizeof(double), hipMemcpyHostToDevice, ctx->stream));

    // outputs
    const size_t osz = fmt == OPH_DM_OUT_FIELD ? sizeof(float2) : fmt == OPH_DM_OUT_FRINGE32 ? 4 : 8;
    void* dout = out;
    if (!(flags & OPH_DEVICE_PTR)) {
        dout = oph_scratch(ctx, SLOT_OUT, npx * ncolor * osz);
        if (!dout) return OPH_ENOMEM;
    }

    OPH_LAUNCH(ctx, "dm_index", dm_index, dim3((unsigned)((npx + 255) / 256)), dim3(256), 0, ddep, (int)npx,
               dlc + (size_t)3 * L * ncolor + L, didx);

    // truncated-series accuracy at the grid corner (see dm_transfer): the
    // first dropped term is 21/1024 u^6 z/lambda turns
    double lmax = 0;
    for (int c = 0; c < ncolor; ++c) lmax = fmax(lmax, lambdas[c]);
    const double fxm = 0.5 / s->pitch_x, fym = (Ny / 2 + 1.0) / Sy;
    const double umax = lmax * lmax * (fxm * fxm + fym * fym);
    const bool exact = umax >= 0.5 || zmax * pow(umax, 6) * (21.0 / 1024.0) > 1e-7;

    // equally spaced z (no field lens): the chunked recurrence of dm_rows_h
    // applies when every step equals the first to far below a phase ulp
    std::vector<double> zs(L);
    for (int l = 0; l < L; ++l)
        zs[l] = s->field_lens > 0.0 ? -s->field_lens * lev[l] / (lev[l] - s->field_lens) : lev[l];
    const double dz = L > 1 ? zs[1] - zs[0] : 0.0;
    double dev = 0.0;
    for (int l = 1; l < L; ++l) dev = fmax(dev, fabs((zs[l] - zs[l - 1]) - dz));
    const double phimax = lmax * (fxm * fxm + fym * fym) / 2.0 + 0.25 * umax * umax / lmax;  // turns per metre
    const bool horner = !mixed && !exact && L > 1 && hi > lo && dev * phimax < 1e-9;

    for (int c = 0; c < ncolor; ++c) {
        const double lam = lambdas[c];
        DmArgs a{};
        a.horner = horner ? 1 : 0;
        a.dcx = dz * lam / (2.0 * Sx * Sx);
        a.dcy = dz * lam / (2.0 * Sy * Sy);
        a.dK = dz / lam;
        a.w = w; a.h = h; a.Nx = Nx; a.Ny = Ny;
        a.ox = (Nx - w) / 2;
        a.oy = (Ny - h) / 2;
        a.L = L; a.lo = lo; a.hi = hi;
        a.ngroups = ngroups;
        a.img = dimg + npx * c;
        a.idx = didx;
        a.I = I;
        a.K = K;
        a.flags = dflags;
        a.any = dany;
        a.fbits = dfbits;
        a.fwpl = fwpl;
        a.lc = dlc + (size_t)3 * L * c;
        a.ux = (float)(lam * lam / (Sx * Sx));
        a.uy = (float)(lam * lam / (Sy * Sy));
        a.lam2_sx2 = lam * lam / (Sx * Sx);
        a.lam2_sy2 = lam * lam / (Sy * Sy);
        a.inv_lambda = 1.0 / lam;
        a.exact = exact ? 1 : 0;
        a.rho = make_float2((float)s->rho_re, (float)s->rho_im);
        a.encode = fmt != OPH_DM_OUT_FIELD;
        const int cropy = Ny / 2;
        a.cy1 = cropy - cropy / 2 - 1;
        a.cy2 = a.cy1 + cropy - 1;
        a.T = T;
        a.spectrum = nullptr;
        a.scale = 1.0 / ((double)Nx * Ny);
        char* ob = static_cast<char*>(dout) + npx * c * osz;
        a.fringe = fmt == OPH_DM_OUT_FRINGE ? reinterpret_cast<double*>(ob) : nullptr;
        a.fringe32 = fmt == OPH_DM_OUT_FRINGE32 ? reinterpret_cast<float*>(ob) : nullptr;
        a.field = fmt == OPH_DM_OUT_FIELD ? reinterpret_cast<float2*>(ob) : nullptr;

        const int nfl = (int)nfl_bytes;   // flags, any and the flag bits
        OPH_LAUNCH(ctx, "dm_zero", dm_zero, dim3((nfl + 255) / 256), dim3(256), 0, dflags, nfl);
        const int nl = hi - lo + 1;
        // column workgroups: four a CU, eight where each still has 16 layers to
        // spread its loading of the pixels over (2048 rows, 480 column groups:
        // 256 layers in 3 parts 466 us, in 5 442; 256 groups, 16 layers in 4
        // parts 49 us, in 8 78).  A part takes every chunks-th layer, which
        // evens out the layers that a column group has pixels in (in runs of
        // 86 layers: 690 us).
        const auto per_cu = [&](int n) { return (int)(((long long)n * ctx->cu_count + ngroups - 1) / ngroups); };
        int chunks = std::max(per_cu(4), std::min(per_cu(8), nl / 16));
        // Loading the pixels costs as much as some nine layers, so beyond one
        // per CU no part has fewer than four layers; fewer still up to two or,
        // on general lengths (fewer rows a thread), three per CU (480 groups of
        // 3840 rows, 4 layers in 3 parts 168 us, in one 90; 256 groups of 1024,
        // 8 layers in 4 parts 38, in 2 31; 180 groups of 540, 8 layers in 6
        // parts 26, in 4 20).  Below 512 rows a workgroup is less than a wave,
        // and the number of them counts more (32 groups of 256, 64 layers in 8
        // parts 24, in 32 16).
        if (mixed || Ny >= 512)
            chunks = std::min(chunks, std::max({per_cu(1), nl / 4, mixed ? std::min(3 * ctx->cu_count / ngroups, nl / 2)
                                                                         : std::min(2 * ctx->cu_count / ngroups, nl / 3)}));
        if (chunks > nl) chunks = nl;
        if (chunks < 1) chunks = 1;
        if (mixed) {
            switch (Ny) {
#define OPH_DMC(n) case n: rc = launch_dm_cols_m<n>(ctx, a, chunks); break;
                OPH_DM_MIXED_LENGTHS(OPH_DMC)
#undef OPH_DMC
            }
            if (rc) return rc;
            switch (Nx) {
#define OPH_DMR(n) case n: rc = launch_dm_rows_m<n>(ctx, a); break;
                OPH_DM_MIXED_LENGTHS(OPH_DMR)
#undef OPH_DMR
            }
            if (rc) return rc;
            switch (Ny) {
#define OPH_DMF(n) case n: rc = launch_dm_final_m<n>(ctx, a); break;
                OPH_DM_MIXED_LENGTHS(OPH_DMF)
#undef OPH_DMF
            }
            if (rc) return rc;
            continue;
        }
        switch (Ny) {
#define OPH_DMC(n) case n: rc = launch_dm_cols<n>(ctx, a, chunks); break;
            OPH_FFT_LENGTHS(OPH_DMC)
#undef OPH_DMC
        }
        if (rc) return rc;
        switch (Nx) {
#define OPH_DMR(n) case n: rc = launch_dm_rows<n>(ctx, a); break;
            OPH_FFT_LENGTHS(OPH_DMR)
#undef OPH_DMR
        }
        if (rc) return rc;
        switch (Ny) {
#define OPH_DMF(n) case n: rc = launch_dm_final<n>(ctx, a); break;
            OPH_FFT_LENGTHS(OPH_DMF)
#undef OPH_DMF
        }
        if (rc) return rc;
    }
    if (!(flags & OPH_DEVICE_PTR))
        OPH_HIP_CHECK(ctx, hipMemcpyAsync(out, dout, npx * ncolor * osz, hipMemcpyDeviceToHost, ctx->stream));
    return oph_finish(ctx, flags);
}
