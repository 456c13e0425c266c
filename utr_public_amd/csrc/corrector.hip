// corrector.hip -- the learned 3D residual corrector on gfx950: a 3-level
// U-Net (3x3x3 convolutions, 16/32/64 channels, ReLU, average pooling,
// nearest upsampling, skip connections by channel concatenation) applied to
// UTR reconstructions in tiles, trained on the GPU by the kernels below
// (forward, backward, Adam).  Included by utr_api.hip (one translation
// unit).  No counterpart in the reference, which has no learned component;
// the C ABI is utr_corr_* in include/utr_hip.h.
//
// Numbers: activations and activation gradients are BF16 (channels last,
// [n][z][y][x][c]); weights are FP32 masters updated by Adam and repacked to
// BF16 MFMA fragments after every step; all products accumulate in FP32 on
// the matrix cores (v_mfma_f32_16x16x32_bf16); the head (1x1x1
// convolution to one channel plus alpha times the input) and the loss are
// FP32.
//
// Convolution as an implicit GEMM: 16 output channels by 4 x 4 voxels, K =
// (two taps, 16 input channels); each 16-channel slice of a work-group's input
// block with its one-voxel halo is staged in LDS.  The backward pass with
// respect to the input is the same kernel with the taps mirrored and the
// channel roles swapped (weights repacked once per step), its epilogue
// multiplying by the ReLU mask of the layer below.  Weight gradients contract
// over voxels (K = 32: two x rows of 16) with the input slice and the
// output-gradient block both staged in LDS; each work-group sums a fixed
// subset of blocks and a second kernel adds the partial sums in a fixed order,
// so gradients are deterministic.
namespace utr {

typedef short cr_s4 __attribute__((ext_vector_type(4)));
typedef float cr_f4 __attribute__((ext_vector_type(4)));
typedef __bf16 cr_b8 __attribute__((ext_vector_type(8)));

// FP32 to BF16 (round to nearest even; NaN stays NaN)
__host__ __device__ __forceinline__ unsigned short cr_f2bf(float f) {
    union { unsigned u; float f; } v;
    v.f = f;
    unsigned u = v.u;
    if ((u & 0x7f800000u) == 0x7f800000u) return (unsigned short)((u >> 16) | ((u & 0xffffu) ? 0x40u : 0u));
    u += 0x7fffu + ((u >> 16) & 1u);
    return (unsigned short)(u >> 16);
}

constexpr int CR_STEPS = 15;  // K = 32 steps per 16-channel slice: five (dy, dx) tap pairs x three dz

struct CrShape {
    int n, d, h, w;         // batch and spatial extent
};

// Voxel index of (b, z, y, x).
__device__ __forceinline__ size_t cr_vox(const CrShape& s, int b, int z, int y, int x) {
    return (((size_t)b * s.d + z) * s.h + y) * s.w + x;
}

// Four FP32 values rounded to BF16 (nearest even) as one 8-byte word.
__device__ __forceinline__ uint2 cr_pack4(const float* v) {
    typedef float f4 __attribute__((ext_vector_type(4)));
    typedef __bf16 b4 __attribute__((ext_vector_type(4)));
    const f4 f = {v[0], v[1], v[2], v[3]};
    return __builtin_bit_cast(uint2, __builtin_convertvector(f, b4));
}

__device__ __forceinline__ float cr_bflo(unsigned w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float cr_bfhi(unsigned w) { return __builtin_bit_cast(float, w & 0xffff0000u); }
// v[i] = 0 where the BF16 activation i of w is not positive.
__device__ __forceinline__ void cr_relu_mask(float* v, uint2 w) {
    const unsigned h[4] = {w.x & 0xffffu, w.x >> 16, w.y & 0xffffu, w.y >> 16};
#pragma unroll
    for (int i = 0; i < 4; i++)
        if (!(h[i] != 0 && (h[i] & 0x8000u) == 0)) v[i] = 0.f;
}

// Channels of a layer's input: the first nup 16-channel slices are a coarser
// tensor read at half the coordinates (nearest 2x upsampling), the others one
// at the layer's own resolution.  Both are dense, channels last.
struct CrIn {
    const unsigned short* up;
    int up_c, nup;             // channels and 16-channel slices of the coarser tensor
    const unsigned short* p;
    int c;                     // channels of p
};

// 16 bytes (half 0 or 1) of 16-channel slice c at voxel (z, y, x).
__device__ __forceinline__ uint4 cr_load(const CrIn& I, const CrShape& s, int c, int half, int b, int z, int y, int x) {
    if (c < I.nup)
        return *reinterpret_cast<const uint4*>(
            I.up + ((((size_t)b * (s.d >> 1) + (z >> 1)) * (s.h >> 1) + (y >> 1)) * (s.w >> 1) + (x >> 1)) * I.up_c +
            c * 16 + half * 8);
    return *reinterpret_cast<const uint4*>(I.p + cr_vox(s, b, z, y, x) * I.c + (c - I.nup) * 16 + half * 8);
}

// The network's FP32 input: crops [b][T][T][T] (ntx = 0), or crop first + b of
// the tile grid of a volume, covering [t0 - halo, t0 + tile + halo) per axis
// with zeros outside the volume; times scale.
struct CrVol {
    const float* p;
    float scale;
    int nx, ny, nz, tile, halo, ntx, nty, first;
};
__device__ __forceinline__ bool cr_vol_at(const CrVol& V, int T, int b, int z, int y, int x, size_t& at) {
    if (V.ntx == 0) {
        at = (((size_t)b * T + z) * T + y) * T + x;
        return true;
    }
    const int id = V.first + b;
    const int gx = id % V.ntx * V.tile - V.halo + x, gy = id / V.ntx % V.nty * V.tile - V.halo + y,
              gz = id / (V.ntx * V.nty) * V.tile - V.halo + z;
    at = ((size_t)gz * V.ny + gy) * V.nx + gx;
    return (unsigned)gx < (unsigned)V.nx && (unsigned)gy < (unsigned)V.ny && (unsigned)gz < (unsigned)V.nz;
}

// What follows a convolution.
enum CrEpi {
    CR_ACT,    // bias, ReLU; BF16 out
    CR_POOL,   // the same, and its 2x2x2 average to out2 at half resolution
    CR_GRAD,   // BF16 out, times (mask > 0) if a mask is given
    CR_SPLIT,  // gradient of an upsampled-and-concatenated input: blocks below nup summed over 2x2x2 to out2 (mask2
               // > 0 at half resolution), the others to out (mask > 0)
    CR_HEAD,   // bias, ReLU and the head: FP32 alpha x + b1 + sum_c w1[c] act[c] to vout
    CR_LOSS    // the same compared with the target: loss, head gradients (part) and the gradient of act to out
};

struct CrConv {
    CrIn in;
    int cin;
    const uint4* wf;           // weight fragments (k_cr_pack), nbt blocks of 16 output channels
    int nbt;
    const float* bias;
    unsigned short* out;       // out_c channels
    int out_c;
    unsigned short* out2;      // CR_POOL, CR_SPLIT
    int out2_c, nup;
    const unsigned short *mask, *mask2;  // same channels as out, out2
    CrShape s;
    int lo, hi;                // outputs are formed in the cube [lo, hi)^3 (even bounds for CR_POOL and CR_SPLIT)
    int ilo, ihi;              // the input is zero outside [ilo, ihi)^3
    // CR_HEAD, CR_LOSS
    CrVol vol;
    const float* hp;           // {w1[16], b1, alpha}
    float* vout;
    float oscale;              // CR_HEAD: output = value * oscale
    const float* tgt;
    float tscale, inv_count;
    float* part;               // [work-group][20]: {dw1[16], db1, dalpha, loss, 0}
};

constexpr int CR_PX = 2, CR_PY = 2, CR_Z = 4;  // patches in x and y, and planes, of a work-group's block

// Waves per SIMD the register budget is set for.
constexpr int cr_occ(int nb) { return nb == 3 ? 3 : 4; }

// 3x3x3 convolution, stride 1, zero padding 1, as an implicit GEMM: output
// channels are the matrix rows, 16 voxels (a 4 x 4 patch of one z plane) its
// columns, K = 32 is two (dy, dx) taps of 16 input channels.  A work-group
// owns CR_PX x CR_PY patches in x and y, CR_Z planes in z and NB blocks of 16
// output channels; each of its waves takes one patch through all planes (two
// patches a wave spilled registers at four waves per SIMD; eight patches and
// waves, 16 x 8 voxels with 2.1 times the input staged instead of 2.3, took
// 1.0 to 1.4 times the time over the layers of 24^3 to 112^3 crops: waves wait
// for the others of their work-group at every slice).
//
// What bounds it: for 16 channels the activations' traffic, for more the LDS
// reads against the matrix cores.  Rows = channels lets a lane hold four
// consecutive channels of one voxel, so a tile leaves in one 8-byte store per
// lane (the transposed form stored 2 bytes at a time).  With the three dz of a
// tap pair held in registers an input fragment read from LDS serves up to three
// output planes: six reads for twelve matrix instructions a pair and patch
// instead of one each.  Staged voxels keep their two 8-channel halves apart and
// rows padded to an odd multiple of 64 bytes, so that the eight lanes of a read
// phase fall on distinct banks.
//
// The passes around a convolution are its own loads and stores (CrIn, CrEpi):
// upsampling and concatenation, pooling, their adjoints, the head and the loss
// each read and wrote whole activations in kernels of their own before.
template <int NB, int EPI>
__global__ void __launch_bounds__(64 * CR_PX * CR_PY, cr_occ(NB)) k_cr_conv(CrConv A) {
    constexpr int PX = CR_PX, PY = CR_PY;
    constexpr int HX = 4 * PX + 2, HY = 4 * PY + 2, HZ = CR_Z + 2;
    constexpr int PITCH = 4 * PX + 4, HALF = HZ * HY * PITCH + 4;  // 16-byte units; HALF = 4 mod 8
    constexpr int NV = HX * HY * HZ, NT = 64 * PX * PY;
    constexpr int PER = (2 * NV + NT - 1) / NT;
    static_assert(PITCH % 8 == 4 && HALF % 8 == 4, "bank layout");
    __shared__ __align__(16) uint4 xs[2 * HALF];
    const CrShape s = A.s;
    const int ext = A.hi - A.lo;
    const int bxn = (ext + 4 * PX - 1) / (4 * PX), byn = (ext + 4 * PY - 1) / (4 * PY),
              bzn = (ext + CR_Z - 1) / CR_Z;
    int tile, nb0;
    if (!xcd_tile(bxn * byn * bzn * s.n, A.nbt / NB, tile, nb0)) return;
    [[maybe_unused]] const int wg = tile;
    nb0 *= NB;
    const int x0 = A.lo + tile % bxn * (4 * PX); tile /= bxn;
    const int y0 = A.lo + tile % byn * (4 * PY); tile /= byn;
    const int z0 = A.lo + tile % bzn * CR_Z;
    const int b = tile / bzn;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4, mx = m & 3, my = m >> 2;
    cr_f4 acc[CR_Z][NB];
#pragma unroll
    for (int z = 0; z < CR_Z; z++)
#pragma unroll
        for (int nb = 0; nb < NB; nb++) acc[z][nb] = cr_f4{0.f, 0.f, 0.f, 0.f};
    // this lane's fragment address for each tap pair (tap 9 of the last pair
    // does not exist: it reads tap 8's voxel and is set to zero)
    int fa[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const int t = min(2 * q + (kq >> 1), 8);
        fa[q] = (kq & 1) * HALF + (wave / PX * 4 + my + t / 3) * PITCH + wave % PX * 4 + mx + t % 3;
    }
    const int nslice = A.cin >> 4;
    const uint4* wp = A.wf + lane;
    for (int c = 0; c < nslice; c++) {
        uint4 val[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int t = (int)threadIdx.x + NT * k, v = t >> 1;
            const int gx = x0 - 1 + v % HX, gy = y0 - 1 + (v / HX) % HY, gz = z0 - 1 + v / (HX * HY);
            val[k] = uint4{0u, 0u, 0u, 0u};
            if (t < 2 * NV && min(gx, min(gy, gz)) >= A.ilo && max(gx, max(gy, gz)) < A.ihi)
                val[k] = cr_load(A.in, s, c, t & 1, b, gz, gy, gx);
        }
        if (c) __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int t = (int)threadIdx.x + NT * k, v = t >> 1;
            if (t < 2 * NV) xs[(t & 1) * HALF + (v / HX) * PITCH + v % HX] = val[k];
        }
        __syncthreads();
#pragma unroll
        for (int q = 0; q < 5; q++) {
            cr_b8 w[3][NB];
#pragma unroll
            for (int dz = 0; dz < 3; dz++)
#pragma unroll
                for (int nb = 0; nb < NB; nb++)
                    w[dz][nb] = __builtin_bit_cast(
                        cr_b8, wp[(size_t)(((c * 5 + q) * 3 + dz) * A.nbt + nb0 + nb) * 64]);
            const uint4* r = xs + fa[q];
#pragma unroll
            for (int zz = 0; zz < HZ; zz++) {
                uint4 f = r[zz * HY * PITCH];
                if (q == 4 && kq >= 2) f = uint4{0u, 0u, 0u, 0u};
                const cr_b8 xf = __builtin_bit_cast(cr_b8, f);
#pragma unroll
                for (int dz = 0; dz < 3; dz++) {
                    const int z = zz - dz;
                    if (z < 0 || z >= CR_Z) continue;
#pragma unroll
                    for (int nb = 0; nb < NB; nb++)
                        acc[z][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[dz][nb], xf, acc[z][nb], 0, 0, 0);
                }
            }
        }
    }
    // D[row = 4 kq + i][col = m]: channel 16 nb + 4 kq + i of the patch's voxel m
    [[maybe_unused]] float hw[4], hb1 = 0.f, halpha = 0.f, loc[4] = {0.f, 0.f, 0.f, 0.f}, lg = 0.f, lgx = 0.f, ll = 0.f;
    if constexpr (EPI == CR_HEAD || EPI == CR_LOSS) {
#pragma unroll
        for (int i = 0; i < 4; i++) hw[i] = A.hp[4 * kq + i];
        hb1 = A.hp[16];
        halpha = A.hp[17];
    }
    const int x = x0 + wave % PX * 4 + mx, y = y0 + wave / PX * 4 + my;
#pragma unroll
    for (int nb = 0; nb < NB; nb++) {
        const int ch = (nb0 + nb) * 16 + 4 * kq;
        float4 bv = {0.f, 0.f, 0.f, 0.f};
        if constexpr (EPI != CR_GRAD && EPI != CR_SPLIT) bv = *reinterpret_cast<const float4*>(A.bias + ch);
        float sum[4];  // running 2x2x2 sum of a pair of planes
#pragma unroll
        for (int z = 0; z < CR_Z; z++) {
            const bool in = x < A.hi && y < A.hi && z0 + z < A.hi;
            const size_t vox = cr_vox(s, b, z0 + z, y, x);
            float v[4] = {acc[z][nb][0] + bv.x, acc[z][nb][1] + bv.y, acc[z][nb][2] + bv.z,
                          acc[z][nb][3] + bv.w};
            if constexpr (EPI == CR_GRAD) {
                if (!in) continue;
                if (A.mask) cr_relu_mask(v, *reinterpret_cast<const uint2*>(A.mask + vox * A.out_c + ch));
                *reinterpret_cast<uint2*>(A.out + vox * A.out_c + ch) = cr_pack4(v);
                continue;
            }
            const bool pooled = EPI == CR_POOL || (EPI == CR_SPLIT && nb0 + nb < A.nup);
            if constexpr (EPI != CR_SPLIT) {
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = fmaxf(v[i], 0.f);
                const uint2 h = cr_pack4(v);
                if constexpr (EPI == CR_ACT || EPI == CR_POOL)
                    if (in) *reinterpret_cast<uint2*>(A.out + vox * A.out_c + ch) = h;
                // what follows sees the rounded activations
                v[0] = cr_bflo(h.x); v[1] = cr_bfhi(h.x); v[2] = cr_bflo(h.y); v[3] = cr_bfhi(h.y);
            } else if (!pooled && in) {
                const int o = ch - A.nup * 16;
                cr_relu_mask(v, *reinterpret_cast<const uint2*>(A.mask + vox * A.out_c + o));
                *reinterpret_cast<uint2*>(A.out + vox * A.out_c + o) = cr_pack4(v);
            }
            if constexpr (EPI == CR_POOL || EPI == CR_SPLIT) {
                if (!pooled) continue;  // uniform
                // x pairs are lanes m and m ^ 1, y pairs m and m ^ 4, z
                // pairs two of this lane's planes; the cube's bounds are
                // even, so a pair is inside it or outside as a whole
#pragma unroll
                for (int i = 0; i < 4; i++) {
                    v[i] += __shfl_xor(v[i], 1);
                    v[i] += __shfl_xor(v[i], 4);
                    sum[i] = (z & 1) ? sum[i] + v[i] : v[i];
                }
                if ((z & 1) && in && ((mx | my) & 1) == 0) {
                    const size_t vc = (((size_t)b * (s.d >> 1) + ((z0 + z) >> 1)) * (s.h >> 1) + (y >> 1)) *
                                          (s.w >> 1) + (x >> 1);
                    if constexpr (EPI == CR_POOL) {
#pragma unroll
                        for (int i = 0; i < 4; i++) sum[i] *= 0.125f;
                    } else {
                        cr_relu_mask(sum, *reinterpret_cast<const uint2*>(A.mask2 + vc * A.out2_c + ch));
                    }
                    *reinterpret_cast<uint2*>(A.out2 + vc * A.out2_c + ch) = cr_pack4(sum);
                }
            }
            if constexpr (EPI == CR_HEAD || EPI == CR_LOSS) {
                float o = hw[0] * v[0] + hw[1] * v[1] + hw[2] * v[2] + hw[3] * v[3];
                o += __shfl_xor(o, 16);
                o += __shfl_xor(o, 32);
                size_t at = 0;
                const bool have = in && cr_vol_at(A.vol, s.w, b, z0 + z, y, x, at);
                const float xv = have ? A.vol.p[at] * A.vol.scale : 0.f;
                o += hb1 + halpha * xv;
                if constexpr (EPI == CR_HEAD) {
                    if (have && kq == 0) A.vout[at] = o * A.oscale;
                } else if (in) {
                    const float d = o - A.tgt[vox] * A.tscale, g = 2.f * d * A.inv_count;
                    float ga[4];
#pragma unroll
                    for (int i = 0; i < 4; i++) {
                        loc[i] += g * v[i];
                        ga[i] = v[i] > 0.f ? g * hw[i] : 0.f;
                    }
                    *reinterpret_cast<uint2*>(A.out + vox * 16 + 4 * kq) = cr_pack4(ga);
                    lg += g;
                    lgx += g * xv;
                    ll += d * d * A.inv_count;
                }
            }
        }
    }
    if constexpr (EPI == CR_LOSS) {
        // lanes of one channel group by a fixed shuffle tree, then the waves in order
        float* red = reinterpret_cast<float*>(xs);  // [waves][20]
        __syncthreads();
        float t[7] = {loc[0], loc[1], loc[2], loc[3], lg, lgx, ll};
#pragma unroll
        for (int i = 0; i < 7; i++)
            for (int o = 8; o > 0; o >>= 1) t[i] += __shfl_xor(t[i], o);
        if (m == 0) {
#pragma unroll
            for (int i = 0; i < 4; i++) red[wave * 20 + 4 * kq + i] = t[i];
            if (kq == 0) {
#pragma unroll
                for (int i = 0; i < 3; i++) red[wave * 20 + 16 + i] = t[4 + i];
                red[wave * 20 + 19] = 0.f;
            }
        }
        __syncthreads();
        if (threadIdx.x < 20) {
            const int k = threadIdx.x;
            float sum = red[k];
            for (int w = 1; w < PX * PY; w++) sum += red[w * 20 + k];
            A.part[(size_t)wg * 20 + k] = sum;
        }
    }
}

// The first convolution: one input channel, so the 27 taps are one K = 32 step
// (the other 15 channels of its parameters meet zeros and are not read).  The
// FP32 input is read, scaled and rounded here; a lane gathers its eight taps
// from a block of BF16 scalars in LDS.  Bound by the activations it writes.
constexpr int CR_FP = 20;  // LDS row pitch (18 staged)
__device__ __forceinline__ void cr_stage_vol(unsigned short* xs, const CrVol& V, const CrShape& s, int b, int z0, int y0,
                                             int x0, int lo, int hi, int nt) {
    for (int t = threadIdx.x; t < 18 * 10 * 6; t += nt) {
        const int gx = x0 - 1 + t % 18, gy = y0 - 1 + (t / 18) % 10, gz = z0 - 1 + t / 180;
        float v = 0.f;
        size_t at;
        if (min(gx, min(gy, gz)) >= lo && max(gx, max(gy, gz)) < hi && cr_vol_at(V, s.w, b, gz, gy, gx, at))
            v = V.p[at] * V.scale;
        xs[(t / 18) * CR_FP + t % 18] = cr_f2bf(v);
    }
}

__global__ void __launch_bounds__(256) k_cr_first(CrVol V, const uint4* __restrict__ wf, const float* __restrict__ bias,
                                                  unsigned short* __restrict__ out, CrShape s, int lo, int hi) {
    __shared__ unsigned short xs[10 * 6 * CR_FP];
    const int ext = hi - lo;
    const int bxn = (ext + 15) / 16, byn = (ext + 7) / 8, bzn = (ext + 3) / 4;
    int tile, one;
    if (!xcd_tile(bxn * byn * bzn * s.n, 1, tile, one)) return;
    const int x0 = lo + tile % bxn * 16; tile /= bxn;
    const int y0 = lo + tile % byn * 8; tile /= byn;
    const int z0 = lo + tile % bzn * 4;
    const int b = tile / bzn;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4, mx = m & 3, my = m >> 2;
    cr_stage_vol(xs, V, s, b, z0, y0, x0, 0, s.w, 256);
    const cr_b8 w = __builtin_bit_cast(cr_b8, wf[lane]);
    const float4 bv = *reinterpret_cast<const float4*>(bias + 4 * kq);
    int off[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
        const int t = min(kq * 8 + j, 26);
        off[j] = (t / 9 * 10 + t / 3 % 3 + my) * CR_FP + t % 3 + mx;
    }
    __syncthreads();
#pragma unroll
    for (int p = 0; p < 2; p++) {
        const int pid = wave * 2 + p;
        const int x = x0 + (pid & 3) * 4 + mx, y = y0 + (pid >> 2) * 4 + my;
#pragma unroll
        for (int z = 0; z < 4; z++) {
            const unsigned short* r = xs + (z * 10 + (pid >> 2) * 4) * CR_FP + (pid & 3) * 4;
            unsigned h[8];
#pragma unroll
            for (int j = 0; j < 8; j++) h[j] = kq * 8 + j < 27 ? r[off[j]] : 0;
            const uint4 f = {h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16};
            const cr_f4 d = __builtin_amdgcn_mfma_f32_16x16x32_bf16(w, __builtin_bit_cast(cr_b8, f),
                                                                   cr_f4{bv.x, bv.y, bv.z, bv.w}, 0, 0, 0);
            if (x >= hi || y >= hi || z0 + z >= hi) continue;
            const float v[4] = {fmaxf(d[0], 0.f), fmaxf(d[1], 0.f), fmaxf(d[2], 0.f), fmaxf(d[3], 0.f)};
            *reinterpret_cast<uint2*>(out + cr_vox(s, b, z0 + z, y, x) * 16 + 4 * kq) = cr_pack4(v);
        }
    }
}

// Four 16-bit LDS values per lane, transposed over each group of 16 lanes:
// lane 4 r + c of a group reads 8 bytes (row r, columns 4 c .. 4 c + 3) and
// lane j receives column j of rows 0 .. 3.  With a row per voxel and a column
// per channel this turns channels-last data into the K-major fragments of a
// contraction over voxels.
__device__ __forceinline__ cr_s4 cr_read_tr(const unsigned short* p) {
    typedef __attribute__((address_space(3))) cr_s4 lds_s4;
    return __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4*)p);
}
__device__ __forceinline__ cr_b8 cr_frag_tr(const unsigned short* p0, const unsigned short* p1) {
    const cr_s4 a = cr_read_tr(p0), b = cr_read_tr(p1);
    return __builtin_bit_cast(cr_b8, __builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

constexpr int CR_WBX = 16, CR_WBY = 8, CR_WBZ = 4;     // voxel block of a weight-gradient step
constexpr int CR_WHX = CR_WBX + 2, CR_WHY = CR_WBY + 2, CR_WHZ = CR_WBZ + 2;
constexpr int CR_WT = 192;                             // three waves

// Weight and bias gradients of one 16-channel input slice (blockIdx.y) and
// NO blocks of 16 output channels (from blockIdx.z * NO), summed over the
// voxel blocks g, g + G, g + 2 G, ... (g = blockIdx.x) of the cube
// [lo, hi)^3 outside which dy is zero: part[g][tap][ci][co], then
// part[g][27 cin cout + co] (FP32).
//
// Bound by LDS reads: both operands are staged channels last and read through
// the transposing LDS load, 512 bytes an instruction.  K = 32 is two x rows of
// 16 voxels.  A wave owns three of the nine (dy, dx) taps with all three dz:
// it holds the output gradients of the block's four z planes in registers, so
// each input fragment (one of six planes) serves up to three products, 18
// input reads for 36 products.  Staging 16 x 8 x 4 voxels with their halo
// reads 2.1 times the input.  The form before it (one 16-bit LDS read per
// element, K = 16) took 512 us a layer on average for four 80^3 crops.
template <int NO>
__global__ void __launch_bounds__(CR_WT) k_cr_wgrad(CrIn in, int cin, const unsigned short* __restrict__ dy, int cout,
                                                    float* __restrict__ part, CrShape s, int lo, int hi, int G) {
    __shared__ __align__(16) unsigned short xs[CR_WHX * CR_WHY * CR_WHZ * 16];
    __shared__ __align__(16) unsigned short ys[NO][CR_WBX * CR_WBY * CR_WBZ * 16];
    const int g = blockIdx.x, c = blockIdx.y, o0 = blockIdx.z * NO * 16;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4;
    // this lane's part of a transposed read: voxel row m / 4 of its group of
    // four, channels 4 (m % 4) ..; the group's first voxel is x = 8 (kq % 2)
    // of row kq / 2 (the second read takes the next four voxels)
    const int lrow = kq >> 1, lvx = (kq & 1) * 8 + (m >> 2), lch = (m & 3) * 4;
    const int e = hi - lo;
    const int bx_n = (e + CR_WBX - 1) / CR_WBX, by_n = (e + CR_WBY - 1) / CR_WBY, bz_n = (e + CR_WBZ - 1) / CR_WBZ;
    const int nblocks = s.n * bz_n * by_n * bx_n;
    // the input is formed up to one voxel around the cube and no further
    const int ilo = max(lo - 1, 0), ihi = min(hi + 1, s.w);
    cr_f4 acc[9][NO], bacc[NO];
#pragma unroll
    for (int nb = 0; nb < NO; nb++) {
        bacc[nb] = cr_f4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int t = 0; t < 9; t++) acc[t][nb] = cr_f4{0.f, 0.f, 0.f, 0.f};
    }
    cr_b8 ones;
#pragma unroll
    for (int i = 0; i < 8; i++) ones[i] = (__bf16)1.f;
    for (int blk0 = g; blk0 < nblocks; blk0 += G) {
        int blk = blk0;
        const int x0 = lo + blk % bx_n * CR_WBX; blk /= bx_n;
        const int y0 = lo + blk % by_n * CR_WBY; blk /= by_n;
        const int z0 = lo + blk % bz_n * CR_WBZ;
        const int b = blk / bz_n;
        __syncthreads();
        for (int t = threadIdx.x; t < CR_WHX * CR_WHY * CR_WHZ * 2; t += CR_WT) {
            const int v = t >> 1, half = t & 1;
            const int lx = v % CR_WHX, ly = (v / CR_WHX) % CR_WHY, lz = v / (CR_WHX * CR_WHY);
            const int gx = x0 - 1 + lx, gy = y0 - 1 + ly, gz = z0 - 1 + lz;
            uint4 val = {0u, 0u, 0u, 0u};
            if (min(gx, min(gy, gz)) >= ilo && max(gx, max(gy, gz)) < ihi)
                val = cr_load(in, s, c, half, b, gz, gy, gx);
            *reinterpret_cast<uint4*>(xs + t * 8) = val;
        }
#pragma unroll
        for (int nb = 0; nb < NO; nb++)
            for (int t = threadIdx.x; t < CR_WBX * CR_WBY * CR_WBZ * 2; t += CR_WT) {
                const int v = t >> 1, half = t & 1;
                const int lx = v % CR_WBX, ly = (v / CR_WBX) % CR_WBY, lz = v / (CR_WBX * CR_WBY);
                const int gx = x0 + lx, gy = y0 + ly, gz = z0 + lz;
                uint4 val = {0u, 0u, 0u, 0u};
                if (gx < hi && gy < hi && gz < hi)
                    val = *reinterpret_cast<const uint4*>(dy + cr_vox(s, b, gz, gy, gx) * cout + o0 + nb * 16 +
                                                          half * 8);
                *reinterpret_cast<uint4*>(ys[nb] + t * 8) = val;
            }
        __syncthreads();
#pragma unroll 1
        for (int yp = 0; yp < CR_WBY; yp += 2) {
            cr_b8 bf[CR_WBZ][NO];
#pragma unroll
            for (int z = 0; z < CR_WBZ; z++)
#pragma unroll
                for (int nb = 0; nb < NO; nb++) {
                    const unsigned short* q = ys[nb] + ((z * CR_WBY + yp + lrow) * CR_WBX + lvx) * 16 + lch;
                    bf[z][nb] = cr_frag_tr(q, q + 4 * 16);
                }
            if (wave == 0) {
#pragma unroll
                for (int z = 0; z < CR_WBZ; z++)
#pragma unroll
                    for (int nb = 0; nb < NO; nb++)
                        bacc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ones, bf[z][nb], bacc[nb], 0, 0, 0);
            }
#pragma unroll
            for (int k = 0; k < 3; k++) {
                // (dy, dx) = (wave, k) - 1
                const unsigned short* q = xs + ((yp + lrow + wave) * CR_WHX + lvx + k) * 16 + lch;
#pragma unroll
                for (int zz = 0; zz < CR_WHZ; zz++) {
                    const unsigned short* r = q + zz * CR_WHX * CR_WHY * 16;
                    const cr_b8 af = cr_frag_tr(r, r + 4 * 16);
#pragma unroll
                    for (int dz = 0; dz < 3; dz++) {
                        const int z = zz - dz;  // input plane zz (with halo) = output plane z + dz
                        if (z < 0 || z >= CR_WBZ) continue;
#pragma unroll
                        for (int nb = 0; nb < NO; nb++)
                            acc[dz * 3 + k][nb] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(af, bf[z][nb], acc[dz * 3 + k][nb], 0, 0, 0);
                    }
                }
            }
        }
    }
    // D[ci = 4 kq + i][co = m]
    const size_t nw = (size_t)27 * cin * cout;
    float* P = part + (size_t)g * (nw + cout);
#pragma unroll
    for (int nb = 0; nb < NO; nb++) {
        const int co = o0 + nb * 16 + m;
#pragma unroll
        for (int t = 0; t < 9; t++) {
            const int tap = (t / 3) * 9 + wave * 3 + t % 3;
#pragma unroll
            for (int i = 0; i < 4; i++) P[((size_t)tap * cin + c * 16 + 4 * kq + i) * cout + co] = acc[t][nb][i];
        }
        if (c == 0 && wave == 0 && kq == 0) P[nw + co] = bacc[nb][0];
    }
}

// The first layer's weight and bias gradients: one input channel, so the 27
// taps and a row of ones (the bias) are the matrix rows and the contraction
// over voxels runs on two row blocks instead of 27 taps.  part[g][28][16].
__global__ void __launch_bounds__(256) k_cr_wgrad_first(CrVol V, const unsigned short* __restrict__ dy,
                                                        float* __restrict__ part, CrShape s, int lo, int hi, int G) {
    __shared__ unsigned short xs[10 * 6 * CR_FP];
    __shared__ __align__(16) unsigned short ys[CR_WBX * CR_WBY * CR_WBZ * 16];
    const int g = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4;
    const int lrow = kq >> 1, lvx = (kq & 1) * 8 + (m >> 2), lch = (m & 3) * 4;
    const int e = hi - lo;
    const int bx_n = (e + CR_WBX - 1) / CR_WBX, by_n = (e + CR_WBY - 1) / CR_WBY, bz_n = (e + CR_WBZ - 1) / CR_WBZ;
    const int nblocks = s.n * bz_n * by_n * bx_n;
    int off[2];  // tap 16 k + m of the first voxel of this lane's eight
#pragma unroll
    for (int k = 0; k < 2; k++) {
        const int t = min(16 * k + m, 26);
        off[k] = (t / 9 * 10 + t / 3 % 3 + lrow) * CR_FP + t % 3 + (kq & 1) * 8;
    }
    cr_f4 acc[2] = {cr_f4{0.f, 0.f, 0.f, 0.f}, cr_f4{0.f, 0.f, 0.f, 0.f}};
    for (int blk0 = g; blk0 < nblocks; blk0 += G) {
        int blk = blk0;
        const int x0 = lo + blk % bx_n * CR_WBX; blk /= bx_n;
        const int y0 = lo + blk % by_n * CR_WBY; blk /= by_n;
        const int z0 = lo + blk % bz_n * CR_WBZ;
        const int b = blk / bz_n;
        __syncthreads();
        cr_stage_vol(xs, V, s, b, z0, y0, x0, 0, s.w, 256);
        for (int t = threadIdx.x; t < CR_WBX * CR_WBY * CR_WBZ * 2; t += 256) {
            const int v = t >> 1, half = t & 1;
            const int gx = x0 + v % CR_WBX, gy = y0 + (v / CR_WBX) % CR_WBY, gz = z0 + v / (CR_WBX * CR_WBY);
            uint4 val = {0u, 0u, 0u, 0u};
            if (gx < hi && gy < hi && gz < hi)
                val = *reinterpret_cast<const uint4*>(dy + cr_vox(s, b, gz, gy, gx) * 16 + half * 8);
            *reinterpret_cast<uint4*>(ys + t * 8) = val;
        }
        __syncthreads();
        // wave = z plane of the block
#pragma unroll
        for (int yp = 0; yp < CR_WBY; yp += 2) {
            const unsigned short* q = ys + ((wave * CR_WBY + yp + lrow) * CR_WBX + lvx) * 16 + lch;
            const cr_b8 bf = cr_frag_tr(q, q + 4 * 16);
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const unsigned short* r = xs + (wave * 10 + yp) * CR_FP + off[k];
                unsigned h[8];
#pragma unroll
                for (int j = 0; j < 8; j++) h[j] = 16 * k + m < 27 ? r[j] : (16 * k + m == 27 ? 0x3f80u : 0u);
                const uint4 f = {h[0] | h[1] << 16, h[2] | h[3] << 16, h[4] | h[5] << 16, h[6] | h[7] << 16};
                acc[k] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(cr_b8, f), bf, acc[k], 0, 0, 0);
            }
        }
    }
    // the four waves' sums in order
    __syncthreads();
    float* red = reinterpret_cast<float*>(ys);  // [4][32][16]
#pragma unroll
    for (int k = 0; k < 2; k++)
#pragma unroll
        for (int i = 0; i < 4; i++) red[(wave * 32 + 16 * k + 4 * kq + i) * 16 + m] = acc[k][i];
    __syncthreads();
    for (int t = threadIdx.x; t < 28 * 16; t += 256)
        part[(size_t)g * 448 + t] = ((red[t] + red[512 + t]) + red[1024 + t]) + red[1536 + t];
}

// Sum of the G partial gradients of n values into grad.  A work-group takes
// 64 values, four threads a value with a quarter of the partials each; every
// quarter and the four quarters are added in order, so the sum is the same in
// every run.  first: the values are [28][16] of the first layer, whose weights
// [tap][ci][co] with ci > 0 never meet an input and keep a zero gradient.
__global__ void __launch_bounds__(256) k_cr_reduce(const float* __restrict__ part, int G, size_t n,
                                                   float* __restrict__ grad, int first) {
    __shared__ float red[4][64];
    const int l = threadIdx.x & 63, q = threadIdx.x >> 6;
    const size_t t = (size_t)blockIdx.x * 64 + l;
    const int per = (G + 3) / 4, g1 = min(G, (q + 1) * per);
    float sum = 0.f;
    if (t < n) {
#pragma unroll 8
        for (int g = q * per; g < g1; g++) sum += part[(size_t)g * n + t];
    }
    red[q][l] = sum;
    __syncthreads();
    const size_t at = first ? (t >> 4) * 256 + (t & 15) : t;
    if (q == 0 && t < n) grad[at] = ((red[0][l] + red[1][l]) + red[2][l]) + red[3][l];
}

// Gradient of an activation that is both pooled and concatenated: in the cube
// [lo, hi)^3, g = (g inside [glo, ghi)^3, else 0, + gc at half the coordinates
// / 8) where act > 0, else 0.  Eight channels a thread.
__global__ void __launch_bounds__(256) k_cr_pool_bwd(unsigned short* __restrict__ g, const unsigned short* __restrict__ gc,
                                                     const unsigned short* __restrict__ act, int c, CrShape s, int lo,
                                                     int hi, int glo, int ghi) {
    const int ext = hi - lo, c8 = c / 8;
    const unsigned t = blockIdx.x * 256 + threadIdx.x;
    const int k = (int)(t % c8);
    unsigned v = t / c8;
    const int x = lo + (int)(v % ext); v /= ext;
    const int y = lo + (int)(v % ext); v /= ext;
    const int z = lo + (int)(v % ext);
    const int b = (int)(v / ext);
    if (b >= s.n) return;
    const size_t at = cr_vox(s, b, z, y, x) * c + k * 8;
    const size_t ac = ((((size_t)b * (s.d / 2) + z / 2) * (s.h / 2) + y / 2) * (s.w / 2) + x / 2) * c + k * 8;
    const bool have = min(x, min(y, z)) >= glo && max(x, max(y, z)) < ghi;
    uint4 gv = {0u, 0u, 0u, 0u};
    if (have) gv = *reinterpret_cast<const uint4*>(g + at);
    const uint4 cv = *reinterpret_cast<const uint4*>(gc + ac), av = *reinterpret_cast<const uint4*>(act + at);
    const unsigned gw[4] = {gv.x, gv.y, gv.z, gv.w}, cw[4] = {cv.x, cv.y, cv.z, cv.w}, aw[4] = {av.x, av.y, av.z, av.w};
    uint2 r[2];
#pragma unroll
    for (int h = 0; h < 2; h++) {
        float f[4];
#pragma unroll
        for (int i = 0; i < 2; i++) {
            f[2 * i] = cr_bflo(gw[2 * h + i]) + 0.125f * cr_bflo(cw[2 * h + i]);
            f[2 * i + 1] = cr_bfhi(gw[2 * h + i]) + 0.125f * cr_bfhi(cw[2 * h + i]);
        }
        cr_relu_mask(f, uint2{aw[2 * h], aw[2 * h + 1]});
        r[h] = cr_pack4(f);
    }
    *reinterpret_cast<uint4*>(g + at) = uint4{r[0].x, r[0].y, r[1].x, r[1].y};
}

// Sum of nblk partial rows of width 20 in FP64 into res[20] and, of the first
// kHead, into the head's gradient: 32 threads a column, each a strided share
// in order, then the 32 shares in order.
__global__ void __launch_bounds__(640) k_cr_head_reduce(const float* __restrict__ part, int nblk, int nhead,
                                                        float* __restrict__ res, float* __restrict__ ghead) {
    __shared__ double red[32][20];
    const int k = threadIdx.x % 20, q = threadIdx.x / 20;
    double s = 0.0;
    for (int b = q; b < nblk; b += 32) s += part[(size_t)b * 20 + k];
    red[q][k] = s;
    __syncthreads();
    if (q == 0) {
        for (int i = 1; i < 32; i++) s += red[i][k];
        res[k] = (float)s;
        if (k < nhead) ghead[k] = (float)s;
    }
}

// Adam (Kingma & Ba 2015) on the flat parameter vector with bias-corrected
// step lr_t = lr sqrt(1 - b2^t) / (1 - b1^t).
__global__ void k_cr_adam(float* __restrict__ w, const float* __restrict__ g, float* __restrict__ m,
                          float* __restrict__ v, size_t n, float lr_t, float b1, float b2, float eps) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= n) return;
    const float gg = g[t];
    const float mm = b1 * m[t] + (1.f - b1) * gg;
    const float vv = b2 * v[t] + (1.f - b2) * gg * gg;
    m[t] = mm;
    v[t] = vv;
    w[t] -= lr_t * mm / (sqrtf(vv) + eps);
}

// BF16 MFMA fragments of one layer's weights W[27][cin][cout] (FP32):
// forward (fwd != 0: K = (tap, ci), rows = co) or input gradient (K =
// (mirrored tap, co), rows = ci).  Fragment (((slice * 5 + pair) * 3 + dz) * NB
// + nb) * 64 + lane holds, for lane (n = lane % 16, kq = lane / 16), the 8
// values of tap 9 dz + 2 pair + kq / 2, K channels slice * 16 + (kq % 2) * 8
// + j, output channel nb * 16 + n (zero where 2 pair + kq / 2 = 9).
__global__ void k_cr_pack(const float* __restrict__ W, int cin, int cout, int fwd, uint4* __restrict__ wf) {
    const int kin = fwd ? cin : cout, nout = fwd ? cout : cin;
    const int NB = nout / 16, ns = kin / 16;
    const size_t total = (size_t)ns * CR_STEPS * NB * 64;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= total) return;
    const int lane = (int)(t % 64);
    size_t r = t / 64;
    const int nb = (int)(r % NB); r /= NB;
    const int dz = (int)(r % 3); r /= 3;
    const int pair = (int)(r % 5);
    const int c = (int)(r / 5);
    const int n = lane & 15, kq = lane >> 4;
    const int t9 = 2 * pair + (kq >> 1), tap = 9 * dz + t9;
    uint4 q;
    unsigned short* h = reinterpret_cast<unsigned short*>(&q);
    for (int j = 0; j < 8; j++) {
        const int k = c * 16 + (kq & 1) * 8 + j, o = nb * 16 + n;
        float val = 0.f;
        if (t9 < 9) val = fwd ? W[((size_t)tap * cin + k) * cout + o] : W[((size_t)(26 - tap) * cin + o) * cout + k];
        h[j] = cr_f2bf(val);
    }
    wf[t] = q;
}

// The first layer's fragment: lane (n = lane % 16, kq = lane / 16) holds taps
// 8 kq + j (zero from 27 on) of input channel 0, output channel n.
__global__ void k_cr_pack_first(const float* __restrict__ W, uint4* __restrict__ wf) {
    const int lane = threadIdx.x, n = lane & 15, kq = lane >> 4;
    uint4 q;
    unsigned short* h = reinterpret_cast<unsigned short*>(&q);
    for (int j = 0; j < 8; j++) h[j] = kq * 8 + j < 27 ? cr_f2bf(W[(kq * 8 + j) * 256 + n]) : (unsigned short)0;
    wf[lane] = q;
}

}  // namespace utr

namespace {

// Layers of the U-Net (3x3x3 convolutions), in the order of the flat
// parameter vector: W[27][cin][cout] then b[cout] per layer, then the head
// {w1[16], b1, alpha}.
struct CrLayerDef {
    int cin, cout;
};
constexpr CrLayerDef kCrLayers[10] = {
    {16, 16},  // e1a  (input: the volume in channel 0 of 16)
    {16, 16},  // e1b
    {16, 32},  // e2a  (input: pooled e1b)
    {32, 32},  // e2b
    {32, 64},  // e3a  (input: pooled e2b)
    {64, 64},  // e3b
    {96, 32},  // d2a  (input: up(e3b) | e2b)
    {32, 32},  // d2b
    {48, 16},  // d1a  (input: up(d2b) | e1b)
    {16, 16},  // d1b
};
constexpr int kCrHead = 18;

using bf16_t = unsigned short;

struct CrLayer {
    int cin, cout;
    size_t woff, boff;
    DevBuf<uint4> wf, wb;  // forward and input-gradient fragments
};

}  // namespace

struct utr_corr {
    int tile = 64, halo = 8, T = 80, batch = 1, device = 0;
    size_t np = 0, headoff = 0;
    CrLayer L[10];
    DevBuf<float> w, g, m, v, res;
    int step = 0;
    float scale = 1.f;
    // activations (BF16, channels last) at the three resolutions
    DevBuf<bf16_t> e1a, e1b, p1, e2a, e2b, p2, e3a, e3b, d2a, d2b, d1a;
    // activation gradients
    DevBuf<bf16_t> gd1b, gd1a, ge1b, gd2b, gd2a, ge2b, ge3b, ge3a, gp2, ge2a, gp1, ge1a;
    DevBuf<uint4> wfirst;
    DevBuf<float> part, hpart;
    hipStream_t st = nullptr;
    double last_ms = 0.0;
};

namespace {

utr::CrShape cr_shape(int n, int e) {
    utr::CrShape s;
    s.n = n;
    s.d = s.h = s.w = e;
    return s;
}

struct CrCube {
    int lo, hi;
};

// The cubes a network pass over crops of edge T needs when only outputs in
// [h, T - h)^3 count: each is grown by one voxel per convolution behind it,
// halved (rounded outwards) at each coarser level, and made even where a
// pooling or upsampling pairs voxels.  Forward, activation qN is formed on its
// cube from inputs formed on theirs; backward, every gradient is zero outside
// the same cubes.
struct CrCubes {
    CrCube d1b, d1a, c1, d2b, d2a, c2, e3b, e3a, e2b, e2a, e1b, e1a;
};
CrCubes cr_cubes(int T, int h) {
    auto grow = [](CrCube q, int e) { return CrCube{std::max(0, q.lo - 1), std::min(e, q.hi + 1)}; };
    auto half = [](CrCube q) { return CrCube{q.lo / 2, (q.hi + 1) / 2}; };
    auto twice = [](CrCube q) { return CrCube{2 * q.lo, 2 * q.hi}; };
    auto both = [](CrCube a, CrCube b) { return CrCube{std::min(a.lo, b.lo), std::max(a.hi, b.hi)}; };
    CrCubes Q;
    Q.d1b = {h, T - h};
    Q.d1a = grow(Q.d1b, T);
    Q.d2b = half(grow(Q.d1a, T));
    Q.c1 = twice(Q.d2b);  // concatenated input of d1a
    Q.d2a = grow(Q.d2b, T / 2);
    Q.e3b = half(grow(Q.d2a, T / 2));
    Q.c2 = twice(Q.e3b);  // concatenated input of d2a
    Q.e3a = grow(Q.e3b, T / 4);
    Q.e2b = both(Q.c2, twice(grow(Q.e3a, T / 4)));
    Q.e2a = grow(Q.e2b, T / 2);
    Q.e1b = both(Q.c1, twice(grow(Q.e2a, T / 2)));
    Q.e1a = grow(Q.e1b, T);
    return Q;
}

// Work-groups that a cube [lo, hi)^3 of n crops splits into: blocks of px x py
// patches and CR_Z planes.
long cr_tiles(int px, int py, int n, CrCube q) {
    const long e = q.hi - q.lo;
    return n * ((e + 4 * px - 1) / (4 * px)) * ((e + 4 * py - 1) / (4 * py)) * ((e + utr::CR_Z - 1) / utr::CR_Z);
}
long cr_conv_tiles(int n, CrCube q) { return cr_tiles(utr::CR_PX, utr::CR_PY, n, q); }

template <int NB, int EPI>
int cr_conv_launch(utr_corr* c, const utr::CrConv& A) {
    const unsigned tiles = (unsigned)cr_conv_tiles(A.s.n, CrCube{A.lo, A.hi}) * (unsigned)(A.nbt / NB);
    utr::k_cr_conv<NB, EPI><<<utr::xcd_grid(tiles), 64 * utr::CR_PX * utr::CR_PY, 0, c->st>>>(A);
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

// A layer's convolution (forward) or input gradient; the caller fills in what
// its epilogue needs.
utr::CrConv cr_conv_args(const utr_corr* c, int layer, bool fwd, utr::CrIn in, utr::CrShape s, CrCube q, CrCube iq) {
    const CrLayer& Ly = c->L[layer];
    utr::CrConv A{};
    A.in = in;
    A.cin = fwd ? Ly.cin : Ly.cout;
    A.nbt = (fwd ? Ly.cout : Ly.cin) / 16;
    A.wf = fwd ? Ly.wf.p : Ly.wb.p;
    A.bias = c->w.p + Ly.boff;
    A.s = s;
    A.lo = q.lo;
    A.hi = q.hi;
    A.ilo = iq.lo;
    A.ihi = iq.hi;
    return A;
}
utr::CrIn cr_in(const DevBuf<bf16_t>& p, int ch) { return utr::CrIn{nullptr, 0, 0, p.p, ch}; }
utr::CrIn cr_in(const DevBuf<bf16_t>& up, int upc, const DevBuf<bf16_t>& p, int ch) {
    return utr::CrIn{up.p, upc, upc / 16, p.p, ch};
}

int cr_act(utr_corr* c, int layer, utr::CrIn in, bf16_t* out, utr::CrShape s, CrCube q, bf16_t* pooled = nullptr) {
    utr::CrConv A = cr_conv_args(c, layer, true, in, s, q, {0, s.w});
    A.out = out;
    A.out_c = A.out2_c = 16 * A.nbt;
    A.out2 = pooled;
    if (pooled) return A.nbt == 1 ? cr_conv_launch<1, utr::CR_POOL>(c, A) : cr_conv_launch<2, utr::CR_POOL>(c, A);
    return A.nbt == 1 ? cr_conv_launch<1, utr::CR_ACT>(c, A) : cr_conv_launch<2, utr::CR_ACT>(c, A);
}

// Input gradient on cube q of an output gradient that is zero outside gq.
int cr_grad(utr_corr* c, int layer, const DevBuf<bf16_t>& dy, CrCube gq, bf16_t* out, const bf16_t* mask, utr::CrShape s,
            CrCube q) {
    utr::CrConv A = cr_conv_args(c, layer, false, cr_in(dy, c->L[layer].cout), s, q, gq);
    A.out = out;
    A.out_c = 16 * A.nbt;
    A.mask = mask;
    return A.nbt == 1 ? cr_conv_launch<1, utr::CR_GRAD>(c, A) : cr_conv_launch<2, utr::CR_GRAD>(c, A);
}

// The same for a layer whose input is an upsampled tensor of upc channels
// beside one at its own resolution.
int cr_grad_split(utr_corr* c, int layer, const DevBuf<bf16_t>& dy, CrCube gq, bf16_t* gup, const bf16_t* up, int upc,
                  bf16_t* out, const bf16_t* mask, utr::CrShape s, CrCube q) {
    utr::CrConv A = cr_conv_args(c, layer, false, cr_in(dy, c->L[layer].cout), s, q, gq);
    A.nup = upc / 16;
    A.out = out;
    A.out_c = 16 * A.nbt - upc;
    A.mask = mask;
    A.out2 = gup;
    A.out2_c = upc;
    A.mask2 = up;
    return cr_conv_launch<3, utr::CR_SPLIT>(c, A);
}

// Weight-gradient launch of a layer over n cubes [0, e)^3: output blocks per
// work-group, and partial sums G such that about kCrWgradWgs work-groups (two
// to three resident per CU) share the voxel blocks evenly.
constexpr int kCrWgradWgs = 768;
int cr_wgrad_no(int cout) { return cout % 32 == 0 ? 2 : 1; }
int cr_wgrad_groups(int cin, int cout, int n, int e) {
    const int nb = n * ((e + utr::CR_WBX - 1) / utr::CR_WBX) * ((e + utr::CR_WBY - 1) / utr::CR_WBY) *
                   ((e + utr::CR_WBZ - 1) / utr::CR_WBZ);
    const int per_g = (cin / 16) * (cout / 16 / cr_wgrad_no(cout));
    const int want = std::max(1, std::min(nb, (kCrWgradWgs + per_g - 1) / per_g));
    const int each = (nb + want - 1) / want;
    return (nb + each - 1) / each;
}

// dy is zero outside q^3.
int cr_wgrad(utr_corr* c, int layer, utr::CrIn in, const DevBuf<bf16_t>& dy, utr::CrShape s, CrCube q) {
    const CrLayer& Ly = c->L[layer];
    const size_t nw = (size_t)27 * Ly.cin * Ly.cout + Ly.cout;
    const int no = cr_wgrad_no(Ly.cout), G = cr_wgrad_groups(Ly.cin, Ly.cout, s.n, q.hi - q.lo);
    if ((size_t)G * nw > c->part.n) return set_err(UTR_E_STATE, "corrector: gradient workspace too small");
    const dim3 grid(G, Ly.cin / 16, Ly.cout / 16 / no);
    if (no == 2)
        utr::k_cr_wgrad<2><<<grid, utr::CR_WT, 0, c->st>>>(in, Ly.cin, dy.p, Ly.cout, c->part.p, s, q.lo, q.hi, G);
    else
        utr::k_cr_wgrad<1><<<grid, utr::CR_WT, 0, c->st>>>(in, Ly.cin, dy.p, Ly.cout, c->part.p, s, q.lo, q.hi, G);
    UTR_HIP_TRY(hipGetLastError());
    // weights and bias of a layer are contiguous in the gradient vector
    utr::k_cr_reduce<<<(unsigned)((nw + 63) / 64), 256, 0, c->st>>>(c->part.p, G, nw, c->g.p + Ly.woff, 0);
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

int cr_wgrad_first(utr_corr* c, const utr::CrVol& V, const DevBuf<bf16_t>& dy, utr::CrShape s, CrCube q) {
    const int G = cr_wgrad_groups(16, 16, s.n, q.hi - q.lo);
    utr::k_cr_wgrad_first<<<G, 256, 0, c->st>>>(V, dy.p, c->part.p, s, q.lo, q.hi, G);
    UTR_HIP_TRY(hipGetLastError());
    utr::k_cr_reduce<<<7, 256, 0, c->st>>>(c->part.p, G, 448, c->g.p + c->L[0].woff, 1);
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

unsigned cr_blocks(size_t n) { return (unsigned)((n + 255) / 256); }

// Floats the partial sums of any layer's weight gradient need, for any number
// of crops up to the batch and any cube inside the layer's.
size_t cr_part_size() {
    size_t mx = 0;
    for (const auto& d : kCrLayers) {
        const int per_g = (d.cin / 16) * (d.cout / 16 / cr_wgrad_no(d.cout));
        const size_t nw = (size_t)27 * d.cin * d.cout + d.cout;
        mx = std::max(mx, nw * (size_t)((kCrWgradWgs + per_g - 1) / per_g));
    }
    return mx;
}

int cr_alloc(utr_corr* c) {
    const size_t n1 = (size_t)c->batch * c->T * c->T * c->T;
    const size_t n2 = n1 / 8, n3 = n1 / 64;
    // the loss's partial sums: one row per work-group of the last convolution
    const CrCube q = {c->halo, c->T - c->halo};
    const size_t hp = (size_t)cr_conv_tiles(c->batch, q) * 20;
    const hipError_t e[] = {
        c->e1a.alloc(n1 * 16), c->e1b.alloc(n1 * 16), c->p1.alloc(n2 * 16), c->e2a.alloc(n2 * 32),
        c->e2b.alloc(n2 * 32), c->p2.alloc(n3 * 32), c->e3a.alloc(n3 * 64), c->e3b.alloc(n3 * 64),
        c->d2a.alloc(n2 * 32), c->d2b.alloc(n2 * 32), c->d1a.alloc(n1 * 16),
        c->gd1b.alloc(n1 * 16), c->gd1a.alloc(n1 * 16), c->ge1b.alloc(n1 * 16), c->gd2b.alloc(n2 * 32),
        c->gd2a.alloc(n2 * 32), c->ge2b.alloc(n2 * 32), c->ge3b.alloc(n3 * 64), c->ge3a.alloc(n3 * 64),
        c->gp2.alloc(n3 * 32), c->ge2a.alloc(n2 * 32), c->gp1.alloc(n2 * 16), c->ge1a.alloc(n1 * 16),
        c->wfirst.alloc(64), c->part.alloc(cr_part_size()), c->hpart.alloc(hp), c->res.alloc(32)};
    for (hipError_t x : e)
        if (x != hipSuccess)
            return set_err(x == hipErrorOutOfMemory ? UTR_E_NOMEM : UTR_E_DEVICE,
                           std::string("corrector: device allocation failed: ") + hipGetErrorString(x));
    return UTR_OK;
}

int cr_repack(utr_corr* c) {
    utr::k_cr_pack_first<<<1, 64, 0, c->st>>>(c->w.p + c->L[0].woff, c->wfirst.p);
    UTR_HIP_TRY(hipGetLastError());
    for (int l = 1; l < 10; l++) {
        CrLayer& Ly = c->L[l];
        const size_t nf = (size_t)(Ly.cin / 16) * utr::CR_STEPS * (Ly.cout / 16) * 64;
        utr::k_cr_pack<<<cr_blocks(nf), 256, 0, c->st>>>(c->w.p + Ly.woff, Ly.cin, Ly.cout, 1, Ly.wf.p);
        UTR_HIP_TRY(hipGetLastError());
        utr::k_cr_pack<<<cr_blocks(nf), 256, 0, c->st>>>(c->w.p + Ly.woff, Ly.cin, Ly.cout, 0, Ly.wb.p);
        UTR_HIP_TRY(hipGetLastError());
    }
    return UTR_OK;
}

// Forward pass of nb crops of V up to d1a, on the cubes Q.
int cr_forward(utr_corr* c, int nb, const utr::CrVol& V, const CrCubes& Q) {
    const int T = c->T;
    const utr::CrShape s1 = cr_shape(nb, T), s2 = cr_shape(nb, T / 2), s3 = cr_shape(nb, T / 4);
    int rc;
    utr::k_cr_first<<<utr::xcd_grid((unsigned)cr_tiles(4, 2, nb, Q.e1a)), 256, 0, c->st>>>(
        V, c->wfirst.p, c->w.p + c->L[0].boff, c->e1a.p, s1, Q.e1a.lo, Q.e1a.hi);
    UTR_HIP_TRY(hipGetLastError());
    if ((rc = cr_act(c, 1, cr_in(c->e1a, 16), c->e1b.p, s1, Q.e1b, c->p1.p))) return rc;
    if ((rc = cr_act(c, 2, cr_in(c->p1, 16), c->e2a.p, s2, Q.e2a))) return rc;
    if ((rc = cr_act(c, 3, cr_in(c->e2a, 32), c->e2b.p, s2, Q.e2b, c->p2.p))) return rc;
    if ((rc = cr_act(c, 4, cr_in(c->p2, 32), c->e3a.p, s3, Q.e3a))) return rc;
    if ((rc = cr_act(c, 5, cr_in(c->e3a, 64), c->e3b.p, s3, Q.e3b))) return rc;
    if ((rc = cr_act(c, 6, cr_in(c->e3b, 64, c->e2b, 32), c->d2a.p, s2, Q.d2a))) return rc;
    if ((rc = cr_act(c, 7, cr_in(c->d2a, 32), c->d2b.p, s2, Q.d2b))) return rc;
    return cr_act(c, 8, cr_in(c->d2b, 32, c->e1b, 16), c->d1a.p, s1, Q.d1a);
}

// The last convolution with the head: out (laid out like V) = oscale * (alpha x
// + b1 + w1 . d1b) on the cube Q.d1b of each crop.
int cr_head(utr_corr* c, int nb, const utr::CrVol& V, const CrCubes& Q, float* out, float oscale) {
    utr::CrConv A = cr_conv_args(c, 9, true, cr_in(c->d1a, 16), cr_shape(nb, c->T), Q.d1b, {0, c->T});
    A.vol = V;
    A.hp = c->w.p + c->headoff;
    A.vout = out;
    A.oscale = oscale;
    return cr_conv_launch<1, utr::CR_HEAD>(c, A);
}

// Loss and gradients of nb crops V after cr_forward against the targets tgt
// (unscaled): gradient vector in c->g, {dw1, db1, dalpha, loss} in res.
int cr_backward(utr_corr* c, int nb, const utr::CrVol& V, const CrCubes& Q, const float* tgt) {
    const int T = c->T;
    const utr::CrShape s1 = cr_shape(nb, T), s2 = cr_shape(nb, T / 2), s3 = cr_shape(nb, T / 4);
    const double cnt = (double)nb * c->tile * c->tile * c->tile;
    int rc;
    utr::CrConv A = cr_conv_args(c, 9, true, cr_in(c->d1a, 16), s1, Q.d1b, {0, T});
    A.vol = V;
    A.hp = c->w.p + c->headoff;
    A.out = c->gd1b.p;
    A.tgt = tgt;
    A.tscale = c->scale;
    A.inv_count = (float)(1.0 / cnt);
    A.part = c->hpart.p;
    const long nwg = cr_conv_tiles(nb, Q.d1b);
    if ((size_t)nwg * 20 > c->hpart.n) return set_err(UTR_E_STATE, "corrector: loss workspace too small");
    if ((rc = cr_conv_launch<1, utr::CR_LOSS>(c, A))) return rc;
    utr::k_cr_head_reduce<<<1, 640, 0, c->st>>>(c->hpart.p, (int)nwg, kCrHead, c->res.p, c->g.p + c->headoff);
    UTR_HIP_TRY(hipGetLastError());
    auto pool_bwd = [&](DevBuf<bf16_t>& g, const DevBuf<bf16_t>& gc, const DevBuf<bf16_t>& act, int ch, utr::CrShape s,
                        CrCube q, CrCube have) -> int {
        const size_t e = (size_t)(q.hi - q.lo), n = (size_t)nb * e * e * e * (ch / 8);
        utr::k_cr_pool_bwd<<<cr_blocks(n), 256, 0, c->st>>>(g.p, gc.p, act.p, ch, s, q.lo, q.hi, have.lo, have.hi);
        UTR_HIP_TRY(hipGetLastError());
        return UTR_OK;
    };
    // d1b, d1a
    if ((rc = cr_wgrad(c, 9, cr_in(c->d1a, 16), c->gd1b, s1, Q.d1b))) return rc;
    if ((rc = cr_grad(c, 9, c->gd1b, Q.d1b, c->gd1a.p, c->d1a.p, s1, Q.d1a))) return rc;
    if ((rc = cr_wgrad(c, 8, cr_in(c->d2b, 32, c->e1b, 16), c->gd1a, s1, Q.d1a))) return rc;
    if ((rc = cr_grad_split(c, 8, c->gd1a, Q.d1a, c->gd2b.p, c->d2b.p, 32, c->ge1b.p, c->e1b.p, s1, Q.c1))) return rc;
    // d2b, d2a
    if ((rc = cr_wgrad(c, 7, cr_in(c->d2a, 32), c->gd2b, s2, Q.d2b))) return rc;
    if ((rc = cr_grad(c, 7, c->gd2b, Q.d2b, c->gd2a.p, c->d2a.p, s2, Q.d2a))) return rc;
    if ((rc = cr_wgrad(c, 6, cr_in(c->e3b, 64, c->e2b, 32), c->gd2a, s2, Q.d2a))) return rc;
    if ((rc = cr_grad_split(c, 6, c->gd2a, Q.d2a, c->ge3b.p, c->e3b.p, 64, c->ge2b.p, c->e2b.p, s2, Q.c2))) return rc;
    // e3b, e3a
    const CrCube p2 = {Q.e2b.lo / 2, Q.e2b.hi / 2}, p1 = {Q.e1b.lo / 2, Q.e1b.hi / 2};
    if ((rc = cr_wgrad(c, 5, cr_in(c->e3a, 64), c->ge3b, s3, Q.e3b))) return rc;
    if ((rc = cr_grad(c, 5, c->ge3b, Q.e3b, c->ge3a.p, c->e3a.p, s3, Q.e3a))) return rc;
    if ((rc = cr_wgrad(c, 4, cr_in(c->p2, 32), c->ge3a, s3, Q.e3a))) return rc;
    if ((rc = cr_grad(c, 4, c->ge3a, Q.e3a, c->gp2.p, nullptr, s3, p2))) return rc;
    // e2b (skip and pooled paths), e2a
    if ((rc = pool_bwd(c->ge2b, c->gp2, c->e2b, 32, s2, Q.e2b, Q.c2))) return rc;
    if ((rc = cr_wgrad(c, 3, cr_in(c->e2a, 32), c->ge2b, s2, Q.e2b))) return rc;
    if ((rc = cr_grad(c, 3, c->ge2b, Q.e2b, c->ge2a.p, c->e2a.p, s2, Q.e2a))) return rc;
    if ((rc = cr_wgrad(c, 2, cr_in(c->p1, 16), c->ge2a, s2, Q.e2a))) return rc;
    if ((rc = cr_grad(c, 2, c->ge2a, Q.e2a, c->gp1.p, nullptr, s2, p1))) return rc;
    // e1b, e1a
    if ((rc = pool_bwd(c->ge1b, c->gp1, c->e1b, 16, s1, Q.e1b, Q.c1))) return rc;
    if ((rc = cr_wgrad(c, 1, cr_in(c->e1a, 16), c->ge1b, s1, Q.e1b))) return rc;
    if ((rc = cr_grad(c, 1, c->ge1b, Q.e1b, c->ge1a.p, c->e1a.p, s1, Q.e1a))) return rc;
    return cr_wgrad_first(c, V, c->ge1a, s1, Q.e1a);
}

utr::CrVol cr_crops(const utr_corr* c, const float* d_in) {
    utr::CrVol V{};
    V.p = d_in;
    V.scale = c->scale;
    return V;
}

int cr_check(utr_corr* c) {
    if (!c) return set_err(UTR_E_INVALID, "null corrector");
    UTR_HIP_TRY(hipSetDevice(c->device));
    return UTR_OK;
}

}  // namespace

extern "C" {

int utr_corr_create(int tile, int halo, int batch, unsigned long long seed, utr_corr** out) {
    if (!out) return set_err(UTR_E_INVALID, "null output pointer");
    *out = nullptr;
    if (tile < 4 || halo < 0 || batch < 1 || (tile + 2 * halo) % 4 != 0 || tile + 2 * halo > 512)
        return set_err(UTR_E_INVALID,
                       "utr_corr_create: tile >= 4, halo >= 0, batch >= 1 and tile + 2 halo a multiple of 4 up to 512");
    utr_corr* c = new utr_corr;
    auto fail = [&](int rc) {
        utr_corr_destroy(c);
        return rc;
    };
    if (hipGetDevice(&c->device) != hipSuccess) return fail(set_err(UTR_E_DEVICE, "no HIP device"));
    c->tile = tile;
    c->halo = halo;
    c->T = tile + 2 * halo;
    c->batch = batch;
    size_t off = 0;
    for (int l = 0; l < 10; l++) {
        c->L[l].cin = kCrLayers[l].cin;
        c->L[l].cout = kCrLayers[l].cout;
        c->L[l].woff = off;
        off += (size_t)27 * c->L[l].cin * c->L[l].cout;
        c->L[l].boff = off;
        off += c->L[l].cout;
    }
    c->headoff = off;
    c->np = off + kCrHead;
    // He initialisation (seeded): N(0, 2 / fan_in), fan_in = 27 cin (27 for
    // the first layer, whose input has one live channel); biases 0; head
    // w1 ~ N(0, 1e-4), b1 = 0, alpha = 1 (the network starts as the identity).
    std::vector<float> w(c->np, 0.f);
    uint64_t state = seed * 0x9E3779B97F4A7C15ull + 0x632BE59BD9B4E019ull;
    auto gauss = [&]() {
        auto u = [&]() {
            state += 0x9E3779B97F4A7C15ull;
            uint64_t z = state;
            z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
            z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
            return ((double)((z ^ (z >> 31)) >> 11) + 0.5) * (1.0 / 9007199254740992.0);
        };
        const double u1 = u(), u2 = u();
        return std::sqrt(-2.0 * std::log(u1)) * std::cos(2.0 * utr::kPi * u2);
    };
    for (int l = 0; l < 10; l++) {
        const double fan = 27.0 * (l == 0 ? 1 : c->L[l].cin);
        const double sd = std::sqrt(2.0 / fan);
        for (size_t k = 0; k < (size_t)27 * c->L[l].cin * c->L[l].cout; k++) w[c->L[l].woff + k] = (float)(sd * gauss());
    }
    for (int k = 0; k < 16; k++) w[c->headoff + k] = (float)(1e-2 * gauss());
    w[c->headoff + 17] = 1.f;
    if (c->w.alloc(c->np) || c->g.alloc(c->np) || c->m.alloc(c->np) || c->v.alloc(c->np))
        return fail(set_err(UTR_E_NOMEM, "corrector: parameter allocation failed"));
    for (int l = 0; l < 10; l++) {
        const size_t nf = (size_t)(c->L[l].cin / 16) * utr::CR_STEPS * (c->L[l].cout / 16) * 64;
        const size_t nb = (size_t)(c->L[l].cout / 16) * utr::CR_STEPS * (c->L[l].cin / 16) * 64;
        if (c->L[l].wf.alloc(nf) || c->L[l].wb.alloc(nb))
            return fail(set_err(UTR_E_NOMEM, "corrector: fragment allocation failed"));
    }
    if (int rc = cr_alloc(c)) return fail(rc);
    if (hipStreamCreateWithFlags(&c->st, hipStreamNonBlocking) != hipSuccess)
        return fail(set_err(UTR_E_DEVICE, "corrector: stream creation failed"));
    if (hipMemcpy(c->w.p, w.data(), sizeof(float) * c->np, hipMemcpyHostToDevice) != hipSuccess ||
        hipMemset(c->m.p, 0, sizeof(float) * c->np) != hipSuccess ||
        hipMemset(c->v.p, 0, sizeof(float) * c->np) != hipSuccess ||
        hipMemset(c->g.p, 0, sizeof(float) * c->np) != hipSuccess)
        return fail(set_err(UTR_E_DEVICE, "corrector: parameter upload failed"));
    if (int rc = cr_repack(c)) return fail(rc);
    if (hipStreamSynchronize(c->st) != hipSuccess) return fail(set_err(UTR_E_DEVICE, "corrector: set-up failed"));
    *out = c;
    return UTR_OK;
}

int utr_corr_nparams(const utr_corr* c) { return c ? (int)c->np : -1; }

int utr_corr_tile(const utr_corr* c, int* tile, int* halo, int* batch) {
    if (!c) return set_err(UTR_E_INVALID, "null corrector");
    if (tile) *tile = c->tile;
    if (halo) *halo = c->halo;
    if (batch) *batch = c->batch;
    return UTR_OK;
}

int utr_corr_get_params(utr_corr* c, float* host, float* scale) {
    if (int rc = cr_check(c)) return rc;
    if (host) UTR_HIP_TRY(hipMemcpy(host, c->w.p, sizeof(float) * c->np, hipMemcpyDeviceToHost));
    if (scale) *scale = c->scale;
    return UTR_OK;
}

int utr_corr_set_params(utr_corr* c, const float* host, float scale) {
    if (int rc = cr_check(c)) return rc;
    if (!(scale > 0) || !std::isfinite(scale)) return set_err(UTR_E_INVALID, "utr_corr_set_params: scale must be positive");
    c->scale = scale;
    if (host) {
        UTR_HIP_TRY(hipMemcpy(c->w.p, host, sizeof(float) * c->np, hipMemcpyHostToDevice));
        UTR_HIP_TRY(hipMemsetAsync(c->m.p, 0, sizeof(float) * c->np, c->st));
        UTR_HIP_TRY(hipMemsetAsync(c->v.p, 0, sizeof(float) * c->np, c->st));
        c->step = 0;
        if (int rc = cr_repack(c)) return rc;
    }
    UTR_HIP_TRY(hipStreamSynchronize(c->st));
    return UTR_OK;
}

int utr_corr_forward(utr_corr* c, const float* d_in, int nb, float* d_out) {
    if (int rc = cr_check(c)) return rc;
    if (!d_in || !d_out || nb < 1 || nb > c->batch) return set_err(UTR_E_INVALID, "utr_corr_forward: 1 <= nb <= batch crops");
    const utr::CrVol V = cr_crops(c, d_in);
    const CrCubes Q = cr_cubes(c->T, 0);  // the whole crop is returned
    if (int rc = cr_forward(c, nb, V, Q)) return rc;
    if (int rc = cr_head(c, nb, V, Q, d_out, 1.f / c->scale)) return rc;
    UTR_HIP_TRY(hipStreamSynchronize(c->st));
    return UTR_OK;
}

int utr_corr_gradient(utr_corr* c, const float* d_in, const float* d_tgt, int nb, float* loss, float* grad_host) {
    if (int rc = cr_check(c)) return rc;
    if (!d_in || !d_tgt || nb < 1 || nb > c->batch)
        return set_err(UTR_E_INVALID, "utr_corr_gradient: 1 <= nb <= batch crops");
    const utr::CrVol V = cr_crops(c, d_in);
    const CrCubes Q = cr_cubes(c->T, c->halo);
    if (int rc = cr_forward(c, nb, V, Q)) return rc;
    if (int rc = cr_backward(c, nb, V, Q, d_tgt)) return rc;
    float res[20];
    UTR_HIP_TRY(hipMemcpyAsync(res, c->res.p, sizeof(res), hipMemcpyDeviceToHost, c->st));
    UTR_HIP_TRY(hipStreamSynchronize(c->st));
    if (loss) *loss = res[18];
    if (grad_host) UTR_HIP_TRY(hipMemcpy(grad_host, c->g.p, sizeof(float) * c->np, hipMemcpyDeviceToHost));
    return UTR_OK;
}

int utr_corr_train_step(utr_corr* c, const float* d_in, const float* d_tgt, int nb, float lr, float* loss) {
    if (int rc = cr_check(c)) return rc;
    if (!d_in || !d_tgt || nb < 1 || nb > c->batch)
        return set_err(UTR_E_INVALID, "utr_corr_train_step: 1 <= nb <= batch crops");
    if (!(lr > 0) || !std::isfinite(lr)) return set_err(UTR_E_INVALID, "utr_corr_train_step: lr must be positive");
    const utr::CrVol V = cr_crops(c, d_in);
    const CrCubes Q = cr_cubes(c->T, c->halo);
    if (int rc = cr_forward(c, nb, V, Q)) return rc;
    if (int rc = cr_backward(c, nb, V, Q, d_tgt)) return rc;
    c->step++;
    const double b1 = 0.9, b2 = 0.999;
    const double lr_t = lr * std::sqrt(1.0 - std::pow(b2, c->step)) / (1.0 - std::pow(b1, c->step));
    utr::k_cr_adam<<<cr_blocks(c->np), 256, 0, c->st>>>(c->w.p, c->g.p, c->m.p, c->v.p, c->np, (float)lr_t, (float)b1,
                                                        (float)b2, 1e-8f);
    UTR_HIP_TRY(hipGetLastError());
    if (int rc = cr_repack(c)) return rc;
    // returns with the step done, so the caller may reuse the crop buffers
    float res[20];
    UTR_HIP_TRY(hipMemcpyAsync(res, c->res.p, sizeof(res), hipMemcpyDeviceToHost, c->st));
    UTR_HIP_TRY(hipStreamSynchronize(c->st));
    if (loss) *loss = res[18];
    return UTR_OK;
}

int utr_corr_apply(utr_corr* c, const float* d_vol, float* d_out, int nx, int ny, int nz) {
    if (int rc = cr_check(c)) return rc;
    if (!d_vol || !d_out || d_vol == d_out) return set_err(UTR_E_INVALID, "utr_corr_apply: distinct input and output");
    if (nx < 1 || ny < 1 || nz < 1) return set_err(UTR_E_INVALID, "utr_corr_apply: sizes must be positive");
    const int ntx = (nx + c->tile - 1) / c->tile, nty = (ny + c->tile - 1) / c->tile, ntz = (nz + c->tile - 1) / c->tile;
    const int ntiles = ntx * nty * ntz;
    const CrCubes Q = cr_cubes(c->T, c->halo);
    utr::CrVol V = cr_crops(c, d_vol);
    V.nx = nx;
    V.ny = ny;
    V.nz = nz;
    V.tile = c->tile;
    V.halo = c->halo;
    V.ntx = ntx;
    V.nty = nty;
    for (int first = 0; first < ntiles; first += c->batch) {
        const int nb = std::min(c->batch, ntiles - first);
        V.first = first;
        if (int rc = cr_forward(c, nb, V, Q)) return rc;
        if (int rc = cr_head(c, nb, V, Q, d_out, 1.f / c->scale)) return rc;
    }
    UTR_HIP_TRY(hipStreamSynchronize(c->st));
    return UTR_OK;
}

int utr_corr_destroy(utr_corr* c) {
    if (!c) return UTR_OK;
    (void)hipSetDevice(c->device);
    if (c->st) {
        (void)hipStreamSynchronize(c->st);
        (void)hipStreamDestroy(c->st);
    }
    for (auto& Ly : c->L) {
        Ly.wf.release();
        Ly.wb.release();
    }
    DevBuf<bf16_t>* bb[] = {&c->e1a, &c->e1b, &c->p1, &c->e2a, &c->e2b, &c->p2, &c->e3a, &c->e3b, &c->d2a, &c->d2b,
                            &c->d1a, &c->gd1b, &c->gd1a, &c->ge1b, &c->gd2b, &c->gd2a, &c->ge2b, &c->ge3b, &c->ge3a,
                            &c->gp2, &c->ge2a, &c->gp1, &c->ge1a};
    for (auto* b : bb) b->release();
    DevBuf<float>* fb[] = {&c->w, &c->g, &c->m, &c->v, &c->res, &c->part, &c->hpart};
    for (auto* b : fb) b->release();
    c->wfirst.release();
    delete c;
    return UTR_OK;
}

}  // extern "C"
