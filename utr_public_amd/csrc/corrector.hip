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

// BF16 <-> FP32 (round to nearest even; NaN stays NaN)
__host__ __device__ __forceinline__ float cr_bf2f(unsigned short h) {
    union { unsigned u; float f; } v;
    v.u = (unsigned)h << 16;
    return v.f;
}
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

struct CrConv {
    const unsigned short* in;  // cin channels at channel offset in_co of rows of in_cs halves
    int in_cs, in_co, cin;
    const uint4* wf;           // weight fragments (k_cr_pack), nbt blocks of 16 output channels
    int nbt;
    const float* bias;         // may be null
    int relu;                  // max(0, .) after the bias
    const unsigned short* mask;  // may be null: multiply by (mask > 0) at the output voxel and channel
    int mask_cs, mask_co;
    unsigned short* out;
    int out_cs, out_co;
    CrShape s;
};

constexpr int CR_Z = 4;  // output planes of a work-group's block

// 3x3x3 convolution, stride 1, zero padding 1, as an implicit GEMM: output
// channels are the matrix rows, 16 voxels (a 4 x 4 patch of one z plane) its
// columns, K = 32 is two (dy, dx) taps of 16 input channels.  A work-group of
// four waves owns PX x PY patches in x and y, CR_Z planes in z and NB blocks of
// 16 output channels (from blockIdx.y * NB); each wave takes PX PY / 4 patches
// through all planes.
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
template <int PX, int PY, int NB>
__global__ void __launch_bounds__(256) k_cr_conv(CrConv A) {
    constexpr int HX = 4 * PX + 2, HY = 4 * PY + 2, HZ = CR_Z + 2;
    constexpr int PITCH = 4 * PX + 4, HALF = HZ * HY * PITCH + 4;  // 16-byte units; HALF = 4 mod 8
    constexpr int NV = HX * HY * HZ, P = PX * PY / 4;
    constexpr int PER = (2 * NV + 255) / 256;
    static_assert(PITCH % 8 == 4 && HALF % 8 == 4, "bank layout");
    __shared__ __align__(16) uint4 xs[2 * HALF];
    const CrShape s = A.s;
    const int bxn = (s.w + 4 * PX - 1) / (4 * PX), byn = (s.h + 4 * PY - 1) / (4 * PY),
              bzn = (s.d + CR_Z - 1) / CR_Z;
    int tile, nb0;
    if (!xcd_tile(bxn * byn * bzn * s.n, A.nbt / NB, tile, nb0)) return;
    nb0 *= NB;
    const int x0 = tile % bxn * (4 * PX); tile /= bxn;
    const int y0 = tile % byn * (4 * PY); tile /= byn;
    const int z0 = tile % bzn * CR_Z;
    const int b = tile / bzn;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int m = lane & 15, kq = lane >> 4, mx = m & 3, my = m >> 2;
    cr_f4 acc[P][CR_Z][NB];
#pragma unroll
    for (int p = 0; p < P; p++)
#pragma unroll
        for (int z = 0; z < CR_Z; z++)
#pragma unroll
            for (int nb = 0; nb < NB; nb++) acc[p][z][nb] = cr_f4{0.f, 0.f, 0.f, 0.f};
    // this lane's fragment address for each tap pair (tap 9 of the last pair
    // does not exist: it reads tap 8's voxel and is set to zero)
    int fa[5];
#pragma unroll
    for (int q = 0; q < 5; q++) {
        const int t = min(2 * q + (kq >> 1), 8);
        fa[q] = (kq & 1) * HALF + (my + t / 3) * PITCH + mx + t % 3;
    }
    const int nslice = A.cin >> 4;
    const uint4* wp = A.wf + lane;
    for (int c = 0; c < nslice; c++) {
        uint4 val[PER];
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int t = (int)threadIdx.x + 256 * k, v = t >> 1;
            const int gx = x0 - 1 + v % HX, gy = y0 - 1 + (v / HX) % HY, gz = z0 - 1 + v / (HX * HY);
            val[k] = uint4{0u, 0u, 0u, 0u};
            if (t < 2 * NV && (unsigned)gx < (unsigned)s.w && (unsigned)gy < (unsigned)s.h &&
                (unsigned)gz < (unsigned)s.d)
                val[k] = *reinterpret_cast<const uint4*>(A.in + cr_vox(s, b, gz, gy, gx) * A.in_cs + A.in_co +
                                                         c * 16 + (t & 1) * 8);
        }
        if (c) __syncthreads();
#pragma unroll
        for (int k = 0; k < PER; k++) {
            const int t = (int)threadIdx.x + 256 * k, v = t >> 1;
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
#pragma unroll
            for (int p = 0; p < P; p++) {
                const int pid = wave * P + p;
                const uint4* r = xs + fa[q] + (pid / PX) * 4 * PITCH + (pid % PX) * 4;
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
                            acc[p][z][nb] =
                                __builtin_amdgcn_mfma_f32_16x16x32_bf16(w[dz][nb], xf, acc[p][z][nb], 0, 0, 0);
                    }
                }
            }
        }
    }
    // D[row = 4 kq + i][col = m]: channel 16 nb + 4 kq + i of the patch's voxel m
#pragma unroll
    for (int p = 0; p < P; p++) {
        const int pid = wave * P + p;
        const int x = x0 + (pid % PX) * 4 + mx, y = y0 + (pid / PX) * 4 + my;
#pragma unroll
        for (int z = 0; z < CR_Z; z++) {
            if (x >= s.w || y >= s.h || z0 + z >= s.d) continue;
            const size_t vox = cr_vox(s, b, z0 + z, y, x);
#pragma unroll
            for (int nb = 0; nb < NB; nb++) {
                const int ch = (nb0 + nb) * 16 + 4 * kq;
                float v[4];
#pragma unroll
                for (int i = 0; i < 4; i++) v[i] = acc[p][z][nb][i];
                if (A.bias) {
                    const float4 bv = *reinterpret_cast<const float4*>(A.bias + ch);
                    v[0] += bv.x; v[1] += bv.y; v[2] += bv.z; v[3] += bv.w;
                }
                if (A.relu) {
#pragma unroll
                    for (int i = 0; i < 4; i++) v[i] = fmaxf(v[i], 0.f);
                }
                if (A.mask) {
                    const uint2 mv = *reinterpret_cast<const uint2*>(A.mask + vox * A.mask_cs + A.mask_co + ch);
                    const unsigned h[4] = {mv.x & 0xffffu, mv.x >> 16, mv.y & 0xffffu, mv.y >> 16};
#pragma unroll
                    for (int i = 0; i < 4; i++)
                        if (!(h[i] != 0 && (h[i] & 0x8000u) == 0)) v[i] = 0.f;
                }
                *reinterpret_cast<uint2*>(A.out + vox * A.out_cs + A.out_co + ch) = cr_pack4(v);
            }
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
__global__ void __launch_bounds__(CR_WT) k_cr_wgrad(const unsigned short* __restrict__ in, int in_cs, int in_co,
                                                    int cin, const unsigned short* __restrict__ dy, int dy_cs,
                                                    int dy_co, int cout, float* __restrict__ part, CrShape s, int lo,
                                                    int hi, int G) {
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
            if (gx >= 0 && gx < s.w && gy >= 0 && gy < s.h && gz >= 0 && gz < s.d)
                val = *reinterpret_cast<const uint4*>(in + cr_vox(s, b, gz, gy, gx) * in_cs + in_co + c * 16 +
                                                      half * 8);
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
                    val = *reinterpret_cast<const uint4*>(dy + cr_vox(s, b, gz, gy, gx) * dy_cs + dy_co + o0 +
                                                          nb * 16 + half * 8);
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

// Sum of the G partial gradients of n values into grad.  A work-group takes
// 64 values, four threads a value with a quarter of the partials each; every
// quarter and the four quarters are added in order, so the sum is the same in
// every run.
__global__ void __launch_bounds__(256) k_cr_reduce(const float* __restrict__ part, int G, size_t n,
                                                   float* __restrict__ grad) {
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
    if (q == 0 && t < n) grad[t] = ((red[0][l] + red[1][l]) + red[2][l]) + red[3][l];
}

// 2 x 2 x 2 average pooling: out (c channels) from in at half resolution.
__global__ void k_cr_pool(const unsigned short* __restrict__ in, int in_cs, int in_co,
                          unsigned short* __restrict__ out, int out_cs, int out_co, int c, CrShape so) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nvox = (size_t)so.n * so.d * so.h * so.w;
    if (t >= nvox * c) return;
    const int ch = (int)(t % c);
    size_t v = t / c;
    const int x = (int)(v % so.w); v /= so.w;
    const int y = (int)(v % so.h); v /= so.h;
    const int z = (int)(v % so.d);
    const int b = (int)(v / so.d);
    const int W = 2 * so.w, H = 2 * so.h, D = 2 * so.d;
    float sum = 0.f;
    for (int k = 0; k < 8; k++) {
        const int xx = 2 * x + (k & 1), yy = 2 * y + ((k >> 1) & 1), zz = 2 * z + (k >> 2);
        sum += cr_bf2f(in[((((size_t)b * D + zz) * H + yy) * W + xx) * in_cs + in_co + ch]);
    }
    out[(t / c) * out_cs + out_co + ch] = cr_f2bf(0.125f * sum);
}

// Backward of the pooling added to the fine gradient, times the ReLU mask
// of the pooled activation: g[v][c] = (g[v][c] + gc[v/2][c] / 8) * (act > 0).
__global__ void k_cr_pool_bwd(unsigned short* __restrict__ gf, int g_cs, int g_co,
                              const unsigned short* __restrict__ gc, int gc_cs, int gc_co,
                              const unsigned short* __restrict__ act, int a_cs, int a_co, int c, CrShape sf) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nvox = (size_t)sf.n * sf.d * sf.h * sf.w;
    if (t >= nvox * c) return;
    const int ch = (int)(t % c);
    size_t v = t / c;
    const size_t vf = v;
    const int x = (int)(v % sf.w); v /= sf.w;
    const int y = (int)(v % sf.h); v /= sf.h;
    const int z = (int)(v % sf.d);
    const int b = (int)(v / sf.d);
    const size_t vc = (((size_t)b * (sf.d / 2) + z / 2) * (sf.h / 2) + y / 2) * (sf.w / 2) + x / 2;
    const unsigned short a = act[vf * a_cs + a_co + ch];
    float val = cr_bf2f(gf[vf * g_cs + g_co + ch]) + 0.125f * cr_bf2f(gc[vc * gc_cs + gc_co + ch]);
    if (!(a != 0 && (a & 0x8000u) == 0)) val = 0.f;
    gf[vf * g_cs + g_co + ch] = cr_f2bf(val);
}

// Nearest 2x upsampling: out (fine, c channels) from in (coarse).
__global__ void k_cr_up(const unsigned short* __restrict__ in, int in_cs, int in_co,
                        unsigned short* __restrict__ out, int out_cs, int out_co, int c, CrShape sf) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nvox = (size_t)sf.n * sf.d * sf.h * sf.w;
    if (t >= nvox * c) return;
    const int ch = (int)(t % c);
    size_t v = t / c;
    const size_t vf = v;
    const int x = (int)(v % sf.w); v /= sf.w;
    const int y = (int)(v % sf.h); v /= sf.h;
    const int z = (int)(v % sf.d);
    const int b = (int)(v / sf.d);
    const size_t vc = (((size_t)b * (sf.d / 2) + z / 2) * (sf.h / 2) + y / 2) * (sf.w / 2) + x / 2;
    out[vf * out_cs + out_co + ch] = in[vc * in_cs + in_co + ch];
}

// Backward of the upsampling: gc[u][c] = sum of the 8 fine gradients.
__global__ void k_cr_up_bwd(const unsigned short* __restrict__ gf, int g_cs, int g_co,
                            unsigned short* __restrict__ gc, int gc_cs, int gc_co, int c, CrShape sc) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t nvox = (size_t)sc.n * sc.d * sc.h * sc.w;
    if (t >= nvox * c) return;
    const int ch = (int)(t % c);
    size_t v = t / c;
    const int x = (int)(v % sc.w); v /= sc.w;
    const int y = (int)(v % sc.h); v /= sc.h;
    const int z = (int)(v % sc.d);
    const int b = (int)(v / sc.d);
    const int W = 2 * sc.w, H = 2 * sc.h, D = 2 * sc.d;
    float sum = 0.f;
    for (int k = 0; k < 8; k++) {
        const int xx = 2 * x + (k & 1), yy = 2 * y + ((k >> 1) & 1), zz = 2 * z + (k >> 2);
        sum += cr_bf2f(gf[((((size_t)b * D + zz) * H + yy) * W + xx) * g_cs + g_co + ch]);
    }
    gc[(t / c) * gc_cs + gc_co + ch] = cr_f2bf(sum);
}

// Network input: FP32 crops [n][T][T][T] -> x0 (BF16, 16 channels, the value
// times scale in channel 0) and x0f (FP32, the value times scale).
__global__ void k_cr_input(const float* __restrict__ vol, float scale, size_t nvox,
                           unsigned short* __restrict__ x0, float* __restrict__ x0f) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nvox) return;
    const float v = vol[t] * scale;
    x0f[t] = v;
    uint4 z = {0u, 0u, 0u, 0u};
    z.x = cr_f2bf(v);
    *reinterpret_cast<uint4*>(x0 + t * 16) = z;
    *reinterpret_cast<uint4*>(x0 + t * 16 + 8) = uint4{0u, 0u, 0u, 0u};
}

// Head: out = alpha * x0f + b1 + sum_c w1[c] * act[c]  (FP32); hp = {w1[16], b1, alpha}.
__global__ void k_cr_head(const unsigned short* __restrict__ act, const float* __restrict__ x0f,
                          const float* __restrict__ hp, size_t nvox, float* __restrict__ out) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= nvox) return;
    float s = hp[16] + hp[17] * x0f[t];
#pragma unroll
    for (int c = 0; c < 16; c++) s += hp[c] * cr_bf2f(act[t * 16 + c]);
    out[t] = s;
}

// Loss and head backward over the central tile^3 of every T^3 crop
// (halo h): L = sum (out - tgt)^2 / count; g = 2 (out - tgt) / count there and
// 0 in the halo; gact[v][c] = g w1[c] (act > 0); per work-group partial sums
// part[wg][20] = {dw1[16], db1, dalpha, loss, 0}.  Work-groups walk the voxels
// in strides of the grid (CR_HEADG of them), each lane keeping its own sums;
// lanes are added by a fixed shuffle tree, then the waves in order.
constexpr int CR_HEADG = 1024;
__global__ void __launch_bounds__(256) k_cr_head_bwd(const unsigned short* __restrict__ act,
                                                     const float* __restrict__ x0f, const float* __restrict__ out,
                                                     const float* __restrict__ tgt, const float* __restrict__ hp,
                                                     int T, int halo, size_t nvox, float inv_count,
                                                     unsigned short* __restrict__ gact, float* __restrict__ part) {
    __shared__ float red[4][20];
    float w1[16], loc[19];
#pragma unroll
    for (int c = 0; c < 16; c++) w1[c] = hp[c];
#pragma unroll
    for (int k = 0; k < 19; k++) loc[k] = 0.f;
    for (size_t t = (size_t)blockIdx.x * 256 + threadIdx.x; t < nvox; t += (size_t)gridDim.x * 256) {
        const int x = (int)(t % T), y = (int)((t / T) % T), z = (int)((t / ((size_t)T * T)) % T);
        const bool in = x >= halo && x < T - halo && y >= halo && y < T - halo && z >= halo && z < T - halo;
        const float d = out[t] - tgt[t];
        const float g = in ? 2.f * d * inv_count : 0.f;
        uint4 w[2], av4[2];
        unsigned short* wp = reinterpret_cast<unsigned short*>(w);
        const unsigned short* ap = reinterpret_cast<const unsigned short*>(av4);
        av4[0] = *reinterpret_cast<const uint4*>(act + t * 16);
        av4[1] = *reinterpret_cast<const uint4*>(act + t * 16 + 8);
#pragma unroll
        for (int c = 0; c < 16; c++) {
            const unsigned short a = ap[c];
            loc[c] += g * cr_bf2f(a);
            wp[c] = cr_f2bf((a != 0 && (a & 0x8000u) == 0) ? g * w1[c] : 0.f);
        }
        *reinterpret_cast<uint4*>(gact + t * 16) = w[0];
        *reinterpret_cast<uint4*>(gact + t * 16 + 8) = w[1];
        loc[16] += g;
        loc[17] += g * x0f[t];
        loc[18] += in ? d * d * inv_count : 0.f;
    }
#pragma unroll
    for (int k = 0; k < 19; k++) {
        for (int o = 32; o > 0; o >>= 1) loc[k] += __shfl_xor(loc[k], o);
        if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6][k] = loc[k];
    }
    __syncthreads();
    if (threadIdx.x < 20) {
        const int k = threadIdx.x;
        part[(size_t)blockIdx.x * 20 + k] = k < 19 ? ((red[0][k] + red[1][k]) + red[2][k]) + red[3][k] : 0.f;
    }
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

// Tiles of a volume for inference: crop b of the (tz, ty, tx) tile grid
// covers [t0 - halo, t0 + tile + halo) per axis, zeros outside the volume.
__global__ void k_cr_gather(const float* __restrict__ vol, int nx, int ny, int nz, int tile, int halo,
                            int ntx, int nty, int first, int nb, float* __restrict__ crops) {
    const int T = tile + 2 * halo;
    const size_t per = (size_t)T * T * T;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= per * nb) return;
    const int b = (int)(t / per);
    size_t r = t % per;
    const int x = (int)(r % T), y = (int)((r / T) % T), z = (int)(r / ((size_t)T * T));
    const int id = first + b;
    const int tx = id % ntx, ty = (id / ntx) % nty, tz = id / (ntx * nty);
    const int gx = tx * tile - halo + x, gy = ty * tile - halo + y, gz = tz * tile - halo + z;
    float v = 0.f;
    if (gx >= 0 && gx < nx && gy >= 0 && gy < ny && gz >= 0 && gz < nz) v = vol[((size_t)gz * ny + gy) * nx + gx];
    crops[t] = v;
}

// Central tile^3 of each output crop back into the volume (divided by scale).
__global__ void k_cr_scatter(const float* __restrict__ crops, int nx, int ny, int nz, int tile, int halo,
                             int ntx, int nty, int first, int nb, float inv_scale, float* __restrict__ vol) {
    const int T = tile + 2 * halo;
    const size_t per = (size_t)tile * tile * tile;
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t >= per * nb) return;
    const int b = (int)(t / per);
    size_t r = t % per;
    const int x = (int)(r % tile), y = (int)((r / tile) % tile), z = (int)(r / ((size_t)tile * tile));
    const int id = first + b;
    const int tx = id % ntx, ty = (id / ntx) % nty, tz = id / (ntx * nty);
    const int gx = tx * tile + x, gy = ty * tile + y, gz = tz * tile + z;
    if (gx >= nx || gy >= ny || gz >= nz) return;
    const size_t src = (size_t)b * T * T * T + ((size_t)(z + halo) * T + (y + halo)) * T + (x + halo);
    vol[((size_t)gz * ny + gy) * nx + gx] = crops[src] * inv_scale;
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
    {16, 16},  // e1b  -> C1[32:48]
    {16, 32},  // e2a  (input: pooled e1b)
    {32, 32},  // e2b  -> C2[64:96]
    {32, 64},  // e3a  (input: pooled e2b)
    {64, 64},  // e3b
    {96, 32},  // d2a  (input: C2 = up(e3b) | e2b)
    {32, 32},  // d2b
    {48, 16},  // d1a  (input: C1 = up(d2b) | e1b)
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
    DevBuf<bf16_t> x0, e1a, C1, p1, e2a, C2, p2, e3a, e3b, d2a, d2b, d1a, d1b;
    DevBuf<float> x0f, out;
    // activation gradients
    DevBuf<bf16_t> gd1b, gd1a, gC1, gd2b, gd2a, gC2, ge3b, ge3a, gp2, ge2a, gp1, ge1a;
    DevBuf<float> part, hpart, crops_in, crops_out;
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

// Blocks of 16 x 8 voxels in x and y where they make at least two work-groups
// per CU, 8 x 8 otherwise (the coarsest level of a few crops).
template <int PX, int PY>
int cr_conv_launch(utr_corr* c, const utr::CrConv& A) {
    const auto& s = A.s;
    const unsigned tiles = (unsigned)(s.n * ((s.w + 4 * PX - 1) / (4 * PX)) * ((s.h + 4 * PY - 1) / (4 * PY)) *
                                      ((s.d + utr::CR_Z - 1) / utr::CR_Z));
    const int nb = A.nbt % 3 == 0 ? 3 : A.nbt % 2 == 0 ? 2 : 1;
    const unsigned grid = utr::xcd_grid(tiles * (unsigned)(A.nbt / nb));
    if (nb == 3) utr::k_cr_conv<PX, PY, 3><<<grid, 256, 0, c->st>>>(A);
    else if (nb == 2) utr::k_cr_conv<PX, PY, 2><<<grid, 256, 0, c->st>>>(A);
    else utr::k_cr_conv<PX, PY, 1><<<grid, 256, 0, c->st>>>(A);
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

int cr_conv(utr_corr* c, int layer, bool fwd, const bf16_t* in, int in_cs, int in_co, bf16_t* out, int out_cs,
            int out_co, const bf16_t* mask, int mask_cs, int mask_co, utr::CrShape s) {
    const CrLayer& Ly = c->L[layer];
    utr::CrConv A;
    A.in = in;
    A.in_cs = in_cs;
    A.in_co = in_co;
    A.cin = fwd ? Ly.cin : Ly.cout;
    A.nbt = (fwd ? Ly.cout : Ly.cin) / 16;
    A.wf = fwd ? Ly.wf.p : Ly.wb.p;
    A.bias = fwd ? c->w.p + Ly.boff : nullptr;
    A.relu = fwd ? 1 : 0;
    A.mask = mask;
    A.mask_cs = mask_cs;
    A.mask_co = mask_co;
    A.out = out;
    A.out_cs = out_cs;
    A.out_co = out_co;
    A.s = s;
    const long big = (long)s.n * ((s.w + 15) / 16) * ((s.h + 7) / 8) * ((s.d + 3) / 4);
    return big >= 512 ? cr_conv_launch<4, 2>(c, A) : cr_conv_launch<2, 2>(c, A);
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

// dy is zero outside [lo, hi)^3.
int cr_wgrad(utr_corr* c, int layer, const bf16_t* in, int in_cs, int in_co, const bf16_t* dy, int dy_cs,
             int dy_co, utr::CrShape s, int lo, int hi) {
    const CrLayer& Ly = c->L[layer];
    const size_t nw = (size_t)27 * Ly.cin * Ly.cout + Ly.cout;
    const int no = cr_wgrad_no(Ly.cout), G = cr_wgrad_groups(Ly.cin, Ly.cout, s.n, hi - lo);
    if ((size_t)G * nw > c->part.n) return set_err(UTR_E_STATE, "corrector: gradient workspace too small");
    const dim3 grid(G, Ly.cin / 16, Ly.cout / 16 / no);
    if (no == 2)
        utr::k_cr_wgrad<2><<<grid, utr::CR_WT, 0, c->st>>>(in, in_cs, in_co, Ly.cin, dy, dy_cs, dy_co, Ly.cout,
                                                           c->part.p, s, lo, hi, G);
    else
        utr::k_cr_wgrad<1><<<grid, utr::CR_WT, 0, c->st>>>(in, in_cs, in_co, Ly.cin, dy, dy_cs, dy_co, Ly.cout,
                                                           c->part.p, s, lo, hi, G);
    UTR_HIP_TRY(hipGetLastError());
    // weights and bias of a layer are contiguous in the gradient vector
    utr::k_cr_reduce<<<(unsigned)((nw + 63) / 64), 256, 0, c->st>>>(c->part.p, G, nw, c->g.p + Ly.woff);
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
    const hipError_t e[] = {
        c->x0.alloc(n1 * 16), c->e1a.alloc(n1 * 16), c->C1.alloc(n1 * 48), c->p1.alloc(n2 * 16),
        c->e2a.alloc(n2 * 32), c->C2.alloc(n2 * 96), c->p2.alloc(n3 * 32), c->e3a.alloc(n3 * 64),
        c->e3b.alloc(n3 * 64), c->d2a.alloc(n2 * 32), c->d2b.alloc(n2 * 32), c->d1a.alloc(n1 * 16),
        c->d1b.alloc(n1 * 16), c->x0f.alloc(n1), c->out.alloc(n1),
        c->gd1b.alloc(n1 * 16), c->gd1a.alloc(n1 * 16), c->gC1.alloc(n1 * 48), c->gd2b.alloc(n2 * 32),
        c->gd2a.alloc(n2 * 32), c->gC2.alloc(n2 * 96), c->ge3b.alloc(n3 * 64), c->ge3a.alloc(n3 * 64),
        c->gp2.alloc(n3 * 32), c->ge2a.alloc(n2 * 32), c->gp1.alloc(n2 * 16), c->ge1a.alloc(n1 * 16),
        c->part.alloc(cr_part_size()), c->hpart.alloc((size_t)utr::CR_HEADG * 20), c->res.alloc(32),
        c->crops_in.alloc(n1), c->crops_out.alloc(n1)};
    for (hipError_t x : e)
        if (x != hipSuccess)
            return set_err(x == hipErrorOutOfMemory ? UTR_E_NOMEM : UTR_E_DEVICE,
                           std::string("corrector: device allocation failed: ") + hipGetErrorString(x));
    return UTR_OK;
}

int cr_repack(utr_corr* c) {
    for (int l = 0; l < 10; l++) {
        CrLayer& Ly = c->L[l];
        const size_t nf = (size_t)(Ly.cin / 16) * utr::CR_STEPS * (Ly.cout / 16) * 64;
        utr::k_cr_pack<<<cr_blocks(nf), 256, 0, c->st>>>(c->w.p + Ly.woff, Ly.cin, Ly.cout, 1, Ly.wf.p);
        UTR_HIP_TRY(hipGetLastError());
        utr::k_cr_pack<<<cr_blocks(nf), 256, 0, c->st>>>(c->w.p + Ly.woff, Ly.cin, Ly.cout, 0, Ly.wb.p);
        UTR_HIP_TRY(hipGetLastError());
    }
    return UTR_OK;
}

// Forward pass of nb crops already in x0 / x0f; result in c->out.
int cr_forward(utr_corr* c, int nb) {
    const int T = c->T;
    const utr::CrShape s1 = cr_shape(nb, T), s2 = cr_shape(nb, T / 2), s3 = cr_shape(nb, T / 4);
    const size_t n1 = (size_t)nb * T * T * T, n2 = n1 / 8, n3 = n1 / 64;
    int rc;
    if ((rc = cr_conv(c, 0, true, c->x0.p, 16, 0, c->e1a.p, 16, 0, nullptr, 0, 0, s1))) return rc;
    if ((rc = cr_conv(c, 1, true, c->e1a.p, 16, 0, c->C1.p, 48, 32, nullptr, 0, 0, s1))) return rc;
    utr::k_cr_pool<<<cr_blocks(n2 * 16), 256, 0, c->st>>>(c->C1.p, 48, 32, c->p1.p, 16, 0, 16, s2);
    if ((rc = cr_conv(c, 2, true, c->p1.p, 16, 0, c->e2a.p, 32, 0, nullptr, 0, 0, s2))) return rc;
    if ((rc = cr_conv(c, 3, true, c->e2a.p, 32, 0, c->C2.p, 96, 64, nullptr, 0, 0, s2))) return rc;
    utr::k_cr_pool<<<cr_blocks(n3 * 32), 256, 0, c->st>>>(c->C2.p, 96, 64, c->p2.p, 32, 0, 32, s3);
    if ((rc = cr_conv(c, 4, true, c->p2.p, 32, 0, c->e3a.p, 64, 0, nullptr, 0, 0, s3))) return rc;
    if ((rc = cr_conv(c, 5, true, c->e3a.p, 64, 0, c->e3b.p, 64, 0, nullptr, 0, 0, s3))) return rc;
    utr::k_cr_up<<<cr_blocks(n2 * 64), 256, 0, c->st>>>(c->e3b.p, 64, 0, c->C2.p, 96, 0, 64, s2);
    if ((rc = cr_conv(c, 6, true, c->C2.p, 96, 0, c->d2a.p, 32, 0, nullptr, 0, 0, s2))) return rc;
    if ((rc = cr_conv(c, 7, true, c->d2a.p, 32, 0, c->d2b.p, 32, 0, nullptr, 0, 0, s2))) return rc;
    utr::k_cr_up<<<cr_blocks(n1 * 32), 256, 0, c->st>>>(c->d2b.p, 32, 0, c->C1.p, 48, 0, 32, s1);
    if ((rc = cr_conv(c, 8, true, c->C1.p, 48, 0, c->d1a.p, 16, 0, nullptr, 0, 0, s1))) return rc;
    if ((rc = cr_conv(c, 9, true, c->d1a.p, 16, 0, c->d1b.p, 16, 0, nullptr, 0, 0, s1))) return rc;
    utr::k_cr_head<<<cr_blocks(n1), 256, 0, c->st>>>(c->d1b.p, c->x0f.p, c->w.p + c->headoff, n1, c->out.p);
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

// Loss and gradients of nb crops after cr_forward, targets in tgt (FP32,
// already scaled); gradient vector in c->g, {dw1, db1, dalpha, loss} in res.
int cr_backward(utr_corr* c, int nb, const float* tgt) {
    const int T = c->T;
    const utr::CrShape s1 = cr_shape(nb, T), s2 = cr_shape(nb, T / 2), s3 = cr_shape(nb, T / 4);
    const size_t n1 = (size_t)nb * T * T * T, n2 = n1 / 8, n3 = n1 / 64;
    const double cnt = (double)nb * c->tile * c->tile * c->tile;
    const unsigned hb = std::min(cr_blocks(n1), (unsigned)utr::CR_HEADG);
    int rc;
    utr::k_cr_head_bwd<<<hb, 256, 0, c->st>>>(c->d1b.p, c->x0f.p, c->out.p, tgt, c->w.p + c->headoff, T, c->halo, n1,
                                              (float)(1.0 / cnt), c->gd1b.p, c->hpart.p);
    UTR_HIP_TRY(hipGetLastError());
    utr::k_cr_head_reduce<<<1, 640, 0, c->st>>>(c->hpart.p, (int)hb, kCrHead, c->res.p, c->g.p + c->headoff);
    UTR_HIP_TRY(hipGetLastError());
    // The loss covers [halo, T - halo)^3, so each layer's output gradient is
    // zero outside that cube grown by one voxel per convolution behind it
    // (halved, rounded outwards, at each coarser level); its weight gradient
    // contracts over that cube only.
    struct Cube {
        int lo, hi;
    };
    auto grow = [](Cube q, int e) { return Cube{std::max(0, q.lo - 1), std::min(e, q.hi + 1)}; };
    auto half = [](Cube q) { return Cube{q.lo / 2, (q.hi + 1) / 2}; };
    const Cube q9 = {c->halo, T - c->halo}, q8 = grow(q9, T), qC1 = grow(q8, T);
    const Cube q7 = half(qC1), q6 = grow(q7, T / 2), qC2 = grow(q6, T / 2);
    const Cube q5 = half(qC2), q4 = grow(q5, T / 4), qp2 = grow(q4, T / 4);
    const Cube q3 = {std::min(qC2.lo, 2 * qp2.lo), std::max(qC2.hi, 2 * qp2.hi)};
    const Cube q2 = grow(q3, T / 2), qp1 = grow(q2, T / 2);
    const Cube q1 = {std::min(qC1.lo, 2 * qp1.lo), std::max(qC1.hi, 2 * qp1.hi)}, q0 = grow(q1, T);
    // d1b, d1a
    if ((rc = cr_wgrad(c, 9, c->d1a.p, 16, 0, c->gd1b.p, 16, 0, s1, q9.lo, q9.hi))) return rc;
    if ((rc = cr_conv(c, 9, false, c->gd1b.p, 16, 0, c->gd1a.p, 16, 0, c->d1a.p, 16, 0, s1))) return rc;
    if ((rc = cr_wgrad(c, 8, c->C1.p, 48, 0, c->gd1a.p, 16, 0, s1, q8.lo, q8.hi))) return rc;
    if ((rc = cr_conv(c, 8, false, c->gd1a.p, 16, 0, c->gC1.p, 48, 0, c->C1.p, 48, 0, s1))) return rc;
    // up(d2b) -> d2b, d2a
    utr::k_cr_up_bwd<<<cr_blocks(n2 * 32), 256, 0, c->st>>>(c->gC1.p, 48, 0, c->gd2b.p, 32, 0, 32, s2);
    if ((rc = cr_wgrad(c, 7, c->d2a.p, 32, 0, c->gd2b.p, 32, 0, s2, q7.lo, q7.hi))) return rc;
    if ((rc = cr_conv(c, 7, false, c->gd2b.p, 32, 0, c->gd2a.p, 32, 0, c->d2a.p, 32, 0, s2))) return rc;
    if ((rc = cr_wgrad(c, 6, c->C2.p, 96, 0, c->gd2a.p, 32, 0, s2, q6.lo, q6.hi))) return rc;
    if ((rc = cr_conv(c, 6, false, c->gd2a.p, 32, 0, c->gC2.p, 96, 0, c->C2.p, 96, 0, s2))) return rc;
    // up(e3b) -> e3b, e3a
    utr::k_cr_up_bwd<<<cr_blocks(n3 * 64), 256, 0, c->st>>>(c->gC2.p, 96, 0, c->ge3b.p, 64, 0, 64, s3);
    if ((rc = cr_wgrad(c, 5, c->e3a.p, 64, 0, c->ge3b.p, 64, 0, s3, q5.lo, q5.hi))) return rc;
    if ((rc = cr_conv(c, 5, false, c->ge3b.p, 64, 0, c->ge3a.p, 64, 0, c->e3a.p, 64, 0, s3))) return rc;
    if ((rc = cr_wgrad(c, 4, c->p2.p, 32, 0, c->ge3a.p, 64, 0, s3, q4.lo, q4.hi))) return rc;
    if ((rc = cr_conv(c, 4, false, c->ge3a.p, 64, 0, c->gp2.p, 32, 0, nullptr, 0, 0, s3))) return rc;
    // pool(e2b) -> e2b (skip and pooled paths), e2a
    utr::k_cr_pool_bwd<<<cr_blocks(n2 * 32), 256, 0, c->st>>>(c->gC2.p, 96, 64, c->gp2.p, 32, 0, c->C2.p, 96, 64, 32,
                                                               s2);
    if ((rc = cr_wgrad(c, 3, c->e2a.p, 32, 0, c->gC2.p, 96, 64, s2, q3.lo, q3.hi))) return rc;
    if ((rc = cr_conv(c, 3, false, c->gC2.p, 96, 64, c->ge2a.p, 32, 0, c->e2a.p, 32, 0, s2))) return rc;
    if ((rc = cr_wgrad(c, 2, c->p1.p, 16, 0, c->ge2a.p, 32, 0, s2, q2.lo, q2.hi))) return rc;
    if ((rc = cr_conv(c, 2, false, c->ge2a.p, 32, 0, c->gp1.p, 16, 0, nullptr, 0, 0, s2))) return rc;
    // pool(e1b) -> e1b, e1a
    utr::k_cr_pool_bwd<<<cr_blocks(n1 * 16), 256, 0, c->st>>>(c->gC1.p, 48, 32, c->gp1.p, 16, 0, c->C1.p, 48, 32, 16,
                                                               s1);
    if ((rc = cr_wgrad(c, 1, c->e1a.p, 16, 0, c->gC1.p, 48, 32, s1, q1.lo, q1.hi))) return rc;
    if ((rc = cr_conv(c, 1, false, c->gC1.p, 48, 32, c->ge1a.p, 16, 0, c->e1a.p, 16, 0, s1))) return rc;
    if ((rc = cr_wgrad(c, 0, c->x0.p, 16, 0, c->ge1a.p, 16, 0, s1, q0.lo, q0.hi))) return rc;
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

int cr_load_crops(utr_corr* c, const float* d_in, int nb) {
    const size_t n1 = (size_t)nb * c->T * c->T * c->T;
    utr::k_cr_input<<<cr_blocks(n1), 256, 0, c->st>>>(d_in, c->scale, n1, c->x0.p, c->x0f.p);
    UTR_HIP_TRY(hipGetLastError());
    return UTR_OK;
}

// Target crops scaled like the input, into crops_out (reused as scratch).
__global__ void k_cr_scale_copy(const float* __restrict__ src, float s, size_t n, float* __restrict__ dst) {
    const size_t t = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < n) dst[t] = src[t] * s;
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
    if (int rc = cr_load_crops(c, d_in, nb)) return rc;
    if (int rc = cr_forward(c, nb)) return rc;
    const size_t n1 = (size_t)nb * c->T * c->T * c->T;
    k_cr_scale_copy<<<cr_blocks(n1), 256, 0, c->st>>>(c->out.p, 1.f / c->scale, n1, d_out);
    UTR_HIP_TRY(hipGetLastError());
    UTR_HIP_TRY(hipStreamSynchronize(c->st));
    return UTR_OK;
}

int utr_corr_gradient(utr_corr* c, const float* d_in, const float* d_tgt, int nb, float* loss, float* grad_host) {
    if (int rc = cr_check(c)) return rc;
    if (!d_in || !d_tgt || nb < 1 || nb > c->batch)
        return set_err(UTR_E_INVALID, "utr_corr_gradient: 1 <= nb <= batch crops");
    const size_t n1 = (size_t)nb * c->T * c->T * c->T;
    if (int rc = cr_load_crops(c, d_in, nb)) return rc;
    k_cr_scale_copy<<<cr_blocks(n1), 256, 0, c->st>>>(d_tgt, c->scale, n1, c->crops_out.p);
    UTR_HIP_TRY(hipGetLastError());
    if (int rc = cr_forward(c, nb)) return rc;
    if (int rc = cr_backward(c, nb, c->crops_out.p)) return rc;
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
    const size_t n1 = (size_t)nb * c->T * c->T * c->T;
    if (int rc = cr_load_crops(c, d_in, nb)) return rc;
    k_cr_scale_copy<<<cr_blocks(n1), 256, 0, c->st>>>(d_tgt, c->scale, n1, c->crops_out.p);
    UTR_HIP_TRY(hipGetLastError());
    if (int rc = cr_forward(c, nb)) return rc;
    if (int rc = cr_backward(c, nb, c->crops_out.p)) return rc;
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
    const size_t per = (size_t)c->T * c->T * c->T;
    for (int first = 0; first < ntiles; first += c->batch) {
        const int nb = std::min(c->batch, ntiles - first);
        utr::k_cr_gather<<<cr_blocks(per * nb), 256, 0, c->st>>>(d_vol, nx, ny, nz, c->tile, c->halo, ntx, nty, first,
                                                                 nb, c->crops_in.p);
        UTR_HIP_TRY(hipGetLastError());
        if (int rc = cr_load_crops(c, c->crops_in.p, nb)) return rc;
        if (int rc = cr_forward(c, nb)) return rc;
        const size_t pt = (size_t)c->tile * c->tile * c->tile;
        utr::k_cr_scatter<<<cr_blocks(pt * nb), 256, 0, c->st>>>(c->out.p, nx, ny, nz, c->tile, c->halo, ntx, nty,
                                                                 first, nb, 1.f / c->scale, d_out);
        UTR_HIP_TRY(hipGetLastError());
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
    DevBuf<bf16_t>* bb[] = {&c->x0, &c->e1a, &c->C1, &c->p1, &c->e2a, &c->C2, &c->p2, &c->e3a, &c->e3b,
                            &c->d2a, &c->d2b, &c->d1a, &c->d1b, &c->gd1b, &c->gd1a, &c->gC1, &c->gd2b,
                            &c->gd2a, &c->gC2, &c->ge3b, &c->ge3a, &c->gp2, &c->ge2a, &c->gp1, &c->ge1a};
    for (auto* b : bb) b->release();
    DevBuf<float>* fb[] = {&c->w, &c->g, &c->m, &c->v, &c->res, &c->x0f, &c->out, &c->part, &c->hpart,
                           &c->crops_in, &c->crops_out};
    for (auto* b : fb) b->release();
    delete c;
    return UTR_OK;
}

}  // extern "C"
